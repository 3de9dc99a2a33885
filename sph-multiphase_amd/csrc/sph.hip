// WCSPH neighbour loops: boundary volume, density + equation of state,
// pressure/viscosity acceleration, symplectic-Euler advance.
// Reference: fluid_system_kern.cu:183-534 (ComputeBoundaryVolume,
// ComputeDensityPressure, ComputeForce, AdvanceParticles) launched by
// fluid_system_host.cu:337-438,510-513.
//
// Kernel family 0 is the reference's poly6/spiky pair with support h
// (fluid_system.cpp:309-312); family 1 swaps in the cubic spline with
// support 2h (kern.cu:637-671) for the dam-break configuration.
#include "nbr.hpp"
#include "rounding.hpp"
#include "wc_rules.hpp"

#include <type_traits>

namespace sphx {

__device__ __forceinline__ float poly6_c3(float r2, float dsq) {
  float c = r2 - dsq;
  return c * c * c;
}

// ComputeBoundaryVolume (kern.cu:249-277): V_b = 1 / (k * sum_b w)
__global__ void k_boundary_volume(KP k, const uint32_t* __restrict__ key,
                                  const int* __restrict__ cs, const float4* __restrict__ pos,
                                  float4* __restrict__ phys) {
  int i = xcd_index();
  if (i >= k.n) return;
  float4 pi = pos[i];
  if (type_of(pi) != SPHX_TYPE_BOUNDARY) return;
  uint32_t gc = key[i];
  if ((int)gc == k.gridtotal) return;
  float sum = 0.f;
  const bool cubic = k.wcsph_kernel == 1;
  for_each_neighbor(k, cs, gc, [&](int j) {
    float4 pj = pos[j];
    if (type_of(pj) != SPHX_TYPE_BOUNDARY) return;
    float dx = (pi.x - pj.x) * k.ss, dy = (pi.y - pj.y) * k.ss, dz = (pi.z - pj.z) * k.ss;
    float dsq = dx * dx + dy * dy + dz * dz;
    if (cubic) {
      sum += cubic_w(sqrtf(dsq), k.inv_h, k.kspline);
    } else if (dsq < k.h2) {
      sum += poly6_c3(k.h2, dsq);
    }
  });
  if (!cubic) sum *= k.kpoly6;
  if (sum == 0.f) sum = 1.f;
  phys[i].y = 1.f / sum;
}

// ---- density and force: L lanes of a wave per particle ----
//
// One thread per particle leaves most of the chip idle below some 100k
// particles and walks its thousand candidates as one serial chain of loads
// (C1's 50k particles: 555 us density, 940 us force).  Here L consecutive
// lanes share a particle: they test its candidates L at a time (a row of
// cells is one contiguous run of the sorted arrays, so the loads coalesce)
// into a hit list in LDS, sum the density over the hits, and leave the list
// in memory for the force pass, which then visits neighbours only.
constexpr int WC_THREADS = 256;
constexpr int WC_WAVES = WC_THREADS / 64;
constexpr int WC_BATCH = 4;   // candidate loads in flight (8: the same time)
// A list entry: neighbour row r (0..8) in the top 4 bits, offset from the
// row's first particle (its dx = -1 cell) in the low 12.
constexpr uint32_t WC_OFF_MAX = 4095;

struct WcList {
  uint16_t* __restrict__ idx;   // [n][cap]
  int* __restrict__ cnt;        // entries; WC_SCAN: no list, scan the cells;
                                // NBR_INVALID: boundary or outside the grid
  int cap;                      // entries per particle, a multiple of 8
};
constexpr int WC_SCAN = -1;

// LDS written by some lanes of a wave and read by others of the same wave.
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <int L>
__device__ __forceinline__ float lanes_sum(float v) {
#pragma unroll
  for (int o = L / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, L);
  return v;
}

// Inclusive sums over L consecutive lanes, by DPP: within rows of 16, then
// the first row's total into the second.
template <int L>
__device__ __forceinline__ int lanes_scan(int v) {
  static_assert(L == 16 || L == 32, "rows of 16");
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);   // row_shr:1
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);
  if (L == 32) v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);   // row_bcast:15
  return v;
}

// Support of the WCSPH kernel family, squared, in stored position units.
__host__ __device__ __forceinline__ float wc_reach2(const KP& k) {
  return (k.wcsph_kernel == 1 ? 4.f * k.h2 : k.h2) / (k.ss * k.ss);
}

// r = |x| and 1/r from r^2, and a / b, rounded as IEEE operations round them
// (rounding.hpp); r of 0 is 0, of a value that is no number that value.
__device__ __forceinline__ void wc_dist(float dsq, float& r, float& ir) {
  const float y = __builtin_amdgcn_rsqf(dsq);
  r = dsq > 0.f ? refine_sqrt(dsq, y) : dsq;
  ir = refine_rcp(r, y);
}
__device__ __forceinline__ float wc_div(float a, float b) {
  return refine_div(a, b, refine_rcp(b, __builtin_amdgcn_rcpf(b)));
}

// The density pass's weight of one neighbour (poly6 without its constant).
__device__ __forceinline__ float wc_weight(const KP& k, bool cubic, float dsq) {
  if (!cubic) {
    // 0 outside the support, and for a distance that is no number
    const float c = fmaxf(k.h2 - dsq, 0.f);
    return c * c * c;
  }
  float r, ir;
  wc_dist(dsq, r, ir);
  return cubic_w(r, k.inv_h, k.kspline);
}

// ComputeDensityPressure (kern.cu:214-318).  Stores 1/rho in dens.  With
// DENSITY false only the list is built; with a capacity of 0 none is and every
// particle scans its cells.  Particles from `first` on.  `prune`: the keys describe the
// current positions, so of the 27 cells only those that the support
// overlaps can hold neighbours (8 for the support h, half a cell wide).
template <int L, bool DENSITY>
__global__ __launch_bounds__(WC_THREADS) void k_wc_density(
    KP k, int first, WcList W, const uint32_t* __restrict__ key, const int* __restrict__ cs,
    const float4* __restrict__ pos, float4* __restrict__ phys, int prune, float3 rad) {
  constexpr int P = 64 / L;   // particles per wave
  extern __shared__ __align__(16) uint16_t wc_q[];
  // by row: its first particle; by reached row: its candidates' begin and
  // end, and which it is
  __shared__ int rows[WC_WAVES][P][4][9];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int g = lane / L, sub = lane % L;
  const int i = first + (xcd_tile() * WC_WAVES + wave) * P + g;
  uint16_t* __restrict__ q = wc_q + (size_t)(wave * P + g) * W.cap;
  int(*__restrict__ rw)[9] = rows[wave][g];
  float4 pi = make_float4(0.f, 0.f, 0.f, 0.f);
  uint32_t gc = 0;
  bool act = false;
  if (i < k.n) {
    pi = pos[i];
    gc = key[i];
    act = type_of(pi) != SPHX_TYPE_BOUNDARY && (int)gc != k.gridtotal;
  }
  const float reach2 = wc_reach2(k);
  int nrow = 0;
  if (act) {
    // Cells d = 0..2 of each axis that hold candidates: with `prune` those
    // the support overlaps, from the place inside the key's cell.
    int x0 = 0, x1 = 2, y0 = 0, ny = 3, z0 = 0, nz = 3;
    if (prune) {
      const float ux = (pi.x - k.gridmin.x) * k.gridfac.x, uy = (pi.y - k.gridmin.y) * k.gridfac.y,
                  uz = (pi.z - k.gridmin.z) * k.gridfac.z;
      const float fx = ux - (float)(int)ux, fy = uy - (float)(int)uy, fz = uz - (float)(int)uz;
      x0 = fx > rad.x;
      x1 = 1 + (fx + rad.x >= 1.f);
      y0 = fy > rad.y;
      ny = 2 + (fy + rad.y >= 1.f) - y0;
      z0 = fz > rad.z;
      nz = 2 + (fz + rad.z >= 1.f) - z0;
    }
    nrow = ny * nz;
    if (sub < nrow) {
      const int yy = sub >= nz ? (sub >= 2 * nz ? 2 : 1) : 0;
      const int r = (y0 + yy) * 3 + z0 + sub - yy * nz;
      const int c0 = (int)gc + k.rowoff[r];
      rw[0][r] = cs[c0];
      rw[1][sub] = cs[c0 + x0];
      rw[2][sub] = cs[c0 + x1 + 1];
      rw[3][sub] = r;
    }
  }
  wave_lds_sync();
  int cnt = 0;
  bool over = W.cap == 0;
  if (act && !over) {
    // The rows' candidates, up to 32 per lane at a time, tested WC_BATCH by
    // WC_BATCH (loads in flight together) into a hit mask: a test enters at
    // bit 0 and moves up; its bit is the sign of d2 - reach2, which is
    // d2 < reach2 exactly.
#pragma unroll 1
    for (int a = 0; a < nrow; ++a) {
      const int r = rw[3][a], base = rw[0][r], jb = rw[1][a], je = rw[2][a];
      over |= je - base > (int)WC_OFF_MAX + 1;
#pragma unroll 1
      for (int j0 = jb; j0 < je; j0 += 32 * L) {
        const int mb = (min(32, (je - j0 + L - 1) / L) + WC_BATCH - 1) & ~(WC_BATCH - 1);
        const int mine = min(32, max(0, (je - j0 - sub + L - 1) / L));
        uint32_t hit = 0;
#pragma unroll 1
        for (int u = 0; u < mb; u += WC_BATCH) {
          float4 pj[WC_BATCH];
#pragma unroll
          for (int v = 0; v < WC_BATCH; ++v)
            pj[v] = load_at(pos, (uint32_t)min(j0 + sub + (u + v) * L, k.n - 1) * 16u);
#pragma unroll
          for (int v = 0; v < WC_BATCH; ++v) {
            const float dx = pi.x - pj[v].x, dy = pi.y - pj[v].y, dz = pi.z - pj[v].z;
            hit = __builtin_amdgcn_alignbit(hit, __float_as_uint(pair_dsq(dx, dy, dz) - reach2), 31);
          }
        }
        hit = mine > 0 ? hit >> (mb - mine) : 0u;   // candidate u now at bit mine - 1 - u
        const int c = __popc(hit);
        const int incl = lanes_scan<L>(c);
        int at = cnt + incl - c;
        cnt += __shfl(incl, L - 1, L);
        const uint32_t tag = ((uint32_t)r << 12) + (uint32_t)(j0 + sub - base);
        while (hit) {
          const int b = 31 - __builtin_clz(hit);
          hit ^= 1u << b;
          if (at < W.cap) q[at] = (uint16_t)(tag + (uint32_t)((mine - 1 - b) * L));
          ++at;
        }
      }
    }
    over |= cnt > W.cap;
  }
  wave_lds_sync();
  if (i < k.n && sub == 0) W.cnt[i] = !act ? NBR_INVALID : (over ? WC_SCAN : cnt);
  if (!act) return;   // whole groups of L lanes
  if (!over) {
    uint16_t* __restrict__ out = W.idx + (size_t)i * W.cap;
    for (int t = sub * 8; t < cnt; t += L * 8)
      *reinterpret_cast<uint4*>(out + t) = *reinterpret_cast<const uint4*>(q + t);
  }
  if (!DENSITY) return;
  float4 qi = phys[i];
  const float rest = qi.w;
  const bool cubic = k.wcsph_kernel == 1;
  float sum = 0.f;
  auto add = [&](const float4& pj, const float4& qj, bool use) {
    // boundary: rho0_i * V_j; any other type uses its own mass (A5)
    const float mj = type_of(pj) == SPHX_TYPE_BOUNDARY ? rest * qj.y : qj.x;
    const float dx = (pi.x - pj.x) * k.ss, dy = (pi.y - pj.y) * k.ss, dz = (pi.z - pj.z) * k.ss;
    const float w = wc_weight(k, cubic, pair_dsq(dx, dy, dz));
    sum += use && w > 0.f ? w * mj : 0.f;
  };
  if (!over) {
    // whole batches of 4 a lane, then what is left
    auto batch = [&](int t, auto whole) {
      constexpr bool W = decltype(whole)::value;
      float4 pj[4], qj[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        if (W || t + u * L < cnt) {
          const uint32_t e = q[t + u * L];
          const uint32_t j = (uint32_t)rw[0][e >> 12] + (e & WC_OFF_MAX);
          pj[u] = load_at(pos, j * 16u);
          qj[u] = load_at(phys, j * 16u);
        } else {
          pj[u] = qj[u] = make_float4(0.f, 0.f, 0.f, 0.f);
        }
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) add(pj[u], qj[u], W || t + u * L < cnt);
    };
    int t0 = 0;
    for (; t0 + 4 * L <= cnt; t0 += 4 * L) batch(t0 + sub, std::true_type{});
    if (t0 < cnt) batch(t0 + sub, std::false_type{});
  } else {
    for (int a = 0; a < nrow; ++a)
      for (int j = rw[1][a] + sub; j < rw[2][a]; j += L) add(pos[j], phys[j], true);
  }
  sum = lanes_sum<L>(sum);
  if (!cubic) sum *= k.kpoly6;
  if (sum == 0.f) sum = 1.f;
  float B = k.eos_B > 0.f ? k.eos_B : 2.5f * rest;
  float x = sum / rest;
  float xp;
  if (k.eos_gamma == 7.f) {
    float x2 = x * x, x4 = x2 * x2;
    xp = x4 * x2 * x;
  } else {
    xp = powf(x, k.eos_gamma);
  }
  float p = B * (xp - 1.f);
  if (p < 0.f) p = 0.f;
  qi.y = 1.f / sum;
  qi.z = p;
  if (sub == 0) phys[i] = qi;
}

// ComputeForce + contributeForce_new (kern.cu:325-424) over the list of the
// density pass, L lanes per particle.
template <int L>
__global__ __launch_bounds__(WC_THREADS) void k_wc_force(
    KP k, int first, WcList W, const uint32_t* __restrict__ key, const int* __restrict__ cs,
    const float4* __restrict__ pos, const float4* __restrict__ vel,
    const float4* __restrict__ phys, float4* __restrict__ accel) {
  constexpr int P = 64 / L;
  __shared__ int rows[WC_WAVES][P][9];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int g = lane / L, sub = lane % L;
  const int i = first + (xcd_tile() * WC_WAVES + wave) * P + g;
  int* __restrict__ rw = rows[wave][g];
  const int cnt = i < k.n ? W.cnt[i] : NBR_INVALID;
  const bool act = cnt != NBR_INVALID;
  const uint32_t gc = act ? key[i] : 0u;
  if (act)
    for (int r = sub; r < 9; r += L) rw[r] = cs[(int)gc + k.rowoff[r]];
  wave_lds_sync();
  if (!act) return;   // whole groups of L lanes
  const float4 pi = pos[i];
  const float4 vi = vel[i];       // the reference reads vel as "iveleval" (:410)
  const float4 qi = phys[i];
  const float idens = qi.y, ipress = qi.z, irest = qi.w, ivisc = vi.w;
  const bool cubic = k.wcsph_kernel == 1;
  const float rsup2 = cubic ? 4.f * k.h2 : k.h2;
  const float fric = k.bvisc * k.h * 0.5f / irest;
  const float bpm = -irest * ipress * idens * idens;
  float fx = 0.f, fy = 0.f, fz = 0.f;
  auto add = [&](const float4& pj, const float4& qj, const float4& vj, bool use) {
    const float dx = (pi.x - pj.x) * k.ss, dy = (pi.y - pj.y) * k.ss, dz = (pi.z - pj.z) * k.ss;
    const float dsq = pair_dsq(dx, dy, dz);
    const int tj = type_of(pj);
    if (!(use && dsq < rsup2 && dsq > 0.f)) return;
    if (tj != SPHX_TYPE_FLUID && tj != SPHX_TYPE_BOUNDARY) return;
    float r, ir;
    wc_dist(dsq, r, ir);
    float cm1;   // grad W = dist * cm1
    if (cubic) {
      cm1 = cubic_gradf(r, ir, k.inv_h, k.kspline);
    } else {
      const float c = k.h - r;
      cm1 = refine_div(k.kspikydiff * c * c, r, ir);
    }
    const float vx = vi.x - vj.x, vy = vi.y - vj.y, vz = vi.z - vj.z;
    const float vdotx = vx * dx + vy * dy + vz * dz;
    // wall friction and artificial viscosity act on approaching pairs only
    const float mu = vdotx < 0.f ? wc_div(vdotx, dsq + 0.01f * k.h2) : 0.f;
    float s;
    if (tj == SPHX_TYPE_FLUID) {
      const float cm = cm1 * qj.x * qj.y;
      const float vm = cm * (ivisc + vj.w) * idens;
      s = -0.5f * cm * qj.z * idens;
      // Pi = -alpha c0 h mu / (mean rho), mean rho = (1/idens + 1/qj.y) / 2;
      // no density yet on either side: an infinite mean
      const float both = idens + qj.y;
      if (k.art_alpha > 0.f && mu < 0.f && both != 0.f)
        s += qj.x * cm1 * (k.art_alpha * k.c0 * k.h) * mu *
             wc_div(2.f * idens * qj.y, both);
      fx += vx * vm;
      fy += vy * vm;
      fz += vz * vm;
    } else {
      s = cm1 * qj.y * bpm;
      if (mu < 0.f) s += cm1 * qj.y * irest * fric * mu;
    }
    fx += dx * s;
    fy += dy * s;
    fz += dz * s;
  };
  if (cnt >= 0) {
    const uint16_t* __restrict__ in = W.idx + (size_t)i * W.cap;
    // whole batches of 4 a lane, then what is left
    auto batch = [&](int t, auto whole) {
      constexpr bool W = decltype(whole)::value;
      float4 pj[4], qj[4], vj[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        if (W || t + u * L < cnt) {
          const uint32_t e = in[t + u * L];
          const uint32_t j = (uint32_t)rw[e >> 12] + (e & WC_OFF_MAX);
          pj[u] = load_at(pos, j * 16u);
          qj[u] = load_at(phys, j * 16u);
          vj[u] = load_at(vel, j * 16u);
        } else {
          pj[u] = qj[u] = vj[u] = make_float4(0.f, 0.f, 0.f, 0.f);
        }
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) add(pj[u], qj[u], vj[u], W || t + u * L < cnt);
    };
    int t0 = 0;
    for (; t0 + 4 * L <= cnt; t0 += 4 * L) batch(t0 + sub, std::true_type{});
    if (t0 < cnt) batch(t0 + sub, std::false_type{});
  } else {
    for (int r = 0; r < 9; ++r) {
      const int je = cs[(int)gc + k.rowoff[r] + 3];
      for (int j = rw[r] + sub; j < je; j += L) add(pos[j], phys[j], vel[j], true);
    }
  }
  fx = lanes_sum<L>(fx);
  fy = lanes_sum<L>(fy);
  fz = lanes_sum<L>(fz);
  if (sub == 0) accel[i] = make_float4(fx, fy, fz, 0.f);
}

// AdvanceParticles (kern.cu:426-534)
__global__ void k_advance(KP k, const uint32_t* __restrict__ key, float4* __restrict__ pos,
                          float4* __restrict__ vel, float4* __restrict__ veleval,
                          const float4* __restrict__ accel) {
  int i = xcd_index();
  if (i >= k.n) return;
  float4 p = pos[i];
  if (type_of(p) == SPHX_TYPE_BOUNDARY) return;
  float4 v = vel[i];
  if ((int)key[i] == k.gridtotal) {
    p.x = p.y = p.z = -1000.f;
    pos[i] = p;
    vel[i] = make_float4(0.f, 0.f, 0.f, v.w);
    return;
  }
  float4 a = accel[i];
  float ax = a.x + k.g.x, ay = a.y + k.g.y, az = a.z + k.g.z;
  float nx = ax * k.dt + v.x, ny = ay * k.dt + v.y, nz = az * k.dt + v.z;
  p.x += nx * k.dt / k.ss;
  p.y += ny * k.dt / k.ss;
  p.z += nz * k.dt / k.ss;
  pos[i] = p;
  veleval[i] = make_float4((v.x + nx) * 0.5f, (v.y + ny) * 0.5f, (v.z + nz) * 0.5f, 0.f);
  vel[i] = make_float4(nx, ny, nz, v.w);
}


static int need_sorted(sphx_context* c, const char* who) {
  SPHX_CHECK(c, who, "null context");
  SPHX_TRY(ensure_device(c));
  SPHX_CHECK(c->sorted_valid, who, "grid not built (call sphx_grid_build first)");
  return 0;
}

static int wc_capacity(const sphx_context* c, const KP& k) {
  const double spacing = std::cbrt((double)c->P.mass / (double)c->P.restdensity) / (double)c->P.simscale;
  return wc_entries(c->num, spacing, std::sqrt((double)wc_reach2(k)),
                    c->O.wcsph_list_max);
}

static int wc_fit(sphx_context* c, const KP& k) {
  c->wl_valid = false;
  c->wl_cap = wc_capacity(c, k);
  SPHX_TRY(c->wl_cnt.alloc((size_t)c->cap));
  const size_t want = (size_t)c->cap * c->wl_cap;
  if (want == 0) return 0;
  // no room for the list: every particle scans its cells; what did not fit is
  // not tried again at each pass
  if ((c->wl_failed && want >= c->wl_failed) || !c->wl_idx.try_alloc(want)) {
    c->wl_failed = want;
    c->wl_cap = 0;
  }
  return 0;
}

// Lists of this capacity or more (135 expected neighbours: the cubic
// spline's support 2h) are "long".
constexpr int WC_LONG = 224;

// The density pass (or the list alone), after wc_fit.
template <bool DENSITY>
static void wc_density(sphx_context* c, const KP& k) {
  const WcList W{c->wl_idx.p, c->wl_cnt.p, c->wl_cap};
  const int most = std::max(k.gridres.x, std::max(k.gridres.y, k.gridres.z));
  const int prune = c->grid_fresh && most <= 16384;   // cell indices exact to 1/100 in float
  // the support in cells, with a slack of 1/100 cell that is far above the
  // rounding of a place in the grid
  const float reach = std::sqrt(wc_reach2(k));
  const float3 rad = make_float3(reach * k.gridfac.x + 0.01f, reach * k.gridfac.y + 0.01f,
                                 reach * k.gridfac.z + 0.01f);
  auto launch = [&](auto l) {
    constexpr int L = decltype(l)::value, per = WC_THREADS / L;
    wc_launches(k.n, [&](int first, int m) {
      k_wc_density<L, DENSITY>
          <<<blocks_for(m, per), WC_THREADS, (size_t)per * W.cap * sizeof(uint16_t), c->stream>>>(
              k, first, W, c->key.p, c->cell_start.p, c->POS(), c->PHYS(), prune, rad);
    });
  };
  // Lanes per particle, 4 to 64 measured (us): 65 neighbours among 1,000
  // candidates at 50k / 675k particles 78 73 56 51 65 / 789 742 674 614 832;
  // 268 among 1,728 at 50k / 675k: 122 80 78 78 90 / 1143 912 896 1017 1231
  // (550 at 630k and 75 at 50k since the two columns in use were tightened:
  // 310M vector instructions instead of 364M, the VALU 94 % busy, and
  // no gathers for lanes past a list's end, a tenth of the L1's accesses).
  if (W.cap >= WC_LONG) launch(std::integral_constant<int, 16>{});
  else launch(std::integral_constant<int, 32>{});
  c->wl_reach2 = wc_reach2(k);
  c->wl_valid = true;
}

}  // namespace sphx

using namespace sphx;

extern "C" {

int sphx_boundary_volume(sphx_context* c) {
  SPHX_TRY(need_sorted(c, "sphx_boundary_volume"));
  KP k = make_kp(c);
  if (k.n == 0) return 0;
  timer_begin(c, "boundary_volume");
  k_boundary_volume<<<blocks_for(k.n, 256), 256, 0, c->stream>>>(k, c->key.p, c->cell_start.p,
                                                                  c->POS(), c->PHYS());
  timer_end(c);
  c->gh_valid = false;   // boundary volumes enter the pressure pass's G_i
  SPHX_HIP(hipGetLastError());
  return 0;
}

int sphx_wcsph_density_pressure(sphx_context* c) {
  SPHX_TRY(need_sorted(c, "sphx_wcsph_density_pressure"));
  c->mf_stress_ok = false;   // phys.y changes
  KP k = make_kp(c);
  if (k.n == 0) return 0;
  SPHX_TRY(wc_fit(c, k));
  timer_begin(c, "wcsph_density");
  wc_density<true>(c, k);
  timer_end(c);
  SPHX_HIP(hipGetLastError());
  return 0;
}

int sphx_wcsph_force(sphx_context* c) {
  SPHX_TRY(need_sorted(c, "sphx_wcsph_force"));
  KP k = make_kp(c);
  if (k.n == 0) return 0;
  timer_begin(c, "wcsph_force");
  if (!c->wl_valid || c->wl_reach2 != wc_reach2(k)) {
    SPHX_TRY(wc_fit(c, k));
    wc_density<false>(c, k);
  }
  const WcList W{c->wl_idx.p, c->wl_cnt.p, c->wl_cap};
  auto launch = [&](auto l) {
    constexpr int L = decltype(l)::value;
    wc_launches(k.n, [&](int first, int m) {
      k_wc_force<L><<<blocks_for(m, WC_WAVES * (64 / L)), WC_THREADS, 0, c->stream>>>(
          k, first, W, c->key.p, c->cell_start.p, c->POS(), c->VEL(), c->PHYS(), c->ACCEL());
    });
  };
  // Lanes per particle, 4 / 8 / 16 / 32 measured (us, fluid without walls).  33
  // neighbours at 2.7k, 12k, 16k, 27k, 47k, 55k, 64k, 157k and 636k particles:
  // 8.3 6.6 4.7 4.4, 8.5 7.2 5.3 5.3, 8.6 7.3 5.8 6.8, 9.4 8.4 7.9 9.0, 10.4
  // 10.0 10.4 12.8, 11.5 12.9 11.5 14.4, 12 14 13 17, 26 29 30 41, 84 102 111
  // 166.  268 neighbours at 2.7k, 12k, 20k, 30k, 47k, 64k, 157k and 636k: 36 21
  // 13 10, 38 24 18 18, 42 30 26 28, 43 39 41 38, 58 57 58 58, 80 80 75 77, 184
  // 170 168 179, 760 683 688 770.  Many lanes until the chip is full, then as
  // few as leave a list in whole batches of 4 a lane.  The L1 binds (one access
  // a gathered lane, 1.0 a clock a CU), so only the lanes of a list's last batch
  // that have an entry gather (630k with walls: 174 -> 155; 50k with 268: 58 ->
  // 55).
  const bool longer = W.cap >= WC_LONG;
  if (k.n <= (longer ? 49152 : 12288)) launch(std::integral_constant<int, 32>{});
  else if (longer || k.n <= 49152) launch(std::integral_constant<int, 16>{});
  else launch(std::integral_constant<int, 4>{});
  timer_end(c);
  SPHX_HIP(hipGetLastError());
  return 0;
}

int sphx_wcsph_advance(sphx_context* c) {
  SPHX_TRY(need_sorted(c, "sphx_wcsph_advance"));
  KP k = make_kp(c);
  if (k.n == 0) return 0;
  positions_changed(c);
  timer_begin(c, "wcsph_advance");
  k_advance<<<blocks_for(k.n, 256), 256, 0, c->stream>>>(k, c->key.p, c->POS(), c->VEL(),
                                                          c->VELEVAL(), c->ACCEL());
  timer_end(c);
  SPHX_HIP(hipGetLastError());
  return 0;
}

int sphx_wcsph_step(sphx_context* c) {
  SPHX_CHECK(c, "sphx_wcsph_step", "null context");
  SPHX_TRY(ensure_device(c));
  SPHX_TRY(grid_build(c));
  SPHX_TRY(sphx_wcsph_density_pressure(c));
  SPHX_TRY(sphx_wcsph_force(c));
  return sphx_wcsph_advance(c);
}

}  // extern "C"
