// Stokesian mobility of spheres (SPH_Solver/stokesian/Mobility.cu).
//
// The polydisperse Rotne-Prager-Yamakawa mobility is applied to K
// right-hand sides, U = M F (M is 3N x 3N, row 3p + a), without storing M:
// each workgroup generates 64 x 32-sphere tiles of the 3x3 pair blocks on
// the VALU, splits them into bf16 pieces in LDS and multiplies them against
// the bf16 pieces of F on MFMA (v_mfma_f32_16x16x32_bf16, FP32
// accumulation).  The dominant self term M_ii = I/(6 pi mu a_i) is applied
// in FP32 outside the MFMA.  Precision modes:
//   1  hi*hi                                  (plain bf16)
//   3  hi*hi + hi*lo + lo*hi                  (bf16x3)
//   6  bf16x3 + lo*lo + hi*F3 + M3*hi         (second-order split terms)
// where x = hi + lo + x3 with each piece bf16 (round to nearest even).
// The reduction over spheres is split over `split` workgroups per row tile
// (partials in FP32, summed by a second kernel) so N = 4096 fills the chip.
//
// Also here: the reference's equal-sphere walkthrough (Kern_getForce
// :257-300, Kern_interpolateVelocity :322-366, Kern_getmobu_walkthrough
// :207-255) and the dense product getMobU (:85-109).
#include "common.hpp"

#include <type_traits>
#include <utility>
#include <vector>

namespace sphx {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;

constexpr int RPY_TP = 64;     // spheres per row tile (4 waves x 16)
constexpr int RPY_TQ = 32;     // spheres per reduction chunk (MFMA K)
constexpr int RPY_THREADS = 256;
constexpr float RPY_PI = 3.14159265358979f;

// round to nearest even to bf16 (finite inputs)
__host__ __device__ __forceinline__ uint16_t bf16_bits(float x) {
  uint32_t u;
  std::memcpy(&u, &x, 4);
  u += 0x7FFFu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}
__host__ __device__ __forceinline__ float bf16_float(uint16_t b) {
  uint32_t u = (uint32_t)b << 16;
  float f;
  std::memcpy(&f, &u, 4);
  return f;
}
// x = hi + lo + r3 (three bf16 pieces)
__device__ __forceinline__ void split3(float x, uint16_t& h, uint16_t& l, uint16_t& r) {
  h = bf16_bits(x);
  float d = x - bf16_float(h);
  l = bf16_bits(d);
  r = bf16_bits(d - bf16_float(l));
}

// F [3n][K] FP32 row-major -> the first `pieces` of FT[b][c][q] (sphere q
// contiguous), zero-padded to np spheres.  A workgroup transposes 16
// right-hand sides of 64 spheres' component b through LDS, so that F is read
// in runs of 64 bytes and written in runs of 128.
__global__ __launch_bounds__(256) void k_rpy_split_f(const float* __restrict__ F, int n, int np,
                                                     int K, int pieces, uint16_t* __restrict__ Fh,
                                                     uint16_t* __restrict__ Fl,
                                                     uint16_t* __restrict__ F3) {
  __shared__ float tile[RPY_TP][17];
  const int q0 = blockIdx.x * RPY_TP, b = blockIdx.y, c0 = blockIdx.z * 16;
  const int cl = threadIdx.x & 15;
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int ql = (threadIdx.x >> 4) + 16 * u, q = q0 + ql;
    tile[ql][cl] = q < n ? F[(3 * (size_t)q + b) * K + c0 + cl] : 0.f;
  }
  __syncthreads();
  const int ql = threadIdx.x & 63;
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int c = (threadIdx.x >> 6) + 4 * u;
    uint16_t h, l, r;
    split3(tile[ql][c], h, l, r);
    const size_t o = ((size_t)b * K + c0 + c) * np + q0 + ql;
    Fh[o] = h;
    if (pieces > 1) Fl[o] = l;
    if (pieces > 2) F3[o] = r;
  }
}

typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;

// Two floats to packed bf16 (element 0 in the low half), round to nearest
// even (v_cvt_pk_bf16_f32).
__device__ __forceinline__ uint32_t pk_bf16(float a, float b) {
  const bf16x2 v = {(__bf16)a, (__bf16)b};
  return __builtin_bit_cast(uint32_t, v);
}
// x0 = hi + lo + r3 and x1 likewise, the pieces of both packed per word.
__device__ __forceinline__ void split3_pk(float x0, float x1, uint32_t& h, uint32_t& l,
                                          uint32_t& r) {
  h = pk_bf16(x0, x1);
  const float d0 = x0 - __uint_as_float(h << 16), d1 = x1 - __uint_as_float(h & 0xFFFF0000u);
  l = pk_bf16(d0, d1);
  const float e0 = d0 - __uint_as_float(l << 16), e1 = d1 - __uint_as_float(l & 0xFFFF0000u);
  r = pk_bf16(e0, e1);
}

// The six distinct entries (00 11 22 01 02 12) of the polydisperse RPY
// pair block for spheres p = {x, y, z, a} and q, zero for q == p or
// outside the set.
__device__ __forceinline__ void rpy_pair(float4 sp, float4 sq, bool valid, float inv8pimu,
                                         float m[6]) {
#pragma unroll
  for (int k = 0; k < 6; ++k) m[k] = 0.f;
  if (!valid) return;
  const float dx = sq.x - sp.x, dy = sq.y - sp.y, dz = sq.z - sp.z;
  const float r2 = dx * dx + dy * dy + dz * dz;
  const float ir2 = 1.f / r2;
  const float c0 = inv8pimu * sqrtf(ir2);
  const float s2 = sp.w * sp.w + sq.w * sq.w;
  const float ci = c0 * (1.f + s2 * ir2 * (1.f / 3.f));
  const float cr = c0 * (1.f - s2 * ir2) * ir2;
  m[0] = ci + cr * dx * dx;
  m[1] = ci + cr * dy * dy;
  m[2] = ci + cr * dz * dz;
  m[3] = cr * dx * dy;
  m[4] = cr * dx * dz;
  m[5] = cr * dy * dz;
}

// Symmetric 3x3 block index: 00 11 22 01 02 12
__device__ __forceinline__ int sym_index(int a, int b) {
  if (a == b) return a;
  int lo = a < b ? a : b, hi = a < b ? b : a;
  return lo == 0 ? (hi == 1 ? 3 : 4) : 5;
}

__device__ __forceinline__ bf16x8 lds8(const uint16_t* p) {
  return *reinterpret_cast<const bf16x8*>(p);
}
__device__ __forceinline__ bf16x8 glb8(const uint16_t* p) {
  return *reinterpret_cast<const bf16x8*>(p);
}

// Partial products of the off-diagonal mobility for row tile blockIdx.x and
// reduction segment blockIdx.y: part[s][a][p][c].
// The pieces planes a precision mode multiplies: hi (mode 1), hi and lo
// (mode 3), all three (mode 6).
template <int MODE>
struct RpyPieces {
  static constexpr int N = MODE == 1 ? 1 : (MODE == 3 ? 2 : 3);
  uint16_t M[N][6][RPY_TP][RPY_TQ];
};

template <int MODE>
__global__ __launch_bounds__(RPY_THREADS, MODE == 1 ? 3 : 2) void k_rpy_tile(
    const float4* __restrict__ sph, int n, int np, float mu, int K, int seg,
    const uint16_t* __restrict__ Fh, const uint16_t* __restrict__ Fl,
    const uint16_t* __restrict__ F3, float* __restrict__ part) {
  constexpr int mode = MODE;
  __shared__ __align__(16) RpyPieces<MODE> P;
  auto& Mh = P.M[0];
  auto& Ml = P.M[MODE >= 3 ? 1 : 0];
  auto& M3 = P.M[MODE == 6 ? 2 : 0];
  const int p0 = blockIdx.x * RPY_TP;
  const int s = blockIdx.y;
  const int q_begin = s * seg, q_end = min(np, q_begin + seg);
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  // pair generation: thread -> spheres q0 + 2 (tid & 15) + {0, 1} and rows
  // p0 + (tid >> 4) + 16 t, t = 0..3; a wave writes 4 consecutive rows of
  // packed words (256 contiguous bytes per store)
  const int qp = 2 * (tid & 15), pr = tid >> 4;
  const float inv8pimu = 1.f / (8.f * RPY_PI * mu);
  // MFMA work of a wave: rows p0 + 32 wr .. +32 (two 16-row tiles) and
  // right-hand sides 32 wc .. +32 (two 16-column tiles), so each F piece is
  // loaded by two waves of the workgroup instead of four
  const int wr = wave & 1, wc = wave >> 1;
  f32x4 acc[3][2][2];
#pragma unroll
  for (int a = 0; a < 3; ++a)
#pragma unroll
    for (int rt = 0; rt < 2; ++rt)
#pragma unroll
      for (int ct = 0; ct < 2; ++ct) acc[a][rt][ct] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int ncb = K / 16;
  // the thread's four row spheres are the same for every chunk; the two
  // column spheres of the next chunk are fetched during this chunk's MFMAs
  float4 sp4[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const int gp = p0 + pr + 16 * t;
    sp4[t] = gp < n ? sph[gp] : make_float4(0.f, 0.f, 0.f, 1.f);
  }
  auto col = [&](int gq) { return gq < n ? sph[gq] : make_float4(0.f, 0.f, 0.f, 1.f); };
  float4 nq0 = col(q_begin + qp), nq1 = col(q_begin + qp + 1);
  for (int q0 = q_begin; q0 < q_end; q0 += RPY_TQ) {
    __syncthreads();
    {
      const int gq0 = q0 + qp, gq1 = gq0 + 1;
      const float4 sq0 = nq0, sq1 = nq1;
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int pl = pr + 16 * t, gp = p0 + pl;
        const float4 sp = sp4[t];
        float m0[6], m1[6];
        rpy_pair(sp, sq0, gp < n && gq0 < n && gq0 != gp, inv8pimu, m0);
        rpy_pair(sp, sq1, gp < n && gq1 < n && gq1 != gp, inv8pimu, m1);
#pragma unroll
        for (int k = 0; k < 6; ++k) {
          uint32_t h, l, r;
          split3_pk(m0[k], m1[k], h, l, r);
          *reinterpret_cast<uint32_t*>(&Mh[k][pl][qp]) = h;
          if (mode >= 3) *reinterpret_cast<uint32_t*>(&Ml[k][pl][qp]) = l;
          if (mode == 6) *reinterpret_cast<uint32_t*>(&M3[k][pl][qp]) = r;
        }
      }
    }
    __syncthreads();
    if (q0 + RPY_TQ < q_end) {
      nq0 = col(q0 + RPY_TQ + qp);
      nq1 = col(q0 + RPY_TQ + qp + 1);
    }
    // MFMA lane layout of v_mfma_f32_16x16x32_bf16: A row = lane % 16,
    // k = 8 (lane / 16) .. +8; B column = lane % 16, same k; D rows
    // 4 (lane / 16) + i, column lane % 16.
    const int kk = 8 * (lane >> 4);
    // all three b unrolled: their F loads issue together
#pragma unroll
    for (int b = 0; b < 3; ++b) {
      bf16x8 fh[2], fl[2], f3[2];
#pragma unroll
      for (int ct = 0; ct < 2; ++ct) {
        const int cb = 2 * wc + ct;
        if (cb >= ncb) break;
        size_t off = ((size_t)b * K + 16 * cb + (lane & 15)) * np + q0 + kk;
        fh[ct] = glb8(Fh + off);
        if (mode >= 3) fl[ct] = glb8(Fl + off);
        if (mode == 6) f3[ct] = glb8(F3 + off);
      }
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        const int k6 = sym_index(a, b);
#pragma unroll
        for (int rt = 0; rt < 2; ++rt) {
          const int arow = 32 * wr + 16 * rt + (lane & 15);
          bf16x8 ah = lds8(&Mh[k6][arow][kk]);
          bf16x8 al = lds8(&Ml[k6][arow][kk]);
          bf16x8 a3;
          if (mode == 6) a3 = lds8(&M3[k6][arow][kk]);
#pragma unroll
          for (int ct = 0; ct < 2; ++ct) {
            if (2 * wc + ct >= ncb) break;
            f32x4 c = acc[a][rt][ct];
            c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, fh[ct], c, 0, 0, 0);
            if (mode >= 3) {
              c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, fl[ct], c, 0, 0, 0);
              c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al, fh[ct], c, 0, 0, 0);
            }
            if (mode == 6) {
              c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al, fl[ct], c, 0, 0, 0);
              c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, f3[ct], c, 0, 0, 0);
              c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a3, fh[ct], c, 0, 0, 0);
            }
            acc[a][rt][ct] = c;
          }
        }
      }
    }
  }
  // partials: part[s][a][p][c]
#pragma unroll
  for (int a = 0; a < 3; ++a)
#pragma unroll
    for (int rt = 0; rt < 2; ++rt)
#pragma unroll
      for (int ct = 0; ct < 2; ++ct) {
        const int cb = 2 * wc + ct;
        if (cb >= ncb) break;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          int p = p0 + 32 * wr + 16 * rt + 4 * (lane >> 4) + i;
          int c = 16 * cb + (lane & 15);
          part[(((size_t)s * 3 + a) * np + p) * K + c] = acc[a][rt][ct][i];
        }
      }
}

// U[3p + a][c] = F/(6 pi mu a_p) + sum_s part[s][a][p][c]
__global__ void k_rpy_reduce(const float4* __restrict__ sph, int n, int np, float mu, int K,
                             int nseg, const float* __restrict__ F,
                             const float* __restrict__ part, float* __restrict__ U) {
  int t = blockIdx.x * blockDim.x + threadIdx.x;   // over 3 n K
  if (t >= 3 * n * K) return;
  int c = t % K, row = t / K, a = row % 3, p = row / 3;
  float v = F[t] / (6.f * RPY_PI * mu * sph[p].w);
  for (int s = 0; s < nseg; ++s) v += part[(((size_t)s * 3 + a) * np + p) * K + c];
  U[t] = v;
}

// ------------------------------------------------------------- reference --
// The walkthrough's two all-pairs sums (near-field force, mobility velocity
// and rotation).  One thread per sphere leaves 16 k spheres on 64 workgroups
// and walks all n partners as one serial chain.  Here a workgroup owns I
// spheres, whose positions are uniform (SGPRs); its threads split the
// partners, load each once for the I spheres, and the I sums are reduced
// over the workgroup at the end.  Bound by VALU issue: 44 instructions a pair
// for the mobility and 8.7 for the force, loads and loops included (counters
// at 16,384 spheres: VALU 122 and 97 % busy, at four clocks an instruction).
constexpr int WALK_THREADS = 256;

// Sums v[0..V) over the workgroup: out[k] (LDS) = sum of v[k].  Lanes first
// exchange halves of the values, so a wave needs about V shuffles and not
// 6 V; every thread calls it, and out is readable after it returns.
template <int V>
__device__ __forceinline__ void walk_reduce(float (&v)[V], float (*part)[V], float* out) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int at = 0;   // index of this lane's v[0] among the V sums
  constexpr int H0 = V % 64 == 0 ? 6 : V % 32 == 0 ? 5 : V % 16 == 0 ? 4 : V % 8 == 0 ? 3 : V % 4 == 0 ? 2 : V % 2 == 0 ? 1 : 0;
  constexpr int H = H0 < 6 ? H0 : 6;   // halving steps
  int n = V;
#pragma unroll
  for (int s = 0; s < H; ++s) {
    const int m = 32 >> s;
    n >>= 1;
    const bool up = (lane & m) != 0;
#pragma unroll
    for (int k = 0; k < (V >> (s + 1)); ++k) {
      const float lo = v[k], hi = v[k + (V >> (s + 1))];
      v[k] = (up ? hi : lo) + __shfl_xor(up ? lo : hi, m, 64);
    }
    at += up ? n : 0;
  }
#pragma unroll
  for (int s = H; s < 6; ++s)
#pragma unroll
    for (int k = 0; k < (V >> H); ++k) v[k] += __shfl_xor(v[k], 32 >> s, 64);
  if ((lane & ((64 >> H) - 1)) == 0)
#pragma unroll
    for (int k = 0; k < (V >> H); ++k) part[wave][at + k] = v[k];
  __syncthreads();
  for (int k = threadIdx.x; k < V; k += WALK_THREADS) {
    float t = 0.f;
    for (int q = 0; q < WALK_THREADS / 64; ++q) t += part[q][k];
    out[k] = t;
  }
  __syncthreads();
}

__device__ __forceinline__ float3 sphere_at(const sphx_displayPack* __restrict__ disp, int i) {
  return f3(disp[i].pos.x, disp[i].pos.y, disp[i].pos.z);
}

// The whole application in FP32 for few spheres, one launch: a workgroup
// owns I row spheres and 16 right-hand sides, its threads split the column
// spheres, and the sums are reduced as the walkthrough's.  About 184 lane
// operations a pair and 16 right-hand sides; the three launches of the tile
// path take about 10 us however few spheres there are.
template <int I>
__global__ __launch_bounds__(WALK_THREADS) void k_rpy_direct(const float4* __restrict__ sph, int n,
                                                             float mu, int K,
                                                             const float* __restrict__ F,
                                                             float* __restrict__ U) {
  constexpr int V = 48 * I;
  __shared__ float part[WALK_THREADS / 64][V], sum[V];
  const int i0 = blockIdx.x * I, c0 = blockIdx.y * 16;
  const float inv8pimu = 1.f / (8.f * RPY_PI * mu);
  float4 p[I];
  float acc[V];
#pragma unroll
  for (int k = 0; k < I; ++k) p[k] = sph[min(i0 + k, n - 1)];
#pragma unroll
  for (int k = 0; k < V; ++k) acc[k] = 0.f;
  for (int q = threadIdx.x; q < n; q += WALK_THREADS) {
    const float4 sq = sph[q];
    const float4* __restrict__ f4 = reinterpret_cast<const float4*>(F + 3 * (size_t)q * K + c0);
    float f[3][16];
#pragma unroll
    for (int b = 0; b < 3; ++b)
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const float4 x = f4[b * (K / 4) + u];
        f[b][4 * u] = x.x; f[b][4 * u + 1] = x.y; f[b][4 * u + 2] = x.z; f[b][4 * u + 3] = x.w;
      }
#pragma unroll
    for (int k = 0; k < I; ++k) {
      float m[6];
      rpy_pair(p[k], sq, q != i0 + k, inv8pimu, m);
      if (q == i0 + k) m[0] = m[1] = m[2] = 1.f / (6.f * RPY_PI * mu * sq.w);   // M_ii
#pragma unroll
      for (int a = 0; a < 3; ++a)
#pragma unroll
        for (int c = 0; c < 16; ++c)
          acc[(3 * k + a) * 16 + c] += m[sym_index(a, 0)] * f[0][c] + m[sym_index(a, 1)] * f[1][c] +
                                       m[sym_index(a, 2)] * f[2][c];
    }
  }
  walk_reduce<V>(acc, part, sum);
  for (int t = threadIdx.x; t < V; t += WALK_THREADS) {
    const int row = 3 * i0 + t / 16;
    if (row < 3 * n) U[(size_t)row * K + c0 + t % 16] = sum[t];
  }
}

// Kern_getForce (:257-300): near-field repulsion added to force.
template <int I>
__global__ __launch_bounds__(WALK_THREADS) void k_walk_force(
    const sphx_displayPack* __restrict__ disp, int n, sphx_float3* __restrict__ force) {
  __shared__ float part[WALK_THREADS / 64][3 * I], sum[3 * I];
  const int i0 = blockIdx.x * I;
  float3 p[I];
  float f[3 * I];
#pragma unroll
  for (int k = 0; k < I; ++k) {
    p[k] = sphere_at(disp, min(i0 + k, n - 1));
    f[3 * k] = f[3 * k + 1] = f[3 * k + 2] = 0.f;
  }
  const float actdist = 1.5f;
  int j = threadIdx.x;
  float3 q = sphere_at(disp, min(j, n - 1));
  for (; j < n; j += WALK_THREADS) {
    const float3 c = q;
    q = sphere_at(disp, min(j + WALK_THREADS, n - 1));   // the next partner
#pragma unroll
    for (int k = 0; k < I; ++k) {
      const float dx = c.x - p[k].x, dy = c.y - p[k].y, dz = c.z - p[k].z;
      const float d2 = dx * dx + dy * dy + dz * dz;
      if (d2 < actdist * actdist) {
        const float dr = sqrtf(d2);
        if (dr < actdist && j != i0 + k) {
          const float fac = 5.f * (expf(actdist / dr) - 2.7128f * dr / actdist);
          f[3 * k] -= dx * fac; f[3 * k + 1] -= dy * fac; f[3 * k + 2] -= dz * fac;
        }
      }
    }
  }
  walk_reduce<3 * I>(f, part, sum);
  const int i = i0 + (int)threadIdx.x;
  if ((int)threadIdx.x < I && i < n) {
    const float* t = sum + 3 * threadIdx.x;
    force[i].x += t[0]; force[i].y += t[1]; force[i].z += t[2];
  }
}

// Kern_interpolateVelocity (:322-366): trilinear background velocity from
// the MPM nodes ({v, m} per node).
__global__ void k_walk_background(const sphx_displayPack* __restrict__ disp, int n,
                                  const float4* __restrict__ nodev, float3 xmin, float cs,
                                  int3 res, float ss, sphx_float3* __restrict__ unew) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  float px = disp[i].pos.x - xmin.x, py = disp[i].pos.y - xmin.y, pz = disp[i].pos.z - xmin.z;
  int ix = (int)(px / cs), iy = (int)(py / cs), iz = (int)(pz / cs);
  float3 v = f3(0.f, 0.f, 0.f);
  for (int c = 0; c < 8; ++c) {
    int x = ix + (c & 1), y = iy + ((c >> 1) & 1), z = iz + (c >> 2);
    if (x < 0 || y < 0 || z < 0 || x >= res.x || y >= res.y || z >= res.z) continue;
    float w = (1.f - fabsf(px - x * cs) / cs) * (1.f - fabsf(py - y * cs) / cs) *
              (1.f - fabsf(pz - z * cs) / cs);
    float4 nv = nodev[((size_t)y * res.z + z) * res.x + x];
    v.x += nv.x * w; v.y += nv.y * w; v.z += nv.z * w;
  }
  unew[i] = {v.x / ss, v.y / ss, v.z / ss};
}

// Kern_getmobu_walkthrough (:207-255): U = U_bg + F + sum A1N F and
// Omega = sum B1N F with PairwiseMobMatrix (:37-82) for equal spheres a = 1:
// with d = x_j - x_i, r = |d| and e = d / r,
//   A1N F = X e (e . F) + Y (F - e (e . F)),  X = 1.5/r - 1/r^3, Y = 0.75/r + 0.5/r^3
//   B1N F = 0.75 / r^2 (e x F).
// Positions are advanced by k_walk_commit, after every workgroup has read
// them (the reference moves them in place while other threads read, A10).
template <int I>
__global__ __launch_bounds__(WALK_THREADS) void k_walk_mob(
    const sphx_displayPack* __restrict__ disp, int n, const sphx_float3* __restrict__ force,
    int background, sphx_float3* __restrict__ unew, sphx_float3* __restrict__ omega) {
  __shared__ float part[WALK_THREADS / 64][6 * I], sum[6 * I];
  const int i0 = blockIdx.x * I;
  float3 p[I];
  float a[6 * I];   // U and Omega of each sphere
#pragma unroll
  for (int k = 0; k < I; ++k) p[k] = sphere_at(disp, min(i0 + k, n - 1));
#pragma unroll
  for (int k = 0; k < 6 * I; ++k) a[k] = 0.f;
  int j = threadIdx.x;
  auto load = [&](int t, float3& q, float3& f) {
    const bool in = t < n;   // past the end: no force, far away
    q = in ? sphere_at(disp, t) : f3(1e15f, 0.f, 0.f);
    f = in ? f3(force[t].x, force[t].y, force[t].z) : f3(0.f, 0.f, 0.f);
  };
  auto pairs = [&](const float3& q, const float3& f, auto self) {
#pragma unroll
    for (int k = 0; k < I; ++k) {
      const float dx = q.x - p[k].x, dy = q.y - p[k].y, dz = q.z - p[k].z;
      float r2 = dx * dx + dy * dy + dz * dz;
      const bool me = decltype(self)::value && j == i0 + k;
      if (decltype(self)::value) r2 = me ? 1.f : r2;
      const float ir = __builtin_amdgcn_rsqf(r2), ir2 = ir * ir;
      float Y = ir * (0.75f + 0.5f * ir2);
      if (decltype(self)::value) Y = me ? 1.f : Y;   // d = 0: only U += F is left
      const float ir3 = ir * ir2;
      const float c = ir3 * (0.75f - 1.5f * ir2) * (dx * f.x + dy * f.y + dz * f.z);
      a[6 * k] += c * dx + Y * f.x;
      a[6 * k + 1] += c * dy + Y * f.y;
      a[6 * k + 2] += c * dz + Y * f.z;
      const float g = 0.75f * ir3;
      a[6 * k + 3] += g * (dy * f.z - dz * f.y);
      a[6 * k + 4] += g * (dz * f.x - dx * f.z);
      a[6 * k + 5] += g * (dx * f.y - dy * f.x);
    }
  };
  float3 q, f;
  load(j, q, f);
  // I divides the partners of one round, so the workgroup's own spheres all
  // meet themselves in the same round
  const int own = i0 / WALK_THREADS * WALK_THREADS;
  for (int j0 = 0; j0 < n; j0 += WALK_THREADS, j += WALK_THREADS) {
    const float3 cq = q, cf = f;
    load(j + WALK_THREADS, q, f);   // the next partner
    if (j0 == own) pairs(cq, cf, std::true_type{});
    else pairs(cq, cf, std::false_type{});
  }
  walk_reduce<6 * I>(a, part, sum);
  const int i = i0 + (int)threadIdx.x;
  if ((int)threadIdx.x < I && i < n) {
    const float* t = sum + 6 * threadIdx.x;
    const float3 bg = background ? f3(unew[i].x, unew[i].y, unew[i].z) : f3(0.f, 0.f, 0.f);
    unew[i] = {bg.x + t[0], bg.y + t[1], bg.z + t[2]};
    omega[i] = {t[3], t[4], t[5]};
  }
}

// x += U dt
__global__ void k_walk_commit(sphx_displayPack* __restrict__ disp, int n,
                              const sphx_float3* __restrict__ u, float dt) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float3 p = sphere_at(disp, i);
  disp[i].pos = {p.x + u[i].x * dt, p.y + u[i].y * dt, p.z + u[i].z * dt};
}

// MVmultiply (:85-98): one wave per row of the dense (6n x 6n) matrix.
__global__ void k_gemv(const float* __restrict__ mat, const float* __restrict__ f,
                       float* __restrict__ u, int dim) {
  int row = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  int lane = threadIdx.x & 63;
  if (row >= dim) return;
  const float* m = mat + (size_t)row * dim;
  double s = 0.0;
  for (int j = lane; j < dim; j += 64) s += (double)m[j] * (double)f[j];
  for (int off = 32; off > 0; off >>= 1) s += __shfl_down(s, off, 64);
  if (lane == 0) u[row] = (float)s;
}

}  // namespace sphx

using namespace sphx;

struct sphx_rpy {
  int n = 0, np = 0, K = 0, split = 0, device = 0;   // split 0: not set
  float mu = 1.f;
  hipStream_t stream = nullptr;
  sphx::DevBuf<float4> sph;
  sphx::DevBuf<uint16_t> Fh, Fl, F3;
  sphx::DevBuf<float> part, F, U;
  // tile-kernel timing: an event pair around each k_rpy_tile launch
  bool timing = false;
  std::vector<std::pair<hipEvent_t, hipEvent_t>> ev;
};

extern "C" {

int sphx_rpy_create(sphx_rpy** out, int n, int nrhs) {
  SPHX_CHECK(out, "sphx_rpy_create", "null argument");
  *out = nullptr;
  SPHX_CHECK(n > 0, "sphx_rpy_create", "n must be positive");
  SPHX_CHECK(nrhs > 0 && nrhs <= 64 && nrhs % 16 == 0, "sphx_rpy_create",
             "nrhs must be 16, 32, 48 or 64");
  int dev = 0;
  SPHX_HIP(hipGetDevice(&dev));
  sphx_rpy* h = new sphx_rpy;
  h->n = n;
  h->np = (n + RPY_TP - 1) / RPY_TP * RPY_TP;
  h->K = nrhs;
  h->device = dev;
  hipError_t e = hipStreamCreateWithFlags(&h->stream, hipStreamNonBlocking);
  if (e != hipSuccess) { delete h; return hip_fail("hipStreamCreate", e); }
  size_t fsz = 3 * (size_t)nrhs * h->np;
  int rc = 0;
  if ((rc = h->sph.alloc(h->np)) || (rc = h->Fh.alloc(fsz)) || (rc = h->Fl.alloc(fsz)) ||
      (rc = h->F3.alloc(fsz)) || (rc = h->F.alloc(3 * (size_t)n * nrhs)) ||
      (rc = h->U.alloc(3 * (size_t)n * nrhs))) {
    (void)hipStreamDestroy(h->stream);
    delete h;
    return rc;
  }
  *out = h;
  return 0;
}

static void rpy_drop_events(sphx_rpy* h) {
  for (auto& e : h->ev) {
    (void)hipEventDestroy(e.first);
    (void)hipEventDestroy(e.second);
  }
  h->ev.clear();
}

int sphx_rpy_destroy(sphx_rpy* h) {
  if (!h) return 0;
  (void)hipStreamSynchronize(h->stream);
  rpy_drop_events(h);
  h->sph.release(); h->Fh.release(); h->Fl.release(); h->F3.release();
  h->part.release(); h->F.release(); h->U.release();
  (void)hipStreamDestroy(h->stream);
  delete h;
  return 0;
}

// Sphere centres [n][3] and radii [n] (host), viscosity mu.
int sphx_rpy_set_spheres(sphx_rpy* h, const float* pos, const float* radius, float mu) {
  SPHX_CHECK(h && pos && radius, "sphx_rpy_set_spheres", "null argument");
  SPHX_CHECK(mu > 0.f, "sphx_rpy_set_spheres", "mu must be positive");
  std::vector<float4> s(h->np, make_float4(0.f, 0.f, 0.f, 1.f));
  for (int i = 0; i < h->n; ++i) {
    SPHX_CHECK(radius[i] > 0.f, "sphx_rpy_set_spheres", "radii must be positive");
    s[i] = make_float4(pos[3 * i], pos[3 * i + 1], pos[3 * i + 2], radius[i]);
  }
  SPHX_HIP(hipSetDevice(h->device));
  SPHX_HIP(hipMemcpy(h->sph.p, s.data(), h->np * sizeof(float4), hipMemcpyHostToDevice));
  h->mu = mu;
  return 0;
}

// Reduction segments per row tile (work split over the spheres); from then
// on every apply of the handle takes the tile path.
int sphx_rpy_set_split(sphx_rpy* h, int split) {
  SPHX_CHECK(h && split >= 1, "sphx_rpy_set_split", "bad argument");
  h->split = split;
  return 0;
}

// U = M F with device arrays dF, dU of [3n][nrhs] FP32 (row 3p + a),
// asynchronous on the handle's stream.  mode 1, 3 or 6 (see above).
int sphx_rpy_apply_device(sphx_rpy* h, const float* dF, float* dU, int mode) {
  SPHX_CHECK(h && dF && dU, "sphx_rpy_apply_device", "null argument");
  SPHX_CHECK(mode == 1 || mode == 3 || mode == 6, "sphx_rpy_apply_device", "mode must be 1, 3 or 6");
  SPHX_HIP(hipSetDevice(h->device));
  const int np = h->np, K = h->K;
  hipEvent_t e0 = nullptr, e1 = nullptr;
  if (h->timing) {
    // timing only: no system-scope fence at the records
    SPHX_HIP(hipEventCreateWithFlags(&e0, hipEventDisableSystemFence));
    SPHX_HIP(hipEventCreateWithFlags(&e1, hipEventDisableSystemFence));
    h->ev.emplace_back(e0, e1);
  }
  // FP32 in one launch where that is faster.  512 workgroups (n/2 times K/16)
  // run at a time and walk the partners 256 at a time: up to four such rounds
  // are, except that at K = 64 two spheres' rows lie 768 bytes apart and the
  // line comes sooner.  us a call, direct / tile path in modes 1, 3 and 6: 512
  // x 16 7.3 / 15 16 17, 1024 x 16 12.9 / 17.6 19 21, 1200 x 16 21 / 19.7 22
  // 25; 433 x 32 9.7 / 14.8 16 18, 512 x 32 11.2 / 15.4 17 18, 513 x 32 16.7 /
  // 15.5 18 21; 340 x 48 8.3 / 14.5 16 18, 512 x 48 13.7 / 16.7 18 20, 513 x 48
  // 16.3 / 16.1 19 23; 256 x 64 7.7 / 13.0 15 16, 306 x 64 13.1 / 13.8 15 17,
  // 433 x 64 17.2 / 15.9 18 19.  Not for a caller who set the tile path's
  // split, nor for arrays that are not aligned for 16-byte loads or that overlap
  // (the tile path may be applied in place: it reads F before its last launch
  // writes U).
  static constexpr int MOST[4] = {1024, 512, 512, 306};   // K = 16, 32, 48, 64
  const bool direct = h->n <= MOST[K / 16 - 1];
  const uintptr_t f0 = reinterpret_cast<uintptr_t>(dF), u0 = reinterpret_cast<uintptr_t>(dU);
  const uintptr_t len = 3 * (uintptr_t)h->n * K * sizeof(float);
  const bool apart = f0 + len <= u0 || u0 + len <= f0;
  if (h->split == 0 && direct && (f0 & 15) == 0 && apart) {
    if (h->timing) SPHX_HIP(hipEventRecord(e0, h->stream));
    k_rpy_direct<2><<<dim3(blocks_for(h->n, 2), K / 16), WALK_THREADS, 0, h->stream>>>(
        h->sph.p, h->n, h->mu, K, dF, dU);
    if (h->timing) SPHX_HIP(hipEventRecord(e1, h->stream));
    SPHX_HIP(hipGetLastError());
    return 0;
  }
  // 16 segments per row tile unless the caller set them: each FP32 sum then
  // runs over a 16th of the spheres, whatever their number.  Fewer, to fill
  // the chip in one round, are as fast or faster and less accurate: mode 3 at
  // 4096 x 64, 12 segments, 87 us instead of 103, error 3.5e-6 instead of
  // 3.3e-6; mode 6 at 8192 and 16384 x 16, 8 and 4 segments, the same time
  // and 9.2e-7 instead of 5.5e-7, 1.9e-6 instead of 7.7e-7.  More cost launches of partials: 24 at 4096 x 64 in mode 6 148
  // us instead of 132.
  const int chunks = np / RPY_TQ, tiles = np / RPY_TP;
  const int want = h->split ? h->split : 16;
  int split = std::max(1, std::min(want, chunks));
  int seg = (chunks + split - 1) / split * RPY_TQ;
  int nseg = (np + seg - 1) / seg;
  SPHX_TRY(h->part.alloc((size_t)nseg * 3 * np * K));
  const int pieces = mode == 1 ? 1 : (mode == 3 ? 2 : 3);
  k_rpy_split_f<<<dim3(tiles, 3, K / 16), 256, 0, h->stream>>>(dF, h->n, np, K, pieces, h->Fh.p, h->Fl.p, h->F3.p);
  dim3 grid(np / RPY_TP, nseg);
  if (h->timing) SPHX_HIP(hipEventRecord(e0, h->stream));
  if (mode == 1)
    k_rpy_tile<1><<<grid, RPY_THREADS, 0, h->stream>>>(h->sph.p, h->n, np, h->mu, K, seg, h->Fh.p,
                                                       h->Fl.p, h->F3.p, h->part.p);
  else if (mode == 3)
    k_rpy_tile<3><<<grid, RPY_THREADS, 0, h->stream>>>(h->sph.p, h->n, np, h->mu, K, seg, h->Fh.p,
                                                       h->Fl.p, h->F3.p, h->part.p);
  else
    k_rpy_tile<6><<<grid, RPY_THREADS, 0, h->stream>>>(h->sph.p, h->n, np, h->mu, K, seg, h->Fh.p,
                                                       h->Fl.p, h->F3.p, h->part.p);
  if (h->timing) SPHX_HIP(hipEventRecord(e1, h->stream));
  int outs = 3 * h->n * K;
  k_rpy_reduce<<<blocks_for(outs, 256), 256, 0, h->stream>>>(h->sph.p, h->n, np, h->mu, K, nseg,
                                                             dF, h->part.p, dU);
  SPHX_HIP(hipGetLastError());
  return 0;
}

// Host arrays F, U of [3n][nrhs]; synchronous.
int sphx_rpy_apply(sphx_rpy* h, const float* F, float* U, int mode) {
  SPHX_CHECK(h && F && U, "sphx_rpy_apply", "null argument");
  SPHX_HIP(hipSetDevice(h->device));
  size_t sz = 3 * (size_t)h->n * h->K * sizeof(float);
  SPHX_HIP(hipMemcpyAsync(h->F.p, F, sz, hipMemcpyHostToDevice, h->stream));
  SPHX_TRY(sphx_rpy_apply_device(h, h->F.p, h->U.p, mode));
  SPHX_HIP(hipMemcpyAsync(U, h->U.p, sz, hipMemcpyDeviceToHost, h->stream));
  SPHX_HIP(hipStreamSynchronize(h->stream));
  return 0;
}

// Time each k_rpy_tile launch with HIP events on the handle's stream (on)
// or stop and forget the recorded launches (off).
int sphx_rpy_timing(sphx_rpy* h, int on) {
  SPHX_CHECK(h, "sphx_rpy_timing", "null handle");
  SPHX_HIP(hipStreamSynchronize(h->stream));
  rpy_drop_events(h);
  h->timing = on != 0;
  return 0;
}

// Total milliseconds and count of the tile launches timed since timing was
// switched on; forgets them.
int sphx_rpy_timing_get(sphx_rpy* h, double* ms, int* count) {
  SPHX_CHECK(h && ms && count, "sphx_rpy_timing_get", "null argument");
  SPHX_HIP(hipStreamSynchronize(h->stream));
  double t = 0.0;
  for (auto& e : h->ev) {
    float f = 0.f;
    SPHX_HIP(hipEventElapsedTime(&f, e.first, e.second));
    t += f;
  }
  *ms = t;
  *count = (int)h->ev.size();
  rpy_drop_events(h);
  return 0;
}

int sphx_rpy_sync(sphx_rpy* h) {
  SPHX_CHECK(h, "sphx_rpy_sync", "null argument");
  SPHX_HIP(hipStreamSynchronize(h->stream));
  return 0;
}

hipStream_t sphx_rpy_stream(sphx_rpy* h) { return h ? h->stream : nullptr; }

}  // extern "C"

namespace {

// The walkthrough's launches on the current device's null stream;
// synchronous.
int walk_run(sphx_context* nodes, const sphx_stokesianBufList* b, int n, int with_force) {
  const int bl = blocks_for(n, 256);
  const bool background = nodes && nodes->mpm.on;
  if (background) {
    const sphx_ParamCarrier& P = nodes->P;
    k_walk_background<<<bl, 256>>>(b->dispBuffer, n, nodes->mpm.nodev.p,
                                   make_float3(P.mpmXmin.x, P.mpmXmin.y, P.mpmXmin.z),
                                   P.mpmcellsize, make_int3(P.mpmRes.x, P.mpmRes.y, P.mpmRes.z),
                                   b->simscale, b->cuUnew);
  }
  auto force = [&](auto spheres) {
    constexpr int I = decltype(spheres)::value;
    k_walk_force<I><<<blocks_for(n, I), WALK_THREADS>>>(b->dispBuffer, n, b->cuForce);
  };
  auto mob = [&](auto spheres) {
    constexpr int I = decltype(spheres)::value;
    k_walk_mob<I><<<blocks_for(n, I), WALK_THREADS>>>(b->dispBuffer, n, b->cuForce, background,
                                                      b->cuUnew, b->cuOmega);
  };
  // Spheres per workgroup 1, 2, 4, 8, 16 measured (us), force / mobility: n =
  // 500 4.4 3.9 4.6 5.4 7.7 / 3.5 3.4 4.0 5.2 7.7; 2,000 13 6.2 6.1 7.7 11 /
  // 8.3 8.3 8.4 11 16; 5,000 52 15 11 13 19 / 39 32 32 38 53; 16,384 481 123
  // 73 60 60 / 428 275 276 290 318 (one thread a sphere: 2,600 / 6,940; at
  // four clocks an instruction the issue alone takes 59 / 299, and some of the
  // mobility's are faster).
  using std::integral_constant;
  if (with_force) {
    if (n <= 1024) force(integral_constant<int, 2>{});
    else if (n <= 8192) force(integral_constant<int, 4>{});
    else force(integral_constant<int, 8>{});
  }
  if (n <= 1024) mob(integral_constant<int, 2>{});
  else mob(integral_constant<int, 4>{});
  k_walk_commit<<<bl, 256>>>(b->dispBuffer, n, b->cuUnew, b->dt);
  SPHX_HIP(hipGetLastError());
  SPHX_HIP(hipDeviceSynchronize());
  return 0;
}

}  // namespace

extern "C" {

// The reference's walkthrough step on device buffers: near-field force
// (added to cuForce), background velocity from the node grid of `nodes`
// (may be NULL: zero background), mobility velocity and rotation,
// positions advanced by U dt.
int sphx_rpy_walkthrough(sphx_context* nodes, const sphx_stokesianBufList* b, int n,
                         int with_force) {
  SPHX_CHECK(b && n >= 0, "sphx_rpy_walkthrough", "bad argument");
  if (n == 0) return 0;
  return walk_run(nodes, b, n, with_force);
}

// Same step under the limit on n that its callers were given.
int sphx_rpy_walkthrough_noalloc(sphx_context* nodes, const sphx_stokesianBufList* b, int n,
                                 int with_force) {
  SPHX_CHECK(b && n >= 0, "sphx_rpy_walkthrough_noalloc", "bad argument");
  SPHX_CHECK(n <= SPHX_WALK_NOALLOC_MAX, "sphx_rpy_walkthrough_noalloc",
             "more spheres than the static scratch held (SPHX_WALK_NOALLOC_MAX)");
  if (n == 0) return 0;
  return walk_run(nodes, b, n, with_force);
}

// MVmultiply / getMobU: u = mat f with mat (6n x 6n) row-major, device.
int sphx_mob_gemv(const float* mat, const float* f, float* u, int nsize) {
  SPHX_CHECK(mat && f && u && nsize >= 0, "sphx_mob_gemv", "bad argument");
  int dim = 6 * nsize;
  if (dim == 0) return 0;
  k_gemv<<<blocks_for(dim, 4), 256>>>(mat, f, u, dim);
  SPHX_HIP(hipGetLastError());
  SPHX_HIP(hipDeviceSynchronize());
  return 0;
}

}  // extern "C"
