// The BSGS multiply-accumulate on the int8 matrix cores, for both prime widths.
//
//   res[c][g][i][l][n] = sum_b pt[g * nb + b][l][n] * baby_b[i][c][l][n]   (mod q_l)
//
// For one coefficient n of one limb this is a matrix product: giants x babies times babies x (input,
// component).  Every canonical word is written as the 64-bit word of its balanced base-256 digits
// (ND of them: 7 below 2^50, 8 below 2^60), so that
//   sum_b x_b w_b = sum_c 256^c C_c,   C_c = sum_b sum_a w_{b,c-a} x_{b,a}.
// For 16 giants x 16 columns x 16 babies, C_c is two v_mfma_i32_16x16x64_i8 (K = 16 babies x 4 digit
// bytes): Q_c times the low halves of the columns' digit words plus Q_{c-4} times their high halves,
// where Q_k holds the plaintext digits w_k, w_{k-1}, w_{k-2}, w_{k-3} of every baby, one byte permute per
// word.  Each Q_k serves both, and those without a digit in range are left out: 3 ND - 2 products
// (19 and 22) instead of 4 ND - 2.  |C_c| <= 16 babies * ND * 2^14 <= 2^21, exact in int32.  The 2 ND - 1 sums of one
// output are folded into its residue once per 16 babies.
//
// What bounds it: one output costs a fold of about 35 (FP64) or 110 (64-bit) VALU instructions per 16
// products, against 7 FP64 operations or four 32 x 32 multiply-adds per product on the VALU.
//
// Tile: a workgroup (8 waves, one per CU) takes 32 consecutive coefficients of one limb (256-byte row
// segments) and walks the 16 x 16 tiles of their (giants x columns) products back and forth (column
// 2 i + c), 16 babies per step.  LDS holds one row group of 16 giants and one of 16 columns, 64 KB each,
// as digit words; a step replaces the one that changes, whose words were loaded into registers while the
// step before it computed.  Each wave computes 4 of the coefficients; the results go back through the
// buffer that the next step replaces, so that they too are written in 256-byte runs.  Rows are
// limbs * 512 KB apart: read in 64-byte runs such a set of rows gives 2.9 TB/s, in 128-byte runs 4.6 to
// 4.9, in 256-byte runs 5.9; written in 64-byte runs 3.0 TB/s, in 128-byte runs 5.6, in 256-byte runs
// 5.8, in single 16-byte stores 2.2.  (16 coefficients and two workgroups per CU: 7.0 ms where 32 take
// 5.7, against 7.9 of the VALU kernel: 16 inputs, 16 babies, 32 giants, 20 limbs.)  The steps' barriers
// leave it at 0.7 of what its HBM traffic takes.
// LDS row r = baby / 4 * 16 + (giant or column) % 16: for every coefficient n a 16-byte chunk 2 n of the
// low words of the four babies' digit words and a chunk 2 n + 1 of their high words -- operands of the
// matrix instruction as they are.  Chunk x sits at x ^ (r & 15) ^ (n >> 2), so that neither the rows that
// a quarter-wave reads at once nor the coefficients that eight lanes write at once share banks.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "internal.hpp"

namespace hck {

typedef int mx_v4i __attribute__((ext_vector_type(4)));
constexpr int kMxThreads = 512;
constexpr int kMxCoef = 32;        // coefficients per unit: 256-byte row segments
constexpr int kMxMaxBabies = 64;

struct MxArgs {
  const uint64_t* c0[kMxMaxBabies];
  const uint64_t* c1[kMxMaxBabies];
  long long baby_stride, pt_stride;
  const uint64_t* pts;
  uint64_t* res;
  int nb, ni, G, limbs;
  int tiles_g, tiles_c;   // row groups of 16 giants / 16 columns
  int units;              // limbs * (N / 32)
  uint8_t prime[kMaxPrimes];
};

// Selector of the bytes w_{k}, w_{k-1}, w_{k-2}, w_{k-3} of an ND-digit word (0 outside it).
template <int ND>
__device__ constexpr uint32_t mx_sel(int k) {
  uint32_t s = 0;
  for (int a = 0; a < 4; ++a) {
    const int d = k - a;
    s |= (uint32_t)(d >= 0 && d < ND ? d : 0x0c) << (8 * a);
  }
  return s;
}
// One step of a workgroup's walk: unit (limb and coefficients), tile, chunk of 16 babies, and which row
// groups it loads.  All uniform.
struct MxStep {
  int unit, tile, ch;
  bool lg, lc;
};
__device__ __forceinline__ int mx_gt(const MxArgs& A, int tile) { return tile / A.tiles_c; }
__device__ __forceinline__ int mx_ct(const MxArgs& A, int tile) {
  const int g = tile / A.tiles_c, c = tile % A.tiles_c;
  return (g & 1) ? A.tiles_c - 1 - c : c;
}
template <bool MULTI>
__device__ __forceinline__ MxStep mx_next(const MxArgs& A, const MxStep& s, int stride) {
  MxStep r = s;
  if (MULTI && (s.ch + 1) * 16 < A.nb) {
    r.ch = s.ch + 1;
    r.lg = r.lc = true;
    return r;
  }
  r.ch = 0;
  r.tile = s.tile + 1;
  r.lg = r.lc = true;
  if (r.tile == A.tiles_g * A.tiles_c) {
    r.tile = 0;
    r.unit = s.unit + stride;
  } else if (!MULTI) {  // one row group changes
    r.lg = mx_gt(A, r.tile) != mx_gt(A, s.tile);
    r.lc = !r.lg;
  }
  return r;
}

// A step's words of a thread: coefficients 2 (t % 16) and the next of row (t / 16) % 16, babies
// 4 (2 j + t / 256) + h.
typedef ulong mx_v2u __attribute__((ext_vector_type(2)));
typedef const mx_v2u __attribute__((address_space(1)))* MxGlobal;  // global, not flat: LDS waits leave it alone
struct MxStage {
  mx_v2u g[2][4], c[2][4];
};
__device__ __forceinline__ void mx_load(MxStage& st, const MxArgs& A, const MxStep& s, int half) {
  const int t = threadIdx.x, rr = (t / (kMxCoef / 2)) & 15;
  const long long off = (long long)(s.unit / (kN / kMxCoef)) * kN + (s.unit % (kN / kMxCoef)) * kMxCoef + 2 * (t % (kMxCoef / 2));
  if (s.lg) {
    const int g = min(16 * mx_gt(A, s.tile) + rr, A.G - 1);  // clamped rows are never stored
    const uint64_t* gp = A.pts + (long long)g * A.nb * A.pt_stride + off;
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int h = 0; h < 4; ++h) {
        const int b = min(s.ch * 16 + 4 * (2 * j + half) + h, A.nb - 1);  // uniform; past the end: zero
        st.g[j][h] = *(MxGlobal)(gp + b * A.pt_stride);
      }
  }
  if (s.lc) {
    const int col = min(16 * mx_ct(A, s.tile) + rr, 2 * A.ni - 1);
    const long long coff = (long long)(col >> 1) * A.baby_stride + off;
    const bool second = (col & 1) != 0;
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int h = 0; h < 4; ++h) {
        const int b = min(s.ch * 16 + 4 * (2 * j + half) + h, A.nb - 1);
        const uint64_t *p0 = A.c0[b], *p1 = A.c1[b];
        asm volatile("" : "+s"(p0), "+s"(p1));  // two scalar loads and a select, not a load per lane
        st.c[j][h] = *(MxGlobal)((second ? p1 : p0) + coff);
      }
  }
}
// The loaded words of one row group, as digit words, into its buffer.
template <class P>
__device__ __forceinline__ void mx_fill(const mx_v2u (&v)[2][4], mx_v4i* Y, int b0, int nb, int half) {
  const int t = threadIdx.x, rr = (t / (kMxCoef / 2)) & 15;
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const int n = 2 * (t % (kMxCoef / 2)) + e, x = 2 * n ^ rr ^ (n >> 2);
      mx_v4i l, h;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const bool live = b0 + 4 * (2 * j + half) + k < nb;  // uniform over the wave
        const uint64_t w = live ? P::digits(e ? v[j][k].y : v[j][k].x) : 0ULL;
        l[k] = (int)(uint32_t)w;
        h[k] = (int)(uint32_t)(w >> 32);
      }
      mx_v4i* y = Y + ((2 * j + half) * 16 + rr) * (2 * kMxCoef);
      y[x] = l;
      y[x ^ 1] = h;
    }
}

// P: the prime width's arithmetic -- ND, digits(word), Consts and its load(tables, prime), Acc, zero(),
// add(acc, a, consts) of one output's ND byte-pair sums a, finish(acc, consts).
template <class P, bool MULTI>
__device__ __forceinline__ void mx_body(const MxArgs& A, const typename P::Tables& T, mx_v4i* Yg, mx_v4i* Yc) {
  constexpr int ND = P::ND, NC = 2 * ND - 1;
  const int t = threadIdx.x, lane = t & 63, q4 = lane >> 4, m = lane & 15;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6) & 7, half = wave >> 2;
  const int xcd = blockIdx.x % kXcds, bi = blockIdx.x / kXcds, bn = gridDim.x / kXcds;
  const int share = (A.units + kXcds - 1) / kXcds;
  const int lo = xcd * share, hi = min(lo + share, A.units);
  if (lo + bi >= hi) return;  // uniform
  const long long is = (long long)A.limbs * kN, gs = (long long)A.ni * is, cs = (long long)A.G * gs;
  MxStage st;
  MxStep s{lo + bi, 0, 0, true, true};
  mx_load(st, A, s, half);
  typename P::Acc acc[4][4];
  typename P::Consts C;
  int limb = -1;
  while (s.unit < hi) {
    if (s.unit / (kN / kMxCoef) != limb) {  // rare: the constants' loads are not waited for in every step
      limb = s.unit / (kN / kMxCoef);
      C.load(T, __builtin_amdgcn_readfirstlane(A.prime[limb]));
    }
    __syncthreads();  // the previous step's readers are done
    if (s.lg) mx_fill<P>(st.g, Yg, s.ch * 16, A.nb, half);
    if (s.lc) mx_fill<P>(st.c, Yc, s.ch * 16, A.nb, half);
    __syncthreads();
    // the next step's words, in flight while this one computes
    const MxStep nx = mx_next<MULTI>(A, s, bn);
    if (nx.unit < hi) mx_load(st, A, nx, half);
    __builtin_amdgcn_sched_barrier(0);
    const mx_v4i* ya = Yg + (q4 * 16 + m) * (2 * kMxCoef);  // babies 4 q4 .. of giant / column m
    const mx_v4i* yb = Yc + (q4 * 16 + m) * (2 * kMxCoef);
#pragma unroll
    for (int e = 0; e < 4; ++e) {  // coefficient 4 wave + e
      const int n = 4 * wave + e, x = 2 * n ^ m ^ (n >> 2);
      const mx_v4i al = ya[x], ah = ya[x ^ 1], bl = yb[x], bh = yb[x ^ 1];
      mx_v4i c[NC];
#pragma unroll
      for (int k = 0; k < ND + 3; ++k) {
        mx_v4i q;
#pragma unroll
        for (int i = 0; i < 4; ++i) q[i] = (int)__builtin_amdgcn_perm((uint32_t)ah[i], (uint32_t)al[i], mx_sel<ND>(k));
        c[k] = __builtin_amdgcn_mfma_i32_16x16x64_i8(q, bl, k < 4 ? mx_v4i{0, 0, 0, 0} : c[k], 0, 0, 0);
        if (k + 4 < NC) c[k + 4] = __builtin_amdgcn_mfma_i32_16x16x64_i8(q, bh, mx_v4i{0, 0, 0, 0}, 0, 0, 0);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        int a[ND];  // a[k] = C_{2k} + 256 C_{2k+1}, |.| < 2^30
#pragma unroll
        for (int k = 0; k < ND; ++k) a[k] = c[2 * k][r] + (2 * k + 1 < NC ? (int)((uint32_t)c[2 * k + 1][r] << 8) : 0);
        if (!MULTI || s.ch == 0) acc[e][r] = P::zero();
        P::add(acc[e][r], a, C);
      }
      if (e & 1) __builtin_amdgcn_sched_barrier(0);  // two coefficients' operands and sums live at a time
    }
    if (!MULTI || nx.ch == 0) {
      // the results through the buffer that the next step replaces: output row 16 giant + column, chunk h at
      // h ^ (column & 7)
      ulonglong2* Y2 = reinterpret_cast<ulonglong2*>(nx.lc ? Yc : Yg);
      __syncthreads();
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int h = 0; h < 2; ++h)
          Y2[((4 * q4 + r) * 16 + m) * (kMxCoef / 2) + ((2 * wave + h) ^ (m & 7))] =
              ulonglong2{P::finish(acc[2 * h][r], C), P::finish(acc[2 * h + 1][r], C)};
      __syncthreads();
      const int g0 = 16 * mx_gt(A, s.tile), c0 = 16 * mx_ct(A, s.tile);
      const long long ln = (long long)(s.unit / (kN / kMxCoef)) * kN + (s.unit % (kN / kMxCoef)) * kMxCoef;
      const int rr = t / (kMxCoef / 2);  // rows rr + 32 j: giant 2 j + rr / 16, column rr % 16
      const int col = c0 + (rr & 15);
      uint64_t* o = A.res + (col & 1) * cs + (long long)(col >> 1) * is + ln + 2 * ((t % (kMxCoef / 2)) ^ (rr & 7));
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int g = g0 + 2 * j + (rr >> 4);
        const ulonglong2 v = Y2[(32 * j + rr) * (kMxCoef / 2) + t % (kMxCoef / 2)];
        if (g < A.G && col < 2 * A.ni) *reinterpret_cast<ulonglong2*>(o + (long long)g * gs) = v;
      }
    }
    s = nx;
  }
}

template <class P, bool MULTI>
__global__ __launch_bounds__(kMxThreads, 2) void k_mac_mx(const MxArgs A, const typename P::Tables T) {
  __shared__ mx_v4i Yg[64 * 2 * kMxCoef], Yc[64 * 2 * kMxCoef];
  mx_body<P, MULTI>(A, T, Yg, Yc);
}

// Where the matrix cores pay: by the share of the 16 x 16 x 16 tiles that holds real giants, columns and
// babies (FP64 words: mx_pays_fp asks for more).  Measured at 8 limbs, VALU kernel against this one, (inputs,
// babies, giants):
//   share   FP64 words                          64-bit words
//   1       3.23 / 2.26 ms (16, 16, 32)         4.72 / 2.70 ms
//           2.99 / 2.40    (8, 64, 16)          4.05 / 2.74
//   0.875   1.59 / 1.22    (7, 16, 32)          2.29 / 1.43
//   0.75    2.39 / 2.09    (16, 16, 24)         3.53 / 2.50
//           2.28 / 2.02    (16, 24, 16)         3.18 / 2.53
//   0.625   2.27 / 1.99    (10, 16, 32)         2.91 / 2.49
//           1.26 / 1.12    (5, 16, 32)          1.75 / 1.36
//           1.53 / 1.12    (16, 16, 10)         1.73 / 1.35
//   0.5     1.00 / 1.12    (16, 8, 16)          1.63 / 1.36
//           0.91 / 1.09    (16, 16, 8)          1.29 / 1.31
//           0.92 / 1.10    (4, 16, 32)          1.29 / 1.34
//   0.44    0.95 / 1.07    (7, 8, 32)           1.53 / 1.32
//   0.375   0.79 / 1.04    (3, 16, 32)          1.21 / 1.28
// (With 8 babies the 64-bit VALU kernel is slow enough that this one wins below the line too.)
inline bool mx_pays(int ni, int nb, int G) {
  auto up = [](int v) { return (v + 15) / 16 * 16; };
  return (double)G * (2 * ni) * nb >= 0.6 * up(G) * up(2 * ni) * up(nb);
}

inline MxArgs mx_args(int limbs, const uint8_t* prime, int ni, int nb, int G, const uint64_t* const* c0,
                      const uint64_t* const* c1, long long baby_stride, const uint64_t* pts, long long pt_stride,
                      uint64_t* res) {
  MxArgs A{};
  for (int b = 0; b < nb; ++b) {
    A.c0[b] = c0[b];
    A.c1[b] = c1[b];
  }
  for (int l = 0; l < limbs; ++l) A.prime[l] = prime[l];
  A.baby_stride = baby_stride;
  A.pt_stride = pt_stride;
  A.pts = pts;
  A.res = res;
  A.nb = nb;
  A.ni = ni;
  A.G = G;
  A.limbs = limbs;
  A.tiles_g = (G + 15) / 16;
  A.tiles_c = (2 * ni + 15) / 16;
  A.units = limbs * (kN / kMxCoef);
  return A;
}

// Whether the vector loads and stores of the matrix-core MAC fit the operands: every row 16-byte aligned.
inline bool mx_aligned(const MxArgs& A) {
  uintptr_t bits = (uintptr_t)A.pts | (uintptr_t)A.res | (uintptr_t)(8 * A.pt_stride) | (uintptr_t)(8 * A.baby_stride);
  for (int b = 0; b < A.nb; ++b) bits |= (uintptr_t)A.c0[b] | (uintptr_t)A.c1[b];
  return (bits & 15) == 0;
}

template <class P>
inline void mx_launch(const MxArgs& A, const typename P::Tables& T, hipStream_t s) {
  constexpr unsigned blocks = 256;  // one per CU; the units of a limb alone are 2048
  if (A.nb <= 16)
    k_mac_mx<P, false><<<blocks, kMxThreads, 0, s>>>(A, T);
  else
    k_mac_mx<P, true><<<blocks, kMxThreads, 0, s>>>(A, T);
}

}  // namespace hck
