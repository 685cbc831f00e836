// BSGS baby-step multiply-accumulate over many inputs at once.
//
//   res[c][g][i][l][n] = sum_{b < nb} pt[g * nb + b][l][n] * baby_b[i][c][l][n]   (mod q_l)
//
// for inputs i < ni, giants g < G, components c in {0, 1}: the partial sums of the diagonal
// method that the giant steps then rotate and add (exact-residue semantics of
// bench/cmp/kernels/holmes_mac.cu:8-12, multi-input tiling of holmes_mac.cu:108-190).
//
// Three kernels: with enough inputs, giants and babies to fill its 16 x 16 x 16 tiles the matrix-core MAC
// of mac_mx.hpp, else k_bsgs_mac on the VALU; k_mac_rows for plaintexts that lack the transform's row pass
// (hck_bsgs_mac_rows).  In k_bsgs_mac a thread owns one coefficient of one limb and
// a TI x 8 tile of (input, giant) accumulators for both components: per baby step it reads 8 plaintext
// words and 2 TI baby words for 16 TI products (the next step's words are loaded while the current step
// computes), so plaintexts stream once per input tile and babies once per giant tile.  Up to 3 inputs HBM
// bounds it (4.5 to 4.9 TB/s with tiles of just these inputs; a tile of 4 ran 1 input's 512 x 17 limbs in
// 1.69 ms, where the products of the 3 empty rows bounded it, against 1.19 ms), from 4 on the VALU.  All tiles
// of one (limb, 128-coefficient) unit are dispatched to the same XCD (workgroups are handed to
// the 8 XCDs round-robin by linear id), so the unit's plaintext and baby data is fetched from HBM
// once and then served from that XCD's L2.
#include <hip/hip_runtime.h>

#include "../../include/holmes_ckks.h"
#include "internal.hpp"
#include "mac_mx.hpp"
#include "tile_layout.hpp"
#include "wide.hpp"
#include "modarith64.hpp"

namespace hck {
namespace {

constexpr int kMacThreads = 128;
constexpr int kTG = 8;  // giants per thread
constexpr int kMaxBabies = 64;

// Inputs per thread: the tile that computes the fewest rows, each row of the tiles of 3 and 2 inputs charged
// with the plaintext words that a smaller tile reads again (an equal count goes to the larger tile).  Tiles
// of 4 against those of 3: 5, 6 and 9 inputs 1.05 to 1.3 times as long; 13 to 15 1.00 to 1.06 with at most 8
// giants, 0.94 to 1.0 with 16; 11 and 12 0.94 to 1.0.  Against those of 2: 10 inputs 1.06 to 1.13 with at
// most 4 giants, 0.90 to 1.0 above with at most 16 babies.  A single input has a tile of its own.
inline int mac_tile_inputs(int ni, int giants) {
  if (ni == 1) return 1;
  const int w3 = giants <= 8 ? 105 : 107, w2 = giants <= 4 ? 113 : 125;
  const int c4 = (ni + 3) / 4 * 4 * 100, c3 = (ni + 2) / 3 * 3 * w3, c2 = (ni + 1) / 2 * 2 * w2;
  return c4 <= c3 && c4 <= c2 ? 4 : c3 <= c2 ? 3 : 2;
}

// Where the matrix cores pay on FP64 words: where the tiles are full (mx_pays), and the VALU kernel's own
// tiles, which need not be, would compute at least `need` of what they compute.  A walk over several tiles keeps
// one row group per step: it pays earlier than a single tile, which loads both.  Measured, VALU time over
// matrix-core time at 2 to 20 limbs, (inputs, babies, giants): single tile (8, 11, 16) 0.90 to 0.97, (8, 12, 16)
// 0.94 to 1.01, (7, 13, 16) 0.94 to 1.05, (8, 14, 16) 1.00 to 1.08, (8, 16, 16) 1.00 to 1.14; two tiles (16, 10,
// 16) 0.97 to 1.00, (8, 11, 32) 1.02 to 1.07, (16, 12, 16) 1.08 to 1.11; four (16, 10, 32) 1.06 to 1.09, (5,
// 16, 32) 1.10 to 1.15, (10, 16, 32) 1.13 to 1.19; two steps of babies (8, 20, 16) 0.94 to 1.03, (16, 20,
// 32) 0.96 to 1.00, (8, 24, 16) 1.08 to 1.15, (16, 33, 16) 1.05 to 1.07.
inline bool mx_pays_fp(int ni, int nb, int giants) {
  if (!mx_pays(ni, nb, giants)) return false;
  auto up = [](int v, int m) { return (v + m - 1) / m * m; };
  const int tiles = (giants + 15) / 16 * ((2 * ni + 15) / 16);
  const double need = nb > 16 ? 0.68 : tiles == 1 ? 0.86 : tiles < 4 ? 0.68 : 0.62;
  const double valu = (double)up(ni, mac_tile_inputs(ni, giants)) * up(giants, kTG) * nb;
  return valu >= need * up(ni, 8) * up(giants, 16) * up(nb, 16);
}

struct BabyPtrs {
  const uint64_t* c0[kMaxBabies];
  const uint64_t* c1[kMaxBabies];
};
struct MacPrimes {
  uint8_t prime[kMaxPrimes];
};

// One baby step's operands for a thread: kTG plaintext words, TI words of each component.
template <int TI>
struct MacOps {
  uint64_t w[kTG], x0[TI], x1[TI];
};

template <int TI>
__device__ __forceinline__ void mac_load(MacOps<TI>& o, const BabyPtrs& babies, int b, int nb, int G, int ni,
                                         int g0, int i0, const uint64_t* __restrict__ pts, long long pt_stride,
                                         long long baby_stride, long long ln) {
#pragma unroll
  for (int g = 0; g < kTG; ++g) {
    const int gg = g0 + g < G ? g0 + g : g0;  // clamp: duplicates are never stored
    o.w[g] = pts[((long long)gg * nb + b) * pt_stride + ln];
  }
  const uint64_t* b0 = babies.c0[b];
  const uint64_t* b1 = babies.c1[b];
#pragma unroll
  for (int t = 0; t < TI; ++t) {
    const int ii = i0 + t < ni ? i0 + t : i0;
    o.x0[t] = b0[(long long)ii * baby_stride + ln];
    o.x1[t] = b1[(long long)ii * baby_stride + ln];
  }
}

template <int TI>
__global__ __launch_bounds__(kMacThreads) void k_bsgs_mac(uint64_t* __restrict__ res, BabyPtrs babies,
                                                          long long baby_stride, int nb, int ni, int G,
                                                          const uint64_t* __restrict__ pts, long long pt_stride,
                                                          int limbs, MacPrimes mp, int units_per_limb,
                                                          int tiles_i, int tiles_g, int total_units, DevTables T) {
  // XCD-aware decode of the linear workgroup id into (unit, tile)
  const int tiles = tiles_i * tiles_g;
  const int lin = blockIdx.x;
  const int xcd = lin % kXcds, k = lin / kXcds;
  const int unit = (k / tiles) * kXcds + xcd;
  const int tile = k % tiles;
  if (unit >= total_units) return;
  const int l = unit / units_per_limb;
  const int n = (unit % units_per_limb) * kMacThreads + threadIdx.x;
  const int i0 = (tile % tiles_i) * TI, g0 = (tile / tiles_i) * kTG;
  const int pi = mp.prime[l];
  const double p = T.p[pi], pinv = T.pinv[pi];
  const long long ln = (long long)l * kN + n;
  double acc[TI][2][kTG];
#pragma unroll
  for (int t = 0; t < TI; ++t)
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int g = 0; g < kTG; ++g) acc[t][c][g] = 0.0;
  // one baby step's products from its loaded words; every 8 steps the sums are reduced
  auto step = [&](const MacOps<TI>& cur, int b) {
    double w[kTG], wp[kTG];
#pragma unroll
    for (int g = 0; g < kTG; ++g) {
      w[g] = u2d(cur.w[g]);
      wp[g] = w[g] * pinv;
    }
#pragma unroll
    for (int t = 0; t < TI; ++t) {
      const double x0 = u2d(cur.x0[t]), x1 = u2d(cur.x1[t]);
#pragma unroll
      for (int g = 0; g < kTG; ++g) {
        acc[t][0][g] += mulc(x0, w[g], wp[g], p);  // canonical operands: |term| <= 0.875 p
        acc[t][1][g] += mulc(x1, w[g], wp[g], p);
      }
    }
    if ((b & 7) == 7) {
#pragma unroll
      for (int t = 0; t < TI; ++t)
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
          for (int g = 0; g < kTG; ++g) acc[t][c][g] = reduce(acc[t][c][g], p, pinv);
    }
  };
  // two-stage software pipeline on two register sets: baby step b + 1's words load into one set while
  // step b computes from the other (the last pair reloads its own words, unused), so the wait before
  // a step's products covers only that step's own loads.
  MacOps<TI> o0, o1;
  mac_load(o0, babies, 0, nb, G, ni, g0, i0, pts, pt_stride, baby_stride, ln);
  int b = 0;
  for (; b + 1 < nb; b += 2) {
    mac_load(o1, babies, b + 1, nb, G, ni, g0, i0, pts, pt_stride, baby_stride, ln);
    // the loads stay ahead of the products they overlap: neither the compiler's IR passes (the
    // memory clobber) nor the scheduler (the barrier) move them below
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    step(o0, b);
    mac_load(o0, babies, b + 2 < nb ? b + 2 : b + 1, nb, G, ni, g0, i0, pts, pt_stride, baby_stride, ln);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    step(o1, b + 1);
  }
  if (b < nb) step(o0, b);  // odd count: the last step's words are in o0
  const long long is = (long long)limbs * kN, gs = (long long)ni * is, cs = (long long)G * gs;
#pragma unroll
  for (int t = 0; t < TI; ++t) {
    if (i0 + t >= ni) break;
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int g = 0; g < kTG; ++g)
        if (g0 + g < G)
          res[c * cs + (long long)(g0 + g) * gs + (long long)(i0 + t) * is + ln] = d2u(canon(acc[t][c][g], p, pinv));
  }
}

// ----------------------------------------------------------------- the MAC with the plaintexts' row pass
// hck_bsgs_mac on plaintext rows that have had the transform's column pass only (hck_encode_cols): a
// 256-word row of the 256 x 256 limb needs stages 8 .. 15, which stay inside it, so the workgroup that
// multiplies the row transforms it.  Written and read back, a transformed plaintext costs 16 bytes of
// HBM traffic per word against the 8 that this kernel reads; with one input the products take 17 FP64
// operations per word and the row pass 36, so it stays near what HBM gives.  512 diagonals x 17 limbs,
// encode and product: one input 4.35 -> 2.86 ms, two 4.59 -> 3.37 ms.  With more inputs the accumulators
// do not fit the registers and the transform would be repeated.
// Workgroup: one row of one limb, SL giants (slot s = t / 16 owns giant g0 + s, lane j = t % 16 of it words
// j + 16 k before the exchange and 16 j + k after it), all babies in turn.  The row's twiddles are the
// same for every plaintext: stages 8..11 in registers (uniform), 12..15 in LDS.  A baby's ciphertext row is
// shared by the slots through LDS (two buffers, word 16 j + k at 17 k + j).  The next baby's words are in
// flight while the current one is transformed.  |v| <= 5.5 p after the transform (centered words, as the
// encoder's column pass takes them): |term| <= 2.6 p, the sums are reduced every two babies.
static_assert(kCentered + 2 * mulv_bound(kFwdOut) < kExact, "two babies on a centered sum");
// SL: with one input 4 giants, a single wave (4, 8, 9, 16 giants x 32 babies: 0.84, 1.49, 1.82, 2.86 ms, 8
// slots 1.03, 1.50, 2.07, 2.92, 16 slots 1.45, 1.88, 2.00, 2.84: fewer slots stand empty in the last
// tile); with two inputs 8, since the two rows' words of a single wave spill (8 and 16 giants 1.73 and 3.37 ms,
// 4 slots 1.88 and 3.72).
constexpr int kMrRow = 272;
constexpr int mr_slots(int inputs) { return inputs == 1 ? 4 : 8; }

template <int NI>
__global__ __launch_bounds__(16 * mr_slots(NI), 2) void k_mac_rows(
    uint64_t* __restrict__ res, BabyPtrs babies, long long baby_stride, int nb, int G,
    const double* __restrict__ pts, long long pt_stride, int limbs, MacPrimes mp, int tiles_g, DevTables T) {
  constexpr int NC = 2 * NI;  // component c of input i: row 2 i + c
  constexpr int SL = mr_slots(NI), TH = 16 * SL, XR = 16 / SL;  // row words per thread and component
  __shared__ double R[SL * kMrRow], X[2][NC][kMrRow], W[15 * 16];
  const int lin = blockIdx.x, xcd = lin % kXcds, q = lin / kXcds;
  const int unit = (q / tiles_g) * kXcds + xcd, tile = q % tiles_g;  // limbs * 256 units, a multiple of 8
  const int l = unit >> 8, row = unit & 255;
  const int t = threadIdx.x, s = t >> 4, j = t & 15;
  const int pi = mp.prime[l];
  const double p = T.p[pi], pinv = T.pinv[pi];
  const double* __restrict__ tw = T.tw_fwd + (size_t)pi * kN;
  const long long ln = (long long)l * kN + row * 256;
  const int g = min(tile * SL + s, G - 1);  // clamped slots are never stored
  const double* prow = pts + (long long)g * nb * pt_stride + ln + j;
  double lo[15];
#pragma unroll
  for (int i = 0; i < 15; ++i) {  // stage 8 + log2(i + 1): entry i + 1 of the row's heap
    const int st = i >= 7 ? 3 : i >= 3 ? 2 : i >= 1 ? 1 : 0;
    lo[i] = tw[(1 << (8 + st)) + (row << st) + (i + 1 - (1 << st))];
  }
  for (int w = t; w < 240; w += TH) {
    const int i = w >> 4, st = i >= 7 ? 3 : i >= 3 ? 2 : i >= 1 ? 1 : 0;
    W[w] = tw[(1 << (12 + st)) + (row << (4 + st)) + (j << st) + (i + 1 - (1 << st))];
  }
  double acc[NC][16], v[16], vn[16];
#pragma unroll
  for (int c = 0; c < NC; ++c)
#pragma unroll
    for (int k = 0; k < 16; ++k) acc[c][k] = 0.0;
  uint64_t xw[NC][XR];
  auto load = [&](double (&d)[16], int b) {
#pragma unroll
    for (int k = 0; k < 16; ++k) d[k] = prow[(long long)b * pt_stride + 16 * k];
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const long long i = c >> 1;
      const uint64_t* base = (c & 1) ? babies.c1[b] : babies.c0[b];
#pragma unroll
      for (int r = 0; r < XR; ++r) xw[c][r] = base[i * baby_stride + ln + t + r * TH];
    }
  };
  auto put = [&](int buf) {
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int r = 0; r < XR; ++r) X[buf][c][17 * (t & 15) + (t >> 4) + r * SL] = u2d(xw[c][r]);
  };
  double* Rs = R + s * kMrRow;
  load(v, 0);
  put(0);
  __syncthreads();
  for (int b = 0; b < nb; ++b) {
    load(vn, b + 1 < nb ? b + 1 : b);  // the last step reloads its own words, unused
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int st = 0; st < 4; ++st) {
      const int h = 8 >> st;
#pragma unroll
      for (int k = 0; k < 16; ++k) {
        if (k & h) continue;
        const double m = mulv(v[k + h], lo[(1 << st) - 1 + (k >> (4 - st))], p, pinv);
        const double a = fwd_reduces(8 + st) ? reduce(v[k], p, pinv) : v[k];
        v[k] = a + m;
        v[k + h] = a - m;
      }
    }
    col_a_to_b(v, Rs, j);
#pragma unroll
    for (int st = 0; st < 4; ++st) {
      const int h = 8 >> st;
#pragma unroll
      for (int k = 0; k < 16; ++k) {
        if (k & h) continue;
        const double m = mulv(v[k + h], W[((1 << st) - 1 + (k >> (4 - st))) * 16 + j], p, pinv);
        const double a = fwd_reduces(12 + st) ? reduce(v[k], p, pinv) : v[k];
        v[k] = a + m;
        v[k + h] = a - m;
      }
    }
    const double(&xb)[NC][kMrRow] = X[b & 1];
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int k = 0; k < 16; ++k) acc[c][k] += mulv(v[k], xb[c][17 * k + j], p, pinv);
    if (b & 1) {
#pragma unroll
      for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int k = 0; k < 16; ++k) acc[c][k] = reduce(acc[c][k], p, pinv);
    }
    put((b + 1) & 1);  // read last in the step before this one
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 16; ++k) v[k] = vn[k];
  }
  const long long is = (long long)limbs * kN, gs = NI * is, cs = (long long)G * gs;
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int i = c >> 1;
#pragma unroll
    for (int k = 0; k < 16; ++k) acc[c][k] = canon(acc[c][k], p, pinv);
    col_b_to_a(acc[c], Rs, j);
    if (tile * SL + s < G) {
      uint64_t* o = res + (c & 1) * cs + (long long)g * gs + (long long)i * is + ln + j;
#pragma unroll
      for (int k = 0; k < 16; ++k) o[16 * k] = d2u(acc[c][k]);
    }
  }
}

// The matrix-core MAC's arithmetic for primes below 2^50 (mac_mx.hpp): canonical words below 2^50 have
// seven balanced digits (the top one at most 4).  The byte-pair sums a_k (|a_k| < 2^29, a_6 the top
// digit's own sum, below 2^9) give d0 + 2^32 d1 + 2^64 d2 with |d0|, |d1| and |d2| < 2^46, taken by
// Horner's rule: u = d1 + (2^32 d2 mod p), then d0 + (2^32 u mod p).  A product by 2^32 is exact, and the FMA
// with its rounded quotient leaves the exact remainder, within 0.51 p for p near 2^50 (for small primes
// the words have fewer digits, the sums are smaller and a quotient off by a few units leaves a few p, far
// below 2^46).  Four steps of 16 babies stay below 4 (2^46 + 1.1 p) < 2^53, so the running sum is
// reduced once, in finish().
struct MxFp {
  static constexpr int ND = 7;
  typedef DevTables Tables;
  typedef double Acc;
  struct Consts {
    double p, pinv, k32;
    __device__ __forceinline__ void load(const DevTables& T, int pi) {
      p = T.p[pi];
      pinv = T.pinv[pi];
      k32 = 4294967296.0 * pinv;
    }
  };
  static __device__ __forceinline__ uint64_t digits(uint64_t x) {
    constexpr uint64_t M = 0x0080808080808080ULL;
    return (x + M) ^ M;
  }
  static __device__ __forceinline__ Acc zero() { return 0.0; }
  static __device__ __forceinline__ void add(Acc& x, const int (&a)[ND], const Consts& C) {
    const double d0 = __builtin_fma(65536.0, (double)a[1], (double)a[0]);
    const double d1 = __builtin_fma(65536.0, (double)a[3], (double)a[2]);
    const double d2 = __builtin_fma(4294967296.0, (double)a[6], __builtin_fma(65536.0, (double)a[5], (double)a[4]));
    const double u = d1 + __builtin_fma(-__builtin_rint(d2 * C.k32), C.p, d2 * 4294967296.0);
    x += d0 + __builtin_fma(-__builtin_rint(u * C.k32), C.p, u * 4294967296.0);
  }
  static __device__ __forceinline__ uint64_t finish(Acc x, const Consts& C) {
    const double r = reduce(x, C.p, C.pinv);  // within p/2 + 2
    return d2u(r < 0.0 ? r + C.p : r);
  }
};

// ----------------------------------------------------------------- the sidecar-shaped MAC
// holmes_mac_multi's layout (bench/cmp/kernels/holmes_mac.cu:359-402): one device pointer per input to
// its baby basis [nb][>= limbs][N] (baby stride bstride words), plaintext rows [groups * nb][>= limbs][N]
// (row stride pstride), res [2][groups][inputs][limbs][N], and the moduli as a device array (limb l uses
// primes[l]).  No context handle is needed: every workgroup derives its limb's Barrett constant from
// the prime (modarith64.hpp), so the entry works for any prime below 2^62 -- the reference's 59/60-bit
// chains included.  Products are reduced one by one and summed canonically.
constexpr int kAbiMaxInputs = 32;
constexpr int kAbiThreads = 128;
constexpr int kAbiTI = 2;
constexpr int kAbiTG = 8;

struct AbiInputs {
  const uint64_t* c0[kAbiMaxInputs];
  const uint64_t* c1[kAbiMaxInputs];
};

__global__ __launch_bounds__(kAbiThreads) void k_mac_multi_abi(uint64_t* __restrict__ res, AbiInputs in,
                                                               long long bstride, int nb, int ni, int G,
                                                               const uint64_t* __restrict__ pts, long long pstride,
                                                               int limbs, const uint64_t* __restrict__ primes,
                                                               int tiles_i) {
  const int l = blockIdx.y;
  const int units = kN / kAbiThreads;
  const int unit = blockIdx.x % units, tile = blockIdx.x / units;
  const int i0 = (tile % tiles_i) * kAbiTI, g0 = (tile / tiles_i) * kAbiTG;
  const long long ln = (long long)l * kN + unit * kAbiThreads + threadIdx.x;
  const Barrett64 br = barrett_make(primes[l]);
  const uint64_t p = br.p;
  uint64_t acc[kAbiTI][2][kAbiTG];
#pragma unroll
  for (int t = 0; t < kAbiTI; ++t)
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int g = 0; g < kAbiTG; ++g) acc[t][c][g] = 0;
  for (int b = 0; b < nb; ++b) {
    uint64_t w[kAbiTG];
#pragma unroll
    for (int g = 0; g < kAbiTG; ++g) {
      const int gg = g0 + g < G ? g0 + g : g0;  // clamped rows are computed but never stored
      w[g] = pts[((long long)gg * nb + b) * pstride + ln];
    }
#pragma unroll
    for (int t = 0; t < kAbiTI; ++t) {
      const int ii = i0 + t < ni ? i0 + t : i0;
      const uint64_t x0 = in.c0[ii][(long long)b * bstride + ln];
      const uint64_t x1 = in.c1[ii][(long long)b * bstride + ln];
#pragma unroll
      for (int g = 0; g < kAbiTG; ++g) {
        acc[t][0][g] = addmod64(acc[t][0][g], mulmod64(x0, w[g], br), p);
        acc[t][1][g] = addmod64(acc[t][1][g], mulmod64(x1, w[g], br), p);
      }
    }
  }
  const long long is = (long long)limbs * kN, gs = (long long)ni * is, cs = (long long)G * gs;
#pragma unroll
  for (int t = 0; t < kAbiTI; ++t) {
    if (i0 + t >= ni) break;
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int g = 0; g < kAbiTG; ++g)
        if (g0 + g < G) res[c * cs + (long long)(g0 + g) * gs + (long long)(i0 + t) * is + ln] = acc[t][c][g];
  }
}

}  // namespace
}  // namespace hck

extern "C" int holmes_mac_multi(uint64_t* res, const uint64_t* const* c0s, const uint64_t* const* c1s,
                                long long bstride, int nb, int inputs, const uint64_t* pts, long long pstride,
                                int groups, int ti, int limbs, const uint64_t* primes, const uint64_t* ratios,
                                const uint64_t* ks, void* stream) {
  (void)ratios;  // the caller's Barrett tables: this entry derives its constants from `primes`
  (void)ks;
  if (inputs < 1 || inputs > hck::kAbiMaxInputs) return -1;
  if (nb < 1) return -2;
  if (groups < 1 || groups > 16 || (groups > 8 && ti != 10116)) return -3;
  static const int kTiles[] = {1, 2, 4, 404, 408, 802, 804, 1601, 1602, 10108, 10116, 10204, 10208, 10402, 10404};
  bool known = false;
  for (int v : kTiles) known |= v == ti;
  if (!known) return -4;  // the reference's tile selector is validated, the tile here is this kernel's own
  if (!res || !c0s || !c1s || !pts || !primes || limbs < 1 || limbs > 65535) return HCK_ERR_ARG;
  hck::AbiInputs in{};
  for (int i = 0; i < inputs; ++i) {
    if (!c0s[i] || !c1s[i]) return HCK_ERR_ARG;
    in.c0[i] = c0s[i];
    in.c1[i] = c1s[i];
  }
  const int tiles_i = (inputs + hck::kAbiTI - 1) / hck::kAbiTI;
  const int tiles_g = (groups + hck::kAbiTG - 1) / hck::kAbiTG;
  const dim3 grid((unsigned)(hck::kN / hck::kAbiThreads * tiles_i * tiles_g), (unsigned)limbs);
  hck::k_mac_multi_abi<<<grid, hck::kAbiThreads, 0, (hipStream_t)stream>>>(res, in, bstride, nb, inputs, groups,
                                                                           pts, pstride, limbs, primes, tiles_i);
  HCK_CHECK_LAUNCH();
  return HCK_OK;
}

extern "C" int hck_bsgs_mac(const hck_context* ctx, int limbs, const int* prime_idx, int inputs, int babies,
                            int giants, const uint64_t* const* baby_c0, const uint64_t* const* baby_c1,
                            int64_t baby_stride, const uint64_t* pts, int64_t pt_stride, uint64_t* res,
                            void* stream) {
  if (!ctx || !prime_idx || !baby_c0 || !baby_c1 || !pts || !res) return HCK_ERR_ARG;
  if (limbs < 1 || limbs > hck::kMaxPrimes || inputs < 1 || babies < 1 || babies > hck::kMaxBabies || giants < 1)
    return HCK_ERR_ARG;
  hck::MacPrimes mp{};
  for (int l = 0; l < limbs; ++l) {
    if (prime_idx[l] < 0 || prime_idx[l] >= ctx->np) return HCK_ERR_ARG;
    mp.prime[l] = (uint8_t)prime_idx[l];
  }
  if (ctx->wide)
    return hck::wide_bsgs_mac(ctx, limbs, prime_idx, inputs, babies, giants, baby_c0, baby_c1, baby_stride, pts,
                              pt_stride, res, (hipStream_t)stream);
  hck::BabyPtrs bp{};
  for (int b = 0; b < babies; ++b) {
    if (!baby_c0[b] || !baby_c1[b]) return HCK_ERR_ARG;
    bp.c0[b] = baby_c0[b];
    bp.c1[b] = baby_c1[b];
  }
  if (hck::mx_pays_fp(inputs, babies, giants)) {
    hck::MxArgs A = hck::mx_args(limbs, mp.prime, inputs, babies, giants, baby_c0, baby_c1, baby_stride, pts, pt_stride, res);
    if (hck::mx_aligned(A)) {
      hck::mx_launch<hck::MxFp>(A, ctx->dev, (hipStream_t)stream);
      HCK_CHECK_LAUNCH();
      return HCK_OK;
    }
  }
  const int units_per_limb = hck::kN / hck::kMacThreads;
  const int total_units = limbs * units_per_limb;
  const int ti = hck::mac_tile_inputs(inputs, giants);
  const int tiles_i = (inputs + ti - 1) / ti, tiles_g = (giants + hck::kTG - 1) / hck::kTG;
  const int tiles = tiles_i * tiles_g;
  const long long units_padded = ((long long)total_units + hck::kXcds - 1) / hck::kXcds * hck::kXcds;
  const long long blocks = units_padded * tiles;
  if (blocks > 0x7fffffffLL) return HCK_ERR_ARG;
  auto k = ti == 1 ? hck::k_bsgs_mac<1> : ti == 2 ? hck::k_bsgs_mac<2> : ti == 3 ? hck::k_bsgs_mac<3> : hck::k_bsgs_mac<4>;
  k<<<dim3((unsigned)blocks), hck::kMacThreads, 0, (hipStream_t)stream>>>(
      res, bp, baby_stride, babies, inputs, giants, pts, pt_stride, limbs, mp, units_per_limb, tiles_i, tiles_g,
      total_units, ctx->dev);
  HCK_CHECK_LAUNCH();
  return HCK_OK;
}

extern "C" int hck_bsgs_mac_rows(const hck_context* ctx, int limbs, const int* prime_idx, int inputs, int babies,
                                 int giants, const uint64_t* const* baby_c0, const uint64_t* const* baby_c1,
                                 int64_t baby_stride, const double* pts, int64_t pt_stride, uint64_t* res,
                                 void* stream) {
  if (!ctx || !prime_idx || !baby_c0 || !baby_c1 || !pts || !res) return HCK_ERR_ARG;
  if (limbs < 1 || limbs > hck::kMaxPrimes || inputs < 1 || babies < 1 || babies > hck::kMaxBabies || giants < 1)
    return HCK_ERR_ARG;
  if (ctx->wide || inputs > HCK_MAC_ROWS_INPUTS) return HCK_ERR_UNSUPPORTED;
  hck::MacPrimes mp{};
  for (int l = 0; l < limbs; ++l) {
    if (prime_idx[l] < 0 || prime_idx[l] >= ctx->np) return HCK_ERR_ARG;
    mp.prime[l] = (uint8_t)prime_idx[l];
  }
  hck::BabyPtrs bp{};
  for (int b = 0; b < babies; ++b) {
    if (!baby_c0[b] || !baby_c1[b]) return HCK_ERR_ARG;
    bp.c0[b] = baby_c0[b];
    bp.c1[b] = baby_c1[b];
  }
  const int slots = hck::mr_slots(inputs), tiles_g = (giants + slots - 1) / slots;
  const long long blocks = (long long)limbs * 256 * tiles_g;
  if (blocks > 0x7fffffffLL) return HCK_ERR_ARG;
  auto k = inputs == 1 ? hck::k_mac_rows<1> : hck::k_mac_rows<2>;
  k<<<dim3((unsigned)blocks), 16 * slots, 0, (hipStream_t)stream>>>(
      res, bp, baby_stride, babies, giants, pts, pt_stride, limbs, mp, tiles_g, ctx->dev);
  HCK_CHECK_LAUNCH();
  return HCK_OK;
}
