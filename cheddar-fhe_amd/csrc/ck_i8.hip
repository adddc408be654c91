// Exact int8 matrix-core forms of the forward negacyclic NTT (4-step,
// 256 x 256) and of the fast BaseConv, plus a vector-unit BaseConv.
//
// Byte splitting. A residue x with |x| < 2^31 - 2^24 has a unique
// balanced base-256 form x = sum_i d_i 2^(8 i), d_i in [-128, 127]: the
// bytes of x + 0x80808080 with their top bit flipped (two instructions,
// pack_c). For a constant matrix T over Z_q the host stores, for every data
// digit i, T^(i) = T 2^(8 i) mod q (centred) split the same way into four
// byte planes T^(i)_j. Then
//   sum_n T[m][n] x_n  ==  sum_j 2^(8 j) D_j[m]   (mod q),
//   D_j[m] = sum_{n, i} T^(i)_j[m][n] d_i(x_n),
// and each D_j is one int8 matrix product with int32 accumulation over
// K = (input, digit). With K = 64 every |D_j| <= 64 * 2^14 = 2^20, so
// lo = D_0 + 2^8 D_1 and hi = D_2 + 2^8 D_3 stay within int32 and
// v = hi 2^16 + lo (|v| < 2^45) is exact in FP64; one FP64 reduction
// (k = rint(v / q), r = v - k q, exact) gives |r| <= q/2 + 1. No step
// rounds: the outputs are the exact residues.
//
// Operand layouts (gfx950, checked on the GPU): for
// v_mfma_i32_16x16x64_i8, lane l supplies A[l % 16][16 (l / 16) + b] and
// B[16 (l / 16) + b][l % 16] for byte b of its four registers and receives
// D[4 (l / 16) + v][l % 16] in accumulator v; v_mfma_i32_16x16x32_i8 is the
// same with eight bytes per lane. A lane's register t holds the four digits
// of one value (input 4 (l / 16) + t), so the reduction index k = (input,
// digit) pairs the same digit positions in A and B.
//
// 4-step transform. A limb x is the 256 x 256 matrix X[r][c] = x[c + 256 r].
// With psi the context's 2N-th root, psi1 = psi^256, omega = psi^512 and
// output position p = p_lo + 256 p_hi holding x(psi^(2 brv16(p) + 1)) (the
// order of NTTPhase1/NTTPhase2, src/core/NTT.cu:231-454):
//   column pass  Y[p_hi][c] = sum_r psi1^(r (2 brv8(p_hi) + 1)) X[r][c],
//                 Z = Y psi^(c (2 brv8(p_hi) + 1))        (4-step twiddle),
//   row pass     out[p_hi][p_lo] = sum_c omega^(c brv8(p_lo)) Z[p_hi][c].
// Each 256-point matrix is applied as two 16-point matrix stages
// (r = r0 + 16 r1, p_hi = p0 + 16 p1; c = c0 + 16 c1, p_lo = q0 + 16 q1):
//   A1[p1][r1]     = psi1^(16 r1 (2 brv4(p1) + 1)),
//   B1_p1[p0][r0]  = psi1^(r0 (2 brv4(p1) + 1) + 32 r0 brv4(p0)),
//   A3[q1][c1]     = omega^(16 c1 brv4(q1)),
//   B3_q1[q0][c0]  = omega^(c0 brv4(q1) + 16 c0 brv4(q0)),
// the inner twiddles folded into the second stage's 16 matrices. Between
// the two stages of a pass the values go through LDS (the matrix cores
// leave a stage's output index where the next stage needs its input index).
// The column pass reads canonical input as x - 2^30 (fits the digit range)
// and adds 2^30 * rowsum(A1) back through the accumulator's initial value.
// Intermediate values between the passes are centred int32 in dst, in
// 16 x 16 tiles (tile_word).
#include "ck_i8.h"
#include "ck_i8_arith.h"
#include "ck_radix16.h"

#include <algorithm>
#include <cstring>

namespace ck {
namespace {

constexpr int kN = 65536;
constexpr int kXs = 324;  // LDS words per 16 x 16 block of the exchange

typedef int v4i __attribute__((ext_vector_type(4)));

using i8::combine;
using i8::pack_c;
using i8::pack_off;
using i8::reduce_q;

// workgroup b runs on XCD b % 8: give each XCD a contiguous range of
// virtual blocks, so workgroups of one prime (adjacent jobs) share an L2
__device__ __forceinline__ int xcd_block(int b, int nwg) {
  const int x = b & 7, i = b >> 3;
  const int per = nwg >> 3, rem = nwg & 7;
  return x * per + (x < rem ? x : rem) + i;
}

__device__ __forceinline__ v4i mfma64(v4i a, v4i b, v4i c) {
  return __builtin_amdgcn_mfma_i32_16x16x64_i8(a, b, c, 0, 0, 0);
}

typedef const __attribute__((address_space(4))) Ntt8Job CJob;
typedef uint32_t v4u __attribute__((ext_vector_type(4)));

// data that streams through once (the intermediate tiles, the outputs):
// non-temporal accesses keep it from evicting the twiddle table and operand
// matrices, which every limb of a prime re-reads. The column pass reads its
// input with ordinary loads: it uses each 128-byte line in two 64-byte
// halves, and a line kept in L2 serves the second half.
__device__ __forceinline__ v4u ld4_nt(const uint32_t *p) {
  return __builtin_nontemporal_load((const v4u *)p);
}
__device__ __forceinline__ void st_nt(uint32_t *p, uint32_t v) {
  __builtin_nontemporal_store(v, p);
}
__device__ __forceinline__ void st4_nt(uint32_t *p, v4u v) {
  __builtin_nontemporal_store(v, (v4u *)p);
}

// Intermediate layout between the passes: 16 x 16 tiles of 1 KiB, tile
// (p1, cb) = rows 16 p1 .. 16 p1 + 15, columns 16 cb .. 16 cb + 15 at word
// (16 p1 + cb) * 256; inside a tile, row p0 = 4 g + v and column n sit at
// word (16 g + n) * 4 + v. The column pass writes a tile with one 16-byte
// store per lane (1 KiB per wave), the row pass of rows 16 p1.. reads the
// 16 KiB of its 16 tiles contiguously.
__device__ __forceinline__ int tile_word(int p1, int cb, int g, int n) {
  return (16 * p1 + cb) * 256 + (16 * g + n) * 4;
}

// Four planes of one 16 x 16 output tile (matrix a[j] times packed data b,
// plane 0 starting from c0).
struct Acc4 {
  v4i d[4];
};
__device__ __forceinline__ Acc4 mfma_tile(const v4i *a, v4i b, v4i c0) {
  const v4i zero = {0, 0, 0, 0};
  Acc4 r;
  r.d[0] = mfma64(a[0], b, c0);
  r.d[1] = mfma64(a[1], b, zero);
  r.d[2] = mfma64(a[2], b, zero);
  r.d[3] = mfma64(a[3], b, zero);
  return r;
}
// data as the A operand (rows = data vectors), matrix as B
__device__ __forceinline__ Acc4 mfma_tile_t(v4i a, const v4i *b) {
  const v4i zero = {0, 0, 0, 0};
  Acc4 r;
  r.d[0] = mfma64(a, b[0], zero);
  r.d[1] = mfma64(a, b[1], zero);
  r.d[2] = mfma64(a, b[2], zero);
  r.d[3] = mfma64(a, b[3], zero);
  return r;
}
// the four outputs of a lane, recombined and reduced, each step over all
// four before the next (four independent dependency chains)
__device__ __forceinline__ void reduce4(const Acc4 &A, double q, double qr, double r[4]) {
  double v[4];
#pragma unroll
  for (int i = 0; i < 4; i++) v[i] = combine(A.d[0][i], A.d[1][i], A.d[2][i], A.d[3][i]);
#pragma unroll
  for (int i = 0; i < 4; i++) r[i] = reduce_q(v[i], q, qr);
}

// Column pass: workgroup part of a limb's `parts` = 16 / cbs workgroups
// takes the 16-column blocks part, part + parts, ...: with two parts the
// workgroups of a limb (adjacent, so on one XCD and started together) read
// the two 64-byte halves of each 128-byte input line at about the same
// time. Wave w runs the first stage for r0 = 4w..4w+3 and the second stage for
// p1 = 4w..4w+3, so it keeps A1 and four B1 matrices in registers. Each
// stage is software-pipelined over its four tiles: the next tile's matrix
// products (and LDS reads) are issued before the current tile's
// recombination, and the next block's inputs load during the block.
__global__ __launch_bounds__(256, 3) void ntt8_cols_kernel(const Ntt8Job *__restrict__ jobs,
                                                           int nwg, int cbs, I8NttTabs T,
                                                           PrimeTab P) {
  __shared__ __align__(16) int xs[2][16 * kXs];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int g = lane >> 4, n = lane & 15;
  const int vb = xcd_block(blockIdx.x, nwg);
  const int parts = 16 / cbs;
  const int job = vb / parts, part = vb - job * parts;
  CJob &J = ((CJob *)jobs)[job];
  const int pr = J.prime, mont = J.mont;
  const uint32_t *__restrict__ src = J.src;
  uint32_t *__restrict__ dst = J.dst;

  const v4i *pl = (const v4i *)T.planes + (size_t)pr * kI8Ctx * 256;
  const int ca = mont ? kI8CtxA1Mont : kI8CtxA1;
  v4i a1[4], b1[4][4];
#pragma unroll
  for (int j = 0; j < 4; j++) a1[j] = pl[(ca * 4 + j) * 64 + lane];
#pragma unroll
  for (int k = 0; k < 4; k++)
#pragma unroll
    for (int j = 0; j < 4; j++) b1[k][j] = pl[((kI8CtxB1 + 4 * w + k) * 4 + j) * 64 + lane];
  const int *cp = T.corr + (pr * 2 + mont) * 16 + 4 * g;
  const v4i corr = {cp[0], cp[1], cp[2], cp[3]};
  const v4i zero = {0, 0, 0, 0};
  const double q = P.qd[pr], qr = P.qr[pr];
  // the twiddle table is tiled like the intermediate: one 16-byte load
  // gives a lane the four twiddles of its outputs in tile (p1, cb)
  const uint32_t *__restrict__ tw0 = T.tw + (size_t)pr * kN + (16 * g + n) * 4;
  // lane's first input word of a block: row 4w + 64 g, column n
  const uint32_t *in0 = src + (4 * w + 64 * g) * 256 + n;
  // this lane's 16-byte slot of tile (p1, cb)
  uint32_t *out0 = dst + (16 * g + n) * 4;

  uint32_t raw[4][4];
#pragma unroll
  for (int k = 0; k < 4; k++)
#pragma unroll
    for (int t = 0; t < 4; t++) raw[k][t] = in0[(k + 16 * t) * 256 + part * 16];

  for (int it = 0; it < cbs; it++) {
    const int cb = part + parts * it;
    int *X = xs[it & 1];
    // first stage: 16-point transforms along r1, tile r0 = 4w + k
    Acc4 acc[2];
    {
      const v4i b = {pack_off(raw[0][0]), pack_off(raw[0][1]), pack_off(raw[0][2]),
                     pack_off(raw[0][3])};
      acc[0] = mfma_tile(a1, b, corr);
    }
#pragma unroll
    for (int k = 0; k < 4; k++) {
      if (k < 3) {
        const v4i b = {pack_off(raw[k + 1][0]), pack_off(raw[k + 1][1]),
                       pack_off(raw[k + 1][2]), pack_off(raw[k + 1][3])};
        acc[(k + 1) & 1] = mfma_tile(a1, b, corr);
      }
      double r[4];
      reduce4(acc[k & 1], q, qr, r);
#pragma unroll
      for (int v = 0; v < 4; v++) X[(4 * g + v) * kXs + (4 * w + k) * 20 + n] = pack_c((int)r[v]);
    }
    // next block's inputs, in flight during the second stage (the last
    // iteration reloads its own block)
    {
      const int cbn = it + 1 < cbs ? cb + parts : cb;
#pragma unroll
      for (int k = 0; k < 4; k++)
#pragma unroll
        for (int t = 0; t < 4; t++) raw[k][t] = in0[(k + 16 * t) * 256 + cbn * 16];
    }
    __syncthreads();
    // second stage along r0 (tile p1 = 4w + k), then the 4-step twiddle;
    // one 16-byte store per lane writes the tile (p1, cb)
    v4u twv[2];
    twv[0] = *(const v4u *)(tw0 + (16 * (4 * w) + cb) * 256);
    v4i bx[2];
    const int *Xl = X + (4 * w) * kXs + (4 * g) * 20 + n;
    bx[0] = v4i{Xl[0], Xl[20], Xl[40], Xl[60]};
    acc[0] = mfma_tile(b1[0], bx[0], zero);
#pragma unroll
    for (int k = 0; k < 4; k++) {
      if (k < 3) {
        const int *Xk = Xl + (k + 1) * kXs;
        bx[(k + 1) & 1] = v4i{Xk[0], Xk[20], Xk[40], Xk[60]};
        twv[(k + 1) & 1] = *(const v4u *)(tw0 + (16 * (4 * w + k + 1) + cb) * 256);
        acc[(k + 1) & 1] = mfma_tile(b1[k + 1], bx[(k + 1) & 1], zero);
      }
      double r[4];
      reduce4(acc[k & 1], q, qr, r);
      v4u out;
#pragma unroll
      for (int v = 0; v < 4; v++)
        out[v] = (uint32_t)(int)mulmod_fq(r[v], (double)twv[k & 1][v], q, qr);
      st4_nt(out0 + (16 * (4 * w + k) + cb) * 256, out);
    }
  }
}

// Row pass (in place on dst): workgroup = one limb's 16-row blocks
// [part * rbs, +rbs). Wave w runs the first stage for rows 16 rb + 4w + k
// (one 16-byte load per lane and tile gives its four rows) and the second
// stage for q1 = 4w + k with the data as the A operand, so each lane ends
// with four rows of one output column. Software-pipelined like the column
// pass; the next block's tiles load while the current one is transformed.
__global__ __launch_bounds__(256, 3) void ntt8_rows_kernel(const Ntt8Job *__restrict__ jobs,
                                                           int nwg, int rbs, I8NttTabs T,
                                                           PrimeTab P) {
  __shared__ __align__(16) int xs[2][16 * kXs];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int g = lane >> 4, n = lane & 15;
  const int vb = xcd_block(blockIdx.x, nwg);
  const int parts = 16 / rbs;
  const int job = vb / parts, part = vb - job * parts;
  CJob &J = ((CJob *)jobs)[job];
  const int pr = J.prime;
  uint32_t *__restrict__ Z = J.dst;

  const v4i *pl = (const v4i *)T.planes + (size_t)pr * kI8Ctx * 256;
  v4i a3[4], b3[4][4];
#pragma unroll
  for (int j = 0; j < 4; j++) a3[j] = pl[(kI8CtxA3 * 4 + j) * 64 + lane];
#pragma unroll
  for (int k = 0; k < 4; k++)
#pragma unroll
    for (int j = 0; j < 4; j++) b3[k][j] = pl[((kI8CtxB3 + 4 * w + k) * 4 + j) * 64 + lane];
  const v4i zero = {0, 0, 0, 0};
  const double q = P.qd[pr], qr = P.qr[pr];

  const int rb0 = part * rbs, rb1 = rb0 + rbs;
  // tile (rb, c1 = 4g + t), rows 4w + k (k = 0..3 in one load), column c0 = n
  const uint32_t *in0 = Z + tile_word(0, 4 * g, w, n);
  v4u raw[4];
#pragma unroll
  for (int t = 0; t < 4; t++) raw[t] = ld4_nt(in0 + (16 * rb0 + t) * 256);

  for (int rb = rb0; rb < rb1; rb++) {
    int *W = xs[rb & 1];
    // first stage along c1 (row 16 rb + 4w + k): V[q1 = 4g + v][c0 = n]
    Acc4 acc[2];
    {
      const v4i b = {pack_c((int)raw[0][0]), pack_c((int)raw[1][0]), pack_c((int)raw[2][0]),
                     pack_c((int)raw[3][0])};
      acc[0] = mfma_tile(a3, b, zero);
    }
#pragma unroll
    for (int k = 0; k < 4; k++) {
      if (k < 3) {
        const v4i b = {pack_c((int)raw[0][k + 1]), pack_c((int)raw[1][k + 1]),
                       pack_c((int)raw[2][k + 1]), pack_c((int)raw[3][k + 1])};
        acc[(k + 1) & 1] = mfma_tile(a3, b, zero);
      }
      double r[4];
      reduce4(acc[k & 1], q, qr, r);
#pragma unroll
      for (int v = 0; v < 4; v++) W[(4 * w + k) * kXs + (4 * g + v) * 20 + n] = pack_c((int)r[v]);
    }
    // next block's tiles, in flight during the second stage
    {
      const int rbn = rb + 1 < rb1 ? rb + 1 : rb;
#pragma unroll
      for (int t = 0; t < 4; t++) raw[t] = ld4_nt(in0 + (16 * rbn + t) * 256);
    }
    __syncthreads();
    // the row block's tiles are all read: the outputs may overwrite them
    // second stage along c0 (q1 = 4w + k): rows as A (row n, c0 = 4g + t)
    const v4i *Wl = (const v4i *)&W[n * kXs + (4 * w) * 20 + 4 * g];
    uint32_t *out0 = Z + (16 * rb + 4 * g) * 256 + n + 16 * (4 * w);
    v4i ax[2];
    ax[0] = Wl[0];
    acc[0] = mfma_tile_t(ax[0], b3[0]);
#pragma unroll
    for (int k = 0; k < 4; k++) {
      if (k < 3) {
        ax[(k + 1) & 1] = Wl[5 * (k + 1)];  // + (k + 1) * 20 words
        acc[(k + 1) & 1] = mfma_tile_t(ax[(k + 1) & 1], b3[k + 1]);
      }
      double r[4];
      reduce4(acc[k & 1], q, qr, r);
#pragma unroll
      for (int v = 0; v < 4; v++) st_nt(out0 + v * 256 + 16 * k, canon_small(r[v], q));
    }
  }
}

// ---- one-pass transform -------------------------------------------------------

// Exchange between the two 16-point stages of a pass: 16 blocks of 16 x 16
// words, 20 words a row.
constexpr int kXb = 324;
// the same for 32 columns: blocks of 16 rows of 36 words
constexpr int kXc = 16 * 36;

// the modulus of a limb and the factor of fold_q
struct FoldQ {
  uint32_t q;
  int qinv, c;
};
__device__ __forceinline__ FoldQ fold_consts(const PrimeTab &P, int pr) {
  return FoldQ{P.q[pr], P.qinv[pr],
               __builtin_amdgcn_readfirstlane(i8::fold_factor(P.qr[pr]))};
}
// a lane's four outputs of a tile mod q (|r| < 0.71 q)
__device__ __forceinline__ void fold4(const Acc4 &A, const FoldQ &f, int r[4]) {
#pragma unroll
  for (int i = 0; i < 4; i++)
    r[i] = i8::fold_q(A.d[0][i], A.d[1][i], A.d[2][i], A.d[3][i], f.q, f.c);
}
__device__ __forceinline__ uint32_t canon_i(int r, uint32_t q) {  // |r| < q
  const uint32_t u = (uint32_t)r, v = u + q;
  return u < v ? u : v;
}

// Global access at a uniform base plus a 32-bit lane offset (scalar base
// addressing: no 64-bit lane addresses to keep in registers).
template <typename V>
__device__ __forceinline__ V ld_at(const void *base, uint32_t off) {
  typedef const __attribute__((address_space(1))) char gchar;
  return *(const __attribute__((address_space(1))) V *)((gchar *)base + off);
}
__device__ __forceinline__ void st4_at(void *base, uint32_t off, v4u v) {
  typedef __attribute__((address_space(1))) char gchar;
  *(__attribute__((address_space(1))) v4u *)((gchar *)base + off) = v;
}

// Forward transform of a whole limb by one workgroup of 8 waves: the column
// pass's output (128 packed words a lane) stays in registers. Wave w runs the
// first stage of a pass for tiles 2w, 2w + 1 and the second stage for the same
// pair, so that its second-stage matrices stay in registers and, in the column
// pass, its results are rows 32w .. 32w + 31 whole: the row pass then needs one
// 4 x 4 transpose between lane groups and no exchange of the limb.
//
// Column pass in blocks of 32 columns: a lane's 16-byte load holds the four
// columns 4 cq + e of one row, which are the same vector n = (cq, r0 & 1) of
// four tiles e. Software pipeline: between two barriers a wave runs the second
// stage of one block (two in the row pass) and the first stage of the next;
// blocks are loaded two ahead.
//
// Reads a limb and writes it once (the two-pass forms move it twice each way,
// at 4.4 to 4.8 TB/s), about 48 vector instructions an element against 61
// with FP64 recombination and 90 of the vector form. 2048 limbs: 470 -> 318
// us. A limb takes a CU 38 us: two waves per SIMD (235 registers hold the
// limb) keep the vector unit 55 % busy, the rest is waiting at barriers and
// for memory (252 us with loads and stores out of the way). A loop over limbs
// with the next one's loads issued early (256 registers, spills) took 350 us,
// one column block per barrier 343 us, non-temporal stores 326 us.
__global__ __launch_bounds__(512, 2) void ntt1p_fwd_kernel(const Ntt8Job *__restrict__ jobs,
                                                           int njobs, I8NttTabs T, PrimeTab P) {
  // two 32-column blocks of the column pass, four row blocks of the row pass
  static_assert(4 * kXb >= 2 * kXc, "exchange size");
  __shared__ __align__(16) int xs[4 * 16 * kXb];
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int g = lane >> 4, n = lane & 15;
  const v4i zero = {0, 0, 0, 0};
  CJob &J = ((CJob *)jobs)[xcd_block(blockIdx.x, njobs)];
  const int pr = J.prime, mont = J.mont;
  const uint32_t *src = J.src;
  uint32_t *dst = J.dst;
  const FoldQ f = fold_consts(P, pr);
  const uint32_t lane16 = 16 * lane;
  const int32_t *pl = T.planes + (size_t)pr * kI8Ctx * 1024;
  auto matrices = [&](int ca, int cb, v4i a[4], v4i b[2][4]) {
#pragma unroll
    for (int j = 0; j < 4; j++) a[j] = ld_at<v4i>(pl + (ca * 4 + j) * 256, lane16);
#pragma unroll
    for (int k = 0; k < 2; k++)
#pragma unroll
      for (int j = 0; j < 4; j++)
        b[k][j] = ld_at<v4i>(pl + ((cb + 2 * w + k) * 4 + j) * 256, lane16);
  };
  int Z[2][16][4];
  {
    // vector n = 2 cq + r0l: rows 2w + r0l + 16 (4 g + t), columns 4 cq + e
    const int cq = n >> 1, r0l = n & 1;
    const uint32_t in_off = 4 * ((64 * g + r0l) * 256 + 4 * cq);
    v4u raw[2][4];
    auto load = [&](int B) {
#pragma unroll
      for (int t = 0; t < 4; t++)
        raw[B & 1][t] = ld_at<v4u>(src + (2 * w + 16 * t) * 256 + 32 * B, in_off);
    };
    load(0);
    v4i a1[4], b1[2][4];
    matrices(mont ? kI8CtxA1Mont : kI8CtxA1, kI8CtxB1, a1, b1);
    const v4i corr = ld_at<v4i>(T.corr + (pr * 2 + mont) * 16, 16 * g);
    load(1);
    const int *tw0 = T.twm + (size_t)pr * kN + (size_t)(2 * w) * 4096;
    v4i tw[2][2][2];
    auto load_tw = [&](int B) {
#pragma unroll
      for (int c = 0; c < 2; c++)
#pragma unroll
        for (int k = 0; k < 2; k++)
          tw[B & 1][c][k] = ld_at<v4i>(tw0 + (16 * k + 2 * B + c) * 256, lane16);
    };
    load_tw(0);
    keep_loads();
    auto stage1 = [&](int B) {
      int r[4][4];
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const v4u *x = raw[B & 1];
        const v4i b = {pack_off(x[0][e]), pack_off(x[1][e]), pack_off(x[2][e]),
                       pack_off(x[3][e])};
        fold4(mfma_tile(a1, b, corr), f, r[e]);
      }
      int *X = &xs[(B & 1) * 16 * kXc + 4 * g * kXc + (2 * w + r0l) * 36 + 4 * cq];
#pragma unroll
      for (int v = 0; v < 4; v++)
        *(v4i *)(X + v * kXc) = v4i{pack_c(r[0][v]), pack_c(r[1][v]), pack_c(r[2][v]),
                                    pack_c(r[3][v])};
    };
    stage1(0);
    __syncthreads();
#pragma unroll
    for (int B = 0; B < 8; B++) {
      if (B + 1 < 8) load_tw(B + 1);
      if (B + 2 < 8) load(B + 2);
      keep_loads();
      if (B + 1 < 8) stage1(B + 1);
#pragma unroll
      for (int c = 0; c < 2; c++)
#pragma unroll
        for (int k = 0; k < 2; k++) {
          const int *X = &xs[(B & 1) * 16 * kXc + (2 * w + k) * kXc + 4 * g * 36 + 16 * c + n];
          const v4i bx = {X[0], X[36], X[72], X[108]};
          int y[4];
          fold4(mfma_tile(b1[k], bx, zero), f, y);
#pragma unroll
          for (int v = 0; v < 4; v++)
            Z[k][2 * B + c][v] =
                pack_c(i8::mont_centred(y[v], tw[B & 1][c][k][v], f.q, f.qinv));
        }
      __syncthreads();
    }
  }
  v4i a3[4], b3[2][4];
  matrices(kI8CtxA3, kI8CtxB3, a3, b3);
  keep_loads();
  // rows 16 (2w + k) + 4 g + v, columns 16 cb + n -> lane group = cb / 4
#pragma unroll
  for (int k = 0; k < 2; k++)
#pragma unroll
    for (int cl = 0; cl < 4; cl++)
#pragma unroll
      for (int v = 0; v < 4; v++)
        transpose_groups(Z[k][cl][v], Z[k][4 + cl][v], Z[k][8 + cl][v], Z[k][12 + cl][v]);
  auto stage3 = [&](int s) {  // rows 16 (2w + k) + s
    const int h = s >> 2, v0 = s & 3;
#pragma unroll
    for (int k = 0; k < 2; k++) {
      const v4i b = {Z[k][4 * h][v0], Z[k][4 * h + 1][v0], Z[k][4 * h + 2][v0],
                     Z[k][4 * h + 3][v0]};
      int r[4];
      fold4(mfma_tile(a3, b, zero), f, r);
      int *W = &xs[(s & 3) * 16 * kXb + 4 * g * kXb + (2 * w + k) * 20 + n];
#pragma unroll
      for (int v = 0; v < 4; v++) W[v * kXb] = pack_c(r[v]);
    }
  };
  stage3(0);
  stage3(1);
  __syncthreads();
  // rows s + 16 n, columns 16 (2w + k) + 4 g + v: 16 bytes a lane
  const uint32_t out_off = 4 * (16 * n * 256 + 4 * g);
#pragma unroll
  for (int s = 0; s < 16; s++) {
    if (s + 2 < 16) stage3(s + 2);
#pragma unroll
    for (int k = 0; k < 2; k++) {
      const v4i bx = *(const v4i *)&xs[(s & 3) * 16 * kXb + (2 * w + k) * kXb + n * 20 + 4 * g];
      int r[4];
      fold4(mfma_tile(b3[k], bx, zero), f, r);
      st4_at(dst + s * 256 + 32 * w + 16 * k, out_off,
                v4u{canon_i(r[0], f.q), canon_i(r[1], f.q), canon_i(r[2], f.q),
                    canon_i(r[3], f.q)});
    }
    if (s & 1) __syncthreads();
  }
}

// Inverse transform of a whole limb, the mirror image: row pass (contract
// q0, then q1), the inverse 4-step twiddle, the transpose between lane groups,
// column pass (contract p0, then p1), then the limb's constant. 2048 limbs: 540
// (two FP64 passes) -> 333 us, bound as the forward transform. Step s of the
// row pass takes rows s + 16 n, vector n of every tile; step c1 of the column
// pass columns 16 c1 .. 16 c1 + 15. PROD: the input is src (*) src2 (Montgomery).
template <bool PROD>
__global__ __launch_bounds__(512, 2) void ntt1p_inv_kernel(const Inv1pJob *__restrict__ jobs,
                                                           int njobs, I8InvTabs T, PrimeTab P) {
  __shared__ __align__(16) int xs[4 * 16 * kXb];
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int g = lane >> 4, n = lane & 15;
  const v4i zero = {0, 0, 0, 0};
  typedef const __attribute__((address_space(4))) Inv1pJob CInv;
  CInv &J = ((CInv *)jobs)[xcd_block(blockIdx.x, njobs)];
  const int pr = J.prime;
  const uint32_t *src = J.src, *src2 = J.src2;
  uint32_t *dst = J.dst;
  const FoldQ f = fold_consts(P, pr);
  const uint32_t lane16 = 16 * lane;
  const int32_t *pl = T.planes + (size_t)pr * kI8InvCtx * 1024;
  // the common matrix, and the second-stage matrices 2w, 2w + 1 from context cb
  v4i a[4], b[2][4];
  auto second = [&](int cb) {
#pragma unroll
    for (int k = 0; k < 2; k++)
#pragma unroll
      for (int j = 0; j < 4; j++)
        b[k][j] = ld_at<v4i>(pl + ((cb + 2 * w + k) * 4 + j) * 256, lane16);
  };
  int Z[2][16][4];
  {
    // row s + 16 n, columns 16 (2w + k) + 4 g + t
    const uint32_t in_off = 4 * (16 * n * 256 + 4 * g);
    constexpr int kAhead = PROD ? 3 : 4;
    v4u raw[4][2], raw2[4][2];
    auto load = [&](int s) {
#pragma unroll
      for (int k = 0; k < 2; k++) {
        raw[s & 3][k] = ld_at<v4u>(src + s * 256 + 32 * w + 16 * k, in_off);
        if (PROD) raw2[s & 3][k] = ld_at<v4u>(src2 + s * 256 + 32 * w + 16 * k, in_off);
      }
    };
    const int *tw0 = T.twm + (size_t)pr * kN + (size_t)(2 * w) * 4096;
    v4i tw[2][2];
    auto load_tw = [&](int s) {
#pragma unroll
      for (int k = 0; k < 2; k++)
        tw[s & 1][k] = ld_at<v4i>(tw0 + (16 * k + s) * 256, lane16);
    };
    load(0);
    load(1);
#pragma unroll
    for (int j = 0; j < 4; j++) a[j] = ld_at<v4i>(pl + j * 256, lane16);
    second(kI8InvCtxRow);
    const v4i corr = ld_at<v4i>(T.corr + pr * 16, 16 * g);
#pragma unroll
    for (int s = 2; s < kAhead; s++) load(s);
    load_tw(0);
    keep_loads();
    auto stage1 = [&](int s) {
      int r[2][4];
#pragma unroll
      for (int k = 0; k < 2; k++) {
        v4u x = raw[s & 3][k];
        if (PROD)
#pragma unroll
          for (int t = 0; t < 4; t++)
            x[t] = sum_reduce((uint64_t)x[t] * raw2[s & 3][k][t], f.q, f.qinv);
        const v4i d = {pack_off(x[0]), pack_off(x[1]), pack_off(x[2]), pack_off(x[3])};
        fold4(mfma_tile(a, d, corr), f, r[k]);
      }
      int *X = &xs[(s & 3) * 16 * kXb + 4 * g * kXb + n * 20 + 2 * w];
#pragma unroll
      for (int v = 0; v < 4; v++)
        *(int2 *)(X + v * kXb) = make_int2(pack_c(r[0][v]), pack_c(r[1][v]));
    };
    stage1(0);
    stage1(1);
    __syncthreads();
#pragma unroll
    for (int s = 0; s < 16; s++) {
      if (s + 1 < 16) load_tw(s + 1);
      if (s + kAhead < 16) load(s + kAhead);
      keep_loads();
      if (s + 2 < 16) stage1(s + 2);
#pragma unroll
      for (int k = 0; k < 2; k++) {
        const v4i d = *(const v4i *)&xs[(s & 3) * 16 * kXb + (2 * w + k) * kXb + n * 20 + 4 * g];
        int y[4];
        fold4(mfma_tile(b[k], d, zero), f, y);
#pragma unroll
        for (int v = 0; v < 4; v++)
          Z[k][s][v] = pack_c(i8::mont_centred(y[v], tw[s & 1][k][v], f.q, f.qinv));
      }
      if (s & 1) __syncthreads();
    }
  }
  second(kI8InvCtxCol);
  keep_loads();
  // columns 2w + k + 16 (4 g + v), rows s + 16 n -> lane group = s / 4
#pragma unroll
  for (int k = 0; k < 2; k++)
#pragma unroll
    for (int sl = 0; sl < 4; sl++)
#pragma unroll
      for (int v = 0; v < 4; v++)
        transpose_groups(Z[k][sl][v], Z[k][4 + sl][v], Z[k][8 + sl][v], Z[k][12 + sl][v]);
  auto stage3 = [&](int c1) {  // columns 16 c1 + 2w + k
    const int h = c1 >> 2, v0 = c1 & 3;
#pragma unroll
    for (int k = 0; k < 2; k++) {
      const v4i d = {Z[k][4 * h][v0], Z[k][4 * h + 1][v0], Z[k][4 * h + 2][v0],
                     Z[k][4 * h + 3][v0]};
      int r[4];
      fold4(mfma_tile(a, d, zero), f, r);
      int *W = &xs[(c1 & 3) * 16 * kXb + 4 * g * kXb + (2 * w + k) * 20 + n];
#pragma unroll
      for (int v = 0; v < 4; v++) W[v * kXb] = pack_c(r[v]);
    }
  };
  stage3(0);
  stage3(1);
  __syncthreads();
  // rows 2w + k + 16 n, columns 16 c1 + 4 g + v: 16 bytes a lane
  const uint32_t out_off = 4 * (16 * n * 256 + 4 * g);
  const int c1m = J.c1m, centred = J.centred;
  const uint32_t above = centred ? (f.q - 1) >> 1 : f.q - 1;
#pragma unroll
  for (int c1 = 0; c1 < 16; c1++) {
    if (c1 + 2 < 16) stage3(c1 + 2);
#pragma unroll
    for (int k = 0; k < 2; k++) {
      const v4i d = *(const v4i *)&xs[(c1 & 3) * 16 * kXb + (2 * w + k) * kXb + n * 20 + 4 * g];
      int r[4];
      fold4(mfma_tile_t(d, b[k]), f, r);
      v4u o;
#pragma unroll
      for (int v = 0; v < 4; v++) {
        const uint32_t u = canon_i(i8::mont_centred(r[v], c1m, f.q, f.qinv), f.q);
        o[v] = u > above ? u - f.q : u;
      }
      st4_at(dst + (2 * w + k) * 256 + 16 * c1, out_off, o);
    }
    if (c1 & 1) __syncthreads();
  }
}

// ---- BaseConv ---------------------------------------------------------------

typedef const __attribute__((address_space(4))) BconvI8Inst CBInst;

// int8 form: workgroup = 256 positions of one instance (64 per wave, four
// 16-position tiles). Rows = 16 destinations per tile, K = 8 sources x 4
// digits per v_mfma_i32_16x16x32_i8 (KS <= 3 k-steps for up to 8 KS
// sources: each plane sums at most 96 digit products, |D_j| < 2^21).
// Source indices past S are clamped to 0 (their plane bytes are 0), so every
// load is unconditional.
template <int KS, class Inst>
__device__ __forceinline__ void bconv_i8_body(Inst &I, const PrimeTab &P) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int g = lane >> 4, n = lane & 15;
  const int S = I.S, D = I.D, canonical = I.canonical;
  const int base = blockIdx.x * 256 + w * 64 + n;
  const int32_t *__restrict__ src = I.src;
  const int64_t *__restrict__ planes = I.planes;

  int raw[4][KS][2];
#pragma unroll
  for (int ks = 0; ks < KS; ks++)
#pragma unroll
    for (int e = 0; e < 2; e++) {
      const int k = 8 * ks + 2 * g + e;
      const int32_t *sp = src + (size_t)(k < S ? k : 0) * kN + base;
#pragma unroll
      for (int t = 0; t < 4; t++) raw[t][ks][e] = sp[16 * t];
    }
  int64_t b[4][KS];
#pragma unroll
  for (int t = 0; t < 4; t++)
#pragma unroll
    for (int ks = 0; ks < KS; ks++)
      b[t][ks] = (int64_t)(uint32_t)pack_c(raw[t][ks][0]) |
                 ((int64_t)(uint32_t)pack_c(raw[t][ks][1]) << 32);

  const int nks = (S + 7) >> 3;  // this instance's k-steps (plane layout)
  const v4i zero = {0, 0, 0, 0};
  for (int mt = 0; mt * 16 < D; mt++) {
    int64_t a[KS][4];
#pragma unroll
    for (int ks = 0; ks < KS; ks++)
#pragma unroll
      for (int j = 0; j < 4; j++)
        a[ks][j] = ks < nks ? planes[((mt * nks + ks) * 4 + j) * 64 + lane] : 0;
    double qv[4], qrv[4];
    uint32_t *dp[4];
#pragma unroll
    for (int v = 0; v < 4; v++) {
      const int d = mt * 16 + 4 * g + v;
      const bool ok = d < D;
      const int dd = ok ? d : 0;
      const int p = I.dst_prime[dd];
      qv[v] = P.qd[p];
      qrv[v] = P.qr[p];
      dp[v] = ok ? I.dst + (size_t)I.dst_limb[dd] * kN : nullptr;
    }
#pragma unroll
    for (int t = 0; t < 4; t++) {
      v4i d[4];
#pragma unroll
      for (int j = 0; j < 4; j++) {
        v4i acc = zero;
#pragma unroll
        for (int ks = 0; ks < KS; ks++)
          acc = __builtin_amdgcn_mfma_i32_16x16x32_i8(a[ks][j], b[t][ks], acc, 0, 0, 0);
        d[j] = acc;
      }
#pragma unroll
      for (int v = 0; v < 4; v++) {
        if (dp[v]) {
          const double r = reduce_q(combine(d[0][v], d[1][v], d[2][v], d[3][v]), qv[v], qrv[v]);
          dp[v][base + 16 * t] = canonical ? canon_small(r, qv[v]) : (uint32_t)(int)r;
        }
      }
    }
  }
}

template <int KS>
__global__ __launch_bounds__(256) void bconv_i8_kernel(const BconvI8Inst *__restrict__ insts,
                                                       PrimeTab P) {
  CBInst &I = ((CBInst *)insts)[blockIdx.y];
  bconv_i8_body<KS>(I, P);
}

template <int KS>
__global__ __launch_bounds__(256) void bconv_i8_arg_kernel(const BconvI8Launch L,
                                                           PrimeTab P) {
  bconv_i8_body<KS>(L.inst[blockIdx.y], P);
}

// Vector-unit form: one position per thread, the table row of each
// destination from scalar loads; per destination sum_i v_i hi_i and
// sum_i v_i lo_i in exact FP64 (|v| < 2^30, halves < 2^16, S <= 24 terms:
// below 2^51), then hi 2^16 + lo reduced as in the fused column pass.
__global__ __launch_bounds__(256) void bconv_valu_kernel(const BconvI8Inst *__restrict__ insts,
                                                         PrimeTab P) {
  CBInst &I = ((CBInst *)insts)[blockIdx.y];
  const int pos = blockIdx.x * 256 + threadIdx.x;
  const int S = I.S, D = I.D, canonical = I.canonical;
  double v[kMaxBconvSrc];
#pragma unroll
  for (int i = 0; i < kMaxBconvSrc; i++) {
    const int32_t x = I.src[(size_t)(i < S ? i : 0) * kN + pos];
    v[i] = i < S ? (double)x : 0.0;
  }
  typedef const __attribute__((address_space(4))) double CD;
  for (int d = 0; d < D; d++) {
    CD *row = (CD *)I.ftab + (size_t)d * S * 2;
    double hi = 0.0, lo = 0.0;
#pragma unroll
    for (int i = 0; i < kMaxBconvSrc; i++) {
      if (i < S) {
        hi = __builtin_fma(v[i], row[2 * i], hi);
        lo = __builtin_fma(v[i], row[2 * i + 1], lo);
      }
    }
    const int p = I.dst_prime[d];
    const ModF mf{P.qd[p], P.qr[p]};
    const double big = hi * 65536.0;
    const double k = __builtin_rint(big * mf.qinv);
    const double r = reduce_f(__builtin_fma(-k, mf.q, big) + lo, mf);
    I.dst[(size_t)I.dst_limb[d] * kN + pos] =
        canonical ? canon_small(r, mf.q) : (uint32_t)(int32_t)r;
  }
}

// ---- BaseConv fused with the forward column stages -------------------------

struct BcolsByValue {
  BcolsLaunch L;
  __device__ __forceinline__ BcolsQuad quad(int y) const { return L.quad[y]; }
};
struct BcolsTable {
  const BcolsQuad *__restrict__ quads;
  __device__ __forceinline__ BcolsQuad quad(int y) const {
    typedef const __attribute__((address_space(4))) BcolsQuad CQuad;
    CQuad *p = (CQuad *)quads + y;
    BcolsQuad q;
    q.src = p->src;
    q.planes = p->planes;
    for (int i = 0; i < 4; i++) {
      q.dst[i] = p->dst[i];
      q.prime[i] = p->prime[i];
    }
    q.S = p->S;
    return q;
  }
};

// BaseConv of 16 rows (16 k apart) at one column for the lane's destination:
// STEPS products of PER sources a lane (bconv_quad_planes), 16x16x32 for one
// step of up to 2, else 16x16x64. Sources past S re-read source 0 (their
// plane bytes are 0), so every load is unconditional and a batch of them is
// in flight before its first product.
template <int STEPS, int PER>
__device__ __forceinline__ void bconv_rows16(const int32_t *src, uint32_t off, int S,
                                             const int32_t *planes, int lane, double x[16]) {
  const int g = lane >> 4;
  const v4i zero = {0, 0, 0, 0};
  typedef const __attribute__((address_space(1))) char gchar;
  typedef const __attribute__((address_space(1))) int gint;
  gchar *base = (gchar *)src;
  uint32_t o[STEPS][PER];
#pragma unroll
  for (int ks = 0; ks < STEPS; ks++)
#pragma unroll
    for (int t = 0; t < PER; t++) {
      const int s = 4 * PER * ks + PER * g + t;
      o[ks][t] = off + (uint32_t)(s < S ? s : 0) * (4 * kN);
    }
  constexpr bool kNarrow = STEPS == 1 && PER <= 2;
  int64_t a32 = 0;
  v4i a64[STEPS];
#pragma unroll
  for (int ks = 0; ks < STEPS; ks++)
    if (kNarrow)
      a32 = ((const int64_t *)planes)[lane];
    else
      a64[ks] = ((const v4i *)planes)[64 * ks + lane];
  constexpr int kB = STEPS * PER <= 2 ? 16 : STEPS * PER <= 4 ? 8 : 4;  // rows of a load batch
#pragma unroll
  for (int k0 = 0; k0 < 16; k0 += kB) {
    int raw[kB][STEPS][PER];
#pragma unroll
    for (int k = 0; k < kB; k++)
#pragma unroll
      for (int ks = 0; ks < STEPS; ks++)
#pragma unroll
        for (int t = 0; t < PER; t++)
          raw[k][ks][t] = *(gint *)(base + 16384 * (k0 + k) + o[ks][t]);
#pragma unroll
    for (int k = 0; k < kB; k++) {
      v4i d = zero;
#pragma unroll
      for (int ks = 0; ks < STEPS; ks++) {
        int b[4] = {0, 0, 0, 0};
#pragma unroll
        for (int t = 0; t < PER; t++) b[t] = pack_c(raw[k][ks][t]);
        if (kNarrow) {
          const int64_t b32 = (int64_t)(uint32_t)b[0] | ((int64_t)(uint32_t)b[1] << 32);
          d = __builtin_amdgcn_mfma_i32_16x16x32_i8(a32, b32, d, 0, 0, 0);
        } else {
          d = mfma64(a64[ks], v4i{b[0], b[1], b[2], b[3]}, d);
        }
      }
      x[k0 + k] = combine(d[0], d[1], d[2], d[3]);
    }
  }
}

// ModSwitchMatrixMult (src/core/ModSwitch.cu:23-171) and the column stages of
// NTTPhase1 (src/core/NTT.cu:231-330) for four destination limbs at once.
//
// A workgroup of NC waves owns NC columns of a quad. One matrix product
// gives a wave the BaseConv of 16 positions for the quad's four
// destinations, lane group g holding destination g (bconv_quad_planes), so
// the sources are read once per four destinations and the lanes keep their
// values in registers for the column stages: lane (g, n) transforms column
// n % NC, first phase rows rb + 16 k with rb = (16 / NC) wave + n / NC,
// second phase rows 16 rb + j. The BaseConv sums enter the butterflies
// unreduced: below 2^46 in magnitude, they stay below 2^47 on the path that
// is only added to (eight sums of products below 2^31), inside the 2^50 of
// mulmod_fq and reduce_f.
//
// Bound by vector issue: about 850 instructions a wave (512 of them the
// butterflies) at the 1.9 GHz that FP64 runs at, 83 % of the time of a full
// chip. The form before it, one limb per workgroup with the BaseConv in FP64
// on the vector unit, took 1260 and read the sources for every destination:
// 72 limbs of 8 sources 19.9 -> 16.3 us, 42 of 15 sources 20.8 -> 14.5 us;
// against BaseConv as its own int8 step and a plain column pass, 4128 limbs
// of 8 sources 970 -> 739 us. Handing the phases over as int32 (half the
// LDS, three workgroups per CU) cost 10 % more instructions and 13 % time.
template <class D, int NC, int WIDTH>
__global__ __launch_bounds__(64 * NC, 4) void bconv_i8_cols(const D desc, const PrimeTab P,
                                                           const uint32_t *__restrict__ tw) {
  constexpr int kRows = 16 / NC;           // row groups rb of one wave
  constexpr int kShare = 32 / NC;          // column tiles in a 128-byte line
  constexpr int kTiles = 256 / NC;
  __shared__ double ldsd[4 * 256 * NC];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int g = lane >> 4, n = lane & 15;
  // workgroup i runs on XCD i mod 8: the tiles of one line share an XCD
  const int b = blockIdx.x;
  const int c0 = (((b & 7) * kShare) | ((b >> 3) & (kShare - 1))) * NC;
  const BcolsQuad Q = desc.quad(b / kTiles);
  const int cc = n % NC, rl = n / NC;
  const int rb = wave * kRows + rl;
  // the lane's destination
  uint32_t *dst = g == 0 ? Q.dst[0] : g == 1 ? Q.dst[1] : g == 2 ? Q.dst[2] : Q.dst[3];
  const int prime = g == 0 ? Q.prime[0] : g == 1 ? Q.prime[1] : g == 2 ? Q.prime[2] : Q.prime[3];
  const double q = P.qd[prime], qr = P.qr[prime];
  const ModF m{q, qr};
  const uint32_t *__restrict__ w = tw + (size_t)prime * kN;
  uint32_t t1[15], t2[15];
#pragma unroll
  for (int s = 0; s < 4; s++)
#pragma unroll
    for (int blk = 0; blk < (1 << s); blk++) {
      t1[(1 << s) - 1 + blk] = w[(1 << s) + blk];
      t2[(1 << s) - 1 + blk] = w[(16 << s) + (rb << s) + blk];
    }
  double x[16];
  const uint32_t off = 4u * (uint32_t)(rb * 256 + c0 + cc);
  const int S = Q.S;
  if (S <= 4)
    bconv_rows16<1, 1>(Q.src, off, S, Q.planes, lane, x);
  else if (WIDTH == 0 || S <= 8)
    bconv_rows16<1, 2>(Q.src, off, S, Q.planes, lane, x);
  else if (S <= 12)
    bconv_rows16<1, 3>(Q.src, off, S, Q.planes, lane, x);
  else if (WIDTH == 1 || S <= 16)
    bconv_rows16<1, 4>(Q.src, off, S, Q.planes, lane, x);
  else if constexpr (WIDTH == 2)
    bconv_rows16<2, 3>(Q.src, off, S, Q.planes, lane, x);
  ct16(x, t1, q, qr);
  // hand-off in LDS, rows of NC doubles; within 16 lanes (one LDS cycle of
  // 128 bytes) the writes cover kRows adjacent rows and the reads kRows rows
  // 16 apart: rows are swapped by their block number so that both cover all
  // banks
  double *tile = ldsd + g * 256 * NC + cc;
#pragma unroll
  for (int k = 0; k < 16; k++) tile[(16 * k + (rb ^ (k & (kRows - 1)))) * NC] = x[k];
  __syncthreads();
#pragma unroll
  for (int j = 0; j < 16; j++) x[j] = tile[(16 * rb + (j ^ rl)) * NC];
  ct16(x, t2, q, qr);
  if (dst) {
    typedef __attribute__((address_space(1))) uint32_t guint;
    guint *o = (guint *)dst + (size_t)(16 * rb) * 256 + c0 + cc;
#pragma unroll
    for (int j = 0; j < 16; j++) o[j * 256] = (uint32_t)(int32_t)reduce_f(x[j], m);
  }
}

// ---- host tables ------------------------------------------------------------

uint32_t brv_n(uint32_t x, int bits) {
  uint32_t r = 0;
  for (int i = 0; i < bits; i++) r |= ((x >> i) & 1u) << (bits - 1 - i);
  return r;
}

}  // namespace

int ntt8_tables(Context &c, I8NttTabs *out) {
  std::lock_guard<std::mutex> lock(c.tables_mu);
  if (c.i8_planes) {
    *out = I8NttTabs{c.i8_planes, c.i8_corr, c.i8_tw, c.i8_twm};
    return kOk;
  }
  const int np = c.num_primes;
  std::vector<int32_t> planes((size_t)np * kI8Ctx * 1024);
  std::vector<int32_t> corr((size_t)np * 32);
  std::vector<uint32_t> tw((size_t)np * kN);
  std::vector<int32_t> twm((size_t)np * kN);
  uint32_t T[16][16];
  for (int pi = 0; pi < np; pi++) {
    const uint32_t q = c.primes[pi];
    const uint32_t psi = c.psi[pi];
    const uint32_t psi1 = h_powmod(psi, 256, q), om = h_powmod(psi, 512, q);
    const uint32_t rmod = (uint32_t)((1ull << 32) % q);
    int32_t *pp = planes.data() + (size_t)pi * kI8Ctx * 1024;
    // A1 (plain and times R) with its offset corrections
    for (int mont = 0; mont < 2; mont++) {
      for (int p1 = 0; p1 < 16; p1++)
        for (int r1 = 0; r1 < 16; r1++) {
          uint32_t v = h_powmod(psi1, 16ull * r1 * (2 * brv_n(p1, 4) + 1), q);
          T[p1][r1] = mont ? h_mulmod(v, rmod, q) : v;
        }
      i8::ctx_planes(T, q, pp + (size_t)(kI8CtxA1 + mont) * 1024);
      for (int m = 0; m < 16; m++) {
        uint64_t s = 0;
        for (int r1 = 0; r1 < 16; r1++) s += T[m][r1];
        corr[(size_t)pi * 32 + mont * 16 + m] =
            i8::centre_h((uint64_t)h_mulmod((uint32_t)(s % q), (1u << 30) % q, q), q);
      }
    }
    for (int p1 = 0; p1 < 16; p1++) {
      for (int p0 = 0; p0 < 16; p0++)
        for (int r0 = 0; r0 < 16; r0++)
          T[p0][r0] = h_powmod(psi1, (uint64_t)r0 * (2 * brv_n(p1, 4) + 1) +
                                         32ull * r0 * brv_n(p0, 4), q);
      i8::ctx_planes(T, q, pp + (size_t)(kI8CtxB1 + p1) * 1024);
    }
    for (int q1 = 0; q1 < 16; q1++)
      for (int c1 = 0; c1 < 16; c1++) T[q1][c1] = h_powmod(om, 16ull * c1 * brv_n(q1, 4), q);
    i8::ctx_planes(T, q, pp + (size_t)kI8CtxA3 * 1024);
    for (int q1 = 0; q1 < 16; q1++) {
      for (int q0 = 0; q0 < 16; q0++)
        for (int c0 = 0; c0 < 16; c0++)
          T[q0][c0] = h_powmod(om, (uint64_t)c0 * brv_n(q1, 4) + 16ull * c0 * brv_n(q0, 4), q);
      i8::ctx_planes(T, q, pp + (size_t)(kI8CtxB3 + q1) * 1024);
    }
    // 4-step twiddle psi^(c (2 brv8(p) + 1)) of row p, column c, stored in
    // the tiled layout of the intermediate (tile_word)
    uint32_t *tp = tw.data() + (size_t)pi * kN;
    for (int p = 0; p < 256; p++) {
      const uint32_t step = h_powmod(psi, 2 * brv_n(p, 8) + 1, q);
      uint64_t x = 1;
      const int p1 = p >> 4, p0 = p & 15;
      for (int col = 0; col < 256; col++) {
        const int cb = col >> 4, cn = col & 15;
        const int at = (16 * p1 + cb) * 256 + (16 * (p0 >> 2) + cn) * 4 + (p0 & 3);
        tp[at] = (uint32_t)x;
        twm[(size_t)pi * kN + at] = i8::centre_h(x * rmod, q);
        x = x * step % q;
      }
    }
  }
  auto up = [&](auto **dst, const auto &v) {
    int rc = check_hip(hipMalloc((void **)dst, v.size() * sizeof(v[0])), "hipMalloc(int8 tables)");
    if (rc) return rc;
    c.allocations.push_back((void *)*dst);
    return check_hip(hipMemcpy((void *)*dst, v.data(), v.size() * sizeof(v[0]),
                               hipMemcpyHostToDevice),
                     "hipMemcpy(int8 tables)");
  };
  int32_t *dp = nullptr, *dc = nullptr;
  uint32_t *dt = nullptr;
  int32_t *dm = nullptr;
  int rc = up(&dp, planes);
  if (!rc) rc = up(&dc, corr);
  if (!rc) rc = up(&dt, tw);
  if (!rc) rc = up(&dm, twm);
  if (rc) return rc;
  c.i8_planes = dp;
  c.i8_corr = dc;
  c.i8_tw = dt;
  c.i8_twm = dm;
  *out = I8NttTabs{dp, dc, dt, dm};
  return kOk;
}

// Tables of the one-pass inverse transform: with omega = psi^512,
//   context 0          A[c0][q0]  = omega^(-16 c0 brv4(q0)), both passes,
//   kI8InvCtxRow + c0  [c1][q1]   = omega^(-(c0 + 16 c1) brv4(q1)),
//   kI8InvCtxCol + r0  [r1][p1]   = psi^(-256 (r0 + 16 r1)(2 brv4(p1) + 1)),
// twm: psi^(-c (2 brv8(p) + 1)) 2^32, centred, for column c = c0 + 16 (4 g + v)
// and row p = s + 16 n at word ((16 c0 + s) 64 + 16 g + n) 4 + v.
int ntt1p_inv_tables(Context &c, I8InvTabs *out) {
  std::lock_guard<std::mutex> lock(c.tables_mu);
  if (c.i8_inv_planes) {
    *out = I8InvTabs{c.i8_inv_planes, c.i8_inv_corr, c.i8_inv_twm};
    return kOk;
  }
  const int np = c.num_primes;
  std::vector<int32_t> planes((size_t)np * kI8InvCtx * 1024), corr((size_t)np * 16);
  std::vector<int32_t> twm((size_t)np * kN);
  uint32_t M[16][16];
  std::vector<uint32_t> pw(2 * kN);  // psi^-k
  for (int pi = 0; pi < np; pi++) {
    const uint32_t q = c.primes[pi], inv = h_invmod(c.psi[pi], q);
    const uint32_t rmod = (uint32_t)((1ull << 32) % q);
    pw[0] = 1;
    for (int k = 1; k < 2 * kN; k++) pw[k] = (uint32_t)((uint64_t)pw[k - 1] * inv % q);
    auto at = [&](uint64_t k) { return pw[k & (2 * kN - 1)]; };
    int32_t *pp = planes.data() + (size_t)pi * kI8InvCtx * 1024;
    for (int m = 0; m < 16; m++) {
      uint64_t s = 0;
      for (int k = 0; k < 16; k++) s += M[m][k] = at(8192ull * m * brv_n(k, 4));
      corr[(size_t)pi * 16 + m] =
          i8::centre_h((uint64_t)h_mulmod((uint32_t)(s % q), (1u << 30) % q, q), q);
    }
    i8::ctx_planes(M, q, pp);
    for (int x = 0; x < 16; x++) {
      for (int m = 0; m < 16; m++)
        for (int k = 0; k < 16; k++) M[m][k] = at(512ull * (x + 16 * m) * brv_n(k, 4));
      i8::ctx_planes(M, q, pp + (size_t)(kI8InvCtxRow + x) * 1024);
      for (int m = 0; m < 16; m++)
        for (int k = 0; k < 16; k++)
          M[m][k] = at(256ull * (x + 16 * m) * (2 * brv_n(k, 4) + 1));
      i8::ctx_planes(M, q, pp + (size_t)(kI8InvCtxCol + x) * 1024);
    }
    int32_t *tp = twm.data() + (size_t)pi * kN;
    for (int col = 0; col < 256; col++)
      for (int p = 0; p < 256; p++) {
        const int c1 = col >> 4, word = ((16 * (col & 15) + (p & 15)) * 64 + 16 * (c1 >> 2) +
                                         (p >> 4)) * 4 + (c1 & 3);
        tp[word] = i8::centre_h((uint64_t)at((uint64_t)col * (2 * brv_n(p, 8) + 1)) * rmod, q);
      }
  }
  const int32_t **dst[3] = {&c.i8_inv_planes, &c.i8_inv_corr, &c.i8_inv_twm};
  const std::vector<int32_t> *src[3] = {&planes, &corr, &twm};
  const int32_t *dev[3];
  for (int i = 0; i < 3; i++) {
    int32_t *d = nullptr;
    int rc = check_hip(hipMalloc((void **)&d, src[i]->size() * 4), "hipMalloc(int8 tables)");
    if (rc) return rc;
    c.allocations.push_back(d);
    rc = check_hip(hipMemcpy(d, src[i]->data(), src[i]->size() * 4, hipMemcpyHostToDevice),
                   "hipMemcpy(int8 tables)");
    if (rc) return rc;
    dev[i] = d;
  }
  for (int i = 0; i < 3; i++) *dst[i] = dev[i];
  *out = I8InvTabs{dev[0], dev[1], dev[2]};
  return kOk;
}

void launch_ntt8_cols(const Context &c, const I8NttTabs &T, const Ntt8Job *jobs, int n,
                      int col_blocks, hipStream_t st) {
  if (n <= 0) return;
  const int nwg = n * (16 / col_blocks);
  launch(c, "ntt8_cols", n, ntt8_cols_kernel, dim3(nwg), dim3(256), st, jobs, nwg,
         col_blocks, T, c.ptab);
}

void launch_ntt8_rows(const Context &c, const I8NttTabs &T, const Ntt8Job *jobs, int n,
                      int row_blocks, hipStream_t st) {
  if (n <= 0) return;
  const int nwg = n * (16 / row_blocks);
  launch(c, "ntt8_rows", n, ntt8_rows_kernel, dim3(nwg), dim3(256), st, jobs, nwg,
         row_blocks, T, c.ptab);
}

void launch_ntt1p_fwd(const Context &c, const I8NttTabs &T, const Ntt8Job *jobs, int n,
                      hipStream_t st) {
  if (n <= 0) return;
  launch(c, "ntt1p_fwd", n, ntt1p_fwd_kernel, dim3(n), dim3(512), st, jobs, n,
         T, c.ptab);
}

void launch_ntt1p_inv(const Context &c, const I8InvTabs &T, const Inv1pJob *jobs, int n,
                      bool prod, hipStream_t st) {
  if (n <= 0) return;
  if (prod)
    launch(c, "ntt1p_inv+tensor", n, ntt1p_inv_kernel<true>, dim3(n), dim3(512), st, jobs, n, T,
           c.ptab);
  else
    launch(c, "ntt1p_inv", n, ntt1p_inv_kernel<false>, dim3(n), dim3(512), st, jobs, n, T,
           c.ptab);
}

void launch_bconv_i8_table(const Context &c, const BconvI8Inst *insts, int n, int dsts,
                           int max_s, int, hipStream_t st) {
  if (n <= 0) return;
  if (max_s <= 8)
    launch(c, "bconv_i8", dsts, bconv_i8_kernel<1>, dim3(kN / 256, n), dim3(256), st, insts,
           c.ptab);
  else if (max_s <= 16)
    launch(c, "bconv_i8", dsts, bconv_i8_kernel<2>, dim3(kN / 256, n), dim3(256), st, insts,
           c.ptab);
  else
    launch(c, "bconv_i8", dsts, bconv_i8_kernel<3>, dim3(kN / 256, n), dim3(256), st, insts,
           c.ptab);
}

void launch_bconv_i8(const Context &c, const BconvI8Launch &L, hipStream_t st) {
  if (L.n <= 0) return;
  int dsts = 0, max_s = 1;
  for (int i = 0; i < L.n; i++) {
    dsts += L.inst[i].D;
    max_s = std::max(max_s, L.inst[i].S);
  }
  if (max_s <= 8)
    launch(c, "bconv_i8", dsts, bconv_i8_arg_kernel<1>, dim3(kN / 256, L.n), dim3(256), st,
           L, c.ptab);
  else if (max_s <= 16)
    launch(c, "bconv_i8", dsts, bconv_i8_arg_kernel<2>, dim3(kN / 256, L.n), dim3(256), st,
           L, c.ptab);
  else
    launch(c, "bconv_i8", dsts, bconv_i8_arg_kernel<3>, dim3(kN / 256, L.n), dim3(256), st,
           L, c.ptab);
}

const int64_t *bconv_i8_planes_for(const Context &c, const double *d_ftab, int S, int D,
                                   const uint8_t *dst_prime) {
  std::lock_guard<std::mutex> lock(c.tables_mu);
  for (auto &e : c.i8_bconv_planes)
    if (e.first == d_ftab) return e.second;
  std::vector<double> f((size_t)2 * S * D);
  if (check_hip(hipMemcpy(f.data(), d_ftab, f.size() * sizeof(double), hipMemcpyDeviceToHost),
                "hipMemcpy(BaseConv table)"))
    return nullptr;
  std::vector<uint32_t> tab((size_t)S * D), dq(D);
  for (int d = 0; d < D; d++) {
    dq[d] = c.primes[dst_prime[d]];
    for (int i = 0; i < S; i++)
      tab[(size_t)d * S + i] = (uint32_t)f[2 * ((size_t)d * S + i)] * 65536u +
                               (uint32_t)f[2 * ((size_t)d * S + i) + 1];
  }
  const std::vector<int64_t> pl = i8::bconv_i8_planes(tab, S, D, dq);
  int64_t *dp = nullptr;
  if (check_hip(hipMalloc((void **)&dp, pl.size() * sizeof(int64_t)), "hipMalloc(int8 planes)"))
    return nullptr;
  if (check_hip(hipMemcpy(dp, pl.data(), pl.size() * sizeof(int64_t), hipMemcpyHostToDevice),
                "hipMemcpy(int8 planes)")) {
    (void)hipFree(dp);
    return nullptr;
  }
  c.i8_bconv_planes.emplace_back(d_ftab, dp);
  return dp;
}

bool to_i8_inst(const Context &c, const BconvInst &in, BconvI8Inst *out) {
  std::memset(out, 0, sizeof(*out));
  out->planes = bconv_i8_planes_for(c, in.tab, in.S, in.D, in.dst_prime);
  if (!out->planes) return false;
  out->src = in.src;
  out->dst = in.dst;
  out->S = in.S;
  out->D = in.D;
  out->canonical = in.canonical;
  for (int m = 0; m < in.D; m++) {
    out->dst_limb[m] = in.dst_limb[m];
    out->dst_prime[m] = in.dst_prime[m];
  }
  return true;
}

void add_bcols_quads(std::vector<BcolsQuad> &out, const int32_t *src, int S,
                     const int32_t *quads, const std::vector<uint32_t *> &dst,
                     const std::vector<int> &prime) {
  const size_t D = dst.size();
  for (size_t d0 = 0; d0 < D; d0 += 4) {
    BcolsQuad Q;
    std::memset(&Q, 0, sizeof(Q));
    Q.src = src;
    Q.planes = quads + d0 / 4 * i8::bconv_quad_words(S);
    Q.S = S;
    for (size_t i = 0; i < 4; i++) {
      Q.dst[i] = d0 + i < D ? dst[d0 + i] : nullptr;
      Q.prime[i] = (uint8_t)prime[d0 + i < D ? d0 + i : d0];
    }
    out.push_back(Q);
  }
}

namespace {

template <class D, int NC>
void bconv_cols_nc(const Context &c, const D &d, int n, int limbs, int max_s, hipStream_t st) {
  const dim3 grid(256 / NC * n), block(64 * NC);
  const uint32_t *tw = c.d_tw_fwd;
  const char *name = "ntt_fwd_cols+bconv";
  if (max_s <= 8)
    launch(c, name, limbs, bconv_i8_cols<D, NC, 0>, grid, block, st, d, c.ptab, tw);
  else if (max_s <= 16)
    launch(c, name, limbs, bconv_i8_cols<D, NC, 1>, grid, block, st, d, c.ptab, tw);
  else
    launch(c, name, limbs, bconv_i8_cols<D, NC, 2>, grid, block, st, d, c.ptab, tw);
}

// Columns per workgroup. 8 (two workgroups of 8 waves on a CU) measured
// faster with up to 8 sources: 72 limbs 16.3 us against 18.3 us with 16
// columns (one workgroup of 16 waves), 4128 limbs 739 against 815 us; 4
// columns lose to their 16-byte row segments (72 limbs 20.7 us). With more
// sources the loads weigh more and whole 64-byte segments win once ten quads
// fill the chip: 42 limbs of 15 sources 14.5 against 16.9 us, 114 of 12
// sources 23.5 against 24.5 us; 4 limbs of 9 sources 10.2 against 7.5 us.
// Nine sources lie on the line: with 16 / 8 columns 28 limbs of 8 polynomials
// 10.8 / 12.1 us, 48 limbs of 6 12.0 / 13.3, 192 limbs of 128 65.6 / 82.4, but 92
// limbs of 4 23.5 / 19.8, 254 limbs of 12 51.5 / 44.7, 506 limbs of 22 90 / 81: a
// polynomial's quads share its sources in a cache, which the few limbs of the
// first three do not.
template <class D>
void bconv_cols(const Context &c, const D &d, int n, int limbs, int max_s, hipStream_t st) {
  if (n <= 0) return;
  if (max_s > 8 && n >= 10)
    bconv_cols_nc<D, 16>(c, d, n, limbs, max_s, st);
  else
    bconv_cols_nc<D, 8>(c, d, n, limbs, max_s, st);
}

}  // namespace

void launch_bconv_cols(const Context &c, const BcolsLaunch &L, int n, int limbs, int max_s,
                       hipStream_t st) {
  bconv_cols(c, BcolsByValue{L}, n, limbs, max_s, st);
}

void launch_bconv_cols_table(const Context &c, const BcolsQuad *quads, int n, int limbs,
                             int max_s, hipStream_t st) {
  bconv_cols(c, BcolsTable{quads}, n, limbs, max_s, st);
}

void launch_bconv_valu_table(const Context &c, const BconvI8Inst *insts, int n, int dsts,
                             int, hipStream_t st) {
  if (n <= 0) return;
  launch(c, "bconv_valu", dsts, bconv_valu_kernel, dim3(kN / 256, n), dim3(256), st, insts,
         c.ptab);
}

}  // namespace ck
