// Negacyclic NTT / INTT over 32-bit RNS limbs for N = 2^16 on gfx950.
//
// Transform definition (the reference's, src/core/NTT.cu:231-454 and
// NTTUtils.cuh:19-58): forward Cooley-Tukey with bit-reversed powers of psi
// (psi = g^((q-1)/2N), g the smallest generator); stage m (= 2^s) pairs
// (j, j + N/2^(s+1)) in block i = j / (N/2^s) with twiddle psi_rev[m + i];
// output position k holds a(psi^(2 brv(k) + 1)). The inverse is the
// Gentleman-Sande mirror with psi^-1 and no N^-1 factor; the per-limb
// constant fused after it carries N^-1 and whatever else the caller folds.
//
// MI355X mapping. A limb of 2^16 u32 is a 256 x 256 matrix (row = 256
// consecutive coefficients).
//   * row kernels (forward stages 8..15, inverse stages 0..7): a wave owns one
//     row, four values a lane, without a barrier, or for many limbs a
//     workgroup 16 rows, 16 values a thread; the transformed side moves with
//     16-byte accesses, the other with 4-byte accesses over 256 (or four times
//     64) contiguous bytes.
//   * column kernels (forward stages 0..7, inverse 8..15): a workgroup owns all
//     256 rows of 4, 8 or 16 columns (four values a thread, or 16 at 16
//     columns), read and written straight from registers.
// A wave with 16 values a thread works 1.4 us by itself, and a transform of a
// few limbs leaves most of the chip idle meanwhile; four values a thread make
// four times the waves and a fraction of the time: one limb, both passes,
// 7.3 -> 5.0 us forward, 7.7 -> 5.1 us inverse.
// Register phases are radix 4 (or 16); between them the lazy doubles move over
// lane transposes or padded LDS words. Twiddles are read as u32 and issued
// before the data loads. Butterflies use the exact FP64 modular
// product of ck_arith.h with lazy ranges (integer doubles below 2^40); the
// intermediate between the two passes of a transform is stored as a lazy
// int32 in (-0.75 q, 0.75 q) and only final outputs are made canonical.
#include "ck_elem.h"
#include "ck_internal.h"
#include "ck_radix16.h"

namespace ck {
namespace {

constexpr int kN = 65536;
constexpr int kRowThreads = 256;
constexpr int kRowTile = 4;                // rows per row-kernel workgroup
constexpr int kRowTiles = 256 / kRowTile;  // per limb
constexpr int kRow16Tile = 16;             // rows of a 16-value workgroup
constexpr int kRow16Tiles = 256 / kRow16Tile;
constexpr int kColThreads = 256;
constexpr int kColTile = 16;               // columns of a 16-value workgroup
constexpr int kColTiles = 256 / kColTile;  // per limb

// Launch descriptors: every kernel asks its descriptor for the LimbJob of
// limb y (uniform per workgroup). JobByValue unpacks the kernel-argument
// plan of a single operation; JobTable reads a batched plan's device table.
struct JobByValue {
  NttLaunch L;
  __device__ __forceinline__ LimbJob job(int y) const {
    const NttLimb &R = L.limb[y];
    const int sel = R.sel;
    LimbJob J;
    J.src = L.src[sel & 3] + (size_t)R.src_limb * kN;
    J.dst = L.dst[(sel >> 2) & 3] + (size_t)R.dst_limb * kN;
    const uint32_t *s2 = L.src2[(sel >> 4) & 3];
    J.src2 = (s2 && R.src2_limb >= 0) ? s2 + (size_t)R.src2_limb * kN : nullptr;
    J.c1 = R.c1;
    J.c2 = R.c2;
    J.c3 = R.c3;
    J.prime = R.prime;
    J.flags = L.flags;
    return J;
  }
};

struct JobTable {
  const LimbJob *__restrict__ jobs;
  // the record is read-only and uniform per workgroup: scalar loads
  // through the constant address space
  __device__ __forceinline__ LimbJob job(int y) const {
    typedef const __attribute__((address_space(4))) LimbJob CJob;
    CJob *p = (CJob *)jobs + y;
    LimbJob J;
    J.src = p->src;
    J.dst = p->dst;
    J.src2 = p->src2;
    J.c1 = p->c1;
    J.c2 = p->c2;
    J.c3 = p->c3;
    J.prime = p->prime;
    J.flags = p->flags;
    return J;
  }
};

// Column tile of the 16-value kernels: 16 tiles of 16 columns per limb; workgroup i
// runs on XCD i mod 8, and tiles 2x and 2x + 1 (which share 128-byte lines)
// are placed on the same XCD so a line is fetched into one L2 only.
struct ColTile {
  int y, c0;
};
__device__ __forceinline__ ColTile col_tile() {
  const int t = ((blockIdx.x & 7) << 1) | ((blockIdx.x >> 3) & 1);
  return ColTile{(int)(blockIdx.x >> 4), t * kColTile};
}

// Final value of an element: canonical u32, or lazy int32 in
// (-0.75 q, 0.75 q) for a pass-1 intermediate that pass 2 reads back.
__device__ __forceinline__ int32_t lazy_i32(double x, const ModF &m) {
  return (int32_t)reduce_f(x, m);
}

// ---------------------------------------------------------------------------
// Column passes: stages 0..7 of the forward transform, 8..15 of the inverse
// ---------------------------------------------------------------------------
//
// A workgroup of NC waves owns NC columns, four rows a thread; with 16 / NC
// values of `extra` in a lane's low four bits, e = wave 16 / NC + extra runs
// over 0..15. The lane groups a = lane / 16 hold the row bits next to the
// four registers', so two of the three hand-offs between radix-4 phases are
// lane transposes and one goes through LDS. With few limbs a launch lasts as
// long as one wave, and this form's waves work a quarter as long; which NC is
// taken, and when 16 values a thread, stands at fwd_passes.
template <int NC>
struct ColLane {
  int y, c, e, a;  // limb slot, column, e, lane group
  __device__ __forceinline__ ColLane() {
    // workgroup i runs on XCD i mod 8: the tiles of a 128-byte line share one
    constexpr int kShare = 32 / NC, kTiles = 256 / NC;
    const int b = blockIdx.x, l = threadIdx.x & 63, wv = threadIdx.x >> 6;
    y = b / kTiles;
    c = (((b & 7) * kShare) | ((b >> 3) & (kShare - 1))) * NC + l % NC;
    e = wv * (16 / NC) + (l & 15) / NC;
    a = l >> 4;
  }
};
// LDS word of a row: one spare row after every 16 keeps both sides of the
// hand-off on distinct banks
template <int NC>
__device__ __forceinline__ int col_word(int row, int lane) {
  return (row + (row >> 4)) * NC + lane % NC;
}

template <class D, int NC>
__global__ __launch_bounds__(64 * NC) void ntt_fwd_cols4(const D desc, const PrimeTab P,
                                                         const uint32_t *__restrict__ tw) {
  __shared__ double lds[272 * NC];
  const ColLane<NC> L;
  const LimbJob J = desc.job(L.y);
  const double q = P.qd[J.prime], qr = P.qr[J.prime];
  const ModF m{q, qr};
  const uint32_t *__restrict__ w = tw + (size_t)J.prime * kN;
  const int e = L.e, a = L.a, C = 4 * e + a;
  const uint32_t t0[3] = {w[1], w[2], w[3]};
  const uint32_t t1[3] = {w[4 + a], w[8 + 2 * a], w[9 + 2 * a]};
  const uint32_t t2[3] = {w[16 + e], w[32 + 2 * e], w[33 + 2 * e]};
  const uint32_t t3[3] = {w[64 + C], w[128 + 2 * C], w[129 + 2 * C]};
  // canonical residues (< 2^31) or a lazy signed BaseConv output, as int32
  const int32_t *__restrict__ g =
      reinterpret_cast<const int32_t *>(J.src) + (16 * a + e) * 256 + L.c;
  double x[4];
#pragma unroll
  for (int i = 0; i < 4; i++) x[i] = (double)g[i * 64 * 256];
  if (J.flags & kNttPreMul) {
    const double cv = (double)J.c1, cq = cv * qr;
#pragma unroll
    for (int i = 0; i < 4; i++) x[i] = mulmod_f(x[i], cv, cq, q);
  }
  ct4(x, t0[0], t0 + 1, q, qr);  // rows 64 i + 16 a + e
  transpose_groups(x);
  ct4(x, t1[0], t1 + 1, q, qr);  // rows 64 a + 16 i + e
#pragma unroll
  for (int i = 0; i < 4; i++) lds[col_word<NC>(64 * a + 16 * i + e, threadIdx.x & 63)] = x[i];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 4; i++) x[i] = lds[col_word<NC>(16 * e + 4 * i + a, threadIdx.x & 63)];
  ct4(x, t2[0], t2 + 1, q, qr);  // rows 16 e + 4 i + a
  transpose_groups(x);
  ct4(x, t3[0], t3 + 1, q, qr);  // rows 16 e + 4 a + i
  uint32_t *__restrict__ o = J.dst + (16 * e + 4 * a) * 256 + L.c;
#pragma unroll
  for (int i = 0; i < 4; i++) o[i * 256] = (uint32_t)lazy_i32(x[i], m);
}

template <class D, int NC>
__global__ __launch_bounds__(64 * NC) void intt_cols4(const D desc, const PrimeTab P,
                                                      const uint32_t *__restrict__ tw) {
  __shared__ double lds[272 * NC];
  const ColLane<NC> L;
  const LimbJob J = desc.job(L.y);
  const double q = P.qd[J.prime], qr = P.qr[J.prime];
  const uint32_t *__restrict__ w = tw + (size_t)J.prime * kN;
  const int e = L.e, a = L.a, C = 4 * e + a;
  const uint32_t t0[3] = {w[128 + 2 * C], w[129 + 2 * C], w[64 + C]};
  const uint32_t t1[3] = {w[32 + 2 * e], w[33 + 2 * e], w[16 + e]};
  const uint32_t t2[3] = {w[8 + 2 * a], w[9 + 2 * a], w[4 + a]};
  const uint32_t t3[3] = {w[2], w[3], w[1]};
  // the pass-1 intermediate (in dst) is lazy signed int32
  const int32_t *__restrict__ g =
      reinterpret_cast<const int32_t *>(J.dst) + (16 * e + 4 * a) * 256 + L.c;
  double x[4];
#pragma unroll
  for (int i = 0; i < 4; i++) x[i] = (double)g[i * 256];
  gs4(x, t0, t0[2], q, qr);  // rows 16 e + 4 a + i
  transpose_groups(x);
  gs4(x, t1, t1[2], q, qr);  // rows 16 e + 4 i + a
#pragma unroll
  for (int i = 0; i < 4; i++) lds[col_word<NC>(16 * e + 4 * i + a, threadIdx.x & 63)] = x[i];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 4; i++) x[i] = lds[col_word<NC>(64 * a + 16 * i + e, threadIdx.x & 63)];
  gs4(x, t2, t2[2], q, qr);  // rows 64 a + 16 i + e
  transpose_groups(x);
  gs4(x, t3, t3[2], q, qr);  // rows 64 i + 16 a + e
  const double cv = (double)J.c1, cq = cv * qr;
  // x * c1 lands in (-0.75 q, 0.75 q): canonical [0, q) (above: never,
  // below 0: + q) or centred [-(q-1)/2, (q-1)/2] (one fix-up either side)
  // (integer fix-ups on the exact int32 conversion)
  const int32_t qi = (int32_t)P.q[J.prime];
  const bool centred = (J.flags & kInttCentred) != 0;
  const int32_t above = centred ? (qi - 1) >> 1 : qi - 1;
  const int32_t below = centred ? -((qi - 1) >> 1) : 0;
  uint32_t *__restrict__ o = J.dst + (16 * a + e) * 256 + L.c;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    int32_t v = (int32_t)mulmod_f(x[i], cv, cq, q);
    v = v > above ? v - qi : v;
    v = v < below ? v + qi : v;
    o[i * 64 * 256] = (uint32_t)v;
  }
}

// Many limbs: 16 values a thread, two radix-16 phases with one hand-off and no
// lane transposes. Bound by vector issue (FP64 butterflies): 129 limbs take
// 21.0 us (67 MB, 3.2 TB/s) where the four-value form takes 23.3.
template <class D>
__global__ __launch_bounds__(kColThreads, 5) void ntt_fwd_cols(
    const D desc, const PrimeTab P, const uint32_t *__restrict__ tw) {
  __shared__ double ldsd[256 * kColTile];
  const ColTile ct = col_tile();
  const int c0 = ct.c0;
  const LimbJob J = desc.job(ct.y);
  const double q = P.qd[J.prime], qr = P.qr[J.prime];
  const ModF m{q, qr};
  const uint32_t *__restrict__ w = tw + (size_t)J.prime * kN;
  const int cc = threadIdx.x & 15;
  const int rb = threadIdx.x >> 4;  // 0..15

  // phase 1 twiddles psi_rev[2^s + blk] (uniform), phase 2 psi_rev[2^(4+s)
  // + rb 2^s + blk]
  uint32_t t1[15], t2[15];
#pragma unroll
  for (int s = 0; s < 4; s++)
#pragma unroll
    for (int blk = 0; blk < (1 << s); blk++) {
      t1[(1 << s) - 1 + blk] = w[(1 << s) + blk];
      t2[(1 << s) - 1 + blk] = w[(16 << s) + (rb << s) + blk];
    }
  // phase 1 holds rows rb + 16 k of column c0 + cc: canonical residues
  // (< 2^31) or a lazy signed BaseConv output, as int32
  double x[16];
  {
    const int32_t *__restrict__ g =
        reinterpret_cast<const int32_t *>(J.src) + c0 + cc;
    int32_t v[16];
#pragma unroll
    for (int k = 0; k < 16; k++) v[k] = g[(rb + 16 * k) * 256];
    // all loads before the first conversion: left alone, the scheduler puts
    // half of them after a wait for the first two (96 limbs 14.4 -> 15.1 us,
    // 256 limbs 28.3 -> 29.4)
    keep_loads();
#pragma unroll
    for (int k = 0; k < 16; k++) x[k] = (double)v[k];
  }
  if (J.flags & kNttPreMul) {
    const double cv = (double)J.c1, cq = cv * qr;
#pragma unroll
    for (int k = 0; k < 16; k++) x[k] = mulmod_f(x[k], cv, cq, q);
  }
  ct16(x, t1, q, qr);
#pragma unroll
  for (int k = 0; k < 16; k++) ldsd[(rb + 16 * k) * kColTile + cc] = x[k];
  __syncthreads();
#pragma unroll
  for (int j = 0; j < 16; j++) x[j] = ldsd[(rb * 16 + j) * kColTile + cc];
  ct16(x, t2, q, qr);
  // rows rb * 16 + j, lazy int32 for the row pass
  uint32_t *__restrict__ o = J.dst + c0 + cc;
#pragma unroll
  for (int j = 0; j < 16; j++)
    o[(rb * 16 + j) * 256] = (uint32_t)lazy_i32(x[j], m);
}

template <class D>
__global__ __launch_bounds__(kColThreads, 5) void intt_cols(
    const D desc, const PrimeTab P, const uint32_t *__restrict__ tw) {
  __shared__ double ldsd[256 * kColTile];
  const ColTile ct = col_tile();  // same XCD-aware order as ntt_fwd_cols
  const int c0 = ct.c0;
  const LimbJob J = desc.job(ct.y);
  const double q = P.qd[J.prime], qr = P.qr[J.prime];
  const ModF m{q, qr};
  const uint32_t *__restrict__ w = tw + (size_t)J.prime * kN;
  const int cc = threadIdx.x & 15;
  const int rb = threadIdx.x >> 4;

  // phase 1 psi_inv_rev[2^(7-u) + rb 2^(3-u) + blk],
  // phase 2 psi_inv_rev[2^(3-u) + blk] (uniform)
  uint32_t t1[15], t2[15];
#pragma unroll
  for (int u = 0; u < 4; u++)
#pragma unroll
    for (int blk = 0; blk < (8 >> u); blk++) {
      t1[16 - (16 >> u) + blk] = w[(128 >> u) + (rb << (3 - u)) + blk];
      t2[16 - (16 >> u) + blk] = w[(8 >> u) + blk];
    }
  // the pass-1 intermediate (in dst) is lazy signed int32; phase 1 holds
  // rows rb * 16 + j of column c0 + cc
  double x[16];
  {
    const int32_t *__restrict__ g =
        reinterpret_cast<const int32_t *>(J.dst) + c0 + cc;
#pragma unroll
    for (int j = 0; j < 16; j++) x[j] = (double)g[(rb * 16 + j) * 256];
  }
  gs16(x, t1, q, qr);
  // lazy inputs (|x| < 0.75 q) grow below 2^39 over the eight stages
#pragma unroll
  for (int j = 0; j < 16; j++) ldsd[(rb * 16 + j) * kColTile + cc] = x[j];
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 16; k++) x[k] = ldsd[(rb + 16 * k) * kColTile + cc];
  gs16(x, t2, q, qr);
  const double cv = (double)J.c1, cq = cv * qr;
  uint32_t *__restrict__ o = J.dst + c0 + cc;
  // x * c1 lands in (-0.75 q, 0.75 q): canonical [0, q) (above: never,
  // below 0: + q) or centred [-(q-1)/2, (q-1)/2] (one fix-up either side)
  // (integer fix-ups on the exact int32 conversion)
  const int32_t qi = (int32_t)P.q[J.prime];
  const bool centred = (J.flags & kInttCentred) != 0;
  const int32_t above = centred ? (qi - 1) >> 1 : qi - 1;
  const int32_t below = centred ? -((qi - 1) >> 1) : 0;
#pragma unroll
  for (int k = 0; k < 16; k++) {
    int32_t v = (int32_t)mulmod_f(x[k], cv, cq, q);
    v = v > above ? v - qi : v;
    v = v < below ? v + qi : v;
    o[(rb + 16 * k) * 256] = (uint32_t)v;
  }
}

// ---------------------------------------------------------------------------
// Row passes: stages 8..15 of the forward transform, 0..7 of the inverse
// ---------------------------------------------------------------------------
//
// A wave owns a row, four values a lane: one hand-off between the radix-4
// phases is a lane transpose, two go through the wave's own LDS words, and no
// barrier is needed. Against 16 rows a workgroup and 16 values a thread, both
// passes of a forward transform: 1 limb 7.3 -> 6.0 us, 24 limbs 14.6 -> 12.6,
// 59 limbs 26.5 -> 23.4. Many limbs take the 16-value kernels below.
constexpr int kRowPad = 320;  // doubles of a row: 4 spare ones after every 16
__device__ __forceinline__ int pad16(int j) { return j + 4 * (j >> 4); }

// twiddles of a forward row: phase p's three in t[p]
struct RowTw {
  uint32_t t[4][3];
};
__device__ __forceinline__ RowTw row_twiddles(const uint32_t *w, int r, int l) {
  const int A = l >> 4, B = l >> 2;
  const uint32_t *w1 = w + 1024 + 4 * r + A, *w1b = w + 2048 + 8 * r + 2 * A;
  const uint32_t *w2 = w + 4096 + 16 * r + B, *w2b = w + 8192 + 32 * r + 2 * B;
  const uint32_t *w3 = w + 16384 + 64 * r + l, *w3b = w + 32768 + 128 * r + 2 * l;
  return RowTw{{{w[256 + r], w[512 + 2 * r], w[513 + 2 * r]},
                {w1[0], w1b[0], w1b[1]},
                {w2[0], w2b[0], w2b[1]},
                {w3[0], w3b[0], w3b[1]}}};
}
// elements 64 i + l of a row in, elements 4 l + i of its transform (lazy) out
__device__ __forceinline__ void row_forward(double x[4], const RowTw &T, int l, double *X,
                                            double q, double qr) {
  const int A = l >> 4, B = l >> 2;
  ct4(x, T.t[0][0], T.t[0] + 1, q, qr);
  transpose_groups(x);  // elements 64 A + 16 i + (l & 15)
  ct4(x, T.t[1][0], T.t[1] + 1, q, qr);
  wave_sync();
#pragma unroll
  for (int i = 0; i < 4; i++) X[pad16(64 * A + 16 * i + (l & 15))] = x[i];
  wave_sync();
#pragma unroll
  for (int i = 0; i < 4; i++) x[i] = X[pad16(16 * B + 4 * i + (l & 3))];
  ct4(x, T.t[2][0], T.t[2] + 1, q, qr);
  wave_sync();
#pragma unroll
  for (int i = 0; i < 4; i++) X[pad16(16 * B + 4 * i + (l & 3))] = x[i];
  wave_sync();
#pragma unroll
  for (int i = 0; i < 4; i++) x[i] = X[pad16(4 * l) + i];
  ct4(x, T.t[3][0], T.t[3] + 1, q, qr);
}

template <class D>
__global__ __launch_bounds__(kRowThreads) void ntt_fwd_rows(const D desc, const PrimeTab P,
                                                            const uint32_t *__restrict__ tw) {
  __shared__ double rows[kRowTile][kRowPad];
  const LimbJob J = desc.job(blockIdx.y);
  const double q = P.qd[J.prime], qr = P.qr[J.prime];
  const ModF m{q, qr};
  const int l = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int r = blockIdx.x * kRowTile + wv;
  const RowTw T = row_twiddles(tw + (size_t)J.prime * kN, r, l);
  // the pass-1 intermediate (in dst) is lazy signed int32
  const int32_t *g = reinterpret_cast<const int32_t *>(J.dst) + r * 256 + l;
  double x[4];
#pragma unroll
  for (int i = 0; i < 4; i++) x[i] = (double)g[64 * i];
  // the ModDown epilogue's second operand, issued with the data loads
  const bool has2 = (J.flags & kNttModDownEpilogue) && J.src2;
  uint4 s2 = make_uint4(0, 0, 0, 0);
  if (has2) s2 = *reinterpret_cast<const uint4 *>(J.src2 + r * 256 + 4 * l);
  row_forward(x, T, l, rows[wv], q, qr);
  uint32_t out[4];
  if (J.flags & kNttModDownEpilogue) {
    // NTTPhase2ForModDown (NTT.cu:456-601): out = (src2 * pad - y) * ip
    const double ip = (double)J.c3, ipq = ip * qr;
    double a2[4] = {(double)s2.x, (double)s2.y, (double)s2.z, (double)s2.w};
    if (J.flags & kNttEpiloguePad) {
      const double pv = (double)J.c2, pq = pv * qr;
#pragma unroll
      for (int i = 0; i < 4; i++) a2[i] = mulmod_f(a2[i], pv, pq, q);
    }
#pragma unroll
    for (int i = 0; i < 4; i++)
      out[i] = canon_small(mulmod_f(a2[i] - x[i], ip, ipq, q), q);
  } else {
#pragma unroll
    for (int i = 0; i < 4; i++) out[i] = canon_f(x[i], m);
  }
  *reinterpret_cast<uint4 *>(J.dst + r * 256 + 4 * l) =
      make_uint4(out[0], out[1], out[2], out[3]);
}

template <class D>
__global__ __launch_bounds__(kRowThreads) void intt_rows(const D desc, const PrimeTab P,
                                                         const uint32_t *__restrict__ tw) {
  __shared__ double rows[kRowTile][kRowPad];
  const LimbJob J = desc.job(blockIdx.y);
  const double q = P.qd[J.prime], qr = P.qr[J.prime];
  const ModF m{q, qr};
  const uint32_t *__restrict__ w = tw + (size_t)J.prime * kN;
  const int l = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int r = blockIdx.x * kRowTile + wv;
  const int A = l >> 4, B = l >> 2;
  const uint32_t *w0 = w + 32768 + 128 * r + 2 * l, *w0b = w + 16384 + 64 * r + l;
  const uint32_t *w1 = w + 8192 + 32 * r + 2 * B, *w1b = w + 4096 + 16 * r + B;
  const uint32_t *w2 = w + 2048 + 8 * r + 2 * A, *w2b = w + 1024 + 4 * r + A;
  const uint32_t t0[3] = {w0[0], w0[1], w0b[0]};
  const uint32_t t1[3] = {w1[0], w1[1], w1b[0]};
  const uint32_t t2[3] = {w2[0], w2[1], w2b[0]};
  const uint32_t t3[3] = {w[512 + 2 * r], w[513 + 2 * r], w[256 + r]};
  const uint4 u = *reinterpret_cast<const uint4 *>(J.src + r * 256 + 4 * l);
  uint32_t in[4] = {u.x, u.y, u.z, u.w};
  if (J.flags & kInttLoadProduct) {
    // Tensor's a1 (*) a2 (ElementWise.cu:504-546) fused into the load
    const uint4 v = *reinterpret_cast<const uint4 *>(J.src2 + r * 256 + 4 * l);
    const uint32_t V[4] = {v.x, v.y, v.z, v.w};
    const uint32_t qu = P.q[J.prime];
    const int32_t qinv = P.qinv[J.prime];
#pragma unroll
    for (int i = 0; i < 4; i++) in[i] = mont_mul(in[i], V[i], qu, qinv);
  }
  double x[4] = {(double)in[0], (double)in[1], (double)in[2], (double)in[3]};
  double *X = rows[wv];
  gs4(x, t0, t0[2], q, qr);
#pragma unroll
  for (int i = 0; i < 4; i++) X[pad16(4 * l) + i] = x[i];
  wave_sync();
#pragma unroll
  for (int i = 0; i < 4; i++) x[i] = X[pad16(16 * B + 4 * i + (l & 3))];
  gs4(x, t1, t1[2], q, qr);
  wave_sync();
#pragma unroll
  for (int i = 0; i < 4; i++) X[pad16(16 * B + 4 * i + (l & 3))] = x[i];
  wave_sync();
#pragma unroll
  for (int i = 0; i < 4; i++) x[i] = X[pad16(64 * A + 16 * i + (l & 15))];
  gs4(x, t2, t2[2], q, qr);
  transpose_groups(x);  // elements 64 i + l
  gs4(x, t3, t3[2], q, qr);
  int32_t *o = reinterpret_cast<int32_t *>(J.dst) + r * 256 + l;
#pragma unroll
  for (int i = 0; i < 4; i++) o[64 * i] = lazy_i32(x[i], m);
}

// Many limbs: 16 values a thread, 16 rows a workgroup (a contiguous 16 KiB), two
// radix-16 phases with one hand-off. Bound by memory and FP64 issue together:
// 2048 limbs inverse 244 us (4.4 TB/s) where four values a lane take 286,
// forward 257 against 285. The lines between the two stand at fwd_passes.
//
// Row-tile LDS index: row rl, in-row offset b, the low nibble swizzled by the
// high nibble (b = t + 16 k and b = 16 t + j both hit 16 distinct banks).
__device__ __forceinline__ int row16_word(int rl, int b) {
  return rl * 256 + (b ^ ((b >> 4) & 15));
}

// no ModDown epilogue
template <class D>
__global__ __launch_bounds__(kRowThreads, 5) void ntt_fwd_rows16(
    const D desc, const PrimeTab P, const uint32_t *__restrict__ tw) {
  __shared__ double lds[kRow16Tile * 256];
  const LimbJob J = desc.job(blockIdx.y);
  const double q = P.qd[J.prime], qr = P.qr[J.prime];
  const ModF m{q, qr};
  const uint32_t *__restrict__ w = tw + (size_t)J.prime * kN;
  const int rl = threadIdx.x >> 4, t = threadIdx.x & 15;
  const int r = blockIdx.x * kRow16Tile + rl;
  // phase 1 twiddles psi_rev[2^(8+s) + r 2^s + blk], phase 2
  // psi_rev[2^(12+s) + r 2^(4+s) + t 2^s + blk]
  uint32_t t1[15], t2[15];
#pragma unroll
  for (int s = 0; s < 4; s++)
#pragma unroll
    for (int blk = 0; blk < (1 << s); blk++) {
      t1[(1 << s) - 1 + blk] = w[(256 << s) + (r << s) + blk];
      t2[(1 << s) - 1 + blk] = w[(4096 << s) + (r << (4 + s)) + (t << s) + blk];
    }
  // the pass-1 intermediate (in dst) is lazy signed int32; elements t + 16 k
  const int32_t *g = reinterpret_cast<const int32_t *>(J.dst) + r * 256 + t;
  double x[16];
#pragma unroll
  for (int k = 0; k < 16; k++) x[k] = (double)g[16 * k];
  ct16(x, t1, q, qr);
#pragma unroll
  for (int k = 0; k < 16; k++) lds[row16_word(rl, t + 16 * k)] = x[k];
  __syncthreads();
#pragma unroll
  for (int j = 0; j < 16; j++) x[j] = lds[row16_word(rl, 16 * t + j)];
  ct16(x, t2, q, qr);
  uint4 *o = reinterpret_cast<uint4 *>(J.dst + r * 256 + 16 * t);
#pragma unroll
  for (int i = 0; i < 4; i++)
    o[i] = make_uint4(canon_f(x[4 * i], m), canon_f(x[4 * i + 1], m),
                      canon_f(x[4 * i + 2], m), canon_f(x[4 * i + 3], m));
}

// no product input
template <class D>
__global__ __launch_bounds__(kRowThreads, 5) void intt_rows16(
    const D desc, const PrimeTab P, const uint32_t *__restrict__ tw) {
  __shared__ double lds[kRow16Tile * 256];
  const LimbJob J = desc.job(blockIdx.y);
  const double q = P.qd[J.prime], qr = P.qr[J.prime];
  const ModF m{q, qr};
  const uint32_t *__restrict__ w = tw + (size_t)J.prime * kN;
  const int rl = threadIdx.x >> 4, t = threadIdx.x & 15;
  const int r = blockIdx.x * kRow16Tile + rl;
  // phase 1 psi_inv_rev[2^(15-u) + r 2^(7-u) + t 2^(3-u) + blk],
  // phase 2 psi_inv_rev[2^(11-u) + r 2^(3-u) + blk]
  uint32_t t1[15], t2[15];
#pragma unroll
  for (int u = 0; u < 4; u++)
#pragma unroll
    for (int blk = 0; blk < (8 >> u); blk++) {
      t1[16 - (16 >> u) + blk] = w[(32768 >> u) + (r << (7 - u)) + (t << (3 - u)) + blk];
      t2[16 - (16 >> u) + blk] = w[(2048 >> u) + (r << (3 - u)) + blk];
    }
  // twiddles first: with the data in front of them 108 limbs take 16.2 us, not 14.9
  keep_loads();
  const uint4 *g = reinterpret_cast<const uint4 *>(J.src + r * 256 + 16 * t);
  double x[16];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const uint4 u = g[i];
    x[4 * i + 0] = (double)u.x;
    x[4 * i + 1] = (double)u.y;
    x[4 * i + 2] = (double)u.z;
    x[4 * i + 3] = (double)u.w;
  }
  // sums double every stage: from inputs below 2^31 they stay below 2^39
  gs16(x, t1, q, qr);
#pragma unroll
  for (int j = 0; j < 16; j++) lds[row16_word(rl, 16 * t + j)] = x[j];
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 16; k++) x[k] = lds[row16_word(rl, t + 16 * k)];
  gs16(x, t2, q, qr);
  int32_t *o = reinterpret_cast<int32_t *>(J.dst) + r * 256 + t;
#pragma unroll
  for (int k = 0; k < 16; k++) o[16 * k] = lazy_i32(x[k], m);
}

// ---------------------------------------------------------------------------
// Forward row stages fused with the key inner product (MultKeyNoModDown,
// src/core/Context.cpp:609-712: the ModUp's last NTT stages, then
// ElementWise::PAccum / CAccum, src/core/ElementWise.cu:225-366)
// ---------------------------------------------------------------------------
//
// One wave owns a row of output limb y (prime p). For every ModUp group g it
// takes limb y of that group's ModUp output straight from the column pass
// (lazy int32 in `modup`), runs the row stages in registers and multiplies the
// four values each lane holds by the key limbs, so the ModUp output never goes
// back to memory in NTT form. A group's own limbs are the ModUp source itself
// (x, or the Tensor product a1 (*) a2). The row outputs are made canonical and
// the products summed in 64 bits (sum_fold, sum_reduce), as Montgomery
// products of the stored data:
//   acc_x[y] = R^-1 (sum_g m_g * key_x,g + P R * fold_x)  mod q,
// fold_b = d0 = b1 (*) b2 (HMult) or add_b, fold_a likewise, which is exactly
// the key_accum kernel's sum.
//
// Bound by memory: the keys, 50 MB for 32 limbs and three groups, pass by
// once, 111 MB in all at least. Products reduced one by one in FP64 -> sums in
// 64 bits -> four values a lane instead of 16: 11 limbs 8.6 -> 6.8 us (last step), 32 limbs 26.8 -> 23.4 ->
// 22.8, 59 limbs 47 -> 42, 382 limbs of a batch 218 -> 195 -> 164.
template <class Args>
__device__ __forceinline__ void key_rows_body(const EwNp &np, const PrimeTab &P,
                                              Args &A, const uint32_t *tw, int y,
                                              double *X, int wv) {
  const int p = y < np.num_q ? np.q_prime0 + y : np.aux_prime0 + (y - np.num_q);
  const double q = P.qd[p], qr = P.qr[p];
  const ModF m{q, qr};
  const uint32_t qu = P.q[p];
  const int32_t qinv = P.qinv[p];
  const int l = threadIdx.x & 63;
  const int r = blockIdx.x * kRowTile + wv;
  const size_t tot_stride = (size_t)np.num_total * kN;
  const uint32_t off = r * 256 + 4 * l;  // this thread's 4 outputs
  const size_t my = (size_t)y * kN + off;
  const int kl = y < np.num_q ? A.key_q0 + y : A.key_aux0 + (y - np.num_q);
  const size_t kp = (size_t)kl * kN + off;
  const bool tens = A.use_tensor && y < np.num_q;
  const RowTw T = row_twiddles(tw + (size_t)p * kN, r, l);

  uint64_t sb[4] = {0, 0, 0, 0}, sa[4] = {0, 0, 0, 0};
  for (int gi = 0; gi < A.ngroups; gi++) {
    const int g = A.group[gi];
    const bool own = (y >= A.own0[g] && y < A.own1[g]);
    // key limbs first: their loads overlap the row stages
    const uint4 kb = *reinterpret_cast<const uint4 *>(A.key_b[g] + kp);
    const uint4 ka = *reinterpret_cast<const uint4 *>(A.key_a[g] + kp);
    uint32_t v[4];
    if (own) {
      if (tens) {
        // d2 = a1 (*) a2
        const uint4 a1 = *reinterpret_cast<const uint4 *>(A.tensor[1] + my);
        const uint4 a2 = *reinterpret_cast<const uint4 *>(A.tensor[3] + my);
        v[0] = sum_reduce((uint64_t)a1.x * a2.x, qu, qinv);
        v[1] = sum_reduce((uint64_t)a1.y * a2.y, qu, qinv);
        v[2] = sum_reduce((uint64_t)a1.z * a2.z, qu, qinv);
        v[3] = sum_reduce((uint64_t)a1.w * a2.w, qu, qinv);
      } else {
        const uint4 u = *reinterpret_cast<const uint4 *>(A.x + my);
        v[0] = u.x;
        v[1] = u.y;
        v[2] = u.z;
        v[3] = u.w;
      }
    } else {
      const int32_t *src = reinterpret_cast<const int32_t *>(
          A.modup + (size_t)g * tot_stride + (size_t)y * kN + r * 256 + l);
      double x[4];
#pragma unroll
      for (int i = 0; i < 4; i++) x[i] = (double)src[64 * i];
      row_forward(x, T, l, X, q, qr);
#pragma unroll
      for (int i = 0; i < 4; i++) v[i] = canon_f(x[i], m);
    }
    const uint32_t KB[4] = {kb.x, kb.y, kb.z, kb.w}, KA[4] = {ka.x, ka.y, ka.z, ka.w};
#pragma unroll
    for (int i = 0; i < 4; i++) {
      sb[i] += (uint64_t)v[i] * KB[i];
      sa[i] += (uint64_t)v[i] * KA[i];
    }
    if (gi & 1) {  // two products between folds
#pragma unroll
      for (int i = 0; i < 4; i++) {
        sb[i] = sum_fold(sb[i], qu);
        sa[i] = sum_fold(sa[i], qu);
      }
    }
  }

  // the P fold on q limbs: one more product (at most two since a fold)
  const uint32_t pp = y < np.num_q ? A.p_prod[p] : 0u;
  if (tens) {
    const uint4 u1 = *reinterpret_cast<const uint4 *>(A.tensor[0] + my);
    const uint4 v1 = *reinterpret_cast<const uint4 *>(A.tensor[1] + my);
    const uint4 u2 = *reinterpret_cast<const uint4 *>(A.tensor[2] + my);
    const uint4 v2 = *reinterpret_cast<const uint4 *>(A.tensor[3] + my);
    const uint32_t B1[4] = {u1.x, u1.y, u1.z, u1.w}, A1[4] = {v1.x, v1.y, v1.z, v1.w};
    const uint32_t B2[4] = {u2.x, u2.y, u2.z, u2.w}, A2[4] = {v2.x, v2.y, v2.z, v2.w};
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const uint32_t d0 = sum_reduce((uint64_t)B1[i] * B2[i], qu, qinv);
      const uint32_t d1 =
          sum_reduce((uint64_t)B1[i] * A2[i] + (uint64_t)A1[i] * B2[i], qu, qinv);
      sb[i] += (uint64_t)pp * d0;
      sa[i] += (uint64_t)pp * d1;
    }
  } else if (y < np.num_q && (A.add_b || A.add_a)) {
    if (A.add_b) {
      const uint4 u = *reinterpret_cast<const uint4 *>(A.add_b + my);
      const uint32_t U[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
      for (int i = 0; i < 4; i++) sb[i] += (uint64_t)pp * U[i];
    }
    if (A.add_a) {
      const uint4 u = *reinterpret_cast<const uint4 *>(A.add_a + my);
      const uint32_t U[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
      for (int i = 0; i < 4; i++) sa[i] += (uint64_t)pp * U[i];
    }
  }

  uint32_t vb[4], va[4];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    vb[i] = sum_reduce(sum_fold(sb[i], qu), qu, qinv);
    va[i] = sum_reduce(sum_fold(sa[i], qu), qu, qinv);
  }
  *reinterpret_cast<uint4 *>(A.out_b + my) = make_uint4(vb[0], vb[1], vb[2], vb[3]);
  *reinterpret_cast<uint4 *>(A.out_a + my) = make_uint4(va[0], va[1], va[2], va[3]);
}

__global__ __launch_bounds__(kRowThreads) void key_rows_kernel(
    const EwNp np, const PrimeTab P, const KeyAccumArgs A, const uint32_t *__restrict__ tw) {
  __shared__ double rows[kRowTile][kRowPad];
  const int wv = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  key_rows_body(np, P, A, tw, blockIdx.y, rows[wv], wv);
}

__global__ __launch_bounds__(kRowThreads) void key_rows_table_kernel(
    const KeyAccumItem *__restrict__ items, const EwJob *__restrict__ jobs,
    const PrimeTab P, const uint32_t *__restrict__ tw) {
  __shared__ double rows[kRowTile][kRowPad];
  const int wv = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  typedef const __attribute__((address_space(4))) KeyAccumItem CItem;
  typedef const __attribute__((address_space(4))) EwJob CJob;
  CJob &jb = ((CJob *)jobs)[blockIdx.y];
  const int item = jb.item, y = jb.y;
  CItem &it = ((CItem *)items)[item];
  const EwNp np{it.np.num_q, it.np.num_total, it.np.q_prime0, it.np.aux_prime0};
  key_rows_body(np, P, it.A, tw, y, rows[wv], wv);
}

const char *fwd_rows_name(int flags) {
  return (flags & kNttModDownEpilogue) ? "ntt_fwd_rows+epilogue" : "ntt_fwd_rows";
}
const char *inv_rows_name(int flags) {
  return (flags & kInttLoadProduct) ? "intt_rows+tensor" : "intt_rows";
}

// Column pass over n limbs. A small launch lasts as long as one wave, so few
// limbs take four values a thread over four (n <= 4) or eight columns a
// workgroup, more the 16-value form. Both passes of a forward transform
// with four columns / eight columns / 16 values, us: 1 limb 5.0 / 5.3 / 6.0,
// 4 limbs 5.7 / 5.8 / 6.6, 8 limbs 7.1 / 6.9 / 7.6, 24 limbs 12.8 / 12.4 / 12.6,
// 59 limbs 24.0 / 23.3 / 23.4; inverse 1 limb 5.1 / 5.4 / 6.4, 24 limbs 13.2 /
// 12.6 / 13.3. The inverse line lies lower, since this pass is the lighter one:
// eight columns / 16 values, the column pass alone, 40 limbs 7.8 / 8.4, 48 limbs
// 9.2 / 8.8, 56 limbs 10.5 / 10.3, 64 limbs 11.7 / 11.1, and 48 limbs within a batch
// of products 10.8 / 9.5.
constexpr int kCols4 = 4, kFwdCols8 = 64, kInvCols8 = 40;
// Row pass over n limbs: four values a lane up to these, 16 above. Four / 16
// values, us, row pass alone: inverse 72 limbs 10.6 / 12.7, 84 limbs 11.9 / 13.5,
// 96 limbs 14.7 / 14.6, 144 limbs 18.0 / 17.4, 256 limbs 32 / 29, 512 limbs 68 /
// 57, and 144 limbs within a batch of products 22.8 / 20.0; forward 256 limbs
// 32.4 / 32.4, 320 limbs 38.7 / 38.5, 384 limbs 48.8 / 45.4, 512 limbs 68 / 61.
// With a product input (at most 191 limbs) four values stay better: 133 limbs
// 24.1 / 25.5, 189 limbs 32.4 / 33.2; with the ModDown epilogue the two are equal
// (506 limbs 75 / 74).
constexpr int kFwdRows4 = 352, kInvRows4 = 88;

template <class D>
void fwd_passes(const Context &ctx, const D &d, int n, int flags, hipStream_t st) {
  const uint32_t *tw = ctx.d_tw_fwd;
  if (!(flags & kNttRowsOnly)) {
    auto cols = [&](auto kernel, int wgs, int threads) {
      launch(ctx, "ntt_fwd_cols", n, kernel, dim3(wgs * n), dim3(threads), st, d, ctx.ptab, tw);
    };
    if (n <= kCols4)
      cols(ntt_fwd_cols4<D, 4>, 64, 256);
    else if (n <= kFwdCols8)
      cols(ntt_fwd_cols4<D, 8>, 32, 512);
    else
      cols(ntt_fwd_cols<D>, kColTiles, kColThreads);
  }
  auto rows = [&](auto kernel, int wgs) {
    launch(ctx, fwd_rows_name(flags), n, kernel, dim3(wgs, n), dim3(kRowThreads), st, d,
           ctx.ptab, tw);
  };
  if (flags & kNttColsOnly) return;
  if (n > kFwdRows4 && !(flags & kNttModDownEpilogue))
    rows(ntt_fwd_rows16<D>, kRow16Tiles);
  else
    rows(ntt_fwd_rows<D>, kRowTiles);
}

template <class D>
void inv_passes(const Context &ctx, const D &d, int n, int flags,
                hipStream_t st) {
  const uint32_t *tw = ctx.d_tw_inv;
  auto rows = [&](auto kernel, int wgs) {
    launch(ctx, inv_rows_name(flags), n, kernel, dim3(wgs, n), dim3(kRowThreads), st, d,
           ctx.ptab, tw);
  };
  if (n > kInvRows4 && !(flags & kInttLoadProduct))
    rows(intt_rows16<D>, kRow16Tiles);
  else
    rows(intt_rows<D>, kRowTiles);
  auto cols = [&](auto kernel, int wgs, int threads) {
    launch(ctx, "intt_cols", n, kernel, dim3(wgs * n), dim3(threads), st, d, ctx.ptab, tw);
  };
  if (n <= kCols4)
    cols(intt_cols4<D, 4>, 64, 256);
  else if (n <= kInvCols8)
    cols(intt_cols4<D, 8>, 32, 512);
  else
    cols(intt_cols<D>, kColTiles, kColThreads);
}

}  // namespace

// Forward NTT of L.n limbs: column stages into dst, then row stages in place
// on dst (with the optional ModDown epilogue).
void launch_ntt_fwd(const Context &ctx, const NttLaunch &L, hipStream_t st) {
  if (L.n <= 0) return;
  fwd_passes(ctx, JobByValue{L}, L.n, L.flags, st);
}

// Inverse NTT of L.n limbs: row stages into dst, then column stages in
// place on dst with the post constant c1 (plain form) and optional centring.
void launch_intt(const Context &ctx, const NttLaunch &L, hipStream_t st) {
  if (L.n <= 0) return;
  inv_passes(ctx, JobByValue{L}, L.n, L.flags, st);
}

void launch_ntt_fwd_table(const Context &ctx, const LimbJob *jobs, int n,
                          int flags_any, hipStream_t st) {
  if (n <= 0) return;
  fwd_passes(ctx, JobTable{jobs}, n, flags_any, st);
}

void launch_key_rows(const Context &ctx, const EwNp &np, const KeyAccumArgs &A,
                     hipStream_t st) {
  if (np.num_total <= 0) return;
  launch(ctx, "ntt_fwd_rows+key", np.num_total, key_rows_kernel, dim3(kRowTiles, np.num_total),
         dim3(kRowThreads), st, np, ctx.ptab, A, (const uint32_t *)ctx.d_tw_fwd);
}

void launch_key_rows_table(const Context &ctx, const KeyAccumItem *items, const EwJob *jobs,
                           int njobs, hipStream_t st) {
  if (njobs <= 0) return;
  launch(ctx, "ntt_fwd_rows+key[batch]", njobs, key_rows_table_kernel, dim3(kRowTiles, njobs),
         dim3(kRowThreads), st, items, jobs, ctx.ptab, (const uint32_t *)ctx.d_tw_fwd);
}

void launch_intt_table(const Context &ctx, const LimbJob *jobs, int n,
                       int flags_any, hipStream_t st) {
  if (n <= 0) return;
  inv_passes(ctx, JobTable{jobs}, n, flags_any, st);
}

}  // namespace ck
