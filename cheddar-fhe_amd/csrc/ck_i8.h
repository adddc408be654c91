// Exact int8 matrix-core forms of the forward NTT and of BaseConv (see
// ck_i8.hip), and a vector-unit BaseConv used as their baseline.
#pragma once

#include "ck_bconv.h"
#include "ck_i8_arith.h"
#include "ck_internal.h"

namespace ck {

// ---- 4-step NTT on the int8 matrix cores ----------------------------------

// Per-prime constant matrices of the 4-step transform ("contexts"), each a
// 16 x 16 matrix over Z_q in MFMA operand order (see ck_i8.hip):
constexpr int kI8CtxA1 = 0;      // column pass, first 16-point stage
constexpr int kI8CtxA1Mont = 1;  // the same times R (Montgomery conversion)
constexpr int kI8CtxB1 = 2;      // + p1: column pass, second stage (twiddled)
constexpr int kI8CtxA3 = 18;     // row pass, first stage
constexpr int kI8CtxB3 = 19;     // + q1: row pass, second stage (twiddled)
constexpr int kI8Ctx = 35;

// Device tables of the int8 transform for every prime of a context, built
// on first use (ntt8_tables).
struct I8NttTabs {
  const int32_t *planes = nullptr;  // [prime][kI8Ctx][4 planes][64 lanes][4]
  const int32_t *corr = nullptr;    // [prime][2][16] offset corrections
  const uint32_t *tw = nullptr;     // [prime] psi^(c (2 brv8(p) + 1)), 16 x 16 tiles
  const int32_t *twm = nullptr;     // the same times 2^32, centred
};

// One limb of a batched int8 transform: dst = NTT(src) (x R when mont).
struct Ntt8Job {
  const uint32_t *src;
  uint32_t *dst;
  int32_t prime;
  int32_t mont;
};
static_assert(sizeof(Ntt8Job) == 24, "Ntt8Job is one 24-byte record");

// Builds (once) and returns the int8 transform tables of every prime.
int ntt8_tables(Context &c, I8NttTabs *out);
// Column pass then row pass over n jobs; col_blocks = 16-column blocks per
// workgroup of the column pass (and 16-row blocks of the row pass), a
// divisor of 16.
void launch_ntt8_cols(const Context &c, const I8NttTabs &T, const Ntt8Job *jobs, int n,
                      int col_blocks, hipStream_t st);
void launch_ntt8_rows(const Context &c, const I8NttTabs &T, const Ntt8Job *jobs, int n,
                      int row_blocks, hipStream_t st);

// The same transform in one pass, a workgroup per limb: rounds of 256 limbs
// (one per CU) of 38-41 us each however full. A batch of at least 192 limbs
// takes it; of the limbs past its whole rounds, 128 and more too, fewer run
// as two passes (7.5 us and 0.25 us a limb). Measured for 192 / 256 / 512 /
// 2048 limbs, against two vector passes: forward 38 / 37 / 74 / 318 us against
// 49 / 62 / 126 / 559, inverse 42 / 40 / 78 / 334 us against 47 / 60 / 120 /
// 544; at 264 limbs a second round for 8 of them costs 63 and 70 us in all.
// With the product input a round takes 53 us at 192 limbs and 57-60 at 240 to
// 256, against 60 and 73-75 of the two vector passes.
constexpr int kOnePassLimbs = 192, kOnePassRound = 256, kOnePassTail = 128;
inline size_t one_pass_limbs(size_t n) {  // how many of n limbs, the first ones
  if (n < (size_t)kOnePassLimbs) return 0;
  const size_t tail = n % kOnePassRound;
  return n < (size_t)kOnePassRound || tail >= (size_t)kOnePassTail ? n : n - tail;
}
void launch_ntt1p_fwd(const Context &c, const I8NttTabs &T, const Ntt8Job *jobs, int n,
                      hipStream_t st);

// Device tables of the one-pass inverse transform (ntt1p_inv_tables).
constexpr int kI8InvCtxRow = 1;   // + c0
constexpr int kI8InvCtxCol = 17;  // + r0
constexpr int kI8InvCtx = 33;
struct I8InvTabs {
  const int32_t *planes = nullptr;  // [prime][kI8InvCtx][4 planes][64 lanes][4]
  const int32_t *corr = nullptr;    // [prime][16] offset corrections
  const int32_t *twm = nullptr;     // [prime] inverse 4-step twiddles
};
// One limb: dst = INTT(src, or src (*) src2) c1 with c1m = c1 2^32 mod q
// centred; canonical, or centred in [-(q - 1)/2, (q - 1)/2].
struct Inv1pJob {
  const uint32_t *src, *src2;
  uint32_t *dst;
  int32_t c1m;
  int16_t prime, centred;
};
static_assert(sizeof(Inv1pJob) == 32, "Inv1pJob is one 32-byte record");
int ntt1p_inv_tables(Context &c, I8InvTabs *out);
// prod: every job has src2
void launch_ntt1p_inv(const Context &c, const I8InvTabs &T, const Inv1pJob *jobs, int n,
                      bool prod, hipStream_t st);

// ---- BaseConv on the int8 matrix cores / on the vector unit ----------------

constexpr int kI8MaxDst = 64;

// One BaseConv instance: S centred int32 source limbs -> D destination limbs.
// i8: planes holds the byte planes of the table (ck_i8.hip, bconv_i8_planes);
// valu: ftab holds D x S x {hi, lo} 16-bit halves of the same table.
struct BconvI8Inst {
  const int32_t *src;
  uint32_t *dst;
  const int64_t *planes;
  const double *ftab;
  int S, D;
  int canonical;  // 1: outputs in [0, t); 0: lazy int32 within (-t, t)
  int pad_;
  uint16_t dst_limb[kI8MaxDst];
  uint8_t dst_prime[kI8MaxDst];
};

constexpr int kMaxBconvI8Inst = 4;  // instances per kernel-argument launch
struct BconvI8Launch {
  int n;
  BconvI8Inst inst[kMaxBconvI8Inst];
};

void launch_bconv_i8_table(const Context &c, const BconvI8Inst *insts, int n, int dsts,
                           int max_s, int max_d, hipStream_t st);
// kernel-argument form (single operations: no device table)
void launch_bconv_i8(const Context &c, const BconvI8Launch &L, hipStream_t st);

// ---- BaseConv fused with the forward column stages -------------------------

// Four destination limbs of one BaseConv: S centred int32 source limbs, the
// quad's operand planes, and for each destination its limb (nullptr past the
// last one) and prime.
struct BcolsQuad {
  const int32_t *src;
  const int32_t *planes;
  uint32_t *dst[4];
  int32_t S;
  uint8_t prime[4];
  int64_t pad_;
};
static_assert(sizeof(BcolsQuad) == 64, "BcolsQuad is one 64-byte record");

constexpr int kMaxBcolsQuads = 48;  // quads of a kernel-argument launch
struct BcolsLaunch {
  BcolsQuad quad[kMaxBcolsQuads];
};

// The quads of one BaseConv, in destination order; quads = the table's
// operand planes (bconv_quad_planes).
void add_bcols_quads(std::vector<BcolsQuad> &out, const int32_t *src, int S,
                     const int32_t *quads, const std::vector<uint32_t *> &dst,
                     const std::vector<int> &prime);
// dst = the column stages of the forward transform of the BaseConv (lazy
// int32, as the column pass leaves it); limbs / max_s = destinations in all
// quads / the largest S among them
void launch_bconv_cols(const Context &c, const BcolsLaunch &L, int n, int limbs, int max_s,
                       hipStream_t st);
void launch_bconv_cols_table(const Context &c, const BcolsQuad *quads, int n, int limbs,
                             int max_s, hipStream_t st);

// The int8 operand planes of a context BaseConv table (a ModUp group's or a
// ModDown plan's FP64 {hi, lo} table on the device, S sources x D
// destinations), built on first use from the table's words and kept in the
// context. Returns nullptr (with the error set) on failure.
const int64_t *bconv_i8_planes_for(const Context &c, const double *d_ftab, int S, int D,
                                   const uint8_t *dst_prime);
// The int8 form of a FP64-table BaseConv instance (same source, outputs
// and destinations); false on failure.
bool to_i8_inst(const Context &c, const BconvInst &in, BconvI8Inst *out);
void launch_bconv_valu_table(const Context &c, const BconvI8Inst *insts, int n, int dsts,
                             int max_s, hipStream_t st);

}  // namespace ck
