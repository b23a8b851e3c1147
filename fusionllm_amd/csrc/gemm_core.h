// gemm_core.h — building blocks of the gfx950 bf16 GEMM main loop shared by the
// grouped expert products.
//
// Tile: 256 x 256 outputs per 512-thread workgroup (8 waves, 4 x 2, each wave a
// 64 x 128 sub-tile of 4 x 8 blocks of v_mfma_f32_16x16x32_bf16), K stepped by
// 64 through two LDS stages of 64 KB.
//
// * Global -> LDS copies use global_load_lds_dwordx4 (16 bytes per lane written
//   straight into LDS, no VGPR round trip), issued from inline assembly so that
//   the compiler neither reorders them nor waits for them: every wait on them
//   is explicit.  Operands whose rows are K-contiguous (128-byte rows in LDS)
//   have the 16-byte chunks of a row XOR-swizzled (slot = chunk ^ (row & 7),
//   swzk below) by choosing which global chunk a lane fetches, which makes the
//   fragment reads free of bank conflicts.
// * A stage is four 16 KB units A0, A1, B0, B1: half of each wave's rows (A)
//   and columns (B), with all 64 k.  A K step is four quarters of a wave's
//   block, (A0, B0), (A0, B1), (A1, B0), (A1, B1), 16 MFMAs each.  A unit is in
//   registers a quarter or two after it was first read, and its slot is then
//   refilled with the stage after the next: five to six units (80 - 96 KB) are
//   in flight at any time, against 64 KB for half of the time when a whole
//   stage was consumed before its slot was refilled.
// * Every quarter is a read phase (its LDS reads, two copies, a wait) and an
//   MFMA phase, each ended by a workgroup barrier.  Waves 4 - 7 run one phase
//   behind waves 0 - 3, so the two waves of a SIMD alternate: one issues MFMAs
//   while the other reads and copies.  The phases hold no branches (past the
//   last step the copies repeat the last stage instead of stopping; stores of
//   an epilogue are waited for like the copies): a few scalar instructions
//   more in each read phase cost 10-25 % of the loop.
//   Measured on MI355X, share of a product's cycles in which the MFMA units are
//   busy (hardware counters), with one barrier and eight copies per step and
//   both waves of a SIMD in step -> in this form: C2 (49152 rows, d = 768, I =
//   2048) gate/up forward 0.40 -> 0.50, down forward 0.41 -> 0.58, gate/up dX
//   0.48 -> 0.57; C5 (229376 rows, d = 2048, I = 1408) 0.45 -> 0.70, 0.41 -> 0.73,
//   0.49 -> 0.66.  The clock falls with it, at C5 from 2.0 - 2.1 to 1.65 - 1.9 GHz.
//   Times: C2 355 -> 305 us, 178 -> 148, 304 -> 277; C5 2770 -> 2140, 1490 -> 1045,
//   2560 -> 2140; outputs bit-identical.
// * MFMA operands are swapped (srcA = B fragment, srcB = A fragment), so that a
//   lane's 4 accumulators hold 4 consecutive output columns of one row:
//   acc[i][j] of lane l = C[16 i + l % 16][16 j + 4 (l / 16) + 0..3].
#pragma once

#include "fmoe_common.h"

namespace fmoe {
namespace core {

constexpr int BM = 256, BN = 256, BK = 64, NT = 512;
constexpr int RB = BK * 2;                  // LDS bytes per operand row
constexpr int A_BYTES = BM * RB;            // 32 KB
constexpr int STAGE = (BM + BN) * RB;       // 64 KB
constexpr int EPI = 4096;                   // epilogue staging bytes per wave
constexpr int SMEM = 2 * STAGE + 8 * EPI;   // 160 KB: the whole LDS of a CU
constexpr int WM = 4, WN = 2;               // wave grid
constexpr int WTM = BM / WM, WTN = BN / WN; // 64 x 128 per wave
constexpr int FM = WTM / 16, FN = WTN / 16; // 4 x 8 blocks of 16 x 16
constexpr int LT = 8;                       // copy instructions per lane per stage
constexpr int LU = LT / 4;                  // ... per unit
constexpr int UNIT = 16384;                 // bytes of a unit (half of an operand's stage)
constexpr int UNIT_ROW = 256;               // bytes of a k row of a unit copied as it lies (128 columns)

// Operand stages: 16-byte chunk c of 128-byte row r sits at slot c ^ swzk(r).
// With this swizzle the fragment reads below (lane l: row l % 16 of a
// 16-row group, chunk l / 16 [+4]) are free of LDS bank conflicts on gfx950
// (measured with SQ_LDS_BANK_CONFLICT; folding bit 3 of the row into the
// swizzle gave 2-way conflicts).
__device__ __forceinline__ int swzk(int r) { return r & 7; }
// Epilogue staging of 128-byte rows: slot c ^ swz(r).
__device__ __forceinline__ int swz(int r) { return (r ^ (r >> 3)) & 7; }

__device__ __forceinline__ uint32_t lds_addr(const void* p) {
  // generic -> LDS address space (a C-style cast is the only form clang accepts)
  return static_cast<uint32_t>(reinterpret_cast<uintptr_t>((const __attribute__((address_space(3))) uint8_t*)p));
}

// One 16-byte-per-lane copy global -> LDS.  lds: wave-uniform LDS byte address
// of the 1 KB the wave writes; base: wave-uniform global address; voff: this
// lane's byte offset from base.
__device__ __forceinline__ void copy16(uint32_t lds, const void* base, uint32_t voff) {
  asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, %2\n" ::"s"(lds), "v"(voff), "s"(base)
               : "memory");
}

// One 4-byte-per-lane copy global -> LDS (lane l writes LDS bytes lds + 4 l).
__device__ __forceinline__ void copy4(uint32_t lds, const void* base, uint32_t voff) {
  asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dword %1, %2\n" ::"s"(lds), "v"(voff), "s"(base) : "memory");
}

// Workgroup barrier (no waits).
__device__ __forceinline__ void barrier() { asm volatile("s_barrier" ::: "memory"); }

// Wait until at most N vector-memory operations of this wave are in flight and
// its LDS reads are done, then synchronise the workgroup.
template <int N>
__device__ __forceinline__ void wait_vm_barrier() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier\n" ::"n"(N) : "memory");
}
// The same, waiting for the LDS reads only.
__device__ __forceinline__ void wait_lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier\n" ::: "memory"); }

// LDS address of a lane's fragment 0 of one operand: its row (l % 16 of the
// wave's block) at chunk l / 16, swizzled.  For rows r = base + 16 f + l % 16
// with base % 16 == 0, swzk(r) = l & 7, so fragment f is 2048 f further on and
// the second 32-deep half of the stage is one XOR of 64 (chunk bit 2).
__device__ __forceinline__ uint32_t frag_base(int row0, int lane) {
  const int t = (lane >> 4) ^ (lane & 7);
  return static_cast<uint32_t>((row0 + (lane & 15)) * RB + (t << 4));
}

// ---- operands read as they lie ([K, N] row-major, N contiguous): the weights
// of the backward dX products (dh = d_out * w2, dx = [da | db] * [w1; w3]) and
// both operands of the weight gradients, without a transposed copy.
// A unit is 64 k rows of 256 bytes (128 columns), copied as they lie (32-byte
// windows of a k row XOR-swizzled by wsw(k row)); fragments are read with
// ds_read_b64_tr_b16, which returns to lane (h = l / 16, i = l % 16) column i
// of the 4 x 4 block of 16-bit values that the group's source lanes 4 j + q
// address (row j, 4 values at column 4 q); two such reads, 4 k rows apart,
// give a lane 8 consecutive k of one column.
__device__ __forceinline__ int wsw(int r) { return (r & 3) | (((r >> 3) & 1) << 2); }

// Lane's address of fragment 0 (k 0..31) of a unit copied as it lies, relative
// to the unit: k row 8 h + jq (+4 for the second read), the wave's first
// window win0 (a multiple of the fragments it reads there), swizzled by
// wsw(8 h + jq).  Fragment f: ^ (f << 5); the second 32 k rows: + TR_KHALF.
__device__ __forceinline__ uint32_t tr_base(int win0, int lane) {
  const int h = lane >> 4, jq = (lane >> 2) & 3, q = lane & 3;
  const int fr = jq | ((h & 1) << 2);
  return static_cast<uint32_t>((8 * h + jq) * UNIT_ROW + ((win0 ^ fr) << 5) + 8 * q);
}
constexpr uint32_t TR_KHALF = 32 * UNIT_ROW;

typedef short s16x4 __attribute__((ext_vector_type(4)));
// One fragment of a unit copied as it lies: 8 consecutive k of the lane's
// column (two transposing reads).
__device__ __forceinline__ bf16x8 tr_frag(uint32_t addr) {
  typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
  const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(uintptr_t)addr);
  const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(uintptr_t)(addr + 4u * UNIT_ROW));
  return __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
}

// ---- the K step -------------------------------------------------------------
// Fragments of one half of an operand's stage: [k half][block].
typedef bf16x8 AFrag[2][FM / 2];
typedef bf16x8 BFrag[2][FN / 2];

#define FMOE_MF(c, a, b) "v_mfma_f32_16x16x32_bf16 " c ", " a ", " b ", " c "\n"
// Four MFMAs: two column blocks (p) x two row blocks (q).  The statement is
// ordered against the fragment reads and the copies around it (memory
// clobber), which fixes the interleaving; the fragment reads are compiler
// loads, so the compiler waits for exactly those that a statement consumes.
__device__ __forceinline__ void mfma4(f32x4& c00, f32x4& c10, f32x4& c01, f32x4& c11, const bf16x8& p0,
                                      const bf16x8& p1, const bf16x8& q0, const bf16x8& q1) {
  asm volatile(FMOE_MF("%[c00]", "%[p0]", "%[q0]") FMOE_MF("%[c10]", "%[p0]", "%[q1]")
               FMOE_MF("%[c01]", "%[p1]", "%[q0]") FMOE_MF("%[c11]", "%[p1]", "%[q1]")
               : [c00] "+v"(c00), [c10] "+v"(c10), [c01] "+v"(c01), [c11] "+v"(c11)
               : [p0] "v"(p0), [p1] "v"(p1), [q0] "v"(q0), [q1] "v"(q1)
               : "memory");
}
#undef FMOE_MF

// Quarter (I, J) of the wave's block, 64 deep: rows 32 I .. +31, columns
// 64 J .. +63; every accumulator adds k 0..31 of the stage, then k 32..63.
template <int I, int J>
__device__ __forceinline__ void quarter(f32x4 (&acc)[FM][FN], const AFrag& a, const BFrag& b) {
  __builtin_amdgcn_s_setprio(1);
#pragma unroll
  for (int x = 0; x < 4; ++x) {
    const int kh = x >> 1, n = (x & 1) * 2;
    mfma4(acc[2 * I][4 * J + n], acc[2 * I + 1][4 * J + n], acc[2 * I][4 * J + n + 1], acc[2 * I + 1][4 * J + n + 1],
          b[kh][n], b[kh][n + 1], a[kh][0], a[kh][1]);
  }
  __builtin_amdgcn_s_setprio(0);
  barrier();
}

}  // namespace core
}  // namespace fmoe
