// gemm.hip — grouped bf16 GEMMs on CDNA4 matrix cores
// (v_mfma_f32_16x16x32_bf16) for the expert SwiGLU products of FusionLLM's
// DeepSeekMoE.
//
// Replaces SwiGLUExpert.forward (models/moe.py:20-21) called once per active
// expert in the loop of moe.py:66-76 and once for the shared expert
// (moe.py:86), and the autograd of those calls.  All experts (and the shared
// expert as one more group) go into a single launch per product; the tile ->
// (expert, rows) mapping is computed on the device from offsets[], so no
// host synchronisation is needed for the ragged, skewed expert sizes.
//
// Row-grouped products (rows_gemm_kernel, modes below): persistent
// workgroups of 8 waves walk 256 x 256 output tiles in an XCD-contiguous
// order.  Both operands are K-contiguous in memory and reach LDS through
// global_load_lds copies (no registers) into a two-stage ring of 64-deep K
// steps that runs on across tile boundaries; a wave owns a 64 x 128 block
// and runs the hand-scheduled K step of gemm_core.h.  The epilogue stages
// each 16-row slice through LDS for 16-byte stores and fuses the SwiGLU
// (forward: a | b and h = silu(a) * b; backward: da, db from dh, a, b).  The
// tiles of the last, partial round of the plain-output products are split
// along K, with fp32 partials summed in range order by split_reduce_kernel.
//
// Weight gradients (wgrad_tr_kernel): work units (group, K chunk, tile);
// both operands are MN-contiguous, copied as they lie and read with
// ds_read_b64_tr_b16 (transposing LDS reads); multi-chunk groups write fp32
// partials that wgrad_reduce_kernel adds in chunk order.
//
// Decode-sized launches send groups of at most kSmallM rows to
// small_gemm_kernel, which streams the weights once (when no group of the
// launch can exceed 2 kSmallM rows, every group, in slabs of kSmallM).
#include <atomic>
#include <type_traits>

#include "fmoe_common.h"
#include "gemm_core.h"

namespace fmoe {

// ---- row-grouped products ---------------------------------------------------
// The activations are row-major [rows, K] (K-contiguous).  The weights are
// the nn.Linear weights as they lie: [out, in] with K = in for the forward
// products (K-contiguous, read like the activations), and [K, N] row-major
// for the backward dX products (dh = d_out * w2 reads w2 [dim, inter];
// dx = [da | db] * [w1; w3] reads w1, w3 [inter, dim]), whose B stages are
// copied as they lie and read with transposing LDS reads (gemm_core.h).
enum GemmMode { GATEUP_FWD = 0, DOWN_FWD = 1, DOWN_BWD = 2, GATEUP_BWD = 3 };

struct GemmArgs {
  const uint16_t* a_routed;  // [rows_routed, K], or with gather: x [T, K]
  const int32_t* gather;     // GATEUP_FWD tiled kernel: routed row r reads a_routed row gather[r] / gather_k
                             // (nullptr: row r; launches of more than kSmallLaunchRows rows only)
  int gather_k;
  uint64_t gather_magic;     // slot_div_magic(gather_k)
  const uint16_t* a_shared;  // [rows_shared, K] (nullptr: rows follow the routed rows)
  int64_t lda;
  const int32_t* offsets;  // [E+1], device
  int E;
  int rows_routed;
  int rows_shared;
  int K;        // reduction length
  int N;        // output columns (GATEUP_FWD: inter = h columns)
  int inter;    // SwiGLU width (GATEUP_FWD, DOWN_BWD)
  int64_t ldb;  // leading dimension of the weight operand (row length as it lies in memory)
  uint16_t* c0;  // main output (ab / out / d_ab / dx_rows)
  uint16_t* c1;  // GATEUP_FWD: h
  const uint16_t* aux;  // DOWN_BWD: ab
  int64_t ldc0, ldc1, ldaux;
  const uint16_t* b0[FMOE_MAX_EXPERTS + 1];  // w1 (GATEUP_*) / w2 (DOWN_*)
  const uint16_t* b1[FMOE_MAX_EXPERTS + 1];  // w3 (GATEUP_*)
  int small_max;  // groups with 1 .. small_max rows go to small_gemm_kernel (0: none)
  int small_compact;  // DOWN_FWD small kernel: the grid covers only groups with rows
  float* split_ws;  // fp32 partials of the K-split tiles of the last round (nullptr: no split)
};

// ---- tiled row-grouped kernel ----------------------------------------------
// Persistent: a grid of at most one workgroup per CU walks the tiles
// t = blockIdx.x, blockIdx.x + gridDim.x, ...  Tiles are enumerated group by
// group (experts 0..E-1, then the shared expert), m tile major; the tile ->
// (group, rows) map comes from offsets[] on the device.  The global -> LDS
// copies run as one continuous two-stage ring over all K steps of all of a
// workgroup's tiles, so the next tile's first operands arrive while the current
// tile finishes and writes its epilogue.  Rows past a group's end and weight
// rows past N are clamped to the last valid one (their products are never
// stored), so no operand is read out of bounds.

// Tile -> (group, rows) map of a launch, held by the lanes of each wave: lane
// e < E has expert e's first row, rows and first tile, so that a tile is found
// with one ballot and three lane reads.  (A walk over the groups with a scalar
// load each took 2-3 us per tile at E = 64, twice per tile: in the copy cursor
// and in the epilogue.)
struct TileMap {
  int row, rows, start;  // of expert `lane` (start: INT_MAX past the last expert)
  int routed, total;     // tiles of the routed groups, of all groups
};

struct Tile {
  int g, tm, tn, row_base, M;  // group, m tile, n tile, the group's first row and rows
};

__device__ __forceinline__ TileMap tile_map(const GemmArgs& a, const int32_t* __restrict__ offsets, int tiles_n,
                                            int lane) {
  TileMap m;
  const int lo = offsets[min(lane, a.E)], hi = offsets[min(lane + 1, a.E)];
  m.row = lo;
  m.rows = hi - lo;  // 0 past the last expert
  const int nt = (m.rows <= a.small_max) ? 0 : ((m.rows + core::BM - 1) / core::BM) * tiles_n;
  const int incl = wave_incl_scan(nt, lane);
  m.start = lane < a.E ? incl - nt : INT32_MAX;
  m.routed = __builtin_amdgcn_readlane(incl, 63);
  m.total = m.routed + ((a.rows_shared <= a.small_max) ? 0 : ((a.rows_shared + core::BM - 1) / core::BM) * tiles_n);
  return m;
}

// Tile t < total: the last expert whose first tile is at most t (experts
// without tiles start where the next one does, or past t).
__device__ __forceinline__ Tile locate_tile(const GemmArgs& a, const TileMap& m, int tiles_n, int t) {
  Tile r;
  if (t >= m.routed) {
    r.g = a.E;
    r.row_base = a.rows_routed;
    r.M = a.rows_shared;
    t -= m.routed;
  } else {
    r.g = 63 - __builtin_clzll(__ballot(m.start <= t));
    r.row_base = __builtin_amdgcn_readlane(m.row, r.g);
    r.M = __builtin_amdgcn_readlane(m.rows, r.g);
    t -= __builtin_amdgcn_readlane(m.start, r.g);
  }
  r.tm = t / tiles_n;
  r.tn = t - r.tm * tiles_n;
  return r;
}

// K-split of the last, partial round of tiles.  With T tiles on P
// workgroups, the T mod P tiles of the last round would run on a fraction of
// the CUs; instead each is split into S K ranges (S <= 8, R * S <= P, at
// least 8 K steps per range) whose fp32 partials a split reduction adds in
// range order before the product's epilogue.  Work items: tiles 0 .. full-1
// whole, then R * S ranges.  A launch of fewer tiles than CUs takes every CU
// for its ranges.  Measured on MI355X (d = 768, I = 2048, 8 experts; the grid
// of such a launch was its tile count, which split nothing): gate/up dX at T
// = 300 83 -> 40 us, T = 1021 84 -> 47, T = 2048 84 -> 59; dense T = 6100 84
// -> 57.  Ranges of 4 steps (K = 768: three of 12) cost more in partials
// (256 KB per range, written and read once) and in the reduction's launch
// than they save: gate/up forward, dense T = 6100 64 -> 49 us without.
// Only for runs of fewer than kSplitMaxRounds full rounds: over many rounds
// the workgroups' finishing times spread by about a tile anyway (d = 2048, I =
// 1408, 64 experts, 21 to 38 rounds: 1 to 15 us lost on every product).
struct SplitPlan {
  int full, R, S;
  __device__ __forceinline__ int items() const { return full + R * S; }
};
constexpr int kSplitMaxS = 8;       // K ranges per split tile
constexpr int kSplitMinSteps = 8;   // K steps per range
constexpr int kSplitBatch = 4;      // ranges whose partials a split reduction loads together
constexpr int kSplitMaxRounds = 8;  // full rounds above which no tile is split
constexpr int kReduceParts = 16;  // blocks of a split reduction per split tile, 16 rows each

template <int MODE>
__device__ __forceinline__ SplitPlan split_plan(const GemmArgs& a, int T, int P, int nk) {
  SplitPlan sp{T, 0, 1};
  if (a.split_ws == nullptr || T <= 0) return sp;
  const int R = T % P;
  if (R == 0 || T / P >= kSplitMaxRounds) return sp;
  const int S = min(min(P / R, kSplitMaxS), nk / kSplitMinSteps);
  if (S < 2) return sp;
  sp.full = T - R;
  sp.R = R;
  sp.S = S;
  return sp;
}
// Workgroup b runs on XCD b % 8 (round-robin dispatch over the 8 XCDs of an
// MI355X, each with its own L2).  Item i of round r of workgroup b is
// r * P + xcd_slot(b): the workgroups of one XCD take a contiguous range of
// items, so the tiles that share operand rows (consecutive n tiles of one m
// tile) meet in the same L2.
__device__ __forceinline__ int xcd_slot(int b, int P) {
  return (P % 8 == 0) ? (b % 8) * (P / 8) + b / 8 : b;
}

// Work item -> tile, first K step, K steps, partial slot (-1: whole tile).
__device__ __forceinline__ void split_item(const SplitPlan& sp, int nk, int item, int& tile, int& k0, int& kn,
                                           int& slot) {
  if (item < sp.full) {
    tile = item;
    k0 = 0;
    kn = nk;
    slot = -1;
  } else {
    const int j = item - sp.full;
    const int s = j % sp.S;
    tile = sp.full + j / sp.S;
    k0 = s * nk / sp.S;
    kn = (s + 1) * nk / sp.S - k0;
    slot = j;
  }
}

// 16-byte global store / load; nt marks data streamed through once (the
// SwiGLU activations a|b and h, read again only in the backward pass, and
// their gradient), so it does not displace operands from the caches.
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ void store16(uint16_t* p, const uint4& v, bool nt) {
  if (nt) {
    const u32x4 q = {v.x, v.y, v.z, v.w};
    __builtin_nontemporal_store(q, reinterpret_cast<u32x4*>(p));
  } else {
    *reinterpret_cast<uint4*>(p) = v;
  }
}
__device__ __forceinline__ uint4 load16(const uint16_t* p, bool nt) {
  if (nt) {
    const u32x4 q = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p));
    return make_uint4(q.x, q.y, q.z, q.w);
  }
  return *reinterpret_cast<const uint4*>(p);
}

// SwiGLU backward of 8 columns (h = s * b, s = bf16(silu(a)); dh arrives
// bf16-rounded): da = bf16(bf16(dh * b) * silu'(a)), db = bf16(dh * s), with
// silu(a) = a * sg and silu'(a) = sg * (1 + a (1 - sg)) = sg + silu(a) (1 - sg).
__device__ __forceinline__ void swiglu_bwd8(const uint4& dhv, const uint4& av, const uint4& bv, uint4& dav,
                                            uint4& dbv) {
  float dh[8], af[8], bfv[8], da[8], db[8];
  unpack8(dhv, dh);
  unpack8(av, af);
  unpack8(bv, bfv);
#pragma unroll
  for (int e = 0; e < 8; e += 2) {
    const float sg0 = fast_sigmoid(af[e]), sg1 = fast_sigmoid(af[e + 1]);
    const float sa0 = af[e] * sg0, sa1 = af[e + 1] * sg1;
    float sv0 = sa0, sv1 = sa1, ds0 = dh[e] * bfv[e], ds1 = dh[e + 1] * bfv[e + 1];
    bf_round2(sv0, sv1);
    bf_round2(ds0, ds1);
    da[e] = ds0 * fmaf(sa0, 1.0f - sg0, sg0);
    da[e + 1] = ds1 * fmaf(sa1, 1.0f - sg1, sg1);
    db[e] = dh[e] * sv0;
    db[e + 1] = dh[e + 1] * sv1;
  }
  dav = pack8(da);
  dbv = pack8(db);
}

// Down-backward epilogue of a full tile (this wave's 64 x 128 block of dh in
// acc).  The SwiGLU backward costs about as many instructions per element as
// the block has accumulators, so the block is first staged whole: dh rounded
// to bf16, through the wave's 4 KB of LDS one 16-row slice at a time, read
// back as 16-byte row segments (64 registers, the accumulators are then
// free); then the slices' a|b are loaded, computed and stored one after
// another; the slice loop is unrolled and the compiler issues a slice's loads
// ahead of the stores before it.  The copies' offsets and the fragment
// addresses of the main loop are formed again after it instead of kept (11
// registers spilled with them, none without: C2 238 -> 232 us, C5 1401 -> 1372, T
// = 9001, d = 1024, I = 1536 218 -> 213).  Two slices of loads issued up front
// spill 51 beside them (C2 302 us, C5 1855 against 1500 in that session).  Row
// pointers are uniform (scalar registers); a lane adds one offset.
__device__ __forceinline__ void down_bwd_full_epilogue(const GemmArgs& args, const f32x4 (&acc)[core::FM][core::FN],
                                                       uint8_t* ep, int el, int64_t grow0, int col0) {
  using namespace core;
  uint4 dhv[FM][4];
  {
    const int r = el & 15;
#pragma unroll
    for (int i = 0; i < FM; ++i) {
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        // chunk c of row r at slot c ^ r (256-byte rows)
        const int col = j * 16 + (el >> 4) * 4;
        const uint32_t off = r * 256 + ((((col >> 3) ^ r)) << 4) + (col & 7) * 2;
        *reinterpret_cast<uint2*>(ep + off) =
            make_uint2(pack2(acc[i][j][0], acc[i][j][1]), pack2(acc[i][j][2], acc[i][j][3]));
      }
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int rr = t * 4 + (el >> 4), c = el & 15;
        dhv[i][t] = *reinterpret_cast<const uint4*>(ep + rr * 256 + ((c ^ rr) << 4));
      }
    }
  }
  // lane: rows 4 t + el / 16 of each slice, columns col0 + 8 (el % 16) .. +7
  const uint8_t* abase = reinterpret_cast<const uint8_t*>(args.aux + grow0 * args.ldaux + col0);
  const uint32_t aoff = static_cast<uint32_t>((el >> 4) * static_cast<int>(args.ldaux) + (el & 15) * 8) * 2u;
  const int64_t astep = args.ldaux * 2 * 4;  // bytes per 4 rows
  uint8_t* cbase = reinterpret_cast<uint8_t*>(args.c0 + grow0 * args.ldc0 + col0);
  const uint32_t coff = static_cast<uint32_t>((el >> 4) * static_cast<int>(args.ldc0) + (el & 15) * 8) * 2u;
  const int64_t cstep = args.ldc0 * 2 * 4;
  const int64_t binter = args.inter * 2;  // bytes from a to b (and from da to db)
  uint4 pa[FM][4], pb[FM][4];
  auto load_slice = [&](int i) {
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const uint8_t* rp = abase + (i * 4 + t) * astep;
      pa[i][t] = load16(reinterpret_cast<const uint16_t*>(rp + aoff), true);
      pb[i][t] = load16(reinterpret_cast<const uint16_t*>(rp + binter + aoff), true);
    }
  };
  asm volatile("" ::: "memory");  // the loads are not hoisted into the staging above
  load_slice(0);
#pragma unroll
  for (int i = 0; i < FM; ++i) {
    if (i > 0) load_slice(i);
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      uint4 dav, dbv;
      swiglu_bwd8(dhv[i][t], pa[i][t], pb[i][t], dav, dbv);
      uint8_t* rp = cbase + (i * 4 + t) * cstep;
      store16(reinterpret_cast<uint16_t*>(rp + coff), dav, true);
      store16(reinterpret_cast<uint16_t*>(rp + binter + coff), dbv, true);
    }
  }
}

// GATHER (GATEUP_FWD only): args.gather is set; a separate instantiation, so
// that the plain kernel carries none of the gathered path's code.
template <int MODE, bool GATHER = false>
__global__ __launch_bounds__(core::NT, 1) void rows_gemm_kernel(const GemmArgs args,
                                                                 const int32_t* __restrict__ offsets) {
  using namespace core;
  constexpr bool GA = MODE == GATEUP_FWD && GATHER;
  __shared__ __attribute__((aligned(1024))) uint8_t smem[SMEM];
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = w / WN, wn = w % WN;
  const uint32_t sbase = lds_addr(smem);

  // GATEUP_FWD: a tile covers 128 h columns (128 rows of w1 and of w3).
  constexpr int TN_COLS = (MODE == GATEUP_FWD) ? BN / 2 : BN;
  // The backward dX products read the weights as they lie ([K, N]) with
  // transposing LDS reads.
  constexpr bool BTR = (MODE == DOWN_BWD || MODE == GATEUP_BWD);
  const int tiles_n = (args.N + TN_COLS - 1) / TN_COLS;
  const TileMap map = tile_map(args, offsets, tiles_n, lane);
  const int total_tiles = map.total;
  const int NP = static_cast<int>(gridDim.x), b = xcd_slot(static_cast<int>(blockIdx.x), NP);
  const int nk = args.K / BK;
  const SplitPlan sp = split_plan<MODE>(args, total_tiles, NP, nk);
  {
    // descriptors of the split tiles for the split reduction (after the
    // partials): first row, valid rows, first output column, valid columns
    // (GATEUP_FWD: h columns, 128 per tile)
    const int r = static_cast<int>(blockIdx.x);
    if (args.split_ws != nullptr) {
      int4* hdr = reinterpret_cast<int4*>(args.split_ws + static_cast<int64_t>(NP) * BM * BN);
      if (r == 0 && threadIdx.x == 0) hdr[0] = make_int4(sp.R, sp.S, 0, 0);
      if (r < sp.R) {
        const Tile t = locate_tile(args, map, tiles_n, sp.full + r);
        if (threadIdx.x == 0)
          hdr[1 + r] = make_int4(t.row_base + t.tm * BM, min(t.M - t.tm * BM, BM), t.tn * TN_COLS,
                                 min(args.N - t.tn * TN_COLS, TN_COLS));
      }
    }
  }
  const int my_items = (sp.items() - b + NP - 1) / NP;  // items b, b + NP, ...
  if (my_items <= 0) return;
  // K steps of 64 over all of this workgroup's items (only the last can be a range)
  int total = (my_items - 1) * nk;
  {
    int t_, k0_, kn_, s_;
    split_item(sp, nk, b + (my_items - 1) * NP, t_, k0_, kn_, s_);
    total += kn_;
  }

  // ---- global -> LDS copy cursor
  // A stage is copied in halves of four instructions: half u holds rows 32 u ..
  // +31 of every wave's 64 A rows and rows (columns of the output) 64 u .. +63
  // of every wave's 128 B rows.  Instruction i of wave w writes eight LDS rows,
  // lane l fetches row l / 8 of them, global chunk dchunk (the swizzled slot
  // l % 8).
  const uint32_t lds_a = sbase + (64 * (w >> 2) + 8 * (w & 3)) * RB;
  const uint32_t lds_b = sbase + A_BYTES + w * 1024;
  int c_ti = 0, c_kt = 0, c_kn = 0;  // item ordinal, step within it, its steps
  const uint8_t* c_a = nullptr;      // A rows of the tile being copied, at the step's k
  const uint8_t* c_b0 = nullptr;     // B operand(s), at the step's k
  const uint8_t* c_b1 = nullptr;
  int c_ksw = 0;                     // GATEUP_BWD: the step at which B goes on in w3
  // this lane's byte offsets from c_a / c_b* of the tile (rows and columns past
  // the end clamped to the last valid one), formed once per tile; [2 u + i]
  constexpr int NBO = (MODE == GATEUP_FWD) ? 2 : 4;
  uint32_t a_off[4], b_off[NBO];
  const int lda = static_cast<int>(args.lda), ldb = static_cast<int>(args.ldb);
  auto form_offsets = [&](const Tile& t) __attribute__((always_inline)) {
    const bool gathered = GA && t.g < args.E;
    const int last_row = min(t.M - t.tm * BM, BM) - 1, n0 = t.tn * TN_COLS;
    // the lane as an opaque value: what follows is formed here, not kept in
    // registers through the main loop
    int l = lane;
    asm volatile("" : "+v"(l));
    const int dchunk = (l & 7) ^ swzk(l >> 3);
    if constexpr (BTR) {
      // B as it lies: unit u holds columns 64 u .. +63 of every wave's 128;
      // instruction i of wave w writes its k rows 32 i + krow, 16-byte chunk
      // cb of a row (wsw(32 i + krow) == wsw(krow))
      const int krow = 4 * w + (l >> 4);
      const int cb = ((((l & 15) >> 1) ^ wsw(krow)) << 1) | (l & 1);
      const int col = 128 * (cb >> 3) + 8 * (cb & 7);  // + 64 u: its column of the tile
#pragma unroll
      for (int q = 0; q < 4; ++q)
        b_off[q] = static_cast<uint32_t>((32 * (q & 1) + krow) * ldb + min(n0 + 64 * (q >> 1) + col, args.N - 8)) * 2u;
    } else {
      // GATEUP_FWD: the wave's first 64 B rows are w1 rows, the others the w3 rows of the same h columns
#pragma unroll
      for (int q = 0; q < NBO; ++q) {
        const int n = min(n0 + ((MODE == GATEUP_FWD) ? 64 * q : 128 * (q & 1) + 64 * (q >> 1)) + 8 * w + (l >> 3), args.N - 1);
        b_off[q] = static_cast<uint32_t>(n * ldb + dchunk * 8) * 2u;
      }
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int r = min(64 * (w >> 2) + 8 * (w & 3) + (l >> 3) + 128 * (q & 1) + 32 * (q >> 1), last_row);
      // gathered: the routed rows are token rows of x, row r: x row gather[r] / gather_k
      // (the index loads are waited for here, once per tile)
      if (gathered) {
        const uint32_t slot = static_cast<uint32_t>(args.gather[t.row_base + t.tm * BM + r]);
        a_off[q] = (slot_token(slot, args.gather_magic) * static_cast<uint32_t>(lda) + static_cast<uint32_t>(dchunk * 8)) * 2u;
      } else {
        a_off[q] = static_cast<uint32_t>(r * lda + dchunk * 8) * 2u;
      }
    }
  };
  auto copy_tile = [&](int ti) __attribute__((always_inline)) {
    int tile, slot, k0;
    split_item(sp, nk, b + ti * NP, tile, k0, c_kn, slot);
    const Tile t = locate_tile(args, map, tiles_n, tile);
    const bool gathered = GA && t.g < args.E;
    const uint16_t* A = gathered ? args.a_routed
                        : (t.g < args.E || args.a_shared == nullptr)
                            ? args.a_routed + static_cast<int64_t>(t.row_base) * args.lda
                            : args.a_shared;
    if (!gathered) A += static_cast<int64_t>(t.tm) * BM * args.lda;
    c_a = reinterpret_cast<const uint8_t*>(A + k0 * BK);
    if constexpr (BTR) {
      // GATEUP_BWD: k < inter from w1, else from w3
      const int kb = k0 * BK;
      const bool hi = MODE == GATEUP_BWD && kb >= args.inter;
      c_b0 = reinterpret_cast<const uint8_t*>((hi ? args.b1[t.g] : args.b0[t.g]) +
                                              static_cast<int64_t>(hi ? kb - args.inter : kb) * args.ldb);
      c_b1 = reinterpret_cast<const uint8_t*>(args.b1[t.g]);
      c_ksw = hi ? INT32_MAX : args.inter / BK - k0;
    } else {
      c_b0 = reinterpret_cast<const uint8_t*>(args.b0[t.g] + k0 * BK);
      if constexpr (MODE == GATEUP_FWD) c_b1 = reinterpret_cast<const uint8_t*>(args.b1[t.g] + k0 * BK);
    }
    form_offsets(t);
  };
  copy_tile(0);
  // Unit u of step it's stage (two instructions): a stage's units are issued
  // in the order A0, B0, B1, A1, and A1 moves the cursor on.  Past the last
  // step the last stage is copied again (into slots that are free and not read
  // any more), so that every wait counts the same operations.
  auto issue_a = [&](int it, int u) __attribute__((always_inline)) {
    const uint32_t st = lds_a + (it & 1) * STAGE;
#pragma unroll
    for (int i = 0; i < 2; ++i) copy16(st + (128 * i + 32 * u) * RB, c_a, a_off[2 * u + i]);
    if (u == 0) return;
    const int64_t bstep = BTR ? 2 * BK * args.ldb : RB;
    c_a += RB;
    c_b0 += bstep;
    if constexpr (MODE == GATEUP_FWD) c_b1 += RB;
    if (__builtin_expect(++c_kt == c_kn, 0)) {
      if (c_ti + 1 < my_items) {
        c_kt = 0;
        copy_tile(++c_ti);
      } else {  // past the end: the last stage again
        --c_kt;
        c_a -= RB;
        c_b0 -= bstep;
        if constexpr (MODE == GATEUP_FWD) c_b1 -= RB;
      }
    } else if (MODE == GATEUP_BWD && c_kt == c_ksw) {
      c_b0 = c_b1;  // (a range that ends at the last row of w1 never gets here)
    }
  };
  auto issue_b = [&](int it, int u) __attribute__((always_inline)) {
    const uint32_t st = lds_b + (it & 1) * STAGE;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      if constexpr (BTR)
        copy16(st + u * UNIT + i * 8192, c_b0, b_off[2 * u + i]);
      else if constexpr (MODE == GATEUP_FWD)
        copy16(st + (128 * i + 64 * u) * RB, u ? c_b1 : c_b0, b_off[i]);
      else
        copy16(st + (128 * i + 64 * u) * RB, c_b0, b_off[2 * u + i]);
    }
  };

  // ---- fragments: A rows 16 f of the wave's 64 (units a0, a1: f 0..1, 2..3),
  // B rows 16 f of its 128 (b0, b1: f 0..3, 4..7)
  uint32_t xa = frag_base(wm * WTM, lane);
  uint32_t xb = A_BYTES + (BTR ? tr_base(4 * wn, lane) : frag_base(wn * WTN, lane));
  AFrag a0, a1;
  BFrag b0, b1;
  typedef __attribute__((address_space(3))) bf16x8 lds_bf16x8;
  auto lds_frag = [&](uint32_t x, uint32_t src, int kh, int f) {
    return *(const lds_bf16x8*)(uintptr_t)((x ^ (kh * 64u)) + src + 2048u * f);
  };
  auto read_a = [&](AFrag& f, int u, uint32_t src, int kh, int m) { f[kh][m] = lds_frag(xa, src, kh, 2 * u + m); };
  auto read_b = [&](BFrag& f, int u, uint32_t src, int kh, int n) {
    if constexpr (BTR)
      f[kh][n] = tr_frag(((src + xb) ^ (n << 5)) + u * UNIT + kh * TR_KHALF);
    else
      f[kh][n] = lds_frag(xb, src, kh, 4 * u + n);
  };

  // The fragments a tile starts with: A0 whole, B0's first 32-deep half.
  auto read_first = [&](uint32_t src) {
#pragma unroll
    for (int kh = 0; kh < 2; ++kh)
#pragma unroll
      for (int m = 0; m < 2; ++m) read_a(a0, 0, src, kh, m);
#pragma unroll
    for (int n = 0; n < 4; ++n) read_b(b0, 0, src, 0, n);
  };

  issue_a(0, 0);
  issue_b(0, 0);
  issue_b(0, 1);
  issue_a(0, 1);
  issue_a(1, 0);
  issue_b(1, 0);
  issue_b(1, 1);
  wait_vm_barrier<5 * LU>();
  read_first(sbase);
  const bool late = w >= 4;  // this wave's SIMD partner is one phase ahead
  if (late) barrier();

  f32x4 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  uint8_t* ep = smem + 2 * STAGE + w * EPI;  // this wave's epilogue staging (4 KB)
  int e_ti = 0, e_kt = 0, e_kn = c_kn, e_slot = -1, e_tile = 0;
  {
    int k0_;
    split_item(sp, nk, b, e_tile, k0_, e_kn, e_slot);
  }
  // At a step's waits, only the units issued after the ones waited for may be
  // in flight (counting the stores of the last epilogue as well, so that they
  // need not have completed, measured no faster and takes branches).
  for (int it = 0; it < total; ++it) {
    // keep the per-step fragment addresses from being hoisted out of the loop
    asm volatile("" : "+v"(xa), "+v"(xb));
    const uint32_t cur = sbase + (it & 1) * STAGE, nxt = sbase + ((it + 1) & 1) * STAGE;
    // (0, 0)
#pragma unroll
    for (int n = 0; n < 4; ++n) read_b(b0, 0, cur, 1, n);
    issue_a(it + 1, 1);
    wait_vm_barrier<5 * LU>();  // B1 of this stage
    quarter<0, 0>(acc, a0, b0);
    // (0, 1)
#pragma unroll
    for (int kh = 0; kh < 2; ++kh)
#pragma unroll
      for (int n = 0; n < 4; ++n) read_b(b1, 1, cur, kh, n);
    issue_a(it + 2, 0);
    wait_vm_barrier<5 * LU>();  // A1 of this stage
    quarter<0, 1>(acc, a0, b1);
    // (1, 0)
#pragma unroll
    for (int kh = 0; kh < 2; ++kh)
#pragma unroll
      for (int m = 0; m < 2; ++m) read_a(a1, 1, cur, kh, m);
    issue_b(it + 2, 0);
    wait_vm_barrier<4 * LU>();  // A0, B0 of the next stage
    quarter<1, 0>(acc, a1, b0);
    // (1, 1): the next step's first fragments (at a tile's end they are read
    // again after its epilogue, which needs the registers)
    read_first(nxt);
    issue_b(it + 2, 1);
    wait_lds_barrier();
    quarter<1, 1>(acc, a1, b1);

    if (++e_kt < e_kn) continue;
    // ---- tile epilogue: this wave's 64 x 128 block (both wave groups together)
    if (!late) barrier();
    e_kt = 0;
    asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 3\n" ::: "memory");  // MFMA results -> VALU reads
    // lane index as an opaque value: keeps the epilogue's address arithmetic
    // from being hoisted out of the main loop (where it would occupy registers)
    int el = lane;
    asm volatile("" : "+v"(el));
    if (e_slot >= 0) {
      // K-split range: fp32 partial of the 256 x 256 tile (local row-major),
      // 16-row slices without valid rows left out (the reduction reads none)
      float* part = args.split_ws + static_cast<int64_t>(e_slot) * BM * BN;
      const Tile t = locate_tile(args, map, tiles_n, e_tile);
      const int rows_valid = t.M - t.tm * BM;
#pragma unroll
      for (int i = 0; i < FM; ++i)
        if (wm * WTM + i * 16 < rows_valid)
#pragma unroll
          for (int j = 0; j < FN; ++j)
            *reinterpret_cast<f32x4*>(part + (wm * WTM + i * 16 + (el & 15)) * BN + wn * WTN + j * 16 + (el >> 4) * 4) =
                acc[i][j];
    } else {
      const Tile t = locate_tile(args, map, tiles_n, e_tile);
      const int rows_valid = min(t.M - t.tm * BM, BM);
      const int col0 = t.tn * TN_COLS + wn * (TN_COLS / WN);  // first output column of this wave
      const bool full = rows_valid == BM && (t.tn + 1) * TN_COLS <= args.N;
      const int64_t grow0 = static_cast<int64_t>(t.row_base) + t.tm * BM + wm * WTM;
      bool epi_done = false;
      if constexpr (MODE == DOWN_BWD) {
        if (full) {
          down_bwd_full_epilogue(args, acc, ep, el, grow0, col0);
          epi_done = true;
        }
      }
      if (!epi_done)
  #pragma unroll
      for (int i = 0; i < FM; ++i) {
        // DOWN_BWD (partial tiles; full ones took down_bwd_full_epilogue): a|b
        // of the 16 rows go in flight before the staging below, all 8 loads at
        // once (rows and columns clamped into the tile, so the addresses stay
        // valid for a partial tile; such values are not stored)
        uint4 pa[4], pb[4];
        if constexpr (MODE == DOWN_BWD) {
  #pragma unroll
          for (int t = 0; t < 4; ++t) {
            const int r = t * 4 + (el >> 4), c = el & 15;
            const int64_t growc = grow0 - wm * WTM + min(wm * WTM + i * 16 + r, rows_valid - 1);
            const uint16_t* src = args.aux + growc * args.ldaux + min(col0 + c * 8, args.N - 8);
            pa[t] = load16(src, true);
            pb[t] = load16(src + args.inter, true);
          }
        }
        // stage rows 16 i .. 16 i + 15 of the wave block, 128 accumulator columns
        // (256 bytes per row; chunk c of row r at slot c ^ r); GATEUP_FWD keeps
        // the packed a | b values for h below
        uint2 pk[FN];
        {
          const int r = el & 15;
  #pragma unroll
          for (int j = 0; j < FN; ++j) {
            const int col = j * 16 + (el >> 4) * 4;
            const uint32_t off = r * 256 + ((((col >> 3) ^ r)) << 4) + (col & 7) * 2;
            pk[j].x = pack2(acc[i][j][0], acc[i][j][1]);
            pk[j].y = pack2(acc[i][j][2], acc[i][j][3]);
            *reinterpret_cast<uint2*>(ep + off) = pk[j];
          }
        }
  #pragma unroll
        for (int t = 0; t < 4; ++t) {
          const int r = t * 4 + (el >> 4), c = el & 15;
          const uint4 v = *reinterpret_cast<const uint4*>(ep + r * 256 + ((c ^ r) << 4));
          const int lrow = wm * WTM + i * 16 + r;
          const int64_t grow = grow0 + i * 16 + r;
          if constexpr (MODE == GATEUP_FWD) {
            // columns 0..63: a, 64..127: b for h columns col0 .. col0 + 63
            const int hc = col0 + (c & 7) * 8;
            if (full || (lrow < rows_valid && hc < args.N)) {
              store16(args.c0 + grow * args.ldc0 + (c < 8 ? 0 : args.inter) + hc, v, true);
            }
          } else if constexpr (MODE == DOWN_BWD) {
            // h = s * b, s = bf16(silu(a)); dh arrives bf16-rounded:
            // da = bf16(bf16(dh * b) * silu'(a)), db = bf16(dh * s)
            const int hc = col0 + c * 8;
            if (full || (lrow < rows_valid && hc < args.N)) {
              uint4 dav, dbv;
              swiglu_bwd8(v, pa[t], pb[t], dav, dbv);
              store16(args.c0 + grow * args.ldc0 + hc, dav, true);
              store16(args.c0 + grow * args.ldc0 + args.inter + hc, dbv, true);
            }
          } else {
            const int oc = col0 + c * 8;
            if (full || (lrow < rows_valid && oc < args.N))
              *reinterpret_cast<uint4*>(args.c0 + grow * args.ldc0 + oc) = v;
          }
        }
        if constexpr (MODE == GATEUP_FWD) {
          // h = bf16(bf16(silu(a)) * b) for the 16 rows x 64 h columns, staged as
          // 128-byte rows (chunk c of row r at slot c ^ swz(r))
          const int r = el & 15;
  #pragma unroll
          for (int j = 0; j < 4; ++j) {
            // a = bf16(acc) and b likewise, as staged above
            const float a[4] = {__uint_as_float(pk[j].x << 16), __uint_as_float(pk[j].x & 0xffff0000u),
                                __uint_as_float(pk[j].y << 16), __uint_as_float(pk[j].y & 0xffff0000u)};
            const float b[4] = {__uint_as_float(pk[j + 4].x << 16), __uint_as_float(pk[j + 4].x & 0xffff0000u),
                                __uint_as_float(pk[j + 4].y << 16), __uint_as_float(pk[j + 4].y & 0xffff0000u)};
            float hv[4];
  #pragma unroll
            for (int e = 0; e < 4; ++e) hv[e] = a[e] * fast_sigmoid(a[e]);
            bf_round2(hv[0], hv[1]);
            bf_round2(hv[2], hv[3]);
  #pragma unroll
            for (int e = 0; e < 4; ++e) hv[e] = hv[e] * b[e];
            const int col = j * 16 + (el >> 4) * 4;
            const uint32_t off = r * 128 + ((((col >> 3) ^ swz(r))) << 4) + (col & 7) * 2;
            uint2 v;
            v.x = pack2(hv[0], hv[1]);
            v.y = pack2(hv[2], hv[3]);
            *reinterpret_cast<uint2*>(ep + off) = v;
          }
  #pragma unroll
          for (int t = 0; t < 2; ++t) {
            const int rr = t * 8 + (el >> 3), c = el & 7;
            const uint4 v = *reinterpret_cast<const uint4*>(ep + rr * 128 + ((c ^ swz(rr)) << 4));
            const int lrow = wm * WTM + i * 16 + rr;
            const int hc = col0 + c * 8;
            if (full || (lrow < rows_valid && hc < args.N))
              store16(args.c1 + (grow0 + i * 16 + rr) * args.ldc1 + hc, v, true);
          }
        }
      }
    }  // whole tile
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    asm volatile("s_nop 1" ::: "memory");  // VALU writes -> MFMA reads of the accumulators
    if constexpr (MODE == DOWN_BWD) {
      // the copies' offsets and the fragment addresses are formed again: kept
      // across this epilogue they made it spill 11 registers
      int tile_, k0_, kn_, slot_;
      split_item(sp, nk, b + c_ti * NP, tile_, k0_, kn_, slot_);
      form_offsets(locate_tile(args, map, tiles_n, tile_));
      xa = frag_base(wm * WTM, el);
      xb = A_BYTES + tr_base(4 * wn, el);
    }
    // the next tile's first fragments (after the last tile a harmless re-read)
    read_first(sbase + ((it + 1) & 1) * STAGE);
    if (late && it + 1 < total) barrier();
    if (++e_ti < my_items) {
      int k0_;
      split_item(sp, nk, b + e_ti * NP, e_tile, k0_, e_kn, e_slot);
    }
  }
  // the copies past the end have landed before the workgroup's LDS is given back
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

// ---- split reductions
// The product wrote, after the P tiles of partials, a header {R, S} and one
// descriptor {first row, valid rows, first output column, valid output
// columns} per split tile.  A reduction sums a split tile's S partials in
// range order and writes the tile through the product's epilogue.  Block =
// (split tile r, sixteenth of its rows); a thread takes units of 8
// consecutive partial columns of one row.  Every partial slot is a whole
// BM x BN region, so the loads need no bounds; only valid rows and columns
// are stored.

struct SplitTile {
  bool active;
  int S;
  int4 d;
  const float* src0;  // the tile's first partial
};

__device__ __forceinline__ SplitTile split_tile(const float* ws, int P) {
  using namespace core;
  const int4* hdr = reinterpret_cast<const int4*>(ws + static_cast<int64_t>(P) * BM * BN);
  const int4 h0 = hdr[0];
  const int r = blockIdx.x / kReduceParts;
  SplitTile t;
  t.S = h0.y;
  t.d = r < h0.x ? hdr[1 + r] : make_int4(0, 0, 0, 0);
  t.active = static_cast<int>(blockIdx.x % kReduceParts) * 16 < t.d.y;  // the block has valid rows
  t.src0 = ws + static_cast<int64_t>(r) * h0.y * BM * BN;
  return t;
}

// Partial values o .. o + 7 of the S ranges, summed in range order from 0 (the
// loads of kSplitBatch ranges issued together; ranges past S re-read range
// S - 1 and are not added).
__device__ __forceinline__ void sum_ranges8(const SplitTile& t, int o, float* acc) {
  using namespace core;
#pragma unroll
  for (int e = 0; e < 8; ++e) acc[e] = 0.0f;
  for (int s0 = 0; s0 < t.S; s0 += kSplitBatch) {
    float4 u[kSplitBatch][2];
#pragma unroll
    for (int s = 0; s < kSplitBatch; ++s) {
      const float* p = t.src0 + static_cast<int64_t>(min(s0 + s, t.S - 1)) * BM * BN + o;
      u[s][0] = *reinterpret_cast<const float4*>(p);
      u[s][1] = *reinterpret_cast<const float4*>(p + 4);
    }
#pragma unroll
    for (int s = 0; s < kSplitBatch; ++s) {
      const float v[8] = {u[s][0].x, u[s][0].y, u[s][0].z, u[s][0].w, u[s][1].x, u[s][1].y, u[s][1].z, u[s][1].w};
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[e] = (s0 + s < t.S) ? acc[e] + v[e] : acc[e];
    }
  }
}

// DOWN_FWD, GATEUP_BWD: the bf16 tile.  Two units per thread.
__global__ __launch_bounds__(256) void split_reduce_kernel(const float* __restrict__ ws, int P,
                                                           uint16_t* __restrict__ out, int64_t ldo) {
  using namespace core;
  const SplitTile t = split_tile(ws, P);
  if (!t.active) return;
  const int row0 = (blockIdx.x % kReduceParts) * 16;
  float acc[2][8];
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int u = threadIdx.x + q * 256;
    sum_ranges8(t, (row0 + u / 32) * BN + (u % 32) * 8, acc[q]);
  }
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int u = threadIdx.x + q * 256, row = row0 + u / 32, col = (u % 32) * 8;
    if (row < t.d.y && col < t.d.w)
      *reinterpret_cast<uint4*>(out + static_cast<int64_t>(t.d.x + row) * ldo + t.d.z + col) = pack8(acc[q]);
  }
}

// GATEUP_FWD: a|b = bf16(acc), h = bf16(bf16(silu(a)) * b), as the tile
// epilogue.  The partial columns of wave half w hold a for h columns
// 64 w .. 64 w + 63, then b for the same columns.  One unit per thread.
__global__ __launch_bounds__(256) void split_reduce_gateup_kernel(const GemmArgs args, int P) {
  using namespace core;
  const SplitTile t = split_tile(args.split_ws, P);
  if (!t.active) return;
  const int row = (blockIdx.x % kReduceParts) * 16 + threadIdx.x / 16, hc = (threadIdx.x % 16) * 8;
  const int pa = (hc / 64) * 128 + hc % 64;
  float a[8], b[8];
  sum_ranges8(t, row * BN + pa, a);
  sum_ranges8(t, row * BN + pa + 64, b);
  if (row >= t.d.y || hc >= t.d.w) return;
  const uint4 pka = pack8(a), pkb = pack8(b);
  const int64_t grow = static_cast<int64_t>(t.d.x) + row;
  const int col = t.d.z + hc;
  store16(args.c0 + grow * args.ldc0 + col, pka, true);
  store16(args.c0 + grow * args.ldc0 + args.inter + col, pkb, true);
  float ar[8], br[8], hv[8];
  unpack8(pka, ar);
  unpack8(pkb, br);
#pragma unroll
  for (int e = 0; e < 8; e += 2) {
    float h0v = ar[e] * fast_sigmoid(ar[e]), h1v = ar[e + 1] * fast_sigmoid(ar[e + 1]);
    bf_round2(h0v, h1v);
    hv[e] = h0v * br[e];
    hv[e + 1] = h1v * br[e + 1];
  }
  store16(args.c1 + grow * args.ldc1 + col, pack8(hv), true);
}

// DOWN_BWD: dh = bf16(acc), then the SwiGLU backward of the tile epilogue
// with a|b read from args.aux (rows and columns clamped into the tile for
// the loads).  Two units per thread.
__global__ __launch_bounds__(256) void split_reduce_down_bwd_kernel(const GemmArgs args, int P) {
  using namespace core;
  const SplitTile t = split_tile(args.split_ws, P);
  if (!t.active) return;
  const int row0 = (blockIdx.x % kReduceParts) * 16;
  float acc[2][8];
  uint4 la[2], lb[2];
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int u = threadIdx.x + q * 256, row = row0 + u / 32, c = (u % 32) * 8;
    const int64_t lrow = static_cast<int64_t>(t.d.x) + min(row, t.d.y - 1);
    const uint16_t* src = args.aux + lrow * args.ldaux + t.d.z + min(c, t.d.w - 8);
    la[q] = load16(src, true);
    lb[q] = load16(src + args.inter, true);
    sum_ranges8(t, row * BN + c, acc[q]);
  }
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int u = threadIdx.x + q * 256, row = row0 + u / 32, c = (u % 32) * 8;
    if (row >= t.d.y || c >= t.d.w) continue;
    const int64_t grow = static_cast<int64_t>(t.d.x) + row;
    const int hc = t.d.z + c;
    uint4 dav, dbv;
    swiglu_bwd8(pack8(acc[q]), la[q], lb[q], dav, dbv);  // dh arrives bf16-rounded, as in the tile epilogue
    store16(args.c0 + grow * args.ldc0 + hc, dav, true);
    store16(args.c0 + grow * args.ldc0 + args.inter + hc, dbv, true);
  }
}

// ---- small groups (decode-sized batches) -------------------------------------
// A group of at most kSmallM rows would leave a 256 x 256 tile nearly empty
// and run its whole K loop in one workgroup; such a product is bound by
// streaming the weights, so the aim is to have all of them in flight at once.
// One workgroup owns 16 output columns of one group (GATEUP_FWD: 16 h
// columns, i.e. the same 16 rows of w1 and of w3, two accumulators); its
// waves (4 for the gate/up product, 8 for the down product, whose K is the
// longer one in the reference's shapes: the faster counts measured) split
// the K steps of 32 evenly, and each wave issues the loads of up to CH steps
// before their MFMAs (v_mfma_f32_16x16x32_bf16, operands read straight from
// memory: the weights once, the few activation rows from L2).  The partial
// tiles are added in wave order through LDS.  MB = 16-row blocks the kernel is built for (the
// host picks it from a bound on the group sizes; with MB > 2 fewer K steps
// are in flight, the activation fragments take the registers; a group of
// more than 16 MB rows runs as slabs of 16 MB rows); a slab that needs fewer
// blocks runs the 2- or 4-block variant, with more K steps in flight.  Rows past a group's end repeat its last row and are not stored.
constexpr int kSmallM = 128;
// The host knows the shared expert's row count, so the small kernel takes the
// shared group as slabs of kSharedSlab rows in workgroups of their own (more
// workgroups, each with more K steps of loads in flight).
constexpr int kSharedSlab = 64;

template <int MODE>
constexpr int small_waves() { return MODE == GATEUP_FWD ? 4 : 8; }

template <int MODE>
constexpr int small_nb() { return MODE == GATEUP_FWD ? 2 : 1; }  // weight matrices
constexpr int kSmallPass = 2;  // m blocks reduced per LDS pass

// One slab of at most 16 MB rows of one group: the K loop with CH steps of
// loads in flight, then the wave-order reduction through LDS and the stores.
// The MFMA chain of every accumulator runs over the wave's K steps in order,
// whatever MB and CH are, so the result does not depend on them.
template <int MODE, int MB>
__device__ __forceinline__ void small_slab(const GemmArgs& args,
                                           float (*red)[kSmallPass][small_nb<MODE>()][4][64], int wave,
                                           int lane, int cb, const uint16_t* A, int M, int row_base,
                                           const uint16_t* w0, const uint16_t* w1, int s_begin, int s_end) {
  constexpr int kSmallWaves = small_waves<MODE>();
  constexpr int NB = small_nb<MODE>();
  constexpr int CH = MB <= 2 ? 8 : (MB == 4 ? 4 : 2);
  constexpr int PASS = kSmallPass;
  const int r16 = lane & 15, kq = (lane >> 4) * 8;
  const int mb_n = (M + 15) / 16;  // 1 .. MB
  const uint16_t* ap[MB];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb)
    ap[mb] = A + static_cast<int64_t>(min(16 * mb + r16, M - 1)) * args.lda + kq;

  f32x4 acc[MB][NB];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb)
#pragma unroll
    for (int b = 0; b < NB; ++b) acc[mb][b] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
  for (int s0 = s_begin; s0 < s_end; s0 += CH) {
    bf16x8 bw[CH][NB], af[CH][MB];
#pragma unroll
    for (int u = 0; u < CH; ++u) {
      if (s0 + u < s_end) {
        const int k = 32 * (s0 + u);
        bw[u][0] = *reinterpret_cast<const bf16x8*>(w0 + k);
        if constexpr (NB == 2) bw[u][1] = *reinterpret_cast<const bf16x8*>(w1 + k);
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
          if (mb < mb_n) af[u][mb] = *reinterpret_cast<const bf16x8*>(ap[mb] + k);
      }
    }
#pragma unroll
    for (int u = 0; u < CH; ++u) {
      if (s0 + u < s_end) {
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
          if (mb < mb_n)
#pragma unroll
            for (int b = 0; b < NB; ++b)
              acc[mb][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bw[u][b], af[u][mb], acc[mb][b], 0, 0, 0);
      }
    }
  }
  // Passes of PASS m blocks: every wave parks its partials, wave p of the pass
  // adds the eight partials of m block (pass base + p) in wave order and stores.
  const int m = lane & 15, n0 = cb * 16 + (lane >> 4) * 4;
  for (int base = 0; base < mb_n; base += PASS) {
#pragma unroll
    for (int p = 0; p < PASS; ++p) {
      const int mb = base + p;
#pragma unroll
      for (int q = 0; q < MB; ++q)  // static register index
        if (q == mb)
#pragma unroll
          for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int r = 0; r < 4; ++r) red[wave][p][b][r][lane] = acc[q][b][r];
    }
    __syncthreads();
    const int mb = base + wave;
    if (wave < PASS && mb < mb_n && 16 * mb + m < M) {
      float v[NB][4];
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          float t = red[0][wave][b][r][lane];
#pragma unroll
          for (int w = 1; w < kSmallWaves; ++w) t = t + red[w][wave][b][r][lane];
          v[b][r] = t;
        }
      const int64_t row = row_base + 16 * mb + m;
      if constexpr (MODE == GATEUP_FWD) {
        float hv[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          v[0][r] = bf_round(v[0][r]);
          v[1][r] = bf_round(v[1][r]);
          hv[r] = bf_round(v[0][r] * fast_sigmoid(v[0][r])) * v[1][r];
        }
        uint16_t* ab = args.c0 + row * args.ldc0;
        *reinterpret_cast<uint2*>(ab + n0) = make_uint2(pack2(v[0][0], v[0][1]), pack2(v[0][2], v[0][3]));
        *reinterpret_cast<uint2*>(ab + args.inter + n0) =
            make_uint2(pack2(v[1][0], v[1][1]), pack2(v[1][2], v[1][3]));
        *reinterpret_cast<uint2*>(args.c1 + row * args.ldc1 + n0) =
            make_uint2(pack2(hv[0], hv[1]), pack2(hv[2], hv[3]));
      } else {
        *reinterpret_cast<uint2*>(args.c0 + row * args.ldc0 + n0) =
            make_uint2(pack2(v[0][0], v[0][1]), pack2(v[0][2], v[0][3]));
      }
    }
    __syncthreads();
  }
}

// The 2- and 4-block variants are held to 3 (gate/up) or 4 (down) waves per
// SIMD, one more than the compiler picks by itself, without spills: a
// decode launch of a few thousand waves then needs fewer rounds (C3 M = 32:
// gate/up 15.8 -> 14.1 us, down 13.0 -> 11.6 us).  The 1-block variant is
// faster without the bound, the 8-block gate/up variant would spill.
template <int MODE, int MB>
__global__ __launch_bounds__(small_waves<MODE>() * 64)
__attribute__((amdgpu_waves_per_eu((MB == 2 || MB == 4) ? (MODE == GATEUP_FWD ? 3 : 4) : 1))) void small_gemm_kernel(
    const GemmArgs args) {
  static_assert(MODE == GATEUP_FWD || MODE == DOWN_FWD, "forward products only");
  constexpr int kSmallWaves = small_waves<MODE>();
  __shared__ float red[kSmallWaves][kSmallPass][small_nb<MODE>()][4][64];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ncb = args.N / 16;
  const int cb = blockIdx.x % ncb;
  int g, row_base, M, shared_off = 0;
  if (MODE == DOWN_FWD && args.small_compact) {
    // Fewer routed rows than experts: workgroup -> (group, column block) over
    // the groups this kernel takes (1 .. small_max rows: routed experts in
    // order, then the shared expert), so that the grid holds no workgroups
    // of empty experts (empty 8-wave workgroups ahead of the busy ones cost
    // up to 2 us at M = 1).  Lane e < E reads expert e's rows, the wave ranks
    // the qualifying experts with a ballot and takes the rank-th.
    const int rank = blockIdx.x / ncb, lane_e = threadIdx.x & 63;
    int lo = 0, m_e = 0;
    if (lane_e < args.E) {
      lo = args.offsets[lane_e];
      m_e = args.offsets[lane_e + 1] - lo;
    }
    const bool qual = m_e > 0 && m_e <= args.small_max;
    const uint64_t qmask = __ballot(qual);
    const int nq = __popcll(qmask);
    if (rank < nq) {
      const uint64_t below = lane_e == 0 ? 0ull : (qmask & (~0ull >> (64 - lane_e)));
      g = __ffsll(static_cast<unsigned long long>(__ballot(qual && __popcll(below) == rank))) - 1;
      row_base = __shfl(lo, g, 64);
      M = __shfl(m_e, g, 64);
    } else {
      // the shared expert, slab rank - nq
      shared_off = (rank - nq) * kSharedSlab;
      if (args.rows_shared > args.small_max || shared_off >= args.rows_shared) return;
      g = args.E;
      row_base = args.rows_routed + shared_off;
      M = min(kSharedSlab, args.rows_shared - shared_off);
    }
  } else {
    // one workgroup per (routed group or shared slab, column block); empty
    // groups return at once
    g = blockIdx.x / ncb;
    if (g < args.E) {
      row_base = args.offsets[g];
      M = args.offsets[g + 1] - row_base;
      if (M == 0 || M > args.small_max) return;
    } else {
      shared_off = (g - args.E) * kSharedSlab;
      if (args.rows_shared > args.small_max || shared_off >= args.rows_shared) return;
      g = args.E;
      row_base = args.rows_routed + shared_off;
      M = min(kSharedSlab, args.rows_shared - shared_off);
    }
  }
  const uint16_t* A_group = (g < args.E || args.a_shared == nullptr)
                                ? args.a_routed + static_cast<int64_t>(row_base) * args.lda
                                : args.a_shared + static_cast<int64_t>(shared_off) * args.lda;
  // Fragments (operands swapped: srcA = weight rows, srcB = activation rows):
  // lane l supplies row l % 16 of each, K elements 8 (l / 16) .. +7 of a step,
  // and gets C[m = l % 16][n = 4 (l / 16) + 0..3].
  const int r16 = lane & 15, kq = (lane >> 4) * 8;
  const uint16_t* w0 = args.b0[g] + static_cast<int64_t>(cb * 16 + r16) * args.ldb + kq;
  const uint16_t* w1 = (MODE == GATEUP_FWD) ? args.b1[g] + static_cast<int64_t>(cb * 16 + r16) * args.ldb + kq
                                            : nullptr;
  const int nsteps = args.K / 32;
  const int s_begin = wave * nsteps / kSmallWaves, s_end = (wave + 1) * nsteps / kSmallWaves;
  // A group of more than 16 MB rows (at most small_max = 2 kSmallM) runs as
  // slabs of 16 MB rows, each streaming the weights again.
  const int M_group = M, row_base_group = row_base;
  for (int slab = 0; slab < M_group; slab += 16 * MB) {
    const int M = min(16 * MB, M_group - slab), row_base = row_base_group + slab;
    const uint16_t* A = A_group + static_cast<int64_t>(slab) * args.lda;
    const int mb_n = (M + 15) / 16;  // 1 .. MB
    // A launch built for MB blocks runs a smaller slab with fewer blocks and
    // more K steps in flight.
    if constexpr (MB >= 4) {
      if (mb_n <= 2) {
        small_slab<MODE, 2>(args, red, wave, lane, cb, A, M, row_base, w0, w1, s_begin, s_end);
        continue;
      }
    }
    if constexpr (MB >= 8) {
      if (mb_n <= 4) {
        small_slab<MODE, 4>(args, red, wave, lane, cb, A, M, row_base, w0, w1, s_begin, s_end);
        continue;
      }
    }
    small_slab<MODE, MB>(args, red, wave, lane, cb, A, M, row_base, w0, w1, s_begin, s_end);
  }
}

// ---- weight gradients (K-grouped) -------------------------------------------
// G_e = A_e^T B_e with A_e [M_e, m_out], B_e [M_e, n_out] (both MN-contiguous).
// Work unit = (group, K chunk of kc rows, output tile).  A group whose rows fit
// in one chunk writes its tile directly; otherwise every chunk writes an fp32
// partial and wgrad_reduce_kernel adds the chunks of a group in chunk order.
struct WgradArgs {
  const uint16_t* a_routed;
  const uint16_t* a_shared;
  int64_t lda;
  const uint16_t* b_routed;  // [rows_routed, n_out], or with b_gather: x [T, n_out]
  const uint16_t* b_shared;
  int64_t ldb;
  const int32_t* b_gather;   // routed row r of B is b_routed row b_gather[r] / gather_k (nullptr: row r)
  int gather_k;
  uint64_t gather_magic;     // slot_div_magic(gather_k)
  const int32_t* offsets;
  int E;
  int rows_routed;
  int rows_shared;
  int m_out, n_out, m_split;
  int kc;
  int out_dtype;
  float* partial;
  void* out_lo[FMOE_MAX_EXPERTS + 1];
  void* out_hi[FMOE_MAX_EXPERTS + 1];
};

// K chunks of a group of M rows: kc rows each, to the nearest count, so that
// they can be made equally long (a multiple of 64 rows; the last may be
// shorter or empty) and a group somewhat larger than kc stays whole.
__host__ __device__ __forceinline__ int wgrad_chunks(int64_t M, int kc) {
  const int n = static_cast<int>((M + kc / 2) / kc);
  return n < 1 ? 1 : n;
}

__device__ __forceinline__ void group_rows(const WgradArgs& a, int g, int& row_base, int& M) {
  if (g < a.E) {
    row_base = a.offsets[g];
    M = a.offsets[g + 1] - row_base;
  } else {
    row_base = a.rows_routed;
    M = a.rows_shared;
  }
}

// ---- weight gradients on the shared core ------------------------------------
// Both operands are MN-contiguous ([rows, m_out] and [rows, n_out]), so their
// 64 x 256 stage tiles are copied as they lie in memory (K-major: 64 k rows of
// 512 bytes) with the same global -> LDS copies as the row products, and the
// MFMA fragments are read with ds_read_b64_tr_b16, which returns to lane
// (h = l / 16, i = l % 16) of each 16-lane group the i-th column of the 4 x 4
// block of 16-bit values that source lanes 4 j + q address (row j, 4 values at
// column 4 q): two such reads give a lane 8 consecutive k of one output row.
// The 32-byte windows of a k row are XOR-swizzled by wsw(row) so that the 16
// rows x 32 bytes a read instruction touches fall on distinct banks.
// GATHER: args.b_gather is set (a separate instantiation, so that the plain
// kernel carries none of the gathered path's code).
template <bool GATHER>
__global__ __launch_bounds__(core::NT, 1) void wgrad_tr_kernel(const WgradArgs args,
                                                               const int32_t* __restrict__ offsets) {
  using namespace core;
  __shared__ __attribute__((aligned(1024))) uint8_t smem[2 * STAGE];
  // Gathered B rows: the slot indices of each stage's 64 k rows, a ring of eight
  // stages per wave, so that every wave issues the same operations and the
  // waits can count them (of one ring that wave 0 fills they can't, and waiting
  // for all copies instead drains the ring of stages every step: dW1|dW3 823
  // -> 350 us at C2, 5500 -> 2549 at C5, 622 -> 308 at T = 9001, d = 1024, I = 1536,
  // 16 experts; with the rows copied beforehand 335, 2392 and 290).  Filled by
  // global -> LDS copies three stages ahead of a stage's copies and read when
  // its first B unit is issued, by the wave that filled it, after a wait that
  // covers them; a slot is refilled stages after its last read.
  __shared__ int32_t idx_ring[GATHER ? 8 : 1][8][BK];
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = w / WN, wn = w % WN;  // wave block: 64 m x 128 n
  const uint32_t sbase = lds_addr(smem);
  const int tiles_m = (args.m_out + BM - 1) / BM, tiles_n = (args.n_out + BN - 1) / BN;
  const int tiles = tiles_m * tiles_n;

  // ---- work unit -> (group, K chunk, output tile): the shared group's chunks
  // first (it is the largest group unless the routing is very skewed: at C5,
  // 512 steps against 48, its units dispatched last left 168 CUs idle for
  // 600 us), then the experts'.  The hardware hands the next unit to the next
  // free CU, which balances the uneven units.  Lane e < E holds expert e's
  // rows and first unit, as the tile map of the row products.
  int g, row_base, M, chunks, pbase, unit = blockIdx.x;
  {
    const int s_chunks = args.rows_shared > 0 ? wgrad_chunks(args.rows_shared, args.kc) : 0;
    if (unit < s_chunks * tiles) {
      g = args.E;
      row_base = args.rows_routed;
      M = args.rows_shared;
      chunks = s_chunks;
      pbase = 0;
    } else {
      unit -= s_chunks * tiles;
      const int lo = offsets[min(lane, args.E)], rows = offsets[min(lane + 1, args.E)] - lo;
      const int nc = lane < args.E ? wgrad_chunks(rows, args.kc) : 0;
      const int npart = nc > 1 ? nc : 0;
      const int u_incl = wave_incl_scan(nc * tiles, lane), p_incl = wave_incl_scan(npart, lane);
      if (unit >= __builtin_amdgcn_readlane(u_incl, 63)) return;
      g = __builtin_ctzll(__ballot(u_incl > unit));
      row_base = __builtin_amdgcn_readlane(lo, g);
      M = __builtin_amdgcn_readlane(rows, g);
      chunks = __builtin_amdgcn_readlane(nc, g);
      pbase = (s_chunks > 1 ? s_chunks : 0) + __builtin_amdgcn_readlane(p_incl - npart, g);
      unit -= __builtin_amdgcn_readlane(u_incl - nc * tiles, g);
    }
  }
  const int chunk = unit / tiles, tile = unit - chunk * tiles;
  int tm = tile / tiles_n, tn = tile - tm * tiles_n;
  if (tiles % 8 == 0) {
    // A chunk's units start at a multiple of 8, so workgroup b runs on XCD
    // tile % 8 (workgroups go to the 8 XCDs round-robin).  Each XCD takes whole
    // column blocks of one operand (its L2 then serves them to all of that
    // XCD's tiles of the chunk) and the same share of every chunk.
    const int xcd = tile & 7, j = tile >> 3;
    if (tiles_m % 8 == 0) {
      tm = xcd + 8 * (j / tiles_n);
      tn = j % tiles_n;
    } else if (tiles_n % 8 == 0) {
      tn = xcd + 8 * (j / tiles_m);
      tm = j % tiles_m;
    }
  }
  const int m0 = tm * BM, n0 = tn * BN;
  const int len = ((M + chunks - 1) / chunks + BK - 1) / BK * BK;  // rows of a chunk
  const int k_begin = chunk * len;
  const int k_end = min(M, k_begin + len);
  // <= 0: no rows (a group without rows, whose gradient is zero, or an empty last chunk)
  const int nk = (k_end - k_begin + BK - 1) / BK;
  const bool shared_sep = (g >= args.E);
  const uint16_t* A = (shared_sep && args.a_shared) ? args.a_shared : args.a_routed + static_cast<int64_t>(row_base) * args.lda;
  const bool gathered = GATHER && !shared_sep;
  const uint16_t* B = (shared_sep && args.b_shared) ? args.b_shared
                      : gathered ? args.b_routed
                                 : args.b_routed + static_cast<int64_t>(row_base) * args.ldb;
  const int lda = static_cast<int>(args.lda), ldb = static_cast<int>(args.ldb);
  const int wr = GATHER ? w : 0;
  const uint32_t ring = lds_addr(&idx_ring[wr][0][0]);
  // stage kt's slot indices into ring slot kt % 8 (rows past k_end repeat the
  // last valid one; the shared group, whose rows are not gathered, fetches a
  // value that it does not use, so that its count is the same)
  const int32_t* idx_src = gathered ? args.b_gather + row_base : offsets;
  auto fetch_idx = [&](int kt) {
    const int r = gathered ? min(k_begin + kt * BK + lane, k_end - 1) : 0;
    copy4(ring + (kt & 7) * (BK * 4), idx_src, static_cast<uint32_t>(r) * 4u);
  };
  // ---- copies: a unit is 128 columns of a stage's 64 k rows (A0, A1, B0, B1
  // in LDS); instruction i of wave w writes its k rows 32 i + drow (1 KB = 4
  // rows of 256 B), lane chunk p = l % 16 holds logical chunk c of the row
  const int drow = 4 * w + (lane >> 4);
  const int p = lane & 15;
  const int c = (((p >> 1) ^ wsw(drow)) << 1) | (p & 1);  // wsw(32 i + drow) == wsw(drow)
  const uint32_t lds_copy = sbase + w * 1024;
  if (gathered) {
    // stages 0..2 before the first copies (stage kt's last unit fetches stage kt + 3)
    for (int q = 0; q < 3 && q < nk; ++q) fetch_idx(q);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  }

  // Unit u of a stage (two instructions); a stage's units are issued in the
  // order A0, B0, B1, A1, and A1 moves on to the next stage.  Past the last
  // stage the last one is copied again (into slots that are free and not read
  // any more), so that every wait counts the same operations.
  // The lane's byte offsets from the stage's first rows (pa, pb): columns past
  // the end clamped to the last ones, rows past k_end to the last valid row
  // (only the last stage can have some).
  const uint8_t* pa = reinterpret_cast<const uint8_t*>(A + static_cast<int64_t>(k_begin) * lda);
  const uint8_t* pb = reinterpret_cast<const uint8_t*>(gathered ? B : B + static_cast<int64_t>(k_begin) * ldb);
  uint32_t a_off[4], b_off[4];  // [2 u + i]
  auto form_rows = [&](int kt) {
    const int last = k_end - 1 - (k_begin + kt * BK);  // >= 0 for kt < nk
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int r = min(32 * (q & 1) + drow, last);
      a_off[q] = static_cast<uint32_t>(r * lda + min(m0 + 128 * (q >> 1) + 8 * c, args.m_out - 8)) * 2u;
      if (!gathered) b_off[q] = static_cast<uint32_t>(r * ldb + min(n0 + 128 * (q >> 1) + 8 * c, args.n_out - 8)) * 2u;
    }
  };
  // gathered B: k row r of a stage is x row (slot of group row k0 + r) / k, from
  // the stage's ring slot
  auto form_gathered = [&](int kt) {
    const int last = k_end - 1 - (k_begin + kt * BK);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int r = min(32 * i + drow, last);
      const uint32_t tok = slot_token(static_cast<uint32_t>(idx_ring[wr][kt & 7][r]), args.gather_magic);
#pragma unroll
      for (int u = 0; u < 2; ++u)
        b_off[2 * u + i] = (tok * static_cast<uint32_t>(ldb) +
                            static_cast<uint32_t>(min(n0 + 128 * u + 8 * c, args.n_out - 8))) * 2u;
    }
  };
  form_rows(0);
  auto issue_a = [&](int kt, int u) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 2; ++i) copy16(lds_copy + (kt & 1) * STAGE + u * UNIT + i * 8192, pa, a_off[2 * u + i]);
    if (u == 0) return;
    if (GATHER) fetch_idx(kt + 3);
    if (kt + 1 < nk) {
      pa += 2 * BK * args.lda;
      if (!gathered) pb += 2 * BK * args.ldb;
      if (kt + 2 == nk) form_rows(kt + 1);
    }
  };
  auto issue_b = [&](int kt, int u) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
      copy16(lds_copy + (kt & 1) * STAGE + A_BYTES + u * UNIT + i * 8192, pb, b_off[2 * u + i]);
  };
  // Rows past k_end in a stage hold copies of the last valid row: zero their A
  // side (after this wave's copies have landed) so that they add nothing.
  auto zero_tail = [&](int kt, int u) {
    const int k0 = k_begin + kt * BK;
    if (kt >= nk || k_end - k0 >= BK) return;
    uint8_t* st = smem + (kt & 1) * STAGE + u * UNIT + w * 1024 + lane * 16;
#pragma unroll
    for (int i = 0; i < 2; ++i)
      if (k0 + 32 * i + drow >= k_end) *reinterpret_cast<uint4*>(st + i * 8192) = make_uint4(0, 0, 0, 0);
  };
  // All but the newest copies of this wave have landed: those of UNITS units,
  // and the FETCHES index fetches among them (one follows each A1).
  auto wait_copies = [&](auto units, auto fetches) {
    constexpr int N = decltype(units)::value * LU + (GATHER ? decltype(fetches)::value : 0);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
  };
  constexpr std::integral_constant<int, 1> n1{};
  constexpr std::integral_constant<int, 2> n2{};
  constexpr std::integral_constant<int, 4> n4{};
  constexpr std::integral_constant<int, 5> n5{};

  // ---- fragment addresses within a unit: the wave's 32 A columns (2 windows), 64 B columns (4)
  uint32_t xa = tr_base(2 * wm, lane), xb = A_BYTES + tr_base(4 * wn, lane);
  AFrag a0, a1;
  BFrag b0, b1;
  auto read_a = [&](AFrag& f, uint32_t unit, int kh, int m) { f[kh][m] = tr_frag(((unit + xa) ^ (m << 5)) + kh * TR_KHALF); };
  auto read_b = [&](BFrag& f, uint32_t unit, int kh, int n) { f[kh][n] = tr_frag(((unit + xb) ^ (n << 5)) + kh * TR_KHALF); };
  auto read_first = [&](uint32_t src) {
#pragma unroll
    for (int kh = 0; kh < 2; ++kh)
#pragma unroll
      for (int m = 0; m < 2; ++m) read_a(a0, src, kh, m);
#pragma unroll
    for (int n = 0; n < 4; ++n) read_b(b0, src, 0, n);
  };

  f32x4 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  asm volatile("s_nop 1" ::: "memory");  // VALU writes -> MFMA reads of the accumulators
  if (nk > 0) {
    if (gathered) form_gathered(0);
    issue_a(0, 0);
    issue_b(0, 0);
    issue_b(0, 1);
    issue_a(0, 1);
    if (gathered) form_gathered(min(1, nk - 1));
    issue_a(1, 0);
    issue_b(1, 0);
    issue_b(1, 1);
    wait_copies(n5, n1);  // A0, B0 of stage 0
    zero_tail(0, 0);
    wait_lds_barrier();
    read_first(sbase);
    const bool late = w >= 4;
    if (late) barrier();

    for (int kt = 0; kt < nk; ++kt) {
      asm volatile("" : "+v"(xa), "+v"(xb));
      const uint32_t cur = sbase + (kt & 1) * STAGE, nxt = sbase + ((kt + 1) & 1) * STAGE;
      // (0, 0)
#pragma unroll
      for (int n = 0; n < 4; ++n) read_b(b0, cur, 1, n);
      issue_a(kt + 1, 1);
      wait_copies(n5, n2);  // B1 of this stage
      wait_lds_barrier();
      quarter<0, 0>(acc, a0, b0);
      // (0, 1)
#pragma unroll
      for (int kh = 0; kh < 2; ++kh)
#pragma unroll
        for (int n = 0; n < 4; ++n) read_b(b1, cur + UNIT, kh, n);
      issue_a(kt + 2, 0);
      wait_copies(n5, n2);  // A1 of this stage (its own fetch may be in flight)
      zero_tail(kt, 1);
      wait_lds_barrier();
      quarter<0, 1>(acc, a0, b1);
      // (1, 0)
#pragma unroll
      for (int kh = 0; kh < 2; ++kh)
#pragma unroll
        for (int m = 0; m < 2; ++m) read_a(a1, cur + UNIT, kh, m);
      // gathered B: the offsets of stage kt + 2, whose ring slot landed a step ago
      if (gathered) form_gathered(min(kt + 2, nk - 1));
      issue_b(kt + 2, 0);
      wait_copies(n4, n1);  // A0, B0 of the next stage
      zero_tail(kt + 1, 0);
      wait_lds_barrier();
      quarter<1, 0>(acc, a1, b0);
      // (1, 1)
      read_first(nxt);  // past the last stage: a harmless read
      issue_b(kt + 2, 1);
      wait_lds_barrier();
      quarter<1, 1>(acc, a1, b1);
    }
    if (!late) barrier();
    asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 3\n" ::: "memory");  // MFMA results -> VALU reads
    // the copies past the end have landed before the workgroup's LDS is given back
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  }

  // ---- epilogue: lane holds C[m0 + 128 (i / 2) + 32 wm + 16 (i % 2) + l % 16]
  //                           [n0 + 128 (j / 4) + 64 wn + 16 (j % 4) + 4 (l / 16) + 0..3]
  const int64_t mn = static_cast<int64_t>(args.m_out) * args.n_out;
  float* part = (chunks > 1) ? args.partial + static_cast<int64_t>(pbase + chunk) * mn : nullptr;
#pragma unroll
  for (int i = 0; i < FM; ++i) {
    const int m = m0 + (i >> 1) * 128 + wm * 32 + (i & 1) * 16 + (lane & 15);
    if (m >= args.m_out) continue;
    const bool lo = m < args.m_split;
    void* base = lo ? args.out_lo[g] : args.out_hi[g];
    const int64_t orow = static_cast<int64_t>(lo ? m : m - args.m_split) * args.n_out;
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      const int n = n0 + (j >> 2) * 128 + wn * 64 + (j & 3) * 16 + (lane >> 4) * 4;
      if (n >= args.n_out) continue;
      const f32x4 v = acc[i][j];
      if (part) {
        *reinterpret_cast<f32x4*>(part + static_cast<int64_t>(m) * args.n_out + n) = v;
      } else if (args.out_dtype == FMOE_BF16) {
        uint2 u;
        u.x = pack2(v[0], v[1]);
        u.y = pack2(v[2], v[3]);
        *reinterpret_cast<uint2*>(static_cast<uint16_t*>(base) + orow + n) = u;
      } else {
        *reinterpret_cast<f32x4*>(static_cast<float*>(base) + orow + n) = v;
      }
    }
  }
}

// Adds the chunk partials of each multi-chunk group in chunk order; 8
// consecutive outputs of one row per thread (m_out and n_out are multiples of
// 64), written with 16-byte stores.  The loads of kWgradReduceBatch chunks are
// issued together (a loop that waited for each chunk's loads before the next
// paid one memory latency per chunk); the sums still run in chunk order,
// from 0.
constexpr int kWgradReduceBatch = 8;

__device__ __forceinline__ void store_grad8(const WgradArgs& a, int g, int64_t i0, const float (&v)[8]) {
  const int m = static_cast<int>(i0 / a.n_out), n = static_cast<int>(i0 - static_cast<int64_t>(m) * a.n_out);
  const bool lo = m < a.m_split;
  const int64_t o = static_cast<int64_t>(lo ? m : m - a.m_split) * a.n_out + n;
  void* base = lo ? a.out_lo[g] : a.out_hi[g];
  if (a.out_dtype == FMOE_BF16) {
    *reinterpret_cast<uint4*>(static_cast<uint16_t*>(base) + o) = pack8(v);
  } else {
    float4* dst = reinterpret_cast<float4*>(static_cast<float*>(base) + o);
    dst[0] = make_float4(v[0], v[1], v[2], v[3]);
    dst[1] = make_float4(v[4], v[5], v[6], v[7]);
  }
}

__global__ __launch_bounds__(256) void wgrad_reduce_kernel(const WgradArgs args) {
  const int g = blockIdx.y;
  int row_base, M;
  group_rows(args, g, row_base, M);
  const int chunks = wgrad_chunks(M, args.kc);
  const int64_t mn = static_cast<int64_t>(args.m_out) * args.n_out;
  const int64_t i0 = (static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x) * 8;
  if (i0 >= mn || chunks <= 1) return;
  float acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  {
    // first partial: the shared group's come first, then the experts'
    int pbase = 0;
    if (g < args.E) {
      const int sc = wgrad_chunks(args.rows_shared, args.kc);
      if (sc > 1) pbase = sc;
      for (int q = 0; q < g; ++q) {
        int rb, Mq;
        group_rows(args, q, rb, Mq);
        const int cq = wgrad_chunks(Mq, args.kc);
        if (cq > 1) pbase += cq;
      }
    }
    const float* src0 = args.partial + static_cast<int64_t>(pbase) * mn + i0;
    for (int c0 = 0; c0 < chunks; c0 += kWgradReduceBatch) {
      float4 u[kWgradReduceBatch][2];
#pragma unroll
      for (int b = 0; b < kWgradReduceBatch; ++b) {
        // chunks past the last re-read the last one and are not added
        const float4* src = reinterpret_cast<const float4*>(src0 + min(c0 + b, chunks - 1) * mn);
        u[b][0] = src[0];
        u[b][1] = src[1];
      }
#pragma unroll
      for (int b = 0; b < kWgradReduceBatch; ++b) {
        if (c0 + b < chunks) {
          acc[0] = acc[0] + u[b][0].x; acc[1] = acc[1] + u[b][0].y;
          acc[2] = acc[2] + u[b][0].z; acc[3] = acc[3] + u[b][0].w;
          acc[4] = acc[4] + u[b][1].x; acc[5] = acc[5] + u[b][1].y;
          acc[6] = acc[6] + u[b][1].z; acc[7] = acc[7] + u[b][1].w;
        }
      }
    }
  }
  store_grad8(args, g, i0, acc);
}

// ---- host side --------------------------------------------------------------
int check_common(int n_experts, int64_t rows_routed, int64_t rows_shared, int64_t dim, int64_t inter) {
  if (n_experts <= 0 || n_experts > FMOE_MAX_EXPERTS) return FMOE_ERR_TOO_MANY_EXPERTS;
  if (rows_routed < 0 || rows_shared < 0 || dim <= 0 || inter <= 0) return FMOE_ERR_INVALID_ARG;
  if (dim % 64 != 0 || inter % 64 != 0) return FMOE_ERR_SHAPE;
  if (rows_routed + rows_shared > INT32_MAX / 2) return FMOE_ERR_SHAPE;
  return FMOE_OK;
}

// The four row products.  Their tile copies address a lane's operand row
// with a 32-bit byte offset from the tile's base: up to 255 rows of at most
// 2 * inter (or dim) elements for the activations, any row of the weight for
// the forward products (n * K + 56 < dim * inter elements).  So a row holds
// fewer than 2^22 elements and a weight matrix fewer than 2^31.
int check_row_product(int n_experts, int64_t rows_routed, int64_t rows_shared, int64_t dim, int64_t inter) {
  const int st = check_common(n_experts, rows_routed, rows_shared, dim, inter);
  if (st) return st;
  constexpr int64_t kMaxRow = int64_t(1) << 22;
  if (dim >= kMaxRow || inter >= kMaxRow || dim * inter >= (int64_t(1) << 31)) return FMOE_ERR_SHAPE;
  return FMOE_OK;
}

// Row counts up to which a launch sends groups of <= kSmallM rows to the
// small-group kernel (decode-sized batches), if they have at most kSmallAvgRows
// routed rows per expert, or no group can exceed 2 kSmallM rows, or an operand
// is not 16-byte aligned (a weight that is a view into a larger buffer); all
// other launches use the tiled kernel for every group.  Both kernels cost their
// share when groups of both kinds occur, and the tiled one is the faster from
// about 8 rows per group: it reads a weight once per 256 rows, the small one
// once per 16 to 128.  Measured (gate/up + down forward, MI355X, small kernel
// for groups of <= 128 rows -> tiled kernel): 64 experts, d = 2048, I = 1408,
// top-6: T = 200 367 -> 285 us, T = 340 452 -> 289, T = 580 592 -> 298 (T = 64, 6
// rows per expert: 271 against 295 us); 8 experts, d = 768, I = 2048, top-2: T =
// 150 82 -> 59, T = 300 104 -> 62; 16 experts, top-4: T = 400 161 -> 72.
constexpr int64_t kSmallLaunchRows = 4096;
constexpr int64_t kSmallAvgRows = 8;

// Compute units of the current device (the persistent grid size), cached per
// device ordinal.
int device_cus() {
  static std::atomic<int> cache[64];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  int v = cache[dev].load(std::memory_order_relaxed);
  if (v > 0) return v;
  if (hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || v <= 0) v = 256;
  cache[dev].store(v, std::memory_order_relaxed);
  return v;
}

// 16-row blocks of the small-group kernel for a launch whose groups have at
// most max_rows rows (1, 2, 4 or 8; the down product stops at 4, so that
// its larger groups run as 64-row slabs: measured faster, as its 8-block
// variant holds fewer waves per SIMD).
template <int MODE>
inline int small_blocks(int64_t max_rows) {
  const int64_t mb = ceil_div(max_rows < kSmallM ? max_rows : kSmallM, 16);
  return mb <= 1 ? 1 : mb <= 2 ? 2 : (mb <= 4 || MODE == DOWN_FWD) ? 4 : 8;
}

// Whether the operands of a launch are 16-byte aligned, as the tiled kernel's
// copies of 16 bytes into LDS expect (the small-group kernel's loads take any
// address that a bf16 may have).
template <int MODE>
bool aligned_operands(const GemmArgs& a, int groups) {
  bool ok = aligned16(a.a_routed) && aligned16(a.a_shared);
  for (int g = 0; g < groups; ++g) ok = ok && aligned16(a.b0[g]) && (MODE != GATEUP_FWD || aligned16(a.b1[g]));
  return ok;
}

template <int MODE>
int launch_rows(GemmArgs& a, int64_t rows_routed, int64_t rows_shared, int E, void* stream) {
  constexpr int TN_COLS = (MODE == GATEUP_FWD) ? core::BN / 2 : core::BN;
  const int64_t tiles_n = ceil_div(a.N, TN_COLS);
  constexpr bool kHasSmall = (MODE == GATEUP_FWD || MODE == DOWN_FWD);
  a.small_max = (kHasSmall && rows_routed + rows_shared <= kSmallLaunchRows &&
                 (rows_routed <= kSmallAvgRows * E || (rows_routed <= 2 * kSmallM && rows_shared <= kSmallM) ||
                  !aligned_operands<MODE>(a, E + (rows_shared > 0 ? 1 : 0))))
                    ? kSmallM
                    : 0;
  // A routed group has at most rows_routed rows: when no group can exceed
  // 2 kSmallM rows (the small kernel takes a larger group as two slabs), the
  // tiled kernel (and its split reduction) would have nothing to do.  This
  // is the case for a decode step of up to 128 tokens at top-2, whose groups
  // the host cannot bound more tightly.
  const bool all_small = a.small_max > 0 && rows_routed <= 2 * kSmallM && rows_shared <= kSmallM;
  if (all_small) a.small_max = 2 * kSmallM;
  // Upper bound of sum over groups of ceil(M_g / BM): floor(rows/BM) + groups.
  const int64_t tiles = (rows_routed / core::BM + E + ceil_div(rows_shared, core::BM)) * tiles_n;
  if (tiles <= 0) return FMOE_OK;
  if (!all_small) {
    // A launch of fewer tiles than CUs still takes every CU if its tiles can be
    // split along K (ranges of kSplitMinSteps steps at least).
    const int64_t cus = device_cus();
    if (a.K / core::BK < 2 * kSplitMinSteps) a.split_ws = nullptr;
    const int64_t grid = (a.split_ws == nullptr && tiles < cus) ? tiles : cus;
    // A run of kSplitMaxRounds full rounds or more never splits (split_plan);
    // sum over groups of ceil(M_g / BM) >= ceil(rows / BM) bounds the tile
    // count from below, so such a run skips the header and the reduction.
    const int64_t tiles_lo = (ceil_div(rows_routed, core::BM) + ceil_div(rows_shared, core::BM)) * tiles_n;
    if (a.small_max == 0 && tiles_lo / grid >= kSplitMaxRounds) a.split_ws = nullptr;
    bool gathered = false;
    if constexpr (MODE == GATEUP_FWD) {
      gathered = a.gather != nullptr;
      if (gathered) rows_gemm_kernel<MODE, true><<<dim3(grid), dim3(core::NT), 0, as_stream(stream)>>>(a, a.offsets);
    }
    if (!gathered) rows_gemm_kernel<MODE, false><<<dim3(grid), dim3(core::NT), 0, as_stream(stream)>>>(a, a.offsets);
    if (a.split_ws != nullptr) {
      // at most half of the CUs' tiles are split (R S <= grid, S >= 2)
      const dim3 rgrid((tiles < cus / 2 ? tiles : cus / 2) * kReduceParts);
      if constexpr (MODE == DOWN_FWD || MODE == GATEUP_BWD)
        split_reduce_kernel<<<rgrid, dim3(256), 0, as_stream(stream)>>>(a.split_ws, static_cast<int>(grid), a.c0,
                                                                       a.ldc0);
      else if constexpr (MODE == GATEUP_FWD)
        split_reduce_gateup_kernel<<<rgrid, dim3(256), 0, as_stream(stream)>>>(a, static_cast<int>(grid));
      else
        split_reduce_down_bwd_kernel<<<rgrid, dim3(256), 0, as_stream(stream)>>>(a, static_cast<int>(grid));
    }
  }
  if constexpr (kHasSmall) {
    if (a.small_max > 0) {
      // DOWN_FWD with fewer routed rows than experts: the grid covers the
      // at most rows_routed routed groups that have rows
      a.small_compact = (MODE == DOWN_FWD && rows_routed < E) ? 1 : 0;
      const int64_t Gr = a.small_compact ? rows_routed : E;
      const int64_t shared_slabs =
          (rows_shared > 0 && rows_shared <= a.small_max) ? ceil_div(rows_shared, kSharedSlab) : 0;
      const int64_t G = Gr + shared_slabs;
      if (G == 0) return launch_status();
      const dim3 grid(G * (a.N / 16)), block(small_waves<MODE>() * 64);
      hipStream_t s = as_stream(stream);
      const int64_t shared_bound = rows_shared < kSharedSlab ? rows_shared : kSharedSlab;
      switch (small_blocks<MODE>(rows_routed > shared_bound ? rows_routed : shared_bound)) {
        case 1: small_gemm_kernel<MODE, 1><<<grid, block, 0, s>>>(a); break;
        case 2: small_gemm_kernel<MODE, 2><<<grid, block, 0, s>>>(a); break;
        case 4: small_gemm_kernel<MODE, 4><<<grid, block, 0, s>>>(a); break;
        default:
          if constexpr (MODE != DOWN_FWD) small_gemm_kernel<MODE, 8><<<grid, block, 0, s>>>(a);
          break;
      }
    }
  }
  return launch_status();
}

void fill_groups(GemmArgs& a, const int32_t* offsets, int E, int64_t rows_routed, int64_t rows_shared) {
  a.offsets = offsets;
  a.E = E;
  a.rows_routed = static_cast<int>(rows_routed);
  a.rows_shared = static_cast<int>(rows_shared);
}

}  // namespace fmoe

using namespace fmoe;

extern "C" size_t fmoe_split_workspace_bytes(void) {
  const size_t P = static_cast<size_t>(device_cus());
  return P * core::BM * core::BN * sizeof(float) + (P + 1) * 16;  // partials + descriptors
}

extern "C" int fmoe_gateup_fwd(const void* x_routed, const int32_t* gather, int gather_k, int64_t gather_tokens,
                               const void* x_shared, const int32_t* offsets,
                               int n_experts, int64_t rows_routed, int64_t rows_shared, int64_t dim,
                               int64_t inter, const void* const* w1, const void* const* w3,
                               void* ab, void* h, void* workspace, size_t workspace_bytes, void* stream) {
  int st = check_row_product(n_experts, rows_routed, rows_shared, dim, inter);
  if (st) return st;
  if (rows_routed + rows_shared == 0) return FMOE_OK;
  if (!offsets || !w1 || !w3 || !ab || !h || (rows_routed && !x_routed) ||
      (rows_shared && !x_shared))
    return FMOE_ERR_INVALID_ARG;
  if (!aligned16(ab) || !aligned16(h)) return FMOE_ERR_ALIGN;
  if (gather) {
    // routed row r reads x_routed ([gather_tokens, dim]) row gather[r] / gather_k;
    // the tiled kernel reads the indices in windows of 8 and forms 32-bit offsets
    if (gather_k <= 0 || gather_k > FMOE_MAX_TOPK || gather_tokens <= 0 || rows_routed < 8 ||
        rows_routed + rows_shared <= kSmallLaunchRows || gather_tokens * dim * 2 >= (int64_t(1) << 31) ||
        rows_routed >= (int64_t(1) << 29))
      return FMOE_ERR_SHAPE;
  }
  GemmArgs a = {};
  a.a_routed = static_cast<const uint16_t*>(x_routed);
  a.gather = gather;
  a.gather_k = gather ? gather_k : 1;
  a.gather_magic = slot_div_magic(a.gather_k);
  a.a_shared = static_cast<const uint16_t*>(x_shared);
  a.lda = dim;
  fill_groups(a, offsets, n_experts, rows_routed, rows_shared);
  a.K = static_cast<int>(dim);
  a.N = static_cast<int>(inter);
  a.inter = static_cast<int>(inter);
  a.ldb = dim;
  a.c0 = static_cast<uint16_t*>(ab);
  a.c1 = static_cast<uint16_t*>(h);
  a.ldc0 = 2 * inter;
  a.ldc1 = inter;
  a.split_ws = (workspace && workspace_bytes >= fmoe_split_workspace_bytes()) ? static_cast<float*>(workspace) : nullptr;
  const int G = n_experts + (rows_shared > 0 ? 1 : 0);
  for (int g = 0; g < G; ++g) {
    if (!w1[g] || !w3[g]) return FMOE_ERR_INVALID_ARG;
    a.b0[g] = static_cast<const uint16_t*>(w1[g]);
    a.b1[g] = static_cast<const uint16_t*>(w3[g]);
  }
  return launch_rows<GATEUP_FWD>(a, rows_routed, rows_shared, n_experts, stream);
}

extern "C" int fmoe_down_fwd(const void* h, const int32_t* offsets, int n_experts,
                             int64_t rows_routed, int64_t rows_shared, int64_t dim, int64_t inter,
                             const void* const* w2, void* out, void* workspace, size_t workspace_bytes,
                             void* stream) {
  int st = check_row_product(n_experts, rows_routed, rows_shared, dim, inter);
  if (st) return st;
  if (rows_routed + rows_shared == 0) return FMOE_OK;
  if (!h || !offsets || !w2 || !out) return FMOE_ERR_INVALID_ARG;
  if (!aligned16(out)) return FMOE_ERR_ALIGN;
  GemmArgs a = {};
  a.a_routed = static_cast<const uint16_t*>(h);
  a.a_shared = nullptr;
  a.lda = inter;
  fill_groups(a, offsets, n_experts, rows_routed, rows_shared);
  a.K = static_cast<int>(inter);
  a.N = static_cast<int>(dim);
  a.inter = static_cast<int>(inter);
  a.ldb = inter;
  a.c0 = static_cast<uint16_t*>(out);
  a.ldc0 = dim;
  a.split_ws = (workspace && workspace_bytes >= fmoe_split_workspace_bytes()) ? static_cast<float*>(workspace) : nullptr;
  const int G = n_experts + (rows_shared > 0 ? 1 : 0);
  for (int g = 0; g < G; ++g) {
    if (!w2[g]) return FMOE_ERR_INVALID_ARG;
    a.b0[g] = static_cast<const uint16_t*>(w2[g]);
  }
  return launch_rows<DOWN_FWD>(a, rows_routed, rows_shared, n_experts, stream);
}

extern "C" int fmoe_down_bwd_dx(const void* d_out_routed, const void* d_out_shared,
                                const int32_t* offsets, int n_experts, int64_t rows_routed,
                                int64_t rows_shared, int64_t dim, int64_t inter, const void* const* w2,
                                const void* ab, void* d_ab, void* workspace, size_t workspace_bytes,
                                void* stream) {
  int st = check_row_product(n_experts, rows_routed, rows_shared, dim, inter);
  if (st) return st;
  if (rows_routed + rows_shared == 0) return FMOE_OK;
  if (!offsets || !w2 || !ab || !d_ab || (rows_routed && !d_out_routed) ||
      (rows_shared && !d_out_shared))
    return FMOE_ERR_INVALID_ARG;
  if (!aligned16(ab) || !aligned16(d_ab)) return FMOE_ERR_ALIGN;
  GemmArgs a = {};
  a.a_routed = static_cast<const uint16_t*>(d_out_routed);
  a.a_shared = static_cast<const uint16_t*>(d_out_shared);
  a.lda = dim;
  fill_groups(a, offsets, n_experts, rows_routed, rows_shared);
  a.K = static_cast<int>(dim);
  a.N = static_cast<int>(inter);
  a.inter = static_cast<int>(inter);
  a.ldb = inter;  // w2[g] is [dim, inter] as nn.Linear keeps it: k row = dim index, inter contiguous
  a.c0 = static_cast<uint16_t*>(d_ab);
  a.ldc0 = 2 * inter;
  a.aux = static_cast<const uint16_t*>(ab);
  a.ldaux = 2 * inter;
  a.split_ws = (workspace && workspace_bytes >= fmoe_split_workspace_bytes()) ? static_cast<float*>(workspace) : nullptr;
  const int G = n_experts + (rows_shared > 0 ? 1 : 0);
  for (int g = 0; g < G; ++g) {
    if (!w2[g]) return FMOE_ERR_INVALID_ARG;
    if (!aligned16(w2[g])) return FMOE_ERR_ALIGN;
    a.b0[g] = static_cast<const uint16_t*>(w2[g]);
  }
  return launch_rows<DOWN_BWD>(a, rows_routed, rows_shared, n_experts, stream);
}

extern "C" int fmoe_gateup_bwd_dx(const void* d_ab, const int32_t* offsets, int n_experts,
                                  int64_t rows_routed, int64_t rows_shared, int64_t dim,
                                  int64_t inter, const void* const* w1, const void* const* w3, void* dx_rows,
                                  void* workspace, size_t workspace_bytes, void* stream) {
  int st = check_row_product(n_experts, rows_routed, rows_shared, dim, inter);
  if (st) return st;
  if (rows_routed + rows_shared == 0) return FMOE_OK;
  if (!d_ab || !offsets || !w1 || !w3 || !dx_rows) return FMOE_ERR_INVALID_ARG;
  if (!aligned16(d_ab) || !aligned16(dx_rows)) return FMOE_ERR_ALIGN;
  GemmArgs a = {};
  a.a_routed = static_cast<const uint16_t*>(d_ab);
  a.a_shared = nullptr;
  a.lda = 2 * inter;
  fill_groups(a, offsets, n_experts, rows_routed, rows_shared);
  a.K = static_cast<int>(2 * inter);
  a.N = static_cast<int>(dim);
  a.inter = static_cast<int>(inter);
  a.ldb = dim;  // w1[g], w3[g] are [inter, dim]: k rows 0..inter-1 from w1, inter.. from w3
  a.c0 = static_cast<uint16_t*>(dx_rows);
  a.ldc0 = dim;
  a.split_ws = (workspace && workspace_bytes >= fmoe_split_workspace_bytes()) ? static_cast<float*>(workspace) : nullptr;
  const int G = n_experts + (rows_shared > 0 ? 1 : 0);
  for (int g = 0; g < G; ++g) {
    if (!w1[g] || !w3[g]) return FMOE_ERR_INVALID_ARG;
    if (!aligned16(w1[g]) || !aligned16(w3[g])) return FMOE_ERR_ALIGN;
    a.b0[g] = static_cast<const uint16_t*>(w1[g]);
    a.b1[g] = static_cast<const uint16_t*>(w3[g]);
  }
  return launch_rows<GATEUP_BWD>(a, rows_routed, rows_shared, n_experts, stream);
}

namespace fmoe {
// Rows per K chunk of the weight gradient (wgrad_chunks rounds a group to the
// nearest count).  A work unit is (group, chunk, output tile); the chunk is
// two thirds of one CU's average share (tiles * rows / 64 K steps over the
// CUs), so that skewed groups do not leave a long tail, and at least 768 rows:
// a split tile costs 256 KB of fp32 partial per chunk, written and read once,
// about six K steps' time.  Measured (dW2 + dW1|dW3, MI355X): T = 1021, d =
// 768, 8 experts 136 -> 81 us, T = 4100 215 -> 185, T = 8192 332 -> 296, C2
// 500 -> 482 us (one third of the share, rounded up: the left figures; the
// whole share 532 us at C2, 172 at T = 4100).
//
// A launch of one group (a dense layer) knows its rows on the host: it takes
// the chunk count n with the least rounds * (K steps + 6) + the reduction's
// n * tiles / 25 + 3 (in K steps' time), so that its n * tiles equal units fill
// whole rounds of the CUs: 48 tiles of 6100 rows in 8 chunks were 384 units,
// two rounds of which the second half empty, in 5 they are 240, one round.
// Forward and backward of the layer, d = 768, I = 2048: T = 6100 311 -> 289 us,
// T = 9001 454 -> 407, T = 16384 594 -> 547; d = 2048, I = 1408: T = 2048 282 ->
// 270, T = 6100 460 -> 417, T = 16384 870 -> 850; up to T = 1500 unchanged.
int64_t wgrad_kc(int64_t rows_routed, int64_t rows_shared, int n_experts, int64_t m_out, int64_t n_out) {
  const int64_t rows = rows_routed + rows_shared;
  const int64_t tiles = ceil_div(m_out, 256) * ceil_div(n_out, 256), cus = device_cus();
  if (n_experts == 1 && rows_shared == 0) {
    const int64_t n_max = (rows + 384) / 768 < 512 ? (rows + 384) / 768 : 512;
    int64_t best_n = 1, best = 0;
    for (int64_t n = 1; n <= n_max; ++n) {
      const int64_t steps = ceil_div(ceil_div(rows, n), 64) + (n > 1 ? 6 : 0);
      const int64_t cost = ceil_div(n * tiles, cus) * steps * 25 + (n > 1 ? n * tiles + 75 : 0);
      if (n == 1 || cost < best) {
        best = cost;
        best_n = n;
      }
    }
    const int64_t kc = ceil_div(rows, best_n);
    return kc < 384 ? 384 : kc;
  }
  const int64_t kc = (2 * tiles * rows / (3 * cus)) / 64 * 64;
  return kc < 768 ? 768 : kc;
}
}  // namespace fmoe

extern "C" size_t fmoe_weight_grad_workspace_bytes(int64_t rows_routed, int64_t rows_shared,
                                                   int n_experts, int64_t m_out, int64_t n_out) {
  if (rows_routed < 0 || rows_shared < 0 || n_experts <= 0 || m_out <= 0 || n_out <= 0) return 0;
  const int64_t kc = wgrad_kc(rows_routed, rows_shared, n_experts, m_out, n_out);
  // sum over groups of wgrad_chunks(M_g, kc) <= floor(rows / kc) + groups
  const int64_t chunks = (rows_routed + rows_shared) / kc + n_experts + 1;
  return static_cast<size_t>(chunks * m_out * n_out) * sizeof(float);
}

extern "C" int fmoe_weight_grad(const void* a_routed, const void* a_shared, int64_t lda,
                                const void* b_routed, const void* b_shared, int64_t ldb,
                                const int32_t* b_gather, int gather_k, int64_t gather_tokens,
                                const int32_t* offsets, int n_experts, int64_t rows_routed,
                                int64_t rows_shared, int64_t m_out, int64_t n_out, int64_t m_split,
                                void* const* out_lo, void* const* out_hi, int out_dtype,
                                void* workspace, size_t workspace_bytes, void* stream) {
  int st = check_common(n_experts, rows_routed, rows_shared, m_out, n_out);
  if (st) return st;
  if (out_dtype != FMOE_BF16 && out_dtype != FMOE_F32) return FMOE_ERR_DTYPE;
  if (m_split <= 0 || m_split > m_out) return FMOE_ERR_SHAPE;
  if (rows_routed + rows_shared == 0) return FMOE_OK;
  if (!offsets || !out_lo || (m_split < m_out && !out_hi) || (rows_routed && (!a_routed || !b_routed)))
    return FMOE_ERR_INVALID_ARG;
  if (lda % 8 != 0 || ldb % 8 != 0) return FMOE_ERR_ALIGN;
  // rows of at least m_out (n_out) elements; the stage copies address up to
  // 63 rows past a stage's first with a 32-bit byte offset
  if (lda < m_out || ldb < n_out || lda >= (int64_t(1) << 24) || ldb >= (int64_t(1) << 24))
    return FMOE_ERR_SHAPE;
  if (workspace_bytes < fmoe_weight_grad_workspace_bytes(rows_routed, rows_shared, n_experts, m_out, n_out))
    return FMOE_ERR_WORKSPACE;
  if (!workspace) return FMOE_ERR_INVALID_ARG;
  WgradArgs a = {};
  a.a_routed = static_cast<const uint16_t*>(a_routed);
  a.a_shared = static_cast<const uint16_t*>(a_shared);
  a.lda = lda;
  a.b_routed = static_cast<const uint16_t*>(b_routed);
  a.b_shared = static_cast<const uint16_t*>(b_shared);
  a.ldb = ldb;
  if (b_gather) {
    // routed row r of B is b_routed ([gather_tokens, n_out]) row b_gather[r] / gather_k
    if (gather_k <= 0 || gather_k > FMOE_MAX_TOPK || gather_tokens <= 0 ||
        gather_tokens * ldb * 2 >= (int64_t(1) << 31) || rows_routed >= (int64_t(1) << 29))
      return FMOE_ERR_SHAPE;
  }
  a.b_gather = b_gather;
  a.gather_k = b_gather ? gather_k : 1;
  a.gather_magic = slot_div_magic(a.gather_k);
  a.offsets = offsets;
  a.E = n_experts;
  a.rows_routed = static_cast<int>(rows_routed);
  a.rows_shared = static_cast<int>(rows_shared);
  a.m_out = static_cast<int>(m_out);
  a.n_out = static_cast<int>(n_out);
  a.m_split = static_cast<int>(m_split);
  a.kc = static_cast<int>(wgrad_kc(rows_routed, rows_shared, n_experts, m_out, n_out));
  a.out_dtype = out_dtype;
  a.partial = static_cast<float*>(workspace);
  const int G = n_experts + (rows_shared > 0 ? 1 : 0);
  for (int g = 0; g < G; ++g) {
    if (!out_lo[g] || (m_split < m_out && !out_hi[g])) return FMOE_ERR_INVALID_ARG;
    if (!aligned16(out_lo[g]) || (m_split < m_out && !aligned16(out_hi[g]))) return FMOE_ERR_ALIGN;
    a.out_lo[g] = out_lo[g];
    a.out_hi[g] = (m_split < m_out) ? out_hi[g] : nullptr;
  }
  const int64_t tiles = ceil_div(m_out, core::BM) * ceil_div(n_out, core::BN);
  // sum over groups of wgrad_chunks(M_g) <= floor(rows / kc) + groups
  const int64_t max_chunks = (rows_routed + rows_shared) / a.kc + G;
  hipStream_t s = as_stream(stream);
  if (b_gather)
    wgrad_tr_kernel<true><<<dim3(max_chunks * tiles), dim3(core::NT), 0, s>>>(a, offsets);
  else
    wgrad_tr_kernel<false><<<dim3(max_chunks * tiles), dim3(core::NT), 0, s>>>(a, offsets);
  // (no group can have two chunks: nothing to reduce)
  if (wgrad_chunks(rows_routed, a.kc) == 1 && wgrad_chunks(rows_shared, a.kc) == 1) return launch_status();
  const int64_t mn = m_out * n_out;
  wgrad_reduce_kernel<<<dim3(ceil_div(mn, 256 * 8), G), dim3(256), 0, s>>>(a);
  return launch_status();
}
