// Dual asymmetric grouped GEMM and the fused dual-expert SwiGLU FFN for gfx950 (bf16 MFMA, fp32 accumulate).
//
// One persistent launch covers the tiles of BOTH experts: the grid is one workgroup per CU, the tile list is
// derived on the device from the per-expert row counts (host values, or the partition's device-side
// expert_offsets), and the tile id -> (expert, tile_m, tile_n) map keeps the 32 tiles that run concurrently on one
// XCD inside a compact patch of the output so they share operand slabs through that XCD's L2.  A skewed pair
// (thousands of VL rows next to tens of action rows, or an empty group) is just a longer or shorter tile list.
//
// Workgroup tile 256 x 256, K step 32, one workgroup per CU: eight wavefronts (two per SIMD) as 2 x 4, wave tile
// 128 x 64 = 8 x 4 MFMA 16x16x32 accumulator blocks (128 accumulator registers per lane), of which one per SIMD
// issues the global -> LDS loads; the projection that rotates heads in its epilogue runs the same tile with the
// wavefronts as 4 x 2 (wave tile 64 x 128: a wavefront holds whole heads).  Problems whose 256 x 256
// tiles would leave most CUs idle (a denoise step of a few thousand action tokens) run the same kernel with a
// 128 x 128 tile, two workgroups per CU.  A ragged last round of the fused FFN launches (tiles left over after the
// whole rounds of one tile per CU) runs in that small shape too, in a second launch, when it then fits the chip in
// one go.  The FFN of few rows (a denoise step of one robot) has tiles of its own, see few_rows_body.
// Operands are K-contiguous, so both MFMA fragments are 16-byte LDS reads.
// Global -> LDS uses buffer loads that write LDS directly (no register staging) into a ring of four K-step slots
// per operand; the load stream runs four K steps ahead of the MFMAs and crosses tile boundaries, with one
// workgroup barrier per K step.  LDS rows are 64 bytes; chunk c of row r sits in slot c ^ ((r >> 2) & 3), which
// makes the 16-byte fragment reads bank-conflict free.
//
// Operand layouts:
//   generic  (wx_dual_gemm)            A, B, C row-major; loads touch 16 rows x 64 bytes per instruction.  An
//                                      operand stored with K as its slow dimension (A as [k, m], B as [k, n]: the
//                                      backward GEMMs) is loaded as K rows of 256 columns and transposed by the LDS
//                                      reads (ds_read_b64_tr_b16), so no layout needs a transposed copy.  An
//                                      addend of C's shape can be summed in the epilogue (wx_dual_gemm_add).
//   gate/up  (wx_dual_swiglu_gate_up)  A = K-tiled activations, B = K-tiled gate and up weights (the B tile is 128
//                                      gate rows + 128 up rows of the same output columns, so gate and up of an
//                                      output element meet in one lane), C = K-tiled intermediate, SwiGLU epilogue.
//   down     (wx_dual_down_proj)       A = K-tiled intermediate, B = K-tiled down weights, C row-major; with a row
//                                      id list the rows go straight to their token positions (the unpermute), and
//                                      a residual matrix can be added there on the way (the layer's closing add).
//   qkv+rope (wx_qkv_rope_proj)        A, B, C row-major like the generic mode, one group; bias and the rotary
//                                      embedding of the q and k heads are applied to the accumulators.
// With K-tiled operands every load instruction moves one contiguous KiB (tiled_layout.h).
// Results leave through a per-wave LDS staging area so that global stores are full 16-byte lanes on contiguous
// runs (whole 1 KiB blocks for the tiled intermediate, 256-byte row segments for row-major outputs).
#include <type_traits>

#include "common.h"
#include "k_major.h"
#include "tiled_layout.h"

namespace wx {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4_word __attribute__((ext_vector_type(4), aligned(4)));  // four words at any word's address

constexpr int BK = 32;
constexpr int kStages = 4;                     // ring slots per operand
constexpr int kRowBytes = BK * 2;              // 64 bytes of K per LDS row

// Workgroup tile shapes.  Everything else (wave tile, loads per step, LDS footprint, resident workgroups per CU)
// follows from the two numbers.
// LW_: how many of the wavefronts (the first LW_) issue the global -> LDS loads; 0 = all of them.
template <int BM_, int BN_, int WM_, int WN_, int LW_ = 0>
struct TileShape {
  static constexpr int BM = BM_, BN = BN_;
  static constexpr int kWavesM = WM_, kWavesN = WN_;  // wavefront grid over the tile
  static constexpr int kWaves = kWavesM * kWavesN;
  static constexpr int kLoadWaves = LW_ > 0 ? LW_ : kWaves;
  static constexpr int kThreads = kWaves * 64;
  static constexpr int FM = BM / kWavesM / 16;        // 16x16 accumulator blocks per wave along M
  static constexpr int FN = BN / kWavesN / 16;        // ... and along N
  static constexpr int kLoadRowsA = BM / kLoadWaves;  // LDS rows of A one loading wave loads per K step
  static constexpr int kLoadRowsB = BN / kLoadWaves;  // ... and of B
  static constexpr int kLoadsA = kLoadRowsA / 16;     // 16-row load instructions per wave per K step: A
  static constexpr int kLoadsB = kLoadRowsB / 16;     // ... and B
  static constexpr int kSlotBytesA = BM * kRowBytes;  // bytes of A per K step
  static constexpr int kSlotBytesB = BN * kRowBytes;
  static constexpr int kStageBytes = FN * 512;        // per-wave staging for the epilogue: 16 rows of the wave tile
  static constexpr int kLdsBytes = kStages * (kSlotBytesA + kSlotBytesB) + kWaves * kStageBytes;
  static constexpr int kWgPerCu = kLdsBytes <= 80 * 1024 && FM * FN * 4 <= 128 ? 2 : 1;
  static_assert(kLdsBytes <= 160 * 1024, "LDS budget");
  static_assert(FM >= 2 && FN >= 4 && FM % 2 == 0 && FN % 4 == 0 && kLoadsA >= 1 && kLoadsB >= 1 && kLoadsB <= kLoadsA, "tile shape");
};
// eight wavefronts (two per SIMD) as 2 x 4: wave tile 128 x 64, 128 accumulator registers per lane, and only the
// first four (one per SIMD) issue the global -> LDS loads.  A wavefront that issues a load stalls while the CU's load
// path takes the instruction in; here its partner on the same SIMD issues no loads and keeps the MFMA pipe fed
// meanwhile.  Against four wavefronts of 128 x 128, on the config 3 shapes: gate/up 4-7 % faster, down 3 %, the
// row-major op 2-6 %.  (With all eight loading on one schedule, both partners stall together: that form was 2 % ahead
// of the four wavefronts on gate/up and behind them elsewhere.)
using BigTile = TileShape<256, 256, 2, 4, 4>;
// The small tile, for problems with too few large tiles to fill the chip: two workgroups per CU, each eight
// wavefronts as 4 x 2 (wave tile 32 x 64), four of them loading, like the large tile.  (Measured with 32x32x16 products:
// four wavefronts of 64 x 64 are 6 % slower on a denoise step; timestamps inside that kernel put 254 ns on a K step whose
// MFMAs need 110, and 169 ns with the loads taken out.)
using SmallTile = TileShape<128, 128, 4, 2, 4>;
// the same eight wavefronts as 4 x 2: wave tile 64 x 128, for the epilogue that needs a wavefront to hold whole
// 128-column heads (the rotation partner of a channel is 64 columns away)
using BigTileQ = TileShape<256, 256, 4, 2, 4>;
// The large tile of a launch.
template <int MODE>
using BigTileFor = std::conditional_t<MODE == 3 || MODE == 4 /* kQkvRope, kQkvRopeFull */, BigTileQ, BigTile>;
// the shape that runs the ragged last round of a launch (see tail_plan): BigTile cut in four.  (Cut in two,
// 256 x 128 with one workgroup per CU, measures the same.)
using TailTile = SmallTile;
// ... and for the projection that rotates heads: four wavefronts as 4 x 1, wave tile 32 x 128, so that a wavefront
// still holds whole heads of 128 channels (all four load)
using TailTileQ = TileShape<128, 128, 4, 1>;
template <int MODE>
using TailTileFor = std::conditional_t<MODE == 3 || MODE == 4 /* kQkvRope, kQkvRopeFull */, TailTileQ, TailTile>;

constexpr int kXcds = 8;
constexpr int kGroupM = 8;                     // tile rows per patch in the tile order

// kQkvRopeFull: kQkvRope reading a rotary table with one entry per channel (an instantiation of its own: both table
// forms in one kernel cost the K loop registers)
enum Mode { kGeneric = 0, kGateUp = 1, kDown = 2, kQkvRope = 3, kQkvRopeFull = 4 };

struct Group {
  const __bf16* a;   // generic: [m, k] row-major (lda).  tiled: base of the K-tiled matrix
  const __bf16* b0;  // generic: [n, k] row-major (ldb).  tiled: K-tiled weights (gate for kGateUp)
  const __bf16* b1;  // kGateUp: K-tiled up weights
  __bf16* c;         // row-major [m, n] (ldc), or base of the K-tiled intermediate (kGateUp)
  int m, n, k;
  int lda, ldb, ldc;  // row-major: leading dimension in elements.  tiled: number of 16-row blocks of the matrix
  int a_row0;         // tiled A: first row of this group inside the tiled matrix (a multiple of 256)
  const __bf16* add;  // generic: optional [m, n] row-major (ldc) matrix added to the product (may be c itself)
};

// The two launches of a problem of more than one round of large tiles (tail_plan).
struct TailPlan {
  int rows[2];  // row blocks of 256 of each expert that are large tiles
  int first;    // large tiles of the first launch
  bool split;   // whether there is a second one
};

struct Params {
  Group g[2];
  const int32_t* offsets;  // device int32[3]: rows of expert e are [offsets[e], offsets[e+1]); null for kGeneric
  // Tile-shape choice made on the device, for launches where the host cannot tell (the split of the rows between
  // the experts lives in `offsets`): both tile shapes are launched and each kernel returns at once unless the
  // number of 256 x 256 tiles is on its side of `gate_tiles`.  0 = always run, 1 = run if at most gate_tiles,
  // 2 = run if more.
  int gate, gate_tiles;
  // Tail split (see tail_plan): 0 = off; 1 = this launch does the whole rounds of 256 x 256 tiles and leaves
  // the ragged last round to a second launch, with 128 x 128 tiles (ROLE 4).
  // split_cus = workgroups of the first launch (one per CU).
  int split, split_cus;
  // kDown only: when set (the partition's sorted_row_id), row r of the sorted result is stored to row scatter[r] of
  // the output instead of row r -- the unpermute folded into the store.
  const int32_t* scatter;
  // kDown with scatter only: when set, a [tokens, n] matrix laid out like the output whose rows are added to the
  // result before the store (out[t] = residual[t] + y[t], each term bf16, one rounding) -- the decoder layer's
  // closing residual add.  May be the output itself.
  const __bf16* residual;
  // kQkvRope only (group 0 is the projection, row-major operands): bias[n] (may be null), the packed rotary table
  // [m, rope_width] (bf16 cos | bf16 sin << 16 per token and channel: rope_width 64 when channels d and d + 64 share
  // an entry, 128 when every channel has its own) and the number of leading output columns that are rotated (whole
  // heads of 128: the q and k heads; the v heads behind them only take the bias).
  const __bf16* bias;
  const uint32_t* rope_table;
  int rope_cols, rope_width;
  // One place for what only one kind of launch has (the one launch of both GEMMs on few rows takes two of these structs: 16 bytes
  // more in each cost a denoise step of 36 layers 10 us of 564).
  union {
    // kGateUp only (training): when set, the two projections themselves (gate and up, rounded to bf16, before the SwiGLU) are
    // stored as well, K-tiled with the geometry of the intermediate, so that a backward pass need not recompute them.
    __bf16* keep[2];
    // kGeneric, kQkvRope, kQkvRopeFull: the plan of the two launches, which the host alone makes there.  (Made again by every
    // workgroup of both launches: 1656 rows of 11008 columns, contractions of 64 to 4096, 0.6 us longer.)
    TailPlan plan;
  };
};

#define LDS_PTR(p) ((__attribute__((address_space(3))) void*)(p))
#define LDS_TR_PTR(p) ((__attribute__((address_space(3))) bf16x4*)(p))

// Buffer descriptor for `bytes` readable bytes at `base`.  Both are wave-uniform by construction; passing them
// through readfirstlane pins the descriptor to scalar registers.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* base, uint32_t bytes) {
  const uint64_t v = reinterpret_cast<uint64_t>(base);
  const uint32_t lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v));
  const uint32_t hi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v >> 32));
  void* p = reinterpret_cast<void*>((static_cast<uint64_t>(hi) << 32) | lo);
  return __builtin_amdgcn_make_buffer_rsrc(p, 0, static_cast<int>(__builtin_amdgcn_readfirstlane(bytes)), 0x00020000);
}

// s_waitcnt immediate for gfx9: vmcnt in bits [3:0] and [15:14], expcnt [6:4] (left at "no wait"), lgkmcnt [11:8]
constexpr int waitcnt_imm(int vm, int lgkm) { return (vm & 15) | ((vm >> 4) << 14) | (7 << 4) | (lgkm << 8); }

struct TileCoord {
  int group, tm, tn;
  int part;  // split contraction: which part of it (PartsRule)
};

// Linear tile id -> coordinates.  Ids are first spread so that each XCD (workgroup id mod 8) walks its own
// contiguous range of "virtual" ids; virtual ids then sweep patches of kGroupM tile rows column by column.
// Integer division runs on the vector ALU even for uniform operands, so the results are handed back through
// readfirstlane to keep everything derived from them (descriptors, branches) scalar.
__device__ __forceinline__ void tile_coords(int v, const int* tiles_m, const int* tiles_n, TileCoord& tc) {
  int g = 0;
  const int c0 = tiles_m[0] * tiles_n[0];
  if (v >= c0) { g = 1; v -= c0; }
  const int tmn = g ? tiles_m[1] : tiles_m[0], tnn = g ? tiles_n[1] : tiles_n[0];
  const int patch = kGroupM * tnn;
  const int first_m = __builtin_amdgcn_readfirstlane(v / patch) * kGroupM;
  const int rows = tmn - first_m < kGroupM ? tmn - first_m : kGroupM;
  const int in_patch = v - (first_m / kGroupM) * patch;
  const int q = __builtin_amdgcn_readfirstlane(in_patch / rows);
  tc.group = g;
  tc.tm = first_m + (in_patch - q * rows);
  tc.tn = q;
}
// The share of `n` tiles that XCD `x` walks when they are dealt out as evenly as possible, the XCDs taking their
// places in the dealing order from `first` on (the first n % 8 places get one tile more): how many, and the index of
// the first one (every XCD's share is a contiguous range).
__device__ __forceinline__ void xcd_share(int n, int x, int first, int& count, int& start) {
  const int q = n / kXcds, r = n % kXcds;
  const int pos = (x - first + kXcds) % kXcds;
  count = q + (pos < r ? 1 : 0);
  start = pos * q + (pos < r ? pos : r);
}
// Workgroup slot t (XCD t % 8, place t / 8 among that XCD's workgroups and rounds) -> tile.  Each expert's tiles
// are dealt to the XCDs separately, expert 1's starting at the XCD where expert 0's remainder ended, so every XCD
// walks its share of expert 0 and then its share of expert 1, at most ceil(total / 8) tiles in all.  With one list
// cut into eight ranges instead, a short second expert would sit at the end of the last XCD's range alone: cheap
// tiles (the action expert's down projection, a tenth of the contraction) then replace expensive ones on one XCD
// only, and the other seven run a longer list.
__device__ __forceinline__ bool map_tile(int t, int total, const int* tiles_m, const int* tiles_n, TileCoord& tc) {
  const int all0 = tiles_m[0] * tiles_n[0];
  const int n0 = all0 < total ? all0 : total, n1 = total - n0;  // (a first launch of a tail split stops at `total`)
  const int x = t % kXcds, j = t / kXcds;
  int count, start;
  xcd_share(n0, x, 0, count, start);
  int v = start + j;
  if (j >= count) {
    const int j1 = j - count;
    xcd_share(n1, x, n0 % kXcds, count, start);
    if (j1 >= count) return false;
    v = n0 + start + j1;
  }
  tile_coords(v, tiles_m, tiles_n, tc);
  return true;
}

// The ragged last round.  `total` 256 x 256 tiles on `cus` workgroups take ceil(total / cus) rounds however few
// tiles the last round holds.  When the tiles left over after the whole rounds (in virtual-id order: the last tile
// rows of expert 0, then expert 1) fit the chip as 128 x 128 tiles in one go -- four per large tile, two workgroups
// per CU -- the first launch stops at the whole rounds and a second launch runs the rest in the small shape.
// Tiles of an expert whose contraction is at most half as long as the other's are cheap enough to ride along
// as a second helping and are not counted.  Returns the number of tiles of the first launch
// (== total: no split).  Evaluated identically by the host (when it knows the row counts) and by both launches.
__host__ __device__ inline int tail_split_point(int tiles0, int tiles1, int k0, int k1, int cus) {
  const int total = tiles0 + tiles1;
  if (cus <= 0 || total <= cus) return total;
  const int full = total / cus * cus, tail = total - full;
  if (tail == 0) return total;
  const int tail1 = tail < tiles1 ? tail : tiles1, tail0 = tail - tail1;
  const int counted = (tiles1 > 0 && tiles0 > 0 && 2ll * k1 <= k0) ? tail0 : tail;
  return 2 * counted <= cus ? full : total;
}

// The two launches of a problem of more than one round of large tiles: the split above, or one that leaves an expert's last
// rows to the second launch where they are 128 at most (`strips`).  As large tiles such a row block is half padding, and its
// tiles take part in the whole rounds like any other: 880 rows of an expert of 11008 are 344 large gate/up tiles, one round
// and 88 left over that take 37 us as small ones, where three whole row blocks and a strip are one round, two large tiles
// and 172 small ones: us a layer 158 -> 146, 2310 to 2400 rows 318 to 323 -> 307 to 311, 1656 rows 240 -> 230.
// The rounds are counted in kTailRound-ths of a round of large tiles: kTailOne for a launch of small tiles with one to a CU,
// kTailTwo with two (contractions of 2048, us: 47 to 56, 20 to 25, 37; row-major 45, 30, 41), none with more (384 rows of 76800
// columns as 776 small tiles behind one round in place of 352 behind two: 147 -> 158).  What a launch costs beside its contraction, 10 us
// with two to a CU against 4 of a round behind another, makes two the dearer below contractions of `length`: row-major, 3704
// rows of 11008 columns, a round and 446 small tiles, us: K 256 31 and 36, 512 46 and 49, 1024 level, 1280 90.8 and 90.3, 2048 129
// and 127; 2150 rows 23.2 and 25.3, 32.2 and 33.7, level, 58.1 and 57.3, 84 and 80; gate/up of the same tiles, us a layer, K 1280
// 105.2 and 106.5, 1536 119.0 and 118.4, 2048 161 and 160.  (One to a CU in place of two pays at any: 880 rows of 22016 columns,
// K 256, 24.0 -> 23.0.)
constexpr int kTailRound = 10, kTailOne = 4, kTailTwo = 8, kTailNever = 1 << 28;
constexpr int kTailLongRows = 1280, kTailLongTiled = 1536;  // `length` of the row-major and the K-tiled operands
__host__ __device__ inline TailPlan tail_plan(int m0, int m1, int cols0, int cols1, int k0, int k1, int cus, bool strips, int length) {
  TailPlan p;
  p.rows[0] = (m0 + 255) >> 8;
  p.rows[1] = (m1 + 255) >> 8;
  const int tiles0 = p.rows[0] * cols0, tiles1 = p.rows[1] * cols1, total = tiles0 + tiles1;
  p.first = tail_split_point(tiles0, tiles1, k0, k1, cus);
  p.split = p.first != total;
  // (experts whose tiles differ in length: the rule above, which does not count the short ones)
  if (!strips || cus <= 0 || total <= cus || (tiles0 > 0 && tiles1 > 0 && (2ll * k1 <= k0 || 2ll * k0 <= k1))) return p;
  const int strip0 = ((m0 - 1) & 255) < 128 && tiles0 > 0 ? 1 : 0, strip1 = ((m1 - 1) & 255) < 128 && tiles1 > 0 ? 1 : 0;
  const int pieces = 2 * (strip0 * cols0 + strip1 * cols1);
  if (pieces == 0) return p;
  const int large = total - pieces / 2, full = large / cus, left = large - full * cus, whole = total / cus;
  const int two = (tiles0 == 0 ? k1 : (tiles1 == 0 || k0 < k1 ? k0 : k1)) >= length ? kTailTwo : kTailRound + 2;
  auto small = [&](int n) { return n <= 0 ? 0 : (n <= cus ? kTailOne : (n <= 2 * cus ? two : kTailNever)); };
  const int as_is = whole * kTailRound + (p.split ? small(4 * (total - p.first)) : (total > whole * cus ? kTailRound : 0));
  const int both = full > 0 ? full * kTailRound + small(4 * left + pieces) : as_is;  // strips and what the whole rounds leave
  const int alone = (full + (left > 0 ? 1 : 0)) * kTailRound + small(pieces);       // strips alone
  if (both >= as_is && alone >= as_is) return p;
  p.rows[0] -= strip0;
  p.rows[1] -= strip1;
  p.first = both <= alone ? full * cus : large;
  p.split = true;
  return p;
}

// The tile count that decides between the two tile shapes.  The small shape pays when the large tiles would leave
// half of the CUs idle.  Tiles of an expert whose contraction is at most half as long as the other's do not count:
// in the small shape they ride along as a cheap second helping of the first workgroups (4096 VL rows next to a
// handful of action rows in the down launch: 128 tiles of K = 11008 and 8 of K = 1024 are one round of small tiles
// plus a tenth, not 136 large tiles on 256 CUs).  Evaluated identically by the host and by both launches.
__host__ __device__ inline long long shape_deciding_tiles(long long tiles0, long long tiles1, int k0, int k1) {
  if (tiles0 > 0 && tiles1 > 0) {
    if (2ll * k1 <= k0) return tiles0;
    if (2ll * k0 <= k1) return tiles1;
  }
  return tiles0 + tiles1;
}

// The down launch's contraction in parts.  A 128 x 128 tile's K step takes 250 ns however many CUs work and however deep the
// ring is, so 513 .. 1024 rows of an expert of 11008 -- 80 .. 128 tiles of 344 steps -- took 87 us with half of the CUs or more
// idle.  The tiles of the expert that decides the launch's length (both experts', unless one's contraction is at most half as
// long as the other's) are cut into two or four parts (1 << lg) along K while all parts have a CU of their own and 2048 of K;
// the part that finishes last adds them up: at hidden 2048 (two parts) 513 .. 880 rows 87 -> 52 .. 55 us, 1024 rows 87 -> 56,
// 100 rows of the expert of 11008 beside 900 of one of 1024 (four) 92 -> 35.  From half as many tiles as CUs on, two parts on
// every CU take what one did (1760 rows: 90 us; parts of 250 tiles would be at 470 ns a step, two workgroups to a CU).
// Where 256 x 256 tiles would be a quarter to half as many as CUs, two parts of 4096 and more of them beat one part of four
// times as many small tiles, two workgroups to a CU: 2640 + 96 rows 140 -> 115 us, 3520 + 128 159 -> 132, an expert of 8192 and
// 2410 rows 94 -> 88 (of 4096 they do not: 2200 rows 50 -> 55, 565 + 1353 of two 34 -> 58).  The other expert's tiles count there: a
// workgroup that takes one as a second helping costs what the parts gained (4050 + 65 rows, 128 tiles and 8, alone 162 -> 160,
// in four layers of a prefill 17 us a layer slower).
// Asked with the same numbers on the host and on the device, so that the sums' order does not depend on which of them knows the
// row counts, of sizes that may_split lets through (more rows than the one launch for both GEMMs takes without knowing the
// counts, and no more than fill half of the CUs with large tiles: where a host that does not know the counts would make these
// launches for parts that hardly ever are, 4115 rows, of 5 x 823, 4 us a layer); not where the one launch takes the rows
// with their counts known.  Every workgroup of a launch on unknown counts asks first, so what depends on the sizes alone is
// worked out on the host, and the rest is 32-bit.
struct DownParts {
  int lg;      // 1 << lg parts
  bool large;  // of 256 x 256 tiles
  bool cut[2]; // expert e's tiles are cut
};
struct PartsRule {
  int cus, cols;      // CUs; column tiles of 128
  int steps[2];       // column tiles of the gate/up launch, expert e
  int beside[2];      // expert e is cut beside rows of the other one
  int lg_most[2];     // parts that expert e's contraction has room for
  __host__ __device__ inline DownParts parts(int m0, int m1) const {
    DownParts d{};
    const int rb0 = (m0 + 127) >> 7, rb1 = (m1 + 127) >> 7;
    if (rb0 * steps[0] + rb1 * steps[1] <= cus && (rb0 + rb1) * cols <= cus) return d;
    d.cut[0] = rb0 > 0 && (rb1 == 0 || beside[0] != 0);
    d.cut[1] = rb1 > 0 && (rb0 == 0 || beside[1] != 0);
    const int most0 = d.cut[0] ? lg_most[0] : 2, most1 = d.cut[1] ? lg_most[1] : 2, most = most0 < most1 ? most0 : most1;
    const int count = ((d.cut[0] ? rb0 : 0) + (d.cut[1] ? rb1 : 0)) * cols;
    d.lg = count * 4 <= cus ? 2 : (count * 2 <= cus ? 1 : 0);
    if (d.lg > most) d.lg = most;
    const int large_cols = (cols + 1) >> 1, large0 = ((rb0 + 1) >> 1) * large_cols, large1 = ((rb1 + 1) >> 1) * large_cols;
    const int large = (d.cut[0] ? large0 : 0) + (d.cut[1] ? large1 : 0);
    d.large = d.lg == 0 && most > 1 && 4 * large > cus && large0 + large1 + large <= cus;
    if (d.large) d.lg = 1;
    return d;
  }
};

// fp32 sums of the parts, a tile's size each, at most as many as CUs, and a counter per slot, all zero
struct DownSplit {
  float* sums;
  int* count;
  PartsRule rule;
};

// Memory that no launch writes while it reads it: scalar loads, wherever they stand.
using ScalarInts = const __attribute__((address_space(4))) int32_t*;

// Workgroup barrier without the fences of __syncthreads().  Those fences make the compiler wait for EVERY
// outstanding LDS-direct load (vmcnt(0)) at the barrier, which drains the prefetch ring on each K step; the waits
// the data flow needs (own LDS reads returned, own loads of the next slot landed) are written out before each call.
// The empty asm statements keep the compiler from moving memory accesses across the barrier.
__device__ __forceinline__ void barrier_no_fence() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// ... and behind this wavefront's own LDS writes.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(waitcnt_imm(63, 0));
  barrier_no_fence();
}

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t pack_bf16x2(float lo, float hi) {
  const bf16x2 v = {static_cast<__bf16>(lo), static_cast<__bf16>(hi)};  // one packed convert
  return __builtin_bit_cast(uint32_t, v);
}

// One LDS array per (size, alignment, index).
template <int BYTES, int ALIGN, int ID>
__device__ __forceinline__ unsigned char* lds_array() {
  __shared__ __attribute__((aligned(ALIGN))) unsigned char s[BYTES];
  return s;
}

// The fused FFN launch: gate/up tiles (producers) and down tiles (consumers) in one grid.  A down tile of row block
// rb reads the intermediate rows that the gate/up tiles of the same row block write, so it waits until `ready[rb]`
// has reached the number of those tiles.  An XCD places its share of a launch's workgroups in index order and the
// producers come first, so on every XCD the producers have their places before a consumer gets one, and producers
// never wait: a launch alone on the chip always makes progress.  So do two of them in flight together on their own
// workspaces.  Where a launch's producers still wait for a place on an XCD, it has no consumer there, and the other launch's
// consumers leave one:
//   two workgroups per CU (128 x 128 tiles, the few-rows form's smaller ones): an XCD has 64 places, a launch at most 32
//     consumers for it (one per CU in all);
//   one workgroup per CU (the few-rows form's larger tiles, at hidden 2048 129 .. 256 rows): 32 places, at most 31 consumers (the limit of
//     kXcds less than a workgroup per CU in launch_ffn_fused), so a whole CU is left, for a workgroup of either kind;
//   one launch of each kind: consumers of the first kind, one on each of 32 CUs, can keep workgroups of the second out, but
//     their own producers find the CU that the second kind leaves, so they end, and the second launch goes on.
// Three or more launches have no such guarantee (two others' consumers can take every place of an XCD), and the kind of one
// per CU has the smaller margin: at 217 rows a launch has 28 consumers to an XCD.  The wait is bounded for them
// (kFusedWaitTicks of the 100 MHz clock; then `*error` is set and the tile goes ahead on whatever is there).  The last consumer
// past the wait of a row block clears the row block's counters, so a launch leaves the workspace as it found it: all zero.
// The producers can read their A operand from the token rows themselves (AROWS below: `x` through `gather`), which
// makes the permute into the K-tiled activation matrix part of the launch.
constexpr int kFusedMaxRowBlocks = 256;   // 128-row blocks per expert
constexpr long long kFusedWaitTicks = 500000000ll;  // 5 s
constexpr int kFusedCounterStride = 64;   // ints between two counters: 256 bytes, so that the polls of different row
                                          // blocks (and the increments) spread over the memory channels
constexpr int kFusedCounters = 2 * kFusedMaxRowBlocks * kFusedCounterStride;  // ints of one counter array
struct FusedSync {
  int* ready;     // [2 * kFusedMaxRowBlocks] x stride: gate/up tiles finished, by expert and row block
  int* passed;    // ... down tiles past their wait
  int* error;     // set to 1 when a wait ran into its bound
  int need[2];    // gate/up tiles per row block of expert e
  const __bf16* warm_b[2][2];  // the producers' weights (gate, up of expert e), K-tiled; null: nothing to warm
  int warm_ldb[2];             // their row blocks per column block
  int warm_k;                  // their contraction length
  int consumers;  // down tiles per row block
  // AROWS: the activations in token order, [tokens, hidden] bf16 row-major, and the partition's sorted_row_id
  // (sorted position -> token)
  const __bf16* x;
  const int32_t* gather;
  int guess[2];  // few-rows form: the rows per expert that the host sized the grid for
  // few-rows form with the norm folded in: the token rows pass through an RMSNorm on their way to the MFMAs
  const __bf16* norm_weight;
  float norm_eps;
};

// Fused launch: what this workgroup wrote for row block `rb` is in memory (its stores are write-through and every
// wavefront has waited for its own before the barrier); one lane counts it.
__device__ __forceinline__ void count_done(const FusedSync& fs, int tid, int rb) {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __builtin_amdgcn_s_waitcnt(waitcnt_imm(0, 0));
  __syncthreads();
  if (tid == 0)
    __hip_atomic_fetch_add(fs.ready + rb * kFusedCounterStride, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Fused launch: wait (bounded) until ready[rb] has reached `need`, and take a number among the workgroups that
// get past this wait (`before`: how many were past it already; the answer travels while the tile is computed).
// No cache is invalidated afterwards: the launch began with clean caches, and no line of what the wait is for is
// read anywhere before it is complete (whole cache lines belong to one writer), so no cache can hold an older
// version of it.
__device__ __forceinline__ void wait_for_count(const FusedSync& fs, int tid, int rb, int need, int& before) {
  if (tid == 0) {
    const int* flag = fs.ready + rb * kFusedCounterStride;
    const long long start = __builtin_amdgcn_s_memrealtime();
    while (__hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < need) {
      if (static_cast<long long>(__builtin_amdgcn_s_memrealtime()) - start > kFusedWaitTicks) {
        __hip_atomic_store(fs.error, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        break;
      }
      __builtin_amdgcn_s_sleep(2);
    }
    before = __hip_atomic_fetch_add(fs.passed + rb * kFusedCounterStride, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  barrier_no_fence();  // (no wait for the counter's answer here)
}
// The same two for the few-rows form, whose launch is a chain of latencies.  A row block has up to 64 gate/up tiles and as
// many down tiles here, and one counter for all of them was worth a queue: 64 increments and 64 pollers of one word took
// 4.2 us from the last increment to the end of the wait (32 rows, hidden 2048, expert 1024), the words of a counter's 256
// bytes, one per gate/up tile and stored, not added to, take 2.4.  A poll is one load of all 64 words by a wavefront.
// (More than 64 tiles of a row block share the words, tile ct the word ct % 64, and add.)
__device__ __forceinline__ void flag_done(const FusedSync& fs, int tid, int rb, int ct, int tiles) {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __builtin_amdgcn_s_waitcnt(waitcnt_imm(0, 0));
  __syncthreads();
  if (tid == 0) {
    int* const word = fs.ready + rb * kFusedCounterStride + ct % kFusedCounterStride;
    if (tiles <= kFusedCounterStride) __hip_atomic_store(word, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else __hip_atomic_fetch_add(word, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}
// A first look at the words, ahead of the tile's other loads; `seen` of wait_for_flags.
__device__ __forceinline__ int poll_flags(const FusedSync& fs, int tid, int rb) {
  return tid < 64 ? __hip_atomic_load(fs.ready + rb * kFusedCounterStride + tid, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0;
}
__device__ __forceinline__ void wait_for_flags(const FusedSync& fs, int tid, int rb, int tiles, int seen, int& before) {
  if (tid < 64) {
    const int need = (tiles - tid + kFusedCounterStride - 1) / kFusedCounterStride;
    if (__ballot(seen < need) != 0) {
      const long long start = __builtin_amdgcn_s_memrealtime();
      do {
        if (static_cast<long long>(__builtin_amdgcn_s_memrealtime()) - start > kFusedWaitTicks) {
          if (tid == 0) __hip_atomic_store(fs.error, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          break;
        }
        __builtin_amdgcn_s_sleep(1);
        seen = poll_flags(fs, tid, rb);
      } while (__ballot(seen < need) != 0);
    }
    if (tid == 0)
      before = __hip_atomic_fetch_add(fs.passed + rb * kFusedCounterStride, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  barrier_no_fence();
}
__device__ __forceinline__ void clear_flags_if_last(const FusedSync& fs, int tid, int rb, int before, int waiters) {
  if (tid >= 64) return;
  if (__builtin_amdgcn_readfirstlane(before) != waiters - 1) return;
  __hip_atomic_store(fs.ready + rb * kFusedCounterStride + tid, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (tid == 0) __hip_atomic_store(fs.passed + rb * kFusedCounterStride, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// ... and once the tile is done: the workgroup that was the last of its row block to get past the wait (everything
// the wait was for is done, and every other waiter is past its wait as well) leaves the two counters at zero for
// the next launch
__device__ __forceinline__ void clear_if_last(const FusedSync& fs, int tid, int rb, int before, int waiters) {
  if (tid == 0 && before == waiters - 1) {
    __hip_atomic_store(fs.ready + rb * kFusedCounterStride, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(fs.passed + rb * kFusedCounterStride, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

// SwiGLU of a gate and an up accumulator like eager bf16 code (act.py:80-82): gate, up and silu(gate) are each rounded
// to bf16 here, the product by the caller's pack.
__device__ __forceinline__ float swiglu_bf16(float gate, float up) {
  const uint32_t gu = pack_bf16x2(gate, up);  // one convert for both
  const float g = __uint_as_float(gu << 16);
  return round_bf16(g * __builtin_amdgcn_rcpf(1.0f + __expf(-g))) * __uint_as_float(gu & 0xffff0000u);
}

// ---- few rows ------------------------------------------------------------------------------------------------
// A denoise step of one robot is 32 rows.  As 128 x 128 tiles its two GEMMs occupy 16 CUs each, and every K step of those
// waits for the one before it (~250 ns, 96 of them).  This form makes the tiles small and cuts the contraction instead:
// a workgroup computes 16 FM rows x 16 NB operand rows of B (half gate and half up, or output columns), its eight wavefronts
// take an eighth of the K steps each, and the partial sums meet in LDS.  Fragments go from memory to registers (a block
// of a K-tiled matrix is one fragment of a 16x16x32 MFMA), a wavefront's whole share of a contraction of 2048 at once, so a
// tile costs a few memory latencies in place of K / 32 barriers.  Each row block reads the weights again (through L2: the
// tiles of a column are on one XCD where the column tiles are a multiple of eight), which is why many rows keep the large
// tiles.
// A layer's launch is a chain of latencies (timestamps at 32 rows with the norm, weights from HBM, us after the first workgroup's
// entry): arguments 0.6, row ids and first weights requested 1.6, rows requested 3.4, squares of the rows 6.0, products 7.1,
// sums 8.0, stored 8.4, in memory 8.8, flags seen 12, intermediate multiplied 12.6, stored 13.  36 layers with distinct weights
// from a graph, us per layer, as two kernels' worth of 128 registers with the norm's pass over the rows in front of the
// products, a counter per row block and tiles of 16 or 32 rows x 64 / as it is: with the norm inside 32 rows 20.9 / 15.4, 64 rows
// 21.0 / 16.5, 128 rows 22.5 / 19.4, 217 rows (the norm was a launch) 29.8 / 23.2; without a norm 18.8 / 13.6, 18.6 / 14.5,
// 20.5 / 16.8, 24.2 / 18.8.
constexpr int kFewThreads = 512;   // eight wavefronts

// Whether the few-rows form takes the problem: at most a row per CU, where with every row on the narrower expert the tiles of 32
// rows x 64 rows of B of each GEMM are at most one per CU; and up to kFewMaxRows where they are for any split of the rows.  The
// split itself does not enter, so the host always knows, and every launch form adds up in the same order.  At hidden 2048, experts
// 11008 / 1024, the line is 256 rows: 36 layers with the norm 910 us at 256 rows, as two rounds of tiles 1520 at 512 where the
// 128 x 128 tiles take 1460.
// Rows on the wide expert are many tiles per workgroup.  Layers with weights of their own (700 MB in turn), us a layer, 128 x 128
// tiles / this form: 32 rows, all on the expert of 11008, 118 / 91, 64 of 128 120 / 100, 192 134 / 122, 256 134 / 136, 248 of 256
// 135 / 137; none on it 28 / 22 at 256 rows.  Beyond a row per CU, at narrower sizes, they cost more than the form gains: hidden
// 512, experts 2048 / 256, 504 of 512 rows on the wide one 24 / 47, none 13 / 9; hidden 256, 11008 / 64, 384 of 768 53 / 231.
// Where both experts are narrow there is no such split: hidden 256, experts 64 / 32, 257 .. 992 rows 10.9 .. 11.5 / 7.9 .. 8.5
// however they are split, 256 / 256 up to 512 rows 12 / 8.7; hidden 512, 256 / 256 14 / 9.5 at 384 rows, at 992 of which half are
// on either 15.0 / 16.5, the one place where it is behind without a norm (with it from 768 rows of 256 / 256 on, 15.3 / 16.5).
constexpr int kFewMaxRows = 1024;
inline bool few_rows(int64_t rows, int64_t inter0, int64_t inter1, int64_t hidden, int cus) {
  auto one_per_cu = [&](int64_t blocks, int64_t inter) { return blocks * (inter / 32) <= cus && blocks * ((hidden + 63) / 64) <= cus; };
  const int64_t blocks = (rows + 31) / 32, wide = inter0 > inter1 ? inter0 : inter1, narrow = inter0 + inter1 - wide;
  return rows <= cus ? one_per_cu(blocks, narrow) : rows <= kFewMaxRows && one_per_cu(blocks + 1, wide);  // (+ 1: rows on both)
}

// One row's bf16 pair through the RMSNorm: w * bf16(x * inv), rounded, as the norm's own kernel has it (w_lo, w_hi: the pair of
// weights).  A tile of 32 rows x 2048 spends 3 us of its CU's vector ALU on this and on the squares, so both roundings are one
// packed convert each and the squares are fused multiply-adds (the square of a bf16 value is exact in fp32: the same sum).
__device__ __forceinline__ uint32_t rms_scale(uint32_t x, float w_lo, float w_hi, float inv) {
  const uint32_t n = pack_bf16x2(__uint_as_float(x << 16) * inv, __uint_as_float(x & 0xffff0000u) * inv);
  return pack_bf16x2(w_lo * __uint_as_float(n << 16), w_hi * __uint_as_float(n & 0xffff0000u));
}

// MODE, ROLE, AROWS as in dual_gemm_body.  512 threads.
// FM: row blocks of 16 per tile.  NB: blocks of 16 rows of B per tile (half gate, half up; or output columns).  R: K steps in
// flight per wavefront, of which RL hold their B in LDS (the registers of a tile of 32 x 64 do not hold eight steps).
// None of the four decides what is added to what, so every shape gives the same bits: wavefront w takes every other K step of
// a quarter of the contraction (w / 2 the quarter, w % 2 the step's parity), in order, and the eight partial sums are added in
// the order of the wavefronts.
// NORM (with AROWS; k a multiple of 256, at most 32 * 8 R): the rows are normalised here.  A wavefront holds its share of the
// rows, so it reads them once, for the squares and for the products.  The quarters and parities are those of the lanes of
// rmsnorm_permute_tiled128_kernel, and the squares are added in its order: the same values.
// NBP (ROLE 2): NB of the producers.
// ROUNDS: there may be more tiles than workgroups by much.  (The search for their places, if it is not needed, costs the kernels
// with the largest tiles the registers of 20 scalars: 225 .. 256 rows at hidden 2048 21.8 us a layer, with the norm 25.3; with the
// search in the down part 22.4 and 26.1.)
template <int MODE, int FM, int NB, int R, int RV, int RL, int ROLE, bool AROWS, bool NORM = false, int NBP = NB, bool ROUNDS = true>
__device__ __forceinline__ void few_rows_body(const Params& p, const int wg, const int n_wg, const FusedSync& fs) {
#if defined(__HIP_DEVICE_COMPILE__)
  static_assert(MODE == kGateUp || MODE == kDown, "the FFN's two GEMMs");
  static_assert(!NORM || AROWS, "the norm reads token rows");
  constexpr bool SWIGLU = MODE == kGateUp;
  constexpr int kRows = 16 * FM;
  static_assert(RV + RL == R || (RL == 0 && R % RV == 0), "steps of B in flight");
  // where the finished blocks go: block q of the tile (row block q / NB, column block q % NB) is summed by wavefront q % 8
  constexpr int kSums = SWIGLU ? 1 : (FM * NB + 7) / 8;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, lq = lane >> 4;
  // one KiB per 16 x 16 block of partial sums (or per fragment of B) and wavefront: eight blocks in the first array, eight more
  // in the second
  constexpr int kBlocksLds = FM * NB > RL * NB ? FM * NB : RL * NB;
  static_assert(kBlocksLds <= 16, "LDS of a wavefront");
  constexpr bool kMore = kBlocksLds > 8;
  unsigned char* const part = lds_array<65536, 1024, 0>();
  unsigned char* const more = lds_array<kMore ? 65536 : 16, 1024, 1>();
  unsigned char* const norm_lds = lds_array<NORM ? 4096 : 16, 16, 2>();              // the norm's weights
  float* const ss_of = reinterpret_cast<float*>(lds_array<NORM ? kRows * 32 : 16, 16, 3>());  // [row][wavefront]
  auto own_block = [&](int q) { return (q < 8 ? part + q * 1024 : more + (q - 8) * 1024) + wave * 8192; };

  constexpr int kTileN = SWIGLU ? 8 * NB : 16 * NB;  // output columns per tile
  const int cols[2] = {(p.g[0].n + kTileN - 1) / kTileN, (p.g[1].n + kTileN - 1) / kTileN};
  const int frag = (l16 << 6) + ((lq ^ ((l16 >> 2) & 3)) << 4);  // this lane's 16 bytes of a K-tiled block

  // The row counts, and this workgroup's tiles: t, t + step, .. below end, in the order expert, row block, column tile, and then
  // (if behind is not negative) behind, behind + n_wg, .. of the other expert.  At most one tile each where there are workgroups
  // enough; else a workgroup stays with a row block, whose rows it then reads (and normalises) once, and the row blocks'
  // workgroups of one column are on one XCD, which takes them in eights: where that leaves many without a row block (nine blocks
  // of 256 workgroups: 24 each, 15 tiles of 344; 248 rows of the expert of 11008 and 8 of the other 159 us a layer), the expert
  // with less to do comes behind the other, a tile or a few for every workgroup (eight blocks of 32: 11 tiles and one; 137 us).
  int m[2], blocks[2], total0, t, step, end, behind;
  auto go_behind = [&](int& next) {
    if (!ROUNDS || behind < 0) return;
    next = behind;
    step = n_wg;
    end = behind < total0 ? total0 : total0 + blocks[1] * cols[1];
    behind = -1;
  };
  auto place = [&](int m0, int m1) {
    m[0] = m0;
    m[1] = m1;
    blocks[0] = (m0 + kRows - 1) / kRows;
    blocks[1] = (m1 + kRows - 1) / kRows;
    total0 = blocks[0] * cols[0];
    t = wg;
    step = n_wg;
    end = total0 + blocks[1] * cols[1];
    behind = -1;
    if (ROUNDS && __builtin_expect(end > n_wg, 0)) {
      const int total1 = end - total0;
      auto slots_of = [&](int e, int i) { return ((e ? cols[1] : cols[0]) + 8 * i - 1) / (8 * i) * 8; };
      // tiles per workgroup: with both experts' row blocks side by side, and with those of `big` alone
      const int big = static_cast<int64_t>(total1) * p.g[1].k > static_cast<int64_t>(total0) * p.g[0].k ? 1 : 0;
      // (fewer do not fit; and none do where there are more row blocks than eights of workgroups: finding that out by trying, 64
      // turns of divisions ahead of every workgroup's first load, was 11 us of a launch of 22)
      int both = (blocks[0] + blocks[1]) * 8 <= n_wg ? (end + n_wg - 1) / n_wg : 64, alone = 0;
      while (both < 64 && blocks[0] * slots_of(0, both) + blocks[1] * slots_of(1, both) > n_wg) ++both;
      if (total0 > 0 && total1 > 0) {
        const int k_big = big ? p.g[1].k : p.g[0].k, k_less = big ? p.g[0].k : p.g[1].k;
        const int b = big ? blocks[1] : blocks[0], less = ((big ? total0 : total1) + n_wg - 1) / n_wg;
        alone = b * 8 <= n_wg ? ((big ? total1 : total0) + n_wg - 1) / n_wg : 64;
        while (alone < 64 && b * slots_of(big, alone) > n_wg) ++alone;
        const int64_t most = k_big > k_less ? k_big : k_less;
        if (alone >= 64 || (both < 64 && static_cast<int64_t>(alone) * k_big + static_cast<int64_t>(less) * k_less >= both * most)) alone = 0;
      }
      if (alone > 0 || both < 64) {
        const int per = alone > 0 ? alone : both;
        const int slots0 = slots_of(0, per), slots1 = slots_of(1, per);
        const int used0 = alone > 0 && big ? 0 : blocks[0] * slots0, used1 = alone > 0 && !big ? 0 : blocks[1] * slots1;
        const int e = wg >= used0 ? 1 : 0, nct = e ? cols[1] : cols[0];
        const int w = e ? wg - used0 : wg;
        step = e ? slots1 : slots0;
        const int rb = __builtin_amdgcn_readfirstlane(w / step);
        const int first = (e ? total0 : 0) + rb * nct;
        t = first + w - rb * step;
        end = rb * step < (e ? used1 : used0) ? first + nct : 0;
        if (alone > 0) {  // (workgroups without a row block first)
          const int at = wg - (used0 + used1) < 0 ? wg - (used0 + used1) + n_wg : wg - (used0 + used1);
          if (at < (big ? total0 : total1)) behind = (big ? 0 : total0) + at;
          if (t >= end) go_behind(t);
        }
      }
    }
  };
  struct Tile {
    int e, rb, ct;
  };
  auto tile_of = [&](int at) {
    Tile x;
    x.e = at >= total0 ? 1 : 0;
    const int te = x.e ? at - total0 : at, nct = x.e ? cols[1] : cols[0];
    x.rb = __builtin_amdgcn_readfirstlane(te / nct);
    x.ct = te - x.rb * nct;
    return x;
  };
  // Where a tile's B comes from.  A K step's descriptor begins at that step (scalar work) and ends with it, so the lanes'
  // offsets are the same in every step; steps past a wavefront's share have an empty descriptor and read as zeros.  A wavefront's
  // steps are k_first + 2 i, i < share.
  struct Stream {
    const char *b0, *b1;
    uint32_t step, off;
    int steps, share, k_first;
  };
  auto stream_of = [&](const Tile& x) {
    const Group& G = x.e ? p.g[1] : p.g[0];
    Stream b;
    b.b0 = reinterpret_cast<const char*>(G.b0);
    b.b1 = reinterpret_cast<const char*>(SWIGLU ? G.b1 : G.b0);
    b.step = static_cast<uint32_t>(G.ldb) << 10;  // (blocks past the matrix's last row of B are past it)
    b.off = (static_cast<uint32_t>(x.ct * kTileN / kBlkRows) << 10) + frag;
    b.steps = G.k / 32;
    b.share = (b.steps + 7) / 8;
    b.k_first = 2 * b.share * (wave >> 1) + (wave & 1);
    return b;
  };
  u32x4 fa[R][FM], fb[RV][NB];
  auto b_rsrc = [&](const Stream& b, int i, bool up) {
    const int ks = b.k_first + 2 * i;
    return make_rsrc((up ? b.b1 : b.b0) + static_cast<int64_t>(ks) * b.step, i < b.share && ks < b.steps ? b.step : 0u);
  };
  auto b_block = [&](const Stream& b, int j) { return b.off + (SWIGLU ? j % (NB / 2) : j) * kBlkBytes; };
  auto load_b = [&](const Stream& b, int slot, int i) {
    const __amdgpu_buffer_rsrc_t r0 = b_rsrc(b, i, false), r1 = SWIGLU ? b_rsrc(b, i, true) : r0;
#pragma unroll
    for (int j = 0; j < NB; ++j) fb[slot][j] = __builtin_amdgcn_raw_buffer_load_b128(SWIGLU && j >= NB / 2 ? r1 : r0, b_block(b, j), 0, 0);
  };
  auto load_b_lds = [&](const Stream& b, int slot, int i) {
    const __amdgpu_buffer_rsrc_t r0 = b_rsrc(b, i, false), r1 = SWIGLU ? b_rsrc(b, i, true) : r0;
#pragma unroll
    for (int j = 0; j < NB; ++j)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(SWIGLU && j >= NB / 2 ? r1 : r0, LDS_PTR(own_block(slot * NB + j)), 16, b_block(b, j), 0, 0, 0);
  };
  // The first loads of a tile.  Loads return in the order they are issued, so what the next address or the wait needs goes out
  // first: the flags of the row block, the row ids; then weights, which come from HBM.
  int flags = 0, row_id[AROWS ? FM : 1], out_row[kSums];
  u32x2 norm_w = {0u, 0u};
  const bool sums = wave < FM * (SWIGLU ? NB / 2 : NB);
  constexpr int kBFirst = AROWS ? 2 : RV;
  auto begin = [&](const Tile& x) {
    const Group& G = x.e ? p.g[1] : p.g[0];
    const int me = x.e ? m[1] : m[0], first_row = x.e ? m[0] : 0, row0 = x.rb * kRows;
    if constexpr (ROLE == 2) flags = poll_flags(fs, tid, x.e * kFusedMaxRowBlocks + x.rb);
    if constexpr (AROWS) {
#pragma unroll
      for (int f = 0; f < FM; ++f) {
        const int r = row0 + 16 * f + l16;
        row_id[f] = fs.gather[first_row + (r < me ? r : 0)];
      }
    }
    if constexpr (!SWIGLU) {
#pragma unroll
      for (int u = 0; u < kSums; ++u) {
        const int q = wave + 8 * u, r = row0 + (q / NB) * 16 + l16, c = x.ct * kTileN + (q % NB) * 16 + 4 * lq;
        out_row[u] = -1;
        if (sums && r < me && c < G.n) out_row[u] = p.scatter != nullptr ? p.scatter[first_row + r] : first_row + r;
      }
    }
    if constexpr (NORM) norm_w = __builtin_amdgcn_raw_buffer_load_b64(make_rsrc(fs.norm_weight, static_cast<uint32_t>(G.k) * 2u), tid * 8, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
    const Stream b = stream_of(x);
#pragma unroll
    for (int i = 0; i < kBFirst; ++i) load_b(b, i, i);
    __builtin_amdgcn_sched_barrier(0);
  };

  // (as a vector load: scalar loads return in any order, and a wait for the launch's arguments would be one for these as well)
  const u32x4 off = __builtin_amdgcn_raw_buffer_load_b128(make_rsrc(p.offsets, 12), 0, 0, 0);
  __builtin_amdgcn_sched_barrier(0);
  auto offset = [&](int q) { return static_cast<int>(__builtin_amdgcn_readfirstlane(off[q])); };
  if constexpr (ROLE != 0) {
    // The offsets are a memory latency away.  The row counts the host took for granted when it sized the grid are in the
    // launch's arguments: the first tile begins with them, and begins again where they turn out not to be the device's.
    place(fs.guess[0], fs.guess[1]);
    if (t < end) begin(tile_of(t));
    if (offset(0) != 0 || offset(1) != fs.guess[0] || offset(2) - offset(1) != fs.guess[1]) {
      place(offset(1) - offset(0), offset(2) - offset(1));
      if (t < end) begin(tile_of(t));
    }
  } else {
    place(offset(1) - offset(0), offset(2) - offset(1));
    if (t < end) begin(tile_of(t));
  }
  const int pad0 = static_cast<int>(round_up_256(m[0])), pad1 = static_cast<int>(round_up_256(m[1]));
  int held = -1;  // the row block whose rows `fa` holds

  while (t < end) {
    const Tile x = tile_of(t);
    int next = t + step;
    if (next >= end) go_behind(next);
    const int e = x.e, rb = x.rb, ct = x.ct;
    const Group G = e ? p.g[1] : p.g[0];
    const int nct = e ? cols[1] : cols[0], me = e ? m[1] : m[0], pad_e = e ? pad1 : pad0;
    const int row0 = rb * kRows, col0 = ct * kTileN;
    const int counter = e * kFusedMaxRowBlocks + rb;
    const Stream B = stream_of(x);
    const bool fresh = !SWIGLU || held != counter;
    held = B.share <= R ? counter : -1;

    // A: K-tiled rows (the activations, or the intermediate of this expert), or the token rows themselves
    const char* a_base;
    uint32_t a_off[FM], a_step, a_bytes;
    auto load_a = [&](int slot, int i) {
      const int ks = B.k_first + 2 * i;
      const int64_t adv = static_cast<int64_t>(ks) * a_step;
      const __amdgpu_buffer_rsrc_t r = make_rsrc(a_base + adv, i < B.share && ks < B.steps ? (AROWS ? a_bytes - static_cast<uint32_t>(adv) : a_bytes) : 0u);
      // (the intermediate inside a fused launch: read past this XCD's L2, since a cache line of it may have two writers)
#pragma unroll
      for (int f = 0; f < FM; ++f) fa[slot][f] = __builtin_amdgcn_raw_buffer_load_b128(r, a_off[f], 0, ROLE == 2 ? 16 /* sc1 */ : 0);
    };
    if constexpr (!AROWS) {
#pragma unroll
      for (int i = R - RL; i < R; ++i) load_b_lds(B, i - RV, i);
    }
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (AROWS) {
      a_base = reinterpret_cast<const char*>(fs.x);
      a_step = 64;
      a_bytes = static_cast<uint32_t>(m[0] + m[1]) * static_cast<uint32_t>(G.k) * 2u;
#pragma unroll
      for (int f = 0; f < FM; ++f)
        a_off[f] = row0 + 16 * f + l16 < me ? static_cast<uint32_t>(row_id[f]) * static_cast<uint32_t>(G.k) * 2u + lq * 16u : 0x80000000u;
    } else {
      const int a_blocks = SWIGLU ? G.lda : pad_e / kBlkRows;
      const int first = (SWIGLU && e ? pad0 : 0) / kBlkRows + row0 / kBlkRows;
      a_base = reinterpret_cast<const char*>(SWIGLU ? G.a : G.a + (e ? static_cast<int64_t>(pad0) * p.g[0].k : 0));
      a_step = a_bytes = static_cast<uint32_t>(a_blocks) << 10;
#pragma unroll
      for (int f = 0; f < FM; ++f) a_off[f] = (static_cast<uint32_t>(first + f) << 10) + frag;
    }
    int before = 0;
    if constexpr (ROLE == 2) wait_for_flags(fs, tid, counter, (e ? p.g[1].k : p.g[0].k) / (8 * NBP), flags, before);
    if (fresh) {
#pragma unroll
      for (int i = 0; i < R; ++i) load_a(i, i);
    }
    u32x2 res[kSums];
    if constexpr (!SWIGLU) {
#pragma unroll
      for (int u = 0; u < kSums; ++u) {
        res[u] = u32x2{0u, 0u};
        if (p.residual != nullptr && out_row[u] >= 0)
          res[u] = *reinterpret_cast<const u32x2*>(p.residual + static_cast<int64_t>(out_row[u]) * G.ldc + col0 + ((wave + 8 * u) % NB) * 16 + 4 * lq);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = kBFirst; i < RV; ++i) load_b(B, i, i);
    if constexpr (AROWS) {
#pragma unroll
      for (int i = R - RL; i < R; ++i) load_b_lds(B, i - RV, i);
    }
    __builtin_amdgcn_sched_barrier(0);
    float inv[FM];
    if constexpr (NORM) {
      if (fresh) {
#pragma unroll
        for (int f = 0; f < FM; ++f) {
          float ss = 0.f;
#pragma unroll
          for (int i = 0; i < R; ++i)
#pragma unroll
            for (int w = 0; w < 4; ++w) {
              const float lo = __uint_as_float(fa[i][f][w] << 16), hi = __uint_as_float(fa[i][f][w] & 0xffff0000u);
              ss = __builtin_fmaf(lo, lo, ss);
              ss = __builtin_fmaf(hi, hi, ss);
            }
          ss += __shfl_xor(ss, 16);
          ss += __shfl_xor(ss, 32);
          if (lane < 16) ss_of[(16 * f + l16) * 8 + wave] = ss;
        }
        *reinterpret_cast<u32x2*>(norm_lds + tid * 8) = norm_w;  // (zeros past the row's end)
        lds_barrier();  // (the weights' loads stay in flight)
#pragma unroll
        for (int f = 0; f < FM; ++f) {
          const f32x4 a = *reinterpret_cast<const f32x4*>(ss_of + (16 * f + l16) * 8), b = *reinterpret_cast<const f32x4*>(ss_of + (16 * f + l16) * 8 + 4);
          inv[f] = __frsqrt_rn(((a[0] + a[1]) + (a[2] + a[3]) + (b[0] + b[1]) + (b[2] + b[3])) / static_cast<float>(G.k) + fs.norm_eps);
        }
      }
    }
    f32x4 acc[FM][NB];
#pragma unroll
    for (int f = 0; f < FM; ++f)
#pragma unroll
      for (int j = 0; j < NB; ++j) acc[f][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int base = 0; base < B.share; base += R) {  // (once, for a contraction of at most 256 R)
#pragma unroll
      for (int i = 0; i < R; ++i) {
        if constexpr (NORM) {
          if (fresh) {
            const u32x4 w4 = *reinterpret_cast<const u32x4*>(norm_lds + (B.k_first + 2 * i) * 64 + lq * 16);
#pragma unroll
            for (int w = 0; w < 4; ++w) {
              const float w_lo = __uint_as_float(w4[w] << 16), w_hi = __uint_as_float(w4[w] & 0xffff0000u);
#pragma unroll
              for (int f = 0; f < FM; ++f) fa[i][f][w] = rms_scale(fa[i][f][w], w_lo, w_hi, inv[f]);
            }
          }
        }
        if (RL > 0 && i == RV) {
          asm volatile("" ::: "memory");
          __builtin_amdgcn_s_waitcnt(waitcnt_imm(0, 15));
          asm volatile("" ::: "memory");
        }
#pragma unroll
        for (int j = 0; j < NB; ++j) {
          const bf16x8 b = i < R - RL ? __builtin_bit_cast(bf16x8, fb[i % RV][j]) : *reinterpret_cast<const bf16x8*>(own_block((i - RV) * NB + j) + lane * 16);
#pragma unroll
          for (int f = 0; f < FM; ++f)
            acc[f][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b, __builtin_bit_cast(bf16x8, fa[i][f]), acc[f][j], 0, 0, 0);
        }
        if (RV < R && RL == 0 && i + RV < R) load_b(B, i % RV, base + i + RV);
        if (!NORM && base + R < B.share) {
          if (i >= R - RL - RV && i < R - RL) load_b(B, i % RV, base + R + i % RV);
          load_a(i, base + i + R);
        }
      }
      if (RL > 0 && !NORM && base + R < B.share) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the fragments in LDS have been read
#pragma unroll
        for (int i = R - RL; i < R; ++i) load_b_lds(B, i - RV, base + i + R);
      }
    }
    // (the last tile's sums need what `begin` changes)
    int out_now[kSums];
#pragma unroll
    for (int u = 0; u < kSums; ++u) out_now[u] = out_row[u];
    if (next < end) begin(tile_of(next));  // the next tile's first loads, while this one's sums meet
    // partial sums: lane l of a block holds row l % 16, columns 4 (l / 16) .. + 3
    if constexpr (RL > 0) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int f = 0; f < FM; ++f)
#pragma unroll
      for (int j = 0; j < NB; ++j) *reinterpret_cast<f32x4*>(own_block(f * NB + j) + lane * 16) = acc[f][j];
    __syncthreads();
    auto sum_of = [&](int block) {
      const unsigned char* const at = (!kMore || block < 8 ? part + block * 1024 : more + (block - 8) * 1024) + lane * 16;
      f32x4 v = *reinterpret_cast<const f32x4*>(at);
#pragma unroll
      for (int w = 1; w < 8; ++w) v += *reinterpret_cast<const f32x4*>(at + w * 8192);
      return v;
    };
    if constexpr (SWIGLU) {
      if (sums) {  // wavefront (NB / 2) i + j: row block i, columns 16 j .. of the tile
        const int i = wave / (NB / 2), j = wave % (NB / 2);
        const f32x4 g = sum_of(i * NB + j), u = sum_of(i * NB + j + NB / 2);
        float h[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) h[r] = swiglu_bf16(g[r], u[r]);
        // four columns of a row of the K-tiled intermediate, written through where another XCD waits for them
        const int c16 = (col0 >> 4) + j, chunk = 2 * (c16 & 1) + (lq >> 1);
        const int in_block = l16 * 64 + ((chunk ^ ((l16 >> 2) & 3)) << 4) + (lq & 1) * 8;
        const int64_t block = (e ? static_cast<int64_t>(pad0) * p.g[0].n * 2 : 0) +
                              ((static_cast<int64_t>(c16 >> 1) * (pad_e / kBlkRows) + row0 / kBlkRows + i) << 10);
        const u32x2 v = {pack_bf16x2(h[0], h[1]), pack_bf16x2(h[2], h[3])};
        unsigned char* const dst = reinterpret_cast<unsigned char*>(p.g[0].c) + block;
        // (a last tile of half a gate and half an up block more than the matrix has: nothing to store)
        if (col0 + 16 * j < G.n) {
          if constexpr (ROLE == 1) __builtin_amdgcn_raw_buffer_store_b64(v, make_rsrc(dst, kBlkBytes), in_block, 0, 16 /* sc1 */);
          else *reinterpret_cast<u32x2*>(dst + in_block) = v;
          if constexpr (ROLE == 0) {  // the projections themselves, for a backward pass
            if (p.keep[0] != nullptr) {
              *reinterpret_cast<u32x2*>(reinterpret_cast<unsigned char*>(p.keep[0]) + block + in_block) = u32x2{pack_bf16x2(g[0], g[1]), pack_bf16x2(g[2], g[3])};
              *reinterpret_cast<u32x2*>(reinterpret_cast<unsigned char*>(p.keep[1]) + block + in_block) = u32x2{pack_bf16x2(u[0], u[1]), pack_bf16x2(u[2], u[3])};
            }
          }
        }
      }
      if constexpr (ROLE == 1) flag_done(fs, tid, counter, ct, nct);
    } else {
#pragma unroll
      for (int u = 0; u < kSums; ++u) {
        if (out_now[u] < 0) continue;
        const int q = wave + 8 * u;
        const f32x4 y = sum_of(q);
        u32x2 v = {pack_bf16x2(y[0], y[1]), pack_bf16x2(y[2], y[3])};
        if (p.residual != nullptr) {
#pragma unroll
          for (int w = 0; w < 2; ++w)
            v[w] = pack_bf16x2(__uint_as_float(v[w] << 16) + __uint_as_float(res[u][w] << 16),
                               __uint_as_float(v[w] & 0xffff0000u) + __uint_as_float(res[u][w] & 0xffff0000u));
        }
        *reinterpret_cast<u32x2*>(p.g[0].c + static_cast<int64_t>(out_now[u]) * G.ldc + col0 + (q % NB) * 16 + 4 * lq) = v;
      }
      if constexpr (ROLE == 2) clear_flags_if_last(fs, tid, counter, before, nct);
    }
    __syncthreads();  // the partial sums' LDS is written by the next tile
    t = next;
  }
#endif
}

// KA / KB (generic mode only): the operand is stored with K as its slow dimension -- A as [k, m], B as [k, n] --
// and is transposed on the way from LDS to the MFMA registers.
//
// The kernel's body is a function of its own so that one launch can run two of them side by side (the fused FFN
// launch below: some workgroups run the gate/up form, the others the down form).  `wg` of `n_wg` is the workgroup's
// place among those that share this body's tile list (blockIdx.x of gridDim.x in a plain launch).
// ROLE: 0 = a plain launch; 1 / 2 = producer / consumer of a fused launch (see FusedSync); 3 = the contraction in parts, as
// `parts` says, with the scratch `split`; 4 = the second launch of a tail split, an instantiation of its own (a launch of small
// tiles alone that carries its code too runs 0.2 to 0.3 us longer: o projection of 512 rows, hidden 2048, 16.3 -> 15.95).  AROWS (gate/up form of a fused launch): the A operand is read from the token rows themselves,
// fs.x through fs.gather, instead of from a K-tiled copy of them.
template <int MODE, typename TS, bool KA, bool KB, int ROLE, bool AROWS = false>
__device__ __forceinline__ void dual_gemm_body(const Params& p, const int wg, const int n_wg, const FusedSync& fs,
                                               const DownParts parts = DownParts{}, const DownSplit& split = DownSplit{}) {
#if defined(__HIP_DEVICE_COMPILE__)  // the host pass only needs the launch stub; the body uses gfx950-only builtins
  constexpr int BM = TS::BM, BN = TS::BN, FM = TS::FM, FN = TS::FN;
  constexpr int kWavesN = TS::kWavesN, kWaves = TS::kWaves;
  constexpr int kLoadRowsA = TS::kLoadRowsA, kLoadRowsB = TS::kLoadRowsB, kLoadsA = TS::kLoadsA, kLoadsB = TS::kLoadsB;
  constexpr int kLoadsPerStep = kLoadsA + kLoadsB;
  constexpr int kSlotBytesA = TS::kSlotBytesA, kSlotBytesB = TS::kSlotBytesB, kStageBytes = TS::kStageBytes;
  constexpr bool SWIGLU = MODE == kGateUp;
  constexpr bool TILED_IN = MODE == kGateUp || MODE == kDown;   // A and B are K-tiled
  constexpr bool TILED_OUT = MODE == kGateUp;   // C is K-tiled
  static_assert(MODE == kGeneric || (!KA && !KB), "K-major operands exist in the generic mode only");
  // kStages ring slots per operand, each one K step (256 rows x 32 bf16).  Separate arrays let the compiler
  // see that a read of one slot never waits for a buffer load that targets another.
  // Row-major operands with K contiguous (the NT layout of the generic mode): the ring's slots live in PAIRS.  A load instruction then fetches 8 rows x 128 bytes -- the K chunks of two consecutive K steps,
  // i.e. whole cache lines -- where one slot's worth would be 16 rows x 64 bytes (sixteen half lines, which hold the
  // loading wavefront's issue slot about twice as long).  A pair is one array of 1 KiB blocks, block = 8 rows x
  // [512 bytes of the even step | 512 bytes of the odd step], so the instruction's 64 lanes land on consecutive LDS
  // addresses; inside a step's half, rows are 64 bytes with the same chunk swizzle as everywhere else.
  // (The projection that rotates heads reads row-major operands too and keeps the slot-by-slot ring: with pairs its
  // launches measured 3 % slower inside a forward pass.)
  constexpr bool kPair = MODE == kGeneric && !KA && !KB;
  // NN (a row-major A beside a K-major B: dX, dHm, the op's default layout): A alone lives in pairs, B keeps its slots
  constexpr bool kPairAOnly = MODE == kGeneric && !KA && KB;
  constexpr bool kPA = kPair || kPairAOnly, kPB = kPair;
  constexpr int kRingA = kPA ? 16 : kSlotBytesA, kRingB = kPB ? 16 : kSlotBytesB;  // the form not in use shrinks
  constexpr int kPairA = kPA ? 2 * kSlotBytesA : 16, kPairB = kPB ? 2 * kSlotBytesB : 16;
  constexpr int kRingAlignA = kPA ? 16 : 1024, kPairAlignA = kPA ? 1024 : 16;
  constexpr int kRingAlignB = kPB ? 16 : 1024, kPairAlignB = kPB ? 1024 : 16;
  // (one LDS object per (size, alignment, index): the two bodies of a fused launch name the same objects, so the
  // launch needs the LDS of one of them)
  unsigned char* const s_a0 = lds_array<kRingA, kRingAlignA, 0>();
  unsigned char* const s_a1 = lds_array<kRingA, kRingAlignA, 1>();
  unsigned char* const s_a2 = lds_array<kRingA, kRingAlignA, 2>();
  unsigned char* const s_b0 = lds_array<kRingB, kRingAlignB, 3>();
  unsigned char* const s_b1 = lds_array<kRingB, kRingAlignB, 4>();
  unsigned char* const s_b2 = lds_array<kRingB, kRingAlignB, 5>();
  unsigned char* const s_a3 = lds_array<kRingA, kRingAlignA, 6>();
  unsigned char* const s_b3 = lds_array<kRingB, kRingAlignB, 7>();
  unsigned char* const s_pa0 = lds_array<kPairA, kPairAlignA, 8>();  // slots 0 and 1 of A
  unsigned char* const s_pa1 = lds_array<kPairA, kPairAlignA, 9>();  // slots 2 and 3
  unsigned char* const s_pb0 = lds_array<kPairB, kPairAlignB, 10>();
  unsigned char* const s_pb1 = lds_array<kPairB, kPairAlignB, 11>();
  unsigned char* const s_out = lds_array<kWaves * kStageBytes, 1024, 12>();
  // ring slot s of each operand (s is a constant after unrolling)
  static_assert(kStages == 4, "ring slots are declared one by one");
  auto slot_a = [&](int s) -> unsigned char* {
    if constexpr (kPA) return (s < 2 ? s_pa0 : s_pa1) + (s & 1) * 512;
    else return s == 0 ? s_a0 : (s == 1 ? s_a1 : (s == 2 ? s_a2 : s_a3));
  };
  auto slot_b = [&](int s) -> unsigned char* {
    if constexpr (kPB) return (s < 2 ? s_pb0 : s_pb1) + (s & 1) * 512;
    else return s == 0 ? s_b0 : (s == 1 ? s_b1 : (s == 2 ? s_b2 : s_b3));
  };

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform: keeps descriptors and LDS bases scalar
  const int wm = wave / kWavesN, wn = wave % kWavesN;
  // MFMA fragment: row (column) l16, 16-byte K chunk lq of the step's four.  Any order of the chunks over the four lane
  // groups will do as long as both operands use it; in this one a ds_read_b128 of 16 swizzled rows, which is served 16
  // lanes at a time -- 0-3, 12-15, 20-27, then 4-11, 16-19, 28-31, and the same above -- touches every bank once each
  // time (in the plain order 0, 1, 2, 3 every read takes twice as long).
  const int l16 = lane & 15, lq = (0x9c >> (2 * (lane >> 4))) & 3;  // 0, 3, 1, 2
  // With more wavefronts than SIMDs only the first kLoadWaves (one per SIMD) issue the global -> LDS loads.  A
  // wavefront that issues a load is held while the CU's load path takes the instruction in; its partner on the same
  // SIMD, which issues none, keeps the MFMA pipe fed meanwhile.  When both partners load on the same schedule they
  // stall together and the pipe idles.
  constexpr int kLoadWaves = TS::kLoadWaves;
  constexpr bool ASYM = kLoadWaves != kWaves;
  const bool loads = !ASYM || wave < kLoadWaves;

  // ---- problem table (uniform) ------------------------------------------------------------------
  // (kept as two named structs, selected per tile, so everything stays in scalar registers)
  Group g0 = p.g[0], g1 = p.g[1];
  int sorted_first[2] = {0, 0};  // tiled modes: sorted position of each expert's first row
  int sorted_total = 0;          // ... and the number of sorted rows
  if constexpr (TILED_IN) {
    // (Behind the asm statements of down_split_kernel they would be vector loads.  A fused launch's are scalar as they stand, and
    // the other type moves its prologue about: 2048 rows 0.2 us a layer slower.)
    using Offsets = std::conditional_t<ROLE == 1 || ROLE == 2, const int32_t*, ScalarInts>;
    const Offsets offsets = (Offsets)p.offsets;
    const int o0 = offsets[0], o1 = offsets[1], o2 = offsets[2];
    g0.m = o1 - o0;
    g1.m = o2 - o1;
    const int pad0 = static_cast<int>(round_up_256(g0.m)), pad1 = static_cast<int>(round_up_256(g1.m));
    if constexpr (MODE == kGateUp) {
      // A: one tiled activation matrix, expert 1 starts at the next multiple of 256 rows.
      // C: per-expert tiled intermediates, packed one after the other
      g0.a_row0 = 0;
      g1.a_row0 = pad0;
      g0.ldc = pad0 / kBlkRows;
      g1.ldc = pad1 / kBlkRows;
      g1.c = g0.c + static_cast<int64_t>(pad0) * g0.n;
    } else {
      // A: per-expert tiled intermediates;  C: row-major, expert e's rows start at offsets[e]
      g0.a_row0 = 0;
      g1.a_row0 = 0;
      g0.lda = pad0 / kBlkRows;
      g1.lda = pad1 / kBlkRows;
      g1.a = g0.a + static_cast<int64_t>(pad0) * g0.k;
      if (p.scatter == nullptr) {
        g0.c += static_cast<int64_t>(o0) * g0.ldc;
        g1.c += static_cast<int64_t>(o1) * g1.ldc;
      }
    }
    sorted_first[0] = o0;
    sorted_first[1] = o1;
    sorted_total = o2;
  }
  constexpr int kTileN = SWIGLU ? BN / 2 : BN;  // output columns per tile
  int tiles_m[2], tiles_n[2];
  tiles_m[0] = (g0.m + BM - 1) / BM;
  tiles_n[0] = (g0.n + kTileN - 1) / kTileN;
  if (g0.m <= 0 || g0.n <= 0) tiles_m[0] = tiles_n[0] = 0;
  tiles_m[1] = (g1.m + BM - 1) / BM;
  tiles_n[1] = (g1.n + kTileN - 1) / kTileN;
  if (g1.m <= 0 || g1.n <= 0) tiles_m[1] = tiles_n[1] = 0;
  // split contraction: part q of a column tile is a column tile of its own, all columns' part 0 first
  // (lg of expert 0, and of expert 1 four bits up: one register across the K loop)
  const int lg_parts = ROLE == 3 ? (parts.cut[0] ? parts.lg : 0) | (parts.cut[1] ? parts.lg : 0) << 4 : 0;
  auto lg_of = [&](int group) { return lg_parts >> (4 * group) & 3; };
  auto cols_of = [&](int group) { return ((group ? g1.n : g0.n) + kTileN - 1) / kTileN; };
  if (ROLE != 3 && p.gate != 0) {
    constexpr int kBigN = SWIGLU ? BigTile::BN / 2 : BigTile::BN;
    auto big = [](int m, int n) { return (m <= 0 || n <= 0) ? 0 : ((m + BigTile::BM - 1) / BigTile::BM) * ((n + kBigN - 1) / kBigN); };
    const bool few = shape_deciding_tiles(big(g0.m, g0.n), big(g1.m, g1.n), g0.k, g1.k) <= p.gate_tiles;
    if (few != (p.gate == 1)) return;  // uniform: the other tile shape's launch does this problem
  }
  if constexpr (ROLE == 3) {
    tiles_n[0] <<= lg_of(0);
    tiles_n[1] <<= lg_of(1);
  }
  int total = tiles_m[0] * tiles_n[0] + tiles_m[1] * tiles_n[1];  // the host bounds this below 2^31
  // tail split (tail_plan): the first launch (256 x 256 tiles) stops at `split_at`; the second (this shape: 128 x 128)
  // takes virtual tiles [split_at, all) of the 256 x 256 tiling, kSubM x kSubN pieces each, and then the strips
  constexpr bool kIsTail = ROLE == 4, kIsBig = ROLE == 0 && std::is_same_v<TS, BigTileFor<MODE>>;
  static_assert(!kIsTail || std::is_same_v<TS, TailTileFor<MODE>>, "the second launch's tile");
  constexpr int kSubM = BigTile::BM / BM, kSubN = BigTile::BN / BN;
  int big_m[2], big_n[2], split_at = 0, pieces = 0, strip_cols[2] = {0, 0};
  if (kIsTail || (kIsBig && p.split == 1)) {
    constexpr int kBigN = SWIGLU ? BigTile::BN / 2 : BigTile::BN;
    big_n[0] = (g0.n + kBigN - 1) / kBigN;
    big_n[1] = (g1.n + kBigN - 1) / kBigN;
    const bool any0 = g0.m > 0 && g0.n > 0, any1 = g1.m > 0 && g1.n > 0;
    TailPlan plan;
    if constexpr (MODE == kGateUp || MODE == kDown)
      plan = tail_plan(any0 ? g0.m : 0, any1 ? g1.m : 0, any0 ? big_n[0] : 0, any1 ? big_n[1] : 0, g0.k, g1.k, p.split_cus, MODE != kDown, kTailLongTiled);
    else
      plan = p.plan;
    if (!any0) big_n[0] = 0;
    if (!any1) big_n[1] = 0;
    big_m[0] = plan.rows[0];
    big_m[1] = plan.rows[1];
    split_at = plan.first;
    if constexpr (kIsBig) {
      total = split_at;
      if (MODE != kDown) {
        tiles_m[0] = big_m[0];
        tiles_m[1] = big_m[1];
      }
    } else {
      if (!plan.split) return;  // the first launch did everything
      pieces = kSubM * kSubN * (big_m[0] * big_n[0] + big_m[1] * big_n[1] - split_at);
      if (MODE != kDown) {  // strips: the row of small tiles behind an expert's large ones
        strip_cols[0] = kSubM * big_m[0] < tiles_m[0] ? tiles_n[0] : 0;
        strip_cols[1] = kSubM * big_m[1] < tiles_m[1] ? tiles_n[1] : 0;
      }
    }
  }
  const int padded = (total + kXcds - 1) / kXcds * kXcds;

  // ---- per-lane constants -----------------------------------------------------------------------
  // row-major loader: one instruction fills 16 LDS rows of 64 bytes; lane -> (row lane/4, slot lane%4).
  // Instruction i of this wave covers rows [wave*64 + 16i, +16) of A.  Chunk c of row r lives in slot c ^ ((r >> 2) & 3).
  const int ld_row0 = wave * kLoadRowsA + (lane >> 2);
  const int ld_chunk = (lane & 3) ^ ((lane >> 4) & 3);
  // fragment reads: row = base + l16, K chunk lq; 16 rows x 64 bytes, i.e. one whole KiB per read
  const int sw = (l16 >> 2) & 3;
  const int frag_off = (lq ^ sw) << 4;
  const int a_row_off = (wm * (FM * 16) + l16) * kRowBytes + frag_off;
  // paired slots: row r of a step's half sits at block r / 8 (1 KiB each), row r % 8 inside it
  const int pair_lane_off = ((l16 >> 3) << 10) + ((l16 & 7) << 6) + frag_off;
  const int a_pair_off = wm * (FM * 16) * 128 + pair_lane_off;
  // paired loader: lane -> (row lane / 4 % 8 of the instruction's 8 rows, step half lane / 32, slot lane % 4)
  constexpr int kPairLoadsA = kLoadRowsA / 8, kPairLoadsB = kLoadRowsB / 8;
  const int pl_row = (lane >> 2) & 7, pl_half = lane >> 5, pl_slot = lane & 3;
  // K chunk (of the 8 in a 128-byte line) this lane fetches in instruction i: the instruction's rows are 8 i + pl_row
  // past a multiple of 32, and the slot holds chunk slot ^ ((row >> 2) & 3) of its step -- one value for even i, one
  // for odd i, so a lane's byte offsets are two bases plus i times the (uniform) pitch of 8 rows
  const int pair_chunk_even = 4 * pl_half + (pl_slot ^ ((pl_row >> 2) & 3));
  const int pair_chunk_odd = 4 * pl_half + (pl_slot ^ (((pl_row >> 2) + 2) & 3));
  auto pair_chunk = [&](int i) { return (i & 1) ? pair_chunk_odd : pair_chunk_even; };
  // B fragment j of this wave starts at LDS row b_row(j): plain tiles hold 256 weight rows; SwiGLU tiles hold 128
  // gate rows then the 128 up rows of the same output columns, and fragments [0, FN/2) are gate, [FN/2, FN) up
  auto b_row = [&](int j) {
    if constexpr (SWIGLU) return (j < FN / 2 ? 0 : BN / 2) + wn * (FN / 2 * 16) + (j % (FN / 2)) * 16;
    else return wn * (FN * 16) + j * 16;
  };
  const int b_lane_off = l16 * kRowBytes + frag_off;
  // K-major operand (KA / KB): a slot holds BK rows of K, each a run of BM (BN) columns, as whole 16-byte chunks.
  // ds_read_b64_tr_b16 works on groups of 16 lanes: lane j of a group supplies the address of 4 consecutive columns of
  // row (j >> 2), and receives column j of the 4 rows.  A group covers one 16-column block (32 bytes of a row); group
  // lq takes K rows [8 lq, +8) in two reads of four.  The 32-byte unit u of row k sits at position
  // u ^ (2 (k & 3)) ^ ((k >> 3) & 1): the four rows of one group and the two groups that are served together (rows
  // 8 apart) fall into different banks.
  const int tr_row = l16 >> 2;
  auto tr_lane_base = [&](int row_bytes, int first_block) {  // first_block: this wave's first 16-column block
    return (8 * lq + tr_row) * row_bytes + ((first_block ^ (2 * tr_row) ^ (lq & 1)) << 5) + (l16 & 3) * 8;
  };
  const int tr_base_a = KA ? tr_lane_base(BM * 2, wm * FM) : 0;
  const int tr_base_b = KB ? tr_lane_base(BN * 2, wn * FN) : 0;

  // K-major loads (k_major.h): a loading wavefront fills K rows [8 wave, +8) of the slot.  Columns past the matrix
  // edge read whatever follows (the next row, or zero past the end): they only reach output rows / columns that are
  // never stored.  Rows past K are out of the descriptor's range and read as zero.  (The offset is worked out at each
  // use -- `step` keeps it from being held in registers across the loop, which has none to spare.)
  static_assert((!KA || kLoadsA * 1024 == 8 * BM * 2) && (!KB || kLoadsB * 1024 == 8 * BN * 2), "8 rows of K per wave");
  auto k_major_voff = [&](int i, int cols, uint32_t row_bytes, int step) {
    int l = lane;
    asm("" : "+v"(l) : "s"(step));
    return k_major_offset(l, wave, i, cols, row_bytes);
  };
  // ---- per-tile state ------------------------------------------------------------------------------
  struct Loader {   // where this wave's kLoadsA + kLoadsB loads per K step come from
    const __bf16 *a_base, *b_base;
    uint32_t a_bytes, b_bytes;        // readable bytes from the base (row-major) / from the current block (tiled)
    uint32_t voff_a[kPA ? 2 : kLoadsA], voff_b[kPB ? 2 : kLoadsB];  // paired slots: [even i, odd i] of instruction 0
    uint32_t pitch_a, pitch_b;        // paired slots: bytes between the rows of consecutive load instructions; K-major:
                                      // bytes of a row
    int64_t a_step, b_step;           // tiled, K-major: bytes between consecutive K steps
    // tiled, K-major: the load stream walks a tile's K steps in order, so the step's base and the bytes readable from it are
    // kept as running values (one add and one saturating subtract per step) instead of products with the step index
    const char *a_cur, *b_cur;
    uint32_t a_left, b_left, a_dec, b_dec;
    int K, nk;      // nk: K steps of the tile, rounded up to a multiple of kStages (padding steps read zeros)
  };
  struct Store {    // where the finished tile goes
    __bf16* c_base;
    const int32_t* row_id;  // kDown with scatter: output row of each of the tile's rows (c_base is then row 0)
    const __bf16* res;      // kDown with scatter and a residual: the residual's column col0 of row 0; generic with
                            // an addend: its element under c_base; else null
    int rows, cols_left, ldc, nk;
    int row0, col0;         // first row / column of the tile inside its group's output
    int row_block;          // fused launch: index of the tile's (expert, row block) counters
    int split;              // split contraction: (logarithm of the number of parts, this part, the slot of the tile's first)
  };

  // K steps of a tile rounded up to whole ring rounds (padding steps read zeros).  The host never launches this
  // kernel with k == 0 and a non-empty output: the tile loop below advances only from inside the K loop.
  auto padded_steps = [](int k) { return ((k + BK - 1) / BK + kStages - 1) / kStages * kStages; };
  // split contraction: the K steps of a part (whole ring rounds; the last part has what is left)
  auto part_steps = [&](int k, int lg) { return (((k / BK + (1 << lg) - 1) >> lg) + kStages - 1) / kStages * kStages; };
  auto part_k = [&](int k, int lg, int part) {
    const int left = k - part * part_steps(k, lg) * BK, most = part_steps(k, lg) * BK;
    return left < most ? left : most;
  };
  auto setup_store = [&](const TileCoord& tc, Store& S) {
    const Group G = tc.group ? g1 : g0;
    const int row0 = tc.tm * BM, col0 = tc.tn * kTileN;
    if constexpr (TILED_OUT) {
      // block (row block, column block) of the tiled intermediate: [column block][row block], 1 KiB each
      S.c_base = G.c + ((static_cast<int64_t>(col0 / kBlkCols) * G.ldc + row0 / kBlkRows) << 9);
    } else {
      S.c_base = G.c + static_cast<int64_t>(row0) * G.ldc + col0;
    }
    S.row_id = nullptr;
    S.res = nullptr;
    if constexpr (MODE == kDown) {
      if (p.scatter != nullptr) {
        S.c_base = G.c + col0;
        S.row_id = p.scatter + sorted_first[tc.group] + row0;
        if (p.residual != nullptr) S.res = p.residual + col0;
      }
    }
    if constexpr (MODE == kGeneric) {
      if (G.add != nullptr) S.res = G.add + static_cast<int64_t>(row0) * G.ldc + col0;
    }
    S.rows = G.m - row0 < BM ? G.m - row0 : BM;
    S.cols_left = G.n - col0;
    S.row0 = row0;
    S.col0 = col0;
    S.row_block = tc.group * kFusedMaxRowBlocks + tc.tm;
    S.ldc = G.ldc;
    S.nk = padded_steps(G.k);
    if constexpr (ROLE == 3) {
      const int lg = lg_of(tc.group);
      const int slot = lg == 0 ? 0 : (tc.group && lg_of(0) > 0 ? tiles_m[0] * tiles_n[0] : 0) + ((tc.tm * cols_of(tc.group) + tc.tn) << lg);
      S.split = lg | tc.part << 4 | slot << 8;
      S.nk = padded_steps(part_k(G.k, lg, tc.part));
    }
  };
  auto setup_loader = [&](const TileCoord& tc, Loader& L) {
    const Group G = tc.group ? g1 : g0;
    const int row0 = tc.tm * BM, col0 = tc.tn * kTileN;
    L.K = G.k;
    int64_t first = 0;  // the tile's first K step
    if constexpr (ROLE == 3) {
      const int lg = lg_of(tc.group);
      L.K = part_k(G.k, lg, tc.part);
      first = static_cast<int64_t>(tc.part) * part_steps(G.k, lg);
    }
    L.nk = padded_steps(L.K);
    constexpr int kHalfWaves = kLoadWaves / 2;  // SwiGLU: the first half of the loading waves load gate rows, the rest up rows
    const bool up_half = SWIGLU && wave >= kHalfWaves;
    const __bf16* b_src = up_half ? G.b1 : G.b0;
    const int b_wave = SWIGLU ? wave % kHalfWaves : wave;
    if constexpr (TILED_IN) {
      // this wave's row blocks of the A tile and of the B tile at K step 0; a K step later they sit one column
      // block further, i.e. (row blocks of the matrix) KiB ahead
      const int64_t b_blk = first * G.ldb + col0 / kBlkRows + b_wave * kLoadsB;
      L.b_base = b_src + (b_blk << 9);
      L.b_step = static_cast<int64_t>(G.ldb) << 10;
      const int64_t b_left = (static_cast<int64_t>(G.k / kBlkCols) * G.ldb - b_blk) << 10;
      L.b_bytes = static_cast<uint32_t>(b_left < 0 ? 0 : (b_left > 0x7fffff00ll ? 0x7fffff00ll : b_left));
      L.b_cur = reinterpret_cast<const char*>(L.b_base);
      L.b_left = L.b_bytes;
      L.b_dec = static_cast<uint32_t>(L.b_step > 0x7fffff00ll ? 0x7fffff00ll : L.b_step);
#pragma unroll
      for (int i = 0; i < kLoadsB; ++i) L.voff_b[i] = static_cast<uint32_t>(i * kBlkBytes + lane * 16);
      if constexpr (AROWS) {
        // A from the token rows: sorted row r of the tile is row gather[...] of the row-major activations; a load
        // instruction fetches 64 bytes of 16 such rows (lane -> row lane / 4, and the chunk that belongs in LDS slot
        // lane % 4), rows past the expert's last row read as zero.  The host keeps the matrix below 2 GiB.
        const int rows_a = G.m - row0 < BM ? G.m - row0 : BM;
        L.a_base = fs.x;
        L.a_bytes = static_cast<uint32_t>(sorted_total) * static_cast<uint32_t>(G.k) * 2u;
        L.a_step = 0;
        L.a_cur = nullptr;
        L.a_left = L.a_dec = 0;
#pragma unroll
        for (int i = 0; i < kLoadsA; ++i) {
          const int r = ld_row0 + 16 * i;
          uint32_t v = 0x80000000u;
          if (r < rows_a)
            v = static_cast<uint32_t>(fs.gather[sorted_first[tc.group] + row0 + r]) * static_cast<uint32_t>(G.k) * 2u + ld_chunk * 16u;
          L.voff_a[i] = v;
        }
      } else {
        const int64_t a_blk = first * G.lda + (G.a_row0 + row0) / kBlkRows + wave * kLoadsA;
        L.a_base = G.a + (a_blk << 9);
        L.a_step = static_cast<int64_t>(G.lda) << 10;
        const int64_t a_left = (static_cast<int64_t>(G.k / kBlkCols) * G.lda - a_blk) << 10;
        L.a_bytes = static_cast<uint32_t>(a_left < 0 ? 0 : (a_left > 0x7fffff00ll ? 0x7fffff00ll : a_left));
        L.a_cur = reinterpret_cast<const char*>(L.a_base);
        L.a_left = L.a_bytes;
        L.a_dec = static_cast<uint32_t>(L.a_step > 0x7fffff00ll ? 0x7fffff00ll : L.a_step);
#pragma unroll
        for (int i = 0; i < kLoadsA; ++i) L.voff_a[i] = static_cast<uint32_t>(i * kBlkBytes + lane * 16);
      }
    } else {
      const int rows_a = G.m - row0 < BM ? G.m - row0 : BM;
      const int rows_b = G.n - col0 < kTileN ? G.n - col0 : kTileN;
      L.a_step = L.b_step = 0;
      if constexpr (KA) {
        L.a_base = G.a + row0;
        const int64_t left = (static_cast<int64_t>(G.k) * G.lda - row0) * 2;
        L.a_bytes = static_cast<uint32_t>(left < 0 ? 0 : left);
        L.a_step = static_cast<int64_t>(G.lda) * (2 * BK);
        L.a_cur = reinterpret_cast<const char*>(L.a_base);
        L.a_left = L.a_bytes;
        L.a_dec = static_cast<uint32_t>(L.a_step);  // (below 2^32: k_major_fits)
        L.pitch_a = 2u * static_cast<uint32_t>(G.lda);
      } else {
        L.a_base = G.a + static_cast<int64_t>(row0) * G.lda;
        L.a_bytes = static_cast<uint32_t>(rows_a) * G.lda * 2u;
        if constexpr (kPA) {
          const uint32_t row_off = static_cast<uint32_t>(wave * kLoadRowsA + pl_row) * G.lda * 2u;
          L.voff_a[0] = row_off + pair_chunk_even * 16u;
          L.voff_a[1] = row_off + pair_chunk_odd * 16u;
          L.pitch_a = 16u * static_cast<uint32_t>(G.lda);
        } else {
#pragma unroll
          for (int i = 0; i < kLoadsA; ++i) L.voff_a[i] = static_cast<uint32_t>(ld_row0 + 16 * i) * G.lda * 2u + ld_chunk * 16u;
        }
      }
      if constexpr (KB) {
        L.b_base = b_src + col0;
        const int64_t left = (static_cast<int64_t>(G.k) * G.ldb - col0) * 2;
        L.b_bytes = static_cast<uint32_t>(left < 0 ? 0 : left);
        L.b_step = static_cast<int64_t>(G.ldb) * (2 * BK);
        L.b_cur = reinterpret_cast<const char*>(L.b_base);
        L.b_left = L.b_bytes;
        L.b_dec = static_cast<uint32_t>(L.b_step);
        L.pitch_b = 2u * static_cast<uint32_t>(G.ldb);
      } else {
        L.b_base = b_src + static_cast<int64_t>(col0) * G.ldb;
        L.b_bytes = static_cast<uint32_t>(rows_b) * G.ldb * 2u;
        if constexpr (kPair) {
          const uint32_t row_off = static_cast<uint32_t>(b_wave * kLoadRowsB + pl_row) * G.ldb * 2u;
          L.voff_b[0] = row_off + pair_chunk_even * 16u;
          L.voff_b[1] = row_off + pair_chunk_odd * 16u;
          L.pitch_b = 16u * static_cast<uint32_t>(G.ldb);
        } else {
          const int b_ld_row0 = b_wave * kLoadRowsB + (lane >> 2);
#pragma unroll
          for (int i = 0; i < kLoadsB; ++i) L.voff_b[i] = static_cast<uint32_t>(b_ld_row0 + 16 * i) * G.ldb * 2u + ld_chunk * 16u;
        }
      }
    }
  };

  // One K step of global -> LDS for this wave: rows [wave*64, +64) of the A slot, [wave*kLoadRowsB, +kLoadRowsB) of B.
  // The A half goes out right after the barrier that frees the slot, the B half one MFMA group later (spreading
  // the loads keeps the CU's L2 port, 64 bytes per clock, from backing up into the wave's in-order issue);
  // `Pending` carries what the B half needs across that gap, which may include a change of tile.
  struct Pending {
    __amdgpu_buffer_rsrc_t rb;
    uint32_t voff_b[kPB ? 2 : kLoadsB];
    uint32_t pitch_b;  // paired slots, K-major
  };
  // Paired slots: the loads of K steps ks and ks + 1 (ks even) of this wave's rows, A here and B through `Pending`.
  auto issue_pair_a = [&](Loader& L, int ks, unsigned char* pa, Pending& P) {
    const int k0 = ks * BK;
    const uint32_t adv = 2u * static_cast<uint32_t>(k0);
    // as in issue_a: the base advances along K and keeps the absolute end of the readable range, so rows past the
    // matrix read as zero; K chunks at or past the row end are pushed out of range lane by lane
    const __amdgpu_buffer_rsrc_t ra = make_rsrc(L.a_base + k0, L.a_bytes > adv ? L.a_bytes - adv : 0u);
    const bool k_tail = k0 + 2 * BK > L.K;
    const uint32_t oob_even = (k_tail && k0 + pair_chunk_even * 8 >= L.K) ? 0x80000000u : 0u;
    const uint32_t oob_odd = (k_tail && k0 + pair_chunk_odd * 8 >= L.K) ? 0x80000000u : 0u;
    if constexpr (kPB) {
      P.rb = make_rsrc(L.b_base + k0, L.b_bytes > adv ? L.b_bytes - adv : 0u);
      P.voff_b[0] = L.voff_b[0] | oob_even;
      P.voff_b[1] = L.voff_b[1] | oob_odd;
      P.pitch_b = L.pitch_b;
    }
    const uint32_t va_even = L.voff_a[0] | oob_even, va_odd = L.voff_a[1] | oob_odd;
#pragma unroll
    for (int i = 0; i < kPairLoadsA; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, LDS_PTR(pa + (wave * kPairLoadsA + i) * 1024), 16,
                                               ((i & 1) ? va_odd : va_even) + static_cast<uint32_t>(i) * L.pitch_a, 0, 0, 0);
  };
  auto issue_pair_b = [&](const Pending& P, unsigned char* pb) {
#pragma unroll
    for (int i = 0; i < kPairLoadsB; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(P.rb, LDS_PTR(pb + (wave * kPairLoadsB + i) * 1024), 16,
                                               P.voff_b[i & 1] + static_cast<uint32_t>(i) * P.pitch_b, 0, 0, 0);
  };
  auto issue_a = [&](Loader& L, int ks, unsigned char* sa, Pending& P) {
    __amdgpu_buffer_rsrc_t ra;
    uint32_t oob = 0;
    if constexpr (TILED_IN) {
      // steps past K (ring padding) and blocks past the end of the matrix read as zero through the bounds check
      const bool real = ks * BK < L.K;
      P.rb = make_rsrc(L.b_cur, real ? L.b_left : 0u);
      // on to the next K step.  The byte counts are clamped for huge matrices; a clamped count is far above what
      // one step reads and stays as it is.
      L.b_cur += L.b_step;
      if (L.b_left != 0x7fffff00u) L.b_left = L.b_left > L.b_dec ? L.b_left - L.b_dec : 0u;
      if constexpr (AROWS) {  // token rows: the base advances along K and keeps the absolute end of the readable range
        const uint32_t adv = 2u * static_cast<uint32_t>(ks * BK);
        ra = make_rsrc(L.a_base + ks * BK, real && L.a_bytes > adv ? L.a_bytes - adv : 0u);
      } else {
        ra = make_rsrc(L.a_cur, real ? L.a_left : 0u);
        L.a_cur += L.a_step;
        if (L.a_left != 0x7fffff00u) L.a_left = L.a_left > L.a_dec ? L.a_left - L.a_dec : 0u;
      }
    } else {
      const int k0 = ks * BK;
      // advancing the base keeps the absolute end of the readable range, so rows past the matrix read as zero;
      // K chunks at or past the row end are pushed out of range per lane (this also zero-fills padding steps).
      // A K-major operand advances by whole rows of K instead, and its rows past K are past the end by themselves.
      const uint32_t adv = 2u * static_cast<uint32_t>(k0);
      if constexpr (KA) {
        ra = make_rsrc(L.a_cur, L.a_left);
        L.a_cur += L.a_step;
        L.a_left = k_major_left(L.a_left, L.a_dec);
      } else {
        ra = make_rsrc(L.a_base + k0, L.a_bytes > adv ? L.a_bytes - adv : 0u);
      }
      if constexpr (KB) {
        P.rb = make_rsrc(L.b_cur, L.b_left);
        L.b_cur += L.b_step;
        L.b_left = k_major_left(L.b_left, L.b_dec);
        P.pitch_b = L.pitch_b;
      } else {
        P.rb = make_rsrc(L.b_base + k0, L.b_bytes > adv ? L.b_bytes - adv : 0u);
      }
      const bool k_tail = k0 + BK > L.K;
      oob = (k_tail && k0 + ld_chunk * 8 >= L.K) ? 0x80000000u : 0u;
    }
    if constexpr (!kPB && !KB) {
#pragma unroll
      for (int i = 0; i < kLoadsB; ++i) P.voff_b[i] = L.voff_b[i] | oob;
    }
    if constexpr (!kPA) {  // (A in pairs: this call only prepares the step's B descriptor)
#pragma unroll
      for (int i = 0; i < kLoadsA; ++i)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, LDS_PTR(sa + (wave * kLoadRowsA + 16 * i) * kRowBytes), 16,
                                                 KA ? k_major_voff(i, BM, L.pitch_a, ks) : L.voff_a[i] | oob, 0, 0, 0);
    }
  };
  auto issue_b = [&](const Pending& P, unsigned char* sb, int step = 0) {
#pragma unroll
    for (int i = 0; i < kLoadsB; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(P.rb, LDS_PTR(sb + (wave * kLoadRowsB + 16 * i) * kRowBytes), 16,
                                               KB ? k_major_voff(i, BN, P.pitch_b, step) : P.voff_b[i], 0, 0, 0);
  };

  // Fused launch, consumer: the B half of K step `s` of a tile that has not started yet (s < kStages), leaving the
  // loader's running values alone.
  auto issue_b_ahead = [&](const Loader& L, int s, unsigned char* sb) {
    uint32_t left = L.b_left;
    for (int i = 0; i < s; ++i)
      if (left != 0x7fffff00u) left = left > L.b_dec ? left - L.b_dec : 0u;
    Pending P;
    P.rb = make_rsrc(L.b_cur + s * L.b_step, s * BK < L.K ? left : 0u);
#pragma unroll
    for (int i = 0; i < kLoadsB; ++i) P.voff_b[i] = L.voff_b[i];
    issue_b(P, sb);
  };
  // Fused launch, consumer, wavefronts that issue no loads: while the workgroup waits for its row block they pull
  // a share of the PRODUCERS' weights through this XCD's L2, so that weights which come from HBM (every layer of a
  // model has its own) are on their way before the producers' ring, four K steps deep, asks for them.  Workgroup c
  // of the consumers sits on the XCD of producer workgroup c and takes that producer's tile: the K steps
  // k = tm (mod kGroupM) of its gate and up column blocks (the producers of an XCD that share a column tile are the
  // kGroupM tile rows of a patch).  The loads are LDS-direct into the still unused first A slot and are waited for
  // before the barrier that ends the wait.  fs.warm_b is null when the host expects the weights in the caches.
  bool warm_pending = true;
  auto warm_producer_weights = [&]() {
    if constexpr (ROLE == 2) {
      const int total_g = tiles_m[0] * fs.need[0] + tiles_m[1] * fs.need[1];
      TileCoord tg;
      if (wg < total_g && map_tile(wg, total_g, tiles_m, fs.need, tg)) {
        const int e = tg.group;
        static_assert(TS::kWaves - kLoadWaves == 4, "two wavefronts per matrix, each every other K step of the share");
        const int q = wave - kLoadWaves;  // 0 .. 3: matrix q & 1, half q >> 1 of the share
        const __bf16* base = fs.warm_b[e][q & 1];
        if (base != nullptr) {
          const int ldb = fs.warm_ldb[e];
          const int nkb = fs.warm_k / kBlkCols;
          const int64_t bytes = (static_cast<int64_t>(nkb) * ldb) << 10;
          if (bytes < 0x7fffff00ll) {
            const __amdgpu_buffer_rsrc_t r = make_rsrc(base, static_cast<uint32_t>(bytes));
            unsigned char* dummy = slot_a(0) + q * 1024;
            constexpr int kGuBlocks = TS::BN / 2 / kBlkRows;  // row blocks of a gate/up column tile, per matrix
            const int blk0 = tg.tn * kGuBlocks;
            for (int ks = tg.tm % kGroupM + kGroupM * (q >> 1); ks < nkb; ks += 2 * kGroupM) {
#pragma unroll
              for (int i = 0; i < kGuBlocks; ++i) {
                const uint32_t off = static_cast<uint32_t>((static_cast<int64_t>(ks) * ldb + blk0 + i) << 10) + lane * 16;
                __builtin_amdgcn_raw_ptr_buffer_load_lds(r, LDS_PTR(dummy), 16, off, 0, 0, 0);
              }
            }
            __builtin_amdgcn_s_waitcnt(waitcnt_imm(0, 15));
          }
        }
      }
    }
  };
  int passed_before = 0;

  // A K step is one MFMA deep (16x16x32) and its FM x FN products go out in two halves around the step's barrier.
  // The operand with more blocks is the one that is cut: its first half and all of the other operand are needed for the
  // first half of the products, its second half only for the second.  So the cut operand has one register set (each
  // half is refilled while the other half's products run) and the other one has two, by the step's parity.
  // Why 16x16x32 and not 32x32x16 (the same operations per cycle): on normally distributed operands the chip holds a
  // clock that depends on what the instructions switch, and back-to-back MFMAs reach 1.96 PFLOP/s in this shape
  // against 1.77 in the other; 2.06 when each differs from the one before in one operand only (the serpentine below);
  // probe.hip measures all three.
  // 28160 + 1024 rows, before and after on one chip: gate/up 1.892 -> 1.757 ms (1.35 -> 1.45 PFLOP/s), down 0.950 ->
  // 0.887 ms; the row-major op at 28160 x 11008 x 2048: forward 0.967 -> 0.900 ms, dX 0.967 -> 0.917, dW (half the
  // tokens) 0.540 -> 0.511.  On all-zero operands, where the clock is the same for both shapes, neither is faster.
  // The operands go in as (B, A), so a lane's four accumulator registers are four consecutive COLUMNS of one row of C:
  // the epilogue packs them into 8 bytes without exchanging anything between lanes.
  constexpr bool kCutA = FM >= FN;
  // The FFN's small tile has the registers for all of two K steps' fragments and does not cut its products: k_step_whole.
  constexpr bool kWhole = TILED_IN && std::is_same_v<TS, SmallTile>;
  constexpr int kFirstReads = (kCutA ? FM / 2 : FM) * (KA ? 2 : 1) + (kCutA ? FN : FN / 2) * (KB ? 2 : 1);
  constexpr int kSecondReads = kCutA ? FM / 2 * (KA ? 2 : 1) : FN / 2 * (KB ? 2 : 1);
  f32x4 acc[FM][FN];
  bf16x8 fa[kCutA && !kWhole ? 1 : 2][FM], fb[kCutA || kWhole ? 2 : 1][FN];

  // K-major slot: K values [8 lq, +8) for the lane's column of 16-column block `blk` (counted from the wave's first
  // block): two transposing reads of four rows each.
  // (`step` keeps the compiler from holding the FM + FN addresses in registers across the loop, which it does not have:
  // one exclusive-or per read instead)
  auto read_k_major = [&](const unsigned char* slot, int lane_base, int row_bytes, int blk, int step) {
    asm("" : "+v"(lane_base) : "s"(step));
    const unsigned char* at = slot + (lane_base ^ (blk << 5));
    const bf16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(LDS_TR_PTR(at));
    const bf16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(LDS_TR_PTR(at + 4 * row_bytes));
    return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  };
  auto read_a = [&](const unsigned char* sa, int i, int step) {
    if constexpr (KA) return read_k_major(sa, tr_base_a, BM * 2, i, step);
    else if constexpr (kPA) return *reinterpret_cast<const bf16x8*>(sa + a_pair_off + i * 16 * 128);
    else return *reinterpret_cast<const bf16x8*>(sa + a_row_off + i * 16 * kRowBytes);
  };
  auto read_b = [&](const unsigned char* sb, int j, int step) {
    if constexpr (KB) return read_k_major(sb, tr_base_b, BN * 2, j, step);
    else if constexpr (kPB) return *reinterpret_cast<const bf16x8*>(sb + b_row(j) * 128 + pair_lane_off);
    else return *reinterpret_cast<const bf16x8*>(sb + b_row(j) * kRowBytes + b_lane_off);
  };
  // What the first half of the products of the step in slot (sa, sb), of parity `par`, needs, in first-use order ...
  auto read_first = [&](const unsigned char* sa, const unsigned char* sb, int par, int step) {
    if constexpr (kCutA) {
      fa[0][0] = read_a(sa, 0, step);
#pragma unroll
      for (int j = 0; j < FN; ++j) fb[par][j] = read_b(sb, j, step);
#pragma unroll
      for (int i = 1; i < FM / 2; ++i) fa[0][i] = read_a(sa, i, step);
    } else {
      fb[0][0] = read_b(sb, 0, step);
#pragma unroll
      for (int i = 0; i < FM; ++i) fa[par][i] = read_a(sa, i, step);
#pragma unroll
      for (int j = 1; j < FN / 2; ++j) fb[0][j] = read_b(sb, j, step);
    }
  };
  // ... and the second half's rest
  auto read_second = [&](const unsigned char* sa, const unsigned char* sb, int step) {
    if constexpr (kCutA) {
#pragma unroll
      for (int i = FM / 2; i < FM; ++i) fa[0][i] = read_a(sa, i, step);
    } else {
#pragma unroll
      for (int j = FN / 2; j < FN; ++j) fb[0][j] = read_b(sb, j, step);
    }
  };
  auto mma = [&](int half, int par) {
    if constexpr (kCutA) {
#pragma unroll
      for (int ii = 0; ii < FM / 2; ++ii)
#pragma unroll
        for (int jj = 0; jj < FN; ++jj) {
          const int i = half * (FM / 2) + ii, j = (ii & 1) ? FN - 1 - jj : jj;
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[par][j], fa[0][i], acc[i][j], 0, 0, 0);
        }
    } else {
#pragma unroll
      for (int jj = 0; jj < FN / 2; ++jj)
#pragma unroll
        for (int ii = 0; ii < FM; ++ii) {
          const int j = half * (FN / 2) + jj, i = (jj & 1) ? FM - 1 - ii : ii;
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[0][j], fa[par][i], acc[i][j], 0, 0, 0);
        }
    }
  };
  // Scheduling hints.  Before the barrier: the LDS reads of the step's second half and the B half of the previous
  // slot's refill go out among the first MFMAs of this half; the rest of them cover the read latency, so the wait in
  // front of the barrier finds the reads done.  After it: the loads of the refill are spread over the whole half, the
  // next slot's fragment reads over three quarters of it.  (Other shares of the MFMAs, a quarter to all of them, measure
  // within 1 % of these.)
  auto schedule_half = [&](auto n_reads, auto n_loads, auto n_read_carry, auto n_carry) {
    constexpr int kReads = decltype(n_reads)::value, kLoads = decltype(n_loads)::value;
    constexpr int kMfma = FM * FN / 2, kReadCarry = decltype(n_read_carry)::value, kCarry = decltype(n_carry)::value;  // MFMAs that carry reads / loads
#pragma unroll
    for (int m = 0; m < kMfma; ++m) {
      // the m-th MFMA is preceded by an even share of the reads and of the loads
      const int reads = m < kReadCarry ? (m + 1) * kReads / kReadCarry - m * kReads / kReadCarry : 0;
      const int loads = m < kCarry ? (m + 1) * kLoads / kCarry - m * kLoads / kCarry : 0;
#pragma unroll
      for (int q = 0; q < reads; ++q) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
#pragma unroll
      for (int q = 0; q < loads; ++q) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  constexpr int kHalfMfma = FM * FN / 2;
  auto schedule_before = [&](auto n_loads) {
    schedule_half(std::integral_constant<int, kSecondReads>{}, n_loads, std::integral_constant<int, kHalfMfma / 2>{}, std::integral_constant<int, kHalfMfma / 2>{});
  };
  auto schedule_after = [&](auto n_loads) {
    schedule_half(std::integral_constant<int, kFirstReads>{}, n_loads, std::integral_constant<int, kHalfMfma * 3 / 4>{}, std::integral_constant<int, kHalfMfma>{});
  };

  // One K step on slot S of the ring (step S of a ring round).  On entry the registers hold what the first half of its
  // products needs.  After the barrier every wave has finished reading this slot, so its refill with the K step kStages
  // ahead in the load stream (step `ld_ks` + S of tile `L`) starts at once: the A half here, the B half in the next
  // step's first half.  The next slot's data was issued kStages - 1 steps ago.
  // A wavefront that does not load runs the same step without the load instructions (and its counted wait passes
  // at once: it has no loads in flight).
  Pending pend;
  auto k_step_as = [&](auto with_loads, auto step_c, Loader& L, int ld_ks) {
    constexpr bool LD = decltype(with_loads)::value;
    constexpr int S = decltype(step_c)::value;
    read_second(slot_a(S), slot_b(S), ld_ks);
    if constexpr (LD) issue_b(pend, slot_b((S + kStages - 1) % kStages), ld_ks);
    mma(0, S & 1);
    schedule_before(std::integral_constant<int, LD ? kLoadsB : 0>{});
    // my LDS reads have returned; of my loads at most the kStages - 2 youngest K steps' worth are still in flight,
    // i.e. the next slot is complete
    __builtin_amdgcn_s_waitcnt(waitcnt_imm(LD ? (kStages - 2) * kLoadsPerStep : 63, 0));
    barrier_no_fence();
    if constexpr (LD) issue_a(L, ld_ks + S, slot_a(S), pend);
    read_first(slot_a((S + 1) % kStages), slot_b((S + 1) % kStages), (S + 1) & 1, ld_ks);
    mma(1, S & 1);
    schedule_after(std::integral_constant<int, LD ? kLoadsA : 0>{});
  };
  // The same step on paired slots (slots 0, 1 are pair 0, slots 2, 3 pair 1).  A pair is
  // free once its odd slot has been read, i.e. after the barrier of steps 1 and 3: its A refill (the K steps one ring
  // round ahead) goes out there, its B refill at the start of the following step, and everything must have landed
  // by the barrier two steps on, which is the only load still in flight then -- the counted wait becomes vmcnt(0) on
  // odd steps and none on even ones.
  auto k_step_pair = [&](auto with_loads, auto step_c, Loader& L, int ld_ks) {
    constexpr bool LD = decltype(with_loads)::value;
    constexpr int S = decltype(step_c)::value;
    constexpr bool kOdd = (S & 1) != 0;
    read_second(slot_a(S), slot_b(S), ld_ks);
    if constexpr (LD && !kOdd) issue_pair_b(pend, S == 0 ? s_pb1 : s_pb0);
    mma(0, S & 1);
    schedule_before(std::integral_constant<int, (LD && !kOdd) ? kPairLoadsB : 0>{});
    __builtin_amdgcn_s_waitcnt(waitcnt_imm((LD && kOdd) ? 0 : 63, 0));
    barrier_no_fence();
    if constexpr (LD && kOdd) issue_pair_a(L, ld_ks + (S == 1 ? 0 : 2), S == 1 ? s_pa0 : s_pa1, pend);
    read_first(slot_a((S + 1) % kStages), slot_b((S + 1) % kStages), (S + 1) & 1, ld_ks);
    mma(1, S & 1);
    schedule_after(std::integral_constant<int, (LD && kOdd) ? kPairLoadsA : 0>{});
  };
  // The same step with whole fragment sets: on entry set S & 1 holds all of slot S, every wavefront has read it, and slot
  // S + 1 is complete.  Slot S is refilled and slot S + 1 read into the other set while the products run, and one wait and
  // barrier end the step.  A step cut in two waits for the LDS twice, one after the other (the reads behind its first
  // products are held up by the wait for those products' operands), which shows where few CUs are busy and the memory is
  // quick: gate/up by itself at 512 rows (hidden 2048, expert 1024) 14.6 -> 13.8 us, down 10.1 -> 9.9, at 2048 rows 17.4 -> 17.0
  // and 12.2 -> 11.9; 36 layers, the block alone, 640 rows 1198 -> 1183 us.  The reads go out among the first half of the
  // products and the loads, at which a loading wavefront stalls, behind them, one at a time (all of them among the first
  // products: 14.4; among the last: 15.1; the reads among the first quarter 15.3, three quarters 14.6).
  auto read_whole = [&](const unsigned char* sa, const unsigned char* sb, int par, int step) {
    fb[par][0] = read_b(sb, 0, step);
#pragma unroll
    for (int i = 0; i < FM; ++i) fa[par][i] = read_a(sa, i, step);
#pragma unroll
    for (int j = 1; j < FN; ++j) fb[par][j] = read_b(sb, j, step);
  };
  auto k_step_whole = [&](auto with_loads, auto step_c, Loader& L, int ld_ks) {
    constexpr bool LD = decltype(with_loads)::value;
    constexpr int S = decltype(step_c)::value, kMfma = FM * FN, kReads = FM + FN;
    if constexpr (LD) {
      issue_a(L, ld_ks + S, slot_a(S), pend);
      issue_b(pend, slot_b(S), ld_ks);
    }
    read_whole(slot_a((S + 1) % kStages), slot_b((S + 1) % kStages), (S + 1) & 1, ld_ks);
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int ii = 0; ii < FM; ++ii) {
        const int i = (j & 1) ? FM - 1 - ii : ii;
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[S & 1][j], fa[S & 1][i], acc[i][j], 0, 0, 0);
      }
    constexpr unsigned kLoadBefore = 0x74;  // one load each before products 2, 4, 5 and 6 (of 0 .. 7)
    static_assert(!kWhole || (kMfma == 8 && kLoadsPerStep == 4), "the loads' places");
#pragma unroll
    for (int m = 0; m < kMfma; ++m) {
      const int reads = m < kMfma / 2 ? (m + 1) * kReads / (kMfma / 2) - m * kReads / (kMfma / 2) : 0;
#pragma unroll
      for (int q = 0; q < reads; ++q) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      if (LD && (kLoadBefore >> m & 1)) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
    // my reads of slot S + 1 have returned; slot S + 2 is complete (the loads of this step and the one before may be in flight)
    __builtin_amdgcn_s_waitcnt(waitcnt_imm(LD ? (kStages - 2) * kLoadsPerStep : 63, 0));
    barrier_no_fence();
  };
  // ... and with A alone in pairs (NN).  B keeps the slot-by-slot schedule of k_step_as (the refill of slot S - 1 at
  // the start of step S, its descriptor prepared after the barrier of step S - 1), A the pairs' (after the barrier of
  // odd steps).  In flight behind what the barrier of step S needs: the B refills of the two youngest steps, and on
  // even steps the A pair issued one step ago as well.
  auto k_step_mixed = [&](auto with_loads, auto step_c, Loader& L, int ld_ks) {
    constexpr bool LD = decltype(with_loads)::value;
    constexpr int S = decltype(step_c)::value;
    constexpr bool kOdd = (S & 1) != 0;
    read_second(slot_a(S), slot_b(S), ld_ks);
    if constexpr (LD) issue_b(pend, slot_b((S + kStages - 1) % kStages), ld_ks);
    mma(0, S & 1);
    schedule_before(std::integral_constant<int, LD ? kLoadsB : 0>{});
    __builtin_amdgcn_s_waitcnt(waitcnt_imm(LD ? (kOdd ? 2 * kLoadsB : 2 * kLoadsB + kPairLoadsA) : 63, 0));
    barrier_no_fence();
    if constexpr (LD) {
      issue_a(L, ld_ks + S, nullptr, pend);
      if constexpr (kOdd) issue_pair_a(L, ld_ks + S - 1, S == 1 ? s_pa0 : s_pa1, pend);
    }
    read_first(slot_a((S + 1) % kStages), slot_b((S + 1) % kStages), (S + 1) & 1, ld_ks);
    mma(1, S & 1);
    schedule_after(std::integral_constant<int, (LD && kOdd) ? kPairLoadsA : 0>{});
  };
  // ---- epilogue ------------------------------------------------------------------------------------------
  // Lane l of a 16x16 block holds row l % 16, columns 4 (l / 16) .. + 3.  Values are rounded to bf16, written to this
  // wave's staging area 8 bytes at a time, and read back as 16-byte lanes laid out the way the destination wants them.
  unsigned char* stage = s_out + wave * kStageBytes;

  // The row-major half of the epilogue.  `with_res`: the addend's form is one of its own, chosen once per tile -- with a
  // test at each of the addend's loads and uses the compiler sees the loads still in flight on paths around their use
  // and makes every wavefront wait for ALL of its loads at the head of the K loop, once per ring round.
  auto store_rows = [&](const Store& S, const int lane_e, auto with_res) {
    constexpr bool RES = decltype(with_res)::value;
    const int e16 = lane_e & 15, eq = lane_e >> 4;
    // wave output: FM row blocks of 16 rows x kOutCols columns, row-major, staged one row block at a time.  Row r of
    // the staging area keeps 16-byte chunk c in slot c ^ swz(r): both the 8-byte writes (16 rows x one chunk) and the
    // 16-byte reads (whole rows) then touch every bank once.
    constexpr int kOutCols = FN * 16;
    constexpr int kPitch = kOutCols * 2;
    static_assert(kStageBytes == 16 * kPitch && (kPitch == 128 || kPitch == 256), "staging holds one row block");
    constexpr int kLanesPerRow = kPitch / 16, kRowsPerStore = 64 / kLanesPerRow, kStores = 16 / kRowsPerStore;
    auto swz = [](int r) { return kPitch == 128 ? (r >> 1) & 7 : r & 15; };
    // a row is kPitch bytes = kLanesPerRow lanes; one store instruction writes kRowsPerStore rows
    const int rl = lane_e / kLanesPerRow, cc = lane_e % kLanesPerRow;
    const int col = wn * kOutCols + cc * 8;
    // What the stores need from memory is asked for ahead of the first of them: the row ids of the whole tile, and the addend's
    // chunks kAhead row blocks in front of their use.  (Asked for row block by row block, a tile of 256 rows waited for eight
    // memory latencies one after the other, twice over with row ids and an addend: q / k / v and o projections of 14592 rows with
    // the rotary table's loads a row block ahead as well 291.6 -> 283.9 us, four layers of 912 rows 627 -> 618; training and a
    // prefill of 29184 rows level.)  Three row blocks where the row ids take registers, two in the kernel with the
    // parts, which spills 24 bytes with three (56 with four): layers of 2049 to 3500 rows on device-side counts 0.6 % longer.
    // Rows past the tile's end read a row that is there.
    constexpr int kMost = ROLE == 3 ? 2 : (MODE == kDown ? 3 : 4), kAhead = FM < kMost ? FM : kMost;
    auto row_of = [&](int i, int q) { return (wm * FM + i) * 16 + q * kRowsPerStore + rl; };
    // (a wavefront's ids: a lane has those of rows lane, lane + 64, .. of its share, and hands them out)
    constexpr int kIds = MODE == kDown ? (FM * 16 + 63) / 64 : 1;
    int ids[kIds];
    if constexpr (MODE == kDown) {
#pragma unroll
      for (int r = 0; r < kIds; ++r) {
        const int row = wm * FM * 16 + 64 * r + lane_e;
        ids[r] = row < S.rows ? row : 0;
      }
      if (S.row_id != nullptr) {
#pragma unroll
        for (int r = 0; r < kIds; ++r) ids[r] = S.row_id[ids[r]];
      }
      // The ids are waited for here, whether or not this lane stores a row.  (A row block with nothing to store skips
      // the stores and with them the wait; the compiler then keeps the registers of the ids from being written again
      // before the loads are back, with a wait of its own in the first K step of every ring round, which drains the
      // ring: the one-launch layer of 260 .. 2048 rows took 28.3 us in place of 26.4 at 512 rows, hidden 2048, expert
      // 1024.)
#pragma unroll
      for (int r = 0; r < kIds; ++r) asm volatile("" : "+v"(ids[r]));
    }
    auto out_row = [&](int i, int q) {
      if constexpr (MODE == kDown) return __shfl(ids[(i * 16 + q * kRowsPerStore) / 64], (i * 16 + q * kRowsPerStore) % 64 + rl);
      else return row_of(i, q) < S.rows ? row_of(i, q) : 0;
    };
    u32x4 resv[RES ? kAhead : 1][kStores];
    auto load_res = [&](int i) {
#pragma unroll
      for (int q = 0; q < kStores; ++q) {
        resv[i % kAhead][q] = *reinterpret_cast<const u32x4*>(S.res + static_cast<int64_t>(out_row(i, q)) * S.ldc + (col < S.cols_left ? col : 0));
      }
    };
    if constexpr (RES) {
#pragma unroll
      for (int i = 0; i < kAhead; ++i) load_res(i);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int i = 0; i < FM; ++i) {
#pragma unroll
      for (int j = 0; j < FN; ++j)
        *reinterpret_cast<u32x2*>(stage + e16 * kPitch + (((2 * j + (eq >> 1)) ^ swz(e16)) << 4) + (eq & 1) * 8) =
            u32x2{pack_bf16x2(acc[i][j][0], acc[i][j][1]), pack_bf16x2(acc[i][j][2], acc[i][j][3])};
      __builtin_amdgcn_s_waitcnt(waitcnt_imm(63, 0));
#pragma unroll
      for (int q = 0; q < kStores; ++q) {
        const int srow = q * kRowsPerStore + rl;
        u32x4 v = *reinterpret_cast<const u32x4*>(stage + srow * kPitch + ((cc ^ swz(srow)) << 4));
        const int row = (wm * FM + i) * 16 + srow, to = MODE == kDown ? out_row(i, q) : row;
        if constexpr (RES) {  // bf16(y) + bf16(residual), summed in fp32 and rounded once, like the eager add
          asm volatile("" : "+v"(resv[i % kAhead][q]));  // (waited for whether or not this lane stores a row, like the ids)
#pragma unroll
          for (int w = 0; w < 4; ++w) {
            const float lo = __builtin_bit_cast(float, v[w] << 16) + __builtin_bit_cast(float, resv[i % kAhead][q][w] << 16);
            const float hi = __builtin_bit_cast(float, v[w] & 0xFFFF0000u) +
                             __builtin_bit_cast(float, resv[i % kAhead][q][w] & 0xFFFF0000u);
            v[w] = pack_bf16x2(lo, hi);
          }
        }
        if (row < S.rows && col < S.cols_left)
          *reinterpret_cast<u32x4*>(S.c_base + static_cast<int64_t>(to) * S.ldc + col) = v;
      }
      if constexpr (RES) {
        if (i + kAhead < FM) load_res(i + kAhead);
        __builtin_amdgcn_sched_barrier(0);
      }
      __builtin_amdgcn_s_waitcnt(waitcnt_imm(63, 0));
    }
  };

  auto epilogue = [&](const Store& S) {
    // The lane id is laundered through an empty asm so the address arithmetic is redone here each tile instead
    // of being hoisted out of the persistent loop and held in registers across the K loop.
    int lane_e = lane;
    asm volatile("" : "+v"(lane_e));
    const int e16 = lane_e & 15, eq = lane_e >> 4;
    if constexpr (SWIGLU) {
      // wave output: FM row blocks x kColBlocks column blocks of the tiled intermediate (16 x 32, 1 KiB each).  The
      // staging area holds blocks in their final layout (16-byte chunk c of row r in slot c ^ ((r >> 2) & 3)), so a
      // block is read back and stored as it lies; kRound row blocks go through it at a time.
      constexpr int kColBlocks = FN / 4;
      constexpr int kRound = kStageBytes / (kColBlocks * kBlkBytes);
      static_assert(FN % 4 == 0 && kRound >= 1 && FM % kRound == 0, "staging holds whole rounds of blocks");
      // what == 0: the intermediate h; 1 / 2: the gate / up projections themselves, when the caller keeps them
      const int n_what = p.keep[0] != nullptr ? 3 : 1;
      const int64_t keep_off[3] = {0, reinterpret_cast<unsigned char*>(p.keep[0]) - reinterpret_cast<unsigned char*>(p.g[0].c),
                                   reinterpret_cast<unsigned char*>(p.keep[1]) - reinterpret_cast<unsigned char*>(p.g[0].c)};
#pragma unroll
      for (int round = 0; round < FM / kRound; ++round) {
        for (int what = 0; what < n_what; ++what) {
#pragma unroll
          for (int ii = 0; ii < kRound; ++ii) {
            const int i = round * kRound + ii;
#pragma unroll
            for (int j = 0; j < FN / 2; ++j) {
              float h[4];
#pragma unroll
              for (int r = 0; r < 4; ++r) {
                const float gate = acc[i][j][r], up = acc[i][j + FN / 2][r];
                h[r] = what == 0 ? swiglu_bf16(gate, up) : (what == 1 ? gate : up);  // (rounded by the pack)
              }
              const int chunk = 2 * (j & 1) + (eq >> 1);  // of the 32-column block j / 2
              *reinterpret_cast<u32x2*>(stage + (ii * kColBlocks + j / 2) * kBlkBytes + e16 * 64 +
                                        ((chunk ^ ((e16 >> 2) & 3)) << 4) + (eq & 1) * 8) =
                  u32x2{pack_bf16x2(h[0], h[1]), pack_bf16x2(h[2], h[3])};
            }
          }
          __builtin_amdgcn_s_waitcnt(waitcnt_imm(63, 0));
#pragma unroll
          for (int rbl = 0; rbl < kRound; ++rbl) {
#pragma unroll
            for (int kbl = 0; kbl < kColBlocks; ++kbl) {
              const u32x4 v = *reinterpret_cast<const u32x4*>(stage + (rbl * kColBlocks + kbl) * kBlkBytes + lane_e * 16);
              const int row = (wm * FM + round * kRound + rbl) * 16;     // first row of the block inside the tile
              const int col = (wn * kColBlocks + kbl) * 32;              // first column of the block inside the tile
              // rows past the expert's last row are padding of the tiled matrix: harmless to write, never read
              if (col < S.cols_left) {
                unsigned char* dst = reinterpret_cast<unsigned char*>(S.c_base) + keep_off[what] +
                                     ((static_cast<int64_t>(col / kBlkCols) * S.ldc + row / kBlkRows) << 10);
                if constexpr (ROLE == 1) {
                  // fused launch: written through to memory (agent-scope store), so that the tile is visible to
                  // the other XCDs once the stores have completed, without a write-back of this XCD's L2
                  __builtin_amdgcn_raw_buffer_store_b128(v, make_rsrc(dst, kBlkBytes), lane_e * 16, 0, 16 /* sc1 */);
                } else {
                  *reinterpret_cast<u32x4*>(dst + lane_e * 16) = v;
                }
              }
            }
          }
          __builtin_amdgcn_s_waitcnt(waitcnt_imm(63, 0));  // staging is rewritten by the next round
        }
      }
    } else {
      if constexpr (MODE == kQkvRope || MODE == kQkvRopeFull) {
        // Bias and rotary embedding on the accumulators, before they are staged.  A wavefront's 128 columns are one
        // head; channel d of the head sits in block d / 16, so its rotation partner d +/- 64 is four blocks away in
        // the same lane and register.  Evaluated like eager bf16 code: the projection (with its bias) rounded once,
        // then q * cos + rotate_half(q) * sin with each product and the sum rounded (vl.py:771-772).
        static_assert(FN == 8, "a wavefront covers whole heads of 128 channels");
        const int col_w = S.col0 + wn * 128;  // first output column of this wavefront's head
        const bool live = wn * 128 < S.cols_left;
        u32x2 bias_v[FN];  // this lane's four columns of each block, bf16
#pragma unroll
        for (int j = 0; j < FN; ++j) bias_v[j] = u32x2{0u, 0u};
        if (p.bias != nullptr && live) {
          const uint16_t* b = reinterpret_cast<const uint16_t*>(p.bias) + col_w + 4 * eq;
          if ((reinterpret_cast<uintptr_t>(p.bias) & 7) == 0) {
#pragma unroll
            for (int j = 0; j < FN; ++j) bias_v[j] = *reinterpret_cast<const u32x2*>(b + j * 16);
          } else {
#pragma unroll
            for (int j = 0; j < FN; ++j)
              bias_v[j] = u32x2{b[j * 16] | static_cast<uint32_t>(b[j * 16 + 1]) << 16,
                                b[j * 16 + 2] | static_cast<uint32_t>(b[j * 16 + 3]) << 16};
          }
        }
        auto bias_of = [&](int j, int r) {
          return __uint_as_float((r & 1) ? (bias_v[j][r >> 1] & 0xffff0000u) : (bias_v[j][r >> 1] << 16));
        };
        const bool rotate = live && col_w < p.rope_cols;  // wave-uniform: q and k heads rotate, v heads do not
        constexpr int kWidth = MODE == kQkvRope ? 64 : 128;  // table entries per token: shared by d and d + 64, or one each
        // cos | sin of this lane's channels, four per load (the table need only be word-aligned), a row block ahead of their use
        // (the table with an entry per channel: ahead of their first use, there are no registers for two row blocks of it; and a
        // tile of two row blocks, where nothing is left to run ahead of and the fence only holds the loads back: 512 rows 22.4 ->
        // 22.1 us, together with the stores' own row numbers)
        constexpr int kCs = kWidth == 64 && FM > 2 ? 2 : 1;
        u32x4 cs[kCs][kWidth / 16];
        auto load_cs = [&](int i) {
          const int row = (wm * FM + i) * 16 + e16;
          const uint32_t* t = p.rope_table + static_cast<int64_t>(S.row0 + (row < S.rows ? row : 0)) * kWidth + 4 * eq;
#pragma unroll
          for (int j = 0; j < kWidth / 16; ++j) cs[i % kCs][j] = *reinterpret_cast<const u32x4_word*>(t + j * 16);
        };
        if (rotate && kCs > 1) load_cs(0);
#pragma unroll
        for (int i = 0; i < FM; ++i) {
          if (rotate && i + kCs - 1 < FM) load_cs(i + kCs - 1);
          if constexpr (kCs > 1) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int j = 0; j < 4; ++j) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const float lo = round_bf16(acc[i][j][r] + bias_of(j, r));
              const float hi = round_bf16(acc[i][j + 4][r] + bias_of(j + 4, r));
              if (rotate) {
                const uint32_t t_lo = cs[i % kCs][j][r], t_hi = cs[i % kCs][MODE == kQkvRope ? j : j + 4][r];
                const float c_lo = __uint_as_float(t_lo << 16), s_lo = __uint_as_float(t_lo & 0xffff0000u);
                const float c_hi = __uint_as_float(t_hi << 16), s_hi = __uint_as_float(t_hi & 0xffff0000u);
                acc[i][j][r] = round_bf16(lo * c_lo) - round_bf16(hi * s_lo);
                acc[i][j + 4][r] = round_bf16(hi * c_hi) + round_bf16(lo * s_hi);
              } else {
                acc[i][j][r] = lo;
                acc[i][j + 4][r] = hi;
              }
            }
          }
        }
      }
      if constexpr (MODE == kDown || MODE == kGeneric) {
        if (S.res != nullptr) {
          store_rows(S, lane_e, std::true_type{});
          return;
        }
      }
      store_rows(S, lane_e, std::false_type{});
    }
  };

  // Split contraction: leaves this part's sums in its slot and says whether it was the tile's last to do so; the sums of all
  // parts, in their order, are then in the accumulators.  The slots are written through to memory and counted once they are
  // there (like the fused launch's intermediate); nobody waits for anybody.
  auto last_part = [&](const Store& S) {
    if constexpr (ROLE == 3) {
      constexpr uint32_t kWaveBytes = FM * FN * 1024;
      const int parts = 1 << (S.split & 15), this_part = S.split >> 4 & 15, slot = S.split >> 8;
      auto sums_of = [&](int part) {
        return make_rsrc(reinterpret_cast<char*>(split.sums) + (static_cast<int64_t>(slot + part) * kWaves + wave) * kWaveBytes, kWaveBytes);
      };
      const __amdgpu_buffer_rsrc_t mine = sums_of(this_part);
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
          __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, acc[i][j]), mine, (i * FN + j) * 1024 + lane * 16, 0, 16 /* sc1 */);
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
      __builtin_amdgcn_s_waitcnt(waitcnt_imm(0, 0));
      __syncthreads();
      volatile int* const s_before = reinterpret_cast<volatile int*>(s_out);  // (the staging area is free between tiles)
      if (tid == 0) *s_before = __hip_atomic_fetch_add(split.count + slot, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __syncthreads();
      const bool last = __builtin_amdgcn_readfirstlane(*s_before) == parts - 1;
      __syncthreads();
      if (!last) return false;
      if (tid == 0) __hip_atomic_store(split.count + slot, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if constexpr (FM * FN > 16) {  // (two parts; no registers for a second set of sums)
        const __amdgpu_buffer_rsrc_t from = sums_of(1 - this_part);
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
          for (int j = 0; j < FN; ++j)
            acc[i][j] += __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(from, (i * FN + j) * 1024 + lane * 16, 0, 16 /* sc1 */));
        return true;
      }
      // (a row of blocks at a time: the sums of all of them at once, and the parts on their way, would take the registers that
      // a second workgroup on the CU needs)
#pragma unroll 1
      for (int i = 0; i < FM; ++i) {
        f32x4 own[FN], sum[FN];
#pragma unroll
        for (int j = 0; j < FN; ++j) own[j] = acc[FM - 1][j];
        for (int q = 0; q < parts; ++q) {
          const __amdgpu_buffer_rsrc_t from = sums_of(q);
#pragma unroll
          for (int j = 0; j < FN; ++j) {
            const f32x4 v = q == this_part ? own[j]
                : __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(from, ((FM - 1 - i) * FN + j) * 1024 + lane * 16, 0, 16 /* sc1 */));
            sum[j] = q == 0 ? v : sum[j] + v;
          }
        }
        // the rows of blocks move up by one, the finished one to the front: after FM turns each is in its place
#pragma unroll
        for (int r = FM - 1; r > 0; --r)
#pragma unroll
          for (int j = 0; j < FN; ++j) acc[r][j] = acc[r - 1][j];
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[0][j] = sum[j];
      }
    }
    return true;
  };

  // ---- persistent loop -------------------------------------------------------------------------------
  // The load stream runs kStages K steps ahead of the MFMAs and crosses tile boundaries: the last kStages steps
  // of a tile refill the ring with the first kStages steps of the next tile, so the pipeline never drains and
  // the next tile's data lands while this tile's results are stored.  After the last tile the stream continues
  // with an empty descriptor (every load out of range, nothing fetched), which keeps the in-flight accounting
  // of the waits uniform.
  int next_t = wg;
  auto next_tile = [&](TileCoord& tc) {
    bool have = false;
    if constexpr (kIsTail) {
      for (; next_t < pieces && !have; next_t += n_wg) {
        const int piece = next_t % (kSubM * kSubN);
        tile_coords(split_at + next_t / (kSubM * kSubN), big_m, big_n, tc);
        tc.tm = kSubM * tc.tm + piece / kSubN;
        tc.tn = kSubN * tc.tn + piece % kSubN;
        // pieces past a ragged last row / column of tiles are empty
        have = tc.tm < (tc.group ? tiles_m[1] : tiles_m[0]) && tc.tn < (tc.group ? tiles_n[1] : tiles_n[0]);
      }
      if (MODE != kDown && !have && next_t < pieces + strip_cols[0] + strip_cols[1]) {
        const int at = next_t - pieces;
        tc.group = at >= strip_cols[0] ? 1 : 0;
        tc.tm = kSubM * (tc.group ? big_m[1] : big_m[0]);
        tc.tn = tc.group ? at - strip_cols[0] : at;
        next_t += n_wg;
        have = true;
      }
      return have;
    }
    for (; next_t < padded && !have; next_t += n_wg) have = map_tile(next_t, total, tiles_m, tiles_n, tc);
    if constexpr (ROLE == 3) {
      tc.part = 0;
      const int cols = cols_of(tc.group);
      while (have && tc.tn >= cols) {  // (four parts at most)
        tc.tn -= cols;
        ++tc.part;
      }
    }
    return have;
  };
  TileCoord tc;
  bool have = next_tile(tc);
  if (!have) return;
  // The whole tile loop exists in two forms, with and without the load instructions; a wavefront picks its form
  // once (all of them the first, unless only some wavefronts load).
  auto run = [&](auto with_loads) {
    constexpr bool LD = decltype(with_loads)::value;
    Loader L;
    Store S;
    if constexpr (LD) setup_loader(tc, L);
    setup_store(tc, S);
    // Consumer of a fused launch: every tile starts from an empty ring.  The weights of the first ring slots are
    // fetched at once, the intermediate only after the row block's producers have finished; then the ring is as the
    // plain prologue leaves it, with every load landed.
    auto consumer_prologue = [&]() {
      static_assert(ROLE != 2 || kWhole, "the fused launch runs the FFN's small tile");
      if constexpr (LD) {
#pragma unroll
        for (int s = 0; s < kStages; ++s) issue_b_ahead(L, s, slot_b(s));
      }
      if constexpr (!LD && ASYM) {
        if (warm_pending) {
          warm_pending = false;
          warm_producer_weights();
        }
      }
      wait_for_count(fs, tid, S.row_block, fs.need[tc.group], passed_before);
      if constexpr (LD) {
#pragma unroll
        for (int s = 0; s < kStages; ++s) issue_a(L, s, slot_a(s), pend);
        __builtin_amdgcn_s_waitcnt(waitcnt_imm(0, 15));
      }
    };
    if constexpr (ROLE == 2) {
      consumer_prologue();
    } else if constexpr (LD && kPair) {
      issue_pair_a(L, 0, s_pa0, pend);
      issue_pair_b(pend, s_pb0);
      issue_pair_a(L, 2, s_pa1, pend);  // this pair's B half goes out in the first K step
      // pair 0 must be complete before its first fragments are read: pair 1's A half may remain in flight
      __builtin_amdgcn_s_waitcnt(waitcnt_imm(kPairLoadsA, 15));
    } else if constexpr (LD && kPairAOnly) {
      // in the order the steps keep: A's first pair, B's slots 0 and 1, A's second pair, B's slot 2 (slot 3 goes out in
      // the first K step)
      issue_a(L, 0, nullptr, pend);
      issue_pair_a(L, 0, s_pa0, pend);
      issue_b(pend, slot_b(0));
      issue_a(L, 1, nullptr, pend);
      issue_b(pend, slot_b(1));
      issue_pair_a(L, 2, s_pa1, pend);
      issue_a(L, 2, nullptr, pend);
      issue_b(pend, slot_b(2));
      issue_a(L, 3, nullptr, pend);
      // slot 0 of both operands must be complete: everything behind B's slot 0 may remain in flight
      __builtin_amdgcn_s_waitcnt(waitcnt_imm(2 * kLoadsB + kPairLoadsA, 15));
    } else if constexpr (LD) {
#pragma unroll
      for (int s = 0; s < kStages; ++s) {
        issue_a(L, s, slot_a(s), pend);
        if (kWhole || s + 1 < kStages) issue_b(pend, slot_b(s));  // (else the last slot's B half goes out in the first K step)
      }
      // slot 0 (and 1, where the first K step reads it) must be complete: the younger loads may remain in flight
      __builtin_amdgcn_s_waitcnt(waitcnt_imm((kStages - 2) * kLoadsPerStep + (kWhole ? 0 : kLoadsA), 15));
    }
    auto read_slot_0 = [&]() {
      if constexpr (kWhole) {
        barrier_no_fence();  // (the loads of slots 2 and 3 stay in flight)
        read_whole(slot_a(0), slot_b(0), 0, 0);
        __builtin_amdgcn_s_waitcnt(waitcnt_imm(63, 0));
        barrier_no_fence();  // slot 0 has been read: the first K step refills it
      } else {
        __syncthreads();
        read_first(slot_a(0), slot_b(0), 0, 0);
      }
    };
    read_slot_0();

    while (have) {
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[i][j][r] = 0.f;

      const Store done = S;
      const int nk = S.nk;
      for (int ks = 0; ks < nk; ks += kStages) {
        int ld_ks = ks + kStages;
        if (ld_ks == nk) {  // the loader moves on to the next tile (or to the empty descriptor)
          // (a consumer of a fused launch lets the ring run empty: its next tile has a wait of its own in front)
          have = ROLE == 2 ? false : next_tile(tc);
          if (have) {
            if constexpr (LD) setup_loader(tc, L);
            setup_store(tc, S);
          } else if constexpr (LD) {
            L.a_bytes = L.a_left = 0;
            L.b_bytes = L.b_left = 0;
            L.K = 0;
          }
          ld_ks = 0;
        }
        if constexpr (kPairAOnly) {
          k_step_mixed(with_loads, std::integral_constant<int, 0>{}, L, ld_ks);
          k_step_mixed(with_loads, std::integral_constant<int, 1>{}, L, ld_ks);
          k_step_mixed(with_loads, std::integral_constant<int, 2>{}, L, ld_ks);
          k_step_mixed(with_loads, std::integral_constant<int, 3>{}, L, ld_ks);
        } else if constexpr (kPair) {
          k_step_pair(with_loads, std::integral_constant<int, 0>{}, L, ld_ks);
          k_step_pair(with_loads, std::integral_constant<int, 1>{}, L, ld_ks);
          k_step_pair(with_loads, std::integral_constant<int, 2>{}, L, ld_ks);
          k_step_pair(with_loads, std::integral_constant<int, 3>{}, L, ld_ks);
        } else if constexpr (kWhole) {
          k_step_whole(with_loads, std::integral_constant<int, 0>{}, L, ld_ks);
          k_step_whole(with_loads, std::integral_constant<int, 1>{}, L, ld_ks);
          k_step_whole(with_loads, std::integral_constant<int, 2>{}, L, ld_ks);
          k_step_whole(with_loads, std::integral_constant<int, 3>{}, L, ld_ks);
        } else {
          k_step_as(with_loads, std::integral_constant<int, 0>{}, L, ld_ks);
          k_step_as(with_loads, std::integral_constant<int, 1>{}, L, ld_ks);
          k_step_as(with_loads, std::integral_constant<int, 2>{}, L, ld_ks);
          k_step_as(with_loads, std::integral_constant<int, 3>{}, L, ld_ks);
        }
      }
      if constexpr (ROLE == 3) {
        if ((done.split & 15) == 0 || last_part(done)) epilogue(done);
      } else {
        epilogue(done);
      }
      if constexpr (ROLE == 1) count_done(fs, tid, done.row_block);
      if constexpr (ROLE == 2) {
        clear_if_last(fs, tid, done.row_block, passed_before, fs.consumers);
        have = next_tile(tc);
        if (have) {  // (one tile per consumer unless the host's row counts were not the device's)
          if constexpr (LD) setup_loader(tc, L);
          setup_store(tc, S);
          consumer_prologue();
          read_slot_0();
        }
      }
    }
  };
  if constexpr (!ASYM) {
    run(std::true_type{});
  } else {
    if (loads) run(std::true_type{});
    else run(std::false_type{});
  }
#endif
}

template <int MODE, typename TS, bool KA = false, bool KB = false, int ROLE = 0>
__global__ __launch_bounds__(TS::kThreads, TS::kWgPerCu) void dual_gemm_kernel(Params p) {
  dual_gemm_body<MODE, TS, KA, KB, ROLE>(p, blockIdx.x, gridDim.x, FusedSync{});
}

// The down launch whose contraction may be in parts: the plain form or the parts', by the row counts.  Rows that are not cut
// pay for the question alone, and their launch's arguments and offsets stay scalar loads that are asked for together: 960 rows
// of the narrow expert on unknown counts 9.9 us, the plain kernel 9.7 (one body for both forms, asked in 64-bit numbers, 10.7;
// two bodies that share their arguments 10.4).
// (Bounded by the wavefronts per SIMD that TS is made for: with 147 registers, no second workgroup on a CU, 4050 rows on unknown
// counts, whose tiles stay whole, took 180 us in place of 161.)
template <typename TS>
__global__ __launch_bounds__(TS::kThreads, TS::kWgPerCu * TS::kWaves / 4) void down_split_kernel(Params p, DownSplit split) {
#if defined(__HIP_DEVICE_COMPILE__)
  // (every line of the launch's arguments, asked for at once, as the plain form does in front of its first wait)
  const int n_wg = gridDim.x;
  const ScalarInts offsets = (ScalarInts)p.offsets;
  asm volatile("" ::"s"(p.g[0].a), "s"(p.g[1].a), "s"(p.gate), "s"(split.rule.cus), "s"(split.rule.lg_most[1]), "s"(n_wg), "s"(offsets));
  const DownParts parts = split.rule.parts(offsets[1] - offsets[0], offsets[2] - offsets[1]);
  // Each form reads its arguments for itself (they are the launch's first): values that both want, held across the question,
  // are more than the scalar registers take.
  using Arguments = const __attribute__((address_space(4))) Params*;
  Arguments args = (Arguments)__builtin_amdgcn_kernarg_segment_ptr();
  const bool other_shape = parts.lg > 0 && parts.large != std::is_same_v<TS, BigTile>;
  if (other_shape && p.gate != 0) return;  // uniform: the other tile shape's launch does this problem
  if (parts.lg == 0 || other_shape) {  // (the only launch, made for row counts that are not the device's: its tiles stay whole)
    asm volatile("" : "+s"(args));
    dual_gemm_body<kDown, TS, false, false, 0>(*(const Params*)args, blockIdx.x, n_wg, FusedSync{});
  } else {
    asm volatile("" : "+s"(args));
    dual_gemm_body<kDown, TS, false, false, 3>(*(const Params*)args, blockIdx.x, n_wg, FusedSync{}, parts, split);
  }
#endif
}

// The few-rows form of the same launch (MODE: gate/up or down).
template <int MODE, int FM, int NB>
__global__ __launch_bounds__(kFewThreads, 2) void dual_gemm_few_rows_kernel(Params p) {
  constexpr int R = MODE == kGateUp ? 8 : 4;
  constexpr int RL = MODE == kGateUp && NB == 4 ? 4 : 0;
  few_rows_body<MODE, FM, NB, R, R - RL, RL, 0, false>(p, blockIdx.x, gridDim.x, FusedSync{});
}

// The fused FFN launch (see FusedSync): workgroups [0, producers) run the gate/up form on `pg`, the rest the down
// form on `pd`, both in the small tile shape.  `producers` is a multiple of 8, so a workgroup's index among its
// form's workgroups names the same XCD as its index in the grid.  (A workgroup that waits is a consumer, and what
// it waits for belongs to workgroups with lower indices, which never wait: whatever part of the grid is resident,
// the launch makes progress.)
// AROWS: the producers read the token rows (fs.x through fs.gather) in place of the K-tiled activations.
template <bool AROWS>
__global__ __launch_bounds__(SmallTile::kThreads, SmallTile::kWgPerCu) void ffn_fused_kernel(Params pg, Params pd, FusedSync fs, int producers) {
  const int wg = blockIdx.x, consumers = static_cast<int>(gridDim.x) - producers;
  if (wg < producers) dual_gemm_body<kGateUp, SmallTile, false, false, 1, AROWS>(pg, wg, producers, fs);
  else dual_gemm_body<kDown, SmallTile, false, false, 2>(pd, wg - producers, consumers, fs);
}

// The one launch in the few-rows form.  NB / NBC: the blocks of a gate/up and of a down tile.  WG: workgroups per CU that the
// registers are divided among.  ffn_few_rows_norm_kernel: with the RMSNorm in front of the FFN inside.
template <int FM, int NB, int NBC, int WG, bool AROWS, bool NORM>
__device__ __forceinline__ void ffn_few_rows(const Params& pg, const Params& pd, const FusedSync& fs, int producers) {
  const int wg = blockIdx.x, consumers = static_cast<int>(gridDim.x) - producers;
  if (wg < producers) {
    if constexpr (WG == 2) few_rows_body<kGateUp, FM, NB, NORM || NB == 2 ? 8 : 4, NB == 2 ? 8 : 4, 0, 1, AROWS, NORM>(pg, wg, producers, fs);
    else few_rows_body<kGateUp, FM, NB, 8, NB == 4 ? 4 : 8, NB == 4 ? 4 : 0, 1, AROWS, NORM>(pg, wg, producers, fs);
  } else {
    // (few_rows leaves at most 256 of the largest down tiles, and more than 192 from hidden 12320 on)
    few_rows_body<kDown, FM, NBC, 4, NBC == 8 ? 2 : 4, NBC == 8 ? 2 : 0, 2, false, false, NB, NBC != 8>(pd, wg - producers, consumers, fs);
  }
}
template <int FM, int NB, int NBC, int WG, bool AROWS>
__global__ __launch_bounds__(kFewThreads, 2 * WG) void ffn_few_rows_kernel(Params pg, Params pd, FusedSync fs, int producers) {
  ffn_few_rows<FM, NB, NBC, WG, AROWS, false>(pg, pd, fs, producers);
}
template <int FM, int NB, int NBC, int WG>
__global__ __launch_bounds__(kFewThreads, 2 * WG) void ffn_few_rows_norm_kernel(Params pg, Params pd, FusedSync fs, int producers) {
  ffn_few_rows<FM, NB, NBC, WG, true, true>(pg, pd, fs, producers);
}

// ---- plain FMA tiles: any transpose combination, any k --------------------------------------------------------
// Used for what the MFMA kernel does not take: K-major operands of 4 GiB or more.
__global__ __launch_bounds__(256) void dual_gemm_reference_layout_kernel(Params p, int trans_a, int trans_b) {
  __shared__ float s_a[32][33];
  __shared__ float s_b[32][33];
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;  // 32 x 8 threads, 32 x 32 output tile
  for (int e = 0; e < 2; ++e) {
    const Group& G = p.g[e];
    if (G.m <= 0 || G.n <= 0) continue;
    const int tiles_n = (G.n - 1) / 32 + 1, tiles_m = (G.m - 1) / 32 + 1;  // (m up to INT32_MAX)
    for (int64_t t = blockIdx.x; t < static_cast<int64_t>(tiles_m) * tiles_n; t += gridDim.x) {
      const int row0 = static_cast<int>(t / tiles_n) * 32, col0 = static_cast<int>(t % tiles_n) * 32;
      float acc[4] = {0.f, 0.f, 0.f, 0.f};
      for (int k0 = 0; k0 < G.k; k0 += 32) {
        for (int r = ty; r < 32; r += 8) {
          const int m = row0 + r, n = col0 + r, k = k0 + tx;
          float av = 0.f, bv = 0.f;
          if (k < G.k && m < G.m)
            av = static_cast<float>(trans_a ? G.a[static_cast<int64_t>(k) * G.lda + m] : G.a[static_cast<int64_t>(m) * G.lda + k]);
          if (k < G.k && n < G.n)
            bv = static_cast<float>(trans_b ? G.b0[static_cast<int64_t>(n) * G.ldb + k] : G.b0[static_cast<int64_t>(k) * G.ldb + n]);
          s_a[r][tx] = av;  // s_a[m][k]
          s_b[r][tx] = bv;  // s_b[n][k]
        }
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < 32; ++kk) {
          const float bv = s_b[tx][kk];
#pragma unroll
          for (int q = 0; q < 4; ++q) acc[q] = fmaf(s_a[ty + 8 * q][kk], bv, acc[q]);
        }
        __syncthreads();
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int m = row0 + ty + 8 * q, n = col0 + tx;
        if (m < G.m && n < G.n) {
          __bf16 v = static_cast<__bf16>(acc[q]);
          if (G.add != nullptr) v = static_cast<__bf16>(static_cast<float>(v) + static_cast<float>(G.add[static_cast<int64_t>(m) * G.ldc + n]));
          G.c[static_cast<int64_t>(m) * G.ldc + n] = v;
        }
      }
    }
  }
}

// Row-major [rows, cols] bf16 -> K-tiled (rows padded to 16 with zeros).  One thread per 16-byte chunk.
__global__ __launch_bounds__(256) void pack_tiled_kernel(const u32x4* __restrict__ src, unsigned char* __restrict__ dst,
                                                         int64_t rows, int64_t cols) {
  const int64_t chunks_per_row = cols / 8;
  const int64_t row_blocks = tiled_row_blocks(rows);
  const int64_t n = row_blocks * kBlkRows * chunks_per_row;
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    const int64_t row = i / chunks_per_row, c = i - row * chunks_per_row;
    const u32x4 v = row < rows ? src[i] : u32x4{0, 0, 0, 0};
    *reinterpret_cast<u32x4*>(dst + tiled_chunk_offset(row, c * 8, row_blocks)) = v;
  }
}

// Zeros for the output of an empty contraction (k == 0): a fill kernel rather than a memset node, so that the call
// stays capturable in a HIP graph like every other launch here.  n16 = number of 16-byte chunks.
__global__ __launch_bounds__(256) void zero_fill_kernel(u32x4* __restrict__ dst, int64_t n16) {
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n16;
       i += static_cast<int64_t>(gridDim.x) * blockDim.x)
    dst[i] = u32x4{0, 0, 0, 0};
}

// k_in_rows: both operands are stored with K as the slow dimension, so K needs no alignment
int check_dims(const char* who, int64_t m, int64_t n, int64_t k, bool k_in_rows = false) {
  if (m < 0 || n < 0 || k < 0) return fail(WX_ERR_INVALID_ARGUMENT, "%s: negative dimension", who);
  if (m > INT32_MAX || n > INT32_MAX || k > INT32_MAX) return fail(WX_ERR_UNSUPPORTED, "%s: dimension exceeds int32", who);
  if (n % 8 != 0 || (k % 8 != 0 && !k_in_rows))
    return fail(WX_ERR_UNSUPPORTED, "%s: n (%lld) and k (%lld) must be multiples of 8", who, static_cast<long long>(n),
                static_cast<long long>(k));
  // 256 rows of one operand must stay addressable through a 31-bit buffer offset
  if (k * 2 * 256 >= (1ll << 31) || n * 2 * 256 >= (1ll << 31)) return fail(WX_ERR_UNSUPPORTED, "%s: row too long", who);
  // the tile list is indexed with 32-bit integers
  if (((m + SmallTile::BM - 1) / SmallTile::BM) * ((n + SmallTile::BN / 2 - 1) / (SmallTile::BN / 2)) >= (1ll << 30))
    return fail(WX_ERR_UNSUPPORTED, "%s: too many tiles", who);
  return WX_OK;
}

int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

// The problem has between `tiles_lo` and `tiles_hi` 256 x 256 tiles (equal when the host knows the row counts).
// When they would occupy at most half of the CUs, the 128 x 128 tile gives four times as many workgroups to spread
// over the chip.  If the bounds fall on both sides of that threshold the choice is made on the device: both
// shapes are launched and the one on the wrong side returns immediately.
// tiles_by_expert: the host's exact 256 x 256 tile counts per expert, or null when only the device knows the row
// split (the bounds are then on the plain sum of the tiles; where they straddle the threshold and the device
// chooses, it chooses by shape_deciding_tiles like the host would).  A launch of large tiles uses the tail split: a
// second launch with 128 x 128 tiles takes the ragged last round when that pays (the row-major op, whose sizes the
// host knows, decides it on the host); when the host cannot tell, both launches are made and the device decides (the
// second returns at once if there is nothing to split).
// few: the few-rows form takes the problem; its number of rows, or 0.
// parts: the down launch's contraction may be in parts (PartsRule), with this scratch.
// rows: with tiles_by_expert, the rows of each expert (0 for one without columns), for the plan with strips (always for kGeneric).
template <int MODE, bool KA = false, bool KB = false>
int launch_mfma(Params p, int64_t tiles_lo, int64_t tiles_hi, hipStream_t s, const char* who,
                const int64_t* tiles_by_expert = nullptr, int64_t few = 0, const DownSplit* parts = nullptr,
                const int64_t* rows = nullptr) {
  const int cus = device_cu_count();
  const int threshold = cus / 2;
  if constexpr (MODE == kGateUp || MODE == kDown) {
    if (few > 0) {
      p.gate = p.split = 0;
      if (few <= 64) hipLaunchKernelGGL((dual_gemm_few_rows_kernel<MODE, 1, 2>), dim3(cus), dim3(kFewThreads), 0, s, p);
      else hipLaunchKernelGGL((dual_gemm_few_rows_kernel<MODE, 2, 4>), dim3(cus), dim3(kFewThreads), 0, s, p);
      return check_launch(who);
    }
  }
  bool small = tiles_lo <= threshold, big = tiles_hi > threshold;
  if (tiles_by_expert != nullptr) {  // the host knows the split: the count that decides is shape_deciding_tiles'
    small = shape_deciding_tiles(tiles_by_expert[0], tiles_by_expert[1], p.g[0].k, p.g[1].k) <= threshold;
    big = !small;
  } else if (!small && tiles_lo <= cus && (2ll * p.g[0].k <= p.g[1].k || 2ll * p.g[1].k <= p.g[0].k)) {
    // at most one round of large tiles, and one expert's tiles may not count: the device has to choose
    small = true;
  }
  if (MODE == kDown && parts != nullptr) {  // parts of large tiles, if the tiles that count can be enough for them
    const bool one_counts = 2ll * p.g[0].k <= p.g[1].k || 2ll * p.g[1].k <= p.g[0].k;
    if ((parts->rule.lg_most[0] > 1 || parts->rule.lg_most[1] > 1) && 4 * (one_counts ? tiles_lo : tiles_hi) > cus) big = true;
  }
  p.gate_tiles = threshold;
  p.split = 0;
  p.split_cus = cus;
  if (small) {
    p.gate = big ? 1 : 0;
    if (MODE == kDown && parts != nullptr)
      hipLaunchKernelGGL(down_split_kernel<SmallTile>, dim3(cus * SmallTile::kWgPerCu), dim3(SmallTile::kThreads), 0, s, p, *parts);
    else
      hipLaunchKernelGGL((dual_gemm_kernel<MODE, SmallTile, KA, KB>), dim3(cus * SmallTile::kWgPerCu), dim3(SmallTile::kThreads), 0, s, p);
  }
  if (big) {
    p.gate = small ? 2 : 0;
    using Big = BigTileFor<MODE>;
    static_assert(Big::kWgPerCu == 1, "the split counts one large tile per CU and round");
    bool split = (MODE != kGeneric || tiles_by_expert != nullptr) && tiles_hi > cus;
    if (split && tiles_by_expert != nullptr) {
      const int64_t all = tiles_by_expert[0] + tiles_by_expert[1];
      if (all >= INT32_MAX) {
        split = false;
      } else if (rows != nullptr) {
        auto cols = [&](int e) { return rows[e] > 0 ? static_cast<int>(tiles_by_expert[e] / ceil_div(rows[e], BigTile::BM)) : 0; };
        const TailPlan plan = tail_plan(static_cast<int>(rows[0]), static_cast<int>(rows[1]), cols(0), cols(1), p.g[0].k, p.g[1].k, cus, true, MODE == kGateUp ? kTailLongTiled : kTailLongRows);
        split = plan.split;
        if (MODE == kGeneric) p.plan = plan;
      } else {
        split = tail_split_point(static_cast<int>(tiles_by_expert[0]), static_cast<int>(tiles_by_expert[1]), p.g[0].k, p.g[1].k, cus) != all;
      }
    }
    p.split = split ? 1 : 0;
    if (MODE == kDown && parts != nullptr)
      hipLaunchKernelGGL(down_split_kernel<BigTile>, dim3(cus), dim3(BigTile::kThreads), 0, s, p, *parts);
    else
      hipLaunchKernelGGL((dual_gemm_kernel<MODE, Big, KA, KB>), dim3(cus), dim3(Big::kThreads), 0, s, p);
    if (split)
      hipLaunchKernelGGL((dual_gemm_kernel<MODE, TailTile, KA, KB, 4>), dim3(cus * TailTile::kWgPerCu), dim3(TailTile::kThreads), 0, s, p);
  }
  return check_launch(who);
}

}  // namespace
}  // namespace wx

using namespace wx;

namespace {
int dual_gemm_impl(const void* in0, const void* in1, const void* w0, const void* w1, void* out0, void* out1,
                   const void* add0, const void* add1, int64_t m0, int64_t n0, int64_t k0, int64_t m1, int64_t n1,
                   int64_t k1, int trans_a, int trans_b, wx_stream_t stream);
}

extern "C" int wx_dual_gemm(const void* in0, const void* in1, const void* w0, const void* w1, void* out0, void* out1,
                            int64_t m0, int64_t n0, int64_t k0, int64_t m1, int64_t n1, int64_t k1, int trans_a,
                            int trans_b, wx_stream_t stream) {
  return dual_gemm_impl(in0, in1, w0, w1, out0, out1, nullptr, nullptr, m0, n0, k0, m1, n1, k1, trans_a, trans_b, stream);
}

extern "C" int wx_dual_gemm_add(const void* in0, const void* in1, const void* w0, const void* w1, void* out0,
                                void* out1, const void* add0, const void* add1, int64_t m0, int64_t n0, int64_t k0,
                                int64_t m1, int64_t n1, int64_t k1, int trans_a, int trans_b, wx_stream_t stream) {
  if ((reinterpret_cast<uintptr_t>(add0) | reinterpret_cast<uintptr_t>(add1)) & 15)
    return fail(WX_ERR_INVALID_ARGUMENT, "wx_dual_gemm_add: buffers must be 16-byte aligned");
  return dual_gemm_impl(in0, in1, w0, w1, out0, out1, add0, add1, m0, n0, k0, m1, n1, k1, trans_a, trans_b, stream);
}

namespace {
int dual_gemm_impl(const void* in0, const void* in1, const void* w0, const void* w1, void* out0, void* out1,
                   const void* add0, const void* add1, int64_t m0, int64_t n0, int64_t k0, int64_t m1, int64_t n1,
                   int64_t k1, int trans_a, int trans_b, wx_stream_t stream) {
  const void* adds[2] = {add0, add1};
  gemm_path_reset();
  const bool k_in_rows = trans_a && !trans_b;  // A [k, m] and B [k, n]
  if (int rc = check_dims("wx_dual_gemm", m0, n0, k0, k_in_rows)) return rc;
  if (int rc = check_dims("wx_dual_gemm", m1, n1, k1, k_in_rows)) return rc;
  const void* ptrs[2][3] = {{in0, w0, out0}, {in1, w1, out1}};
  const int64_t dims[2][3] = {{m0, n0, k0}, {m1, n1, k1}};
  Params p{};
  for (int e = 0; e < 2; ++e) {
    const int64_t m = dims[e][0], n = dims[e][1], k = dims[e][2];
    if (m > 0 && n > 0 && (!ptrs[e][2] || (k > 0 && (!ptrs[e][0] || !ptrs[e][1]))))
      return fail(WX_ERR_INVALID_ARGUMENT, "wx_dual_gemm: null pointer for expert %d", e);
    for (int q = 0; q < 3; ++q)
      if (reinterpret_cast<uintptr_t>(ptrs[e][q]) & 15)
        return fail(WX_ERR_INVALID_ARGUMENT, "wx_dual_gemm: buffers must be 16-byte aligned");
    if (trans_a && m % 8 != 0) return fail(WX_ERR_UNSUPPORTED, "wx_dual_gemm: trans_a needs m to be a multiple of 8");
    Group& g = p.g[e];
    g.a = static_cast<const __bf16*>(ptrs[e][0]);
    g.b0 = static_cast<const __bf16*>(ptrs[e][1]);
    g.b1 = nullptr;
    g.c = static_cast<__bf16*>(const_cast<void*>(ptrs[e][2]));
    g.m = static_cast<int>(m); g.n = static_cast<int>(n); g.k = static_cast<int>(k);
    g.lda = static_cast<int>(trans_a ? m : k);
    g.ldb = static_cast<int>(trans_b ? k : n);
    g.ldc = static_cast<int>(n);
    g.a_row0 = 0;
    g.add = static_cast<const __bf16*>(adds[e]);
  }
  p.offsets = nullptr;
  if ((m0 == 0 || n0 == 0) && (m1 == 0 || n1 == 0)) return WX_OK;
  hipStream_t s = as_stream(stream);
  // an empty contraction (k == 0) has zeros as its result: a fill launch writes them and the group leaves the
  // problem, so the other expert still runs on the MFMA kernel (a training batch without action tokens has k == 0
  // in the action expert's weight gradients next to the VL expert's full-size ones)
  for (int e = 0; e < 2; ++e) {
    const int64_t m = dims[e][0], n = dims[e][1];
    if (dims[e][2] != 0 || m <= 0 || n <= 0) continue;
    if (adds[e] != nullptr) {  // 0 + addend
      if (adds[e] != ptrs[e][2] &&
          hipMemcpyAsync(const_cast<void*>(ptrs[e][2]), adds[e], static_cast<size_t>(m) * n * 2, hipMemcpyDeviceToDevice, s) != hipSuccess)
        return fail(WX_ERR_LAUNCH, "wx_dual_gemm_add: copy of the addend failed");
      gemm_path_note(WX_GEMM_PATH_ADD_COPY);
      p.g[e].m = 0;
      continue;
    }
    const int64_t n16 = m * n / 8;  // n is a multiple of 8 and the buffer 16-byte aligned
    const int64_t want = (n16 + 255) / 256, cap = static_cast<int64_t>(device_cu_count()) * 8;
    hipLaunchKernelGGL(zero_fill_kernel, dim3(static_cast<unsigned>(want < cap ? want : cap)), dim3(256), 0, s,
                       static_cast<u32x4*>(const_cast<void*>(ptrs[e][2])), n16);
    if (int rc = check_launch("zero_fill_kernel")) return rc;
    gemm_path_note(WX_GEMM_PATH_ZERO_FILL);
    p.g[e].m = 0;
  }
  if ((p.g[0].m == 0 || n0 == 0) && (p.g[1].m == 0 || n1 == 0)) return WX_OK;
  const int64_t mm0 = p.g[0].m, mm1 = p.g[1].m;  // row counts left after the empty contractions are done
  // K-major operands (A stored [k, m], B stored [k, n]) advance by whole rows of K through 32-bit byte counts
  bool fits = true;
  for (int e = 0; e < 2; ++e) {
    if (p.g[e].m == 0 || p.g[e].n == 0) continue;
    if (trans_a && !k_major_fits(dims[e][2], dims[e][0])) fits = false;
    if (!trans_b && !k_major_fits(dims[e][2], dims[e][1])) fits = false;
  }
  if (fits) {
    const int64_t tiles = ceil_div(mm0, BigTile::BM) * ceil_div(n0, BigTile::BN) + ceil_div(mm1, BigTile::BM) * ceil_div(n1, BigTile::BN);
    const char* who = "dual_gemm_kernel<generic>";
    gemm_path_note(WX_GEMM_PATH_MFMA);
    // (the host knows both problems' sizes: it settles the tile shape and the split of a ragged last round itself)
    const int64_t by_expert[2] = {ceil_div(mm0, BigTile::BM) * ceil_div(n0, BigTile::BN),
                                  ceil_div(mm1, BigTile::BM) * ceil_div(n1, BigTile::BN)};
    const int64_t by_rows[2] = {n0 > 0 ? mm0 : 0, n1 > 0 ? mm1 : 0};
    if (!trans_a && trans_b) return launch_mfma<kGeneric, false, false>(p, tiles, tiles, s, who, by_expert, 0, nullptr, by_rows);
    if (!trans_a && !trans_b) return launch_mfma<kGeneric, false, true>(p, tiles, tiles, s, who, by_expert, 0, nullptr, by_rows);
    if (trans_a && trans_b) return launch_mfma<kGeneric, true, false>(p, tiles, tiles, s, who, by_expert, 0, nullptr, by_rows);
    return launch_mfma<kGeneric, true, true>(p, tiles, tiles, s, who, by_expert, 0, nullptr, by_rows);
  }
  gemm_path_note(WX_GEMM_PATH_FMA);
  hipLaunchKernelGGL(dual_gemm_reference_layout_kernel, dim3(device_cu_count() * 4), dim3(256), 0, s, p, trans_a, trans_b);
  return check_launch("dual_gemm_reference_layout_kernel");
}
}  // namespace

extern "C" int wx_qkv_rope_proj(const void* x, const void* weight, const void* bias, const uint32_t* rope_table,
                                int table_width, void* out, int64_t num_tokens, int64_t hidden, int n_q_heads,
                                int n_kv_heads, int head_dim, wx_stream_t stream) {
  const char* who = "wx_qkv_rope_proj";
  if (n_q_heads < 0 || n_kv_heads < 0) return fail(WX_ERR_INVALID_ARGUMENT, "%s: negative head count", who);
  if (head_dim != 128)
    return fail(WX_ERR_UNSUPPORTED, "%s: head_dim %d; the epilogue rotates heads of 128 channels", who, head_dim);
  if (table_width != head_dim / 2 && table_width != head_dim)
    return fail(WX_ERR_INVALID_ARGUMENT, "%s: table_width %d must be %d (channels d and d + %d share an entry) or %d", who,
                table_width, head_dim / 2, head_dim / 2, head_dim);
  const int64_t n = static_cast<int64_t>(n_q_heads + 2 * n_kv_heads) * head_dim;
  if (int rc = check_dims(who, num_tokens, n, hidden)) return rc;
  if (num_tokens == 0 || n == 0) return WX_OK;
  if (hidden == 0) return fail(WX_ERR_UNSUPPORTED, "%s: hidden must be positive", who);
  if (!x || !weight || !out || !rope_table) return fail(WX_ERR_INVALID_ARGUMENT, "%s: null pointer", who);
  if ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(weight) | reinterpret_cast<uintptr_t>(out)) & 15)
    return fail(WX_ERR_INVALID_ARGUMENT, "%s: buffers must be 16-byte aligned", who);
  if ((reinterpret_cast<uintptr_t>(bias) & 1) || (reinterpret_cast<uintptr_t>(rope_table) & 3))
    return fail(WX_ERR_INVALID_ARGUMENT, "%s: misaligned bias or table", who);
  Params p{};
  Group& g = p.g[0];
  g.a = static_cast<const __bf16*>(x);
  g.b0 = static_cast<const __bf16*>(weight);
  g.c = static_cast<__bf16*>(out);
  g.m = static_cast<int>(num_tokens); g.n = static_cast<int>(n); g.k = static_cast<int>(hidden);
  g.lda = g.ldb = static_cast<int>(hidden);
  g.ldc = static_cast<int>(n);
  p.bias = static_cast<const __bf16*>(bias);
  p.rope_table = rope_table;
  p.rope_cols = (n_q_heads + n_kv_heads) * head_dim;
  p.rope_width = table_width;
  // Tiles whose wavefronts cover whole heads only (a 64-column wave tile would split a rotation pair): the large
  // tile, and for a ragged last round (see tail_plan) a second launch of 128 x 128 tiles with 32 x 128 wave tiles
  using Tile = BigTileFor<kQkvRope>;
  using Tail = TailTileFor<kQkvRope>;
  const int cus = device_cu_count();
  const int64_t tiles = ceil_div(num_tokens, Tile::BM) * ceil_div(n, Tile::BN);
  // Too few large tiles for half of the CUs (a denoise step, a short prefill): 128 x 128 tiles alone, as in launch_mfma.
  // The table, this launch and the o projection at n 2560, k 2048: 32 rows 66 -> 45 us, 1024 rows 70 -> 48, 2048 rows
  // 73 -> 63, 3072 rows 83 -> 76; one more row of large tiles is past the line.
  const bool small = tiles <= cus / 2;
  p.plan = TailPlan{};
  if (!small && tiles < INT32_MAX) p.plan = tail_plan(g.m, 0, static_cast<int>(ceil_div(g.n, Tile::BN)), 0, g.k, 0, cus, true, kTailLongRows);
  const bool split = p.plan.split;
  p.split = split ? 1 : 0;
  p.split_cus = cus;
  hipStream_t s = as_stream(stream);
  auto launch = [&](auto large, auto alone, auto second) {
    if (small) hipLaunchKernelGGL(alone, dim3(cus * Tail::kWgPerCu), dim3(Tail::kThreads), 0, s, p);
    else hipLaunchKernelGGL(large, dim3(cus), dim3(Tile::kThreads), 0, s, p);
    if (split) hipLaunchKernelGGL(second, dim3(cus * Tail::kWgPerCu), dim3(Tail::kThreads), 0, s, p);
  };
  if (table_width == head_dim)
    launch(dual_gemm_kernel<kQkvRopeFull, Tile>, dual_gemm_kernel<kQkvRopeFull, Tail>, dual_gemm_kernel<kQkvRopeFull, Tail, false, false, 4>);
  else
    launch(dual_gemm_kernel<kQkvRope, Tile>, dual_gemm_kernel<kQkvRope, Tail>, dual_gemm_kernel<kQkvRope, Tail, false, false, 4>);
  return check_launch("dual_gemm_kernel<qkv_rope>");
}

extern "C" size_t wx_tiled_bytes(int64_t rows, int64_t cols) {
  if (rows < 0 || cols < 0) return 0;
  return static_cast<size_t>(tiled_bytes(rows, (cols + kBlkCols - 1) / kBlkCols * kBlkCols));
}

extern "C" int64_t wx_padded_sorted_rows(int64_t rows) { return rows < 0 ? 0 : padded_sorted_rows(rows); }

extern "C" int wx_pack_tiled(const void* src, void* dst, int64_t rows, int64_t cols, wx_stream_t stream) {
  if (rows < 0 || cols < 0) return fail(WX_ERR_INVALID_ARGUMENT, "wx_pack_tiled: negative size");
  if (cols % kBlkCols != 0)
    return fail(WX_ERR_UNSUPPORTED, "wx_pack_tiled: cols (%lld) must be a multiple of 32", static_cast<long long>(cols));
  if (rows == 0 || cols == 0) return WX_OK;
  if (!src || !dst) return fail(WX_ERR_INVALID_ARGUMENT, "wx_pack_tiled: null pointer");
  if ((reinterpret_cast<uintptr_t>(src) | reinterpret_cast<uintptr_t>(dst)) & 15)
    return fail(WX_ERR_INVALID_ARGUMENT, "wx_pack_tiled: buffers must be 16-byte aligned");
  const int64_t chunks = tiled_row_blocks(rows) * kBlkRows * (cols / 8);
  const int64_t want = (chunks + 255) / 256;
  const int64_t cap = static_cast<int64_t>(device_cu_count()) * 16;
  hipLaunchKernelGGL(pack_tiled_kernel, dim3(static_cast<unsigned>(want < cap ? want : cap)), dim3(256), 0,
                     as_stream(stream), static_cast<const u32x4*>(src), static_cast<unsigned char*>(dst), rows, cols);
  return check_launch("pack_tiled_kernel");
}

namespace {

struct FfnArgs {
  const void *x, *gate[2], *up[2], *down[2];
  void *out, *hmid;
  const int64_t* host_rows;  // optional: rows of each expert as the caller knows them on the host
  const int32_t* offsets;
  int64_t rows, hidden, inter[2];
  const int32_t* out_row_id = nullptr;  // optional: sorted row r of the result goes to row out_row_id[r] of `out`
  void *keep_gate = nullptr, *keep_up = nullptr;  // optional: the gate / up projections, K-tiled like hmid
  const void* residual = nullptr;  // optional (with out_row_id): rows added to the result, laid out like `out`
  const void* norm_weight = nullptr;  // optional (with x_rows): the rows pass through an RMSNorm first; few rows only
  float norm_eps = 0.f;
  const void* x_rows = nullptr;    // optional: the activations in token order; `x` is then built by the fused launch
  void* split_scratch = nullptr;   // optional: wx_ffn_split_scratch_bytes() for the down launch's parts
};

int check_ffn(const char* who, const FfnArgs& a, bool need_gate_up, bool need_down) {
  if (int rc = check_dims(who, a.rows, a.inter[0], a.hidden)) return rc;
  if (int rc = check_dims(who, a.rows, a.hidden, a.inter[1])) return rc;
  if (a.hidden % kBlkCols != 0 || a.inter[0] % kBlkCols != 0 || a.inter[1] % kBlkCols != 0)
    return fail(WX_ERR_UNSUPPORTED, "%s: hidden and intermediate sizes must be multiples of 32", who);
  if (a.host_rows != nullptr && (a.host_rows[0] < 0 || a.host_rows[1] < 0 || a.host_rows[0] + a.host_rows[1] != a.rows))
    return fail(WX_ERR_INVALID_ARGUMENT, "%s: host_rows_per_expert must be non-negative and sum to num_rows", who);
  if (a.hidden == 0 || a.inter[0] == 0 || a.inter[1] == 0)
    return fail(WX_ERR_UNSUPPORTED, "%s: hidden and both intermediate sizes must be positive", who);
  if (a.rows == 0) return WX_OK;
  if (!a.offsets || !a.hmid || (need_gate_up && !a.x) || (need_down && !a.out))
    return fail(WX_ERR_INVALID_ARGUMENT, "%s: null pointer", who);
  for (int e = 0; e < 2; ++e) {
    if (a.inter[e] == 0) continue;
    if ((need_gate_up && (!a.gate[e] || !a.up[e])) || (need_down && !a.down[e]))
      return fail(WX_ERR_INVALID_ARGUMENT, "%s: null weight pointer for expert %d", who, e);
  }
  const int64_t max_inter = a.inter[0] > a.inter[1] ? a.inter[0] : a.inter[1];
  if (padded_sorted_rows(a.rows) * max_inter * 2 >= (1ll << 40))
    return fail(WX_ERR_UNSUPPORTED, "%s: intermediate too large", who);
  return WX_OK;
}

// hmid_e = silu(x_e @ gate_e^T) * (x_e @ up_e^T), K-tiled per expert
Params gate_up_params(const FfnArgs& a) {
  Params p{};
  for (int e = 0; e < 2; ++e) {
    Group& g = p.g[e];
    g.a = static_cast<const __bf16*>(a.x);
    g.b0 = static_cast<const __bf16*>(a.gate[e]);
    g.b1 = static_cast<const __bf16*>(a.up[e]);
    g.c = static_cast<__bf16*>(a.hmid);
    g.m = 0; g.n = static_cast<int>(a.inter[e]); g.k = static_cast<int>(a.hidden);
    g.lda = static_cast<int>(padded_sorted_rows(a.rows) / kBlkRows);  // row blocks of the tiled activations
    g.ldb = static_cast<int>(tiled_row_blocks(a.inter[e]));           // row blocks of the tiled weights
    g.ldc = 0;                                                        // set on the device from the row counts
    g.a_row0 = 0;
  }
  p.offsets = a.offsets;
  p.keep[0] = static_cast<__bf16*>(a.keep_gate);
  p.keep[1] = static_cast<__bf16*>(a.keep_up);
  return p;
}

// The number of rows if the few-rows form takes this FFN, else 0.  Not with matrices beyond 31-bit byte offsets.  (Where the
// projections are kept for a backward pass it does, as everywhere: a block's forward is the same with and without gradients.)
int64_t few_rows_of(const FfnArgs& a) {
  const int64_t max_inter = a.inter[0] > a.inter[1] ? a.inter[0] : a.inter[1];
  if ((max_inter + 16) * (a.hidden + 32) * 2 >= (1ll << 31) ||
      padded_sorted_rows(a.rows) * (a.hidden > max_inter ? a.hidden : max_inter) * 2 >= (1ll << 31))
    return 0;
  return few_rows(a.rows, a.inter[0], a.inter[1], a.hidden, device_cu_count()) ? a.rows : 0;
}

int launch_gate_up(const FfnArgs& a, hipStream_t s) {
  const Params p = gate_up_params(a);
  const int64_t t0 = ceil_div(a.inter[0], BigTile::BN / 2), t1 = ceil_div(a.inter[1], BigTile::BN / 2);
  if (a.host_rows != nullptr) {  // the caller knows the split: one launch of the right tile shape
    const int64_t by_expert[2] = {ceil_div(a.host_rows[0], BigTile::BM) * t0, ceil_div(a.host_rows[1], BigTile::BM) * t1};
    const int64_t tiles = by_expert[0] + by_expert[1];
    return launch_mfma<kGateUp>(p, tiles, tiles, s, "dual_gemm_kernel<gate_up>", by_expert, few_rows_of(a), nullptr, a.host_rows);
  }
  // the split of the rows between the experts is only known on the device: bound the tile count from the total
  const int64_t row_tiles = ceil_div(a.rows, BigTile::BM);
  return launch_mfma<kGateUp>(p, row_tiles * (t0 < t1 ? t0 : t1), (row_tiles + 1) * (t0 > t1 ? t0 : t1), s,
                              "dual_gemm_kernel<gate_up>", nullptr, few_rows_of(a));
}

// out_e = hmid_e @ down_e^T, row-major, expert e's rows start at offsets[e]
Params down_params(const FfnArgs& a) {
  Params p{};
  for (int e = 0; e < 2; ++e) {
    Group& g = p.g[e];
    g.a = static_cast<const __bf16*>(a.hmid);
    g.b0 = static_cast<const __bf16*>(a.down[e]);
    g.b1 = nullptr;
    g.c = static_cast<__bf16*>(a.out);
    g.m = 0; g.n = static_cast<int>(a.hidden); g.k = static_cast<int>(a.inter[e]);
    g.lda = 0;  // set on the device from the row counts
    g.ldb = static_cast<int>(tiled_row_blocks(a.hidden));
    g.ldc = static_cast<int>(a.hidden);
    g.a_row0 = 0;
  }
  p.offsets = a.offsets;
  p.scatter = a.out_row_id;
  p.residual = static_cast<const __bf16*>(a.residual);
  return p;
}

constexpr size_t kSplitSlotBytes = static_cast<size_t>(BigTile::BM) * BigTile::BN * sizeof(float);
// counters, a word per slot, in front of the slots
size_t split_count_bytes() { return (static_cast<size_t>(device_cu_count()) * sizeof(int) + 1023) / 1024 * 1024; }

// Whether the down launch's contraction is cut for some split of the rows (PartsRule): more than 2 * cus rows, half a round of
// large tiles at most, contractions of 4096 at least.  (The few-rows form takes none of them: of so many rows only
// where both experts are far narrower.)
bool may_split(const FfnArgs& a) {
  const int cus = device_cu_count();
  return a.rows > 2ll * cus && 2 * (ceil_div(a.rows, BigTile::BM) * ceil_div(a.hidden, BigTile::BN)) <= cus &&
         (a.inter[0] >= 4096 || a.inter[1] >= 4096);
}

// (of sizes that may_split lets through: at most 32768 rows)
PartsRule parts_rule(const FfnArgs& a) {
  PartsRule r{};
  r.cus = device_cu_count();
  r.cols = static_cast<int>(ceil_div(a.hidden, SmallTile::BN));
  for (int e = 0; e < 2; ++e) {
    const int64_t steps = ceil_div(a.inter[e], SmallTile::BN / 2);
    r.steps[e] = static_cast<int>(steps <= r.cus ? steps : r.cus + 1);  // (more than one per CU is all that is asked)
    r.beside[e] = 2 * a.inter[e] > a.inter[1 - e];
    r.lg_most[e] = a.inter[e] >= 8192 ? 2 : (a.inter[e] >= 4096 ? 1 : 0);
  }
  return r;
}

int launch_down(const FfnArgs& a, hipStream_t s) {
  const Params p = down_params(a);
  const int64_t col_tiles = ceil_div(a.hidden, BigTile::BN);
  const int cus = device_cu_count();
  const bool rows_known = a.host_rows != nullptr;
  DownSplit parts_of{};
  const DownSplit* split = nullptr;
  if (a.split_scratch != nullptr && may_split(a)) {
    parts_of.count = static_cast<int*>(a.split_scratch);
    parts_of.sums = reinterpret_cast<float*>(static_cast<char*>(a.split_scratch) + split_count_bytes());
    parts_of.rule = parts_rule(a);
    if (rows_known) {
      const DownParts parts = parts_of.rule.parts(static_cast<int>(a.host_rows[0]), static_cast<int>(a.host_rows[1]));
      if (parts.large) hipLaunchKernelGGL(down_split_kernel<BigTile>, dim3(cus), dim3(BigTile::kThreads), 0, s, p, parts_of);
      else if (parts.lg > 0)
        hipLaunchKernelGGL(down_split_kernel<SmallTile>, dim3(cus * SmallTile::kWgPerCu), dim3(SmallTile::kThreads), 0, s, p, parts_of);
      if (parts.lg > 0) return check_launch("down_split_kernel");
    } else {
      split = &parts_of;  // the launches decide by the same rule
    }
  }
  if (a.host_rows != nullptr) {
    const int64_t by_expert[2] = {ceil_div(a.host_rows[0], BigTile::BM) * col_tiles, ceil_div(a.host_rows[1], BigTile::BM) * col_tiles};
    const int64_t tiles = by_expert[0] + by_expert[1];
    return launch_mfma<kDown>(p, tiles, tiles, s, "dual_gemm_kernel<down>", by_expert, few_rows_of(a));
  }
  const int64_t row_tiles = ceil_div(a.rows, BigTile::BM);
  return launch_mfma<kDown>(p, row_tiles * col_tiles, (row_tiles + 1) * col_tiles, s, "dual_gemm_kernel<down>", nullptr,
                            few_rows_of(a), split);
}

// Both launches as one (ffn_fused_kernel), for the shapes where each is a single round of small tiles with the row
// counts known on the host -- a denoise step.  With a.x_rows the gate/up tiles read the token rows themselves (the
// permute happens in their loads; a.x is not touched).  Returns 1 when the shape is not of that kind (nothing launched).
// Whether the one launch that last used workspace `ws` from this thread ran on the same weights (they are then
// taken to be in the caches still, and the launch does not pull them in ahead of its K loops: in a loop over one
// layer that would cost 0.9 us per launch, where for a model's layers, each with weights of its own, it saves 2).
// A guess that only decides this; a few workspaces (streams) per thread are remembered.
bool weights_of_last_launch(const void* ws, const FfnArgs& a) {
  struct Seen { const void* ws; const void* w[6]; };
  constexpr int kSeen = 8;
  thread_local Seen seen[kSeen] = {};
  thread_local int next = 0;
  const void* w[6] = {a.gate[0], a.up[0], a.down[0], a.gate[1], a.up[1], a.down[1]};
  for (Seen& s : seen) {
    if (s.ws != ws) continue;
    bool same = true;
    for (int i = 0; i < 6; ++i) { same = same && s.w[i] == w[i]; s.w[i] = w[i]; }
    return same;
  }
  Seen& s = seen[next];
  next = (next + 1) % kSeen;
  s.ws = ws;
  for (int i = 0; i < 6; ++i) s.w[i] = w[i];
  return false;
}

// Tiles of the one launch in the few-rows form: row blocks of 16, blocks of 16 weight rows of a gate/up tile (half gate, half
// up) and of a down tile, workgroups per CU.
constexpr int kFewShapes = 4;
constexpr int kFewShape[kFewShapes][4] = {{1, 2, 2, 2}, {1, 4, 4, 2}, {2, 4, 4, 1}, {2, 4, 8, 1}};
using FfnKernel = void (*)(Params, Params, FusedSync, int);
template <int Q>
FfnKernel few_rows_kernel(bool x_rows, bool norm) {
  constexpr int fm = kFewShape[Q][0], nb = kFewShape[Q][1], nbc = kFewShape[Q][2], wg = kFewShape[Q][3];
  if (norm) return ffn_few_rows_norm_kernel<fm, nb, nbc, wg>;
  if constexpr (wg == 1)
    if (!x_rows) return ffn_few_rows_kernel<fm, nb, nbc, wg, false>;
  return ffn_few_rows_kernel<fm, nb, nbc, wg, true>;
}

constexpr size_t kFusedWorkspaceInts = 2 * static_cast<size_t>(kFusedCounters) + 1;  // two counter arrays, then the error flag
int launch_ffn_fused(const FfnArgs& a, int* ws, hipStream_t s) {
  if (ws == nullptr || a.keep_gate != nullptr) return 1;
  // (whatever the real split of the rows: the counters hold this many row blocks per expert)
  if (a.rows > static_cast<int64_t>(kFusedMaxRowBlocks) * SmallTile::BM) return 1;
  // (token rows are addressed with 31-bit byte offsets)
  if (a.x_rows != nullptr && (a.out_row_id == nullptr || a.rows * a.hidden * 2 >= (1ll << 31))) return 1;
  const int cus = device_cu_count();
  int64_t gate_tiles = 0, down_tiles = 0;
  int need[2] = {0, 0};
  const int64_t down_cols = ceil_div(a.hidden, SmallTile::BN);
  for (int e = 0; e < 2; ++e) {
    need[e] = static_cast<int>(ceil_div(a.inter[e], SmallTile::BN / 2));
    if (a.host_rows != nullptr) {
      const int64_t row_blocks = ceil_div(a.host_rows[e], SmallTile::BM);
      gate_tiles += row_blocks * need[e];
      down_tiles += row_blocks * down_cols;
    }
  }
  const bool rows_known = a.host_rows != nullptr;
  const bool few = few_rows_of(a) > 0;
  if (a.norm_weight != nullptr && !few) return 1;
  int shape = kFewShapes - 1, guess[2] = {0, 0};
  int64_t places = cus;
  if (few) {
    // Where the split of the rows is not known on the host it is taken to be all rows on the narrower expert.  The launch is
    // right for any split (a workgroup takes as many tiles as there are).
    const int narrow = a.inter[1] <= a.inter[0] ? 1 : 0;
    const int64_t rows[2] = {rows_known ? a.host_rows[0] : (narrow ? 0 : a.rows), rows_known ? a.host_rows[1] : (narrow ? a.rows : 0)};
    guess[0] = static_cast<int>(rows[0]);
    guess[1] = static_cast<int>(rows[1]);
    // the smallest tile with at most one gate/up tile per CU whose down tiles have a place beside them, or (as the registers of
    // the larger tiles leave no such place) behind them; for K-tiled rows of the larger tiles only
    for (int q = a.x_rows != nullptr ? 0 : kFewShapes - 2; q < kFewShapes; ++q) {
      const int fm = kFewShape[q][0], nb = kFewShape[q][1], nbc = kFewShape[q][2];
      const int64_t r0 = ceil_div(rows[0], 16 * fm), r1 = ceil_div(rows[1], 16 * fm);
      gate_tiles = r0 * ceil_div(a.inter[0], 8 * nb) + r1 * ceil_div(a.inter[1], 8 * nb);
      down_tiles = (r0 + r1) * ceil_div(a.hidden, 16 * nbc);
      places = static_cast<int64_t>(cus) * kFewShape[q][3];
      shape = q;
      if (gate_tiles <= cus && down_tiles <= (places == cus ? cus - kXcds : cus)) break;
    }
    // (a row block more where rows are on both experts)
    if (!rows_known) down_tiles += ceil_div(a.hidden, 16 * kFewShape[shape][2]);
    // (Fewer down tiles in the grid than an XCD has places: see FusedSync.)
    const int64_t most = places == cus ? cus - kXcds : cus;
    down_tiles = down_tiles < most ? down_tiles : most;
    if (!rows_known) {  // (for rows that are on the wide expert after all)
      const int64_t spare = places - ceil_div(down_tiles, kXcds) * kXcds;
      gate_tiles = gate_tiles < spare ? spare : cus;
    }
    gate_tiles = gate_tiles < cus ? gate_tiles : cus;
  } else if (!rows_known) {
    // The split of the rows is only known on the device.  The launch is right for any split (workgroups take as
    // many tiles as there are), so what the host has to settle is whether it is the faster form whatever the split.
    // Up to two rows per CU it is: 24-27 against 29-34 us with every row on the narrow expert, 2-9 % ahead with a
    // mix, within 4 % with every row on the wide expert (256 and 512 rows, experts 11008 / 1024).  Beyond that, rows
    // on the wide expert cost the one workgroup of producers per CU more than they cost the separate launches' large
    // tiles (+12 % at 1024 rows, +19 % at 2048, against -25 % / -31 % with none); with two workgroups of producers
    // per CU the consumers land wherever a producer has left, two of them on one CU while others idle (+25 % on a
    // half-and-half split of 1024 rows).  So larger problems take the one launch only with the host's row counts.
    if (a.rows > 2 * cus) return 1;
    gate_tiles = down_tiles = cus;
  }
  if (gate_tiles == 0 || gate_tiles > cus || down_tiles > cus) return 1;
  Params pg = gate_up_params(a), pd = down_params(a);
  pg.gate = pd.gate = 0;
  pg.split = pd.split = 0;
  FusedSync fs{};
  fs.ready = ws;
  fs.passed = ws + kFusedCounters;
  fs.error = ws + 2 * kFusedCounters;
  fs.need[0] = need[0];
  fs.need[1] = need[1];
  fs.consumers = static_cast<int>(down_cols);
  if (!weights_of_last_launch(ws, a)) {
    for (int e = 0; e < 2; ++e) {
      fs.warm_b[e][0] = pg.g[e].b0;
      fs.warm_b[e][1] = pg.g[e].b1;
      fs.warm_ldb[e] = pg.g[e].ldb;
    }
    fs.warm_k = static_cast<int>(a.hidden);
  }
  fs.x = static_cast<const __bf16*>(a.x_rows);
  fs.gather = a.out_row_id;
  const int producers = static_cast<int>((gate_tiles + kXcds - 1) / kXcds * kXcds);
  const int consumers = static_cast<int>((down_tiles + kXcds - 1) / kXcds * kXcds);
  if (few) {
    fs.guess[0] = guess[0];
    fs.guess[1] = guess[1];
    fs.norm_weight = static_cast<const __bf16*>(a.norm_weight);
    fs.norm_eps = a.norm_eps;
    const bool x_rows = a.x_rows != nullptr, norm = a.norm_weight != nullptr;
    const FfnKernel kernel = shape == 0   ? few_rows_kernel<0>(x_rows, norm)
                             : shape == 1 ? few_rows_kernel<1>(x_rows, norm)
                             : shape == 2 ? few_rows_kernel<2>(x_rows, norm)
                                          : few_rows_kernel<3>(x_rows, norm);
    hipLaunchKernelGGL(kernel, dim3(producers + consumers), dim3(kFewThreads), 0, s, pg, pd, fs, producers);
    return check_launch("ffn_few_rows_kernel");
  }
  const FfnKernel kernel = a.x_rows != nullptr ? ffn_fused_kernel<true> : ffn_fused_kernel<false>;
  hipLaunchKernelGGL(kernel, dim3(producers + consumers), dim3(SmallTile::kThreads), 0, s, pg, pd, fs, producers);
  return check_launch("ffn_fused_kernel");
}

}  // namespace

namespace wx {
int launch_norm_ffn_few_rows(const void* x, const void* x_tiled, void* out, const void* residual, const int32_t* sorted_row_id,
                             const int32_t* expert_offsets, const void* const* weights0, const void* const* weights1, void* hmid,
                             int64_t num_rows, int64_t hidden, int64_t inter0, int64_t inter1, const int64_t* host_rows,
                             const void* norm_weight, float eps, void* workspace, hipStream_t stream) {
  // (hidden: what the norm's kernel takes in its whole-line form)
  if (!x || !x_tiled || !out || !sorted_row_id || !norm_weight || !workspace || !(eps >= 0.f) || num_rows <= 0 ||
      hidden <= 0 || hidden % 256 != 0 || hidden > 2048)
    return 1;
  if ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(x_tiled) | reinterpret_cast<uintptr_t>(norm_weight) |
       reinterpret_cast<uintptr_t>(residual) | reinterpret_cast<uintptr_t>(out)) & 15)
    return 1;
  if (reinterpret_cast<uintptr_t>(workspace) & 3) return 1;
  FfnArgs a{x_tiled, {weights0[0], weights1[0]}, {weights0[1], weights1[1]}, {weights0[2], weights1[2]},
            out, hmid, host_rows, expert_offsets, num_rows, hidden, {inter0, inter1}, sorted_row_id};
  if (check_ffn("wx_moe_block_forward", a, true, true) != WX_OK) return 1;
  a.residual = residual;
  a.x_rows = x;
  a.norm_weight = norm_weight;
  a.norm_eps = eps;
  return launch_ffn_fused(a, static_cast<int*>(workspace), stream);
}
}  // namespace wx

extern "C" size_t wx_ffn_fused_workspace_bytes(void) { return kFusedWorkspaceInts * sizeof(int); }

extern "C" int wx_ffn_may_split(int64_t num_rows, int64_t hidden, int64_t inter0, int64_t inter1) {
  FfnArgs a{};
  a.rows = num_rows;
  a.hidden = hidden;
  a.inter[0] = inter0;
  a.inter[1] = inter1;
  return may_split(a) ? 1 : 0;
}

extern "C" size_t wx_ffn_split_scratch_bytes(void) { return split_count_bytes() + device_cu_count() * kSplitSlotBytes; }

extern "C" int wx_dual_swiglu_ffn_fused(const void* x_rows, void* x_tiled, void* out, const void* residual,
                                        const int32_t* expert_offsets, const void* gate0, const void* up0,
                                        const void* down0, const void* gate1, const void* up1, const void* down1,
                                        void* hmid, int64_t num_rows, int64_t hidden, int64_t inter0, int64_t inter1,
                                        const int64_t* host_rows_per_expert, const int32_t* out_row_id,
                                        void* workspace, wx_stream_t stream) {
  return wx::ffn_fused(x_rows, x_tiled, out, residual, expert_offsets, gate0, up0, down0, gate1, up1, down1, hmid, num_rows, hidden,
                       inter0, inter1, host_rows_per_expert, out_row_id, workspace, nullptr, stream);
}

int wx::ffn_fused(const void* x_rows, void* x_tiled, void* out, const void* residual, const int32_t* expert_offsets, const void* gate0,
                  const void* up0, const void* down0, const void* gate1, const void* up1, const void* down1, void* hmid,
                  int64_t num_rows, int64_t hidden, int64_t inter0, int64_t inter1, const int64_t* host_rows_per_expert,
                  const int32_t* out_row_id, void* workspace, void* split_scratch, wx_stream_t stream) {
  const char* who = "wx_dual_swiglu_ffn_fused";
  FfnArgs a{x_tiled, {gate0, gate1}, {up0, up1}, {down0, down1}, out, hmid, host_rows_per_expert, expert_offsets,
            num_rows, hidden, {inter0, inter1}, out_row_id};
  if (int rc = check_ffn(who, a, true, true)) return rc;
  if (num_rows == 0) return WX_OK;
  if (residual != nullptr) {
    if (!out_row_id) return fail(WX_ERR_INVALID_ARGUMENT, "%s: a residual needs out_row_id (the sum is formed in token order)", who);
    if (reinterpret_cast<uintptr_t>(residual) & 15) return fail(WX_ERR_INVALID_ARGUMENT, "%s: residual must be 16-byte aligned", who);
    a.residual = residual;
  }
  if (x_rows != nullptr) {
    if (!out_row_id) return fail(WX_ERR_INVALID_ARGUMENT, "%s: x_rows needs out_row_id (the rows are gathered through it)", who);
    if (reinterpret_cast<uintptr_t>(x_rows) & 15) return fail(WX_ERR_INVALID_ARGUMENT, "%s: x_rows must be 16-byte aligned", who);
    a.x_rows = x_rows;
  }
  if (reinterpret_cast<uintptr_t>(workspace) & 3) return fail(WX_ERR_INVALID_ARGUMENT, "%s: workspace must be 4-byte aligned", who);
  a.split_scratch = split_scratch;
  const int rc = launch_ffn_fused(a, static_cast<int*>(workspace), as_stream(stream));
  if (rc <= 0) return rc;
  if (x_rows != nullptr)
    if (int rc2 = wx_permute_rows_tiled(x_rows, x_tiled, nullptr, out_row_id, expert_offsets, num_rows, hidden, stream)) return rc2;
  if (int rc2 = launch_gate_up(a, as_stream(stream))) return rc2;
  return launch_down(a, as_stream(stream));
}

extern "C" int wx_dual_swiglu_gate_up(const void* x_tiled, void* hmid, const int32_t* expert_offsets,
                                      const void* gate0, const void* up0, const void* gate1, const void* up1,
                                      int64_t num_rows, int64_t hidden, int64_t inter0, int64_t inter1,
                                      const int64_t* host_rows_per_expert, wx_stream_t stream) {
  const FfnArgs a{x_tiled, {gate0, gate1}, {up0, up1}, {nullptr, nullptr}, nullptr, hmid, host_rows_per_expert, expert_offsets,
                  num_rows, hidden, {inter0, inter1}};
  if (int rc = check_ffn("wx_dual_swiglu_gate_up", a, true, false)) return rc;
  if (num_rows == 0) return WX_OK;
  return launch_gate_up(a, as_stream(stream));
}

extern "C" int wx_dual_swiglu_gate_up_keep(const void* x_tiled, void* hmid, void* gate_keep, void* up_keep,
                                           const int32_t* expert_offsets, const void* gate0, const void* up0,
                                           const void* gate1, const void* up1, int64_t num_rows, int64_t hidden,
                                           int64_t inter0, int64_t inter1, const int64_t* host_rows_per_expert,
                                           wx_stream_t stream) {
  FfnArgs a{x_tiled, {gate0, gate1}, {up0, up1}, {nullptr, nullptr}, nullptr, hmid, host_rows_per_expert, expert_offsets,
            num_rows, hidden, {inter0, inter1}};
  if (int rc = check_ffn("wx_dual_swiglu_gate_up_keep", a, true, false)) return rc;
  if (num_rows == 0) return WX_OK;
  if (!gate_keep || !up_keep) return fail(WX_ERR_INVALID_ARGUMENT, "wx_dual_swiglu_gate_up_keep: null pointer");
  if ((reinterpret_cast<uintptr_t>(gate_keep) | reinterpret_cast<uintptr_t>(up_keep)) & 15)
    return fail(WX_ERR_INVALID_ARGUMENT, "wx_dual_swiglu_gate_up_keep: buffers must be 16-byte aligned");
  a.keep_gate = gate_keep;
  a.keep_up = up_keep;
  return launch_gate_up(a, as_stream(stream));
}

extern "C" int wx_dual_down_proj(const void* hmid, void* out, const int32_t* expert_offsets, const void* down0,
                                 const void* down1, int64_t num_rows, int64_t hidden, int64_t inter0,
                                 int64_t inter1, const int64_t* host_rows_per_expert, const int32_t* out_row_id,
                                 wx_stream_t stream) {
  const FfnArgs a{nullptr, {nullptr, nullptr}, {nullptr, nullptr}, {down0, down1}, out, const_cast<void*>(hmid),
                  host_rows_per_expert, expert_offsets, num_rows, hidden, {inter0, inter1}, out_row_id};
  if (int rc = check_ffn("wx_dual_down_proj", a, false, true)) return rc;
  if (num_rows == 0) return WX_OK;
  return launch_down(a, as_stream(stream));
}

extern "C" int wx_dual_down_proj_residual(const void* hmid, void* out, const void* residual,
                                          const int32_t* expert_offsets, const void* down0, const void* down1,
                                          int64_t num_rows, int64_t hidden, int64_t inter0, int64_t inter1,
                                          const int64_t* host_rows_per_expert, const int32_t* out_row_id,
                                          wx_stream_t stream) {
  const char* who = "wx_dual_down_proj_residual";
  FfnArgs a{nullptr, {nullptr, nullptr}, {nullptr, nullptr}, {down0, down1}, out, const_cast<void*>(hmid),
            host_rows_per_expert, expert_offsets, num_rows, hidden, {inter0, inter1}, out_row_id};
  if (int rc = check_ffn(who, a, false, true)) return rc;
  if (num_rows == 0) return WX_OK;
  if (!residual || !out_row_id)
    return fail(WX_ERR_INVALID_ARGUMENT, "%s: residual and out_row_id are required (the sum is formed in token order)", who);
  if (reinterpret_cast<uintptr_t>(residual) & 15) return fail(WX_ERR_INVALID_ARGUMENT, "%s: residual must be 16-byte aligned", who);
  a.residual = residual;
  return launch_down(a, as_stream(stream));
}

extern "C" int wx_dual_down_proj_split(const void* hmid, void* out, const void* residual, const int32_t* expert_offsets,
                                       const void* down0, const void* down1, int64_t num_rows, int64_t hidden,
                                       int64_t inter0, int64_t inter1, const int64_t* host_rows_per_expert,
                                       const int32_t* out_row_id, void* split_scratch, wx_stream_t stream) {
  const char* who = "wx_dual_down_proj_split";
  FfnArgs a{nullptr, {nullptr, nullptr}, {nullptr, nullptr}, {down0, down1}, out, const_cast<void*>(hmid),
            host_rows_per_expert, expert_offsets, num_rows, hidden, {inter0, inter1}, out_row_id};
  if (int rc = check_ffn(who, a, false, true)) return rc;
  if (num_rows == 0) return WX_OK;
  if (residual != nullptr && !out_row_id)
    return fail(WX_ERR_INVALID_ARGUMENT, "%s: a residual needs out_row_id (the sum is formed in token order)", who);
  if ((reinterpret_cast<uintptr_t>(residual) | reinterpret_cast<uintptr_t>(split_scratch)) & 15)
    return fail(WX_ERR_INVALID_ARGUMENT, "%s: residual and split_scratch must be 16-byte aligned", who);
  a.residual = residual;
  a.split_scratch = split_scratch;
  return launch_down(a, as_stream(stream));
}

extern "C" int wx_dual_swiglu_ffn(const void* x_tiled, void* out, const int32_t* expert_offsets, const void* gate0,
                                  const void* up0, const void* down0, const void* gate1, const void* up1,
                                  const void* down1, void* hmid, int64_t num_rows, int64_t hidden, int64_t inter0,
                                  int64_t inter1, const int64_t* host_rows_per_expert, const int32_t* out_row_id,
                                  wx_stream_t stream) {
  const FfnArgs a{x_tiled, {gate0, gate1}, {up0, up1}, {down0, down1}, out, hmid, host_rows_per_expert, expert_offsets,
                  num_rows, hidden, {inter0, inter1}, out_row_id};
  if (int rc = check_ffn("wx_dual_swiglu_ffn", a, true, true)) return rc;
  if (num_rows == 0) return WX_OK;
  if (int rc = launch_gate_up(a, as_stream(stream))) return rc;
  return launch_down(a, as_stream(stream));
}
