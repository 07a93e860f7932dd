// GQA-native prefill attention for gfx950 (MFMA, fp32 softmax).
//
// Reference semantics: the prefill branch of threadcut/attention.py:43-46 —
// SDPA of q [b, hq, L, d] against repeat_kv(k), repeat_kv(v) (each KV head
// expanded g = hq/hkv times) with the boolean attention mask, or is_causal
// when there is no mask and L == n; output transposed to [b, L, hq, d].
// Here the KV heads are never expanded: a work-group owns 64 or 128 query rows
// (Shape; plan() says which shape a call takes) that are (query token, query head of the group) pairs of ONE KV head, so every
// K/V tile it stages in LDS is read once and shared by the g heads.
//
// Per tile, each wave (32 query rows, 32 or 64 of the tile's keys) computes
//   S^T = K . Q^T   with v_mfma_f32_32x32x16: A = K rows from LDS, B = Q^T
//                   from registers; lane l then holds 16 of the 32 keys of
//                   each 32-key half for query row l%32 (the other 16 sit in
//                   lane l^32), so a row's max and sum need one lane swap;
//   O^T += V^T . P^T with P^T fed straight from those registers (fp16/bf16)
//                   and V^T read from the V rows in LDS with the
//                   transposing read (ds_read_b64_tr_b16), so P never moves
//                   between lanes.
// The online softmax runs per query row in fp32, log2 domain, as
// p = exp2(s * c - m) with c = |scale| * log2(e) (a negative scale flips the
// sign bits of Q instead). The running maximum m moves only when a tile's
// maximum exceeds it by more than a factor 2^8, so the accumulators are
// rescaled rarely. The K and V^T fragments are read from LDS ahead of the
// MFMAs that use them.
//
// Every tile is classified for the whole work-group: SKIP (no row sees any
// of its keys: not loaded), FULL (every row sees every key: no per-element
// test), CAUSAL (per-element test by the end-aligned causal rule) or MIXED
// (per-element test against the mask bytes). Without a mask the class
// follows from n and the causal diagonal; with a boolean mask it is read
// from a map that tc_prefill_mask_tiles builds in one pass over the mask,
// once per mask.
// Tiles are double-buffered and loaded straight into LDS (16-byte buffer
// loads with the LDS bit, no registers, no LDS stores): the next active
// tile's loads are in flight while the current one is multiplied.
#include <algorithm>
#include <cmath>

#include "tc_common.hpp"

namespace tc {
namespace {

#ifndef TC_PREFILL_STAMPS
#define TC_PREFILL_STAMPS 0  // 1: the measurement build; every prefill wave records its tile phases
#endif
constexpr int kHeadDim = 128;
constexpr int kMapRows = 128;      // query rows per row of the mask's tile map
constexpr int kKeys = 64;          // keys per tile of the map
constexpr int kRowBytes = 2 * kHeadDim;  // a K or V row in LDS (unpadded)

// TILE_CAUSAL: the tile's mask is exactly the end-aligned causal rule
// (key <= n - q_len + token), so its elements are tested arithmetically.
enum : int { TILE_SKIP = 0, TILE_FULL = 1, TILE_MIXED = 2, TILE_CAUSAL = 3 };

// Waves per SIMD the register allocation targets: 2 leaves 256 registers a lane
// and matches what the 160 KB LDS of a CU holds, two work-groups of four waves
// (64 KB of tile buffers each) or one of eight (128 KB).
#ifndef TC_PREFILL_WAVES
#define TC_PREFILL_WAVES 2
#endif

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float float16v __attribute__((ext_vector_type(16)));

struct PrefillArgs {
  const uint16_t* q;
  const uint16_t* k;
  const uint16_t* v;
  const uint8_t* mask;      // null, or [mb, L, n] booleans, keys contiguous (batch stride 0 broadcasts)
  const uint8_t* tiles;     // null, or the tile classes of `mask` [mb][nblk][pitch]
  uint16_t* out;            // [b, L, hq, d]
  int64_t sq_b, sq_h, sq_t;
  int64_t sk_b, sk_h, sk_t;
  int64_t sv_b, sv_h, sv_t;
  int64_t sm_b, sm_q;
  int64_t so_b, so_t, so_h;
  int64_t q_len, n;         // query tokens, keys (the queries sit at positions n - q_len ..)
  int64_t nblk;             // query blocks per (batch, KV head)
  int64_t map_nblk;         // rows of the tile map per mask: blocks of kMapRows query rows
  int64_t pitch;            // tile map row length: ntiles rounded up to 8 (padding reads as SKIP)
  int64_t split_tiles;      // tiles per key split
  float* o_part;            // splits > 1: [b, splits, L, hq, d] fp32, normalized per split
  float* lse_part;          // splits > 1: [b, splits, L, hq] log2-sum-exp of the split (-inf if empty)
  int kv_heads, batch, causal, neg, splits;
  int descend;              // query blocks from the last to the first (later rows see more keys)
  int by_block;             // a query block of every sequence before the next block (else a sequence at a time)
  int mask_words;           // mask rows 4-byte aligned: a tile's mask bytes load as words
  int whole;                // contiguous K/V: (n + 128) rows of each fit 31 bits (one buffer range a slab)
  int fold_cus;             // > 0: pair work items w and W-1-w on one CU (see the kernel), W <= 2 x this
  float c;                  // |scale| * log2(e), > 0 (neg: 1 for a negative scale, -1 for scale 0)
  // Paged K/V (prefill_kernel<DT, G, true>): k and v are page pools whose head
  // slabs start at k + h * sk_h (v + h * sv_h); the row of sequence b's
  // logical key t sits tok_off[b * tok_pitch + t] bytes into the slab (the
  // same offset in K and V). pool_bytes_k / _v bound the buffer ranges from
  // the slab start, so a wrong offset reads zeros, not another allocation.
  const int32_t* tok_off;
  int64_t tok_pitch;
  int64_t pool_bytes_k, pool_bytes_v;
#if TC_PREFILL_STAMPS
  // The shapes of one key group only (Wide). Per wave (work-group * 4 + wave),
  // kStampWords words: a header of 8 (shader
  // clock and realtime clock at the start, the same at the end, HW_REG_HW_ID
  // | HW_REG_XCC_ID << 32, tiles recorded), then 5 shader-clock stamps per
  // tile (its start, QK^T issued, softmax done, P.V issued, its loads landed).
  unsigned long long* stamps;
#endif
};
#if TC_PREFILL_STAMPS
constexpr int kStampTiles = 256;
constexpr int kStampWords = 8 + 5 * kStampTiles;
#endif

template <int DT> struct Mfma;
template <> struct Mfma<TC_DTYPE_F16> {
  static __device__ __forceinline__ float16v mma(const uint4& a, const uint4& b, const float16v& c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8, a), __builtin_bit_cast(half8, b), c, 0,
                                                  0, 0);
  }
};
template <> struct Mfma<TC_DTYPE_BF16> {
  static __device__ __forceinline__ float16v mma(const uint4& a, const uint4& b, const float16v& c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c,
                                                   0, 0, 0);
  }
};

// Two fp32 values rounded to nearest even into one word of two 16-bit
// elements (v_cvt_pk_f16_f32 / v_cvt_pk_bf16_f32), the first in the low half.
template <int DT> __device__ __forceinline__ uint32_t pack2(float x, float y);
template <> __device__ __forceinline__ uint32_t pack2<TC_DTYPE_F16>(float x, float y) {
  typedef _Float16 h2 __attribute__((ext_vector_type(2)));
  const h2 v = {static_cast<_Float16>(x), static_cast<_Float16>(y)};
  return __builtin_bit_cast(uint32_t, v);
}
template <> __device__ __forceinline__ uint32_t pack2<TC_DTYPE_BF16>(float x, float y) {
  typedef __bf16 b2 __attribute__((ext_vector_type(2)));
  const b2 v = {static_cast<__bf16>(x), static_cast<__bf16>(y)};
  return __builtin_bit_cast(uint32_t, v);
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const void* p, int64_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0,
                                           static_cast<int32_t>(bytes < 0 ? 0 : (bytes > 0x7fffffff ? 0x7fffffff : bytes)),
                                           0x00020000);
}

// Paged: the offset of a key past n (as an unsigned offset, 2^31: past every
// buffer range, so the row reads zeros).
constexpr int32_t kNoRow = INT32_MIN;

// x combined with its value in lane l ^ 32 (v_permlane32_swap leaves both
// halves' values in its two results).
__device__ __forceinline__ float pair_max(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float pair_sum(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// The running maximum moves only when a tile's maximum exceeds it by more
// than this (log2 units), so p = exp2(s*c - m) <= 2^kLazy.
constexpr float kLazy = 8.f;

// (1, 1) as two 16-bit elements: dot2(p, kOnes) is the sum of a packed pair.
template <int DT> constexpr uint32_t kOnes = 0;
template <> constexpr uint32_t kOnes<TC_DTYPE_F16> = 0x3C003C00u;
template <> constexpr uint32_t kOnes<TC_DTYPE_BF16> = 0x3F803F80u;

// Key offset (within a 32-key half) of accumulator v of a lane in half `hi`.
__device__ __forceinline__ int acc_key(int v, int hi) { return 8 * (v >> 2) + 4 * hi + (v & 3); }

// Query rows and keys of a work-group. Its ROWS x KEYGROUPS waves run on the
// four SIMDs of a CU; row group rg holds 32 query rows, key group kg takes
// HALVES x 32 keys of every tile, and the key groups' partial results are
// merged through LDS at the end.
template <int ROWGROUPS, int KEYGROUPS, int HALVES>
struct Shape {
  static constexpr int kRowGroups = ROWGROUPS;
  static constexpr int kKeyGroups = KEYGROUPS;
  static constexpr int kWaves = ROWGROUPS * KEYGROUPS;
  static constexpr int kRows = 32 * ROWGROUPS;        // query rows per work-group
  static constexpr int kWaveKeys = 32 * HALVES;       // a wave's keys of a tile
  static constexpr int kTileKeys = kWaveKeys * KEYGROUPS;
};

template <int DT, int G, bool PAGED, class S>
__global__ __launch_bounds__(64 * S::kWaves) __attribute__((amdgpu_waves_per_eu(TC_PREFILL_WAVES, TC_PREFILL_WAVES))) void prefill_kernel(
    const PrefillArgs a) {
  constexpr int kTileKeys = S::kTileKeys;
  constexpr int kHalves = S::kWaveKeys / 32;       // 32-key halves of a wave's keys
  constexpr int kSteps = 2 * kHalves;              // 16-key steps of P.V
  constexpr int kMapTiles = kTileKeys / kKeys;     // 64-key tiles (mask map, 64-key classes) per tile
  constexpr int kDmaRows = kTileKeys / S::kWaves;  // K rows (and V rows) a wave loads per tile
  constexpr int kDma = kDmaRows / 4;               // loads a thread issues for them
  constexpr int kTokens = S::kRows / G;            // query tokens per work-group
  // Tile buffers: K and V rows of 256 B, unpadded (a 16-byte load into LDS
  // writes 64 lanes x 16 B in one run); chunk x of row r sits in slot
  // x ^ sw(r), sw(r) = 4 (r % 4) + (r / 4) % 4, which spreads the K reads
  // (16 rows, one chunk) and the transposing V reads (8 rows, 4 chunks)
  // over all banks.
  __shared__ __attribute__((aligned(1024))) uint16_t s_k0[kTileKeys * kHeadDim];
  __shared__ __attribute__((aligned(1024))) uint16_t s_k1[kTileKeys * kHeadDim];
  __shared__ __attribute__((aligned(1024))) uint16_t s_v0[kTileKeys * kHeadDim];
  __shared__ __attribute__((aligned(1024))) uint16_t s_v1[kTileKeys * kHeadDim];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int rg = wave % S::kRowGroups;
  const int kg = wave / S::kRowGroups;
  const int hi = lane >> 5;            // which 16 keys of each 32-key half this lane holds
  const int r32 = lane & 31;           // the lane's query row within the row group
#if TC_PREFILL_STAMPS
  unsigned long long* stw = a.stamps && S::kKeyGroups == 1
                                ? a.stamps + (static_cast<int64_t>(blockIdx.x) * 4 + wave) * kStampWords
                                : nullptr;
  int st_tile = 0;
  auto stamp = [&](int k) {
    if (stw && st_tile < kStampTiles) {
      const unsigned long long now = __builtin_amdgcn_s_memtime();
      if (lane == 0) stw[8 + 5 * st_tile + k] = now;
    }
  };
  if (stw && lane == 0) {
    stw[0] = __builtin_amdgcn_s_memtime();
    stw[1] = __builtin_amdgcn_s_memrealtime();
    unsigned hw, xcc;
    __asm__ volatile("s_getreg_b32 %0, hwreg(HW_REG_HW_ID)" : "=s"(hw));
    __asm__ volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID)" : "=s"(xcc));
    stw[4] = hw | (static_cast<unsigned long long>(xcc) << 32);
  }
#else
  auto stamp = [](int) {};
#endif

  // Work item (KV head fastest, then key split, then sequence and query block,
  // by_block telling which of the two is faster): consecutive work-groups go
  // to different XCDs round-robin, so with 8 | kv_heads each XCD's L2 streams
  // one head's K/V.
  // With C CUs and a grid of C < W <= 2C work-groups (two fit a CU), the
  // dispatcher puts work-groups i and i + C on the same CU (measured on this
  // part). When the work grows along the items (causal rows see more keys),
  // fold_cus = C hands work-group i >= C item W-1-(i-C), so each CU runs item
  // i next to item W-1-i and the CUs finish together. Only the speed depends
  // on that placement.
  // The grid fits 31 bits, so the item is taken apart in 32-bit arithmetic (a
  // 64-bit division is 140 scalar instructions, and nothing can load before).
  uint32_t rest = blockIdx.x;
  const uint32_t heads = a.kv_heads, splits = a.splits, batch = a.batch;
  if (a.fold_cus > 0 && rest >= static_cast<uint32_t>(a.fold_cus))
    rest = heads * splits * batch * static_cast<uint32_t>(a.nblk) - 1 - (rest - a.fold_cus);
  const int h = static_cast<int>(rest % heads);
  rest /= heads;
  const int split = static_cast<int>(rest % splits);
  rest /= splits;
  const uint32_t inner = a.by_block ? batch : static_cast<uint32_t>(a.nblk);
  const uint32_t slow = rest / inner, fast = rest - slow * inner;
  const int b = static_cast<int>(a.by_block ? fast : slow);
  int32_t blk = static_cast<int32_t>(a.by_block ? slow : fast);
  if (a.descend) blk = static_cast<int32_t>(a.nblk) - 1 - blk;  // longest rows first
  // Key and query positions and tile indices fit 32 bits (the host keeps n
  // below 2^30), so the loop's bookkeeping is 32-bit scalar arithmetic.
  const int32_t n32 = static_cast<int32_t>(a.n), q_len32 = static_cast<int32_t>(a.q_len);
  const int32_t tok0 = blk * kTokens;
  const int32_t past = n32 - q_len32;
  const int64_t bm = a.sm_b ? b : 0;

  // The wave's 32 rows: row = (token, head of the group).
  const int row = rg * 32 + r32;
  const int32_t tok = tok0 + row / G;
  const int hq = h * G + row % G;
  const bool row_ok = tok < q_len32;
  const uint8_t* mrow = a.mask ? a.mask + bm * a.sm_b + (row_ok ? tok : 0) * a.sm_q : nullptr;
  const char* kslab = reinterpret_cast<const char*>(a.k + (PAGED ? 0 : b * a.sk_b) + h * a.sk_h);
  const char* vslab = reinterpret_cast<const char*>(a.v + (PAGED ? 0 : b * a.sv_b) + h * a.sv_h);
  const int64_t row_k = a.sk_t * 2, row_v = a.sv_t * 2;
  // Buffer ranges from this head's slab on: paged, over the pools (and the
  // offsets of the wave's rows of a tile, one per lane, kNoRow past n);
  // contiguous with `whole`, over the n rows (the rows past n read zeros).
  const __amdgpu_buffer_rsrc_t prk =
      rsrc(kslab, PAGED ? a.pool_bytes_k - h * a.sk_h * 2 : (a.whole ? static_cast<int64_t>(n32) * row_k : 0));
  const __amdgpu_buffer_rsrc_t prv =
      rsrc(vslab, PAGED ? a.pool_bytes_v - h * a.sv_h * 2 : (a.whole ? static_cast<int64_t>(n32) * row_v : 0));
  const int32_t* toff = PAGED ? a.tok_off + b * a.tok_pitch : nullptr;
  auto tile_rows = [&](int32_t tile) -> int32_t {
    const int32_t key = tile * kTileKeys + kDmaRows * wave + (lane & (kDmaRows - 1));
    return key < n32 ? toff[key] : kNoRow;
  };
  // Paged: when the wave's rows of a tile are consecutive rows of one page
  // (row k at offset first + k * row), the offset of its first row, else -1
  // (also where the tile runs past n). Wave-uniform.
  auto contiguous_from = [&](int32_t idx) -> int32_t {
    const int32_t first = __builtin_amdgcn_readfirstlane(idx);
    const bool apart = static_cast<uint32_t>(idx) !=
                       static_cast<uint32_t>(first) + (lane & (kDmaRows - 1)) * static_cast<uint32_t>(row_k);
    return (first >= 0 && __builtin_amdgcn_ballot_w64(apart) == 0) ? first : -1;
  };
  // Load c of the 2 kDma a thread issues per tile (c < kDma: K, else V),
  // straight into LDS: rows R = kDmaRows wave + 4 (c % kDma) + lane / 16, the
  // lane filling slot lane % 16 of its row with chunk (lane % 16) ^ sw(R).
  // Paged: a row's offset is first + its row of the wave's for a contiguous
  // run (first >= 0), else taken from the lane of idx that holds it.
  // Contiguous: the slab's range with the tile's first row in the load's
  // scalar offset (first >= 0, `whole`), else a range over the tile's rows.
  const int dma_r = lane >> 4;
  auto dma_part = [&](uint16_t* dk, uint16_t* dv, int32_t tile, int32_t idx, int32_t first, int c) {
    const int i = c % kDma;
    const int Rw = 4 * i + dma_r;              // row of the wave's
    const int R = kDmaRows * wave + Rw;
    const int x = (lane & 15) ^ (4 * dma_r + ((kDmaRows / 4 * wave + i) & 3));
    __attribute__((address_space(3))) void* dst =
        (__attribute__((address_space(3))) void*)(reinterpret_cast<char*>(c < kDma ? dk : dv) +
                                                  (kDmaRows * wave + 4 * i) * kRowBytes);
    if constexpr (PAGED) {
      if (first >= 0) {
        const int32_t rb = static_cast<int32_t>(row_k);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(c < kDma ? prk : prv, dst, 16, Rw * rb + 16 * x, first, 0, 0);
      } else {
        const int32_t off = __builtin_amdgcn_ds_bpermute(4 * Rw, idx) + 16 * x;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(c < kDma ? prk : prv, dst, 16, off, 0, 0, 0);
      }
    } else if (first >= 0) {
      const int32_t rb = static_cast<int32_t>(c < kDma ? row_k : row_v);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(c < kDma ? prk : prv, dst, 16, R * rb + 16 * x, tile * kTileKeys * rb, 0, 0);
    } else {
      const int32_t key0 = tile * kTileKeys;
      const int32_t rows = n32 - key0 < kTileKeys ? n32 - key0 : kTileKeys;
      if (c < kDma)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc(kslab + key0 * row_k, rows * row_k), dst, 16,
                                                 static_cast<int32_t>(R * row_k + 16 * x), 0, 0, 0);
      else
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc(vslab + key0 * row_v, rows * row_v), dst, 16,
                                                 static_cast<int32_t>(R * row_v + 16 * x), 0, 0, 0);
    }
  };
  // The loads of a tile. The test for a one-page run (paged) or a slab in one
  // range (contiguous) is taken once for the burst (a test per load left the
  // compiler branching and waiting between the loads).
  auto dma_tile = [&](uint16_t* dk, uint16_t* dv, int32_t tile, int32_t idx, int32_t first) {
    if (!PAGED) first = a.whole ? 0 : -1;
    if (__builtin_expect(first >= 0, 1)) {
#pragma unroll
      for (int c = 0; c < 2 * kDma; ++c) dma_part(dk, dv, tile, idx, first, c);
    } else {
#pragma unroll
      for (int c = 0; c < 2 * kDma; ++c) dma_part(dk, dv, tile, idx, -1, c);
    }
  };
  // The map's rows are blocks of kMapRows query rows, of which this block is one or a part.
  const uint8_t* tcls = a.tiles ? a.tiles + (bm * a.map_nblk + blk * S::kRows / kMapRows) * a.pitch : nullptr;

  // Tiles this work-group may need: its split's share of all n keys, cut at
  // its last query's position when causal.
  const int32_t last_tok = min(tok0 + kTokens, q_len32) - 1;
  const int32_t key_end = a.causal ? min(n32, past + last_tok + 1) : n32;
  const int32_t split_tiles = static_cast<int32_t>(a.split_tiles);
  const int32_t t_begin = split * split_tiles;
  const int32_t nt = min((key_end + kTileKeys - 1) / kTileKeys, t_begin + split_tiles);
  // The classes of a window of 64 tiles from `base` on, one bit a tile: lane i
  // works out tile base + i, and ballots leave the window in scalar registers,
  // so that finding the next active tile and its class takes a shift and a
  // few bit tests (testing tile by tile took 490 cycles of a 2500-cycle tile
  // in jumps). act: some row of the work-group sees a key of the tile; cls0 and
  // cls1: the low and the high bit of the class of this wave's keys (with one
  // key group they are the tile's, and act follows from them).
  int32_t base = 0;
  uint64_t act = 0, cls0 = 0, cls1 = 0;
  // The map's classes of a window are loaded a window ahead.
  auto map_load = [&](int32_t tile) -> uint32_t {
    if (tile >= nt) return 0;
    if constexpr (kMapTiles == 1) return tcls[tile];
    return *reinterpret_cast<const uint16_t*>(tcls + tile * kMapTiles);
  };
  uint32_t map_next = tcls ? map_load(t_begin + lane) : 0u;
  auto window = [&](int32_t first) {
    base = first;
    const int32_t tile = first + lane;
    const int32_t key0 = tile * kTileKeys + kg * S::kWaveKeys;
    const bool on = tile < nt;
    bool some = on;
    int c = TILE_MIXED;
    if (tcls) {
      some = map_next != 0;
      c = static_cast<int>(kMapTiles == 1 ? map_next : (map_next >> (8 * (key0 / kKeys % kMapTiles))) & 0xffu);
      map_next = map_load(tile + 64);
    } else if (!a.mask && key0 + S::kWaveKeys <= n32) {
      c = a.causal ? TILE_CAUSAL : TILE_FULL;
    }
    if (c == TILE_CAUSAL && (S::kKeyGroups > 1 || !tcls)) {
      c = key0 + S::kWaveKeys - 1 > past + tok0 ? TILE_CAUSAL : TILE_FULL;
      if (S::kKeyGroups > 1 && key0 > past + last_tok) c = TILE_SKIP;
    }
    if (!on || (S::kKeyGroups > 1 && key0 >= n32)) c = TILE_SKIP;
    cls0 = __builtin_amdgcn_ballot_w64(c & 1);
    cls1 = __builtin_amdgcn_ballot_w64(c & 2);
    act = S::kKeyGroups > 1 ? __builtin_amdgcn_ballot_w64(on && some) : cls0 | cls1;
  };
  // First active tile at or after t >= base (nt if none), and its class.
  auto next_active = [&](int32_t t, int& cls) -> int32_t {
    uint64_t r = t - base < 64 ? act >> (t - base) : 0;
    while (__builtin_expect(r == 0, 0)) {
      t = base + 64;
      if (t >= nt) {
        cls = TILE_SKIP;
        return nt;
      }
      window(t);
      r = act;
    }
    t += __builtin_ctzll(r);
    const int k = t - base;
    cls = static_cast<int>((cls0 >> k) & 1) | static_cast<int>((cls1 >> k) & 1) << 1;
    return t;
  };

  float m = neg_inf(), l = 0.f;
  float16v o[4];
#pragma unroll
  for (int dt = 0; dt < 4; ++dt)
#pragma unroll
    for (int v = 0; v < 16; ++v) o[dt][v] = 0.f;

  // Byte offsets of the lane's K reads (chunk 2c + hi of row 32 kt + r32 of
  // the wave's keys, kt adding 8 KB) and transposing V reads (rows
  // 16p + 8rr + 4hi + j, chunk 4dt + 2(g&1) + q/2, byte 8(q&1) for lane 4j + q
  // of 16-lane group g; p adding 4 KB).
  int kaddr[8], vaddr[2][4];
  {
    const int base = kg * S::kWaveKeys * kRowBytes;
    const int swk = ((r32 & 3) << 2) | ((r32 >> 2) & 3);
#pragma unroll
    for (int c = 0; c < 8; ++c) kaddr[c] = base + r32 * kRowBytes + 16 * ((2 * c + hi) ^ swk);
    const int j = (lane & 15) >> 2, q = lane & 3, e = 2 * ((lane >> 4) & 1) + (q >> 1);
#pragma unroll
    for (int rr = 0; rr < 2; ++rr)
#pragma unroll
      for (int dt = 0; dt < 4; ++dt)
        vaddr[rr][dt] = base + (8 * rr + 4 * hi + j) * kRowBytes +
                        16 * ((4 * dt + e) ^ ((j << 2) | (2 * rr + hi))) + 8 * (q & 1);
  }

  // Active tiles t (in LDS), tn (loading) and the class of each, found one
  // iteration ahead. The first tile of the range is loaded before its class
  // is known: it is nearly always active.
  auto load_first = [&](int32_t tile) {
    int32_t rows_t = kNoRow, first_t = -1;
    if constexpr (PAGED) {
      rows_t = tile_rows(tile);
      first_t = contiguous_from(rows_t);
    }
    dma_tile(s_k0, s_v0, tile, rows_t, first_t);
  };
  if (t_begin < nt) load_first(t_begin);
  // Q^T as the MFMA B operand: dims 16c + 8*hi .. +8 of the lane's row, loaded
  // behind the first tile.
  uint4 qb[8];
  {
    const uint16_t* qp = a.q + b * a.sq_b + hq * a.sq_h + (row_ok ? tok : 0) * a.sq_t + 8 * hi;
#pragma unroll
    for (int c = 0; c < 8; ++c)
      qb[c] = row_ok ? *reinterpret_cast<const uint4*>(qp + 16 * c) : make_uint4(0u, 0u, 0u, 0u);
    if (a.neg > 0) {
#pragma unroll
      for (int c = 0; c < 8; ++c) {
        qb[c].x ^= 0x80008000u; qb[c].y ^= 0x80008000u; qb[c].z ^= 0x80008000u; qb[c].w ^= 0x80008000u;
      }
    } else if (a.neg < 0) {
      // Scale 0, as Q = 0 with c = 1 (an infinity or NaN times 0 is NaN): the
      // scores stay products with c > 0.
      auto zero = [](uint32_t w) {
        constexpr uint32_t e = DT == TC_DTYPE_F16 ? 0x7c00u : 0x7f80u;
        return ((w & e) == e ? 0x7fffu : 0u) | ((w >> 16 & e) == e ? 0x7fff0000u : 0u);
      };
#pragma unroll
      for (int c = 0; c < 8; ++c)
        qb[c] = make_uint4(zero(qb[c].x), zero(qb[c].y), zero(qb[c].z), zero(qb[c].w));
    }
  }
  int cls_t = TILE_SKIP, cls_n = TILE_SKIP;
  int32_t t = nt, tn = nt;
  if (t_begin < nt) {
    window(t_begin);
    t = next_active(t_begin, cls_t);
    if (t > t_begin && t < nt) {
      __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the buffer is written again
      load_first(t);
    }
    if (t < nt) tn = next_active(t + 1, cls_n);
  }
  // Paged: the row offsets of the tile loaded next, fetched one tile ahead.
  int32_t rows_n = kNoRow;
  if constexpr (PAGED) rows_n = tn < nt ? tile_rows(tn) : kNoRow;
  __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();

  // The wave's keys of one tile from (lk, lv).
  auto attend = [&](const uint16_t* lk, const uint16_t* lv, const int cls) {
    // S^T of the tile in two independent MFMA chains: the 32-key halves, or
    // with one half the even and the odd 16-dim chunks, added at the end.
    // The K fragments are read four chunks ahead of their MFMAs; the
    // scheduling barriers keep the compiler from pulling the reads back next
    // to their use (it otherwise waits out each read's latency).
    float16v s[2];
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int v = 0; v < 16; ++v) s[kt][v] = 0.f;
    {
      auto kfrag = [&](int c, int kt) {
        return *reinterpret_cast<const uint4*>(reinterpret_cast<const char*>(lk) + kaddr[c] + 32 * kRowBytes * kt);
      };
      uint4 kf[4][kHalves];
#pragma unroll
      for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int kt = 0; kt < kHalves; ++kt) kf[c][kt] = kfrag(c, kt);
#pragma unroll
      for (int c = 0; c < 8; ++c) {
        uint4 kc[kHalves];
#pragma unroll
        for (int kt = 0; kt < kHalves; ++kt) {
          kc[kt] = kf[c & 3][kt];
          if (c + 4 < 8) kf[c & 3][kt] = kfrag(c + 4, kt);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int kt = 0; kt < kHalves; ++kt) {
          const int chain = kHalves == 2 ? kt : c & 1;
          s[chain] = Mfma<DT>::mma(kc[kt], qb[c], s[chain]);
        }
      }
    }
    typedef short vs4 __attribute__((ext_vector_type(4)));
    auto vfrag = [&](int p, int dt) {
      const char* vb = reinterpret_cast<const char*>(lv) + 16 * kRowBytes * p;
      const vs4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) vs4*)(vb + vaddr[0][dt]));
      const vs4 up = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) vs4*)(vb + vaddr[1][dt]));
      const uint2 l2 = __builtin_bit_cast(uint2, lo), u2 = __builtin_bit_cast(uint2, up);
      return make_uint4(l2.x, l2.y, u2.x, u2.y);
    };
    uint4 vf[3][4];
    if constexpr (kHalves == 1) {
      // The registers that the second half would take hold V^T: its reads
      // run under the softmax.
#pragma unroll
      for (int p0 = 0; p0 < 2; ++p0)
#pragma unroll
        for (int dt = 0; dt < 4; ++dt) vf[p0][dt] = vfrag(p0, dt);
      __builtin_amdgcn_sched_barrier(0);
      s[0] += s[1];
    }

    stamp(1);
    uint4 pb[kHalves][2];
    {
      // Hidden keys of this lane's row (none on a FULL tile) score -inf, and
      // their exponentials are 0. Key 32 kt + 8 q + 4 hi + j of the wave's.
      const int32_t key0 = t * kTileKeys + kg * S::kWaveKeys;
      if (cls == TILE_MIXED && a.mask) {
        // By the row's mask bytes, read as one batch of loads (one wait, no
        // branch per key): aligned words (word q of half kt at byte
        // 32 kt + 8 q + 4 hi) when the rows are 4-byte aligned and the keys
        // lie inside the row, else bytes, keys past the row reading its last
        // byte and counting as hidden.
        const uint8_t* mt = mrow + key0;
        uint32_t mw[4 * kHalves];
        if (a.mask_words && key0 + S::kWaveKeys <= n32) {
#pragma unroll
          for (int q = 0; q < 4 * kHalves; ++q) mw[q] = reinterpret_cast<const uint32_t*>(mt)[2 * q + hi];
        } else {
          const int32_t lim = n32 - key0;
#pragma unroll
          for (int q = 0; q < 4 * kHalves; ++q) {
            mw[q] = 0;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              const int key = 32 * (q >> 2) + 8 * (q & 3) + 4 * hi + j;
              const uint32_t x = mt[min(key, lim - 1)];
              mw[q] |= (key < lim ? x : 0u) << (8 * j);
            }
          }
        }
#pragma unroll
        for (int kt = 0; kt < kHalves; ++kt)
#pragma unroll
          for (int v = 0; v < 16; ++v)
            s[kt][v] = ((mw[4 * kt + (v >> 2)] >> (8 * (v & 3))) & 0xffu) != 0 ? s[kt][v] : neg_inf();
      } else if (cls != TILE_FULL) {
        // By position: from the row's own key on (causal), or from n on.
        int32_t lim = n32 - key0 - 4 * hi;
        if (a.causal || cls == TILE_CAUSAL) lim = min(lim, past + tok + 1 - key0 - 4 * hi);
#pragma unroll
        for (int kt = 0; kt < kHalves; ++kt)
#pragma unroll
          for (int v = 0; v < 16; ++v) s[kt][v] = 32 * kt + acc_key(v, 0) < lim ? s[kt][v] : neg_inf();
      }
      // Four independent max chains (fmax is exact in any order).
      float m4[4] = {s[0][0], s[0][1], s[0][2], s[0][3]};
#pragma unroll
      for (int kt = 0; kt < kHalves; ++kt)
#pragma unroll
        for (int v = kt ? 0 : 4; v < 16; ++v) m4[v & 3] = fmaxf(m4[v & 3], s[kt][v]);
      float mx = fmaxf(fmaxf(m4[0], m4[1]), fmaxf(m4[2], m4[3]));

      // Running maximum, moved only when the tile's maximum exceeds it by
      // more than 2^kLazy: p = exp2(s*c - m) then stays below 2^kLazy (exact
      // in fp16/bf16 range) and the accumulators are rescaled rarely.
      mx = pair_max(mx);
      const float tmax = mx == neg_inf() ? neg_inf() : mx * a.c;
      const bool move = tmax > m + kLazy;
      const float mn = move ? tmax : m;
      const float alpha = move ? __builtin_amdgcn_exp2f(m - mn) : 1.f;
      m = mn;
      const float ms = (mn == neg_inf()) ? 0.f : mn;
      if (__builtin_amdgcn_ballot_w64(move)) {
#pragma unroll
        for (int dt = 0; dt < 4; ++dt)
#pragma unroll
          for (int v = 0; v < 16; ++v) o[dt][v] *= alpha;
        l *= alpha;
      }

      // P^T operand of half kt, chunk c2: accumulators 8*c2 .. 8*c2+7 are keys
      // 16*c2 + {4hi..4hi+3, 8+4hi..8+4hi+3} of the half, the order in which
      // V^T is read. All the exponentials come first, in one block with no
      // branch between them (c > 0, so a hidden key's is exp2(-inf)). The row
      // sum takes the rounded P, as the MFMA does, in one chain per 32-key half.
#pragma unroll
      for (int kt = 0; kt < kHalves; ++kt)
#pragma unroll
        for (int v = 0; v < 16; ++v) s[kt][v] = __builtin_amdgcn_exp2f(fmaf(s[kt][v], a.c, -ms));
      float lh[kHalves];
#pragma unroll
      for (int kt = 0; kt < kHalves; ++kt) {
        lh[kt] = 0.f;
#pragma unroll
        for (int c2 = 0; c2 < 2; ++c2) {
          uint32_t w[4];
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const int v0 = 8 * c2 + 2 * j;
            w[j] = pack2<DT>(s[kt][v0], s[kt][v0 + 1]);
            lh[kt] = Elem<DT>::dot2(w[j], kOnes<DT>, lh[kt]);
          }
          pb[kt][c2] = make_uint4(w[0], w[1], w[2], w[3]);
        }
      }
      if constexpr (kHalves == 2)
        l += lh[0] + lh[1];
      else
        l += lh[0];
    }

    stamp(2);
    // O^T += V^T . P^T. The four fragments of a 16-key step are read two steps ahead.
    {
      if constexpr (kHalves == 2) {
#pragma unroll
        for (int p0 = 0; p0 < 2; ++p0)
#pragma unroll
          for (int dt = 0; dt < 4; ++dt) vf[p0][dt] = vfrag(p0, dt);
      }
#pragma unroll
      for (int p = 0; p < kSteps; ++p) {
        if (p + 2 < kSteps) {
#pragma unroll
          for (int dt = 0; dt < 4; ++dt) vf[(p + 2) % 3][dt] = vfrag(p + 2, dt);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int dt = 0; dt < 4; ++dt) o[dt] = Mfma<DT>::mma(vf[p % 3][dt], pb[p >> 1][p & 1], o[dt]);
      }
    }
  };

  // One tile from (lk, lv) while the next one loads into (dk, dv).
  auto body = [&](const uint16_t* lk, const uint16_t* lv, uint16_t* dk, uint16_t* dv) {
    stamp(0);
    const bool more = tn < nt;
    const int32_t rows_tn = rows_n;  // paged: the row offsets of tile tn, whose rows load at this tile's start
    int32_t first_tn = -1;
    if constexpr (PAGED) first_tn = more ? contiguous_from(rows_tn) : -1;
    int cls_nn = TILE_SKIP;
    const int32_t tnn = next_active(tn + 1, cls_nn);
    if constexpr (PAGED) rows_n = tnn < nt ? tile_rows(tnn) : kNoRow;
    const int cls = cls_t;

    // The next tile's loads go out first, in one burst: spread between the
    // MFMAs below they stall the MFMA issue.
    if (more) {
      dma_tile(dk, dv, tn, rows_tn, first_tn);
    }
    // With several key groups a wave's own keys may all be hidden.
    if (S::kKeyGroups == 1 || cls != TILE_SKIP) attend(lk, lv, cls);

    stamp(3);
    // This thread's loads of tile tn have landed in LDS; then everyone's.
    __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");
    stamp(4);
#if TC_PREFILL_STAMPS
    ++st_tile;
#endif
    __syncthreads();
    t = tn;
    cls_t = cls_n;
    tn = tnn;
    cls_n = cls_nn;
  };
  while (t < nt) {
    body(s_k0, s_v0, s_k1, s_v1);
    if (t >= nt) break;
    body(s_k1, s_v1, s_k0, s_v0);
  }

#if TC_PREFILL_STAMPS
  if (stw && lane == 0) {
    stw[2] = __builtin_amdgcn_s_memtime();
    stw[3] = __builtin_amdgcn_s_memrealtime();
    stw[5] = static_cast<unsigned long long>(min(st_tile, kStampTiles));
  }
#endif
  float lt = pair_sum(l);
  if constexpr (S::kKeyGroups > 1) {
    // Merge the key groups of each row group: key group kg ends up with
    // 4 / kKeyGroups of the four 32-dim slices; the others' parts of them go
    // through the tile buffers (free after the loop's last barrier), 4 KB a
    // part, in the accumulators' own lane layout (16-byte accesses, no bank
    // conflicts).
    constexpr int kOwn = 4 / S::kKeyGroups;
    constexpr int kSlots = kTileKeys * kRowBytes / 4096;  // parts a tile buffer holds
    static_assert(S::kRowGroups * 4 * (S::kKeyGroups - 1) <= 4 * kSlots, "the parts fit the tile buffers");
    __shared__ float s_m[S::kWaves][32], s_l[S::kWaves][32];
    auto part = [&](int dt, int from) -> float4* {  // row group rg's slice dt as key group `from` holds it
      const int own = dt / kOwn;
      const int slot = (rg * 4 + dt) * (S::kKeyGroups - 1) + (from < own ? from : from - 1);
      const int buf = slot / kSlots;
      uint16_t* p = buf == 0 ? s_k0 : buf == 1 ? s_k1 : buf == 2 ? s_v0 : s_v1;
      return reinterpret_cast<float4*>(p) + (slot % kSlots) * 256 + lane;
    };
    if (hi == 0) {
      s_m[wave][r32] = m;
      s_l[wave][r32] = lt;
    }
#pragma unroll
    for (int dt = 0; dt < 4; ++dt) {
      if (dt / kOwn != kg) {
        float4* p = part(dt, kg);
#pragma unroll
        for (int j = 0; j < 4; ++j)
          p[64 * j] = make_float4(o[dt][4 * j], o[dt][4 * j + 1], o[dt][4 * j + 2], o[dt][4 * j + 3]);
      }
    }
    __syncthreads();
    float mx = neg_inf(), f[S::kKeyGroups];
#pragma unroll
    for (int k = 0; k < S::kKeyGroups; ++k) mx = fmaxf(mx, s_m[k * S::kRowGroups + rg][r32]);
    const float ms = mx == neg_inf() ? 0.f : mx;
    lt = 0.f;
#pragma unroll
    for (int k = 0; k < S::kKeyGroups; ++k) {
      f[k] = __builtin_amdgcn_exp2f(s_m[k * S::kRowGroups + rg][r32] - ms);
      lt += f[k] * s_l[k * S::kRowGroups + rg][r32];
    }
    const float mine = __builtin_amdgcn_exp2f(m - ms);
    m = mx;
#pragma unroll
    for (int dt = 0; dt < 4; ++dt) {
      if (dt / kOwn == kg) {
#pragma unroll
        for (int v = 0; v < 16; ++v) o[dt][v] *= mine;
#pragma unroll
        for (int k = 0; k < S::kKeyGroups; ++k) {
          if (k != kg) {
            const float4* p = part(dt, k);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              const float4 x = p[64 * j];
              o[dt][4 * j] += f[k] * x.x;
              o[dt][4 * j + 1] += f[k] * x.y;
              o[dt][4 * j + 2] += f[k] * x.z;
              o[dt][4 * j + 3] += f[k] * x.w;
            }
          }
        }
      }
    }
  }
  // Normalize and write the wave's outputs (or, of several splits, its partial,
  // merged by prefill_combine_kernel). A lane holds pieces of 4 dims of its
  // row, whose stores would touch 32 rows an instruction (3500 cycles of a
  // short call); the rows are laid out in LDS first (16-byte chunk c of row r
  // at slot c ^ (r % chunks), so that the pieces spread over the banks) and
  // leave 16 bytes a lane, whole rows together.
  const float inv = lt > 0.f ? 1.f / lt : 0.f;
  constexpr int kOwnDims = kHeadDim / S::kKeyGroups;  // dims d_lo .. of this wave
  constexpr int kStage = 32 * kOwnDims * 4;           // staging bytes of a wave (fp32 rows)
  constexpr int kBuf = kTileKeys * kRowBytes;
  static_assert(S::kKeyGroups == 1 || S::kRowGroups * 4 * (S::kKeyGroups - 1) * 4096 + S::kWaves * kStage <= 4 * kBuf,
                "the staged rows lie behind the key groups' parts");
  static_assert(kBuf % kStage == 0 && 4 * kBuf >= S::kWaves * kStage, "a wave's rows fit one tile buffer");
  char* stage;
  {
    const int at = 4 * kBuf - (S::kWaves - wave) * kStage;
    uint16_t* p = at < kBuf ? s_k0 : at < 2 * kBuf ? s_k1 : at < 3 * kBuf ? s_v0 : s_v1;
    stage = reinterpret_cast<char*>(p) + at % kBuf;
  }
  // The lanes of a wave read rows that other lanes of it have written: its LDS
  // accesses run in order, and this keeps the compiler to that order.
  auto staged = [] {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };
  const int d0 = kOwnDims * kg;  // the wave's first dim
  const bool partial = a.splits > 1;
  const int64_t prow0 = ((static_cast<int64_t>(b) * splits + split) * a.q_len) * (a.kv_heads * G);
  if (partial && hi == 0 && kg == 0 && row_ok)
    a.lse_part[prow0 + static_cast<int64_t>(tok) * (a.kv_heads * G) + hq] = lt > 0.f ? m + __log2f(lt) : neg_inf();
  if (!partial) {
    constexpr int kC = kOwnDims / 8;  // 16-byte chunks of a row
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
      if (S::kKeyGroups == 1 || dt / (4 / S::kKeyGroups) == kg) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int c = (4 * dt + j) % kC;
          const uint32_t w0 = pack2<DT>(o[dt][4 * j] * inv, o[dt][4 * j + 1] * inv);
          const uint32_t w1 = pack2<DT>(o[dt][4 * j + 2] * inv, o[dt][4 * j + 3] * inv);
          *reinterpret_cast<uint2*>(stage + r32 * (16 * kC) + 16 * (c ^ (r32 & (kC - 1))) + 8 * hi) = make_uint2(w0, w1);
        }
      }
    staged();
    uint16_t* const ob = a.out + b * a.so_b + static_cast<int64_t>(h) * G * a.so_h + d0;
#pragma unroll
    for (int i = 0; i < kC / 2; ++i) {
      const int r = (64 * i + lane) / kC, x = lane & (kC - 1);
      const int tk = tok0 + (rg * 32 + r) / G, g = (rg * 32 + r) % G;
      const uint4 y = *reinterpret_cast<const uint4*>(stage + r * (16 * kC) + 16 * x);
      if (tk < q_len32) *reinterpret_cast<uint4*>(ob + tk * a.so_t + g * a.so_h + 8 * (x ^ (r & (kC - 1)))) = y;
    }
  } else {
    constexpr int kC = kOwnDims / 4;
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
      if (S::kKeyGroups == 1 || dt / (4 / S::kKeyGroups) == kg) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int c = (8 * dt + 2 * j + hi) % kC;
          *reinterpret_cast<float4*>(stage + r32 * (16 * kC) + 16 * (c ^ (r32 & (kC - 1)))) = make_float4(
              o[dt][4 * j] * inv, o[dt][4 * j + 1] * inv, o[dt][4 * j + 2] * inv, o[dt][4 * j + 3] * inv);
        }
      }
    staged();
    float* const ob = a.o_part + prow0 * kHeadDim + d0;
#pragma unroll
    for (int i = 0; i < kC / 2; ++i) {
      const int r = (64 * i + lane) / kC, x = lane & (kC - 1);
      const int tk = tok0 + (rg * 32 + r) / G, g = (rg * 32 + r) % G;
      const float4 y = *reinterpret_cast<const float4*>(stage + r * (16 * kC) + 16 * x);
      if (tk < q_len32)
        *reinterpret_cast<float4*>(ob + (static_cast<int64_t>(tk) * (a.kv_heads * G) + h * G + g) * kHeadDim +
                                   4 * (x ^ (r & (kC - 1)))) = y;
    }
  }
}

// out[b, tok, hq, :] = sum_s 2^(lse_s - M) o_s / sum_s 2^(lse_s - M) over the key
// splits (M = max_s lse_s); zeros when no split saw a key. 8 rows of one KV
// head per 256-thread work-group, 4 dims per thread, the KV head fastest in the
// grid: like the splits' work-groups of head h, those of its combine then run
// on XCD h (8 KV heads), whose L2 holds the partials. Bound: one launch and one
// round trip. Rows of all heads in a work-group and a 64-bit division for the
// token cost more, whole call us: 40 tokens on 1000 of two sequences 16.5
// against 14.2 now, 93 on 5000 of 16 heads 20.1, 18.5, 600 on 2400 of 8 heads
// 24.5, 23.6, 300 on 9700 66.2-68.2, 65.8-66.8. Every split's log-sum-exp and
// partial are one batch of loads, then the merge in split order. N is the
// smallest compiled count >= splits (a split past the count reads the last
// one again and weighs nothing): with one kernel for 16, three splits of a
// 600-token chunk took 9.4 us, five sixths of it for rereads.
template <int DT, int N>
__global__ __launch_bounds__(256) void prefill_combine_kernel(const float* o_part, const float* lse_part,
                                                              int splits, int64_t q_len, int kv_heads, int gshift,
                                                              uint16_t* out, int64_t so_b, int64_t so_t,
                                                              int64_t so_h) {
  const uint32_t blk = blockIdx.x / static_cast<uint32_t>(kv_heads);
  const int h = static_cast<int>(blockIdx.x - blk * kv_heads);
  const int64_t r = static_cast<int64_t>(blk) * 8 + (threadIdx.x >> 5);  // the row among the KV head's
  const int64_t tok = r >> gshift;
  const int b = blockIdx.y;
  if (tok >= q_len) return;
  const int hq = (h << gshift) + static_cast<int>(r & ((1 << gshift) - 1));
  const int64_t rows = q_len * (static_cast<int64_t>(kv_heads) << gshift);
  const int64_t row = tok * (static_cast<int64_t>(kv_heads) << gshift) + hq;
  const int d0 = 4 * (threadIdx.x & 31);
  const float* lp = lse_part + static_cast<int64_t>(b) * splits * rows + row;
  const float* opp = o_part + (static_cast<int64_t>(b) * splits * rows + row) * kHeadDim + d0;
  float ls[N];
  float4 x[N];
#pragma unroll
  for (int s = 0; s < N; ++s) {
    const int si = s < splits ? s : splits - 1;
    ls[s] = lp[si * rows];
    x[s] = *reinterpret_cast<const float4*>(opp + si * rows * kHeadDim);
  }
  float mx = neg_inf();
#pragma unroll
  for (int s = 0; s < N; ++s) mx = s < splits ? fmaxf(mx, ls[s]) : mx;
  float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
  float wsum = 0.f;
  if (mx != neg_inf()) {
#pragma unroll
    for (int s = 0; s < N; ++s) {
      if (s < splits) {
        const float w = __builtin_amdgcn_exp2f(ls[s] - mx);
        acc.x += w * x[s].x; acc.y += w * x[s].y; acc.z += w * x[s].z; acc.w += w * x[s].w;
        wsum += w;
      }
    }
  }
  const float inv = wsum > 0.f ? 1.f / wsum : 0.f;
  uint16_t* op = out + b * so_b + tok * so_t + hq * so_h + d0;
  *reinterpret_cast<uint2*>(op) = make_uint2(pack2<DT>(acc.x * inv, acc.y * inv), pack2<DT>(acc.z * inv, acc.w * inv));
}

constexpr int kMaxPrefillSplits = 32;

// The combine compiled for N splits or the next larger count.
template <int DT, int N = 2>
void launch_combine(const PrefillArgs& a, dim3 grid, int gshift, hipStream_t stream) {
  constexpr int kNext = N < 4 ? N + 1 : N < 8 ? N + 2 : N < 16 ? N + 4 : N + 8;
  if constexpr (N < kMaxPrefillSplits)
    if (a.splits > N) return launch_combine<DT, kNext>(a, grid, gshift, stream);
  static_assert(N <= kMaxPrefillSplits, "the largest count is compiled");
  hipLaunchKernelGGL((prefill_combine_kernel<DT, N>), grid, dim3(256), 0, stream, a.o_part, a.lse_part, a.splits,
                     a.q_len, a.kv_heads, gshift, a.out, a.so_b, a.so_t, a.so_h);
}

// The classes of eight tiles (512 keys) of one query block: a thread reads 16
// keys of every eighth row, 16 bytes at any alignment, and keeps three flags;
// ballots and LDS join the 32 threads of a tile. Bound: the mask's bytes, read
// once. (One wave a tile, a byte a lane and row, took 23-26 us for 2048 x 9764;
// this 4.6 on a mask in cache, 7.3 on one just written.)
constexpr int kMapKeys = 512;
__global__ __launch_bounds__(256) void mask_tiles_kernel(const uint8_t* mask, int64_t sm_b, int64_t sm_q, int64_t q_len,
                                                         int64_t n, int tokens, int64_t nblk, int64_t pitch,
                                                         uint8_t* tiles) {
  constexpr uint32_t kHigh = 0x80808080u;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t blk = blockIdx.y, bm = blockIdx.z;
  const int64_t key0 = static_cast<int64_t>(blockIdx.x) * kMapKeys + 16 * (threadIdx.x & 31);
  const int64_t tok0 = blk * tokens;
  const int rows = static_cast<int>(min(static_cast<int64_t>(tokens), q_len - tok0));
  const int64_t past = n - q_len;
  const uint8_t* p0 = mask + bm * sm_b + tok0 * sm_q + key0;
  uint32_t some = 0, every = kHigh, apart = 0;  // bytes' high bits over the rows and keys
  auto row = [&](int r, const uint32_t (&w)[4]) {
    // Keys key0 .. that the causal rule shows row tok0 + r.
    const int64_t seen = past + tok0 + r + 1 - key0;
    const int c = static_cast<int>(max(static_cast<int64_t>(0), min(static_cast<int64_t>(16), seen)));
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      // High bit of each byte: the byte is not 0.
      const uint32_t t = (((w[i] & ~kHigh) + ~kHigh) | w[i]) & kHigh;
      const int ci = max(0, min(4, c - 4 * i));
      const uint32_t shown = kHigh & static_cast<uint32_t>((uint64_t(1) << (8 * ci)) - 1);
      some |= t;
      every &= t;
      apart |= t ^ shown;
    }
  };
  if (key0 + 16 <= n) {
#pragma unroll 4
    for (int r = threadIdx.x >> 5; r < rows; r += 8) {
      uint32_t w[4];
      __builtin_memcpy(w, p0 + r * sm_q, 16);
      row(r, w);
    }
  } else {  // keys past n count as hidden, by the mask and by the causal rule
    for (int r = threadIdx.x >> 5; r < rows; r += 8) {
      uint32_t w[4] = {0, 0, 0, 0};
#pragma unroll
      for (int i = 0; i < 16; ++i)
        if (key0 + i < n) w[i >> 2] |= static_cast<uint32_t>(p0[r * sm_q + i]) << (8 * (i & 3));
      row(r, w);
    }
    if (key0 >= n) every = 0;
  }
  __shared__ uint64_t s_flags[4][3];
  const uint64_t b_some = __builtin_amdgcn_ballot_w64(some != 0);
  const uint64_t b_hidden = __builtin_amdgcn_ballot_w64(every != kHigh);
  const uint64_t b_apart = __builtin_amdgcn_ballot_w64(apart != 0);
  if (lane == 0) {
    s_flags[wave][0] = b_some;
    s_flags[wave][1] = b_hidden;
    s_flags[wave][2] = b_apart;
  }
  __syncthreads();
  if (threadIdx.x < kMapKeys / kKeys) {
    const int j = threadIdx.x;
    bool f[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const uint64_t x = s_flags[0][k] | s_flags[1][k] | s_flags[2][k] | s_flags[3][k];
      f[k] = ((x >> (4 * j)) & 0xf0000000full) != 0;
    }
    const int cls = !f[0] ? TILE_SKIP : !f[1] ? TILE_FULL : !f[2] ? TILE_CAUSAL : TILE_MIXED;
    tiles[(bm * nblk + blk) * pitch + blockIdx.x * (kMapKeys / kKeys) + j] = static_cast<uint8_t>(cls);
  }
}

#if TC_PREFILL_STAMPS
unsigned long long* g_prefill_stamps = nullptr;  // the buffer prefill launches record into (null: none)
#endif

typedef Shape<4, 1, 2> Wide;    // 128 rows, 64-key tiles, 4 waves: two work-groups a CU
typedef Shape<4, 2, 2> Tall;    // 128 rows, 128-key tiles, 8 waves: one work-group a CU
typedef Shape<2, 4, 1> Deep;    // 64 rows, 128-key tiles, 8 waves: one work-group a CU
typedef Shape<2, 2, 1> Narrow;  // 64 rows, 64-key tiles, 4 waves: two work-groups a CU
enum : int { SHAPE_WIDE = 0, SHAPE_TALL = 1, SHAPE_DEEP = 2, SHAPE_NARROW = 3 };

template <int DT, bool PAGED, class S>
void launch_attention(const PrefillArgs& a_in, int group, dim3 grid, hipStream_t stream) {
  PrefillArgs a = a_in;
#if TC_PREFILL_STAMPS
  a.stamps = g_prefill_stamps;
#endif
  const dim3 block(64 * S::kWaves);
  switch (group) {
    case 1: hipLaunchKernelGGL((prefill_kernel<DT, 1, PAGED, S>), grid, block, 0, stream, a); break;
    case 2: hipLaunchKernelGGL((prefill_kernel<DT, 2, PAGED, S>), grid, block, 0, stream, a); break;
    case 4: hipLaunchKernelGGL((prefill_kernel<DT, 4, PAGED, S>), grid, block, 0, stream, a); break;
    default: hipLaunchKernelGGL((prefill_kernel<DT, 8, PAGED, S>), grid, block, 0, stream, a); break;
  }
}

template <int DT, class S>
void launch_shape(const PrefillArgs& a, int group, dim3 grid, hipStream_t stream) {
  if (a.tok_off)
    launch_attention<DT, true, S>(a, group, grid, stream);
  else
    launch_attention<DT, false, S>(a, group, grid, stream);
}

template <int DT>
hipError_t launch_dt(const PrefillArgs& a, int shape, int group, int batch, hipStream_t stream) {
  const dim3 grid(static_cast<unsigned>(a.nblk * a.kv_heads * batch * a.splits));
  switch (shape) {
    case SHAPE_TALL: launch_shape<DT, Tall>(a, group, grid, stream); break;
    case SHAPE_DEEP: launch_shape<DT, Deep>(a, group, grid, stream); break;
    case SHAPE_NARROW: launch_shape<DT, Narrow>(a, group, grid, stream); break;
    default: launch_shape<DT, Wide>(a, group, grid, stream);
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || a.splits == 1) return e;
  const dim3 cgrid(static_cast<unsigned>((a.q_len * group + 7) / 8 * a.kv_heads), static_cast<unsigned>(batch));
  launch_combine<DT>(a, cgrid, __builtin_ctz(group), stream);
  return hipGetLastError();
}

int check3(const char* what, const int64_t* st) {
  if (!st) return fail(TC_ERR_INVALID_ARGUMENT, "%s strides are null", what);
  for (int i = 0; i < 3; ++i) {
    if (st[i] < 0) return fail(TC_ERR_INVALID_ARGUMENT, "%s stride %d negative", what, i);
    if (st[i] % 8) return fail(TC_ERR_ALIGNMENT, "%s stride %d (%lld) not a multiple of 8", what, i, (long long)st[i]);
  }
  return TC_OK;
}

int check_group(int q_heads, int kv_heads, int* group) {
  if (kv_heads < 1 || kv_heads > 65535 || q_heads < 1)
    return fail(TC_ERR_INVALID_ARGUMENT, "q_heads %d, kv_heads %d", q_heads, kv_heads);
  if (q_heads % kv_heads)
    return fail(TC_ERR_INVALID_ARGUMENT, "q_heads %d not a multiple of kv_heads %d", q_heads, kv_heads);
  *group = q_heads / kv_heads;
  if (*group != 1 && *group != 2 && *group != 4 && *group != 8)
    return fail(TC_ERR_UNSUPPORTED, "group %d unsupported (1, 2, 4 or 8)", *group);
  return TC_OK;
}

int check_mask_strides(const int64_t* st) {
  if (!st) return fail(TC_ERR_INVALID_ARGUMENT, "mask strides are null");
  if (st[0] < 0 || st[1] < 0 || st[2] < 0) return fail(TC_ERR_INVALID_ARGUMENT, "mask strides must be non-negative");
  if (st[2] != 1) return fail(TC_ERR_UNSUPPORTED, "mask keys must be contiguous (key stride %lld)", (long long)st[2]);
  return TC_OK;
}

// Tile map geometry: query blocks of 128/g tokens, 64-key tiles.
int64_t map_pitch(int64_t ntiles) { return (ntiles + 7) & ~int64_t(7); }

void tile_geometry(int64_t q_len, int64_t n, int group, int64_t* nblk, int64_t* ntiles) {
  const int64_t tokens = kMapRows / group;
  *nblk = (q_len + tokens - 1) / tokens;
  *ntiles = (n + kKeys - 1) / kKeys;
}

constexpr int kMinSplitTiles = 4;    // keys per split: at least 256

struct Plan {
  int shape;
  int64_t nblk;          // query blocks
  int64_t split_tiles;   // tiles of the shape per key split
  int splits;
};

// Shape of the work-groups and key splits of a call. A tile costs a wave about
// the same whatever share of its MFMAs it holds (its chain of LDS reads, MFMAs
// and exponentials is what takes the time), so what decides is how many tiles
// in a row the longest work-group walks and whether every CU has eight waves.
// With W and W64 the work-groups of 128 and of 64 query rows, C CUs and T
// 64-key tiles (us, 32 query over 8 KV heads if not said otherwise):
// - A prompt (at least half of the keys are its own) is never split over
//   work-groups: the combine costs more than it saves.
//   - T <= 10, W <= C: Narrow (64 rows, two key groups). 300 tokens 10.1 against
//     11.8 Wide, 10.7 Deep; four prompts of 300 (W > C): Wide, 13.6 against 16.4.
//   - No mask and not causal, so that every block walks all tiles: a work-group more
//     than the CUs costs a round. Deep for W64 <= C, Tall for W <= C, else Wide. 656
//     of 32 heads (W64 = 328): 18.1 Tall, 27.3 Deep, 20.0 Wide; 1329 of 32 over 8 (W
//     = 336): 48 Wide, 52 Tall.
//   - W64 <= 4/3 C: Deep, a quarter of the tiles in a row. 1100 tokens of 16
//     heads over 8: 18.3 against 26.8 Wide, 22.4 Tall; 1300: 21.5, 30.5, 24.2.
//   - W > 2 C, or W > C with few tiles: Wide, two independent work-groups a CU.
//     Four prompts of 1500, 16 over 8: 46.0 against 54.4 Tall; two of 800: 23.7,
//     24.8; 1300 of 64 over 8: 41.9, 50.6.
//   - else Tall, half of the tiles in a row. 1100: 23.8 against 28.3 Wide, 32.7
//     Deep; 2048: 46.6, 51.2, 65.4.
// - A chunk on a longer cache is split to fill the CUs once (a second round
//   would double the call), into at most 32 splits of at least 256 keys.
//   - T <= 5: Narrow, Wide where W64 > C. A Deep tile of 128 keys is mostly empty
//     there: 14 tokens on 43 of 32 heads 6.5 us against 7.8 Deep, 6.3 Wide; 0.92 of
//     Deep's time at T = 2 (366 shapes), 0.97 at 5, 1.02 at 6 and 7.
//   - Deep for few rows (W64 <= C / 6) or short caches (n <= 4096 and two splits, W64
//     <= C / 2; n <= 3072, W64 <= 7/8 C: 0.78 of Wide's time with T in [16, 24), 1.03
//     in [56, 64)):
//     3 tokens on 9000: 15.6 against 17.3 Wide, 16.9 Tall; 150 on 1500: 19.7,
//     22.3, 22.2; 400 on 3000: 38.1, 43.0, 41.7.
//   - Tall where its splits fill at least 0.85 as much of the CUs as Wide's fill of
//     their two slots: 93 on 9000: 29.8 against 31.6 Wide, 31.0 Deep; 1024 on 9000:
//     169, 183; 300 on 9700: 65.8, 68.9. With W = 96 (2 splits Tall, 5 Wide): 189 on
//     16238 142 Tall, 132 Wide.
//   - else Wide: 600 on 7600 (W = 152): 99.7 in 3 splits against 114 Tall.
// requested > 0 fixes the splits. Trailing empty splits are dropped: the result
// times its tiles covers n. Shapes other than Wide address a tile by one 32-bit
// range over the slab (one_range); without it Wide walks the very splits that
// the call would have had, so that tc_prefill_num_splits, which does not know
// the strides, tells the count of either.
// even: every query sees every key (the splits do not depend on it).
int plan(int batch, int64_t q_len, int64_t n, int group, int kv_heads, int requested, bool one_range, bool even,
         Plan* out) {
  int cus32 = 0;
  const int rc = current_device_cus(&cus32);
  if (rc != TC_OK) return rc;
  const int64_t cus = cus32, pairs = static_cast<int64_t>(kv_heads) * batch;
  const int64_t T = ceil_div(n, kKeys);
  const int64_t w = ceil_div(q_len, 128 / group) * pairs, w64 = ceil_div(q_len, 64 / group) * pairs;
  const int64_t most = std::max<int64_t>(1, std::min<int64_t>(kMaxPrefillSplits, T / kMinSplitTiles));
  auto fill = [&](int64_t wgs, int64_t slots) { return std::max<int64_t>(1, std::min(most, wgs > 0 ? slots / wgs : 1)); };
  int shape;
  int64_t s = 1;
  if (2 * q_len >= n) {
    if (T <= 10)
      shape = w <= cus ? SHAPE_NARROW : SHAPE_WIDE;
    else if (even)
      shape = w64 <= cus ? SHAPE_DEEP : w <= cus ? SHAPE_TALL : SHAPE_WIDE;
    else if (3 * w64 <= 4 * cus)
      shape = SHAPE_DEEP;
    else
      shape = w > 2 * cus || (w > cus && T <= 16) ? SHAPE_WIDE : SHAPE_TALL;
  } else if (T <= 5) {
    shape = w64 <= cus ? SHAPE_NARROW : SHAPE_WIDE;
  } else if (6 * w64 <= cus || (n <= 4096 && 2 * w64 <= cus) || (n <= 3072 && 8 * w64 <= 7 * cus)) {
    shape = SHAPE_DEEP;
    s = fill(w64, cus);
  } else if (w <= cus && 40 * fill(w, cus) >= 17 * fill(w, 2 * cus)) {
    shape = SHAPE_TALL;
    s = fill(w, cus);
  } else {
    shape = SHAPE_WIDE;
    s = fill(w, 2 * cus);
  }
  const int64_t rows = shape == SHAPE_WIDE || shape == SHAPE_TALL || !one_range ? 128 : 64;
  const int64_t keys = shape == SHAPE_WIDE || shape == SHAPE_NARROW ? 64 : 128;
  if (requested > 0) s = std::min<int64_t>(requested, kMaxPrefillSplits);
  const int64_t ntiles = std::max<int64_t>(1, ceil_div(n, keys));
  int64_t st = ceil_div(ntiles, std::min(s, ntiles));
  const int64_t splits = ceil_div(ntiles, st);
  if (!one_range) {
    st *= keys / 64;
    shape = SHAPE_WIDE;
  }
  *out = Plan{shape, ceil_div(q_len, rows / group), st, static_cast<int>(splits)};
  return TC_OK;
}

size_t workspace_bytes(int batch, int64_t q_len, int q_heads, int splits) {
  if (splits <= 1) return 0;
  return static_cast<size_t>(batch) * splits * q_len * q_heads * (kHeadDim + 1) * sizeof(float);
}

}  // namespace
}  // namespace tc

using namespace tc;

extern "C" int tc_prefill_num_splits(int batch, int64_t q_len, int64_t n_tokens, int q_heads, int kv_heads) {
  clear_error();
  int group = 0, rc;
  if (batch < 1 || q_len < 0 || n_tokens < q_len) return -fail(TC_ERR_INVALID_ARGUMENT, "batch %d, q_len %lld, n %lld", batch, (long long)q_len, (long long)n_tokens);
  if ((rc = check_group(q_heads, kv_heads, &group)) != TC_OK) return -rc;
  Plan p;
  if ((rc = plan(batch, q_len, n_tokens, group, kv_heads, 0, true, false, &p)) != TC_OK) return -rc;
  return p.splits;
}

extern "C" size_t tc_prefill_workspace_bytes(int batch, int64_t q_len, int q_heads, int num_splits) {
  if (batch < 1 || q_len < 0 || q_heads < 1) return 0;
  return workspace_bytes(batch, q_len, q_heads, num_splits);
}

extern "C" size_t tc_prefill_tiles_bytes(int64_t q_len, int64_t n_tokens, int mask_batch, int q_heads,
                                         int kv_heads) {
  int group = 0;
  if (q_len < 0 || n_tokens < q_len || mask_batch < 1 || check_group(q_heads, kv_heads, &group) != TC_OK) return 0;
  int64_t nblk, ntiles;
  tile_geometry(q_len, n_tokens, group, &nblk, &ntiles);
  return static_cast<size_t>(mask_batch * nblk * map_pitch(ntiles));
}

extern "C" int tc_prefill_mask_tiles(const uint8_t* mask_dev, const int64_t mask_strides[3], int mask_batch,
                                     int64_t q_len, int64_t n_tokens, int q_heads, int kv_heads, uint8_t* tiles_dev,
                                     size_t tiles_bytes, void* stream) {
  clear_error();
  int group = 0, rc;
  if ((rc = check_group(q_heads, kv_heads, &group)) != TC_OK) return rc;
  if (mask_batch < 1 || mask_batch > 65535) return fail(TC_ERR_INVALID_ARGUMENT, "mask_batch %d", mask_batch);
  if (q_len < 0 || n_tokens < q_len)
    return fail(TC_ERR_INVALID_ARGUMENT, "q_len %lld must be in [0, n_tokens %lld]", (long long)q_len,
                (long long)n_tokens);
  if ((rc = check_mask_strides(mask_strides)) != TC_OK) return rc;
  if (mask_batch > 1 && mask_strides[0] == 0)
    return fail(TC_ERR_INVALID_ARGUMENT, "mask_batch %d with a broadcast (stride 0) mask batch", mask_batch);
  int64_t nblk, ntiles;
  tile_geometry(q_len, n_tokens, group, &nblk, &ntiles);
  const int64_t pitch = map_pitch(ntiles);
  const size_t need = static_cast<size_t>(mask_batch * nblk * pitch);
  if (need == 0) return TC_OK;
  if (!mask_dev || !tiles_dev) return fail(TC_ERR_INVALID_ARGUMENT, "null mask or tile map pointer");
  if (tiles_bytes < need)
    return fail(TC_ERR_WORKSPACE, "tile map holds %zu bytes, needs %zu", tiles_bytes, need);
  if (ntiles > 0x7fffffff || nblk > 65535)
    return fail(TC_ERR_UNSUPPORTED, "mask of %lld x %lld exceeds the tile grid", (long long)q_len,
                (long long)n_tokens);
  if (reinterpret_cast<uintptr_t>(tiles_dev) & 7u) return fail(TC_ERR_ALIGNMENT, "tile map must be 8-byte aligned");
  // The padding tiles (keys past n) classify as SKIP, so whole rows are written.
  static_assert(kMapKeys == 8 * kKeys, "a work-group writes the eight tiles that a map row is a multiple of");
  const dim3 grid(static_cast<unsigned>(pitch / 8), static_cast<unsigned>(nblk), static_cast<unsigned>(mask_batch));
  hipLaunchKernelGGL(mask_tiles_kernel, grid, dim3(256), 0, static_cast<hipStream_t>(stream), mask_dev, mask_strides[0],
                     mask_strides[1], q_len, n_tokens, kMapRows / group, nblk, pitch, tiles_dev);
  return hip_status(hipGetLastError(), "mask tile launch");
}

namespace tc {
namespace {

// The page pools of a paged prefill call.
struct PagedPools {
  const int32_t* tok_off;  // [batch, tok_pitch] byte offsets of each logical key's row in its head slab
  int64_t tok_pitch;
  int64_t pool_bytes;      // bytes of one pool (K and V pools share the shape)
};

int prefill_impl(const void* q_dev, const int64_t q_strides[3], const void* k_dev, const int64_t k_strides[3],
                 const void* v_dev, const int64_t v_strides[3], const uint8_t* mask_dev,
                 const int64_t mask_strides[3], const uint8_t* mask_tiles_dev, size_t mask_tiles_bytes, int causal,
                 int64_t q_len, int64_t n_tokens, int batch, int q_heads, int kv_heads, int head_dim, int dtype,
                 float scale, int num_splits, void* workspace_dev, size_t workspace_bytes_in, void* out_dev,
                 const int64_t out_strides[3], void* stream, const PagedPools* pools) {
  int group = 0, rc;
  if (batch < 1 || batch > 65535) return fail(TC_ERR_INVALID_ARGUMENT, "batch %d", batch);
  if ((rc = check_group(q_heads, kv_heads, &group)) != TC_OK) return rc;
  if (head_dim != kHeadDim) return fail(TC_ERR_UNSUPPORTED, "head_dim %d unsupported (kernels are built for 128)", head_dim);
  if (dtype != TC_DTYPE_F16 && dtype != TC_DTYPE_BF16) return fail(TC_ERR_UNSUPPORTED, "dtype %d unsupported", dtype);
  if (q_len < 0 || n_tokens < q_len)
    return fail(TC_ERR_INVALID_ARGUMENT, "q_len %lld must be in [0, n_tokens %lld]", (long long)q_len,
                (long long)n_tokens);
  if (q_len == 0) return TC_OK;
  // Key positions and tile indices are 32-bit in the kernel.
  if (n_tokens >= (int64_t(1) << 30))
    return fail(TC_ERR_UNSUPPORTED, "n_tokens %lld: the prefill kernels take fewer than 2^30 keys", (long long)n_tokens);
  if (!q_dev || !k_dev || !v_dev || !out_dev) return fail(TC_ERR_INVALID_ARGUMENT, "null tensor pointer");
  if (!aligned16(q_dev) || !aligned16(k_dev) || !aligned16(v_dev) || !aligned16(out_dev))
    return fail(TC_ERR_ALIGNMENT, "q/k/v/out base pointers must be 16-byte aligned");
  if ((rc = check3("q", q_strides)) != TC_OK) return rc;
  if ((rc = check3("k", k_strides)) != TC_OK) return rc;
  if ((rc = check3("v", v_strides)) != TC_OK) return rc;
  if ((rc = check3("out", out_strides)) != TC_OK) return rc;
  // A 64-key tile is addressed with 32-bit buffer offsets: 64 rows of at most 2^24 elements.
  constexpr int64_t kMaxTokenStride = int64_t(1) << 24;
  if (k_strides[2] < head_dim || v_strides[2] < head_dim || k_strides[2] >= kMaxTokenStride ||
      v_strides[2] >= kMaxTokenStride)
    return fail(TC_ERR_INVALID_ARGUMENT, "k/v token strides outside [%d, 2^24)", head_dim);
  if (!std::isfinite(scale)) return fail(TC_ERR_INVALID_ARGUMENT, "scale is not finite");
  int64_t nblk, ntiles;
  tile_geometry(q_len, n_tokens, group, &nblk, &ntiles);
  // 2^27 query blocks; the grid that the splits make of them is checked with the plan.
  if (nblk * kv_heads * batch * 16 > 0x7fffffff) return fail(TC_ERR_UNSUPPORTED, "grid too large");
  if (mask_dev) {
    if (causal) return fail(TC_ERR_INVALID_ARGUMENT, "pass either a mask or causal, not both");
    if ((rc = check_mask_strides(mask_strides)) != TC_OK) return rc;
    if (mask_tiles_dev) {
      const size_t need = static_cast<size_t>((mask_strides[0] ? batch : 1) * nblk * map_pitch(ntiles));
      if (reinterpret_cast<uintptr_t>(mask_tiles_dev) & 7u)
        return fail(TC_ERR_ALIGNMENT, "tile map must be 8-byte aligned");
      if (mask_tiles_bytes < need)
        return fail(TC_ERR_WORKSPACE, "tile map holds %zu bytes, this call reads %zu", mask_tiles_bytes, need);
    }
  } else if (mask_tiles_dev) {
    return fail(TC_ERR_INVALID_ARGUMENT, "a tile map without its mask");
  }

  // One 32-bit buffer range over a head's slab, with room for the tiles' rows past n.
  const bool whole = !pools && (n_tokens + 2 * kKeys) * 2 * std::max(k_strides[2], v_strides[2]) < (int64_t(1) << 31);
  Plan p;
  if ((rc = plan(batch, q_len, n_tokens, group, kv_heads, num_splits, pools || whole, !causal && !mask_dev,
                 &p)) != TC_OK) return rc;
  const int splits = p.splits;
  if (p.nblk * kv_heads * batch * splits > 0x7fffffff) return fail(TC_ERR_UNSUPPORTED, "grid too large");
  const size_t need = workspace_bytes(batch, q_len, q_heads, splits);
  if (need > 0 && (!workspace_dev || workspace_bytes_in < need))
    return fail(TC_ERR_WORKSPACE, "%d key splits need %zu workspace bytes, got %zu", splits, need,
                workspace_dev ? workspace_bytes_in : size_t(0));
  if (need > 0 && (reinterpret_cast<uintptr_t>(workspace_dev) & 15u))
    return fail(TC_ERR_ALIGNMENT, "workspace must be 16-byte aligned");

  PrefillArgs a;
  a.split_tiles = p.split_tiles;
  a.splits = splits;
  a.o_part = static_cast<float*>(workspace_dev);
  a.lse_part = splits > 1 ? a.o_part + static_cast<size_t>(batch) * splits * q_len * q_heads * kHeadDim : nullptr;
  a.q = static_cast<const uint16_t*>(q_dev);
  a.k = static_cast<const uint16_t*>(k_dev);
  a.v = static_cast<const uint16_t*>(v_dev);
  a.mask = mask_dev;
  a.tiles = mask_dev ? mask_tiles_dev : nullptr;
  a.out = static_cast<uint16_t*>(out_dev);
  a.sq_b = q_strides[0]; a.sq_h = q_strides[1]; a.sq_t = q_strides[2];
  a.sk_b = k_strides[0]; a.sk_h = k_strides[1]; a.sk_t = k_strides[2];
  a.sv_b = v_strides[0]; a.sv_h = v_strides[1]; a.sv_t = v_strides[2];
  a.sm_b = mask_dev ? mask_strides[0] : 0;
  a.sm_q = mask_dev ? mask_strides[1] : 0;
  a.mask_words = mask_dev && reinterpret_cast<uintptr_t>(mask_dev) % 4 == 0 && a.sm_b % 4 == 0 && a.sm_q % 4 == 0;
  a.whole = whole;
  a.so_b = out_strides[0]; a.so_t = out_strides[1]; a.so_h = out_strides[2];
  a.q_len = q_len;
  a.n = n_tokens;
  a.nblk = p.nblk;
  a.map_nblk = nblk;
  a.pitch = map_pitch(ntiles);
  a.kv_heads = kv_heads;
  a.batch = batch;
  a.causal = causal ? 1 : 0;
  a.descend = causal || mask_dev;
  a.by_block = 0;
  a.fold_cus = 0;
  if (splits == 1 && (causal || mask_dev)) {
    int cus = 0;
    if ((rc = current_device_cus(&cus)) != TC_OK) return rc;
    const int64_t wgs = p.nblk * kv_heads * batch, slots = TC_PREFILL_WAVES * static_cast<int64_t>(cus);
    // The longest blocks of all sequences first where a block's length varies
    // much (prompts) and there are few rounds, so that the last round is short:
    // 3 to 6% less time than a sequence at a time for C < W <= 4 C (730 shapes).
    // With more rounds, or a chunk on a cache, the blocks in flight should share
    // a sequence's K/V: 16 x 61 tokens on 2176 of 32 KV heads 222 us by block,
    // 181 by sequence; 16 x 1398 on 2669, W = 22 C, 1106 and 854.
    a.by_block = 2 * q_len >= n_tokens && wgs <= 4 * static_cast<int64_t>(cus);
    // One round of two work-groups per CU with rows that see more keys further down.
    if (p.shape == SHAPE_WIDE && wgs > cus && wgs <= slots) a.fold_cus = cus;
  }
  a.c = static_cast<float>(std::fabs(static_cast<double>(scale)) * 1.4426950408889634);
  a.neg = a.c == 0.f ? -1 : scale < 0.f ? 1 : 0;
  if (a.c == 0.f) a.c = 1.f;
  a.tok_off = pools ? pools->tok_off : nullptr;
  a.tok_pitch = pools ? pools->tok_pitch : 0;
  a.pool_bytes_k = a.pool_bytes_v = pools ? pools->pool_bytes : 0;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const hipError_t e = dtype == TC_DTYPE_F16 ? launch_dt<TC_DTYPE_F16>(a, p.shape, group, batch, s)
                                             : launch_dt<TC_DTYPE_BF16>(a, p.shape, group, batch, s);
  return hip_status(e, "prefill launch");
}

}  // namespace
}  // namespace tc

extern "C" int tc_prefill_attention(const void* q_dev, const int64_t q_strides[3], const void* k_dev,
                                    const int64_t k_strides[3], const void* v_dev, const int64_t v_strides[3],
                                    const uint8_t* mask_dev, const int64_t mask_strides[3],
                                    const uint8_t* mask_tiles_dev, size_t mask_tiles_bytes, int causal,
                                    int64_t q_len, int64_t n_tokens, int batch, int q_heads, int kv_heads,
                                    int head_dim, int dtype, float scale, int num_splits, void* workspace_dev,
                                    size_t workspace_bytes_in, void* out_dev, const int64_t out_strides[3],
                                    void* stream) {
  clear_error();
  return prefill_impl(q_dev, q_strides, k_dev, k_strides, v_dev, v_strides, mask_dev, mask_strides, mask_tiles_dev,
                      mask_tiles_bytes, causal, q_len, n_tokens, batch, q_heads, kv_heads, head_dim, dtype, scale,
                      num_splits, workspace_dev, workspace_bytes_in, out_dev, out_strides, stream, nullptr);
}

extern "C" int tc_prefill_paged_attention(const void* q_dev, const int64_t q_strides[3], const void* k_pool_dev,
                                          const void* v_pool_dev, const int64_t pool_strides[3], int num_pages,
                                          const int32_t* tok_off_dev, int64_t tok_pitch, const uint8_t* mask_dev,
                                          const int64_t mask_strides[3], const uint8_t* mask_tiles_dev,
                                          size_t mask_tiles_bytes, int causal, int64_t q_len, int64_t n_tokens,
                                          int batch, int q_heads, int kv_heads, int head_dim, int dtype, float scale,
                                          int num_splits, void* workspace_dev, size_t workspace_bytes_in,
                                          void* out_dev, const int64_t out_strides[3], void* stream) {
  clear_error();
  if (!pool_strides) return fail(TC_ERR_INVALID_ARGUMENT, "null pool strides");
  if (num_pages < 1) return fail(TC_ERR_INVALID_ARGUMENT, "pool of %d pages", num_pages);
  if (q_len > 0 && (!tok_off_dev || tok_pitch < n_tokens))
    return fail(TC_ERR_INVALID_ARGUMENT, "token offsets: null or a row of %lld for %lld keys", (long long)tok_pitch,
                (long long)n_tokens);
  if (reinterpret_cast<uintptr_t>(tok_off_dev) & 3u) return fail(TC_ERR_ALIGNMENT, "token offsets not 4-byte aligned");
  // Rows are found by 32-bit byte offsets from a head's slab.
  const int64_t pool_bytes = static_cast<int64_t>(num_pages) * pool_strides[0] * 2;
  if (pool_strides[0] < 1 || pool_bytes >= (int64_t(1) << 31) ||
      static_cast<int64_t>(kv_heads - 1) * pool_strides[1] * 2 >= pool_bytes)
    return fail(TC_ERR_UNSUPPORTED, "pool of %lld bytes (page stride %lld): paged prefill needs a pool under 2 GiB",
                (long long)pool_bytes, (long long)pool_strides[0]);
  const PagedPools pools{tok_off_dev, tok_pitch, pool_bytes};
  return prefill_impl(q_dev, q_strides, k_pool_dev, pool_strides, v_pool_dev, pool_strides, mask_dev, mask_strides,
                      mask_tiles_dev, mask_tiles_bytes, causal, q_len, n_tokens, batch, q_heads, kv_heads, head_dim,
                      dtype, scale, num_splits, workspace_dev, workspace_bytes_in, out_dev, out_strides, stream,
                      &pools);
}

#if TC_PREFILL_STAMPS
// Measurement build only (libthreadcut_stamps.so): the device buffer that the
// prefill kernels launched from now on record their per-wave, per-tile phase
// stamps into (kStampWords words per wave, see PrefillArgs::stamps), or null.
extern "C" void tc_prefill_set_stamps(void* stamps_dev) {
  tc::g_prefill_stamps = static_cast<unsigned long long*>(stamps_dev);
}
#endif
