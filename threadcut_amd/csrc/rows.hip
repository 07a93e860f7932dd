// New tokens' K/V rows written into the cache: the append of
// threadcut/kv.py:68-77 (two strided copies per layer there) as one launch for
// K and V of one or more layers, into contiguous buffers (rows row0 .. of
// every head strip) or into the page slots that a paged cache reserved.
//
// A model hands the rows over as transposed views ([b, heads, n, d] over
// [b, n, heads, d] memory), so a head's rows are 256-byte pieces a few KB
// apart. Bound: HBM (each byte read and written once). A thread moves 16-byte
// chunks, 16 lanes a row, so every access is a whole 256-byte row piece, and
// keeps kPasses rows' loads in flight before it stores. Loads and stores are
// non-temporal (24 layers, rows read from HBM: 6620 rows 11.8 us, 4.6 TB/s,
// against 13.3 cached, 12.5 with either one; 1000 rows 3.05 against 3.8; two
// passes 13.1, eight 15.0, row tiles fastest 14.3). torch's strided copy
// of such a view (its elementwise kernel, 8 elements a thread with per-element
// index arithmetic) moved 6620 rows x 8 heads at 2.0 TB/s.
#include "tc_common.hpp"

namespace tc {
namespace {

constexpr int kHeadDim = 128;
constexpr int kThreads = 256;
constexpr int kChunks = kHeadDim / 8;               // 16-byte chunks (lanes) per row
constexpr int kRowsPerPass = kThreads / kChunks;    // 16
constexpr int kPasses = 4;                          // rows a thread has in flight
constexpr int kTileRows = kRowsPerPass * kPasses;   // rows of one head per work-group
constexpr int kMaxLayers = 64;

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef int64_t i64x2 __attribute__((ext_vector_type(2)));

template <int LAYERS>
struct RowArgs {
  const uint16_t* src[2 * LAYERS];  // K of every layer, then V
  uint16_t* dst[2 * LAYERS];
  int64_t s_b[2], s_h[2], s_t[2];   // source strides of K and V
  int64_t d_b, d_h, d_t;            // destination strides (paged: page, head, slot)
  const int64_t* slots;             // paged: [batch, rows, 2] of (page, slot); null: contiguous
  int64_t rows;
  int layers;
  int pages, page_tokens;
};

// Grid (heads, row tiles, batch * jobs), the head fastest: the work-groups in
// flight together read the same tokens' neighbouring row pieces.
template <int LAYERS, bool PAGED>
__global__ __launch_bounds__(kThreads) void write_rows_kernel(const RowArgs<LAYERS> a) {
  const int h = blockIdx.x;
  const int jobs = 2 * a.layers;
  const int job = LAYERS == 1 ? static_cast<int>(blockIdx.z) & 1 : static_cast<int>(blockIdx.z) % jobs;
  const int64_t b = LAYERS == 1 ? blockIdx.z >> 1 : blockIdx.z / jobs;
  const int is_v = job >= a.layers ? 1 : 0;
  const int chunk = 8 * (threadIdx.x & (kChunks - 1));
  const int64_t tile0 = static_cast<int64_t>(blockIdx.y) * kTileRows;
  const int64_t r0 = tile0 + threadIdx.x / kChunks;
  const uint16_t* src = a.src[job] + b * a.s_b[is_v] + h * a.s_h[is_v] + chunk;
  uint16_t* dst = a.dst[job] + (PAGED ? 0 : b * a.d_b) + h * a.d_h + chunk;

  const int64_t st = a.s_t[is_v];
  const int64_t* slots = PAGED ? a.slots + 2 * b * a.rows : nullptr;
  // Where row r goes, -1 for a slot outside the pool.
  auto place = [&](int64_t r, const i64x2& s) -> int64_t {
    if constexpr (!PAGED) return r * a.d_t;
    const bool ok = (s.x >= 0) & (s.x < a.pages) & (s.y >= 0) & (s.y < a.page_tokens);
    return ok ? s.x * a.d_b + s.y * a.d_t : -1;
  };
  if (tile0 + kTileRows <= a.rows) {
    // A whole tile: every load goes out before the first store, with no
    // branch between them. (Loads under a per-row branch made the compiler
    // keep x in LDS and cost 22.8 us for 6620 rows x 8 heads against 8.6 us.)
    u32x4 x[kPasses];
    i64x2 s[kPasses];
#pragma unroll
    for (int i = 0; i < kPasses; ++i) {
      const int64_t r = r0 + i * kRowsPerPass;
      s[i] = i64x2{0, 0};
      if constexpr (PAGED) s[i] = *reinterpret_cast<const i64x2*>(slots + 2 * r);
      x[i] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(src + r * st));
    }
#pragma unroll
    for (int i = 0; i < kPasses; ++i) {
      const int64_t off = place(r0 + i * kRowsPerPass, s[i]);
      if (!PAGED || off >= 0) __builtin_nontemporal_store(x[i], reinterpret_cast<u32x4*>(dst + off));
    }
  } else {
    for (int64_t r = r0; r < a.rows; r += kRowsPerPass) {
      i64x2 s{0, 0};
      if constexpr (PAGED) s = *reinterpret_cast<const i64x2*>(slots + 2 * r);
      const u32x4 x = *reinterpret_cast<const u32x4*>(src + r * st);
      const int64_t off = place(r, s);
      if (!PAGED || off >= 0) *reinterpret_cast<u32x4*>(dst + off) = x;
    }
  }
}

int check_strides(const char* what, const int64_t* st) {
  if (!st) return fail(TC_ERR_INVALID_ARGUMENT, "%s strides are null", what);
  for (int i = 0; i < 3; ++i) {
    if (st[i] < 0) return fail(TC_ERR_INVALID_ARGUMENT, "%s stride %d is negative", what, i);
    if (st[i] % 8) return fail(TC_ERR_ALIGNMENT, "%s stride %d (%lld) not a multiple of 8", what, i, (long long)st[i]);
  }
  return TC_OK;
}

template <int LAYERS>
void launch(const RowArgs<LAYERS>& a, dim3 grid, hipStream_t s) {
  if (a.slots)
    hipLaunchKernelGGL((write_rows_kernel<LAYERS, true>), grid, dim3(kThreads), 0, s, a);
  else
    hipLaunchKernelGGL((write_rows_kernel<LAYERS, false>), grid, dim3(kThreads), 0, s, a);
}

struct Dest {
  const int64_t* strides;
  const int64_t* slots = nullptr;
  int pages = 0, page_tokens = 0;
};

int write_rows(const void* const* ks, const int64_t* k_st, const void* const* vs, const int64_t* v_st,
               void* const* kd, void* const* vd, const Dest& d, int64_t row0, int layers, int batch, int heads,
               int64_t rows, int head_dim, int dtype, hipStream_t s) {
  int rc;
  if (layers < 0) return fail(TC_ERR_INVALID_ARGUMENT, "num_layers %d is negative", layers);
  if (batch < 1 || heads < 1) return fail(TC_ERR_INVALID_ARGUMENT, "batch %d, heads %d", batch, heads);
  if (head_dim != kHeadDim) return fail(TC_ERR_UNSUPPORTED, "head_dim %d unsupported (kernels are built for 128)", head_dim);
  if (dtype != TC_DTYPE_F16 && dtype != TC_DTYPE_BF16) return fail(TC_ERR_UNSUPPORTED, "dtype %d unsupported", dtype);
  if (rows < 0) return fail(TC_ERR_INVALID_ARGUMENT, "rows %lld is negative", (long long)rows);
  if (rows == 0 || layers == 0) return TC_OK;
  if ((rc = check_strides("k rows", k_st)) != TC_OK) return rc;
  if ((rc = check_strides("v rows", v_st)) != TC_OK) return rc;
  if ((rc = check_strides("cache", d.strides)) != TC_OK) return rc;
  if (d.strides[2] < kHeadDim)
    return fail(TC_ERR_INVALID_ARGUMENT, "cache token stride %lld overlaps rows", (long long)d.strides[2]);
  if (!ks || !vs || !kd || !vd) return fail(TC_ERR_INVALID_ARGUMENT, "null pointer array");
  for (int l = 0; l < layers; ++l) {
    if (!ks[l] || !vs[l] || !kd[l] || !vd[l]) return fail(TC_ERR_INVALID_ARGUMENT, "null pointer of layer %d", l);
    if (!aligned16(ks[l]) || !aligned16(vs[l]) || !aligned16(kd[l]) || !aligned16(vd[l]))
      return fail(TC_ERR_ALIGNMENT, "layer %d: rows or cache not 16-byte aligned", l);
  }
  const int64_t tiles = ceil_div(rows, kTileRows);
  if (tiles > 65535) return fail(TC_ERR_UNSUPPORTED, "%lld rows exceed the grid", (long long)rows);
  if (static_cast<int64_t>(batch) * 2 * (layers < kMaxLayers ? layers : kMaxLayers) > 65535)
    return fail(TC_ERR_UNSUPPORTED, "batch %d exceeds the grid", batch);
  auto fill = [&](auto& a, int l0, int nl) {
    constexpr int kCap = sizeof(a.src) / sizeof(a.src[0]);
    for (int i = 0; i < kCap; ++i) { a.src[i] = nullptr; a.dst[i] = nullptr; }
    for (int i = 0; i < nl; ++i) {
      a.src[i] = static_cast<const uint16_t*>(ks[l0 + i]);
      a.src[nl + i] = static_cast<const uint16_t*>(vs[l0 + i]);
      a.dst[i] = static_cast<uint16_t*>(kd[l0 + i]) + row0 * d.strides[2];
      a.dst[nl + i] = static_cast<uint16_t*>(vd[l0 + i]) + row0 * d.strides[2];
    }
    a.s_b[0] = k_st[0]; a.s_h[0] = k_st[1]; a.s_t[0] = k_st[2];
    a.s_b[1] = v_st[0]; a.s_h[1] = v_st[1]; a.s_t[1] = v_st[2];
    a.d_b = d.strides[0]; a.d_h = d.strides[1]; a.d_t = d.strides[2];
    a.slots = d.slots;
    a.rows = rows;
    a.layers = nl;
    a.pages = d.pages;
    a.page_tokens = d.page_tokens;
    launch(a, dim3(heads, static_cast<unsigned>(tiles), static_cast<unsigned>(batch * 2 * nl)), s);
    return hip_status(hipGetLastError(), "row write launch");
  };
  if (layers == 1) {  // the usual call: 200 bytes of arguments instead of 2 KB
    RowArgs<1> a;
    return fill(a, 0, 1);
  }
  for (int l0 = 0; l0 < layers; l0 += kMaxLayers) {
    RowArgs<kMaxLayers> a;
    if ((rc = fill(a, l0, layers - l0 < kMaxLayers ? layers - l0 : kMaxLayers)) != TC_OK) return rc;
  }
  return TC_OK;
}

}  // namespace
}  // namespace tc

using namespace tc;

extern "C" int tc_append_rows(const void* k_rows_dev, const int64_t k_strides[3], const void* v_rows_dev,
                              const int64_t v_strides[3], void* k_cache_dev, void* v_cache_dev,
                              const int64_t cache_strides[3], int64_t capacity, int64_t row0, int batch, int heads,
                              int64_t rows, int head_dim, int dtype, void* stream) {
  clear_error();
  if (row0 < 0 || rows < 0 || row0 > capacity - rows)
    return fail(TC_ERR_INVALID_ARGUMENT, "rows [%lld, %lld) outside the capacity %lld", (long long)row0,
                (long long)(row0 + rows), (long long)capacity);
  const Dest d{cache_strides};
  return write_rows(&k_rows_dev, k_strides, &v_rows_dev, v_strides, &k_cache_dev, &v_cache_dev, d, row0, 1, batch,
                    heads, rows, head_dim, dtype, static_cast<hipStream_t>(stream));
}

extern "C" int tc_paged_append_rows(const void* const* k_rows_host, const int64_t k_strides[3],
                                    const void* const* v_rows_host, const int64_t v_strides[3],
                                    void* const* k_pools_host, void* const* v_pools_host,
                                    const int64_t pool_strides[3], int num_pages, int page_tokens,
                                    const int64_t* slots_dev, int num_layers, int batch, int heads, int64_t rows,
                                    int head_dim, int dtype, void* stream) {
  clear_error();
  if (num_pages < 1 || page_tokens < 1)
    return fail(TC_ERR_INVALID_ARGUMENT, "pool of %d pages of %d tokens", num_pages, page_tokens);
  if (rows > 0 && num_layers > 0 && !slots_dev) return fail(TC_ERR_INVALID_ARGUMENT, "null slot list");
  if (!aligned16(slots_dev)) return fail(TC_ERR_ALIGNMENT, "slot list not 16-byte aligned");
  const Dest d{pool_strides, slots_dev, num_pages, page_tokens};
  return write_rows(k_rows_host, k_strides, v_rows_host, v_strides, k_pools_host, v_pools_host, d, 0, num_layers,
                    batch, heads, rows, head_dim, dtype, static_cast<hipStream_t>(stream));
}
