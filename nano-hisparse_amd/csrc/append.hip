// Decode-time append into one pool page, fused: the new K/V rows are
// written to the page's pool block and (through the pinned host alias) to
// its host block, the page's running per-element key minimum / maximum fold
// in the new keys, and its fp32 mean key is recomputed over every valid row.
//
// append_page_rows_kernel (a prompt's pages: several rows of whole 16-byte
// chunks): some workgroups copy the rows to the pool and the host block, a
// chunk per lane and four loads in flight; others load the page's keys into
// LDS and fold them, one wave each for the sum, the minimum and the maximum.
// What bounds it is the PCIe write of the mirror (a page of 64 x 4 KB is
// 262144 host bytes: 4.6 us at 57 GB/s), the ordered fold (4.5 us of 64 rows)
// and ~2 us of launch. A full page takes 6.6 us; it took 24 to 36 when one
// thread walked all rows of its element, a store after each load.
//
// append_element (any other row): one thread owns one element of a row
// (kv_heads * head_dim elements), so every access of a wave is contiguous.
//
// The mean is summed in double in row order and rounded to fp32 once (the
// oracle sums in the same order). Min/max propagate NaN like torch.minimum
// / torch.maximum.
#include <math.h>

#include <type_traits>

#include "nhs_common.h"

namespace nhs {

constexpr int kAppendThreads = 256;
constexpr int kAppendBatch = 64;  // earlier rows loaded together for the page mean (one round for P <= 64)

struct AppendArgs {
  const void* k;
  const void* v;
  int64_t token_stride;  // elements between consecutive tokens of k and v
  int dtype;
  int row_elems;
  int64_t plane_elems;   // page_size * row_elems
  char* pool_block;      // the page's pool block [2, P, row_elems]
  char* host_block;      // its host block, or null
  int within, count;
  float* summary;
  void* minimum;
  void* maximum;
};

__device__ __forceinline__ float nan_min(float a, float b) { return (a != a || b != b) ? a + b : (b < a ? b : a); }
__device__ __forceinline__ float nan_max(float a, float b) { return (a != a || b != b) ? a + b : (b > a ? b : a); }

// Element e of every appended row of one page (T: the KV storage type, so
// every load below is a plain load of a known width).
template <typename T>
__device__ __forceinline__ void append_element(const AppendArgs& a, int e) {
  constexpr int esize = T::bytes;
  float lo = load_elem(a.minimum, T::dtype, e);
  float hi = load_elem(a.maximum, T::dtype, e);
  double sum = 0.0;
  // the earlier keys of the page, loaded kAppendBatch at a time before they
  // are summed (in row order)
  // Loads are unconditional (rows past `within` re-read the last earlier
  // row, which is in bounds) so that no branch separates them; only the
  // sum is masked.
  for (int r0 = 0; r0 < a.within; r0 += kAppendBatch) {
    float keys[kAppendBatch];
#pragma unroll
    for (int j = 0; j < kAppendBatch; ++j) {
      const int r = min(r0 + j, a.within - 1);
      keys[j] = load_elem(a.pool_block, T::dtype, (int64_t)r * a.row_elems + e);
    }
#pragma unroll
    for (int j = 0; j < kAppendBatch; ++j)
      if (r0 + j < a.within) sum += (double)keys[j];
  }
  for (int t = 0; t < a.count; ++t) {
    const int64_t src = (int64_t)t * a.token_stride + e;
    const int64_t row = (int64_t)(a.within + t) * a.row_elems + e;
    // copy the raw element bits: no conversion touches the stored values
    if (esize == 4) {
      const uint32_t kb = static_cast<const uint32_t*>(a.k)[src], vb = static_cast<const uint32_t*>(a.v)[src];
      reinterpret_cast<uint32_t*>(a.pool_block)[row] = kb;
      reinterpret_cast<uint32_t*>(a.pool_block)[a.plane_elems + row] = vb;
      if (a.host_block) {
        reinterpret_cast<uint32_t*>(a.host_block)[row] = kb;
        reinterpret_cast<uint32_t*>(a.host_block)[a.plane_elems + row] = vb;
      }
    } else {
      const uint16_t kb = static_cast<const uint16_t*>(a.k)[src], vb = static_cast<const uint16_t*>(a.v)[src];
      reinterpret_cast<uint16_t*>(a.pool_block)[row] = kb;
      reinterpret_cast<uint16_t*>(a.pool_block)[a.plane_elems + row] = vb;
      if (a.host_block) {
        reinterpret_cast<uint16_t*>(a.host_block)[row] = kb;
        reinterpret_cast<uint16_t*>(a.host_block)[a.plane_elems + row] = vb;
      }
    }
    const float key = load_elem(a.k, T::dtype, src);
    lo = nan_min(lo, key);
    hi = nan_max(hi, key);
    sum += (double)key;
  }
  store_elem(a.minimum, T::dtype, e, lo);
  store_elem(a.maximum, T::dtype, e, hi);
  a.summary[e] = (float)(sum / (double)(a.within + a.count));
}

template <typename T>
__global__ __launch_bounds__(kAppendThreads) void append_page_kernel(AppendArgs a) {
  const int e = blockIdx.x * kAppendThreads + threadIdx.x;
  if (e < a.row_elems) append_element<T>(a, e);
}

// Fewest new rows of a call that append_page_rows_kernel takes. us per call
// (bf16, 1024 elements a row), it against append_page_kernel: 1 row 3.1
// against 2.1 and 6.5 against 3.7 with 63 earlier rows to fold; 8 rows 3.1
// against 4.4 and 6.5 against 6.1; 16 rows 3.1 against 7.2 and 6.5 against 8.9.
constexpr int kRowsCount = 10;
constexpr int kRowChunks = 8;                               // 16-byte chunks of a row per folding workgroup
constexpr int kRowsPerPass = kAppendThreads / kRowChunks;   // 32
constexpr int kRowsHeld = 2 * kRowsPerPass;                 // rows folded between two barriers
constexpr int kFoldBatch = 16;                              // rows read from LDS together
constexpr int kCopyChunks = 4;                              // chunks per thread of a copying workgroup

typedef uint32_t append_u4 __attribute__((ext_vector_type(4)));

template <typename T, typename Elem>
__device__ __forceinline__ float widen(Elem bits) {
  if constexpr (T::dtype == NHS_F32) return bits;
  else return T::dtype == NHS_BF16 ? bf16_bits_to_f32(bits) : f16_bits_to_f32(bits);
}
template <typename T>
__device__ __forceinline__ std::conditional_t<T::bytes == 4, float, uint16_t> narrow(float v) {
  if constexpr (T::dtype == NHS_F32) return v;
  else return T::dtype == NHS_BF16 ? f32_to_bf16_bits(v) : f32_to_f16_bits(v);
}

// 16-byte chunk `chunk` of new row `row` of one plane.
__device__ __forceinline__ const NHS_GLOBAL append_u4* new_chunk(const AppendArgs& a, int plane, uint32_t row,
                                                                 uint32_t chunk, int esize) {
  const NHS_GLOBAL char* src = to_global(static_cast<const char*>(plane ? a.v : a.k));
  return (const NHS_GLOBAL append_u4*)(src + (int64_t)row * a.token_stride * esize + (int64_t)chunk * 16);
}

// A store that leaves the caches at once (system scope). Plain stores to
// pinned host memory stay in L2 until the kernel ends, and the PCIe writes
// then follow everything else: a page took 10.9 us, against 6.6 with the
// fold beside the writes. The builtin spelling (a volatile store) would wait
// after every store. s_nop: the data registers must outlive the issue.
__device__ __forceinline__ void store_through(NHS_GLOBAL char* p, append_u4 v) {
  asm volatile("global_store_dwordx4 %0, %1, off sc0 sc1\n\ts_nop 1" ::"v"(p), "v"(v) : "memory");
}

// Copies the new rows to the pool and the host block, kCopyChunks * 256
// consecutive chunks of a plane per workgroup: the rows are consecutive in
// both blocks, so a wave's store covers 1 KB of one span. Written 128 bytes a
// row (by the workgroups that fold them) the mirror reached half the rate.
template <typename T>
__device__ __forceinline__ void copy_rows(const AppendArgs& a, int group, int plane, FastDiv chunks) {
  const int64_t first = (plane * a.plane_elems + (int64_t)a.within * a.row_elems) * T::bytes;
  NHS_GLOBAL char* pool = to_global(a.pool_block) + first;
  NHS_GLOBAL char* host = to_global(a.host_block) + first;
  const uint32_t n = (uint32_t)a.count * chunks.d, at = (uint32_t)group * kCopyChunks * kAppendThreads + threadIdx.x;
  append_u4 v[kCopyChunks];
#pragma unroll
  for (int i = 0; i < kCopyChunks; ++i) {  // unconditional (past the end they re-read the last chunk)
    const uint32_t x = min(at + i * kAppendThreads, n - 1), row = chunks.div(x);
    v[i] = *new_chunk(a, plane, row, x - row * chunks.d, T::bytes);
  }
#pragma unroll
  for (int i = 0; i < kCopyChunks; ++i) {
    const uint32_t x = at + i * kAppendThreads;
    if (x >= n) break;
    if (a.host_block) store_through(host + (int64_t)x * 16, v[i]);
    *(NHS_GLOBAL append_u4*)(pool + (int64_t)x * 16) = v[i];
  }
}

// Folds the keys of the workgroup's 8 chunks (from chunk 8 * group): 64 rows
// at a time are loaded together (a thread one chunk of two rows) and held in
// LDS, and one wave each walks them in row order for the sum, the minimum and
// the maximum (a thread per element).
template <typename T>
__device__ __forceinline__ void fold_rows(const AppendArgs& a, int group, int chunks) {
  constexpr int E = 16 / T::bytes;  // elements per chunk
  constexpr int kCols = kRowChunks * E;
  using Elem = std::conditional_t<T::bytes == 4, float, uint16_t>;
  __shared__ append_u4 held[kRowsHeld * kRowChunks];
  const int tid = threadIdx.x, slot = tid % kRowChunks, lane_row = tid / kRowChunks;
  const int chunk = min(group * kRowChunks + slot, chunks - 1);
  const int64_t row_bytes = (int64_t)a.row_elems * T::bytes;
  const NHS_GLOBAL char* pool = to_global(a.pool_block) + (int64_t)chunk * 16;
  const int total = a.within + a.count;
  const int role = tid / kWave, col = tid % kWave, e = group * kCols + col;  // 0: sum, 1: minimum, 2: maximum
  const bool folds = role < 3 && col < kCols && e < a.row_elems;
  NHS_GLOBAL Elem* bound = to_global(static_cast<Elem*>(role == 1 ? a.minimum : a.maximum));
  Elem page = 0;
  if (folds && role) page = bound[e];
  float best = role == 1 ? INFINITY : -INFINITY;  // over the new keys
  double sum = 0.0;
  for (int r0 = 0; r0 < total; r0 += kRowsHeld) {
    // unconditional loads (past the end they re-read the last row), so that no branch or wait separates them
    append_u4 v[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int r = min(r0 + lane_row + i * kRowsPerPass, total - 1);
      v[i] = r < a.within ? *(const NHS_GLOBAL append_u4*)(pool + r * row_bytes)
                          : *new_chunk(a, 0, r - a.within, chunk, T::bytes);
    }
    held[lane_row * kRowChunks + slot] = v[0];
    held[(lane_row + kRowsPerPass) * kRowChunks + slot] = v[1];
    __syncthreads();
    if (folds) {
      // kFoldBatch LDS reads in flight at a time; rows past the end (copies of the last) are masked
      const Elem* keys = reinterpret_cast<const Elem*>(held) + col;
      const int n = min(kRowsHeld, total - r0), fresh = a.within - r0;
#pragma unroll 1
      for (int j0 = 0; j0 < n; j0 += kFoldBatch) {
        float key[kFoldBatch];
#pragma unroll
        for (int j = 0; j < kFoldBatch; ++j) key[j] = widen<T>(keys[(j0 + j) * kCols]);
        if (role == 0) {
#pragma unroll
          for (int j = 0; j < kFoldBatch; ++j) sum = j0 + j < n ? sum + (double)key[j] : sum;
        } else {
          // the first NaN stays, as in nan_min / nan_max
#pragma unroll
          for (int j = 0; j < kFoldBatch; ++j) {
            const bool better = role == 1 ? key[j] < best : key[j] > best;
            const bool takes = better || (key[j] != key[j] && best == best);
            best = takes && j0 + j < n && j0 + j >= fresh ? key[j] : best;
          }
        }
      }
    }
    __syncthreads();  // the next rows overwrite the held ones
  }
  if (!folds) return;
  if (role == 0)
    to_global(a.summary)[e] = (float)(sum / (double)total);
  else
    bound[e] = narrow<T>(role == 1 ? nan_min(widen<T>(page), best) : nan_max(widen<T>(page), best));
}

// The first fold_groups workgroups fold, the others copy (the planes' groups
// one after another).
template <typename T>
__global__ __launch_bounds__(kAppendThreads) void append_page_rows_kernel(AppendArgs a, FastDiv chunks,
                                                                          int fold_groups, int copy_groups) {
  int group = blockIdx.x;
  if (group < fold_groups) return fold_rows<T>(a, group, (int)chunks.d);
  group -= fold_groups;
  const int plane = group >= copy_groups;
  copy_rows<T>(a, group - plane * copy_groups, plane, chunks);
}

struct AppendItemsArgs {
  const char* k;
  const char* v;
  int64_t token_stride;  // elements between the items' rows
  int dtype, row_elems, page_size;
  char* pool;
  int64_t pool_block_bytes;  // the pool's block stride (host blocks are contiguous)
  char* host;
  const nhs_layer_item* items;
  const int64_t* lengths;
};

// Item blockIdx.y appends its one token; its page and row follow from its
// length and its page tables.
template <typename T>
__global__ __launch_bounds__(kAppendThreads) void append_items_kernel(AppendItemsArgs g) {
  const int e = blockIdx.x * kAppendThreads + threadIdx.x;
  if (e >= g.row_elems) return;
  const int b = blockIdx.y;
  const nhs_layer_item& item = g.items[b];
  const int64_t length = g.lengths[b];
  const int64_t page = length / g.page_size;
  constexpr int esize = T::bytes;
  const int64_t plane = (int64_t)g.page_size * g.row_elems;
  const int64_t block_bytes = 2 * plane * esize;
  const int64_t page_offset = page * g.row_elems;
  AppendArgs a;
  a.k = g.k + (int64_t)b * g.token_stride * esize;
  a.v = g.v + (int64_t)b * g.token_stride * esize;
  a.token_stride = g.token_stride;
  a.dtype = g.dtype;
  a.row_elems = g.row_elems;
  a.plane_elems = plane;
  a.pool_block = g.pool + (int64_t)item.resident[page] * g.pool_block_bytes;
  a.host_block = g.host ? g.host + (int64_t)item.source[page] * block_bytes : nullptr;
  a.within = (int)(length - page * g.page_size);
  a.count = 1;
  a.summary = item.summaries + page_offset;
  a.minimum = static_cast<char*>(item.minimum) + page_offset * esize;
  a.maximum = static_cast<char*>(item.maximum) + page_offset * esize;
  append_element<T>(a, e);
}

// Whether rows are whole 16-byte chunks wherever append_page_rows_kernel touches them.
static bool whole_chunks(const void* k, const void* v, const void* pool, const void* host, int64_t pool_block_stride,
                         int64_t token_stride, int64_t row_elems, int esize) {
  return row_elems * esize % 16 == 0 && token_stride * esize % 16 == 0 && pool_block_stride % 16 == 0 &&
         ((uintptr_t)k | (uintptr_t)v | (uintptr_t)pool | (uintptr_t)host) % 16 == 0;
}

}  // namespace nhs

extern "C" int nhs_append_page(const void* k, const void* v, int64_t token_stride, int32_t kv_dtype,
                               int32_t row_elems, int32_t page_size, void* pool, int64_t pool_block_stride,
                               int64_t block, int32_t within,
                               int32_t count, void* host_alias, int64_t host_page, float* summary, void* minimum,
                               void* maximum, void* stream) {
  using namespace nhs;
  const LaunchEvents ev = take_launch_events();
  if (!k || !v || !pool || !summary || !minimum || !maximum) return fail(NHS_ERR_INVALID, "nhs_append_page: null pointer");
  if (!valid_dtype(kv_dtype)) return fail(NHS_ERR_INVALID, "nhs_append_page: bad dtype");
  if (row_elems < 1 || page_size < 1 || block < 0 || within < 0 || count < 1 || within + count > page_size ||
      token_stride < row_elems || (host_alias && host_page < 0))
    return fail(NHS_ERR_INVALID, "nhs_append_page: invalid page, rows or strides");
  AppendArgs a;
  a.k = k;
  a.v = v;
  a.token_stride = token_stride;
  a.dtype = kv_dtype;
  a.row_elems = row_elems;
  a.plane_elems = (int64_t)page_size * row_elems;
  const int64_t block_bytes = 2 * a.plane_elems * elem_size(kv_dtype);
  if (pool_block_stride == 0) pool_block_stride = block_bytes;
  if (pool_block_stride < block_bytes || pool_block_stride % elem_size(kv_dtype))
    return fail(NHS_ERR_INVALID, "nhs_append_page: pool_block_stride below a block or not a whole element");
  a.pool_block = static_cast<char*>(pool) + block * pool_block_stride;
  a.host_block = host_alias ? static_cast<char*>(host_alias) + host_page * block_bytes : nullptr;
  a.within = within;
  a.count = count;
  a.summary = summary;
  a.minimum = minimum;
  a.maximum = maximum;
  const dim3 threads(kAppendThreads);
  const int64_t chunks = (int64_t)row_elems * elem_size(kv_dtype) / 16;
  if (count >= kRowsCount && chunks * count < (1ll << 30) &&
      whole_chunks(k, v, pool, host_alias, pool_block_stride, token_stride, row_elems, elem_size(kv_dtype))) {
    const int fold_groups = (int)((chunks + kRowChunks - 1) / kRowChunks);
    const int copy_groups = (int)((chunks * count + kCopyChunks * kAppendThreads - 1) / (kCopyChunks * kAppendThreads));
    const dim3 grid((unsigned)(fold_groups + 2 * copy_groups));
    const FastDiv div((uint32_t)chunks);
    if (kv_dtype == NHS_BF16)
      launch(append_page_rows_kernel<BF16>, grid, threads, 0, (hipStream_t)stream, ev.start, ev.stop, a, div,
             fold_groups, copy_groups);
    else if (kv_dtype == NHS_F16)
      launch(append_page_rows_kernel<F16>, grid, threads, 0, (hipStream_t)stream, ev.start, ev.stop, a, div,
             fold_groups, copy_groups);
    else
      launch(append_page_rows_kernel<F32>, grid, threads, 0, (hipStream_t)stream, ev.start, ev.stop, a, div,
             fold_groups, copy_groups);
    return launch_status("nhs_append_page");
  }
  const dim3 grid((unsigned)((row_elems + kAppendThreads - 1) / kAppendThreads));
  if (kv_dtype == NHS_BF16)
    launch(append_page_kernel<BF16>, grid, threads, 0, (hipStream_t)stream, ev.start, ev.stop, a);
  else if (kv_dtype == NHS_F16)
    launch(append_page_kernel<F16>, grid, threads, 0, (hipStream_t)stream, ev.start, ev.stop, a);
  else
    launch(append_page_kernel<F32>, grid, threads, 0, (hipStream_t)stream, ev.start, ev.stop, a);
  return launch_status("nhs_append_page");
}

extern "C" int nhs_append_items(int32_t batch, const void* k, const void* v, int64_t token_stride, int32_t kv_dtype,
                                int32_t row_elems, int32_t page_size, void* pool, int64_t pool_block_stride,
                                void* host_alias,
                                const nhs_layer_item* items, const int64_t* lengths, void* stream) {
  using namespace nhs;
  const LaunchEvents ev = take_launch_events();
  if (!k || !v || !pool || !items || !lengths) return fail(NHS_ERR_INVALID, "nhs_append_items: null pointer");
  if (!valid_dtype(kv_dtype)) return fail(NHS_ERR_INVALID, "nhs_append_items: bad dtype");
  if (batch < 0 || batch > 65535 || row_elems < 1 || page_size < 1 || token_stride < row_elems)
    return fail(NHS_ERR_INVALID, "nhs_append_items: invalid batch, rows or strides");
  if (batch == 0) return NHS_OK;
  AppendItemsArgs g;
  g.k = static_cast<const char*>(k);
  g.v = static_cast<const char*>(v);
  g.token_stride = token_stride;
  g.dtype = kv_dtype;
  g.row_elems = row_elems;
  g.page_size = page_size;
  g.pool = static_cast<char*>(pool);
  const int64_t block_bytes = 2 * (int64_t)page_size * row_elems * elem_size(kv_dtype);
  if (pool_block_stride == 0) pool_block_stride = block_bytes;
  if (pool_block_stride < block_bytes || pool_block_stride % elem_size(kv_dtype))
    return fail(NHS_ERR_INVALID, "nhs_append_items: pool_block_stride below a block or not a whole element");
  g.pool_block_bytes = pool_block_stride;
  g.host = static_cast<char*>(host_alias);
  g.items = items;
  g.lengths = lengths;
  const dim3 grid((unsigned)((row_elems + kAppendThreads - 1) / kAppendThreads), (unsigned)batch), block(kAppendThreads);
  if (kv_dtype == NHS_BF16)
    launch(append_items_kernel<BF16>, grid, block, 0, (hipStream_t)stream, ev.start, ev.stop, g);
  else if (kv_dtype == NHS_F16)
    launch(append_items_kernel<F16>, grid, block, 0, (hipStream_t)stream, ev.start, ev.stop, g);
  else
    launch(append_items_kernel<F32>, grid, block, 0, (hipStream_t)stream, ev.start, ev.stop, g);
  return launch_status("nhs_append_items");
}
