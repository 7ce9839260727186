// Deterministic segmented row reduction (the weight-gradient scatter of
// rte/kernels/cluster_pool_ffn.py:218-241 and of every index/gather backward):
//   out[v] (+)= sum over pairs p with keys[p] = v of w[p] * rows[p / row_div]
// The pairs are counting-sorted by key (stable: ascending p), each key's run is summed in chunks by
// one wave per 128 columns, and chunk partials are added in chunk order; up to 4096 pairs over up to
// 1024 keys take a one-launch path (per-key pair lists, summed in ascending p).  No floating-point
// atomics: the result is bitwise repeatable for a given input.
//
// Bounds, at the shortlist head's 2.1 M pairs over 8192 keys (rows of 1024 bf16): the sums read 4.3 GB of
// rows.  A wave takes 128 columns and the waves of one column slab run on one XCD, whose 4 MB L2 then
// holds that slab of every row, so the reads run at L2 and not at memory rate (573 us with whole
// rows).  The sort moves a histogram of sort blocks x keys, kept block-major so it is written and
// read in whole lines (312 us key-major with 1024-pair blocks).
#include "common.hpp"

namespace rte {

namespace {

constexpr int kSortSub = 256;         // pairs ranked together inside a sort block
constexpr int kMaxSortKeys = 32768;   // LDS histogram of the sort: 128 KB
constexpr int kSlab = 128;            // columns of a wave in the sums

// Pairs per sort block and per partial sum.  Few pairs: more, shorter pieces (latency); many: fewer
// histograms and partials.  Whole call in us, blocks of 1024 / 4096 (chunks of 128): 2^18 pairs 49 / 62,
// 72 / 86 and 245 / 260 over 2048, 8192 and 32768 keys (512, 512 and 1024 columns); 2^19 64 / 77, 86 / 97
// and 332 / 277; 2^20 97 / 99, 129 / 129 and 509 / 318; 2^21 179 / 164, 236 / 196 and 1020 / 519: the line
// costs least where it is wrong.  Chunks of 64 / 128 (blocks of 1024, the same keys): 2^16 37.4 / 38.0, 63.9
// / 64.1, 247 / 246; 2^18 50.6 / 49.1, 71.7 / 71.6, 245 / 245; 2^19 66.5 / 64.3, 94.2 / 86.2, 333 / 332; a
// tie up to 2^18, 2 - 8% from there.
int sort_block(int64_t P) { return P > (1 << 19) ? 4096 : 1024; }
int seg_chunk(int64_t P) { return P >= (1 << 18) ? 128 : 64; }

// hist[b * V + v] = pairs of sort block b whose key is v.

__global__ void __launch_bounds__(256) sort_count_kernel(const int32_t* __restrict__ keys, int P, int V, int per,
                                                         int32_t* __restrict__ hist) {
  extern __shared__ int32_t hcount[];
  for (int c = threadIdx.x; c < V; c += 256) hcount[c] = 0;
  __syncthreads();
  const int64_t p0 = (int64_t)blockIdx.x * per;
  for (int i = threadIdx.x; i < per; i += 256) {
    const int64_t p = p0 + i;
    if (p < P) {
      const int k = keys[p];
      if (k >= 0 && k < V) atomicAdd(&hcount[k], 1);
    }
  }
  __syncthreads();
  int32_t* row = hist + (int64_t)blockIdx.x * V;
  for (int c = threadIdx.x; c < V; c += 256) row[c] = hcount[c];
}

// Exclusive scan of each key's column of hist, totals[v] = column sum.  A workgroup takes 32 keys
// (whole 128-byte lines) in 8 ranges of sort blocks.
__global__ void __launch_bounds__(256) sort_rowscan_kernel(int32_t* __restrict__ hist, int V, int nblk,
                                                           int32_t* __restrict__ totals) {
  __shared__ int32_t part[8][33];
  const int vi = threadIdx.x & 31, seg = threadIdx.x >> 5;
  const int v = blockIdx.x * 32 + vi;
  const int per = (nblk + 7) / 8, b0 = seg * per, b1 = min(nblk, b0 + per);
  int32_t sum = 0;
  if (v < V) {
    int b = b0;
    for (; b + 8 <= b1; b += 8) {
      int32_t x[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) x[u] = hist[(int64_t)(b + u) * V + v];
#pragma unroll
      for (int u = 0; u < 8; ++u) sum += x[u];
    }
    for (; b < b1; ++b) sum += hist[(int64_t)b * V + v];
  }
  part[seg][vi] = sum;
  __syncthreads();
  if (v >= V) return;
  int32_t run = 0;
  for (int q = 0; q < seg; ++q) run += part[q][vi];
  int b = b0;
  for (; b + 8 <= b1; b += 8) {
    int32_t x[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) x[u] = hist[(int64_t)(b + u) * V + v];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      hist[(int64_t)(b + u) * V + v] = run;
      run += x[u];
    }
  }
  for (; b < b1; ++b) {
    const int32_t x = hist[(int64_t)b * V + v];
    hist[(int64_t)b * V + v] = run;
    run += x;
  }
  if (seg == 7) totals[v] = run;
}

// offsets = exclusive scan of totals, chunk_off = exclusive scan of ceil(totals / chunk).
__global__ void __launch_bounds__(1024) sort_keyscan_kernel(const int32_t* __restrict__ totals, int V, int chunk,
                                                            int32_t* __restrict__ offsets,
                                                            int32_t* __restrict__ chunk_off) {
  __shared__ int32_t ws[16], wc[16];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int seg = (V + 1023) / 1024;
  const int b0 = tid * seg, b1 = min(V, b0 + seg);
  int32_t s = 0, sc = 0;
  for (int v = b0; v < b1; ++v) {
    s += totals[v];
    sc += (totals[v] + chunk - 1) / chunk;
  }
  int32_t is = s, ic = sc;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int32_t y = __shfl_up(is, o, 64), yc = __shfl_up(ic, o, 64);
    if (lane >= o) {
      is += y;
      ic += yc;
    }
  }
  if (lane == 63) {
    ws[wave] = is;
    wc[wave] = ic;
  }
  __syncthreads();
  int32_t run = is - s, runc = ic - sc;
  for (int q = 0; q < wave; ++q) {
    run += ws[q];
    runc += wc[q];
  }
  for (int v = b0; v < b1; ++v) {
    offsets[v] = run;
    chunk_off[v] = runc;
    run += totals[v];
    runc += (totals[v] + chunk - 1) / chunk;
  }
  if (tid == 1023) {
    offsets[V] = run;
    chunk_off[V] = runc;
  }
}

// Stable scatter: pair p of block b with key v goes to slot offsets[v] + hist[b, v] +
// (pairs of block b before p with key v).  Writes the pair's row (p / row_div) and weight.  A wave finds
// the lanes that share a key with one ballot per key bit; the waves take the cursors in turn.  Also
// item_key[i] = the key whose run chunk i of the sums belongs to.
__global__ void __launch_bounds__(256) sort_scatter_kernel(const int32_t* __restrict__ keys, int P, int V, int per,
                                                           int row_div, const int32_t* __restrict__ hist,
                                                           const int32_t* __restrict__ offsets,
                                                           const float* __restrict__ g, int2* __restrict__ pairs,
                                                           const int32_t* __restrict__ chunk_off,
                                                           int32_t* __restrict__ item_key) {
  extern __shared__ int32_t cursor[];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int32_t* row = hist + (int64_t)blockIdx.x * V;
  for (int c = tid; c < V; c += 256) cursor[c] = offsets[c] + row[c];
  const int64_t p0 = (int64_t)blockIdx.x * per;
  const int bits = V > 1 ? 32 - __clz(V - 1) : 0;
  const int nsub = (int)((P - p0 < per ? P - p0 : per) + kSortSub - 1) / kSortSub;
  int next = p0 + tid < P ? keys[p0 + tid] : -1;
  const int items = chunk_off[V];
  for (int i = blockIdx.x * 256 + tid; i < items; i += gridDim.x * 256) {
    int lo = 0, hi = V;  // largest v with chunk_off[v] <= i
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      if (chunk_off[mid] <= i) lo = mid; else hi = mid;
    }
    item_key[i] = lo;
  }
  __syncthreads();
  for (int q = 0; q < nsub; ++q) {
    const int64_t p = p0 + (int64_t)q * kSortSub + tid;
    const int k = next;
    if (q + 1 < nsub) next = p + kSortSub < P && (q + 1) * kSortSub + tid < per ? keys[p + kSortSub] : -1;
    const bool valid = k >= 0 && k < V;
    unsigned long long same = __ballot(valid);
    for (int b = 0; b < bits; ++b) {
      const bool one = (k >> b) & 1;
      const unsigned long long m = __ballot(one);
      same &= one ? m : ~m;
    }
    const int rank = __popcll(same & ((1ull << lane) - 1ull)), count = __popcll(same);
    int slot = 0;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      if (wave == w && valid) {
        slot = cursor[k] + rank;
        __builtin_amdgcn_wave_barrier();  // every lane has read its cursor
        if (rank == 0) cursor[k] = slot + count;
      }
      __syncthreads();
    }
    if (valid) {
      const float wp = g ? g[p] : 1.0f;
      pairs[slot] = make_int2((int32_t)(p / row_div), __float_as_int(wp));
    }
  }
}

__device__ __forceinline__ void load8(const bf16* p, float* v) {
  const uint4 u = *reinterpret_cast<const uint4*>(p);
  const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    v[2 * i] = __uint_as_float(w[i] << 16);
    v[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
  }
}

__device__ __forceinline__ void load8(const float* p, float* v) {
  const float4 a = reinterpret_cast<const float4*>(p)[0], b = reinterpret_cast<const float4*>(p)[1];
  v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
  v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
}

__device__ __forceinline__ float2 load2(const bf16* p) {
  const uint32_t w = *reinterpret_cast<const uint32_t*>(p);
  return make_float2(__uint_as_float(w << 16), __uint_as_float(w & 0xffff0000u));
}
__device__ __forceinline__ float2 load2(const float* p) { return *reinterpret_cast<const float2*>(p); }

// One wave per chunk of one key's run and slab of 128 columns (two per lane): sum_s w[s] * rows[tok[s]], the
// pairs read a batch ahead of their rows (2.1 M pairs of 1024 columns: 269 us without, 236 us).  A
// key with a single chunk writes out directly; otherwise the chunk's partial goes to part[item].
// Dispatch id b runs on XCD b % 8: each XCD takes an equal, contiguous run of the (slab, chunk) pairs
// that exist, in slab order.  The launch is sized by a bound on the chunks; with the bound shared out
// instead of chunk_off[V], the XCDs of a sum of few slabs had unequal work (whole call, 8192 keys, 512
// columns: 2^19 pairs 188 us and now 174, 2^20 146 and 129; 8192 pairs over 2048 keys 36.6 and 35.4).
template <typename RowT>
__global__ void __launch_bounds__(256) sort_segsum_kernel(const int32_t* __restrict__ offsets,
                                                          const int32_t* __restrict__ chunk_off,
                                                          const int32_t* __restrict__ item_key, int V, int chunk,
                                                          int nslab, const int2* __restrict__ pairs,
                                                          const RowT* __restrict__ hidden, int d,
                                                          float* __restrict__ part, float* __restrict__ dW,
                                                          int accumulate) {
  const int lane = threadIdx.x & 63;
  const int items = chunk_off[V];
  const int nb = (int)(((int64_t)items * nslab + 3) / 4);  // workgroups with work: at most the grid
  const int xcd = blockIdx.x & 7, q8 = nb >> 3, r8 = nb & 7, at = blockIdx.x >> 3;
  if (at >= q8 + (xcd < r8 ? 1 : 0)) return;
  const int64_t id = (int64_t)(xcd * q8 + (xcd < r8 ? xcd : r8) + at) * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int slab = (int)(id / items), item = (int)(id - (int64_t)slab * items);
  if (slab >= nslab) return;
  const int v = item_key[item];
  const int first = chunk_off[v], nq = chunk_off[v + 1] - first;
  const int s0 = offsets[v] + (item - first) * chunk;
  const int s1 = min(offsets[v + 1], s0 + chunk);
  const int col = slab * kSlab + lane * 2;
  const bool on = col < d;
  const RowT* base = hidden + (on ? col : 0);
  float2 acc = make_float2(0.0f, 0.0f);
  int s = s0;
  if (s + 8 <= s1) {  // 8 rows in flight, the next 8 pairs on their way
    int2 pr[8], nx[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) pr[j] = pairs[s + j];
    for (; s + 8 <= s1; s += 8) {
      float2 x[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) x[j] = load2(base + (int64_t)pr[j].x * d);
      const int n = s + 16 <= s1 ? s + 8 : s;
#pragma unroll
      for (int j = 0; j < 8; ++j) nx[j] = pairs[n + j];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        acc.x += __int_as_float(pr[j].y) * x[j].x;
        acc.y += __int_as_float(pr[j].y) * x[j].y;
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) pr[j] = nx[j];
    }
  }
  for (; s < s1; ++s) {
    const int2 pr = pairs[s];
    const float2 x = load2(base + (int64_t)pr.x * d);
    acc.x += __int_as_float(pr.y) * x.x;
    acc.y += __int_as_float(pr.y) * x.y;
  }
  if (!on) return;
  float2* o = reinterpret_cast<float2*>((nq == 1 ? dW + (int64_t)v * d : part + (int64_t)item * d) + col);
  if (nq == 1 && accumulate) {
    const float2 old = *o;
    acc.x += old.x;
    acc.y += old.y;
  }
  *o = acc;
}

// Keys with zero or several chunks: dW[v] (+)= sum of the key's partials in chunk order.
__global__ void __launch_bounds__(256) sort_final_kernel(const int32_t* __restrict__ chunk_off, int V, int d,
                                                         const float* __restrict__ part, float* __restrict__ dW,
                                                         int accumulate) {
  const int64_t idx4 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int d4 = d >> 2;
  if (idx4 >= (int64_t)V * d4) return;
  const int v = (int)(idx4 / d4), c = (int)(idx4 % d4) * 4;
  const int q0 = chunk_off[v], q1 = chunk_off[v + 1];
  if (q1 - q0 == 1) return;
  if (q1 == q0 && accumulate) return;
  float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
  for (int q = q0; q < q1; ++q) {
    const float4 x = *reinterpret_cast<const float4*>(part + (int64_t)q * d + c);
    s.x += x.x; s.y += x.y; s.z += x.z; s.w += x.w;
  }
  float4* o = reinterpret_cast<float4*>(dW + (int64_t)v * d + c);
  if (accumulate) {
    const float4 a = *o;
    s.x += a.x; s.y += a.y; s.z += a.z; s.w += a.w;
  }
  *o = s;
}

template <typename K>
int set_lds_limit(K kernel, size_t bytes, const char* what) {
  if (bytes <= 65536) return 0;
  const hipError_t err = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
  if (err != hipSuccess) {
    set_error("%s: cannot reserve %zu bytes of LDS: %s", what, bytes, hipGetErrorString(err));
    return -1;
  }
  return 0;
}

// Bound on the chunks of all keys: every chunk holds a pair, and all but each key's last are full.
// (Without the first, 5000 pairs over 32768 keys of 2048 columns kept 270 MB of partials, 42 now, and
// started half a million waves with nothing to do: 249 us, 210 now.)
size_t max_chunks(int64_t P, int V) {
  const size_t n = ((size_t)P + seg_chunk(P) - 1) / seg_chunk(P) + (size_t)V;
  return n < (size_t)P ? n : (size_t)P;
}

struct SegCarve {
  int32_t* hist;
  int32_t* totals;
  int32_t* offsets;
  int32_t* chunk_off;
  int32_t* item_key;
  int2* pairs;
  float* part;
  size_t bytes;
};

SegCarve carve(void* base, int64_t P, int V, int d) {
  const size_t per = sort_block(P);
  const size_t nblk = ((size_t)P + per - 1) / per;
  const size_t max_items = max_chunks(P, V);
  SegCarve c{};
  size_t off = 0;
  auto take = [&](size_t bytes) {
    char* p = base ? static_cast<char*>(base) + off : nullptr;
    off += ((bytes + 255) / 256) * 256;
    return static_cast<void*>(p);
  };
  c.hist = static_cast<int32_t*>(take((size_t)V * (nblk ? nblk : 1) * 4));
  c.totals = static_cast<int32_t*>(take((size_t)V * 4));
  c.offsets = static_cast<int32_t*>(take((size_t)(V + 1) * 4));
  c.chunk_off = static_cast<int32_t*>(take((size_t)(V + 1) * 4));
  c.item_key = static_cast<int32_t*>(take(max_items * 4));
  c.pairs = static_cast<int2*>(take((size_t)P * 8));
  c.part = static_cast<float*>(take(max_items * (size_t)d * 4));
  c.bytes = off;
  return c;
}

// Few pairs (P <= kSmallPairs) and few keys: one workgroup per key lists its pairs in
// ascending order (ballot compaction into LDS), then each thread sums 8 columns over the list
// in that order.  One launch instead of the sort pipeline; still deterministic.
constexpr int kSmallPairs = 4096;
constexpr int kSmallKeys = 1024;

template <typename RowT>
__global__ void __launch_bounds__(256) segsum_small_kernel(const int32_t* __restrict__ keys, int P, int row_div,
                                                           const float* __restrict__ w,
                                                           const RowT* __restrict__ rows, int d,
                                                           float* __restrict__ out, int accumulate) {
  __shared__ int32_t list[kSmallPairs];
  __shared__ int32_t wcnt[4];
  const int v = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  int n = 0;
  for (int base = 0; base < P; base += 256) {
    const int p = base + tid;
    const bool hit = p < P && keys[p] == v;
    const unsigned long long m = __ballot(hit);
    if (lane == 0) wcnt[wave] = __popcll(m);
    __syncthreads();
    int off = n;
    for (int q = 0; q < wave; ++q) off += wcnt[q];
    if (hit) list[off + __popcll(m & ((1ull << lane) - 1ull))] = p;
    n += ((wcnt[0] + wcnt[1]) + wcnt[2]) + wcnt[3];
    __syncthreads();
  }
  for (int col = tid * 8; col < d; col += 256 * 8) {
    float acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    for (int i = 0; i < n; ++i) {
      const int p = list[i];
      const float wp = w ? w[p] : 1.0f;
      float r[8];
      load8(rows + (int64_t)(p / row_div) * d + col, r);
#pragma unroll
      for (int t = 0; t < 8; ++t) acc[t] += wp * r[t];
    }
    float* o = out + (int64_t)v * d + col;
    if (accumulate) {
      float prev[8];
      load8(o, prev);
#pragma unroll
      for (int t = 0; t < 8; ++t) acc[t] += prev[t];
    }
    *reinterpret_cast<float4*>(o) = make_float4(acc[0], acc[1], acc[2], acc[3]);
    *reinterpret_cast<float4*>(o + 4) = make_float4(acc[4], acc[5], acc[6], acc[7]);
  }
}

}  // namespace

size_t segreduce_workspace_bytes(int64_t P, int V, int d) {
  if (P < 0 || V < 1 || d < 1) return 0;
  return carve(nullptr, P, V, d).bytes;
}

int segreduce_rows(const int32_t* keys, int64_t P, int V, int row_div, const float* w, const void* rows, int rows_f32,
                   int d, float* out, int accumulate, void* ws, size_t ws_bytes, hipStream_t s) {
  RTE_REQUIRE(V >= 1 && V <= kMaxSortKeys, "segment_reduce: key count must be in [1, %d]", kMaxSortKeys);
  RTE_REQUIRE(d >= 8 && d % 8 == 0 && d <= 2048, "segment_reduce: d must be a multiple of 8 in [8, 2048]");
  RTE_REQUIRE(P >= 0 && P < (1LL << 31) && row_div >= 1, "segment_reduce: bad pair count / row divisor");
  RTE_REQUIRE(((uintptr_t)rows & 15) == 0 && ((uintptr_t)out & 15) == 0 && ((uintptr_t)ws & 255) == 0,
              "segment_reduce: rows / out need 16-byte and workspace 256-byte alignment");
  const SegCarve c = carve(ws, P, V, d);
  RTE_REQUIRE(ws_bytes >= c.bytes, "segment_reduce: workspace too small (%zu < %zu)", ws_bytes, c.bytes);
  if (P == 0) {
    if (!accumulate) return fill_f32(out, 0.0f, (int64_t)V * d, s);
    return 0;
  }
  const int Pi = (int)P;
  if (Pi <= kSmallPairs && V <= kSmallKeys) {
    if (rows_f32)
      hipLaunchKernelGGL(segsum_small_kernel<float>, dim3(V), dim3(256), 0, s, keys, Pi, row_div, w,
                         static_cast<const float*>(rows), d, out, accumulate);
    else
      hipLaunchKernelGGL(segsum_small_kernel<bf16>, dim3(V), dim3(256), 0, s, keys, Pi, row_div, w,
                         static_cast<const bf16*>(rows), d, out, accumulate);
    return check_launch("segment_reduce_small");
  }
  const int per = sort_block(P), chunk = seg_chunk(P);
  const int nblk = (Pi + per - 1) / per;
  const dim3 block(256);
  const size_t lds_hist = (size_t)V * sizeof(int32_t);
  RTE_TRY(set_lds_limit(sort_count_kernel, lds_hist, "segment_reduce"));
  RTE_TRY(set_lds_limit(sort_scatter_kernel, lds_hist, "segment_reduce"));
  hipLaunchKernelGGL(sort_count_kernel, dim3(nblk), block, lds_hist, s, keys, Pi, V, per, c.hist);
  RTE_TRY(check_launch("segment_reduce_count"));
  hipLaunchKernelGGL(sort_rowscan_kernel, dim3((V + 31) / 32), block, 0, s, c.hist, V, nblk, c.totals);
  RTE_TRY(check_launch("segment_reduce_rowscan"));
  hipLaunchKernelGGL(sort_keyscan_kernel, dim3(1), dim3(1024), 0, s, c.totals, V, chunk, c.offsets, c.chunk_off);
  RTE_TRY(check_launch("segment_reduce_keyscan"));
  // the chunk count lives on the device: launch its upper bound, extra waves exit at once
  const int64_t max_items = (int64_t)max_chunks(P, V);
  hipLaunchKernelGGL(sort_scatter_kernel, dim3(nblk), block, lds_hist, s, keys, Pi, V, per, row_div, c.hist, c.offsets,
                     w, c.pairs, c.chunk_off, c.item_key);
  RTE_TRY(check_launch("segment_reduce_scatter"));
  const int nslab = (d + kSlab - 1) / kSlab;
  const int64_t nwg = (max_items * nslab + 3) / 4;
  RTE_REQUIRE(nwg < ((int64_t)1 << 31), "segment_reduce: too many partial sums");
  if (rows_f32)
    hipLaunchKernelGGL(sort_segsum_kernel<float>, dim3((unsigned)nwg), block, 0, s, c.offsets, c.chunk_off, c.item_key, V,
                       chunk, nslab, c.pairs, static_cast<const float*>(rows), d, c.part, out,
                       accumulate);
  else
    hipLaunchKernelGGL(sort_segsum_kernel<bf16>, dim3((unsigned)nwg), block, 0, s, c.offsets, c.chunk_off, c.item_key, V,
                       chunk, nslab, c.pairs, static_cast<const bf16*>(rows), d, c.part, out,
                       accumulate);
  RTE_TRY(check_launch("segment_reduce_sum"));
  const int64_t n4 = (int64_t)V * (d / 4);
  hipLaunchKernelGGL(sort_final_kernel, dim3((unsigned)((n4 + 255) / 256)), block, 0, s, c.chunk_off, V, d, c.part,
                     out, accumulate);
  return check_launch("segment_reduce_final");
}

}  // namespace rte
