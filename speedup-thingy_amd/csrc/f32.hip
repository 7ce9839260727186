// fp32 arithmetic for training.precision = "fp32" (the reference's default precision, where every
// matmul runs in float32 and nothing is cast to bf16).
//
//  * rte_gemm_f32: C = alpha op(A) op(B)^T + beta C on v_mfma_f32_32x32x2_f32 with fp32 operands and
//    accumulation.  One kernel covers the dense products, batched products (two-level batch
//    strides: the attention's (sample, head) pairs read straight out of the packed QKV rows), and
//    grouped products over device-side group offsets: GROUP_M (each group a row range with its own
//    weight block: routed / banked pools, per-key macro products) and GROUP_K (each group a
//    reduction range writing its own output block: their weight gradients, summed in row order or,
//    with a workspace, in chunks whose partials are added in order, so results repeat bitwise).  Rows of A and B
//    may be gathered through index arrays and scaled per row; rows of C may be scattered.
//  * causal softmax over score rows (scaled, optional per-(batch) output scale), forward and backward
//  * SwiGLU over [up | gate] rows, forward and backward
//  * pair combine (out[t] = resid[t] + sum_j w[t, j] rows[slot(t, j)]) and the pair row dots of its
//    weight gradient
//
// Tile: 64 x 64 outputs per 256-thread workgroup (four waves of 32 x 32), k steps of 32 staged
// through two LDS buffers k-major (each MFMA operand a contiguous 32-float LDS row segment): while
// step s multiplies, step s + 1 is written to the other buffer and step s + 2 is on its way from
// memory, with one barrier per step.  These products are bound by the latency of their k steps and
// by too few workgroups, not by the matrix cores, so long reductions are cut into k ranges whose
// fp32 partials a second kernel adds in order: a 32 x 256 x 8192 weight gradient took 4 workgroups
// 512 serial steps before.  fp32 routed pool layer (T 8192, d 256, 32 x 32, top-4) forward + backward:
// 1335 us with 16-k steps of one buffer and unsplit reductions, 440 now.
#include "common.hpp"

namespace rte {
namespace {

typedef __attribute__((__vector_size__(16 * sizeof(float)))) float f32x16;

constexpr int kBM = 64, kBN = 64, kBK = 32, kThreads = 256;
constexpr int kPitch = kBM + 4;

struct GemmF32 {
  const float* A;
  int64_t lda;
  int a_t;
  const int32_t* a_rows;
  const float* a_scale;
  const float* B;
  int64_t ldb;
  int b_t;
  const int32_t* b_rows;
  const float* b_scale;
  float* C;
  int64_t ldc;
  const int32_t* c_rows;
  int M, N, K;
  float alpha, beta;
  // batch z = z1 * Z2 + z2: operand offsets z1 * s1 + z2 * s2
  int Z2;
  int64_t sA1, sA2, sB1, sB2, sC1, sC2;
  // groups: mode 1 = GROUP_M (rows), 2 = GROUP_K (reduction); goff[G + 1] device offsets
  int mode;
  const int32_t* goff;
  int G;
  const int64_t* b_goff;  // GROUP_M: B element offset of group g (else g * b_gstride)
  int64_t b_gstride, b_rows_gstride;
  const int64_t* c_goff;  // GROUP_K: C element offset of group g (else g * c_gstride)
  int64_t c_gstride, c_rows_gstride;
  // split reductions: dense (mode 0, one batch) split blockIdx.z covers k [z chunk, (z + 1) chunk);
  // GROUP_K work item blockIdx.z is a chunk of its group (an empty group has one item, a group of
  // one chunk stores directly).  part holds fp32 [item][M][N].
  int chunk;
  float* part;
};

// One 64 x 32 operand tile through registers, eight elements per thread.  Non-transposed operands
// are contiguous along k (thread: one row, eight k), transposed ones along the row index (thread:
// one k, eight rows).  Rows outside [r0, r_end) and k outside [k_lo, k_end) read as 0.
template <bool T>
struct TileF32 {
  const float* base;
  const float* row_ptr;  // layout N: this thread's row, nullptr past the end
  float row_scale;
  int next_row;  // layout T: the memory row of the next step's k (gathers are looked up a step ahead)
  float next_scale;
  float v[8];

  __device__ __forceinline__ static int sub() { return T ? threadIdx.x >> 3 : threadIdx.x >> 2; }
  __device__ __forceinline__ static int at() { return T ? (threadIdx.x & 7) * 8 : (threadIdx.x & 3) * 8; }

  __device__ __forceinline__ void look(const int32_t* rows, const float* scale, int k0, int k_end) {
    const int k = k0 + sub();
    next_row = k;
    next_scale = 1.0f;
    if (k < k_end) {
      if (rows) next_row = rows[k];
      if (scale) next_scale = scale[k];
    }
  }
  __device__ __forceinline__ void init(const float* X, int64_t ld, const int32_t* rows, const float* scale, int r0,
                                       int r_end, int k_lo, int k_end) {
    base = X;
    if constexpr (T) {
      look(rows, scale, k_lo, k_end);
    } else {
      const int r = r0 + sub();
      row_ptr = r < r_end ? X + (int64_t)(rows ? rows[r] : r) * ld : nullptr;
      row_scale = (scale && r < r_end) ? scale[r] : 1.0f;
    }
  }
  // the tile starting at k0; vec: 16-byte loads are aligned
  __device__ __forceinline__ void load(int64_t ld, const int32_t* rows, const float* scale, int r0, int r_end, int k0,
                                       int k_end, bool vec) {
    const float* p;
    float sc;
    int n;  // valid elements from p on
    if constexpr (T) {
      p = base + (int64_t)next_row * ld + r0 + at();
      sc = next_scale;
      n = k0 + sub() < k_end ? r_end - r0 - at() : 0;
      look(rows, scale, k0 + kBK, k_end);
    } else {
      p = row_ptr + k0 + at();
      sc = row_scale;
      n = row_ptr ? k_end - k0 - at() : 0;
    }
    if (n >= 8 && vec) {
      const float4 x = *reinterpret_cast<const float4*>(p), y = *reinterpret_cast<const float4*>(p + 4);
      v[0] = x.x; v[1] = x.y; v[2] = x.z; v[3] = x.w;
      v[4] = y.x; v[5] = y.y; v[6] = y.z; v[7] = y.w;
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) v[i] = i < n ? p[i] : 0.0f;
    }
    if (scale) {
#pragma unroll
      for (int i = 0; i < 8; ++i) v[i] *= sc;
    }
  }
  __device__ __forceinline__ void store(float (*S)[kPitch]) const {
    if constexpr (T) {
      float* d = &S[sub()][at()];
      *reinterpret_cast<float4*>(d) = make_float4(v[0], v[1], v[2], v[3]);
      *reinterpret_cast<float4*>(d + 4) = make_float4(v[4], v[5], v[6], v[7]);
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) S[at() + i][sub()] = v[i];
    }
  }
};

// Group and position of element x of the sequence that lists, group by group, ceil(count / per)
// entries (at least `least`): 64 groups at a time by one wave.  Returns {group or -1, index within
// the group, entries of the group}.
__device__ __forceinline__ int3 find_group(const int32_t* goff, int G, int per, int least, int x, int lane) {
  int base = 0;
  for (int c0 = 0; c0 < G; c0 += 64) {
    const int g = c0 + lane;
    int cnt = 0;
    if (g < G) {
      cnt = (goff[g + 1] - goff[g] + per - 1) / per;
      if (cnt < least) cnt = least;
    }
    int incl = cnt;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int y = __shfl_up(incl, off, 64);
      if (lane >= off) incl += y;
    }
    const unsigned long long hit = __ballot(cnt > 0 && x >= base + incl - cnt && x < base + incl);
    if (hit) {
      const int l = __ffsll((long long)hit) - 1;
      const int n = __shfl(cnt, l, 64);
      return make_int3(c0 + l, x - base - __shfl(incl, l, 64) + n, n);
    }
    base += __shfl(incl, 63, 64);
  }
  return make_int3(-1, 0, 0);
}

template <bool AT, bool BT>
__global__ void __launch_bounds__(kThreads) gemm_f32_kernel(GemmF32 p) {
  __shared__ __align__(16) float As[2][kBK][kPitch];
  __shared__ __align__(16) float Bs[2][kBK][kPitch];
  const float* A = p.A;
  const float* B = p.B;
  float* C = p.C;
  const int32_t* b_rows = p.b_rows;
  const int32_t* c_rows = p.c_rows;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int m0, m_end = p.M, k_lo = 0, k_hi = p.K;
  const int n0 = blockIdx.y * kBN;
  float* part = nullptr;
  if (p.mode == 1) {
    // GROUP_M: the x index enumerates each group's row tiles in group order
    const int3 f = find_group(p.goff, p.G, kBM, 0, blockIdx.x, lane);
    const int g = f.x;
    if (g < 0) return;
    m0 = p.goff[g] + f.y * kBM;
    m_end = p.goff[g + 1];
    B += p.b_goff ? p.b_goff[g] : (int64_t)g * p.b_gstride;
    if (b_rows) b_rows += (int64_t)g * p.b_rows_gstride;
  } else if (p.mode == 2) {
    int g = blockIdx.z;
    m0 = blockIdx.x * kBM;
    if (p.part) {
      const int3 f = find_group(p.goff, p.G, p.chunk, 1, blockIdx.z, lane);
      g = f.x;
      if (g < 0) return;
      k_lo = p.goff[g] + f.y * p.chunk;
      k_hi = k_lo + p.chunk < p.goff[g + 1] ? k_lo + p.chunk : p.goff[g + 1];
      if (f.z > 1) part = p.part + (int64_t)blockIdx.z * p.M * p.N;
    } else {
      k_lo = p.goff[g];
      k_hi = p.goff[g + 1];
    }
    C += p.c_goff ? p.c_goff[g] : (int64_t)g * p.c_gstride;
    if (c_rows) c_rows += (int64_t)g * p.c_rows_gstride;
  } else {
    m0 = blockIdx.x * kBM;
    if (p.part) {
      k_lo = blockIdx.z * p.chunk;
      k_hi = k_lo + p.chunk < p.K ? k_lo + p.chunk : p.K;
      part = p.part + (int64_t)blockIdx.z * p.M * p.N;
    } else {
      const int z = blockIdx.z, z1 = z / p.Z2, z2 = z - z1 * p.Z2;
      A += z1 * p.sA1 + z2 * p.sA2;
      B += z1 * p.sB1 + z2 * p.sB2;
      C += z1 * p.sC1 + z2 * p.sC2;
    }
  }
  if (m0 >= m_end || n0 >= p.N) return;
  const int wm = wave >> 1, wn = wave & 1;
  f32x16 acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
  // a_t: A's memory rows run over k; else over m (rows gathered / scaled by the logical index)
  const bool avec = (((uintptr_t)A | ((uintptr_t)p.lda << 2)) & 15) == 0 && (AT || (k_lo & 3) == 0);
  const bool bvec = (((uintptr_t)B | ((uintptr_t)p.ldb << 2)) & 15) == 0 && (BT || (k_lo & 3) == 0);
  TileF32<AT> ta;
  TileF32<BT> tb;
  auto load = [&](int k0) {
    ta.load(p.lda, p.a_rows, p.a_scale, m0, m_end, k0, k_hi, avec);
    tb.load(p.ldb, b_rows, p.b_scale, n0, p.N, k0, k_hi, bvec);
  };
  auto store = [&](int b) {
    ta.store(As[b]);
    tb.store(Bs[b]);
  };
  if (k_lo < k_hi) {
    ta.init(A, p.lda, p.a_rows, p.a_scale, m0, m_end, k_lo, k_hi);
    tb.init(B, p.ldb, b_rows, p.b_scale, n0, p.N, k_lo, k_hi);
    load(k_lo);
    store(0);
    if (k_lo + kBK < k_hi) load(k_lo + kBK);
    __syncthreads();
    int buf = 0;
    for (int k0 = k_lo; k0 < k_hi; k0 += kBK) {
      if (k0 + kBK < k_hi) {
        store(buf ^ 1);
        if (k0 + 2 * kBK < k_hi) load(k0 + 2 * kBK);
      }
#pragma unroll
      for (int kk = 0; kk < kBK; kk += 2) {
        const float a = As[buf][kk + (lane >> 5)][wm * 32 + (lane & 31)];
        const float b = Bs[buf][kk + (lane >> 5)][wn * 32 + (lane & 31)];
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, acc, 0, 0, 0);
      }
      __syncthreads();
      buf ^= 1;
    }
  }
  const int col = n0 + wn * 32 + (lane & 31);
  if (col >= p.N) return;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int m = m0 + wm * 32 + (lane >> 5) * 4 + (r >> 2) * 8 + (r & 3);
    if (m < m_end) {
      if (part) {
        part[(int64_t)m * p.N + col] = acc[r];
        continue;
      }
      const int64_t row = c_rows ? (int64_t)c_rows[m] : (int64_t)m;
      float* c = C + row * p.ldc + col;
      const float v = p.alpha * acc[r];
      *c = p.beta != 0.0f ? v + p.beta * *c : v;
    }
  }
}

// The partials of a split reduction, added in k order.  Grid (elements / 256, groups or 1).
__global__ void __launch_bounds__(256) gemm_f32_reduce_kernel(GemmF32 p, int items) {
  const int g = blockIdx.y;
  int q0 = 0, n = items;
  float* C = p.C;
  const int32_t* c_rows = p.c_rows;
  if (p.mode == 2) {
    // the group's items: entries of the groups before it, and its own
    __shared__ int s_q[2];
    if (threadIdx.x < 64) {
      int before = 0, own = 0;
      for (int h = threadIdx.x; h <= g; h += 64) {
        int cnt = (p.goff[h + 1] - p.goff[h] + p.chunk - 1) / p.chunk;
        if (cnt < 1) cnt = 1;
        if (h < g) before += cnt;
        else own = cnt;
      }
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) {
        before += __shfl_xor(before, o, 64);
        own += __shfl_xor(own, o, 64);
      }
      if (threadIdx.x == 0) {
        s_q[0] = before;
        s_q[1] = own;
      }
    }
    __syncthreads();
    q0 = s_q[0];
    n = s_q[1];
    if (n == 1) return;  // stored by the product itself
    C += p.c_goff ? p.c_goff[g] : (int64_t)g * p.c_gstride;
    if (c_rows) c_rows += (int64_t)g * p.c_rows_gstride;
  }
  const int64_t plane = (int64_t)p.M * p.N;
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= plane) return;
  const float* src = p.part + q0 * plane + i;
  float v = 0.0f;
  int q = 0;
  for (; q + 8 <= n; q += 8) {  // eight partials in flight
    float x[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) x[u] = src[(q + u) * plane];
#pragma unroll
    for (int u = 0; u < 8; ++u) v += x[u];
  }
  for (; q < n; ++q) v += src[q * plane];
  const int m = (int)(i / p.N), col = (int)(i - (int64_t)m * p.N);
  float* c = C + (int64_t)(c_rows ? c_rows[m] : m) * p.ldc + col;
  v *= p.alpha;
  *c = p.beta != 0.0f ? v + p.beta * *c : v;
}

// k range of one workgroup of a split dense product (0: not split): about 512 workgroups of at least
// 256 k.  Only for weight gradients (A transposed: the reduction runs over tokens), so a row of
// activations keeps its one sum whatever shares its call.
int dense_chunk(int M, int N, int K) {
  const int64_t tiles = (int64_t)((M + kBM - 1) / kBM) * ((N + kBN - 1) / kBN);
  if (tiles >= 256 || K < 512) return 0;
  int64_t s = (512 + tiles - 1) / tiles;
  if (s > K / 256) s = K / 256;
  if (s > 64) s = 64;
  const int64_t kc = ((K + s - 1) / s + kBK - 1) / kBK * kBK;
  return kc < K ? (int)kc : 0;
}

// k chunk of a grouped reduction: 256 (8192 slots of 32 groups, 64 x 256 outputs: 512 workgroups of 8
// steps), longer where the partials would pass 256 MiB.
constexpr size_t kGroupPartBytes = (size_t)256 << 20;
int group_chunk(int M, int N, int K, int G) {
  int64_t c = 256;
  while (c < K && ((size_t)(K / c) + 1 + G) * M * N * 4 > kGroupPartBytes) c *= 2;
  return (int)c;
}

size_t group_bytes(int M, int N, int K, int G) {
  const int64_t c = group_chunk(M, N, K, G);
  if (c >= K) return 0;
  const size_t b = ((size_t)((K + c - 1) / c) + G) * M * N * 4;
  return b <= kGroupPartBytes + (size_t)M * N * 4 ? b : 0;
}

int launch_f32(const GemmF32& p, dim3 grid, hipStream_t stream) {
  if (!p.a_t && !p.b_t) hipLaunchKernelGGL((gemm_f32_kernel<false, false>), grid, dim3(kThreads), 0, stream, p);
  else if (!p.a_t) hipLaunchKernelGGL((gemm_f32_kernel<false, true>), grid, dim3(kThreads), 0, stream, p);
  else if (!p.b_t) hipLaunchKernelGGL((gemm_f32_kernel<true, false>), grid, dim3(kThreads), 0, stream, p);
  else hipLaunchKernelGGL((gemm_f32_kernel<true, true>), grid, dim3(kThreads), 0, stream, p);
  return check_launch("gemm_f32");
}

// ---------------------------------------------------------------------------------------------
// causal softmax over rows of [Z, S, S] scores: P = softmax(scale * s, keys <= query); the output
// is oscale[z] * P (oscale optional).  One wave per row, the row read in 64-column chunks.

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o));
  return v;
}
__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  return v;
}

__global__ void softmax_causal_fwd_kernel(const float* s, int64_t rows, int S, float scale, const float* oscale,
                                          float* p_out, float* y_out) {
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;
  const int lane = threadIdx.x & 63;
  const int q = (int)(row % S);
  const int64_t z = row / S;
  const float* x = s + row * S;
  float mx = -INFINITY;
  for (int c = lane; c <= q; c += 64) mx = fmaxf(mx, x[c] * scale);
  mx = wave_max(mx);
  float sum = 0.0f;
  for (int c = lane; c <= q; c += 64) sum += __expf(x[c] * scale - mx);
  sum = wave_sum(sum);
  const float inv = 1.0f / sum;
  const float os = oscale ? oscale[z] : 1.0f;
  float* pr = p_out + row * S;
  float* yr = y_out + row * S;
  for (int c = lane; c < S; c += 64) {
    const float v = c <= q ? __expf(x[c] * scale - mx) * inv : 0.0f;
    pr[c] = v;
    yr[c] = v * os;
  }
}

// ds = scale * P (g - sum_c P g) with g = oscale * dy
__global__ void softmax_causal_bwd_kernel(const float* P, const float* dy, int64_t rows, int S, float scale,
                                          const float* oscale, float* ds) {
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;
  const int lane = threadIdx.x & 63;
  const int64_t z = row / S;
  const float os = oscale ? oscale[z] : 1.0f;
  const float* pr = P + row * S;
  const float* gr = dy + row * S;
  float dot = 0.0f;
  for (int c = lane; c < S; c += 64) dot += pr[c] * gr[c];
  dot = wave_sum(dot) * os;
  float* o = ds + row * S;
  for (int c = lane; c < S; c += 64) o[c] = scale * pr[c] * (os * gr[c] - dot);
}

// ---------------------------------------------------------------------------------------------
// SwiGLU over rows [up (n) | gate (n)] of width ld: z = up silu(gate)

__global__ void swiglu_f32_fwd_kernel(const float* ug, int64_t rows, int n, int64_t ld, float* z) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= rows * n) return;
  const int64_t r = i / n;
  const int j = (int)(i - r * n);
  const float u = ug[r * ld + j], g = ug[r * ld + n + j];
  z[i] = u * g * sigmoidf_(g);
}

__global__ void swiglu_f32_bwd_kernel(const float* ug, const float* dz, int64_t rows, int n, int64_t ld, float* dug) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= rows * n) return;
  const int64_t r = i / n;
  const int j = (int)(i - r * n);
  const float u = ug[r * ld + j], g = ug[r * ld + n + j], d = dz[i];
  const float sg = sigmoidf_(g);
  dug[r * ld + j] = d * g * sg;
  dug[r * ld + n + j] = d * u * sg * (1.0f + g * (1.0f - sg));
}

// ---------------------------------------------------------------------------------------------
// pair combine: out[t] = resid[t] + sum_j w[t, j] rows[slot[t k + j]] (slot < 0: no pair; w
// optional = 1), the pairs summed in j order.  One workgroup of 64 lanes per token row, lanes
// over the columns.
__global__ void combine_f32_kernel(const float* rows, const int32_t* slot, const float* w, int T, int k, int d,
                                   const float* resid, float* out) {
  const int t = blockIdx.x;
  for (int c = threadIdx.x; c < d; c += blockDim.x) {
    float acc = resid ? resid[(int64_t)t * d + c] : 0.0f;
    for (int j = 0; j < k; ++j) {
      const int s = slot[(int64_t)t * k + j];
      if (s >= 0) acc += (w ? w[(int64_t)t * k + j] : 1.0f) * rows[(int64_t)s * d + c];
    }
    out[(int64_t)t * d + c] = acc;
  }
}

// dw[t, j] = sum_c dout[t, c] rows[slot[t k + j], c]  (0 for an absent pair): one wave per pair
__global__ void pair_dot_f32_kernel(const float* dout, const float* rows, const int32_t* slot, int64_t pairs, int k,
                                    int d, float* dw) {
  const int64_t pr = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (pr >= pairs) return;
  const int lane = threadIdx.x & 63;
  const int s = slot[pr];
  float acc = 0.0f;
  if (s >= 0) {
    const float* a = dout + (pr / k) * d;
    const float* b = rows + (int64_t)s * d;
    for (int c = lane; c < d; c += 64) acc += a[c] * b[c];
  }
  acc = wave_sum(acc);
  if (lane == 0) dw[pr] = acc;
}

}  // namespace
}  // namespace rte

using namespace rte;

extern "C" {

size_t rte_gemm_f32_workspace_bytes(int M, int N, int K) {
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  const int kc = dense_chunk(M, N, K);
  return kc ? (size_t)((K + kc - 1) / kc) * M * N * 4 : 0;
}

int rte_gemm_f32_ws(const float* A, int64_t lda, int a_t, const int32_t* a_rows, const float* a_scale, const float* B,
                    int64_t ldb, int b_t, const int32_t* b_rows, const float* b_scale, float* C, int64_t ldc,
                    const int32_t* c_rows, int M, int N, int K, float alpha, float beta, int Z1, int Z2, int64_t sA1,
                    int64_t sA2, int64_t sB1, int64_t sB2, int64_t sC1, int64_t sC2, void* ws, size_t ws_bytes,
                    void* stream) {
  RTE_REQUIRE(M >= 0 && N >= 0 && K >= 0 && Z1 >= 1 && Z2 >= 1, "gemm_f32: bad sizes");
  RTE_REQUIRE(A && B && C, "gemm_f32: null operand");
  RTE_REQUIRE((int64_t)Z1 * Z2 <= 65535, "gemm_f32: at most 65535 batches");
  if (M == 0 || N == 0) return 0;
  GemmF32 p{A, lda, a_t, a_rows, a_scale, B, ldb, b_t, b_rows, b_scale, C, ldc, c_rows, M, N, K, alpha, beta,
            Z2, sA1, sA2, sB1, sB2, sC1, sC2, 0, nullptr, 0, nullptr, 0, 0, nullptr, 0, 0, 0, nullptr};
  dim3 grid((M + kBM - 1) / kBM, (N + kBN - 1) / kBN, Z1 * Z2);
  RTE_REQUIRE(grid.y <= 65535, "gemm_f32: N too large");
  const size_t need = a_t && Z1 * Z2 == 1 ? rte_gemm_f32_workspace_bytes(M, N, K) : 0;
  if (!need || !ws || ws_bytes < need) return launch_f32(p, grid, static_cast<hipStream_t>(stream));
  p.chunk = dense_chunk(M, N, K);
  p.part = static_cast<float*>(ws);
  grid.z = (K + p.chunk - 1) / p.chunk;
  RTE_TRY(launch_f32(p, grid, static_cast<hipStream_t>(stream)));
  hipLaunchKernelGGL(gemm_f32_reduce_kernel, dim3((unsigned)(((int64_t)M * N + 255) / 256)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), p, (int)grid.z);
  return check_launch("gemm_f32_reduce");
}

int rte_gemm_f32(const float* A, int64_t lda, int a_t, const int32_t* a_rows, const float* a_scale, const float* B,
                 int64_t ldb, int b_t, const int32_t* b_rows, const float* b_scale, float* C, int64_t ldc,
                 const int32_t* c_rows, int M, int N, int K, float alpha, float beta, int Z1, int Z2, int64_t sA1,
                 int64_t sA2, int64_t sB1, int64_t sB2, int64_t sC1, int64_t sC2, void* stream) {
  return rte_gemm_f32_ws(A, lda, a_t, a_rows, a_scale, B, ldb, b_t, b_rows, b_scale, C, ldc, c_rows, M, N, K, alpha,
                         beta, Z1, Z2, sA1, sA2, sB1, sB2, sC1, sC2, nullptr, 0, stream);
}

size_t rte_gemm_f32_grouped_workspace_bytes(int mode, int M, int N, int K, int G) {
  if (mode != 2 || M <= 0 || N <= 0 || K <= 0 || G <= 0) return 0;
  return group_bytes(M, N, K, G);
}

// Grouped products.  mode 1 (GROUP_M): group g owns rows [goff[g], goff[g+1]) of the M total and
// reads B at b_goff[g] (or g * b_gstride) with b_rows shifted by g * b_rows_gstride.  mode 2
// (GROUP_K): group g reduces over k in [goff[g], goff[g+1]) and writes C at c_goff[g] (or
// g * c_gstride) with c_rows shifted by g * c_rows_gstride; with a workspace, in chunks.
int rte_gemm_f32_grouped_ws(int mode, const int32_t* goff, int G, const float* A, int64_t lda, int a_t,
                            const int32_t* a_rows, const float* a_scale, const float* B, int64_t ldb, int b_t,
                            const int32_t* b_rows, const float* b_scale, const int64_t* b_goff, int64_t b_gstride,
                            int64_t b_rows_gstride, float* C, int64_t ldc, const int32_t* c_rows,
                            const int64_t* c_goff, int64_t c_gstride, int64_t c_rows_gstride, int M, int N, int K,
                            float alpha, float beta, void* ws, size_t ws_bytes, void* stream) {
  RTE_REQUIRE(mode == 1 || mode == 2, "gemm_f32_grouped: mode must be 1 (rows) or 2 (reduction)");
  RTE_REQUIRE(G >= 0 && M >= 0 && N >= 0 && K >= 0, "gemm_f32_grouped: bad sizes");
  RTE_REQUIRE(goff && A && B && C, "gemm_f32_grouped: null argument");
  if (G == 0 || N == 0 || (mode == 1 && M == 0) || (mode == 2 && M == 0)) return 0;
  GemmF32 p{A, lda, a_t, a_rows, a_scale, B, ldb, b_t, b_rows, b_scale, C, ldc, c_rows, M, N, K, alpha, beta,
            1, 0, 0, 0, 0, 0, 0, mode, goff, G, b_goff, b_gstride, b_rows_gstride, c_goff, c_gstride,
            c_rows_gstride, 0, nullptr};
  const hipStream_t st = static_cast<hipStream_t>(stream);
  if (mode == 1) {
    // a bound on the groups' row tiles
    return launch_f32(p, dim3((M + kBM - 1) / kBM + G, (N + kBN - 1) / kBN, 1), st);
  }
  RTE_REQUIRE(G <= 65535, "gemm_f32_grouped: at most 65535 reduction groups");
  dim3 grid((M + kBM - 1) / kBM, (N + kBN - 1) / kBN, G);
  const size_t need = group_bytes(M, N, K, G);
  const int64_t chunk = group_chunk(M, N, K, G), items = ((int64_t)K + chunk - 1) / chunk + G;
  if (!need || !ws || ws_bytes < need || items > 65535) return launch_f32(p, grid, st);
  p.chunk = (int)chunk;
  p.part = static_cast<float*>(ws);
  grid.z = (unsigned)items;
  RTE_TRY(launch_f32(p, grid, st));
  hipLaunchKernelGGL(gemm_f32_reduce_kernel, dim3((unsigned)(((int64_t)M * N + 255) / 256), (unsigned)G), dim3(256), 0,
                     st, p, 0);
  return check_launch("gemm_f32_reduce");
}

int rte_gemm_f32_grouped(int mode, const int32_t* goff, int G, const float* A, int64_t lda, int a_t,
                         const int32_t* a_rows, const float* a_scale, const float* B, int64_t ldb, int b_t,
                         const int32_t* b_rows, const float* b_scale, const int64_t* b_goff, int64_t b_gstride,
                         int64_t b_rows_gstride, float* C, int64_t ldc, const int32_t* c_rows, const int64_t* c_goff,
                         int64_t c_gstride, int64_t c_rows_gstride, int M, int N, int K, float alpha, float beta,
                         void* stream) {
  return rte_gemm_f32_grouped_ws(mode, goff, G, A, lda, a_t, a_rows, a_scale, B, ldb, b_t, b_rows, b_scale, b_goff,
                                 b_gstride, b_rows_gstride, C, ldc, c_rows, c_goff, c_gstride, c_rows_gstride, M, N, K,
                                 alpha, beta, nullptr, 0, stream);
}

int rte_softmax_causal_f32_fwd(const float* s, int64_t rows, int S, float scale, const float* oscale, float* p,
                               float* y, void* stream) {
  RTE_REQUIRE(rows >= 0 && S >= 1 && s && p && y, "softmax_causal_f32_fwd: bad arguments");
  if (rows == 0) return 0;
  hipLaunchKernelGGL(softmax_causal_fwd_kernel, dim3((unsigned)((rows + 3) / 4)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), s, rows, S, scale, oscale, p, y);
  return check_launch("softmax_causal_f32_fwd");
}

int rte_softmax_causal_f32_bwd(const float* p, const float* dy, int64_t rows, int S, float scale,
                               const float* oscale, float* ds, void* stream) {
  RTE_REQUIRE(rows >= 0 && S >= 1 && p && dy && ds, "softmax_causal_f32_bwd: bad arguments");
  if (rows == 0) return 0;
  hipLaunchKernelGGL(softmax_causal_bwd_kernel, dim3((unsigned)((rows + 3) / 4)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), p, dy, rows, S, scale, oscale, ds);
  return check_launch("softmax_causal_f32_bwd");
}

int rte_swiglu_f32_fwd(const float* ug, int64_t rows, int n, int64_t ld, float* z, void* stream) {
  RTE_REQUIRE(rows >= 0 && n >= 1 && ld >= 2 * (int64_t)n && ug && z, "swiglu_f32_fwd: bad arguments");
  const int64_t total = rows * n;
  if (total == 0) return 0;
  hipLaunchKernelGGL(swiglu_f32_fwd_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), ug, rows, n, ld, z);
  return check_launch("swiglu_f32_fwd");
}

int rte_swiglu_f32_bwd(const float* ug, const float* dz, int64_t rows, int n, int64_t ld, float* dug, void* stream) {
  RTE_REQUIRE(rows >= 0 && n >= 1 && ld >= 2 * (int64_t)n && ug && dz && dug, "swiglu_f32_bwd: bad arguments");
  const int64_t total = rows * n;
  if (total == 0) return 0;
  hipLaunchKernelGGL(swiglu_f32_bwd_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), ug, dz, rows, n, ld, dug);
  return check_launch("swiglu_f32_bwd");
}

int rte_combine_f32(const float* rows, const int32_t* slot, const float* w, int T, int k, int d, const float* resid,
                    float* out, void* stream) {
  RTE_REQUIRE(T >= 0 && k >= 1 && d >= 1 && rows && slot && out, "combine_f32: bad arguments");
  if (T == 0) return 0;
  hipLaunchKernelGGL(combine_f32_kernel, dim3(T), dim3(d >= 256 ? 256 : 64), 0, static_cast<hipStream_t>(stream),
                     rows, slot, w, T, k, d, resid, out);
  return check_launch("combine_f32");
}

int rte_pair_dot_f32(const float* dout, const float* rows, const int32_t* slot, int64_t pairs, int k, int d, float* dw,
                     void* stream) {
  RTE_REQUIRE(pairs >= 0 && k >= 1 && d >= 1 && dout && rows && slot && dw, "pair_dot_f32: bad arguments");
  if (pairs == 0) return 0;
  hipLaunchKernelGGL(pair_dot_f32_kernel, dim3((unsigned)((pairs + 3) / 4)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), dout, rows, slot, pairs, k, d, dw);
  return check_launch("pair_dot_f32");
}

}  // extern "C"
