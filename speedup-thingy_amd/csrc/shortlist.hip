// Shortlist output head (rte/output.py:46-136, rte/kernels/reference.py:141-147):
// candidate build with first-occurrence dedupe, shortlist logits fused with the
// cross-entropy at target position 0, and the backward with a deterministic
// vocabulary-row gradient reduction.
//
// build   : one wave64 per token walks the candidate sequence
//             [target | members of its top vocab clusters | hard negatives arange(H) % V |
//              random negatives | filler arange(L) % V | (target + arange(2L)) % V]
//           64 candidates at a time.  A candidate is new when its bit is clear in the
//           wave's LDS bitmap of the vocabulary and no earlier lane of the chunk holds
//           it: one ballot per id bit finds the lanes that share an id (16384 tokens of
//           705 candidates: 58 us; 154 us when each lane was compared with every other
//           in turn).  New candidates take the next positions (ballot prefix count),
//           so the shortlist holds the first L distinct ids in candidate order -- the
//           order the reference obtains from scatter_reduce(amin) over [T, V] first
//           positions followed by topk(largest=False, sorted=True).
// fwd     : logits[t, j] = hidden[t] . W[shortlist[t, j]]; 8 lanes per vocab row, 8 rows
//           per wave pass; lse[t] = logsumexp_j logits[t, j]; loss[t] = lse[t] - logits[t, 0].
// bwd     : g[t, j] = dloss[t] (softmax_j - [j == 0]) + dlogits_ext[t, j]
//           dhidden[t] = sum_j g[t, j] W[shortlist[t, j]]: four sums over j mod 4, each
//           in ascending j, added as (0 + 1) + (2 + 3)
//           dW[v]      = sum over pairs (t, j) with shortlist[t, j] = v of g[t, j] hidden[t]
//           The pairs are counting-sorted by vocab row (stable: ascending pair index),
//           each row's run is summed in chunks by one wave per column slab, and chunk
//           partials are added in chunk order: no floating-point atomics, bitwise repeatable.
#include "common.hpp"

namespace rte {

size_t segreduce_workspace_bytes(int64_t P, int V, int d);
int segreduce_rows(const int32_t* keys, int64_t P, int V, int row_div, const float* w, const void* rows, int rows_f32,
                   int d, float* out, int accumulate, void* ws, size_t ws_bytes, hipStream_t s);

namespace {

constexpr int kMaxBuildVocab = 65536;  // 4 waves x 8 KB bitmap per block
constexpr int kMaxSortVocab = 32768;   // key range of the segmented reduction

// ----------------------------------------------------------------------------- build

__global__ void __launch_bounds__(256) shortlist_build_kernel(
    const int64_t* __restrict__ targets, const int32_t* __restrict__ top_clusters, int tc,
    const int64_t* __restrict__ members, int n_clusters, int per_cluster, const int64_t* __restrict__ random_negs,
    int R, int H, int L, int V, int T, int32_t* __restrict__ shortlist, int32_t* __restrict__ dup_per_token) {
  extern __shared__ uint32_t bitmap_all[];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int t = blockIdx.x * 4 + wave;
  const int words = (V + 31) / 32;
  uint32_t* bm = bitmap_all + wave * words;
  for (int w = lane; w < words; w += 64) bm[w] = 0u;
  __syncthreads();
  if (t >= T) return;  // no block-wide barrier below
  const int64_t tgt = targets[t];
  const int n_members = tc * per_cluster;
  const int width = 1 + n_members + H + R + L + 2 * L;
  const int bits = V > 1 ? 32 - __clz(V - 1) : 0;
  int count = 0;
  for (int c0 = 0; c0 < width; c0 += 64) {
    const int i = c0 + lane;
    int64_t cand = -1;
    if (i < width) {
      int rem = i;
      if (rem == 0) {
        cand = tgt;
      } else if ((rem -= 1) < n_members) {
        const int32_t cl = top_clusters[(int64_t)t * tc + rem / per_cluster];
        cand = (cl >= 0 && cl < n_clusters) ? members[(int64_t)cl * per_cluster + rem % per_cluster] : -1;
      } else if ((rem -= n_members) < H) {
        cand = rem % V;
      } else if ((rem -= H) < R) {
        cand = random_negs[(int64_t)t * R + rem];
      } else if ((rem -= R) < L) {
        cand = rem % V;
      } else {
        rem -= L;
        cand = ((tgt + rem) % V + V) % V;
      }
    }
    const int cv = (cand >= 0 && cand < V) ? (int)cand : -1;
    unsigned long long same = __ballot(cv >= 0);
    for (int b = 0; b < bits; ++b) {
      const bool one = (cv >> b) & 1;
      const unsigned long long m = __ballot(one);
      same &= one ? m : ~m;
    }
    const bool dup_in_chunk = (same & ((1ull << lane) - 1ull)) != 0;
    const bool fresh = cv >= 0 && !dup_in_chunk && !((bm[cv >> 5] >> (cv & 31)) & 1u);
    const unsigned long long mask = __ballot(fresh);
    const int rank = __popcll(mask & ((1ull << lane) - 1ull));
    if (fresh) {
      const int pos = count + rank;
      if (pos < L) shortlist[(int64_t)t * L + pos] = cv;
      atomicOr(&bm[cv >> 5], 1u << (cv & 31));
    }
    count += __popcll(mask);
  }
  if (lane == 0) dup_per_token[t] = width - count;
}

// ----------------------------------------------------------------------------- logits + CE

__device__ __forceinline__ float dot8(uint4 a, uint4 b) {
  const uint32_t aw[4] = {a.x, a.y, a.z, a.w};
  const uint32_t bw[4] = {b.x, b.y, b.z, b.w};
  float s = 0.0f;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    s += __uint_as_float(aw[i] << 16) * __uint_as_float(bw[i] << 16);
    s += __uint_as_float(aw[i] & 0xffff0000u) * __uint_as_float(bw[i] & 0xffff0000u);
  }
  return s;
}

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, 64));
  return v;
}

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// One wave per token.  Lane = G * grp + sub: group grp handles vocab row j0 + grp of the
// current pass (64 / G rows per pass), lane sub holds the 16-byte chunks sub, sub + G, ...
// of the row, so each load instruction reads whole 128-byte segments.  A lane holds at most
// NCMAX chunks: G grows with d so that the row chunks stay in registers.
template <int G, int NCMAX>
__global__ void __launch_bounds__(256) shortlist_fwd_kernel(const bf16* __restrict__ hidden,
                                                            const bf16* __restrict__ W, int d, int V,
                                                            const int32_t* __restrict__ sl, int L, int T,
                                                            float* __restrict__ logits, float* __restrict__ lse_out,
                                                            float* __restrict__ loss_out) {
  extern __shared__ float lg_all[];
  constexpr int RP = 64 / G;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int t = blockIdx.x * 4 + wave;
  const bool active = t < T;
  float* lg = lg_all + wave * L;
  const int grp = lane / G, sub = lane % G;
  const int nch = d >> 3;
  if (active) {
    uint4 h[NCMAX];
    const bf16* hrow = hidden + (int64_t)t * d;
#pragma unroll
    for (int i = 0; i < NCMAX; ++i)
      h[i] = sub + G * i < nch ? *reinterpret_cast<const uint4*>(hrow + (sub + G * i) * 8) : make_uint4(0u, 0u, 0u, 0u);
    for (int j0 = 0; j0 < L; j0 += RP) {
      const int j = j0 + grp;
      float s = 0.0f;
      if (j < L) {
        const int v = sl[(int64_t)t * L + j];
        if (v >= 0 && v < V) {
          const bf16* row = W + (int64_t)v * d;
          uint4 w[NCMAX];
#pragma unroll
          for (int i = 0; i < NCMAX; ++i)
            if (sub + G * i < nch) w[i] = *reinterpret_cast<const uint4*>(row + (sub + G * i) * 8);
#pragma unroll
          for (int i = 0; i < NCMAX; ++i)
            if (sub + G * i < nch) s += dot8(h[i], w[i]);
        } else {
          s = __builtin_nanf("");
        }
      }
#pragma unroll
      for (int off = 1; off < G; off <<= 1) s += __shfl_xor(s, off, 64);
      if (sub == 0 && j < L) {
        lg[j] = s;
        logits[(int64_t)t * L + j] = s;
      }
    }
  }
  __syncthreads();
  if (!active) return;
  float mx = -__builtin_inff();
  for (int j = lane; j < L; j += 64) mx = fmaxf(mx, lg[j]);
  mx = wave_max(mx);
  float se = 0.0f;
  for (int j = lane; j < L; j += 64) se += __expf(lg[j] - mx);
  se = wave_sum(se);
  if (lane == 0) {
    const float lse = mx + logf(se);
    lse_out[t] = lse;
    loss_out[t] = lse - lg[0];
  }
}

// g[t, :] and dhidden[t] = sum_j g[t, j] W[sl[t, j]].  One wave per token and slab of 128 columns (64
// ids and g values at a time in its lanes); 16 lanes of 8 columns take a row, the four groups of lanes
// every fourth row.  The waves of a slab run together on an XCD (dispatch id b runs on XCD b % 8), whose
// L2 then holds that slab of W: 16384 tokens of 128 rows of 1024, V 8192: 196 us, 226 with whole
// rows (330 with two columns per lane and one row per load).
__global__ void __launch_bounds__(256) shortlist_bwd_dh_kernel(
    const float* __restrict__ dloss, const float* __restrict__ dlext, const bf16* __restrict__ W, int d, int V,
    const int32_t* __restrict__ sl, int L, int T, const float* __restrict__ logits, const float* __restrict__ lse,
    float* __restrict__ g_out, bf16* __restrict__ dh, int nslab) {
  const int lane = threadIdx.x & 63;
  const int nb = gridDim.x, xcd = blockIdx.x & 7, q8 = nb >> 3, r8 = nb & 7;
  const int blk = xcd * q8 + (xcd < r8 ? xcd : r8) + (blockIdx.x >> 3);
  const int64_t id = (int64_t)blk * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int slab = (int)(id / T), t = (int)(id - (int64_t)slab * T);
  if (slab >= nslab) return;
  const float gt = dloss ? dloss[t] : 0.0f;
  const float ls = lse[t];
  const int grp = lane >> 4, col = slab * 128 + (lane & 15) * 8;
  const bool on = dh != nullptr && col < d;
  const bf16* base = W + (on ? col : 0);
  float acc[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
  for (int j0 = 0; j0 < L; j0 += 64) {
    const int j = j0 + lane;
    int vid = -1;
    float gj = 0.0f;
    if (j < L) {
      const int64_t o = (int64_t)t * L + j;
      vid = sl[o];
      if (dloss) gj = gt * (__expf(logits[o] - ls) - (j == 0 ? 1.0f : 0.0f));
      if (dlext) gj += dlext[o];
      if (slab == 0) g_out[o] = gj;
    }
    if (vid >= V) vid = -1;
    if (dh == nullptr) continue;
    const int n = L - j0 < 64 ? L - j0 : 64;
    for (int q0 = 0; q0 < n; q0 += 16) {
      uint4 u[4];
      float gq[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int q = q0 + 4 * i + grp, v = __shfl(vid, q, 64);
        gq[i] = __shfl(gj, q, 64);
        u[i] = on && v >= 0 ? *reinterpret_cast<const uint4*>(base + (int64_t)v * d) : make_uint4(0u, 0u, 0u, 0u);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint32_t w[4] = {u[i].x, u[i].y, u[i].z, u[i].w};
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          acc[2 * k] += gq[i] * __uint_as_float(w[k] << 16);
          acc[2 * k + 1] += gq[i] * __uint_as_float(w[k] & 0xffff0000u);
        }
      }
    }
  }
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    acc[i] += __shfl_xor(acc[i], 16, 64);
    acc[i] += __shfl_xor(acc[i], 32, 64);
  }
  if (!on || grp) return;
  *reinterpret_cast<uint4*>(dh + (int64_t)t * d + col) =
      make_uint4(pack_bf2(acc[0], acc[1]), pack_bf2(acc[2], acc[3]), pack_bf2(acc[4], acc[5]), pack_bf2(acc[6], acc[7]));
}

}  // namespace

int shortlist_build(const int64_t* targets, const int32_t* top_clusters, int tc, const int64_t* members,
                    int n_clusters, int per_cluster, const int64_t* random_negs, int R, int H, int L, int V, int T,
                    int32_t* shortlist, int32_t* dup_per_token, hipStream_t s) {
  RTE_REQUIRE(V >= 1 && V <= kMaxBuildVocab, "shortlist_build: vocab size must be in [1, %d]", kMaxBuildVocab);
  RTE_REQUIRE(L >= 1 && L <= V, "shortlist_build: need 1 <= L <= V (got L=%d, V=%d)", L, V);
  RTE_REQUIRE(tc >= 0 && per_cluster >= 0 && R >= 0 && H >= 0 && T >= 0, "shortlist_build: negative size");
  RTE_REQUIRE(tc == 0 || (n_clusters >= 1 && per_cluster >= 1), "shortlist_build: empty member table");
  RTE_REQUIRE((int64_t)tc * per_cluster + H + R + 3LL * L + 1 < (1LL << 30), "shortlist_build: too many candidates");
  if (T == 0) return 0;
  const size_t lds = (size_t)4 * ((V + 31) / 32) * sizeof(uint32_t);
  hipLaunchKernelGGL(shortlist_build_kernel, dim3((T + 3) / 4), dim3(256), lds, s, targets, top_clusters, tc,
                     members, n_clusters, per_cluster, random_negs, R, H, L, V, T, shortlist, dup_per_token);
  return check_launch("shortlist_build");
}

int shortlist_fwd(const bf16* hidden, const bf16* W, int d, int V, const int32_t* sl, int L, int T, float* logits,
                  float* lse, float* loss, hipStream_t s) {
  RTE_REQUIRE(d >= 8 && d % 8 == 0 && d <= 2048, "shortlist_fwd: d must be a multiple of 8 in [8, 2048]");
  RTE_REQUIRE(L >= 1 && L <= 4096 && V >= 1, "shortlist_fwd: need 1 <= L <= 4096");
  RTE_REQUIRE(((uintptr_t)hidden & 15) == 0 && ((uintptr_t)W & 15) == 0, "shortlist_fwd: 16-byte alignment");
  if (T == 0) return 0;
  const size_t lds = (size_t)4 * L * sizeof(float);
  const dim3 grid((T + 3) / 4), block(256);
#define RTE_SL_FWD(G, NC) \
  hipLaunchKernelGGL((shortlist_fwd_kernel<G, NC>), grid, block, lds, s, hidden, W, d, V, sl, L, T, logits, lse, loss)
  if (d <= 256)
    RTE_SL_FWD(8, 4);
  else if (d <= 512)
    RTE_SL_FWD(8, 8);
  else if (d <= 1024)
    RTE_SL_FWD(16, 8);
  else
    RTE_SL_FWD(32, 8);
#undef RTE_SL_FWD
  return check_launch("shortlist_fwd");
}

size_t shortlist_bwd_workspace_bytes(int T, int L, int V, int d) {
  if (T < 0 || L < 1 || V < 1 || d < 1) return 0;
  const size_t g_bytes = (((size_t)T * L * 4 + 255) / 256) * 256;
  return g_bytes + segreduce_workspace_bytes((int64_t)T * L, V, d);
}

int shortlist_bwd(const float* dloss, const float* dlext, const bf16* hidden, const bf16* W, int d, int V,
                  const int32_t* sl, int L, int T, const float* logits, const float* lse, bf16* dhidden, float* dW,
                  int dW_accumulate, void* ws, size_t ws_bytes, hipStream_t s) {
  RTE_REQUIRE(d >= 8 && d % 8 == 0 && d <= 2048, "shortlist_bwd: d must be a multiple of 8 in [8, 2048]");
  RTE_REQUIRE(L >= 1 && L <= 4096 && V >= 1, "shortlist_bwd: need 1 <= L <= 4096");
  RTE_REQUIRE(dW == nullptr || V <= kMaxSortVocab, "shortlist_bwd: dW needs vocab size <= %d", kMaxSortVocab);
  RTE_REQUIRE((int64_t)T * L < (1LL << 31), "shortlist_bwd: T * L must fit in int32");
  RTE_REQUIRE(((uintptr_t)hidden & 15) == 0 && ((uintptr_t)W & 15) == 0 && ((uintptr_t)ws & 255) == 0,
              "shortlist_bwd: hidden / W need 16-byte and workspace 256-byte alignment");
  const size_t need = shortlist_bwd_workspace_bytes(T, L, V, d);
  RTE_REQUIRE(ws_bytes >= need, "shortlist_bwd: workspace too small (%zu < %zu)", ws_bytes, need);
  if (T == 0) {
    if (dW && !dW_accumulate) return fill_f32(dW, 0.0f, (int64_t)V * d, s);
    return 0;
  }
  float* g = static_cast<float*>(ws);
  const size_t g_bytes = (((size_t)T * L * 4 + 255) / 256) * 256;
  const int nslab = dhidden ? (d + 127) / 128 : 1;
  const int64_t nwg = ((int64_t)T * nslab + 3) / 4;
  RTE_REQUIRE(nwg < ((int64_t)1 << 31), "shortlist_bwd: too many tokens");
  hipLaunchKernelGGL(shortlist_bwd_dh_kernel, dim3((unsigned)nwg), dim3(256), 0, s, dloss, dlext, W, d, V, sl, L, T,
                     logits, lse, g, dhidden, nslab);
  RTE_TRY(check_launch("shortlist_bwd_dhidden"));
  if (!dW) return 0;
  // dW[v] = sum over pairs (t, j) with sl[t, j] = v of g[t, j] hidden[t]: key = sl, row = p / L
  return segreduce_rows(sl, (int64_t)T * L, V, L, g, hidden, 0, d, dW, dW_accumulate,
                        static_cast<char*>(ws) + g_bytes, ws_bytes - g_bytes, s);
}

}  // namespace rte
