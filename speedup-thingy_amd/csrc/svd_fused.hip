// SVD low-rank SwiGLU FFN with the wide activations kept on chip (rte/layers.py:342-643, the
// low-rank factor products of SVDFactorSparseFFN, with U diag(S) V^T as the up, gate and down
// weights):
//
//   a    = x @ [A_up | A_gate]                  [T, 2r]   (A = U diag(S), GEMM)
//   u, g = a_up V_up^T, a_gate V_gate^T         [T, F]    never written
//   z    = u * silu(g)                          [T, F]    never written
//   b    = z @ V_dn                             [T, r]
//   y    = resid + b @ A_dn^T                   [T, d]    (GEMM)
//
// The middle part runs per 32 x 32 (token, neuron) block on v_mfma_f32_32x32x16_bf16 with the
// neuron index as the MFMA row dimension: the u / g / dz blocks then sit in the accumulators
// with the token index across lanes and the neuron index across registers, which is exactly the
// B-operand layout of the next product that sums over neurons (b, da) or, computed the other
// way round (token index as the row dimension), over tokens (the weight gradients).  The order
// in which the 32 neurons of a block enter that reduction is the accumulator's register order;
// the A operand is read from LDS in the same order.  Nothing of width F reaches HBM.
//
// Backward:
//   db = dy @ A_dn, dA_dn = dy^T b                                       (GEMMs)
//   bwdx (per token tile):  recompute u, g; dz = db V_dn^T; du = dz silu(g);
//                           dg = dz u silu'(g); da = [du V_up | dg V_gate]
//   bwdw (per neuron tile, split over tokens): recompute u, g, dz, z, du, dg and
//                           dV_up = du^T a_up, dV_gate = dg^T a_gate, dV_dn = z^T db
//   dx = da @ [A_up | A_gate]^T, d[A_up | A_gate] = x^T da                (GEMMs)
// Split partial sums (over neuron ranges in fwd / bwdx, over token ranges in bwdw) are fp32 and
// added in split order by a separate kernel: results are bitwise repeatable.
//
// MFMA lane layout (32x32x16): lane l supplies A row l % 32 and B column l % 32 with k values
// 8 (l / 32) .. +7 of each 16-step; output register r of lane l holds row 8 (r / 4) + 4 (l / 32)
// + r % 4, column l % 32.
#include "common.hpp"
#include "gemm_dev.hpp"

namespace rte {
namespace {

__device__ __forceinline__ f32x16_v sv_mfma(bf16x8_v a, bf16x8_v b, f32x16_v c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ bf16x8_v sv_ld8(const bf16* p) {
  return __builtin_bit_cast(bf16x8_v, *reinterpret_cast<const uint4*>(p));
}

__device__ __forceinline__ f32x16_v sv_zero() {
  f32x16_v z;
#pragma unroll
  for (int i = 0; i < 16; ++i) z[i] = 0.0f;
  return z;
}

// logistic function through the hardware exp and reciprocal (about 1 ulp each; the results
// feed bf16 MFMA operands)
__device__ __forceinline__ float sv_sigmoid(float x) { return __builtin_amdgcn_rcpf(1.0f + __expf(-x)); }

// A 32-row tile of one operand in LDS: rows of R bf16 as the matrix has them, 16-byte chunk c of
// row r stored at c ^ swz(r).  The operand reads of 16 consecutive rows (one chunk each) and the
// transposing reads (four consecutive rows, 64 bytes each) then both cover all banks once.
template <int R>
struct SvTile {
  static constexpr int CPR = R / 8, BYTES = 32 * R * 2, NV = R / 64;
  __device__ __forceinline__ static int swz(int r) {
    return CPR == 16 ? ((r & 3) << 2) | ((r >> 2) & 3) : (((r >> 1) & 1) << 2) | ((r >> 2) & 3);
  }
};

// The loop over 32-row tiles that the three kernels share.  Tile i of three matrices (m0, m1, m2:
// rows 32 i .. of `rows`, R columns at the given pitch) meets the wave's 32 columns (bu, bg, bd):
//   u = m0 bu, g = m1 bg, dz = m2 bd                              (rows x columns, over R)
//   acc_u += m0^T du, acc_g += m1^T dg (UG), acc_d += m2^T z (D)  (R x columns, over rows)
// Rows at or past `rows` read as zeros and add nothing.
//
// Tiles go from memory straight into LDS and serve both products: the second reads its operand
// transposed (ds_read_b64_tr_b16) from the same rows.  (With transposed copies of the matrices in
// memory a tile took 64 bytes from each of R rows that lie a power of two apart, all in one L2
// channel: 5300 - 9500 cycles a tile against 1300 - 1500 of matrix instructions.)  The accumulators leave
// room for one wave per SIMD in the backward kernels, so nothing else hides an LDS read or the
// vector work: both are spread by hand over slots of matrix instructions (without: 300 / 247 us for
// bwdw / bwdx).  What is left is issue: a wave issues about 400 instructions of 4 cycles a tile.
//
// T 32768, F 4096, R 128, us before and now: fwd 141, 108; bwdx 288, 186; bwdw 509, 217; and four
// transposes (22) gone.
template <int R, bool GRAD, bool UG, bool D>
struct SvMid {
  static constexpr int KS = R / 16, JB = R / 32, NV = SvTile<R>::NV, CPR = SvTile<R>::CPR, TB = SvTile<R>::BYTES;
  static constexpr int NM = 3;                               // matrices
  static constexpr int NB = (UG ? 2 : 0) + (D ? 1 : 0);          // second products
  static constexpr int NG = KS / 4, NU = GRAD ? KS / 2 : KS / 4;  // slots of the gate and up products
  static constexpr int NS = JB / 2;                              // slots of a step of the second
  f32x16_v acc_u[UG ? JB : 1], acc_g[UG ? JB : 1], acc_d[D ? JB : 1];
  bf16x8_v bu[KS], bg[KS], bd[GRAD ? KS : 1];
  f32x16_v u, g, dz, sl;         // of the tile in work; sl: silu(g)
  uint32_t pz[8], pu[8], pg[8];  // bf16 pairs of z, du, dg by accumulator row
  int ra[KS], ta[JB][2];
  const bf16* m[NM];
  int pitch[NM];
  uint32_t voff[NM][NV];
  int rows, wave;

  __device__ __forceinline__ void init(const bf16* m0, int p0, const bf16* m1, int p1, const bf16* m2, int p2,
                                       int nrows) {
    const int tid = threadIdx.x, lane = tid & 63, h = lane >> 5, l32 = lane & 31;
    wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    rows = nrows;
    m[0] = m0; m[1] = m1; m[2] = m2;
    pitch[0] = p0; pitch[1] = p1; pitch[2] = p2;
#pragma unroll
    for (int k = 0; k < NM; ++k)
#pragma unroll
      for (int q = 0; q < NV; ++q) {
        const int r = (tid + 256 * q) / CPR, c = (tid + 256 * q) % CPR;
        voff[k][q] = (uint32_t)(r * pitch[k] + (c ^ SvTile<R>::swz(r)) * 8) * 2;
      }
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) ra[ks] = (l32 * CPR + ((2 * ks + h) ^ SvTile<R>::swz(l32))) * 16;
    const int i = lane & 15, sub = (lane >> 4) & 1;
#pragma unroll
    for (int jb = 0; jb < JB; ++jb)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int r = 8 * j + 4 * h + (i >> 2), col = 32 * jb + 16 * sub + 4 * (i & 3);
        ta[jb][j] = (r * CPR + ((col >> 3) ^ SvTile<R>::swz(r))) * 16 + (col & 7) * 2;
      }
#pragma unroll
    for (int jb = 0; jb < JB; ++jb) {
      if constexpr (UG) acc_u[jb] = acc_g[jb] = sv_zero();
      if constexpr (D) acc_d[jb] = sv_zero();
    }
  }

  // tile i into a stage; tiles at or past `end` load nothing (zero-length descriptors)
  __device__ __forceinline__ void load(unsigned char* st, int i, int end) const {
    const int left = rows - i * 32, nr = i < end ? (left < 32 ? left : 32) : 0;
#pragma unroll
    for (int k = 0; k < NM; ++k) {
      const BufferRsrc rs = buffer_rsrc(m[k] + (int64_t)(i < end ? i : 0) * 32 * pitch[k],
                                        nr ? (uint32_t)((nr - 1) * pitch[k] + R) * 2 : 0u);
#pragma unroll
      for (int q = 0; q < NV; ++q) lds_dma16_buf(rs, st + k * TB + (q * 256 + wave * 64) * 16, voff[k][q], 0);
    }
  }

  // Operands of a slot and its matrix instructions.  Gate: k steps 4n .. 4n + 3 of g = m1 bg.
  __device__ __forceinline__ void read_gate(const unsigned char* st, int n, bf16x8_v* f) const {
#pragma unroll
    for (int e = 0; e < 4; ++e) f[e] = *reinterpret_cast<const bf16x8_v*>(st + TB + ra[4 * n + e]);
  }
  __device__ __forceinline__ void mm_gate(const bf16x8_v* f, int n) {
#pragma unroll
    for (int e = 0; e < 4; ++e) g = sv_mfma(f[e], bg[4 * n + e], n + e == 0 ? sv_zero() : g);
  }
  // Up: k steps 2n, 2n + 1 of u = m0 bu and dz = m2 bd (4n .. 4n + 3 without dz).
  __device__ __forceinline__ void read_up(const unsigned char* st, int n, bf16x8_v* f) const {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int k = GRAD ? e & 1 : 0, ks = GRAD ? 2 * n + (e >> 1) : 4 * n + e;
      f[e] = *reinterpret_cast<const bf16x8_v*>(st + 2 * k * TB + ra[ks]);
    }
  }
  __device__ __forceinline__ void mm_up(const bf16x8_v* f, int n) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int ks = GRAD ? 2 * n + (e >> 1) : 4 * n + e;
      if (GRAD && (e & 1)) dz = sv_mfma(f[e], bd[GRAD ? ks : 0], ks == 0 ? sv_zero() : dz);
      else u = sv_mfma(f[e], bu[ks], ks == 0 ? sv_zero() : u);
    }
  }
  // Second products of step s (accumulator rows 8 s ..), blocks 2n, 2n + 1: rows of the tile turned
  // into columns, in the accumulators' row order.
  __device__ __forceinline__ void read_second(const unsigned char* st, int s, int n, bf16x8_v* f) const {
#pragma unroll
    for (int e = 0; e < 2; ++e)
#pragma unroll
      for (int k = 0; k < NB; ++k) {
        const unsigned char* t = st + (UG ? k : 2) * TB + s * 16 * CPR * 16;
        const short4_v lo = lds_read_tr4(t + ta[2 * n + e][0]), hi = lds_read_tr4(t + ta[2 * n + e][1]);
        typedef short short8_v __attribute__((ext_vector_type(8)));
        f[e * NB + k] = __builtin_bit_cast(bf16x8_v, (short8_v)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
      }
  }
  __device__ __forceinline__ void mm_second(const bf16x8_v* f, int s, int n) {
#pragma unroll
    for (int e = 0; e < 2; ++e)
#pragma unroll
      for (int k = 0; k < NB; ++k) {
        const uint32_t* p = (UG ? (k == 0 ? pu : k == 1 ? pg : pz) : pz) + 4 * s;
        const bf16x8_v b = __builtin_bit_cast(bf16x8_v, make_uint4(p[0], p[1], p[2], p[3]));
        f32x16_v& acc = UG ? (k == 0 ? acc_u[2 * n + e] : k == 1 ? acc_g[2 * n + e] : acc_d[D ? 2 * n + e : 0])
                           : acc_d[D ? 2 * n + e : 0];
        acc = sv_mfma(f[e * NB + k], b, acc);
      }
  }

  // Vector work on accumulator rows r0 .. r0 + N - 1: silu(g) and silu'(g) (left in g) ...
  template <int N>
  __device__ __forceinline__ void gate(int r0) {
#pragma unroll
    for (int r = r0; r < r0 + N; ++r) {
      const float sg = sv_sigmoid(g[r]);
      sl[r] = g[r] * sg;
      if constexpr (UG) g[r] = sg + sl[r] * (1.0f - sg);
    }
  }
  // ... and the bf16 operands of the second products.
  template <int N>
  __device__ __forceinline__ void act(int r0) {
#pragma unroll
    for (int r = r0; r < r0 + N; r += 2) {
      if constexpr (D) pz[r / 2] = pack_bf2(u[r] * sl[r], u[r + 1] * sl[r + 1]);
      if constexpr (UG) {
        pu[r / 2] = pack_bf2(dz[r] * sl[r], dz[r + 1] * sl[r + 1]);
        pg[r / 2] = pack_bf2(dz[r] * u[r] * g[r], dz[r + 1] * u[r + 1] * g[r + 1]);
      }
    }
  }

  __device__ __forceinline__ static void fence() {
#if defined(__HIP_DEVICE_COMPILE__)
    __builtin_amdgcn_sched_barrier(0);
#endif
  }
  // Order within a slot: M matrix instructions, V vector and X exp / reciprocal instructions after each.
  template <int M, int V, int X, int L>
  __device__ __forceinline__ static void weave() {
#if defined(__HIP_DEVICE_COMPILE__)
    constexpr int kVector = 0x2, kMatrix = 0x8, kLdsRead = 0x100, kTrans = 0x400;
#pragma unroll
    for (int n = 0; n < M; ++n) {
      __builtin_amdgcn_sched_group_barrier(kMatrix, 1, 0);
      __builtin_amdgcn_sched_group_barrier(kLdsRead, L, 0);
      if constexpr (X > 0) __builtin_amdgcn_sched_group_barrier(kTrans, X, 0);
      if constexpr (V > 0) __builtin_amdgcn_sched_group_barrier(kVector, V, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
#endif
  }

  // Tile i in slots of 4 to 6 matrix instructions.  A slot begins with the LDS reads of the slot after it
  // and carries a share of the vector work, so that a wave alone on its SIMD keeps the matrix cores
  // busy.  Order: gate products; up products (gate functions of the vector unit); second products of
  // step 1 of tile i - 1 (operands of step 0); barrier; second products of step 0 (operands of step 1).
  template <bool START>
  __device__ __forceinline__ void tile(const unsigned char* cur, unsigned char* prev, const unsigned char* next, int i,
                                       int end, bf16x8_v (*f)[6]) {
    constexpr int GV = UG ? 5 : 3;                       // vector instructions per gate row
    constexpr int AV = (UG ? 4 : 0) + (D ? 2 : 0);       // per operand row, about
    constexpr int UR = 16 / NU, SR = 8 / NS;             // rows per slot
    int q = 0;
#pragma unroll
    for (int n = 0; n < NG; ++n, ++q) {
      if (n + 1 < NG) read_gate(cur, n + 1, f[(q + 1) & 1]);
      else read_up(cur, 0, f[(q + 1) & 1]);
      mm_gate(f[q & 1], n);
      weave<4, 0, 0, 1>();
    }
#pragma unroll
    for (int n = 0; n < NU; ++n, ++q) {
      if (n + 1 < NU) read_up(cur, n + 1, f[(q + 1) & 1]);
      else if (START) read_second(cur, 0, 0, f[(q + 1) & 1]);
      else read_second(prev, 1, 0, f[(q + 1) & 1]);
      mm_up(f[q & 1], n);
      gate<UR>(n * UR);
      weave<4, (UR * GV + 3) / 4, (UR * 2 + 3) / 4, 1>();
    }
#pragma unroll
    for (int n = 0; n < NS; ++n) {
      if (!START) {
        if (n + 1 < NS) read_second(prev, 1, n + 1, f[(q + 1) & 1]);
        else read_second(cur, 0, 0, f[(q + 1) & 1]);
        mm_second(f[q & 1], 1, n);
        ++q;
      }
      act<SR>(n * SR);
      if (!START) weave<2 * NB, (SR * AV + 2 * NB - 1) / (2 * NB), 0, 2>();
    }
    wait_vmcnt_lgkm0<0>();
    wg_barrier();  // tile i + 1 is in LDS, every wave is done with tile i - 1
    load(prev, i + 2, end);
    fence();
    bf16x8_v ahead[4];
#pragma unroll
    for (int n = 0; n < NS; ++n, ++q) {
      if (n + 1 < NS) read_second(cur, 0, n + 1, f[(q + 1) & 1]);
      else read_gate(next, 0, ahead);
      mm_second(f[q & 1], 0, n);
      act<SR>(8 + n * SR);
      weave<2 * NB, (SR * AV + 2 * NB - 1) / (2 * NB), 0, 2>();
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) f[0][e] = ahead[e];
  }
  __device__ __forceinline__ void run(unsigned char* s0, unsigned char* s1, unsigned char* s2, int i0, int i1) {
    if (i0 >= i1) return;
    load(s0, i0, i1);
    load(s1, i0 + 1, i1);
    bf16x8_v f[2][6];
    wait_vmcnt_lgkm0<NM * NV>();
    wg_barrier();
    read_gate(s0, 0, f[0]);
    tile<true>(s0, s2, s1, i0, i1, f);
    int i = i0 + 1;
    for (; i + 2 < i1; i += 3) {
      tile<false>(s1, s0, s2, i, i1, f);
      tile<false>(s2, s1, s0, i + 1, i1, f);
      tile<false>(s0, s2, s1, i + 2, i1, f);
    }
    if (i < i1) tile<false>(s1, s0, s2, i, i1, f);
    if (i + 1 < i1) tile<false>(s2, s1, s0, i + 1, i1, f);
    const int last = (i1 - 1 - i0) % 3;
    const unsigned char* st = last == 0 ? s0 : last == 1 ? s1 : s2;
#pragma unroll
    for (int n = 0; n < NS; ++n) {  // step 1 of the last tile
      read_second(st, 1, n, f[0]);
      mm_second(f[0], 1, n);
    }
    wait_vmcnt<0>();
  }
};

// One row of a wave's R x 32 accumulator blocks per lane column: element j of row `out` (16-byte
// fp32 or 8-byte bf16 stores)
template <int JB>
__device__ __forceinline__ void sv_store(const f32x16_v* acc, int h, float* f32_row, bf16* bf16_row) {
#pragma unroll
  for (int jb = 0; jb < JB; ++jb) {
    const f32x16_v& a = acc[jb];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int j = jb * 32 + 8 * q + 4 * h;
      if (f32_row != nullptr)
        *reinterpret_cast<float4*>(f32_row + j) = make_float4(a[4 * q], a[4 * q + 1], a[4 * q + 2], a[4 * q + 3]);
      else
        *reinterpret_cast<uint2*>(bf16_row + j) =
            make_uint2(pack_bf2(a[4 * q], a[4 * q + 1]), pack_bf2(a[4 * q + 2], a[4 * q + 3]));
    }
  }
}

// Stages are arrays of their own: from one array the transposing reads wait for every load in flight.
#define SVD_STAGE(name) __shared__ __align__(1024) unsigned char name[3 * SvTile<R>::BYTES]

// Forward middle: b (or fp32 partials over neuron splits) from a = [a_up | a_gate].
// grid (ceil(T / 128), splits), 256 threads; wave w owns tokens blockIdx.x * 128 + 32 w + (0..31);
// split y covers neuron chunks [y cps, (y + 1) cps) of 32 neurons.
template <int R>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void svd_mid_fwd_kernel(
    const bf16* __restrict__ a_ug, const bf16* __restrict__ v_ug, const bf16* __restrict__ v_dn, int T, int F, int cps,
    bf16* __restrict__ b_out, float* __restrict__ part) {
  SVD_STAGE(s0);
  SVD_STAGE(s1);
  SVD_STAGE(s2);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, h = lane >> 5, l32 = lane & 31;
  const int t = blockIdx.x * 128 + w * 32 + l32;
  const int tl = t < T ? t : T - 1;
  const int nc = F / 32;
  const int c0 = blockIdx.y * cps;
  const int c1 = c0 + cps < nc ? c0 + cps : nc;
  SvMid<R, false, false, true> k;
  k.init(v_ug, R, v_ug + (int64_t)F * R, R, v_dn, R, F);
  const bf16* arow = a_ug + (int64_t)tl * 2 * R + 8 * h;
#pragma unroll
  for (int ks = 0; ks < k.KS; ++ks) {
    k.bu[ks] = sv_ld8(arow + 16 * ks);
    k.bg[ks] = sv_ld8(arow + R + 16 * ks);
  }
  k.run(s0, s1, s2, c0, c1);
  if (t >= T) return;
  sv_store<R / 32>(k.acc_d, h, part ? part + ((int64_t)blockIdx.y * T + t) * R : nullptr, b_out + (int64_t)t * R);
}

// Backward to the low-rank codes: da = [du V_up | dg V_gate] per token tile (fp32 partials over
// neuron splits when splits > 1).  Layout and grid as svd_mid_fwd_kernel.
template <int R>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) void svd_mid_bwdx_kernel(
    const bf16* __restrict__ a_ug, const bf16* __restrict__ db, const bf16* __restrict__ v_ug,
    const bf16* __restrict__ v_dn, int T, int F, int cps, bf16* __restrict__ da_out, float* __restrict__ part) {
  SVD_STAGE(s0);
  SVD_STAGE(s1);
  SVD_STAGE(s2);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, h = lane >> 5, l32 = lane & 31;
  const int t = blockIdx.x * 128 + w * 32 + l32;
  const int tl = t < T ? t : T - 1;
  const int nc = F / 32;
  const int c0 = blockIdx.y * cps;
  const int c1 = c0 + cps < nc ? c0 + cps : nc;
  SvMid<R, true, true, false> k;
  k.init(v_ug, R, v_ug + (int64_t)F * R, R, v_dn, R, F);
  const bf16* arow = a_ug + (int64_t)tl * 2 * R + 8 * h;
  const bf16* drow = db + (int64_t)tl * R + 8 * h;
#pragma unroll
  for (int ks = 0; ks < k.KS; ++ks) {
    k.bu[ks] = sv_ld8(arow + 16 * ks);
    k.bg[ks] = sv_ld8(arow + R + 16 * ks);
    k.bd[ks] = sv_ld8(drow + 16 * ks);
  }
  k.run(s0, s1, s2, c0, c1);
  if (t >= T) return;
  float* prow = part ? part + ((int64_t)blockIdx.y * T + t) * 2 * R : nullptr;
  bf16* orow = da_out + (int64_t)t * 2 * R;
  sv_store<R / 32>(k.acc_u, h, prow, orow);
  sv_store<R / 32>(k.acc_g, h, prow ? prow + R : nullptr, orow + R);
}

// Backward to the factors V_up, V_gate, V_dn: grid (splits, F / 128), 256 threads; wave w owns
// neurons blockIdx.y * 128 + 32 w + (0..31) (the lane index); split x reduces token tiles
// [x tps, (x + 1) tps) of 32 tokens (consecutive workgroups run on different XCDs, so one L2 mostly
// sees one token range).  Writes [dV_up; dV_gate] ([2F][R]) and dV_dn ([F][R]) in fp32, or fp32
// partials [split][3F][R] when splits > 1.
template <int R>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) void svd_mid_bwdw_kernel(
    const bf16* __restrict__ a_ug, const bf16* __restrict__ db, const bf16* __restrict__ v_ug,
    const bf16* __restrict__ v_dn, int T, int F, int tps, float* __restrict__ dv_ug, float* __restrict__ dv_dn,
    float* __restrict__ part) {
  SVD_STAGE(s0);
  SVD_STAGE(s1);
  SVD_STAGE(s2);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, h = lane >> 5, l32 = lane & 31;
  const int64_t f = (int64_t)blockIdx.y * 128 + w * 32 + l32;
  const int nt = (T + 31) / 32;
  const int t0 = blockIdx.x * tps;
  const int t1 = t0 + tps < nt ? t0 + tps : nt;
  SvMid<R, true, true, true> k;
  k.init(a_ug, 2 * R, a_ug + R, 2 * R, db, R, T);
#pragma unroll
  for (int ks = 0; ks < k.KS; ++ks) {
    k.bu[ks] = sv_ld8(v_ug + f * R + 16 * ks + 8 * h);
    k.bg[ks] = sv_ld8(v_ug + (F + f) * R + 16 * ks + 8 * h);
    k.bd[ks] = sv_ld8(v_dn + f * R + 16 * ks + 8 * h);
  }
  k.run(s0, s1, s2, t0, t1);
  float* p = part ? part + ((int64_t)blockIdx.x * 3 * F + f) * R : nullptr;
  sv_store<R / 32>(k.acc_u, h, p ? p : dv_ug + f * R, nullptr);
  sv_store<R / 32>(k.acc_g, h, p ? p + (int64_t)F * R : dv_ug + (F + f) * R, nullptr);
  sv_store<R / 32>(k.acc_d, h, p ? p + (int64_t)2 * F * R : dv_dn + f * R, nullptr);
}

// out = sum over splits y (in order) of part[y][e]; elements e < n0 go to out0 (fp32 or bf16),
// the rest to out1 (same type) at e - n0.  n0 and n are multiples of 4.
__global__ __launch_bounds__(256) void svd_split_sum_kernel(const float* __restrict__ part, int splits, int64_t n,
                                                            int64_t n0, void* out0, void* out1, int out_bf16) {
  const int64_t e = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
  if (e >= n) return;
  float4 s = *reinterpret_cast<const float4*>(part + e);
  for (int y = 1; y < splits; ++y) {
    const float4 v = *reinterpret_cast<const float4*>(part + (int64_t)y * n + e);
    s.x += v.x;
    s.y += v.y;
    s.z += v.z;
    s.w += v.w;
  }
  const bool first = e < n0;
  const int64_t o = first ? e : e - n0;
  void* base = first ? out0 : out1;
  if (out_bf16) {
    *reinterpret_cast<uint2*>(static_cast<bf16*>(base) + o) = make_uint2(pack_bf2(s.x, s.y), pack_bf2(s.z, s.w));
  } else {
    *reinterpret_cast<float4*>(static_cast<float*>(base) + o) = s;
  }
}

int split_sum(const float* part, int splits, int64_t n, int64_t n0, void* out0, void* out1, int out_bf16,
              hipStream_t s) {
  const int64_t blocks = (n / 4 + 255) / 256;
  hipLaunchKernelGGL(svd_split_sum_kernel, dim3((unsigned)blocks), dim3(256), 0, s, part, splits, n, n0, out0, out1,
                     out_bf16);
  return check_launch("svd_split_sum");
}

Operand op_plain(const void* p, int64_t ld) {
  Operand o;
  o.ptr = static_cast<const bf16*>(p);
  o.ld = ld;
  return o;
}

size_t align256(size_t n) { return (n + 255) & ~(size_t)255; }

// neuron-range splits of the per-token-tile kernels: enough workgroups for one per CU, at least 2
// chunks of 32 neurons per split
int mid_splits(int T, int F, int target) {
  const int gx = (T + 127) / 128;
  int fs = (target + gx - 1) / gx;
  const int cap = F / 64 > 1 ? F / 64 : 1;
  if (fs > cap) fs = cap;
  return fs < 1 ? 1 : fs;
}

int w_splits(int T, int F) {
  const int gx = F / 128;
  const int nt = (T + 31) / 32;
  int ts = (256 + gx - 1) / gx;
  if (ts > nt) ts = nt;
  return ts < 1 ? 1 : ts;
}

struct FusedWs {
  size_t gemm = 0, part = 0, total = 0;
};

FusedWs fused_layout(int T, int d, int F, int r) {
  FusedWs L;
  size_t g = gemm_splitk_bytes(d, 2 * r, T);
  const size_t g2 = gemm_splitk_bytes(d, r, T);
  L.gemm = align256(g > g2 ? g : g2);
  const size_t p_fwd = (size_t)mid_splits(T, F, 512) * T * r * 4;
  const size_t p_bx = (size_t)mid_splits(T, F, 256) * T * 2 * r * 4;
  const size_t p_bw = (size_t)w_splits(T, F) * 3 * F * r * 4;
  size_t p = p_fwd > p_bx ? p_fwd : p_bx;
  p = p > p_bw ? p : p_bw;
  L.part = align256(p);
  L.total = L.gemm + L.part;
  return L;
}

}  // namespace
}  // namespace rte

using namespace rte;

extern "C" {

size_t rte_svd_ffn_fused_workspace_bytes(int T, int d, int F, int r) {
  if (T <= 0 || d <= 0 || F <= 0 || r <= 0) return 256;
  return fused_layout(T, d, F, r).total;
}

int rte_svd_ffn_fused_fwd(const void* x, int T, int d, int F, int r, const void* us_ug, const void* v_ug,
                          const void* v_dn, const void* us_dn, const float* resid, void* a_ug, void* b, void* y,
                          int y_f32, void* workspace, size_t workspace_bytes, void* stream) {
  RTE_REQUIRE(r == 64 || r == 128, "svd_ffn_fused: rank must be 64 or 128 (got %d)", r);
  RTE_REQUIRE(F % 128 == 0 && d % 8 == 0 && T % 8 == 0 && T >= 0,
              "svd_ffn_fused: need F %% 128, d %% 8, T %% 8 == 0 (F=%d d=%d T=%d)", F, d, T);
  if (T == 0) return 0;
  const FusedWs L = fused_layout(T, d, F, r);
  RTE_REQUIRE(workspace != nullptr && workspace_bytes >= L.total,
              "svd_ffn_fused: workspace of %zu bytes needed", L.total);
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  char* ws = static_cast<char*>(workspace);
  float* part = reinterpret_cast<float*>(ws + L.gemm);
  {
    GemmArgs p;  // a_ug = x @ us_ug : B(n=j, k=dcol) = us_ug[dcol][j]
    p.M = T;
    p.N = 2 * r;
    p.K = d;
    p.a = op_plain(x, d);
    p.b = op_plain(us_ug, 2 * r);
    p.b_t = 1;
    p.epi.c = a_ug;
    p.epi.ldc = 2 * r;
    RTE_TRY(gemm_launch(p, EPI_STORE, st));
  }
  const int fs = mid_splits(T, F, 512);
  const int nc = F / 32;
  const int cps = (nc + fs - 1) / fs;
  dim3 grid((T + 127) / 128, fs);
  float* pp = fs > 1 ? part : nullptr;
  if (r == 128)
    hipLaunchKernelGGL(svd_mid_fwd_kernel<128>, grid, dim3(256), 0, st, static_cast<const bf16*>(a_ug),
                       static_cast<const bf16*>(v_ug), static_cast<const bf16*>(v_dn), T, F, cps, static_cast<bf16*>(b), pp);
  else
    hipLaunchKernelGGL(svd_mid_fwd_kernel<64>, grid, dim3(256), 0, st, static_cast<const bf16*>(a_ug),
                       static_cast<const bf16*>(v_ug), static_cast<const bf16*>(v_dn), T, F, cps, static_cast<bf16*>(b), pp);
  RTE_TRY(check_launch("svd_mid_fwd"));
  if (fs > 1) RTE_TRY(split_sum(part, fs, (int64_t)T * r, (int64_t)T * r, b, b, 1, st));
  {
    GemmArgs p;  // y = resid + b @ us_dn^T : B(n=dcol, k=j) = us_dn[dcol][j]
    p.M = T;
    p.N = d;
    p.K = r;
    p.a = op_plain(b, r);
    p.b = op_plain(us_dn, r);
    p.epi.c = y;
    p.epi.ldc = d;
    p.epi.c_f32 = y_f32;
    p.epi.resid = resid;
    p.epi.ld_resid = d;
    RTE_TRY(gemm_launch(p, EPI_STORE, st));
  }
  return 0;
}

int rte_svd_ffn_fused_bwd(const void* dy, const void* x, int T, int d, int F, int r, const void* us_ug,
                          const void* v_ug, const void* v_dn, const void* us_dn, const void* a_ug, const void* b,
                          void* db, void* da_ug, void* dx, float* dus_ug, float* dv_ug, float* dv_dn, float* dus_dn,
                          void* workspace, size_t workspace_bytes, void* stream) {
  RTE_REQUIRE(r == 64 || r == 128, "svd_ffn_fused: rank must be 64 or 128 (got %d)", r);
  RTE_REQUIRE(F % 128 == 0 && d % 8 == 0 && T % 8 == 0 && T >= 0,
              "svd_ffn_fused: need F %% 128, d %% 8, T %% 8 == 0 (F=%d d=%d T=%d)", F, d, T);
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  if (T == 0) {
    RTE_TRY(fill_f32(dus_ug, 0.0f, (int64_t)d * 2 * r, st));
    RTE_TRY(fill_f32(dv_ug, 0.0f, (int64_t)2 * F * r, st));
    RTE_TRY(fill_f32(dv_dn, 0.0f, (int64_t)F * r, st));
    return fill_f32(dus_dn, 0.0f, (int64_t)d * r, st);
  }
  const FusedWs L = fused_layout(T, d, F, r);
  RTE_REQUIRE(workspace != nullptr && workspace_bytes >= L.total,
              "svd_ffn_fused: workspace of %zu bytes needed", L.total);
  char* ws = static_cast<char*>(workspace);
  void* gws = ws;
  float* part = reinterpret_cast<float*>(ws + L.gemm);
  {
    GemmArgs p;  // db = dy @ us_dn : B(n=j, k=dcol) = us_dn[dcol][j]
    p.M = T;
    p.N = r;
    p.K = d;
    p.a = op_plain(dy, d);
    p.b = op_plain(us_dn, r);
    p.b_t = 1;
    p.epi.c = db;
    p.epi.ldc = r;
    RTE_TRY(gemm_launch(p, EPI_STORE, st));
  }
  {
    GemmArgs p;  // dus_dn[dcol, j] = sum_t dy[t, dcol] b[t, j]
    p.M = d;
    p.N = r;
    p.K = T;
    p.a = op_plain(dy, d);
    p.a_t = 1;
    p.b = op_plain(b, r);
    p.b_t = 1;
    p.epi.c = dus_dn;
    p.epi.ldc = r;
    p.epi.c_f32 = 1;
    RTE_TRY(gemm_launch(p, EPI_STORE, st, gws, L.gemm));
  }
  {
    const int fs = mid_splits(T, F, 256);
    const int nc = F / 32;
    const int cps = (nc + fs - 1) / fs;
    dim3 grid((T + 127) / 128, fs);
    float* pp = fs > 1 ? part : nullptr;
    if (r == 128)
      hipLaunchKernelGGL(svd_mid_bwdx_kernel<128>, grid, dim3(256), 0, st, static_cast<const bf16*>(a_ug),
                         static_cast<const bf16*>(db), static_cast<const bf16*>(v_ug),
                         static_cast<const bf16*>(v_dn), T, F, cps, static_cast<bf16*>(da_ug), pp);
    else
      hipLaunchKernelGGL(svd_mid_bwdx_kernel<64>, grid, dim3(256), 0, st, static_cast<const bf16*>(a_ug),
                         static_cast<const bf16*>(db), static_cast<const bf16*>(v_ug),
                         static_cast<const bf16*>(v_dn), T, F, cps, static_cast<bf16*>(da_ug), pp);
    RTE_TRY(check_launch("svd_mid_bwdx"));
    if (fs > 1) RTE_TRY(split_sum(part, fs, (int64_t)T * 2 * r, (int64_t)T * 2 * r, da_ug, da_ug, 1, st));
  }
  {
    const int ts = w_splits(T, F);
    const int nt = (T + 31) / 32;
    const int tps = (nt + ts - 1) / ts;
    dim3 grid(ts, F / 128);
    float* pp = ts > 1 ? part : nullptr;
    if (r == 128)
      hipLaunchKernelGGL(svd_mid_bwdw_kernel<128>, grid, dim3(256), 0, st, static_cast<const bf16*>(a_ug),
                         static_cast<const bf16*>(db), static_cast<const bf16*>(v_ug),
                         static_cast<const bf16*>(v_dn), T, F, tps, dv_ug, dv_dn, pp);
    else
      hipLaunchKernelGGL(svd_mid_bwdw_kernel<64>, grid, dim3(256), 0, st, static_cast<const bf16*>(a_ug),
                         static_cast<const bf16*>(db), static_cast<const bf16*>(v_ug),
                         static_cast<const bf16*>(v_dn), T, F, tps, dv_ug, dv_dn, pp);
    RTE_TRY(check_launch("svd_mid_bwdw"));
    if (ts > 1) RTE_TRY(split_sum(part, ts, (int64_t)3 * F * r, (int64_t)2 * F * r, dv_ug, dv_dn, 0, st));
  }
  {
    GemmArgs p;  // dx = da_ug @ us_ug^T : B(n=dcol, k=j) = us_ug[dcol][j]
    p.M = T;
    p.N = d;
    p.K = 2 * r;
    p.a = op_plain(da_ug, 2 * r);
    p.b = op_plain(us_ug, 2 * r);
    p.epi.c = dx;
    p.epi.ldc = d;
    RTE_TRY(gemm_launch(p, EPI_STORE, st));
  }
  {
    GemmArgs p;  // dus_ug[dcol, j] = sum_t x[t, dcol] da_ug[t, j]
    p.M = d;
    p.N = 2 * r;
    p.K = T;
    p.a = op_plain(x, d);
    p.a_t = 1;
    p.b = op_plain(da_ug, 2 * r);
    p.b_t = 1;
    p.epi.c = dus_ug;
    p.epi.ldc = 2 * r;
    p.epi.c_f32 = 1;
    RTE_TRY(gemm_launch(p, EPI_STORE, st, gws, L.gemm));
  }
  return 0;
}

}  // extern "C"
