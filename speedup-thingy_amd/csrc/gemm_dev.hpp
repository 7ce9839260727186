// Device helpers shared by the GEMM kernels (gemm.hip, gemm_tile.hip): operand addressing, output
// chunks, direct-to-LDS loads, LDS swizzles and waits.
#pragma once

#include "gemm.hpp"

namespace rte {
namespace {

__device__ __forceinline__ int64_t ilv_row(int64_t r, int32_t half) {
  return ((r & 63) < 32 ? 0 : half) + (r >> 6) * 32 + (r & 31);
}

__device__ __forceinline__ int log2i(int v) { return 31 - __clz(v); }

__device__ __forceinline__ int64_t row_off(const Operand& o, int64_t r) {
  if (o.ilv) r = ilv_row(r, o.ilv);
  if (o.rows) r = o.rows[r];
  if (o.rdiv) return (r >> log2i(o.rdiv)) * o.rs_hi + (r & (o.rdiv - 1)) * o.ld;
  return r * o.ld;
}

__device__ __forceinline__ int64_t col_off(const Operand& o, int c) {
  if (o.cdiv) return (int64_t)(c >> log2i(o.cdiv)) * o.cs_hi + (c & (o.cdiv - 1));
  return c;
}

// ------------------------------------------------------------------ output chunks

// Writes W consecutive outputs (row m of the tile space, columns n..n+W-1) applying
// alpha, row_scale, output-row mapping, residual and beta.  vec: 16-byte path allowed.
template <int W>
__device__ __forceinline__ void store_chunk(const Epilogue& e, int g, int m, int n, int N, float* v, bool vec) {
  const float rs = e.row_scale ? e.row_scale[m] : 1.0f;
  int64_t orow = m + (int64_t)g * e.c_growstride;
  if (e.c_ilv) orow = ilv_row(orow, e.c_ilv);
  if (e.c_rows) orow = e.c_rows[orow];
  const int nv = N - n < W ? N - n : W;
#pragma unroll
  for (int t = 0; t < W; ++t) v[t] *= e.alpha * rs;
  if (e.resid) {
    const float* rp = e.resid + orow * e.ld_resid + n;
    if (vec && nv == W) {
#pragma unroll
      for (int t = 0; t < W; t += 4) {
        const float4 x = *reinterpret_cast<const float4*>(rp + t);
        v[t] += x.x; v[t + 1] += x.y; v[t + 2] += x.z; v[t + 3] += x.w;
      }
    } else {
      for (int t = 0; t < nv; ++t) v[t] += rp[t];
    }
  }
  // W-column chunks start at multiples of W and never cross a 32-column run of the interleave
  const int64_t ocol = e.c_col_ilv ? ilv_row((int64_t)g * e.c_gstride + n, e.c_col_ilv) : (int64_t)g * e.c_gstride + n;
  if (e.c_f32) {
    float* cp = reinterpret_cast<float*>(e.c) + orow * e.ldc + ocol;
    if (vec && nv == W) {
#pragma unroll
      for (int t = 0; t < W; t += 4) {
        if (e.beta != 0.0f) {
          const float4 o = *reinterpret_cast<const float4*>(cp + t);
          v[t] += e.beta * o.x; v[t + 1] += e.beta * o.y; v[t + 2] += e.beta * o.z; v[t + 3] += e.beta * o.w;
        }
        *reinterpret_cast<float4*>(cp + t) = make_float4(v[t], v[t + 1], v[t + 2], v[t + 3]);
      }
    } else {
      for (int t = 0; t < nv; ++t) cp[t] = v[t] + (e.beta != 0.0f ? e.beta * cp[t] : 0.0f);
    }
  } else {
    bf16* cp = reinterpret_cast<bf16*>(e.c) + orow * e.ldc + ocol;
    if (vec && nv == W && W == 8) {
      if (e.beta != 0.0f) {
        const uint4 o = *reinterpret_cast<const uint4*>(cp);
        const uint32_t ow[4] = {o.x, o.y, o.z, o.w};
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          v[2 * t] += e.beta * __uint_as_float(ow[t] << 16);
          v[2 * t + 1] += e.beta * __uint_as_float(ow[t] & 0xffff0000u);
        }
      }
      uint4 o;
      o.x = pack_bf2(v[0], v[1]);
      o.y = pack_bf2(v[2], v[3]);
      o.z = pack_bf2(v[4], v[5]);
      o.w = pack_bf2(v[6], v[7]);
      *reinterpret_cast<uint4*>(cp) = o;
    } else {
      for (int t = 0; t < nv; ++t) cp[t] = f2bf(v[t] + (e.beta != 0.0f ? e.beta * bf2f(cp[t]) : 0.0f));
    }
  }
}

struct EpiFlags {
  int vec;  // 16-byte stores / residual loads are aligned
};

// Direct-to-LDS stage layout: a tile row holds BK k values = CPR chunks of 16 bytes, chunk c
// stored at position c ^ swz(row), so that 32 lanes reading the same logical chunk of 32
// consecutive rows (the MFMA operand reads) spread over all LDS banks.  Both swizzles were
// chosen by measurement (SQ_LDS_BANK_CONFLICT of ds_read_b128 patterns on gfx950: zero
// conflicts for these two, conflicts for the unswizzled rows and for (row & 7), (row >> 1) & 3).
template <int CPR>
__device__ __forceinline__ int dl_swz(int row) {
  if constexpr (CPR == 8) return (row ^ (row >> 3)) & 7;  // 128-byte rows
  else return (row >> 2) & 3;                             // 64-byte rows
}

// 16 bytes per lane from global memory straight into LDS at (LDS base + 16 * lane); the LDS
// base must be wave-uniform.  The host pass of the compiler has no such builtin and never
// runs kernel bodies, so it only sees the declaration.
__device__ __forceinline__ void lds_dma16(const void* src, void* lds_base) {
#if defined(__HIP_DEVICE_COMPILE__)
  __builtin_amdgcn_global_load_lds(src, lds_base, 16, 0, 0);
#else
  (void)src;
  (void)lds_base;
#endif
}

// The same through a buffer descriptor (raw, `bytes` long; loads past the end are refused by the
// hardware): the k advance is one scalar added to per-lane byte offsets, and the compiler tracks
// the load by vmcnt alone (a global_load_lds also counts as a pending flat access, which turns
// every later LDS wait into a wait for all).
#if defined(__HIP_DEVICE_COMPILE__)
typedef __amdgpu_buffer_rsrc_t BufferRsrc;
#else
typedef int BufferRsrc;
#endif
__device__ __forceinline__ BufferRsrc buffer_rsrc(const void* base, uint32_t bytes) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, bytes, 0x00020000);
#else
  (void)base;
  (void)bytes;
  return 0;
#endif
}
__device__ __forceinline__ void lds_dma16_buf(BufferRsrc r, void* lds_base, uint32_t voff, int soff) {
#if defined(__HIP_DEVICE_COMPILE__)
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)lds_base, 16, voff, soff, 0, 0);
#else
  (void)r;
  (void)lds_base;
  (void)voff;
  (void)soff;
#endif
}

// Four bf16 of a k-major LDS tile, transposed across the 16 lanes of each lane group
// (ds_read_b64_tr_b16, gfx950).  Measured lane layout: within a group of 16 lanes, lane i
// receives element (i % 4) of the 8-byte rows that lanes 4j + i / 4 (j = 0..3) point at, in j
// order.  So if lane s of the group points at k-row (kb + s / 4) and columns (cb + 4 (s % 4))..+3,
// lane i gets column cb + i at k-rows kb..kb + 3: an MFMA operand fragment.
typedef short short4_v __attribute__((ext_vector_type(4)));

// 16 zero bytes in global memory: the source of direct loads past the end of a k range (a
// layout-T tile's rows beyond the group of a grouped-K problem), so LDS gets exact zeros.
__device__ __align__(16) unsigned int kDlZero[4] = {0u, 0u, 0u, 0u};  // never written
__device__ __forceinline__ short4_v lds_read_tr4(const unsigned char* lds_byte_ptr) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) short4_v*)lds_byte_ptr);
#else
  (void)lds_byte_ptr;
  return short4_v{0, 0, 0, 0};
#endif
}

// s_waitcnt with vmcnt <= n and the other counters unconstrained (gfx9 encoding).
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}

// The same with every LDS operation of the wave done (lgkmcnt 0).
template <int N>
__device__ __forceinline__ void wait_vmcnt_lgkm0() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4));
}

// Workgroup barrier without the waits of __syncthreads (loads into LDS may stay in flight); the
// caller waits for what the barrier has to cover.
__device__ __forceinline__ void wg_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

__device__ __forceinline__ bf16x8_v ld_frag16(const bf16* p) {
  return __builtin_bit_cast(bf16x8_v, *reinterpret_cast<const uint4*>(p));
}

__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

}  // namespace
}  // namespace rte
