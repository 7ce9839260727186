// bf16 MFMA products with a register-pipelined main loop (gfx950), fp32 accumulation: dense ones, the
// grouped SwiGLU products (GROUP_M) and the grouped weight gradients (GROUP_K); at the end of the file the
// products of grouped rows with a short-k weight (gemm_rows_kernel).
//
// One workgroup owns a BM x BN output tile; each of its WM x WN waves holds a (BM / WM) x
// (BN / WN) block in v_mfma_f32_32x32x16_bf16 accumulators.  K advances in tiles of BK through ST
// LDS stages filled through buffer descriptors (buffer_load_dwordx4 ... lds, no registers; loads past
// an operand's end come back as zeros), and the MFMA operands of the next 16-k step are read from LDS
// while the current step's products run, across tile boundaries too:
//
//   step (kt, last): wait until tile kt + 1 has landed; barrier; refill tile kt's stage with tile
//                    kt + ST; read the operands of (kt + 1, 0); products of (kt, last)
//
// so a barrier is passed with a whole step's products still to issue, and a load has ST - 1 tiles
// of products to arrive.
#include "gemm_dev.hpp"
#include "gemm_tile.hpp"

#include <type_traits>

namespace rte {

namespace {

// One operand: R tile rows (the output index) by BK k per stage.  Layout N (k contiguous): LDS
// rows are output rows of BK k, 16-byte chunk c at c ^ dl_swz(row).  Layout T (output index
// contiguous): LDS rows are k rows of R elements, chunk c at c ^ tswz(k), so the four k rows of a
// ds_read_b64_tr_b16 sit in distinct 64-byte windows of the 256 bytes the banks cover.
template <int R, int NT, int BK, bool T>
struct TileOperand {
  static constexpr int ROWB = T ? R * 2 : BK * 2;
  static constexpr int CPR = ROWB / 16;
  static constexpr int BYTES = R * BK * 2;
  static constexpr int INS = BYTES / 16 / NT;
  static_assert(INS >= 1 && BYTES == INS * 16 * NT, "whole 16-byte loads per thread");
  static_assert(!T || CPR >= 8, "layout-T tiles hold at least 64 columns");

  uint32_t off[INS];  // byte offset of this thread's loads in the operand (under 2^31: host check)

  __device__ __forceinline__ static int tswz(int krow) { return CPR >= 16 ? (krow & 3) * 4 : ((krow >> 1) & 1) * 4; }
  __device__ __forceinline__ static int krow(int u, int tid) { return (u * NT + tid) / CPR; }

  // group: the operand's group (row and element shifts); rows_later: layout T, leave the k row out
  __device__ __forceinline__ void init(const Operand& o, int group, int i0, int ilim, int tid, bool rows_later) {
    const int64_t shift = (int64_t)group * o.growstride, base = (int64_t)group * o.gstride;
#pragma unroll
    for (int u = 0; u < INS; ++u) {
      const int q = u * NT + tid, row = q / CPR, pc = q % CPR;
      if constexpr (!T) {
        int i = i0 + row;
        if (i >= ilim) i = ilim - 1;  // rows past the end re-read the last one; never stored
        off[u] = (uint32_t)(base + row_off(o, i + shift) + (pc ^ dl_swz<CPR>(row)) * 8) * 2;
      } else {
        int i = i0 + (pc ^ tswz(row)) * 8;
        if (i + 8 > ilim) i = ilim - 8;  // layout-T extents are multiples of 8
        const int64_t krow = (o.ilv && row >= 32) ? (int64_t)(row - 32) + o.ilv : row;
        off[u] = (uint32_t)(base + (rows_later ? 0 : krow * o.ld) + i) * 2;
      }
    }
  }
  // byte offset of the tile starting at k0 (a multiple of BK past a multiple of 64)
  __device__ __forceinline__ static int advance(int ld, int ilv, int k0) {
    if constexpr (!T) return k0 * 2;
    return (ilv ? (k0 >> 6) * 32 + ((k0 >> 5) & 1) * ilv : k0) * ld * 2;
  }
  // LDS byte offset of this lane's part of 32-row block b at k-step ks
  __device__ __forceinline__ static int frag_off(int rb, int lane, int b, int ks) {
    if constexpr (!T) {
      const int r = rb + 32 * b + (lane & 31);
      return r * ROWB + (((ks * 2 + (lane >> 5)) ^ dl_swz<CPR>(r)) << 4);
    } else {
      const int g = lane >> 4, s = lane & 15;
      const int kr = 8 * (g >> 1) + (s >> 2);
      const int col = rb + 32 * b + 16 * (g & 1) + 4 * (s & 3);
      return (kr + 16 * ks) * ROWB + (((col >> 3) ^ tswz(kr)) << 4) + (col & 7) * 2;
    }
  }
  __device__ __forceinline__ static bf16x8_v frag(const unsigned char* at) {
    if constexpr (!T) {
      return *reinterpret_cast<const bf16x8_v*>(at);
    } else {
      const short4_v lo = lds_read_tr4(at);
      const short4_v hi = lds_read_tr4(at + 4 * ROWB);
      typedef short short8_v __attribute__((ext_vector_type(8)));
      return __builtin_bit_cast(bf16x8_v, (short8_v)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    }
  }
};

constexpr int kBand = 4;  // tile rows walked together (4, 8 and 16 are within 2% but for long-k layout T: 413, 427, 504 us)
constexpr int kPatchPitch = 68;  // floats per row of a wave's 32 x 64 output patch
constexpr int kPatchBytes = 32 * kPatchPitch * 4;

constexpr int kIdxRows = kTileGroupChunk;  // gathered rows of a grouped reduction held in LDS

template <int BM, int BN, int WM, int WN, int BK, int ST, int MODE>
constexpr int tile_wgs() {
  constexpr int by_lds = 163840 / (ST * (BM + BN) * BK * 2 + (MODE == MODE_GROUP_K ? kIdxRows * 4 : 0));
  constexpr int by_regs = ((BM / WM) * (BN / WN) >= 128 * 128 ? 4 : (BM / WM) * (BN / WN) >= 128 * 64 ? 8 : 16) / (WM * WN);
  return by_lds < by_regs ? by_lds : by_regs;
}

// Group and position of element x of the sequence that lists, group by group, ceil(rows / per) entries
// (at least `least`): {group or -1, index in the group, entries of the group}.  One wave looks at 64
// groups at a time.
__device__ __forceinline__ int3 tile_group(const int32_t* goff, int G, int per, int least, int x, int lane) {
  int base = 0;
  for (int c0 = 0; c0 < G; c0 += 64) {
    const int gg = c0 + lane;
    int cnt = 0;
    if (gg < G) {
      cnt = (goff[gg + 1] - goff[gg] + per - 1) / per;
      if (cnt < least) cnt = least;
    }
    int incl = cnt;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int y = __shfl_up(incl, o, 64);
      if (lane >= o) incl += y;
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

// SwiGLU backward of neurons n .. n + 7 of row m: v holds their dZ; up / gate values sit 32 columns
// apart.  Writes dUG, returns the neurons' part of <z, dZ>.
__device__ __forceinline__ float swiglu_bwd8(const Epilogue& e, int m, int n, const float* v) {
  const int64_t at = (int64_t)m * e.ld_ug + (int64_t)(n >> 5) * 64 + (n & 31);
  const uint4 uq = *reinterpret_cast<const uint4*>(e.ug_in + at);
  const uint4 gq = *reinterpret_cast<const uint4*>(e.ug_in + at + 32);
  const uint32_t uw[4] = {uq.x, uq.y, uq.z, uq.w}, gw[4] = {gq.x, gq.y, gq.z, gq.w};
  const float rs = e.row_scale ? e.row_scale[m] : 1.0f;
  uint32_t du[4], dg[4];
  float part = 0.0f;
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const float2 d2 = *reinterpret_cast<const float2*>(v + 2 * t);
    float a[2], b[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const float up = h ? __uint_as_float(uw[t] & 0xffff0000u) : __uint_as_float(uw[t] << 16);
      const float gt = h ? __uint_as_float(gw[t] & 0xffff0000u) : __uint_as_float(gw[t] << 16);
      const float draw = h ? d2.y : d2.x;
      const float s = sigmoidf_(gt), silu = gt * s, dz = draw * rs;
      a[h] = dz * silu;
      b[h] = dz * up * s * (1.0f + gt * (1.0f - s));
      part += up * silu * draw;
    }
    du[t] = pack_bf2(a[0], a[1]);
    dg[t] = pack_bf2(b[0], b[1]);
  }
  *reinterpret_cast<uint4*>(e.ug + at) = make_uint4(du[0], du[1], du[2], du[3]);
  *reinterpret_cast<uint4*>(e.ug + at + 32) = make_uint4(dg[0], dg[1], dg[2], dg[3]);
  return part;
}

template <int BM, int BN, int WM, int WN, int BK, int ST, bool AT, bool BT, int EPI, int MODE>
__global__ void __launch_bounds__(WM* WN * 64, (tile_wgs<BM, BN, WM, WN, BK, ST, MODE>() * WM * WN / 4))
    gemm_tile_kernel(GemmArgs p, int vec) {
  constexpr int NT = WM * WN * 64;
  constexpr int WTM = BM / WM, WTN = BN / WN, TM = WTM / 32, TN = WTN / 32, KS = BK / 16;
  static_assert(TN % 2 == 0, "output patches are 64 columns");
  static_assert(ST >= 2 && ST <= 4 && KS % 2 == 0, "stages and k-steps");
  using OpA = TileOperand<BM, NT, BK, AT>;
  using OpB = TileOperand<BN, NT, BK, BT>;
  constexpr int INS = OpA::INS + OpB::INS;
  constexpr int A_BYTES = OpA::BYTES, STAGE = OpA::BYTES + OpB::BYTES;
  constexpr int PPS = STAGE / kPatchBytes;  // output patches per stage
  static_assert(PPS * ST >= WM * WN, "the stages hold every wave's output patch");

  // One LDS array per stage, each addressed by name: the compiler then knows that the operand
  // reads of one stage do not touch the stages being filled and waits for no load it need not
  // (from one array, a ds_read_b64_tr_b16 waits for every load in flight).
  __shared__ __align__(16) unsigned char st0[STAGE], st1[STAGE], st2[ST > 2 ? STAGE : 16], st3[ST > 3 ? STAGE : 16];
  auto stage_of = [&](auto s) -> unsigned char* {
    constexpr int S = decltype(s)::value % ST;
    if constexpr (S == 0) return st0;
    else if constexpr (S == 1) return st1;
    else if constexpr (S == 2) return st2;
    else return st3;
  };
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WN, wn = wave % WN;

  const int gy = (p.N + BN - 1) / BN;
  int g = 0, m0, n0, mlim = p.M, kbeg = 0, kend = p.K;
  float* partial = nullptr;
  if constexpr (MODE == MODE_DENSE) {
    // Tile order: dispatch id d runs on XCD d % 8, so each XCD takes a contiguous run of tiles, and
    // a run walks kBand tile rows column by column: the tiles an XCD works on at one time share
    // few A and B panels of its L2.
    const int gx = (p.M + BM - 1) / BM, total = gx * gy;
    int lin = blockIdx.x;
    {
      const int q = total >> 3, r = total & 7, xcd = lin & 7;
      lin = xcd * q + (xcd < r ? xcd : r) + (lin >> 3);
    }
    const int bw = kBand * gy, bi = lin / bw;
    const int rows = gx - bi * kBand < kBand ? gx - bi * kBand : kBand;
    m0 = (bi * kBand + (lin - bi * bw) % rows) * BM;
    n0 = ((lin - bi * bw) / rows) * BN;
    if (p.splits > 1) {
      kbeg = blockIdx.y * p.k_chunk;
      kend = kbeg + p.k_chunk < p.K ? kbeg + p.k_chunk : p.K;
      partial = p.splitk_ws + (int64_t)blockIdx.y * p.M * p.N;
    }
  } else {
    // Grouped: of every 256 dispatch ids, an XCD takes 32 consecutive tiles, so the tiles of a group
    // meet in one L2.
    const int lin = (blockIdx.x & ~255) + (blockIdx.x & 7) * 32 + ((blockIdx.x & 255) >> 3);
    if constexpr (MODE == MODE_GROUP_M) {
      const int3 f = tile_group(p.goff, p.G, BM, 0, lin / gy, lane);
      g = f.x;
      if (g < 0) return;
      m0 = p.goff[g] + f.y * BM;
      n0 = (lin % gy) * BN;
      mlim = p.goff[g + 1];
    } else {
      const int per = (p.M + BM - 1) / BM * gy, item = lin / per, tile = lin - item * per;
      if (blockIdx.x == 0 && wave == 0) {  // the groups' first items, for the sum of the partials
        int base = 0;
        for (int c0 = 0; c0 < p.G; c0 += 64) {
          const int gg = c0 + lane;
          int cnt = 0;
          if (gg < p.G) {
            cnt = (p.goff[gg + 1] - p.goff[gg] + p.gk_chunk - 1) / p.gk_chunk;
            if (cnt < 1) cnt = 1;
          }
          int incl = cnt;
#pragma unroll
          for (int o = 1; o < 64; o <<= 1) {
            const int y = __shfl_up(incl, o, 64);
            if (lane >= o) incl += y;
          }
          if (gg < p.G) const_cast<int32_t*>(p.gk_first)[gg] = base + incl - cnt;
          base += __shfl(incl, 63, 64);
        }
        if (lane == 0) const_cast<int32_t*>(p.gk_first)[p.G] = base;
      }
      const int3 f = tile_group(p.goff, p.G, p.gk_chunk, 1, item, lane);
      g = f.x;
      if (g < 0) return;
      m0 = (tile / gy) * BM;
      n0 = (tile % gy) * BN;
      kbeg = p.goff[g] + f.y * p.gk_chunk;
      kend = kbeg + p.gk_chunk < p.goff[g + 1] ? kbeg + p.gk_chunk : p.goff[g + 1];
      if (f.z > 1) partial = p.gk_part + (int64_t)item * p.M * p.N;
    }
  }

  f32x16_v acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

  OpA la;
  OpB lb;
  // a grouped reduction's output rows and columns are shifted by the epilogue, its operands are not
  la.init(p.a, MODE == MODE_GROUP_M ? g : 0, m0, mlim, tid, MODE == MODE_GROUP_K);
  lb.init(p.b, MODE == MODE_GROUP_M ? g : 0, n0, p.N, tid, MODE == MODE_GROUP_K);
  const int alda = (int)p.a.ld, blda = (int)p.b.ld, ailv = p.a.ilv, bilv = p.b.ilv;
  const BufferRsrc ra = buffer_rsrc(p.a.ptr, p.a_bytes), rb = buffer_rsrc(p.b.ptr, p.b_bytes);

  // Grouped reductions gather the memory rows of one operand (or none): the range's indices sit in
  // LDS, and the rows of the next refill are looked up a tile ahead.
  __shared__ int s_idx[MODE == MODE_GROUP_K ? kIdxRows : 1];
  const bool a_gather = MODE == MODE_GROUP_K && p.a.rows, b_gather = MODE == MODE_GROUP_K && p.b.rows;
  const int klen = kend - kbeg;
  uint32_t ar[OpA::INS], br[OpB::INS];  // byte offsets of the next refill's rows (past the range: no row)
  auto look = [&](int kt) {
    if constexpr (MODE == MODE_GROUP_K) {
#pragma unroll
      for (int u = 0; u < OpA::INS; ++u) {
        const int k = kt * BK + OpA::krow(u, tid);
        const int row = a_gather ? s_idx[k < klen ? k : 0] : kbeg + k;
        ar[u] = k < klen ? (uint32_t)row * (uint32_t)alda * 2u + la.off[u] : 0x80000000u;
      }
#pragma unroll
      for (int u = 0; u < OpB::INS; ++u) {
        const int k = kt * BK + OpB::krow(u, tid);
        const int row = b_gather ? s_idx[k < klen ? k : 0] : kbeg + k;
        br[u] = k < klen ? (uint32_t)row * (uint32_t)blda * 2u + lb.off[u] : 0x80000000u;
      }
    }
  };
  if constexpr (MODE == MODE_GROUP_K) {
    const int32_t* rows = p.a.rows ? p.a.rows : p.b.rows;
    if (rows)
      for (int i = tid; i < klen; i += NT) s_idx[i] = rows[kbeg + i];
    if (klen <= 0 && tid == 0) s_idx[0] = 0;
    __syncthreads();
  }

  // A ragged dense reduction (both operands layout T) reads k rows past its end in its last tile:
  // they lie past the operands' buffer bounds, as the rows past a group's range are made to, and the
  // hardware turns them into zeros.
  auto issue = [&](unsigned char* st, int kt) {
    unsigned char* dst = st + wave * 1024;
    if constexpr (MODE == MODE_GROUP_K) {
#pragma unroll
      for (int u = 0; u < OpA::INS; ++u) lds_dma16_buf(ra, dst + u * NT * 16, ar[u], 0);
#pragma unroll
      for (int u = 0; u < OpB::INS; ++u) lds_dma16_buf(rb, dst + A_BYTES + u * NT * 16, br[u], 0);
    } else {
      const int k0 = kbeg + kt * BK;
      const int ao = OpA::advance(alda, ailv, k0), bo = OpB::advance(blda, bilv, k0);
#pragma unroll
      for (int u = 0; u < OpA::INS; ++u) lds_dma16_buf(ra, dst + u * NT * 16, la.off[u], ao);
#pragma unroll
      for (int u = 0; u < OpB::INS; ++u) lds_dma16_buf(rb, dst + A_BYTES + u * NT * 16, lb.off[u], bo);
    }
  };

  int aof[TM], bof[TN];
#pragma unroll
  for (int i = 0; i < TM; ++i) aof[i] = OpA::frag_off(wm * WTM, lane, i, 0);
#pragma unroll
  for (int j = 0; j < TN; ++j) bof[j] = OpB::frag_off(wn * WTN, lane, j, 0);
  // layout N: k-step ks of a row sits at chunk (2 ks + half) ^ swz, i.e. the offset XOR 32 ks;
  // layout T: 16 k rows further
  auto at_step = [&](int off, int ks, bool t, int rowb) { return t ? off + ks * 16 * rowb : off ^ (ks * 32); };

  bf16x8_v af[2][TM], bfr[2][TN];
  auto read = [&](auto set, const unsigned char* st, int ks) {
    constexpr int S = decltype(set)::value;
#pragma unroll
    for (int j = 0; j < TN; ++j) bfr[S][j] = OpB::frag(st + A_BYTES + at_step(bof[j], ks, BT, OpB::ROWB));
#pragma unroll
    for (int i = 0; i < TM; ++i) af[S][i] = OpA::frag(st + at_step(aof[i], ks, AT, OpA::ROWB));
  };
  auto mul = [&](auto set) {
    constexpr int S = decltype(set)::value;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[S][i], bfr[S][j], acc[i][j], 0, 0, 0);
  };
  using S0 = std::integral_constant<int, 0>;
  using S1 = std::integral_constant<int, 1>;

  // Tile kt sits in stage (kt + off) % ST, with off so that the last round ends at stage ST - 1:
  // a first round of ST - off tiles, full rounds, and a last one that fetches nothing.  The host
  // gives every dense k range at least ST tiles.
  int nk = (kend - kbeg + BK - 1) / BK;
  if (MODE == MODE_GROUP_K && nk < ST) nk = ST;  // few rows: the missing ones read zeros
  const int rounds = (nk + ST - 1) / ST, off = rounds * ST - nk;

  // One operand read after each product: the LDS and the matrix cores work at the same time.
  auto interleave = [&] {
    constexpr int READS = (AT ? 2 : 1) * TM + (BT ? 2 : 1) * TN, MULS = TM * TN;
    constexpr int PER = (READS + MULS - 1) / MULS;
#pragma unroll
    for (int m = 0; m < MULS; ++m) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, PER, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
  };

  // Products of the tile in stage S; then the next tile: wait for it (YOUNGER tiles' loads may
  // still be in flight), refill this stage with tile `refill`, read its first operands.
  auto step = [&](auto s, auto younger, auto more, int refill) {
    constexpr int S = decltype(s)::value;
    const unsigned char* st = stage_of(s);
    if constexpr (decltype(more)::value) look(refill);
#pragma unroll
    for (int ks = 0; ks < KS - 1; ++ks) {
      if ((ks & 1) == 0) {
        read(S1{}, st, ks + 1);
        mul(S0{});
      } else {
        read(S0{}, st, ks + 1);
        mul(S1{});
      }
      interleave();
    }
    if constexpr (decltype(younger)::value >= 0) {
      wait_vmcnt_lgkm0<decltype(younger)::value * INS>();
      wg_barrier();
      if constexpr (decltype(more)::value) issue(stage_of(s), refill);
      read(S0{}, stage_of(std::integral_constant<int, (S + 1) % ST>{}), 0);
    }
    mul(S1{});
    interleave();
  };
  auto each_stage = [&](auto f) {
    f(std::integral_constant<int, 0>{});
    f(std::integral_constant<int, 1>{});
    if constexpr (ST > 2) f(std::integral_constant<int, 2>{});
    if constexpr (ST > 3) f(std::integral_constant<int, 3>{});
  };
  using Young = std::integral_constant<int, ST - 2>;

  each_stage([&](auto s) {
    const int t = decltype(s)::value - off;
    look(t < 0 ? t + ST : t);
    issue(stage_of(s), t < 0 ? t + ST : t);
  });
  if (off == 0) wait_vmcnt_lgkm0<(ST - 1) * INS>();  // tile 0 came first
  else wait_vmcnt_lgkm0<0>();
  wg_barrier();
  each_stage([&](auto s) {
    if (decltype(s)::value == off) read(S0{}, stage_of(s), 0);
  });
  int kt = -off;  // the tile of stage 0 in the current round
  if (off > 0) {
    each_stage([&](auto s) {
      if (decltype(s)::value >= off) step(s, Young{}, std::true_type{}, kt + decltype(s)::value + ST);
    });
    kt += ST;
  }
  for (; kt + ST < nk; kt += ST)
    each_stage([&](auto s) { step(s, Young{}, std::true_type{}, kt + decltype(s)::value + ST); });
  each_stage([&](auto s) {
    step(s, std::integral_constant<int, ST - 2 - decltype(s)::value>{}, std::false_type{}, 0);
  });
  __syncthreads();  // the output patches reuse the stages

  // ---------------------------------------------------------------- output: 32 x 64 wave patches
  const Epilogue& e = p.epi;
  unsigned char* pst = wave < PPS ? st0 : (wave < 2 * PPS ? st1 : (wave < 3 * PPS ? st2 : st3));
  float* pt = reinterpret_cast<float*>(pst + (wave % PPS) * kPatchBytes);
  const int half = lane >> 5, l32 = lane & 31;
#pragma unroll
  for (int jp = 0; jp < TN / 2; ++jp) {
    const int nb = n0 + wn * WTN + jp * 64;
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int mb = m0 + wm * WTM + i * 32;
      wave_lds_fence();
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          pt[(8 * (r >> 2) + 4 * half + (r & 3)) * kPatchPitch + j * 32 + l32] = acc[i][jp * 2 + j][r];
      wave_lds_fence();
      if constexpr (EPI == EPI_STORE) {
        if (partial || e.c_f32) {
          const int cc = (lane & 15) * 4, n = nb + cc;
#pragma unroll
          for (int u = 0; u < 8; ++u) {
            const int row = u * 4 + (lane >> 4), m = mb + row;
            if (m >= mlim || n >= p.N) continue;
            const float4 x = *reinterpret_cast<const float4*>(pt + row * kPatchPitch + cc);
            if (partial) {
              float* dst = partial + (int64_t)m * p.N + n;
              if (vec && n + 4 <= p.N) {
                *reinterpret_cast<float4*>(dst) = x;
              } else {
                const float v[4] = {x.x, x.y, x.z, x.w};
                for (int t = 0; t < 4 && n + t < p.N; ++t) dst[t] = v[t];
              }
            } else {
              float v[4] = {x.x, x.y, x.z, x.w};
              store_chunk<4>(e, g, m, n, p.N, v, vec);
            }
          }
          continue;
        }
      }
      const int cc = (lane & 7) * 8;
      if constexpr (EPI == EPI_SWIGLU_FWD) {
        // patch columns 0..31 are the up values, 32..63 the gates of the same neurons
        const int c8 = (lane & 3) * 8;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const int row = u * 16 + (lane >> 2), m = mb + row;
          if (m >= mlim || nb >= p.N) continue;
          const float* src = pt + row * kPatchPitch + c8;
          const float rs = e.row_scale ? e.row_scale[m] : 1.0f;
          uint32_t uw[4], gw[4], zw[4];
#pragma unroll
          for (int t = 0; t < 4; ++t) {
            const float2 a = *reinterpret_cast<const float2*>(src + 2 * t);
            const float2 b = *reinterpret_cast<const float2*>(src + 32 + 2 * t);
            uw[t] = pack_bf2(a.x, a.y);
            gw[t] = pack_bf2(b.x, b.y);
            const float u0 = __uint_as_float(uw[t] << 16), u1 = __uint_as_float(uw[t] & 0xffff0000u);
            const float g0 = __uint_as_float(gw[t] << 16), g1 = __uint_as_float(gw[t] & 0xffff0000u);
            zw[t] = pack_bf2(u0 * g0 * sigmoidf_(g0) * rs, u1 * g1 * sigmoidf_(g1) * rs);
          }
          bf16* up = e.ug + (int64_t)m * e.ld_ug + nb + c8;
          *reinterpret_cast<uint4*>(up) = make_uint4(uw[0], uw[1], uw[2], uw[3]);
          *reinterpret_cast<uint4*>(up + 32) = make_uint4(gw[0], gw[1], gw[2], gw[3]);
          *reinterpret_cast<uint4*>(e.z + (int64_t)m * e.ld_z + nb / 2 + c8) = make_uint4(zw[0], zw[1], zw[2], zw[3]);
        }
      } else {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int row = u * 8 + (lane >> 3), m = mb + row, n = nb + cc;
          if constexpr (EPI == EPI_SWIGLU_BWD && MODE == MODE_GROUP_M) {
            // <z, dZ> of the row (the pair weight's gradient): all of its neurons are in this patch
            float part = 0.0f;
            const bool here = m < mlim && n < p.N;
            if (here) part = swiglu_bwd8(e, m, n, pt + row * kPatchPitch + cc);
#pragma unroll
            for (int o = 1; o <= 4; o <<= 1) part += __shfl_xor(part, o, 64);
            if (e.dw_row && m < mlim && (lane & 7) == 0) e.dw_row[m] = part;
            continue;
          }
          if (m >= mlim || n >= p.N) continue;
          if constexpr (EPI == EPI_SWIGLU_BWD && MODE != MODE_GROUP_M) {
            swiglu_bwd8(e, m, n, pt + row * kPatchPitch + cc);
            continue;
          }
          const float4 x = *reinterpret_cast<const float4*>(pt + row * kPatchPitch + cc);
          const float4 y = *reinterpret_cast<const float4*>(pt + row * kPatchPitch + cc + 4);
          float v[8] = {x.x, x.y, x.z, x.w, y.x, y.y, y.z, y.w};
          if constexpr (EPI == EPI_STORE) {
            store_chunk<8>(e, g, m, n, p.N, v, vec);
          } else if constexpr (EPI == EPI_ROPE_QKV) {  // 8 columns of one head; RoPE pairs (2i, 2i + 1)
            const int part = n / e.dmodel, within = n - part * e.dmodel;
            const int hh = within / e.hd, dim = within - hh * e.hd;
            const int b = m / e.S, s = m - b * e.S;
            if (part < 2) {
              const float* cp = e.cos_t + (int64_t)s * e.hd + dim;
              const float* sp = e.sin_t + (int64_t)s * e.hd + dim;
#pragma unroll
              for (int t = 0; t < 4; ++t) {
                const float2 c = *reinterpret_cast<const float2*>(cp + 2 * t);
                const float2 sn = *reinterpret_cast<const float2*>(sp + 2 * t);
                const float xe = v[2 * t], xo = v[2 * t + 1];
                v[2 * t] = xe * c.x - xo * sn.x;
                v[2 * t + 1] = xo * c.y + xe * sn.y;
              }
            }
            bf16* dst = part == 0 ? e.q : (part == 1 ? e.k : e.v);
            *reinterpret_cast<uint4*>(dst + (((int64_t)b * e.H + hh) * e.S + s) * e.hd + dim) =
                make_uint4(pack_bf2(v[0], v[1]), pack_bf2(v[2], v[3]), pack_bf2(v[4], v[5]), pack_bf2(v[6], v[7]));
          }
        }
      }
    }
  }
}

template <int BM, int BN, int WM, int WN, int BK, int ST, bool AT, bool BT, int EPI, int MODE = MODE_DENSE>
int launch(const GemmArgs& p, hipStream_t stream, int vec) {
  auto fn = gemm_tile_kernel<BM, BN, WM, WN, BK, ST, AT, BT, EPI, MODE>;
  const int64_t gx = (p.M + BM - 1) / BM, gy = (p.N + BN - 1) / BN;
  int64_t tiles = gx * gy;
  if (MODE == MODE_GROUP_M) tiles = p.max_tiles_m * gy;
  if (MODE == MODE_GROUP_K) tiles *= ((int64_t)p.K + p.gk_chunk - 1) / p.gk_chunk + p.G;
  if (MODE != MODE_DENSE) tiles = (tiles + 255) / 256 * 256;
  RTE_REQUIRE(tiles < ((int64_t)1 << 31), "gemm: too many tiles");
  hipLaunchKernelGGL(fn, dim3((unsigned)tiles, (unsigned)(p.splits > 1 ? p.splits : 1)), dim3(WM * WN * 64), 0, stream,
                     p, vec);
  return check_launch("gemm_tile");
}

template <int BM, int BN, int WM, int WN, int BK, int ST, int EPI>
int layouts(const GemmArgs& p, hipStream_t stream, int vec) {
  if (!p.a_t && !p.b_t) return launch<BM, BN, WM, WN, BK, ST, false, false, EPI>(p, stream, vec);
  if constexpr (EPI == EPI_STORE || EPI == EPI_SWIGLU_BWD) {
    if (!p.a_t) return launch<BM, BN, WM, WN, BK, ST, false, true, EPI>(p, stream, vec);
  }
  if constexpr (EPI == EPI_STORE) {
    if (p.b_t) return launch<BM, BN, WM, WN, BK, ST, true, true, EPI>(p, stream, vec);
  }
  set_error("gemm_tile: operand layouts not taken by this epilogue");
  return -1;
}


// Tile and split choice: the estimated time of each (tile, splits) pair, in us.  A 256x256 tile alone on
// its CU takes 0.0235 us per k; a 128x128 tile 0.0144 with two on its CU, 0.0107 alone and 0.0088 with most
// of the chip idle (both operands layout T, half as much k per stage: 0.0275, 0.0179, 0.0111 and 0.0099); a
// round of workgroups 4 us (256) or 2.7 us besides (first loads, output); the launch that adds the partials
// 3.85, 0.07 for each of them, and their bytes at 1.78 TB/s.  Fitted to 10611 measured (layouts, M, N, K,
// tile, splits), M and N 65 to 32768, K 256 to 32768: the pick of 1246 shapes takes 0.6% more than their
// best pair on average and 19% at most (8192 x 128 x 2048: 24.1 us, 20.2 in 3 splits).  The estimate before
// set that launch at 6 us, counted bytes alone, split from 256 k and went 29% wrong (weight gradients of
// 200 x 512 x 1024: 12.7 us unsplit, 10.1 in 8; 6000 x 3072 x 256 31 us in large tiles, 24 in small ones;
// 512 x 128 x 8192 16.0 us in 32 splits, 13.7 in 16).  Large tiles where the grid fills the chip (16384 x
// 3072 x 1024: 104 us against 118), small ones where it does not (8192 x 512 x 4096: 46 against 81).
struct TilePick {
  int tile, splits;
  double us;
};

TilePick pick_tile(int M, int N, int K, bool a_t, int lo, int hi) {
  TilePick best{128, 1, 1e30};
  for (int tile : {256, 128}) {
    const int64_t tiles = (int64_t)((M + tile - 1) / tile) * ((N + tile - 1) / tile);
    const int64_t slots = tile == 256 ? 256 : 512;
    for (int s = lo; s <= hi; ++s) {
      const int kc = ((K + s - 1) / s + 63) / 64 * 64;
      if (s > 1 && (kc < kTileMinK || (K + kc - 1) / kc != s || K - (s - 1) * kc < kTileMinK)) continue;
      if (tiles * s > 2 * slots && s > lo) break;  // two rounds of splits never pay
      const int64_t wgs = tiles * s, rounds = (wgs + slots - 1) / slots;
      const double per_k = tile == 256  ? (a_t ? 0.0275 : 0.0235)
                           : wgs <= 64  ? (a_t ? 0.0099 : 0.0088)
                           : wgs <= 256 ? (a_t ? 0.0111 : 0.0107)
                                        : (a_t ? 0.0179 : 0.0144);
      const double round = per_k * (s > 1 ? kc : K) + (tile == 256 ? 4.0 : 2.7);
      const double us = rounds * round + (s > 1 ? 3.85 + s * (0.07 + 4.0 * M * N / 1.78e6) : 0.0);
      if (us < best.us) best = {tile, s, us};
    }
  }
  return best;
}

// Rows of activations: the number of splits sets the order of an element's sum, so it is chosen for
// the power of two nearest to M (a bucket of rows: from 1 / 1.4142 to 1.4142 times it).
int row_bucket(int M) {
  int m2 = 64;
  while (m2 < (1 << 30) && (double)M > 1.4142 * m2) m2 *= 2;
  return m2;
}

// Splits of a product with room for its partials, by the shape alone: the same call gives the same
// bits whatever ran before it, and so do a sample's rows beside others of their bucket.
int tile_splits(int M, int N, int K, bool a_t) {
  if (a_t) return pick_tile(M, N, K, true, 1, kTileMaxSplits).splits;
  return K > kTileRowK ? pick_tile(row_bucket(M), N, K, false, 1, kTileMaxSplits).splits : 1;
}

template <int EPI>
int launch_tile(const GemmArgs& p, hipStream_t stream, int vec, int tile) {
  if (tile == 256) return layouts<256, 256, 2, 4, 64, 2, EPI>(p, stream, vec);
  // both operands layout T: rows are long whatever BK is, four short stages hide more latency
  // (512 x 2048 x 8192 in 4 splits: 31 us against 33); layout N wants whole 128-byte lines per row
  // (8192 x 2048 x 8192: 258 us against 316)
  if constexpr (EPI == EPI_STORE) {
    if (p.a_t) return launch<128, 128, 2, 2, 32, 4, true, true, EPI>(p, stream, vec);
  }
  return layouts<128, 128, 2, 2, 64, 2, EPI>(p, stream, vec);
}

// Grouped rows times a short-k weight (the pools' output and input-gradient pairs): C[row] = A[row] B_g
// for K = 64 KT, bf16 out, rows optionally scattered.  Bound by writing C (N values per row against K
// read).  A workgroup keeps 256 columns of one group's weight in LDS and its four waves stream
// `chunk` rows past it, 32 at a time, with the next rows on their way: no load, barrier or wait of one
// block of rows stands in front of the next one's stores.  With a tile of 128 x 128 per workgroup each
// tile paid a load and a store latency in turn (262144 rows of 1024 columns, 537 MB written: K 64 240 us
// and now 134, K 128 324 us and now 181).  The weight is the product's row operand, so a lane holds one row's
// columns in fours and 64 columns of 32 rows leave through a 4 KB patch in whole 128-byte lines.
constexpr int kRowsCols = 256;
template <int KT, bool BT>
__global__ void __launch_bounds__(256, KT == 1 ? 3 : 2) gemm_rows_kernel(GemmArgs p, int chunk) {
  using OpB = TileOperand<kRowsCols, 256, 64, BT>;
  __shared__ __align__(16) unsigned char slab[KT * OpB::BYTES];
  __shared__ __align__(16) unsigned char patches[4 * 4096];
  const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int gy = (p.N + kRowsCols - 1) / kRowsCols;
  const int lin = (blockIdx.x & ~255) + (blockIdx.x & 7) * 32 + ((blockIdx.x & 255) >> 3);  // as the tiles
  const int3 f = tile_group(p.goff, p.G, chunk, 0, lin / gy, lane);
  const int g = f.x;
  if (g < 0) return;
  const int n0 = (lin % gy) * kRowsCols;
  const int mbeg = p.goff[g] + f.y * chunk;
  const int mend = mbeg + chunk < p.goff[g + 1] ? mbeg + chunk : p.goff[g + 1];

  // layout T leaves the group's k rows (whole interleave periods of 64) to the descriptor
  const int64_t shift = BT ? (int64_t)g * (p.b.ilv ? p.b.growstride / 2 : p.b.growstride) * p.b.ld : 0;
  OpB lb;
  lb.init(p.b, g, n0, p.N, tid, false);
  const BufferRsrc rb = buffer_rsrc(p.b.ptr + shift, p.b_bytes - (uint32_t)(shift * 2));
#pragma unroll
  for (int kt = 0; kt < KT; ++kt) {
    const int bo = OpB::advance((int)p.b.ld, p.b.ilv, kt * 64);
#pragma unroll
    for (int u = 0; u < OpB::INS; ++u)
      lds_dma16_buf(rb, slab + kt * OpB::BYTES + wave * 1024 + u * 4096, lb.off[u], bo);
  }
  int bof[kRowsCols / 32];
#pragma unroll
  for (int j = 0; j < kRowsCols / 32; ++j) bof[j] = OpB::frag_off(0, lane, j, 0);

  bf16x8_v x[KT * 4];
  auto rows_of = [&](int m) {  // rows past the chunk repeat its last one and are not stored
    const int r = m + l32 < mend ? m + l32 : mend - 1;
    const bf16* a = p.a.ptr + (int64_t)r * p.a.ld + 8 * h;
#pragma unroll
    for (int k = 0; k < KT * 4; ++k) x[k] = ld_frag16(a + 16 * k);
  };
  int m = mbeg + wave * 32;
  if (m < mend) rows_of(m);
  wait_vmcnt_lgkm0<0>();
  wg_barrier();  // the slab is in LDS

  unsigned char* patch = patches + wave * 4096;
  bf16* c = static_cast<bf16*>(p.epi.c);
  for (; m < mend; m += 128) {
    bf16x8_v cur[KT * 4];
#pragma unroll
    for (int k = 0; k < KT * 4; ++k) cur[k] = x[k];
    int64_t at[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = m + i * 8 + (lane >> 3);
      at[i] = r < mend ? (int64_t)(p.epi.c_rows ? p.epi.c_rows[r] : r) * p.epi.ldc : -1;
    }
    if (m + 128 < mend) rows_of(m + 128);
#pragma unroll
    for (int j = 0; j < kRowsCols / 64; ++j) {
      if (n0 + j * 64 >= p.N) break;
      f32x16_v acc[2];
#pragma unroll
      for (int e = 0; e < 2; ++e)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[e][r] = 0.0f;
#pragma unroll
      for (int k = 0; k < KT * 4; ++k)
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          const int off = bof[2 * j + e];
          const unsigned char* w = slab + (k >> 2) * OpB::BYTES + (BT ? off + (k & 3) * 16 * OpB::ROWB : off ^ ((k & 3) * 32));
          acc[e] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(OpB::frag(w), cur[k], acc[e], 0, 0, 0);
        }
#pragma unroll
      for (int e = 0; e < 2; ++e)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          *reinterpret_cast<uint2*>(patch + l32 * 128 + (((4 * e + q) ^ (l32 & 7)) << 4) + h * 8) =
              make_uint2(pack_bf2(acc[e][4 * q], acc[e][4 * q + 1]), pack_bf2(acc[e][4 * q + 2], acc[e][4 * q + 3]));
      wave_lds_fence();
      const int ch = lane & 7, col = n0 + j * 64 + ch * 8;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int r = i * 8 + (lane >> 3);
        const uint4 v = *reinterpret_cast<const uint4*>(patch + r * 128 + ((ch ^ (r & 7)) << 4));
        if (at[i] >= 0 && col < p.N) *reinterpret_cast<uint4*>(c + at[i] + col) = v;
      }
      wave_lds_fence();
    }
  }
}

int launch_rows(const GemmArgs& p, hipStream_t stream) {
  // rows per workgroup: 512 unless that leaves fewer than four workgroups per CU
  const int gy = (p.N + kRowsCols - 1) / kRowsCols;
  int chunk = 512;
  while (chunk > 128 && (int64_t)p.M / chunk * gy < 1024) chunk /= 2;
  const int64_t items = ((int64_t)p.M / chunk + p.G) * gy;
  const int64_t grid = (items + 255) / 256 * 256;
  RTE_REQUIRE(grid < ((int64_t)1 << 31), "gemm: too many row chunks");
  if (p.K == 64)
    hipLaunchKernelGGL((p.b_t ? gemm_rows_kernel<1, true> : gemm_rows_kernel<1, false>), dim3((unsigned)grid), dim3(256),
                       0, stream, p, chunk);
  else
    hipLaunchKernelGGL((p.b_t ? gemm_rows_kernel<2, true> : gemm_rows_kernel<2, false>), dim3((unsigned)grid), dim3(256),
                       0, stream, p, chunk);
  return check_launch("gemm_rows");
}

}  // namespace

int gemm_tile_group_launch(const GemmArgs& p, int epi_kind, hipStream_t stream, int vec) {
  if (p.mode == MODE_GROUP_M) {
    if (epi_kind == EPI_STORE) return launch_rows(p, stream);
    if (epi_kind == EPI_SWIGLU_FWD)
      return launch<128, 128, 2, 2, 64, 2, false, false, EPI_SWIGLU_FWD, MODE_GROUP_M>(p, stream, vec);
    return launch<128, 64, 4, 1, 64, 2, false, true, EPI_SWIGLU_BWD, MODE_GROUP_M>(p, stream, vec);
  }
  if (p.M <= 64) return launch<64, 128, 2, 2, 32, 4, true, true, EPI_STORE, MODE_GROUP_K>(p, stream, vec);
  if (p.N <= 64) return launch<128, 64, 4, 1, 32, 4, true, true, EPI_STORE, MODE_GROUP_K>(p, stream, vec);
  return launch<128, 128, 2, 2, 32, 4, true, true, EPI_STORE, MODE_GROUP_K>(p, stream, vec);
}

size_t gemm_tile_split_bytes(int M, int N, int K) {
  if (M <= 0 || N <= 0 || K < 2 * kTileMinK) return 0;
  const int wgrad = tile_splits(M, N, K, true), rows = tile_splits(M, N, K, false);
  const int most = wgrad > rows ? wgrad : rows;
  return most > 1 ? (size_t)most * M * N * sizeof(float) : 0;
}

int gemm_tile_launch(const GemmArgs& p0, int epi_kind, hipStream_t stream, int vec, void* ws, size_t ws_bytes,
                     int* splits) {
  GemmArgs p = p0;
  p.splits = epi_kind == EPI_STORE && ws ? tile_splits(p.M, p.N, p.K, p.a_t) : 1;
  if ((size_t)p.splits * p.M * p.N * sizeof(float) > ws_bytes) p.splits = 1;
  const int tile = pick_tile(p.M, p.N, p.K, p.a_t, p.splits, p.splits).tile;
  if (p.splits > 1) {
    p.k_chunk = ((p.K + p.splits - 1) / p.splits + 63) / 64 * 64;
    p.splitk_ws = static_cast<float*>(ws);
  }
  *splits = p.splits;
  switch (epi_kind) {
    case EPI_STORE: return launch_tile<EPI_STORE>(p, stream, vec, tile);
    case EPI_SWIGLU_FWD: return launch_tile<EPI_SWIGLU_FWD>(p, stream, vec, tile);
    case EPI_SWIGLU_BWD: return launch_tile<EPI_SWIGLU_BWD>(p, stream, vec, tile);
    default: return launch_tile<EPI_ROPE_QKV>(p, stream, vec, tile);
  }
}

}  // namespace rte
