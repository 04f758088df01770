#pragma once
// The fused encoder's smaller tiles, for problems that 256x256 tiles cannot spread over the
// chip: few tokens (where the call is one pass over W_enc and latency decides), ragged or
// middling shapes whose 256x256 tiles fill the CUs unevenly, and row-contiguous W_enc whose rows
// are not 16-B aligned (an odd d_sae). Same x' workspace, MFMA instruction, operand order and
// accumulation order per output as gemm_kernel (encode_kernels.h), so results are bit-identical
// to it; only the tile, the pipeline and the epilogue's staging differ.
#include "encode_kernels.h"

namespace sfenc {

// How a slim tile's W arrives: the two DMA paths of the 256x256 kernels, or through registers
// for rows that are contiguous along features / along d_in at any alignment.
enum SlimW { S_NMAJOR = 0, S_KMAJOR = 1, S_NROWS = 2, S_KROWS = 3 };

// A tile: WM x WN waves of (32 MB tokens x 32 NB features), K-steps of KC 16-B chunks per x'
// row, NS stage buffers.
template <int MB_, int NB_, int WM_, int WN_, int KC_, int NS_>
struct SlimTile {
  static constexpr int MB = MB_, NB = NB_, WM = WM_, WN = WN_, KC = KC_, NS = NS_;
  static constexpr int NW = WM * WN, NT = 64 * NW;
  static constexpr int TM = 32 * MB * WM, TN = 32 * NB * WN;
  static constexpr int WT = TN * KC * 16, XT = TM * KC * 16, ST = WT + XT;  // stage bytes
  static constexpr int PW = WT / 16 / NT, PX = XT / 16 / NT;                // chunks per thread
  static_assert(PW * 16 * NT == WT && PX * 16 * NT == XT, "whole DMAs per thread");
};
// What bounds them: up to a few hundred tokens the pass over W (the stages in flight times the
// latency of HBM), so the panels are narrow enough to give every CU one; above that the barrier and
// LDS latency of a K-step, which two workgroups per CU overlap (26-36% of the MFMA rate in 16 bits,
// 87-100% in fp32, against 69% / 95% of a 256x256 tile). Rates at each size beside pick_slim
// (encode.hip).
// Up to 32 tokens: two waves of 32 features each, 128-B W rows, five stages in flight and two
// workgroups per CU.
typedef SlimTile<1, 1, 1, 2, 8, 6> Slim32;
// 128 tokens: 4 waves of 64 x 32 over a 64-feature panel, or of 64 x 64 over 128 features.
typedef SlimTile<2, 1, 2, 2, 8, 3> Slim128;
typedef SlimTile<2, 2, 2, 2, 4, 4> Slim128w;
// 128-feature panels, and a 256-feature one for up to 160 tokens (256- and 512-B W rows).
typedef SlimTile<1, 1, 1, 4, 8, 3> Slim32w;
typedef SlimTile<2, 1, 1, 4, 8, 3> Slim64w;
typedef SlimTile<5, 2, 1, 4, 8, 3> Slim160x;
// Register-staged W: three stages.
typedef SlimTile<1, 1, 1, 2, 8, 3> Slim32r;
typedef SlimTile<2, 2, 2, 2, 4, 3> Slim128wr;

// dma16 with a cache policy: AUX_NT streams past L2, for a W that each launch reads once.
constexpr int AUX_NT = 2;
template <int AUX>
__device__ __forceinline__ void dma16_w(__amdgpu_buffer_rsrc_t r, char* wave_base, uint32_t voff, uint32_t soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void*)wave_base, 16, (int)voff, (int)soff, 0, AUX);
}

// s_waitcnt vmcnt(N) lgkmcnt(0)
template <int N>
__device__ __forceinline__ void wait_vm_lgkm0() {
  static_assert(N >= 0 && N < 64, "vmcnt immediate");
  __builtin_amdgcn_s_waitcnt(0x0070 | (N & 15) | ((N >> 4) << 14));
}

template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt immediate");
  __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14));
}

// Memory operations stay on their side of it, in the compiler's passes and its scheduler.
__device__ __forceinline__ void order_vmem() {
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  __builtin_amdgcn_sched_barrier(0);
}

// LDS layouts, conflict free on 64 banks of 4 B (encode_kernels.h's swizzles for other row
// lengths). x' and a K-contiguous W: rows of KC chunks.
template <int KC>
__device__ __forceinline__ int slim_swz(int row) {
  return KC == 8 ? (row ^ (row >> 3)) & 7 : (row >> 2) & 3;
}
// A feature-contiguous W: rows of TN features. 16-bit transpose reads touch 4 rows x 4 chunks
// (aligned) per clock: rows of 256 or 512 B all start at bank 0 and are spread by 4 (k % 4);
// 128-B rows (TN 64) k and k + 1 already sit in different bank halves and k, k + 2 are spread
// by 4. fp32 reads touch rows k and k + 4, 128 B each.
template <int DT, int TN>
__device__ __forceinline__ int slim_wswz(int k) {
  if constexpr (DT == SF_F32) return 8 * ((k >> 2) & 1);
  else if constexpr (TN >= 128) return 4 * (k & 3);
  else return 4 * ((k >> 1) & 1);
}

// Row-candidate epilogue of a wave's (32 MB x 32 NB) tile; as epilogue_rows (encode_kernels.h)
// with the output type and the floor taken at run time.
template <int MB, int NB>
__device__ __forceinline__ void slim_rows(const GemmArgs& a, f32x16 (&acc)[NB][MB], int64_t m0, int64_t n0, int lane,
                                          const float* s_t) {
  uint32_t km[MB];
  int cnt[MB], old[MB];
  uint32_t colok = 0;
#pragma unroll
  for (int q = 0; q < NB * 16; ++q) {
    const int64_t n = n0 + (q >> 4) * 32 + ((q >> 2) & 3) * 8 + (lane >> 5) * 4 + (q & 3);
    colok |= n < a.N ? 1u << q : 0u;
  }
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) {
    const int64_t m = m0 + mb * 32 + (lane & 31);
    float fl = -__builtin_inff();
    if (a.row_floor != nullptr && m < a.M) {
      const float F = a.row_floor[m];
      fl = a.out_dt == SF_F32 ? floor_lo<SF_F32>(F) : (a.out_dt == SF_BF16 ? floor_lo<SF_BF16>(F) : floor_lo<SF_F16>(F));
    }
    km[mb] = 0;
#pragma unroll
    for (int idx = 0; idx < NB * 4; ++idx) {
      const float4 th = *(const float4*)(s_t + (idx >> 2) * 32 + (idx & 3) * 8 + (lane >> 5) * 4);
      const float thv[4] = {th.x, th.y, th.z, th.w};
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float pre = acc[idx >> 2][mb][(idx & 3) * 4 + r];
        km[mb] |= !(pre <= thv[r]) && !(pre < fl) ? 1u << (idx * 4 + r) : 0u;  // a NaN is kept
      }
    }
    km[mb] = m < a.M ? km[mb] & colok : 0u;
    cnt[mb] = __popc(km[mb]);
    const int tot = cnt[mb] + __shfl_xor(cnt[mb], 32);
    old[mb] = 0;
    if (lane < 32 && tot > 0) old[mb] = atomicAdd(a.cand_cnt + m, tot);
  }
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) {
    const int64_t m = m0 + mb * 32 + (lane & 31);
    const int o = __shfl(old[mb], lane & 31), c = __shfl(cnt[mb], lane & 31);
    int64_t j = o + (lane >= 32 ? c : 0);
#pragma unroll
    for (int idx = 0; idx < NB * 4; ++idx) {
      const uint32_t nib = (km[mb] >> (idx * 4)) & 15u;
      if (__ballot(nib != 0) == 0) continue;  // wave-uniform: most groups hold nothing
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        if (nib & (1u << r)) {
          if (j < a.cap) {
            a.cand_idx[m * a.cap + j] = (int32_t)(n0 + (idx >> 2) * 32 + (idx & 3) * 8 + (lane >> 5) * 4 + r);
            const uint32_t b = f32_to_bits(acc[idx >> 2][mb][(idx & 3) * 4 + r], a.out_dt);
            if (a.out_dt == SF_F32) ((uint32_t*)a.cand_val)[m * a.cap + j] = b;
            else ((u16*)a.cand_val)[m * a.cap + j] = (u16)b;
          }
          ++j;
        }
      }
    }
  }
}

// Dense epilogue of a wave's tile, 32 tokens at a time through `reg` (32 rows of 32 NB features
// of this wave); the arithmetic of epilogue2. Aligned output rows are written as 16-B units,
// others one element per lane with consecutive lanes on consecutive features.
template <int OES, int MB, int NB>
__device__ __forceinline__ void slim_dense(const GemmArgs& a, f32x16 (&acc)[NB][MB], int64_t m0, int64_t n0, int lane,
                                           const float* s_t, char* reg) {
  constexpr int RB = NB * 32 * OES, UPR = RB / 16, RPI = 64 / UPR, EPU = 16 / OES;
  const bool count = a.row_nnz != nullptr;
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) {
    const int rl = lane & 31;
    const int64_t m = m0 + mb * 32 + rl;
    int cnt = 0;
#pragma unroll
    for (int idx = 0; idx < NB * 4; ++idx) {
      const int cl = (idx >> 2) * 32 + (idx & 3) * 8 + (lane >> 5) * 4;  // feature within the wave tile
      const float4 th = *(const float4*)(s_t + cl);
      const float thv[4] = {th.x, th.y, th.z, th.w};
      float o[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float pre = acc[idx >> 2][mb][(idx & 3) * 4 + r];
        const bool keep = !(pre <= thv[r]);
        o[r] = keep ? pre : 0.f;
        // columns past N have threshold +inf: only a NaN there would pass, and is not counted
        cnt += keep && n0 + cl + r < a.N ? 1 : 0;
      }
      char* dst = reg + rl * RB + ((((cl * OES) >> 4) ^ (rl & (UPR - 1))) << 4);
      if constexpr (OES == 4)
        *(float4*)dst = float4{o[0], o[1], o[2], o[3]};
      else if (a.out_dt == SF_F16)
        *(u32x2*)(dst + ((cl >> 2) & 1) * 8) = u32x2{pack2<SF_F16>(o[0], o[1]), pack2<SF_F16>(o[2], o[3])};
      else
        *(u32x2*)(dst + ((cl >> 2) & 1) * 8) = u32x2{pack2<SF_BF16>(o[0], o[1]), pack2<SF_BF16>(o[2], o[3])};
    }
    if (count) {
      const int c = cnt + __shfl_xor(cnt, 32);
      if (lane < 32 && m < a.M && c > 0) atomicAdd(a.row_nnz + m, c);
    }
    __builtin_amdgcn_wave_barrier();  // the staged rows are this wave's own (in-order LDS)
    if (a.vec_store && n0 + NB * 32 <= a.N) {
#pragma unroll
      for (int it = 0; it < 32 / RPI; ++it) {
        const int row = it * RPI + lane / UPR, u = lane % UPR;
        const u32x4 v = *(const u32x4*)(reg + row * RB + ((u ^ (row & (UPR - 1))) << 4));
        const int64_t mr = m0 + mb * 32 + row;
        if (mr < a.M) *(u32x4*)((char*)a.out + (mr * a.som + n0 + u * EPU) * OES) = v;
      }
    } else {
      constexpr int CPR = NB * 32, RPE = 64 / CPR;  // features and rows per 64 lanes
#pragma unroll 4
      for (int it = 0; it < 32 / RPE; ++it) {
        const int row = it * RPE + lane / CPR, col = lane % CPR;
        const char* src = reg + row * RB + ((((col * OES) >> 4) ^ (row & (UPR - 1))) << 4) + (col % EPU) * OES;
        const int64_t mr = m0 + mb * 32 + row, n = n0 + col;
        if (mr < a.M && n < a.N) {
          char* dst = (char*)a.out + (mr * a.som + n * a.son) * OES;
          if constexpr (OES == 2) *(u16*)dst = *(const u16*)src;
          else *(uint32_t*)dst = *(const uint32_t*)src;
        }
      }
    }
    __builtin_amdgcn_wave_barrier();
  }
}

// A W that a launch reads once (one token tile) streams past L2 (AUX_NT): d_in 2304 bf16, d_sae
// 65536, 1 token 58 -> 53 us a call; with several token tiles it is 2-60% slower, so those keep it.
//
// One workgroup per tile. Stage kt + NS - 1 is issued at K-step kt, right after the barrier that
// ends every wave's reads of the buffer it goes to, so NS - 1 stages are in flight; a thread
// waits only for its oldest stage (vmcnt counts in issue order) before the next barrier. Stages
// past the last K-step are issued with an empty range (zeros, no memory access), which keeps the
// count the same on every step. Register-staged W (S_NROWS, S_KROWS): the chunks of K-step kt + 1
// go from registers to LDS at step kt and those of kt + 3 are loaded (two sets of registers); x'
// stays on DMA, two steps ahead.
template <int DT, int SW, typename TL, int EPI, int AUX>
__global__ __launch_bounds__(TL::NT, TL::ST * TL::NS > 81920 ? TL::NW / 4 : TL::NW / 2) void gemm_slim_kernel(GemmArgs a) {
  constexpr int E = Traits<DT>::E, EPC = Traits<DT>::EPC;
  constexpr int MB = TL::MB, NB = TL::NB, KC = TL::KC, NS = TL::NS, NW = TL::NW, TN = TL::TN, TM = TL::TM;
  constexpr int PW = TL::PW, PX = TL::PX, BK = KC * EPC, KS = KC / 2;  // KS k16 (fp32: k8) steps per K-step
  constexpr bool NROW = SW == S_NMAJOR || SW == S_NROWS;  // W tile [k][n] in LDS, else [n][k]
  constexpr bool REG = SW == S_NROWS || SW == S_KROWS;
  constexpr int CPR = TN / EPC;  // 16-B chunks per [k][n] row
  static_assert((NS == 3 || NS == 4 || NS == 6) && (!REG || NS == 3), "stage buffers");
  // distinct LDS objects, so the compiler's wait-count pass can tell the DMA targets from the
  // buffer that fragments are read from
  __shared__ __attribute__((aligned(1024))) char s0[TL::ST];
  __shared__ __attribute__((aligned(1024))) char s1[TL::ST];
  __shared__ __attribute__((aligned(1024))) char s2[TL::ST];
  __shared__ __attribute__((aligned(1024))) char s3[NS > 3 ? TL::ST : 16];
  __shared__ __attribute__((aligned(1024))) char s4[NS > 4 ? TL::ST : 16];
  __shared__ __attribute__((aligned(1024))) char s5[NS > 5 ? TL::ST : 16];
  __shared__ __attribute__((aligned(16))) float s_benc[TN];
  __shared__ __attribute__((aligned(16))) float s_thr[TN];

  const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int wm = w / TL::WN, wn = w % TL::WN;
  // XCD-aware remap, as gemm_kernel
  const int total = a.tiles_m * a.tiles_n;
  const int b = blockIdx.x, per = total / 8, rem = total % 8, xcd = b % 8, loc = b / 8;
  const TilePos tp = tile_of(a, xcd * per + min(xcd, rem) + loc);
  const int64_t m0 = (int64_t)tp.m * TM, n0 = (int64_t)tp.n * TN;
  const int KT = a.ksteps;

  uint32_t xo[PX], wo[PW];
  int kcw[PW];
  const int64_t xbytes = min((int64_t)TM, a.M - m0) * a.Kp * E;
#pragma unroll
  for (int i = 0; i < PX; ++i) {
    const int P = (i * NW + w) * 64 + lane, m = P / KC;
    xo[i] = (uint32_t)(m * a.Kp * E + ((P % KC) ^ slim_swz<KC>(m)) * 16);
  }
#pragma unroll
  for (int i = 0; i < PW; ++i) {
    const int P = (i * NW + w) * 64 + lane;
    kcw[i] = 0;
    wo[i] = 0;
    if constexpr (SW == S_NMAJOR) {
      const int k = P / CPR, c = (P % CPR) ^ slim_wswz<DT, TN>(k);
      wo[i] = (uint32_t)((k * a.swk + min((int64_t)c * EPC, a.N - EPC - n0)) * E);  // past N: valid data again
    } else if constexpr (SW == S_KMAJOR) {
      const int n = P / KC;
      kcw[i] = (P % KC) ^ slim_swz<KC>(n);
      wo[i] = (uint32_t)(min((int64_t)n, a.N - 1 - n0) * a.swn * E + kcw[i] * 16);
    }
  }
  auto issue_x = [&](int kt, char* st) {
    const __amdgpu_buffer_rsrc_t xr = rsrc(a.xw + m0 * a.Kp * E, kt < KT ? xbytes : 0);
#pragma unroll
    for (int i = 0; i < PX; ++i)
      dma16(xr, st + TL::WT + (i * NW + w) * 1024, xo[i], (uint32_t)((int64_t)kt * BK * E));
  };
  auto issue = [&](int kt, char* st) {
    const int64_t k0 = (int64_t)kt * BK;
    issue_x(kt, st);
    if constexpr (SW == S_NMAJOR) {
      const int64_t rows = min((int64_t)BK, a.K - k0);  // rows past K read zero; <= 0 past the last step
      const __amdgpu_buffer_rsrc_t wr =
          rsrc(a.w + (k0 * a.swk + n0) * E, rows > 0 ? (rows - 1) * a.swk * E + (a.N - n0) * E : 0);
#pragma unroll
      for (int i = 0; i < PW; ++i) dma16_w<AUX>(wr, st + (i * NW + w) * 1024, wo[i], 0);
    } else if constexpr (SW == S_KMAJOR) {
      const __amdgpu_buffer_rsrc_t wr =
          rsrc(a.w + n0 * a.swn * E, kt < KT ? (min((int64_t)TN, a.N - n0) - 1) * a.swn * E + a.K * E : 0);
#pragma unroll
      for (int i = 0; i < PW; ++i)
        dma16_w<AUX>(wr, st + (i * NW + w) * 1024, k0 + kcw[i] * EPC >= a.K ? OOB : wo[i], (uint32_t)(k0 * E));
    }
  };
  // Register-staged W: this thread's chunks of K-step kt. Each is one 16-B load at any alignment;
  // a chunk that reaches past its row's end (`whole` is false for its tile or K-step) loads the
  // row's last 16 B instead and is shifted into place, zeros behind it, when it goes to LDS. Rows
  // past K load row K - 1 and go in as zeros; features past N are not stored, so theirs may hold
  // anything. Rows shorter than a chunk (`narrow`) are read element by element.
  u32x4 rw[2][REG ? PW : 1];
  const int64_t row_len = SW == S_NROWS ? a.N : a.K;
  const bool narrow = row_len < EPC;  // uniform
  auto whole = [&](int kt) { return SW == S_NROWS ? n0 + TN <= a.N : (int64_t)(kt + 1) * BK <= a.K; };
  // chunk i of K-step kt: its row and its first element within the row
  auto w_at = [&](int kt, int i, int64_t& row, int64_t& at) {
    const int P = (i * NW + w) * 64 + lane;
    if constexpr (SW == S_NROWS) {
      const int kr = P / CPR;
      row = (int64_t)kt * BK + kr;
      at = n0 + ((P % CPR) ^ slim_wswz<DT, TN>(kr)) * EPC;
    } else {
      const int nr = P / KC;
      row = n0 + nr;
      at = (int64_t)kt * BK + ((P % KC) ^ slim_swz<KC>(nr)) * EPC;
    }
  };
  // chunk addresses of K-step 0; a step adds k_step bytes per element of d_in while it lies inside K
  const int64_t k_step = (SW == S_NROWS ? a.swk : 1) * E;
  const char* w0[REG ? PW : 1];
  if constexpr (REG) {
#pragma unroll
    for (int i = 0; i < PW; ++i) {
      int64_t row, at;
      w_at(0, i, row, at);
      w0[i] = SW == S_NROWS ? a.w + (row * a.swk + min(at, a.N - EPC)) * E : a.w + (min(row, a.N - 1) * a.swn + at) * E;
    }
  }
  auto load_w = [&](int kt, u32x4 (&r)[REG ? PW : 1]) {
    if constexpr (REG) {
      const int64_t k0 = (int64_t)kt * BK;
      if (!narrow && k0 + BK <= a.K) {  // uniform
#pragma unroll
        for (int i = 0; i < PW; ++i) __builtin_memcpy(&r[i], __builtin_assume_aligned(w0[i] + k0 * k_step, E), 16);
        return;
      }
#pragma unroll
      for (int i = 0; i < PW; ++i) {
        int64_t row, at;
        w_at(kt, i, row, at);
        const char* p = a.w + min(row, (SW == S_NROWS ? a.K : a.N) - 1) * (SW == S_NROWS ? a.swk : a.swn) * E;
        if (!narrow) {
          __builtin_memcpy(&r[i], __builtin_assume_aligned(p + min(at, row_len - EPC) * E, E), 16);
        } else {
          u32x4 v = {0, 0, 0, 0};
#pragma unroll
          for (int e = 0; e < EPC; ++e)
            if (at + e < row_len) {
              if constexpr (E == 4) v[e] = ((const uint32_t*)p)[at + e];
              else v[e >> 1] |= (uint32_t)((const u16*)p)[at + e] << ((e & 1) * 16);
            }
          r[i] = v;
        }
      }
    }
  };
  auto put_w = [&](int kt, char* st, const u32x4 (&r)[REG ? PW : 1]) {
    if constexpr (REG) {
      const bool shift = !narrow && !whole(kt);                              // uniform
      const bool tail = SW == S_NROWS && (int64_t)(kt + 1) * BK > a.K;       // uniform
      if (!shift && !tail) {
#pragma unroll
        for (int i = 0; i < PW; ++i) *(u32x4*)(st + ((i * NW + w) * 64 + lane) * 16) = r[i];
        return;
      }
#pragma unroll
      for (int i = 0; i < PW; ++i) {
        int64_t row, at;
        w_at(kt, i, row, at);
        u32x4 v = r[i];
        if (shift) {
          const int64_t past = at - (row_len - EPC);  // elements by which the load was moved back
          const int sh = past <= 0 ? 0 : (past >= EPC ? 16 : (int)past * E);  // in bytes; 16: no element left
          const uint32_t q[5] = {v[0], v[1], v[2], v[3], 0};
          uint32_t u[5];
#pragma unroll
          for (int d = 0; d < 5; ++d) {
            u[d] = 0;
#pragma unroll
            for (int o = 0; o < 4; ++o)
              if (d + o < 4 && (sh >> 2) == o) u[d] = q[d + o];
          }
#pragma unroll
          for (int d = 0; d < 4; ++d) v[d] = (sh & 2) ? (u[d] >> 16) | (u[d + 1] << 16) : u[d];
        }
        if (tail && row >= a.K) v = u32x4{0, 0, 0, 0};
        *(u32x4*)(st + ((i * NW + w) * 64 + lane) * 16) = v;
      }
    }
  };

  f32x16 acc[NB][MB];
  struct Frag {
    u32x4 a[NB], b[MB];
  };
  auto load_frag = [&](Frag& f, const char* st, int s) {
    const char* xs = st + TL::WT;
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      const int row = (wm * MB + mb) * 32 + (lane & 31);
      f.b[mb] = *(const u32x4*)(xs + row * KC * 16 + (((2 * s + (lane >> 5)) ^ slim_swz<KC>(row)) << 4));
    }
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      const int c0 = (wn * NB + nb) * 32;
      if constexpr (NROW && DT != SF_F32) {  // transposing reads, as load_a
        const int g = lane >> 4, p = lane & 15;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int k = s * 16 + 8 * (g >> 1) + 4 * h + (p >> 2), col = c0 + 16 * (g & 1) + 4 * (p & 3);
          const int off = k * TN * 2 + (((col >> 3) ^ slim_wswz<DT, TN>(k)) << 4) + ((col >> 2) & 1) * 8;
          const u32x2 u = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(st + off)));
          f.a[nb][2 * h] = u[0];
          f.a[nb][2 * h + 1] = u[1];
        }
      } else if constexpr (NROW) {
        const int n = c0 + (lane & 31), kq = (2 * s + (lane >> 5)) * 4;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int k = kq + e;
          f.a[nb][e] = *(const uint32_t*)(st + k * TN * 4 + (((n >> 2) ^ slim_wswz<DT, TN>(k)) << 4) + (n & 3) * 4);
        }
      } else {
        const int row = c0 + (lane & 31);
        f.a[nb] = *(const u32x4*)(st + row * KC * 16 + (((2 * s + (lane >> 5)) ^ slim_swz<KC>(row)) << 4));
      }
    }
  };

  // raw bias and threshold bits of feature n0 + t % TN, loaded before the first stages so that
  // awaiting them does not await those
  const int64_t nb_ = min(n0 + t % TN, a.N - 1);
  const uint32_t rb = load_bits(a.b_enc, a.benc_dt, nb_);
  const uint32_t rt = a.act == SF_ACT_JUMPRELU ? load_bits(a.thr, a.thr_dt, nb_) : 0u;
  // the first stages
  if constexpr (REG) {
    load_w(0, rw[0]);
    load_w(1, rw[1]);
    issue_x(0, s0);
    issue_x(1, s1);
    wait_vmcnt0();
    put_w(0, s0, rw[0]);
    load_w(2, rw[0]);
    order_vmem();
  } else {
    issue(0, s0);
    issue(1, s1);
    if constexpr (NS > 3) issue(2, s2);
    if constexpr (NS > 4) issue(3, s3);
    if constexpr (NS > 5) issue(4, s4);
  }
  // bias and keep-threshold of the tile's features, as gemm_kernel
  if (t < TN) {
    const int64_t n = n0 + t;
    const float h = a.out_dt == SF_F32 ? 0.f : (a.out_dt == SF_BF16 ? 0x1p-126f : 0x1p-25f);
    float tv = a.act == SF_ACT_NONE ? __builtin_nanf("") : h;
    if (n >= a.N) {
      tv = __builtin_inff();
    } else if (a.act == SF_ACT_JUMPRELU) {
      const float th = bits_as_f32(rt, a.thr_dt);
      tv = th != th ? __builtin_inff() : fmaxf(th, h);
    }
    s_benc[t] = n < a.N ? bits_as_f32(rb, a.benc_dt) : 0.f;
    s_thr[t] = tv;
  }
  wait_lgkmcnt0();
  barrier_no_fence();
#pragma unroll
  for (int nb = 0; nb < NB; ++nb)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const float4 be = *(const float4*)(s_benc + (wn * NB + nb) * 32 + g * 8 + (lane >> 5) * 4);
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) {
        acc[nb][mb][g * 4 + 0] = be.x;
        acc[nb][mb][g * 4 + 1] = be.y;
        acc[nb][mb][g * 4 + 2] = be.z;
        acc[nb][mb][g * 4 + 3] = be.w;
      }
    }

  // K-step kt: its stage in `cur`; `nxt` takes stage kt + NS - 1 (DMA) or, with register-staged W,
  // `wnx` the W of kt + 1 and `nxt` the x' of kt + 2 (NS = 3; ODD: kt is odd).
  auto step = [&](auto odd_tag, int kt, char* cur, char* nxt, char* wnx) {
    constexpr int ODD = decltype(odd_tag)::value;
    if constexpr (!REG) {
      wait_vm_lgkm0<(NS - 2) * (PW + PX)>();
      barrier_no_fence();
      issue(kt + NS - 1, nxt);
    } else {
      wait_lgkmcnt0();
      barrier_no_fence();
      // This thread's x' of kt + 1 (issued a step ago) and W registers of kt + 1 (two steps ago);
      // only the W loads of kt + 2, issued after both, may still be in flight. vmcnt counts in issue
      // order, so a step's DMAs must all precede its W loads and none of these may slip behind the
      // next step's wait; no data ties them, so order_vmem keeps the compiler from moving either.
      if (!narrow) wait_vmcnt<PW>();
      else wait_vmcnt0();
      put_w(kt + 1, wnx, rw[1 - ODD]);
      issue_x(kt + 2, nxt);
      order_vmem();
      load_w(kt + 3, rw[1 - ODD]);
      order_vmem();
    }
    Frag f[2];
    load_frag(f[0], cur, 0);
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      if (s + 1 < KS) load_frag(f[(s + 1) & 1], cur, s + 1);
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) mfma_chunk<DT>(acc[nb][mb], f[s & 1].a[nb], f[s & 1].b[mb]);
    }
  };
  using S0 = std::integral_constant<int, 0>;
  using S1 = std::integral_constant<int, 1>;
  for (int kt = 0;;) {  // KT >= 1; the buffers (and the W register sets) rotate statically
    step(S0{}, kt, s0, NS == 3 ? s2 : (NS == 4 ? s3 : s5), s1);
    if (++kt >= KT) break;
    step(S1{}, kt, s1, s0, s2);
    if (++kt >= KT) break;
    step(S0{}, kt, s2, s1, NS == 3 ? s0 : s3);
    if (++kt >= KT) break;
    if constexpr (REG) {
      step(S1{}, kt, s0, s2, s1);
      if (++kt >= KT) break;
      step(S0{}, kt, s1, s0, s2);
      if (++kt >= KT) break;
      step(S1{}, kt, s2, s1, s0);
      if (++kt >= KT) break;
    }
    if constexpr (NS > 3) {
      step(S0{}, kt, s3, s2, NS == 4 ? s0 : s4);
      if (++kt >= KT) break;
    }
    if constexpr (NS > 4) {
      step(S0{}, kt, s4, s3, s5);
      if (++kt >= KT) break;
    }
    if constexpr (NS > 5) {
      step(S0{}, kt, s5, s4, s0);
      if (++kt >= KT) break;
    }
  }
  const int64_t mw = m0 + wm * MB * 32, nw = n0 + wn * NB * 32;
  const float* st = s_thr + wn * NB * 32;
  wait_vmcnt0();  // no DMA (the empty-range ones included) outlives its wave or hits the staging
  if constexpr (EPI != EPI_DENSE) {
    slim_rows<MB, NB>(a, acc, mw, nw, lane, st);
  } else {
    __syncthreads();
    constexpr int RG = 32 * NB * 32 * 4, WPS = TL::ST / RG;  // staging bytes per wave, waves per buffer
    static_assert(NW <= 2 * WPS, "epilogue staging");
    char* reg = w < WPS ? s0 + w * RG : s1 + (w - WPS) * RG;
    if (a.out_dt == SF_F32) slim_dense<4, MB, NB>(a, acc, mw, nw, lane, st, reg);
    else slim_dense<2, MB, NB>(a, acc, mw, nw, lane, st, reg);
  }
}

// The compiled shapes, by index (sf_encode's tile_cfg names them by BLOCK_M x BLOCK_N).
constexpr int SLIM_SHAPES = 6, SLIM_DMA_ONLY = 5;  // from SLIM_DMA_ONLY on: no register-staged W
struct SlimShape {
  int tm, tn, kc, nw;
};
template <typename TL>
constexpr SlimShape slim_shape_of() {
  return SlimShape{TL::TM, TL::TN, TL::KC, TL::NW};
}
constexpr SlimShape slim_shape(int i) {
  constexpr SlimShape all[SLIM_SHAPES] = {
      slim_shape_of<Slim32>(),  slim_shape_of<Slim128>(), slim_shape_of<Slim128w>(),
      slim_shape_of<Slim32w>(), slim_shape_of<Slim64w>(), slim_shape_of<Slim160x>()};
  return all[i];
}

template <int DT, int SW, typename TL>
hipError_t launch_slim_tile(const GemmArgs& a, int epi, hipStream_t s) {
  const dim3 grid(a.tiles_m * a.tiles_n), block(TL::NT);
  auto go = [&](auto aux_tag) {
    constexpr int AUX = decltype(aux_tag)::value;
    if (epi == EPI_DENSE) hipLaunchKernelGGL((gemm_slim_kernel<DT, SW, TL, EPI_DENSE, AUX>), grid, block, 0, s, a);
    else hipLaunchKernelGGL((gemm_slim_kernel<DT, SW, TL, EPI_ROWS, AUX>), grid, block, 0, s, a);
  };
  // one token tile: every W element is read once
  if (SW == S_NMAJOR && a.tiles_m == 1) go(std::integral_constant<int, SW == S_NMAJOR ? AUX_NT : 0>{});
  else go(std::integral_constant<int, 0>{});
  return hipGetLastError();
}

// Launches shape `shape` (tiles_m, tiles_n, ksteps and the group set for it). Defined where
// SF_SLIM_DEFINE is set, one instantiation per translation unit.
template <int DT, int SW>
hipError_t launch_slim(const GemmArgs& a, int shape, int epi, hipStream_t s);
#ifdef SF_SLIM_DEFINE
template <int DT, int SW>
hipError_t launch_slim(const GemmArgs& a, int shape, int epi, hipStream_t s) {
  constexpr bool REG = SW == S_NROWS || SW == S_KROWS;
  switch (shape) {
    case 0: return launch_slim_tile<DT, SW, std::conditional_t<REG, Slim32r, Slim32>>(a, epi, s);
    case 1: return launch_slim_tile<DT, SW, Slim128>(a, epi, s);
    case 2: return launch_slim_tile<DT, SW, std::conditional_t<REG, Slim128wr, Slim128w>>(a, epi, s);
    case 3: return launch_slim_tile<DT, SW, Slim32w>(a, epi, s);
    case 4: return launch_slim_tile<DT, SW, Slim64w>(a, epi, s);
    default: break;
  }
  if constexpr (!REG) return launch_slim_tile<DT, SW, Slim160x>(a, epi, s);
  return hipErrorInvalidValue;
}
#endif

}  // namespace sfenc
