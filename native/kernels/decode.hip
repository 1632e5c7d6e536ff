// Decode-path kernels for gfx950: the memory-bound half of LLM serving (one new
// token per sequence per step), written around layouts chosen for the MFMA
// operand maps so that every hot load is a contiguous 1 KB wave access.
//
//   * skinny GEMM   y[M, N] = x[M, K] . W[N, K]^T for a decode batch M <= 256.
//                   W is PREPACKED once (kgs/ops/decode.py pack_weight) into
//                   16-row x 32-k MFMA A-fragments: [N/16][K/32][64 lanes][8],
//                   so a wave streams its rows as back-to-back 1 KB loads
//                   straight into registers (no LDS round trip for the weight
//                   bytes). x (small, L2-resident) is staged through LDS in
//                   fragment order, read from global in whole rows, and shared
//                   by the 4 waves of a workgroup. Split-K across workgroups
//                   when N alone cannot fill 256 CUs: the last workgroup of a
//                   strip (agent-scope release/acquire ticket) reduces the fp32
//                   slabs and writes bf16 -- one launch, graph-capturable.
//   * rope_cache    rotate-half RoPE on the q and k heads of a fused QKV row and
//                   scatter k, v into the paged KV cache (one launch for both).
//   * paged decode attention: one wave per (sequence, KV head, context split);
//                   the GQA group's query heads are the 16 columns of
//                   S^T = K . Q^T (v_mfma_f32_16x16x32_bf16) and O^T = V^T . P^T
//                   takes the S^T accumulator as its B operand with no lane
//                   movement. The cache page layout is the MFMA fragment order
//                   itself (kv_k_index / kv_v_index) -- 16 contiguous 1 KB loads
//                   per 32-token page -- and context splits are merged
//                   (log-sum-exp) by the split that finishes last, in-launch.
#include "decode_common.h"

#include <type_traits>

namespace kgs {
namespace dec {

// ---------------------------------------------------------------------------
// skinny GEMM
// ---------------------------------------------------------------------------
// Workgroup = 4 waves = a strip of 64*R rows of W (wave w: 16-row tiles
// (strip*4 + w)*R .. +R-1) x all Mp = 16*MT columns, over one K range.
// x chunk per stage: KC k-steps of 32 x Mp rows, double buffered in LDS. The
// next chunk's x loads are issued a whole chunk (16 k-steps, ~2 us of weight
// streaming) before they are needed -- shorter distances stall on L2 latency
// (measured: KC 4 at Mp 64 ran 1.4x slower); W fragments stream through a
// register ring PF k-steps deep. Mp > 64 keeps KC 2 (VGPR-bound; the serving
// engine routes those batches to hipBLASLt, profiles/decode_kernels.md).
template <int MT, int KC_>
struct SkinnyCfg {
  static constexpr int KC = KC_;                    // k-steps per x chunk
  static constexpr int CHUNK_SLOTS = KC * MT * 64;  // 16-B slots per chunk
  static constexpr int LOADS = CHUNK_SLOTS / 256;   // per thread per chunk
};

// W8 (weight-only fp8, "W8A16"): W is OCP e4m3 in the same fragment order, 8 B
// per lane per fragment (512 B wave loads: half the HBM bytes), dequantised to
// bf16 in registers (v_cvt_pk_f32_fp8, times the lane's row scale, RNE to
// bf16); x, the MFMA and every epilogue stay bf16/fp32.
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
template <bool W8>
using WFrag = typename std::conditional<W8, u32x2, bf16x8>::type;

// 8 floats -> 8 OCP e4m3 bytes (saturating at +-448, RNE)
__device__ __forceinline__ uint2 tfm_e4m3x8(const float* v) {
  float c[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) c[e] = fminf(fmaxf(v[e], -448.f), 448.f);
  unsigned lo = __builtin_amdgcn_cvt_pk_fp8_f32(c[0], c[1], 0, false);
  lo = __builtin_amdgcn_cvt_pk_fp8_f32(c[2], c[3], lo, true);
  unsigned hi = __builtin_amdgcn_cvt_pk_fp8_f32(c[4], c[5], 0, false);
  hi = __builtin_amdgcn_cvt_pk_fp8_f32(c[6], c[7], hi, true);
  return make_uint2(lo, hi);
}

__device__ __forceinline__ bf16x8 dequant8(u32x2 v, float s) {
  bf16x8 o;
#pragma unroll
  for (int w = 0; w < 2; ++w) {
    const auto lo = __builtin_amdgcn_cvt_pk_f32_fp8((int)v[w], false);  // bytes 0, 1
    const auto hi = __builtin_amdgcn_cvt_pk_f32_fp8((int)v[w], true);   // bytes 2, 3
    o[4 * w + 0] = (short)f2bf(lo[0] * s);
    o[4 * w + 1] = (short)f2bf(lo[1] * s);
    o[4 * w + 2] = (short)f2bf(hi[0] * s);
    o[4 * w + 3] = (short)f2bf(hi[1] * s);
  }
  return o;
}

// EROPE: the EPI_ROPE instantiation (qkv of the fused decode layer only, so
// the other projections keep the lean epilogue's registers); its RoPE tables,
// positions and cache slots are loaded at kernel start, under the main loop.
// KIN (batch <= 64): the four waves share one strip of 16 R rows and
// split its K range four ways instead of each taking its own rows, so a
// 4096-row projection fills 256 CUs with no cross-workgroup split-K (the slab
// stores, the ticket and the last arriver's reduce are ~3-4 us of a 12-14 us
// batch-1 launch); the waves' partial tiles are summed through LDS. x comes
// straight from global/L2 through the W ring (no LDS staging): chunk = KC
// k-steps per wave, k_per_chunk = 4 * 32 * KC.
// SUMS: the instantiations with EPI_SUMS_IN and EPI_SUMS_OUT (bf16 weights, batch <= 64), apart because
// what they add moves the main loop's register allocation. The rows' scales are made once per workgroup, under the
// first weights' way from memory, and a workgroup's tiles are summed in LDS before they are added (with each
// tile's atomics and each output's conversion 1.2 us more a launch). us at 30 rows, floats / exact sums:
// 28672x4096 43.4 / 43.6, 4096x14336 29.5 / 29.1, 4096x4096 16.9 / 16.5.
// OWN (EPI_OWN; bf16 weights, batch <= 64): EPI_RMS by statistics that the workgroup makes itself from the operands as they pass
// (add_squares; decode_few.hip has the reason). KIN: each wave of its K quarter; else wave c of column tile c, and with cross-workgroup
// split-K (not KIN) the splits' sums go behind their slabs.
template <int R, int MT, int KC_, bool W8 = false, bool EROPE = false, bool KIN = false, bool SUMS = false, bool OWN = false>
__global__ __launch_bounds__(256, (MT * KC_ > 32 || R * MT >= 16) ? 1 : 2) void skinny(const void* __restrict__ wpv, const unsigned short* __restrict__ x,
                                                 unsigned short* __restrict__ y, float* __restrict__ ws,
                                                 int* __restrict__ cnt, int M, int N, int K, long ldx, long ldy,
                                                 int ksplit, int chunks_per_split, SkinnyEpi ep) {
  using C = SkinnyCfg<MT, KC_>;
  constexpr int KC = C::KC;
  // W ring depth in k-steps (divides KC); fp8 fragments are half the bytes, so
  // twice the depth keeps the same bytes in flight (a 16-deep bf16 ring at
  // batch 1 measured the same per launch: the fixed launch / split-K costs, not
  // the bytes in flight, set a batch-1 launch's time)
  constexpr int PF = KC < (W8 ? 16 : 8) ? KC : (W8 ? 16 : 8);
  // the only __shared__ object (a second one can make hipcc drain vmcnt before
  // every ds_read, cdna_hip_programming.md s5 trap 4a); the split-K "last
  // arriver" flag reuses its first word after the main loop
  static_assert(!KIN || PF == KC, "KIN: one ring round per chunk");
  __shared__ __attribute__((aligned(16))) bf16x8 xs[2][KIN ? 2 * R * MT * 64 : C::CHUNK_SLOTS];
  // SUMS: the rows' scales; a wave's sums of squares in [1 + wave]. OWN: a wave's (KIN), the rows'
  __shared__ typename std::conditional<OWN, double, float>::type stat[SUMS ? 5 : OWN && KIN ? 4 : 1][16 * MT];

  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int nstrip = N / ((KIN ? 16 : 64) * R);
  const int strip = blockIdx.x % nstrip, split = blockIdx.x / nstrip;
  if constexpr (SUMS) {
    if (ep.ss_zero != nullptr && blockIdx.x == 0)
      for (int i = tid; i < ep.zero_words; i += 256) ep.ss_zero[i] = 0.f;
  } else {
    if (ep.ss_zero != nullptr && blockIdx.x == 0 && tid < M) ep.ss_zero[tid] = 0.f;
  }
  const int nkk = K / 32;
  // k-steps (of 32) of this wave and where they start
  const int nsteps = chunks_per_split * KC;
  const int kk0 = KIN ? (split * 4 + w) * nsteps : split * nsteps;
  const int nt0 = KIN ? strip * R : (strip * 4 + w) * R;  // first 16-row tile of this wave
  const WFrag<W8>* wp = (const WFrag<W8>*)wpv;
  const WFrag<W8>* wrow[R];
  float wsc[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    wrow[r] = wp + ((long)(nt0 + r) * nkk + kk0) * 64 + lane;
    wsc[r] = W8 ? ep.wscale[16 * (nt0 + r) + (lane & 15)] : 1.f;
  }
  // EROPE: per (column tile c, row tile r) the lane's 4 cos / sin values and its
  // row's cache slot, fetched now so their latency hides under the main loop
  float rcs[EROPE ? MT : 1][EROPE ? R : 1][4], rsn[EROPE ? MT : 1][EROPE ? R : 1][4];
  int rslot[EROPE ? MT : 1];
  if constexpr (EROPE) {
    const int gq = lane >> 4;
#pragma unroll
    for (int c = 0; c < MT; ++c) {
      const int mr = min(16 * c + (lane & 15), M - 1);
      const int p = ep.pos[mr];
      rslot[c] = 16 * c + (lane & 15) < M ? ep.slot[mr] : -1;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int T = nt0 + r, t = T & 7;
        const int dd = gq < 2 ? 8 * t + 4 * gq : 8 * t + 4 * (gq - 2);  // dim within the rotated half
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          rcs[c][r][i] = ep.cosv[(long)p * (HD / 2) + dd + i];
          rsn[c][r][i] = ep.sinv[(long)p * (HD / 2) + dd + i];
        }
      }
    }
  }

  // x chunk staging: element e = tid + 256 i of the chunk, row-major over
  // (row m, 16-B column q) so global reads are whole-row runs; the LDS position
  // is the fragment slot ((kk*MT + ct)*64 + g*16 + r). Rows >= M re-read row
  // M-1 (their output columns are never stored).
  constexpr int QPR = KC * 4;  // 16-B columns per row per chunk
  bf16x8 xstage[C::LOADS];
  auto load_x = [&](int chunk) {
#pragma unroll
    for (int i = 0; i < C::LOADS; ++i) {
      const int e = tid + 256 * i, m = e / QPR, q = e - m * QPR;
      const int mr = m < M ? m : M - 1;
      xstage[i] = *(const bf16x8*)(x + (long)mr * ldx + (long)(kk0 + chunk * KC) * 32 + 8 * q);
    }
  };
  auto store_x = [&](int buf) {
#pragma unroll
    for (int i = 0; i < C::LOADS; ++i) {
      const int e = tid + 256 * i, m = e / QPR, q = e - m * QPR;
      const int kk = q >> 2, g = q & 3, ct = m >> 4, r = m & 15;
      xs[buf][(kk * MT + ct) * 64 + g * 16 + r] = xstage[i];
    }
  };

  f32x4v acc[R][MT];
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int c = 0; c < MT; ++c) acc[r][c] = f32x4v{0.f, 0.f, 0.f, 0.f};

  [[maybe_unused]] double own[OWN && KIN ? MT : 1] = {};  // OWN: this lane's part of its rows' sums of squares, of all column tiles (KIN) or the wave's own

  // Loads in the loops below are unconditional, so that hipcc can count vmcnt instead of draining the ring before
  // each MFMA. The last round, which sends for nothing more, stands behind them (PEEL): the last k-steps fetched again
  // were waited for at the end. us, fetched again / so: 3072x2048 at 48 rows 11.1 / 10.2, 2048x8192 at 24 15.0 / 13.7, 16384x2048 at 32
  // 16.3 / 14.9, 32000x2048 at 16 24.8 / 23.5. Eight tiles a wave and more spill, and four (K not split) are 3 % slower so at long K: these keep the clamped loads.
  constexpr bool PEEL = R * MT < (KIN ? 8 : 4);
  WFrag<W8> wf[PF][R];
  // OWN, KIN: the k-steps' order is fixed, else the compiler gives up the ring for the statistic's sake (84 registers instead of 167, every load in
  // flight waited for several times a chunk). us at 24 rows, given statistics / own, loose / own, fixed: 8192x2048 11.7 / 15.5 / 10.9, 3072x2048
  // 7.9 / 9.6 / 8.5, there with MFMAs of x with itself for the statistic; fixed with those / add_squares in one run 10.4 / 10.4, 7.9 / 7.6, two column
  // tiles of 6144x4096 18.9 / 19.9, four of 3072x2048 at 64 rows 12.3 / 12.7.
  constexpr bool PINNED = OWN && KIN && MT <= 2;
  if constexpr (!PINNED) {
#pragma unroll
    for (int p = 0; p < PF; ++p)
#pragma unroll
      for (int r = 0; r < R; ++r) wf[p][r] = __builtin_nontemporal_load(wrow[r] + (long)min(p, nsteps - 1) * 64);
  }

  if constexpr (SUMS) {
    if ((ep.mode & EPI_RMS) && tid < M) {
      const float ss = (ep.mode & EPI_SUMS_IN) ? exact_sum((const unsigned long long*)ep.ss_in + tid, M) : ep.ss_in[tid];
      stat[0][tid] = rsqrtf(ss * ep.inv_k + ep.eps);  // read after the barriers below
    }
  }
  if constexpr (KIN) {
    // B fragment of k-step s: lane (column m = 16 c + (lane & 15), k = 8 (lane >> 4) ..)
    // e4m3 weights with up to 16 rows in a form of its own: from the general one the compiler drains every load in
    // the middle of a chunk (us at 1 / 16 rows: 4096x4096 8.0 / 9.8, here 7.4 / 8.5; 6144x4096 10.2 / 14.5, here 9.6 / 13.0)
    if constexpr (W8 && MT == 1) {
      const unsigned short* xr = x + (long)min(lane & 15, M - 1) * ldx + (long)kk0 * 32 + 8 * (lane >> 4);
      bf16x8 xf[PF];
#pragma unroll
      for (int p = 0; p < PF; ++p) xf[p] = *(const bf16x8*)(xr + p * 32);
      auto round = [&](int s0, auto more) {
#pragma unroll
        for (int p = 0; p < PF; ++p) {
#pragma unroll
          for (int r = 0; r < R; ++r) acc[r][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(dequant8(wf[p][r], wsc[r]), xf[p], acc[r][0], 0, 0, 0);
          if constexpr (decltype(more)::value) {
            const int sn = s0 + p + PF;
#pragma unroll
            for (int r = 0; r < R; ++r) wf[p][r] = __builtin_nontemporal_load(wrow[r] + (long)sn * 64);
            xf[p] = *(const bf16x8*)(xr + sn * 32);
          }
        }
      };
      int s0 = 0;
      for (; s0 + PF < nsteps; s0 += PF) round(s0, std::true_type{});
      round(s0, std::false_type{});
    } else {
      const unsigned short* xr[MT];
#pragma unroll
      for (int c = 0; c < MT; ++c) xr[c] = x + (long)min(16 * c + (lane & 15), M - 1) * ldx + (long)kk0 * 32 + 8 * (lane >> 4);
      bf16x8 xf[PF][MT];
#pragma unroll
      for (int p = 0; p < PF; ++p) {
        if constexpr (PINNED) {
#pragma unroll
          for (int r = 0; r < R; ++r) wf[p][r] = __builtin_nontemporal_load(wrow[r] + p * 64);
        }
#pragma unroll
        for (int c = 0; c < MT; ++c) xf[p][c] = *(const bf16x8*)(xr[c] + p * 32);
        if constexpr (PINNED) __builtin_amdgcn_sched_barrier(0);
      }
      auto round = [&](int s0, auto more) {
#pragma unroll
        for (int p = 0; p < PF; ++p) {
#pragma unroll
          for (int r = 0; r < R; ++r) {
            bf16x8 wdq;
            if constexpr (W8) wdq = dequant8(wf[p][r], wsc[r]);
            else wdq = wf[p][r];
#pragma unroll
            for (int c = 0; c < MT; ++c) acc[r][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wdq, xf[p][c], acc[r][c], 0, 0, 0);
          }
          if constexpr (OWN) {
#pragma unroll
            for (int c = 0; c < MT; ++c) own[c] = add_squares(own[c], xf[p][c]);
          }
          if constexpr (decltype(more)::value) {
            const int sn = PEEL ? s0 + p + PF : min(s0 + p + PF, nsteps - 1);
#pragma unroll
            for (int r = 0; r < R; ++r) wf[p][r] = __builtin_nontemporal_load(wrow[r] + (long)sn * 64);
#pragma unroll
            for (int c = 0; c < MT; ++c) xf[p][c] = *(const bf16x8*)(xr[c] + sn * 32);
          }
          if constexpr (PINNED) __builtin_amdgcn_sched_barrier(0);
        }
      };
      int s0 = 0;
      for (; s0 + (PEEL ? PF : 0) < nsteps; s0 += PF) round(s0, std::true_type{});
      if constexpr (PEEL) round(s0, std::false_type{});
    }
    // the four K quarters of the strip: waves 1-3 hand theirs to wave 0 (slot 0
    // of xs stays free for the split-K flag); summed in wave order
    f32x4v* red = (f32x4v*)&xs[0][1];
    if constexpr (OWN) {
#pragma unroll
      for (int c = 0; c < MT; ++c) {
        const double s = wsum16(own[c]);
        if (lane < 16) stat[w][16 * c + lane] = s;
      }
    }
    if (w > 0) {
#pragma unroll
      for (int r = 0; r < R; ++r)
#pragma unroll
        for (int c = 0; c < MT; ++c) red[(((w - 1) * R + r) * MT + c) * 64 + lane] = acc[r][c];
    }
    __syncthreads();
    if (w == 0) {
#pragma unroll
      for (int r = 0; r < R; ++r)
#pragma unroll
        for (int c = 0; c < MT; ++c) {
          f32x4v t = acc[r][c];
#pragma unroll
          for (int v = 0; v < 3; ++v) t += red[((v * R + r) * MT + c) * 64 + lane];
          acc[r][c] = t;
        }
    }
  } else {
  load_x(0);
  store_x(0);
  __syncthreads();
  const int nchunks = chunks_per_split;
  auto round = [&](int chunk, auto more) {
    constexpr bool MORE = decltype(more)::value;
    if constexpr (MORE) load_x(PEEL ? chunk + 1 : min(chunk + 1, nchunks - 1));
    const bf16x8* xb = xs[chunk & 1] + lane;
#pragma unroll
    for (int kk = 0; kk < KC; ++kk) {
      const int p = kk % PF;
      if constexpr (OWN) {
        own[0] = add_squares(own[0], xb[(kk * MT + (w < MT ? w : 0)) * 64]);
      }
      bf16x8 wdq[R];
#pragma unroll
      for (int r = 0; r < R; ++r) {
        if constexpr (W8) wdq[r] = dequant8(wf[p][r], wsc[r]);
        else wdq[r] = wf[p][r];
      }
#pragma unroll
      for (int c = 0; c < MT; ++c) {
        const bf16x8 bfrag = xb[(kk * MT + c) * 64];
#pragma unroll
        for (int r = 0; r < R; ++r)
          acc[r][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wdq[r], bfrag, acc[r][c], 0, 0, 0);
      }
      if (MORE || kk + PF < KC) {
        const long sn = PEEL ? chunk * KC + kk + PF : min(chunk * KC + kk + PF, nsteps - 1);
#pragma unroll
        for (int r = 0; r < R; ++r) wf[p][r] = __builtin_nontemporal_load(wrow[r] + sn * 64);
      }
    }
    if constexpr (MORE) {
      store_x((chunk + 1) & 1);
      __syncthreads();
    }
  };
  int chunk = 0;
  for (; chunk + PEEL < nchunks; ++chunk) round(chunk, std::true_type{});
  if constexpr (PEEL) round(chunk, std::false_type{});
  if constexpr (OWN) {
    const double s = wsum16(own[0]);
    if (w < MT && lane < 16) stat[0][16 * w + lane] = s;
    __syncthreads();
  }
  }  // !KIN

  // C^T tile (r, c): lane holds column m = 16c + (lane & 15), rows n = 16*(nt0+r) + 4*(lane>>4) + i
  const int g = lane >> 4, mc = lane & 15;
  // store one lane's 4 consecutive outputs; every lane of the wave calls it
  // (the SWIGLU / RESID exchanges are cross-lane)
  auto emit = [&](f32x4v v, int m, int r) {
    const int ms = m < M ? m : M - 1;
    if constexpr (OWN) {
      double ss = stat[0][ms];
      if constexpr (KIN) ss = ((ss + stat[1][ms]) + stat[2][ms]) + stat[3][ms];
      v *= rsqrtf((float)ss * ep.inv_k + ep.eps);
    } else {
      if (ep.mode & EPI_RMS) v *= SUMS ? stat[0][ms] : rsqrtf(ep.ss_in[ms] * ep.inv_k + ep.eps);
    }
    if (ep.mode & EPI_SWIGLU) {
      f32x4v u;
#pragma unroll
      for (int i = 0; i < 4; ++i) u[i] = lane_xor32(v[i]);
      if (m < M && g < 2) {
        f32x4v o;
#pragma unroll
        for (int i = 0; i < 4; ++i)
          o[i] = (ep.mode & EPI_CLAMPED) ? gate_clamped(v[i], u[i], ep.limit)
                 : ((ep.mode & EPI_GELU) ? gate_act<GATE_GELU>(v[i]) : gate_act<GATE_SILU>(v[i])) * u[i];
        uint2 pk;
        pk.x = pack_bf16x2(o[0], o[1]);
        pk.y = pack_bf16x2(o[2], o[3]);
        *(uint2*)(y + (long)m * ldy + 8 * (nt0 + r) + 4 * g) = pk;
      }
    } else if (ep.mode & EPI_RESID) {
      float sq = 0.f;
      if (m < M) {
        uint2* yp = (uint2*)(y + (long)m * ldy + 16 * (nt0 + r) + 4 * g);
        const uint2 old = *yp;
        float o[4] = {bf2f(old.x & 0xffff) + v[0], bf2f(old.x >> 16) + v[1], bf2f(old.y & 0xffff) + v[2],
                      bf2f(old.y >> 16) + v[3]};
        uint2 pk;
        pk.x = pack_bf16x2(o[0], o[1]);
        pk.y = pack_bf16x2(o[2], o[3]);
        *yp = pk;
        // statistic of the stored (bf16-rounded) values, as add_rmsnorm computes it
        const float r0 = bf2f(pk.x & 0xffff), r1 = bf2f(pk.x >> 16), r2 = bf2f(pk.y & 0xffff), r3 = bf2f(pk.y >> 16);
        sq = r0 * r0 + r1 * r1 + r2 * r2 + r3 * r3;
      }
      sq = wsum16(sq);  // lanes of one column m (g = 0..3)
      if (m < M && g == 0 && ep.ss_out) {
        if (SUMS && (ep.mode & EPI_SUMS_OUT)) stat[1 + w][m] = r ? stat[1 + w][m] + sq : sq;
        else atomicAdd(ep.ss_out + m, sq);
      }
    } else if (EROPE) {
      const int c = m >> 4;
      const int T = nt0 + r, hh = T >> 3, t = T & 7;  // head and 16-row tile within it
      const bool rot = hh < ep.H + ep.HKV;
      f32x4v vb, pb;  // this lane's and its partner's (lane ^ 32) values, bf16-rounded
#pragma unroll
      for (int i = 0; i < 4; ++i) vb[i] = bf2f(f2bf(v[i]));
#pragma unroll
      for (int i = 0; i < 4; ++i) pb[i] = lane_xor32(vb[i]);
      // original dim of element 0: rotated heads hold (d, d + 64) pairs in a tile
      const int d0 = rot ? (g < 2 ? 8 * t + 4 * g : 64 + 8 * t + 4 * (g - 2)) : 16 * t + 4 * g;
      if (m < M) {
        f32x4v o = vb;
        if (rot) {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float cs = rcs[c][r][i], sn = rsn[c][r][i];
            o[i] = g < 2 ? rope_lo(vb[i], pb[i], cs, sn) : rope_hi(pb[i], vb[i], cs, sn);
          }
        }
        uint2 pk;
        pk.x = pack_bf16x2(o[0], o[1]);
        pk.y = pack_bf16x2(o[2], o[3]);
        *(uint2*)(y + (long)m * ldy + hh * HD + d0) = pk;
        const int sl = hh >= ep.H ? rslot[c] : -1;
        if (sl >= 0) {
          const int page = sl / PAGE, tau = sl - page * PAGE;
          const bool isv = hh >= ep.H + ep.HKV;
          const int kvh = isv ? hh - ep.H - ep.HKV : hh - ep.H;
          unsigned short* pg = ep.cache + (((long)page * ep.HKV + kvh) * 2 + (isv ? 1 : 0)) * PAGE_ELEMS;
          if (!isv) {
            *(uint2*)(pg + kv_k_index(tau, d0)) = pk;  // 4 consecutive dims: one 8-B run of the K fragment
          } else {
            pg[kv_v_index(tau, d0 + 0)] = (unsigned short)(pk.x & 0xffff);
            pg[kv_v_index(tau, d0 + 1)] = (unsigned short)(pk.x >> 16);
            pg[kv_v_index(tau, d0 + 2)] = (unsigned short)(pk.y & 0xffff);
            pg[kv_v_index(tau, d0 + 3)] = (unsigned short)(pk.y >> 16);
          }
        }
      }
    } else if (m < M) {
      uint2 pk;
      pk.x = pack_bf16x2(v[0], v[1]);
      pk.y = pack_bf16x2(v[2], v[3]);
      *(uint2*)(y + (long)m * ldy + 16 * (nt0 + r) + 4 * g) = pk;
    }
  };
  // the workgroup's sums of squares, in the order of its waves (KIN: wave 0's alone), to the rows' exact sums
  auto add_sums = [&] {
    if constexpr (SUMS) {
      if (!(ep.mode & EPI_RESID) || !(ep.mode & EPI_SUMS_OUT)) return;
      if constexpr (KIN) {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // other lanes' values, by the wave's own LDS order
        __builtin_amdgcn_wave_barrier();
      } else {
        __syncthreads();
      }
      if (tid < M) {
        float sq = stat[1][tid];
        if constexpr (!KIN) sq = ((sq + stat[2][tid]) + stat[3][tid]) + stat[4][tid];
        add_exact((unsigned long long*)ep.ss_out + tid, M, sq);
      }
    }
  };
  // Above 128 rows the unrolled epilogues are 25 thousand instructions, and a product that has none fetched its way
  // through them, 2 to 3 us of a launch: it stores by itself. us at 256 rows, through them / so: 4096x4096 63.6 /
  // 59.9, 6144x4096 68.9 / 63.5, 5120x5120 79.5 / 76.5. (Apart from the rest: a change to what fewer rows' kernels hold
  // here moves their register allocation, 28672x4096 at 16 rows 44 / 79.)
  [[maybe_unused]] auto store = [&](f32x4v v, int m, int r) {
    uint2 pk;
    pk.x = pack_bf16x2(v[0], v[1]);
    pk.y = pack_bf16x2(v[2], v[3]);
    if (m < M) *(uint2*)(y + (long)m * ldy + 16 * (nt0 + r) + 4 * g) = pk;
  };
  if constexpr (MT > 8) {
    if (ksplit == 1 && ep.mode == 0) {
#pragma unroll
      for (int c = 0; c < MT; ++c)
#pragma unroll
        for (int r = 0; r < R; ++r) store(acc[r][c], 16 * c + mc, r);
      return;
    }
  }
  if (ksplit == 1) {
    if (KIN && w != 0) return;
#pragma unroll
    for (int c = 0; c < MT; ++c)
#pragma unroll
      for (int r = 0; r < R; ++r) emit(acc[r][c], 16 * c + mc, r);
    add_sums();
    return;
  }
  // split-K: fp32 slabs ws[split][m][n] stored write-through (sc1); every wave
  // drains, the workgroup takes a ticket; the last arriver of the strip reads
  // every slab with sc1 loads and reduces -- no release/acquire fences.
  const long mstride = N, sstride = (long)16 * MT * N;
  const __amdgpu_buffer_rsrc_t wr = rsrc(ws, (unsigned)(ksplit * sstride * 4));
#pragma unroll
  for (int c = 0; c < MT; ++c) {
    const int m = 16 * c + mc;
    if (m < M && (!KIN || w == 0)) {
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int n = 16 * (nt0 + r) + 4 * g;
        st_sc1(wr, (unsigned)((split * sstride + m * mstride + n) * 4), acc[r][c]);
      }
    }
  }
  constexpr int SR = 16 * MT;  // OWN: sums of squares [split][strip][SR] behind the slabs
  const __amdgpu_buffer_rsrc_t sr = rsrc(ws + ksplit * sstride, OWN ? (unsigned)(ksplit * nstrip * SR * 8) : 0);
  if constexpr (OWN && !KIN) {
    if (tid < SR) st2_sc1(sr, (unsigned)(((split * nstrip + strip) * SR + tid) * 8), stat[0][tid]);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  int* flag = (int*)&xs[0][0];
  if (tid == 0) {
    const int prev = __hip_atomic_fetch_add(cnt + strip, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const int last = prev == ksplit - 1;
    if (last) {
      __hip_atomic_store(cnt + strip, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // re-arm
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    *flag = last;
  }
  __syncthreads();
  if (!*flag || (KIN && w != 0)) return;
  if constexpr (OWN && !KIN) {
    if (tid < SR) {
      double ss = 0.;
      for (int sp = 0; sp < ksplit; ++sp) ss += ld2_sc1(sr, (unsigned)(((sp * nstrip + strip) * SR + tid) * 8));
      stat[0][tid] = ss;
    }
    __syncthreads();
  }
  if constexpr (MT > 8) {
    if (ep.mode == 0) {
#pragma unroll
      for (int c = 0; c < MT; ++c) {
        const int m = 16 * c + mc;
#pragma unroll
        for (int r = 0; r < R; ++r) {
          const unsigned at = (unsigned)((min(m, M - 1) * mstride + 16 * (nt0 + r) + 4 * g) * 4);
          f32x4v t = f32x4v{0.f, 0.f, 0.f, 0.f};
          for (int sp0 = 0; sp0 < ksplit; sp0 += 4) {  // four slabs' loads in flight, as below
            f32x4v pv[4];
#pragma unroll
            for (int j = 0; j < 4; ++j)
              if (sp0 + j < ksplit) pv[j] = ld_sc1(wr, at + (unsigned)((sp0 + j) * sstride * 4));
#pragma unroll
            for (int j = 0; j < 4; ++j)
              if (sp0 + j < ksplit) t += pv[j];
          }
          store(t, m, r);
        }
      }
      return;
    }
  }
#pragma unroll
  for (int c = 0; c < MT; ++c) {
    const int m = 16 * c + mc;
    const int ms = m < M ? m : M - 1;  // every lane joins the epilogue exchanges
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int n = 16 * (nt0 + r) + 4 * g;
      f32x4v t = f32x4v{0.f, 0.f, 0.f, 0.f};
      // four slabs' loads in flight at a time (a load-add chain pays one L2
      // round trip per slab); summed in slab order as before
      for (int sp0 = 0; sp0 < ksplit; sp0 += 4) {
        f32x4v pv[4];
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (sp0 + j < ksplit) pv[j] = ld_sc1(wr, (unsigned)(((sp0 + j) * sstride + ms * mstride + n) * 4));
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (sp0 + j < ksplit) t += pv[j];
      }
      emit(t, m, r);
    }
  }
  add_sums();
}

// ---------------------------------------------------------------------------
// RoPE + KV-cache write
// ---------------------------------------------------------------------------
// k / v head h (H <= h < H + 2 HKV), dims (8c.., 64+8c..) = (a, b), into cache
// slot sl (page sl / 32, offset sl % 32) in the MFMA operand order of the pages
template <bool KV8>
__device__ __forceinline__ void kv_write(void* __restrict__ cache, int sl, int h, int H, int HKV, int c, bf16x8 a,
                                         bf16x8 b) {
  const int page = sl / PAGE, tau = sl - page * PAGE;
  const bool isv = h >= H + HKV;
  const int kvh = isv ? h - H - HKV : h - H;
  const long region = (((long)page * HKV + kvh) * 2 + (isv ? 1 : 0)) * PAGE_ELEMS;
  const int d1 = 8 * c, d2 = HD / 2 + 8 * c;
  if constexpr (KV8) {
    unsigned char* pg = (unsigned char*)cache + region;
    float fa[8], fb[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      fa[e] = bf2f((unsigned short)a[e]);
      fb[e] = bf2f((unsigned short)b[e]);
    }
    if (!isv) {
      *(uint2*)(pg + kv_k_index(tau, d1)) = tfm_e4m3x8(fa);
      *(uint2*)(pg + kv_k_index(tau, d2)) = tfm_e4m3x8(fb);
    } else {
      const uint2 qa = tfm_e4m3x8(fa), qb = tfm_e4m3x8(fb);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        pg[kv_v_index(tau, d1 + e)] = (unsigned char)(((e < 4 ? qa.x : qa.y) >> (8 * (e & 3))) & 0xff);
        pg[kv_v_index(tau, d2 + e)] = (unsigned char)(((e < 4 ? qb.x : qb.y) >> (8 * (e & 3))) & 0xff);
      }
    }
  } else {
    unsigned short* pg = (unsigned short*)cache + region;
    if (!isv) {
      *(bf16x8*)(pg + kv_k_index(tau, d1)) = a;
      *(bf16x8*)(pg + kv_k_index(tau, d2)) = b;
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        pg[kv_v_index(tau, d1 + e)] = (unsigned short)a[e];
        pg[kv_v_index(tau, d2 + e)] = (unsigned short)b[e];
      }
    }
  }
}

// qkv row t: [H q heads | HKV k heads | HKV v heads] x 128. Thread = (token,
// head among H + 2 HKV, chunk c < 8): q/k heads rotate dims (8c.., 64+8c..) in
// place; k and v heads are also written into page slot[t] (skipped when < 0).
// KV8: the cache holds OCP e4m3 bytes (scale 1, saturating) in the same
// element order -- a page region is 4 KB instead of 8 KB.
// SK: the projection arrives as nslice fp32 split-K partials P[s][t][nh * 128]
// (gemm_nt_w4x without its reduce); they are summed in slice order and rounded
// to bf16 exactly as kgs::splitk_reduce would, then rotated and stored to qkv
// and the cache -- one launch instead of reduce + rope_cache. NSL > 0: the
// slice count at compile time (all partial loads issued before the first add).
// PK (SK): the partials' columns are in the order of a weight packed with rope_rows (kgs/ops/decode.py), and rows of a raw residual
// stream: they are scaled by its RMSNorm, rsqrt(sq[row] * inv_k + eps).
template <bool KV8, bool SK = false, int NSL = 0, bool PK = false>
__global__ __launch_bounds__(256) void rope_cache(unsigned short* __restrict__ qkv, const float* __restrict__ cosv,
                                                  const float* __restrict__ sinv, const int* __restrict__ pos,
                                                  const int* __restrict__ slot, void* __restrict__ cache,
                                                  long tokens, int H, int HKV, long ld,
                                                  const float* __restrict__ P = nullptr, int nslice = 0,
                                                  const int* __restrict__ rows = nullptr, long prows = 0,
                                                  const float* __restrict__ sq = nullptr, float inv_k = 0.f, float eps = 0.f) {
  const int nh = H + 2 * HKV;
  const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= tokens * nh * 8) return;
  const long t = idx / (nh * 8);
  const int rem = (int)(idx - t * nh * 8);
  const int h = rem >> 3, c = rem & 7;
  const long row = rows ? rows[t] : t;
  if (row < 0) return;
  unsigned short* base = qkv + row * ld + (long)h * HD + 8 * c;
  bf16x8* p1 = (bf16x8*)base;
  bf16x8* p2 = (bf16x8*)(base + HD / 2);
  // position and cache slot first: the cos/sin loads hang off pos[t], so its
  // latency overlaps the qkv / partial loads instead of following them
  const int p = pos[t];
  const int sl = slot[t];
  bf16x8 a, b;
  if constexpr (SK) {
    const bool turned = PK && h < H + HKV;  // dims 8 c.. and 64 + 8 c.. side by side
    const long MN = prows * nh * HD, e = row * nh * HD + (long)h * HD + (turned ? 16 : 8) * c;
    const int far = turned ? 8 : HD / 2;
    const float scale = PK ? rsqrtf(sq[row] * inv_k + eps) : 1.f;
    f32x4 s[4];
    if constexpr (NSL > 0) {
      f32x4 ps[NSL][4];
#pragma unroll
      for (int sl = 0; sl < NSL; ++sl)
#pragma unroll
        for (int q = 0; q < 4; ++q) ps[sl][q] = *(const f32x4*)(P + sl * MN + e + (q >> 1) * far + (q & 1) * 4);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        s[q] = ps[0][q];
#pragma unroll
        for (int sl = 1; sl < NSL; ++sl) s[q] += ps[sl][q];
      }
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q) s[q] = *(const f32x4*)(P + e + (q >> 1) * far + (q & 1) * 4);
      for (int sl = 1; sl < nslice; ++sl)
#pragma unroll
        for (int q = 0; q < 4; ++q) s[q] += *(const f32x4*)(P + sl * MN + e + (q >> 1) * far + (q & 1) * 4);
    }
    if constexpr (PK) {
#pragma unroll
      for (int q = 0; q < 4; ++q) s[q] *= scale;
    }
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      a[k] = (short)f2bf(s[k >> 2][k & 3]);
      b[k] = (short)f2bf(s[2 + (k >> 2)][k & 3]);
    }
    if (h >= H + HKV) {  // v heads are not rotated: store them here
      *p1 = a;
      *p2 = b;
    }
  } else {
    a = *p1;
    b = *p2;
  }
  if (h < H + HKV) {
    const f32x4* cp = (const f32x4*)(cosv + (long)p * (HD / 2) + 8 * c);
    const f32x4* sp = (const f32x4*)(sinv + (long)p * (HD / 2) + 8 * c);
    const f32x4 c0 = cp[0], c1 = cp[1], s0 = sp[0], s1 = sp[1];
    bf16x8 o1, o2;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float cs = e < 4 ? c0[e] : c1[e - 4];
      const float sn = e < 4 ? s0[e] : s1[e - 4];
      const float x1 = bf2f((unsigned short)a[e]), x2 = bf2f((unsigned short)b[e]);
      o1[e] = (short)f2bf(rope_lo(x1, x2, cs, sn));
      o2[e] = (short)f2bf(rope_hi(x1, x2, cs, sn));
    }
    *p1 = o1;
    *p2 = o2;
    a = o1;
    b = o2;
  }
  if (h < H) return;
  if (sl < 0) return;
  kv_write<KV8>(cache, sl, h, H, HKV, c, a, b);
}

// Prompt-pass form (the projection in qkv, (H + 2 HKV) % 8 == 0): thread =
// (token, group of 8 heads, chunk c). The cos / sin of (pos[t], c) are loaded
// once for the 8 heads -- the per-head form above loads them once per head, as
// many bytes again as the qkv rows, all through L1 -- and the 8 heads' 16 row
// loads are issued before the first rotation. Same arithmetic per element
// (bitwise the per-head form's result).
// VSEP: the v heads are left to v_cache_pages (below): this kernel neither
// loads nor writes them.
template <bool KV8, bool VSEP = false>
__global__ __launch_bounds__(256) void rope_cache_g8(unsigned short* __restrict__ qkv, const float* __restrict__ cosv,
                                                     const float* __restrict__ sinv, const int* __restrict__ pos,
                                                     const int* __restrict__ slot, void* __restrict__ cache,
                                                     long tokens, int H, int HKV, long ld,
                                                     const int* __restrict__ rows) {
  const int ng = (H + 2 * HKV) >> 3;
  const long idx = (long)blockIdx.x * 256 + threadIdx.x;
  if (idx >= tokens * ng * 8) return;
  const long t = idx / (ng * 8);
  const int rem = (int)(idx - t * ng * 8);
  const int g = rem >> 3, c = rem & 7;
  if (VSEP && g * 8 >= H + HKV) return;  // a group of v heads only
  const long row = rows ? rows[t] : t;
  if (row < 0) return;
  const int p = pos[t];
  const int sl = slot[t];
  unsigned short* base = qkv + row * ld + (long)g * 8 * HD + 8 * c;
  bf16x8 a[8], b[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    a[j] = *(const bf16x8*)(base + j * HD);
    b[j] = *(const bf16x8*)(base + j * HD + HD / 2);
  }
  const f32x4* cp = (const f32x4*)(cosv + (long)p * (HD / 2) + 8 * c);
  const f32x4* sp = (const f32x4*)(sinv + (long)p * (HD / 2) + 8 * c);
  const f32x4 c0 = cp[0], c1 = cp[1], s0 = sp[0], s1 = sp[1];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const int h = g * 8 + j;
    if (h < H + HKV) {
      bf16x8 o1, o2;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float cs = e < 4 ? c0[e] : c1[e - 4];
        const float sn = e < 4 ? s0[e] : s1[e - 4];
        const float x1 = bf2f((unsigned short)a[j][e]), x2 = bf2f((unsigned short)b[j][e]);
        o1[e] = (short)f2bf(rope_lo(x1, x2, cs, sn));
        o2[e] = (short)f2bf(rope_hi(x1, x2, cs, sn));
      }
      *(bf16x8*)(base + j * HD) = o1;
      *(bf16x8*)(base + j * HD + HD / 2) = o2;
      a[j] = o1;
      b[j] = o2;
    }
    if (h >= H && sl >= 0 && !(VSEP && h >= H + HKV)) kv_write<KV8>(cache, sl, h, H, HKV, c, a[j], b[j]);
  }
}

// The prompt pass's V rows into the paged bf16 cache, one (run of 32 tokens,
// KV head) per workgroup. The V page layout is transposed (kv_v_index: a 16-B
// chunk holds one dim of 8 tokens), so a per-token writer stores 2 bytes at a
// time. Here the run's 32 x 128 values are staged in LDS and, when its slots
// fill one page in order (a prompt written from a page boundary), written as
// the page's 512 whole chunks; any other run goes element by element, exactly
// as kv_write.
__global__ __launch_bounds__(256) void v_cache_pages(const unsigned short* __restrict__ qkv,
                                                     const int* __restrict__ slot, unsigned short* __restrict__ cache,
                                                     long tokens, int H, int HKV, long ld,
                                                     const int* __restrict__ rows) {
  __shared__ unsigned short vs[PAGE][HD + 8];
  __shared__ int sl[PAGE];
  __shared__ int fast;
  const long t0 = (long)blockIdx.x * PAGE;
  const int kvh = blockIdx.y, tid = threadIdx.x;
  if (tid < PAGE) sl[tid] = t0 + tid < tokens && (!rows || rows[t0 + tid] >= 0) ? slot[t0 + tid] : -1;
  for (int k = tid; k < PAGE * (HD / 8); k += 256) {
    const int r = k / (HD / 8), ch = k % (HD / 8);
    const long t = t0 + r, row = t >= tokens ? -1 : rows ? rows[t] : t;
    const uint4 v = row >= 0 ? *(const uint4*)(qkv + row * ld + (long)(H + HKV + kvh) * HD + ch * 8)
                               : make_uint4(0, 0, 0, 0);
    *(uint4*)&vs[r][ch * 8] = v;
  }
  __syncthreads();
  if (tid == 0) {
    int ok = sl[0] >= 0 && sl[0] % PAGE == 0;
    for (int i = 1; i < PAGE && ok; ++i) ok = sl[i] == sl[0] + i;
    fast = ok;
  }
  __syncthreads();
  if (fast) {
    unsigned short* pg = cache + (((long)(sl[0] / PAGE) * HKV + kvh) * 2 + 1) * PAGE_ELEMS;
    for (int k = tid; k < PAGE_ELEMS / 8; k += 256) {  // chunk k = dt * 64 + g * 16 + m
      const int d = (k >> 6) * 16 + (k & 15), g = (k >> 4) & 3;
      bf16x8 o;
#pragma unroll
      for (int j = 0; j < 8; ++j) o[j] = (short)vs[4 * g + (j & 3) + 16 * (j >> 2)][d];
      *(bf16x8*)(pg + k * 8) = o;
    }
  } else {
    for (int k = tid; k < PAGE * HD; k += 256) {
      const int r = k / HD, d = k % HD, s = sl[r];
      if (s < 0) continue;
      unsigned short* pg = cache + (((long)(s / PAGE) * HKV + kvh) * 2 + 1) * PAGE_ELEMS;
      pg[kv_v_index(s % PAGE, d)] = vs[r][d];
    }
  }
}

// The first `ctx` cached tokens of a sequence as row-major K and V, [rows, HKV * 128] each, rows from
// ctx on zero: the keys a prompt chunk attends to. A workgroup per (page, KV head): both regions go
// through LDS as they lie, so that the rows leave as 256-byte runs. Bound by memory: 16384 tokens
// of 8 heads (67 MB read, as much written) take 24 us, 5.5 TB/s, against 176 for the same gather
// by tensor operations (an index, transpose, zero padding and conversion pass each); 4096
// tokens, where the launch is most of it, 9 against 70.
template <bool KV8>
__global__ __launch_bounds__(256) void gather_kv(const void* __restrict__ cache, const int* __restrict__ pages,
                                                 unsigned short* __restrict__ ko, unsigned short* __restrict__ vo, int ctx,
                                                 int rows, int HKV, int npages, long ld) {
  __shared__ __attribute__((aligned(16))) unsigned short sk[PAGE_ELEMS], sv[PAGE_ELEMS];
  const int t0 = blockIdx.x * PAGE, kvh = blockIdx.y, tid = threadIdx.x;
  int valid = ctx - t0;  // tokens of this page
  const int pg = valid > 0 ? pages[blockIdx.x] : 0;
  if ((unsigned)pg >= (unsigned)npages) valid = 0;
  if (valid > 0) {
    const long region = ((long)pg * HKV + kvh) * 2 * PAGE_ELEMS;
#pragma unroll
    for (int i = tid * 8; i < PAGE_ELEMS; i += 256 * 8) {
      if constexpr (KV8) {
        const unsigned char* p = (const unsigned char*)cache + region + i;
        *(bf16x8*)&sk[i] = dequant8(*(const u32x2*)p, 1.f);
        *(bf16x8*)&sv[i] = dequant8(*(const u32x2*)(p + PAGE_ELEMS), 1.f);
      } else {
        const unsigned short* p = (const unsigned short*)cache + region + i;
        *(bf16x8*)&sk[i] = *(const bf16x8*)p;
        *(bf16x8*)&sv[i] = *(const bf16x8*)(p + PAGE_ELEMS);
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int i = tid; i < PAGE_ELEMS / 8; i += 256) {
    const int tau = i >> 4, d = (i & 15) * 8;
    if (t0 + tau >= rows) continue;
    bf16x8 k = {0, 0, 0, 0, 0, 0, 0, 0}, v = k;
    if (tau < valid) {
      k = *(const bf16x8*)&sk[kv_k_index(tau, d)];
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = (short)sv[kv_v_index(tau, d + e)];
    }
    const long at = (long)(t0 + tau) * ld + kvh * HD + d;
    *(bf16x8*)(ko + at) = k;
    *(bf16x8*)(vo + at) = v;
  }
}

// ---------------------------------------------------------------------------
// paged decode attention
// ---------------------------------------------------------------------------
struct AttnArgs {
  const unsigned short* q;      // [B, ldq]: head h at q + h*128
  const unsigned short* cache;  // layer base: [pages][HKV][2][4096]
  const int* block_tables;      // [B, max_pages]
  const int* ctx_lens;          // [B] tokens in the cache (incl. the new one)
  unsigned short* o;            // [B, ldo]
  float* po;                    // [B, H, nsplit, 128] (nsplit > 1)
  float* pml;                   // [B, H, nsplit, 2]
  int* cnt;                     // [B * HKV] split tickets (in-launch merge), zero / re-armed
  long ldq, ldo;
  int B, H, HKV, max_pages, pages_per_split, nsplit;
  int merge;                    // nsplit > 1: 1 = last split merges in-launch, 0 = paged_reduce follows
  float sl2;                    // scale * log2(e)
  // RP (rope prologue): q / k / v arrive as nslice fp32 split-K partials of the
  // fused qkv projection, P[s][B][(H + 2 HKV) * 128]; the wave reduces, rotates
  // and caches its own (sequence, KV head) rows -- rope_cache folded in
  const float* P;
  int nslice;
  const float* cosv;            // [max_pos, 64]
  const float* sinv;
  const int* pos;               // [B]
  const int* slot;              // [B] cache slot of the new token (< 0: no write)
  void* cache_w;                // the same layer base as cache, writable
  // parts by length (paged_parts): units (parts of a sequence) to deal the pages to, a part's least pages, units at most
  int target, least, units;
};

// store O^T[dim 16dt + 4g + i][head] * inv for the lane's head
__device__ __forceinline__ void store_o(unsigned short* op, const f32x4v* acc, float inv) {
#pragma unroll
  for (int dt = 0; dt < 8; ++dt) {
    uint2 pk;
    pk.x = pack_bf16x2(acc[dt][0] * inv, acc[dt][1] * inv);
    pk.y = pack_bf16x2(acc[dt][2] * inv, acc[dt][3] * inv);
    *(uint2*)(op + 16 * dt) = pk;
  }
}

// One wave per (sequence, KV head, context split). With nsplit > 1 the partial (m, l, O)
// go to a workspace and the split that arrives last (agent-scope ticket per
// (sequence, KV head)) merges them -- no separate reduction launch.
// PIPE (small grids, e.g. batch 1-16): the next page's loads are issued before
// the current page is computed. With a few dozen waves on the chip no other wave
// hides a page's HBM latency, so a split otherwise pays it once per page.
//
// RP: the rope_cache work of this (sequence, KV head) runs first, in the wave:
// lane (hs = lane / 8, c = lane % 8) takes head slot hs (G q heads, then the k
// and the v head) and dims (8c.., 64+8c..), reduces the nslice partials in
// slice order, rounds to bf16 and rotates exactly as rope_cache does. The q
// heads go to LDS (the q fragments below are read from there), k and v to the
// cache slot -- written by the split whose pages hold the new token, which
// reads them back after its own stores have drained (vmcnt(0) before that
// page's loads only; nothing on this CU has that line in L1). Every split
// rotates q for itself. RP = the slice count (2, 4 or 8): all partial loads
// are issued before the first add, next to the position / slot loads.
template <bool KV8, bool PIPE = false, int RP = 0>
__global__ __launch_bounds__(64) void paged_decode(AttnArgs a) {
  const int lane = threadIdx.x;
  const int G = a.H / a.HKV;
  int id = blockIdx.x;
  const int sp = id % a.nsplit;
  id /= a.nsplit;
  const int kvh = id % a.HKV, b = id / a.HKV;
  const int g = lane >> 4, n = lane & 15;
  const int ctx = a.ctx_lens[b];
  const int npages = (ctx + PAGE - 1) / PAGE;
  const int p0 = sp * a.pages_per_split, p1 = min(npages, p0 + a.pages_per_split);
  const int h = kvh * G + n;
  __shared__ __attribute__((aligned(16))) unsigned short qs[RP ? 6 * HD : 8];  // RP: G <= 6 (host check)

  if constexpr (RP) {
    const int hs = lane >> 3, c = lane & 7;
    if (p0 < p1 && hs < G + 2) {
      const int nh = a.H + 2 * a.HKV;
      const int hh = hs < G ? kvh * G + hs : (hs == G ? a.H + kvh : a.H + a.HKV + kvh);
      const int p = a.pos[b];
      const int sl = a.slot[b];
      const long MN = (long)a.B * nh * HD, e = (long)b * nh * HD + (long)hh * HD + 8 * c;
      f32x4 ps[RP][4];
#pragma unroll
      for (int si = 0; si < RP; ++si)
#pragma unroll
        for (int q = 0; q < 4; ++q) ps[si][q] = *(const f32x4*)(a.P + si * MN + e + (q >> 1) * (HD / 2) + (q & 1) * 4);
      f32x4 s4[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        s4[q] = ps[0][q];
#pragma unroll
        for (int si = 1; si < RP; ++si) s4[q] += ps[si][q];
      }
      bf16x8 ra, rb;
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        ra[k] = (short)f2bf(s4[k >> 2][k & 3]);
        rb[k] = (short)f2bf(s4[2 + (k >> 2)][k & 3]);
      }
      if (hs <= G) {  // q and k heads: rotate-half RoPE at position p
        const f32x4* cp = (const f32x4*)(a.cosv + (long)p * (HD / 2) + 8 * c);
        const f32x4* spp = (const f32x4*)(a.sinv + (long)p * (HD / 2) + 8 * c);
        const f32x4 c0 = cp[0], c1 = cp[1], s0 = spp[0], s1 = spp[1];
        bf16x8 o1, o2;
#pragma unroll
        for (int e2 = 0; e2 < 8; ++e2) {
          const float cs = e2 < 4 ? c0[e2] : c1[e2 - 4];
          const float sn = e2 < 4 ? s0[e2] : s1[e2 - 4];
          const float x1 = bf2f((unsigned short)ra[e2]), x2 = bf2f((unsigned short)rb[e2]);
          o1[e2] = (short)f2bf(rope_lo(x1, x2, cs, sn));
          o2[e2] = (short)f2bf(rope_hi(x1, x2, cs, sn));
        }
        ra = o1;
        rb = o2;
      }
      if (hs < G) {
        *(bf16x8*)(qs + hs * HD + 8 * c) = ra;
        *(bf16x8*)(qs + hs * HD + HD / 2 + 8 * c) = rb;
      } else if (sl >= 0 && (ctx - 1) / PAGE >= p0 && (ctx - 1) / PAGE < p1) {
        kv_write<KV8>(a.cache_w, sl, hh, a.H, a.HKV, c, ra, rb);
      }
    }
    __syncthreads();  // q in LDS (the cache stores drain before the last page's loads)
  }
  const int last_page = (ctx - 1) / PAGE;  // RP: the page that holds the new token

  float m = -INFINITY, lsum = 0.f;
  f32x4v acc[8];
#pragma unroll
  for (int dt = 0; dt < 8; ++dt) acc[dt] = f32x4v{0.f, 0.f, 0.f, 0.f};

  if (p0 < p1) {
    bf16x8 qf[4];
    if constexpr (RP) {
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) qf[ks] = n < G ? *(const bf16x8*)(qs + n * HD + 8 * g + 32 * ks) : bf16x8{};
    } else {
      const unsigned short* qp = a.q + (long)b * a.ldq + (long)h * HD + 8 * g;
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) qf[ks] = n < G ? *(const bf16x8*)(qp + 32 * ks) : bf16x8{};
    }
    const int* bt = a.block_tables + (long)b * a.max_pages;
    auto load_page = [&](bf16x8 (&kf)[8], bf16x8 (&vf)[8], int pi) {
      if constexpr (RP != 0)
        if (pi == last_page) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // own k / v stores landed
      const long region = ((long)bt[pi] * a.HKV + kvh) * 2 * PAGE_ELEMS;  // elements of the K region
      if constexpr (KV8) {  // e4m3 pages: 8 B per lane per fragment, dequantised in registers
        const u32x2* kp = (const u32x2*)((const unsigned char*)a.cache + region) + lane;
        u32x2 kr[8], vr[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) kr[i] = __builtin_nontemporal_load(kp + 64 * i);
#pragma unroll
        for (int i = 0; i < 8; ++i) vr[i] = __builtin_nontemporal_load(kp + PAGE_ELEMS / 8 + 64 * i);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          kf[i] = dequant8(kr[i], 1.f);
          vf[i] = dequant8(vr[i], 1.f);
        }
      } else {
        const bf16x8* kp = (const bf16x8*)(a.cache + region) + lane;
#pragma unroll
        for (int i = 0; i < 8; ++i) kf[i] = __builtin_nontemporal_load(kp + 64 * i);
#pragma unroll
        for (int i = 0; i < 8; ++i) vf[i] = __builtin_nontemporal_load(kp + PAGE_ELEMS / 8 + 64 * i);
      }
    };
    auto page = [&](const bf16x8 (&kf)[8], const bf16x8 (&vf)[8], int pi) {
      f32x4v s[2];
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        s[t] = f32x4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < 4; ++ks)
          s[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[t * 4 + ks], qf[ks], s[t], 0, 0, 0);
      }
      // lane holds S^T[token 16t + 4g + i][head n]
      const int tok0 = pi * PAGE + 4 * g;
      float bm = -INFINITY;
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float v = (tok0 + 16 * t + i) < ctx ? s[t][i] * a.sl2 : -INFINITY;
          s[t][i] = v;
          bm = fmaxf(bm, v);
        }
      bm = wmax16(bm);
      const float mn = fmaxf(m, bm);
      const float alpha = __builtin_amdgcn_exp2f(m - mn);
      m = mn;
      bf16x8 pf;
      float ps = 0.f;
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float p = __builtin_amdgcn_exp2f(s[t][i] - mn);
          ps += p;
          pf[4 * t + i] = (short)f2bf(p);
        }
      lsum = lsum * alpha + ps;
#pragma unroll
      for (int dt = 0; dt < 8; ++dt) {
        acc[dt] *= alpha;
        acc[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[dt], pf, acc[dt], 0, 0, 0);
      }
    };
    if constexpr (PIPE) {
      // two register sets: page pi + 1 is in flight while page pi is computed
      bf16x8 ka[8], va[8], kb[8], vb[8];
      load_page(ka, va, p0);
      for (int pi = p0; pi < p1; pi += 2) {
        if (pi + 1 < p1) load_page(kb, vb, pi + 1);
        page(ka, va, pi);
        if (pi + 1 < p1) {
          if (pi + 2 < p1) load_page(ka, va, pi + 2);
          page(kb, vb, pi + 1);
        }
      }
    } else {
      // one page at a time: the loads of other waves on the SIMD hide this one's
      // latency (a two-register-set pipeline measured slower here: 208 VGPRs cost
      // a wave of occupancy, 47 -> 59 us at batch 64 x 1024)
      for (int pi = p0; pi < p1; ++pi) {
        bf16x8 kf[8], vf[8];
        load_page(kf, vf, pi);
        page(kf, vf, pi);
      }
    }
  }
  lsum = wsum16(lsum);
  // lane holds O^T[dim 16dt + 4g + i][head n]
  unsigned short* op = a.o + (long)b * a.ldo + (long)h * HD + 4 * g;
  if (a.nsplit == 1) {
    if (n < G) store_o(op, acc, lsum > 0.f ? 1.f / lsum : 0.f);
    return;
  }
  const long row = ((long)b * a.H + h) * a.nsplit;  // this head's first split slot
  const long nrows = (long)a.B * a.H * a.nsplit;
  const __amdgpu_buffer_rsrc_t por = rsrc(a.po, (unsigned)(nrows * HD * 4));
  const __amdgpu_buffer_rsrc_t mlr = rsrc(a.pml, (unsigned)(nrows * 8));
  if (n < G) {
#pragma unroll
    for (int dt = 0; dt < 8; ++dt) st_sc1(por, (unsigned)(((row + sp) * HD + 16 * dt + 4 * g) * 4), acc[dt]);
    if (g == 0) {
      st1_sc1(mlr, (unsigned)((row + sp) * 8), m);
      st1_sc1(mlr, (unsigned)((row + sp) * 8 + 4), lsum);
    }
  }
  if (!a.merge) return;  // paged_reduce merges after the kernel boundary
  // publish (write-through stores drained), take a ticket; the last split of
  // (b, kvh) merges with sc1 loads
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  int last = 0;
  if (lane == 0) {
    int* c = a.cnt + (long)b * a.HKV + kvh;
    last = __hip_atomic_fetch_add(c, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == a.nsplit - 1;
    if (last) {
      __hip_atomic_store(c, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // re-arm
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
  }
  last = __shfl(last, 0, 64);
  if (!last) return;
  if constexpr (PIPE) {
    // one pass with an online rescale (as over pages), the (m, l, O) loads of
    // four splits in flight together: the serial two-pass loop below pays an
    // L2 round trip per split (it stays for the large-grid variant, whose
    // occupancy the 128 extra VGPRs would cost)
    if (n >= G) return;
    float M = -INFINITY, L = 0.f;
    f32x4v o[8];
#pragma unroll
    for (int dt = 0; dt < 8; ++dt) o[dt] = f32x4v{0.f, 0.f, 0.f, 0.f};
    for (int s0 = 0; s0 < a.nsplit; s0 += 4) {
      float mv[4], lv[4];
      f32x4v part[4][8];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        mv[j] = -INFINITY;
        lv[j] = 0.f;
        if (s0 + j < a.nsplit) {
          mv[j] = ld1_sc1(mlr, (unsigned)((row + s0 + j) * 8));
          lv[j] = ld1_sc1(mlr, (unsigned)((row + s0 + j) * 8 + 4));
#pragma unroll
          for (int dt = 0; dt < 8; ++dt)
            part[j][dt] = ld_sc1(por, (unsigned)(((row + s0 + j) * HD + 16 * dt + 4 * g) * 4));
        }
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (lv[j] <= 0.f) continue;
        const float mn = fmaxf(M, mv[j]);
        const float sc = __builtin_amdgcn_exp2f(M - mn), f = __builtin_amdgcn_exp2f(mv[j] - mn);
        L = L * sc + f * lv[j];
#pragma unroll
        for (int dt = 0; dt < 8; ++dt) o[dt] = o[dt] * sc + f * part[j][dt];
        M = mn;
      }
    }
    store_o(op, o, L > 0.f ? 1.f / L : 0.f);
    return;
  }
  if (n >= G) return;
  float M = -INFINITY;
  for (int s2 = 0; s2 < a.nsplit; ++s2) M = fmaxf(M, ld1_sc1(mlr, (unsigned)((row + s2) * 8)));
  float L = 0.f;
  f32x4v o[8];
#pragma unroll
  for (int dt = 0; dt < 8; ++dt) o[dt] = f32x4v{0.f, 0.f, 0.f, 0.f};
  for (int s2 = 0; s2 < a.nsplit; ++s2) {
    const float ms = ld1_sc1(mlr, (unsigned)((row + s2) * 8));
    const float ls = ld1_sc1(mlr, (unsigned)((row + s2) * 8 + 4));
    if (ls <= 0.f) continue;
    const float f = __builtin_amdgcn_exp2f(ms - M);
    L += f * ls;
#pragma unroll
    for (int dt = 0; dt < 8; ++dt) o[dt] += f * ld_sc1(por, (unsigned)(((row + s2) * HD + 16 * dt + 4 * g) * 4));
  }
  store_o(op, o, L > 0.f ? 1.f / L : 0.f);
}

// Inclusive sums over the wave's lanes, all of them active: shifts by 1, 2, 4 and 8 within rows of 16, then the last
// lane of row 0 (of 2) to row 1 (3) and of lane 31 to the upper half
__device__ __forceinline__ int scan64(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, true);
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, true);
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, true);
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, true);
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);
  return v;
}

// Decode attention by workgroups: W waves share a (sequence, KV head), or one of nsplit equal
// parts of its pages. paged_decode gives every (sequence, KV head, fixed number of pages) one wave,
// so a batch of unequal contexts waits for the longest one's wave, and at small batches a split
// costs a merge through memory. Here the pages are dealt to the waves by the sequence's own length
// (wave w takes pages w, w + W, ..) and the waves merge in LDS. Bound by the HBM reads of K and V:
// 100 sequences of 60 to 2800 tokens (4 KV heads) 60 -> 38 us, one of 4000 (8 KV heads)
// 22 -> 11 us, 256 unequal ones around 1024 329 -> 171 us; 256 equal ones of 1024, which the single
// waves already read at 6.9 TB/s, 156 -> 163 us (the host, which sees the table's width and not the
// lengths, cannot tell the two; equal lengths lose 4 %, unequal ones gain half). Narrow tables take
// fewer waves or the single-wave kernel by a rule on the host.
//
// A wave's page ids lie in its lanes (64 at a time, one load), so that no page waits for its id.
// bf16 pages: eight waves, four on a SIMD hide each other's loads. e4m3 pages (PIPE): four waves
// that keep the next page on its way in registers while they widen and multiply one (64 sequences
// around 700 tokens, 8 KV heads: 22 us, 31 without). Fewer waves where the table holds few pages
// (kgs/ops/decode.py workgroup_waves).
template <bool KV8>
struct PageRegs;  // a page's K and V as loaded: fragment order, e4m3 pages 8 bytes a lane
template <>
struct PageRegs<false> {
  bf16x8 k[8], v[8];
  __device__ void load(const void* cache, long region, int lane) {
    const bf16x8* p = (const bf16x8*)((const unsigned short*)cache + region) + lane;
#pragma unroll
    for (int i = 0; i < 8; ++i) k[i] = __builtin_nontemporal_load(p + 64 * i);
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = __builtin_nontemporal_load(p + PAGE_ELEMS / 8 + 64 * i);
  }
  __device__ bf16x8 kf(int i) const { return k[i]; }
  __device__ bf16x8 vf(int i) const { return v[i]; }
};
template <>
struct PageRegs<true> {
  u32x2 k[8], v[8];
  __device__ void load(const void* cache, long region, int lane) {
    const u32x2* p = (const u32x2*)((const unsigned char*)cache + region) + lane;
#pragma unroll
    for (int i = 0; i < 8; ++i) k[i] = __builtin_nontemporal_load(p + 64 * i);
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = __builtin_nontemporal_load(p + PAGE_ELEMS / 8 + 64 * i);
  }
  __device__ bf16x8 kf(int i) const { return dequant8(k[i], 1.f); }
  __device__ bf16x8 vf(int i) const { return dequant8(v[i], 1.f); }
};

// The attention itself, as described above at PageRegs. BAL (paged_parts): the parts follow the lengths, so that a long context is no longer one workgroup's (100
// sequences of 60 to 2800 tokens, 4 KV heads: 38.1 -> 29.9 us, 70 of 4000 at most 44.9 -> 31.2; the rules are part_target and length_parts). All workgroups read
// all of them (a lane holds BAL of each 64) and cut every sequence into equal parts of at most P pages, P such that `target` parts of P hold
// them all (at least `least`): unit u of the grid is the u-th such part. Partial results and tickets are the caller's, of a call and a step.
template <bool KV8, int W, bool PIPE, int BAL>
__device__ __forceinline__ void paged_waves(const AttnArgs& a) {
  constexpr int LDO = HD + 4;  // a row of partial outputs: 16 heads' rows start on different banks
  __shared__ __attribute__((aligned(16))) float part[W][16][LDO];
  __shared__ float mls[W][16][2];
  __shared__ int is_last;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int G = a.H / a.HKV;
  int id = blockIdx.x, sp, kvh, b, nsplit = a.nsplit, first = 0;  // first: the sequence's first unit (BAL)
  const int g = lane >> 4, n = lane & 15;
  if constexpr (BAL) {
    kvh = id % a.HKV;
    id /= a.HKV;
    int pages[BAL], total = 0;
#pragma unroll
    for (int i = 0; i < BAL; ++i) {
      const int at = 64 * i + lane;
      pages[i] = at < a.B ? max(0, min((a.ctx_lens[at] + PAGE - 1) / PAGE, a.max_pages)) : 0;
      total += pages[i];
    }
    total = __builtin_amdgcn_readlane(scan64(total), 63);
    const int P = (max(a.least, (int)((unsigned)(total + a.target - 1) / (unsigned)a.target)) + W - 1) / W * W;  // whole rounds of the waves
    b = -1;
    int before = 0;
#pragma unroll
    for (int i = 0; i < BAL; ++i) {
      const int parts = 64 * i + lane < a.B ? max(1u, (unsigned)(pages[i] + P - 1) / (unsigned)P) : 0;
      const int upto = before + scan64(parts);
      const unsigned long long hit = __ballot(parts && id >= upto - parts && id < upto);
      if (hit) {
        const int l = __builtin_ctzll(hit);
        b = 64 * i + l;
        nsplit = __builtin_amdgcn_readlane(parts, l);
        first = __builtin_amdgcn_readlane(upto, l) - nsplit;
        sp = id - first;
        break;
      }
      before = __builtin_amdgcn_readlane(upto, 63);
    }
    if (b < 0) return;
  } else {
    sp = id % nsplit;
    id /= nsplit;
    kvh = id % a.HKV;
    b = id / a.HKV;
  }
  const int ctx = a.ctx_lens[b];
  const int npages = min((ctx + PAGE - 1) / PAGE, a.max_pages);
  const int per = (npages + nsplit - 1) / nsplit;
  const int p0 = sp * per, p1 = min(npages, p0 + per);
  const int h = kvh * G + n;
  const int mine = p1 > p0 + w ? (p1 - p0 - w + W - 1) / W : 0;  // this wave's pages

  float m = -INFINITY, lsum = 0.f;
  f32x4v acc[8];
#pragma unroll
  for (int dt = 0; dt < 8; ++dt) acc[dt] = f32x4v{0.f, 0.f, 0.f, 0.f};
  if (mine) {
    const int* bt = a.block_tables + (long)b * a.max_pages + p0 + w;
    int ids = lane < mine ? bt[W * lane] : 0;
    bf16x8 qf[4];
    const unsigned short* qp = a.q + (long)b * a.ldq + (long)h * HD + 8 * g;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) qf[ks] = n < G ? *(const bf16x8*)(qp + 32 * ks) : bf16x8{};
    auto load_page = [&](PageRegs<KV8>& r, int j) {
      if (j && (j & 63) == 0) ids = j + lane < mine ? bt[W * (j + lane)] : 0;
      r.load(a.cache, ((long)__builtin_amdgcn_readlane(ids, j & 63) * a.HKV + kvh) * 2 * PAGE_ELEMS, lane);
    };
    auto page = [&](const PageRegs<KV8>& r, int j) {
      f32x4v s[2];
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        s[t] = f32x4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) s[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(r.kf(t * 4 + ks), qf[ks], s[t], 0, 0, 0);
      }
      const int tok0 = (p0 + w + W * j) * PAGE + 4 * g;  // lane holds S^T[token 16t + 4g + i][head n]
      float bm = -INFINITY;
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float v = (tok0 + 16 * t + i) < ctx ? s[t][i] * a.sl2 : -INFINITY;
          s[t][i] = v;
          bm = fmaxf(bm, v);
        }
      bm = wmax16(bm);
      const float mn = fmaxf(m, bm), alpha = __builtin_amdgcn_exp2f(m - mn);
      m = mn;
      bf16x8 pf;
      float ps = 0.f;
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float p = __builtin_amdgcn_exp2f(s[t][i] - mn);
          ps += p;
          pf[4 * t + i] = (short)f2bf(p);
        }
      lsum = lsum * alpha + ps;
#pragma unroll
      for (int dt = 0; dt < 8; ++dt) {
        acc[dt] *= alpha;
        acc[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(r.vf(dt), pf, acc[dt], 0, 0, 0);
      }
    };
    if constexpr (PIPE) {
      PageRegs<KV8> ra, rb;
      load_page(ra, 0);
      for (int j = 0; j < mine; j += 2) {
        if (j + 1 < mine) load_page(rb, j + 1);
        page(ra, j);
        if (j + 1 < mine) {
          if (j + 2 < mine) load_page(ra, j + 2);
          page(rb, j + 1);
        }
      }
    } else {
      for (int j = 0; j < mine; ++j) {
        PageRegs<KV8> r;
        load_page(r, j);
        page(r, j);
      }
    }
    lsum = wsum16(lsum);
  }
  // lane holds O^T[dim 16dt + 4g + i][head n]
  if (n < G) {
#pragma unroll
    for (int dt = 0; dt < 8; ++dt) *(f32x4v*)&part[w][n][16 * dt + 4 * g] = acc[dt];
    if (g == 0) {
      mls[w][n][0] = m;
      mls[w][n][1] = lsum;
    }
  }
  __syncthreads();
  // rows of partial results: part s of head hh
  const long nrows = (long)(BAL ? a.units : a.B * nsplit) * a.H;
  const unsigned next = BAL ? a.H : 1;
  auto row_of = [&](int hh) { return BAL ? (unsigned)(first * a.H + hh) : (unsigned)(((long)b * a.H + hh) * nsplit); };
  const __amdgpu_buffer_rsrc_t por = rsrc(a.po, (unsigned)(nrows * HD * 4));
  const __amdgpu_buffer_rsrc_t mlr = rsrc(a.pml, (unsigned)(nrows * 8));
  // a thread's four dims of one head
  for (int i = threadIdx.x; i < G * (HD / 4); i += 64 * W) {
    const int hn = i >> 5, d = (i & 31) * 4;
    float M = -INFINITY;
#pragma unroll
    for (int x = 0; x < W; ++x) M = fmaxf(M, mls[x][hn][0]);
    float L = 0.f;
    f32x4v o = f32x4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int x = 0; x < W; ++x) {
      const float l = mls[x][hn][1];
      if (l <= 0.f) continue;
      const float f = __builtin_amdgcn_exp2f(mls[x][hn][0] - M);
      L += f * l;
      o += f * *(const f32x4v*)&part[x][hn][d];
    }
    const int hh = kvh * G + hn;
    if (nsplit == 1) {
      const float inv = L > 0.f ? 1.f / L : 0.f;
      *(uint2*)(a.o + (long)b * a.ldo + (long)hh * HD + d) =
          make_uint2(pack_bf16x2(o[0] * inv, o[1] * inv), pack_bf16x2(o[2] * inv, o[3] * inv));
    } else {
      const unsigned row = row_of(hh) + sp * next;
      st_sc1(por, (row * HD + d) * 4, o);
      if (d == 0) {
        st1_sc1(mlr, row * 8, M);
        st1_sc1(mlr, row * 8 + 4, L);
      }
    }
  }
  if (nsplit == 1) return;
  // the split that arrives last merges: partial results written through, then a ticket
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (threadIdx.x == 0) {
    int* c = a.cnt + (long)b * a.HKV + kvh;
    const int last = __hip_atomic_fetch_add(c, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == nsplit - 1;
    if (last) {
      __hip_atomic_store(c, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // re-arm
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    is_last = last;
  }
  __syncthreads();
  if (!is_last) return;
  if constexpr (!BAL) {
    for (int i = threadIdx.x; i < G * (HD / 4); i += 64 * W) {
      const int hn = i >> 5, d = (i & 31) * 4, hh = kvh * G + hn;
      const unsigned row = (unsigned)(((long)b * a.H + hh) * a.nsplit);
      float M = -INFINITY, L = 0.f;
      f32x4v o = f32x4v{0.f, 0.f, 0.f, 0.f};
      for (int s0 = 0; s0 < a.nsplit; s0 += 4) {
        float mv[4], lv[4];
        f32x4v pv[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          mv[j] = -INFINITY;
          lv[j] = 0.f;
          if (s0 + j < a.nsplit) {
            mv[j] = ld1_sc1(mlr, (row + s0 + j) * 8);
            lv[j] = ld1_sc1(mlr, (row + s0 + j) * 8 + 4);
            pv[j] = ld_sc1(por, ((row + s0 + j) * HD + d) * 4);
          }
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          if (lv[j] <= 0.f) continue;
          const float mn = fmaxf(M, mv[j]);
          const float sc = __builtin_amdgcn_exp2f(M - mn), f = __builtin_amdgcn_exp2f(mv[j] - mn);
          L = L * sc + f * lv[j];
          o = o * sc + f * pv[j];
          M = mn;
        }
      }
      const float inv = L > 0.f ? 1.f / L : 0.f;
      *(uint2*)(a.o + (long)b * a.ldo + (long)hh * HD + d) =
          make_uint2(pack_bf16x2(o[0] * inv, o[1] * inv), pack_bf16x2(o[2] * inv, o[3] * inv));
    }
    return;
  }
  const int tasks = G * (HD / 4);  // a thread's four dims of one head
  // parts pg, pg + groups, ..: four rows on their way at once
  auto merge = [&](int ii, int pg, int groups, float& M, float& L, f32x4v& o) {
    const unsigned row = row_of(kvh * G + (ii >> 5)), d = (ii & 31) * 4;
    M = -INFINITY, L = 0.f;
    o = f32x4v{0.f, 0.f, 0.f, 0.f};
    for (int s0 = pg; s0 < nsplit; s0 += 4 * groups) {
      float mv[4], lv[4];
      f32x4v pv[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        mv[j] = -INFINITY;
        lv[j] = 0.f;
        const int sj = s0 + j * groups;
        if (sj < nsplit) {
          mv[j] = ld1_sc1(mlr, (row + sj * next) * 8);
          lv[j] = ld1_sc1(mlr, (row + sj * next) * 8 + 4);
          pv[j] = ld_sc1(por, ((row + sj * next) * HD + d) * 4);
        }
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (lv[j] <= 0.f) continue;
        const float mn = fmaxf(M, mv[j]);
        const float sc = __builtin_amdgcn_exp2f(M - mn), f = __builtin_amdgcn_exp2f(mv[j] - mn);
        L = L * sc + f * lv[j];
        o = o * sc + f * pv[j];
        M = mn;
      }
    }
  };
  auto store = [&](int ii, float L, const f32x4v& o) {
    const float inv = L > 0.f ? 1.f / L : 0.f;
    *(uint2*)(a.o + (long)b * a.ldo + (long)(kvh * G + (ii >> 5)) * HD + (ii & 31) * 4) =
        make_uint2(pack_bf16x2(o[0] * inv, o[1] * inv), pack_bf16x2(o[2] * inv, o[3] * inv));
  };
  float M, L;
  f32x4v o;
  if (nsplit <= 8) {
    for (int i = threadIdx.x; i < tasks; i += 64 * W) {
      merge(i, 0, 1, M, L, o);
      store(i, L, o);
    }
    return;
  }
  // many parts by as many groups of threads as there are, then through LDS
  const int groups = max(1, min(W, 64 * W / tasks));
  for (int i = threadIdx.x; i < tasks * groups; i += 64 * W) {
    const int pg = i / tasks, ii = i - pg * tasks;
    merge(ii, pg, groups, M, L, o);
    *(f32x4v*)&part[pg][ii >> 5][(ii & 31) * 4] = o;
    if ((ii & 31) == 0) {
      mls[pg][ii >> 5][0] = M;
      mls[pg][ii >> 5][1] = L;
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < tasks; i += 64 * W) {
    const int hn = i >> 5;
    M = -INFINITY, L = 0.f;
    o = f32x4v{0.f, 0.f, 0.f, 0.f};
    for (int x = 0; x < groups; ++x) M = fmaxf(M, mls[x][hn][0]);
    for (int x = 0; x < groups; ++x) {
      const float l = mls[x][hn][1];
      if (l <= 0.f) continue;
      const float f = __builtin_amdgcn_exp2f(mls[x][hn][0] - M);
      L += f * l;
      o += f * *(const f32x4v*)&part[x][hn][(i & 31) * 4];
    }
    store(i, L, o);
  }
}

template <bool KV8, int W = KV8 ? 4 : 8, bool PIPE = KV8>
__global__ __launch_bounds__(64 * W) __attribute__((amdgpu_waves_per_eu(PIPE ? 2 : 4, PIPE ? 2 : 4))) void paged_wg(AttnArgs a) {
  paged_waves<KV8, W, PIPE, 0>(a);
}

template <bool KV8, int BAL>
__global__ __launch_bounds__(KV8 ? 256 : 512) __attribute__((amdgpu_waves_per_eu(KV8 ? 2 : 4, KV8 ? 2 : 4))) void paged_parts(AttnArgs a) {
  paged_waves<KV8, KV8 ? 4 : 8, KV8, BAL>(a);
}

// merge nsplit partials (m in log2 units, l, unnormalised O) of one (b, h):
// the launch-boundary variant, for batches with many (sequence, KV head)
// groups -- there an in-launch last-arriver merge costs one L2-invalidating
// acquire per group (measured 47 -> 58 us at batch 64 x 1024)
__global__ __launch_bounds__(64) void paged_reduce(const float* __restrict__ po, const float* __restrict__ pml,
                                                   unsigned short* __restrict__ o, int H, int nsplit, long ldo) {
  const int bh = blockIdx.x, lane = threadIdx.x;
  const int b = bh / H, h = bh - b * H;
  const float* ml = pml + (long)bh * nsplit * 2;
  float M = -INFINITY;
  for (int s = 0; s < nsplit; ++s) M = fmaxf(M, ml[2 * s]);
  float L = 0.f, o0 = 0.f, o1 = 0.f;
  // the writer stores O^T in 16-dim tiles: lane's dims d = 2*lane, 2*lane + 1
  const float* pb = po + (long)bh * nsplit * HD + 2 * lane;
#pragma unroll 4
  for (int s = 0; s < nsplit; ++s) {
    const float l = ml[2 * s + 1];
    if (l <= 0.f) continue;
    const float f = __builtin_amdgcn_exp2f(ml[2 * s] - M);
    L += f * l;
    const float2 v = *(const float2*)(pb + (long)s * HD);
    o0 += f * v.x;
    o1 += f * v.y;
  }
  const float inv = L > 0.f ? 1.f / L : 0.f;
  *(unsigned*)(o + (long)b * ldo + (long)h * HD + 2 * lane) = pack_bf16x2(o0 * inv, o1 * inv);
}

}  // namespace dec
}  // namespace kgs

namespace {
inline bool al16(const void* p) { return ((uintptr_t)p & 15) == 0; }

// Tile variants (R = 16-row W tiles per wave, MT = 16-column x tiles, KC =
// k-steps per x chunk). 0 = the measured default for the batch size.
struct SkinnyVariant {
  int r, mt, kc, kin;
};
constexpr SkinnyVariant kVariants[] = {
    {0, 0, 0},                                      // 0: auto
    {1, 1, 16}, {1, 1, 8}, {2, 1, 16},              // 1-3:  M <= 16
    {1, 2, 16}, {1, 2, 8}, {2, 2, 8}, {2, 2, 16},   // 4-7:  M <= 32
    {1, 4, 16}, {1, 4, 4}, {1, 4, 8}, {2, 4, 4}, {2, 4, 8},  // 8-12: M <= 64
    {2, 8, 2}, {2, 8, 4}, {4, 8, 2}, {1, 8, 4},     // 13-16: M <= 128
    {2, 16, 2}, {1, 16, 4}, {1, 16, 2},             // 17-19: M <= 256
    {1, 1, 8, 1}, {2, 1, 8, 1},                     // 20-21: M <= 16, K split inside the workgroup
    {1, 2, 8, 1}, {2, 2, 8, 1},                     // 22-23: M <= 32
    {1, 4, 8, 1}, {2, 4, 8, 1},                     // 24-25: M <= 64
};
constexpr int kNumVariants = sizeof(kVariants) / sizeof(kVariants[0]);

int mt_for(int M) { return M <= 16 ? 1 : M <= 32 ? 2 : M <= 64 ? 4 : M <= 128 ? 8 : 16; }
int default_variant(int mt) { return mt == 1 ? 1 : mt == 2 ? 4 : mt == 4 ? 8 : mt == 8 ? 13 : 17; }

template <int R, int MT, int KC, bool W8, bool KIN = false>
hipError_t launch_skinny(const void* wp, const void* x, void* y, float* ws, int* cnt, int M, int N, int K, long ldx,
                         long ldy, int ksplit, int cps, const kgs::dec::SkinnyEpi& ep, hipStream_t s) {
  using namespace kgs::dec;
  const dim3 grid(N / ((KIN ? 16 : 64) * R) * ksplit);
  auto run = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, dim3(256), 0, s, wp, (const unsigned short*)x, (unsigned short*)y, ws, cnt, M, N, K, ldx, ldy,
                       ksplit, cps, ep);
    return hipGetLastError();
  };
  const bool rope = ep.mode & EPI_ROPE, sums = ep.mode & (EPI_SUMS_IN | EPI_SUMS_OUT);
  if (ep.mode & EPI_OWN) {
    if constexpr (!W8 && MT <= 4) {
      if ((KIN && ksplit != 1) || sums) return hipErrorInvalidValue;
      if constexpr (R == 1) {
        if (rope) return run(skinny<R, MT, KC, false, true, KIN, false, true>);
      }
      if (!rope) return run(skinny<R, MT, KC, false, false, KIN, false, true>);
    }
    return hipErrorInvalidValue;
  }
  if constexpr (!W8 && MT <= 4 && R == 1) {  // the fused layer's qkv variants (kgs/ops/decode.py rope_variant)
    if (rope) return sums ? run(skinny<R, MT, KC, false, true, KIN, true>) : run(skinny<R, MT, KC, false, true, KIN>);
  }
  if (rope) return hipErrorInvalidValue;  // no RoPE instantiation for this variant
  if constexpr (!W8 && MT <= 4) {
    if (sums) return run(skinny<R, MT, KC, false, false, KIN, true>);
  }
  if (sums) return hipErrorInvalidValue;
  return run(skinny<R, MT, KC, W8, false, KIN>);
}
}  // namespace

// Geometry of tile variant `variant` (0 = default) for a batch of M rows:
// rows of W per workgroup strip, k elements per x chunk, padded batch. Lets the
// host size split-K and the workspace (kgs/ops/decode.py). Returns
// KGS_ERR_ARG when the variant does not cover M's column-tile count.
KGS_EXPORT int kgs_skinny_variant_geometry(int variant, int M, int* rows_per_strip, int* k_per_chunk, int* mpad) {
  if (M <= 0 || M > 256) return KGS_ERR_SHAPE;
  const int mt = mt_for(M);
  if (variant == 0) variant = default_variant(mt);
  if (variant < 0 || variant >= kNumVariants || kVariants[variant].mt != mt) return KGS_ERR_ARG;
  *mpad = 16 * mt;
  const int kin = kVariants[variant].kin;
  *rows_per_strip = (kin ? 16 : 64) * kVariants[variant].r;
  *k_per_chunk = (kin ? 4 : 1) * 32 * kVariants[variant].kc;
  return 0;
}

KGS_EXPORT int kgs_skinny_geometry(int M, int* rows_per_strip, int* k_per_chunk, int* mpad) {
  return kgs_skinny_variant_geometry(0, M, rows_per_strip, k_per_chunk, mpad);
}

// y[M, N] (bf16, row stride ldy) = x[M, K] (row stride ldx) . W^T with W
// prepacked ([N/16][K/32][64][8] bf16). ksplit must divide K / k_per_chunk;
// with ksplit > 1, ws holds ksplit * mpad * N floats (OWN: and 2 ksplit * mpad * N / rows_per_strip) and cnt N / rows_per_strip
// zero-initialised ints (left zeroed on return). epi: EPI_* flags (SWIGLU: y is
// [M, N/2]; RMS needs ss_in[M], or OWN; RESID accumulates into y and, unless null, ss_out[M]);
// ss_zero (optional, [M] floats) is cleared at kernel start. With EPI_SUMS_IN ss_in, with EPI_SUMS_OUT
// ss_out and ss_zero hold 64-bit integers [8][M] (16-B aligned), N at most 8192 for ss_out.
namespace {
int skinny_fused(const void* wp, const void* x, void* y, float* ws, int* cnt, int M, int N, int K, long ldx, long ldy,
                 int ksplit, int variant, int epi, const float* ss_in, float* ss_out, float* ss_zero, float inv_k,
                 float eps, const float* wscale, const kgs::dec::SkinnyEpi& rope, hipStream_t s);
}

KGS_EXPORT int kgs_skinny_gemm_bf16_fused(const void* wp, const void* x, void* y, float* ws, int* cnt, int M, int N,
                                         int K, long ldx, long ldy, int ksplit, int variant, int epi,
                                         const float* ss_in, float* ss_out, float* ss_zero, float inv_k, float eps,
                                         const float* wscale, float limit, hipStream_t s) {
  if (epi & kgs::dec::EPI_ROPE) return KGS_ERR_ARG;  // kgs_skinny_gemm_bf16_rope
  kgs::dec::SkinnyEpi ep{};
  ep.limit = limit;
  return skinny_fused(wp, x, y, ws, cnt, M, N, K, ldx, ldy, ksplit, variant, epi, ss_in, ss_out, ss_zero, inv_k, eps,
                      wscale, ep, s);
}

// The fused qkv projection with RoPE + the KV-cache write in its epilogue
// (EPI_ROPE; W packed with kgs/ops/decode.py rope_rows): y [M, (H + 2 HKV) 128]
// gets the rotated q, k and the v rows in the original order, and k / v land
// in the bf16 cache slot slot[m] (< 0: no write). cos / sin: fp32 [max_pos, 64].
// epi may add EPI_RMS (ss_in, inv_k, eps as in kgs_skinny_gemm_bf16_fused).
KGS_EXPORT int kgs_skinny_gemm_bf16_rope(const void* wp, const void* x, void* y, float* ws, int* cnt, int M, int N,
                                        int K, long ldx, long ldy, int ksplit, int variant, int epi,
                                        const float* ss_in, float inv_k, float eps, const float* cosv,
                                        const float* sinv, const int* pos, const int* slot, void* cache, int H,
                                        int HKV, hipStream_t s) {
  using namespace kgs::dec;
  if (epi & ~(EPI_RMS | EPI_SUMS_IN | EPI_OWN)) return KGS_ERR_ARG;
  if (H <= 0 || HKV <= 0 || H % HKV || N != (H + 2 * HKV) * HD) return KGS_ERR_SHAPE;
  if (!cosv || !sinv || !pos || !slot || !al16(cache)) return KGS_ERR_ARG;
  SkinnyEpi r{};
  r.cosv = cosv;
  r.sinv = sinv;
  r.pos = pos;
  r.slot = slot;
  r.cache = (unsigned short*)cache;
  r.H = H;
  r.HKV = HKV;
  return skinny_fused(wp, x, y, ws, cnt, M, N, K, ldx, ldy, ksplit, variant, epi | EPI_ROPE, ss_in, nullptr, nullptr,
                      inv_k, eps, nullptr, r, s);
}

namespace {
int skinny_fused(const void* wp, const void* x, void* y, float* ws, int* cnt, int M, int N, int K, long ldx, long ldy,
                 int ksplit, int variant, int epi, const float* ss_in, float* ss_out, float* ss_zero, float inv_k,
                 float eps, const float* wscale, const kgs::dec::SkinnyEpi& rope, hipStream_t s) {
  using namespace kgs::dec;
  int rps, kpc, mpad;
  const int rc = kgs_skinny_variant_geometry(variant, M, &rps, &kpc, &mpad);
  if (rc) return rc;
  if (variant == 0) variant = default_variant(mt_for(M));
  if (epi & ~(EPI_SWIGLU | EPI_RMS | EPI_RESID | EPI_ROPE | EPI_GELU | EPI_CLAMPED | EPI_SUMS_IN | EPI_SUMS_OUT | EPI_OWN) ||
      ((epi & (EPI_GELU | EPI_CLAMPED)) && !(epi & EPI_SWIGLU)) || ((epi & EPI_SWIGLU) && (epi & EPI_RESID)))
    return KGS_ERR_ARG;
  if ((epi & EPI_ROPE) && (rope.cache == nullptr || (epi & (EPI_SWIGLU | EPI_RESID)) || wscale != nullptr))
    return KGS_ERR_ARG;
  if ((epi & EPI_RMS) && !(epi & EPI_OWN) && ss_in == nullptr) return KGS_ERR_ARG;
  if ((epi & EPI_OWN) && (!(epi & EPI_RMS) || (epi & (EPI_RESID | EPI_SUMS_IN | EPI_SUMS_OUT)) || M > 64 || wscale)) return KGS_ERR_ARG;
  if ((epi & EPI_SUMS_OUT) && (epi & EPI_RESID) && ss_out == nullptr) return KGS_ERR_ARG;
  if (N <= 0 || K <= 0 || N % rps || K % kpc || ldx < K || ldy < ((epi & EPI_SWIGLU) ? N / 2 : N))
    return KGS_ERR_SHAPE;
  if ((epi & EPI_RESID) && (epi & EPI_SUMS_OUT) && N > SUM_MAX_N) return KGS_ERR_SHAPE;
  if (((epi & EPI_SUMS_IN) && !al16(ss_in)) || ((epi & EPI_SUMS_OUT) && (!al16(ss_out) || !al16(ss_zero)))) return KGS_ERR_ALIGN;
  const int nchunks = K / kpc;
  if (ksplit <= 0 || nchunks % ksplit) return KGS_ERR_ARG;
  if (ksplit > 1 && (ws == nullptr || cnt == nullptr)) return KGS_ERR_ARG;
  if (!al16(wp) || !al16(x) || ((uintptr_t)y & 7) || ((uintptr_t)ws & 15) || ldx % 8 || ldy % 4) return KGS_ERR_ALIGN;
  const int cps = nchunks / ksplit;
  SkinnyEpi ep = rope;
  ep.mode = epi;
  ep.ss_in = ss_in;
  ep.ss_out = ss_out;
  ep.ss_zero = ss_zero;
  ep.zero_words = (epi & EPI_SUMS_OUT) ? 2 * SUM_WORDS * M : M;
  ep.inv_k = inv_k;
  ep.eps = eps;
  ep.wscale = wscale;
  const bool w8 = wscale != nullptr;
  if (w8 && variant > 12 && variant < 20) return KGS_ERR_ARG;  // fp8 weights: batch buckets <= 64
  switch (variant * 2 + (w8 ? 1 : 0)) {
#define KGS_SKV(id, R, MT, KC)                                                                                       \
  case 2 * id: return (int)launch_skinny<R, MT, KC, false>(wp, x, y, ws, cnt, M, N, K, ldx, ldy, ksplit, cps, ep, s); \
  case 2 * id + 1:                                                                                                    \
    if constexpr (id <= 12) return (int)launch_skinny<R, MT, KC, true>(wp, x, y, ws, cnt, M, N, K, ldx, ldy, ksplit,  \
                                                                        cps, ep, s);                                  \
    return KGS_ERR_ARG;
    KGS_SKV(1, 1, 1, 16) KGS_SKV(2, 1, 1, 8) KGS_SKV(3, 2, 1, 16)
    KGS_SKV(4, 1, 2, 16) KGS_SKV(5, 1, 2, 8) KGS_SKV(6, 2, 2, 8) KGS_SKV(7, 2, 2, 16)
    KGS_SKV(8, 1, 4, 16) KGS_SKV(9, 1, 4, 4) KGS_SKV(10, 1, 4, 8) KGS_SKV(11, 2, 4, 4) KGS_SKV(12, 2, 4, 8)
    KGS_SKV(13, 2, 8, 2) KGS_SKV(14, 2, 8, 4) KGS_SKV(15, 4, 8, 2) KGS_SKV(16, 1, 8, 4)
    KGS_SKV(17, 2, 16, 2) KGS_SKV(18, 1, 16, 4) KGS_SKV(19, 1, 16, 2)
#undef KGS_SKV
    case 2 * 20: return (int)launch_skinny<1, 1, 8, false, true>(wp, x, y, ws, cnt, M, N, K, ldx, ldy, ksplit, cps, ep, s);
    case 2 * 20 + 1: return (int)launch_skinny<1, 1, 8, true, true>(wp, x, y, ws, cnt, M, N, K, ldx, ldy, ksplit, cps, ep, s);
    case 2 * 21: return (int)launch_skinny<2, 1, 8, false, true>(wp, x, y, ws, cnt, M, N, K, ldx, ldy, ksplit, cps, ep, s);
    case 2 * 21 + 1: return (int)launch_skinny<2, 1, 8, true, true>(wp, x, y, ws, cnt, M, N, K, ldx, ldy, ksplit, cps, ep, s);
    case 2 * 22: return (int)launch_skinny<1, 2, 8, false, true>(wp, x, y, ws, cnt, M, N, K, ldx, ldy, ksplit, cps, ep, s);
    case 2 * 22 + 1: return (int)launch_skinny<1, 2, 8, true, true>(wp, x, y, ws, cnt, M, N, K, ldx, ldy, ksplit, cps, ep, s);
    case 2 * 23: return (int)launch_skinny<2, 2, 8, false, true>(wp, x, y, ws, cnt, M, N, K, ldx, ldy, ksplit, cps, ep, s);
    case 2 * 23 + 1: return (int)launch_skinny<2, 2, 8, true, true>(wp, x, y, ws, cnt, M, N, K, ldx, ldy, ksplit, cps, ep, s);
    case 2 * 24: return (int)launch_skinny<1, 4, 8, false, true>(wp, x, y, ws, cnt, M, N, K, ldx, ldy, ksplit, cps, ep, s);
    case 2 * 24 + 1: return (int)launch_skinny<1, 4, 8, true, true>(wp, x, y, ws, cnt, M, N, K, ldx, ldy, ksplit, cps, ep, s);
    case 2 * 25: return (int)launch_skinny<2, 4, 8, false, true>(wp, x, y, ws, cnt, M, N, K, ldx, ldy, ksplit, cps, ep, s);
    case 2 * 25 + 1: return (int)launch_skinny<2, 4, 8, true, true>(wp, x, y, ws, cnt, M, N, K, ldx, ldy, ksplit, cps, ep, s);
    default: return KGS_ERR_ARG;
  }
}
}  // namespace

KGS_EXPORT int kgs_skinny_gemm_bf16_ex(const void* wp, const void* x, void* y, float* ws, int* cnt, int M, int N,
                                      int K, long ldx, long ldy, int ksplit, int variant, int epi, hipStream_t s) {
  return kgs_skinny_gemm_bf16_fused(wp, x, y, ws, cnt, M, N, K, ldx, ldy, ksplit, variant, epi, nullptr, nullptr,
                                    nullptr, 0.f, 0.f, nullptr, 0.f, s);
}

KGS_EXPORT int kgs_skinny_gemm_bf16_v(const void* wp, const void* x, void* y, float* ws, int* cnt, int M, int N, int K,
                                     long ldx, long ldy, int ksplit, int variant, hipStream_t s) {
  return kgs_skinny_gemm_bf16_ex(wp, x, y, ws, cnt, M, N, K, ldx, ldy, ksplit, variant, 0, s);
}

KGS_EXPORT int kgs_skinny_gemm_bf16(const void* wp, const void* x, void* y, float* ws, int* cnt, int M, int N, int K,
                                   long ldx, long ldy, int ksplit, hipStream_t s) {
  return kgs_skinny_gemm_bf16_v(wp, x, y, ws, cnt, M, N, K, ldx, ldy, ksplit, 0, s);
}

// qkv: [tokens, ld] fused projection rows (H q heads, HKV k heads, HKV v heads
// of 128); pos/slot: int32 [tokens]; cache: this layer's pages
// [pages][HKV][2][4096] bf16. q and k are rotated in place; k, v land in the cache.
// kv8: the cache holds e4m3 bytes ([pages][HKV][2][4096] B) instead of bf16.
// P != nullptr: the projection is given as nslice fp32 split-K partials
// [nslice][prows][(H + 2 HKV) * hd] instead of in qkv (prows: its rows, tokens without a map); the reduced, rotated
// rows are written to qkv (which is then output only).
// rows != nullptr: token t is row rows[t] of qkv, none where negative: prompts padded
// to whole pages whose padding has no rows, so that a page's run still leaves in 16-byte chunks.
KGS_EXPORT int kgs_rope_cache_bf16(void* qkv, const float* cosv, const float* sinv, const int* pos, const int* slot,
                                  void* cache, long tokens, int H, int HKV, int hd, long ld, int kv8, const float* P,
                                  int nslice, const int* rows, long prows, hipStream_t s) {
  if (tokens < 0 || H <= 0 || HKV <= 0 || H % HKV || hd != kgs::dec::HD) return KGS_ERR_SHAPE;
  if (ld < (long)(H + 2 * HKV) * hd) return KGS_ERR_SHAPE;
  if (!al16(qkv) || !al16(cosv) || !al16(sinv) || !al16(cache) || ld % 8) return KGS_ERR_ALIGN;
  if (P != nullptr && (nslice <= 0 || !al16(P) || prows <= 0 || (!rows && prows != tokens))) return KGS_ERR_ARG;
  const long n = tokens * (H + 2 * HKV) * 8;
  if (n == 0) return 0;
  // small grids: a wave per workgroup, so that every CU takes part (us of 256 / 64 threads, 24 heads, 8 slices: 40 tokens 3.9 / 3.2,
  // 128 4.5 / 3.9; 48 heads: 90 5.05 / 4.6, 30 without slices 3.2 / 2.9; two slices up to 24k threads only: 80 heads 51 tokens 3.4 / 3.7,
  // 48 150 5.1 / 5.5)
  const int wg = n <= (P != nullptr && nslice == 2 ? 96 : 256) * 256 ? 64 : 256;
  const dim3 g((unsigned)((n + wg - 1) / wg)), b(wg);
  auto q = (unsigned short*)qkv;
  if (P != nullptr) {
#define KGS_RCS(KV, NSL)                                                                                           \
  hipLaunchKernelGGL((kgs::dec::rope_cache<KV, true, NSL>), g, b, 0, s, q, cosv, sinv, pos, slot, cache, tokens, H, \
                     HKV, ld, P, nslice, rows, prows)
#define KGS_RCS_KV(KV)                \
  switch (nslice) {                   \
    case 2: KGS_RCS(KV, 2); break;    \
    case 4: KGS_RCS(KV, 4); break;    \
    case 8: KGS_RCS(KV, 8); break;    \
    case 16: KGS_RCS(KV, 16); break;  \
    default: KGS_RCS(KV, 0); break;   \
  }
    if (kv8) {
      KGS_RCS_KV(true);
    } else {
      KGS_RCS_KV(false);
    }
#undef KGS_RCS_KV
#undef KGS_RCS
  } else if ((H + 2 * HKV) % 8 == 0 && !kv8 && tokens >= 1024) {
    // prompt-sized: the v heads go through the page-run writer
    const dim3 g8((unsigned)((n / 8 + 255) / 256));
    hipLaunchKernelGGL((kgs::dec::rope_cache_g8<false, true>), g8, dim3(256), 0, s, q, cosv, sinv, pos, slot, cache, tokens, H,
                       HKV, ld, rows);
    const dim3 gv((unsigned)((tokens + kgs::dec::PAGE - 1) / kgs::dec::PAGE), (unsigned)HKV);
    hipLaunchKernelGGL(kgs::dec::v_cache_pages, gv, dim3(256), 0, s, (const unsigned short*)q, slot, (unsigned short*)cache,
                       tokens, H, HKV, ld, rows);
  } else if ((H + 2 * HKV) % 8 == 0 && n > 2 * 256 * 256) {
    // more than two workgroups of the per-head form on every CU: eight heads a thread share the
    // cos / sin loads; below, their serial work is what takes the time (24 heads, us of
    // per-head / eight-head: 8 tokens 3.6 / 5.9, 100 4.1 / 6.9, 512 7.0 / 8.3, 1000 10.2 / 10.0)
    const dim3 g8((unsigned)((n / 8 + 255) / 256));
    if (kv8)
      hipLaunchKernelGGL(kgs::dec::rope_cache_g8<true>, g8, dim3(256), 0, s, q, cosv, sinv, pos, slot, cache, tokens, H, HKV,
                         ld, rows);
    else
      hipLaunchKernelGGL(kgs::dec::rope_cache_g8<false>, g8, dim3(256), 0, s, q, cosv, sinv, pos, slot, cache, tokens, H, HKV,
                         ld, rows);
  } else if (kv8) {
    hipLaunchKernelGGL(kgs::dec::rope_cache<true>, g, b, 0, s, q, cosv, sinv, pos, slot, cache, tokens, H, HKV, ld,
                       nullptr, 0, rows);
  } else {
    hipLaunchKernelGGL(kgs::dec::rope_cache<false>, g, b, 0, s, q, cosv, sinv, pos, slot, cache, tokens, H, HKV, ld,
                       nullptr, 0, rows);
  }
  return (int)hipGetLastError();
}

// kgs_rope_cache_bf16 of the partials (1 to 16, a power of two) of a weight packed with rope_rows, on rows of the raw residual stream
// with sums of squares sq [tokens]: scaled by their RMSNorm, over inv_k^-1 columns. bf16 pages.
KGS_EXPORT int kgs_rope_cache_packed_bf16(void* qkv, const float* cosv, const float* sinv, const int* pos, const int* slot, void* cache,
                                         long tokens, int H, int HKV, long ld, const float* P, int nslice, const float* sq,
                                         float inv_k, float eps, hipStream_t s) {
  if (tokens < 0 || H <= 0 || HKV <= 0 || H % HKV || ld < (long)(H + 2 * HKV) * kgs::dec::HD) return KGS_ERR_SHAPE;
  if (!al16(qkv) || !al16(cosv) || !al16(sinv) || !al16(cache) || !al16(P) || ld % 8) return KGS_ERR_ALIGN;
  if (!P || !sq || !pos || !slot) return KGS_ERR_ARG;
  const long n = tokens * (H + 2 * HKV) * 8;
  if (n == 0) return 0;
  const int wg = n <= (nslice == 2 ? 96 : 256) * 256 ? 64 : 256;  // as kgs_rope_cache_bf16
  const dim3 g((unsigned)((n + wg - 1) / wg)), b(wg);
#define KGS_RCP(NSL)                                                                                                                  \
  hipLaunchKernelGGL((kgs::dec::rope_cache<false, true, NSL, true>), g, b, 0, s, (unsigned short*)qkv, cosv, sinv, pos, slot, cache, \
                     tokens, H, HKV, ld, P, nslice, nullptr, tokens, sq, inv_k, eps)
  switch (nslice) {
    case 1: KGS_RCP(1); break;
    case 2: KGS_RCP(2); break;
    case 4: KGS_RCP(4); break;
    case 8: KGS_RCP(8); break;
    case 16: KGS_RCP(16); break;
    default: return KGS_ERR_ARG;
  }
#undef KGS_RCP
  return (int)hipGetLastError();
}

// Paged decode attention for one new query token per sequence. q: [B, ldq]
// (query heads at 128-element blocks); cache: layer base; block_tables
// [B, max_pages] int32; ctx_lens [B] int32 (>= 1). nsplit > 1 needs po
// (B*H*nsplit*128 f32), pml (B*H*nsplit*2 f32) and cnt (B*HKV zeroed ints, left
// zeroed); the splits are merged in the same launch.
KGS_EXPORT int kgs_paged_decode_bf16_ex(const void* q, const void* cache, const int* block_tables,
                                       const int* ctx_lens, void* o, float* po, float* pml, int* cnt, int B, int H,
                                       int HKV, int hd, int max_pages, int pages_per_split, int nsplit, long ldq,
                                       long ldo, float scale, int kv8, int pipe_mode, hipStream_t s);

KGS_EXPORT int kgs_paged_decode_bf16(const void* q, const void* cache, const int* block_tables, const int* ctx_lens,
                                    void* o, float* po, float* pml, int* cnt, int B, int H, int HKV, int hd,
                                    int max_pages, int pages_per_split, int nsplit, long ldq, long ldo, float scale,
                                    int kv8, hipStream_t s) {
  return kgs_paged_decode_bf16_ex(q, cache, block_tables, ctx_lens, o, po, pml, cnt, B, H, HKV, hd, max_pages,
                                  pages_per_split, nsplit, ldq, ldo, scale, kv8, -1, s);
}

// pipe_mode: -1 = automatic (the two-page register pipeline for small grids),
// 0 / 1 = force it off / on (measurement)
KGS_EXPORT int kgs_paged_decode_bf16_ex(const void* q, const void* cache, const int* block_tables,
                                       const int* ctx_lens, void* o, float* po, float* pml, int* cnt, int B, int H,
                                       int HKV, int hd, int max_pages, int pages_per_split, int nsplit, long ldq,
                                       long ldo, float scale, int kv8, int pipe_mode, hipStream_t s) {
  using namespace kgs::dec;
  if (B <= 0 || H <= 0 || HKV <= 0 || H % HKV || H / HKV > 16 || hd != HD) return KGS_ERR_SHAPE;
  if (max_pages <= 0 || pages_per_split <= 0 || nsplit <= 0) return KGS_ERR_SHAPE;
  if ((long)pages_per_split * nsplit < max_pages) return KGS_ERR_ARG;
  if (ldq < (long)H * HD || ldo < (long)H * HD) return KGS_ERR_SHAPE;
  if (!al16(q) || !al16(cache) || !al16(o) || ldq % 8 || ldo % 8) return KGS_ERR_ALIGN;
  if (nsplit > 1 && (po == nullptr || pml == nullptr || !al16(po))) return KGS_ERR_ARG;
  const long nwg = (long)B * HKV * nsplit;
  if (nwg > 0x7fffffff) return KGS_ERR_SHAPE;
  // in-launch merge only when there are few (sequence, KV head) groups: it saves
  // the reduce launch but costs each group's last split an acquire
  const int merge = nsplit > 1 && cnt != nullptr && (long)B * HKV <= 32;
  AttnArgs a{(const unsigned short*)q, (const unsigned short*)cache, block_tables, ctx_lens, (unsigned short*)o, po,
             pml, cnt, ldq, ldo, B, H, HKV, max_pages, pages_per_split, nsplit, merge, scale * 1.4426950408889634f,
             nullptr, 0, nullptr, nullptr, nullptr, nullptr, nullptr};
  // up to 4 waves per CU (1024 on the chip) other waves cannot hide a page's
  // latency: pipeline inside the wave there. Round 3 measured the pipeline at
  // 1.2-1.9x for 512-1024-wave grids (batch 64-128 at 528-2000 cached
  // tokens) and +-2 % at 2048 waves (profiles/r3/decode/paged_sweep_ctx*.log)
  const bool pipe = pipe_mode < 0 ? nwg <= 1024 : pipe_mode != 0;
  if (kv8) {
    if (pipe) hipLaunchKernelGGL((paged_decode<true, true>), dim3((unsigned)nwg), dim3(64), 0, s, a);
    else hipLaunchKernelGGL((paged_decode<true, false>), dim3((unsigned)nwg), dim3(64), 0, s, a);
  } else {
    if (pipe) hipLaunchKernelGGL((paged_decode<false, true>), dim3((unsigned)nwg), dim3(64), 0, s, a);
    else hipLaunchKernelGGL((paged_decode<false, false>), dim3((unsigned)nwg), dim3(64), 0, s, a);
  }
  if (nsplit > 1 && !merge)
    hipLaunchKernelGGL(paged_reduce, dim3((unsigned)(B * H)), dim3(64), 0, s, po, pml, (unsigned short*)o, H, nsplit,
                       ldo);
  return (int)hipGetLastError();
}

// Paged decode attention by workgroups of `waves` waves (bf16 pages 2, 4 or 8, e4m3 pages 2 or 4), nsplit equal parts
// of every sequence's pages (paged_wg). Arguments as kgs_paged_decode_bf16; nsplit > 1 needs po, pml and cnt, and
// merges in the same launch.
KGS_EXPORT int kgs_paged_decode_wg_ex(const void* q, const void* cache, const int* block_tables, const int* ctx_lens, void* o,
                                      float* po, float* pml, int* cnt, int B, int H, int HKV, int hd, int max_pages,
                                      int nsplit, long ldq, long ldo, float scale, int kv8, int waves, hipStream_t s) {
  using namespace kgs::dec;
  if (B <= 0 || H <= 0 || HKV <= 0 || H % HKV || H / HKV > 16 || hd != HD || max_pages <= 0 || nsplit <= 0) return KGS_ERR_SHAPE;
  if (ldq < (long)H * HD || ldo < (long)H * HD) return KGS_ERR_SHAPE;
  if (!al16(q) || !al16(cache) || !al16(o) || ldq % 8 || ldo % 8) return KGS_ERR_ALIGN;
  if (nsplit > 1 && (!po || !pml || !cnt || !al16(po))) return KGS_ERR_ARG;
  const long nwg = (long)B * HKV * nsplit;
  if (nwg > 0x7fffffff || (long)B * H * nsplit * HD * 4 > 0xffffffffL) return KGS_ERR_SHAPE;
  AttnArgs a{(const unsigned short*)q, (const unsigned short*)cache, block_tables, ctx_lens, (unsigned short*)o, po,
             pml, cnt, ldq, ldo, B, H, HKV, max_pages, 0, nsplit, 1, scale * 1.4426950408889634f,
             nullptr, 0, nullptr, nullptr, nullptr, nullptr, nullptr};
  auto fn = kv8 ? (waves == 4 ? paged_wg<true> : waves == 2 ? paged_wg<true, 2> : nullptr)
                : (waves == 8 ? paged_wg<false> : waves == 4 ? paged_wg<false, 4> : waves == 2 ? paged_wg<false, 2> : nullptr);
  if (!fn) return KGS_ERR_ARG;
  hipLaunchKernelGGL(fn, dim3((unsigned)nwg), dim3(64 * waves), 0, s, a);
  return (int)hipGetLastError();
}

// The same with parts by the sequences' lengths (paged_parts): at most 128 sequences, 8 (e4m3: 4) waves; po and pml hold
// B + target rows of H heads.
KGS_EXPORT int kgs_paged_decode_wg_bal(const void* q, const void* cache, const int* block_tables, const int* ctx_lens, void* o,
                                       float* po, float* pml, int* cnt, int B, int H, int HKV, int hd, int max_pages, int target,
                                       int least, long ldq, long ldo, float scale, int kv8, hipStream_t s) {
  using namespace kgs::dec;
  if (B <= 0 || B > 128 || H <= 0 || HKV <= 0 || H % HKV || H / HKV > 16 || hd != HD || max_pages <= 0) return KGS_ERR_SHAPE;
  if (target <= 0 || target > 1 << 16 || least <= 0 || max_pages > 1 << 22) return KGS_ERR_SHAPE;
  if (ldq < (long)H * HD || ldo < (long)H * HD) return KGS_ERR_SHAPE;
  if (!al16(q) || !al16(cache) || !al16(o) || ldq % 8 || ldo % 8) return KGS_ERR_ALIGN;
  if (!po || !pml || !cnt || !al16(po)) return KGS_ERR_ARG;
  // parts of at most P pages: sum of ceil(pages / P) <= B + total / P <= B + target
  const int units = B + target;
  if ((long)units * HKV > 0x7fffffff || (long)units * H * HD * 4 > 0xffffffffL) return KGS_ERR_SHAPE;
  AttnArgs a{(const unsigned short*)q, (const unsigned short*)cache, block_tables, ctx_lens, (unsigned short*)o, po,
             pml, cnt, ldq, ldo, B, H, HKV, max_pages, 0, 1, 1, scale * 1.4426950408889634f,
             nullptr, 0, nullptr, nullptr, nullptr, nullptr, nullptr, target, least, units};
  auto fn = kv8 ? (B > 64 ? paged_parts<true, 2> : paged_parts<true, 1>)
                : (B > 64 ? paged_parts<false, 2> : paged_parts<false, 1>);
  hipLaunchKernelGGL(fn, dim3((unsigned)(units * HKV)), dim3(kv8 ? 256 : 512), 0, s, a);
  return (int)hipGetLastError();
}

KGS_EXPORT int kgs_paged_decode_wg(const void* q, const void* cache, const int* block_tables, const int* ctx_lens, void* o,
                                   float* po, float* pml, int* cnt, int B, int H, int HKV, int hd, int max_pages,
                                   int nsplit, long ldq, long ldo, float scale, int kv8, hipStream_t s) {
  return kgs_paged_decode_wg_ex(q, cache, block_tables, ctx_lens, o, po, pml, cnt, B, H, HKV, hd, max_pages, nsplit, ldq, ldo,
                                scale, kv8, kv8 ? 4 : 8, s);
}

// Rows 0 .. rows - 1 of a sequence's cached keys and values, row-major with rows ld apart (16-B
// aligned): the first ctx from its pages (int32, at least ceil(ctx / 32) of them), the others zero.
KGS_EXPORT int kgs_gather_kv(const void* cache, const int* pages, void* k, void* v, int ctx, int rows, int HKV, int hd, int npages,
                             long ld, int kv8, hipStream_t s) {
  using namespace kgs::dec;
  if (ctx < 0 || rows < ctx || rows <= 0 || npages <= 0 || HKV <= 0 || HKV > 65535 || hd != HD || ld < (long)HKV * HD) return KGS_ERR_SHAPE;
  if (!al16(cache) || !al16(k) || !al16(v) || ld % 8) return KGS_ERR_ALIGN;
  const dim3 grid((unsigned)((rows + PAGE - 1) / PAGE), (unsigned)HKV);
  auto ko = (unsigned short*)k;
  auto vo = (unsigned short*)v;
  if (kv8) hipLaunchKernelGGL(gather_kv<true>, grid, dim3(256), 0, s, cache, pages, ko, vo, ctx, rows, HKV, npages, ld);
  else hipLaunchKernelGGL(gather_kv<false>, grid, dim3(256), 0, s, cache, pages, ko, vo, ctx, rows, HKV, npages, ld);
  return (int)hipGetLastError();
}

// rope_cache + paged decode attention in one launch: the fused qkv projection
// arrives as nslice fp32 split-K partials P [nslice][B][(H + 2 HKV) * 128]
// (gemm_nt_w4x_partials); each attention wave reduces, rotates and caches its
// own (sequence, KV head) rows (paged_decode RP) -- the same bits as
// kgs_rope_cache_bf16(P) followed by kgs_paged_decode_bf16 on the rotated q.
// slot[b]: the new token's cache slot; its page must be the last one of
// ctx_lens[b] in block_tables (as the engine assigns it).
KGS_EXPORT int kgs_paged_decode_rope_bf16(const float* P, int nslice, const float* cosv, const float* sinv,
                                         const int* pos, const int* slot, void* cache, const int* block_tables,
                                         const int* ctx_lens, void* o, float* po, float* pml, int* cnt, int B, int H,
                                         int HKV, int hd, int max_pages, int pages_per_split, int nsplit, long ldo,
                                         float scale, int kv8, int pipe_mode, hipStream_t s) {
  using namespace kgs::dec;
  if (B <= 0 || H <= 0 || HKV <= 0 || H % HKV || H / HKV > 6 || hd != HD) return KGS_ERR_SHAPE;
  if (max_pages <= 0 || pages_per_split <= 0 || nsplit <= 0) return KGS_ERR_SHAPE;
  if (nslice != 2 && nslice != 4 && nslice != 8) return KGS_ERR_ARG;  // compile-time slice counts
  if ((long)pages_per_split * nsplit < max_pages) return KGS_ERR_ARG;
  if (ldo < (long)H * HD || ldo % 8) return KGS_ERR_SHAPE;
  if (P == nullptr || pos == nullptr || slot == nullptr) return KGS_ERR_ARG;
  if (!al16(P) || !al16(cosv) || !al16(sinv) || !al16(cache) || !al16(o)) return KGS_ERR_ALIGN;
  if (nsplit > 1 && (po == nullptr || pml == nullptr || !al16(po))) return KGS_ERR_ARG;
  const long nwg = (long)B * HKV * nsplit;
  if (nwg > 0x7fffffff) return KGS_ERR_SHAPE;
  const int merge = nsplit > 1 && cnt != nullptr && (long)B * HKV <= 32;
  AttnArgs a{nullptr, (const unsigned short*)cache, block_tables, ctx_lens, (unsigned short*)o, po, pml, cnt, 0, ldo,
             B, H, HKV, max_pages, pages_per_split, nsplit, merge, scale * 1.4426950408889634f,
             P, nslice, cosv, sinv, pos, slot, cache};
  const bool pipe = pipe_mode < 0 ? nwg <= 1024 : pipe_mode != 0;
#define KGS_PDR(KV, PP, NS) hipLaunchKernelGGL((paged_decode<KV, PP, NS>), dim3((unsigned)nwg), dim3(64), 0, s, a)
#define KGS_PDR_NS(KV, PP)         \
  switch (nslice) {                \
    case 2: KGS_PDR(KV, PP, 2); break; \
    case 4: KGS_PDR(KV, PP, 4); break; \
    default: KGS_PDR(KV, PP, 8); break; \
  }
  if (kv8) {
    if (pipe) { KGS_PDR_NS(true, true); } else { KGS_PDR_NS(true, false); }
  } else {
    if (pipe) { KGS_PDR_NS(false, true); } else { KGS_PDR_NS(false, false); }
  }
#undef KGS_PDR_NS
#undef KGS_PDR
  if (nsplit > 1 && !merge)
    hipLaunchKernelGGL(paged_reduce, dim3((unsigned)(B * H)), dim3(64), 0, s, po, pml, (unsigned short*)o, H, nsplit,
                       ldo);
  return (int)hipGetLastError();
}
