// Skinny products of up to 16 rows (plain ones 32): y[M, N] = x[M, K] . W^T, W packed as for decode.hip's skinny
// ([N/16][K/32][64][8]), with that kernel's epilogues and one statistic of its own.
//
// A workgroup of NW waves takes R 16-row tiles of W; the waves share out K, stream their part of W and of x (in
// MFMA operand order, straight from memory) through a ring of PF k-steps and add their sums in LDS, in the order of the waves.
// Loads are buffer loads, so that a step waits for exactly its own.
//
// OWN: the RMSNorm of x from x itself. Every wave holds its part of all rows anyway and adds up its squares (add_squares). Where the producer of x adds them up instead, 256 workgroups' atomics
// meet on one address, 12.5 ns each, at the end of a launch that nothing hides: a layer's o and down took 1.6 us longer at 1
// row, 2.0 at 16. Nothing here depends on the order in which workgroups arrive.
//
// Bound by memory where W is large (28672 x 4096 at 1 row 39 us, 6.0 TB/s), else by the launch and one trip through
// memory, the ring and LDS (4096 x 4096 7.8 us). The split by the number of strips (few_split): short grids need the waves,
// long ones lose by them (us at 1 row with 8 / 4 / 2 waves: 2048x8192 9.1 / 12.5 / 11.5, 4096x14336 20.8 / 21.1 / 22.7, 6144x4096 11.9 /
// 10.2 / 10.2, 28672x4096 42.0 / 40.6 / 39.8, 32000x4096 48.3 / 45.9 / 44.5). Two tiles a workgroup from 5 rows on where one makes
// a little more than one round of the CUs: every workgroup reads all of x (6144x4096 at 12 rows 12.7 / 12.1). Any K of 64, for products that
// were the library's: us at 1 / 32 rows, library / here: 2048x128 3.3, 3.8 / 2.1, 2.5; 2048x768 5.0, 6.8 / 2.8, 5.3; 832x2048 7.9 / 3.6 at 1 row. From 17
// rows on the way of x bounds K (kgs/ops/decode.py few_route).
#include "decode_common.h"

#include <type_traits>

namespace kgs {
namespace dec {

struct FewArgs {
  const unsigned short* x;
  const unsigned short* w;
  unsigned short* y;
  int M, N, K, ldx;
  long ldy;
  int mode;
  float inv_k, eps, limit;
  const float* cosv;
  const float* sinv;
  const int* pos;
  const int* slot;
  unsigned short* cache;
  int H, HKV;
  // a second product of the same sizes (the grid's y), plain ones only
  const unsigned short* x2;
  const unsigned short* w2;
  unsigned short* y2;
};

template <int AUX>
__device__ __forceinline__ bf16x8 ld_frag(__amdgpu_buffer_rsrc_t r, int v, int s) {
  return __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(r, v, s, AUX));
}

// MT column tiles of 16 rows of x; ROPE and OWN of one
template <int R, int MT, int NW, int PF, bool ROPE, bool OWN>
__global__ __launch_bounds__(64 * NW) void few(FewArgs a) {
  static_assert(MT == 1 || (!ROPE && !OWN && R == 1));
  __shared__ __attribute__((aligned(16))) f32x4v red[NW * R * MT * 64];
  __shared__ double stat[OWN ? NW : 1][16];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), fr = lane & 15, fq = lane >> 4;
  const int M = a.M, nkk = a.K / 32, nsteps = nkk / NW, kk0 = w * nsteps, nt0 = blockIdx.x * R;
  if constexpr (!ROPE && !OWN) {
    if (blockIdx.y) {
      a.x = a.x2;
      a.w = a.w2;
      a.y = a.y2;
    }
  }
  const auto rw = rsrc(a.w + (long)nt0 * nkk * 512, (unsigned)(R * nkk * 1024));
  const auto rx = rsrc(a.x, (unsigned)(((M - 1) * a.ldx + a.K) * 2));
  const int wo = lane * 16;
  int xo[MT];
#pragma unroll
  for (int c = 0; c < MT; ++c) xo[c] = 2 * (min(16 * c + fr, M - 1) * a.ldx + fq * 8);  // rows from M on repeat the last one: never stored
  bf16x8 wf[PF][R], xf[PF][MT];
  auto load = [&](int p, int s) {  // k-step s of this wave; W past the caches, it comes once
#pragma unroll
    for (int r = 0; r < R; ++r) wf[p][r] = ld_frag<2>(rw, wo, (r * nkk + kk0 + s) * 1024);
#pragma unroll
    for (int c = 0; c < MT; ++c) xf[p][c] = ld_frag<0>(rx, xo[c], (kk0 + s) * 64);
  };
#pragma unroll
  for (int p = 0; p < PF; ++p) load(p, p);

  // what the epilogue needs, under the main loop's way: old values or rotation of tile (r, c) = (w / MT, w % MT)
  const int nt = nt0 + (w < R * MT ? w / MT : 0), m = 16 * (w % MT) + fr;
  unsigned short* const yt = a.y + (long)min(m, M - 1) * a.ldy + 16 * nt + 4 * fq;
  uint2 old = make_uint2(0, 0);
  if (!ROPE && (a.mode & EPI_RESID) && w < R * MT) old = *(const uint2*)yt;
  float cs[4], sn[4];
  int slot = -1;
  if constexpr (ROPE) {
    const int mr = min(fr, M - 1), p = a.pos[mr], t = nt & 7, dd = 8 * t + 4 * (fq & 1);  // dim within the rotated half
    slot = fr < M ? a.slot[mr] : -1;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      cs[i] = a.cosv[(long)p * (HD / 2) + dd + i];
      sn[i] = a.sinv[(long)p * (HD / 2) + dd + i];
    }
  }

  f32x4v acc[R][MT];
  [[maybe_unused]] double own = 0.;
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int c = 0; c < MT; ++c) acc[r][c] = f32x4v{0.f, 0.f, 0.f, 0.f};
  for (int s0 = 0; s0 < nsteps; s0 += PF) {
    const int next = min(s0 + PF, nsteps - PF);  // past the end: the last round again, from the caches
#pragma unroll
    for (int p = 0; p < PF; ++p) {
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int r = 0; r < R; ++r)
#pragma unroll
        for (int c = 0; c < MT; ++c) acc[r][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[p][r], xf[p][c], acc[r][c], 0, 0, 0);
      if constexpr (OWN) own = add_squares(own, xf[p][0]);
      load(p, next + p);
    }
  }
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int c = 0; c < MT; ++c) red[((w * R + r) * MT + c) * 64 + lane] = acc[r][c];
  if constexpr (OWN) {
    own = wsum16(own);
    if (fq == 0) stat[w][fr] = own;
  }
  __syncthreads();
  if (w >= R * MT) return;

  // lane: row m of x, rows 16 nt + 4 fq + i of W
  f32x4v v = red[w * 64 + lane];
#pragma unroll
  for (int j = 1; j < NW; ++j) v += red[(j * R * MT + w) * 64 + lane];
  if constexpr (OWN) {
    double ss = stat[0][fr];
#pragma unroll
    for (int j = 1; j < NW; ++j) ss += stat[j][fr];
    v *= rsqrtf((float)ss * a.inv_k + a.eps);
  }
  const bool in = m < M;
  if constexpr (ROPE) {
    const int hh = nt >> 3, t = nt & 7;  // head and tile within it
    const bool rot = hh < a.H + a.HKV;
    f32x4v vb, pb;  // this lane's and its partner's (lane ^ 32) values, rounded to bf16
#pragma unroll
    for (int i = 0; i < 4; ++i) vb[i] = bf2f(f2bf(v[i]));
#pragma unroll
    for (int i = 0; i < 4; ++i) pb[i] = lane_xor32(vb[i]);
    if (!in) return;
    const int d0 = rot ? (fq < 2 ? 8 * t + 4 * fq : 64 + 8 * t + 4 * (fq - 2)) : 16 * t + 4 * fq;
    f32x4v o = vb;
    if (rot) {
#pragma unroll
      for (int i = 0; i < 4; ++i) o[i] = fq < 2 ? rope_lo(vb[i], pb[i], cs[i], sn[i]) : rope_hi(pb[i], vb[i], cs[i], sn[i]);
    }
    const uint2 pk{pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3])};
    *(uint2*)(a.y + (long)fr * a.ldy + hh * HD + d0) = pk;
    if (hh < a.H || slot < 0) return;
    const int page = slot / PAGE, tau = slot - page * PAGE;
    const bool isv = hh >= a.H + a.HKV;
    const int kvh = isv ? hh - a.H - a.HKV : hh - a.H;
    unsigned short* pg = a.cache + (((long)page * a.HKV + kvh) * 2 + (isv ? 1 : 0)) * PAGE_ELEMS;
    if (!isv) {
      *(uint2*)(pg + kv_k_index(tau, d0)) = pk;  // 4 consecutive dims: one 8-B run of the K fragment
    } else {
      pg[kv_v_index(tau, d0 + 0)] = (unsigned short)(pk.x & 0xffff);
      pg[kv_v_index(tau, d0 + 1)] = (unsigned short)(pk.x >> 16);
      pg[kv_v_index(tau, d0 + 2)] = (unsigned short)(pk.y & 0xffff);
      pg[kv_v_index(tau, d0 + 3)] = (unsigned short)(pk.y >> 16);
    }
  } else if (a.mode & EPI_SWIGLU) {
    f32x4v u, o;
#pragma unroll
    for (int i = 0; i < 4; ++i) u[i] = lane_xor32(v[i]);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      o[i] = (a.mode & EPI_CLAMPED) ? gate_clamped(v[i], u[i], a.limit)
             : ((a.mode & EPI_GELU) ? gate_act<GATE_GELU>(v[i]) : gate_act<GATE_SILU>(v[i])) * u[i];
    if (in && fq < 2) *(uint2*)(a.y + (long)m * a.ldy + 8 * nt + 4 * fq) = uint2{pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3])};
  } else if (in) {
    if (a.mode & EPI_RESID) {
      v[0] += bf2f(old.x & 0xffff);
      v[1] += bf2f(old.x >> 16);
      v[2] += bf2f(old.y & 0xffff);
      v[3] += bf2f(old.y >> 16);
    }
    *(uint2*)yt = uint2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
  }
}

}  // namespace dec
}  // namespace kgs

namespace {
constexpr int FEW_CUS = 256;

// Tiles of W (of 16 rows) and waves of a workgroup, and the k-steps of its ring; r 0: not for this kernel. Sums that neither divide as the
// first lines' nor are short: 8, 4 or 2 waves, and as much of a wave's part in the ring as divides it.
struct FewSplit {
  int r, nw, pf;
};
FewSplit few_split(int M, int N, int K) {
  if (M < 1 || M > 32 || N <= 0 || K <= 0 || N % 16 || K % 64 || (long)N * K > (1l << 31)) return {0, 0, 0};
  const int strips = N / 16;
  if (M <= 16 && K % 512 == 0) {
    if (strips <= FEW_CUS && K % 1024 == 0) return {1, 8, 4};
    if (strips <= 2 * FEW_CUS) return M > 4 && strips > FEW_CUS && strips % 2 == 0 ? FewSplit{2, 4, 4} : FewSplit{1, 4, 4};
    return {1, 2, 8};
  }
  const int nw = K % 256 == 0 ? 8 : K % 128 == 0 ? 4 : 2, steps = K / 32 / nw;
  return {1, nw, steps % 4 == 0 ? 4 : steps % 3 == 0 ? 3 : steps % 2 == 0 ? 2 : 1};
}
}  // namespace

// Whether kgs_skinny_few runs M rows of an [N, K] weight: up to 16 rows, N a multiple of 16 and K of 512; without a norm and a rotation up to 32 rows and K of 64.
KGS_EXPORT int kgs_skinny_few_ok(int M, int N, int K, int plain) { return few_split(M, N, K).r > 0 && (plain || (M <= 16 && K % 512 == 0)); }

namespace {
int launch_few(const kgs::dec::FewArgs& a, const FewSplit& f, bool rope, bool own, int products, hipStream_t s) {
  using namespace kgs::dec;
  const int M = a.M, N = a.N, K = a.K;
  auto run = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(N / (16 * f.r), products), dim3(64 * f.nw), 0, s, a);
    return (int)hipGetLastError();
  };
  auto pick = [&](auto ro, auto ow) {
    constexpr bool RO = decltype(ro)::value, OW = decltype(ow)::value;
    if (f.r == 2) return run(few<2, 1, 4, 4, RO, OW>);
    if (f.nw == 8) return run(few<1, 1, 8, 4, RO, OW>);
    if (f.nw == 4) return run(few<1, 1, 4, 4, RO, OW>);
    return run(few<1, 1, 2, 8, RO, OW>);
  };
  using T = std::true_type;
  using F = std::false_type;
  if (M <= 16 && K % 512 == 0) return rope ? (own ? pick(T{}, T{}) : pick(T{}, F{})) : own ? pick(F{}, T{}) : pick(F{}, F{});
  auto odd = [&](auto mt, auto nw) {
    constexpr int MT = decltype(mt)::value, NW = decltype(nw)::value;
    return f.pf == 4 ? run(few<1, MT, NW, 4, false, false>) : f.pf == 3 ? run(few<1, MT, NW, 3, false, false>)
           : f.pf == 2 ? run(few<1, MT, NW, 2, false, false>) : run(few<1, MT, NW, 1, false, false>);
  };
  auto waves = [&](auto mt) {
    return f.nw == 8 ? odd(mt, std::integral_constant<int, 8>{}) : f.nw == 4 ? odd(mt, std::integral_constant<int, 4>{})
                                                                             : odd(mt, std::integral_constant<int, 2>{});
  };
  return M <= 16 ? waves(std::integral_constant<int, 1>{}) : waves(std::integral_constant<int, 2>{});
}
}  // namespace

// y[M, N] (bf16, rows ldy apart) = x[M, K] (rows ldx apart) . W^T, W packed as for kgs_skinny_gemm_bf16. epi: EPI_SWIGLU (with
// EPI_GELU or EPI_CLAMPED and limit; y is [M, N / 2]), EPI_RESID (y += the product), EPI_RMS (the product of x's RMSNorm: its
// rows' statistics are made here), EPI_ROPE (as kgs_skinny_gemm_bf16_rope, with cosv .. HKV).
KGS_EXPORT int kgs_skinny_few(const void* wp, const void* x, void* y, int M, int N, int K, long ldx, long ldy, int epi, float eps,
                              float limit, const float* cosv, const float* sinv, const int* pos, const int* slot, void* cache,
                              int H, int HKV, hipStream_t s) {
  using namespace kgs::dec;
  const FewSplit f = few_split(M, N, K);
  if (!f.r) return KGS_ERR_SHAPE;
  const bool rope = epi & EPI_ROPE, own = epi & EPI_RMS;
  if ((rope || own) && (M > 16 || K % 512)) return KGS_ERR_SHAPE;
  if (ldx < K || ldy < (epi & EPI_SWIGLU ? N / 2 : N) || ldx > 1l << 25) return KGS_ERR_SHAPE;
  if ((uintptr_t)wp % 16 || (uintptr_t)x % 16 || (uintptr_t)y % 8 || ldx % 8 || ldy % 4) return KGS_ERR_ALIGN;
  if (epi & ~(EPI_SWIGLU | EPI_GELU | EPI_CLAMPED | EPI_RMS | EPI_RESID | EPI_ROPE)) return KGS_ERR_ARG;
  if (((epi & EPI_SWIGLU) != 0) + ((epi & EPI_RESID) != 0) + rope > 1) return KGS_ERR_ARG;
  if (rope) {
    if (H <= 0 || HKV <= 0 || H % HKV || N != (H + 2 * HKV) * HD) return KGS_ERR_SHAPE;
    if (!cosv || !sinv || !pos || !slot || !cache || (uintptr_t)cache % 16) return KGS_ERR_ARG;
  }
  const FewArgs a{(const unsigned short*)x, (const unsigned short*)wp, (unsigned short*)y, M, N, K, (int)ldx, ldy, epi, 1.f / K, eps, limit,
                  cosv, sinv, pos, slot, (unsigned short*)cache, H, HKV};
  return launch_few(a, f, rope, own, 1, s);
}

// y = x . W^T and y2 = x2 . W2^T in one launch: sizes and strides shared, as kgs_skinny_few with epi 0.
KGS_EXPORT int kgs_skinny_few_two(const void* wp, const void* x, void* y, const void* wp2, const void* x2, void* y2, int M, int N, int K,
                                  long ldx, long ldy, hipStream_t s) {
  using namespace kgs::dec;
  const FewSplit f = few_split(M, N, K);
  if (!f.r || ldx < K || ldy < N || ldx > 1l << 25) return KGS_ERR_SHAPE;
  if (((uintptr_t)wp | (uintptr_t)x | (uintptr_t)wp2 | (uintptr_t)x2) % 16 || ((uintptr_t)y | (uintptr_t)y2) % 8 || ldx % 8 || ldy % 4)
    return KGS_ERR_ALIGN;
  FewArgs a{(const unsigned short*)x, (const unsigned short*)wp, (unsigned short*)y, M, N, K, (int)ldx, ldy};
  a.x2 = (const unsigned short*)x2;
  a.w2 = (const unsigned short*)wp2;
  a.y2 = (unsigned short*)y2;
  return launch_few(a, f, false, false, 2, s);
}
