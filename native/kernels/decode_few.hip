// Skinny products of up to 32 rows (with a norm or a rotation of K of 512, from 17 rows on of 1024): y[M, N] = x[M, K] . W^T, W packed as for decode.hip's skinny
// ([N/16][K/32][64][8]), with that kernel's epilogues and one statistic of its own.
//
// A workgroup of NW waves takes R 16-row tiles of W; the waves share out K, stream their part of W and of x through a ring of PF k-steps and add
// their sums in LDS, in the order of K's parts (few_parts). Loads are buffer loads, so that a step waits for exactly its own. The last round sends for nothing:
// the last k-steps fetched again, as the ring did, were waited for at the end of the launch, 0.5 to 1 us of a short one and a
// tenth of a long one.
//
// x: up to 16 rows straight from memory in MFMA operand order. There a load instruction costs by its distinct rows (137 bytes a ns and CU at 1 row, 60
// at 8, 37 at 16, where whole lines come at 120), so that from 17 rows on (LX) x comes by LDS-DMA, 8 rows of 128 bytes a piece, into stages of
// the wave's own: no barrier. Below, LDS on the way costs more than it gives (us at 16 rows direct / so: 2048x2048 4.8 / 4.9, 4096x4096 8.1 / 8.9).
//
// OWN: the RMSNorm of x from x itself. Every wave holds its part of all rows anyway and adds up its squares (add_squares). Where the producer of x adds them up instead, 256 workgroups' atomics
// meet on one address, 12.5 ns each, at the end of a launch that nothing hides: a layer's o and down took 1.6 us longer at 1
// row, 2.0 at 16. Nothing here depends on the order in which workgroups arrive.
//
// Bound by memory where W is large (28672 x 4096 at 1 row 36.4 us, 6.5 TB/s; 40.6 before), else by the launch and one trip through
// memory and the ring (4096 x 4096 7.1 us, before 7.5; 2048 x 2048 3.6, 4.3). The split (few_split): few waves with long rings, whose loads are all in flight
// at once and whose sums are soon added -- us at 8 rows with 8 / 4 / 2 / 1 waves, as long rings as fit: 2048x2048 4.3 / 4.2 / 4.0 / 4.6, 4096x4096 7.4 / 7.2 /
// 7.0 / 8.4, 6144x4096 12.4 / 11.7 / 10.9 / 10.2, 16384x2048 12.3 / 13.6 / 12.4 / 12.2, 28672x4096 36.2 / 39.7 / 36.6 / 36.2; eight for long sums of up to 4 rows (4096x14336 at 1
// row 18.5, by two 19.8; at 8 20.7, 19.2). Two tiles a workgroup where x counts: 6144x4096 at 16 rows 12.1 / 11.0, 28672x4096 at 16 40.8 / 40.3. At 24 / 32 rows, skinny / here:
// 6144x4096 19.7, 19.8 / 12.6, 13.2; 4096x4096 12.3, 13.7 / 9.1, 10.1; 2048x2048 7.4, 8.1 / 5.5, 6.0; 12288x2048 16.0, 15.9 / 12.3, 12.7. Any K of 64, for products that
// were the library's: us at 1 / 32 rows, library / here: 2048x128 3.3, 3.8 / 2.0, 2.5; 2048x768 5.0, 6.8 / 2.6, 4.0; 832x2048 7.9 / 3.3 at 1 row. Which products come here:
// kgs/ops/decode.py few_route, few_wide.
#include "decode_common.h"

#include <type_traits>
#include <utility>

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

__device__ __forceinline__ void dma16(__amdgpu_buffer_rsrc_t r, void* lds, int v, int s) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (KGS_LDS void*)lds, 16, v, s, 0, 0);
}

template <int... I, typename F>
__device__ __forceinline__ void each_of(std::integer_sequence<int, I...>, F&& f) { (f(std::integral_constant<int, I>{}), ...); }
template <int N, typename F>
__device__ __forceinline__ void each(F&& f) { each_of(std::make_integer_sequence<int, N>{}, f); }

// MT column tiles of 16 rows of x. LX: x by LDS, in XP pieces of 8 rows of 64 values for two k-steps; else straight from memory in operand order. PARTS: K's
// parts, which are summed apart and added in their order (few_parts); a wave takes as many as are left for it one after the other
template <int R, int MT, int NW, int PF, bool LX, bool ROPE, bool OWN, int PARTS = NW>
__global__ __launch_bounds__(64 * NW) void few(FewArgs a) {
  static_assert(!LX || PF % 2 == 0);
  static_assert(PARTS % NW == 0 && (PARTS == NW || (!LX && PF % 4 == 0)));
  constexpr int XP = LX ? 2 * MT : 0, NX = PF / 2 + 1;  // NX: stages of two k-steps of x, a wave's own: no barrier
  __shared__ __attribute__((aligned(16))) f32x4v red[PARTS * R * MT * 64];
  __shared__ double stat[OWN ? NW : 1][16 * MT];
  __shared__ __attribute__((aligned(16))) bf16x8 xs[LX ? NW * NX * XP * 64 : 1];
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
  // rows from M on repeat the last one: never stored. By LDS: row 8 j + lane / 8 of piece j, its 16-byte chunk c at c ^ (row / 2 % 8), so that a
  // fragment's reads touch every bank evenly
  int xo[LX ? XP : MT];
  if constexpr (!LX) {
#pragma unroll
    for (int c = 0; c < MT; ++c) xo[c] = 2 * (min(16 * c + fr, M - 1) * a.ldx + fq * 8);
  } else {
#pragma unroll
    for (int j = 0; j < XP; ++j) {
      const int row = 8 * j + (lane >> 3);
      xo[j] = 2 * (min(row, M - 1) * a.ldx + ((lane & 7) ^ ((row >> 1) & 7)) * 8);
    }
  }
  bf16x8* const xw = xs + (LX ? w * NX * XP * 64 : 0);
  const int ro[2] = {fr * 8 + (fq ^ (fr >> 1)), fr * 8 + ((4 + fq) ^ (fr >> 1))};  // a fragment's 16 bytes: even and odd k-steps
  bf16x8 wf[PF][R], xf[LX ? 2 : PF][MT];
  auto load_w = [&](int p, int s) {  // k-step s of this wave; W past the caches, it comes once
#pragma unroll
    for (int r = 0; r < R; ++r) wf[p][r] = ld_frag<2>(rw, wo, (r * nkk + kk0 + s) * 1024);
  };
  auto load_x = [&](int p, int s) {
#pragma unroll
    for (int c = 0; c < MT; ++c) xf[p][c] = ld_frag<0>(rx, xo[c], (kk0 + s) * 64);
  };
  auto send_x = [&](int stage, int s) {
#pragma unroll
    for (int j = 0; j < XP; ++j) dma16(rx, xw + (stage * XP + j) * 64, xo[j], (kk0 + s) * 64);
  };
#pragma unroll
  for (int p = 0; p < PF; ++p) {
    if constexpr (!LX) {
      load_w(p, p);
      load_x(p, p);
    } else {
      if (p % 2 == 0) {
        __builtin_amdgcn_sched_barrier(0);
        send_x(p / 2, p);
        __builtin_amdgcn_sched_barrier(0);
      }
      load_w(p, p);
    }
  }

  // what the epilogue needs of its first tile (r, c) = (w / MT, w % MT), under the main loop's way: old values or rotation
  auto out = [&](int t) { return a.y + (long)min(16 * (t % MT) + fr, M - 1) * a.ldy + 16 * (nt0 + t / MT) + 4 * fq; };
  const int t0 = w < R * MT ? w : 0;
  uint2 old = make_uint2(0, 0);
  if (!ROPE && (a.mode & EPI_RESID) && w < R * MT) old = *(const uint2*)out(t0);
  float cs[4], sn[4];
  int slot = -1;
  auto turn = [&](int t) {
    const int m = 16 * (t % MT) + fr, mr = min(m, M - 1), p = a.pos[mr], dd = 8 * ((nt0 + t / MT) & 7) + 4 * (fq & 1);  // dim within the rotated half
    slot = m < M ? a.slot[mr] : -1;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      cs[i] = a.cosv[(long)p * (HD / 2) + dd + i];
      sn[i] = a.sinv[(long)p * (HD / 2) + dd + i];
    }
  };
  if constexpr (ROPE) turn(t0);

  f32x4v acc[R][MT];
  [[maybe_unused]] double own[MT] = {};
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int c = 0; c < MT; ++c) acc[r][c] = f32x4v{0.f, 0.f, 0.f, 0.f};
  auto step = [&](int p, const bf16x8 (&x)[MT]) {
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int c = 0; c < MT; ++c) acc[r][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[p][r], x[c], acc[r][c], 0, 0, 0);
    if constexpr (OWN) {
#pragma unroll
      for (int c = 0; c < MT; ++c) own[c] = add_squares(own[c], x[c]);
    }
  };
  // a part's sums to LDS, at its last k-step (a part has a multiple of four)
  const int psteps = nkk / PARTS;
  int part = w * (PARTS / NW);
  [[maybe_unused]] int end = psteps;
  auto hand_over = [&] {
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int c = 0; c < MT; ++c) {
        red[((part * R + r) * MT + c) * 64 + lane] = acc[r][c];
        acc[r][c] = f32x4v{0.f, 0.f, 0.f, 0.f};
      }
    ++part;
    end += psteps;
  };
  [[maybe_unused]] int from = 0, to = NX - 1;  // stages being read and sent for
  // a round of the ring; the last one sends for nothing: what it would fetch again is waited for, up to 1 us of a launch
  auto round = [&](int s0, auto more) {
    constexpr bool MORE = decltype(more)::value;
    each<PF>([&](auto pc) {
      constexpr int p = decltype(pc)::value;
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (!LX) {
        step(p, xf[p]);
        if constexpr (MORE) {
          load_w(p, s0 + PF + p);
          load_x(p, s0 + PF + p);
        }
        if constexpr (PARTS > NW && p % 4 == 3) {
          if constexpr (OWN) asm volatile("" : "+v"(own[0]));  // here: else the squares wait behind the branch, with x in 64 registers more
          if (s0 + p + 1 == end) hand_over();
        }
      } else {
        if constexpr (p % 2 == 0) {
          if constexpr (MORE) {
            send_x(to, s0 + PF + p);  // into the stage whose fragments the step before last took
            to = to == NX - 1 ? 0 : to + 1;
          }
          // these k-steps' pieces: the weights of two k-steps, and the pieces and weights of the ring's others, were sent for after them
          constexpr int AFTER = PF / 2 - (MORE ? 0 : p / 2 + 1);
          asm volatile("s_waitcnt vmcnt(%0)" ::"n"(AFTER * (XP + 2 * R) + (MORE ? 0 : 2 * R)) : "memory");
          const bf16x8* st = xw + from * XP * 64;
          from = from == NX - 1 ? 0 : from + 1;
#pragma unroll
          for (int e = 0; e < 2; ++e)
#pragma unroll
            for (int c = 0; c < MT; ++c) xf[e][c] = st[c * 128 + ro[e]];
          __builtin_amdgcn_sched_barrier(0);
        }
        step(p, xf[p % 2]);
        if constexpr (MORE) load_w(p, s0 + PF + p);
      }
    });
  };
  int s0 = 0;
  for (; s0 + PF < nsteps; s0 += PF) round(s0, std::true_type{});
  round(s0, std::false_type{});
  if constexpr (PARTS == NW) hand_over();
  if constexpr (OWN) {
#pragma unroll
    for (int c = 0; c < MT; ++c) {
      own[c] = wsum16(own[c]);
      if (fq == 0) stat[w][16 * c + fr] = own[c];
    }
  }
  __syncthreads();
  for (int t = w; t < R * MT; t += NW) {
    const int nt = nt0 + t / MT, m = 16 * (t % MT) + fr;
    if (R * MT > NW && t != w) {
      if (!ROPE && (a.mode & EPI_RESID)) old = *(const uint2*)out(t);
      if constexpr (ROPE) turn(t);
    }
    // lane: row m of x, rows 16 nt + 4 fq + i of W
    f32x4v v = red[t * 64 + lane];
#pragma unroll
    for (int j = 1; j < PARTS; ++j) v += red[(j * R * MT + t) * 64 + lane];
    if constexpr (OWN) {
      const int col = 16 * (t % MT) + fr;
      double ss = stat[0][col];
#pragma unroll
      for (int j = 1; j < NW; ++j) ss += stat[j][col];
      v *= rsqrtf((float)ss * a.inv_k + a.eps);
    }
    const bool in = m < M;
    if constexpr (ROPE) {
      const int hh = nt >> 3, i8 = nt & 7;  // head and tile within it
      const bool rot = hh < a.H + a.HKV;
      f32x4v vb, pb;  // this lane's and its partner's (lane ^ 32) values, rounded to bf16
#pragma unroll
      for (int i = 0; i < 4; ++i) vb[i] = bf2f(f2bf(v[i]));
#pragma unroll
      for (int i = 0; i < 4; ++i) pb[i] = lane_xor32(vb[i]);
      if (!in) continue;
      const int d0 = rot ? (fq < 2 ? 8 * i8 + 4 * fq : 64 + 8 * i8 + 4 * (fq - 2)) : 16 * i8 + 4 * fq;
      f32x4v o = vb;
      if (rot) {
#pragma unroll
        for (int i = 0; i < 4; ++i) o[i] = fq < 2 ? rope_lo(vb[i], pb[i], cs[i], sn[i]) : rope_hi(pb[i], vb[i], cs[i], sn[i]);
      }
      const uint2 pk{pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3])};
      *(uint2*)(a.y + (long)m * a.ldy + hh * HD + d0) = pk;
      if (hh < a.H || slot < 0) continue;
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
      *(uint2*)out(t) = uint2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
    }
  }
}

}  // namespace dec
}  // namespace kgs

namespace {
constexpr int FEW_CUS = 256;

// Tiles of W (of 16 rows) and waves of a workgroup, the k-steps of its ring, and whether x comes by LDS; r 0: not for this kernel. Sums that neither
// divide as the first lines' nor are short: 8, 4 or 2 waves, and as much of a wave's part in the ring as divides it.
struct FewSplit {
  int r, nw, pf, lx;
};
FewSplit few_split(int M, int N, int K) {
  if (M < 1 || M > 32 || N <= 0 || K <= 0 || N % 16 || K % 64 || (long)N * K > (1l << 31)) return {0, 0, 0, 0};
  const int strips = N / 16;
  if (M <= 16 && K % 512 == 0) {
    if (strips <= FEW_CUS) return M <= 4 && K >= 8192 && K % 1024 == 0 ? FewSplit{1, 8, 4, 0} : FewSplit{1, 2, K % 1024 == 0 ? 16 : 8, 0};
    // two tiles a workgroup share x: where one makes little more than one round of the CUs, and where 13 rows and more bound a long grid
    if (strips % 2 == 0 && (strips <= 2 * FEW_CUS ? M > 4 || strips <= 5 * FEW_CUS / 4 : M > 12 && strips >= 4 * FEW_CUS)) return {2, 2, 8, 0};
    return {1, 1, 16, 0};
  }
  if (M > 16 && K % 1024 == 0) {
    if (strips <= FEW_CUS) return {1, 8, 4, 1};
    if (strips % 2 == 0) return strips <= 2 * FEW_CUS ? FewSplit{2, 8, 4, 1} : FewSplit{2, 4, 4, 1};
  }
  const int nw = K % 256 == 0 ? 8 : K % 128 == 0 ? 4 : 2, steps = K / 32 / nw;
  return {1, nw, steps % 4 == 0 ? 4 : steps % 3 == 0 ? 3 : steps % 2 == 0 ? 2 : 1, 0};
}
// Parts of K that a product of up to 16 rows and K of 512 sums apart, whatever its waves: one chain a wave would be up to four times as long. rms error of
// sums that cancel, against 64 bits, a chain a wave / so: 4096x4096 2.1e-7 / 1.2e-7, 4096x14336 4.3e-7 / 2.4e-7, 2048x1024 1.0e-7 / 0.65e-7, 6144x4096 2.1e-7 / 1.7e-7. us, the
// same: 4096x4096 at 1 / 8 / 16 rows 7.0, 7.2, 7.9 / 7.1, 7.3, 8.1; 28672x4096 and 16384x2048 do not differ.
int few_parts(int N, int K) { return N <= 16 * FEW_CUS && K % 1024 == 0 ? 8 : N <= 32 * FEW_CUS ? 4 : 2; }
// With a norm or a rotation: only by the splits of the first lines
bool few_normed(const FewSplit& f, int M, int K) { return f.r && (M <= 16 ? K % 512 == 0 : f.lx != 0); }
}  // namespace

// Whether kgs_skinny_few runs M rows of an [N, K] weight: up to 32 rows, N a multiple of 16, K of 64. With a norm or a rotation (!plain) up to 16 rows
// and K of 512; kgs_skinny_few_wide_ok has 17 to 32.
KGS_EXPORT int kgs_skinny_few_ok(int M, int N, int K, int plain) { return few_split(M, N, K).r > 0 && (plain || (M <= 16 && K % 512 == 0)); }

// Whether it runs 17 to 32 rows with x by LDS, and so with a norm and a rotation too: N a multiple of 32, or of 16 up to a strip a CU, K of 1024.
KGS_EXPORT int kgs_skinny_few_wide_ok(int M, int N, int K) { return M > 16 && few_split(M, N, K).lx; }

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
    if (f.lx) return f.r == 1 ? run(few<1, 2, 8, 4, true, RO, OW>) : f.nw == 8 ? run(few<2, 2, 8, 4, true, RO, OW>) : run(few<2, 2, 4, 4, true, RO, OW>);
    const bool four = few_parts(N, K) == 4;
    if (f.r == 2) return four ? run(few<2, 1, 2, 8, false, RO, OW, 4>) : run(few<2, 1, 2, 8, false, RO, OW>);
    if (f.nw == 1) return four ? run(few<1, 1, 1, 16, false, RO, OW, 4>) : run(few<1, 1, 1, 16, false, RO, OW, 2>);
    if (f.nw == 8) return run(few<1, 1, 8, 4, false, RO, OW>);
    return f.pf == 16 ? run(few<1, 1, 2, 16, false, RO, OW, 8>) : run(few<1, 1, 2, 8, false, RO, OW, 4>);
  };
  using T = std::true_type;
  using F = std::false_type;
  if (f.lx || (M <= 16 && K % 512 == 0)) return rope ? (own ? pick(T{}, T{}) : pick(T{}, F{})) : own ? pick(F{}, T{}) : pick(F{}, F{});
  auto odd = [&](auto mt, auto nw) {
    constexpr int MT = decltype(mt)::value, NW = decltype(nw)::value;
    return f.pf == 4 ? run(few<1, MT, NW, 4, false, false, false>) : f.pf == 3 ? run(few<1, MT, NW, 3, false, false, false>)
           : f.pf == 2 ? run(few<1, MT, NW, 2, false, false, false>) : run(few<1, MT, NW, 1, false, false, false>);
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
  if ((rope || own) && !few_normed(f, M, K)) return KGS_ERR_SHAPE;
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
