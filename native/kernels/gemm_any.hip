// bf16 NT GEMM for any M, N and K % 8 == 0 on the four-wave K-step of gemm_w4.h: the kernel
// behind kgs_gemm_bf16_nt wherever the persistent 256x256 grid does not apply -- ragged sizes,
// and products of too few 256x256 tiles to fill the chip.
//
//   C[M, N] = epilogue(A[M, K] . B[N, K]^T + bias)
//
// What bounds such a product is the number of CUs that get a tile and the length of one
// workgroup's serial chain of K-steps, so the tile (64x64, or 128x128 to 256x256 in steps of 32 and 64) and the number
// of K slices are chosen by sizes (plan below). 128x128 tiles keep a quarter of the AGPRs, so
// two workgroups share a CU and one's barriers and loads hide behind the other's MFMAs.
//
// Ragged sizes cost two selects per K-step: rows past M or N lie outside the buffer resources,
// which end at the last valid element, and a lane whose 16-byte chunk of K lies past K gets an
// offset outside them too; all of these arrive in LDS as zeros. K is walked in whole pairs of
// 64-wide steps. Stores are predicated by row and column; a C whose rows are not 16-byte aligned
// takes 2-byte stores.
//
// The order of the products in every accumulator is gemm_w4.h's, so without K slices the result
// is bitwise the aligned kernels'. With slices each one writes fp32 partial tiles, which
// any_reduce sums in a fixed order before the epilogue.
#include <utility>

#include "gemm_w4p.h"
#include "tile_queue.h"

namespace kgs {
int cu_count();  // gemm_bf16.hip
namespace any {

using w4::BK;
using w4::Ctx;
using w4::Frag;

typedef long i64x2 __attribute__((ext_vector_type(2)));
constexpr int OOB = w4::OOB_OFFSET;  // above every buffer resource's size (gemm_any_ok)

// What a launch stores. DUAL: C gets bf16(acc + bias) and C2 the activation of that bf16 value
// (a training forward pass, whose backward pass needs both).
struct Args {
  const unsigned short* A;
  const unsigned short* B;
  void* C;                     // bf16 [M, ldc], or fp32 partials [slices][M][ldc]
  unsigned short* C2;          // DUAL
  const unsigned short* bias;  // null: none
  int M, N, K, lda, ldb, ldc;
  int ks;                      // K of a slice, a multiple of 128
  int tall;                    // tile groups along N (M > N): see launch
  int vec;                     // 16-B stores: ldc % 8 == 0 and C (C2) 16-B aligned
  float alpha;                 // e4m3: a factor of the sums, times *alpha_ptr if that is given
  const float* alpha_ptr;
};

// The launch's arguments, read anew: behind the asm the compiler cannot know them for the ones that it has
__device__ __forceinline__ Args again() {
  typedef const Args __attribute__((address_space(4)))* Kernarg;
  Kernarg p = (Kernarg)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  Args g;
  __builtin_memcpy(&g, p, sizeof g);
  return g;
}

template <int BM, int BN>
constexpr int waves_per_simd() { return BM == 128 && BN == 128 ? 2 : 1; }

// LDS stages of a tile with a CU to itself (ONE): 128 columns leave room for more than two, and so for one barrier a K-step (w4::kstep1). Of 192
// columns three fit too and give nothing (1762 x 6144 x 4096 67.8, 68.3). Medians of runs in turn, us, two stages / so: 128x128 tiles 2048^3 21.7 / 19.8
// (three stages 20.4, five 20.7), 1024 x 4096 x 4096 40.4 / 36.7, 1024 x 1024 x 8192 49.0 / 42.2; 192x128 1536 x 4096 x 4096 47.6 / 44.9;
// 224x128 1762 x 4096 x 4096 55.3 / 53.2, K 14336 185 / 181, 3580 x 2048 x 2048 27.4 / 26.5; 256x128 2048 x 4096 x 4096 57.5 / 54.4. What is left there is
// the matrix cores' clock and the operands' way in: MFMAs alone 49 us of the last.
template <int BM, int BN, bool ONE>
constexpr int lds_stages() { return !ONE || BN != 128 ? 2 : BM == 128 ? 4 : 3; }

template <int EPI>
__device__ __forceinline__ unsigned pack_epi(float a, float b, float ba, float bb) {
  return pack_bf16x2(epilogue<EPI>(a, ba), epilogue<EPI>(b, bb));
}

// the activation of an already rounded pre-activation; a NaN stays one
template <int EPI>
__device__ __forceinline__ float act_of(unsigned short z) {
  const float v = bf2f(z);
  if constexpr (EPI == EPI_BIAS_RELU) return v < 0.f ? 0.f : v;
  return epilogue<EPI>(v, 0.f);
}
template <int EPI>
__device__ __forceinline__ unsigned act_pair(unsigned z) {
  return pack_bf16x2(act_of<EPI>((unsigned short)(z & 0xffff)), act_of<EPI>((unsigned short)(z >> 16)));
}

// 8 columns from `col` of a row: one 16-B store, or the valid columns one by one
__device__ __forceinline__ void store8(unsigned short* row, int col, int N, int vec, uint4 v) {
  if (vec && col + 8 <= N) {
    *(uint4*)(row + col) = v;
    return;
  }
  const unsigned u[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
  for (int e = 0; e < 8; ++e)
    if (col + e < N) row[col + e] = (unsigned short)(u[e >> 1] >> (16 * (e & 1)));
}

// A lane's part of a tile's rows: NB fragments of 16 columns, four of each from `col`
template <int EPI, int NB>
__device__ __forceinline__ void load_bias(const Args& a, int col, float (&bv)[NB][4]) {
#pragma unroll
  for (int n = 0; n < NB; ++n)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      bv[n][e] = 0.f;
      if constexpr (epi_bias<EPI>())
        if (a.bias && col + n * 16 + e < a.N) bv[n][e] = bf2f(a.bias[col + n * 16 + e]);
    }
}
// EPI_ADDC's old values, 8 columns from `col` of each fragment pair (N % 8 == 0 and 16-B rows)
template <int EPI, int NB>
__device__ __forceinline__ void load_old(const Args& a, int r, int col, uint4 (&old)[NB / 2]) {
  if constexpr (EPI == EPI_ADDC) {
    const unsigned short* crow = (const unsigned short*)a.C + (long)r * a.ldc;
#pragma unroll
    for (int p = 0; p < NB / 2; ++p)
      old[p] = r < a.M && col + p * 32 < a.N ? *(const uint4*)(crow + col + p * 32) : make_uint4(0, 0, 0, 0);
  }
}
// Row r of a tile through the epilogue; `col` as in load_old
template <int EPI, int NB, bool DUAL>
__device__ __forceinline__ void store_row(const Args& a, int r, int col, const f32x4 (&v)[NB], const float (&bv)[NB][4],
                                          const uint4 (&old)[NB / 2]) {
  unsigned short* crow = (unsigned short*)a.C + (long)r * a.ldc;
#pragma unroll
  for (int n = 0; n < NB; n += 2) {
    uint2 o[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      constexpr int E = DUAL ? EPI_BIAS : EPI;
      o[h].x = pack_epi<E>(v[n + h][0], v[n + h][1], bv[n + h][0], bv[n + h][1]);
      o[h].y = pack_epi<E>(v[n + h][2], v[n + h][3], bv[n + h][2], bv[n + h][3]);
    }
    auto sx = __builtin_amdgcn_permlane16_swap(o[0].x, o[1].x, false, false);
    auto sy = __builtin_amdgcn_permlane16_swap(o[0].y, o[1].y, false, false);
    uint4 q = make_uint4(sx[0], sy[0], sx[1], sy[1]);
    const int c = col + n * 16;
    if (r < a.M && c < a.N) {
      if constexpr (EPI == EPI_ADDC) q = add_bf16x8(old[n / 2], q);
      store8(crow, c, a.N, a.vec, q);
      if constexpr (DUAL)
        store8(a.C2 + (long)r * a.ldc, c, a.N, a.vec,
               make_uint4(act_pair<EPI>(q.x), act_pair<EPI>(q.y), act_pair<EPI>(q.z), act_pair<EPI>(q.w)));
    }
  }
}

// SW (a GateAct): B is a fused gate|up weight of N rows, gate rows first, and C [M, N / 2] holds
// act(gate) * up; a tile stages both halves' rows in turn (gemm_w4.h). `bias` then points to the
// clamped gate's limit.
//
// Two-stage tiles of a workgroup a CU take turns in one launch of a workgroup a CU (TURNS, turns_pay): the last two K-steps of a tile send for the
// first two K-tiles of the next and read its first fragments, so that between tiles a wave only has its epilogue. us, a
// workgroup a tile / so: 3001 x 7000 x 200 23.4 / 21.3, 5000 x 5000 x 1000 56.1 / 54.1, 6000 x 9000 x 1000 120.8 / 114.6, 8192 x 14336 x 1024 227 / 213. Bound by
// the matrix cores' power: what the gaps no longer cost comes off the clock. Tiles and resources are worked out from the arguments read anew at each turn:
// held through the K loop and the stores they spilled 26 to 53 scalar registers, and up to 8 in kernels of one tile that shared the loop.
// A workgroup's first tile is its own, the others are tickets of its XCD label in the launch's row q (tile_queue.h), so that a CU held by another
// stream's kernel leaves its share to the others. us with 16 CUs held for a millisecond, a fixed list / tickets / a workgroup a tile: 8192 x 14336 x 1024 336 /
// 212 / 241, 6000 x 9000 x 1000 156 / 135 / 119 (a late workgroup still has its first tile); else as the list (2049 x 8200 x 64 12.6 / 13.1 / 13.6, 6000 x 9000 x 1000 112 / 111 /
// 118). A ticket is drawn one tile ahead and handed over between the last two K-steps, whose waits and barriers are all that it needs.
template <int EPI, int BM, int BN, bool SPLIT, bool DUAL, int SW, int NS, bool TURNS = false>
__device__ __forceinline__ void tile_product(const Args& a, [[maybe_unused]] int* q = nullptr) {
  constexpr int X = SW * 1000000, TN = SW ? BN / 2 : BN;  // TN: output columns of a tile
  using S = w4::Shape<BM, BN>;
  using Kn = w4::Knobs<BM, BN>;
  constexpr int MA = S::MA, NB = S::NB, ND = w4::dma_per_stage<BM, BN>();
  static_assert(!TURNS || (NS == 2 && !SPLIT));
  // TURNS: and a ticket. One object: with a second one each fragment read waits for every DMA
  __shared__ __attribute__((aligned(1024))) char smem[NS * S::STAGE + (TURNS ? 16 : 0)];
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // TURNS: the next ticket, through an address that is not known to be uniform (for a uniform one the compiler waits at once, for everything in flight)
  const int label = (int)blockIdx.x & 7;
  [[maybe_unused]] int zero = 0, ticket = 0;
  [[maybe_unused]] int* const slot = (int*)(smem + NS * S::STAGE);
  if constexpr (TURNS) asm volatile("v_mov_b32 %0, 0" : "=v"(zero));
  auto draw = [&] {
    if (threadIdx.x == 0) ticket = atomicAdd(q + label * TQ_INTS + zero, 1);
  };
  if constexpr (TURNS) draw();
  int slice = 0, m0, n0;
  auto rows = [](const Args& g) { return (g.M + BM - 1) / BM; };  // of tiles, and their columns
  auto columns = [](const Args& g) { return ((SW ? g.N / 2 : g.N) + TN - 1) / TN; };
  auto locate = [&](const Args& g, int id, int& m, int& n) {
    const int ntm = rows(g), ntn = columns(g);
    int tm, tn;
    if (g.tall) w4::tile_of<40000000, SPLIT>(id, (int)gridDim.x, ntm, ntn, slice, tm, tn);
    else w4::tile_of<0, SPLIT>(id, (int)gridDim.x, ntm, ntn, slice, tm, tn);
    m = tm * BM;
    n = tn * TN;
  };
  locate(a, (int)blockIdx.x, m0, n0);
  const int k0 = SPLIT ? slice * a.ks : 0;
  int kn = SPLIT ? min(a.K - k0, a.ks) : a.K;  // this slice's valid K

  Ctx c;
  c.smem = smem;
  c.w = w;
  c.wr = w >> 1;
  c.wc = w & 1;
  // resources end with the last valid element: nothing outside the operands is ever read
  auto bind = [&](const Args& g, int m, int n) {
    if constexpr (TURNS) kn = g.K;
    c.nt = NS > 2 ? (kn + BK - 1) / BK : (kn + 2 * BK - 1) / (2 * BK) * 2;
    c.sa32 = 32 * g.lda * 2;
    c.sb32 = 32 * g.ldb * 2;
    const int cols = SW ? g.N / 2 : g.N, ra = min(g.M - m, BM), rb = min(cols - n, TN);
    c.ra = __builtin_amdgcn_make_buffer_rsrc((void*)(g.A + (long)m * g.lda + k0), 0, ((ra - 1) * g.lda + kn) * 2, 0x00020000);
    c.rb = __builtin_amdgcn_make_buffer_rsrc((void*)(g.B + (long)n * g.ldb + k0), 0, ((rb - 1) * g.ldb + kn) * 2, 0x00020000);
    if constexpr (SW != 0)
      c.rb2 = __builtin_amdgcn_make_buffer_rsrc((void*)(g.B + ((long)cols + n) * g.ldb + k0), 0, ((rb - 1) * g.ldb + kn) * 2, 0x00020000);
  };
  bind(a, m0, n0);
  const int row = w * 8 + (lane >> 3);
  const int ch = ((lane & 7) ^ ((row >> 1) & 7)) * 8;  // first column of this lane's chunk in a K-tile
  const int voa = (row * a.lda + ch) * 2, vob = (row * a.ldb + ch) * 2;
  const int fr = lane & 15, fq = lane >> 4;
  c.ro0 = fr * 128 + ((fq ^ (fr >> 1)) * 16);
  c.ro1 = fr * 128 + (((4 + fq) ^ (fr >> 1)) * 16);
  // offsets of the next DMAs: outside the resources where K-tile kt's chunk lies past K, so that nothing is fetched (a fetch is waited for at the end)
  auto aim = [&](int kt) {
    const bool in = kt * BK + ch < kn;
    c.voa = in ? voa : OOB;
    c.vob = in ? vob : OOB;
  };

  if constexpr (BM == 128 && BN == 128) KGS_ACC_RESERVE_QUARTER();
  else KGS_ACC_RESERVE();
  w4::static_for<0, MA * NB>([](auto q) { accr::zero<decltype(q)::value>(); });

#pragma unroll
  for (int st = 0; st < (NS > 2 ? NS - 1 : 2); ++st) {
    aim(st);
#pragma unroll
    for (int j = 0; j < ND; ++j) w4::dma_any<BM, BN, X>(c, st, j, min(st, c.nt - 1) * BK);
  }
  w4::wait_vm<(NS > 2 ? NS - 2 : 1) * ND>();
  w4::bar();
  Frag<MA, NB> f0, f1;
  {
    const char* pa = w4::abase<BM, BN, 0>(c, 0);
    const char* pb = w4::bbase<BM, BN, 0>(c, 0);
#pragma unroll
    for (int e = 0; e < S::NR; ++e) {
      const int x = w4::rd_idx(Kn::ORD, MA, NB, e);
      if (w4::rd_isa(Kn::ORD, MA, NB, e)) f0.a[x] = w4::frag(pa + x * 2048);
      else f0.b[x] = w4::frag(pb + x * 2048);
    }
  }
  __builtin_amdgcn_s_waitcnt(0xc07f);

  // K-steps of K-tiles t, t + 1, which send for K-tiles s and s + 1; between them `middle`
  auto pair = [&](int s, auto&& middle) {
    aim(s);
    w4::kstep<BM, BN, 0, Kn::B1, Kn::R, Kn::P, Kn::ORD, X>(c, f0, f1, s - 2);
    middle();
    aim(s + 1);
    w4::kstep<BM, BN, 1, Kn::B1, Kn::R, Kn::P, Kn::ORD, X>(c, f0, f1, s - 1);
  };
  auto steady = [&](int s) { pair(s, [] {}); };
  auto store = [&](const Args& g, int m, int n) {
    const int mw = m + c.wr * (BM / 2) + fr, nw = n + c.wc * (TN / 2);
    const int lc = (fq & 1) * 16 + (fq >> 1) * 8;  // this lane's 8 of a fragment pair's 32 columns
    if constexpr (SW != 0) {
      // output fragment q: gate fragment ng = 4 (q / 2) + q % 2 and the up fragment two further
      const int cols = g.N / 2;
      const float limit = SW == GATE_CLAMPED ? *(const float*)g.bias : 0.f;
      w4::static_for<0, MA>([&](auto ic) {
        constexpr int i = decltype(ic)::value;
        f32x4 v[NB];
        w4::read_row<NB, i>(v);
        if (mw + i * 16 >= g.M) return;
        unsigned short* crow = (unsigned short*)g.C + (long)(mw + i * 16) * g.ldc;
#pragma unroll
        for (int q = 0; q < NB / 2; q += 2) {
          uint2 o[2];
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const int ng = 4 * ((q + h) / 2) + (q + h) % 2;
            float r[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) r[e] = gated<SW>(v[ng][e], v[ng + 2][e], limit);
            o[h] = make_uint2(pack_bf16x2(r[0], r[1]), pack_bf16x2(r[2], r[3]));
          }
          auto sx = __builtin_amdgcn_permlane16_swap(o[0].x, o[1].x, false, false);
          auto sy = __builtin_amdgcn_permlane16_swap(o[0].y, o[1].y, false, false);
          const int col = nw + q * 16 + lc;
          if (col < cols) store8(crow, col, cols, g.vec, make_uint4(sx[0], sy[0], sx[1], sy[1]));
        }
      });
    } else if constexpr (SPLIT) {
      // ldc is a multiple of 8: a fragment's four columns are inside the row or all outside
      float* part = (float*)g.C + (long)slice * g.M * g.ldc;
      w4::static_for<0, MA>([&](auto ic) {
        constexpr int i = decltype(ic)::value;
        f32x4 v[NB];
        w4::read_row<NB, i>(v);
        if (mw + i * 16 >= g.M) return;
        float* prow = part + (long)(mw + i * 16) * g.ldc;
#pragma unroll
        for (int q = 0; q < NB; ++q) {
          const int col = nw + q * 16 + fq * 4;
          if (col < g.ldc) *(f32x4*)(prow + col) = v[q];
        }
      });
    } else {
      float bv[NB][4];
      load_bias<EPI, NB>(g, nw + fq * 4, bv);
      w4::static_for<0, MA>([&](auto ic) {
        constexpr int i = decltype(ic)::value;
        const int r = mw + i * 16;
        uint4 old[NB / 2];
        load_old<EPI, NB>(g, r, nw + lc, old);
        f32x4 v[NB];
        w4::read_row<NB, i>(v);
        store_row<EPI, NB, DUAL>(g, r, nw + lc, v, bv, old);
      });
    }
  };
  auto settle = [] { asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 3" ::: "memory"); };  // MFMA -> v_accvgpr_read hazard

  if constexpr (!TURNS) {
    if constexpr (NS > 2) {
      for (int t = 0; t < c.nt; t += NS) {
        w4::static_for<0, NS>([&](auto st) {
          constexpr int ST = decltype(st)::value;
          if (ST && t + ST >= c.nt) return;
          aim(t + ST + NS - 1);
          w4::kstep1<BM, BN, ST, Kn::R, Kn::P, Kn::ORD, X, NS>(c, f0, f1, t + ST);
        });
      }
    } else {
      for (int t = 0; t < c.nt; t += 2) steady(t + 2);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the tail's DMAs (zeros) land before LDS is released
    settle();
    store(a, m0, n0);
  } else {
    // tickets of a label are numbered behind its workgroups' first tiles; its tile t is label + 8 t
    const int first = ((int)gridDim.x - label + 7) >> 3;
    auto limit = [&](const Args& g) { return (rows(g) * columns(g) - label + 7) >> 3; };
    auto hand_over = [&] {
      if (threadIdx.x == 0) *slot = ticket;
    };
    // unsigned: a ticket that no launch can have issued ends the workgroup, no address comes of it
    auto taken = [&](int lim) {
      const int raw = __builtin_amdgcn_readfirstlane(*slot);
      w4p::mark_bad_ticket(q + label * TQ_INTS, raw, lim);
      if (raw == lim - 1 && threadIdx.x == 0) atomicExch(q + label * TQ_INTS, 0);  // the label's last draw: each tile of it and each end of a workgroup is one
      return first + raw;
    };
    bool begun = false;
    for (int next = 0;;) {
      for (int t = 0; t + 2 < c.nt; t += 2) steady(t + 2);
      // the arguments again, instead of registers that hold them through the K-steps
      const Args g = again();
      const int lim = limit(g);
      if (!begun) {
        hand_over();
        __builtin_amdgcn_s_waitcnt(0xc07f);
        w4::bar();
        next = taken(lim);
        if ((unsigned)next < (unsigned)lim) draw();
        begun = true;
      }
      const bool more = (unsigned)next < (unsigned)lim;
      int m1 = 0, n1 = 0;
      if (more) {
        locate(g, label + 8 * next, m1, n1);
        bind(g, m1, n1);
      }
      pair(more ? 0 : c.nt, hand_over);
      if (!more) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // as above
      settle();
      const Args h = again();
      store(h, m0, n0);
      if (!more) break;
      m0 = m1;
      n0 = n1;
      const Args k = again();  // again: not held through the stores
      bind(k, m0, n0);
      const int most = limit(k);
      next = taken(most);
      if ((unsigned)next < (unsigned)most) draw();
      w4::static_for<0, MA * NB>([](auto q) { accr::zero<decltype(q)::value>(); });
      asm volatile("s_nop 7" ::: "memory");
      __builtin_amdgcn_s_waitcnt(0xc07f);
    }
  }
}

// gemm_nt_any: the tiles of plan, with or without slices; gemm_nt_mid: those between them (refine), one workgroup a CU, on two stages; gemm_nt_deep: tiles
// of 128 columns on the stages of lds_stages, 128x128 ones where they are no more than the CUs; gemm_nt_turn: tiles that take turns, kernels of their own,
// since a launch of one round loses up to 0.5 us by it (2080 x 5504 x 128 11.7 / 12.2)
template <int EPI, int BM, int BN, bool SPLIT, bool DUAL, int SW = 0>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(waves_per_simd<BM, BN>(), waves_per_simd<BM, BN>())))
void gemm_nt_any(Args a) {
  tile_product<EPI, BM, BN, SPLIT, DUAL, SW, lds_stages<BM, BN, waves_per_simd<BM, BN>() == 1>()>(a);
}
template <int EPI, int BM, int BN, bool DUAL, int SW = 0>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) void gemm_nt_mid(Args a) {
  tile_product<EPI, BM, BN, false, DUAL, SW, 2>(a);
}
template <int EPI, int BM, int BN, bool DUAL, int SW = 0, bool SPLIT = false>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) void gemm_nt_deep(Args a) {
  tile_product<EPI, BM, BN, SPLIT, DUAL, SW, lds_stages<BM, BN, true>()>(a);
}
template <int EPI, int BM, int BN, bool DUAL, int SW = 0>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) void gemm_nt_turn(Args a, int* q) {
  tile_product<EPI, BM, BN, false, DUAL, SW, 2, true>(a, q);
}

// The same product on 64x64 tiles, for grids that leave CUs idle at 128x128. What bounds such a
// launch is each workgroup's chain of K-steps; a step of this tile takes 0.26 us in a lone workgroup and
// 0.27 with one on every CU, against 0.34 and 0.49 (LDS traffic: half the bytes; operands in L2, cost()
// below has weights from HBM), and four times the workgroups share the epilogue. Four stages of 64-wide
// K-tiles keep three on their way with one barrier per step (eight: the same time; 64x128 tiles with
// three stages 0.44 us a step). Accumulators are plain registers, in gemm_w4.h's order of products per
// element: bitwise the larger tiles' results. us, 128x128 / here: 1024^3 9.4 / 7.4, 256 x 3072 x 2048 15.1 /
// 11.6, 128 x 5757 x 2080 19.8 / 13.5, 168 x 1760 x 1032 9.7 / 7.2.
// F8: e4m3 operands, seen as rows of 16-bit words (lda, ldb, K in words). A lane's 16-byte chunk is 16
// values of K, its halves the operands of two MFMAs: which K they are does not matter as long as
// both operands agree.
// NT: B past the caches, for one row tile of a B of whole 128-byte lines and 64 column tiles or more (launch), which is read once: 5.9 TB/s of a large one
// where the default policy reaches 5.0. Off the lines each would come twice (64 x 3000 x 1032 9.1 / 12.1 us), of a few tiles such loads cost 0.2 us (17 x
// 448 x 256 3.4 / 3.6). A kernel of its own: chosen at run time inside, the others lost 2 to 8 % (e4m3 8 x 512 x 5120 13.7 / 14.5 us, 32 x 1152 x 1280 with
// both outputs 9.0 / 9.8).
template <int EPI, bool DUAL, bool F8 = false, bool NT = false>
__global__ __launch_bounds__(256) void gemm_small(Args a) {
  constexpr int BM = 64, BN = 64, ST = 4;
  constexpr int FM = BM / 32, FN = BN / 32, LA = BM / 32, LB = BN / 32, STAGE = (BM + BN) * 128;
  __shared__ __attribute__((aligned(1024))) char smem[ST * STAGE];
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ntm = (a.M + BM - 1) / BM, ntn = (a.N + BN - 1) / BN;
  int none, tm, tn;
  w4::tile_of<0, false>((int)blockIdx.x, (int)gridDim.x, ntm, ntn, none, tm, tn);
  const int m0 = tm * BM, n0 = tn * BN, K = a.K, nt = (K + BK - 1) / BK;
  const int na = min(a.M - m0, BM), nb = min(a.N - n0, BN);
  const auto ra = __builtin_amdgcn_make_buffer_rsrc((void*)(a.A + (long)m0 * a.lda), 0, ((na - 1) * a.lda + K) * 2, 0x00020000);
  const auto rb = __builtin_amdgcn_make_buffer_rsrc((void*)(a.B + (long)n0 * a.ldb), 0, ((nb - 1) * a.ldb + K) * 2, 0x00020000);
  const int row = w * 8 + (lane >> 3), ch = ((lane & 7) ^ ((row >> 1) & 7)) * 8;
  const int va = (row * a.lda + ch) * 2, vb = (row * a.ldb + ch) * 2, sa = 64 * a.lda, sb = 64 * a.ldb;
  auto load = [&](int t) {  // K-tile t (zeros past K) into its stage
    char* dst = smem + (t % ST) * STAGE;
    const bool in = t * BK + ch < K;
    const int oa = in ? va : OOB, ob = in ? vb : OOB;
#pragma unroll
    for (int j = 0; j < LA; ++j)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (KGS_LDS void*)(dst + (j * 4 + w) * 1024), 16, oa, j * sa + t * 128, 0, 0);
#pragma unroll
    for (int j = 0; j < LB; ++j)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, (KGS_LDS void*)(dst + BM * 128 + (j * 4 + w) * 1024), 16, ob, j * sb + t * 128, 0, NT ? 2 : 0);
  };
  const int fr = lane & 15, fq = lane >> 4;
  const int ro = fr * 128 + ((fq ^ (fr >> 1)) * 16);
  const int pa = (w >> 1) * (BM / 2) * 128 + ro, pb = BM * 128 + (w & 1) * (BN / 2) * 128 + ro;
  f32x4 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int n = 0; n < FN; ++n) acc[i][n] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int t = 0; t < ST - 1; ++t) load(t);
  for (int t = 0; t < nt; ++t) {
    w4::wait_vm<(ST - 2) * (LA + LB)>();  // own part of K-tile t
    w4::bar();  // every wave's part, and every wave has read K-tile t - 1
    load(t + ST - 1);
    const char* st = smem + (t % ST) * STAGE;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      bf16x8 fa[FM], fb[FN];
#pragma unroll
      for (int i = 0; i < FM; ++i) fa[i] = *(const bf16x8*)(st + ((pa + i * 2048) ^ (ks * 64)));
#pragma unroll
      for (int n = 0; n < FN; ++n) fb[n] = *(const bf16x8*)(st + ((pb + n * 2048) ^ (ks * 64)));
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int n = 0; n < FN; ++n) {
          if constexpr (F8) {
            const auto x = __builtin_bit_cast(i64x2, fa[i]), y = __builtin_bit_cast(i64x2, fb[n]);
            acc[i][n] = __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(y[0], x[0], acc[i][n], 0, 0, 0);
            acc[i][n] = __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(y[1], x[1], acc[i][n], 0, 0, 0);
          } else {
            acc[i][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[n], fa[i], acc[i][n], 0, 0, 0);
          }
        }
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the tail's loads land before LDS is released
  if constexpr (F8) {
    const float f = a.alpha_ptr ? a.alpha * *a.alpha_ptr : a.alpha;
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int n = 0; n < FN; ++n) acc[i][n] *= f;
  }
  const int mw = m0 + (w >> 1) * (BM / 2) + fr, nw = n0 + (w & 1) * (BN / 2);
  const int lc = (fq & 1) * 16 + (fq >> 1) * 8;
  float bv[FN][4];
  load_bias<EPI, FN>(a, nw + fq * 4, bv);
#pragma unroll
  for (int i = 0; i < FM; ++i) {
    uint4 old[FN / 2];
    load_old<EPI, FN>(a, mw + i * 16, nw + lc, old);
    store_row<EPI, FN, DUAL>(a, mw + i * 16, nw + lc, acc[i], bv, old);
  }
}

// act(A . gate^T) * (A . up^T) of few rows, B = [gate; up] of 2 I rows: BM rows by 32 outputs, whose gate and up columns
// (16 of each in turn) one wave holds. For grids that 128-wide tiles leave short of the CUs: what else fills them
// there, K slices, costs their fp32 partial products' way through memory and a launch that sums them. Four stages and one
// barrier per K-step as gemm_small, and its order of products per element. Bound by the operands' way into LDS: A comes
// whole to every workgroup, 16384x2048 at 100 rows 20 us where 23.6 (0.4 us a K-step). B's loads are non-temporal where its rows are whole
// 128-byte lines (21.0 by default; kgs/ops/decode.py gate_rule has the rule and its other side).
template <int BM, int SW>
__global__ __launch_bounds__(256) void gemm_gate(Args a) {
  constexpr int BN = 64, ST = 4, FM = BM / 32, LA = BM / 32, LB = BN / 32, STAGE = (BM + BN) * 128;
  __shared__ __attribute__((aligned(1024))) char smem[ST * STAGE];
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int I = a.N / 2, ntm = (a.M + BM - 1) / BM, ntn = (I + 31) / 32;
  int none, tm, tn;
  w4::tile_of<0, false>((int)blockIdx.x, (int)gridDim.x, ntm, ntn, none, tm, tn);
  const int m0 = tm * BM, n0 = tn * 32, K = a.K, nt = (K + BK - 1) / BK;
  const int na = min(a.M - m0, BM), nb = min(I - n0, 32);
  // waves 0 and 1 stage gate rows, 2 and 3 up rows: 16 of each per 32-row group
  const auto ra = __builtin_amdgcn_make_buffer_rsrc((void*)(a.A + (long)m0 * a.lda), 0, ((na - 1) * a.lda + K) * 2, 0x00020000);
  const auto rb = __builtin_amdgcn_make_buffer_rsrc((void*)(a.B + ((long)(w >> 1) * I + n0) * a.ldb), 0, ((nb - 1) * a.ldb + K) * 2, 0x00020000);
  const int row = w * 8 + (lane >> 3), ch = ((lane & 7) ^ ((row >> 1) & 7)) * 8;
  const int va = (row * a.lda + ch) * 2, vb = ((row & 15) * a.ldb + ch) * 2, sa = 64 * a.lda, sb = 32 * a.ldb;
  auto load = [&](int t) {  // K-tile t (zeros past K) into its stage
    char* dst = smem + (t % ST) * STAGE;
    const bool in = t * BK + ch < K;
    const int oa = in ? va : OOB, ob = in ? vb : OOB;
#pragma unroll
    for (int j = 0; j < LA; ++j)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (KGS_LDS void*)(dst + (j * 4 + w) * 1024), 16, oa, j * sa + t * 128, 0, 0);
    if (a.ldb % 64 == 0) {
#pragma unroll
      for (int j = 0; j < LB; ++j)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, (KGS_LDS void*)(dst + BM * 128 + (j * 4 + w) * 1024), 16, ob, j * sb + t * 128, 0, 2);
    } else {
#pragma unroll
      for (int j = 0; j < LB; ++j)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, (KGS_LDS void*)(dst + BM * 128 + (j * 4 + w) * 1024), 16, ob, j * sb + t * 128, 0, 0);
    }
  };
  const int fr = lane & 15, fq = lane >> 4;
  const int ro = fr * 128 + ((fq ^ (fr >> 1)) * 16);
  const int pa = (w >> 1) * (BM / 2) * 128 + ro, pb = BM * 128 + (w & 1) * (BN / 2) * 128 + ro;
  f32x4 acc[FM][2];
#pragma unroll
  for (int i = 0; i < FM; ++i) acc[i][0] = acc[i][1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int t = 0; t < ST - 1; ++t) load(t);
  for (int t = 0; t < nt; ++t) {
    w4::wait_vm<(ST - 2) * (LA + LB)>();  // this wave's part of K-tile t
    w4::bar();                            // every wave's part, and every wave has read K-tile t - 1
    load(t + ST - 1);
    const char* st = smem + (t % ST) * STAGE;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      bf16x8 fa[FM], fb[2];
#pragma unroll
      for (int i = 0; i < FM; ++i) fa[i] = *(const bf16x8*)(st + ((pa + i * 2048) ^ (ks * 64)));
#pragma unroll
      for (int n = 0; n < 2; ++n) fb[n] = *(const bf16x8*)(st + ((pb + n * 2048) ^ (ks * 64)));
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int n = 0; n < 2; ++n) acc[i][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[n], fa[i], acc[i][n], 0, 0, 0);
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the tail's loads land before LDS is released
  const float limit = SW == GATE_CLAMPED ? *(const float*)a.bias : 0.f;
  const int col = n0 + (w & 1) * 16 + fq * 4;
#pragma unroll
  for (int i = 0; i < FM; ++i) {
    const int r = m0 + (w >> 1) * (BM / 2) + i * 16 + fr;
    if (r >= a.M || col >= I) continue;
    float y[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) y[e] = gated<SW>(acc[i][0][e], acc[i][1][e], limit);
    *(uint2*)((unsigned short*)a.C + (long)r * a.ldc + col) = make_uint2(pack_bf16x2(y[0], y[1]), pack_bf16x2(y[2], y[3]));
  }
}

// Products with operands stored K-major (A as [K, M], B as [K, N]): Linear's backward pass, whose
// dX = dY . W reads W that way and dW = dY^T . X both operands, at the sizes where transposing them
// first costs more than a smaller tile does (layout_plan below). 128x128 tiles, two workgroups
// per CU, one barrier per 64-wide K-step: K-tile t + 1 is on its way while t is multiplied.
//
// A K-major K-tile is 64 rows of 128 columns (256 B). The 16-byte chunk c of row r lies at
// c ^ 2 (r & 3 | (r >> 3 & 1) << 2), so that the 16 chunks that a half wave of transposed reads
// touches are on 16 bank groups. Rows past K lie outside the resource and arrive as zeros; columns
// past M or N only reach outputs that are not stored. Rows hold whole chunks: sizes of no multiple
// of 8 come with rows padded to one (zeros where they are contracted over).
struct TrArgs {
  const unsigned short* A;
  const unsigned short* B;
  void* C;
  int M, N, K, lda, ldb, ldc, ks, vec;
};

// Four fragments (16 columns each) of k-sub KS of a K-major operand: eight transposed reads and
// their wait in one block, so that no read is in flight where the compiler does not see it.
template <int KS>
__device__ __forceinline__ void tr_read4(bf16x8 (&f)[4], const unsigned (&ad)[4]) {
  bf16x4 v[8];
  asm volatile(
      "ds_read_b64_tr_b16 %0, %8 offset:%c12\n\tds_read_b64_tr_b16 %1, %8 offset:%c13\n\t"
      "ds_read_b64_tr_b16 %2, %9 offset:%c12\n\tds_read_b64_tr_b16 %3, %9 offset:%c13\n\t"
      "ds_read_b64_tr_b16 %4, %10 offset:%c12\n\tds_read_b64_tr_b16 %5, %10 offset:%c13\n\t"
      "ds_read_b64_tr_b16 %6, %11 offset:%c12\n\tds_read_b64_tr_b16 %7, %11 offset:%c13\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]), "=&v"(v[4]), "=&v"(v[5]), "=&v"(v[6]), "=&v"(v[7])
      : "v"(ad[0]), "v"(ad[1]), "v"(ad[2]), "v"(ad[3]), "n"(KS * 8192), "n"(KS * 8192 + 1024)
      : "memory");
#pragma unroll
  for (int i = 0; i < 4; ++i) f[i] = __builtin_shufflevector(v[2 * i], v[2 * i + 1], 0, 1, 2, 3, 4, 5, 6, 7);
}

// One operand of the K-major kernel: TR as described, else K-contiguous as in gemm_nt_any.
template <bool TR>
struct Operand {
  __amdgpu_buffer_rsrc_t r;
  int vo, step, kstep;  // lane's byte offset, bytes between DMA instructions and between K-tiles
  int ch, kn;
  unsigned ro[4];       // fragment reads: byte offsets inside a stage's operand

  __device__ void init(const unsigned short* P, int ld, int p0, int rows, int k0, int kn_, int w, int lane, int half) {
    kn = kn_;
    const int fr = lane & 15, fq = lane >> 4;
    const int n = min(rows - p0, 128);
    if constexpr (TR) {
      r = __builtin_amdgcn_make_buffer_rsrc((void*)(P + (long)k0 * ld + p0), 0, ((kn - 1) * ld + (n + 7) / 8 * 8) * 2, 0x00020000);
      const int row = w * 4 + (lane >> 4);  // of the 16 rows that the four waves' instruction brings
      const int c = (lane & 15) ^ (2 * ((row & 3) | ((row >> 3) & 1) << 2));
      vo = row * ld * 2 + c * 16;
      step = 16 * ld * 2;
      kstep = BK * ld * 2;
      const int q = (lane >> 2) & 3, p = lane & 3, kr = 8 * fq + q;  // a read's row, and its place in it
      const int x = 2 * ((kr & 3) | ((kr >> 3) & 1) << 2);
#pragma unroll
      for (int i = 0; i < 4; ++i) ro[i] = kr * 256 + (((half * 8 + 2 * i) ^ x) + (p >> 1)) * 16 + (p & 1) * 8;
    } else {
      kn = (kn + 7) / 8 * 8;
      r = __builtin_amdgcn_make_buffer_rsrc((void*)(P + (long)p0 * ld + k0), 0, ((n - 1) * ld + kn) * 2, 0x00020000);
      const int row = w * 8 + (lane >> 3);
      ch = ((lane & 7) ^ ((row >> 1) & 7)) * 8;
      vo = (row * ld + ch) * 2;
      step = 32 * ld * 2;
      kstep = BK * 2;
#pragma unroll
      for (int i = 0; i < 4; ++i) ro[i] = (half * 64 + i * 16 + fr) * 128 + ((fq ^ (fr >> 1)) * 16);
    }
  }
  // K-tile t into the 16 KiB at dst
  __device__ void load(char* dst, int t, int w) const {
    const int v = TR || t * BK + ch < kn ? vo : OOB;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (KGS_LDS void*)(dst + (j * 4 + w) * 1024), 16, v, j * step + t * kstep, 0, 0);
  }
  template <int KS>
  __device__ void read(bf16x8 (&f)[4], const char* src) const {
    if constexpr (TR) {
      const unsigned b = (unsigned)(uintptr_t)(const KGS_LDS char*)src;
      const unsigned ad[4] = {b + ro[0], b + ro[1], b + ro[2], b + ro[3]};
      tr_read4<KS>(f, ad);
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) f[i] = *(const bf16x8*)(src + (KS ? ro[i] ^ 64 : ro[i]));
    }
  }
};

// workgroup `id` of the product's `wgs`
template <bool TA, bool TB, bool SPLIT>
__device__ __forceinline__ void tr_tile(const TrArgs& a, char* smem, int id, int wgs) {
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ntm = (a.M + 127) / 128, ntn = (a.N + 127) / 128;
  int slice, tm, tn;
  w4::tile_of<0, SPLIT>(id, wgs, ntm, ntn, slice, tm, tn);
  const int m0 = tm * 128, n0 = tn * 128, k0 = SPLIT ? slice * a.ks : 0;
  const int kn = SPLIT ? min(a.K - k0, a.ks) : a.K, nt = (kn + BK - 1) / BK;
  Operand<TA> oa;
  Operand<TB> ob;
  oa.init(a.A, a.lda, m0, a.M, k0, kn, w, lane, w >> 1);
  ob.init(a.B, a.ldb, n0, a.N, k0, kn, w, lane, w & 1);
  f32x4 acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int n = 0; n < 4; ++n) acc[i][n] = f32x4{0.f, 0.f, 0.f, 0.f};
  oa.load(smem, 0, w);
  ob.load(smem + 16384, 0, w);
  for (int t = 0; t < nt; ++t) {
    char* st = smem + (t & 1) * 32768;
    char* nx = smem + ((t & 1) ^ 1) * 32768;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // own part of K-tile t
    w4::bar();  // every wave's part, and every wave has read K-tile t - 1
    if (t + 1 < nt) {
      oa.load(nx, t + 1, w);
      ob.load(nx + 16384, t + 1, w);
    }
    bf16x8 fa[4], fb[4];
    oa.template read<0>(fa, st);
    ob.template read<0>(fb, st + 16384);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int n = 0; n < 4; ++n) acc[i][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[n], fa[i], acc[i][n], 0, 0, 0);
    bf16x8 ga[4], gb[4];
    oa.template read<1>(ga, st);
    ob.template read<1>(gb, st + 16384);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int n = 0; n < 4; ++n) acc[i][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(gb[n], ga[i], acc[i][n], 0, 0, 0);
  }
  const int fr = lane & 15, fq = lane >> 4;
  const int mw = m0 + (w >> 1) * 64 + fr, nw = n0 + (w & 1) * 64;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = mw + i * 16;
    if constexpr (SPLIT) {
      float* prow = (float*)a.C + ((long)slice * a.M + r) * a.ldc;
#pragma unroll
      for (int n = 0; n < 4; ++n) {
        const int col = nw + n * 16 + fq * 4;
        if (r < a.M && col < a.ldc) *(f32x4*)(prow + col) = acc[i][n];
      }
    } else {
      unsigned short* crow = (unsigned short*)a.C + (long)r * a.ldc;
#pragma unroll
      for (int n = 0; n < 4; n += 2) {
        uint2 o[2];
#pragma unroll
        for (int h = 0; h < 2; ++h)
          o[h] = make_uint2(pack_bf16x2(acc[i][n + h][0], acc[i][n + h][1]), pack_bf16x2(acc[i][n + h][2], acc[i][n + h][3]));
        auto sx = __builtin_amdgcn_permlane16_swap(o[0].x, o[1].x, false, false);
        auto sy = __builtin_amdgcn_permlane16_swap(o[0].y, o[1].y, false, false);
        const int col = nw + n * 16 + (fq & 1) * 16 + (fq >> 1) * 8;
        if (r < a.M && col < a.N) store8(crow, col, a.N, a.vec, make_uint4(sx[0], sy[0], sx[1], sy[1]));
      }
    }
  }
}

template <bool TA, bool TB, bool SPLIT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void gemm_tr(TrArgs a) {
  __shared__ __attribute__((aligned(1024))) char smem[2 * 32768];
  tr_tile<TA, TB, SPLIT>(a, smem, (int)blockIdx.x, (int)gridDim.x);
}

// A layer's two gradient products in one launch, dX = dY . W (its workgroups first) and dW = dY^T . X, the tiles of
// gemm_tr and their bits. Layers of up to about a thousand rows are bound by the launches (some 4 us of host time each), and leave CUs
// idle in either product. us, a training step by two launches / one: 64 rows, three layers, 512 - 2048 - 512 216 / 204;
// 256 rows, three of 1024 219 / 202; 777 rows 768 - 3072 - 768 230 / 214; 1024 rows, two layers, 1024 - 4096 - 1024 186 / 175; from 2048 rows the
// same time, and large grids go one by one (gemm_tr_pair below).
template <bool SPLIT0, bool SPLIT1>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void gemm_tr_pair(TrArgs x, TrArgs w, int wgx) {
  __shared__ __attribute__((aligned(1024))) char smem[2 * 32768];
  const int id = (int)blockIdx.x;
  if (id < wgx) tr_tile<false, true, SPLIT0>(x, smem, id, wgx);
  else tr_tile<true, true, SPLIT1>(w, smem, id - wgx, (int)gridDim.x - wgx);
}

// Sum of the K slices' partial tiles (fp32 [ns][M][ldp]) and the epilogue: a thread's 8 columns
// of one row, every slice's loads issued before the first add. Bound by memory: ns + 0.5 passes.
template <int EPI, bool DUAL>
__global__ __launch_bounds__(256) void any_reduce(const float* __restrict__ P, unsigned short* __restrict__ C,
                                                  unsigned short* __restrict__ C2, const unsigned short* __restrict__ bias,
                                                  int M, int N, int ldc, int ldp, int ns, int vec) {
  const int per = ldp / 8;
  const long id = (long)blockIdx.x * 256 + threadIdx.x;
  if (id >= (long)M * per) return;
  const int row = (int)(id / per), col = (int)(id - (long)row * per) * 8;
  const float* p = P + (long)row * ldp + col;
  const long step = (long)M * ldp;
  f32x4 s0 = *(const f32x4*)p, s1 = *(const f32x4*)(p + 4);
  for (int s = 1; s < ns; s += 4) {
    f32x4 u[4], v[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float* q = p + min(s + e, ns - 1) * step;
      u[e] = *(const f32x4*)q;
      v[e] = *(const f32x4*)(q + 4);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (s + e < ns) {
        s0 += u[e];
        s1 += v[e];
      }
  }
  float b[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    b[e] = 0.f;
    if constexpr (epi_bias<EPI>())
      if (bias && col + e < N) b[e] = bf2f(bias[col + e]);
  }
  constexpr int E = DUAL ? EPI_BIAS : EPI;
  uint4 q = make_uint4(pack_epi<E>(s0[0], s0[1], b[0], b[1]), pack_epi<E>(s0[2], s0[3], b[2], b[3]),
                       pack_epi<E>(s1[0], s1[1], b[4], b[5]), pack_epi<E>(s1[2], s1[3], b[6], b[7]));
  unsigned short* crow = C + (long)row * ldc;
  if constexpr (EPI == EPI_ADDC) q = add_bf16x8(*(const uint4*)(crow + col), q);
  store8(crow, col, N, vec, q);
  if constexpr (DUAL)
    store8(C2 + (long)row * ldc, col, N, vec,
           make_uint4(act_pair<EPI>(q.x), act_pair<EPI>(q.y), act_pair<EPI>(q.z), act_pair<EPI>(q.w)));
}

typedef short bf16x8u __attribute__((ext_vector_type(8), aligned(2)));

// Rows of any length at any 2-byte alignment into rows of whole 16-byte chunks, zeros past the
// last column, of one or two matrices: what the kernels' 16-byte loads can read. Bound by memory
// (6624 x 2243 5.1 TB/s; small ones the launch, 2.6 us). us by the kernel that reads such operands
// element by element / by this and the fast tiles: 16 x 64 x 2467 162 / 11, 128 x 128 x 401 55 / 10,
// 4096 x 4096 x 2467 1204 / 92; they meet near K = 32 (16 x 64 x 33 5.2 / 5.8).
struct PadArgs {
  const unsigned short* src[2];
  unsigned short* dst[2];
  long rows[2];
  int cols[2];
  long ld[2];
};
__global__ __launch_bounds__(256) void pad_rows(PadArgs a) {
  const int per[2] = {(a.cols[0] + 7) / 8, (a.cols[1] + 7) / 8};
  const long first = a.rows[0] * per[0], all = first + a.rows[1] * per[1];
  for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < all; i += (long)gridDim.x * 256) {
    const int o = i >= first;
    const long j = o ? i - first : i, n = o ? per[1] : per[0], row = j / n;
    const int c = (int)(j - row * n) * 8, cols = o ? a.cols[1] : a.cols[0];
    const unsigned short* s = (o ? a.src[1] : a.src[0]) + row * (o ? a.ld[1] : a.ld[0]) + c;
    bf16x8 v = {0, 0, 0, 0, 0, 0, 0, 0};
    if (c + 8 <= cols) {
      v = *(const bf16x8u*)s;
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (c + e < cols) v[e] = (short)s[e];
    }
    *(bf16x8*)((o ? a.dst[1] : a.dst[0]) + j * 8) = v;
  }
}

struct Plan {
  int bm, bn, ns;
};

inline int ceil_div(long a, long b) { return (int)((a + b - 1) / b); }

// Whether the two-stage tiles of an unsliced launch take turns (tile_product) when they are more than a round: not for long sums over rows off the
// 128-byte lines (us, a workgroup a tile / taking turns: 4000 x 6000 x 2000 108 / 116, of 2048 91.5 / 91.6; 6000 x 9000 x 3000 295 / 304.5, 6144 x 9216 x 3072 278 / 272)
inline bool turns_pay(const void* A, const void* B, int K, int lda, int ldb) {
  return (lda % 64 == 0 && ldb % 64 == 0 && ((uintptr_t)A | (uintptr_t)B) % 128 == 0) || K <= 1024;
}

// An unsliced launch of tiles with a CU each. Those of 128 columns run on lds_stages but for K of 65 to 128, all of which two stages hold: there is no
// difference (192x128 tiles of 965 x 5456 x 72 and x 128 9.8, 9.8 us on two, 9.8, 9.7 on three), while of one K-tile two stages walk two (x 64 9.9 / 8.9; 4000 x 6000 x 64 by
// 224x128 20.2 / 18.2).
template <int EPI, int BM, int BN, bool DUAL, int SW = 0>
void launch_mid(const Args& a, hipStream_t s) {
  const long tiles = (long)ceil_div(a.M, BM) * (SW ? ceil_div(a.N / 2, BN / 2) : ceil_div(a.N, BN));
  if constexpr (BN != 128) {
    if (tiles > cu_count() && turns_pay(a.A, a.B, a.K, a.lda, a.ldb))
      if (int* q = tile_queue_row(s)) {  // null in a capture: a workgroup a tile
        hipLaunchKernelGGL((gemm_nt_turn<EPI, BM, BN, DUAL, SW>), dim3((unsigned)cu_count()), dim3(256), 0, s, a, q);
        return;
      }
  } else if (a.K <= BK || a.K > 2 * BK) {
    hipLaunchKernelGGL((gemm_nt_deep<EPI, BM, BN, DUAL, SW>), dim3((unsigned)tiles), dim3(256), 0, s, a);
    return;
  }
  if constexpr (BM == 256 && BN == 256) hipLaunchKernelGGL((gemm_nt_any<EPI, BM, BN, false, DUAL, SW>), dim3((unsigned)tiles), dim3(256), 0, s, a);
  else hipLaunchKernelGGL((gemm_nt_mid<EPI, BM, BN, DUAL, SW>), dim3((unsigned)tiles), dim3(256), 0, s, a);
}

// Microseconds of a launch, as measured on an MI355X (weights streamed from HBM).
inline double cost(long M, long N, long K, int bm, int bn, int ns, int cus) {
  const int pairs = ceil_div(K, 128), steps = 2 * ceil_div(pairs, ns);
  const long wg = (long)ceil_div(M, bm) * ceil_div(N, bn) * ns;
  const int share = bm == 128 && bn == 128 ? 2 : 1;  // workgroups that one CU runs at a time
  const double full = (double)wg / cus;
  // a K-step's time by how full the chip is, one workgroup per CU
  const double busy = full < 1 ? full : 1;
  double step = bm == 256 ? (bn == 256 ? 0.92 + 0.30 * busy : 0.62 + 0.18 * busy) : 0.46 + 0.08 * busy;
  double rounds = ceil_div(wg, cus);
  if (share == 2 && full > 1) {  // pairs of workgroups overlap
    const int two = (int)(wg / (2L * cus)), rest = (int)(wg - 2L * cus * two);
    rounds = two * 1.5 + (rest > cus ? 1.5 : rest > 0 ? 1 : 0);
  }
  double t = 4 + rounds * steps * step;
  if (ns > 1) t += 4 + (2.0 * ns + 0.5) * M * N * 4 / 5.5e6;
  return t;
}

// The tile and the slices of a product. A slice keeps at least 512 of K: the partial tiles of
// shorter ones cost as much as they save (300 x 304 x 2400: 10.6 us in slices of 640, 9.9 of 384).
// Slices have to promise 15 %: below that the estimate is not sure of them (1024 x 768 x 2048), and
// without them the result keeps the bits that it has in every other layout.
inline Plan plan(long M, long N, long K, bool split, int cus) {
  Plan best{256, 256, 1};
  double t0 = 1e30;
  const int shapes[3][2] = {{256, 256}, {256, 128}, {128, 128}};
  for (auto& s : shapes)
    for (int ns = 1; ns <= 16; ++ns) {
      if (ns > 1 && (!split || K < 512L * ns)) break;
      const double t = cost(M, N, K, s[0], s[1], ns, cus) * (ns > 1 ? 1.15 : 1.0);
      if (t < t0) {
        t0 = t;
        best = {s[0], s[1], ns};
      }
    }
  // 64x64 tiles: a cheaper step, twice as many bytes per product; several share a CU. Up to 64 rows a B of whole 128-byte lines is read once, past
  // the caches, where there are tiles for most CUs: us at 1 to 16 rows by larger tiles / so 32000x4096 57 / 45, 32000x2048 33 / 28,
  // 14336x4096 28 / 25, 128256x4096 at 40 192 / 179, but at 64 196 / 207; off the lines each line comes twice, 89600x1872 at 32 78 / 83
  const bool few = M <= 64 && K % 64 == 0;
  if (few) t0 = t0 > 4 + 2.0 * N * K / 5.0e6 ? t0 : 4 + 2.0 * N * K / 5.0e6;  // few rows: B's way from memory
  const double full = (double)ceil_div(M, 64) * ceil_div(N, 64) / cus, steps = ceil_div(K, 64);
  const double t = few && full >= 0.75 && (M <= 48 || full <= 4) ? 4 + steps * (full <= 1 ? 0.20 + 0.13 * full : 0.33 * full)
                                                                 : 3.5 + steps * (full <= 1 ? 0.34 + 0.06 * full : 0.06 + (few ? 0.43 : 0.38) * full);
  if (t < t0) best = {64, 64, 1};
  return best;
}

// A tile's time in an unsliced product, us, fitted to 310 sizes of 160 to 10000 rows (half of the errors below 6 %; the
// tile that these estimates choose takes 0.8 % more than the best one): start, what each round of workgroups
// after the first adds, and a K-step alone on a CU and what the chip's filling adds to it. 128x128 tiles: of two
// workgroups on a CU, and of the single ones that remain. Tiles of 128 columns (of 128x128 ones the single) scaled to their K-steps of one barrier, by 48
// sizes: 0.33 + 0.13 full where 0.37 + 0.16, of 192 rows 0.40 + 0.25 / 0.42 + 0.29, 224 0.44 + 0.29 / 0.45 + 0.32, 256 0.46 + 0.35 / 0.49 + 0.36. turn: what a
// further round costs tiles that take turns (turns_pay), 1.5 to 2 us less.
struct Tile {
  int bm, bn;
  double start, again, turn, step, fill;
};
constexpr Tile TILES[] = {{256, 256, 7.12, 7.31, 5.3, 0.88, 0.50}, {256, 128, 4.61, 4.53, 4.53, 0.53, 0.28}, {128, 128, 3.5, 3.2, 3.2, 0.97, 0},
                          {192, 128, 4.15, 2.97, 2.97, 0.42, 0.22}, {224, 128, 4.27, 3.53, 3.53, 0.48, 0.25}, {192, 192, 5.02, 4.65, 3.3, 0.56, 0.29},
                          {224, 192, 5.40, 5.14, 3.6, 0.61, 0.35}, {256, 192, 5.90, 5.94, 4.3, 0.67, 0.38}, {224, 256, 6.49, 6.69, 4.9, 0.78, 0.43}};
// The persistent and the eight-wave kernels of 256x256 tiles, as finer and turn_b see them. With the 5.3 us of tiles that take turns for a further round, 36
// products with a K-major B that read it faster on average (up to 29 %: 3584 x 11264 x 384 48.0 us, transposed first 61.9) were transposed first, and 24
// of ragged rows kept to persistent tiles that lose 2 % to finer ones on average (0.92 to 1.03 of their time).
constexpr Tile LARGE = {256, 256, 7.12, 7.31, 7.31, 0.88, 0.50};
inline double tile_cost(const Tile& t, long M, long N, long K, int cus, bool turns) {
  const long wg = (long)ceil_div(M, t.bm) * ceil_div(N, t.bn);
  const int steps = 2 * ceil_div(K, 128);
  if (t.bm == 128) {
    const int two = (int)(wg / (2L * cus)), rest = (int)(wg - 2L * cus * two), pairs = two + (rest > cus);
    const double one = rest > 0 && rest <= cus ? 0.30 + 0.21 * rest / cus : 0;
    return t.start + steps * (pairs * t.step + one) + (two ? t.again * (two - (rest == 0)) : 0);
  }
  const int full = (int)(wg / cus), rest = (int)(wg - (long)full * cus), rounds = full + (rest > 0);
  return t.start + (rounds - 1) * (turns ? t.turn : t.again) + steps * (rounds * t.step + (full + (double)rest / cus) * t.fill);
}
inline double tile_cost(int bm, int bn, long M, long N, long K, int cus, bool turns) {
  for (const Tile& t : TILES)
    if (t.bm == bm && t.bn == bn) return tile_cost(t, M, N, K, cus, turns);
  return 1e30;
}

// The tile of an unsliced product: plan's, or one between its three that leaves fewer CUs idle in the last round. What
// such a product loses is that round (7 x 24 tiles of 256x256 are 168 of 256 CUs, 8 x 32 of 224x192 all of them);
// a K-step of any of these tiles is bound by its operands' way into LDS, 60 bytes per ns and CU, so that the smaller ones are little
// slower per product. The bits are the same. us, plan's tile / this one: 1762 x 6144 x 4096 81 / 66, 2830 x 6144 x 5504 199 / 145,
// 1762 x 28672 x 4096 349 / 309, 590 x 11776 x 3472 75 / 57, 1382 x 6144 x 1152 28 / 21. sw: a gated product's tiles, whose
// waves hold gate and up columns in turn, are 128 or 256 wide.
inline Plan refine(Plan p, long M, long N, long K, int cus, bool turns, bool sw = false) {
  if (p.ns > 1 || p.bm == 64) return p;
  double t0 = tile_cost(p.bm, p.bn, M, N, K, cus, turns) * 0.97;
  for (const Tile& t : TILES) {
    if (sw && t.bn == 192) continue;
    const double c = tile_cost(t, M, N, K, cus, turns);
    if (c < t0) {
      t0 = c;
      p.bm = t.bm;
      p.bn = t.bn;
    }
  }
  return p;
}

// The tile of a gated product (B of N rows, gate and up)
inline Plan gated_plan(long M, long N, long K, int cus, bool turns) {
  const Plan p = plan(M, N, K, false, cus);
  return refine(p.bm == 64 ? Plan{128, 128, 1} : p, M, N, K, cus, turns, true);
}

inline int tile_of_rows(int M, int N, int K, int lda, int ldb, int gated) {
  const bool turns = turns_pay(nullptr, nullptr, K, lda, ldb);
  const int cus = cu_count();
  const Plan p = gated ? gated_plan(M, N, K, cus, turns) : refine(plan(M, N, K, false, cus), M, N, K, cus, turns);
  return p.bm << 16 | p.bn;
}

// Whether a product that the aligned, the persistent or the eight-wave 256x256 kernels take is better off on refine's
// tile here: those keep a little (persistent tiles 3 % on average, 9 % at most) that a tile has to win back first. Of 90 such products whose estimate
// promises 7 to 20 % the tile is 6 % faster on average, 4 % slower at worst (2902 x 13312 x 1536 107 / 112 us, ragged rows). off: rows off the
// 128-byte lines (wide below), where a K-step waits for twice the lines: 20 % have to be promised. us by eight waves / so: 2129 x 3728 x 4616
// 103 / 89 (27 %), 1598 x 5680 x 4144 87 / 86 (22 %); below, what 55 products gain 1 % from on average 7756 x 6320 x 3816 loses 7 % of (349 / 372),
// 3567 x 15328 x 928 6 % (108 / 114).
inline bool finer(long M, long N, long K, int cus, bool turns, bool sw, bool off) {
  const Plan p = refine({256, 256, 1}, M, N, K, cus, turns, sw);
  return p.bm * p.bn < 65536 && tile_cost(p.bm, p.bn, M, N, K, cus, turns) < (off ? 0.80 : 0.93) * tile_cost(LARGE, M, N, K, cus, false);
}

// Whether 256x256 tiles are plan's choice, or so near it that the eight-wave kernel of such tiles
// (gemm_pipeline.h: the same bits) is the faster one where the rows of A start off the 128-byte lines. A K-step of
// the tiles here then waits for twice the lines: 4 to 15 % of a product, of smaller tiles more; the
// eight-wave kernel's loads do not show it. us, tiles by plan / eight waves, A's rows 16 bytes off a line or more
// (both on lines): 3812 x 2240 x 4208 90 / 84 (80 / 80), 7738 x 1320 x 7584 163 / 141, 3653 x 2784 x 712 25.3 / 24.3, 10155 x 4216
// x 3424 256 / 239 (222 / 228); where plan takes smaller tiles 1653 x 14544 x 3552 194 / 157, 3495 x 5248 x 4944 222 / 203, but
// 3508 x 4928 x 888 47 / 49, 1752 x 9960 x 520 32 / 37: the estimates may differ by 3 % above K = 512, 14 % from
// 3072 on, and shorter sums than 256 keep plan's tiles (8121 x 1312 x 160 13.5 / 14.9). B's rows do not matter
// (72.3 / 71.9).
inline bool wide(long M, long N, long K, bool split, int cus) {
  const Plan p = plan(M, N, K, split, cus);
  if (K < 256 || p.ns > 1 || p.bm == 64) return false;
  return cost(M, N, K, 256, 256, 1, cus) <= cost(M, N, K, p.bm, p.bn, 1, cus) * (K >= 3072 ? 1.14 : K > 512 ? 1.03 : 1);
}

// The 256x256 kernel that reads a K-major B transposed (kgs_gemm_bf16), us; sizes of whole tiles. Measured: 2048 x 1024 x 4096 65,
// 4096 x 2048 x 8192 132, 3072^3 58, 4096^3 95, 4096 x 8192 x 2048 106, 4096 x 14336 x 4096 347.
inline double tr256_cost(long M, long N, long K, int cus) {
  const long g = (M / 256) * (N / 256), full = g / cus;
  const double rest = (double)(g - full * cus) / cus, b4 = rest * rest * rest * rest;
  return 8 * (full + (rest > 0)) + K / 64 * (full * 1.36 + (rest > 0 ? 0.88 + 0.15 * rest + 0.33 * b4 : 0));
}

// Whether that kernel loses to a transpose of B (4 bytes a value at 6.4 TB/s) and the product as gemm_nt runs it: where its tiles leave
// most of the CUs idle. us, transposed read / transpose and tiles: 2048 x 1024 x 4096 65 / 38, 4096 x 512 x 4096 65 / 36, 4096 x
// 2048 x 8192 132 / 118; 4096 x 8192 x 2048 106 / 114, 2048 x 14336 x 4096 172 / 217, 8192 x 2048 x 2048 52 / 59. Aligned products of more
// 256x256 tiles than CUs run on these (gemm_bf16.hip aligned_finer): 2304 x 8192 x 6912 255 / 296, 3072 x 6656 x 1536 69 / 83. Of 117 sizes of
// more than 4096 rows that read transposed now 7 % on average, none loses more than 7 (11520 x 10752 x 384 119 / 111).
inline bool turn_b(long M, long N, long K, int cus) {
  const Plan p = refine(plan(M, N, K, true, cus), M, N, K, cus, true);  // rows of a transposed B: as long as the plan takes them
  const bool aligned = M % 256 == 0 && N % 256 == 0 && K % 128 == 0 && (M / 256) * (N / 256) > cus;
  const double nt = aligned ? tile_cost(LARGE, M, N, K, cus, false)
                    : p.ns > 1 || p.bm == 64 ? cost(M, N, K, p.bm == 64 ? 128 : p.bm, p.bm == 64 ? 128 : p.bn, p.ns, cus)
                                             : tile_cost(p.bm, p.bn, M, N, K, cus, true);
  return nt + 2.5 + 4.0 * N * K / 6.4e6 < tr256_cost(M, N, K, cus);
}

// Slices with which gemm_tr is the fastest way to a product with K-major operands, 0 where
// another one is. The others transpose the operands first (a launch and a pass over memory each)
// and run cost()'s best tile, or, for aligned sizes and a K-major B alone, the 256x256 kernel that
// reads it transposed. Measured, us: 2048^3 both K-major 26 here, 42 with transposes; 4096^3 128
// and 105; 64 x 512 x 2048 9.5 in 8 slices and 33. Slices have to promise a quarter of the time
// here: they cost the result the bits that it has in every other layout.
inline int layout_plan(long M, long N, long K, int ta, int tb, int cus) {
  const long wg = (long)ceil_div(M, 128) * ceil_div(N, 128);
  double t0 = 1e30;
  int best = 1;
  for (int ns = 1; ns <= 16; ++ns) {
    if (ns > 1 && K < 512L * ns) break;
    const long n = wg * ns;
    const double busy = n < cus ? (double)n / cus : 1, step = 0.58 + 0.12 * busy;
    const int two = (int)(n / (2L * cus)), rest = (int)(n - 2L * cus * two);
    const double rounds = two * 1.42 + (rest > cus ? 1.42 : rest > 0 ? 1 : 0);
    double t = 4 + rounds * 2 * ceil_div(ceil_div(K, 128), ns) * step;
    if (ns > 1) t = 1.35 * (t + 4 + (2.0 * ns + 0.5) * M * N * 4 / 5.5e6);
    if (t < t0) {
      t0 = t;
      best = ns;
    }
  }
  const double turn_a = ta ? 4 + 4.0 * M * K / 5e6 : 0, turn_b = tb ? 4 + 4.0 * N * K / 5e6 : 0;
  double nt = 1e30;
  for (auto& s : {std::pair<int, int>{256, 256}, {256, 128}, {128, 128}}) {
    const double t = cost(M, N, K, s.first, s.second, 1, cus);
    nt = t < nt ? t : nt;
  }
  if (K % 8) return best;  // nothing else reads such operands 16 bytes at a time
  if (t0 > nt + turn_a + turn_b) return 0;
  // (3 %: few rows of tiles read a K-major B less well than that estimate; 1280 x 5376 x 11776 182 here, 208 there)
  if (M % 256 == 0 && N % 256 == 0 && K % 128 == 0 && tb && t0 > 1.03 * tr256_cost(M, N, K, cus) + turn_a) return 0;
  return best;
}

template <int EPI, int BM, int BN, bool DUAL>
void launch_tile(const Args& a, int ns, hipStream_t s) {
  const dim3 grid((unsigned)(ceil_div(a.M, BM) * ceil_div(a.N, BN) * ns));
  if constexpr (BM == 128 && BN == 128)
    if ((int)grid.x <= cu_count()) {
      if (ns > 1) hipLaunchKernelGGL((gemm_nt_deep<EPI_NONE, BM, BN, false, 0, true>), grid, dim3(256), 0, s, a);
      else hipLaunchKernelGGL((gemm_nt_deep<EPI, BM, BN, DUAL>), grid, dim3(256), 0, s, a);
      return;
    }
  if (ns > 1) hipLaunchKernelGGL((gemm_nt_any<EPI_NONE, BM, BN, true, false>), grid, dim3(256), 0, s, a);
  else if constexpr (BN == 256) launch_mid<EPI, BM, BN, DUAL>(a, s);
  else hipLaunchKernelGGL((gemm_nt_any<EPI, BM, BN, false, DUAL>), grid, dim3(256), 0, s, a);
}

template <int EPI, bool DUAL>
int launch(Args a, Plan p, float* ws, hipStream_t s) {
  if (p.bm == 64) {
    const dim3 grid((unsigned)(ceil_div(a.M, 64) * ceil_div(a.N, 64)));
    if constexpr (!DUAL)
      if (a.M <= 64 && grid.x >= 64 && a.ldb % 64 == 0) {
        hipLaunchKernelGGL((gemm_small<EPI, false, false, true>), grid, dim3(256), 0, s, a);
        return (int)hipGetLastError();
      }
    hipLaunchKernelGGL((gemm_small<EPI, DUAL>), grid, dim3(256), 0, s, a);
    return (int)hipGetLastError();
  }
  Args g = a;
  const int ldp = (a.N + 7) / 8 * 8;
  g.ks = ceil_div(ceil_div(a.K, 128), p.ns) * 128;
  p.ns = ceil_div(a.K, g.ks);  // no empty slice
  if (p.ns > 1) {
    g.C = ws;
    g.ldc = ldp;
  }
  if (p.ns > 1 && (p.bn == 192 || (p.bm != 128 && p.bm != 256))) return KGS_ERR_ARG;  // slices run on plan's tiles
#define KGS_MID(BM, BN) \
  case BM << 16 | BN: launch_mid<EPI, BM, BN, DUAL>(g, s); break
  switch (p.bm << 16 | p.bn) {
    case 128 << 16 | 128: launch_tile<EPI, 128, 128, DUAL>(g, p.ns, s); break;
    case 256 << 16 | 128: launch_tile<EPI, 256, 128, DUAL>(g, p.ns, s); break;
    case 256 << 16 | 256: launch_tile<EPI, 256, 256, DUAL>(g, p.ns, s); break;
    KGS_MID(192, 128);
    KGS_MID(224, 128);
    KGS_MID(192, 192);
    KGS_MID(224, 192);
    KGS_MID(256, 192);
    KGS_MID(224, 256);
    default: return KGS_ERR_ARG;
  }
#undef KGS_MID
  if (p.ns > 1)
    hipLaunchKernelGGL((any_reduce<EPI, DUAL>), dim3((unsigned)ceil_div((long)a.M * (ldp / 8), 256)), dim3(256), 0, s, ws,
                       (unsigned short*)a.C, a.C2, a.bias, a.M, a.N, a.ldc, ldp, p.ns, a.vec);
  return (int)hipGetLastError();
}

}  // namespace any

// The operands gemm_tr takes: rows of whole 16-byte chunks, readable (and zero where contracted
// over) to the next one, 32-bit offsets over K.
int gemm_tr_ok(const void* A, const void* B, int M, int N, int K, int lda, int ldb, int ta, int tb) {
  // lda, ldb are multiples of 8 and so hold the padded rows too
  if (M <= 0 || N <= 0 || K <= 0 || lda % 8 || ldb % 8 || lda < (ta ? M : K) || ldb < (tb ? N : K)) return 0;
  if ((uintptr_t)A % 16 || (uintptr_t)B % 16) return 0;
  const long ea = ta ? (long)(K + 128) * lda : 256L * lda, eb = tb ? (long)(K + 128) * ldb : 256L * ldb;
  if (2 * ea >= any::OOB || 2 * eb >= any::OOB) return 0;
  return ((long)M + 127) / 128 * (((long)N + 127) / 128) * 64 < (1L << 31);
}

// A product's arguments, its slices as they come out (of ns asked for) and its workgroups
inline any::TrArgs tr_args(const void* A, const void* B, void* C, int M, int N, int K, int lda, int ldb, int ldc, int& ns, float* ws,
                           unsigned& wgs) {
  using namespace any;
  TrArgs a{(const unsigned short*)A, (const unsigned short*)B, C, M, N, K, lda, ldb, ldc, 0,
           ldc % 8 == 0 && (uintptr_t)C % 16 == 0};
  a.ks = ceil_div(ceil_div(K, 128), ns) * 128;
  ns = ceil_div(K, a.ks);
  if (ns > 1) {
    a.C = ws;
    a.ldc = (N + 7) / 8 * 8;
  }
  wgs = (unsigned)(ceil_div(M, 128) * ceil_div(N, 128) * ns);
  return a;
}

inline void tr_reduce(const any::TrArgs& a, void* C, int ldc, int ns, float* ws, hipStream_t s) {
  using namespace any;
  if (ns < 2) return;
  hipLaunchKernelGGL((any_reduce<EPI_NONE, false>), dim3((unsigned)ceil_div((long)a.M * (a.ldc / 8), 256)), dim3(256), 0, s, ws,
                     (unsigned short*)C, nullptr, nullptr, a.M, a.N, ldc, a.ldc, ns, a.vec);
}

int gemm_tr(const void* A, const void* B, void* C, int M, int N, int K, int lda, int ldb, int ldc, int ta, int tb, int ns,
            float* ws, hipStream_t s) {
  using namespace any;
  unsigned wgs;
  const TrArgs a = tr_args(A, B, C, M, N, K, lda, ldb, ldc, ns, ws, wgs);
  if (ns > 1 && !ws) return KGS_ERR_ARG;
#define KGS_TR(TA, TB)                                                                            \
  if (ns > 1) hipLaunchKernelGGL((any::gemm_tr<TA, TB, true>), dim3(wgs), dim3(256), 0, s, a);    \
  else hipLaunchKernelGGL((any::gemm_tr<TA, TB, false>), dim3(wgs), dim3(256), 0, s, a)
  if (ta && tb) { KGS_TR(true, true); }
  else if (ta) { KGS_TR(true, false); }
  else if (tb) { KGS_TR(false, true); }
  else return KGS_ERR_ARG;
#undef KGS_TR
  tr_reduce(a, C, ldc, ns, ws, s);
  return (int)hipGetLastError();
}

// dX [m, k] = dY [m, n] . W [n, k] and dW [n, k] = dY^T . X [m, k]
int gemm_tr_pair(const void* dY, const void* W, const void* X, void* dX, void* dW, int m, int n, int k, int ldy, int ldw, int ldx,
                 int nsx, int nsw, float* wsx, float* wsw, hipStream_t s) {
  using namespace any;
  unsigned gx, gw;
  const TrArgs x = tr_args(dY, W, dX, m, k, n, ldy, ldw, k, nsx, wsx, gx), w = tr_args(dY, X, dW, n, k, m, ldy, ldx, k, nsw, wsw, gw);
  if ((nsx > 1 && !wsx) || (nsw > 1 && !wsw)) return KGS_ERR_ARG;
  // Two rounds of two workgroups a CU: beyond, neither launch leaves CUs idle for long and the mixed one loses (us, two launches / one: 1500
  // rows, three layers of 2048, 448 tiles each, 266 / 229; 3000 rows, 1536 - 6144 - 1536, up to 1728 tiles, 540 / 544)
  if ((long)gx + gw > 4L * cu_count()) {
    const int rc = gemm_tr(dY, W, dX, m, k, n, ldy, ldw, k, 0, 1, nsx, wsx, s);
    return rc ? rc : gemm_tr(dY, X, dW, n, k, m, ldy, ldx, k, 1, 1, nsw, wsw, s);
  }
  const dim3 grid(gx + gw);
  if (nsx > 1 && nsw > 1) hipLaunchKernelGGL((any::gemm_tr_pair<true, true>), grid, dim3(256), 0, s, x, w, (int)gx);
  else if (nsx > 1) hipLaunchKernelGGL((any::gemm_tr_pair<true, false>), grid, dim3(256), 0, s, x, w, (int)gx);
  else if (nsw > 1) hipLaunchKernelGGL((any::gemm_tr_pair<false, true>), grid, dim3(256), 0, s, x, w, (int)gx);
  else hipLaunchKernelGGL((any::gemm_tr_pair<false, false>), grid, dim3(256), 0, s, x, w, (int)gx);
  tr_reduce(x, dX, k, nsx, wsx, s);
  tr_reduce(w, dW, k, nsw, wsw, s);
  return (int)hipGetLastError();
}

// The operands the kernel takes: 16-byte rows and chunks, 32-bit offsets over a tile's rows.
int gemm_any_ok(const void* A, const void* B, int M, int N, int K, int lda, int ldb) {
  if (M <= 0 || N <= 0 || K <= 0 || K % 8 || lda % 8 || ldb % 8) return 0;
  if ((uintptr_t)A % 16 || (uintptr_t)B % 16) return 0;
  if ((long)lda * 512 >= any::OOB || (long)ldb * 512 >= any::OOB) return 0;
  return ((long)M + 127) / 128 * (((long)N + 127) / 128) * 16 < (1L << 31);
}

// C2: DUAL's second output, else null. bm, bn, ns: 0 for the plan's choice. ws: fp32 scratch for
// the plan's slices (kgs_gemm_bf16_nt_scratch), null: no slices.
int gemm_any(const void* A, const void* B, void* C, void* C2, const void* bias, int M, int N, int K, int lda, int ldb,
             int ldc, int epi, int bm, int bn, int ns, float* ws, hipStream_t s) {
  using namespace any;
  const int vec = ldc % 8 == 0 && (uintptr_t)C % 16 == 0 && (uintptr_t)C2 % 16 == 0;
  if (epi == EPI_ADDC && (!vec || N % 8)) return KGS_ERR_ALIGN;
  const Plan p = bm ? Plan{bm, bn, ns} : refine(plan(M, N, K, ws != nullptr, cu_count()), M, N, K, cu_count(), turns_pay(A, B, K, lda, ldb));
  if (p.ns > 1 && ws == nullptr) return KGS_ERR_ARG;
  const Args a{(const unsigned short*)A, (const unsigned short*)B, C, (unsigned short*)C2, (const unsigned short*)bias,
               M, N, K, lda, ldb, ldc, 0, M > N, vec, 1.f, nullptr};
  if (C2) {
    switch (epi) {
      case EPI_BIAS_GELU: return launch<EPI_BIAS_GELU, true>(a, p, ws, s);
      case EPI_BIAS_RELU: return launch<EPI_BIAS_RELU, true>(a, p, ws, s);
      case EPI_BIAS_SILU: return launch<EPI_BIAS_SILU, true>(a, p, ws, s);
      default: return KGS_ERR_ARG;
    }
  }
  switch (epi) {
    case EPI_NONE: return launch<EPI_NONE, false>(a, p, ws, s);
    case EPI_BIAS: return launch<EPI_BIAS, false>(a, p, ws, s);
    case EPI_BIAS_GELU: return launch<EPI_BIAS_GELU, false>(a, p, ws, s);
    case EPI_BIAS_RELU: return launch<EPI_BIAS_RELU, false>(a, p, ws, s);
    case EPI_BIAS_SILU: return launch<EPI_BIAS_SILU, false>(a, p, ws, s);
    case EPI_ADDC: return launch<EPI_ADDC, false>(a, p, ws, s);
    default: return KGS_ERR_ARG;
  }
}

// C [M, N / 2] = act(A . gate^T) * (A . up^T), B = [gate; up] of N rows (launch_w4p_swiglu for
// prompts): the largest tile whose grid fills the chip
int gemm_any_swiglu(const void* A, const void* B, void* C, int M, int N, int K, int lda, int ldb, int ldc, int act,
                    const float* limit, hipStream_t s) {
  using namespace any;
  const Args a{(const unsigned short*)A, (const unsigned short*)B, C, nullptr, (const unsigned short*)limit,
               M, N, K, lda, ldb, ldc, 0, M > N, ldc % 8 == 0 && (uintptr_t)C % 16 == 0, 1.f, nullptr};
  const Plan p = gated_plan(M, N, K, cu_count(), turns_pay(A, B, K, lda, ldb));
  const dim3 grid((unsigned)(ceil_div(M, p.bm) * ceil_div(N / 2, p.bn / 2)));
  const bool one = (int)grid.x <= cu_count();
#define KGS_SWT(ACT)                                                                                                                     \
  switch (p.bm << 16 | p.bn) {                                                                                                          \
    case 128 << 16 | 128:                                                                                                               \
      if (one) hipLaunchKernelGGL((gemm_nt_deep<EPI_NONE, 128, 128, false, ACT>), grid, dim3(256), 0, s, a);                            \
      else hipLaunchKernelGGL((gemm_nt_any<EPI_NONE, 128, 128, false, false, ACT>), grid, dim3(256), 0, s, a);                          \
      break;                                                                                                                            \
    case 256 << 16 | 128: hipLaunchKernelGGL((gemm_nt_any<EPI_NONE, 256, 128, false, false, ACT>), grid, dim3(256), 0, s, a); break;    \
    case 256 << 16 | 256: launch_mid<EPI_NONE, 256, 256, false, ACT>(a, s); break;                                                      \
    case 192 << 16 | 128: launch_mid<EPI_NONE, 192, 128, false, ACT>(a, s); break;                                                      \
    case 224 << 16 | 128: launch_mid<EPI_NONE, 224, 128, false, ACT>(a, s); break;                                                      \
    case 224 << 16 | 256: launch_mid<EPI_NONE, 224, 256, false, ACT>(a, s); break;                                                      \
    default: return KGS_ERR_ARG;                                                                                                        \
  }
  if (act == GATE_CLAMPED) {
    KGS_SWT(GATE_CLAMPED)
  } else if (act == GATE_GELU) {
    KGS_SWT(GATE_GELU)
  } else {
    KGS_SWT(GATE_SILU)
  }
#undef KGS_SWT
  return (int)hipGetLastError();
}

// C [M, I] = act(A . gate^T) * (A . up^T), B = [gate; up] of N = 2 I rows, on tiles of bm (64, 128) rows by 32 outputs
int gemm_gate(const void* A, const void* B, void* C, int M, int N, int K, int lda, int ldb, int ldc, int bm, int act,
              const float* limit, hipStream_t s) {
  using namespace any;
  const Args a{(const unsigned short*)A, (const unsigned short*)B, C, nullptr, (const unsigned short*)limit,
               M, N, K, lda, ldb, ldc, 0, 0, 1, 1.f, nullptr};
  const dim3 grid((unsigned)(ceil_div(M, bm) * ceil_div(N / 2, 32)));
#define KGS_GATE(ACT)                                                                                  \
  if (bm == 64) hipLaunchKernelGGL((any::gemm_gate<64, ACT>), grid, dim3(256), 0, s, a);               \
  else hipLaunchKernelGGL((any::gemm_gate<128, ACT>), grid, dim3(256), 0, s, a)
  if (act == GATE_CLAMPED) { KGS_GATE(GATE_CLAMPED); }
  else if (act == GATE_GELU) { KGS_GATE(GATE_GELU); }
  else { KGS_GATE(GATE_SILU); }
#undef KGS_GATE
  return (int)hipGetLastError();
}

// e4m3 operands on 64x64 tiles, sizes in 16-bit words (kgs_gemm_fp8_nt_dev)
int gemm_any_f8(const void* A, const void* B, void* C, const void* bias, int M, int N, int Kw, int lda, int ldb, int ldc,
                float alpha, const float* alpha_ptr, int epi, hipStream_t s) {
  using namespace any;
  if (!gemm_any_ok(A, B, M, N, Kw, lda, ldb)) return KGS_ERR_ALIGN;
  const Args a{(const unsigned short*)A, (const unsigned short*)B, C, nullptr, (const unsigned short*)bias, M, N, Kw, lda, ldb,
               ldc, 0, 0, ldc % 8 == 0 && (uintptr_t)C % 16 == 0, alpha, alpha_ptr};
  const dim3 grid((unsigned)(ceil_div(M, 64) * ceil_div(N, 64)));
#define KGS_F8(E) hipLaunchKernelGGL((gemm_small<E, false, true>), grid, dim3(256), 0, s, a)
  switch (epi) {
    case EPI_NONE: KGS_F8(EPI_NONE); break;
    case EPI_BIAS: KGS_F8(EPI_BIAS); break;
    case EPI_BIAS_GELU: KGS_F8(EPI_BIAS_GELU); break;
    case EPI_BIAS_RELU: KGS_F8(EPI_BIAS_RELU); break;
    case EPI_BIAS_SILU: KGS_F8(EPI_BIAS_SILU); break;
    default: return KGS_ERR_ARG;
  }
#undef KGS_F8
  return (int)hipGetLastError();
}

bool gemm_any_finer(const void* A, const void* B, int M, int N, int K, int lda, int ldb, bool sw, bool off) {
  return any::finer(M, N, K, cu_count(), any::turns_pay(A, B, K, lda, ldb), sw, off);
}

bool gemm_any_wide(int M, int N, int K, bool split) { return any::wide(M, N, K, split, cu_count()); }

// fp32 values of scratch that a product's slices need (0: it has none)
long gemm_any_ws(int M, int N, int K) {
  const any::Plan p = any::plan(M, N, K, true, cu_count());
  return p.ns > 1 ? (long)p.ns * M * ((N + 7) / 8 * 8) : 0;
}

}  // namespace kgs

// Copies of one or two (src2 null: one) bf16 matrices with rows of cols rounded up to 8, zeros in
// the added columns. dst 16-B aligned, contiguous.
KGS_EXPORT int kgs_pad_rows_bf16(const void* src, void* dst, long rows, int cols, long ld, const void* src2, void* dst2,
                                 long rows2, int cols2, long ld2, hipStream_t s) {
  using namespace kgs::any;
  if (!src2) rows2 = cols2 = 0;
  if (rows <= 0 || cols <= 0 || ld < cols || (src2 && (rows2 <= 0 || cols2 <= 0 || ld2 < cols2))) return KGS_ERR_SHAPE;
  if ((uintptr_t)src % 2 || (uintptr_t)dst % 16 || (uintptr_t)src2 % 2 || (uintptr_t)dst2 % 16) return KGS_ERR_ALIGN;
  const PadArgs a{{(const unsigned short*)src, (const unsigned short*)src2}, {(unsigned short*)dst, (unsigned short*)dst2},
                  {rows, rows2}, {cols, cols2}, {ld, ld2}};
  const long n = rows * ((cols + 7) / 8) + rows2 * ((cols2 + 7) / 8), wg = (n + 255) / 256;
  hipLaunchKernelGGL(pad_rows, dim3((unsigned)(wg < 4096 ? wg : 4096)), dim3(256), 0, s, a);
  return (int)hipGetLastError();
}

// A product with K-major operands (ta, tb: stored [K][rows]) read in place on 128 x 128 tiles over
// ns K slices (ws: ns M (N rounded up to 8) fp32 values when ns > 1).
KGS_EXPORT int kgs_gemm_bf16_tr(const void* A, const void* B, void* C, int M, int N, int K, int lda, int ldb, int ldc,
                                int ta, int tb, int ns, float* ws, hipStream_t s) {
  if (M <= 0 || N <= 0 || K <= 0 || ldc < N || ns < 1 || ns > 64) return KGS_ERR_SHAPE;
  if (!kgs::gemm_tr_ok(A, B, M, N, K, lda, ldb, ta, tb) || (uintptr_t)ws % 16) return KGS_ERR_ALIGN;
  return kgs::gemm_tr(A, B, C, M, N, K, lda, ldb, ldc, ta, tb, ns, ws, s);
}

// A linear layer's gradients in one launch, as two kgs_gemm_bf16_tr calls leave them: dX [m, k] = dY [m, n] . W [n, k] over nsx slices
// of n (wsx: nsx m (k rounded up to 8) fp32 values if nsx > 1) and dW [n, k] = dY^T . X [m, k] over nsw of m (wsw alike).
KGS_EXPORT int kgs_gemm_bf16_tr_pair(const void* dY, const void* W, const void* X, void* dX, void* dW, int m, int n, int k, int ldy,
                                     int ldw, int ldx, int nsx, int nsw, float* wsx, float* wsw, hipStream_t s) {
  if (m <= 0 || n <= 0 || k <= 0 || nsx < 1 || nsx > 64 || nsw < 1 || nsw > 64) return KGS_ERR_SHAPE;
  if (!kgs::gemm_tr_ok(dY, W, m, k, n, ldy, ldw, 0, 1) || !kgs::gemm_tr_ok(dY, X, n, k, m, ldy, ldx, 1, 1)) return KGS_ERR_ALIGN;
  if ((uintptr_t)wsx % 16 || (uintptr_t)wsw % 16) return KGS_ERR_ALIGN;
  return kgs::gemm_tr_pair(dY, W, X, dX, dW, m, n, k, ldy, ldw, ldx, nsx, nsw, wsx, wsw, s);
}

// The tile that gemm_any chooses without scratch, for a gated product (N rows of gate and up) if gated: rows << 16 | columns.
KGS_EXPORT int kgs_gemm_bf16_nt_tile(int M, int N, int K, int gated) {
  return M > 0 && N > 0 && K > 0 ? kgs::any::tile_of_rows(M, N, K, 64, 64, gated) : 0;
}

// The same of rows lda and ldb apart.
KGS_EXPORT int kgs_gemm_bf16_nt_tile_rows(int M, int N, int K, int lda, int ldb, int gated) {
  return M > 0 && N > 0 && K > 0 && lda >= K && ldb >= K ? kgs::any::tile_of_rows(M, N, K, lda, ldb, gated) : 0;
}

// Whether the kernels of 256x256 tiles leave a product (gated: of a gated projection; off: A's rows off the 128-byte lines) to a finer tile.
KGS_EXPORT int kgs_gemm_bf16_nt_finer(int M, int N, int K, int gated, int off) {
  return M > 0 && N > 0 && K > 0 && kgs::gemm_any_finer(nullptr, nullptr, M, N, K, off ? 8 : 64, 64, gated != 0, off != 0);
}

// Whether a K-major B is better transposed first than read by kgs_gemm_bf16 (turn_b).
KGS_EXPORT int kgs_gemm_bf16_turn_b(int M, int N, int K) {
  return M > 0 && N > 0 && K > 0 && kgs::any::turn_b(M, N, K, kgs::cu_count());
}

// Slices for kgs_gemm_bf16_tr, 0 where another route is faster (layout_plan).
KGS_EXPORT int kgs_gemm_bf16_tr_slices(int M, int N, int K, int ta, int tb) {
  return M > 0 && N > 0 && K > 0 ? kgs::any::layout_plan(M, N, K, ta, tb, kgs::cu_count()) : 0;
}

// Z = bf16(A . B^T + bias) and Y = act(Z) from one launch (epi: the activations' epilogues; bias
// may be null), both [M, N] with rows ldc apart. ws: kgs_gemm_bf16_nt_scratch values, or null.
KGS_EXPORT int kgs_gemm_bf16_nt_act(const void* A, const void* B, void* Z, void* Y, const void* bias, int M, int N, int K,
                                    int lda, int ldb, int ldc, int epi, float* ws, hipStream_t s) {
  if (M <= 0 || N <= 0 || K <= 0 || lda < K || ldb < K || ldc < N) return KGS_ERR_SHAPE;
  if (!Y || epi < kgs::EPI_BIAS_GELU || epi > kgs::EPI_BIAS_SILU) return KGS_ERR_ARG;
  if (!kgs::gemm_any_ok(A, B, M, N, K, lda, ldb) || (uintptr_t)ws % 16) return KGS_ERR_ALIGN;
  return kgs::gemm_any(A, B, Z, Y, bias, M, N, K, lda, ldb, ldc, epi, 0, 0, 0, ws, s);
}

// C [M, N / 2] = act(A . gate^T) * (A . up^T), B = [gate; up] of N rows, both products rounded to bf16 first: tiles of bm (64
// or 128) rows by 32 outputs. act: a GateAct (limit: the clamped gate's, on the device). N / 2 and K multiples of 8.
KGS_EXPORT int kgs_gemm_bf16_nt_gate(const void* A, const void* B, void* C, int M, int N, int K, int lda, int ldb, int ldc, int bm,
                                     int act, const void* limit, hipStream_t s) {
  if (M <= 0 || N <= 0 || K <= 0 || N % 16 || lda < K || ldb < K || ldc < N / 2) return KGS_ERR_SHAPE;
  if ((bm != 64 && bm != 128) || (act != kgs::GATE_SILU && act != kgs::GATE_GELU && act != kgs::GATE_CLAMPED)) return KGS_ERR_ARG;
  if (act == kgs::GATE_CLAMPED && (!limit || (uintptr_t)limit % 4)) return KGS_ERR_ARG;
  if (!kgs::gemm_any_ok(A, B, M, N, K, lda, ldb) || (uintptr_t)C % 16 || ldc % 8) return KGS_ERR_ALIGN;
  return kgs::gemm_gate(A, B, C, M, N, K, lda, ldb, ldc, bm, act, (const float*)limit, s);
}
