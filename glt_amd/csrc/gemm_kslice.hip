// Segment-list GEMM for launches with too few 256 x 256 tiles to fill the
// chip: small output tiles whose reduction is split over the wavefronts of
// one workgroup.
#include <algorithm>
#include <atomic>
#include <cmath>

#include "gemm.hpp"
#include "gemm_dev.hpp"
#include "layout.hpp"

namespace glt {

// =========================================================================
// gfx950 MFMA kernel with the K-steps dealt over wavefront groups: bf16 x
// bf16 -> f32, v_mfma_f32_32x32x16_bf16.
//
// One workgroup owns one output tile of 32 TI rows x 32 TJ NWN B-rows (dual:
// a wavefront's first TJ/2 blocks are gate columns, the others the up columns
// of the same outputs). It has NG groups of NWN wavefronts; the wavefronts of
// a group share the columns, and group g runs K-steps g, g + NG, g + 2 NG, ...
// of the tile's segments. The NG partial tiles are added, in group order,
// through LDS in f32 before the epilogue: no scratch memory and no second
// launch.
//
// A (row-major) comes by direct-to-LDS loads into the group's ring of PA
// chunks of 32 RB rows x 64 K (128-byte rows, 16-byte chunk ^ swz_key(row) as
// in the persistent kernel; chunks of 64-byte rows moved every line twice and
// were 20 % slower), B from the fragment layout straight into registers, PB
// steps ahead. A step is NP = TI / RB passes over the rows, so that the ring
// turns over in pieces smaller than a step. With NWN = 1 the loop has no
// barrier, only counted waits on the wavefront's own loads; else one per pass.
//
// What bounds it: a wavefront blocked at a load's issue issues no MFMAs, so
// one wavefront per SIMD pays for its loads and its MFMAs one after the other
// (4 wavefronts of 64 x 128: loads alone 24 us, MFMAs alone 14, together 48 at
// 512 x 4096 x 8192); the eight wavefronts here put two on each SIMD.
//
// ONCE loads B non-temporally (read_once below says when).
// =========================================================================
constexpr int min63(int n) { return n < 63 ? n : 63; }  // vmcnt holds 6 bits

template <int TI, int TJ, int RB, int NWN, int NG, int PA, int PB, typename TO, int MODE, bool DUAL, bool ONCE>
__global__ void __launch_bounds__(64 * NWN * NG) gemm_kslice_kernel(const GArgs args) {
  extern __shared__ __attribute__((aligned(16))) uint16_t smem[];
  constexpr int BM = 32 * TI, BNW = DUAL ? 16 * TJ : 32 * TJ, BN = BNW * NWN;
  constexpr int NP = TI / RB;                // passes of a step
  constexpr int NA = 4 * RB / NWN;           // a wavefront's A loads per chunk: 8 rows x 128 bytes each
  static_assert(NA == 4, "one A load per substep");
  constexpr int kStage = 32 * RB * kBK;      // elements of one A chunk
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int grp = wave / NWN, wn = wave % NWN;
  // The four substeps of a K-step are 1 KB apart in a B fragment block and one
  // K-step is 4 KB, so wavefronts in step would all read the same quarter of
  // the L2's channels: each takes the substeps in an order of its own (M = 512
  // of the shape above: 98 -> 90 us).
  const int rot = __builtin_amdgcn_readfirstlane((wave + (blockIdx.x >> 3)) & 3);
  // consecutive tiles on one XCD (workgroups are dealt round-robin over the
  // eight): they share A and B rows in its L2
  const int G = gridDim.x, b = blockIdx.x;
  const int q8 = G >> 3, r8 = G & 7, xcd = b & 7;
  const int tile = xcd * q8 + min(xcd, r8) + (b >> 3);
  int tm, tn;
  const int pi = locate_tile(args, tile, tm, tn, BM >= 128 ? kGroupM : 8);
  const GProb& P = args.p[pi];
  const int m0 = tm * BM, n0 = tn * BN, send = P.seg0 + P.nseg;

  auto next_active = [&](int s) __attribute__((always_inline)) {
    ++s;
    while (s < send && !seg_hits(args.s[s], P, n0, BN)) ++s;
    return s;
  };
  int T = 0;  // K-steps of the tile
  for (int s = next_active(P.seg0 - 1); s < send; s = next_active(s)) T += args.s[s].K / kBK;
  // this group's steps; wavefronts that meet at barriers all run the same
  // number (a step past the end multiplies zeros)
  const int Tg = NWN > 1 ? (T + NG - 1) / NG : (T - grp + NG - 1) / NG;

  // ---- stream positions: segment s, K offset k in it. Past the end every
  // offset is kOob, so the loads of the last steps deliver zeros without
  // touching memory and the load counts behind the waits stay the same.
  constexpr int kNoEnd = 1 << 30;
  struct Pos {
    int s, k, K;
  };
  auto settle = [&](Pos& q) __attribute__((always_inline)) {
    while (q.k >= q.K) {
      q.k -= q.K;
      q.s = q.s < send ? next_active(q.s) : send;
      if (q.s >= send) {
        q.k = 0;
        q.K = kNoEnd;
        return;
      }
      q.K = args.s[q.s].K;
    }
  };
  Pos pa{P.seg0 - 1, grp * kBK, 0};
  settle(pa);
  Pos pb = pa;

  // A: the group's wavefronts split the rows of each chunk evenly
  const void* pA = nullptr;
  uint32_t voA[NP * NA];
  auto setup_a = [&]() __attribute__((always_inline)) {
    if (pa.s >= send) {
#pragma unroll
      for (int i = 0; i < NP * NA; ++i) voA[i] = kOob;
      return;
    }
    const GSeg& S = args.s[pa.s];
    pA = S.A;
#pragma unroll
    for (int i = 0; i < NP * NA; ++i) {
      const int row = 32 * RB * (i / NA) + 8 * (NA * wn + i % NA) + (lane >> 3);
      const int kc = (lane & 7) ^ swz_key(row);
      const int m = m0 + row;
      voA[i] = m < P.M ? (uint32_t)(((int64_t)m * S.lda + S.a_col + kc * 8) * 2) : kOob;
    }
  };
  const void *pB0 = nullptr, *pB1 = nullptr;
  uint32_t nB0 = 0, nB1 = 0, voB[TJ];
  auto setup_b = [&]() __attribute__((always_inline)) {
    if (pb.s >= send) {
#pragma unroll
      for (int j = 0; j < TJ; ++j) voB[j] = kOob;
      return;
    }
    const GSeg& S = args.s[pb.s];
    pB0 = S.B0;
    pB1 = DUAL ? S.B1 : S.B0;
    nB0 = pB0 ? kExtent : 0;
    nB1 = pB1 ? kExtent : 0;
    const int nlo = S.n_lo, nhi = min(S.n_hi, P.N), nw0 = n0 + wn * BNW;
    auto voff = [&](int f0, int64_t ld, int r0) {
      const int n = f0 + (lane & 31);
      return (n >= nlo && n < nhi) ? (uint32_t)((int64_t)((f0 - r0) >> 5) * ld * 64 + lane * 16) : kOob;
    };
    constexpr int J0 = DUAL ? TJ / 2 : TJ;
#pragma unroll
    for (int j = 0; j < J0; ++j) voB[j] = voff(nw0 + 32 * j, S.ldb0, S.b0_row0);
#pragma unroll
    for (int j = J0; j < TJ; ++j) voB[j] = voff(nw0 + 32 * (j - J0), S.ldb1, S.b1_row0);
  };
  auto adv = [&](Pos& q, auto&& setup) __attribute__((always_inline)) {
    q.k += NG * kBK;
    if (__builtin_expect(q.k >= q.K, 0)) {
      settle(q);
      setup();
    }
  };

  uint16_t* const ring = smem + (size_t)grp * PA * kStage;
  auto load_a = [&](int slot, int p, int i) {  // load i of the chunk of row pass p
    load_lds16(uni_rsrc(pA, kExtent), ring + slot * kStage + (NA * wn + i) * 8 * kBK, voA[NA * p + i],
               (uint32_t)pa.k * 2);
  };
  uint32_t sub[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) sub[s] = (s + rot) & 3;
  constexpr int kAux = ONCE ? 2 : 0;  // 2: non-temporal
  bf16x8 fb[PB][4][TJ];
  auto load_b = [&](int u, int s, int j) {
    const __amdgpu_buffer_rsrc_t r = (DUAL && j >= TJ / 2) ? uni_rsrc(pB1, nB1) : uni_rsrc(pB0, nB0);
    const uint32_t so = (uint32_t)pb.k * 64 + sub[s] * 1024;  // 1 KB per fragment of 16 K
    fb[u][s][j] = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(r, voB[j], so, kAux));
  };

  f32x16 acc[TI][TJ];
#pragma unroll
  for (int i = 0; i < TI; ++i)
#pragma unroll
    for (int j = 0; j < TJ; ++j) acc[i][j] = f32x16{};
  const int lr = lane & 31, lkh = lane >> 5;
  int aoff[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) aoff[s] = lr * kBK + (((sub[s] * 2 + lkh) ^ swz_key(lr)) << 3);
  bf16x8 fa[2][RB];
  auto read_a = [&](int slot, int ks, int f, int i) {
    fa[f][i] = *reinterpret_cast<const bf16x8*>(ring + slot * kStage + 32 * i * kBK + aoff[ks]);
  };
  // chunks published (and the last reads of the one before done) across the
  // wavefronts that share them
  auto publish = [&]() __attribute__((always_inline)) {
    if constexpr (NWN > 1) asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    else asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };

  if (Tg > 0) {
    // fill: B of steps 0 .. PB-1, then A chunks 0 .. PA-2
    static_assert((PA - 1) % NP == 0 && PA >= 3, "the ring leads by whole steps");
    setup_a();
    setup_b();
#pragma unroll
    for (int u = 0; u < PB; ++u) {
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int j = 0; j < TJ; ++j) load_b(u, s, j);
      adv(pb, setup_b);
    }
#pragma unroll
    for (int c = 0; c < PA - 1; ++c) {
#pragma unroll
      for (int i = 0; i < NA; ++i) load_a(c, c % NP, i);
      if (c % NP == NP - 1) adv(pa, setup_a);
    }
    __builtin_amdgcn_s_waitcnt(vmcnt_enc((PA - 2) * NA));
    publish();
#pragma unroll
    for (int i = 0; i < RB; ++i) read_a(0, 0, 0, i);

    // Chunk c = pass p of step t sits in slot c % PA. Per substep of 16 K:
    // its MFMAs beside the A reads of the next substep (in substep 3 of the
    // next chunk), a quarter of chunk c + PA - 1 into the slot that chunk
    // c - 1 left, and in the last pass each B fragment reloaded for step
    // t + PB once used. Loads land in order: chunk c + 1 was loaded in pass
    // c + 2 - PA, with PA - 3 whole passes and three substeps of loads behind
    // it (while it came in the fill: with A loads only).
    constexpr int kPasses = (PA - 3) * NA + (NP == 1 ? PA - 3 : (PA - 3) / NP) * 4 * TJ;
    constexpr int kWaitFill = (PA - 3) * NA + 3, kWaitMid = min63(kPasses + 3), kWaitLast = min63(kPasses + 3 + 3 * TJ);
    int slot = 0;
    auto step = [&](int u, int t, bool tail) __attribute__((always_inline)) {
#pragma unroll
      for (int p = 0; p < NP; ++p) {
        const int nslot = slot + 1 == PA ? 0 : slot + 1, pslot = slot == 0 ? PA - 1 : slot - 1;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          if (s == 3) {
            if (tail || __builtin_expect(t * NP + p < PA - 2, 0)) __builtin_amdgcn_s_waitcnt(vmcnt_enc(kWaitFill));
            else if (p == NP - 1) __builtin_amdgcn_s_waitcnt(vmcnt_enc(kWaitLast));
            else __builtin_amdgcn_s_waitcnt(vmcnt_enc(kWaitMid));
            publish();
          }
#pragma unroll
          for (int j = 0; j < TJ; ++j) {
#pragma unroll
            for (int i = 0; i < RB; ++i)
              acc[RB * p + i][j] =
                  __builtin_amdgcn_mfma_f32_32x32x16_bf16(fb[u][s][j], fa[s & 1][i], acc[RB * p + i][j], 0, 0, 0);
            // the next fragments, spread over the column blocks
#pragma unroll
            for (int i = j * RB / TJ; i < (j + 1) * RB / TJ; ++i)
              read_a(s == 3 ? nslot : slot, (s + 1) & 3, (s & 1) ^ 1, i);
            if (p == NP - 1) load_b(u, s, j);
            if (j == 0) load_a(pslot, p, s);
            __builtin_amdgcn_sched_barrier(0);
          }
        }
        slot = nslot;
      }
      adv(pa, setup_a);
      adv(pb, setup_b);
    };
    // Whole groups of PB steps, then the rest apart: with an exit between the
    // copies the compiler sees a way from one copy's loads back to its own
    // uses one step later, and waits for everything older than that.
    int t = 0;
#pragma unroll 1
    for (; t + PB <= Tg; t += PB) {
#pragma unroll
      for (int u = 0; u < PB; ++u) step(u, t + u, false);
    }
    // (in these last steps the compiler drops the B loads, which nothing uses
    // any more: the waits may count A loads only)
    if constexpr (PB > 1) {
#pragma unroll
      for (int u = 0; u < PB - 1; ++u)
        if (t + u < Tg) step(u, t + u, true);
    }
    // trailing (zero) loads must land before the ring is reused
    __builtin_amdgcn_s_waitcnt(vmcnt_enc(0));
  }

  // ---- sum over the groups and epilogue, one 32-row block at a time.
  // acc[i][j] is the transposed 32 x 32 product: lane l holds row 32 i +
  // (l & 31), columns 32 j + 8 q + 4 (l >> 5) .. +3 in elements 4 q .. +3.
  // Each group writes its block as 16-byte chunks (chunk c of row r at
  // c ^ rkey(r): 16 consecutive rows of one chunk, and the chunks of one row,
  // both cover all 64 banks); threads then add the NG copies of a chunk.
  constexpr int CW = 8 * TJ, CH = CW * NWN;  // chunks of a row: a wavefront's, the tile's
  constexpr int kBlk = 32 * CH * 16;         // bytes of one group's block
  auto rkey = [](int r) { return CH >= 16 ? r & 15 : (r >> 1) & 7; };
  char* const red = reinterpret_cast<char*>(smem);
  constexpr int CO = DUAL ? CH / 2 : CH;     // output chunks of a row
#pragma unroll
  for (int i = 0; i < TI; ++i) {
    __syncthreads();
#pragma unroll
    for (int j = 0; j < TJ; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const f32x16& a = acc[i][j];
        const int c = CW * wn + 8 * j + 2 * q + lkh;
        *reinterpret_cast<f32x4*>(red + grp * kBlk + lr * (CH * 16) + ((c ^ rkey(lr)) << 4)) =
            f32x4{a[4 * q], a[4 * q + 1], a[4 * q + 2], a[4 * q + 3]};
      }
    __syncthreads();
#pragma unroll 2
    for (int e = tid; e < 32 * CO; e += 64 * NWN * NG) {
      const int row = e / CO, c = e % CO;
      const int m = m0 + 32 * i + row, n = n0 + 4 * c;
      if (m >= P.M || n >= P.N) continue;
      auto sum = [&](int ch) {
        const char* src = red + row * (CH * 16) + ((ch ^ rkey(row)) << 4);
        f32x4 v = *reinterpret_cast<const f32x4*>(src);
#pragma unroll
        for (int w = 1; w < NG; ++w) v += *reinterpret_cast<const f32x4*>(src + w * kBlk);
        return v;
      };
      // dual: output chunk c is gate chunk c of its wavefront's CW / 2, up CW / 2 on
      const int cg = DUAL ? c / (CW / 2) * CW + c % (CW / 2) : c;
      const f32x4 v = sum(cg);
      const int64_t o = (int64_t)m * P.ldo + n;
      auto st = [&](void* p, float a0, float a1, float a2, float a3) {
        if constexpr (sizeof(TO) == 4) *reinterpret_cast<f32x4*>(static_cast<float*>(p) + o) = f32x4{a0, a1, a2, a3};
        else *reinterpret_cast<u32x2*>(static_cast<uint16_t*>(p) + o) = u32x2{pack2_hw(a0, a1), pack2_hw(a2, a3)};
      };
      auto ld4 = [](const void* p, int64_t off, float* f) {
        const u32x2 w = *reinterpret_cast<const u32x2*>(static_cast<const uint16_t*>(p) + off);
        f[0] = __uint_as_float(w.x << 16);
        f[1] = __uint_as_float(w.x & 0xFFFF0000u);
        f[2] = __uint_as_float(w.y << 16);
        f[3] = __uint_as_float(w.y & 0xFFFF0000u);
      };
      if constexpr (MODE == EPI_STORE) {
        st(P.out0, P.alpha * v.x, P.alpha * v.y, P.alpha * v.z, P.alpha * v.w);
      } else if constexpr (MODE == EPI_RESID) {
        static_assert(MODE != EPI_RESID || sizeof(TO) == 2, "the residual epilogue here is bf16");
        float x[4];
        ld4(P.out0, o, x);
        st(P.out0, x[0] + round_like<TO>(P.alpha * v.x), x[1] + round_like<TO>(P.alpha * v.y),
           x[2] + round_like<TO>(P.alpha * v.z), x[3] + round_like<TO>(P.alpha * v.w));
      } else if constexpr (MODE == EPI_SILU) {
        const f32x4 u4 = sum(cg + CW / 2);
        float g[4], u[4], r[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          g[k] = round_like<TO>(v[k]);
          u[k] = round_like<TO>(u4[k]);
          r[k] = g[k] * sigmoid_fast(g[k]) * u[k];
        }
        st(P.out0, r[0], r[1], r[2], r[3]);
        if (P.out1) st(P.out1, g[0], g[1], g[2], g[3]);
        if (P.out2) st(P.out2, u[0], u[1], u[2], u[3]);
      } else {
        float g[4], u[4], dg[4], du[4];
        const int64_t oa = (int64_t)m * P.ldaux + n;
        ld4(P.aux0, oa, g);
        ld4(P.aux1, oa, u);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const float sg = sigmoid_fast(g[k]);
          dg[k] = v[k] * u[k] * (sg * (1.0f + g[k] * (1.0f - sg)));
          du[k] = v[k] * (g[k] * sg);
        }
        st(P.out0, dg[0], dg[1], dg[2], dg[3]);
        st(P.out1, du[0], du[1], du[2], du[3]);
      }
    }
  }
}

// ------------------------------------------------------------------ host
// Tile shapes: id, TI, TJ, RB, NWN, NG, PA, PB, and the cost model of the
// dispatch: us per round of one tile per CU = fix + per_k * K / 1000.
// Measured over M = 8 .. 5056 at N x K = 4096 x 15360, 4096 x 30720 and 15360
// x 4096 (MI355X); the same constants for the persistent kernel below.
#define GLT_KS_SHAPES(X)                                                       \
  X(0, 1, 1, 1, 1, 4, 5, 4, 3.f, 2.0f)  /* 32 x 32, the fewest rows */         \
  X(1, 2, 2, 1, 1, 8, 5, 4, 5.f, 4.0f)  /* 64 x 64 */                          \
  X(2, 2, 2, 2, 2, 4, 5, 4, 6.f, 5.6f)  /* 64 x 128 */                         \
  X(3, 4, 2, 2, 2, 4, 5, 2, 10.f, 8.0f) /* 128 x 128 */                        \
  X(4, 4, 2, 4, 4, 2, 4, 2, 16.f, 12.5f) /* 128 x 256 */
constexpr int kShapeCount = 5;
struct KsShape {
  int ti, tj, nwn;
  float fix, per_k;
};
static const KsShape kShapes[kShapeCount] = {
#define GLT_KS_ROW(ID, TI, TJ, RB, NWN, NG, PA, PB, FIX, PERK) {TI, TJ, NWN, FIX, PERK},
    GLT_KS_SHAPES(GLT_KS_ROW)
#undef GLT_KS_ROW
};
static int ks_rows(const KsShape& s) { return 32 * s.ti; }
static int ks_cols(const KsShape& s, bool dual) {
  return s.nwn * (dual ? (s.tj == 1 ? 32 : 16 * s.tj) : 32 * s.tj);
}

// The tile shape with the least estimated time, or -1 for the persistent 256
// x 256 kernel. A launch runs in rounds of one tile per CU, each round the
// time of its longest reduction; large tiles move fewer bytes per product,
// small ones leave no CU idle (4096 output columns are 16 tiles of 256 for
// 256 CUs: M = 8, K = 15360 took 247 us on the persistent kernel, 32 us on 32
// x 32 tiles; M = 512: 282 and 90 on 64 x 128; M = 2048: 288 and 211 on 128 x
// 256; M = 4096, one full round: 372 and 424, so the persistent kernel stays).
// Weights are read once from HBM whatever the shape (about 5.2 TB/s in these
// launches). The sum over K-slices rounds in another order than the persistent
// kernel's, so a row of a small call may differ from the same row of a large
// one in the last f32 bits of its sums. Outputs narrower than kMinCols stay on
// the persistent kernel, where the rows of every call agree bit for bit:
// nothing is lost there, as no layer is that narrow.
constexpr int kMinCols = 512;
int pick_kslice(const GemmPlan& plan, int cus) {
  const GArgs& a = plan.args;
  const int mode = a.p[0].mode, of32 = a.p[0].out_f32;
  if (!((mode == EPI_SILU && plan.dual && !of32) ||
        (!plan.dual && (mode == EPI_STORE || ((mode == EPI_DGDU || mode == EPI_RESID) && !of32)))))
    return -1;
  for (int p = 0; p < a.nprob; ++p)
    if (a.p[p].N < kMinCols) return -1;
  auto cost = [&](int rows, int cols, float fix, float per_k) {
    double tiles = 0, kmax = 0, bytes = 0;
    for (int p = 0; p < a.nprob; ++p) {
      const GProb& P = a.p[p];
      double k = 0;  // the longest reduction of any tile of the problem: at most all its segments
      for (int i = P.seg0; i < P.seg0 + P.nseg; ++i) {
        const GSeg& s = a.s[i];
        const double span = (double)std::max(0, std::min(s.n_hi, P.N) - s.n_lo);
        bytes += span * s.K * 2 * (plan.dual ? 2 : 1);
        k = std::max(k, (double)s.K);
        // segments over the same columns add up, those side by side do not
        for (int j = P.seg0; j < i; ++j)
          if (a.s[j].n_lo < s.n_hi && s.n_lo < a.s[j].n_hi) k = std::max(k, (double)s.K + a.s[j].K);
      }
      double same = 0;
      for (int i = P.seg0; i < P.seg0 + P.nseg; ++i)
        if (a.s[i].n_lo <= 0 && a.s[i].n_hi >= P.N) same += a.s[i].K;
      kmax = std::max(kmax, std::max(k, same));
      tiles += (double)cdiv(P.M, rows) * cdiv(P.N, cols);
    }
    const float epi = mode == EPI_SILU ? 10.f : mode == EPI_DGDU ? 6.f : 0.f;
    const double rounds = std::ceil(tiles / cus);
    const double run = rounds * (fix + epi + per_k * kmax / 1000.);
    return std::max(run, bytes / 5.2e6) + 0.2 * run;  // bytes / us; ties go to the shorter run
  };
  int best = -1;
  double least = cost(256, plan.dual ? 128 : 256, 12.f, 19.5f);
  for (int i = 0; i < kShapeCount; ++i) {
    const KsShape& s = kShapes[i];
    const double c = cost(ks_rows(s), ks_cols(s, plan.dual),
                          s.fix, plan.dual && s.tj == 1 ? 1.5f * s.per_k : s.per_k);
    if (c < least) {
      least = c;
      best = i;
    }
  }
  return best;
}

template <int TI, int TJ, int RB, int NWN, int NG, int PA, int PB, typename TO, int MODE, bool DUAL, bool ONCE>
static glt_status launch_ks_as(const GArgs& a, hipStream_t st, const char* label) {
  static std::atomic<bool> attr_set[64];
  // dual tiles pair gate with up blocks (a 1 x 1 shape takes one of each)
  constexpr int TJ_ = DUAL && TJ == 1 ? 2 : TJ;
  auto fn = gemm_kslice_kernel<TI, TJ_, RB, NWN, NG, PA, PB, TO, MODE, DUAL, ONCE>;
  int dev = 0;
  GLT_TRY_HIP(hipGetDevice(&dev));
  GLT_CHECK(dev >= 0 && dev < 64, GLT_ERR_HIP, "gemm: device index %d out of range", dev);
  constexpr size_t ring = (size_t)NG * PA * 32 * RB * kBK * 2, red = (size_t)NG * 32 * TJ_ * NWN * 32 * 4;
  constexpr size_t lds = ring > red ? ring : red;
  static_assert(lds <= 160 * 1024, "LDS of one CU");
  if (!attr_set[dev].load(std::memory_order_acquire)) {
    GLT_TRY_HIP(
        hipFuncSetAttribute(reinterpret_cast<const void*>(fn), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    attr_set[dev].store(true, std::memory_order_release);
  }
  GLT_LAUNCH(label, fn, dim3(a.total_tiles), dim3(64 * NWN * NG), lds, st, a);
  GLT_LAUNCH_CHECK("gemm_kslice");
  return GLT_OK;
}

// Whether B is read once and gone: a single row of tiles (no other workgroup
// reads the same part of B), and more than half of the 256 MB last-level cache
// of it, so that the next call would not find it there whatever the loads say.
// Non-temporal loads then stream faster and leave the cache to the others'
// operands: MLP forward of 4096 x 15360, one layer called again and again, 8
// tokens 81 -> 65 us, 64 tokens 91 -> 72; four layers in turn 80 -> 76 and 92
// -> 86. Below that size repeated calls lose the cached weights (2048 x 11008,
// 8 tokens: 34 -> 41 us), and with several row tiles the B that they share
// comes twice (4096 x 15360, 200 tokens: 180 -> 222 us).
static bool read_once(const GArgs& a, bool dual) {
  int64_t bytes = 0;
  for (int p = 0; p < a.nprob; ++p) {
    const GProb& P = a.p[p];
    if (P.tiles_m > 1) return false;
    for (int i = P.seg0; i < P.seg0 + P.nseg; ++i)
      bytes += (int64_t)std::max(0, std::min(a.s[i].n_hi, P.N) - a.s[i].n_lo) * a.s[i].K * (dual ? 4 : 2);
  }
  return bytes > (int64_t)128 << 20;
}

template <int TI, int TJ, int RB, int NWN, int NG, int PA, int PB, typename TO, int MODE, bool DUAL>
static glt_status launch_ks(const GArgs& a, hipStream_t st, const char* label) {
  return read_once(a, DUAL) ? launch_ks_as<TI, TJ, RB, NWN, NG, PA, PB, TO, MODE, DUAL, true>(a, st, label)
                            : launch_ks_as<TI, TJ, RB, NWN, NG, PA, PB, TO, MODE, DUAL, false>(a, st, label);
}

glt_status run_kslice(GemmPlan& plan, int shape, hipStream_t st) {
  GArgs& a = plan.args;
  const KsShape& S = kShapes[shape];
  const int bm = ks_rows(S), bn = ks_cols(S, plan.dual);
  const int mode = a.p[0].mode, of32 = a.p[0].out_f32;
  int tiles = 0;
  for (int p = 0; p < a.nprob; ++p) {
    GProb& P = a.p[p];
    GLT_CHECK(P.mode == mode && P.out_f32 == of32, GLT_ERR_INVALID_ARG, "run_gemm: mixed epilogues in one launch");
    P.tiles_m = (int)cdiv(P.M, bm);
    P.tiles_n = (int)cdiv(P.N, bn);
    P.tile_begin = tiles;
    tiles += P.tiles_m * P.tiles_n;
  }
  a.total_tiles = tiles;
  if (tiles == 0) return GLT_OK;
#define GLT_KS_RUN(ID, TI, TJ, RB, NWN, NG, PA, PB, FIX, PERK)                                                                        \
  if (shape == ID) {                                                                                             \
    if (mode == EPI_SILU && plan.dual)                                                                           \
      return launch_ks<TI, TJ, RB, NWN, NG, PA, PB, uint16_t, EPI_SILU, true>(a, st, plan.label);                  \
    if (mode == EPI_DGDU && !plan.dual)                                                                          \
      return launch_ks<TI, TJ, RB, NWN, NG, PA, PB, uint16_t, EPI_DGDU, false>(a, st, plan.label);                 \
    if (mode == EPI_STORE && !plan.dual)                                                                         \
      return of32 ? launch_ks<TI, TJ, RB, NWN, NG, PA, PB, float, EPI_STORE, false>(a, st, plan.label)             \
                  : launch_ks<TI, TJ, RB, NWN, NG, PA, PB, uint16_t, EPI_STORE, false>(a, st, plan.label);         \
    if (mode == EPI_RESID && !plan.dual && !of32)                                                                \
      return launch_ks<TI, TJ, RB, NWN, NG, PA, PB, uint16_t, EPI_RESID, false>(a, st, plan.label);                \
  }
  GLT_KS_SHAPES(GLT_KS_RUN)
#undef GLT_KS_RUN
  set_error("run_gemm: no K-sliced kernel for mode %d dual %d", mode, (int)plan.dual);
  return GLT_ERR_UNSUPPORTED;
}

}  // namespace glt
