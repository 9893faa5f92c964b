// Segment-list GEMM for launches with too few 256 x 256 tiles to fill the
// chip: small output tiles, summed in the persistent kernel's order.
#include <algorithm>
#include <atomic>
#include <cmath>

#include "gemm.hpp"
#include "gemm_dev.hpp"
#include "layout.hpp"

namespace glt {

// =========================================================================
// gfx950 MFMA kernel: bf16 x bf16 -> f32, v_mfma_f32_32x32x16_bf16.
//
// One workgroup of NWN wavefronts owns one output tile of 32 TI rows x 32 TJ
// NWN B-rows (dual: a wavefront's first TJ/2 blocks are gate columns, the
// others the up columns of the same outputs); each wavefront takes all rows of
// its own columns.
//
// Every output is the sum of the same MFMAs in the same order as in the
// persistent kernel (gemm.hip): segments in order, one accumulator along K. So
// a row has the same bits whatever the rows beside it and whichever kernel a
// launch of that size takes. Dealing the K-steps over wavefront groups and
// adding the partial tiles, which gives up that order, measured 0 to 10 % less
// at 8 to 2048 rows (N = 4096, K = 15360: M = 8 31 against 37 us, M = 512 90
// against 99, M = 2048 199 against 207; N = 15360, K = 4096: the same).
//
// A (row-major) comes by direct-to-LDS loads into a ring of PA chunks of 32 RB
// rows x 64 K (128-byte rows, 16-byte chunk ^ swz_key(row) as in the persistent
// kernel; chunks of 64-byte rows moved every line twice and were 20 % slower),
// B from the fragment layout straight into registers, PB steps ahead. A step
// is NP = TI / RB passes over the rows, so that the ring turns over in pieces
// smaller than a step.
//
// What bounds it: few rows, the chain of dependent MFMAs (32 rows x 32 columns
// a wavefront, K = 15360: 960 MFMAs in 37 us; with the A fragments read one
// substep ahead instead of two, 48: the LDS read's latency); more rows, the
// operands' way to a CU, which moves 24 to 26 bytes per clock at every tile
// shape, row split and depth of the rings tried. Rows split over wavefronts
// too (eight wavefronts of 32 x 32 for 64 x 128) measured 1.2 times slower.
//
// ONCE loads B non-temporally (read_once below says when).
// =========================================================================
constexpr int min63(int n) { return n < 63 ? n : 63; }  // vmcnt holds 6 bits

template <int TI, int TJ, int RB, int NWN, int PA, int PB, typename TO, int MODE, bool DUAL, bool ONCE>
__global__ void __launch_bounds__(64 * NWN) gemm_small_kernel(const GArgs args) {
  extern __shared__ __attribute__((aligned(16))) uint16_t smem[];
  constexpr int BM = 32 * TI, BNW = DUAL ? 16 * TJ : 32 * TJ, BN = BNW * NWN;
  constexpr int NP = TI / RB;                // passes of a step
  constexpr int NA = 4 * RB / NWN;           // a wavefront's A loads per chunk: 8 rows x 128 bytes each
  static_assert(NA == 4 || NA == 2 || NA == 1, "A loads spread evenly over the substeps");
  constexpr int kStage = 32 * RB * kBK;      // elements of one A chunk
  const int tid = threadIdx.x, lane = tid & 63;
  const int wn = __builtin_amdgcn_readfirstlane(tid >> 6);
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
  Pos pa{P.seg0 - 1, 0, 0};
  settle(pa);
  Pos pb = pa;

  // A: the wavefronts split the rows of each chunk evenly
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
    q.k += kBK;
    if (__builtin_expect(q.k >= q.K, 0)) {
      settle(q);
      setup();
    }
  };

  auto load_a = [&](int slot, int p, int i) {  // load i of the chunk of row pass p
    load_lds16(uni_rsrc(pA, kExtent), smem + slot * kStage + (NA * wn + i) * 8 * kBK, voA[NA * p + i],
               (uint32_t)pa.k * 2);
  };
  constexpr int kAux = ONCE ? 2 : 0;  // 2: non-temporal
  bf16x8 fb[PB][4][TJ];
  auto load_b = [&](int u, int s, int j) {
    const __amdgpu_buffer_rsrc_t r = (DUAL && j >= TJ / 2) ? uni_rsrc(pB1, nB1) : uni_rsrc(pB0, nB0);
    const uint32_t so = (uint32_t)pb.k * 64 + s * 1024;  // 1 KB per fragment of 16 K
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
  for (int s = 0; s < 4; ++s) aoff[s] = lr * kBK + (((s * 2 + lkh) ^ swz_key(lr)) << 3);
  bf16x8 fa[4][RB];
  auto read_a = [&](int slot, int ks, int i) {
    fa[ks][i] = *reinterpret_cast<const bf16x8*>(smem + slot * kStage + 32 * i * kBK + aoff[ks]);
  };
  // chunks that this wavefront has waited for, published to the wavefronts
  // that share them
  auto publish = [&]() __attribute__((always_inline)) {
    if constexpr (NWN > 1) asm volatile("s_barrier" ::: "memory");
    else asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };

  if (T > 0) {
    // fill: B of steps 0 .. PB-1, then A chunks 0 .. PA-3
    static_assert((PA - 2) % NP == 0 && PA >= 4, "the ring leads by whole steps");
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
    for (int c = 0; c < PA - 2; ++c) {
#pragma unroll
      for (int i = 0; i < NA; ++i) load_a(c, c % NP, i);
      if (c % NP == NP - 1) adv(pa, setup_a);
    }
    __builtin_amdgcn_s_waitcnt(vmcnt_enc((PA - 3) * NA));
    publish();
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int i = 0; i < RB; ++i) read_a(0, s, i);

    // Chunk c = pass p of step t sits in slot c % PA. Per substep of 16 K: its
    // MFMAs beside the A reads of the substep after next (in substeps 2 and 3
    // of the next chunk), in the last pass each B fragment reloaded for step t
    // + PB once used, and a share of chunk c + PA - 2 into the slot of chunk c
    // - 2: every wavefront consumed its last reads of that one (by its MFMAs
    // of pass c - 2) before the barrier of pass c - 1, so no wait for LDS reads
    // is needed. Loads land in order: chunk c + 1 was loaded in pass c + 3 -
    // PA, with PA - 4 whole passes and the loads of substeps 0 and 1 behind it
    // (while it came in the fill: with A loads only).
    constexpr int kA = NA / 2 > 0 ? NA / 2 : 1;  // A loads of substeps 0 and 1
    constexpr int kPasses = (PA - 4) * NA + (NP == 1 ? PA - 4 : (PA - 4) / NP) * 4 * TJ;
    constexpr int kWaitFill = (PA - 4) * NA + kA, kWaitMid = min63(kPasses + kA), kWaitLast = min63(kPasses + kA + 2 * TJ);
    int slot = 0;
    auto step = [&](int u, int t, bool tail) __attribute__((always_inline)) {
#pragma unroll
      for (int p = 0; p < NP; ++p) {
        const int nslot = slot + 1 == PA ? 0 : slot + 1, pslot = slot < 2 ? slot + PA - 2 : slot - 2;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          if (s == 2) {
            if (tail || __builtin_expect(t * NP + p < PA - 3, 0)) __builtin_amdgcn_s_waitcnt(vmcnt_enc(kWaitFill));
            else if (p == NP - 1) __builtin_amdgcn_s_waitcnt(vmcnt_enc(kWaitLast));
            else __builtin_amdgcn_s_waitcnt(vmcnt_enc(kWaitMid));
            publish();
          }
#pragma unroll
          for (int j = 0; j < TJ; ++j) {
#pragma unroll
            for (int i = 0; i < RB; ++i)
              acc[RB * p + i][j] =
                  __builtin_amdgcn_mfma_f32_32x32x16_bf16(fb[u][s][j], fa[s][i], acc[RB * p + i][j], 0, 0, 0);
            // the next fragments, spread over the column blocks
#pragma unroll
            for (int i = j * RB / TJ; i < (j + 1) * RB / TJ; ++i)
              read_a(s >= 2 ? nslot : slot, (s + 2) & 3, i);
            if (p == NP - 1) load_b(u, s, j);
            if (j == 0 && s % (4 / NA) == 0) load_a(pslot, p, s / (4 / NA));
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
    for (; t + PB <= T; t += PB) {
#pragma unroll
      for (int u = 0; u < PB; ++u) step(u, t + u, false);
    }
    // (in these last steps the compiler drops the B loads, which nothing uses
    // any more: the waits may count A loads only)
    if constexpr (PB > 1) {
#pragma unroll
      for (int u = 0; u < PB - 1; ++u)
        if (t + u < T) step(u, t + u, true);
    }
    // trailing (zero) loads must land before the ring is reused
    __builtin_amdgcn_s_waitcnt(vmcnt_enc(0));
  }

  // ---- epilogue, one 32-row block at a time. acc[i][j] is the transposed 32
  // x 32 product: lane l holds row 32 i + (l & 31), columns 32 j + 8 q + 4 (l
  // >> 5) .. +3 in elements 4 q .. +3. The block goes through LDS in 16-byte
  // chunks (chunk c of row r at c ^ rkey(r): 16 consecutive rows of one chunk,
  // and the chunks of one row, both cover all 64 banks) and comes back
  // row-wise.
  constexpr int CW = 8 * TJ, CH = CW * NWN;  // chunks of a row: a wavefront's, the tile's
  auto rkey = [](int r) { return CH >= 16 ? r & 15 : (r >> 1) & 7; };
  char* const red = reinterpret_cast<char*>(smem);
  constexpr int CO = DUAL ? CH / 2 : CH;     // output chunks of a row
  constexpr int NE = CO / (2 * NWN);         // a thread's chunks of the block
  auto ld4 = [](const u32x2& w, float* f) {
    f[0] = __uint_as_float(w.x << 16);
    f[1] = __uint_as_float(w.x & 0xFFFF0000u);
    f[2] = __uint_as_float(w.y << 16);
    f[3] = __uint_as_float(w.y & 0xFFFF0000u);
  };
#pragma unroll
  for (int i = 0; i < TI; ++i) {
    int64_t off[NE], offx[NE];  // element offsets of the chunks in the outputs and in what is read, -1 outside
#pragma unroll
    for (int k = 0; k < NE; ++k) {
      const int e = tid + 64 * NWN * k, m = m0 + 32 * i + e / CO, n = n0 + 4 * (e % CO);
      const bool in = m < P.M && n < P.N;
      off[k] = in ? (int64_t)m * P.ldo + n : -1;
      offx[k] = in ? (int64_t)m * (MODE == EPI_DGDU ? P.ldaux : P.ldo) + n : -1;
    }
    // what the outputs are formed from in memory, all in flight while the
    // block goes through LDS (one chunk after the other, their latencies added
    // up: dInter of 512 rows 87 us)
    u32x2 xa[NE], xb[NE];
    if constexpr (MODE == EPI_DGDU || MODE == EPI_RESID) {
      const void* const p0 = MODE == EPI_DGDU ? P.aux0 : P.out0;
#pragma unroll
      for (int k = 0; k < NE; ++k) {
        xa[k] = xb[k] = u32x2{0u, 0u};
        if (offx[k] < 0) continue;
        xa[k] = *reinterpret_cast<const u32x2*>(static_cast<const uint16_t*>(p0) + offx[k]);
        if constexpr (MODE == EPI_DGDU)
          xb[k] = *reinterpret_cast<const u32x2*>(static_cast<const uint16_t*>(P.aux1) + offx[k]);
      }
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < TJ; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const f32x16& a = acc[i][j];
        const int c = CW * wn + 8 * j + 2 * q + lkh;
        *reinterpret_cast<f32x4*>(red + lr * (CH * 16) + ((c ^ rkey(lr)) << 4)) =
            f32x4{a[4 * q], a[4 * q + 1], a[4 * q + 2], a[4 * q + 3]};
      }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < NE; ++k) {
      const int64_t o = off[k];
      if (o < 0) continue;
      const int e = tid + 64 * NWN * k, row = e / CO, c = e % CO;
      auto chunk = [&](int ch) {
        return *reinterpret_cast<const f32x4*>(red + row * (CH * 16) + ((ch ^ rkey(row)) << 4));
      };
      // dual: output chunk c is gate chunk c of its wavefront's CW / 2, up CW / 2 on
      const int cg = DUAL ? c / (CW / 2) * CW + c % (CW / 2) : c;
      const f32x4 v = chunk(cg);
      auto st = [&](void* p, float a0, float a1, float a2, float a3) {
        if constexpr (sizeof(TO) == 4) *reinterpret_cast<f32x4*>(static_cast<float*>(p) + o) = f32x4{a0, a1, a2, a3};
        else *reinterpret_cast<u32x2*>(static_cast<uint16_t*>(p) + o) = u32x2{pack2_hw(a0, a1), pack2_hw(a2, a3)};
      };
      if constexpr (MODE == EPI_STORE) {
        st(P.out0, P.alpha * v.x, P.alpha * v.y, P.alpha * v.z, P.alpha * v.w);
      } else if constexpr (MODE == EPI_RESID) {
        static_assert(MODE != EPI_RESID || sizeof(TO) == 2, "the residual epilogue here is bf16");
        float x[4];
        ld4(xa[k], x);
        st(P.out0, x[0] + round_like<TO>(P.alpha * v.x), x[1] + round_like<TO>(P.alpha * v.y),
           x[2] + round_like<TO>(P.alpha * v.z), x[3] + round_like<TO>(P.alpha * v.w));
      } else if constexpr (MODE == EPI_SILU) {
        const f32x4 u4 = chunk(cg + CW / 2);
        float g[4], u[4], r[4];
#pragma unroll
        for (int e4 = 0; e4 < 4; ++e4) {
          g[e4] = round_like<TO>(v[e4]);
          u[e4] = round_like<TO>(u4[e4]);
          r[e4] = g[e4] * sigmoid_fast(g[e4]) * u[e4];
        }
        st(P.out0, r[0], r[1], r[2], r[3]);
        if (P.out1) st(P.out1, g[0], g[1], g[2], g[3]);
        if (P.out2) st(P.out2, u[0], u[1], u[2], u[3]);
      } else {
        float g[4], u[4], dg[4], du[4];
        ld4(xa[k], g);
        ld4(xb[k], u);
#pragma unroll
        for (int e4 = 0; e4 < 4; ++e4) {
          const float sg = sigmoid_fast(g[e4]);
          dg[e4] = v[e4] * u[e4] * (sg * (1.0f + g[e4] * (1.0f - sg)));
          du[e4] = v[e4] * (g[e4] * sg);
        }
        st(P.out0, dg[0], dg[1], dg[2], dg[3]);
        st(P.out1, du[0], du[1], du[2], du[3]);
      }
    }
  }
}

// ------------------------------------------------------------------ host
// Tile shapes (id, TI, TJ, RB, NWN, PA, PB) and their constants in the cost
// model of pick_small (fix, first, round); there is one for the persistent
// kernel's tiles too.
#define GLT_SMALL_PLAIN(X)                                              \
  X(0, 1, 1, 1, 1, 8, 8, 0.3f, 3.0f, 4.3f)     /* 32 x 32 */            \
  X(1, 2, 1, 2, 2, 6, 6, 3.1f, 8.8f, 6.0f)     /* 64 x 64 */            \
  X(2, 2, 1, 2, 4, 6, 5, 1.4f, 9.9f, 9.3f)     /* 64 x 128 */           \
  X(3, 4, 1, 4, 4, 6, 4, 6.5f, 11.9f, 16.65f)  /* 128 x 128 */          \
  X(4, 4, 2, 4, 4, 5, 2, 18.6f, 18.1f, 23.2f)  /* 128 x 256 */
#define GLT_SMALL_DUAL(X)                                               \
  X(0, 1, 2, 1, 1, 9, 6, 2.1f, 3.2f, 6.6f)     /* 32 x 32 */            \
  X(1, 2, 2, 2, 2, 6, 4, 2.7f, 14.5f, 12.8f)   /* 64 x 64 */            \
  X(2, 4, 2, 2, 2, 8, 4, 8.0f, 18.6f, 16.5f)   /* 128 x 64 */           \
  X(3, 4, 2, 4, 4, 6, 2, 15.3f, 23.1f, 23.1f)  /* 128 x 128 */
struct SmallShape {
  int rows, cols;
  float fix, first, round;
};
static const SmallShape kPlain[] = {
#define GLT_SMALL_ROW(ID, TI, TJ, RB, NWN, PA, PB, FIX, FIRST, ROUND) {32 * TI, 32 * TJ * NWN, FIX, FIRST, ROUND},
    GLT_SMALL_PLAIN(GLT_SMALL_ROW)
#undef GLT_SMALL_ROW
};
static const SmallShape kDual[] = {
#define GLT_SMALL_ROW(ID, TI, TJ, RB, NWN, PA, PB, FIX, FIRST, ROUND) {32 * TI, 16 * TJ * NWN, FIX, FIRST, ROUND},
    GLT_SMALL_DUAL(GLT_SMALL_ROW)
#undef GLT_SMALL_ROW
};
static const SmallShape kPersistentPlain = {256, 256, 11.8f, 7.6f, 34.95f};
static const SmallShape kPersistentDual = {256, 128, 24.1f, 17.4f, 28.9f};

// The tile shape with the least estimated cost, or -1 for the persistent 256 x
// 256 kernel: speed alone decides, every choice gives the same bits. A launch
// runs in rounds of one tile per CU; large tiles move fewer bytes per product,
// small ones leave no CU idle (4096 output columns are 16 tiles of 256 for 256
// CUs: M = 8, K = 15360 takes 247 us on the persistent kernel, 37 on 32 x 32
// tiles; M = 512: 272 and 99 on 64 x 128; M = 2048: 260 and 207 on 128 x 256;
// M = 4096, one full round, stays persistent).
//
// cost = fix + the longest reduction's K / 1000 times `first` (a round in which
// a workgroup has its CU to itself) or all rounds' K / 1000 times `round`,
// whichever is more, + the outputs' share; at least the bytes that must move.
// The constants are fitted, to no unit, so that the shape of least cost is the
// fastest: over 548 launches timed with every shape (MI355X; M = 1 .. 5056, the
// five GEMMs of layers 4096 x 14336 and 2048 x 11008 with appended, stacked and
// in-place slices, LM heads of 6144 to 128256 rows both ways) its choice takes
// 0.7 % more than the fastest on average, 32 % at most (dInter of 1000 x 11008).
int pick_small(const GemmPlan& plan, int cus) {
  const GArgs& a = plan.args;
  const int mode = a.p[0].mode, of32 = a.p[0].out_f32;
  if (!((mode == EPI_SILU && plan.dual && !of32) ||
        (!plan.dual && (mode == EPI_STORE || ((mode == EPI_DGDU || mode == EPI_RESID) && !of32)))))
    return -1;
  double kmax = 0, kelems = 0, elems = 0, bytes = 0;
  for (int p = 0; p < a.nprob; ++p) {
    const GProb& P = a.p[p];
    const double out = mode == EPI_DGDU || mode == EPI_RESID ? (mode == EPI_DGDU ? 8 : 4)
                                                             : (of32 ? 4 : 2) + (P.out1 ? 2 : 0) + (P.out2 ? 2 : 0);
    elems += (double)P.M * P.N;
    bytes += out * P.M * P.N;
    for (int i = P.seg0; i < P.seg0 + P.nseg; ++i) {
      const GSeg& s = a.s[i];
      const double span = std::max(0, std::min(s.n_hi, P.N) - s.n_lo);
      bytes += span * s.K * (plan.dual ? 4 : 2);
      kelems += span * s.K * P.M;
      double k = 0;  // the reduction of the segment's first column
      for (int j = P.seg0; j < P.seg0 + P.nseg; ++j)
        if (a.s[j].n_lo <= s.n_lo && s.n_lo < a.s[j].n_hi) k += a.s[j].K;
      kmax = std::max(kmax, k);
    }
  }
  if (elems == 0) return -1;
  const double kavg = kelems / elems;
  const float out_us = plan.dual ? 8.0f : mode == EPI_DGDU ? 7.7f : of32 ? 7.9f : 5.9f;  // per 32768 outputs
  auto cost = [&](const SmallShape& s) {
    double tiles = 0;
    for (int p = 0; p < a.nprob; ++p) tiles += (double)cdiv(a.p[p].M, s.rows) * cdiv(a.p[p].N, s.cols);
    const double rounds = std::ceil(tiles / cus);
    const double run = s.fix + std::max(s.first * kmax, s.round * (kmax + (rounds - 1) * kavg)) / 1000. +
                       rounds * out_us * s.rows * s.cols / 32768.;
    return std::max(run, bytes / 5.2e6) + 0.2 * run;  // ties go to the shorter run
  };
  int best = -1;
  double least = cost(plan.dual ? kPersistentDual : kPersistentPlain);
  const SmallShape* const shapes = plan.dual ? kDual : kPlain;
  const int n = plan.dual ? (int)(sizeof kDual / sizeof *kDual) : (int)(sizeof kPlain / sizeof *kPlain);
  for (int i = 0; i < n; ++i) {
    const double c = cost(shapes[i]);
    if (c < least) {
      least = c;
      best = i;
    }
  }
  return best;
}

template <int TI, int TJ, int RB, int NWN, int PA, int PB, typename TO, int MODE, bool DUAL, bool ONCE>
static glt_status launch_small_as(const GArgs& a, hipStream_t st, const char* label) {
  static std::atomic<bool> attr_set[64];
  auto fn = gemm_small_kernel<TI, TJ, RB, NWN, PA, PB, TO, MODE, DUAL, ONCE>;
  int dev = 0;
  GLT_TRY_HIP(hipGetDevice(&dev));
  GLT_CHECK(dev >= 0 && dev < 64, GLT_ERR_HIP, "gemm: device index %d out of range", dev);
  constexpr size_t ring = (size_t)PA * 32 * RB * kBK * 2, red = (size_t)32 * TJ * NWN * 32 * 4;
  constexpr size_t lds = ring > red ? ring : red;
  static_assert(lds <= 160 * 1024, "LDS of one CU");
  if (!attr_set[dev].load(std::memory_order_acquire)) {
    GLT_TRY_HIP(
        hipFuncSetAttribute(reinterpret_cast<const void*>(fn), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    attr_set[dev].store(true, std::memory_order_release);
  }
  GLT_LAUNCH(label, fn, dim3(a.total_tiles), dim3(64 * NWN), lds, st, a);
  GLT_LAUNCH_CHECK("gemm_small");
  return GLT_OK;
}

// Whether B is read once and gone: one problem of a single row of tiles (no
// other workgroup reads the same part of B), and more than half of the 256 MB
// last-level cache of it, so that the next call would not find it there
// whatever the loads say. Non-temporal loads then stream faster and leave the
// cache to the others' operands: gate/up of 8 tokens and 4096 x 15360, two
// layers in turn, 48 -> 41 us, of 64 55 -> 43. With several row tiles the B
// that they share came twice (200 tokens: MLP forward 180 -> 222 us), and
// smaller weights called again and again were lost from the cache (2048 x
// 11008, 8 tokens: 34 -> 41 us).
static bool read_once(const GArgs& a, bool dual) {
  const GProb& P = a.p[0];
  if (a.nprob != 1 || P.tiles_m > 1) return false;
  int64_t bytes = 0;
  for (int i = P.seg0; i < P.seg0 + P.nseg; ++i)
    bytes += (int64_t)std::max(0, std::min(a.s[i].n_hi, P.N) - a.s[i].n_lo) * a.s[i].K * (dual ? 4 : 2);
  return bytes > (int64_t)128 << 20;
}

template <int TI, int TJ, int RB, int NWN, int PA, int PB, typename TO, int MODE, bool DUAL>
static glt_status launch_small(const GArgs& a, hipStream_t st, const char* label) {
  // (the non-temporal form only where the cost model can come with so much B:
  // f32 outputs, dX and the head's, are narrow and of 32 x 32 tiles then)
  if constexpr (MODE == EPI_SILU || (MODE == EPI_STORE && (sizeof(TO) == 2 || TI == 1)))
    if (read_once(a, DUAL)) return launch_small_as<TI, TJ, RB, NWN, PA, PB, TO, MODE, DUAL, true>(a, st, label);
  return launch_small_as<TI, TJ, RB, NWN, PA, PB, TO, MODE, DUAL, false>(a, st, label);
}

glt_status run_small(GemmPlan& plan, int shape, hipStream_t st) {
  GArgs& a = plan.args;
  const SmallShape& S = plan.dual ? kDual[shape] : kPlain[shape];
  const int mode = a.p[0].mode, of32 = a.p[0].out_f32;
  int tiles = 0;
  for (int p = 0; p < a.nprob; ++p) {
    GProb& P = a.p[p];
    GLT_CHECK(P.mode == mode && P.out_f32 == of32, GLT_ERR_INVALID_ARG, "run_gemm: mixed epilogues in one launch");
    P.tiles_m = (int)cdiv(P.M, S.rows);
    P.tiles_n = (int)cdiv(P.N, S.cols);
    P.tile_begin = tiles;
    tiles += P.tiles_m * P.tiles_n;
  }
  a.total_tiles = tiles;
  if (tiles == 0) return GLT_OK;
#define GLT_SMALL_RUN(ID, TI, TJ, RB, NWN, PA, PB, FIX, FIRST, ROUND) \
  if (plan.dual && shape == ID && mode == EPI_SILU)                   \
    return launch_small<TI, TJ, RB, NWN, PA, PB, uint16_t, EPI_SILU, true>(a, st, plan.label);
  GLT_SMALL_DUAL(GLT_SMALL_RUN)
#undef GLT_SMALL_RUN
#define GLT_SMALL_RUN(ID, TI, TJ, RB, NWN, PA, PB, FIX, FIRST, ROUND)                                        \
  if (!plan.dual && shape == ID) {                                                                           \
    if (mode == EPI_STORE)                                                                                   \
      return of32 ? launch_small<TI, TJ, RB, NWN, PA, PB, float, EPI_STORE, false>(a, st, plan.label)        \
                  : launch_small<TI, TJ, RB, NWN, PA, PB, uint16_t, EPI_STORE, false>(a, st, plan.label);    \
    if (mode == EPI_DGDU) return launch_small<TI, TJ, RB, NWN, PA, PB, uint16_t, EPI_DGDU, false>(a, st, plan.label); \
    if (mode == EPI_RESID && !of32)                                                                          \
      return launch_small<TI, TJ, RB, NWN, PA, PB, uint16_t, EPI_RESID, false>(a, st, plan.label);           \
  }
  GLT_SMALL_PLAIN(GLT_SMALL_RUN)
#undef GLT_SMALL_RUN
  set_error("run_gemm: no small-tile kernel for mode %d dual %d", mode, (int)plan.dual);
  return GLT_ERR_UNSUPPORTED;
}

}  // namespace glt
