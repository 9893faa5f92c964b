// Segment-list GEMM over strided operands: the f32 path, bf16 shapes that the
// fragment layout does not take, and the graft-GEMM probes.
#include <algorithm>
#include <atomic>

#include "gemm.hpp"
#include "gemm_dev.hpp"

namespace glt {

// Eight-byte or sixteen-byte loads of four consecutive elements as f32.
template <int KIND>
__device__ __forceinline__ f32x4 ld4_kind(const void* p, int64_t i) {
  if constexpr (KIND == LD_BF16) {
    const u32x2 w = *reinterpret_cast<const u32x2*>(static_cast<const uint16_t*>(p) + i);
    return f32x4{__uint_as_float(w.x << 16), __uint_as_float(w.x & 0xFFFF0000u), __uint_as_float(w.y << 16),
                 __uint_as_float(w.y & 0xFFFF0000u)};
  } else {
    f32x4 v = *reinterpret_cast<const f32x4*>(static_cast<const float*>(p) + i);
    if constexpr (KIND == LD_F32_AS_BF16)
      v = f32x4{bf16_to_f32(f32_to_bf16(v.x)), bf16_to_f32(f32_to_bf16(v.y)), bf16_to_f32(f32_to_bf16(v.z)),
                bf16_to_f32(f32_to_bf16(v.w))};
    return v;
  }
}
template <int KIND>
__device__ __forceinline__ float ld_kind(const void* p, int64_t i) {
  if constexpr (KIND == LD_BF16) return bf16_to_f32(static_cast<const uint16_t*>(p)[i]);
  else if constexpr (KIND == LD_F32) return static_cast<const float*>(p)[i];
  else return bf16_to_f32(f32_to_bf16(static_cast<const float*>(p)[i]));
}

template <int V>
struct Kind {
  static constexpr int value = V;
};

// One operand of a segment: element (r, k) = p[(r - r0) * ld + k * ks] for r
// in [lo, hi), zero outside.
struct StridedOp {
  const void* p;
  int64_t ld, ks;
  int r0, lo, hi;
};
// How an operand's 4-element pieces are read: along k, along the rows, or one
// element at a time. Pieces must be aligned and lie wholly inside or outside
// [lo, hi) and [0, K).
enum : int { PIECE_K = 0, PIECE_ROW = 1, PIECE_NONE = 2 };
template <int KIND>
__device__ __forceinline__ int piece_mode(const StridedOp& o, int K) {
  const uint64_t al = (uint64_t)(KIND == LD_BF16 ? 7 : 15);
  if ((reinterpret_cast<uint64_t>(o.p) & al) != 0) return PIECE_NONE;
  if (o.ks == 1 && o.ld % 4 == 0 && K % 4 == 0) return PIECE_K;
  if (o.ld == 1 && o.ks % 4 == 0 && o.r0 % 4 == 0 && o.lo % 4 == 0 && o.hi % 4 == 0) return PIECE_ROW;
  return PIECE_NONE;
}

// =========================================================================
// f32 MFMA kernel (v_mfma_f32_32x32x2_f32: f32 products, f32 sums), operands
// of any stride converted to f32 as they are staged.
//
// Every output is the sum, in order, of 16 partial sums (dual: 8); part p takes
// the groups of 16 K whose number in their segment is p mod 16, each from its
// segments' first group to the last. So a row's bits depend neither on the rows
// beside it nor on which of the forms below a launch of that size takes.
//
// TILE 32: one 32 x 32 output tile per workgroup of NW wavefronts (dual: the
// gate and up columns of it); each wavefront takes 16 K of every chunk of 16
// NW, into its accumulators (one per part) in turn. A chunk costs a load latency
// whatever its size, so launches of few tiles take many wavefronts (M = N = 512,
// K = 3328: 33 us with 16, 98 with 4). TILE 64: one 64 x 64 tile, a 32 x 32
// quadrant per four wavefronts over chunks of 64 K, 16 each: half the operand
// bytes per product, for launches that fill the chip with those.
//
// Operand tiles are staged as [k][row] in two LDS buffers (a row of 32 or 64
// floats plus one: the transposing writes of four k and the reads of 32 rows
// both spread over the banks); the next chunk's global loads are in flight
// during the MFMAs of the current one. Bound by the f32 MFMA rate (64 cycles
// per 4096 FLOP and SIMD) once the loads are 16 bytes wide: the 512-token f32
// layer's GEMMs (hidden 512, base 1408, slice 256) take 125 us, 1286 on an FMA
// kernel with scalar loads. The accumulators of the parts cost little against
// one each (2048 tokens of 1024 x 2816: 1148 us and 1117; dInter 203 and 171,
// its 16-wavefront tiles share no CU) and halve the distance to 64-bit sums
// (6.6e-7 -> 4.1e-7). The dual form of four wavefronts is held to three a SIMD:
// left to itself the compiler takes registers for two (329 -> 383 us).
// =========================================================================
template <bool DUAL, int TILE, int NW>
struct StridedGeom {
  static constexpr int kParts = DUAL ? 8 : 16;
  static constexpr int BK = TILE == 32 ? 16 * NW : 64, NB = DUAL ? 2 : 1, PITCH = TILE + 1;
  static constexpr int kOp = BK * PITCH;           // floats of one staged operand
  static constexpr int kStage = (1 + NB) * kOp;    // one buffer
  static constexpr int kRed = NB * NW * 32 * 33;   // floats of one partial tile of every wavefront
  static constexpr int kLds = (2 * kStage > kRed ? 2 * kStage : kRed) * 4;
  static constexpr int kAcc = kParts * 16 / BK;                       // accumulators of a wavefront
  static constexpr int kPieces = BK * TILE / (4 * 64 * NW);           // 4-element pieces of a thread and operand
  static_assert(TILE == 32 || (TILE == 64 && NW == 16 && !DUAL), "64 x 64 tiles: four quadrants, four wavefronts each");
  static_assert(kLds <= 160 * 1024, "LDS of one CU");
};

template <int LA, int LB, typename TO, int MODE, bool DUAL, int TILE, int NW>
__global__ void __launch_bounds__(64 * NW, DUAL && NW == 4 ? 3 : 1) gemm_strided_kernel(const GArgs args) {
  using Geom = StridedGeom<DUAL, TILE, NW>;
  constexpr int BK = Geom::BK, NB = Geom::NB, PITCH = Geom::PITCH, kOp = Geom::kOp, kThreads = 64 * NW;
  constexpr int NACC = Geom::kAcc, NQ = Geom::kPieces;
  extern __shared__ __attribute__((aligned(16))) float lds[];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  int tm, tn;
  const int64_t t = (int64_t)blockIdx.y * gridDim.x + blockIdx.x;
  if (t >= args.total_tiles) return;
  const int pi = locate_tile(args, (int)t, tm, tn);
  const GProb& P = args.p[pi];
  const int m0 = tm * TILE, n0 = tn * TILE, send = P.seg0 + P.nseg;

  // ---- chunk position: segment s, offset k0 in it
  int s = P.seg0 - 1;
  uint32_t k0 = 0, K = 0;
  // Four-element pieces of one operand's chunk: piece q of a thread is number e
  // = tid + 64 NW q. Along k: a wavefront takes PR rows x PK pieces (256 bytes
  // of a row, and transposing writes that cover all banks). Along the rows:
  // rows fastest. Addresses are formed once per segment and stepped per chunk
  // (formed per chunk they were half of the loop's instructions).
  constexpr int PK = BK / 4 < 16 ? BK / 4 : 16, PR = 64 / PK;
  struct Src {
    const char* p[NQ];  // piece q of the chunk at k0
    uint32_t k[NQ];    // its k within a chunk, or past any K for a row outside the operand
    int off[NQ], inc;  // where its elements go in the staged [k][row] tile
    int mode;
    int64_t step, ks;  // bytes per chunk, per k
  };
  constexpr uint32_t kNoRow = 0x80000000u;  // (k0 + kNoRow + 3 stays in 32 bits: k0 is a multiple of 16 below 2^31)
  Src sa, sb[NB];
  f32x4 ra[NQ], rb[NB][NQ];
  auto setup = [&](auto kind, Src& r, const StridedOp& o, int base) __attribute__((always_inline)) {
    constexpr int KIND = decltype(kind)::value, E = KIND == LD_BF16 ? 2 : 4;
    r.mode = o.p ? piece_mode<KIND>(o, (int)K) : PIECE_NONE;
    r.ks = o.ks * E;
    r.step = r.ks * BK;
    r.inc = r.mode == PIECE_ROW ? 1 : PITCH;
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      const int e = tid + kThreads * q;
      const int row = r.mode == PIECE_ROW ? 4 * (e % (TILE / 4)) : e / PK % PR + PR * (e / 64 / (BK / 4 / PK));
      const int k = r.mode == PIECE_ROW ? e / (TILE / 4) : 4 * (e % PK + PK * (e / 64 % (BK / 4 / PK)));
      const bool in = o.p && base + row >= o.lo && base + row < o.hi;
      r.k[q] = in ? (uint32_t)k : kNoRow;
      r.off[q] = k * PITCH + row;
      r.p[q] = static_cast<const char*>(o.p) + ((int64_t)(base + row - o.r0) * o.ld + (int64_t)k * o.ks) * E;
    }
  };
  auto fetch = [&](auto kind, Src& o, f32x4* r) __attribute__((always_inline)) {
    constexpr int KIND = decltype(kind)::value;
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      r[q] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (o.mode != PIECE_NONE) {
        if (k0 + o.k[q] < K) r[q] = ld4_kind<KIND>(o.p[q], 0);
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (k0 + o.k[q] + i < K) r[q][i] = ld_kind<KIND>(o.p[q] + i * o.ks, 0);
      }
      o.p[q] += o.step;
    }
  };
  auto put = [&](float* dst, const Src& o, const f32x4* r) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < NQ; ++q)
#pragma unroll
      for (int i = 0; i < 4; ++i) dst[o.off[q] + i * o.inc] = r[q][i];
  };
  auto next_seg = [&]() __attribute__((always_inline)) {
    ++s;
    while (s < send && !seg_hits(args.s[s], P, n0, TILE)) ++s;
    k0 = 0;
    if (s >= send) return;
    const GSeg& S = args.s[s];
    K = (uint32_t)S.K;
    const int64_t ae = LA == LD_BF16 ? 2 : 4;
    setup(Kind<LA>{}, sa,
          StridedOp{static_cast<const char*>(S.A) + (int64_t)S.a_col * S.a_ks * ae, S.lda, S.a_ks, 0, 0, P.M}, m0);
#pragma unroll
    for (int h = 0; h < NB; ++h)
      setup(Kind<LB>{}, sb[h],
            StridedOp{h ? S.B1 : S.B0, h ? S.ldb1 : S.ldb0, S.b_ks, h ? S.b1_row0 : S.b0_row0, S.n_lo,
                      min(S.n_hi, P.N)},
            n0);
  };
  auto load = [&]() __attribute__((always_inline)) {
    fetch(Kind<LA>{}, sa, ra);
#pragma unroll
    for (int h = 0; h < NB; ++h) fetch(Kind<LB>{}, sb[h], rb[h]);
  };

  f32x16 acc[NB][NACC];
#pragma unroll
  for (int h = 0; h < NB; ++h)
#pragma unroll
    for (int j = 0; j < NACC; ++j) acc[h][j] = f32x16{};
  const int lr = lane & 31, lk = lane >> 5;
  // this wavefront's first k of a chunk, rows and columns of the tile
  const int kw = 16 * (TILE == 32 ? wave : wave >> 2);
  const int am = TILE == 32 ? 0 : 32 * (wave >> 1 & 1), bn = TILE == 32 ? 0 : 32 * (wave & 1);
  next_seg();
  if (s < send) load();
  int p = 0;
  while (s < send) {
    // the chunks of one turn through the accumulators, or those left of the segment
#pragma unroll
    for (int j = 0; j < NACC; ++j) {
      float* const st = lds + p * Geom::kStage;
      p ^= 1;
      put(st, sa, ra);
#pragma unroll
      for (int h = 0; h < NB; ++h) put(st + (1 + h) * kOp, sb[h], rb[h]);
      k0 += BK;
      const bool last = k0 >= K;
      if (last) next_seg();
      __syncthreads();  // (whoever writes the other buffer next has passed this barrier after reading it)
      if (s < send) load();
#pragma unroll
      for (int k = 0; k < 16; k += 2) {
        const int o = (kw + k + lk) * PITCH + lr;
        const float a = st[o + am];
#pragma unroll
        for (int h = 0; h < NB; ++h)
          acc[h][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a, st[(1 + h) * kOp + o + bn], acc[h][j], 0, 0, 0);
      }
      if (last) break;
    }
  }

  // The parts are added through LDS, an accumulator of every wavefront at a
  // time: lane l holds output column l & 31, rows 8 (e >> 2) + 4 (l >> 5) + (e &
  // 3); [operand][wavefront][32 rows][33].
  constexpr int NV = TILE * TILE / kThreads;  // a thread's outputs
  float v[NV][2];
  SavedGU saved[NV];  // in flight meanwhile
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int e = tid + kThreads * i;
    v[i][0] = v[i][1] = 0.f;
    saved[i] = load_saved<TO, MODE>(P, m0 + e / TILE, n0 + e % TILE);
  }
#pragma unroll
  for (int j = 0; j < NACC; ++j) {
    __syncthreads();
#pragma unroll
    for (int h = 0; h < NB; ++h)
#pragma unroll
      for (int e = 0; e < 16; ++e)
        lds[((h * NW + wave) * 32 + 8 * (e >> 2) + 4 * lk + (e & 3)) * 33 + lr] = acc[h][j][e];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int e = tid + kThreads * i, row = e / TILE, col = e % TILE;
#pragma unroll
      for (int h = 0; h < NB; ++h)
#pragma unroll
        for (int w = 0; w < (TILE == 32 ? NW : 4); ++w) {
          const int from = TILE == 32 ? w : 4 * w + 2 * (row >> 5) + (col >> 5);
          v[i][h] += lds[((h * NW + from) * 32 + (row & 31)) * 33 + (col & 31)];
        }
    }
  }
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int e = tid + kThreads * i;
    epilogue<TO, MODE>(P, m0 + e / TILE, n0 + e % TILE, v[i][0], v[i][1], saved[i]);
  }
}

// ------------------------------------------------------------------ host
template <int LA, int LB, typename TO, int MODE, bool DUAL, int TILE, int NW>
static glt_status launch_strided(GemmPlan& plan, hipStream_t st) {
  static std::atomic<bool> attr_set[64];
  constexpr int lds = StridedGeom<DUAL, TILE, NW>::kLds;
  auto fn = gemm_strided_kernel<LA, LB, TO, MODE, DUAL, TILE, NW>;
  int dev = 0;
  GLT_TRY_HIP(hipGetDevice(&dev));
  GLT_CHECK(dev >= 0 && dev < 64, GLT_ERR_HIP, "gemm: device index %d out of range", dev);
  if (!attr_set[dev].load(std::memory_order_acquire)) {
    GLT_TRY_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(fn), hipFuncAttributeMaxDynamicSharedMemorySize, lds));
    attr_set[dev].store(true, std::memory_order_release);
  }
  GArgs& a = plan.args;
  int64_t tiles = 0;
  for (int p = 0; p < a.nprob; ++p) {
    GProb& P = a.p[p];
    P.tiles_m = (int)cdiv(P.M, TILE);
    P.tiles_n = (int)cdiv(P.N, TILE);
    P.tile_begin = (int)tiles;
    tiles += (int64_t)P.tiles_m * P.tiles_n;
    GLT_CHECK(tiles < INT32_MAX, GLT_ERR_SHAPE, "run_gemm(%s): %lld tiles", plan.label, (long long)tiles);
  }
  a.total_tiles = (int)tiles;
  if (tiles == 0) return GLT_OK;
  // (a grid dimension holds at most 2^32 threads: 2^24 tiles of 256, e.g. 2^29
  // rows of a 1-column layer)
  constexpr int64_t kGridX = 1 << 20;
  const dim3 grid((unsigned)std::min(tiles, kGridX), (unsigned)cdiv(tiles, kGridX));
  GLT_LAUNCH(plan.label, fn, grid, dim3(64 * NW), lds, st, a);
  GLT_LAUNCH_CHECK("gemm_strided");
  return GLT_OK;
}

glt_status run_strided(GemmPlan& plan, hipStream_t st) {
  const GArgs& a = plan.args;
  const int mode = a.p[0].mode, of32 = a.p[0].out_f32, la = plan.a_kind, lb = plan.b_kind;
  int64_t tiles32 = 0, tiles64 = 0;
  for (int p = 0; p < a.nprob; ++p) {
    GLT_CHECK(a.p[p].mode == mode && a.p[p].out_f32 == of32, GLT_ERR_INVALID_ARG,
              "run_gemm: mixed epilogues in one launch");
    tiles32 += cdiv(a.p[p].M, 32) * cdiv(a.p[p].N, 32);
    tiles64 += cdiv(a.p[p].M, 64) * cdiv(a.p[p].N, 64);
  }
  int cus = 0;
  const glt_status rc = device_cus(cus);
  if (rc != GLT_OK) return rc;
  // 64 x 64 tiles where there are several per CU, else 32 x 32, with the more
  // wavefronts where there is less than one per CU
  const bool big = tiles64 >= 3 * (int64_t)cus, few = tiles32 <= cus;
#define GLT_STRIDED(LA_, LB_, TO_, MODE_, DUAL_)                                                          \
  if (la == LA_ && lb == LB_ && (sizeof(TO_) == 4) == (of32 != 0) && mode == MODE_ && plan.dual == DUAL_) \
    return big && !DUAL_   ? launch_strided<LA_, LB_, TO_, MODE_, DUAL_, DUAL_ ? 32 : 64, DUAL_ ? 8 : 16>(plan, st)    \
           : few && !DUAL_ ? launch_strided<LA_, LB_, TO_, MODE_, DUAL_, 32, DUAL_ ? 8 : 16>(plan, st)    \
           : few || !DUAL_ ? launch_strided<LA_, LB_, TO_, MODE_, DUAL_, 32, 8>(plan, st)                 \
                           : launch_strided<LA_, LB_, TO_, MODE_, DUAL_, 32, DUAL_ ? 4 : 8>(plan, st);
  // f32 path
  GLT_STRIDED(LD_F32, LD_F32, float, EPI_STORE, false)
  GLT_STRIDED(LD_F32, LD_F32, float, EPI_RESID, false)
  GLT_STRIDED(LD_F32, LD_F32, float, EPI_SILU, true)
  GLT_STRIDED(LD_F32, LD_F32, float, EPI_DGDU, false)
  // bf16 path on shapes the MFMA kernels do not take
  GLT_STRIDED(LD_BF16, LD_BF16, uint16_t, EPI_STORE, false)
  GLT_STRIDED(LD_BF16, LD_BF16, uint16_t, EPI_RESID, false)
  GLT_STRIDED(LD_BF16, LD_BF16, float, EPI_STORE, false)
  GLT_STRIDED(LD_BF16, LD_BF16, uint16_t, EPI_SILU, true)
  GLT_STRIDED(LD_BF16, LD_BF16, uint16_t, EPI_DGDU, false)
  // graft-GEMM probes (f32 operands rounded to bf16 on load)
  GLT_STRIDED(LD_BF16, LD_F32_AS_BF16, float, EPI_STORE, false)
  GLT_STRIDED(LD_F32_AS_BF16, LD_BF16, float, EPI_STORE, false)
  GLT_STRIDED(LD_F32_AS_BF16, LD_F32_AS_BF16, float, EPI_STORE, false)
#undef GLT_STRIDED
  set_error("run_gemm: no strided kernel for kinds (%d,%d) out_f32 %d mode %d dual %d", la, lb, of32, mode,
            (int)plan.dual);
  return GLT_ERR_UNSUPPORTED;
}

}  // namespace glt
