// Device helpers shared by the segment-list GEMM kernels (gemm.hip,
// gemm_small.hip).
#pragma once

#include "gemm.hpp"

namespace glt {

constexpr int kBK = 64;  // K-step of the MFMA kernels
constexpr uint32_t kExtent = 0x7FFFFFF0u;                // buffer extent below kOob

// ---------------------------------------------------------------- epilogue
// GEMM outputs are rounded with the gfx950 conversion instruction: round to
// nearest even, the same result as the reference's bias-and-shift rounding
// (src/kernels_elementwise_impl.inc:570-580) for every finite value. (The
// bit-exact conversion entry points keep the reference's integer form,
// which also fixes what NaN payloads become.)
__device__ __forceinline__ uint16_t bf16_hw(float v) { return __builtin_bit_cast(uint16_t, (__bf16)v); }
__device__ __forceinline__ uint32_t pack2_hw(float a, float b) {
  typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
  const bf16x2_t v = {(__bf16)a, (__bf16)b};
  return __builtin_bit_cast(uint32_t, v);
}
// sigmoid 1/(1+exp(-g)) from the hardware exp2 and reciprocal (each within
// about 1 ulp in f32) instead of the correctly rounded library sequences,
// which cost some 30 instructions per element in the epilogues; the values
// are rounded to the path dtype right after.
__device__ __forceinline__ float sigmoid_fast(float g) {
  return __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-g * 1.4426950408889634f));
}

template <typename TO>
__device__ __forceinline__ float ld_elem(const void* p, int64_t i) {
  if constexpr (sizeof(TO) == 4) return static_cast<const float*>(p)[i];
  else return bf16_to_f32(static_cast<const uint16_t*>(p)[i]);
}
template <typename TO>
__device__ __forceinline__ void st_elem(void* p, int64_t i, float v) {
  if constexpr (sizeof(TO) == 4) static_cast<float*>(p)[i] = v;
  else static_cast<uint16_t*>(p)[i] = bf16_hw(v);
}
template <typename TO>
__device__ __forceinline__ float round_like(float v) {
  if constexpr (sizeof(TO) == 4) return v;
  else return bf16_to_f32(bf16_hw(v));
}

// The saved pre-activations that the EPI_DGDU form of epilogue() reads.
struct SavedGU {
  float g, u;
};
template <typename TO, int MODE>
__device__ __forceinline__ SavedGU load_saved(const GProb& P, int m, int n) {
  if constexpr (MODE != EPI_DGDU) return SavedGU{};
  if (m >= P.M || n >= P.N) return SavedGU{};
  const int64_t oa = (int64_t)m * P.ldaux + n;
  return SavedGU{ld_elem<TO>(P.aux0, oa), ld_elem<TO>(P.aux1, oa)};
}

// a0 = accumulator (gate accumulator in the dual form), a1 = up accumulator.
template <typename TO, int MODE>
__device__ __forceinline__ void epilogue(const GProb& P, int m, int n, float a0, float a1, SavedGU saved) {
  if (m >= P.M || n >= P.N) return;
  const int64_t o = (int64_t)m * P.ldo + n;
  if constexpr (MODE == EPI_STORE) {
    float v = P.alpha * a0;
    if (P.beta != 0.f) v += P.beta * ld_elem<TO>(P.out0, o);
    st_elem<TO>(P.out0, o, v);
  } else if constexpr (MODE == EPI_RESID) {
    // the layer output is rounded to the path dtype, then added to the
    // residual stream (reference x = x + ffn_out, src/layer_forward_impl.inc:271-275)
    st_elem<TO>(P.out0, o, ld_elem<TO>(P.out0, o) + round_like<TO>(P.alpha * a0));
  } else if constexpr (MODE == EPI_SILU) {
    // gate/up pre-activations leave the accumulator rounded to the path
    // dtype (bf16 in the reference, src/layer_forward_impl.inc:72,122), and
    // silu(g)*u is formed from those values in the reference's f32 order
    // (src/kernels_elementwise_impl.inc:440-446): sg = 1/(1+exp(-g)), (g*sg)*u,
    // with sg from sigmoid_fast.
    const float g = round_like<TO>(a0), u = round_like<TO>(a1);
    const float sg = sigmoid_fast(g);
    st_elem<TO>(P.out0, o, g * sg * u);
    if (P.out1) st_elem<TO>(P.out1, o, g);
    if (P.out2) st_elem<TO>(P.out2, o, u);
  } else {
    // SiLU*up derivative on the dInter accumulator
    // (reference fused_gate_up_bwd_kernel, src/kernels_elementwise_impl.inc:107-117).
    const float g = saved.g, u = saved.u;
    const float sg = sigmoid_fast(g);
    const float gv = g * sg;
    const float sgrad = sg * (1.0f + g * (1.0f - sg));
    st_elem<TO>(P.out0, o, a0 * u * sgrad);
    st_elem<TO>(P.out1, o, a0 * gv);
  }
}

// Locates problem and tile of tile index t. Within a problem tiles run in
// groups of kGroupM M-tiles, so tiles with neighbouring indices share A and
// B rows in L2.
// (4 measured best of 1, 2, 4, 8, 16 on the step's GEMMs: each XCD's 32
// tiles of a round form a 4 x 8 block.)
constexpr int kGroupM = 4;
__device__ __forceinline__ int locate_tile(const GArgs& args, int t, int& tm, int& tn, int group_m = kGroupM) {
  int pi = 0;
  while (pi + 1 < args.nprob && t >= args.p[pi + 1].tile_begin) ++pi;
  const GProb& P = args.p[pi];
  t -= P.tile_begin;
  const int per_group = group_m * P.tiles_n;
  const int g = t / per_group;
  const int first_m = g * group_m;
  const int gm = min(P.tiles_m - first_m, group_m);
  const int r = t - g * per_group;
  tm = first_m + r % gm;
  tn = r / gm;
  return pi;
}

__device__ __forceinline__ bool seg_hits(const GSeg& S, const GProb& P, int n0, int bn) {
  return S.K > 0 && max(S.n_lo, n0) < min(min(S.n_hi, P.N), n0 + bn);
}

// Rows are 64 bf16 = 128 bytes, one cache line each, so every global
// request a tile issues moves a whole line. gfx950 LDS serves a
// 16-byte-per-lane access 16 lanes at a time over 64 banks (256 bytes); a
// 16-lane group reading one logical chunk of 16 consecutive rows touches
// bank group 8*(row&1) + physical chunk, so the physical chunk is the
// logical one XOR (row>>1)&7, which makes the 16 groups distinct.
__device__ __forceinline__ int swz_key(int row) { return (row >> 1) & 7; }

// Buffer descriptor of a wave-uniform base and extent. The compiler loses
// track of their uniformity through the kernel's position bookkeeping and
// would wrap every buffer load in a per-lane loop over descriptor values;
// readfirstlane states it.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t uni_rsrc(const void* p, uint32_t n) {
  const uint64_t v = reinterpret_cast<uint64_t>(p);
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
  return make_rsrc(reinterpret_cast<const void*>(((uint64_t)hi << 32) | lo), __builtin_amdgcn_readfirstlane(n));
}

// s_waitcnt immediate (gfx9 encoding) that waits for vmcnt <= n and leaves
// expcnt / lgkmcnt unconstrained.
constexpr int vmcnt_enc(int n) { return (n & 15) | ((n >> 4) << 14) | (7 << 4) | (15 << 8); }

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

// Orders one wavefront's LDS accesses across lanes: LDS executes a
// wavefront's instructions in order, so only the compiler must not move
// accesses across this point.
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

typedef __attribute__((address_space(3))) void lds_void;
// Direct-to-LDS load of 16 bytes per lane (lane L lands at dst + 16 L). Not a
// template: in one, the host pass drops every kernel that instantiates it
// (the builtin's arguments are checked against the host target).
__device__ __forceinline__ void load_lds16(__amdgpu_buffer_rsrc_t r, void* dst, uint32_t voff, uint32_t soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void*)dst, 16, voff, soff, 0, 0);
}

}  // namespace glt
