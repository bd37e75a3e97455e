// gemm_weights.h -- what the projection kernels share: their arguments, the
// weights' device layout as a wave reads it (gemm.hip describes it) and its
// dequantization into MFMA B fragments, and the SwiGLU store.
#pragma once

#include "../common.h"

namespace tgohip {

struct GemmArgs {
  const void* x;        // [M,K] f16 or f32 (or the hi plane of an XK_X2 pair)
  const void* xlo;      // XK_X2: the lo plane [M,K] f16; null otherwise
  const void* wp;       // packed payload
  const half_t* ws;     // packed scales (form dependent)
  const half_t* wz;     // packed zero+1024 (I4_TGO only)
  void* y;              // output (EPI dependent)
  float* part;          // split-K partials: split s at part + s * pstride, [M][N]
  size_t pstride;
  int M, K, N;
  int ksteps_per_split;
};

__device__ __forceinline__ half2_t as_h2(uint32_t u) {
  union { uint32_t u; half2_t h; } c;
  c.u = u;
  return c.h;
}

// ---- dequantization of one substep's B fragment (8 consecutive k) ----------
__device__ __forceinline__ half8_t deq_i4_sym(uint32_t w, half_t s) {
  const half2_t sp = {s, s};
  // A nibble in bits 0-3 of a 16-bit half merged into 0x6400 (1024.0) reads
  // as 1024 + q; one in bits 4-7 merged into 0x5400 (64.0, whose mantissa bit
  // 4 is worth 1) reads as 64 + q. Subtracting 1032 or 72 leaves q - 8
  // exactly, so substeps 0/1 come from w and 2/3 from w >> 8 with one shift.
  // The masks sit in registers so each mask-and-merge is one v_and_or_b32
  // (its encoding takes no literal constants).
  uint32_t m0 = 0x000F000Fu, m1 = 0x00F000F0u, g0 = 0x64006400u, g1 = 0x54005400u;
  asm("" : "+v"(m0), "+v"(m1), "+v"(g0), "+v"(g1));
  const half2_t b0 = {(half_t)1032.f, (half_t)1032.f}, b1 = {(half_t)72.f, (half_t)72.f};
  const uint32_t w8 = w >> 8;
  const half2_t h[4] = {(as_h2((w & m0) | g0) - b0) * sp, (as_h2((w & m1) | g1) - b1) * sp,
                        (as_h2((w8 & m0) | g0) - b0) * sp, (as_h2((w8 & m1) | g1) - b1) * sp};
  half8_t o;
#pragma unroll
  for (int j = 0; j < 4; j++) {
    o[2 * j] = h[j][0];
    o[2 * j + 1] = h[j][1];
  }
  return o;
}
// The codes q - 8 of one substep's B fragment, unscaled: small integers, exact
// in f16 (the masks and merge constants of deq_i4_sym).
__device__ __forceinline__ half8_t i4_sym_codes(uint32_t w) {
  uint32_t m0 = 0x000F000Fu, m1 = 0x00F000F0u, g0 = 0x64006400u, g1 = 0x54005400u;
  asm("" : "+v"(m0), "+v"(m1), "+v"(g0), "+v"(g1));
  const half2_t b0 = {(half_t)1032.f, (half_t)1032.f}, b1 = {(half_t)72.f, (half_t)72.f};
  const uint32_t w8 = w >> 8;
  const half2_t h[4] = {as_h2((w & m0) | g0) - b0, as_h2((w & m1) | g1) - b1,
                        as_h2((w8 & m0) | g0) - b0, as_h2((w8 & m1) | g1) - b1};
  half8_t o;
#pragma unroll
  for (int j = 0; j < 4; j++) {
    o[2 * j] = h[j][0];
    o[2 * j + 1] = h[j][1];
  }
  return o;
}
__device__ __forceinline__ half8_t deq_i4_asym(uint32_t w, half8_t s, half8_t zz) {
  half8_t o;
#pragma unroll
  for (int j = 0; j < 4; j++) {
    half2_t h = as_h2(((w >> (4 * j)) & 0x000F000Fu) | 0x64006400u);
    const half2_t z2 = {zz[2 * j], zz[2 * j + 1]};
    const half2_t s2 = {s[2 * j], s[2 * j + 1]};
    h = h - z2;
    h = h * s2;
    o[2 * j] = h[0];
    o[2 * j + 1] = h[1];
  }
  return o;
}
__device__ __forceinline__ half8_t deq_i8(uint32_t w0, uint32_t w1, half8_t s) {
  const half2_t bias = {(half_t)1152.f, (half_t)1152.f};
  half8_t o;
  const uint32_t ws[2] = {w0, w1};
#pragma unroll
  for (int u = 0; u < 2; u++) {
    half2_t lo = as_h2((ws[u] & 0x00FF00FFu) | 0x64006400u);
    half2_t hi = as_h2(((ws[u] >> 8) & 0x00FF00FFu) | 0x64006400u);
    const half2_t s0 = {s[4 * u], s[4 * u + 1]}, s1 = {s[4 * u + 2], s[4 * u + 3]};
    lo = (lo - bias) * s0;
    hi = (hi - bias) * s1;
    o[4 * u] = lo[0];
    o[4 * u + 1] = lo[1];
    o[4 * u + 2] = hi[0];
    o[4 * u + 3] = hi[1];
  }
  return o;
}

// The lane's raw material for one (nb, ks): payload plus the scales it needs,
// sized per form so no register is spent on another form's fields.
template <int FORM> struct BRaw;
template <> struct BRaw<TGOHIP_FORM_F16> { uint4 p[4]; };
template <> struct BRaw<TGOHIP_FORM_I8> { uint4 p[2]; uint4 s[4]; };
template <> struct BRaw<TGOHIP_FORM_I4_TGO> { uint4 p; uint4 s[4]; uint4 z[4]; };
template <> struct BRaw<TGOHIP_FORM_I4_SYM> { uint4 p; uint32_t s; };

typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

// A 16-byte weight load; NT: non-temporal (the nt bit), for a launch that
// reads each weight once. The small-M kernel's int4 gate/up at one row went
// from 15.6 to 13.5 us with it, the LM head from 70.7 to 64.8; the pipelined
// kernel's row tiles share weights through L2, and nt loads made its 64- and
// 128-row down 12-18% slower.
template <bool NT>
__device__ __forceinline__ uint4 ldw16(const void* p) {
  if constexpr (NT) {
    const u32x4_t v = __builtin_nontemporal_load((const u32x4_t*)p);
    return make_uint4(v.x, v.y, v.z, v.w);
  } else {
    return *(const uint4*)p;
  }
}

template <bool NT = false>
__device__ __forceinline__ void load_braw(const GemmArgs& g, int nb, int ks, int lane,
                                          BRaw<TGOHIP_FORM_F16>& r) {
  const size_t blk = (size_t)nb * (g.K / 64) + ks;
  const char* pp = (const char*)g.wp + blk * 4096 + (uint32_t)lane * 16u;
#pragma unroll
  for (int i = 0; i < 4; i++) r.p[i] = ldw16<NT>(pp + 1024 * i);
}
template <bool NT = false>
__device__ __forceinline__ void load_braw(const GemmArgs& g, int nb, int ks, int lane,
                                          BRaw<TGOHIP_FORM_I8>& r) {
  const int KS = g.K / 64;
  const size_t blk = (size_t)nb * KS + ks;
  const char* pp = (const char*)g.wp + blk * 2048 + (uint32_t)lane * 16u;
  r.p[0] = ldw16<NT>(pp);
  r.p[1] = ldw16<NT>(pp + 1024);
  const int h = lane >> 5;
#pragma unroll
  for (int j = 0; j < 4; j++) r.s[j] = *(const uint4*)(g.ws + ((((size_t)nb * KS + ks) * 4 + j) * 2 + h) * 8);
}
template <bool NT = false>
__device__ __forceinline__ void load_braw(const GemmArgs& g, int nb, int ks, int lane,
                                          BRaw<TGOHIP_FORM_I4_TGO>& r) {
  const int KS = g.K / 64;
  const size_t slot = ((size_t)nb * KS + ks) * 64 + lane;
  r.p = ldw16<NT>((const char*)g.wp + slot * 16);
  const int h = lane >> 5;
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const size_t o = ((((size_t)nb * KS + ks) * 4 + j) * 2 + h) * 8;
    r.s[j] = *(const uint4*)(g.ws + o);
    r.z[j] = *(const uint4*)(g.wz + o);
  }
}
template <bool NT = false>
__device__ __forceinline__ void load_braw(const GemmArgs& g, int nb, int ks, int lane,
                                          BRaw<TGOHIP_FORM_I4_SYM>& r) {
  // (nb, ks) is uniform across the wave: a scalar base plus a 32-bit lane
  // offset, so the loads need no 64-bit vector address arithmetic.
  const size_t blk = (size_t)nb * (g.K / 64) + ks;
  r.p = ldw16<NT>((const char*)g.wp + blk * 1024 + (uint32_t)lane * 16u);
  r.s = *(const uint32_t*)((const char*)g.ws + blk * 128 + (uint32_t)(lane & 31) * 4u);
}

__device__ __forceinline__ uint32_t word_of(const uint4& p, int j) {
  return j == 0 ? p.x : j == 1 ? p.y : j == 2 ? p.z : p.w;
}

union U16B { uint4 u; half8_t h; };

__device__ __forceinline__ half8_t bfrag(const BRaw<TGOHIP_FORM_F16>& r, int j) {
  U16B c;
  c.u = r.p[j];
  return c.h;
}
__device__ __forceinline__ half8_t bfrag(const BRaw<TGOHIP_FORM_I4_SYM>& r, int j) {
  union { uint32_t u; half2_t h; } sc;
  sc.u = r.s;
  return deq_i4_sym(word_of(r.p, j), j < 2 ? sc.h[0] : sc.h[1]);
}
__device__ __forceinline__ half8_t bfrag(const BRaw<TGOHIP_FORM_I4_TGO>& r, int j) {
  U16B s, z;
  s.u = r.s[j];
  z.u = r.z[j];
  return deq_i4_asym(word_of(r.p, j), s.h, z.h);
}
__device__ __forceinline__ half8_t bfrag(const BRaw<TGOHIP_FORM_I8>& r, int j) {
  const uint4 q = r.p[j >> 1];
  const uint32_t w0 = (j & 1) ? q.z : q.x, w1 = (j & 1) ? q.w : q.y;
  U16B s;
  s.u = r.s[j];
  return deq_i8(w0, w1, s.h);
}

// ---- exact dequantized weights as two f16 fragments ------------------------
// hi = RNE_f16((q - z) * s) and lo = (q - z) * s - hi, each f16, so hi + lo is
// the exact product tgo's CPU path multiplies (the f32 dequantization): (q - z)
// has at most 8 significant bits and s 11, so the residual after hi's 11 bits
// fits lo's (down to f16's subnormal spacing, 2^-24). lo comes from one fused
// multiply-add, q*s - hi, rounded once and exact. An MFMA with each half gives
// the product against the unrounded weight.
__device__ __forceinline__ void split_pair(half2_t d, half2_t s2, half2_t& hi, half2_t& lo) {
  hi = d * s2;
  lo = __builtin_elementwise_fma(d, s2, -hi);
}
__device__ __forceinline__ void pack_pair(half8_t& o, int j, half2_t h) {
  o[2 * j] = h[0];
  o[2 * j + 1] = h[1];
}
template <int FORM>
__device__ __forceinline__ void bfrag_split(const BRaw<FORM>& r, int j, half8_t& hi, half8_t& lo);
template <>
__device__ __forceinline__ void bfrag_split(const BRaw<TGOHIP_FORM_I4_SYM>& r, int j, half8_t& hi,
                                            half8_t& lo) {
  union { uint32_t u; half2_t h; } sc;
  sc.u = r.s;
  const half_t s = j < 2 ? sc.h[0] : sc.h[1];
  const half2_t sp = {s, s};
  const uint32_t w = word_of(r.p, j), w8 = w >> 8;
  const half2_t b0 = {(half_t)1032.f, (half_t)1032.f}, b1 = {(half_t)72.f, (half_t)72.f};
  // q - 8 exactly, as in deq_i4_sym (masks in registers: one v_and_or_b32 each)
  uint32_t m0 = 0x000F000Fu, m1 = 0x00F000F0u, g0 = 0x64006400u, g1 = 0x54005400u;
  asm("" : "+v"(m0), "+v"(m1), "+v"(g0), "+v"(g1));
  const half2_t d[4] = {as_h2((w & m0) | g0) - b0, as_h2((w & m1) | g1) - b1,
                        as_h2((w8 & m0) | g0) - b0, as_h2((w8 & m1) | g1) - b1};
#pragma unroll
  for (int i = 0; i < 4; i++) {
    half2_t h, l;
    split_pair(d[i], sp, h, l);
    pack_pair(hi, i, h);
    pack_pair(lo, i, l);
  }
}
template <>
__device__ __forceinline__ void bfrag_split(const BRaw<TGOHIP_FORM_I4_TGO>& r, int j, half8_t& hi,
                                            half8_t& lo) {
  U16B s, z;
  s.u = r.s[j];
  z.u = r.z[j];
  const uint32_t w = word_of(r.p, j);
  uint32_t m0 = 0x000F000Fu, g0 = 0x64006400u;
  asm("" : "+v"(m0), "+v"(g0));
#pragma unroll
  for (int i = 0; i < 4; i++) {
    // (1024 + q) - (1024 + z) = q - z exactly
    const half2_t d = as_h2(((w >> (4 * i)) & m0) | g0) - half2_t{z.h[2 * i], z.h[2 * i + 1]};
    half2_t h, l;
    split_pair(d, half2_t{s.h[2 * i], s.h[2 * i + 1]}, h, l);
    pack_pair(hi, i, h);
    pack_pair(lo, i, l);
  }
}
template <>
__device__ __forceinline__ void bfrag_split(const BRaw<TGOHIP_FORM_I8>& r, int j, half8_t& hi,
                                            half8_t& lo) {
  const uint4 q = r.p[j >> 1];
  const uint32_t ws[2] = {(j & 1) ? q.z : q.x, (j & 1) ? q.w : q.y};
  U16B s;
  s.u = r.s[j];
  const half2_t bias = {(half_t)1152.f, (half_t)1152.f};
  uint32_t m0 = 0x00FF00FFu, g0 = 0x64006400u;
  asm("" : "+v"(m0), "+v"(g0));
#pragma unroll
  for (int u = 0; u < 2; u++) {
    // (1024 + q + 128) - 1152 = q exactly
    const half2_t dl = as_h2((ws[u] & m0) | g0) - bias;
    const half2_t dh = as_h2(((ws[u] >> 8) & m0) | g0) - bias;
    half2_t h, l;
    split_pair(dl, half2_t{s.h[4 * u], s.h[4 * u + 1]}, h, l);
    pack_pair(hi, 2 * u, h);
    pack_pair(lo, 2 * u, l);
    split_pair(dh, half2_t{s.h[4 * u + 2], s.h[4 * u + 3]}, h, l);
    pack_pair(hi, 2 * u + 1, h);
    pack_pair(lo, 2 * u + 1, l);
  }
}
template <>
__device__ __forceinline__ void bfrag_split(const BRaw<TGOHIP_FORM_F16>& r, int j, half8_t& hi,
                                            half8_t& lo) {
  hi = bfrag(r, j);  // f16 weights are exact as stored
  lo = half8_t{0, 0, 0, 0, 0, 0, 0, 0};
}

// silu(g) = g / (1 + e^-g) (nn/blocks.go:62-66) with the hardware reciprocal
// (v_rcp_f32, 1 ulp) in place of the IEEE division's ten-instruction sequence:
// the SwiGLU epilogue of the C4 gate/up 209 -> 205 us.
__device__ __forceinline__ float silu_f(float g) { return g * __builtin_amdgcn_rcpf(1.f + __expf(-g)); }

// 16-byte slot of (row, k-chunk) in an LDS activation tile of 8 chunks per row.
// The XOR with (row/2) % 8 spreads any 16 consecutive rows of one k-chunk over
// all 64 banks (a bank row is 256 bytes = two tile rows), so the MFMA operand
// reads (16 lanes = 16 rows per LDS cycle) and the row-wise stores are
// conflict-free.
__device__ __forceinline__ int a_slot(int row, int kc) { return row * 8 + (kc ^ ((row >> 1) & 7)); }

// One SwiGLU output at element o of [M, N/2]: f16, f32, or the f16 hi plane
// and the lo plane (f16(v - hi)) M*N/2 elements after it (the activation pair
// the exact down projection reads).
template <int EPI>
__device__ __forceinline__ void store_swiglu(const GemmArgs& g, size_t o, float v) {
  if (EPI == EPI_SWIGLU_F32) {
    ((float*)g.y)[o] = v;
  } else {
    const half_t h = (half_t)v;
    ((half_t*)g.y)[o] = h;
    if (EPI == EPI_SWIGLU_X2) ((half_t*)g.y)[(size_t)g.M * (g.N / 2) + o] = (half_t)(v - (float)h);
  }
}

// Four consecutive SwiGLU outputs at element o (store_swiglu's values).
template <int EPI>
__device__ __forceinline__ void store_swiglu4(const GemmArgs& g, size_t o, float4_t gate, float4_t up) {
  float4_t v;
#pragma unroll
  for (int e = 0; e < 4; e++) v[e] = silu_f(gate[e]) * up[e];
  if (EPI == EPI_SWIGLU_F32) {
    *(float4_t*)((float*)g.y + o) = v;
    return;
  }
  half4_t hv, lv;
#pragma unroll
  for (int e = 0; e < 4; e++) {
    hv[e] = (half_t)v[e];
    lv[e] = (half_t)(v[e] - (float)hv[e]);
  }
  *(half4_t*)((half_t*)g.y + o) = hv;
  if (EPI == EPI_SWIGLU_X2) *(half4_t*)((half_t*)g.y + (size_t)g.M * (g.N / 2) + o) = lv;
}

// A workgroup barrier that orders LDS only: global loads in flight stay in
// flight across it (__syncthreads would wait for them).
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// gemm_rows.hip: cb column blocks per workgroup (2 pairs a SwiGLU's gate and up
// blocks), K in `splits` (the planes in g.part when more than one).
constexpr size_t kRowsPlaneBytes = (size_t)64 << 20;  // most bytes of its split-K planes
// Whether M f32 or pair rows over `ksteps` k-steps fit a CU's LDS beside the
// waves' sums.
bool rows_staged(int M, int ksteps);
int launch_gemm_rows(int form, const GemmArgs& g, int xk, int epi, int cb, int splits, hipStream_t st);

}  // namespace tgohip
