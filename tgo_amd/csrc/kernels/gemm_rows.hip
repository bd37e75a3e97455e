// gemm_rows.hip -- projections over few rows, or over a weight too small to
// fill the chip with the pipelined kernel's 64 x 256 tiles: latency and the
// weight stream are the cost, not the MFMAs.
//
// A workgroup of 8 or 16 waves owns 32 * CB columns and 32 * MB rows. The waves take
// the k-steps (64 deep) of its share of K in turn, each with its own weight
// fragments (registers, two k-steps ahead) and activations (one k-step ahead),
// and meet once, in LDS, where their
// sums are added in wave order: one barrier per launch instead of one per
// k-step, and 8 waves' loads in flight on each CU from the first cycle.
#include "gemm_weights.h"

#include <algorithm>
#include <type_traits>

namespace tgohip {

// k-steps of weight fragments a wave keeps in flight, by what the registers
// allow: 128 with 16 waves (staged) or four waves per SIMD, else 256.
template <int FORM, int CB, bool STG> constexpr int rows_depth() {
  if (FORM == TGOHIP_FORM_I4_TGO && CB == 2) return 1;
  if (STG && CB == 1 && (FORM == TGOHIP_FORM_F16 || FORM == TGOHIP_FORM_I4_SYM)) return 4;
  return 2;
}

// f(integral_constant<0>) ... f(integral_constant<N - 1>), in order.
template <int N, class F>
__device__ __forceinline__ void rows_for(F&& f) {
  if constexpr (N > 0) {
    rows_for<N - 1>(f);
    f(std::integral_constant<int, N - 1>{});
  }
}

constexpr int kRowsLdsMax = 160 << 10;  // a CU's LDS
constexpr int kRowsPersist = 256;       // staged workgroups in flight: one per CU
// The hi and lo planes of M rows over `ksteps` k-steps.
static int64_t rows_stage_bytes(int M, int ksteps) { return (int64_t)2 * M * ksteps * 64 * 2; }
// 16-byte chunk c of staged row r: XOR-swizzled within its k-step's eight, so
// that eight rows' reads of one chunk touch distinct banks.
__device__ __forceinline__ int rows_chunk(int r, int c) { return c ^ (r & 7); }

// XK: how the activation is stored. PACK (at most 16 rows, tgo's arithmetic):
// rows 0-15 of the A operand are the activations' f16 hi parts and rows 16-31
// their lo parts, so one MFMA multiplies both; D rows i and i + 16 sit in one
// lane and are added at the end.
// STG (PACK only): the workgroup's share of the activations goes to LDS once,
// split into hi and lo there, after the first weight loads are issued; the
// weight stream is then the only vector-memory traffic of the loop.
// TURN: a wave loads its rows of a k-step as whole 128-byte lines, eight lanes
// each, and turns them into MFMA operands in its own part of LDS. Operands
// loaded straight from L2 touch a quarter of 32 lines each, and the L1 misses
// bound the launch: [1024, 4096] of f16 weights at 67 pair rows 10.0 -> 6.8 us,
// [3072, 1024] 11.2 -> 8.5, [4096, 6144] at 20 rows 20.6 -> 14.4.
// Neither (PACK, or one k-step per wave): operands from L2.
// Two waves per SIMD where 128 registers are not enough: int8's f32 rows and
// pairs in TURN too (at four, 22 of them went to memory in every k-step: [4096,
// 6144] at 20 pair rows 15.8 us against 12.8). tgo's int4 staged over 16 waves,
// which have 128 registers and no more, spills 9.
template <int FORM, int XK, int MB, int CB, bool PACK, bool STG, int W, bool TURN>
__global__ __launch_bounds__(64 * W, W == 16 || (MB * CB == 1 && FORM != TGOHIP_FORM_I4_TGO && !(FORM == TGOHIP_FORM_I8 && XK != XK_F16 && TURN)) ? 4 : 2) void gemm_rows_kernel(
    GemmArgs g, int epi) {
  constexpr bool EX = XK != XK_F16;                          // tgo's arithmetic
  constexpr bool FX = EX && FORM == TGOHIP_FORM_I4_SYM;      // factored group scales
  constexpr bool BSPLIT = EX && !FX && FORM != TGOHIP_FORM_F16;
  constexpr int AP = EX && !PACK ? 2 : 1;                    // A operands per row block
  constexpr int D = rows_depth<FORM, CB, STG>();
  extern __shared__ __attribute__((aligned(16))) char smem[];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int h = lane >> 5, c32 = lane & 31;
  const int NBT = g.N / 32, KS = g.K / 64;
  const int m0 = blockIdx.y * 32 * MB;
  const int k0 = blockIdx.z * g.ksteps_per_split;
  const int nk = min(KS - k0, g.ksteps_per_split);
  const int n = (nk - wave + W - 1) / W;  // the wave's k-steps: k0 + wave + W i
  // The lane's activation rows; rows past M repeat the last (not stored).
  const bool lolane = PACK && c32 >= 16;
  size_t arow[MB];
#pragma unroll
  for (int mb = 0; mb < MB; mb++)
    arow[mb] = (size_t)min(m0 + (PACK ? (c32 & 15) : mb * 32 + c32), g.M - 1) * g.K + 8 * h;
  const half_t* const xh = (const half_t*)(lolane ? g.xlo : g.x);
  const half_t* const xl = (const half_t*)g.xlo;
  const float* const xf = (const float*)g.x;
  // STG: [hi, lo][rows][nk * 64] halves; the lane's row of its plane
  const int sk = nk * 64, sr = min(c32 & 15, g.M - 1);
  const half_t* const srow = (const half_t*)smem + (size_t)((lolane ? g.M : 0) + sr) * sk;

  // TURN: the wave's rows of a k-step, whole 128-byte lines of 8 lanes each, on
  // their way to its own part of LDS, where they are read as operands.
  half_t* const turn = (half_t*)smem + (size_t)wave * AP * MB * 2048;
  const int tc = lane & 7, tr = lane >> 3;
  uint4 tq[TURN ? 4 * MB : 1][XK == XK_F16 ? 1 : 2];
  auto load_turn = [&](int ks) {
    if constexpr (TURN) {
#pragma unroll
      for (int t = 0; t < 4 * MB; t++) {
        const size_t o = (size_t)min(m0 + 8 * t + tr, g.M - 1) * g.K + (size_t)ks * 64 + 8 * tc;
        if constexpr (XK == XK_F32) {
          tq[t][0] = *(const uint4*)(xf + o);
          tq[t][1] = *(const uint4*)(xf + o + 4);
        } else {
          tq[t][0] = *(const uint4*)(xh + o);
          if constexpr (AP == 2) tq[t][AP - 1] = *(const uint4*)(xl + o);
        }
      }
    }
  };
  // Only this wave reads what it writes here, in its other lanes, and the hardware
  // keeps a wave's LDS operations in order. The compiler sees each lane's own
  // addresses, which hardly ever meet: turn0 (zero, but unknown to it) is in the
  // reads' addresses, so that it cannot tell them from the writes' and keeps the
  // order too. (A wave barrier or an LDS fence on both sides of the writes orders
  // the global loads as well: int8 and symmetric int4 pairs then spill 13 to 55
  // VGPRs.)
  int turn0 = 0;
  if constexpr (TURN) asm volatile("" : "+v"(turn0));
  auto store_turn = [&] {
    if constexpr (TURN) {
#pragma unroll
      for (int t = 0; t < 4 * MB; t++) {
        half_t* const dst = turn + (8 * t + tr) * 64 + 8 * rows_chunk(tr, tc);
        if constexpr (XK == XK_F32) {
          union { uint4 u[2]; float f[8]; } r;
          r.u[0] = tq[t][0];
          r.u[1] = tq[t][1];
          half8_t hv, lv;
#pragma unroll
          for (int e = 0; e < 8; e++) {
            hv[e] = (half_t)r.f[e];
            lv[e] = (half_t)(r.f[e] - (float)hv[e]);
          }
          *(half8_t*)dst = hv;
          *(half8_t*)(dst + MB * 2048) = lv;
        } else {
          U16B u;
          u.u = tq[t][0];
          *(half8_t*)dst = u.h;
          u.u = tq[t][AP - 1];
          if constexpr (AP == 2) *(half8_t*)(dst + MB * 2048) = u.h;
        }
      }
    }
  };

  struct ARaw { uint4 v[XK == XK_F32 ? 2 : AP]; };  // f32: eight floats; else hi (and lo)
  ARaw aq[STG || TURN ? 1 : 4][MB];
  auto load_a = [&](int j, int ks) {
    if constexpr (!STG && !TURN) {
#pragma unroll
      for (int mb = 0; mb < MB; mb++) {
        const size_t o = arow[mb] + (size_t)ks * 64 + 16 * j;
        if constexpr (XK == XK_F32) {
          aq[j][mb].v[0] = *(const uint4*)(xf + o);
          aq[j][mb].v[1] = *(const uint4*)(xf + o + 4);
        } else {
          aq[j][mb].v[0] = *(const uint4*)(xh + o);
          if constexpr (AP == 2) aq[j][mb].v[AP - 1] = *(const uint4*)(xl + o);
        }
      }
    }
  };
  // The A operands of substep j of k-step ks: ah, and al (the lo parts) unless packed.
  auto operand = [&](int j, int ks, half8_t(&ah)[MB], half8_t(&al)[MB]) {
    if constexpr (STG) {
      ah[0] = *(const half8_t*)(srow + (ks - k0) * 64 + 8 * rows_chunk(sr, 2 * j + h));
    } else if constexpr (TURN) {
#pragma unroll
      for (int mb = 0; mb < MB; mb++) {
        const half_t* const src = turn + turn0 + (mb * 32 + c32) * 64 + 8 * rows_chunk(c32, 2 * j + h);
        ah[mb] = *(const half8_t*)src;
        if constexpr (AP == 2) al[mb] = *(const half8_t*)(src + MB * 2048);
      }
    } else {
#pragma unroll
      for (int mb = 0; mb < MB; mb++) {
        if constexpr (XK == XK_F32) {
          union { uint4 u[2]; float f[8]; } r;
          r.u[0] = aq[j][mb].v[0];
          r.u[1] = aq[j][mb].v[1];
#pragma unroll
          for (int e = 0; e < 8; e++) {
            const half_t hv = (half_t)r.f[e];
            ah[mb][e] = hv;
            al[mb][e] = (half_t)(r.f[e] - (float)hv);
          }
          if constexpr (PACK) {
            U16B a, b;
            a.h = ah[mb];
            b.h = al[mb];
            a.u.x = lolane ? b.u.x : a.u.x;
            a.u.y = lolane ? b.u.y : a.u.y;
            a.u.z = lolane ? b.u.z : a.u.z;
            a.u.w = lolane ? b.u.w : a.u.w;
            ah[mb] = a.h;
          }
        } else {
          U16B c;
          c.u = aq[j][mb].v[0];
          ah[mb] = c.h;
          c.u = aq[j][mb].v[AP - 1];
          al[mb] = c.h;
        }
      }
    }
  };

  float16_t acc[MB][CB];
  BRaw<FORM> bq[D][CB];
  int nb0 = blockIdx.x * CB;
  // One row block reads each weight once per launch (non-temporal loads);
  // several row blocks' workgroups share it through L2.
  auto load_b = [&](int d, int ks) {
#pragma unroll
    for (int b = 0; b < CB; b++) load_braw<MB == 1>(g, min(nb0 + b, NBT - 1), ks, lane, bq[d][b]);
  };
  const int ks0 = k0 + wave;
  auto first_b = [&] {
    rows_for<D>([&](auto dc) {
      constexpr int d = decltype(dc)::value;
      if (d < n) load_b(d, ks0 + W * d);
    });
  };
  if (TURN && n > 0) load_turn(ks0);
  first_b();
  if constexpr (STG) {
    // eight elements at a time, four loads of them in flight
    const int per = nk * 8, total = g.M * per;
    half_t* const xs = (half_t*)smem;
    for (int t = tid; t < total; t += 4 * 64 * W) {
      uint4 u[4][2];
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const int c = min(t + q * 64 * W, total - 1), row = c / per;
        const size_t o = (size_t)row * g.K + (size_t)k0 * 64 + (c - row * per) * 8;
        if constexpr (XK == XK_F32) {
          u[q][0] = *(const uint4*)(xf + o);
          u[q][1] = *(const uint4*)(xf + o + 4);
        } else {
          u[q][0] = *(const uint4*)((const half_t*)g.x + o);
          u[q][1] = *(const uint4*)(xl + o);
        }
      }
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const int c = t + q * 64 * W;
        if (c >= total) break;
        const int row = c / per;
        half_t* dst = xs + row * sk + 8 * rows_chunk(row, c - row * per);
        if constexpr (XK == XK_F32) {
          union { uint4 u[2]; float f[8]; } r;
          r.u[0] = u[q][0];
          r.u[1] = u[q][1];
          half8_t hv, lv;
#pragma unroll
          for (int e = 0; e < 8; e++) {
            hv[e] = (half_t)r.f[e];
            lv[e] = (half_t)(r.f[e] - (float)hv[e]);
          }
          *(half8_t*)dst = hv;
          *(half8_t*)(dst + (size_t)g.M * sk) = lv;
        } else {
          *(uint4*)dst = u[q][0];
          *(uint4*)(dst + (size_t)g.M * sk) = u[q][1];
        }
      }
    }
    lds_barrier();
  } else if (!TURN && n > 0) {
#pragma unroll
    for (int j = 0; j < 4; j++) load_a(j, ks0);
  }
  const float16_t zero16 = {};
  // k-step i of the wave, from slot d; its loads for later k-steps are
  // unconditional in the main loop (so a wait counts the loads in flight) and
  // under a uniform branch in the tail.
  auto step = [&](auto dc, auto mainc, int i) {
    constexpr int d = decltype(dc)::value;
    constexpr bool MAIN = decltype(mainc)::value;
    const int ks = ks0 + W * i;
    float16_t accg[FX ? MB : 1][CB];
    store_turn();
    if (MAIN || i + 1 < n) load_turn(ks + W);
#pragma unroll
    for (int j = 0; j < 4; j++) {
      half8_t ah[MB], al[MB];
      operand(j, ks, ah, al);
#pragma unroll
      for (int b = 0; b < CB; b++) {
        half8_t bh, bl;
        if constexpr (FX) bh = i4_sym_codes(word_of(bq[d][b].p, j));
        else if constexpr (BSPLIT) bfrag_split(bq[d][b], j, bh, bl);
        else bh = bfrag(bq[d][b], j);
#pragma unroll
        for (int mb = 0; mb < MB; mb++) {
          if constexpr (FX) {
            accg[mb][b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah[mb], bh, (j & 1) ? accg[mb][b] : zero16, 0, 0, 0);
            if constexpr (!PACK)
              accg[mb][b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(al[mb], bh, accg[mb][b], 0, 0, 0);
          } else {
            acc[mb][b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah[mb], bh, acc[mb][b], 0, 0, 0);
            if constexpr (EX && !PACK)
              acc[mb][b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(al[mb], bh, acc[mb][b], 0, 0, 0);
            if constexpr (BSPLIT)
              acc[mb][b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah[mb], bl, acc[mb][b], 0, 0, 0);
          }
        }
        if constexpr (FX) {
          if (j & 1) {
            union { uint32_t u; half2_t hh; } sc;
            sc.u = bq[d][b].s;
            const float s = (float)sc.hh[j >> 1];
#pragma unroll
            for (int mb = 0; mb < MB; mb++)
#pragma unroll
              for (int r = 0; r < 16; r++) acc[mb][b][r] = __builtin_fmaf(accg[mb][b][r], s, acc[mb][b][r]);
          }
        }
      }
      if (MAIN || i + 1 < n) load_a(j, ks + W);
    }
    if (MAIN || i + D < n) load_b(d, ks + W * D);
  };
  constexpr int R = PACK ? 8 : 16;  // result rows of a lane per 32 x 32 block
  // STG: the sums sit after the staged rows, and the workgroup goes on to
  // further column groups with the rows it staged.
  float* const red = (float*)(smem + (STG ? (size_t)2 * g.M * sk * sizeof(half_t) : 0));
  const int rows = min(32 * MB, g.M - m0);
  const int rstride = STG ? g.M * 32 : MB * 1024;  // floats of a wave's sums of one column block
  auto sum4 = [&](int at) {
    float4_t v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < W; w++) v += *(const float4_t*)&red[w * CB * rstride + at];
    return v;
  };
  const bool swiglu = CB == 2 && (epi == EPI_SWIGLU_F16 || epi == EPI_SWIGLU_X2) && gridDim.z == 1;
  for (;;) {
#pragma unroll
    for (int mb = 0; mb < MB; mb++)
#pragma unroll
      for (int b = 0; b < CB; b++) acc[mb][b] = float16_t{};
    int i = 0;
    for (; i + 2 * D <= n; i += D)
      rows_for<D>([&](auto dc) { step(dc, std::true_type{}, i + decltype(dc)::value); });
    for (; i < n; i += D)
      rows_for<D>([&](auto dc) {
        if (i + decltype(dc)::value < n) step(dc, std::false_type{}, i + decltype(dc)::value);
      });
    const int nbd = nb0;  // the group just summed; its successor's weights are already asked for
    nb0 += gridDim.x * CB;
    const bool last = !STG || nb0 >= NBT;
    if (!last) first_b();

    // The waves' sums, [rows][32] per column block: lane (c32, h) holds rows
    // 8 (r/4) + 4 h + r%4 of each 32 x 32 block.
    if constexpr (STG || TURN) lds_barrier();  // the sums before, or the rows, have been read
#pragma unroll
    for (int b = 0; b < CB; b++)
#pragma unroll
      for (int mb = 0; mb < MB; mb++)
#pragma unroll
        for (int r = 0; r < R; r++) {
          const int row = mb * 32 + 8 * (r >> 2) + 4 * h + (r & 3);
          const float v = PACK ? acc[mb][b][r] + acc[mb][b][r + 8] : acc[mb][b][r];
          if (!STG || row < g.M) red[(wave * CB + b) * rstride + row * 32 + c32] = v;
        }
    lds_barrier();
    for (int t = tid; t < rows * 8 * (swiglu ? 1 : CB); t += 64 * W) {
      const int b = t / (rows * 8), u = t - b * rows * 8, row = u >> 3, c4 = (u & 7) * 4;
      if (nbd + b >= NBT) continue;
      const int at = b * rstride + row * 32 + c4;
      float4_t v = sum4(at);
      if (swiglu) {
        const float4_t up = sum4(at + rstride);
        const size_t o = (size_t)(m0 + row) * (g.N / 2) + (nbd >> 1) * 32 + c4;
        half4_t hv, lv;
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const float s = silu_f(v[e]) * up[e];
          hv[e] = (half_t)s;
          lv[e] = (half_t)(s - (float)hv[e]);
        }
        *(half4_t*)((half_t*)g.y + o) = hv;
        if (epi == EPI_SWIGLU_X2) *(half4_t*)((half_t*)g.y + (size_t)g.M * (g.N / 2) + o) = lv;
        continue;
      }
      const size_t o = (size_t)(m0 + row) * g.N + (nbd + b) * 32 + c4;
      if (gridDim.z > 1) {
        *(float4_t*)(g.part + (size_t)blockIdx.z * g.pstride + o) = v;
      } else if (epi == EPI_F16) {
        *(half4_t*)((half_t*)g.y + o) = half4_t{(half_t)v[0], (half_t)v[1], (half_t)v[2], (half_t)v[3]};
      } else if (epi == EPI_RESID) {
        float4_t y = *(const float4_t*)((float*)g.y + o);
        y += v;
        *(float4_t*)((float*)g.y + o) = y;
      } else {
        *(float4_t*)((float*)g.y + o) = v;
      }
    }
    if (last) break;
  }
}

// Bytes of the staged kernel's sums: 16 waves, or 8 over two column blocks.
static int64_t rows_sum_bytes(int M) { return (int64_t)16 * M * 128; }
bool rows_staged(int M, int ksteps) {
  return M <= 16 && rows_stage_bytes(M, ksteps) + rows_sum_bytes(M) <= kRowsLdsMax;
}

template <int FORM, int XK, int MB, int CB, bool PACK, bool STG, int W, bool TURN = false>
static void launch_rows_one(const GemmArgs& g, int epi, int splits, hipStream_t st) {
  const int groups = (g.N / 32 + CB - 1) / CB;
  dim3 grid((unsigned)groups, (unsigned)((g.M + 32 * MB - 1) / (32 * MB)), (unsigned)splits);
  // the waves' sums, or the rows they turn
  size_t lds = (size_t)W * MB * std::max(CB, TURN && XK != XK_F16 ? 2 : 1) * 4096;
  if (STG) {
    lds = (size_t)(rows_stage_bytes(g.M, g.ksteps_per_split) + rows_sum_bytes(g.M));
    // one workgroup per CU (16 waves of up to 128 registers), each over every
    // 256th column group
    grid.x = (unsigned)std::min(groups, std::max(1, kRowsPersist / splits));
  }
  static const hipError_t attr = hipFuncSetAttribute((const void*)&gemm_rows_kernel<FORM, XK, MB, CB, PACK, STG, W, TURN>,
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, kRowsLdsMax);
  (void)attr;
  hipLaunchKernelGGL((gemm_rows_kernel<FORM, XK, MB, CB, PACK, STG, W, TURN>), grid, dim3(64 * W), lds, st, g, epi);
}

template <int FORM, int XK, int MB, int CB>
static void launch_rows_cb(const GemmArgs& g, int epi, int splits, hipStream_t st) {
  if constexpr (MB == 1 && XK != XK_F16) {
    if (rows_staged(g.M, g.ksteps_per_split))
      return launch_rows_one<FORM, XK, 1, CB, true, true, CB == 1 ? 16 : 8>(g, epi, splits, st);
    if (g.M <= 16) return launch_rows_one<FORM, XK, 1, CB, true, false, 8>(g, epi, splits, st);
  }
  // One k-step a wave over one row block: its operands straight from L2, without
  // the way through LDS ([2048, 1024] of f16 weights at 32 pair rows 7.2 us
  // against 8.2).
  if constexpr (MB == 1)
    if (g.ksteps_per_split <= 8) return launch_rows_one<FORM, XK, MB, CB, false, false, 8>(g, epi, splits, st);
  launch_rows_one<FORM, XK, MB, CB, false, false, 8, true>(g, epi, splits, st);
}

template <int FORM>
static int launch_rows_form(const GemmArgs& g, int xk, int epi, int cb, int splits, hipStream_t st) {
#define ROWS(XK)                                                                    \
  if (g.M <= 32 && cb == 1) launch_rows_cb<FORM, XK, 1, 1>(g, epi, splits, st);     \
  else if (g.M <= 32) launch_rows_cb<FORM, XK, 1, 2>(g, epi, splits, st);           \
  else if (cb == 1) launch_rows_cb<FORM, XK, 2, 1>(g, epi, splits, st);             \
  else if constexpr (FORM == TGOHIP_FORM_F16 && XK != XK_F32)                       \
    launch_rows_cb<FORM, XK, 2, 2>(g, epi, splits, st);                             \
  else return fail(TGOHIP_ESTATE, "linear: the row kernel takes no pair of column blocks here")
  if (xk == XK_F32) { ROWS(XK_F32); }
  else if (xk == XK_X2) { ROWS(XK_X2); }
  else { ROWS(XK_F16); }
#undef ROWS
  return 0;
}

int launch_gemm_rows(int form, const GemmArgs& g, int xk, int epi, int cb, int splits, hipStream_t st) {
  if (epi == EPI_SWIGLU_F32 || (cb == 1 && (epi == EPI_SWIGLU_F16 || epi == EPI_SWIGLU_X2)))
    return fail(TGOHIP_ESTATE, "linear: the row kernel has no such SwiGLU store");
  switch (form) {
    case TGOHIP_FORM_F16: return launch_rows_form<TGOHIP_FORM_F16>(g, xk, epi, cb, splits, st);
    case TGOHIP_FORM_I8: return launch_rows_form<TGOHIP_FORM_I8>(g, xk, epi, cb, splits, st);
    case TGOHIP_FORM_I4_TGO: return launch_rows_form<TGOHIP_FORM_I4_TGO>(g, xk, epi, cb, splits, st);
    default: return launch_rows_form<TGOHIP_FORM_I4_SYM>(g, xk, epi, cb, splits, st);
  }
}

}  // namespace tgohip
