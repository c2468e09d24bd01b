// The generation step's Dense layers for small batches (bf16, prenorm, half_glu1 blocks),
// each with the elementwise work around it: per block
//   in_proj   proj = LayerNorm(x) W_in                   (layers.py:108-160, mamba3.py:210)
//   out_proj  g = gelu(RMSNorm(y) W_out)                 (mamba3.py:281-331; K <= 1024)
//   gate      x' = x + g sigmoid(g W_2 + b_2)            (half_glu1; with the gelu before
//                                                        it where the out_proj is apart)
// in place of three library GEMMs, m3_layer_post, m3_block_gelu and m3_block_act_norm.
// Values are rounded to bf16 where the separate kernels round them.
//
// What bounds it: at one token for 64 sequences a block's weights (9 MB at d_model 768) and
// activations take 2 us from memory, but each of the seven launches around the decode
// kernel takes 5 to 11 us, all latency.  So the work is cut for latency: a workgroup of 8
// waves computes 16 MT rows by 16 NT columns; its waves share the loads along the
// contraction, each requesting every operand of its slice (16 bytes per lane) before it uses
// any, and put them into LDS in MFMA operand order; then one wave per 16 x 16 tile runs the
// whole contraction, k ascending in one accumulator.  (Splitting the contraction over the
// waves and adding their accumulators makes a step of 64 rows 7% faster, but rounds
// differently from the library's products, which the other batch sizes run on.)  The norms' statistics are formed by
// every column block again, one wave per row in the order of m3_block_norm and
// m3_layer_post, from rows that it reads anyway: that costs a few hundred cycles and saves a
// launch.  The mixer's kernels are read where they lie, (in, out) with the output contiguous,
// so no second copy of them is kept: a wave's 32 x 16 tiles are read transposed from LDS
// (ds_read_b64_tr_b16).  A tile's rows are a quarter of a cache line, so neighbouring column
// blocks run on one XCD, whose L2 then serves the rest of the line.  The gate's kernel is
// (out, in), already in operand order.
//
// A captured step (us, library products and single kernels / this): d_model 768, 12 blocks,
// 64 rows 762 / 630; 512, 8 blocks, 64 rows 442 / 301; 256, 8 blocks, 64 rows 347 / 187.
#include "m3_chunk_common.h"

namespace m3 {
namespace {

constexpr int kStepWaves = 8;
enum StepMode { kStepIn, kStepOut, kStepGate, kStepGeluGate };

__device__ __forceinline__ float step_gelu(float x) {    // x sigmoid(2u), as m3_block.hip's
  const float u2 = 1.5957691216057308f * fmaf(0.044715f * x * x, x, x);
  return x * __builtin_amdgcn_rcpf(1.0f + __expf(-u2));
}
__device__ __forceinline__ float step_sigmoid(float x) { return __builtin_amdgcn_rcpf(1.0f + __expf(-x)); }
__device__ __forceinline__ float rbf(float x) { return (float)(bf16)x; }

// LDS bytes of a workgroup: the operands, in 1 KB fragments of 32 x 16.
constexpr int step_lds(int ks, int mt, int nt) { return 1024 * ks * kStepWaves * (mt + nt) + 2 * 16 * mt * 4; }

// Grid (ceil(N / (16 NT)) rounded up to a multiple of 8, ceil(M / (16 MT))).  KS: 32-wide
// k-steps of a wave's share of the loads, K = 256 KS.
template <int MODE, int KS, int MT, int NT>
__global__ __launch_bounds__(64 * kStepWaves)
void step_gemm_kernel(StepGemmArgs a) {
  constexpr int K = 32 * KS * kStepWaves, TM = 16 * MT, TN = 16 * NT;
  static_assert(MT * NT <= kStepWaves && step_lds(KS, MT, NT) <= 160 * 1024, "tile");
  __shared__ float st_s[2][TM];                          // the rows' mean (LayerNorm) and scale
  __shared__ bf16x8 w_s[KS * kStepWaves][NT][64], x_s[KS * kStepWaves][MT][64];   // by k-step
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, g = lane >> 4;
  const int xb = gridDim.x % 8 == 0 ? (blockIdx.x % 8) * (gridDim.x / 8) + blockIdx.x / 8 : blockIdx.x;
  const int nb = (a.N + TN - 1) / TN;
  if (xb >= nb) return;                                  // the grid is rounded up to whole XCD turns
  const int m0 = blockIdx.y * TM, n0 = xb * TN;
  const int k0 = wave * 32 * KS + 8 * g;                 // this lane's first column of its share

  // every operand of the share is requested first: rows and columns past the end read the
  // last ones' and are not stored.  Weights (K, N): lane -> row lane/2 and 8 of the 16
  // columns of a tile (N is a multiple of 8); (N, K): operand order.
  constexpr bool GATE = MODE == kStepGate || MODE == kStepGeluGate, TR = !GATE;
  bf16x8 w[KS][NT];
  const bf16* wt = reinterpret_cast<const bf16*>(a.wt);
#pragma unroll
  for (int s = 0; s < KS; ++s)
#pragma unroll
    for (int j = 0; j < NT; ++j)
      w[s][j] = *reinterpret_cast<const bf16x8*>(
          TR ? wt + (long)(wave * 32 * KS + 32 * s + (lane >> 1)) * a.N + min(n0 + 16 * j + 8 * (lane & 1), a.N - 8)
             : wt + (long)min(n0 + 16 * j + l16, a.N - 1) * K + k0 + 32 * s);
  long row[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) row[t] = (long)min(m0 + 16 * t + l16, a.M - 1) * K + k0;

  // the rows' statistics, one wave per row, two rows per wave and row tile
  if constexpr (MODE == kStepIn) {
    const float* xr = reinterpret_cast<const float*>(a.x);
    const float inv_d = 1.0f / (float)a.K;
#pragma unroll
    for (int i = 0; i < 2 * MT; ++i) {
      const int r = wave + kStepWaves * i;
      const float4* x4 = reinterpret_cast<const float4*>(xr + (long)min(m0 + r, a.M - 1) * K);
      float4 v[KS];
      float s = 0.0f;
#pragma unroll
      for (int k = 0; k < KS; ++k) {
        v[k] = x4[lane + 64 * k];
        s += (v[k].x + v[k].y) + (v[k].z + v[k].w);
      }
      float mean = group_sum<64>(s) * inv_d;
      asm("" : "+v"(mean));     // rounded, as m3_block_norm holds it: not part of the subtraction's FMA
      float ss = 0.0f;
#pragma unroll
      for (int k = 0; k < KS; ++k) {
        const float dx = v[k].x - mean, dy = v[k].y - mean, dz = v[k].z - mean, dw = v[k].w - mean;
        ss += (dx * dx + dy * dy) + (dz * dz + dw * dw);
      }
      const float rs = rsqrtf(group_sum<64>(ss) * inv_d + a.eps);
      if (lane == 0) {
        st_s[0][r] = mean;
        st_s[1][r] = rs;
      }
    }
  } else if constexpr (MODE == kStepOut) {
    const bf16* xr = reinterpret_cast<const bf16*>(a.x);
#pragma unroll
    for (int i = 0; i < 2 * MT; ++i) {
      const int r = wave + kStepWaves * i;
      const bf16* x1 = xr + (long)min(m0 + r, a.M - 1) * K;
      float ss = 0.0f;
#pragma unroll
      for (int k = 0; k < KS / 2; ++k) {
        float f[8];
        Vec8<bf16> v;
        v.load(x1 + 8 * (lane + 64 * k));
        v.to_f(f);
#pragma unroll
        for (int e = 0; e < 8; ++e) ss += f[e] * f[e];
      }
      ss = group_sum<64>(ss);
      if (lane == 0) st_s[1][r] = rbf(rsqrtf(ss / a.K + a.eps));
    }
  }
  if constexpr (!GATE) __syncthreads();

  // the activations in operand order, normalised
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    const int ks = wave * KS + s;
    float sc[8], bi[8];
    if constexpr (!GATE) {
      Vec8<float> v;
      v.load(a.scale + k0 + 32 * s);
      v.to_f(sc);
    }
    if constexpr (MODE == kStepIn) {
      Vec8<float> v;
      v.load(a.bias + k0 + 32 * s);
      v.to_f(bi);
    }
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      bf16x8 x;
      if constexpr (MODE == kStepIn) {
        float f[8];
        Vec8<float> v;
        v.load(reinterpret_cast<const float*>(a.x) + row[t] + 32 * s);
        v.to_f(f);
        const float mean = st_s[0][16 * t + l16], rs = st_s[1][16 * t + l16];
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = (bf16)fmaf((f[e] - mean) * rs, sc[e], bi[e]);
      } else {
        x = *reinterpret_cast<const bf16x8*>(reinterpret_cast<const bf16*>(a.x) + row[t] + 32 * s);
        if constexpr (MODE == kStepOut) {
          // rounded as m3_layer_post rounds it: the rsqrt, the product, the scaled product
          const float ri = st_s[1][16 * t + l16];
#pragma unroll
          for (int e = 0; e < 8; ++e) x[e] = (bf16)(rbf((float)x[e] * ri) * sc[e]);
        } else if constexpr (MODE == kStepGeluGate) {
#pragma unroll
          for (int e = 0; e < 8; ++e) x[e] = (bf16)step_gelu((float)x[e]);
        }
      }
      x_s[ks][t][lane] = x;
    }
#pragma unroll
    for (int j = 0; j < NT; ++j) w_s[ks][j][lane] = w[s][j];
  }
  __syncthreads();

  // one tile per wave: rows = columns of the product (4 consecutive ones per lane), columns
  // = its rows
  if (wave >= MT * NT) return;
  const int t = wave / NT, j = wave % NT;
  f32x4 o = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 8
  for (int ks = 0; ks < KS * kStepWaves; ++ks) {
    const bf16x8 wf = TR ? ld_tr(reinterpret_cast<const bf16*>(&w_s[ks][j][0]), 16, 0, 0, lane) : w_s[ks][j][lane];
    o = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf, x_s[ks][t][lane], o, 0, 0, 0);
  }
  const int m = m0 + 16 * t + l16, n = n0 + 16 * j + 4 * g;
  if (m >= a.M || n >= a.N) return;
  const long at = (long)m * a.N + n;
  if constexpr (GATE) {
    // x + g sigmoid(h2), with the gate's factor g the rows of the product themselves
    const bf16x4 b2 = *reinterpret_cast<const bf16x4*>(reinterpret_cast<const bf16*>(a.b2) + n);
    bf16x4 gv = *reinterpret_cast<const bf16x4*>(reinterpret_cast<const bf16*>(a.x) + at);
    if constexpr (MODE == kStepGeluGate) {
#pragma unroll
      for (int e = 0; e < 4; ++e) gv[e] = (bf16)step_gelu((float)gv[e]);
    }
    const f32x4 sk = *reinterpret_cast<const f32x4*>(a.skip + at);
    f32x4 y;
#pragma unroll
    for (int e = 0; e < 4; ++e) y[e] = sk[e] + rbf((float)gv[e] * rbf(step_sigmoid(rbf(o[e] + (float)b2[e]))));
    *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(a.out) + at) = y;
  } else {
    bf16x4 y;
#pragma unroll
    for (int e = 0; e < 4; ++e) y[e] = (bf16)(MODE == kStepOut ? step_gelu(rbf(o[e])) : o[e]);
    *reinterpret_cast<bf16x4*>(reinterpret_cast<bf16*>(a.out) + at) = y;
  }
}

template <int MODE, int KS, int MT, int NT>
hipError_t launch(const StepGemmArgs& a, hipStream_t st) {
  const int nb = (a.N + 16 * NT - 1) / (16 * NT);
  hipLaunchKernelGGL((step_gemm_kernel<MODE, KS, MT, NT>), dim3((nb + 7) / 8 * 8, (a.M + 16 * MT - 1) / (16 * MT)),
                     dim3(64 * kStepWaves), 0, st, a);
  return hipGetLastError();
}

// The tile (row tiles x column tiles of 16): the smallest of 1x1, 1x2, 2x2 and 4x2 whose
// blocks fit one round of the compute units, since a second round costs as much as the
// first and a larger tile only a little more; where none fits, 2x2.  Measured at d_model
// 768 with the contraction split over the waves (us, 1x1 / 1x2 / 2x2 / 4x2; * chosen): in_proj 16 rows 5.0* / 5.4, 32 rows 7.3 / 5.6* /
// 7.5, 64 rows 12.4 / 8.7 / 7.7* / 11.2, 128 rows 20.6 / 17.0 / 12.1 / 11.5*, 256 rows 40 /
// 28 / 22.2* / 21.5; out_proj 64 rows 5.3* / 6.6 / 9.4, 128 rows 8.8 / 6.7* / 9.4, 256 rows
// 12.5 / 11.3 / 9.4*.  4x2 is for contractions whose operands fit LDS.
template <int MODE, int KS>
hipError_t launch_rows(const StepGemmArgs& a, hipStream_t st) {
  auto fits = [&](int mt, int nt) {
    return (long)((a.M + 16 * mt - 1) / (16 * mt)) * ((a.N + 16 * nt - 1) / (16 * nt)) <= 256;
  };
  if (fits(1, 1)) return launch<MODE, KS, 1, 1>(a, st);
  if (fits(1, 2)) return launch<MODE, KS, 1, 2>(a, st);
  if constexpr (step_lds(KS, 4, 2) <= 160 * 1024) {
    if (!fits(2, 2) && fits(4, 2)) return launch<MODE, KS, 4, 2>(a, st);
  }
  return launch<MODE, KS, 2, 2>(a, st);
}

}  // namespace

bool step_gemm_supported(int mode, int K, int N) {
  return K % 256 == 0 && K >= 256 && K <= 1024 && N >= 8 && N % 8 == 0 &&
         (mode != kStepOut || K % 512 == 0);
}

hipError_t step_gemm_launch(int mode, const StepGemmArgs& a, hipStream_t st) {
  const int ks = a.K / 256;
  if (mode == kStepIn) {
    if (ks == 1) return launch_rows<kStepIn, 1>(a, st);
    if (ks == 2) return launch_rows<kStepIn, 2>(a, st);
    if (ks == 3) return launch_rows<kStepIn, 3>(a, st);
    if (ks == 4) return launch_rows<kStepIn, 4>(a, st);
  } else if (mode == kStepOut) {
    if (ks == 2) return launch_rows<kStepOut, 2>(a, st);
    if (ks == 4) return launch_rows<kStepOut, 4>(a, st);
  } else if (mode == kStepGeluGate) {
    if (ks == 1) return launch_rows<kStepGeluGate, 1>(a, st);
    if (ks == 2) return launch_rows<kStepGeluGate, 2>(a, st);
    if (ks == 3) return launch_rows<kStepGeluGate, 3>(a, st);
    if (ks == 4) return launch_rows<kStepGeluGate, 4>(a, st);
  } else {
    if (ks == 1) return launch_rows<kStepGate, 1>(a, st);
    if (ks == 2) return launch_rows<kStepGate, 2>(a, st);
    if (ks == 3) return launch_rows<kStepGate, 3>(a, st);
    if (ks == 4) return launch_rows<kStepGate, 4>(a, st);
  }
  return hipErrorInvalidValue;
}

}  // namespace m3
