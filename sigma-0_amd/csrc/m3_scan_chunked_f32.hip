// Chunked Mamba3 SISO prefill scan with float32 I/O on CDNA4 matrix cores.
//
// The same operator as m3_scan_chunked.hip (the reference's mamba3_ssd_chunked_jax,
// phases 1-7, src/base_model/models/mamba3_jax.py:327-419), for the float32
// inputs the model hands its scan (mamba3.py:363-367 casts x, z, B and C to float32
// before mamba3_siso_triton), with float32 accuracy and 32-token chunks.
//
// The contractions over d_state and over the keys run on bf16 matrix cores with every
// float32 operand as the exact sum of three bf16 parts and six part products
// (m3_chunk_common.h): 3/8 of the float32 MFMA's time, and against float64 the same
// error (8e-8 in the 2-norm, measured at d_state 64 and 128).  The intra-chunk M V keeps
// v_mfma_f32_16x16x4_f32: its operands are in registers and used once, so splitting them
// would cost more than it saves.  At B=8, L=4096, H=32, d_state 128 (same box): 664 us
// with float32 MFMA throughout, 517 us with the parts, 500 us with the roles below; the
// loads and stores alone take 371 us.  With every compute unit busy the kernel runs into
// the board's power limit (1390 W; the shader clock settles at 2.05 of 2.4 GHz), so what
// it executes costs clock as well as cycles; with fewer blocks the gain is larger (32
// pairs of 1024 tokens at d_state 64: 121 -> 70 us).
//
// One workgroup of 12 waves per (batch, head) walks the chunks in order, in three roles
// that work on different chunks at the same time, so that vector, matrix and memory work
// overlap on every SIMD:
//   preparation waves 8-11: chunk c+1's Q and K rows, read whole into registers one chunk
//     ahead (lane -> 4 columns), biases, rope from a cos/sin table and key scale, split
//     into the planes that the matrix work of the next chunk reads; chunk c+2's angles
//     into the table (lane = token, for the prefix over tokens)
//   state waves 4-7: each owns 16 columns of the value dimension (a p-tile): h^T[:, p-tile]
//     (all N rows) as 16x16 accumulators, that p-tile's Y_off = Q_r h^T and its update
//   output waves 0-3: the three (query block, key block) items of Y_diag (an S^T block,
//     the causal mask or the decay, M V over its keys), then the gate and the store
// A chunk is two phases with a barrier after each (Y_off and the items, then the update
// and the gate that reads their Y).  Every input byte is read from HBM once and the
// output written once.
#include <type_traits>

#include "m3_chunk_block.h"

namespace m3 {
namespace chunked_f32 {

// Two inclusive scans over each 32-lane half of the wavefront on its own: the steps of
// wave_incl_scan without the carry from the lower half into the upper one.
__device__ __forceinline__ void half_incl_scan2(float v[2]) {
#pragma unroll
  for (int j = 0; j < 2; ++j) v[j] += dpp0<kDppRowShr1>(v[j]);
#pragma unroll
  for (int j = 0; j < 2; ++j) v[j] += dpp0<kDppRowShr2>(v[j]);
#pragma unroll
  for (int j = 0; j < 2; ++j) v[j] += dpp0<kDppRowShr4>(v[j]);
#pragma unroll
  for (int j = 0; j < 2; ++j) v[j] += dpp0<kDppRowShr8>(v[j]);
#pragma unroll
  for (int j = 0; j < 2; ++j) v[j] += dpp0<kDppRowBcast15, 0xa>(v[j]);
}

// Compile-time geometry of one instantiation.
template <typename T, int CS_, int N_, int P_, int R_, int NW_, bool SO>
struct Geo : GeoBase<T, CS_, N_, P_, R_, NW_> {
  typedef GeoBase<T, CS_, N_, P_, R_, NW_> B;
  static constexpr int NQK = 0;                             // Q and K are not staged raw
  static constexpr int LDY = B::P;                          // Y tile rows (swizzled, yoff)
  // Element (row, col) of a Y tile: the 16-column blocks are exchanged by row / 4, so
  // that an accumulator tile's stores (rows 4 g + r of lane groups g) miss each other's banks.
  __device__ static int yoff(int row, int col) { return row * LDY + (col ^ (16 * ((row >> 2) & (B::PT - 1)))); }
  // The cos/sin table: a token's R pairs as R / 2 16-byte slots (two pairs each),
  // exchanged within the row so that the angle waves' writes (one slot per lane, lanes on
  // consecutive tokens) touch every bank.
  static constexpr int TSL = B::R / 2;
  __device__ static int toff(int t, int slot) {
    return t * TSL + (slot ^ ((t >> (TSL >= 16 ? 0 : TSL == 8 ? 1 : 2)) & (TSL - 1)));
  }
  // LDS bytes besides the table and the rotation rates.  Those are double-buffered where
  // they fit (all but the full pass at rotation width N/2 and d_state 128): with one
  // table the preparation and the next angles cannot share a phase, with one buffer the
  // rates' loads have one phase instead of a chunk to land.
  static constexpr int FIXED = (SO ? 2 : 4) * 3 * B::CS * B::N * 2 + (SO ? 0 : (2 * B::CS + 16) * LDY * 4) +
                               2 * B::CS * B::SV * 16 + 3 * 6 * B::CS * 4 + 128;
  static constexpr int TAB = B::CS * TSL * 16, RATES = B::CS * B::SA * 16 + 3 * (B::CS + 4) * 4;
  static constexpr int NTAB = FIXED + 2 * (TAB + RATES) <= 160 * 1024 ? 2 : 1;
  static constexpr int NRA = FIXED + NTAB * TAB + 2 * RATES <= 160 * 1024 ? 2 : 1;
  static_assert(B::SPT >= 1 && B::NST % B::PT == 0 && B::LB16 % B::SPT == 0, "state-wave split");
  static_assert(!B::BF && B::CS == 32 && (B::N == 32 || B::N == 64 || B::N == 128), "float32, 32-token chunks");
  static_assert(B::R >= 8 && (TSL & (TSL - 1)) == 0, "rotation widths");
};

template <typename G, bool SO>
struct __attribute__((aligned(16))) Smem {
  typedef float T;
  PlaneTile<G::CS, G::N> k[2];           // rope'd, trapezoid-scaled K rows, in bf16 parts, by chunk parity
  // rope'd Q rows, likewise (not in the state-only pass, as the Y tiles)
  typename std::conditional<SO, char, PlaneTile<G::CS, G::N>>::type q[2];
  // Y before the gate, written by plain stores: the intra-chunk part (output waves, by
  // query block) and Q h^T (state waves, by p-tile; the gate applies its e^{A_cum} row scale)
  alignas(16) T yd[SO ? 4 : G::CS * G::LDY];
  alignas(16) T yo[SO ? 4 : G::CS * G::LDY];
  alignas(16) T ydo[SO ? 4 : 16 * G::LDY];       // the off-diagonal item's part of rows 16..31
  alignas(16) uint4 rv[2][G::CS * G::SV];            // V, by chunk parity
  alignas(16) uint4 ra[G::NRA][G::CS * G::SA];       // rotation rates
  alignas(16) float rs[G::NRA][3][G::CS + 4];        // adt, dt, trap ([CS]: the next chunk's first token)
  alignas(16) float4 tab[G::NTAB][G::CS * G::TSL];   // cos, sin of a token's pairs (Geo::toff)
  float4 one;                                        // 1, 0, 1, 0: the table of columns past the rope
  // per-token chunk constants, of chunk c at c % 3: computed two chunks ahead, while the
  // matrix work of one chunk and the preparation of the next read theirs
  alignas(16) float ac2[3][G::CS];       // A_cum * log2(e)
  alignas(16) float g16[3][G::CS];       // e^{A_e - A_cum}, A_e = A_cum at the end of the token's 16-block
  alignas(16) float expa[3][G::CS];      // e^{A_cum}
  alignas(16) float dg[3][G::CS];        // gamma / scale: turns the S diagonal into the QK skip weight
  alignas(16) float scl[3][G::CS];       // trapezoid key scale gamma_t + dt_{t+1} (1 - sigmoid_{t+1})
  alignas(16) float wdec[3][G::CS];      // e^{A_end - A_cum}
  float dec[4];                          // e^{A_end}
};

// SO (state only): the pass that produces each segment's exit carry from a zero
// entering carry; it skips Q, Y_diag, Y_off, the gate and the output.
// SAVE (full pass): also write each chunk's entering state and angles (chunk_h,
// chunk_th), the residuals the backward reads instead of running the state-only pass,
// and with Z the output before the gate (out_v).
template <typename T, int CS, int N, int P, int R, int NW, bool SO, bool SAVE = false>
__global__ __launch_bounds__(64 * NW, 1)
void scan_chunked_f32_kernel(ScanArgs a) {
  typedef Geo<T, CS, N, P, R, NW, SO> G;
  typedef MF16<T> W;
  static_assert(sizeof(Smem<G, SO>) <= 160 * 1024, "LDS budget");
  __shared__ Smem<G, SO> sm;
  if constexpr (SO) {
    if (a.so_skip_last && blockIdx.y + 1 == gridDim.y) return;   // before any barrier: the whole block
  }

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  __builtin_assume(wave >= 0 && wave < NW);
  const ChunkBlock<T> cb = chunk_block<T, CS, N, P, R>(a);
  const int L = cb.L, Lnx = cb.Lnx, nc = cb.nc;
  const long ch0 = cb.ch0;
  const int ci_in = cb.ci_in, ci_out = cb.ci_out;
  const bool has_init = cb.has_init, fin_here = cb.fin_here, has_z = cb.has_z;
  const float Dh = cb.Dh;
  const int v_stride = cb.v_stride, vz_stride = cb.vz_stride;
  const T* z_base = cb.z_base;
  T* o_base = cb.o_base;
  T* gO = cb.gO;

  // ---- roles: output waves 0-3, state waves 4-7 (state wave sw owns p-tile pr, i.e.
  // h^T[:, 16 pr + lane%16] for all N rows as 16x16 accumulators, and the query blocks
  // lb = part (mod SPT) of Y_off), preparation waves 8-11 (state-only pass: 0-3 too)
  const bool ywave = wave < G::NWY;
  const bool swave = wave >= G::NWY && wave < G::NWY + G::NST;
  const int sw = wave - G::NWY;
  const int pr = swave ? sw % G::PT : 0, part = swave ? sw / G::PT : 0;

  // ---- direct-to-LDS loads, issued by two state waves, which have no other loads to
  // wait for: V of chunk c into rv[c % 2], rotation rates and scalars into ra / rs[c % NRA]
  constexpr int kWA = G::NWY + 2, kWV = G::NWY + 3;
  auto stage_v = [&](int c) { stage_v_chunk<G, kWV>(sm, cb, c, wave, lane); };
  auto stage_ars = [&](int c) { stage_ars_chunk<G, kWA>(sm, cb, c, wave, lane); };

  // ---- preparation waves.  Wave pw takes TPW tokens of a chunk.  Their Q and K rows are
  // read whole into registers (lane -> 4 columns of one row, RPI rows per instruction)
  // one chunk ahead: a register is loaded for the next chunk as soon as it is used.
  constexpr int NPW = SO ? G::NWY + G::NAUX : G::NAUX;
  constexpr int TPW = CS / NPW, LPR = N / 4, RPI = 64 / LPR, NI = TPW / RPI;
  static_assert(NI >= 1 && TPW % RPI == 0, "whole instructions");
  const int pw = ywave ? wave : wave - G::NWY - G::NAUX + (SO ? G::NWY : 0);
  const int cq = lane % LPR, ptok = TPW * pw + lane / LPR;
  f32x4 qraw[NI], kraw[NI];
  f32x4 qb4, kb4;
  const uint32_t rowb = (uint32_t)cb.qk_stride * 4;
  auto load_raw = [&](int c, int i) {
    // rows past the segment end read its last row: their key scale is 0, so they add
    // nothing to S or h, and their outputs are never stored
    const uint32_t off = (uint32_t)min(ptok + RPI * i, L - 1 - c * CS) * rowb + 16u * cq;
    const long row0 = (long)(c * CS) * cb.qk_stride;
    if constexpr (!SO)
      qraw[i] = __builtin_nontemporal_load(
          reinterpret_cast<const f32x4*>(reinterpret_cast<const char*>(cb.q_base + row0) + off));
    kraw[i] = __builtin_nontemporal_load(
        reinterpret_cast<const f32x4*>(reinterpret_cast<const char*>(cb.k_base + row0) + off));
  };
  // cos, sin of the rope pairs 2 cq and 2 cq + 1 of token t (columns past the rope: 1, 0)
  auto table = [&](int c, int t) { return *(cq < G::TSL ? &sm.tab[c % G::NTAB][G::toff(t, cq)] : &sm.one); };
  auto turn = [&](float x[4], const float4& cs) {
    const float co[2] = {cs.x, cs.z}, si[2] = {cs.y, cs.w};
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const float x0 = x[2 * j], x1 = x[2 * j + 1];
      x[2 * j] = x0 * co[j] - x1 * si[j];
      x[2 * j + 1] = x0 * si[j] + x1 * co[j];
    }
  };
  // biases, rope and key scale of chunk c's rows, into the planes; loads of chunk c + 1's
  // (of the last chunk's own again at the end, for the final carry's key)
  auto prep = [&](int c, auto i0_c, auto i1_c) {
    constexpr int I0 = decltype(i0_c)::value, I1 = decltype(i1_c)::value;
    const int c3 = c % 3;
    float scl[NI];
    float4 cs[NI];
#pragma unroll
    for (int i = I0; i < I1; ++i) {
      scl[i] = sm.scl[c3][ptok + RPI * i];
      cs[i] = table(c, ptok + RPI * i);
    }
    float qf[NI][4], kf[NI][4];
#pragma unroll
    for (int i = I0; i < I1; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if constexpr (!SO) qf[i][e] = qraw[i][e] + qb4[e];
        kf[i][e] = kraw[i][e] + kb4[e];
      }
    // the rows' registers are free: the next loads go into the same ones (issued among
    // the uses they would need others, and a copy at the loop's end that waits for them)
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = I0; i < I1; ++i) load_raw(min(c + 1, nc - 1), i);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = I0; i < I1; ++i) {
      const int t = ptok + RPI * i;
      if constexpr (!SO) turn(qf[i], cs[i]);
      turn(kf[i], cs[i]);
#pragma unroll
      for (int e = 0; e < 4; ++e) kf[i][e] *= scl[i];
      if constexpr (!SO) sm.q[c & 1].put4(t, cq, qf[i]);
      sm.k[c & 1].put4(t, cq, kf[i]);
    }
  };
  // in two parts: the second in phase 2, with the angles, or with a single table right
  // after the first
  constexpr bool kPrep2 = G::NTAB > 1 && !SO;
  const std::integral_constant<int, 0> kI0{};
  const std::integral_constant<int, (NI + 1) / 2> kI1{};
  const std::integral_constant<int, NI> kI2{};
  auto prep_rest = [&](int c) {
    if constexpr (NI > 1) {
      __builtin_amdgcn_sched_barrier(0);         // the parts' registers are not live together
      prep(c, kI1, kI2);
    }
  };

  // ---- rotations of chunk c into the table.  Wave pw takes the groups pw + NPW k of four
  // rope pairs; two lanes per token (tkn, hf), each with pairs 4 g + 2 hf + {0, 1}.
  constexpr int NG = R / 4, GPW = (NG + NPW - 1) / NPW;
  const int tkn = lane & (CS - 1), hf = lane / CS;
  float carry[GPW][2];                         // the pairs' angles, revolutions
#pragma unroll
  for (int k = 0; k < GPW; ++k)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int r = 4 * (pw + NPW * k) + 2 * hf + j;
      carry[k][j] = (a.init_theta && has_init && r < R && pw >= 0) ? a.init_theta[(long)ci_in * R + r] * kInvTwoPi : 0.0f;
    }
  auto angles = [&](int cc) {
    const int pb = cc % G::NRA;
    const int t0 = cc * CS;
    // dt = 0 past the end: the angle stays
    const float h_dt = t0 + tkn < L ? sm.rs[pb][1][tkn] : 0.0f;
    const float hdt = 0.5f * h_dt;
#pragma unroll
    for (int k = 0; k < GPW; ++k) {
      const int g = pw + NPW * k;
      if (g < NG) {
        const uint4 rr = staged<G::SA>(sm.ra[pb], tkn, g);
        const float rav[2] = {__uint_as_float(hf ? rr.z : rr.x), __uint_as_float(hf ? rr.w : rr.y)};
        // angle in revolutions: carry + prefix of tanh(rate) pi dt / 2pi = tanh(rate) dt / 2,
        // with tanh(x) = 1 - 2 / (1 + e^{2x}); the fractional part is the reference's
        // mod-2pi wrap, and the hardware sin/cos take revolutions
        float d[2], co[2], si[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) d[j] = fmaf(-h_dt, rcp_fast(1.0f + exp2_fast(2.0f * kLog2e * rav[j])), hdt);
        half_incl_scan2(d);                    // over the tokens, in each half
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const float th = __builtin_amdgcn_fractf(carry[k][j] + d[j]);
          // the angle entering chunk cc (revolutions), for the backward
          if constexpr (SO || SAVE) {
            if (a.chunk_th && tkn == 0) a.chunk_th[(ch0 + cc) * R + 4 * g + 2 * hf + j] = carry[k][j];
          }
          const float c0 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(th), CS - 1));
          const float c1 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(th), 2 * CS - 1));
          carry[k][j] = hf ? c1 : c0;
          co[j] = __builtin_amdgcn_cosf(th);
          si[j] = __builtin_amdgcn_sinf(th);
        }
        sm.tab[cc % G::NTAB][G::toff(tkn, 2 * g + hf)] = make_float4(co[0], si[0], co[1], si[1]);
      }
    }
  };
  // ---- per-token constants of chunk cc (lane = token), by the output wave without an item
  constexpr int kScalarWave = G::NWY - 1;
  float logdec = 0.0f;                     // state-only pass: sum of the chunks' log-decays
  auto scalars = [&](int cc) {
    const int t0 = cc * CS, c3 = cc % 3;
    const bool tok = lane < CS && t0 + lane < L;
    const int tl = lane < CS ? lane : 0;
    const float (&rs)[3][CS + 4] = sm.rs[cc % G::NRA];
    const TokenScalars ts = token_scalars<CS>(rs, tok ? rs[1][tl] : 0.0f, tok, tl, t0, Lnx, lane);
    if (lane < CS) {
      const float ablk = __shfl(ts.acum, lane | 15, 64);
      sm.scl[c3][lane] = ts.scl;
      sm.wdec[c3][lane] = exp2_fast((ts.aend - ts.acum) * kLog2e);
      sm.ac2[c3][lane] = ts.acum * kLog2e;
      sm.expa[c3][lane] = exp2_fast(ts.acum * kLog2e);
      sm.g16[c3][lane] = exp2_fast((ablk - ts.acum) * kLog2e);
      sm.dg[c3][lane] = ts.scl != 0.0f ? ts.gam * rcp_fast(ts.scl) : 0.0f;
      if (lane == 0) sm.dec[c3] = exp2_fast(ts.aend * kLog2e);
      if constexpr (SO) logdec += ts.aend;
    }
  };

  // ---- gate (phase 7), output waves: thread -> (row, 8-column group) of a chunk's Y tile
  constexpr int GROUPS = CS * (P / 8);
  static_assert(GROUPS <= 64 * G::NWY, "the gate on the output waves' threads");
  const int erow = tid / (P / 8), egrp = tid % (P / 8);
  const bool eact = tid < GROUPS;
  Vec8<T> zr;                              // Z of the chunk waiting for its gate
  zr.zero();
  auto load_z = [&](int c) {
    if (has_z && eact && c * CS + erow < L) zr.load(z_base + (long)(c * CS + erow) * vz_stride + 8 * egrp);
  };
  auto gate = [&](int c) {                 // Y of chunk c -> out
    if (eact && c * CS + erow < L) {
      const int off = G::yoff(erow, 8 * egrp);
      Vec8<T> ya, yb;
      ya.load(&sm.yd[off]);
      yb.load(&sm.yo[off]);
      const float ea = sm.expa[c % 3][erow];   // the e^{A_cum} row scale of Q h^T
      float o[8], ob[8];
      ya.to_f(o);
      yb.to_f(ob);
#pragma unroll
      for (int q = 0; q < 8; ++q) o[q] = fmaf(ob[q], ea, o[q]);
      if (erow >= 16) {                    // rows 16..31: the off-diagonal item
        Vec8<T> yc;
        float oc[8];
        yc.load(&sm.ydo[G::yoff(erow - 16, 8 * egrp)]);
        yc.to_f(oc);
#pragma unroll
        for (int q = 0; q < 8; ++q) o[q] += oc[q];
      }
      if constexpr (SAVE) {
        // the training forward: the output before the gate, for the backward's dZ
        if (has_z && a.out_v)
          store8(reinterpret_cast<T*>(a.out_v) + (o_base - gO) + (long)(c * CS + erow) * v_stride + 8 * egrp, o);
      }
      if (has_z) {
        float zf[8];
        zr.to_f(zf);
#pragma unroll
        for (int q = 0; q < 8; ++q) o[q] *= silu_fast(zf[q]);
      }
      store8(o_base + (long)(c * CS + erow) * v_stride + 8 * egrp, o);
    }
  };

  // ---- phase 3 as (query block lb, key block sb <= lb) items, one per output wave:
  // three at 32-token chunks, on three SIMDs (each also holds a state wave).  An item
  // is the 16 x 16 block S^T of keys 16 sb.. against queries 16 lb.., masked -- decayed
  // off the diagonal block; on it causal, with D + gamma QK on the diagonal -- then
  // M V over those 16 keys for every p-tile.  The diagonal items write their rows of
  // Y_diag to yd, the off-diagonal one to ydo, which the gate adds.  The S^T operands
  // are read four k-steps at a time: in step s of a 16-wide block of the d_state axis,
  // k slot i/16 of lane i stands for column k0 + 4 (i/16) + s in both operands (the
  // dot product is the same sum in another order), one 16-byte read per operand per
  // four MFMAs.
  auto diag_item = [&](auto lb_c, auto sb_c, int c) {
    if constexpr (!SO) {
    const uint4* sv = sm.rv[c & 1];
    const PlaneTile<CS, N>&q = sm.q[c & 1], &k = sm.k[c & 1];
    constexpr int lb = decltype(lb_c)::value, sb = decltype(sb_c)::value;
    static_assert(sb <= lb, "causal items only");
    // lane-derived addresses are recomputed here, not kept live across the loop
    int ln = lane;
    asm volatile("" : "+v"(ln));
    const int g4l = 4 * (ln >> 4);
    const int l = 16 * lb + (ln & 15);
    const float al = sm.ac2[c % 3][l];
    f32x4 st = {0.0f, 0.0f, 0.0f, 0.0f}, stl = {0.0f, 0.0f, 0.0f, 0.0f};
    Parts8 ka[1] = {k.row(16 * sb, 0, ln)}, qa[1] = {q.row(16 * lb, 0, ln)};
#pragma unroll
    for (int s = 0; s < N / 32; ++s) {
      Parts8 kn[1], qn[1];
      if (s + 1 < N / 32) {
        kn[0] = k.row(16 * sb, s + 1, ln);
        qn[0] = q.row(16 * lb, s + 1, ln);
      }
      __builtin_amdgcn_sched_barrier(0);
      mma_parts<1>(ka, qa, &st, &stl);
      if (s + 1 < N / 32) {
        ka[0] = kn[0];
        qa[0] = qn[0];
      }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) st[r] += stl[r];
    const int s0 = 16 * sb + g4l;
    if constexpr (sb < lb) {
      // off-diagonal block: e^{A_l - A_s} = e^{A_l - A_e} e^{A_e - A_s}, both <= 1
      const float f = exp2_fast(fminf(al - sm.ac2[c % 3][16 * sb + 15], 0.0f));
      const float4 gg = *reinterpret_cast<const float4*>(&sm.g16[c % 3][s0]);
      st[0] *= f * gg.x; st[1] *= f * gg.y; st[2] *= f * gg.z; st[3] *= f * gg.w;
    } else {
      // diagonal block: causal decay below the diagonal; on it, D plus the
      // QK skip gamma_l (q_l . k_l) (the stored key carries the scale)
      const float dgl = sm.dg[c % 3][l];
      const float4 as = *reinterpret_cast<const float4*>(&sm.ac2[c % 3][s0]);
      const float asv[4] = {as.x, as.y, as.z, as.w};
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float v = st[r] * exp2_fast(fminf(al - asv[r], 0.0f));
        st[r] = (s0 + r < l) ? v : (s0 + r == l ? Dh + st[r] * dgl : 0.0f);
      }
    }
    // M V: the A operand is the masked block itself (lane i, reg j: query l, key
    // 16 sb + 4 (i/16) + j), matched by V's rows
    f32x4 yd[G::PT];
#pragma unroll
    for (int pt = 0; pt < G::PT; ++pt)
#pragma unroll
      for (int r = 0; r < 4; ++r) yd[pt][r] = 0.0f;
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int pt = 0; pt < G::PT; ++pt)
        yd[pt] = W::mma(st[j], W::template vdiag<G::SV>(sv, 16 * pt, 16 * sb, j, ln), yd[pt]);
    T* dst = sb == lb ? sm.yd + 16 * lb * G::LDY : sm.ydo;
#pragma unroll
    for (int pt = 0; pt < G::PT; ++pt)
#pragma unroll
      for (int r = 0; r < 4; r += 2)
        store_pair(&dst[G::yoff(g4l + r, 16 * pt + (ln & 15))], &dst[G::yoff(g4l + r + 1, 16 * pt + (ln & 15))],
                   yd[pt][r], yd[pt][r + 1]);
    }
  };
  f32x4 hs[G::NB16];
  entering_state<G>(hs, a, cb, swave, 16 * pr + (lane & 15), 4 * (lane >> 4));
  // ---- phase 6, state waves: Y_off = Q_r h^T for my p-tile, query blocks lb = part (mod SPT)
  auto state_yoff = [&](int c) {
    if constexpr (!SO) {
    // lane-derived addresses are recomputed here, not kept live across the loop
    int ln = lane;
    asm volatile("" : "+v"(ln));
    const PlaneTile<CS, N>& qp = sm.q[c & 1];
    constexpr int NLB = G::LB16 / G::SPT;
    f32x4 yo[NLB], yl[NLB];
#pragma unroll
    for (int i = 0; i < NLB; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) yo[i][r] = yl[i][r] = 0.0f;
    // a step's query operands are requested before the state's split, which hides them
#pragma unroll
    for (int q = 0; q < N / 32; ++q) {
      Parts8 qa[NLB], hp[NLB];
#pragma unroll
      for (int i = 0; i < NLB; ++i) qa[i] = qp.row(16 * (part + G::SPT * i), q, ln);
      __builtin_amdgcn_sched_barrier(0);
      const float hv[8] = {hs[2 * q][0], hs[2 * q][1], hs[2 * q][2], hs[2 * q][3],
                           hs[2 * q + 1][0], hs[2 * q + 1][1], hs[2 * q + 1][2], hs[2 * q + 1][3]};
      hp[0] = split8(hv);
#pragma unroll
      for (int i = 1; i < NLB; ++i) hp[i] = hp[0];
      mma_parts<NLB>(qa, hp, yo, yl);
    }
    const int pcol = 16 * pr + (ln & 15), g4 = 4 * (ln >> 4);
#pragma unroll
    for (int i = 0; i < NLB; ++i) {
      const int lb = part + G::SPT * i;
#pragma unroll
      for (int r = 0; r < 4; r += 2)
        store_pair(&sm.yo[G::yoff(16 * lb + g4 + r, pcol)], &sm.yo[G::yoff(16 * lb + g4 + r + 1, pcol)],
                   yo[i][r] + yl[i][r], yo[i][r + 1] + yl[i][r + 1]);
    }
    }
  };
  // ---- phases 4-5, state waves: h <- e^{A_end} h + K_s^T (w V) for my p-tile
  auto state_update = [&](int c) {
    int ln = lane;
    asm volatile("" : "+v"(ln));
    const uint4* sv = sm.rv[c & 1];
    const PlaneTile<CS, N>& kt = sm.k[c & 1];
    // the state entering chunk c, [p][n], for the backward
    if constexpr (SO || SAVE) {
      if (a.chunk_h && part == 0) {
        T* dst = reinterpret_cast<T*>(a.chunk_h) + (ch0 + c) * P * N;
#pragma unroll
        for (int nb = 0; nb < G::NB16; ++nb) {
          const float hv[4] = {hs[nb][0], hs[nb][1], hs[nb][2], hs[nb][3]};
          store4(dst + saved_tile_off<N>(pr, nb, lane), hv);
        }
      }
    }
    const float dec = sm.dec[c % 3];
    const float* w = &sm.wdec[c % 3][8 * (ln >> 4)];
    const float4 w0 = *reinterpret_cast<const float4*>(w), w1 = *reinterpret_cast<const float4*>(w + 4);
    const float wv[8] = {w0.x, w0.y, w0.z, w0.w, w1.x, w1.y, w1.z, w1.w};
    float wx[8];                         // w V: tokens 8 (lane/16) + 0..7, column 16 pr + lane%16
#pragma unroll
    for (int j = 0; j < 8; ++j) wx[j] = *staged_elem<G::SV, float>(sv, 8 * (ln >> 4) + j, 16 * pr + (ln & 15)) * wv[j];
    // the key operands, two state tiles at a time, requested a step ahead
    Parts8 kp[2] = {kt.col(0, ln), kt.col(1, ln)}, wp[2];
    wp[0] = wp[1] = split8(wx);
#pragma unroll
    for (int nb = 0; nb < G::NB16; ++nb)
#pragma unroll
      for (int r = 0; r < 4; ++r) hs[nb][r] *= dec;
#pragma unroll
    for (int nb = 0; nb < G::NB16; nb += 2) {
      Parts8 kn[2];
      if (nb + 2 < G::NB16) {
        kn[0] = kt.col(nb + 2, ln);
        kn[1] = kt.col(nb + 3, ln);
      }
      __builtin_amdgcn_sched_barrier(0);
      mma_parts<2>(kp, wp, &hs[nb], &hs[nb]);
      if (nb + 2 < G::NB16) {
        kp[0] = kn[0];
        kp[1] = kn[1];
      }
    }
  };

  // ---- prologue: chunk 0's inputs, its angles and constants, then its planes; chunk 1's
  // angles and constants (the loop works one chunk ahead in the preparation and two in
  // the angles)
  const bool pwave = SO ? !swave : wave >= G::NWY + G::NST;
  zero_staging<G>(sm, tid);
  if (tid == 0) sm.one = make_float4(1.0f, 0.0f, 1.0f, 0.0f);
  if (pwave) {
    const f32x4* qb = reinterpret_cast<const f32x4*>(a.qbias + (long)cb.h * N);
    const f32x4* kb = reinterpret_cast<const f32x4*>(a.kbias + (long)cb.h * N);
    qb4 = qb[cq];
    kb4 = kb[cq];
#pragma unroll
    for (int i = 0; i < NI; ++i) load_raw(0, i);
  }
  __syncthreads();
  stage_v(0);
  stage_ars(0);
  if (G::NRA > 1 && nc > 1) stage_ars(1);
  if (swave) __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  if (pwave) angles(0);
  if (wave == kScalarWave) scalars(0);
  __syncthreads();
  if (pwave) {
    prep(0, kI0, kI1);
    prep_rest(0);
  }
  if (nc > G::NRA) stage_ars(G::NRA);    // chunk 0 is done with its buffer
  if (swave) __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  if (nc > 1) {
    if (pwave) angles(1);
    if (wave == kScalarWave) scalars(1);
  }
  if (!SO && ywave) load_z(0);
  __syncthreads();

  // ---- the chunk loop, one per role: the roles share no loop-carried registers, and
  // every loop passes the same barriers: two per chunk, one in the state-only pass.
  //   phase 1  preparation waves: a first part of chunk c+1's planes (its table, key
  //            scale and rows are there), loading chunk c+2's rows in their place; state
  //            waves: the direct-to-LDS loads of V (chunk c+1) and the rates, then Y_off
  //            of chunk c; output waves: its items
  //   phase 2  preparation waves: the rest of the planes, chunk c+2's angles; state
  //            waves: the update; output waves: the gate, and chunk c+2's constants
  // The state-only pass has no Y, so nothing in it waits within a chunk.
  static_assert(!SO || (G::NTAB == 2 && G::NRA == 2), "one barrier per chunk");
  if (swave) {
    for (int c = 0; c < nc; ++c) {
      if (c + 1 < nc) stage_v(c + 1);
      if (c + G::NRA + 1 < nc) stage_ars(c + G::NRA + 1);
      if constexpr (!SO) {
        state_yoff(c);
        if (G::NRA == 1 && wave == kWA) __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
      }
      state_update(c);
      __builtin_amdgcn_s_waitcnt(0);     // this wave's staged loads are done
      __syncthreads();
    }
    if (a.fin_h && fin_here && part == 0) {
#pragma unroll
      for (int nb = 0; nb < G::NB16; ++nb)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          a.fin_h[((long)ci_out * P + 16 * pr + (lane & 15)) * N + 16 * nb + 4 * (lane >> 4) + r] = hs[nb][r];
    }
  } else if (ywave && !SO) {
    for (int c = 0; c < nc; ++c) {
      static_assert(G::LB16 == 2 && G::NWY >= 3, "three items on three output waves");
      if (wave == 0) diag_item(std::integral_constant<int, 0>{}, std::integral_constant<int, 0>{}, c);
      if (wave == 1) diag_item(std::integral_constant<int, 1>{}, std::integral_constant<int, 1>{}, c);
      if (wave == 2) diag_item(std::integral_constant<int, 1>{}, std::integral_constant<int, 0>{}, c);
      __syncthreads();
      gate(c);
      if (c + 1 < nc) load_z(c + 1);
      if (wave == kScalarWave && c + 2 < nc) scalars(c + 2);
      __syncthreads();
    }
  } else {
    for (int c = 0; c + 1 < nc; ++c) {
      prep(c + 1, kI0, kI1);
      if constexpr (!kPrep2) prep_rest(c + 1);
      if constexpr (!SO) __syncthreads();
      if constexpr (kPrep2) prep_rest(c + 1);
      if (c + 2 < nc) {
        angles(c + 2);
        if (SO && wave == kScalarWave) scalars(c + 2);
      }
      __syncthreads();
    }
    if constexpr (!SO) __syncthreads();          // the last chunk has nothing to prepare
    __syncthreads();
  }

  // the final carry's k (the last token's rope'd key, unscaled: its row is in the last
  // loads, its angles in the table) and v (in the last chunk's staged rows)
  if (a.fin_k && fin_here) {
    if (pwave) {
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const int t = ptok + RPI * i;
        if ((nc - 1) * CS + t == L - 1) {
          float kf[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) kf[e] = kraw[i][e] + kb4[e];
          turn(kf, table(nc - 1, t));
#pragma unroll
          for (int e = 0; e < 4; ++e) a.fin_k[(long)ci_out * N + 4 * cq + e] = kf[e];
        }
      }
    }
    for (int i = tid; i < P; i += G::NT)
      a.fin_v[(long)ci_out * P + i] = *staged_elem<G::SV, T>(sm.rv[(nc - 1) & 1], L - 1 - (nc - 1) * CS, i);
  }
  if constexpr (SO) {
    if (a.fin_logdec && fin_here && wave == kScalarWave && lane == 0) a.fin_logdec[ci_out] = logdec;
  }
  if (a.fin_theta && fin_here && pwave && tkn == 0) {
#pragma unroll
    for (int k = 0; k < GPW; ++k)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int r = 4 * (pw + NPW * k) + 2 * hf + j;
        if (r < R) a.fin_theta[(long)ci_out * R + r] = carry[k][j] * kTwoPi;
      }
  }
}

}  // namespace chunked_f32

// ------------------------------------------------------------------ dispatch
// (chunk, d_state, headdim, rotation width) instantiations with float32 I/O; R is the
// model's rope_fraction 0.5 (R = N/4) or 1.0 (R = N/2) width.  Chunk sizes that are
// multiples of 32 run as 32-token sub-chunks (the chunked form is an exact rewrite of
// the token recurrence for every chunk size: only the rounding differs).
#define M3_F32_SHAPES(X)                                                                       \
  X(32, 128, 64, 32) X(32, 128, 64, 64) X(32, 64, 64, 16) X(32, 64, 64, 32) X(32, 64, 32, 16) \
  X(32, 32, 32, 8) X(32, 32, 64, 8)

constexpr int kF32Waves = 12;

static int f32_kernel_chunk(int CS) { return (CS > 32 && CS % 32 == 0) ? 32 : CS; }

bool scan_chunked_f32_supported(int CS_, int N, int P, int R) {
  const int CS = f32_kernel_chunk(CS_);
#define X(cs, n, p, r) \
  if (CS == cs && N == n && P == p && R == r) return true;
  M3_F32_SHAPES(X)
#undef X
  return false;
}

// shapes whose full pass can also write the chunk states (the backward's float32 shapes)
#define M3_F32_SAVE_SHAPES(X) X(32, 128, 64, 32) X(32, 128, 64, 64) X(32, 64, 64, 16) X(32, 64, 32, 16)

// the state-only pass: the sequence split's first pass and the backward's chunk states
#define M3_F32_STATE_SHAPES(X) X(32, 128, 64, 32) X(32, 128, 64, 64) X(32, 64, 64, 16) X(32, 64, 32, 16)

bool scan_state_f32_supported(int CS_, int N, int P, int R) {
  const int CS = f32_kernel_chunk(CS_);
#define X(cs, n, p, r) \
  if (CS == cs && N == n && P == p && R == r) return true;
  M3_F32_STATE_SHAPES(X)
#undef X
  return false;
}

hipError_t scan_state_f32_launch(const ScanArgs& a, hipStream_t st) {
  const int CS = f32_kernel_chunk(a.CS);
  const int nseg = a.seg_len > 0 ? (a.L + a.seg_len - 1) / a.seg_len : 1;
#define X(cs, n, p, r)                                                                               \
  if (CS == cs && a.N == n && a.P == p && a.R == r) {                                                \
    hipLaunchKernelGGL((chunked_f32::scan_chunked_f32_kernel<float, cs, n, p, r, kF32Waves, true>),  \
                       dim3(a.B * a.H, nseg), dim3(64 * kF32Waves), 0, st, a);                       \
    return hipGetLastError();                                                                        \
  }
  M3_F32_STATE_SHAPES(X)
#undef X
  return hipErrorInvalidValue;
}

hipError_t scan_chunked_f32_launch(const ScanArgs& a, hipStream_t st) {
  const int CS = f32_kernel_chunk(a.CS);
  const int nseg = a.seg_len > 0 ? (a.L + a.seg_len - 1) / a.seg_len : 1;
  if (a.chunk_h) {
#define X(cs, n, p, r)                                                                                 \
  if (CS == cs && a.N == n && a.P == p && a.R == r) {                                                  \
    hipLaunchKernelGGL((chunked_f32::scan_chunked_f32_kernel<float, cs, n, p, r, kF32Waves, false, true>), \
                       dim3(a.B * a.H, nseg), dim3(64 * kF32Waves), 0, st, a);                         \
    return hipGetLastError();                                                                          \
  }
    M3_F32_SAVE_SHAPES(X)
#undef X
    return hipErrorInvalidValue;
  }
#define X(cs, n, p, r)                                                                                 \
  if (CS == cs && a.N == n && a.P == p && a.R == r) {                                                  \
    hipLaunchKernelGGL((chunked_f32::scan_chunked_f32_kernel<float, cs, n, p, r, kF32Waves, false>),   \
                       dim3(a.B * a.H, nseg), dim3(64 * kF32Waves), 0, st, a);                         \
    return hipGetLastError();                                                                          \
  }
  M3_F32_SHAPES(X)
#undef X
  return hipErrorInvalidValue;
}

}  // namespace m3
