// Sequence split of the chunked prefill for few (batch, head) pairs.
//
// With B·H well below the CU count (config 3: B·H = 32 on 256 CUs) one block per
// (b, h) leaves most of the chip idle.  The recurrence is linear in its carry, so a
// sequence can be cut into S segments that run side by side:
//
//   pass 1  the state-only kernel runs every segment from a zero carry and leaves
//           its exit state h_i^0, rope angle advance Δθ_i and total log-decay ΣA_i,
//           with keys rotated by the segment's own angles (starting from zero).  A segment's last
//           token already carries the trapezoid's cross term with the next token
//           (its key scale reads the next token), so h_i^0 is complete;
//   pass 2  the combine chains the segments, one thread per state element: the state entering segment
//           i+1 is  h' = e^{ΣA_i} h + h_i^0 rot(θ)^T  and  θ' = θ + Δθ_i (mod 2π),
//           where rot(θ) turns the rope pairs (2r, 2r+1) of the state's d_state axis
//           by the entering angles (a rotation by θ + φ is rotation by φ, then θ).
//           Only segment 0 enters with a carry that lacks the cross term (a caller's
//           carry from an earlier prefill): there the first summand is
//           e^{ΣA_0} (h + c v ⊗ k) with c = (1 - sigmoid(trap)) dt of the first
//           token, as the kernel forms its entering state;
//   pass 3  the full kernel runs every segment from its entering carry; the carry
//           of segments 1.. has zero k and v, so the kernel adds no cross term again.
//
// This is the reference's sequence-parallel carry algebra (models/mamba3_seqpar.py:
// 67-110) applied across CUs of one GPU; the extra work is pass 1 (no Q, Y or gate).
#include <algorithm>

#include "m3_scan.h"

namespace m3 {
namespace {

constexpr int kCombineThreads = 256;
constexpr int kTargetBlocks = 256;     // MI355X compute units
constexpr int kMinSegment = 64;        // tokens
constexpr int kMaxRounds = 4;          // rounds of blocks on the chip, at most

// Modelled time of one pass of n 64-token steps on nb blocks, in ns: rounds of 256 blocks
// (one per compute unit), each with a start and a time per step that grows a little with
// the blocks and is at least the time that the chip's memory takes for their bytes
// (N: d_state; the value dimension counts little).  Slopes and intercepts of passes
// measured alone (graph replays): per step 2.5 us in bf16 and 6.8 us in float32 at d_state
// 128 (state-only pass 1.4 and 2.1), 3.4 us in bf16 with every compute unit busy.
long pass_ns(bool bf16_io, bool state_only, int N, long nb, long n) {
  const bool wide = N >= 128;
  const long full[2][2] = {{4100, 6800}, {2020, 2480}};
  const long so[2][2] = {{1500, 2050}, {950, 1300}};
  const long base = state_only ? so[bf16_io][wide] : full[bf16_io][wide];
  const long grow10 = state_only ? 20 : 15;                                  // 0.1 ns per step and block
  const long mem10 = (state_only ? (wide ? 67 : 43) : (wide ? 133 : 92)) * (bf16_io ? 1 : 2);
  const long start = state_only ? 5000 : 5700;
  long t = 0;
  for (long left = nb; left > 0; left -= kTargetBlocks) {
    const long b = std::min<long>(left, kTargetBlocks);
    t += start + n * std::max(base + grow10 * b / 10, mem10 * b / 10);
  }
  return t;
}

// Segment length, or 0 for no split.  Segments are whole multiples of 64 tokens, so every
// interior segment ends on a kernel chunk (64 tokens in bf16, 32 in float32).  The segment
// count with the least modelled time (both passes, 10 us for the combine and the gaps, 0.4
// us per segment) is taken if that is 5% below one pass's.  Measured, in us, one pass / the
// former rule (reserved_seg_len, which counts no starts) / this one:
//   bf16  d_state 128: 96 pairs of 1500 tokens 68 / 93 / 68, 128 of 1000 47 / 67 / 47,
//         24 of 4096 166 / 60 / 60, 32 of 2000 87 / 56 / 46, 24 of 613 40 / 44 / 40
//   bf16  d_state 64: 16 of 3000 100 / 100 / 34
//   f32   d_state 128: 24 of 600 66 / 58 / 39;  d_state 64: 16 of 1024 70 / 70 / 31
int seg_len_for(bool bf16_io, int B, int H, int L, int N) {
  const int bh = B * H;
  if (bh <= 0 || bh * 2 > kTargetBlocks || L < 2 * kMinSegment) return 0;
  const int smax = min(L / kMinSegment, kMaxRounds * kTargetBlocks / bh);
  const long one = pass_ns(bf16_io, false, N, bh, (L + 63) / 64);
  int best = 0;
  long best_cost = one - one / 20;
  for (int s = 2; s <= smax; ++s) {
    const int len = ((L + s - 1) / s + 63) / 64 * 64;
    const long ns = (L + len - 1) / len, n = len / 64;
    if (ns < 2) continue;
    const long cost = pass_ns(bf16_io, false, N, bh * ns, n) + pass_ns(bf16_io, true, N, bh * (ns - 1), n) + 10000 +
                      400 * ns;
    if (cost < best_cost) {
      best = len;
      best_cost = cost;
    }
  }
  return best;
}

// The segments of the least workspace that a split call takes (scan_split_ws_bytes), which
// are also those of the backward's state passes: d_state 128 and headdim 64, whole multiples of 128
// tokens, at least 256; the state-only pass counted as half the full pass's time per
// token, starts as nothing.
int reserved_seg_len(int B, int H, int L) {
  const int bh = B * H;
  if (bh <= 0 || bh * 2 > kTargetBlocks || L < 512) return 0;
  const int smax = min(L / 256, kMaxRounds * kTargetBlocks / bh);
  int best = 0;
  long best_cost = 0;
  for (int s = 2; s <= smax; ++s) {
    const int len = ((L + s - 1) / s + 127) / 128 * 128;
    const long ns = (L + len - 1) / len;
    if (ns < 2) continue;
    const long rounds = (bh * ns + kTargetBlocks - 1) / kTargetBlocks;
    const long so_rounds = (bh * (ns - 1) + kTargetBlocks - 1) / kTargetBlocks;
    const long cost = (2 * rounds + so_rounds) * len;     // in half-token units of one block
    if (best == 0 || cost < best_cost) {
      best = len;
      best_cost = cost;
    }
  }
  return best;
}

struct Carries {
  float* h;   // (BH, S, P, N)
  float* k;   // (BH, S, N)   last rope'd key (pass 1 writes it; the combine does not need it)
  float* v;   // (BH, S, P)
  float* th;  // (BH, S, R)
  float* ld;  // (BH, S)      pass 1: the segment's total log-decay
};

size_t align256(size_t x) { return (x + 255) & ~size_t(255); }

// Carve the workspace: the local carries of pass 1, then the entering carries of pass 3.
size_t carve(char* base, long bhs, int N, int P, int R, Carries* loc, Carries* in) {
  size_t off = 0;
  auto take = [&](size_t n) {
    float* p = base ? reinterpret_cast<float*>(base + off) : nullptr;
    off += align256(n * sizeof(float));
    return p;
  };
  Carries* sets[2] = {loc, in};
  for (int set = 0; set < 2; ++set) {
    Carries* c = sets[set];
    Carries t;
    t.h = take((size_t)bhs * P * N);
    t.k = take((size_t)bhs * N);
    t.v = take((size_t)bhs * P);
    t.th = take((size_t)bhs * (R > 0 ? R : 1));
    t.ld = set == 0 ? take((size_t)bhs) : nullptr;
    if (c) *c = t;
  }
  return off;
}

// Grid (P*N / kCombineThreads, B*H): thread -> state element (p, n) of one (b, h),
// walking the segments in order.  Block x == 0 also writes the small carry parts
// (angles, zero k and v of segments 1..).
__global__ __launch_bounds__(kCombineThreads)
void seg_combine_kernel(ScanArgs a, int nseg, Carries loc, Carries in) {
  const int bh = blockIdx.y, tid = threadIdx.x;
  const int N = a.N, P = a.P, R = a.R;
  const long c0 = (long)bh * nseg;                 // carry slot of segment 0
  const int e = blockIdx.x * kCombineThreads + tid;
  if (blockIdx.x == 0) {
    for (int n = tid; n < N; n += kCombineThreads) {
      in.k[c0 * N + n] = a.init_k ? a.init_k[(long)bh * N + n] : 0.0f;
      for (int i = 1; i < nseg; ++i) in.k[(c0 + i) * N + n] = 0.0f;
    }
    for (int p = tid; p < P; p += kCombineThreads) {
      in.v[c0 * P + p] = a.init_v ? a.init_v[(long)bh * P + p] : 0.0f;
      for (int i = 1; i < nseg; ++i) in.v[(c0 + i) * P + p] = 0.0f;
    }
    for (int r = tid; r < R; r += kCombineThreads) {
      float th = a.init_theta ? a.init_theta[(long)bh * R + r] : 0.0f;
      in.th[c0 * R + r] = th;
      for (int i = 0; i + 1 < nseg; ++i) {
        const float x = th + loc.th[(c0 + i) * R + r];
        th = x - kTwoPi * floorf(x * kInvTwoPi);
        in.th[(c0 + i + 1) * R + r] = th;
      }
    }
  }
  if (e >= P * N) return;
  const int p = e / N, n = e % N, r = n >> 1;
  const bool rope = r < R;
  // segment 0 enters with the caller's carry, or zero; its cross term with the
  // previous token (c = (1 - sigmoid(trap_0)) dt_0) is added here, as the kernel
  // adds it to an entering carry
  float h = a.init_h ? a.init_h[(long)bh * P * N + e] : 0.0f;
  in.h[c0 * P * N + e] = h;
  if (a.init_h) {
    const float dt0 = a.dt[(long)bh * a.L], tr0 = a.trap[(long)bh * a.L];
    h += (1.0f - 1.0f / (1.0f + expf(-tr0))) * dt0 * a.init_v[(long)bh * P + p] * a.init_k[(long)bh * N + n];
  }
  float th = rope && a.init_theta ? a.init_theta[(long)bh * R + r] : 0.0f;
  // the segments' values (the element's rope pair of the exit state, the angle advance
  // and the log-decay) are loaded kBatch segments at a time before the chain uses them:
  // the steps are a few operations each, so a load per step would be all latency
  constexpr int kBatch = 8;
  for (int i0 = 0; i0 + 1 < nseg; i0 += kBatch) {
    float2 hp[kBatch];
    float dth[kBatch], ld[kBatch];
#pragma unroll
    for (int j = 0; j < kBatch; ++j) {
      const long ci = c0 + min(i0 + j, nseg - 2);
      hp[j] = *reinterpret_cast<const float2*>(loc.h + ci * P * N + p * N + 2 * r);
      dth[j] = rope ? loc.th[ci * R + r] : 0.0f;
      ld[j] = loc.ld[ci];
    }
#pragma unroll
    for (int j = 0; j < kBatch; ++j) {
      if (i0 + j + 1 >= nseg) break;
      float own = (n & 1) ? hp[j].y : hp[j].x;
      if (rope) {                        // segment-local key frame -> entering frame
        float sn, cs;
        sincosf(th, &sn, &cs);
        own = (n & 1) ? hp[j].x * sn + hp[j].y * cs : hp[j].x * cs - hp[j].y * sn;
        const float x = th + dth[j];
        th = x - kTwoPi * floorf(x * kInvTwoPi);
      }
      h = expf(ld[j]) * h + own;
      in.h[(c0 + i0 + j + 1) * P * N + e] = h;
    }
  }
}

}  // namespace

namespace {
size_t split_bytes(int len, int B, int L, int H, int N, int P, int R) {
  return len == 0 ? 0 : carve(nullptr, (long)B * H * ((L + len - 1) / len), N, P, R, nullptr, nullptr);
}
bool split_supported(bool bf16_io, int N, int P, int R, int CS) {
  // shapes without a state-only pass run one pass
  return scan_state_supported(bf16_io, 64, N, P, R) && scan_chunked_supported(bf16_io, CS, N, P, R);
}
}  // namespace

size_t scan_split_ws_bytes(bool bf16_io, int B, int L, int H, int N, int P, int R, int CS) {
  if (N != 128 || P != 64 || !split_supported(bf16_io, N, P, R, CS)) return 0;
  return split_bytes(reserved_seg_len(B, H, L), B, L, H, N, P, R);
}

size_t scan_split_plan_bytes(bool bf16_io, int B, int L, int H, int N, int P, int R, int CS) {
  if (!split_supported(bf16_io, N, P, R, CS)) return 0;
  const size_t need = split_bytes(seg_len_for(bf16_io, B, H, L, N), B, L, H, N, P, R);
  return need == 0 ? 0 : std::max(need, scan_split_ws_bytes(bf16_io, B, L, H, N, P, R, CS));
}

int scan_split_len(bool bf16_io, int B, int L, int H, int N, int P, int R, int CS, size_t ws_bytes) {
  if (!split_supported(bf16_io, N, P, R, CS)) return 0;
  const int len = seg_len_for(bf16_io, B, H, L, N);
  if (len == 0 || split_bytes(len, B, L, H, N, P, R) <= ws_bytes) return len;
  const size_t reserved = scan_split_ws_bytes(bf16_io, B, L, H, N, P, R, CS);
  return reserved > 0 && reserved <= ws_bytes ? reserved_seg_len(B, H, L) : 0;
}

hipError_t scan_split_launch(const ScanArgs& a, bool bf16_io, int len, void* ws, hipStream_t st) {
  const int nseg = (a.L + len - 1) / len;
  const long bhs = (long)a.B * a.H * nseg;
  Carries loc, in;
  carve(reinterpret_cast<char*>(ws), bhs, a.N, a.P, a.R, &loc, &in);

  ScanArgs p1 = a;                                   // pass 1: exit carries from a zero carry
  p1.seg_len = len;
  p1.init_theta = p1.init_h = p1.init_k = p1.init_v = nullptr;
  p1.fin_h = loc.h; p1.fin_k = loc.k; p1.fin_v = loc.v; p1.fin_theta = a.R > 0 ? loc.th : nullptr;
  p1.fin_logdec = loc.ld;
  p1.fin_per_seg = 1;
  p1.chunk_h = nullptr;                              // the saved residuals come from pass 3
  p1.chunk_th = nullptr;
  p1.out_v = nullptr;
  p1.CS = 64;                                        // 64-token (bf16) or 32-token (float32) sub-chunks
  p1.so_skip_last = 1;                               // no segment reads the last one's exit carry
  hipError_t e = scan_state_launch(p1, bf16_io, st);
  if (e != hipSuccess) return e;

  ScanArgs p2 = a;                                   // pass 2: entering carries
  p2.seg_len = len;
  hipLaunchKernelGGL(seg_combine_kernel, dim3((a.P * a.N + kCombineThreads - 1) / kCombineThreads, a.B * a.H),
                     dim3(kCombineThreads), 0, st, p2, nseg, loc, in);
  e = hipGetLastError();
  if (e != hipSuccess) return e;

  ScanArgs p3 = a;                                   // pass 3: the scan from the entering carries
  p3.seg_len = len;
  p3.init_h = in.h; p3.init_k = in.k; p3.init_v = in.v; p3.init_theta = a.R > 0 ? in.th : nullptr;
  p3.init_per_seg = 1;
  return scan_chunked_launch(p3, bf16_io, st);
}

hipError_t scan_split_state_launch(const ScanArgs& a, bool bf16_io, void* ws, hipStream_t st) {
  const int len = scan_split_len(bf16_io, a.B, a.L, a.H, a.N, a.P, a.R, 64,
                                 scan_split_ws_bytes(bf16_io, a.B, a.L, a.H, a.N, a.P, a.R, 64));
  if (len == 0) return scan_state_launch(a, bf16_io, st);
  const int nseg = (a.L + len - 1) / len;
  const long bhs = (long)a.B * a.H * nseg;
  Carries loc, in;
  carve(reinterpret_cast<char*>(ws), bhs, a.N, a.P, a.R, &loc, &in);

  ScanArgs p1 = a;                                   // pass 1: exit carries from a zero carry
  p1.seg_len = len;
  p1.init_theta = p1.init_h = p1.init_k = p1.init_v = nullptr;
  p1.fin_h = loc.h; p1.fin_k = loc.k; p1.fin_v = loc.v; p1.fin_theta = a.R > 0 ? loc.th : nullptr;
  p1.fin_logdec = loc.ld;
  p1.init_per_seg = 0;
  p1.fin_per_seg = 1;
  p1.chunk_h = nullptr;
  p1.chunk_th = nullptr;
  p1.so_skip_last = 1;                               // no segment reads the last one's exit carry
  hipError_t e = scan_state_launch(p1, bf16_io, st);
  if (e != hipSuccess) return e;

  ScanArgs p2 = a;                                   // pass 2: entering carries (none from the caller)
  p2.seg_len = len;
  p2.init_theta = p2.init_h = p2.init_k = p2.init_v = nullptr;
  hipLaunchKernelGGL(seg_combine_kernel, dim3((a.P * a.N + kCombineThreads - 1) / kCombineThreads, a.B * a.H),
                     dim3(kCombineThreads), 0, st, p2, nseg, loc, in);
  e = hipGetLastError();
  if (e != hipSuccess) return e;

  ScanArgs p3 = a;                                   // pass 3: the states entering every chunk
  p3.seg_len = len;
  p3.init_h = in.h; p3.init_k = in.k; p3.init_v = in.v; p3.init_theta = a.R > 0 ? in.th : nullptr;
  p3.init_per_seg = 1;
  p3.fin_theta = p3.fin_h = p3.fin_k = p3.fin_v = nullptr;
  p3.fin_logdec = nullptr;
  p3.fin_per_seg = 0;
  return scan_state_launch(p3, bf16_io, st);
}

}  // namespace m3
