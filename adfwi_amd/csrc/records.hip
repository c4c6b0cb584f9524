// Record post-processing on the GPU: the per-trace waveform L2 misfit of the FWI drivers,
// optionally with the per-trace max normalisation of the synthetic traces, and its adjoint
// source, in one kernel over the [S][nt][R] records.
//
//   n[s,t,r] = a[s,t,r] / max_t |a[s,.,r]|     (normalize_a; fwi/acoustic_fwi.py:149-150)
//   rsd      = n - b,  e[s,r] = sum_t rsd^2 dt,  trace loss = sqrt(e)   (fwi/misfit/L2.py:26-29)
//   d loss / d n[t] = w rsd[t],  w = dt / sqrt(e)
//   d loss / d a[t] = w rsd[t] / m  -  [t == t*] sign(a[t*]) w (sum_t' rsd[t'] a[t']) / m^2
// with m = max_t |a| reached first at t* (the max's gradient goes to that sample, as torch's
// max over a dimension routes it); d loss / d b = -w rsd.  A trace with zero residual has
// e = 0 and, as in the reference, a NaN gradient.
// Least-squares mode (ADFWI_L2_SQUARED): trace loss = e / 2 and w = dt, the objective
// 1/2 sum (n - b)^2 dt, whose gradient is defined on every trace (no counterpart in the
// reference's misfit set).
//
// One workgroup per shot and RW receivers; its threads take RW receivers times 1024 / RW samples
// side by side and step through time together.  Three passes over the traces: the maximum, the
// residual energy and sum rsd * a, then the gradients; partial maxima and sums are combined through
// shuffles and LDS in a fixed order (of equal maxima the first in time wins), so results do not
// depend on timing.
//
// Bound by reading a three times and b twice; the workgroups in flight together hold few enough
// traces for the later passes to come from the caches.  Eight loads in flight per thread; one lane
// per trace and eighth of the time axis, as before, kept 240 to 700 workgroups of 512 threads waiting
// on four.  us with normalisation, before -> now: 24 shots, 2000 samples, 601 receivers 237 -> 131
// (72 for reading both records and writing the gradient once at 4.8 TB/s); 64 x 3000 x 700 774 -> 714;
// 4 x 1500 x 101 74 -> 11; 1 x 1000 x 200 64 -> 10.
#include <hip/hip_runtime.h>

#include "adfwi_amd.h"
#include "common.hpp"

namespace {

constexpr int NT = 1024;       // threads per workgroup
constexpr int NW = NT / 64;

// x / b from rb = 1.0 / (double)b, for quotients of 2^-126 and more bit for bit: rb and the product are
// within 2^-53 of their exact values, relatively, and a quotient of two floats lies at least 2^-49 of its
// size from any value halfway between two floats.  (Below 2^-126 a quotient can lie on one, and may round
// to the other side.)  Three operations against the division's ten.
__device__ __forceinline__ float quot(float x, double rb) { return (float)((double)x * rb); }

template <int RW>
__global__ __launch_bounds__(NT) void trace_l2(const float *__restrict__ a, const float *__restrict__ b,
                                               int nt, int R, float dt, int normalize, int squared,
                                               float *__restrict__ loss,
                                               float *__restrict__ ga, float *__restrict__ gb) {
  constexpr int TR = NT / RW;   // time samples side by side
  __shared__ float part_m[NW][RW], part_e[NW][RW], part_q[NW][RW];
  __shared__ int part_t[NW][RW];
  const int wv = threadIdx.x >> 6, rl = threadIdx.x % RW, tr = threadIdx.x / RW;
  const int ngr = (R + RW - 1) / RW;
  // neighbouring receivers share cache lines: an XCD takes a contiguous run of the groups
  const int n = (int)gridDim.x, xcd = (int)blockIdx.x & 7, per = n >> 3, rem = n & 7;
  const int blk = xcd * per + min(xcd, rem) + ((int)blockIdx.x >> 3);
  const int s = blk / ngr, r = (blk - s * ngr) * RW + rl;
  const bool act = r < R;   // lanes past the last receiver only take part in the reductions
  const int t_end = act ? nt : 0;
  const long long base = (long long)s * nt * R + r;
  float m = 1.0f;
  int tstar = 0;
  if (normalize) {
    float lm = -1.0f;
    int lt = 0;
#pragma unroll 8
    for (int t = tr; t < t_end; t += TR) {
      const float v = fabsf(a[base + (long long)t * R]);
      if (v > lm) { lm = v; lt = t; }
    }
    // the largest, of equal ones the first in time
    auto take = [](float v, int t, float &m, int &ts) {
      if (v > m || (v == m && t < ts)) { m = v; ts = t; }
    };
#pragma unroll
    for (int o = RW; o < 64; o <<= 1) take(__shfl_xor(lm, o, 64), __shfl_xor(lt, o, 64), lm, lt);
    part_m[wv][rl] = lm;
    part_t[wv][rl] = lt;
    __syncthreads();
    m = part_m[0][rl];
    tstar = part_t[0][rl];
    for (int k = 1; k < NW; ++k) take(part_m[k][rl], part_t[k][rl], m, tstar);
  }
  const double rm = 1.0 / (double)m;
  float e = 0.0f, q = 0.0f;
#pragma unroll 8
  for (int t = tr; t < t_end; t += TR) {
    const long long i = base + (long long)t * R;
    const float av = a[i];
    const float n = normalize ? quot(av, rm) : av;
    const float rsd = n - b[i];
    e += (rsd * rsd) * dt;
    q += rsd * av;
  }
#pragma unroll
  for (int o = RW; o < 64; o <<= 1) {
    e += __shfl_xor(e, o, 64);
    q += __shfl_xor(q, o, 64);
  }
  part_e[wv][rl] = e;
  part_q[wv][rl] = q;
  __syncthreads();
  e = 0.0f;
  q = 0.0f;
  for (int k = 0; k < NW; ++k) {
    e += part_e[k][rl];
    q += part_q[k][rl];
  }
  const float root = sqrtf(e);
  if (act && tr == 0) loss[(long long)s * R + r] = squared ? 0.5f * e : root;
  if (!ga && !gb) return;
  const float w = squared ? dt : dt / root;
#pragma unroll 8
  for (int t = tr; t < t_end; t += TR) {
    const long long i = base + (long long)t * R;
    const float av = a[i];
    const float n = normalize ? quot(av, rm) : av;
    const float g = w * (n - b[i]);
    if (ga) {
      float v = normalize ? quot(g, rm) : g;
      if (normalize && t == tstar) {
        const float sg = av > 0.0f ? 1.0f : (av < 0.0f ? -1.0f : 0.0f);
        v = v - sg * ((w * q) / (m * m));
      }
      ga[i] = v;
    }
    if (gb) gb[i] = -g;
  }
}

}  // namespace

extern "C" int adfwi_trace_l2(const float *a, const float *b, int32_t nshots, int32_t nt, int32_t nrec, float dt,
                              int32_t flags, float *trace_loss, float *grad_a, float *grad_b,
                              adfwi_stream_t stream) {
  if (int rc = adfwi::fault_injected("adfwi_trace_l2")) return rc;
  ADFWI_CHECK_ARG(a && b && trace_loss, "null record or trace-loss pointer");
  ADFWI_CHECK_ARG(nshots >= 1 && nt >= 1 && nrec >= 1, "record shape %d x %d x %d invalid", nshots, nt, nrec);
  ADFWI_CHECK_ARG(dt > 0.0f, "dt must be positive (got %g)", (double)dt);
  ADFWI_CHECK_ARG((flags & ~(ADFWI_L2_NORMALIZE | ADFWI_L2_SQUARED)) == 0, "unknown flags 0x%x", flags);
  // Receivers per workgroup: the fewest that leave at most two workgroups per CU (a trace's samples
  // are then spread over the most threads), else 32: rows of 128 bytes.  Measured, us for 64 / 32 /
  // 16 / 8: 1 shot x 1000 samples x 200 receivers 33 / 18 / 12 / 10; 10 x 2000 x 50 52 / 30 / 23 / 15;
  // 24 x 2000 x 601 144 / 131 / 156 / 224; 32 x 2000 x 640 204 / 189 / 210 / 297; 64 x 3000 x 700
  // 704 / 714 / 723 / 945.
  int rw = 8;
  while (rw < 32 && (long long)nshots * ((nrec + rw - 1) / rw) > 512) rw *= 2;
  const long long nblocks = (long long)nshots * ((nrec + rw - 1) / rw);
  ADFWI_CHECK_ARG(nblocks < (1LL << 31), "record shape %d x %d x %d too large for one launch", nshots, nt, nrec);
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const auto kern = rw == 8 ? trace_l2<8> : rw == 16 ? trace_l2<16> : trace_l2<32>;
  hipLaunchKernelGGL(kern, dim3((unsigned)nblocks), dim3(NT), 0, st, a, b, nt, nrec, dt,
                     (flags & ADFWI_L2_NORMALIZE) ? 1 : 0, (flags & ADFWI_L2_SQUARED) ? 1 : 0, trace_loss,
                     grad_a, grad_b);
  return adfwi::check_launch("trace_l2");
}
