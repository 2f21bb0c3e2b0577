// Fused diagonal SSM for gfx950 (the reference's per-token recurrence,
// src/pssa.rs:1131-1144, and its staged twin, src/gpu_batch.rs:392-437):
//
//   bar_a = exp(delta_ti * rate_ij),  bar_b = delta_ti * B_tj,
//   h_tij = bar_a * h_(t-1)ij + bar_b * x_ti,   y_ti = sum_j h_tij * C_tj.
//
// With lanes*d*s independent channels (6.3M at the 105M prefill shape) a
// time-sequential walk per channel is work-optimal: no scan tree, no
// materialised states.  Mapping: a workgroup owns one lane b and 64
// consecutive channels i; its four waves split a range of 4*J states j, and
// each lane of a wave keeps its J states h_ij and rates in registers for the
// whole sequence.  Per time chunk the workgroup stages delta/x (per i) and
// B/C (per j) in LDS; B_tj and C_tj are read by every lane of a wave at the
// same address (LDS broadcast).  Per element the VALU work is one multiply
// for the exponent, one v_exp_f32, one multiply and two FMAs.  The four
// waves' partial sums over j meet in LDS and are added in a fixed order.
#include "ssm.h"

#include <algorithm>

namespace pssa {

// ---------------------------------------------------------------------------
// Unpipelined variant: with MAT it also writes bar_a, bar_b and every state
// h_t (stage API, small diagnostic shapes); without MAT it serves sequences
// shorter than one pipelined chunk (single-token decode), where it runs
// exactly T steps.
constexpr int MAT_TC = 16;

template <int J, bool MAT>
__global__ __launch_bounds__(256) void ssm_materialize_kernel(SsmArgs a) {
  __shared__ float sD[MAT_TC][64];
  __shared__ float sX[MAT_TC][64];
  __shared__ float sB[MAT_TC][4 * J];
  __shared__ float sC[MAT_TC][4 * J];
  constexpr int GS = J < 16 ? J : 16;  // readout group, as in the production scan
  constexpr int NG = J / GS;
  __shared__ float sY[4 * NG][MAT_TC][64];

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int i0 = blockIdx.x * 64;
  const int b = blockIdx.y;
  const int jb = blockIdx.z * 4 * J;
  const int i = i0 + lane;
  const int jw = jb + wave * J;
  const bool ivalid = i < a.d;
  const int T = a.T, d = a.d, s = a.s;
  const size_t row0 = (size_t)b * T;
  const size_t ds = (size_t)d * s;

  float h[J], r2[J];
  float* carry = a.carry + (size_t)b * a.carry_stride;
  const CarryCol cc = carry_col(jw, i, d, s);
#pragma unroll
  for (int q = 0; q < J; ++q) {
    const int j = jw + q;
    const bool ok = ivalid && j < s;
    h[q] = ok ? carry[cc.base + q * cc.stride] : 0.0f;
    r2[q] = ok ? a.rates2[(size_t)j * d + i] : 0.0f;
  }
  if (MAT && blockIdx.z == 0 && wave == 0 && ivalid)
    for (int j = 0; j < s; ++j) a.states[(size_t)b * (T + 1) * ds + (size_t)i * s + j] = carry[carry_at(j, i, d, s)];

  for (int t0 = 0; t0 < T; t0 += MAT_TC) {
    for (int e = tid; e < MAT_TC * 64; e += 256) {
      const int tt = e >> 6, ii = e & 63;
      const int t = t0 + tt, gi = i0 + ii;
      const bool ok = t < T && gi < d;
      const size_t r = row0 + t;
      sD[tt][ii] = ok ? a.delta[r * a.ld_delta + gi] : 0.0f;
      sX[tt][ii] = ok ? a.xn[r * a.ld_x + gi] : 0.0f;
    }
    for (int e = tid; e < MAT_TC * 4 * J; e += 256) {
      const int tt = e / (4 * J), jj = e % (4 * J);
      const int t = t0 + tt, gj = jb + jj;
      const bool ok = t < T && gj < s;
      const size_t r = row0 + t;
      sB[tt][jj] = ok ? a.bproj[r * a.ld_b + gj] : 0.0f;
      sC[tt][jj] = ok ? a.cproj[r * a.ld_c + gj] : 0.0f;
    }
    __syncthreads();
    const int steps = min(MAT_TC, T - t0);
    for (int tt = 0; tt < steps; ++tt) {
      const float dl = sD[tt][lane];
      const float u = dl * sX[tt][lane];
      // Readout in the production scan's order (groups of GS states, four
      // partial sums each), so that a run of single-token steps equals one
      // prefill bit for bit.
#pragma unroll
      for (int g = 0; g < NG; ++g) {
        float yp4[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int qq = 0; qq < GS; ++qq) {
          const int q = g * GS + qq;
          const float bq = sB[tt][wave * J + q];
          const float ab = __builtin_amdgcn_exp2f(dl * r2[q]);
          h[q] = fmaf(ab, h[q], u * bq);
          yp4[qq & 3] = fmaf(h[q], sC[tt][wave * J + q], yp4[qq & 3]);
          const int j = jw + q;
          if (MAT && ivalid && j < s) {
            const size_t c = (size_t)i * s + j;
            const size_t base = (size_t)b * T * ds + (size_t)(t0 + tt) * ds;
            a.bar_a[base + c] = ab;
            a.bar_b[base + c] = dl * bq;
            a.states[(size_t)b * (T + 1) * ds + (size_t)(t0 + tt + 1) * ds + c] = h[q];
          }
        }
        sY[wave * NG + g][tt][lane] = (yp4[0] + yp4[1]) + (yp4[2] + yp4[3]);
      }
    }
    __syncthreads();
    for (int e = tid; e < steps * 64; e += 256) {
      const int tt = e >> 6, ii = e & 63;
      const int gi = i0 + ii;
      if (gi < d) {
        float v = sY[0][tt][ii];
#pragma unroll
        for (int g = 1; g < 4 * NG; ++g) v += sY[g][tt][ii];
        const size_t r = row0 + t0 + tt;
        if (!MAT && a.y_part)
          a.y_part[((size_t)blockIdx.z * a.rows + r) * a.d + gi] = v;
        else if (gridDim.z > 1)
          atomicAdd(a.y + r * a.ld_y + gi, v);
        else
          a.y[r * a.ld_y + gi] = v;
      }
    }
    __syncthreads();
  }
#pragma unroll
  for (int q = 0; q < J; ++q) {
    const int j = jw + q;
    if (ivalid && j < s) carry[cc.base + q * cc.stride] = h[q];
  }
}

// ---------------------------------------------------------------------------
// One time step (decode): no staging, just the carry update.  A workgroup
// owns LPB lanes and 64 channels, and NB consecutive state blocks of 4*J
// states (four waves each); with NB covering all of d_state it also finishes
// the readout, adding the block sums in block order as the multi-block paths
// do, and writes y (and its bf16 copy) directly.  The arithmetic and the
// readout order are those of the kernels above, so a step here equals the
// same step inside a prefill bit for bit.  The traffic is the carry read and
// written once, streamed past the caches, plus the rates, which the LPB
// lanes of a workgroup share: they load from L2 once per workgroup, and the
// next lane's carry, B/C, delta and x loads are issued before this lane's
// carry stores, so the loads of consecutive lanes overlap.
template <int J, int NB, int LPB>
__global__ __launch_bounds__(NB * 256) void ssm_step_kernel(SsmArgs a) {
  constexpr int GS = J < 16 ? J : 16;
  constexpr int NG = J / GS;
  static_assert(J <= 32, "one B/C load per wave covers at most 32 states");
  __shared__ float sY[LPB][NB * 4 * NG][64];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int i0 = blockIdx.x * 64, b0 = blockIdx.y * LPB;
  const int jw = blockIdx.z * NB * 4 * J + wave * J;
  const int i = i0 + lane;
  const bool ivalid = i < a.d;
  const int d = a.d, s = a.s;
  const int jb = jw + (lane & 31);
  // One lane's step inputs: the wave's B values (lanes 0..J-1) and C values
  // (lanes 32..32+J-1) in one load, broadcast with readlane; delta, the
  // input term u = delta * x and the J carries.
  struct LaneIn {
    float h[J];
    float bc, dl, u;
  };
  auto load_lane = [&](int b, LaneIn& L) {
    const size_t r = b;  // T == 1: lane b's row
    const float* carry = a.carry + (size_t)b * a.carry_stride;
    L.bc = 0.0f;
    if ((lane & 31) < J && jb < s) L.bc = lane < 32 ? a.bproj[r * a.ld_b + jb] : a.cproj[r * a.ld_c + jb];
    L.dl = ivalid ? a.delta[r * a.ld_delta + i] : 0.0f;
    L.u = L.dl * (ivalid ? a.xn[r * a.ld_x + i] : 0.0f);
#pragma unroll
    for (int q = 0; q < J; ++q) {
      const int j = jw + q;
      L.h[q] = (ivalid && j < s) ? __builtin_nontemporal_load(&carry[carry_at(j, i, d, s)]) : 0.0f;
    }
  };
  float r2[J];
  LaneIn cur, nxt;
  load_lane(b0, cur);
#pragma unroll
  for (int q = 0; q < J; ++q) {
    const int j = jw + q;
    r2[q] = (ivalid && j < s) ? a.rates2[(size_t)j * d + i] : 0.0f;
  }
#pragma unroll
  for (int l = 0; l < LPB; ++l) {
    const int b = b0 + l;
    if (b >= a.lanes) break;  // uniform over the workgroup
    LaneIn& L = (l & 1) ? nxt : cur;
    LaneIn& N = (l & 1) ? cur : nxt;
    if (l + 1 < LPB && b + 1 < a.lanes) load_lane(b + 1, N);
    float* carry = a.carry + (size_t)b * a.carry_stride;
    const int bc_bits = __float_as_int(L.bc);
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      float yp4[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int qq = 0; qq < GS; ++qq) {
        const int q = g * GS + qq;
        const int j = jw + q;
        const float bq = __int_as_float(__builtin_amdgcn_readlane(bc_bits, q));
        const float cq = __int_as_float(__builtin_amdgcn_readlane(bc_bits, 32 + q));
        const float ab = __builtin_amdgcn_exp2f(L.dl * r2[q]);
        const float hv = fmaf(ab, L.h[q], L.u * bq);
        yp4[qq & 3] = fmaf(hv, cq, yp4[qq & 3]);
        if (ivalid && j < s) __builtin_nontemporal_store(hv, &carry[carry_at(j, i, d, s)]);
      }
      sY[l][wave * NG + g][lane] = (yp4[0] + yp4[1]) + (yp4[2] + yp4[3]);
    }
  }
  __syncthreads();
  // Wave l finishes lane b0 + l's readout (LPB <= NB * 4 waves).
  static_assert(LPB <= NB * 4, "one wave per lane for the readout");
  const int b = b0 + wave;
  if (wave < LPB && b < a.lanes && ivalid) {
    const size_t r = b;
    float v = 0.0f;
#pragma unroll
    for (int blk = 0; blk < NB; ++blk) {
      float bv = sY[wave][blk * 4 * NG][lane];
#pragma unroll
      for (int g = 1; g < 4 * NG; ++g) bv += sY[wave][blk * 4 * NG + g][lane];
      v = blk == 0 ? bv : v + bv;
    }
    if (a.y_part) {
      a.y_part[((size_t)blockIdx.z * a.rows + r) * a.d + i] = v;
    } else if (gridDim.z > 1) {
      atomicAdd(a.y + r * a.ld_y + i, v);
    } else {
      a.y[r * a.ld_y + i] = v;
      if (a.y16) a.y16[r * a.ld_y16 + i] = bf16_bits_dev(v);
    }
  }
}

// ---------------------------------------------------------------------------
// Production scan.  The next TC time steps' inputs are fetched into registers
// while the current TC steps run out of LDS, so the global-memory latency of
// the staging hides behind the recurrence.  Time steps past the end of a lane
// read delta = x = 0: the update is then h <- exp2(0) h + 0 = h, so whole
// chunks run unguarded and only the stores check t < T.  Per state the inner
// loop batches GS independent exponentials before the dependent FMAs.
//
// NW waves of J states each cover one state block of NW*J states (128 for
// J >= 32 with four waves and J = 16 with eight).  Every variant sums the
// readout in the same order (readout_group_size): per group of GS states four
// partial sums over j = p (mod 4), combined as (p0 + p1) + (p2 + p3), then the
// group sums of the block added one after another in state order.  The
// variant can therefore be chosen by occupancy alone without changing a bit
// of the result, and a run of single-token steps still equals one prefill.
#ifndef PSSA_SSM_TC
#define PSSA_SSM_TC 4
#endif
constexpr int SSM_TC = PSSA_SSM_TC;

// SPANS: the lanes have spans (of the full-batch prefill's scan, whose loop is
// sensitive to every register, a build of its own: 0.5% of the pass).
template <int J, int NW, int WPE, bool SPANS>
__global__ __launch_bounds__(NW * 64) __attribute__((amdgpu_waves_per_eu(WPE))) void ssm_scan_kernel(SsmArgs a) {
  // Steps staged per chunk: with few states per lane a chunk's compute is
  // short, so 16 steps stand between a chunk's input loads and their use.
  constexpr int TC = J <= 8 ? 4 * SSM_TC : SSM_TC;
  constexpr int NT = NW * 64;
  constexpr int GS = J < 16 ? J : 16;        // states per readout group
  constexpr int NG = J / GS;                 // readout groups per wave
  constexpr int SB = NW * J;                 // states per block
  constexpr int NDX = (TC * 64 + NT - 1) / NT;  // delta/x values staged per thread
  constexpr int NBC = (TC * SB + NT - 1) / NT;  // B/C values staged per thread
  __shared__ float sD[TC][64];
  __shared__ float sX[TC][64];
  __shared__ __attribute__((aligned(16))) float sB[TC][SB];
  __shared__ __attribute__((aligned(16))) float sC[TC][SB];
  __shared__ float sY[NW * NG][TC][64];

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int i0 = blockIdx.x * 64;
  const int b = blockIdx.y;
  const int jb = blockIdx.z * SB;
  const int i = i0 + lane;
  const int jw = jb + wave * J;
  const bool ivalid = i < a.d;
  const int T = SPANS ? a.spans[3 * b + 1] : a.T, d = a.d, s = a.s;
  const size_t row0 = SPANS ? (size_t)a.spans[3 * b] : (size_t)b * T;

  float h[J], r2[J];
  float* carry = a.carry + (size_t)(SPANS ? a.spans[3 * b + 2] : b) * a.carry_stride;
  const CarryCol cc = carry_col(jw, i, d, s);
#pragma unroll
  for (int q = 0; q < J; ++q) {
    const int j = jw + q;
    const bool ok = ivalid && j < s;
    h[q] = ok ? carry[cc.base + q * cc.stride] : 0.0f;
    r2[q] = ok ? a.rates2[(size_t)j * d + i] : 0.0f;
  }

  float pd[NDX], px[NDX], pb[NBC], pc[NBC];
  auto load = [&](int t0) {
#pragma unroll
    for (int k = 0; k < NDX; ++k) {
      const int e = tid + NT * k;
      const int t = t0 + (e >> 6), gi = i0 + (e & 63);
      const bool ok = e < TC * 64 && t < T && gi < d;
      const size_t r = row0 + t;
      pd[k] = ok ? a.delta[r * a.ld_delta + gi] : 0.0f;
      px[k] = ok ? a.xn[r * a.ld_x + gi] : 0.0f;
    }
#pragma unroll
    for (int k = 0; k < NBC; ++k) {
      const int e = tid + NT * k;
      const int t = t0 + e / SB, gj = jb + e % SB;
      const bool ok = e < TC * SB && t < T && gj < s;
      const size_t r = row0 + t;
      pb[k] = ok ? a.bproj[r * a.ld_b + gj] : 0.0f;
      pc[k] = ok ? a.cproj[r * a.ld_c + gj] : 0.0f;
    }
  };
  auto store = [&]() {
#pragma unroll
    for (int k = 0; k < NDX; ++k) {
      const int e = tid + NT * k;
      if (e < TC * 64) {
        sD[e >> 6][e & 63] = pd[k];
        sX[e >> 6][e & 63] = px[k];
      }
    }
#pragma unroll
    for (int k = 0; k < NBC; ++k) {
      const int e = tid + NT * k;
      if (e < TC * SB) {
        sB[e / SB][e % SB] = pb[k];
        sC[e / SB][e % SB] = pc[k];
      }
    }
  };

  load(0);
  store();
  __syncthreads();
  for (int t0 = 0; t0 < T; t0 += TC) {
    if (t0 + TC < T) load(t0 + TC);
    if constexpr (J <= 8) {
      // Few states per lane (small d_state, where a grid of few lanes is
      // bound by the step chain): per four steps the exponentials and input
      // terms first, all independent of h, then the recurrence and readout.
      // The same operations as below (one readout group), so the same bits.
      for (int t4 = 0; t4 < TC; t4 += 4) {
        float ab[4][J], ub[4][J];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float dl = sD[t4 + i][lane];
          const float u = dl * sX[t4 + i][lane];
          const float* bt = &sB[t4 + i][wave * J];
#pragma unroll
          for (int q = 0; q < J; ++q) {
            ab[i][q] = __builtin_amdgcn_exp2f(dl * r2[q]);
            ub[i][q] = u * bt[q];
          }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float* ct = &sC[t4 + i][wave * J];
          float yp[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
          for (int q = 0; q < J; ++q) h[q] = fmaf(ab[i][q], h[q], ub[i][q]);
#pragma unroll
          for (int q = 0; q < J; ++q) yp[q & 3] = fmaf(h[q], ct[q], yp[q & 3]);
          sY[wave][t4 + i][lane] = (yp[0] + yp[1]) + (yp[2] + yp[3]);
        }
      }
    } else
    for (int tt = 0; tt < TC; ++tt) {
      const float dl = sD[tt][lane];
      const float u = dl * sX[tt][lane];
      const float* bt = &sB[tt][wave * J];
      const float* ct = &sC[tt][wave * J];
#pragma unroll
      for (int g = 0; g < NG; ++g) {
        const int g0 = g * GS;
        float ab[GS];
        float yp[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int q = 0; q < GS; ++q) ab[q] = dl * r2[g0 + q];
#pragma unroll
        for (int q = 0; q < GS; ++q) ab[q] = __builtin_amdgcn_exp2f(ab[q]);
#pragma unroll
        for (int q = 0; q < GS; ++q) h[g0 + q] = fmaf(ab[q], h[g0 + q], u * bt[g0 + q]);
#pragma unroll
        for (int q = 0; q < GS; ++q) yp[q & 3] = fmaf(h[g0 + q], ct[g0 + q], yp[q & 3]);
        sY[wave * NG + g][tt][lane] = (yp[0] + yp[1]) + (yp[2] + yp[3]);
      }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < NDX; ++k) {
      const int e = tid + NT * k;
      const int tt = e >> 6, gi = i0 + (e & 63);
      const int t = t0 + tt;
      if (e < TC * 64 && t < T && gi < d) {
        float v = sY[0][tt][e & 63];
#pragma unroll
        for (int g = 1; g < NW * NG; ++g) v += sY[g][tt][e & 63];
        const size_t r = row0 + t;
        if (a.y_part)
          a.y_part[((size_t)blockIdx.z * a.rows + r) * a.d + gi] = v;
        else if (gridDim.z > 1)
          atomicAdd(a.y + r * a.ld_y + gi, v);
        else
          a.y[r * a.ld_y + gi] = v;
      }
    }
    if (t0 + TC < T) store();
    __syncthreads();
  }
#pragma unroll
  for (int q = 0; q < J; ++q) {
    const int j = jw + q;
    if (ivalid && j < s) carry[cc.base + q * cc.stride] = h[q];
  }
}

// ---------------------------------------------------------------------------
// The scan of few lanes.  With a wave lane per channel and 16 or 32 states in
// its registers, one 105M lane is 192 waves: most SIMDs idle while each step
// of the busy ones takes 16 states' arithmetic.  Here a wave lane owns one
// channel and one of the four partial sums of a readout group (states
// p, p + 4, ... of the group's 4 * M), so one lane is 768 waves (d_state 256,
// M = 4) or 64 (the small model, M = 2) with M states' arithmetic per step.
// The partial sums meet inside the quad of neighbouring wave lanes by DPP,
// the groups of a state block in LDS, in the same order as above
// ((p0 + p1) + (p2 + p3), then group after group): the same operations on
// the same operands, so the same bits.
//
// Bound: one wave per SIMD issues a step's chain of about 28 instructions
// every ~245 cycles (105M, one lane; ~150 at the rate one wave can issue
// them), against 6 issue slots per state and step at full occupancy.  A
// workgroup's four waves own CH channels and NG = 64 / CH groups, so 192
// workgroups spread a 105M lane over the CUs.  delta and u = delta * x are
// staged as pairs; B and C as four planes (states j with j mod 4 = p), so a
// lane's M values are one LDS read and the staging stores of consecutive
// threads are consecutive; the plane pitch puts the planes' and groups'
// reads of a wave in distinct banks.  Each lane of a quad keeps the sum of
// one of four steps, so four steps are stored by one LDS write.  Measured
// against the scan above, prefill of T = 512: 105M bf16 one lane 3.95 -> 1.39
// ms (scan 265 -> 52 us per layer), four lanes 5.86 -> 2.68, eight 6.64 ->
// 4.42; small fp32 model one lane 0.387 -> 0.244 (scan 110 -> 40 us).
template <int M>
constexpr int quad_block_groups() { return M == 4 ? 8 : 4; }  // readout groups per state block (ssm_state_blocks)

template <int M, int CH, bool VEC>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3))) void ssm_quad_kernel(SsmArgs a) {
  constexpr int NW = 4, NT = NW * 64, TC = 16;
  constexpr int GS = 4 * M, GW = 16 / CH, NG = NW * GW, SB = NG * GS;
  constexpr int NGB = quad_block_groups<M>(), NB = NG / NGB;  // state blocks per workgroup
  static_assert(NB * NGB == NG, "a workgroup covers whole state blocks");
  constexpr int PL = SB / 4 + (M == 4 ? 8 : 4);   // plane pitch (floats)
  constexpr int NBC = TC * SB / 4 / NT;           // float4s of B (and C) staged per thread
  static_assert(TC % 8 == 0 && NBC * NT * 4 == TC * SB && TC * CH <= NT, "whole staging rounds");
  typedef float vm_t __attribute__((ext_vector_type(M)));
  __shared__ __attribute__((aligned(16))) float2 sU[2][TC][CH];
  __shared__ __attribute__((aligned(16))) float sB[2][TC][4 * PL];
  __shared__ __attribute__((aligned(16))) float sC[2][TC][4 * PL];
  __shared__ float sY[2][NG][TC][CH];

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int p = lane & 3, ch = (lane >> 2) & (CH - 1), g = wave * GW + lane / (4 * CH);
  const int i0 = blockIdx.x * CH, b = blockIdx.y, jb = blockIdx.z * SB;
  const int i = i0 + ch, jw = jb + g * GS + p;
  const bool ivalid = i < a.d;
  const int d = a.d, s = a.s;
  const int T = a.spans ? a.spans[3 * b + 1] : a.T;
  const size_t row0 = a.spans ? (size_t)a.spans[3 * b] : (size_t)b * T;

  float h[M], r2[M];
  float* carry = a.carry + (size_t)(a.spans ? a.spans[3 * b + 2] : b) * a.carry_stride;
#pragma unroll
  for (int m = 0; m < M; ++m) {
    const int j = jw + 4 * m;
    const bool ok = ivalid && j < s;
    h[m] = ok ? carry[carry_at(j, i, d, s)] : 0.0f;
    r2[m] = ok ? a.rates2[(size_t)j * d + i] : 0.0f;
  }

  // This thread's step and channel of a chunk (threads past TC * CH repeat
  // the first ones' loads and store nothing).
  const int ett = tid / CH % TC, eci = tid % CH;
  // Offset of row t of this lane in a matrix of leading dimension ld.
  const uint32_t r0 = (uint32_t)row0;
  auto row = [&](int t, int ld) { return (size_t)(r0 + (uint32_t)t) * (uint32_t)ld; };
  // The staged loads are unguarded (a guarded load's zero fill waits for the
  // load before it): a chunk whose channels, states and steps are all in
  // range reads at running pointers, any other at clamped addresses, masked
  // on the way to LDS.
  const bool whole = VEC && i0 + CH <= d && jb + SB <= s;  // uniform
  const float* pdp = a.delta + row(min(ett, T - 1), a.ld_delta) + min(i0 + eci, d - 1);
  const float* pxp = a.xn + row(min(ett, T - 1), a.ld_x) + min(i0 + eci, d - 1);
  const float *pbp[NBC], *pcp[NBC];
#pragma unroll
  for (int k = 0; k < NBC; ++k) {
    const int e = tid + NT * k, t = e / (SB / 4), j = jb + 4 * (e % (SB / 4));
    pbp[k] = a.bproj + row(t, a.ld_b) + j;
    pcp[k] = a.cproj + row(t, a.ld_c) + j;
  }
  const size_t sd = (size_t)TC * (uint32_t)a.ld_delta, sx = (size_t)TC * (uint32_t)a.ld_x,
               sb = (size_t)TC * (uint32_t)a.ld_b, sc = (size_t)TC * (uint32_t)a.ld_c;
  float pd, px;
  float4 pb[NBC], pc[NBC];
  // The chunk at t0; called for t0 = 0, TC, 2 TC, ... in order.
  auto load = [&](int t0) {
    if (whole && t0 + TC <= T) {
      pd = *pdp;
      px = *pxp;
      pdp += sd;
      pxp += sx;
#pragma unroll
      for (int k = 0; k < NBC; ++k) {
        pb[k] = *reinterpret_cast<const float4*>(pbp[k]);
        pc[k] = *reinterpret_cast<const float4*>(pcp[k]);
        pbp[k] += sb;
        pcp[k] += sc;
      }
      return;
    }
    {
      const int t = min(t0 + ett, T - 1), gi = min(i0 + eci, d - 1);
      pd = a.delta[row(t, a.ld_delta) + gi];
      px = a.xn[row(t, a.ld_x) + gi];
    }
#pragma unroll
    for (int k = 0; k < NBC; ++k) {
      const int e = tid + NT * k, t = min(t0 + e / (SB / 4), T - 1), j = jb + 4 * (e % (SB / 4));
      const float* br = a.bproj + row(t, a.ld_b);
      const float* cr = a.cproj + row(t, a.ld_c);
      if constexpr (VEC) {
        pb[k] = *reinterpret_cast<const float4*>(br + min(j, s - 4));
        pc[k] = *reinterpret_cast<const float4*>(cr + min(j, s - 4));
      } else {
        const int j0 = min(j, s - 1), j1 = min(j + 1, s - 1), j2 = min(j + 2, s - 1), j3 = min(j + 3, s - 1);
        pb[k] = make_float4(br[j0], br[j1], br[j2], br[j3]);
        pc[k] = make_float4(cr[j0], cr[j1], cr[j2], cr[j3]);
      }
    }
  };
  auto store = [&](int t0, int buf) {
    if (!(whole && t0 + TC <= T)) {
      const bool oku = t0 + ett < T && i0 + eci < d;
      pd = oku ? pd : 0.0f;
      px = oku ? px : 0.0f;
#pragma unroll
      for (int k = 0; k < NBC; ++k) {
        const int e = tid + NT * k, j = jb + 4 * (e % (SB / 4));
        const int n = t0 + e / (SB / 4) < T ? s - j : 0;  // states of this piece in range
        pb[k].x = n > 0 ? pb[k].x : 0.0f, pc[k].x = n > 0 ? pc[k].x : 0.0f;
        pb[k].y = n > 1 ? pb[k].y : 0.0f, pc[k].y = n > 1 ? pc[k].y : 0.0f;
        pb[k].z = n > 2 ? pb[k].z : 0.0f, pc[k].z = n > 2 ? pc[k].z : 0.0f;
        pb[k].w = n > 3 ? pb[k].w : 0.0f, pc[k].w = n > 3 ? pc[k].w : 0.0f;
      }
    }
    if (tid < TC * CH) sU[buf][ett][eci] = make_float2(pd, pd * px);
#pragma unroll
    for (int k = 0; k < NBC; ++k) {
      const int e = tid + NT * k, tt = e / (SB / 4), q = e % (SB / 4);
      float* pB = &sB[buf][tt][q];
      float* pC = &sC[buf][tt][q];
      pB[0] = pb[k].x, pB[PL] = pb[k].y, pB[2 * PL] = pb[k].z, pB[3 * PL] = pb[k].w;
      pC[0] = pc[k].x, pC[PL] = pc[k].y, pC[2 * PL] = pc[k].z, pC[3 * PL] = pc[k].w;
    }
  };
  const int nz = (s + NGB * GS - 1) / (NGB * GS);  // ssm_state_blocks(s)
  // The readout of the chunk at t0 from its groups' sums.
  auto finish = [&](int t0, int buf) {
    const int t = t0 + ett, gi = i0 + eci;
    if (tid < TC * CH && t < T && gi < d) {
      float v = 0.0f;
#pragma unroll
      for (int blk = 0; blk < NB; ++blk) {
        const int z = blockIdx.z * NB + blk;
        if (blk > 0 && z >= nz) break;
        float bv = sY[buf][blk * NGB][ett][eci];
#pragma unroll
        for (int q = 1; q < NGB; ++q) bv += sY[buf][blk * NGB + q][ett][eci];
        if (a.y_part) a.y_part[(size_t)z * a.rows * d + row(t, d) + gi] = bv;
        v = blk == 0 ? bv : v + bv;
      }
      if (!a.y_part) {
        if (gridDim.z > 1)
          atomicAdd(a.y + row(t, a.ld_y) + gi, v);
        else
          a.y[row(t, a.ld_y) + gi] = v;
      }
    }
  };
  // Four steps' inputs in registers, read from LDS a group ahead of their use.
  struct Quad {
    float2 u[4];
    vm_t b[4], c[4];
  };
  auto read = [&](Quad& q, int buf, int t4) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      q.u[k] = sU[buf][t4 + k][ch];
      q.b[k] = *reinterpret_cast<const vm_t*>(&sB[buf][t4 + k][p * PL + g * M]);
      q.c[k] = *reinterpret_cast<const vm_t*>(&sC[buf][t4 + k][p * PL + g * M]);
    }
  };
  auto steps = [&](const Quad& q, int buf, int t4) {
    float ab[4][M], ub[4][M], sum[4];
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
      for (int m = 0; m < M; ++m) {
        ab[k][m] = __builtin_amdgcn_exp2f(q.u[k].x * r2[m]);
        ub[k][m] = q.u[k].y * q.b[k][m];
      }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      float yp = 0.0f;
#pragma unroll
      for (int m = 0; m < M; ++m) h[m] = fmaf(ab[k][m], h[m], ub[k][m]);
#pragma unroll
      for (int m = 0; m < M; ++m) yp = fmaf(h[m], q.c[k][m], yp);
      sum[k] = yp;
    }
    // (p0 + p1) + (p2 + p3) over the quad: quad_perm [1,0,3,2], [2,3,0,1].
#pragma unroll
    for (int k = 0; k < 4; ++k)
      sum[k] += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(sum[k]), 0xB1, 0xF, 0xF, true));
#pragma unroll
    for (int k = 0; k < 4; ++k)
      sum[k] += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(sum[k]), 0x4E, 0xF, 0xF, true));
    sY[buf][g][t4 + p][ch] = p < 2 ? (p == 0 ? sum[0] : sum[1]) : (p == 2 ? sum[2] : sum[3]);
  };

  // Chunk c computes from buffer c & 1 while the next chunk's inputs move
  // from registers to the other buffer, the one after that is loaded, and the
  // previous chunk's readout is finished: one barrier per chunk.
  load(0);
  store(0, 0);
  load(TC);
  __syncthreads();
  int buf = 0;
  for (int t0 = 0; t0 < T; t0 += TC, buf ^= 1) {
    Quad qa, qb;
    read(qa, buf, 0);
    store(t0 + TC, buf ^ 1);
    if (t0 > 0) finish(t0 - TC, buf ^ 1);  // before the loads: their waits count what was issued after them
    load(t0 + 2 * TC);
    // Steps past T have delta = u = 0 and leave h as it is.
    const int n = min(TC, T - t0);
    for (int t8 = 0; t8 < n; t8 += 8) {
      read(qb, buf, t8 + 4);
      __builtin_amdgcn_sched_barrier(0);
      steps(qa, buf, t8);
      read(qa, buf, (t8 + 8) & (TC - 1));
      __builtin_amdgcn_sched_barrier(0);
      steps(qb, buf, t8 + 4);
    }
    __syncthreads();
  }
  finish((T - 1) / TC * TC, buf ^ 1);
#pragma unroll
  for (int m = 0; m < M; ++m) {
    const int j = jw + 4 * m;
    if (ivalid && j < s) carry[carry_at(j, i, d, s)] = h[m];
  }
}

// y = sum over state blocks of the partial readouts, in block order.
__global__ void ssm_reduce_kernel(const float* __restrict__ part, int nz, size_t rows, int d,
                                  float* __restrict__ y, int ld_y) {
  const size_t n = rows * (size_t)d;
  for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += (size_t)gridDim.x * blockDim.x) {
    float v = part[e];
    for (int z = 1; z < nz; ++z) v += part[(size_t)z * n + e];
    y[(e / d) * ld_y + e % d] = v;
  }
}

static int pick_j(int s) { return s >= 128 ? 32 : (s >= 32 ? 8 : 2); }

bool ssm_step_writes_y(int T, int s) { return T == 1 && ssm_state_blocks(s) <= 2; }

int ssm_state_blocks(int s) {
  const int J = pick_j(s);
  return (s + 4 * J - 1) / (4 * J);
}

bool ssm_needs_zeroed_y(int s) { return ssm_state_blocks(s) == 2; }

// Workgroups at which the four-wave J = 32 scan holds three waves per SIMD on
// the 256 CUs; below that the eight-wave J = 16 variant (same state blocks,
// twice the waves, half the registers per lane) keeps the SIMDs fed.
constexpr long kScanFullGrid = 768;

// The few-lane scan (ssm_quad_kernel) up to this many of its workgroups
// beside another lane group, twice as many alone with M = 4.  Prefill of the
// 105M model, T = 512, old / quad scan: in two groups, 16 lanes (1536
// workgroups a group) 7.65 / 7.37 ms, 18 lanes 7.83 / 8.17, 24 lanes 9.28 /
// 9.93; serialised scan stage, 16 lanes (3072) 4.71 / 4.20 ms, 18 lanes
// 4.73 / 4.82.  Small model, scan stage: 64 lanes x 256 (1024) 0.120 / 0.098
// ms, 128 x 128 (2048) 0.082 / 0.098.
// Under 32 steps a workgroup's loading of its states is much of its work, and
// only grids that are resident at once (three workgroups per CU) gain: whole
// prefills of 6 lanes x 12 (1152) 0.974 / 1.035 ms, 10 x 24 (1920) 1.10 / 1.17,
// but 3 x 33 (576) 1.10 / 1.01; up to 64 the line lies between 5 x 50 (960)
// 1.22 / 1.15 and 16 x 60 (3072) 1.86 / 1.90.
// Lanes of their own lengths count as whole ones by their rows (each some 32
// steps longer, its loading of the states): a lane that ends early leaves its
// CUs to the others, and the longest one's chain is what the pass waits for.
// Ragged prefills of the 105M model, by the lanes / by the rows: one of 1000
// with 31 of 5 9.45 / 3.36 ms, with 20 of 100 10.1 / 4.35; 32 spread over 4 to
// 1024 10.7 / 6.68; 32 over 100 to 700 9.49 / 8.90.
constexpr int kQuadChannels = 8;
constexpr long kQuadMax = 1536;
static long whole_lanes(const SsmArgs& a) {
  const size_t lane = (size_t)a.T + 32;
  return (long)std::min<size_t>(a.lanes, (a.rows + 32 * (size_t)a.lanes + lane - 1) / lane);
}
static long quad_limit(const SsmArgs& a, bool four_states) {
  if (a.T < 32) return kQuadMax / 2;
  return four_states && !a.concurrent && a.T >= 64 ? 2 * kQuadMax : kQuadMax;
}

// From four workgroups per CU up to where the few-lane scan ends.  105M
// prefill, two groups / one: 4 lanes x 512 (768 workgroups) 2.65 / 2.73 ms, 8
// x 512 4.48 / 4.29, 12 x 512 5.76 / 5.47, 16 x 512 (3072) 7.33 / 7.00, 24 x
// 512 9.51 / 10.9; short prompts leave the scan less of the pass: 8 x 128 1.66
// / 1.73, 16 x 128 2.69 / 2.80.  Nine ragged prompts of up to 1000 4.39 /
// 4.19 ms.
bool ssm_one_group(int d, int s, size_t lanes, size_t max_len) {
  if (s < 128 || max_len < 256) return false;
  const size_t wgs = (size_t)((d + kQuadChannels - 1) / kQuadChannels) * lanes * ((s + 127) / 128);
  return wgs >= 1024 && wgs <= 2 * (size_t)kQuadMax;
}

// Lanes per decode-step workgroup (they share the rate loads).
#ifndef PSSA_SSM_STEP_LPB
#define PSSA_SSM_STEP_LPB 4
#endif

// The few-lane scan's grid: kQuadChannels channels and 128 (J = 32) or 64
// (J = 8) states per workgroup.  Returns its workgroups for the rule above.
template <int J>
static long quad_workgroups(const SsmArgs& a, dim3& grid) {
  constexpr int SB = J == 32 ? 128 : 64;
  grid = dim3((a.d + kQuadChannels - 1) / kQuadChannels, a.lanes, (a.s + SB - 1) / SB);
  return (long)grid.x * whole_lanes(a) * grid.z;
}

template <int J, bool SPANS>
static void launch_scan(hipStream_t stream, const SsmArgs& a, dim3 grid) {
  if constexpr (J == 32) {
    if ((long)grid.x * grid.y * grid.z < kScanFullGrid && !a.concurrent)
      ssm_scan_kernel<16, 8, 4, SPANS><<<grid, 512, 0, stream>>>(a);
    else
      ssm_scan_kernel<32, 4, 3, SPANS><<<grid, 256, 0, stream>>>(a);
  } else {
    // Few states per lane: a small model's grid of a few workgroups, each
    // bound by its step chain, so occupancy gives nothing and the register
    // budget of two waves per SIMD keeps the 16-step staging out of scratch.
    ssm_scan_kernel<J, 4, 2, SPANS><<<grid, 256, 0, stream>>>(a);
  }
}

template <int J>
static void launch_j(hipStream_t stream, const SsmArgs& a, bool mat) {
  dim3 grid((a.d + 63) / 64, a.lanes, (a.s + 4 * J - 1) / (4 * J)), qgrid;
  if (mat) {
    ssm_materialize_kernel<J, true><<<grid, 256, 0, stream>>>(a);
  } else if (a.T == 1 && !a.spans) {
    // At most one lane per wave of the workgroup (the readout's waves).
    constexpr int LPB2 = PSSA_SSM_STEP_LPB < 8 ? PSSA_SSM_STEP_LPB : 8;
    constexpr int LPB1 = PSSA_SSM_STEP_LPB < 4 ? PSSA_SSM_STEP_LPB : 4;
    if (grid.z == 2) {
      grid.z = 1;
      grid.y = (a.lanes + LPB2 - 1) / LPB2;
      ssm_step_kernel<J, 2, LPB2><<<grid, 512, 0, stream>>>(a);
    } else {
      grid.y = (a.lanes + LPB1 - 1) / LPB1;
      ssm_step_kernel<J, 1, LPB1><<<grid, 256, 0, stream>>>(a);
    }
  } else if (a.T < SSM_TC && !a.spans) {
    ssm_materialize_kernel<J, false><<<grid, 256, 0, stream>>>(a);
  } else if (J >= 8 && quad_workgroups<J>(a, qgrid) <= quad_limit(a, J == 32)) {
    constexpr int M = J == 32 ? 4 : 2;
    const bool vec = a.s % 4 == 0 && a.ld_b % 4 == 0 && a.ld_c % 4 == 0 && ((uintptr_t)a.bproj & 15) == 0 &&
                     ((uintptr_t)a.cproj & 15) == 0;
    if (vec)
      ssm_quad_kernel<M, kQuadChannels, true><<<qgrid, 256, 0, stream>>>(a);
    else
      ssm_quad_kernel<M, kQuadChannels, false><<<qgrid, 256, 0, stream>>>(a);
  } else if (a.spans) {
    launch_scan<J, true>(stream, a, grid);
  } else {
    launch_scan<J, false>(stream, a, grid);
  }
}

Status launch_ssm_scan(hipStream_t stream, const SsmArgs& a_in) {
  SsmArgs a = a_in;
  if (a.T <= 0 || a.d <= 0 || a.s <= 0 || a.lanes <= 0) return Status::Invalid("ssm: empty shape");
  const bool mat = a.bar_a && a.bar_b && a.states;
  const int nz = ssm_state_blocks(a.s);
  if (!a.spans) a.rows = (size_t)a.lanes * a.T;
  if (mat && a.spans) return Status::Invalid("ssm: the tape is written for lanes of one length");
  if (mat || nz <= 2) {
    a.y_part = nullptr;
  } else if (!a.y_part) {
    return Status::Invalid("ssm: more than two state blocks need a partial-sum buffer");
  }
  switch (pick_j(a.s)) {
    case 32:
      launch_j<32>(stream, a, mat);
      break;
    case 8:
      launch_j<8>(stream, a, mat);
      break;
    default:
      launch_j<2>(stream, a, mat);
      break;
  }
  PSSA_LAUNCH_CHECK("ssm_scan");
  if (a.y_part) {
    const size_t n = a.rows * (size_t)a.d;
    size_t g = (n + 255) / 256;
    if (g > 16384) g = 16384;
    ssm_reduce_kernel<<<(unsigned)g, 256, 0, stream>>>(a.y_part, nz, a.rows, a.d, a.y, a.ld_y);
    PSSA_LAUNCH_CHECK("ssm_reduce");
  }
  return Status::Ok();
}

__global__ void scale_kernel(const float* __restrict__ in, float* __restrict__ out, size_t n,
                             float scale) {
  size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = in[i] * scale;
}

// 32x32 tiles through LDS; blockIdx.z = matrix.
__global__ void transpose_kernel(const float* __restrict__ in, float* __restrict__ out, int rows, int cols,
                                 float scale) {
  __shared__ float tile[32][33];
  const size_t base = (size_t)blockIdx.z * rows * cols;
  const int r0 = blockIdx.y * 32, c0 = blockIdx.x * 32;
  for (int k = threadIdx.y; k < 32; k += blockDim.y) {
    const int r = r0 + k, c = c0 + threadIdx.x;
    if (r < rows && c < cols) tile[k][threadIdx.x] = in[base + (size_t)r * cols + c];
  }
  __syncthreads();
  for (int k = threadIdx.y; k < 32; k += blockDim.y) {
    const int c = c0 + k, r = r0 + threadIdx.x;
    if (r < rows && c < cols) out[base + (size_t)c * rows + r] = tile[threadIdx.x][k] * scale;
  }
}

Status launch_transpose(hipStream_t stream, const float* in, float* out, size_t count, int rows,
                        int cols, float scale) {
  if (!count || rows <= 0 || cols <= 0) return Status::Ok();
  if (count > 65535) return Status::Invalid("transpose: too many matrices");
  dim3 grid((cols + 31) / 32, (rows + 31) / 32, (unsigned)count), block(32, 8);
  transpose_kernel<<<grid, block, 0, stream>>>(in, out, rows, cols, scale);
  PSSA_LAUNCH_CHECK("transpose");
  return Status::Ok();
}

// Carries between the reference's [d, s] per matrix and the device's
// channel-blocked layout (carry_at): one 64-channel x 64-state tile per
// workgroup through LDS, so both sides move contiguous runs.
__global__ __launch_bounds__(256) void carry_convert_kernel(const float* __restrict__ in, float* __restrict__ out,
                                                            int d, int s, int to_device) {
  __shared__ float tile[64][65];
  const size_t m = blockIdx.z, ds = (size_t)d * s;
  const float* src = in + m * ds;
  float* dst = out + m * ds;
  const int i0 = blockIdx.x * 64, j0 = blockIdx.y * 64;
  const int w = min(64, d - i0), hs = min(64, s - j0);
  const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
  if (to_device) {
    for (int r = ty; r < w; r += 4)
      if (tx < hs) tile[r][tx] = src[(size_t)(i0 + r) * s + j0 + tx];
    __syncthreads();
    float* blk = dst + (size_t)i0 * s;  // the channel block's run: state j at + j * w
    for (int r = ty; r < hs; r += 4)
      if (tx < w) blk[(size_t)(j0 + r) * w + tx] = tile[tx][r];
  } else {
    const float* sb = src + (size_t)i0 * s;
    for (int r = ty; r < hs; r += 4)
      if (tx < w) tile[tx][r] = sb[(size_t)(j0 + r) * w + tx];
    __syncthreads();
    for (int r = ty; r < w; r += 4)
      if (tx < hs) dst[(size_t)(i0 + r) * s + j0 + tx] = tile[r][tx];
  }
}

Status launch_carry_convert(hipStream_t stream, const float* in, float* out, size_t count, int d, int s,
                            bool to_device) {
  if (!count || d <= 0 || s <= 0) return Status::Ok();
  for (size_t m0 = 0; m0 < count; m0 += 65535) {
    const size_t cnt = count - m0 < 65535 ? count - m0 : 65535, off = m0 * (size_t)d * s;
    dim3 grid((d + 63) / 64, (s + 63) / 64, (unsigned)cnt);
    carry_convert_kernel<<<grid, 256, 0, stream>>>(in + off, out + off, d, s, to_device ? 1 : 0);
    PSSA_LAUNCH_CHECK("carry_convert");
  }
  return Status::Ok();
}

Status launch_scale(hipStream_t stream, const float* in, float* out, size_t n, float scale) {
  if (n == 0) return Status::Ok();
  scale_kernel<<<(unsigned)((n + 255) / 256), 256, 0, stream>>>(in, out, n, scale);
  PSSA_LAUNCH_CHECK("scale");
  return Status::Ok();
}

}  // namespace pssa
