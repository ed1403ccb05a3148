// encode.h — tail-biting trellis encoder (Viterbi) for gfx950: the counterpart of the
// reference's fused Triton encoder (src/trellis/viterbi_triton.py:34-129) and of
// qtip.viterbi_tb / _viterbi_pass (src/trellis/qtip.py:124-196), for L = 16, T = 256, V = 1.
//
// One 1024-thread workgroup per tile at a time (persistent over tiles):
//   * QTIP's two-pass tail-biting (qtip.py:124-144): pass 1 on the tile rolled by T/2,
//     unconstrained; the overlap (the top L-K bits of the state at rolled position T/2)
//     constrains pass 2 to start and end on that edge.
//   * A pass is the exact DP over the E = 2^(L-K) edges (state s = (q << (L-K)) | e, its
//     predecessor edge s >> K = (q << (L-2K)) | (e >> K)): the cost vector ping-pongs
//     between two LDS buffers (E floats each: 64 KB at K=2), one barrier per step. Runs of
//     2^K edges share their 2^K predecessors, so a thread owns whole runs (or, at K=4, four
//     edges of one): it reads each predecessor's cost once for all of them, and keeps the
//     codebook values of its 2^K candidate states per edge in registers (they do not depend
//     on the step).
//   * fp32 arithmetic in the reference's order without contraction, d = w - v,
//     c = d*d + cost[pred], the smallest q kept on ties, the smallest edge for the free
//     end: the same operations as the CPU restatement, so the paths agree bit for bit.
//   * The kernel is bound by the VALU's issue rate, so the step is written for its count:
//     per candidate the subtract, multiply and add, half a v_min3_f32, and one compare of
//     the candidate with the minimum. The compares' lane masks stay in scalar registers,
//     where the scalar unit (its own issue port) turns them into the bits of the smallest
//     matching q; each bit enters the backpointer word as the carry of one v_addc_co_u32.
//     4.97 VALU operations per candidate at K=3 (318 in the compiled step of 64), against
//     5.75 with a compare and two selects per candidate: 1024 tiles at K=3 MCG took 5.32 ms
//     that way, one lane walking the backpointers, and take 4.19 ms now (244 k tiles/s, the
//     VALU issuing all the time: 2 * 256 steps * 4 waves * 318 * 4 cycles = 1.09 ms per tile
//     and CU at 2.4 GHz, 1.05 measured).
//   * Backpointers (K bits per edge per step, one word per thread) go to a per-workgroup
//     workspace region; one wave walks them back, several steps per memory round trip
//     (vit_walk), then the K-bit symbols are packed into the reference's reversed stream
//     layout (scripts/export_packed.py:27-35) with LDS atomic ORs.
#pragma once

#include "common.h"

namespace trellis {

constexpr int VIT_L = 16;
constexpr int VIT_T = 256;
constexpr int VIT_THREADS = 1024;

// Workspace bytes per workgroup: one word of backpointers per thread and step.
constexpr size_t VIT_BP_BYTES = static_cast<size_t>(VIT_T) * VIT_THREADS * 4;

struct VitArgs {
  const float* w;       // [ntiles][256] targets in tile order t = (row%16)*16 + col%16
  uint32_t* bits;       // [ntiles][8K] packed symbols
  float* dq;            // [ntiles][256] codebook value of each chosen state, or null
  uint32_t* bp;         // workspace: gridDim.x regions of VIT_BP_BYTES
  uint32_t ntiles;
};

// The edges of a thread: runs of GE = min(2^K, EPT) adjacent edges with the same
// predecessors, run i of thread j starting at edge GE * (i * 1024 + j).
template <int K> struct VitEdges {
  static constexpr int Q = 1 << K;
  static constexpr int EPT = (1 << (VIT_L - K)) / VIT_THREADS;   // 16, 8, 4
  static constexpr int GE = Q < EPT ? Q : EPT;                   // 4, 8, 4
  static constexpr int NG = EPT / GE;                            // 4, 1, 1
  static_assert(EPT * K <= 32, "one backpointer word per thread and step");
};

// w = 2w + the lane's bit of `mask`, one VALU operation (the compiler makes it two, a select
// and a shift-or). The mask comes from the scalar unit, so no VALU-write hazard precedes it.
__device__ __forceinline__ uint32_t shift_in(uint32_t w, uint64_t mask) {
  asm("v_addc_co_u32_e64 %0, vcc, %0, %0, %1" : "+v"(w) : "s"(mask) : "vcc");
  return w;
}

// The bits of the smallest q whose lane-mask e[q] is set, the most significant first, shifted
// into w; a lane with no mask set among e[0 .. Q-2] takes Q - 1 (e[Q-1] is not looked at).
template <int K>
__device__ __forceinline__ uint32_t shift_in_first(uint32_t w, const uint64_t (&e)[1 << K]) {
  constexpr int Q = 1 << K;
#pragma unroll
  for (int b = K - 1; b >= 0; --b) {
    // the answer's bit b, from the last run of 2^b candidates to the first: a run with a
    // mask set decides (all of them in the same half of a run of 2^(b+1) give one value)
    uint64_t bit = ~0ull;
#pragma unroll
    for (int run = (Q >> b) - 2; run >= 0; --run) {
      uint64_t any = 0;
#pragma unroll
      for (int q = 0; q < (1 << b); ++q) any |= e[(run << b) + q];
      bit = run & 1 ? bit | any : bit & ~any;
    }
    w = shift_in(w, bit);
  }
  return w;
}

// One wave walks the backpointers from edge `e` after step T - 1 back to step `last`, writing
// states[t]. The D steps t, t-1, .., t-D+1 are read in one memory round trip: the edge that
// step t - d arrives at is one of Q^d, its low bits e >> (K d) and its top bits the d q's that
// the walk has still to learn, so lane l loads the word of candidate l of each of the D steps
// and the walk then picks its way through them by lane reads. (One lane walking one step per
// round trip took ~55 us per pass of a K=3 tile, of ~680.)
template <int K>
__device__ __forceinline__ void vit_walk(const uint32_t* bp, int32_t* states, int e, int last,
                                         int lane) {
  using Ed = VitEdges<K>;
  constexpr int L = VIT_L, Q = 1 << K, EB = L - K;     // EB: bits of an edge
  constexpr int D = K == 2 ? 4 : K == 3 ? 3 : 2;       // Q^(D-1) <= 64 candidates
  for (int t = VIT_T - 1; t >= last; t -= D) {
    uint32_t wd[D];
#pragma unroll
    for (int d = 0; d < D; ++d) {
      // candidate c of step t - d: its low K d bits are the q's of steps t .. t - d + 1, the
      // latest in the lowest bits; they enter the edge from the top
      const int c = lane & ((1 << (K * d)) - 1);
      const int ed = (e >> (K * d)) | (c << (EB - K * d));
      const int j = (ed / Ed::GE) % VIT_THREADS;
      const int step = t - d >= 0 ? t - d : 0;
      const uint32_t w = __builtin_nontemporal_load(bp + static_cast<size_t>(step) * VIT_THREADS + j);
      const int pos = (ed / Ed::GE) / VIT_THREADS * Ed::GE + ed % Ed::GE;
      wd[d] = w >> ((Ed::EPT - 1 - pos) * K);
    }
    int c = 0;
#pragma unroll
    for (int d = 0; d < D; ++d) {
      if (t - d < last) break;
      const int q = static_cast<int>(__builtin_amdgcn_readlane(wd[d], c)) & (Q - 1);
      const int s = (q << EB) | e;
      if (lane == 0) states[t - d] = s;
      e = s >> K;
      c |= q << (K * d);
    }
    e = __builtin_amdgcn_readfirstlane(e);
  }
}

template <int K, int CB>
__global__ __launch_bounds__(VIT_THREADS) void viterbi_kernel(VitArgs a) {
#pragma clang fp contract(off)
  using Ed = VitEdges<K>;
  constexpr int L = VIT_L, T = VIT_T;
  constexpr int E = 1 << (L - K), Q = 1 << K;
  constexpr int GE = Ed::GE, NG = Ed::NG;
  constexpr int NWK = 8 * K;
  __shared__ __align__(16) float cost[2][E];
  __shared__ float wseq[T];
  __shared__ int32_t states[T];
  __shared__ uint32_t packed[NWK];
  __shared__ int32_t edge_sh;
  const int tid = threadIdx.x;
  uint32_t* bp = a.bp + static_cast<size_t>(blockIdx.x) * (VIT_BP_BYTES / 4);

  // the codebook values of this thread's candidate states (independent of the step)
  float cv[NG][GE][Q];
#pragma unroll
  for (int i = 0; i < NG; ++i)
#pragma unroll
    for (int b = 0; b < GE; ++b)
#pragma unroll
      for (int q = 0; q < Q; ++q)
        cv[i][b][q] = cb_exact<CB>(cb_raw<CB>(
            static_cast<uint32_t>((q << (L - K)) | (GE * (i * VIT_THREADS + tid) + b))));

  for (uint32_t tile = blockIdx.x; tile < a.ntiles; tile += gridDim.x) {
    const float* wt = a.w + static_cast<size_t>(tile) * T;
    int overlap = -1;
    for (int pass = 0; pass < 2; ++pass) {
      // pass 0: the tile rolled by T/2 (torch.roll: wr[t] = w[(t - T/2) mod T])
      if (tid < T) wseq[tid] = pass == 0 ? wt[(tid + T / 2) % T] : wt[tid];
#pragma unroll
      for (int i = 0; i < E / VIT_THREADS; ++i) {
        const int e = i * VIT_THREADS + tid;
        cost[0][e] = overlap < 0 || e == overlap ? 0.0f : __FLT_MAX__ / 4.0f;
      }
      __syncthreads();
      int cur = 0;
      for (int t = 0; t < T; ++t) {
        const float w_t = wseq[t];
        uint32_t word = 0u;
#pragma unroll
        for (int i = 0; i < NG; ++i) {
          const int e0 = GE * (i * VIT_THREADS + tid);
          float pc[Q];
#pragma unroll
          for (int q = 0; q < Q; ++q) pc[q] = cost[cur][(q << (L - 2 * K)) | (e0 >> K)];
          float4_t out[GE / 4];
#pragma unroll
          for (int b = 0; b < GE; ++b) {
            float c[Q];
#pragma unroll
            for (int q = 0; q < Q; ++q) {
              const float d = w_t - cv[i][b][q];
              c[q] = d * d + pc[q];
            }
            // best = the smallest candidate below FLT_MAX, in pairs (v_min3_f32); a lane with
            // none (infinite or NaN targets) keeps FLT_MAX and q = 0
            float best = __FLT_MAX__;
#pragma unroll
            for (int q = 0; q < Q; q += 2) best = __builtin_fminf(__builtin_fminf(best, c[q]), c[q + 1]);
            uint64_t eq[Q];
#pragma unroll
            for (int q = 0; q < Q - 1; ++q) eq[q] = __builtin_amdgcn_ballot_w64(c[q] == best);
            eq[Q - 1] = 0;
            eq[0] |= ~__builtin_amdgcn_ballot_w64(best < __FLT_MAX__);
            out[b / 4][b % 4] = best;
            word = shift_in_first<K>(word, eq);
          }
#pragma unroll
          for (int b = 0; b < GE / 4; ++b)
            *reinterpret_cast<float4_t*>(&cost[cur ^ 1][e0 + 4 * b]) = out[b];
        }
        bp[static_cast<size_t>(t) * VIT_THREADS + tid] = word;
        __syncthreads();
        cur ^= 1;
      }
      // the final edge: the smallest-cost edge (ties: the smallest) or the overlap
      if (overlap < 0) {
        // per-thread best of its edges, then a workgroup argmin in edge order
        float best = __FLT_MAX__;
        int be = 0;
#pragma unroll
        for (int i = 0; i < E / VIT_THREADS; ++i) {
          const int e = i * VIT_THREADS + tid;
          const float c = cost[cur][e];
          if (c < best || (c == best && e < be)) {
            best = c;
            be = e;
          }
        }
        __syncthreads();   // every thread has read the final costs
        // reduce (cost, edge) pairs through the now-free other buffer
        float* rc = cost[cur ^ 1];
        int32_t* re = reinterpret_cast<int32_t*>(cost[cur ^ 1] + VIT_THREADS);
        rc[tid] = best;
        re[tid] = be;
        __syncthreads();
        for (int s = VIT_THREADS / 2; s > 0; s >>= 1) {
          if (tid < s) {
            const float c2 = rc[tid + s];
            const int e2 = re[tid + s];
            if (c2 < rc[tid] || (c2 == rc[tid] && e2 < re[tid])) {
              rc[tid] = c2;
              re[tid] = e2;
            }
          }
          __syncthreads();
        }
        if (tid == 0) edge_sh = re[0];
      } else if (tid == 0) {
        edge_sh = overlap;
      }
      // the barrier makes every thread's backpointer stores visible to the walking wave;
      // the first pass is walked only to the state at T/2, the overlap
      __syncthreads();
      if (tid < 64) vit_walk<K>(bp, states, __builtin_amdgcn_readfirstlane(edge_sh), pass == 0 ? T / 2 : 0, tid);
      __syncthreads();
      if (pass == 0) overlap = states[T / 2] >> K;
    }
    // pass 2's states: symbols packed reversed (symbol t at stream bits (255-t)*K), and
    // the dequantized values
    if (tid < NWK) packed[tid] = 0u;
    __syncthreads();
    if (tid < T) {
      const uint32_t sym = static_cast<uint32_t>(states[tid]) & ((1u << K) - 1u);
      const int p = (T - 1 - tid) * K;
      atomicOr(&packed[p >> 5], sym << (p & 31));
      if ((p & 31) + K > 32) atomicOr(&packed[(p >> 5) + 1], sym >> (32 - (p & 31)));
      if (a.dq)
        a.dq[static_cast<size_t>(tile) * T + tid] =
            cb_exact<CB>(cb_raw<CB>(static_cast<uint32_t>(states[tid])));
    }
    __syncthreads();
    if (tid < NWK) a.bits[static_cast<size_t>(tile) * NWK + tid] = packed[tid];
    __syncthreads();
  }
}

}  // namespace trellis
