// bgemm.h — batched packed linear for gfx950: decode once, reuse across the batch. Three
// kernels by the call's rows, each a 128-row output block (the out-dim Hadamard block) x a
// block of batch columns x one k-range per workgroup, one workgroup per CU:
//   bgemm_shared_kernel 16 to 128 columns: 16 waves (12 for exact 128-column blocks), activations
//                     shared through LDS: up to 16 rows, and above where the planner's rule
//                     finds it faster (streams, trellis_amd.hip);
//   bgemm_kernel      32 or 64 columns: 8 waves, each with its own share of the k-range;
//   bgemm_wide_kernel 128 or 256 columns: 4 waves with 64 accumulator tiles each.
// In each a wave decodes a tile once, straight into the A operand of an MFMA (common.h), and
// multiplies it with every column of the block. With one k-range the workgroup applies
// y = sv * osc * Hb_n(t) itself, otherwise it stores its partial block and bfold_kernel (next
// launch) adds the slices in slice order and folds, one wave per batch column: reducing
// inside the kernel leaves the whole reduction to the last workgroup of each block, behind
// device-scope round trips, and measured slower.
//
// Measured on the Qwen3-8B block (K=3, MCG, one MI355X, weights from the last-level cache where
// they fit, in turn on one box), bgemm_shared_kernel and the streaming two:
//   gate+up, 32 / 64 / 128 rows, exact            32.6 / 42-44 / 68.2 -> 28.3 / 38.5 / 64.9 us
//   gate+up, 512 rows, exact                      229-235 -> 205-208 us
//   down, 2048 rows, exact / fp16-weight mode     438-445 / 280-289 -> 333-342 / 236-240 us
// What bounds them: the GPU's power limit sets the clock once the matrix cores work on real
// activations (gate+up at 512 rows ran at 1.56 GHz with 32x32x16 MFMAs, and at 2.33 GHz, 1.4
// times as fast, with all-zero activations), then instruction issue (a wave issues at most
// one operation per 5 cycles; decode, MFMA issue and LDS reads add up to ~1.3 times the
// matrix time of an exact 128-column block).
#pragma once

#include "common.h"

namespace trellis {

// y[b0 + b] = sv * osc * Hb_n(t[b]) for the nbv <= NB batch columns staged in LDS as
// t[b][TLS] (rows padded to TLS), summed over NR regions NR_OFF floats apart. Wave w folds
// columns w, w + WAVES, ..: all of them at once, level by level (fwht_chunks), so their
// lane exchanges overlap (one column after another, the fold of 64 columns measured ~2 us
// at the end of every batched launch); a wave's slots past nbv repeat column nbv - 1 and
// are not stored. so[h] = sv * osc of row 128 ob + min(lane + 64 h, rows - 1), loaded by
// the caller long before (cold, their load took ~1 us when the fold issued it).
template <int CB, int WAVES, int TLS, int NR, int NR_OFF, int NB>
__device__ __forceinline__ void bg_out_fold(const LinArgs& g, const LinMat& m, const float* tl,
                                            int ob, int b0, int nbv, int rows,
                                            const float (&sov)[2]) {
  constexpr int C = (NB + WAVES - 1) / WAVES;   // columns per wave
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  if (wave >= nbv) return;
  const float nrm = m.nrm_out;
  const float so[2] = {sov[0] * nrm, sov[1] * nrm};
  const FwhtLane fl = fwht_lane(lane, m.block_out);
  float lo[C], hi[C];
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const int b = min(wave + WAVES * c, nbv - 1);
    lo[c] = tl[b * TLS + lane];
    hi[c] = tl[b * TLS + lane + 64];
#pragma unroll
    for (int q = 1; q < NR; ++q) {
      lo[c] += tl[q * NR_OFF + b * TLS + lane];
      hi[c] += tl[q * NR_OFF + b * TLS + lane + 64];
    }
    if (lane >= rows) lo[c] = 0.f;
    if (lane + 64 >= rows) hi[c] = 0.f;
    if (CB == CB_1MAD) {
      lo[c] = lo[c] / 147.800537109375f;
      hi[c] = hi[c] / 147.800537109375f;
    }
  }
  fwht_chunks<C>(lo, hi, m.block_out, lane, fl);
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const int b = wave + WAVES * c;
    if (b >= nbv) break;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int rl = lane + 64 * h;
      if (rl < rows) {
        const float v = (h ? hi[c] : lo[c]) * so[h];
        const long long o = static_cast<long long>(b0 + b) * m.ldy + ob * 128 + rl;
        if (g.y_f16)
          st_wt(static_cast<_Float16*>(m.y) + o, static_cast<_Float16>(v));
        else
          st_wt(static_cast<float*>(m.y) + o, v);
      }
    }
  }
}

constexpr int BG_LDS_WORDS = 160 * 1024 / 4;

// LDS regions of bgemm_shared_kernel's epilogue sums, at most one per k-lane.
__host__ __device__ constexpr int bg_regions(int nb, int kl, int tls, int xbuf, int other) {
  const int limit = nb < 64 ? BG_LDS_WORDS / 2 : BG_LDS_WORDS, base = 2 * xbuf;
  int r = kl;
  while (r > 1 && (r * nb * tls > base ? r * nb * tls : base) + other > limit) r /= 2;
  return r;
}

// s_setprio with a value known after unrolling (the instruction takes an immediate)
__device__ __forceinline__ void setprio_n(int v) {
  if (v >= 3) __builtin_amdgcn_s_setprio(3);
  else if (v == 2) __builtin_amdgcn_s_setprio(2);
  else if (v == 1) __builtin_amdgcn_s_setprio(1);
  else __builtin_amdgcn_s_setprio(0);
}

// ---------------------------------------------------------------- shared activations
// A workgroup of 16 (or 12) waves: wave w = (band group bg = w % NG, k-lane kl = w / NG), a band group
// being BW adjacent bands; the waves of a SIMD share a band group and split every k-step's
// tiles between them (tile j of a step belongs to k-lane j % KL):
//   * the B tile of a step (xf[batch cols][KT*16] as (x, x) fp16 pairs written by
//     xfold_kernel) is loaded two steps ahead into registers by all the threads, stored
//     to one half of a double-buffered LDS area, and read by every wave: each fragment
//     serves the BW bands of each of the NG band groups; one barrier per step;
//   * each wave's packed words ride a two-step register ring and a wave-private LDS buffer
//     (for the lanes' window reads);
//   * every load is a range-checked buffer load (batch rows past the call's, tiles past the
//     matrix read zeros), so none is clamped or skipped and the waits stay exact;
//   * the B rows are padded by 8 words (a row stride of 8 mod 64 words: the fragments' reads
//     spread over the banks);
//   * the epilogue adds the k-lanes' sums into t[16 NC][128] in LDS in k-lane order.
// At 16 rows the kernels below measured slower (8B gate+up 28.9 us with 32-column
// blocks, 26.5 with this one; q/k/v 16.5 and 15.9, o 14.7 and 13.2, down 19.5 and 17.3).
//
// Waves per workgroup: 16 (four per SIMD), or 12 (three per SIMD, up to 168 registers each) for
// the exact mode's 128-column blocks, whose 8 fragments and 16 accumulators per wave (~150
// registers) do not fit a quarter of a SIMD's registers.
template <int NC, int F16> struct BgShared {
  static constexpr int WAVES = !F16 && NC == 8 ? 12 : 16;
};

template <int K, int CB, int V, int NC, int F16, bool SINGLE>
__global__ __launch_bounds__((64 * BgShared<NC, F16>::WAVES)) void bgemm_shared_kernel(LinArgs g) {
  constexpr int BG_WAVES = BgShared<NC, F16>::WAVES;
  constexpr int NWK = 8 * K;
  // tile columns per k-step: at 16 columns 16 (half the barriers of 8; the 8B gate+up group 29.1 -> 27.9 us),
  // otherwise 8 (in the fp16-weight mode a pair per k-lane), or 6 for the exact mode's 128
  // columns (two per k-lane over three k-lanes; LDS holds two B steps)
  constexpr int KT = F16 ? 8 : NC == 1 ? 16 : NC <= 4 ? 8 : 6;
  // bands per wave: at 16 columns 4 (8 k-lanes; each B fragment read from LDS feeds 4 bands: 27.8 ->
  // 26.6-27.1 us), otherwise 2
  constexpr int BW = F16 || NC > 1 ? 2 : 4;
  constexpr int NG = 8 / BW;                       // band groups of the block
  constexpr int KL = BG_WAVES / NG;                // k-lanes: waves of one band group
  // tiles per band per k-lane per step: exact mode, tiles kl, kl + KL, ...; fp16-weight
  // mode, the tile pair 2kl, 2kl + 1 (one MFMA per pair)
  constexpr int TPL = F16 ? 2 : KT / KL;
  static_assert(F16 || (KT % KL == 0 && TPL >= 1), "a tile column per k-lane per step");
  constexpr int WPT = F16 ? 8 : 16;                // B words per tile column and batch row
  constexpr int XW = KT * WPT + 8;                 // LDS words per B row (+8: bank spread)
  constexpr int NB = 16 * NC;                      // batch columns per workgroup
  constexpr int RCH = KT * WPT / 4;                // 16-byte chunks per B row per step
  constexpr int XCH = NB * RCH;                    // 16-byte B chunks per step
  constexpr int XLOADS = (XCH + 64 * BG_WAVES - 1) / (64 * BG_WAVES);
  constexpr int XBUF = NB * XW;                    // words per B buffer
  constexpr int CPT = NWK / 4;                     // 16-byte chunks per tile
  constexpr int BCH = BW * TPL * CPT;              // 16-byte chunks per wave per step
  constexpr int BLOADS = (BCH + 63) / 64;
  constexpr int BSW = BLOADS * 256;                // words per wave buffer: every lane's chunks
  static_assert(!F16 || (KT == 2 * KL && BW == 2), "fp16-weight mode: one tile pair per k-lane per step");
  // epilogue: t[NB][TLS] (rows padded like the B rows, so a fragment's float4 writes spread
  // over the banks) in NR regions NR_OFF floats apart over the B buffers (k-lanes
  // k2 .. k2 + NR - 1 add into regions 0 .. NR - 1 in round k2 / NR). As many as
  // the LDS holds, below 64 columns half of it: two workgroups fit a CU (bg_regions)
  constexpr int TLS = 136;
  constexpr int NR = bg_regions(NB, KL, TLS, XBUF, BG_WAVES * BSW);
  constexpr int NR_OFF = NB * TLS;
  constexpr int XSB = 2 * XBUF > NR * NR_OFF ? 2 * XBUF : NR * NR_OFF;
  static_assert(KL % NR == 0 && NB * TLS <= XSB && XSB + BG_WAVES * BSW <= BG_LDS_WORDS, "epilogue regions");
  __shared__ __align__(16) uint32_t xsb[XSB];
  __shared__ __align__(16) uint32_t bst[BG_WAVES * BSW];
  float* tl = reinterpret_cast<float*>(xsb);

  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int bg = wave % NG, kl = wave / NG;
  // a one-matrix launch (SINGLE) reads its matrix's fields in the first argument round
  const int mi = SINGLE ? 0 : locate_mat(g, blockIdx.x, false);
  const LinMat& m = g.m[mi];
  {
    // the matrix's fields that the set-up needs, loaded in one round (the argument segment
    // is cold; used one by one, the loads would go out in several dependent rounds)
    const int f_i0 = m.item0, f_s = m.S, f_t = m.tiles_in, f_n = m.n, f_xw = m.xfw;
    const int f_bt = g.batch, f_kr = g.kr;
    const uint32_t *f_b = m.bits, *f_xf = m.xf;
    const float *f_sv = m.sv, *f_os = m.osc;
    asm volatile("" ::"s"(f_i0), "s"(f_s), "s"(f_t), "s"(f_n), "s"(f_xw), "s"(f_bt), "s"(f_kr),
                 "s"(f_b), "s"(f_xf), "s"(f_sv), "s"(f_os));
  }
  const int local = blockIdx.x - m.item0;
  const int ncb = (g.batch + NB - 1) / NB;
  const int sl = local % m.S, obcb = local / m.S;
  const int ob = obcb / ncb, cb = obcb % ncb;
  const int b0 = cb * NB;                          // first batch row of this column block
  const int nbv = min(NB, g.batch - b0);           // valid batch columns
  const int c0 = sl * g.kr;
  const int ntl = min(g.kr, m.tiles_in - c0);
  const int nsteps = (ntl + KT - 1) / KT;
  const int rows = min(128, m.n - ob * 128);
  uint32_t* mystg = bst + wave * BSW;

  // B: rows b0 .. b0 + nbv - 1 of xf (a batch row past the call's reads zeros; columns
  // past the k-range feed only tiles that are not decoded)
  const rsrc_t r_x = make_rsrc(m.xf + static_cast<size_t>(b0) * m.xfw,
                               static_cast<unsigned>(nbv) * m.xfw * 4);
  unsigned xoff[XLOADS];
#pragma unroll
  for (int q = 0; q < XLOADS; ++q) {
    const int ch = threadIdx.x + 64 * BG_WAVES * q;
    const int n = ch / RCH, off = ch % RCH;        // batch row, 16-byte chunk of its row
    xoff[q] = ch < XCH ? static_cast<unsigned>((n * m.xfw + c0 * WPT + off * 4) * 4) : RSRC_OOB;
  }
  // packed words of the block's bands (bands past the matrix read zeros; the range stays
  // far below 4 GB whatever the matrix); lane chunk -> (band of the pair, tile of the
  // k-lane, chunk)
  const size_t blk0 = static_cast<size_t>(ob) * 8 * m.tiles_in * NWK;
  const int nbands = min(8, m.n / 16 - ob * 8);    // bands of this block in the matrix
  const rsrc_t r_b = make_rsrc(m.bits + blk0, static_cast<unsigned>(nbands * m.tiles_in * NWK * 4));
  unsigned boff[BLOADS];
#pragma unroll
  for (int q = 0; q < BLOADS; ++q) {
    const int ch = lane + 64 * q;
    const int bb = ch / (TPL * CPT), rem = ch % (TPL * CPT);
    const int t = rem / CPT, c = rem % CPT;
    const int tile = c0 + (F16 ? 2 * kl + t : kl + KL * t);
    boff[q] = ch < BCH ? static_cast<unsigned>(((BW * bg + bb) * m.tiles_in + tile) * NWK * 4 + c * 16)
                       : RSRC_OOB;
  }
  u32x4_t xr[2][XLOADS], br[2][BLOADS];
  auto load_step = [&](int s, u32x4_t (&xd)[XLOADS], u32x4_t (&bd)[BLOADS]) {
    // a step past the last reads nothing
    const unsigned sx = s < nsteps ? static_cast<unsigned>(s * KT * WPT * 4) : RSRC_OOB;
    const unsigned sb = s < nsteps ? static_cast<unsigned>(s * KT * NWK * 4) : RSRC_OOB;
#pragma unroll
    for (int q = 0; q < XLOADS; ++q)
      xd[q] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(
                                              r_x, static_cast<int>(xoff[q] + sx), 0, 0));
#pragma unroll
    for (int q = 0; q < BLOADS; ++q)
      bd[q] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(
                                              r_b, static_cast<int>(boff[q] + sb), 0, AUX_NT));
  };
  auto store_b = [&](int buf, const u32x4_t (&xd)[XLOADS]) {
#pragma unroll
    for (int q = 0; q < XLOADS; ++q) {
      const int ch = threadIdx.x + 64 * BG_WAVES * q;
      if (XCH % (64 * BG_WAVES) == 0 || ch < XCH)
        *reinterpret_cast<u32x4_t*>(xsb + buf * XBUF + (ch / RCH) * XW + (ch % RCH) * 4) = xd[q];
    }
  };

  // one k-range: the output fold's scales, loaded now so their latency hides behind the loop
  float sov[2] = {0.f, 0.f};
  if (m.S == 1) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int row = ob * 128 + min(lane + 64 * h, rows - 1);
      sov[h] = m.sv[row] * m.osc[row];
    }
  }

  const int r = lane & 15, gq = lane >> 4;
  const QuadPos qp = quad_pos_v<K, V>(r, gq);
  float4_t acc[BW][NC];
#pragma unroll
  for (int b = 0; b < BW; ++b)
#pragma unroll
    for (int c = 0; c < NC; ++c) acc[b][c] = float4_t{0.f, 0.f, 0.f, 0.f};

  load_step(0, xr[0], br[0]);
  load_step(1, xr[1], br[1]);
  store_b(0, xr[0]);
  __syncthreads();
  __builtin_amdgcn_s_setprio(3);
  // two steps per trip so the register rings keep a fixed shape; a step past the last
  // computes nothing, and its loads read nothing
  for (int s = 0; s < nsteps; s += 2) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int st = s + h;
      // this wave's packed words of step st to its LDS buffer; the B tile of step st + 1
      // (loaded a step ago) to the other buffer, whose step st - 1 every wave finished
      // before the last barrier: its stores drain while this step computes, instead of
      // all waves' stores queueing in front of the barrier; then refill the slots with
      // step st + 2 (the B part of this slot went to LDS a step earlier)
#pragma unroll
      for (int q = 0; q < BLOADS; ++q)
        *reinterpret_cast<u32x4_t*>(mystg + 4 * (lane + 64 * q)) = br[h][q];
      store_b(h ^ 1, xr[h ^ 1]);
      load_step(st + 2, xr[h], br[h]);
      if (st < nsteps) {
        const uint32_t* xb = xsb + h * XBUF + r * XW + 4 * gq;
        if constexpr (F16) {
          // the pair 2kl, 2kl + 1 of the step; past an odd last tile the second tile's
          // words decode to finite values that meet zero activations (xfold_kernel)
          if (st * KT + 2 * kl < ntl) {
            const uint32_t* p0 = mystg;                 // band 2bg: tiles 2kl, 2kl + 1
            const uint32_t* p1 = mystg + TPL * NWK;     // band 2bg + 1
            // the window words and the first two fragments are read before the decode, and
            // each later pair of fragments while the MFMAs of the pair before it run (read
            // just before its own MFMAs, each pair's LDS latency was exposed)
            const uint32_t w0a = p0[qp.wa], w0b = p0[qp.wb], w0c = p0[NWK + qp.wa], w0d = p0[NWK + qp.wb];
            const uint32_t w1a = p1[qp.wa], w1b = p1[qp.wb], w1c = p1[NWK + qp.wa], w1d = p1[NWK + qp.wb];
            constexpr int FP = NC < 2 ? NC : 2;         // fragments per group
            auto frag = [&](int c) {
              return __builtin_bit_cast(half8_t, *reinterpret_cast<const u32x4_t*>(xb + c * 16 * XW + kl * 16));
            };
            half8_t Bn[FP];
#pragma unroll
            for (int f = 0; f < FP; ++f) Bn[f] = frag(f);
            const half8_t A0 = decode_a_pair<K, CB, V>(w0a, w0b, w0c, w0d, qp.sh);
            const half8_t A1 = decode_a_pair<K, CB, V>(w1a, w1b, w1c, w1d, qp.sh);
#pragma unroll
            for (int c0 = 0; c0 < NC; c0 += FP) {
              half8_t Bc[FP];
#pragma unroll
              for (int f = 0; f < FP; ++f) Bc[f] = Bn[f];
              if (c0 + FP < NC) {
#pragma unroll
                for (int f = 0; f < FP; ++f) Bn[f] = frag(c0 + FP + f);
              }
#pragma unroll
              for (int f = 0; f < FP; ++f) {
                acc[0][c0 + f] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A0, Bc[f], acc[0][c0 + f], 0, 0, 0);
                acc[1][c0 + f] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A1, Bc[f], acc[1][c0 + f], 0, 0, 0);
              }
              setprio_n(2 - 4 * (c0 + FP) / NC);
            }
          }
        } else {
#pragma unroll
          for (int t = 0; t < TPL; ++t) {
            const int j = kl + KL * t;               // tile of the step
            if (st * KT + j < ntl) {
              // every LDS read of the tile (window words, the NC B fragments) before the
              // decode, so the fragments' latency hides behind it (read just before each
              // MFMA pair, it was exposed)
              uint32_t wa[BW], wb[BW];
#pragma unroll
              for (int b = 0; b < BW; ++b) {
                const uint32_t* tb = mystg + (b * TPL + t) * NWK;   // band BW * bg + b
                wa[b] = tb[qp.wa];
                wb[b] = tb[qp.wb];
              }
              half8_t Bf[NC];
#pragma unroll
              for (int c = 0; c < NC; ++c)
                Bf[c] = __builtin_bit_cast(half8_t, *reinterpret_cast<const u32x4_t*>(xb + c * 16 * XW + j * 16));
              // no instruction crosses this point (the scheduler would otherwise sink each
              // fragment's read back in front of its MFMAs); with 8 chunks the fragments'
              // registers would spill
              if constexpr (NC <= 4) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
              for (int b = 0; b < BW; ++b) {
                const half8_t A = decode_a<K, CB, V>(wa[b], wb[b], qp.sh);
#pragma unroll
                for (int c = 0; c < NC; ++c)
                  acc[b][c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A, Bf[c], acc[b][c], 0, 0, 0);
                setprio_n(2 - (t * BW + b) * 4 / (TPL * BW));
              }
            }
          }
        }
      }
      // every wave is done with this step's buffer, and the next step's B is stored
      __syncthreads();
      __builtin_amdgcn_s_setprio(3);
    }
  }
  __builtin_amdgcn_s_setprio(0);
  // the rings' last loads (steps past the end) are not consumed: let them land
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

  // ---- t[batch col][row] in LDS, k-lanes added in a fixed order: lane (n, gq) of band
  // b, chunk c holds rows 4gq .. 4gq + 3 (one float4)
  for (int k2 = 0; k2 < KL; k2 += NR) {
    if (kl >= k2 && kl < k2 + NR) {
      float* reg = tl + (kl - k2) * NR_OFF;
#pragma unroll
      for (int b = 0; b < BW; ++b)
#pragma unroll
        for (int c = 0; c < NC; ++c) {
          float4_t* p = reinterpret_cast<float4_t*>(&reg[(c * 16 + r) * TLS + 16 * (BW * bg + b) + 4 * gq]);
          *p = k2 == 0 ? acc[b][c] : *p + acc[b][c];
        }
    }
    __syncthreads();
  }

  if (m.S > 1) {
    // publish this slice's partial block (16-byte write-through stores); bfold_kernel adds
    // the slices and folds
    float* mypart = m.part + (static_cast<size_t>(ob * ncb + cb) * m.S + sl) * NB * 128;
    const float4_t* t4 = reinterpret_cast<const float4_t*>(tl);
    const rsrc_t r_p = make_rsrc(mypart, static_cast<unsigned>(nbv) * 512);
    for (int i = threadIdx.x; i < nbv * 32; i += 64 * BG_WAVES) {
      const int j = (i >> 5) * (TLS / 4) + (i & 31);
      float4_t v = t4[j];
#pragma unroll
      for (int q = 1; q < NR; ++q) v += t4[q * (NR_OFF / 4) + j];
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, v), r_p, i * 16, 0, AUX_SC1);
    }
    return;
  }
  bg_out_fold<CB, BG_WAVES, TLS, NR, NR_OFF, NB>(g, m, tl, ob, b0, nbv, rows, sov);
}

// The work item of a workgroup: workgroups go round the 8 XCDs, so the ones of an XCD (b % 8)
// take a contiguous run of items, in order.
__device__ __forceinline__ int xcd_item(int b, int total) {
  constexpr int XCDS = 8;
  const int q = total / XCDS, rem = total % XCDS, x = b % XCDS;
  return x * q + min(x, rem) + b / XCDS;
}

// y = sv * osc * Hb_n(t) of the nbe columns t[c] (BG_TLS floats apart, summed over NR regions
// NR_OFF floats apart) of batch rows b0 .. b0 + nbe - 1. Eight columns a wave at a time, eight
// lanes a column, 16 rows a lane: the Hadamard's levels 1 to 8 are plain adds in the lane,
// 16 to 64 butterflies over the 8 lanes (signs as in fwht_chunk, joined to the scale), the
// sums read and the rows written 16 bytes at a time. About 35 instructions a column, against
// ~70 with a column across the 64 lanes, which the waves of these kernels, one or two to a
// SIMD, issue at 5 cycles each. so = sv * osc of the lane's rows.
constexpr int BG_TLS = 132;    // floats per column of t (4 mod 64: a wave's writes spread over the banks)
template <int CB, int WAVES, int NR, int NR_OFF, int EC>
__device__ __forceinline__ void bg_fold16(const LinArgs& g, const LinMat& m, const float* tl, int ob,
                                          int b0, int nbe, int rows, const float (&so)[16]) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int l8 = lane & 7;
  const FwhtLane fl = fwht_lane(lane, 8);
  const int B = m.block_out;                    // 16 to 128
  // the sign a(l) that the butterflies leave in the lane
  const int cross = B > 64 ? 7 : B > 32 ? 3 : B > 16 ? 1 : 0;
  const float nrm = (__builtin_popcount(l8 & cross) & 1) ? -m.nrm_out : m.nrm_out;
#pragma unroll
  for (int c0 = 0; c0 < EC; c0 += 8 * WAVES) {
    const int c = c0 + 8 * wave + (lane >> 3);
    if (c0 + 8 * wave >= nbe) break;
    const float4_t* t4 = reinterpret_cast<const float4_t*>(tl + c * BG_TLS + 16 * l8);
    float v[16];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      float4_t q = t4[j];
#pragma unroll
      for (int n = 1; n < NR; ++n) q += t4[n * (NR_OFF / 4) + j];
#pragma unroll
      for (int i = 0; i < 4; ++i) v[4 * j + i] = CB == CB_1MAD ? q[i] / 147.800537109375f : q[i];
    }
#pragma unroll
    for (int d = 1; d < 16; d *= 2)
#pragma unroll
      for (int i = 0; i < 16; ++i)
        if (!(i & d)) {
          const float a = v[i], b = v[i + d];
          v[i] = a + b;
          v[i + d] = a - b;
        }
    if (B > 16)
#pragma unroll
      for (int i = 0; i < 16; i += 2) butterfly<1>(v[i], v[i + 1], fl.s1, lane);
    if (B > 32)
#pragma unroll
      for (int i = 0; i < 16; i += 2) butterfly<2>(v[i], v[i + 1], fl.s2, lane);
    if (B > 64)
#pragma unroll
      for (int i = 0; i < 16; i += 2) butterfly<4>(v[i], v[i + 1], fl.s4, lane);
#pragma unroll
    for (int i = 0; i < 16; ++i) v[i] *= so[i] * nrm;
    // rows of a band past the matrix and columns past the call's are not stored
    const bool keep = c < nbe && 16 * l8 < rows;
    const long long o = static_cast<long long>(b0 + c) * m.ldy + ob * 128 + 16 * l8;
    if (g.y_f16) {
      uint32_t h[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const half2_t p = {static_cast<_Float16>(v[2 * i]), static_cast<_Float16>(v[2 * i + 1])};
        h[i] = __builtin_bit_cast(uint32_t, p);
      }
      _Float16* y = static_cast<_Float16*>(m.y) + o;
      if (!keep) {
      } else if (m.y_words) {
#pragma unroll
        for (int i = 0; i < 2; ++i) st_wt16(y + 8 * i, u32x4_t{h[4 * i], h[4 * i + 1], h[4 * i + 2], h[4 * i + 3]});
      } else {
#pragma unroll
        for (int i = 0; i < 16; ++i) st_wt(y + i, static_cast<_Float16>(v[i]));
      }
    } else if (keep) {
      float* y = static_cast<float*>(m.y) + o;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        st_wt16(y + 4 * i, __builtin_bit_cast(u32x4_t, float4_t{v[4 * i], v[4 * i + 1], v[4 * i + 2], v[4 * i + 3]}));
    }
  }
}

// The epilogue of the kernels below: the KL k-lanes' sums meet in LDS as t[column][row], EC
// columns at a time, in NR regions (one per k-lane, or the k-lanes in KL / NR rounds), added
// in a fixed order; then the output fold, or with split-K the partial block for bfold_kernel.
// put(region, e, add) writes (adds) the calling wave's sums of the e-th EC columns. The rounds
// are separated by barriers that leave the stores in flight (lds_barrier).
template <int CB, int NC, int WAVES, int KL, int NR, class Put>
__device__ __forceinline__ void bg_epilogue(const LinArgs& g, const LinMat& m, uint32_t* lds, int kl,
                                            int ob, int cb, int sl, int rows, Put put) {
  constexpr int NB = 16 * NC, EC = NB < 64 ? NB : 64, NR_OFF = EC * BG_TLS;
  float* tl = reinterpret_cast<float*>(lds);
  const int b0 = cb * NB, ncb = (g.batch + NB - 1) / NB;
  const int nbv = min(NB, g.batch - b0);
  // one k-range: the output scales of the lane's rows (zeros past the matrix); they arrive
  // while the sums meet
  float4_t sv[4], os[4];
  if (m.S == 1) {
    const rsrc_t r_sv = make_rsrc(m.sv + ob * 128, rows * 4), r_os = make_rsrc(m.osc + ob * 128, rows * 4);
    const int o = (threadIdx.x & 7) * 64;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      sv[j] = __builtin_bit_cast(float4_t, __builtin_amdgcn_raw_buffer_load_b128(r_sv, o + 16 * j, 0, 0));
      os[j] = __builtin_bit_cast(float4_t, __builtin_amdgcn_raw_buffer_load_b128(r_os, o + 16 * j, 0, 0));
    }
  }
  lds_barrier();   // every wave is done with its ring: the sums take its place
#pragma unroll
  for (int e = 0; e < NB / EC; ++e) {
    const int nbe = min(EC, nbv - e * EC);
    if (nbe <= 0) break;
    if (e > 0) lds_barrier();
#pragma unroll
    for (int k2 = 0; k2 < KL; k2 += NR) {
      if (kl >= k2 && kl < k2 + NR) put(tl + (kl - k2) * NR_OFF, e, k2 > 0);
      lds_barrier();
    }
    if (m.S > 1) {
      // publish this slice's partial block (16-byte write-through stores)
      float* mypart = m.part + (static_cast<size_t>(ob * ncb + cb) * m.S + sl) * NB * 128 + e * EC * 128;
      const float4_t* t4 = reinterpret_cast<const float4_t*>(tl);
      const rsrc_t r_p = make_rsrc(mypart, static_cast<unsigned>(nbe) * 512);
      for (int i = threadIdx.x; i < nbe * 32; i += 64 * WAVES) {
        const int j = (i >> 5) * (BG_TLS / 4) + (i & 31);
        float4_t v = t4[j];
#pragma unroll
        for (int q = 1; q < NR; ++q) v += t4[q * (NR_OFF / 4) + j];
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, v), r_p, i * 16, 0, AUX_SC1);
      }
    } else {
      float so[16];
#pragma unroll
      for (int i = 0; i < 16; ++i) so[i] = sv[i / 4][i % 4] * os[i / 4][i % 4];
      bg_fold16<CB, WAVES, NR, NR_OFF, EC>(g, m, tl, ob, b0 + e * EC, nbe, rows, so);
    }
  }
}

// ---------------------------------------------------------------- 17 to 64 columns
// One workgroup of 8 waves (two per SIMD, up to 256 registers each) per 128-row output block
// x 32 CC batch columns x k-range, on v_mfma_f32_32x32x16_f16. A wave owns all four band
// pairs x all the columns, and a contiguous share of the k-range, so every fragment of A and
// B is used without another wave's help and nothing in the loop is shared: each wave streams
// its packed words and its B fragments from global memory straight into LDS rings of its own
// (load_lds16) and waits only for its own loads. No barrier, no staging registers, no LDS
// store.
template <int NC> struct BgShape {
  static constexpr int CC = NC / 2;             // 32-column chunks
  static constexpr int RG = 4;                  // band pairs per wave
  static constexpr int WAVES = 8;
  static constexpr int KL = 8;                  // the waves' shares of the k-range
  static constexpr int T = 4;                   // tile columns per stage of packed words
  static constexpr int PB = 4;                  // tile columns of B in flight (ring slots)
};

template <int K, int CB, int V, int NC, int F16, bool SINGLE>
__global__ __launch_bounds__(512) void bgemm_kernel(LinArgs g) {
  using Sh = BgShape<NC>;
  constexpr int CC = Sh::CC, RG = Sh::RG, KL = Sh::KL, T = Sh::T, PB = Sh::PB, WAVES = Sh::WAVES;
  constexpr int NB = 32 * CC;                   // batch columns per workgroup
  constexpr int NWK = 8 * K, CPT = 2 * K;       // words, 16-byte chunks per tile
  constexpr int BW = 2 * RG;                    // bands per wave
  constexpr int BCH = BW * T * CPT;             // chunks of a wave's stage of packed words
  constexpr int BL = (BCH + 63) / 64;           // load instructions for them
  constexpr int BST = BL * 256;                 // words of a stage slot
  constexpr int XST = CC * 256;                 // words of a B slot (one tile column)
  constexpr int RING = 2 * BST + PB * XST;
  // the exact mode: a weight's two halves side by side in one operand, against B's values
  // duplicated in registers (4 v_perm_b32 per quad, shared by the wave's four band pairs)
  constexpr bool SUM = F16 || CB == CB_1MAD;    // one fp16 per weight (1MAD: exactly)
  constexpr int NR = CC == 1 ? KL : 4, EC = NB;   // epilogue regions, columns per round
  constexpr int WORDS = WAVES * RING > NR * EC * BG_TLS ? WAVES * RING : NR * EC * BG_TLS;
  static_assert(WORDS <= BG_LDS_WORDS && KL % NR == 0, "rings and epilogue regions fit the LDS");
  static_assert(T == PB && T % 2 == 0, "static ring slots and read-ahead registers");
  static_assert(PB <= T && PB * CC + BL + CC < 64, "loads in flight");
  __shared__ __align__(16) uint32_t lds[WORDS];

  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int item = xcd_item(blockIdx.x, g.total);
  const int mi = SINGLE ? 0 : locate_mat(g, item, false);
  const LinMat& m = g.m[mi];
  {
    // the matrix's fields that the set-up needs, loaded in one round
    const int f_i0 = m.item0, f_s = m.S, f_t = m.tiles_in, f_n = m.n, f_ob = m.n_ob;
    const int f_bt = g.batch, f_kr = g.kr;
    const uint32_t *f_b = m.bits, *f_xf = m.xf;
    const float *f_sv = m.sv, *f_os = m.osc;
    asm volatile("" ::"s"(f_i0), "s"(f_s), "s"(f_t), "s"(f_n), "s"(f_ob), "s"(f_bt), "s"(f_kr),
                 "s"(f_b), "s"(f_xf), "s"(f_sv), "s"(f_os));
  }
  // items: column blocks outermost, so that the workgroups in flight on an XCD read one
  // block's activations, which its L2 then holds; then output blocks, then k-ranges
  const int local = item - m.item0;
  const int sl = local % m.S, cbob = local / m.S;
  const int cb = cbob / m.n_ob, ob = cbob % m.n_ob;
  const int rows = min(128, m.n - ob * 128);
  const int kl = wave;                          // share of the k-range
  const int ntl = min(g.kr, m.tiles_in - sl * g.kr);
  const int share = (ntl + KL - 1) / KL;
  const int j0 = sl * g.kr + kl * share;        // this wave's tile columns j0 .. j0 + nt - 1
  const int nt = min(share, ntl - kl * share);  // (none: nt <= 0)

  // ---- loads: per-lane offsets, fixed; the column's part is one add
  const size_t blk0 = static_cast<size_t>(ob) * 8 * m.tiles_in * NWK;
  const int nbands = min(8, m.n / 16 - ob * 8);  // bands of this block in the matrix
  const rsrc_t r_b = make_rsrc(m.bits + blk0, static_cast<unsigned>(nbands * m.tiles_in * NWK * 4));
  const int nch32 = (g.batch + XF_CHUNK - 1) / XF_CHUNK;
  const rsrc_t r_x = make_rsrc(reinterpret_cast<const char*>(m.xf) +
                                   static_cast<size_t>(cb) * CC * m.tiles_in * XF_FRAG,
                               static_cast<unsigned>(min(CC, nch32 - cb * CC)) * m.tiles_in * XF_FRAG);
  // packed words: chunk ch of a stage = band ch / (T CPT), then the band's T tiles in order
  unsigned boff[BL], bt[BL];
#pragma unroll
  for (int q = 0; q < BL; ++q) {
    const int ch = lane + 64 * q;
    const int bb = ch / (T * CPT), rem = ch % (T * CPT);
    bt[q] = rem / CPT;                          // tile of the stage
    boff[q] = ch < BCH ? static_cast<unsigned>((bb * m.tiles_in + j0) * NWK * 4 + rem * 16)
                       : RSRC_PAST;
  }
  uint32_t* ring = lds + wave * RING;
  const unsigned ring_base = __builtin_amdgcn_readfirstlane(lds_addr(ring));
  auto load_bits = [&](int s) {
#pragma unroll
    for (int q = 0; q < BL; ++q) {
      // tiles past the wave's share are not read
      const unsigned o = static_cast<int>(s * T + bt[q]) < nt ? boff[q] + static_cast<unsigned>(s * T * NWK * 4) : RSRC_PAST;
      load_lds16<false>(r_b, ring_base + static_cast<unsigned>((s & 1) * BST * 4 + q * 1024), o);
    }
  };
  const unsigned xcs = static_cast<unsigned>(m.tiles_in) * XF_FRAG;   // bytes per chunk
  const unsigned xoff = static_cast<unsigned>(j0) * XF_FRAG + lane * 16;
  auto load_x = [&](int c, int slot) {
    const unsigned o = c < nt ? xoff + static_cast<unsigned>(c) * XF_FRAG : RSRC_PAST;
#pragma unroll
    for (int q = 0; q < CC; ++q)
      load_lds16<false>(r_x, ring_base + static_cast<unsigned>((2 * BST + slot * XST) * 4 + q * 1024), o + q * xcs);
  };

  const int r = lane & 15, h = lane >> 5;
  const QuadPos q0 = quad_pos_v<K, V>(r, h), q1 = quad_pos_v<K, V>(r, h + 2);
  const uint32_t* wbase = ring + ((lane >> 4) & 1) * T * NWK;
  const uint32_t* xbase = ring + 2 * BST + lane * 4;
  float16_t acc[RG][CC];
#pragma unroll
  for (int p = 0; p < RG; ++p)
#pragma unroll
    for (int c = 0; c < CC; ++c)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[p][c][i] = 0.f;

  // every load that the compiler knows of has landed: it puts no wait of its own after the
  // ring's loads, which it cannot count
  __builtin_amdgcn_s_waitcnt(0 | (7 << 4) | (15 << 8));
  asm volatile("" ::: "memory");

  load_bits(0);
#pragma unroll
  for (int c = 0; c < PB; ++c) load_x(c, c);
  // a column's fragments and window words, read from LDS one column ahead of their use
  u32x4_t bx[2][CC];
  uint32_t w[2][RG][4];
  auto read_column = [&](const uint32_t* wst, int t, u32x4_t (&b)[CC], uint32_t (&v)[RG][4]) {
#pragma unroll
    for (int c = 0; c < CC; ++c)
      b[c] = *reinterpret_cast<const u32x4_t*>(xbase + t * XST + c * 256);
#pragma unroll
    for (int p = 0; p < RG; ++p) {
      const uint32_t* tp = wst + (2 * p * T + t) * NWK;
      v[p][0] = tp[q0.wa];
      v[p][1] = tp[q0.wb];
      v[p][2] = tp[q1.wa];
      v[p][3] = tp[q1.wb];
    }
  };
  auto compute = [&](const u32x4_t (&b)[CC], const uint32_t (&v)[RG][4]) {
    if constexpr (SUM) {
#pragma unroll
      for (int p = 0; p < RG; ++p) {
        uint32_t p0[4], p1[4];
        decode_lcg<K, CB, V>(v[p][0], v[p][1], q0.sh, p0);
        decode_lcg<K, CB, V>(v[p][2], v[p][3], q1.sh, p1);
        const half8_t A = operand_sum<CB>(p0, p1);
#pragma unroll
        for (int c = 0; c < CC; ++c)
          acc[p][c] = __builtin_amdgcn_mfma_f32_32x32x16_f16(A, __builtin_bit_cast(half8_t, b[c]), acc[p][c], 0, 0, 0);
      }
    } else {
      half8_t d0[CC], d1[CC];
#pragma unroll
      for (int c = 0; c < CC; ++c) {
        d0[c] = dup_frag(b[c], 0);
        d1[c] = dup_frag(b[c], 1);
      }
#pragma unroll
      for (int p = 0; p < RG; ++p) {
        uint32_t pv[4];
        decode_lcg<K, CB, V>(v[p][0], v[p][1], q0.sh, pv);
        const half8_t A0 = operand_pairs(pv);
#pragma unroll
        for (int c = 0; c < CC; ++c)
          acc[p][c] = __builtin_amdgcn_mfma_f32_32x32x16_f16(A0, d0[c], acc[p][c], 0, 0, 0);
        decode_lcg<K, CB, V>(v[p][2], v[p][3], q1.sh, pv);
        const half8_t A1 = operand_pairs(pv);
#pragma unroll
        for (int c = 0; c < CC; ++c)
          acc[p][c] = __builtin_amdgcn_mfma_f32_32x32x16_f16(A1, d1[c], acc[p][c], 0, 0, 0);
      }
    }
  };
  // loads land in issue order: column 0's fragments (and stage 0's words before them) have
  // landed when at most the other PB - 1 columns' are outstanding
  wait_vmcnt<(PB - 1) * CC>();
  asm volatile("" ::: "memory");
  read_column(wbase, 0, bx[0], w[0]);
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  const int nst = (nt + T - 1) / T;
  for (int s = 0; s < nst; ++s) {
    // a SIMD issues from its older wave first: each wave's priority falls as its share is
    // done, so that the two finish together
    setprio_n((4 * (nst - s) - 1) / nst);
#pragma unroll
    for (int t = 0; t < T; ++t) {
      // the slots refilled here were read into registers in the column (the words: the stage)
      // before, and those reads have returned
      if (t == 0) load_bits(s + 1);
      load_x(s * T + t + PB, t);
      // after the next column's fragments (and its stage's words before them) came PB - 1
      // columns of fragments and, up to column PB - 2, the next stage's words
      if (t + 1 < PB)
        wait_vmcnt<(PB - 1) * CC + BL>();
      else
        wait_vmcnt<(PB - 1) * CC>();
      asm volatile("" ::: "memory");
      read_column(wbase + ((t + 1 < T ? s : s + 1) & 1) * BST, (t + 1) % T, bx[(t + 1) & 1], w[(t + 1) & 1]);
      if (s * T + t < nt) compute(bx[t & 1], w[t & 1]);
      // every LDS read of the slots has returned before they are refilled
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
  }
  __builtin_amdgcn_s_setprio(0);
  // the rings' last loads (past the wave's share) are not consumed: let them land
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  // ---- t[column][row] in LDS: lane (n, h) of band pair p, chunk c holds rows 8 q + 4 h + i of
  // the pair in acc[4 q + i]
  const int col = lane & 31;
  bg_epilogue<CB, NC, WAVES, KL, NR>(g, m, lds, kl, ob, cb, sl, rows, [&](float* reg, int e, bool add) {
#pragma unroll
    for (int p = 0; p < RG; ++p)
#pragma unroll
      for (int c = 0; c < EC / 32; ++c)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          float4_t* d = reinterpret_cast<float4_t*>(&reg[(c * 32 + col) * BG_TLS + 32 * p + 8 * q + 4 * h]);
          const float16_t& a = acc[p][e * (EC / 32) + c];
          const float4_t v = {a[4 * q], a[4 * q + 1], a[4 * q + 2], a[4 * q + 3]};
          *d = add ? *d + v : v;
        }
  });
}

// ---------------------------------------------------------------- more than 64 columns
// One workgroup of 4 waves (one per SIMD, up to 512 registers each) per 128-row output block x
// NB = 16 NC batch columns x k-range, on v_mfma_f32_16x16x32_f16 over tile pairs. The GPU's
// power limit sets the clock here (1.6 to 1.9 GHz with the matrix cores busy; loops of MFMAs
// alone hold 1920 TFLOP/s with this shape and 1690 with 32x32x16), so the kernel is built to
// move and recompute little: a wave holds 64 accumulator tiles, 8 bands x 128 columns with a
// quarter of the k-range, or 4 bands x 256 columns with half of it, so a fragment of B read
// from LDS serves 8 or 4 bands, a decoded operand 8 or 16 column chunks, and no fragment of
// B or word of the stream is read twice by a wave. As above, every wave streams into rings
// of its own and no barrier is in the loop.
template <int NC> struct BgWide {
  static constexpr int WAVES = 4;
  static constexpr int BW = NC == 8 ? 8 : 4;    // bands per wave
  static constexpr int KL = BW / 2;             // waves that share a band, each a share of k
  static constexpr int T = 4;                   // tile columns per stage of packed words (two pairs)
  static constexpr int PB = NC == 8 ? 3 : 2;    // tile pairs of B in flight (ring slots)
  static constexpr int NS = 3;                  // stages of packed words in the ring
};

template <int K, int CB, int V, int NC, int F16, bool SINGLE>
__global__ __launch_bounds__(256) void bgemm_wide_kernel(LinArgs g) {
  using Sh = BgWide<NC>;
  constexpr int BW = Sh::BW, KL = Sh::KL, T = Sh::T, PB = Sh::PB, NS = Sh::NS, WAVES = Sh::WAVES;
  constexpr int XQ = NC / 2;                    // 32-row chunks of B
  constexpr int NWK = 8 * K, CPT = 2 * K;       // words, 16-byte chunks per tile
  constexpr int BCH = BW * T * CPT, BL = (BCH + 63) / 64, BST = BL * 256;
  constexpr int XL = 2 * XQ, XST = XL * 256;    // loads, words of a B slot (one tile pair)
  constexpr int RING = NS * BST + PB * XST;
  constexpr bool SUM = F16 || CB == CB_1MAD;    // one fp16 per weight (1MAD: exactly)
  constexpr int NR = KL, EC = 64;
  constexpr int WORDS = WAVES * RING > NR * EC * BG_TLS ? WAVES * RING : NR * EC * BG_TLS;
  static_assert(WORDS <= BG_LDS_WORDS, "rings and epilogue regions fit the LDS");
  static_assert(PB * XL + 2 * BL < 64, "loads in flight");
  __shared__ __align__(16) uint32_t lds[WORDS];

  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int item = xcd_item(blockIdx.x, g.total);
  const int mi = SINGLE ? 0 : locate_mat(g, item, false);
  const LinMat& m = g.m[mi];
  {
    // the matrix's fields that the set-up needs, loaded in one round
    const int f_i0 = m.item0, f_s = m.S, f_t = m.tiles_in, f_n = m.n, f_ob = m.n_ob;
    const int f_bt = g.batch, f_kr = g.kr;
    const uint32_t *f_b = m.bits, *f_xf = m.xf;
    const float *f_sv = m.sv, *f_os = m.osc;
    asm volatile("" ::"s"(f_i0), "s"(f_s), "s"(f_t), "s"(f_n), "s"(f_ob), "s"(f_bt), "s"(f_kr),
                 "s"(f_b), "s"(f_xf), "s"(f_sv), "s"(f_os));
  }
  // items as in bgemm_kernel
  const int local = item - m.item0;
  const int sl = local % m.S, cbob = local / m.S;
  const int cb = cbob / m.n_ob, ob = cbob % m.n_ob;
  const int rows = min(128, m.n - ob * 128);
  const int kl = wave % KL, bg = wave / KL;     // share of the k-range, band group
  const int ntl = min(g.kr, m.tiles_in - sl * g.kr);
  const int share = ((ntl + KL - 1) / KL + 1) & ~1;
  const int j0 = sl * g.kr + kl * share;        // this wave's tile columns j0 .. j0 + nt - 1
  const int nt = min(share, ntl - kl * share);  // (none: nt <= 0)

  const size_t blk0 = static_cast<size_t>(ob) * 8 * m.tiles_in * NWK;
  const int nbands = min(8, m.n / 16 - ob * 8);
  const rsrc_t r_b = make_rsrc(m.bits + blk0, static_cast<unsigned>(nbands * m.tiles_in * NWK * 4));
  const int nch32 = (g.batch + XF_CHUNK - 1) / XF_CHUNK;
  const rsrc_t r_x = make_rsrc(reinterpret_cast<const char*>(m.xf) +
                                   static_cast<size_t>(cb) * XQ * m.tiles_in * XF_FRAG,
                               static_cast<unsigned>(min(XQ, nch32 - cb * XQ)) * m.tiles_in * XF_FRAG);
  unsigned boff[BL], bt[BL];
#pragma unroll
  for (int q = 0; q < BL; ++q) {
    const int ch = lane + 64 * q;
    const int bb = ch / (T * CPT), rem = ch % (T * CPT);
    bt[q] = rem / CPT;
    boff[q] = ch < BCH ? static_cast<unsigned>(((BW * bg + bb) * m.tiles_in + j0) * NWK * 4 + rem * 16)
                       : RSRC_PAST;
  }
  uint32_t* ring = lds + wave * RING;
  const unsigned ring_base = __builtin_amdgcn_readfirstlane(lds_addr(ring));
  auto load_bits = [&](int s, int slot) {
#pragma unroll
    for (int q = 0; q < BL; ++q) {
      const unsigned o = static_cast<int>(s * T + bt[q]) < nt ? boff[q] + static_cast<unsigned>(s * T * NWK * 4) : RSRC_PAST;
      load_lds16<false>(r_b, ring_base + static_cast<unsigned>(slot * BST * 4 + q * 1024), o);
    }
  };
  const unsigned xcs = static_cast<unsigned>(m.tiles_in) * XF_FRAG;   // bytes per chunk
  const unsigned xoff = static_cast<unsigned>(j0) * XF_FRAG + lane * 16;
  // pair p's fragments: chunk q's two tile columns 1 KB apart; a pair's second column past
  // the share reads zeros, which its words (any finite weights) then meet
  auto load_x = [&](int p, int slot) {
    const unsigned o = 2 * p < nt ? xoff + static_cast<unsigned>(2 * p) * XF_FRAG : RSRC_PAST;
    const unsigned o1 = 2 * p + 1 < nt ? o : RSRC_PAST;
#pragma unroll
    for (int q = 0; q < XQ; ++q)
      load_lds16_pair(r_x, ring_base + static_cast<unsigned>((NS * BST + slot * XST) * 4 + q * 2048), o + q * xcs, o1 + q * xcs);
  };

  // lane (r, gq): row r of a band; quads h and h + 2 of the pair's tile gq / 2, h = gq % 2
  const int r = lane & 15, gq = lane >> 4, h = gq & 1;
  const QuadPos q0 = quad_pos_v<K, V>(r, h), q1 = quad_pos_v<K, V>(r, h + 2);
  const uint32_t* wbase = ring + (gq >> 1) * NWK;
  const uint32_t* xbase = ring + NS * BST + (gq >> 1) * 256 + h * 128 + r * 4;
  float4_t acc[BW][NC];
#pragma unroll
  for (int b = 0; b < BW; ++b)
#pragma unroll
    for (int c = 0; c < NC; ++c) acc[b][c] = float4_t{0.f, 0.f, 0.f, 0.f};

  __builtin_amdgcn_s_waitcnt(0 | (7 << 4) | (15 << 8));
  asm volatile("" ::: "memory");

  load_bits(0, 0);
  load_bits(1, 1);
#pragma unroll
  for (int p = 0; p < PB; ++p) load_x(p, p);
  u32x4_t bx[2][NC];
  uint32_t w[2][BW][4];
  auto read_pair = [&](int bslot, int t2, int xslot, u32x4_t (&b)[NC], uint32_t (&v)[BW][4]) {
    const uint32_t* xp = xbase + xslot * XST;
#pragma unroll
    for (int c = 0; c < NC; ++c)
      b[c] = *reinterpret_cast<const u32x4_t*>(xp + (c >> 1) * 512 + (c & 1) * 64);
    const uint32_t* wp = wbase + bslot * BST;
#pragma unroll
    for (int i = 0; i < BW; ++i) {
      const uint32_t* tp = wp + (i * T + 2 * t2) * NWK;
      v[i][0] = tp[q0.wa];
      v[i][1] = tp[q0.wb];
      v[i][2] = tp[q1.wa];
      v[i][3] = tp[q1.wb];
    }
  };
  auto compute = [&](const u32x4_t (&b)[NC], const uint32_t (&v)[BW][4]) {
    // band i + 1 is decoded between the MFMAs of band i
    half8_t hi[2], lo[2];
    auto operands = [&](int i) {
      uint32_t p0[4], p1[4];
      decode_lcg<K, CB, V>(v[i][0], v[i][1], q0.sh, p0);
      decode_lcg<K, CB, V>(v[i][2], v[i][3], q1.sh, p1);
      if constexpr (SUM)
        hi[i & 1] = operand_sum<CB>(p0, p1);
      else
        operand_planes(p0, p1, hi[i & 1], lo[i & 1]);
    };
    operands(0);
#pragma unroll
    for (int i = 0; i < BW; ++i) {
      if (i + 1 < BW) operands(i + 1);
#pragma unroll
      for (int c = 0; c < NC; ++c)
        acc[i][c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(hi[i & 1], __builtin_bit_cast(half8_t, b[c]), acc[i][c], 0, 0, 0);
      if constexpr (!SUM) {
#pragma unroll
        for (int c = 0; c < NC; ++c)
          acc[i][c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(lo[i & 1], __builtin_bit_cast(half8_t, b[c]), acc[i][c], 0, 0, 0);
      }
      if (i + 1 < BW) {
        constexpr int M = SUM ? NC : 2 * NC, VPM = (40 + M - 1) / M;
#pragma unroll
        for (int c = 0; c < M; ++c) {
          __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);     // an MFMA
          __builtin_amdgcn_sched_group_barrier(0x2, VPM, 0);   // VALU operations
        }
      }
    }
  };
  // loads land in issue order: pair 0's fragments (and stages 0 and 1 before them)
  wait_vmcnt<(PB - 1) * XL>();
  asm volatile("" ::: "memory");
  read_pair(0, 0, 0, bx[0], w[0]);
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  const int nst = (nt + T - 1) / T;
  int bs = 0, xs = 0;                           // ring slots of stage s and pair p
  for (int s = 0; s < nst; ++s) {
#pragma unroll
    for (int t2 = 0; t2 < 2; ++t2) {
      // the slots refilled here were read into registers before, and those reads returned:
      // stage s - 1's words and pair p's fragments
      if (t2 == 0) load_bits(s + 2, bs >= 1 ? bs - 1 : NS - 1);
      load_x(2 * s + t2 + PB, xs);
      // after pair p + 1's fragments (and its stage's words before them) came PB - 1 pairs of
      // fragments and a stage of words, if one was issued in the last PB - 1 pairs
      if (PB == 3 || t2 == 0)
        wait_vmcnt<(PB - 1) * XL + BL>();
      else
        wait_vmcnt<(PB - 1) * XL>();
      asm volatile("" ::: "memory");
      xs = xs + 1 < PB ? xs + 1 : 0;
      if (t2 == 1) bs = bs + 1 < NS ? bs + 1 : 0;
      read_pair(bs, (t2 + 1) & 1, xs, bx[(t2 + 1) & 1], w[(t2 + 1) & 1]);
      if (s * T + 2 * t2 < nt) compute(bx[t2], w[t2]);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  bg_epilogue<CB, NC, WAVES, KL, NR>(g, m, lds, kl, ob, cb, sl, rows, [&](float* reg, int e, bool add) {
#pragma unroll
    for (int i = 0; i < BW; ++i)
#pragma unroll
      for (int c = 0; c < EC / 16; ++c) {
        float4_t* d = reinterpret_cast<float4_t*>(&reg[(c * 16 + r) * BG_TLS + 16 * (BW * bg + i) + 4 * gq]);
        const float4_t v = acc[i][e * (EC / 16) + c];
        *d = add ? *d + v : v;
      }
  });
}

// Split-K reduction of bgemm_kernel: one wave per (matrix, 128-row block, batch column):
// it loads that column's 128 rows of every slice at once (S slices x 2 values per lane in
// flight), adds them in slice order (deterministic), and folds y = sv * osc * Hb_n(t).
// Workgroup = 4 batch columns of one (matrix, block, column block). Runs after
// bgemm_kernel (a kernel boundary), so plain loads see its partial sums.
template <int CB, int NC, bool SINGLE>
__global__ __launch_bounds__(256) void bfold_kernel(LinArgs g) {
  constexpr int NB = 16 * NC, CG = NB / 4;        // workgroups per (block, column block)
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int fi = blockIdx.x / CG, cg = blockIdx.x % CG;
  // a one-matrix launch reads its matrix's fields in the first round of argument loads
  const int mi = SINGLE ? 0 : locate_fold(g, fi);
  const LinMat& m = g.m[mi];
  const int ncb = (g.batch + NB - 1) / NB;
  const int local = fi - m.fold0;
  const int ob = local / ncb, cb = local % ncb;
  const int b0 = cb * NB, nbv = min(NB, g.batch - b0);
  const int n = cg * 4 + wave;                    // batch column of the block
  if (n >= nbv) return;
  const int rows = min(128, m.n - ob * 128);
  const int S = m.S;
  // the output scales first: their loads are in flight with the partial sums'
  float so[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int row = ob * 128 + min(lane + 64 * h, rows - 1);
    so[h] = m.sv[row] * m.osc[row];
  }
  const float* p = m.part + static_cast<size_t>(ob * ncb + cb) * S * NB * 128 + n * 128;
  float lo = 0.f, hi = 0.f;
  for (int s0 = 0; s0 < S; s0 += 8) {
    float q0[8], q1[8];
#pragma unroll
    for (int v = 0; v < 8; ++v) {
      const float* ps = p + static_cast<size_t>(min(s0 + v, S - 1)) * NB * 128;
      q0[v] = ps[lane];
      q1[v] = ps[lane + 64];
    }
#pragma unroll
    for (int v = 0; v < 8; ++v)
      if (s0 + v < S) {
        lo += q0[v];
        hi += q1[v];
      }
  }
  if (CB == CB_1MAD) {
    lo = lo / 147.800537109375f;
    hi = hi / 147.800537109375f;
  }
  fwht_chunk(lo, hi, m.block_out, lane);
  const float nrm = m.nrm_out;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int rl = lane + 64 * h;
    if (rl < rows) {
      const int row = ob * 128 + rl;
      const float v = (h ? hi : lo) * (so[h] * nrm);
      const long long o = static_cast<long long>(b0 + n) * m.ldy + row;
      if (g.y_f16)
        st_wt(static_cast<_Float16*>(m.y) + o, static_cast<_Float16>(v));
      else
        st_wt(static_cast<float*>(m.y) + o, v);
    }
  }
}

}  // namespace trellis
