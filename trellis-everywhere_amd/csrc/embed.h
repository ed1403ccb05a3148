// embed.h — embedding-row lookup from a packed trellis matrix with the full restore:
// out[t, j] = W_hat[tok[t], j] (web/kernels.js:192-249 DECODE_EMBED, web/packed.js:137-146).
//
// W_hat[r, j] = sv[r] osc[r] su[j] isc_scaled[j] / sqrt(B_n B_k)
//               * sum_l H_k[j % B_k, l] * sum_c H_n[r % B_n, c] * zq[rb + c, jb + l]
// (rb, jb: first row / column of r's and j's Hadamard blocks; H entries (-1)^popcount(a&b)).
// The two Hadamard sums commute, so every weight of the B_n x B_k block is decoded once
// per (token, column block): one workgroup per (token, column block), 4 waves.
//   * wave w takes the tile columns 2w, 2w + 1 of the block (of 4 or fewer, column w) in all of
//     its bands, so it holds 8 column sums per lane group and no other wave adds to them; it
//     loads its tiles' packed words as 16-byte chunks into a wave-private LDS buffer (one
//     chunk per lane and load), then lane (row rl = l / 4, column group g = l % 4) decodes 4
//     weights of each tile (the same window/codebook code as the matmul kernels) and
//     accumulates sign(rr, 16b + rl) * w per column. MCG/3INST: one v_dot2_f32_f16 of the raw
//     (hi, lo) fp16 pair with (sign, sign) per weight (the products are exact; hi + lo is the
//     reference's exact fp32 sum); 1MAD: the integer (y - 510) * sign, exact in fp32, divided
//     by 147.800537109375 once per output. The sums, too, are exact (multiples of 2^-13 below
//     2^9), whatever their order;
//   * the 16 rows are summed two values at a time: a permlane swap of two values and one add
//     halve both the lanes and the values that are left (levels 32 and 16), then DPP moves.
//     Bound: VALU, ~69 cycles per tile and SIMD for decode and dot products (36 of the 47 us of
//     512 rows of a K=4 table 4096 wide). With two bands of all 8 tile columns per wave (32 sums
//     a lane, all-reduced by DPP) the reduction cost as much again: 71.5 us;
//   * wave 0 applies the column-side Hadamard (fwht_chunk) and the scales.
// A token id outside [0, n_out) yields a row of zeros.
#pragma once

#include "common.h"

namespace trellis {

struct EmbedArgs {
  const uint32_t* bits;
  const float* su;
  const float* sv;
  const float* isc;     // isc_scaled = f32(isc) * scale
  const float* osc;
  const int32_t* tokens;
  void* out;
  long long ldo;
  int n, k, tiles_in, block_in, block_out, nblk;   // nblk = k / block_in
  float nrm;            // 1/sqrt(block_in) * 1/sqrt(block_out), fp32
  int out_f16;
};

// For lanes l and l ^ H: a's sum in the lower of the two, b's in the upper (one permlane swap
// puts a's pair in the one and b's pair in the other).
template <int H>
__device__ __forceinline__ float swap_add(float a, float b) {
  const uint32_t ia = __builtin_bit_cast(uint32_t, a), ib = __builtin_bit_cast(uint32_t, b);
  uint32_t x, y;
  if constexpr (H == 32) {
    const auto p = __builtin_amdgcn_permlane32_swap(ia, ib, false, false);
    x = p[0];
    y = p[1];
  } else {
    static_assert(H == 16, "partner distance");
    const auto p = __builtin_amdgcn_permlane16_swap(ia, ib, false, false);
    x = p[0];
    y = p[1];
  }
  return __builtin_bit_cast(float, x) + __builtin_bit_cast(float, y);
}

template <int K, int CB, int V>
__global__ __launch_bounds__(256) void embed_kernel(EmbedArgs a) {
  constexpr int NWK = 8 * K;
  constexpr int WBUF = 2 * 8 * NWK;                 // words of two tile columns x 8 bands
  __shared__ float colsum[128];
  __shared__ __align__(16) uint32_t wbuf[4][WBUF];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int t = blockIdx.x / a.nblk, jblk = blockIdx.x % a.nblk;
  const int jb = jblk * a.block_in;                 // first column of the block
  const int tok = a.tokens[t];
  const bool ok = tok >= 0 && tok < a.n;
  const int r = ok ? tok : 0;
  const int rb = r - r % a.block_out, rr = r % a.block_out;
  const int ntc = a.block_in / 16, nbands = a.block_out / 16;
  const int rl = lane >> 2, g = lane & 3;
  const QuadPos qp = quad_pos_v<K, V>(rl, g);

  // this wave's tile columns tc0 .. tc0 + ntw - 1 of every band to LDS, [band][tile][words]
  const int per = (ntc + 3) / 4, tc0 = wave * per, ntw = min(per, ntc - tc0);
  uint32_t* mybuf = wbuf[wave];
  {
    const int cpb = per * NWK / 4;                  // 16-byte chunks per band
    const rsrc_t r_bits = make_rsrc(a.bits + static_cast<size_t>(rb / 16) * a.tiles_in * NWK,
                                    static_cast<unsigned>(nbands * a.tiles_in * NWK * 4));
#pragma unroll
    for (int q = 0; q < (WBUF / 4 + 63) / 64; ++q) {
      const int ch = lane + 64 * q;
      const int band = (per == 2 ? ch >> 1 : ch) / (NWK / 4), c = ch - band * cpb;   // per <= 2
      const bool in = ch < nbands * cpb && c < ntw * (NWK / 4);
      const unsigned off = in ? static_cast<unsigned>(((band * a.tiles_in + jb / 16 + tc0) * NWK + 4 * c) * 4)
                              : RSRC_PAST;
      const u32x4_t v = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(
                                                        r_bits, static_cast<int>(off), 0, AUX_NT));
      if (in) *reinterpret_cast<u32x4_t*>(mybuf + 4 * ch) = v;
    }
  }

  float v8[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};   // [tile column][quad column]
  // the Hadamard sign of row 16 b + rl: the lane's part once, the band's on the scalar side
  const uint32_t lane_sign = (__builtin_popcount(rr & rl) & 1) ? 0xBC00BC00u : 0x3C003C00u;   // +-1, twice
#pragma unroll 2
  for (int b = 0; b < nbands; ++b) {
    const uint32_t flip = (__builtin_popcount((rr >> 4) & b) & 1) ? 0x80008000u : 0u;
    const half2_t s2 = __builtin_bit_cast(half2_t, lane_sign ^ flip);
    const float sgn = static_cast<float>(s2.x);
    const uint32_t* band = mybuf + b * per * NWK;
#pragma unroll
    for (int tc = 0; tc < 2; ++tc) {
      if (tc < ntw) {
        const uint32_t* tp = band + tc * NWK;
        uint32_t raw[4];
        decode_quad<K, CB, V>(tp[qp.wa], tp[qp.wb], qp.sh, raw);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          if constexpr (CB == CB_1MAD)
            v8[4 * tc + q] += sgn * static_cast<float>(static_cast<int>(raw[q]) - 510);
          else
            v8[4 * tc + q] = __builtin_amdgcn_fdot2(__builtin_bit_cast(half2_t, raw[q]), s2,
                                                    v8[4 * tc + q], false);
        }
      }
    }
  }
  // sum over the 16 rows (lane bits 2 to 5). After the swaps a lane of half h5 and row h4 of
  // 16 lanes holds the sums of tile column h5, quad columns 2 h4 and 2 h4 + 1
  float v4[4], v2[2];
#pragma unroll
  for (int i = 0; i < 4; ++i) v4[i] = swap_add<32>(v8[i], v8[i + 4]);
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    v2[i] = swap_add<16>(v4[i], v4[i + 2]);
    v2[i] += lane_xor<8>(v2[i], lane);
    v2[i] += lane_xor<4>(v2[i], lane);
  }
  const int tc = lane >> 5;
  if ((lane & 12) == 0 && tc < ntw) {
    float* d = colsum + 16 * (tc0 + tc) + 4 * g + 2 * ((lane >> 4) & 1);
    d[0] = v2[0];
    d[1] = v2[1];
  }
  __syncthreads();
  if (wave != 0) return;
  float lo = lane < a.block_in ? colsum[lane] : 0.f;
  float hi = lane + 64 < a.block_in ? colsum[lane + 64] : 0.f;
  if (CB == CB_1MAD) {
    lo = lo / 147.800537109375f;
    hi = hi / 147.800537109375f;
  }
  fwht_chunk(lo, hi, a.block_in, lane);
  const float rs = ok ? a.sv[r] * a.osc[r] * a.nrm : 0.f;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int jl = lane + 64 * h;
    if (jl < a.block_in) {
      const int j = jb + jl;
      const float v = (h ? hi : lo) * rs * a.isc[j] * a.su[j];
      const long long o = static_cast<long long>(t) * a.ldo + j;
      if (a.out_f16)
        static_cast<_Float16*>(a.out)[o] = static_cast<_Float16>(v);
      else
        static_cast<float*>(a.out)[o] = v;
    }
  }
}

}  // namespace trellis
