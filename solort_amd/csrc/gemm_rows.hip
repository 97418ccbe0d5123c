// Matrix product of a few rows with a weight matrix, HBM-bound weight
// streams: out[t] = W x[t] for m <= 16 rows (a speculative round's K+1 tokens,
// the shortest prompt bucket), W [N][K] bf16 row-major (the torch Linear
// weight layout), fp32 accumulation, bf16 results, with the layer's
// neighbours fused as in gemv.hip:
//   h  = _rmsnorm(x, in_ln);   qkv = h @ wqkv.T            (NORM, PLAIN)
//   x  = x + ctx @ wo.T                                    (RESID)
//   h2 = _rmsnorm(x, post_ln); gate, up = (h2 @ wgu.T).split
//   x  = x + (silu(gate) * up) @ wd.T                      (NORM + SWIGLU, RESID)
//   _rmsnorm(x, final_norm) @ lm_head.T                    (NORM, PLAIN)
// (src/solort/model/cuda_graph_executor.py:104-135, :245-268), rounding where
// the reference's bf16 tensors round.
//
// Mapping: a workgroup of kWaves wavefronts takes tiles of up to 16 weight rows
// (two row groups of 8; SWIGLU: 8 gate rows and their 8 up rows), the wavefronts
// each a contiguous share of K, and their sums meet in LDS, where the epilogue
// reads them.  Operands go from memory straight into the registers of
// v_mfma_f32_16x16x32_bf16 (weights are used once, so LDS would only add a round
// trip).  A load instruction covers 8 rows x 128 bytes, lane (r, g) (r = lane %
// 16, g = lane / 16) chunk 2g + r / 8 of row r % 8 in a step of 64 k: as operand
// A these are 16 virtual rows, row i its real row's k in chunks of parity i / 8,
// and the 8 x rows laid out the same way are 16 virtual columns.  The two
// products of equal parity are the row's partial sums, added at the end; the
// other two are dropped (the matrix unit is idle otherwise).  Loading 16 rows x
// 64 bytes per instruction, as the operand layout has it without this, streamed
// at 3.9 TB/s instead of 4.6 (gate_up) and 4.9 instead of 6.5 (lm_head).
// RMSNorm: a lane holds the x it will multiply, so the sum of squares is
// collected from those registers (one LDS exchange between the wavefronts)
// while the weight loads are in flight.
// One workgroup per CU: 256 registers a wavefront hold x and two batches of U
// steps of weights, 32 KB x U in flight per CU (K = 2560: U = 5, 160 KB).  (Two workgroups of 128 registers each
// spill: gate_up 25-28 us instead of 18.5.)
// Measured on MI355X, 5 rows, Qwen3-4B, graphs over 12 weight copies, with the
// library product of the same shape (no fused neighbours) behind: qkv 7.9 us
// (10.7), o_proj 6.6 (13.4), gate_up + SwiGLU 18.5 (47.5), down 13.3 (18.3),
// lm_head 118.7 us = 6.6 TB/s (242).  A 5-token verify of 8 such layers and the
// lm_head: 1125 -> 568 us.
#include "common.h"
#include "capi_internal.h"

namespace solort {

enum { kRowsPlain = 0, kRowsResid = 1, kRowsSwiglu = 2 };

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

constexpr int kWaves = 8;  // wavefronts per workgroup

// rows_per: outputs per tile (<= 16, SWIGLU <= 8); n_tiles of them are dealt to
// the grid's workgroups.  MT groups of 8 x rows.  NB > 0: NB batches of U steps
// cover a wavefront's whole share of K (the last one may reach past it); the
// (normalised) x stays in registers for every tile, and two batches of weights
// are in flight.  NB = 0: any share, x travels with the weights (5 rows of a 4B
// down product, 19 steps a share: 18.7 us, against 13.3 with x resident).
// TAIL: K is not a multiple of 64 * kWaves, every chunk is checked.  Lanes of
// absent weight or x rows repeat the last one (their sums are dropped).
template <int U, int NB, int MT, int EPI, bool NORM, bool TAIL>
__global__ __launch_bounds__(64 * kWaves, 2) void gemm_rows_kernel(
    const uint16_t* __restrict__ w, int64_t w_stride, int n_out, int K, int rows_per, int n_tiles, int m,
    const uint16_t* __restrict__ x, int64_t x_stride, const uint16_t* __restrict__ norm_w, float eps, int64_t inter,
    const uint16_t* res, int64_t res_stride, uint16_t* out, int64_t out_stride) {
  __shared__ float s_ss[kWaves][8 * MT];
  __shared__ __align__(16) float s_acc[2][kWaves][128 * MT];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, g = lane >> 4, row8 = r & 7;
  const int nch = K >> 3;
  const int nsteps = (K + 63) >> 6, per = (nsteps + kWaves - 1) / kWaves;
  const int s_beg = wave * per, s_end = min(s_beg + per, nsteps);
  const int c0 = 2 * g + (r >> 3);  // the lane's chunk in a step
  const uint16_t* xr[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) xr[t] = x + (int64_t)min(8 * t + row8, m - 1) * x_stride;

  constexpr bool RES = NB > 0;       // x resident
  constexpr int T = RES ? NB * U : U;  // steps of x per register set
  uint4 wv[2][U][2], xv[RES ? 1 : 2][T][MT], gv[NORM && RES ? T : 1];
  float rs[MT];
  // Every load is issued, without branches (a load that some path skips makes the compiler wait for all of
  // them at the first use: o_proj 8.7 us instead of 6.6 for 5 rows): steps past the share and chunks past K
  // read the last one again, and keep() zeroes them where they are used.  Step index u of a batch can lie past
  // the share only where the template says so.
  auto guarded = [](int u) { return TAIL || (RES ? NB > 1 && u >= (NB - 1) * U : true); };
  auto keep = [&](uint4 v, int s, int u) {
    if (!guarded(u)) return v;
    const bool on = s < s_end && (!TAIL || s * 8 + c0 < nch);
    return make_uint4(on ? v.x : 0u, on ? v.y : 0u, on ? v.z : 0u, on ? v.w : 0u);
  };
  auto ld = [&](const uint16_t* row, int s, int u, bool stream) {
    if (guarded(u)) s = max(min(s, s_end - 1), 0);
    int c = s * 8 + c0;
    if (TAIL) c = min(c, nch - 1);
    return stream ? ld_stream(row + 8 * c) : *reinterpret_cast<const uint4*>(row + 8 * c);
  };
  auto load_x = [&](uint4 (&xb)[T][MT], int sb) {
#pragma unroll
    for (int u = 0; u < T; ++u)
#pragma unroll
      for (int t = 0; t < MT; ++t) xb[u][t] = ld(xr[t], sb + u, u, false);
  };
  auto load_w = [&](uint4 (&wb)[U][2], int tile, int sb, int u0) {
    const uint16_t* wr[2];
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int i = EPI == kRowsSwiglu ? row8 : 8 * q + row8;
      const int o = min(tile * rows_per + min(i, rows_per - 1), n_out - 1);
      wr[q] = w + (o + (EPI == kRowsSwiglu && q ? inter : 0)) * w_stride;
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int q = 0; q < 2; ++q) wb[u][q] = ld(wr[q], sb + u, u0 + u, true);
  };
  auto normed = [&](uint4 b, uint4 gw, float scale) {
    float v[8], gg[8];
    unpack8(b, v);
    unpack8(gw, gg);
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = (v[i] * scale) * gg[i];
    return pack8(v);
  };
  int tile = blockIdx.x;
  load_x(xv[0], s_beg);
  if constexpr (NORM && RES) {
#pragma unroll
    for (int u = 0; u < T; ++u) gv[u] = ld(norm_w, s_beg + u, u, false);
  }
  load_w(wv[0], tile, s_beg, 0);
  if constexpr (NORM) {
    float ss[MT];
    auto squares = [&](const uint4& v, float a) {
      a = dot2bf(v.x, v.x, a);
      a = dot2bf(v.y, v.y, a);
      a = dot2bf(v.z, v.z, a);
      return dot2bf(v.w, v.w, a);
    };
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      ss[t] = 0.f;
#pragma unroll
      for (int u = 0; u < T; ++u) ss[t] = squares(keep(xv[0][u][t], s_beg + u, u), ss[t]);
      if constexpr (!RES)
        for (int s = s_beg + U; s < s_end; ++s) ss[t] = squares(keep(ld(xr[t], s, T, false), s, T), ss[t]);
      ss[t] += row16_swap8(ss[t]);
      ss[t] = xor16_combine(ss[t], [](float a, float b) { return a + b; });
      ss[t] = xor32_combine(ss[t], [](float a, float b) { return a + b; });
      if (lane < 8) s_ss[wave][8 * t + lane] = ss[t];
    }
    lds_barrier();
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      float a = 0.f;
#pragma unroll
      for (int i = 0; i < kWaves; ++i) a += s_ss[i][8 * t + row8];
      rs[t] = 1.0f / __builtin_sqrtf(a / (float)K + eps);
      if constexpr (RES) {
#pragma unroll
        for (int u = 0; u < T; ++u) xv[0][u][t] = normed(xv[0][u][t], gv[u], rs[t]);
      }
    }
  }

  auto mma = [&](f32x4_t (&acc)[2][MT], const uint4 (&wb)[U][2], const uint4 (&xb)[T][MT], int sb, int x0) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      uint4 gw = make_uint4(0u, 0u, 0u, 0u);
      if constexpr (NORM && !RES) gw = ld(norm_w, sb + u, u, false);
      const uint4 w0 = keep(wb[u][0], sb + u, x0 + u), w1 = keep(wb[u][1], sb + u, x0 + u);
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        uint4 b = xb[x0 + u][t];
        if constexpr (NORM && !RES) b = normed(b, gw, rs[t]);
        b = keep(b, sb + u, x0 + u);
        acc[0][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, w0),
                                                            __builtin_bit_cast(bf16x8_t, b), acc[0][t], 0, 0, 0);
        acc[1][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, w1),
                                                            __builtin_bit_cast(bf16x8_t, b), acc[1][t], 0, 0, 0);
      }
    }
  };
  // Sums of one tile: to LDS, then the epilogue.
  auto finish = [&](const f32x4_t (&acc)[2][MT], int tile, int par) {
    // Lane (r, g) holds virtual rows 4g .. 4g + 3 of virtual column r: rows 0-7 (lower half wave) with
    // columns 0-7 are parity 0, rows 8-15 (upper half) with columns 8-15 parity 1.  The sum of both for row
    // group 0 ends in the lower half, for group 1 in the upper: lane (r < 8, g) has rows 4g .. 4g + 3 of the
    // tile.
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      f32x4_t sum;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(acc[0][t][i]), __float_as_uint(acc[1][t][i]),
                                                         false, false);
        const uint32_t p0 = sw[0], p1 = sw[1];
        sum[i] = __uint_as_float(p0) + row16_swap8(__uint_as_float(p1));
      }
      if (r < 8) *reinterpret_cast<f32x4_t*>(&s_acc[par][wave][(8 * t + r) * 16 + 4 * g]) = sum;
    }
    lds_barrier();  // two buffers by turns: it also separates the tile before's reads from the next one's writes
    if (tid < 128 * MT) {
      const int t = tid >> 4, i = tid & 15, o = tile * rows_per + i;
      if (t < m && i < rows_per && o < n_out) {
        float a = 0.f;
#pragma unroll
        for (int q = 0; q < kWaves; ++q) a += s_acc[par][q][tid];
        float y = a;
        if constexpr (EPI == kRowsResid) {
          y = bf2f(res[t * res_stride + o]) + rbf(a);
        } else if constexpr (EPI == kRowsSwiglu) {
          float b = 0.f;
#pragma unroll
          for (int q = 0; q < kWaves; ++q) b += s_acc[par][q][tid + 8];
          const float gt = rbf(a);
          y = rbf(gt / (1.0f + __expf(-gt))) * rbf(b);
        }
        out[t * out_stride + o] = f2bf(y);
      }
    }
  };
  const int step = gridDim.x;
  if constexpr (NB == 1) {
    if (tile + step < n_tiles) load_w(wv[1], tile + step, s_beg, 0);
    for (; tile < n_tiles; tile += 2 * step) {
      f32x4_t acc[2][MT] = {};
      mma(acc, wv[0], xv[0], s_beg, 0);
      if (tile + 2 * step < n_tiles) load_w(wv[0], tile + 2 * step, s_beg, 0);
      finish(acc, tile, 0);
      if (tile + step >= n_tiles) break;
      f32x4_t acc1[2][MT] = {};
      mma(acc1, wv[1], xv[0], s_beg, 0);
      if (tile + 3 * step < n_tiles) load_w(wv[1], tile + 3 * step, s_beg, 0);
      finish(acc1, tile + step, 1);
    }
  } else if constexpr (RES) {
    static_assert(NB % 2 == 0, "the batches of a tile alternate between the two weight buffers");
    load_w(wv[1], tile, s_beg + U, U);
    for (int par = 0; tile < n_tiles; par ^= 1) {
      const int next = tile + step;
      f32x4_t acc[2][MT] = {};
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        mma(acc, wv[b & 1], xv[0], s_beg + b * U, b * U);
        if (b + 2 < NB)
          load_w(wv[b & 1], tile, s_beg + (b + 2) * U, (b + 2) * U);
        else if (next < n_tiles)
          load_w(wv[b & 1], next, s_beg + (b + 2 - NB) * U, (b + 2 - NB) * U);
      }
      finish(acc, tile, par);
      tile = next;
    }
  } else {
    for (int par = 0; tile < n_tiles; par ^= 1) {
      f32x4_t acc[2][MT] = {};
      load_x(xv[1], s_beg + U);
      load_w(wv[1], tile, s_beg + U, 0);
      for (int sb = s_beg; sb < s_end; sb += 2 * U) {
        mma(acc, wv[0], xv[0], sb, 0);
        load_x(xv[0], sb + 2 * U);
        load_w(wv[0], tile, sb + 2 * U, 0);
        mma(acc, wv[1], xv[1], sb + U, 0);
        load_x(xv[1], sb + 3 * U);
        load_w(wv[1], tile, sb + 3 * U, 0);
      }
      const int next = tile + step;
      if (next < n_tiles) {  // the next tile's first loads fly during this one's epilogue
        load_x(xv[0], s_beg);
        load_w(wv[0], next, s_beg, 0);
      }
      finish(acc, tile, par);
      tile = next;
    }
  }
}

}  // namespace solort

using namespace solort;

extern "C" int solort_gemm_rows(const void* w, int64_t w_row_stride, int n_out, int k, const void* x,
                                int64_t x_row_stride, int m, const void* norm_w, float eps, const void* res,
                                int64_t res_row_stride, int mode, int64_t inter, void* out, int64_t out_row_stride,
                                solort_stream_t stream) {
  const char* name = "gemm_rows";
  if (mode != kRowsPlain && mode != kRowsResid && mode != kRowsSwiglu)
    return set_error(SOLORT_EINVAL, "%s: mode %d", name, mode);
  if (!w || !x || !out || (mode == kRowsResid && !res)) return set_error(SOLORT_EINVAL, "%s: null pointer", name);
  if (mode == kRowsSwiglu && inter < n_out)
    return set_error(SOLORT_EINVAL, "%s: swiglu needs inter >= n_out (up rows follow the gate rows)", name);
  if (m < 1 || m > 16 || n_out < 1 || k < 8 || k % 8 != 0 || k > 65536)
    return set_error(SOLORT_EINVAL, "%s: bad shape m=%d n_out=%d k=%d (m <= 16, k a multiple of 8, <= 65536)", name, m,
                     n_out, k);
  if (w_row_stride < k || w_row_stride % 8 != 0 || x_row_stride < k || x_row_stride % 8 != 0 ||
      out_row_stride < n_out || (mode == kRowsResid && res_row_stride < n_out))
    return set_error(SOLORT_EINVAL, "%s: bad row stride", name);
  if (!aligned16(w) || !aligned16(x) || (norm_w && !aligned16(norm_w)) || ((uintptr_t)out & 1u) ||
      (res && ((uintptr_t)res & 1u)))
    return set_error(SOLORT_EINVAL, "%s: w, x and norm_w must be 16-byte aligned", name);
  // Outputs per tile: a full one (16, SWIGLU 8), unless that leaves the last round of tiles over the CUs
  // uneven; then the smallest count with the same number of rounds (2560 outputs: 256 tiles of 10, not 160
  // of 16 on 160 CUs).
  const int tile = mode == kRowsSwiglu ? 8 : 16, cus = cu_count() > 0 ? cu_count() : 256;
  const int rounds = ((n_out + tile - 1) / tile + cus - 1) / cus;
  const int rows_per = (int)(((int64_t)n_out + (int64_t)rounds * cus - 1) / ((int64_t)rounds * cus));
  const int tiles = (n_out + rows_per - 1) / rows_per;
  const int steps = ((k + 63) / 64 + kWaves - 1) / kWaves;
  const bool tail = k % (64 * kWaves) != 0;
  // Shares of the served widths (K = 1024, 2048, 2560, 3072, 4096: 2 to 8 steps) have a batch of their own, the
  // down products (K = 9728, 12288: 19 and 24) 4 and 6 batches; 9-16 rows and the rest go without x resident.
#define SOLORT_ROWS_U(UU, BB, MM, EE, NN, TT)                                                                       \
  hipLaunchKernelGGL((gemm_rows_kernel<UU, BB, MM, EE, NN, TT>), dim3(min(tiles, cus)), dim3(64 * kWaves), 0,      \
                     (hipStream_t)stream, (const uint16_t*)w, w_row_stride, n_out, k, rows_per, tiles, m,          \
                     (const uint16_t*)x, x_row_stride, (const uint16_t*)norm_w, eps, inter, (const uint16_t*)res,  \
                     res_row_stride, (uint16_t*)out, out_row_stride)
#define SOLORT_ROWS_M(MM, EE, NN)                                                        \
  do {                                                                                   \
    if (tail) SOLORT_ROWS_U(2, 0, MM, EE, NN, true);                                     \
    else if (steps == 2) SOLORT_ROWS_U(2, 1, MM, EE, NN, false);                         \
    else if (steps == 4) SOLORT_ROWS_U(4, 1, MM, EE, NN, false);                         \
    else if (steps == 5) SOLORT_ROWS_U(5, 1, MM, EE, NN, false);                         \
    else if (steps == 6) SOLORT_ROWS_U(6, 1, MM, EE, NN, false);                         \
    else if (MM == 1 && steps == 8) SOLORT_ROWS_U(8, 1, 1, EE, NN, false);               \
    else if (MM == 2 && steps == 8) SOLORT_ROWS_U(4, 2, 2, EE, NN, false);               \
    else if (!NN && MM == 1 && steps > 15 && steps <= 20) SOLORT_ROWS_U(5, 4, 1, EE, false, false); \
    else if (!NN && MM == 1 && steps > 20 && steps <= 24) SOLORT_ROWS_U(4, 6, 1, EE, false, false); \
    else SOLORT_ROWS_U(4, 0, MM, EE, NN, false);                                         \
  } while (0)
#define SOLORT_ROWS_N(EE, NN)                                              \
  do {                                                                     \
    if (m <= 8) SOLORT_ROWS_M(1, EE, NN); else SOLORT_ROWS_M(2, EE, NN);   \
  } while (0)
#define SOLORT_ROWS(EE)                                                    \
  do {                                                                     \
    if (norm_w) SOLORT_ROWS_N(EE, true); else SOLORT_ROWS_N(EE, false);    \
  } while (0)
  if (mode == kRowsPlain) SOLORT_ROWS(kRowsPlain);
  else if (mode == kRowsResid) SOLORT_ROWS(kRowsResid);
  else SOLORT_ROWS(kRowsSwiglu);
#undef SOLORT_ROWS
#undef SOLORT_ROWS_N
#undef SOLORT_ROWS_M
#undef SOLORT_ROWS_U
  return check_launch(name);
}
