// Matrix product of a prompt bucket's rows with a weight matrix: X [m][k] W^T,
// W [N][k] bf16 row-major (the torch Linear weight layout), fp32 accumulation.
//   qkv = h @ wqkv.T                             (PLAIN)
//   gate, up = (h @ wgu.T).split; silu(gate) * up (SWIGLU)
//   ctx @ wo.T, act @ wd.T                       (PARTS: fp32 sums over shares
//     of k, added by solort_add_parts_rmsnorm with the residual and the norm)
// (src/solort/model/cuda_graph_executor.py:115, :131-134), rounding where the
// reference's bf16 tensors round.
//
// Bound: up to 256 rows what a CU can load, beyond loads and matrix units alike
// (down of 1024 rows: its loads alone take 81 % of its time, its arithmetic
// alone 71 %).  A workgroup takes a BM x BN tile over a share of k, WM x WN wavefronts of
// v_mfma_f32_16x16x32_bf16 each BM / WM rows x BN / WN weight rows (A = W, B =
// X, so a lane ends with four neighbouring outputs of one row).
// Stages of kBK columns of X and W go from memory straight into LDS (16 bytes
// a lane, no registers), NST - 1 of them in flight over counted waits and one
// barrier a stage.  Each stage buffer is an array of its own: the compiler then
// sees that a stage's reads do not touch the buffers being filled and adds no
// full wait.  A row's 16-byte chunks are stored in the order chunk ^ (row %
// chunks) (rows of four chunks: row / 2), by permuting the lanes' source
// addresses, so the 16 rows of an operand read fall on different banks.
// Up to 256 rows the loads are the time (gate_up of 128 rows 32.3 us, its loads
// alone 31.7, its arithmetic alone 19.8), and those of X and W add up (X alone
// 10.3, W alone 21.6): a CU's requests return in order, so rows of X that hit
// the L2 wait behind weights from HBM, and more stages in flight change
// nothing.  The tile is therefore chosen to give every CU one workgroup and few
// repeated reads of X (304 workgroups instead of 203: 44 us instead of 32); where
// the tiles of N alone leave CUs idle (N = 2560: 40 tiles), k is split.
// Workgroups that share a tile of W run on one XCD (block index mod 8).
// Measured on MI355X, Qwen3-4B widths, normal random values, graphs over 10
// weight copies with one x and one result, 32 / 128 / 1024 rows, the library's
// product behind (us, two runs within 5 %): qkv 10.2 / 17.1 / - (12.0 / 19.2 /
// 40.1), o_proj 5.9 / 8.2 / 28.3 (9.4 / 19.1 / 31.1), gate_up with SwiGLU 23.2 /
// 32.3 / 96 (24.9 / 33.1 / 107 without), down 12.6 / 19.6 / 55 (21.4 / 52.6 /
// 79).  The time depends on the values through the clock: down of 1024 rows
// takes 49 us with zero weights.
#include "common.h"
#include "capi_internal.h"

namespace solort {

enum { kTilePlain = 0, kTileSwiglu = 1, kTileParts = 2 };

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

typedef __attribute__((address_space(3))) void lds_void;

// 64 lanes x 16 bytes from memory into LDS at dst + 16 lane, without a register in between.
__device__ __forceinline__ void lds_load16(__amdgpu_buffer_rsrc_t r, lds_void* dst, int voff, int soff) {
#ifdef __HIP_DEVICE_COMPILE__  // the host pass does not know the 16-byte form
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, dst, 16, voff, soff, 0, 0);
#endif
}

// Waits until at most VM of this wavefront's loads are in flight and its LDS reads have returned, then for the
// other wavefronts: the oldest stage is whole, and nobody reads the buffer of the stage before it any more.
template <int VM>
__device__ __forceinline__ void stage_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt((VM & 15) | (7 << 4) | ((VM >> 4) << 14));
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// out: bf16 [m][out_stride], PARTS: fp32 [splits][m][out_stride].  inter: row distance of a gate row's up row.
template <int BM, int BN, int WM, int WN, int NST, int kBK, int EPI>
__global__ __launch_bounds__(64 * WM * WN) void gemm_tile_kernel(
    const uint16_t* __restrict__ w, const uint16_t* __restrict__ x, int n_out, int k_steps, int m, int w_stride,
    int x_stride, int tiles_m, int tiles_n, int splits,
    int inter, void* __restrict__ out_ptr, int64_t out_stride) {
  constexpr int NW = WM * WN, MT = BM / WM / 16, NT = BN / WN / 16;
  constexpr int ROWS = BM + BN, KC = kBK / 8, RPI = 64 / KC,
                NI = ROWS / RPI, IPW = (NI + NW - 1) / NW;  // load instructions per wavefront and stage
  constexpr int KS = KC == 4 ? 1 : 0;  // rows of four chunks: two rows fill a bank period
  static_assert(ROWS % RPI == 0 && BM % RPI == 0 && BM % (16 * WM) == 0 && BN % (16 * WN) == 0, "tile shape");
  static_assert(EPI != kTileSwiglu || NT % 2 == 0, "gate and up blocks of a column meet in one wavefront");
  constexpr int BO = EPI == kTileSwiglu ? BN / 2 : BN;  // outputs per tile
  constexpr int WORDS = ROWS * kBK;
  __shared__ __align__(1024) uint16_t s0[WORDS], s1[WORDS], s2[WORDS], s3[NST > 3 ? WORDS : 1];
  static_assert(NST == 3 || NST == 4, "three or four stage buffers");
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int b = blockIdx.x, loc = b >> 3, col = (loc / tiles_m) * 8 + (b & 7);
  if (col >= tiles_n * splits) return;
  const int tm = loc % tiles_m, split = col / tiles_n, tn = col % tiles_n;
  const int k_beg = split * k_steps / splits, steps = (split + 1) * k_steps / splits - k_beg;  // >= NST - 1

  // Resources that end with the last row's k: rows past the tile's edge repeat the last one, so nothing reads past.
  const auto rsrc = [&](const uint16_t* p, int rows, int stride) {
    const int nbytes = ((rows - 1) * stride + k_steps * kBK) * 2;  // below 2^31, checked by the caller
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(p), (short)0, nbytes, 0x00020000);
  };
  const __amdgpu_buffer_rsrc_t xr = rsrc(x, m, x_stride);
  const __amdgpu_buffer_rsrc_t wr = rsrc(w, EPI == kTileSwiglu ? inter + n_out : n_out, w_stride);
  // First row of this wavefront's j-th load; past the tile's last one it repeats that (the same bytes to the same place).
  const auto row_of = [&](int j) { return RPI * min(wave + NW * j, NI - 1); };
  int voff[IPW];
#pragma unroll
  for (int j = 0; j < IPW; ++j) {
    const int row0 = row_of(j), row = row0 + lane / KC, ch = (lane ^ (row >> KS)) & (KC - 1);
    int64_t off;
    if (row0 < BM) {
      off = (int64_t)min(tm * BM + row, m - 1) * x_stride;
    } else {
      const int q = row - BM;
      if constexpr (EPI == kTileSwiglu) {
        off = (int64_t)(min(tn * BO + (q >> 5) * 16 + (q & 15), n_out - 1) + ((q >> 4) & 1) * inter) * w_stride;
      } else {
        off = (int64_t)min(tn * BO + q, n_out - 1) * w_stride;
      }
    }
    voff[j] = (int)((off + 8 * ch) * 2);
  }
  auto issue = [&](uint16_t* s, int step) {
    const int soff = (k_beg + step) * (kBK * 2);
#pragma unroll
    for (int j = 0; j < IPW; ++j) {
      const int row0 = row_of(j);
      lds_void* dst = (lds_void*)(__attribute__((address_space(3))) uint16_t*)(s + row0 * kBK);
      lds_load16(row0 < BM ? xr : wr, dst, voff[j], soff);
    }
  };
  const int r = lane & 15, g = lane >> 4;
  const int wm = wave % WM, wn = wave / WM;
  // chunk 4 kk + g of row r sits in slot (4 kk + g) ^ (r % 8)
  const int frag = r * kBK + 8 * (g ^ ((r >> KS) & (KC - 1)));
  const int xbase = wm * (BM / WM) * kBK + frag, wbase = (BM + wn * (BN / WN)) * kBK + frag;
  f32x4_t acc[NT][MT] = {};
  auto compute = [&](const uint16_t* s) {
#pragma unroll
    for (int kk = 0; kk < kBK / 32; ++kk) {
      bf16x8_t xf[MT], wf[NT];
#pragma unroll
      for (int i = 0; i < MT; ++i) xf[i] = *reinterpret_cast<const bf16x8_t*>(s + ((xbase + i * 16 * kBK) ^ (32 * kk)));
#pragma unroll
      for (int i = 0; i < NT; ++i) wf[i] = *reinterpret_cast<const bf16x8_t*>(s + ((wbase + i * 16 * kBK) ^ (32 * kk)));
#pragma unroll
      for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int i = 0; i < MT; ++i)
          acc[n][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[n], xf[i], acc[n][i], 0, 0, 0);
    }
  };
  auto buf = [&](int i) -> uint16_t* { return i == 0 ? s0 : i == 1 ? s1 : i == 2 ? s2 : s3; };
  constexpr int A = NST - 1;  // stages in flight
#pragma unroll
  for (int i = 0; i < A; ++i) issue(buf(i), i);
  int i = 0;
  for (; i + A + NST <= steps; i += NST) {
#pragma unroll
    for (int u = 0; u < NST; ++u) {
      stage_barrier<(A - 1) * IPW>();
      issue(buf((u + A) % NST), i + u + A);
      compute(buf(u));
    }
  }
#pragma unroll
  for (int u = 0; u < A + NST - 1; ++u) {
    if (i + u >= steps) break;
    if (i + u + A <= steps)
      stage_barrier<(A - 1) * IPW>();
    else
      stage_barrier<0>();
    if (i + u + A < steps) issue(buf((u + A) % NST), i + u + A);
    compute(buf(u % NST));
  }

#pragma unroll
  for (int mi = 0; mi < MT; ++mi) {
    const int row = tm * BM + wm * (BM / WM) + mi * 16 + r;
    if (row >= m) continue;
    if constexpr (EPI == kTileSwiglu) {
#pragma unroll
      for (int n = 0; n < NT; n += 2) {
        const int col = tn * BO + wn * (BO / WN) + (n / 2) * 16 + 4 * g;
        float y[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float gt = rbf(acc[n][mi][e]);
          y[e] = rbf(gt / (1.0f + __expf(-gt))) * rbf(acc[n + 1][mi][e]);
        }
        uint16_t* o = reinterpret_cast<uint16_t*>(out_ptr) + row * out_stride + col;
        if (col < n_out) *reinterpret_cast<uint2*>(o) = make_uint2(pack2(y[0], y[1]), pack2(y[2], y[3]));
      }
    } else {
#pragma unroll
      for (int n = 0; n < NT; ++n) {
        const int col = tn * BO + wn * (BO / WN) + n * 16 + 4 * g;
        if (col >= n_out) continue;
        if constexpr (EPI == kTileParts) {
          float* o = reinterpret_cast<float*>(out_ptr) + ((int64_t)split * m + row) * out_stride + col;
          *reinterpret_cast<f32x4_t*>(o) = acc[n][mi];
        } else {
          uint16_t* o = reinterpret_cast<uint16_t*>(out_ptr) + row * out_stride + col;
          *reinterpret_cast<uint2*>(o) =
              make_uint2(pack2(acc[n][mi][0], acc[n][mi][1]), pack2(acc[n][mi][2], acc[n][mi][3]));
        }
      }
    }
  }
}

}  // namespace solort

using namespace solort;

namespace {

// A tile shape and its launch.
template <int BM, int BN, int WM, int WN, int NST, int BK, int EPI>
void launch_tile(const void* w, const void* x, int n_out, int k, int m, int64_t w_stride, int64_t x_stride, int splits,
                 int64_t inter, void* out, int64_t out_stride, hipStream_t stream) {
  constexpr int BO = EPI == kTileSwiglu ? BN / 2 : BN;
  const int tiles_m = (m + BM - 1) / BM, tiles_n = (n_out + BO - 1) / BO;
  const int grid = (tiles_n * splits + 7) / 8 * 8 * tiles_m;
  hipLaunchKernelGGL((gemm_tile_kernel<BM, BN, WM, WN, NST, BK, EPI>), dim3(grid), dim3(64 * WM * WN), 0, stream,
                     (const uint16_t*)w, (const uint16_t*)x, n_out, k / BK, m, (int)w_stride, (int)x_stride, tiles_m,
                     tiles_n, splits, (int)inter, out, out_stride);
}

// Tiles of a PARTS product: 64 weight rows up to 128 rows of x, 128 beyond; rows of x 32, 64, 128, 128 (up to 256),
// 256.
int parts_tiles(int m, int n_out) {
  const int bn = m <= 128 ? 64 : 128, bm = m <= 256 ? 128 : 256;
  return (n_out + bn - 1) / bn * (m <= 128 ? 1 : (m + bm - 1) / bm);
}

bool tile_shape_ok(int m, int n_out, int k) {
  return m >= 1 && m <= (1 << 20) && n_out >= 4 && n_out % 4 == 0 && n_out <= (1 << 24) && k >= 512 && k % 128 == 0 &&
         k <= 65536;
}

}  // namespace

// One workgroup per CU: as many shares of k as the tiles leave CUs for, at least 4 steps of 64 each (the pipeline's
// depth).  (N = 2560, k = 9728, 128 rows: 6 shares on 240 CUs 17.7 us, 3 on 120 28.9, 12 on 480 workgroups 19.4.)
extern "C" int solort_gemm_tile_parts(int m, int n_out, int k) {
  if (!tile_shape_ok(m, n_out, k)) return 0;
  const int cus = cu_count() > 0 ? cu_count() : 256, tiles = parts_tiles(m, n_out);
  const int most = k / 64 / 4;
  const int fit = cus / tiles > 1 ? cus / tiles : 1;
  return fit < most ? fit : most;
}

extern "C" int solort_gemm_tile(const void* w, int64_t w_row_stride, int n_out, int k, const void* x,
                                int64_t x_row_stride, int m, int mode, int64_t inter, int n_parts, void* out,
                                int64_t out_row_stride, solort_stream_t stream) {
  const char* name = "gemm_tile";
  if (mode != kTilePlain && mode != kTileSwiglu && mode != kTileParts)
    return set_error(SOLORT_EINVAL, "%s: mode %d", name, mode);
  if (!w || !x || !out) return set_error(SOLORT_EINVAL, "%s: null pointer", name);
  if (!tile_shape_ok(m, n_out, k))
    return set_error(SOLORT_EINVAL, "%s: bad shape m=%d n_out=%d k=%d (n_out a multiple of 4, k of 128, 512..65536)",
                     name, m, n_out, k);
  if (mode == kTileSwiglu && (inter < n_out || inter > (1 << 24)))
    return set_error(SOLORT_EINVAL, "%s: swiglu needs inter >= n_out (up rows follow the gate rows)", name);
  if (mode == kTileParts && (n_parts < 1 || n_parts > k / 256))
    return set_error(SOLORT_EINVAL, "%s: n_parts=%d outside [1, k / 256]", name, n_parts);
  if (w_row_stride < k || w_row_stride % 8 != 0 || x_row_stride < k || x_row_stride % 8 != 0 ||
      out_row_stride < n_out || out_row_stride % 4 != 0 || (mode == kTileParts && out_row_stride != n_out))
    return set_error(SOLORT_EINVAL, "%s: bad row stride", name);
  // Rows are addressed with 32-bit byte offsets.
  const int64_t w_rows = mode == kTileSwiglu ? inter + n_out : n_out, lim = ((int64_t)1 << 30) - 65536;
  if (w_row_stride > lim / w_rows || x_row_stride > lim / m)
    return set_error(SOLORT_EINVAL, "%s: w or x exceeds 32-bit byte offsets", name);
  if (!aligned16(w) || !aligned16(x) || !aligned16(out))
    return set_error(SOLORT_EINVAL, "%s: pointers must be 16-byte aligned", name);
  const hipStream_t s = (hipStream_t)stream;
#define SOLORT_TILE(...) \
  launch_tile<__VA_ARGS__>(w, x, n_out, k, m, w_row_stride, x_row_stride, mode == kTileParts ? n_parts : 1, inter, out, \
                           out_row_stride, s)
  if (mode == kTilePlain) {
    // 32 weight rows a tile (qkv widths 4096 and 6144: 128 and 192 workgroups; 128 rows, N = 6144: 16.6 us, 24.3 at
    // 64); 256 rows have two tiles of rows, so 64 (20.2 us; library 31.4).
    if (m <= 32) SOLORT_TILE(32, 32, 2, 2, 4, 128, kTilePlain);
    else if (m <= 64) SOLORT_TILE(64, 32, 2, 2, 4, 128, kTilePlain);
    else if (m <= 128) SOLORT_TILE(128, 32, 4, 2, 3, 128, kTilePlain);
    else SOLORT_TILE(128, 64, 4, 2, 3, 128, kTilePlain);
  } else if (mode == kTileSwiglu) {
    // 48 outputs a tile where that gives at least one for every second CU (9728: 203, 12288: 256), else 16 (3072: 192).
    const bool wide = (n_out + 47) / 48 * 2 >= (cu_count() > 0 ? cu_count() : 256);
    if (m <= 32) {
      if (wide) SOLORT_TILE(32, 96, 2, 1, 3, 128, kTileSwiglu);
      else SOLORT_TILE(32, 32, 2, 1, 4, 128, kTileSwiglu);
    } else if (m <= 64) {
      if (wide) SOLORT_TILE(64, 96, 4, 1, 3, 128, kTileSwiglu);
      else SOLORT_TILE(64, 32, 4, 1, 4, 128, kTileSwiglu);
    } else if (m <= 128) {
      if (wide) SOLORT_TILE(128, 96, 4, 1, 4, 64, kTileSwiglu);
      else SOLORT_TILE(128, 32, 4, 1, 3, 128, kTileSwiglu);
    } else if (m > 256) {
      // 256 rows x 160 outputs, the widest that fits: 1024 rows of N = 9728 are 244 workgroups, one round (102 us; 119
      // with 64 outputs, library and SwiGLU 117).
      SOLORT_TILE(256, 320, 4, 2, 3, 32, kTileSwiglu);
    } else {
      if (wide) SOLORT_TILE(256, 96, 4, 1, 3, 64, kTileSwiglu);
      else SOLORT_TILE(128, 64, 4, 2, 3, 128, kTileSwiglu);
    }
  } else {
    if (m <= 32) SOLORT_TILE(32, 64, 1, 4, 4, 64, kTileParts);
    else if (m <= 64) SOLORT_TILE(64, 64, 2, 2, 4, 64, kTileParts);
    else if (m <= 128) SOLORT_TILE(128, 64, 4, 2, 4, 64, kTileParts);
    else if (m <= 256) SOLORT_TILE(128, 128, 4, 2, 4, 64, kTileParts);
    else SOLORT_TILE(256, 128, 4, 2, 3, 64, kTileParts);
  }
#undef SOLORT_TILE
  return check_launch(name);
}
