// Quantisation kernels: X and W to padded e4m3 operand arrays (with the final RMSNorm fused on request), amax scales,
// the bf16 operands of the eval head, byte transposes (internal header).
// Part of the one translation unit sce_kernels.hip, which includes it after the headers it builds on.
#pragma once

namespace sce {

// ------------------------------------------------------------------------------------------
// quantisation
// ------------------------------------------------------------------------------------------
// 16 consecutive elements starting at p as floats after the scaling; elements at or beyond `valid` are 0.  One or two 16/32-byte
// vector loads when the run is complete and 16-byte aligned -- with ANY, aligned or not: for rows of which all or most runs are not
// (element by element, the lanes of a wave touch a different cache line each, 16 times over).  The kernels choose once, by base
// and row length: the choice made for each run was 2 to 4 % slower on aligned rows.
template <typename T, bool ANY>
__device__ __forceinline__ void load16_scaled(const T* __restrict__ p, int64_t valid, const Scaler scale, float (&v)[16]) {
  using VI = std::conditional_t<ANY, v4i_any, v4i>;
  using VF = std::conditional_t<ANY, v4f_any, v4f>;
  if (valid >= 16 && (ANY || (((uintptr_t)p) & 15) == 0)) {
    if constexpr (sizeof(T) == 2) {
      const v4i r0 = *reinterpret_cast<const VI*>(p), r1 = *reinterpret_cast<const VI*>(p + 8);
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        v[2 * m] = scale.apply<T>(__uint_as_float((uint32_t)r0[m] << 16));
        v[2 * m + 1] = scale.apply<T>(__uint_as_float((uint32_t)r0[m] & 0xffff0000u));
        v[8 + 2 * m] = scale.apply<T>(__uint_as_float((uint32_t)r1[m] << 16));
        v[8 + 2 * m + 1] = scale.apply<T>(__uint_as_float((uint32_t)r1[m] & 0xffff0000u));
      }
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const v4f r = *reinterpret_cast<const VF*>(p + 4 * q);
#pragma unroll
        for (int m = 0; m < 4; ++m) v[4 * q + m] = scale.apply<T>(r[m]);
      }
    }
  } else {
#pragma unroll
    for (int m = 0; m < 16; ++m) v[m] = (m < valid) ? scale.apply<T>(Elem<T>::load(p + m)) : 0.f;
  }
}
// every run of 16 elements that starts at a multiple of 16 in a row is aligned
template <typename T>
__device__ __forceinline__ bool rows_aligned(const T* p, int64_t ld) { return (((uintptr_t)p | (uintptr_t)(ld * (int64_t)sizeof(T))) & 15) == 0; }

// dst [rows_p][cols_p] e4m3 = src [rows][cols] / s, zero outside; 16 outputs per thread.  In all the quantising
// kernels inv_scale is the reciprocal 1 / s taken once on the host, or, with scale_dev, s is read from the device.
template <typename T>
__device__ __forceinline__ void quantize_pad(int block, int nblocks, const T* __restrict__ src, int64_t ld, int64_t rows, int64_t cols, uint8_t* __restrict__ dst,
                                             int64_t rows_p, int64_t cols_p, int64_t dst_ld, float inv_scale, const float* __restrict__ scale_dev) {
  const Scaler scale = make_scaler<T>(inv_scale, scale_dev);
  const int64_t chunks_per_row = cols_p / 16;
  const int64_t total = rows_p * chunks_per_row;
  auto walk = [&](auto any) {
    for (int64_t q = (int64_t)block * 256 + threadIdx.x; q < total; q += (int64_t)nblocks * 256) {
      const int64_t r = q / chunks_per_row, c0 = (q - r * chunks_per_row) * 16;
      uint32_t out[4] = {0, 0, 0, 0};
      if (r < rows && c0 < cols) {
        float v[16];
        load16_scaled<T, decltype(any)::value>(src + r * ld + c0, cols - c0, scale, v);
#pragma unroll
        for (int m = 0; m < 4; ++m) out[m] = cvt4_e4m3(v[4 * m], v[4 * m + 1], v[4 * m + 2], v[4 * m + 3]);
      }
      *reinterpret_cast<v4i*>(dst + r * dst_ld + c0) = (v4i){(int)out[0], (int)out[1], (int)out[2], (int)out[3]};
    }
  };
  if (rows_aligned(src, ld)) walk(std::false_type()); else walk(std::true_type());
}

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// The trunk's last operation fused into the quantiser (F.rms_norm without weight, tiny/train.py:397-398,734):
// dst row = e4m3(round_T(h * rstd) / scale) with rstd = 1 / sqrt(mean(h^2) + eps), the normalised row rounded to
// the input's type as the unfused path has it in memory.  One wave per row; rstd is kept for backward.
template <typename T>
__device__ __forceinline__ void rmsnorm_quantize(int block, const T* __restrict__ src, int64_t ld, int64_t rows, int64_t cols, float eps, uint8_t* __restrict__ dst,
                                                 int64_t rows_p, int64_t cols_p, int64_t dst_ld, float inv_scale, const float* __restrict__ scale_dev,
                                                 float* __restrict__ rstd_out) {
  const Scaler scale = make_scaler<T>(inv_scale, scale_dev), one = {1.0f, false};
  const int lane = threadIdx.x & 63;
  const int64_t r = (int64_t)block * 4 + (threadIdx.x >> 6);
  if (r >= rows_p) return;
  const int64_t chunks = cols_p / 16;
  if (r >= rows) {
    for (int64_t c = lane; c < chunks; c += 64) *reinterpret_cast<v4i*>(dst + r * dst_ld + c * 16) = (v4i){0, 0, 0, 0};
    if (lane == 0) rstd_out[r] = 0.f;
    return;
  }
  const T* row = src + r * ld;
  float ss = 0.f;
  for (int64_t c = lane; c * 16 < cols; c += 64) {
    float v[16];
    load16_scaled<T, false>(row + c * 16, cols - c * 16, one, v);      // scaling by 1 is exact: the values themselves
#pragma unroll
    for (int m = 0; m < 16; ++m) ss = fmaf(v[m], v[m], ss);
  }
  ss = wave_sum(ss);
  const float rstd = 1.0f / sqrtf(ss / (float)cols + eps);
  if (lane == 0) rstd_out[r] = rstd;
  for (int64_t c = lane; c < chunks; c += 64) {
    uint32_t out[4] = {0, 0, 0, 0};
    if (c * 16 < cols) {
      float v[16];
      load16_scaled<T, false>(row + c * 16, cols - c * 16, one, v);
#pragma unroll
      for (int m = 0; m < 16; ++m) {
        float y = v[m] * rstd;
        if constexpr (sizeof(T) == 2) y = round_to_bf16(y);
        v[m] = scale.apply<T>(y);
      }
#pragma unroll
      for (int m = 0; m < 4; ++m) out[m] = cvt4_e4m3(v[4 * m], v[4 * m + 1], v[4 * m + 2], v[4 * m + 3]);
    }
    *reinterpret_cast<v4i*>(dst + r * dst_ld + c * 16) = (v4i){(int)out[0], (int)out[1], (int)out[2], (int)out[3]};
  }
}

// 8 consecutive elements as floats, and back; `vec`: the run is 16-byte (bf16) / 32-byte (fp32) aligned.
template <typename T>
__device__ __forceinline__ void load8(const T* __restrict__ p, bool vec, float (&v)[8]) {
  if (vec) {
    if constexpr (sizeof(T) == 2) {
      const v4i r = *reinterpret_cast<const v4i*>(p);
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        v[2 * m] = __uint_as_float((uint32_t)r[m] << 16);
        v[2 * m + 1] = __uint_as_float((uint32_t)r[m] & 0xffff0000u);
      }
    } else {
      const v4f a = *reinterpret_cast<const v4f*>(p), b = *reinterpret_cast<const v4f*>(p + 4);
#pragma unroll
      for (int m = 0; m < 4; ++m) { v[m] = a[m]; v[4 + m] = b[m]; }
    }
  } else {
#pragma unroll
    for (int m = 0; m < 8; ++m) v[m] = Elem<T>::load(p + m);
  }
}
template <typename T>
__device__ __forceinline__ void store8(T* __restrict__ p, bool vec, const float (&v)[8]) {
  if (vec) {
    if constexpr (sizeof(T) == 2) {
      v4i r;
#pragma unroll
      for (int m = 0; m < 4; ++m) r[m] = (int)((uint32_t)float_to_bf16_bits(v[2 * m]) | ((uint32_t)float_to_bf16_bits(v[2 * m + 1]) << 16));
      *reinterpret_cast<v4i*>(p) = r;
    } else {
      *reinterpret_cast<v4f*>(p) = (v4f){v[0], v[1], v[2], v[3]};
      *reinterpret_cast<v4f*>(p + 4) = (v4f){v[4], v[5], v[6], v[7]};
    }
  } else {
#pragma unroll
    for (int m = 0; m < 8; ++m) Elem<T>::store(p + m, v[m]);
  }
}

// Backward of that norm, in place on the finished dX: with xhat = h * rstd and g the gradient of the normalised row,
// dh = rstd * (g - xhat * mean(g * xhat)).  One wave per row; cols is a multiple of 8.
template <typename TG, typename TH>
__global__ __launch_bounds__(256) void rmsnorm_backward_kernel(TG* __restrict__ g, int64_t g_ld, const TH* __restrict__ h,
                                                              int64_t h_ld, const float* __restrict__ rstd_in, int64_t rows,
                                                              int64_t cols) {
  const int lane = threadIdx.x & 63;
  const int64_t r = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (r >= rows) return;
  const float rstd = rstd_in[r];
  TG* grow = g + r * g_ld;
  const TH* hrow = h + r * h_ld;
  const bool gvec = (((uintptr_t)grow) & (8 * sizeof(TG) - 1)) == 0, hvec = (((uintptr_t)hrow) & (8 * sizeof(TH) - 1)) == 0;
  float dot = 0.f;
  for (int64_t c = 8 * lane; c < cols; c += 512) {
    float gv[8], hv[8];
    load8<TG>(grow + c, gvec, gv);
    load8<TH>(hrow + c, hvec, hv);
#pragma unroll
    for (int m = 0; m < 8; ++m) dot = fmaf(gv[m], hv[m] * rstd, dot);
  }
  dot = wave_sum(dot) / (float)cols;
  for (int64_t c = 8 * lane; c < cols; c += 512) {
    float gv[8], hv[8];
    load8<TG>(grow + c, gvec, gv);
    load8<TH>(hrow + c, hvec, hv);
#pragma unroll
    for (int m = 0; m < 8; ++m) gv[m] = rstd * (gv[m] - hv[m] * rstd * dot);
    store8<TG>(grow + c, gvec, gv);
  }
}

// Operands with a long K (the two of dW, and W_q in dX) are stored tile by tile: for every 256 rows, K block
// after K block, 256 rows of 128 bytes each.  A workgroup's load of one K block of one operand is then one
// contiguous 32 KB piece (row-major rows lie Np, Pw or Vp bytes apart, and the dW main loop lost 12 % to that at
// K = 65536).
__device__ __forceinline__ int64_t blocked_offset(int64_t row, int64_t k, int64_t kblocks) {
  return (((row >> 8) * kblocks + (k >> 7)) * 256 + (row & 255)) * 128 + (k & 127);
}
constexpr int BLOCKED_KSTEP = 256 * BK;     // bytes from one K block of a tile to the next

// W (d, V) -> W_q (dq rows, K = Vp, tile by tile) and W_q^T [Vp][dp] (row-major); 128 x 128 tiles through LDS, so that
// every piece of a row that a workgroup reads or writes is at least 128 bytes long (with 64 x 64 tiles and 64-byte
// pieces the kernel reached 3.5 TB/s at V = 131072).
constexpr int QW_TILE = 128;
typedef uint8_t QwTile[QW_TILE][QW_TILE + 4];
template <typename T>
__device__ __forceinline__ void quantize_w(QwTile& tile, int bx, int by, const T* __restrict__ w, int64_t ld, int64_t d, int64_t V, uint8_t* __restrict__ wq,
                                           uint8_t* __restrict__ wqt, int64_t dp, int64_t ldx, int64_t kbv, float inv_scale, const float* __restrict__ scale_dev) {
  const Scaler scale = make_scaler<T>(inv_scale, scale_dev);
  const int t = threadIdx.x;
  const int64_t j0 = (int64_t)by * QW_TILE, v0 = (int64_t)bx * QW_TILE;
  if (sizeof(T) == 4 && v0 + QW_TILE <= V && ((reinterpret_cast<uintptr_t>(w) | (uintptr_t)(ld * 4)) & 15) == 0) {
    // fp32: four elements a load, so that a wave reads 512 bytes of a row in a row (with 16 a thread its loads lay 64 bytes
    // apart: 3.2 TB/s at d = 768)
    v4f x[16];
#pragma unroll
    for (int pass = 0; pass < 16; ++pass) {
      const int64_t j = j0 + (t >> 5) + 8 * pass;
      x[pass] = j < d ? *reinterpret_cast<const v4f*>(reinterpret_cast<const float*>(w) + j * ld + v0 + (t & 31) * 4) : (v4f){0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int pass = 0; pass < 16; ++pass) {
      const int r = (t >> 5) + 8 * pass, c = (t & 31) * 4;
      const uint32_t out = cvt4_e4m3(scale.apply<T>(x[pass][0]), scale.apply<T>(x[pass][1]), scale.apply<T>(x[pass][2]), scale.apply<T>(x[pass][3]));
      *reinterpret_cast<uint32_t*>(wq + blocked_offset(j0 + r, v0 + c, kbv)) = out;
      *reinterpret_cast<uint32_t*>(&tile[r][c]) = out;
    }
  } else {
    auto fill = [&](auto any) {
#pragma unroll
      for (int pass = 0; pass < 4; ++pass) {
        const int r = (t >> 3) + 32 * pass, c = (t & 7) * 16;
        const int64_t j = j0 + r, v = v0 + c;
        uint32_t out[4] = {0, 0, 0, 0};
        if (j < d && v < V) {
          float x[16];
          load16_scaled<T, decltype(any)::value>(w + j * ld + v, V - v, scale, x);
#pragma unroll
          for (int m = 0; m < 4; ++m) out[m] = cvt4_e4m3(x[4 * m], x[4 * m + 1], x[4 * m + 2], x[4 * m + 3]);
        }
        *reinterpret_cast<v4i*>(wq + blocked_offset(j, v, kbv)) = (v4i){(int)out[0], (int)out[1], (int)out[2], (int)out[3]};
#pragma unroll
        for (int m = 0; m < 4; ++m) *reinterpret_cast<uint32_t*>(&tile[r][c + 4 * m]) = out[m];
      }
    };
    if (rows_aligned(w, ld)) fill(std::false_type()); else fill(std::true_type());
  }
  __syncthreads();
  if (j0 < dp) {
#pragma unroll
    for (int pass = 0; pass < 4; ++pass) {
      const int vr = (t >> 3) + 32 * pass, jc = (t & 7) * 16;
      uint32_t out[4];
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        out[m] = (uint32_t)tile[jc + 4 * m][vr] | ((uint32_t)tile[jc + 4 * m + 1][vr] << 8) |
                 ((uint32_t)tile[jc + 4 * m + 2][vr] << 16) | ((uint32_t)tile[jc + 4 * m + 3][vr] << 24);
      }
      *reinterpret_cast<v4i*>(wqt + (v0 + vr) * ldx + j0 + jc) = (v4i){(int)out[0], (int)out[1], (int)out[2], (int)out[3]};
    }
  }
}

// Both operands of the fp8 head in one launch: workgroups [0, nx) the rows of X, with the final norm or without, the rest the tiles of W
// (there are none with a weight cache that is filled already).  The first one also leaves what follows from scales on the device in the
// header (dc, or NULL).  Neither operand needs the other, and on few rows X is all launch and latency.  Measured, in launches of their own
// (quantize_pad_kernel or with the norm rmsnorm_quantize_kernel, quantize_w_kernel, one of one thread for dc) and like this: 2048 rows, d = 768, fp32, V = 50304
// 5.6 + 53 and 54 us; 4096 rows, d = 1600 with norm and device scales 4 + 13 + 65 and 74; 1000 rows, d = 256, V = 4096 5.1 + 8.3
// and 10; 30011 rows, d = 2560 41 + 91 and 127; 2048 rows, d = 1024 with the weight's bytes from a cache 6.5 either way.
struct QuantizeParams {
  const void* x;
  int64_t x_ld, N, d, Np, dp, ldx;
  uint8_t* xq;
  float* rstd;                 // non-NULL: the norm is part of the call
  float eps, inv_xs, inv_ws;
  const float *xs_dev, *ws_dev;
  int nx;
  const void* w;
  int64_t w_ld, V, kbv;
  int nv;                      // tiles of W side by side
  uint8_t *wq, *wqt;
  DevConsts* dc;
  float xs_host, ws_host, cap;
};
template <typename TX, typename TW>
__global__ __launch_bounds__(256) void quantize_operands_kernel(QuantizeParams p) {
  __shared__ QwTile tile;
  const int b = blockIdx.x;
  if (b == 0 && threadIdx.x == 0 && p.dc) dev_consts(p.xs_dev, p.ws_dev, p.xs_host, p.ws_host, p.cap, p.dc);
  if (b >= p.nx) quantize_w<TW>(tile, (b - p.nx) % p.nv, (b - p.nx) / p.nv, (const TW*)p.w, p.w_ld, p.d, p.V, p.wq, p.wqt, p.dp, p.ldx, p.kbv, p.inv_ws, p.ws_dev);
  else if (p.rstd) rmsnorm_quantize<TX>(b, (const TX*)p.x, p.x_ld, p.N, p.d, p.eps, p.xq, p.Np, p.dp, p.ldx, p.inv_xs, p.xs_dev, p.rstd);
  else quantize_pad<TX>(b, p.nx, (const TX*)p.x, p.x_ld, p.N, p.d, p.xq, p.Np, p.dp, p.ldx, p.inv_xs, p.xs_dev);
}

// bf16 operands (the eval head, tiny/train.py:741 under bf16 autocast): no quantisation, only the layout.
// 8 consecutive elements as bf16 bits; `vec`: all 8 are there and the run is 16-byte aligned.  Elements at or beyond `valid` are 0.
template <typename T>
__device__ __forceinline__ v4i load8_bf16(const T* __restrict__ p, int64_t valid, bool vec) {
  if constexpr (sizeof(T) == 2) {
    if (vec) return *reinterpret_cast<const v4i*>(p);
  }
  uint32_t out[4] = {0, 0, 0, 0};
  if (vec) {
    const v4f a = *reinterpret_cast<const v4f*>(p), b = *reinterpret_cast<const v4f*>(p + 4);
#pragma unroll
    for (int m = 0; m < 2; ++m) {
      out[m] = (uint32_t)float_to_bf16_bits(a[2 * m]) | ((uint32_t)float_to_bf16_bits(a[2 * m + 1]) << 16);
      out[2 + m] = (uint32_t)float_to_bf16_bits(b[2 * m]) | ((uint32_t)float_to_bf16_bits(b[2 * m + 1]) << 16);
    }
  } else {
#pragma unroll
    for (int m = 0; m < 8; ++m)
      if (m < valid) out[m >> 1] |= (uint32_t)float_to_bf16_bits(Elem<T>::load(p + m)) << (16 * (m & 1));
  }
  return (v4i){(int)out[0], (int)out[1], (int)out[2], (int)out[3]};
}

// dst [rows_p][cols_p] bf16 = src [rows][cols] rounded to bf16 (RNE, as autocast's cast), zero outside; 8 outputs per thread.
template <typename T>
__global__ __launch_bounds__(256) void prep_x_bf16_kernel(const T* __restrict__ src, int64_t ld, int64_t rows, int64_t cols,
                                                         uint16_t* __restrict__ dst, int64_t rows_p, int64_t cols_p, int64_t dst_ld) {
  const int64_t chunks_per_row = cols_p / 8;
  const int64_t total = rows_p * chunks_per_row;
  for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q < total; q += (int64_t)gridDim.x * blockDim.x) {
    const int64_t r = q / chunks_per_row, c0 = (q - r * chunks_per_row) * 8;
    v4i out = (v4i){0, 0, 0, 0};
    if (r < rows && c0 < cols) {
      const T* p = src + r * ld + c0;
      out = load8_bf16<T>(p, cols - c0, cols - c0 >= 8 && ((uintptr_t)p & 15) == 0);
    }
    *reinterpret_cast<v4i*>(dst + r * dst_ld + c0) = out;
  }
}

// W (d, V) -> W^T [Vp][dp2 / 2] in bf16 (row stride ldw elements), in tiles of 64 rows x 128 columns through LDS: loads and stores of 16
// bytes, whole 256-byte pieces of the rows of W and whole 128-byte lines of W^T.  The transposing read (ds_read_b64_tr_b16: of the 4 x 16
// matrix that 16 lanes point at, 8 bytes each, lane i gets column i) hands a lane eight rows of its column in two reads.
// HBM-bound, 4 bytes an element from bf16: 2560 x 50304 in 197 us with an element to an access (2.6 TB/s), 163 with 16-byte
// accesses and tiles of 128 rows (36 KB of LDS leave a CU four workgroups), 88 with these (5.8 TB/s, eight workgroups).
constexpr int PREP_W_ROWS = 64;
template <typename T>
__global__ __launch_bounds__(256) void prep_w_bf16_kernel(const T* __restrict__ w, int64_t ld, int64_t d, int64_t V,
                                                         uint16_t* __restrict__ wt, int64_t ldw) {
  constexpr int TILE = 128, TJ = PREP_W_ROWS, PITCH = 2 * TILE + 32;
  __shared__ __attribute__((aligned(16))) uint8_t tile[TJ * PITCH];
  const int t = threadIdx.x;
  const int64_t j0 = (int64_t)blockIdx.y * TJ, v0 = (int64_t)blockIdx.x * TILE;
  const bool aligned = ((reinterpret_cast<uintptr_t>(w) | (uintptr_t)(ld * (int64_t)sizeof(T))) & 15) == 0;
  {
    v4i x[TJ / 16];
    const int64_t v = v0 + (t & 15) * 8;
#pragma unroll
    for (int pass = 0; pass < TJ / 16; ++pass) {
      const int64_t j = j0 + (t >> 4) + 16 * pass;
      x[pass] = (v4i){0, 0, 0, 0};
      if (j < d && v < V) x[pass] = load8_bf16<T>(w + j * ld + v, V - v, aligned && v + 8 <= V);
    }
#pragma unroll
    for (int pass = 0; pass < TJ / 16; ++pass) *reinterpret_cast<v4i*>(tile + ((t >> 4) + 16 * pass) * PITCH + (t & 15) * 16) = x[pass];
  }
  __syncthreads();
  typedef short v4s __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) v4s lds_v4s;
  const int lane = t & 63, wave = t >> 6, g = lane >> 4, i = lane & 15;
#pragma unroll
  for (int vb = 0; vb < 2; ++vb) {
    const int vc = wave * 32 + vb * 16;                        // 16 columns of the tile, one for each lane of a group
#pragma unroll
    for (int s = 0; s < TJ / 32; s += 2) {                     // rows 32 s + 8 g on, and 32 (s + 1) + 8 g on
      v4i q[2];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const uint8_t* src = tile + (32 * (s + u) + 8 * g + (i >> 2)) * PITCH + 2 * vc + 8 * (i & 3);
        const v2i lo = __builtin_bit_cast(v2i, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s*)src));
        const v2i hi = __builtin_bit_cast(v2i, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s*)(src + 4 * PITCH)));
        q[u] = (v4i){lo[0], lo[1], hi[0], hi[1]};
      }
      uint16_t* dst = wt + (v0 + vc + i) * ldw + j0 + 32 * s + 8 * g;
      *reinterpret_cast<v4i*>(dst) = q[0];
      *reinterpret_cast<v4i*>(dst + 32) = q[1];
    }
  }
}

// flat cast, for the standalone sce_quantize_e4m3 entry point: 16 elements a thread, their 32 or 64 bytes in 16-byte loads
// and the result in one 16-byte store, at whatever address they lie; element by element at the end.  HBM-bound: 3 bytes an
// element in bf16; 75 us for 2560 x 50257 whether the source is aligned or one element off (four elements a thread in
// 2-byte loads: 145 and 153; 16 a thread one by one: 268).  From the end of the tensor to its start: what a caller has done with the
// tensor before -- taken its maximum, written it -- went from the start to the end, and the 256 MB memory-side cache holds the
// end; and what comes after finds the start of the result there.  2560 x 50304 in bf16 between amax_kernel and transpose_bytes_kernel
// 79 -> 74 us, the transpose 51 -> 44.
template <typename T>
__global__ __launch_bounds__(256) void quantize_flat_kernel(const T* __restrict__ src, uint8_t* __restrict__ dst,
                                                           size_t n, float inv_scale, const float* __restrict__ scale_dev) {
  const Scaler scale = make_scaler<T>(inv_scale, scale_dev);
  for (size_t q = ((size_t)(gridDim.x - 1 - blockIdx.x) * blockDim.x + threadIdx.x) * 16; q < n; q += (size_t)gridDim.x * blockDim.x * 16) {
    const int64_t left = (int64_t)(n - q);
    float v[16];
    load16_scaled<T, true>(src + q, left, scale, v);
    uint32_t w[4];
#pragma unroll
    for (int m = 0; m < 4; ++m) w[m] = cvt4_e4m3(v[4 * m], v[4 * m + 1], v[4 * m + 2], v[4 * m + 3]);
    if (left >= 16) {
      *reinterpret_cast<v4i_any*>(dst + q) = (v4i){(int)w[0], (int)w[1], (int)w[2], (int)w[3]};
    } else {
#pragma unroll
      for (int m = 0; m < 16; ++m)
        if (m < left) dst[q + m] = (uint8_t)(w[m >> 2] >> (8 * (m & 3)));
    }
  }
}

// max |src| / 448 over n elements into *bits, as the bits of a non-negative float (they order like unsigned integers,
// NaN above everything); *bits starts at 0 (amax_begin_kernel).  The division comes before the maximum over the
// workgroups: it is monotonic, so the result is the same and needs no kernel of its own.  HBM-bound: a workgroup walks
// pieces of AMAX_LOADS x 4 KB with all its 16-byte loads in flight (a 2-byte load at a time: 1.8 TB/s).  All the maxima
// meet in one address, which takes them one at a time, so there are AMAX_GRID workgroups, two to a CU, and one whose
// maximum is not above what is there already stays away.  2560 x 50304 bf16, read just before: 38 us with 512 workgroups,
// 45 with 2048, 62 with 4096 (38 with each of them and no maximum stored); 1600 x 50304 26, 39 and 58.
__global__ void amax_begin_kernel(uint32_t* bits) { *bits = 0u; }
constexpr int AMAX_LOADS = 8, AMAX_GRID = 512;
template <typename T>
__global__ __launch_bounds__(256) void amax_kernel(const T* __restrict__ src, size_t n, uint32_t* __restrict__ bits) {
  __shared__ uint32_t smax[4];
  constexpr int PER = 16 / sizeof(T);
  uint32_t m = 0u;
  auto take = [&](uint32_t b) { b &= 0x7fffffffu; m = b > m ? b : m; };
  // the elements before the first 16-byte boundary, and those after the last whole load, one by one
  size_t head = ((16 - ((uintptr_t)src & 15)) & 15) / sizeof(T);
  if (head > n) head = n;
  const size_t loads = (n - head) / PER, tail = head + loads * PER;
  const v4i* vec = reinterpret_cast<const v4i*>(src + head);
  for (size_t q0 = (size_t)blockIdx.x * (256 * AMAX_LOADS) + threadIdx.x; q0 < loads; q0 += (size_t)gridDim.x * (256 * AMAX_LOADS)) {
    v4i r[AMAX_LOADS];
#pragma unroll
    for (int k = 0; k < AMAX_LOADS; ++k) r[k] = vec[q0 + k * 256 < loads ? q0 + k * 256 : q0];
#pragma unroll
    for (int k = 0; k < AMAX_LOADS; ++k)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if constexpr (sizeof(T) == 2) { take((uint32_t)r[k][e] << 16); take((uint32_t)r[k][e] & 0xffff0000u); }
        else take((uint32_t)r[k][e]);
      }
  }
  if (blockIdx.x == 0) {
    for (size_t q = threadIdx.x; q < head; q += 256) take(__float_as_uint(Elem<T>::load(src + q)));
    for (size_t q = tail + threadIdx.x; q < n; q += 256) take(__float_as_uint(Elem<T>::load(src + q)));
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) { const uint32_t x = (uint32_t)__shfl_xor((int)m, o); m = x > m ? x : m; }
  if ((threadIdx.x & 63) == 0) smax[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < 4; ++w) m = smax[w] > m ? smax[w] : m;
    m = __float_as_uint(__uint_as_float(m) / 448.0f);
    if (__hip_atomic_load(bits, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < m) atomicMax(bits, m);
  }
}

// dst (cols, rows) = src (rows, cols)^T, bytes, in 128 x 128 tiles: whole 128-byte lines both ways.  On the way out of
// LDS the transposing read gives a lane eight rows of its column at once (16 lanes point at 8 rows of 16 bytes, 8 bytes
// each, and lane j receives column j).  Both sides move 16 bytes at a time wherever 16 are there, aligned or not; only the
// last few of a row go byte by byte.  HBM-bound, 2 bytes an element: 50 us for
// 2560 x 50304 (164 with every byte an access of its own), 89 for 2561 x 50257 where no row is aligned (131 with bytes, 341
// with a lane's 16 bytes one by one: neighbouring lanes then touch different lines).
constexpr int TB_TILE = 128, TB_PITCH = TB_TILE + 16;
__global__ __launch_bounds__(256) void transpose_bytes_kernel(const uint8_t* __restrict__ src, uint8_t* __restrict__ dst,
                                                             int64_t rows, int64_t cols) {
  __shared__ __attribute__((aligned(16))) uint8_t tile[TB_TILE * TB_PITCH];
  const int t = threadIdx.x;
  const int64_t r0 = (int64_t)blockIdx.y * TB_TILE, c0 = (int64_t)blockIdx.x * TB_TILE;
  {
    v4i raw[4];
#pragma unroll
    for (int pass = 0; pass < 4; ++pass) {
      const int64_t r = r0 + (t >> 3) + 32 * pass, c = c0 + (t & 7) * 16;
      raw[pass] = (v4i){0, 0, 0, 0};
      if (r < rows && c < cols) {
        if (c + 16 <= cols) raw[pass] = *reinterpret_cast<const v4i_any*>(src + r * cols + c);
        else
          for (int m = 0; m < 16 && c + m < cols; ++m) raw[pass][m >> 2] |= (int)((uint32_t)src[r * cols + c + m] << (8 * (m & 3)));
      }
    }
#pragma unroll
    for (int pass = 0; pass < 4; ++pass) *reinterpret_cast<v4i*>(&tile[((t >> 3) + 32 * pass) * TB_PITCH + (t & 7) * 16]) = raw[pass];
  }
  __syncthreads();
  // a wave takes 16 columns at a time: group g of 16 lanes the rows [16 g, +16) and [64 + 16 g, +16) of the tile
  const int lane = t & 63, wave = t >> 6, g = lane >> 4, i = lane & 15;
  typedef __attribute__((address_space(3))) v2i lds_v2i;
#pragma unroll
  for (int pass = 0; pass < 4; ++pass) {
    const int cc = (wave * 2 + (pass & 1)) * 16, rr = 16 * g + 64 * (pass >> 1);
    const uint8_t* s = &tile[(rr + (i >> 1)) * TB_PITCH + cc + 8 * (i & 1)];
    const v2i lo = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_v2i*)s), hi = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_v2i*)(s + 8 * TB_PITCH));
    const int64_t c = c0 + cc + i, r = r0 + rr;
    if (c < cols && r < rows) {
      uint8_t* d = dst + c * rows + r;
      if (r + 16 <= rows) *reinterpret_cast<v4i_any*>(d) = (v4i){lo[0], lo[1], hi[0], hi[1]};
      else {
        const int w[4] = {lo[0], lo[1], hi[0], hi[1]};
#pragma unroll
        for (int m = 0; m < 16; ++m)
          if (r + m < rows) d[m] = (uint8_t)((uint32_t)w[m >> 2] >> (8 * (m & 3)));
      }
    }
  }
}

}  // namespace sce
