// Backward kernels: row factors, transposed scaled X, recompute, dX, dW (with its K-split last round), the one-hot
// part of dW from the sorted targets, finalisation (internal header).
// Part of the one translation unit sce_kernels.hip, which includes it after the headers it builds on.
#pragma once

namespace sce {

// ------------------------------------------------------------------------------------------
// backward
// ------------------------------------------------------------------------------------------
// Up to RANK_MAX (offset, row) entries are put in the order of their targets by counting: entry e goes to the place that is
// the number of entries before it, n compares spread over 16 lanes, all n keys in LDS.  (target, e) is one 32-bit number, so ties
// keep their order, as in the radix sort that larger calls use.  That sort is 3 to 4 launches of 4.8 us each whatever
// the size (20 us at 2048 entries, 16 at 4096); this is blocks of bwd_prep_kernel's own launch, for it needs nothing but the targets, and
// takes that kernel from 5 us to 7 and 9.8.  n^2 grows past the sort soon after.
constexpr int RANK_BITS = 12, RANK_MAX = 1 << RANK_BITS, RANK_PER_BLOCK = 16;
__device__ __forceinline__ void rank_targets(uint32_t* keys, int block, const int64_t* __restrict__ targets, int64_t ignore_index, int N, int Np, int V,
                                             int32_t key_none, int n_predict, int32_t* __restrict__ skeys, int32_t* __restrict__ perm) {
  const int n = N * n_predict, n64 = (n + 63) & ~63, t = threadIdx.x;
  for (int e0 = t; e0 < n64; e0 += 8 * 256) {
    int64_t y[8];                        // (eight loads in flight: one at a time they were the whole time, 13 us for 4096 entries)
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int e = e0 + 256 * u, k = e / N, i = e - k * N + k;
      y[u] = e < n && i < N ? targets[i] : ignore_index;
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int e = e0 + 256 * u;
      const uint32_t key = y[u] != ignore_index && y[u] >= 0 && y[u] < V ? (uint32_t)y[u] : (uint32_t)key_none;
      if (e < n64) keys[e] = e < n ? (key << RANK_BITS) | (uint32_t)e : ~0u;
    }
  }
  __syncthreads();
  const int e = block * RANK_PER_BLOCK + (t >> 4);
  const uint32_t mine = e < n ? keys[e] : 0u;
  int before = 0;
  for (int q = 4 * (t & 15); q < n64; q += 64) {
    const uint4 c = *reinterpret_cast<const uint4*>(keys + q);
    before += (c.x < mine) + (c.y < mine) + (c.z < mine) + (c.w < mine);
  }
#pragma unroll
  for (int o = 8; o > 0; o >>= 1) before += __shfl_xor(before, o);
  if ((t & 15) == 0 && e < n) {
    skeys[before] = (int32_t)(mine >> RANK_BITS);
    perm[before] = (e / N) * Np + e % N;
  }
}

// per row: rho (row factor of the block-scaled dlogits) and h_k (one-hot coefficients).
//   dz_iv = g_i ( S_i p_iv - sum_k w_k [v = y_{i+k}] ),  S_i = sum of w_k over the offsets that take part,
//   S_i p_iv (1 - t^2) = rho_i (D_iv 2^{lam_i})  with  rho_i = g_i S_i e^{cap - lse_i} 2^{-lam_i}.
// The target columns take no part in D (take_target_logits knocks them out where D is formed): their S_i p_iy goes into the
// one-hot coefficient instead, h_ik = g_i (1 - t_y^2) (w_k - S_i p_iy), formed here in fp32 from lse and z_y.
// Through e4m3 the difference S_i p_iy - w_k would carry the rounding error of p_iy alone, a relative
// error of eps p / (1 - p) that grows without bound on rows the model is sure of.  When two offsets of a row
// have the same target, the first one carries the S_i p_iy term.
__global__ __launch_bounds__(256) void bwd_prep_kernel(const float* __restrict__ s_lse,
                                                      const float* __restrict__ s_zy, const int64_t* __restrict__ targets,
                                                      int64_t ignore_index, const int32_t* __restrict__ hdr,
                                                      const float* __restrict__ grad_output, int per_row, float grad_scale,
                                                      const float* __restrict__ mtp_weights, int n_predict,
                                                      float cap, int N, int Np, int V, const float* __restrict__ lam, const float* __restrict__ lam2,
                                                      float* __restrict__ rho, float* __restrict__ hcoef,
                                                      float* __restrict__ blockmax, int32_t* __restrict__ rowinfo, CallMode mode,
                                                      int32_t key_none, int32_t* __restrict__ keys, int32_t* __restrict__ vals,
                                                      int32_t* __restrict__ longlist, int32_t* __restrict__ skeys, int32_t* __restrict__ perm) {
  __shared__ float smax[256];
  __shared__ __attribute__((aligned(16))) uint32_t rank_keys[RANK_MAX];
  // blocks beyond the rows' (there are some with few entries only): the entries' places
  if ((int)blockIdx.x >= Np / 256) return rank_targets(rank_keys, blockIdx.x - Np / 256, targets, ignore_index, N, Np, V, key_none, n_predict, skeys, perm);
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < 3) longlist[i] = 0;         // counters of the long-column lists, filled by column_segments
  float r = 0.f;
  float h[4] = {0.f, 0.f, 0.f, 0.f};
  // the forward call that wrote `saved` was asked for something else (kept dlogits, vocabulary limit, offsets, cap):
  // its state does not fit this call, and every gradient comes out NaN rather than silently wrong
  const CallMode fm = *reinterpret_cast<const CallMode*>(reinterpret_cast<const uint8_t*>(hdr) + HDR_MODE_OFF);
  const bool mismatch = fm.emit != mode.emit || fm.vocab_limit != mode.vocab_limit || fm.n_predict != mode.n_predict || fm.cap_bits != mode.cap_bits;
  // The row's exponent boost.  A forward pass that emitted the dlogits had to estimate the row's sum from a sample of
  // the row (fwd_sample_kernel).  When the dlogits are formed again here in backward, the sum Z = e^{lse - cap} is known, and
  // the boost is what makes the stored value the probability itself, D 2^lam = p (1 - t^2): rows
  // that share a block are then weighed by what their entries contribute, whatever the shapes of their distributions.
  float lam_i = 0.f;
  if (i < N) lam_i = rowinfo ? (cap - s_lse[i]) * LOG2E : row_boost(lam, lam2, i);
  if (!(lam_i >= -64.f && lam_i <= 120.f)) lam_i = 0.f;      // (ignored rows have no lse to speak of)
  if (rowinfo && i < Np) {          // what the recompute kernel wants to know of a row: its boost and its target columns
    rowinfo[i] = __float_as_int(lam_i);
    for (int k = 0; k < 4; ++k)
      rowinfo[(int64_t)(1 + k) * Np + i] = (k < n_predict && i < N && target_valid(targets, ignore_index, i + k, N, V)) ? (int)targets[i + k] : -1;
    for (int k = 0; k < 4; ++k)          // and the target logits as the forward pass saved them: the recompute kernel knows its targets by these values
      rowinfo[(int64_t)(5 + k) * Np + i] = (k < n_predict && i < N) ? __float_as_int(s_zy[(int64_t)k * Np + i]) : 0x7fc00000;
  }
  if (i < N) {
    const float g = (per_row ? grad_output[i] : grad_output[0] / (float)hdr[0]) * grad_scale;
    float sw = 0.f;
    bool ok[4] = {false, false, false, false};
    int64_t yk[4] = {0, 0, 0, 0};
    for (int k = 0; k < n_predict; ++k) {
      ok[k] = target_valid(targets, ignore_index, i + k, N, V);
      if (!ok[k]) continue;
      yk[k] = targets[i + k];
      sw += mtp_weights ? mtp_weights[k] : 1.0f;
    }
    // sort keys of the rows grouped by target (keys == NULL: ranked by this launch's other blocks): one entry per (offset k, row i): key = target y_{i+k} (key_none if the pair
    // takes no part), value = entry id k * Np + i
    for (int k = 0; k < n_predict && keys; ++k) {
      keys[(int64_t)k * N + i] = ok[k] ? (int32_t)yk[k] : key_none;
      vals[(int64_t)k * N + i] = k * Np + i;
    }
    if (ok[0] || ok[1] || ok[2] || ok[3]) {
      const float lse = s_lse[i];
      for (int k = 0; k < n_predict; ++k) {
        if (!ok[k]) continue;
        const float wk = mtp_weights ? mtp_weights[k] : 1.0f;
        const float zy = s_zy[(int64_t)k * Np + i];
        const float ty = zy / cap;
        bool first = true;
        for (int k2 = 0; k2 < k; ++k2) first = first && !(ok[k2] && yk[k2] == yk[k]);
        h[k] = g * (1.0f - ty * ty) * (wk - (first ? sw * expf(zy - lse) : 0.f));
      }
      // the stored dlogits carry the row's boost 2^lam: an integer from the forward pass that emitted them, the real
      // (cap - lse) log2(e) here -- then rho_i 2^-lam_i is g_i times the row's weights and nothing else, the same number for
      // nearly every row of a mean-reduced loss, and the scaled X that dW multiplies with is X_q itself: no second rounding
      r = rowinfo ? g * sw * expf(cap - lse - lam_i * 0.6931471805599453f) : ldexpf(g * sw * expf(cap - lse), -(int)lam_i);
    }
  }
  if (mismatch && i < N) {
    r = NAN;
    for (int k = 0; k < 4; ++k) h[k] = NAN;
  }
  if (i < Np) {
    rho[i] = r;
    for (int k = 0; k < n_predict; ++k) hcoef[(int64_t)k * Np + i] = h[k];
  }
  smax[threadIdx.x] = fabsf(r);
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (threadIdx.x < w) smax[threadIdx.x] = fmaxf(smax[threadIdx.x], smax[threadIdx.x + w]);
    __syncthreads();
  }
  if (threadIdx.x == 0) blockmax[blockIdx.x] = smax[0];
}

// Xt (blocked, dq rows, K = Np) = e4m3( X_q[i][j] * rho_i / xi ), transposed through LDS in 128 x 128 tiles: a row of
// the tile is one whole 128-byte line of the blocked layout on the way out, and 128 bytes of an X_q row on the way in.
// xi, the largest |rho|, is folded from bwd_prep_kernel's block maxima by every workgroup for itself (one load a thread at
// N = 65536, from L2, beside the loads of the tile): a launch of one workgroup for it was 4.7 us of every backward call.
constexpr int XT_TILE = 128;
struct XtShared { uint8_t tile[XT_TILE][XT_TILE + 4]; float wmax[4]; };
__device__ __forceinline__ void xt_tile(XtShared& shared, int bx, int by, const uint8_t* __restrict__ xq, int64_t dp, int64_t ldx, int64_t kbn,
                                        const float* __restrict__ rho, const float* __restrict__ blockmax, int nblk,
                                        float* __restrict__ xi_out, uint8_t* __restrict__ xt) {
  auto& tile = shared.tile;
  auto& wmax = shared.wmax;
  const int t = threadIdx.x;
  float xi = 0.f;
  for (int n = t; n < nblk; n += 256) xi = fmaxf(xi, blockmax[n]);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) xi = fmaxf(xi, __shfl_xor(xi, o));
  if ((t & 63) == 0) wmax[t >> 6] = xi;
  __syncthreads();
  xi = fmaxf(fmaxf(wmax[0], wmax[1]), fmaxf(wmax[2], wmax[3]));
  xi = (xi > 0.f && isfinite(xi)) ? xi : 1.0f;
  if (bx == 0 && by == 0 && t == 0) xi_out[0] = xi;
  const int64_t i0 = (int64_t)bx * XT_TILE, j0 = (int64_t)by * XT_TILE;
  if (j0 < dp) {
#pragma unroll
    for (int pass = 0; pass < 4; ++pass) {
      const int r = (t >> 3) + 32 * pass, c = (t & 7) * 16;
      const v4i raw = *reinterpret_cast<const v4i*>(xq + (i0 + r) * ldx + j0 + c);
      const float f = rho[i0 + r] / xi;
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        const uint32_t w = (uint32_t)raw[m];
        const uint32_t o = cvt4_e4m3(e4m3_to_float<0>(w) * f, e4m3_to_float<1>(w) * f, e4m3_to_float<2>(w) * f,
                                     e4m3_to_float<3>(w) * f);
        *reinterpret_cast<uint32_t*>(&tile[r][c + 4 * m]) = o;
      }
    }
  } else {
    for (int e = t; e < XT_TILE * (XT_TILE + 4) / 4; e += 256) reinterpret_cast<uint32_t*>(&tile[0][0])[e] = 0;
  }
  __syncthreads();
#pragma unroll
  for (int pass = 0; pass < 4; ++pass) {
    const int jr = (t >> 3) + 32 * pass, ic = (t & 7) * 16;
    uint32_t out[4];
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      out[m] = (uint32_t)tile[ic + 4 * m][jr] | ((uint32_t)tile[ic + 4 * m + 1][jr] << 8) |
               ((uint32_t)tile[ic + 4 * m + 2][jr] << 16) | ((uint32_t)tile[ic + 4 * m + 3][jr] << 24);
    }
    *reinterpret_cast<v4i*>(xt + blocked_offset(j0 + jr, i0 + ic, kbn)) = (v4i){(int)out[0], (int)out[1], (int)out[2], (int)out[3]};
  }
}

struct RecomputeParams {
  const uint8_t* xq;     // [Np][dp], already offset to the panel's first row
  const uint8_t* wqt;    // [Vp][dp]
  uint8_t* ghat_t;       // G of the rows this buffer stands for, tile by tile (kbv blocks of 128 columns per tile of 256 rows)
  uint32_t* gexp;        // [Vp / 128][kbw]
  const int32_t* rowinfo;      // [ROWINFO_PLANES][Np], offset to the panel's first row: boosts and targets (bwd_prep_kernel)
  int64_t Np;
  int n_predict;
  int64_t dp, ldx;             // K extent and row stride of xq / wqt
  int64_t kbw, kb0, kbv;       // blocks of 128 rows in the buffer (row stride of gexp), block of this panel's first row, blocks of 128 columns
  int RT, CT, V;
  float k1, c2, sc;      // as in FwdParams
  const DevConsts* dc;   // non-NULL: k1 and sc come from here
};

// Recompute a 256 x 256 logit tile and leave its block-scaled dlogits in G (16-byte stores straight from the registers).
constexpr int ROWINFO_PLANES = 9;                      // per row: exponent boost (a float), the target column of each of 4 offsets (or -1), the target logits
constexpr int SMEM_RECOMPUTE = SMEM_BYTES + 4 * ROWINFO_PLANES * 512;      // two K slots + the row data of 128 rows per wave

__global__ __launch_bounds__(256) void bwd_recompute_kernel(RecomputeParams p_in) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  RecomputeParams p = p_in;
  if (p.dc) { p.k1 = p.dc->k1; p.sc = p.dc->sc; }
  int rt, ct;
  if (!map_tile(blockIdx.x, p.RT, p.CT, rt, ct)) return;
  // The tile order goes through the columns in groups of 8, and it does so from the last group to the first:
  // the dX kernel that follows starts its K loop at column 0, with the part of G that was written last and is
  // still in the memory-side cache.
  ct = p.CT - 1 - ct;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wa = wave >> 1, wb = wave & 1;
  // The boosts and targets of the wave's 128 rows go straight to LDS, behind the two slots: requested before the K
  // loop (whose waits for its own, younger loads cover them), read after it, no register held in between.
  // (Through the compiler's builtin, which knows that the instruction reads M0 and sets it itself; the price -- the
  // compiler makes the first LDS read after it wait for every vector memory load in flight, the tile loads of the
  // main loop's prologue included -- is paid once per tile here.)
  {
    typedef __attribute__((address_space(3))) uint8_t lds_u8;
    typedef const __attribute__((address_space(1))) int32_t global_i32;
    lds_u8* dst = (lds_u8*)(smem + SMEM_BYTES) + wave * (ROWINFO_PLANES * 512);
    const int lane = lane_id();
#pragma unroll
    for (int q = 0; q < ROWINFO_PLANES; ++q) {
      global_i32* src = (global_i32*)(uintptr_t)(p.rowinfo + (int64_t)q * p.Np + rt * 256 + wb * 128 + lane);
      // lane l's dword lands at the LDS base + 4 l; the instruction's offset moves the memory address and the LDS
      // address alike: the second half of the rows
      __builtin_amdgcn_global_load_lds(src, dst + q * 512, 4, 0, 0);
      __builtin_amdgcn_global_load_lds(src, dst + q * 512, 4, 256, 0);
    }
  }
  v16f acc[4][4];
  // (as in the forward kernel: the last pair's MFMAs of row blocks 1 - 3 ride along with the epilogues of row blocks 0 and 1)
  mfma_mainloop<false, NoHook, BK, false, 0, false, true>(p.wqt + (int64_t)ct * 256 * p.ldx, p.ldx, p.xq + (int64_t)rt * 256 * p.ldx, p.ldx, (int)(p.dp / BK), smem, acc, 2 * (rt & 3), ct & 7, wave);
  DeferredTail<> deferred(smem, wa, wb);
  auto tail = [&](int b, int k) { deferred(acc, b, k); };
  const int vlim = p.V - ct * 256;           // columns >= vlim of this tile do not exist
  const bool ragged = vlim < 256;
  const float* lam = reinterpret_cast<const float*>(smem + SMEM_BYTES) + wave * (ROWINFO_PLANES * 128);     // row block b: 32 floats on
  const int* tgt = reinterpret_cast<const int*>(smem + SMEM_BYTES) + wave * (ROWINFO_PLANES * 128) + 128;
  uint8_t* gq = const_cast<uint8_t*>(uniform_ptr(p.ghat_t + ((p.kb0 / 2 + rt) * p.kbv + 2 * ct + wa) * BLOCKED_KSTEP + wb * 128 * BK));      // the wave's quadrant of G
  const int col0 = ct * 256 + wa * 128;
  // The target entries are not looked up in the accumulators (the compiler moves a row block's 64 accumulators around
  // every such lookup): a lane knows the value of a target among its columns -- the forward pass saved it, and this
  // kernel computes the same number -- and keeps it out of the block exponent by that (form_dlogits, EXCL); the bytes
  // are cleared afterwards (fwd_knock_kernel).
  const float* tval = reinterpret_cast<const float*>(tgt + 4 * 128);
  auto target_value = [&](int b) {
    float v = __builtin_nanf("");
    for (int k = 0; k < p.n_predict; ++k) {
      const int rel = tgt[k * 128 + b * 32 + (lane_id() & 31)] - col0;
      if ((unsigned)rel < 128u && ((rel >> 2) & 1) == (lane_id() >> 5)) v = tval[k * 128 + b * 32 + (lane_id() & 31)];
    }
    return v;
  };
  float xc[4];
  if (ragged) strike_columns_beyond<0, 1>(acc, vlim, wa);
  xc[0] = target_value(0);
  uint32_t ew = form_dlogits<false, 32, 32, 0, 1, decltype(tail)&, true>(acc, p.k1, p.c2, 0, gq, wa, wb, nullptr, lam, false, tail, xc, p.sc);
  if (ragged) strike_columns_beyond<1, 2>(acc, vlim, wa);
  xc[1] = target_value(1);
  ew |= form_dlogits<false, 32, 32, 1, 2, decltype(tail)&, true>(acc, p.k1, p.c2, 0, gq, wa, wb, nullptr, lam, false, tail, xc, p.sc);
  if (ragged) strike_columns_beyond<2, 4>(acc, vlim, wa);
  xc[2] = target_value(2); xc[3] = target_value(3);
  NoHook none;
  ew |= form_dlogits<false, 32, 32, 2, 4, NoHook&, true>(acc, p.k1, p.c2, 0, gq, wa, wb, nullptr, lam, false, none, xc, p.sc);
  if (lane_id() == 0) p.gexp[(int64_t)(2 * ct + wa) * p.kbw + p.kb0 + 2 * rt + wb] = ew;
}

struct DxParams {
  const uint8_t* wq;      // dq rows, K = Vp, tile by tile: A side (rows j)
  const uint8_t* ghat_t;  // G, tile by tile (rows i, K = v); already at the tile of the panel's first row    B side (rows i of the panel)
  const uint32_t* gexp;   // its block exponents [Vp / 128][kbw], likewise at the panel's first row
  const uint8_t* wqt;     // [Vp][dp]   for the one-hot gather
  const float* rho;       // offset to the panel
  const float* hcoef;     // [n_predict][Np], offset to the panel
  const int64_t* targets; // offset to the panel
  void* dx;               // offset to the panel's first row
  float* part;            // [ksplit][RT][CT] tiles of fp32 partial sums, as dx_part_offset lays them out (ksplit > 1 only)
  int64_t dx_ld, Vp, ldx, Np, dq;        // Vp: K extent; ldx: row stride of wqt
  int64_t kbw;                           // blocks of 128 rows i that gexp counts per block of 128 columns
  int RT, CT, rows, d, V;  // rows: valid rows in this panel
  int n_predict, rows_left; // rows_left: N - (first row of the panel), bounds the target look-ahead
  int ksplit;              // the K loop (V) is cut into this many parts, one workgroup each
  float w_s;
  const DevConsts* dc;     // non-NULL: w_s comes from here
};

// LDS a wave uses to stage its quadrant of a dX tile on the way out: 128 rows of 64 fp32 (or bf16) plus 16 bytes
constexpr int DX_STAGE_BYTES = 128 * (64 * 4 + 16);
constexpr int SMEM_DX = 4 * DX_STAGE_BYTES > SMEM_BYTES ? 4 * DX_STAGE_BYTES : SMEM_BYTES;
// ... or the two K slots and, behind them, the block exponents of the K loop (one dword per K block and half of the rows)
constexpr int MAX_SCALE_KBLOCKS = (SMEM_MAX - SMEM_BYTES) / 8;      // K blocks of one scaled main loop: 4096
static inline int smem_scaled(int kblocks, int at_least) { const int n = SMEM_BYTES + 8 * kblocks; return n > at_least ? n : at_least; }

// Row scale and one-hot term of four consecutive dX columns j..j+3 of panel row il:
//   dX = rho_i w_s (G W_q^T) - sum_k h_ik w_s W_q^T[y_{i+k}, :]
struct DxRowTerms {
  float rs;
  float hs[4];
  const uint8_t* wrow[4];
  __device__ __forceinline__ DxRowTerms(const DxParams& p, int il) {
    rs = p.rho[il] * p.w_s;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      hs[k] = 0.f; wrow[k] = p.wqt;
      if (k < p.n_predict && il + k < p.rows_left) {
        const float hk = p.hcoef[(int64_t)k * p.Np + il] * p.w_s;
        const int64_t y = p.targets[il + k];
        if (hk != 0.f && y >= 0 && y < p.V) { hs[k] = hk; wrow[k] = p.wqt + y * p.ldx; }
      }
    }
  }
  template <typename T>
  __device__ __forceinline__ void store4(const DxParams& p, T* dst, int j, float o0, float o1, float o2, float o3) const {
    // explicit roundings: the fast path of bwd_dx_kernel forms the same values and must give the same bits
    o0 = __fmul_rn(o0, rs); o1 = __fmul_rn(o1, rs); o2 = __fmul_rn(o2, rs); o3 = __fmul_rn(o3, rs);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      if (k < p.n_predict) {
        const uint32_t w = *reinterpret_cast<const uint32_t*>(wrow[k] + j);
        o0 = __builtin_fmaf(-hs[k], e4m3_to_float<0>(w), o0); o1 = __builtin_fmaf(-hs[k], e4m3_to_float<1>(w), o1);
        o2 = __builtin_fmaf(-hs[k], e4m3_to_float<2>(w), o2); o3 = __builtin_fmaf(-hs[k], e4m3_to_float<3>(w), o3);
      }
    }
    Elem<T>::store(dst + 0, o0); Elem<T>::store(dst + 1, o1);
    Elem<T>::store(dst + 2, o2); Elem<T>::store(dst + 3, o3);
  }
};

// The partial sums of a tile are private to the two kernels, so they lie as the accumulators do: for every 32 rows x 128 columns
// (il / 32, wa) the 16 registers quads (a, q) one behind the other, 64 lanes x 16 bytes each -- a wave's store is 1 KB in a row.
// In row order it was 32 pieces of 32 bytes, and waiting to issue them took two thirds of the kernel at 1000 rows, d = 256,
// V = 4096: 16.8 -> 12.6 us there, 89.5 -> 86 at 2048 rows, d = 1024, V = 50304.
__device__ __forceinline__ int64_t dx_part_offset(int64_t tile, int wb, int b, int wa) { return ((tile * 2 + wb) * 4 + b) * 8192 + wa * 4096; }

// SPLIT = false: one workgroup per 256 x 256 tile of dX, whole K loop, finished values stored.
// SPLIT = true : a panel with too few tiles to fill the chip; each tile's K loop is shared by ksplit
//                workgroups that store raw fp32 partial sums, and bwd_dx_finish_kernel adds them up.
template <typename T, bool SPLIT>
__global__ __launch_bounds__(256) void bwd_dx_kernel(DxParams p_in) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  DxParams p = p_in;
  if (p.dc) p.w_s = p.dc->w_s;
  int rt, ct, ks = 0;
  int64_t k0 = 0;
  int KD = (int)(p.Vp / BK);
  if (!SPLIT) {
    if (!map_tile(blockIdx.x, p.RT, p.CT, rt, ct)) return;
  } else {
    // The parts of the K loop are the slowest index of the order that the XCDs take eighths of: what one L2 serves is all (or
    // many) tiles of the panel over one stretch of K, so both operands come through it once and not once for every row
    // and column of tiles.  With the parts of a tile side by side instead, G was read by four XCDs and W_q by two each
    // (515 MB instead of 154 at N = 2048, d = 1024, V = 50304): 95.4 -> 89.5 us there.
    int lin, none;
    if (!map_tile(blockIdx.x, 1, p.RT * p.CT * p.ksplit, none, lin)) return;
    ks = __builtin_amdgcn_readfirstlane(lin / (p.RT * p.CT));
    tile_from_index(lin - ks * (p.RT * p.CT), p.RT, p.CT, rt, ct);
    rt = __builtin_amdgcn_readfirstlane(rt); ct = __builtin_amdgcn_readfirstlane(ct);
    const int pairs = KD >> 1;
    const int q0 = (int)((int64_t)pairs * ks / p.ksplit), q1 = (int)((int64_t)pairs * (ks + 1) / p.ksplit);
    k0 = (int64_t)q0 * 2 * BK; KD = 2 * (q1 - q0);
  }
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6, wa = wave >> 1, wb = wave & 1;
  // the block exponents of this tile's K loop wait in LDS behind the two K slots: [i half][K block]
  uint32_t* lsc = reinterpret_cast<uint32_t*>(smem + SMEM_BYTES);
  for (int e = t; e < 2 * KD; e += NTHREADS) {
    const int w = e >= KD, kb = e - w * KD;
    lsc[e] = p.gexp[(k0 / BK + kb) * p.kbw + 2 * rt + w];
  }
  __syncthreads();
  v16f acc[4][4];
  // both operands tile by tile with K = v: W_q rows j, G rows i
  mfma_mainloop<false, NoHook, BLOCKED_KSTEP, false, 1>(p.wq + ((int64_t)ct * (p.Vp / BK) + k0 / BK) * BLOCKED_KSTEP, BK,
                                                        p.ghat_t + ((int64_t)rt * (p.Vp / BK) + k0 / BK) * BLOCKED_KSTEP, BK, KD, smem, acc,
                                                        2 * (rt & 3), ct & 7, __builtin_amdgcn_readfirstlane(wave), NoHook(), 0, 0,
                                                        lsc + __builtin_amdgcn_readfirstlane(wb) * KD);
  const int jbase = ct * 256 + wa * 128 + 4 * (lane >> 5);
  T* dx = reinterpret_cast<T*>(p.dx);
  if (!SPLIT && p.n_predict > 1 && ((reinterpret_cast<uintptr_t>(p.dx) | (uintptr_t)(p.dx_ld * (int64_t)sizeof(T))) & 15) == 0) {
    // Several prediction offsets: the same staged way out as below, with the W_q^T words of all offsets loaded for one
    // block of 32 rows and 64 columns at a time (all at once they would not fit the registers; folded into the
    // accumulators beforehand, offset by offset, the whole kernel, main loop included, takes to scratch memory).
    // Values and their order are those of DxRowTerms::store4.
    const int K = p.n_predict;
    float rs[4], hs[4][4];
    int yrow[4][4];
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const int il = rt * 256 + wb * 128 + b * 32 + (lane & 31);
      const bool live = il < p.rows;
      rs[b] = p.rho[live ? il : 0] * p.w_s;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        hs[b][k] = 0.f; yrow[b][k] = 0;
        if (k < K) {
          const bool there = live && il + k < p.rows_left;
          const float hk = there ? p.hcoef[(int64_t)k * p.Np + il] * p.w_s : 0.f;
          const int64_t y = there ? p.targets[il + k] : -1;
          if (hk != 0.f && y >= 0 && y < p.V) { hs[b][k] = hk; yrow[b][k] = (int)y; }
        }
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    constexpr int RB = 64 * (int)sizeof(T), PITCH = RB + 16, CH = RB / 16;     // row bytes, staging pitch, chunks per row
    uint8_t* stg = smem + wave * DX_STAGE_BYTES;
#pragma unroll
    for (int pass = 0; pass < 2; ++pass) {
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        uint32_t wk[4][8];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          if (k < K) {
            const uint8_t* wrow = p.wqt + (int64_t)yrow[b][k] * p.ldx + jbase + pass * 64;
#pragma unroll
            for (int e = 0; e < 8; ++e) wk[k][e] = *reinterpret_cast<const uint32_t*>(wrow + (e >> 2) * 32 + 8 * (e & 3));
          }
        }
        __builtin_amdgcn_sched_barrier(0);
        uint8_t* srow = stg + (b * 32 + (lane & 31)) * PITCH + 4 * (lane >> 5) * (int)sizeof(T);
#pragma unroll
        for (int a2 = 0; a2 < 2; ++a2)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const int a = 2 * pass + a2;
            float o0 = __fmul_rn(acc[a][b][4 * q + 0], rs[b]), o1 = __fmul_rn(acc[a][b][4 * q + 1], rs[b]);
            float o2 = __fmul_rn(acc[a][b][4 * q + 2], rs[b]), o3 = __fmul_rn(acc[a][b][4 * q + 3], rs[b]);
#pragma unroll
            for (int k = 0; k < 4; ++k) {
              if (k < K) {
                const uint32_t w = wk[k][a2 * 4 + q];
                o0 = __builtin_fmaf(-hs[b][k], e4m3_to_float<0>(w), o0); o1 = __builtin_fmaf(-hs[b][k], e4m3_to_float<1>(w), o1);
                o2 = __builtin_fmaf(-hs[b][k], e4m3_to_float<2>(w), o2); o3 = __builtin_fmaf(-hs[b][k], e4m3_to_float<3>(w), o3);
              }
            }
            uint8_t* dst = srow + (a2 * 32 + 8 * q) * (int)sizeof(T);
            if constexpr (sizeof(T) == 2)
              *reinterpret_cast<v2i*>(dst) = (v2i){(int)((uint32_t)float_to_bf16_bits(o0) | ((uint32_t)float_to_bf16_bits(o1) << 16)),
                                                   (int)((uint32_t)float_to_bf16_bits(o2) | ((uint32_t)float_to_bf16_bits(o3) << 16))};
            else
              *reinterpret_cast<v4f*>(dst) = (v4f){o0, o1, o2, o3};
          }
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int n = 0; n < 128 * CH / 64; ++n) {
        const int c = lane + 64 * n, row = c / CH, k16 = c % CH;
        const int il = rt * 256 + wb * 128 + row;
        const int col = ct * 256 + wa * 128 + pass * 64 + k16 * (16 / (int)sizeof(T));
        if (il < p.rows && col < p.d)
          *reinterpret_cast<v4i*>(reinterpret_cast<uint8_t*>(dx) + ((int64_t)il * p.dx_ld + col) * (int64_t)sizeof(T)) =
              *reinterpret_cast<const v4i*>(stg + row * PITCH + k16 * 16);
      }
    }
    return;
  }
  if (!SPLIT && p.n_predict == 1) {
    // One wave per SIMD has nothing to hide a load behind, so the epilogue is written in three phases with all
    // loads of a phase in flight together: the row terms of the lane's four rows, then the 64 words of the four
    // W_q^T rows of their targets, then arithmetic and stores.
    float rs[4], hs[4];
    int64_t yy[4];
    int il4[4];
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const int il = rt * 256 + wb * 128 + b * 32 + (lane & 31);
      const bool live = il < p.rows;
      il4[b] = live ? il : -1;
      const int is = live ? il : 0;                       // row 0 exists whenever any row does
      rs[b] = p.rho[is] * p.w_s;
      hs[b] = p.hcoef[is] * p.w_s;
      yy[b] = p.targets[is];
    }
    __builtin_amdgcn_sched_barrier(0);
    uint32_t wv[4][16];
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const bool hit = il4[b] >= 0 && hs[b] != 0.f && yy[b] >= 0 && yy[b] < p.V;
      if (!hit) hs[b] = 0.f;
      const uint8_t* wrow = p.wqt + (hit ? yy[b] : 0) * p.ldx + jbase;
#pragma unroll
      for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int q = 0; q < 4; ++q) wv[b][4 * a + q] = *reinterpret_cast<const uint32_t*>(wrow + a * 32 + 8 * q);
    }
    __builtin_amdgcn_sched_barrier(0);
    // Out through LDS (free now: every wave is past the closing barrier of the main loop), so that the stores are
    // whole 16-byte runs of a row instead of 8-byte pieces of 32 different rows: each wave stages its own quadrant,
    // 64 columns at a time, and reads only what it wrote itself (no barrier).
    const bool vec = ((reinterpret_cast<uintptr_t>(p.dx) | (uintptr_t)(p.dx_ld * (int64_t)sizeof(T))) & 15) == 0;
    if (vec) {
      constexpr int RB = 64 * (int)sizeof(T), PITCH = RB + 16, CH = RB / 16;     // row bytes, staging pitch, chunks per row
      uint8_t* stg = smem + wave * DX_STAGE_BYTES;
#pragma unroll
      for (int pass = 0; pass < 2; ++pass) {
#pragma unroll
        for (int b = 0; b < 4; ++b) {
          uint8_t* srow = stg + (b * 32 + (lane & 31)) * PITCH + 4 * (lane >> 5) * (int)sizeof(T);
#pragma unroll
          for (int a2 = 0; a2 < 2; ++a2)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              const int a = 2 * pass + a2;
              const uint32_t w = wv[b][4 * a + q];
              const float o0 = __builtin_fmaf(-hs[b], e4m3_to_float<0>(w), __fmul_rn(acc[a][b][4 * q + 0], rs[b]));
              const float o1 = __builtin_fmaf(-hs[b], e4m3_to_float<1>(w), __fmul_rn(acc[a][b][4 * q + 1], rs[b]));
              const float o2 = __builtin_fmaf(-hs[b], e4m3_to_float<2>(w), __fmul_rn(acc[a][b][4 * q + 2], rs[b]));
              const float o3 = __builtin_fmaf(-hs[b], e4m3_to_float<3>(w), __fmul_rn(acc[a][b][4 * q + 3], rs[b]));
              uint8_t* dst = srow + (a2 * 32 + 8 * q) * (int)sizeof(T);
              if constexpr (sizeof(T) == 2)
                *reinterpret_cast<v2i*>(dst) = (v2i){(int)((uint32_t)float_to_bf16_bits(o0) | ((uint32_t)float_to_bf16_bits(o1) << 16)),
                                                     (int)((uint32_t)float_to_bf16_bits(o2) | ((uint32_t)float_to_bf16_bits(o3) << 16))};
              else
                *reinterpret_cast<v4f*>(dst) = (v4f){o0, o1, o2, o3};
            }
        }
#pragma unroll
        for (int n = 0; n < 128 * CH / 64; ++n) {
          const int c = lane + 64 * n, row = c / CH, k16 = c % CH;
          const int il = rt * 256 + wb * 128 + row;
          const int col = ct * 256 + wa * 128 + pass * 64 + k16 * (16 / (int)sizeof(T));
          if (il < p.rows && col < p.d)
            *reinterpret_cast<v4i*>(reinterpret_cast<uint8_t*>(dx) + ((int64_t)il * p.dx_ld + col) * (int64_t)sizeof(T)) =
                *reinterpret_cast<const v4i*>(stg + row * PITCH + k16 * 16);
        }
      }
      return;
    }
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      if (il4[b] < 0) continue;
      T* drow = dx + (int64_t)il4[b] * p.dx_ld;
#pragma unroll
      for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int j = jbase + a * 32 + 8 * q;
          if (j >= p.d) continue;                       // d is a multiple of 4, so j..j+3 are in range together
          const uint32_t w = wv[b][4 * a + q];
          Elem<T>::store(drow + j + 0, __builtin_fmaf(-hs[b], e4m3_to_float<0>(w), __fmul_rn(acc[a][b][4 * q + 0], rs[b])));
          Elem<T>::store(drow + j + 1, __builtin_fmaf(-hs[b], e4m3_to_float<1>(w), __fmul_rn(acc[a][b][4 * q + 1], rs[b])));
          Elem<T>::store(drow + j + 2, __builtin_fmaf(-hs[b], e4m3_to_float<2>(w), __fmul_rn(acc[a][b][4 * q + 2], rs[b])));
          Elem<T>::store(drow + j + 3, __builtin_fmaf(-hs[b], e4m3_to_float<3>(w), __fmul_rn(acc[a][b][4 * q + 3], rs[b])));
        }
    }
    return;
  }
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    const int il = rt * 256 + wb * 128 + b * 32 + (lane & 31);
    if (SPLIT) {
      float* dst = p.part + dx_part_offset(((int64_t)ks * p.RT + rt) * p.CT + ct, wb, b, wa) + lane * 4;
#pragma unroll
      for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          *reinterpret_cast<v4f*>(dst + (4 * a + q) * 256) =
              (v4f){acc[a][b][4 * q + 0], acc[a][b][4 * q + 1], acc[a][b][4 * q + 2], acc[a][b][4 * q + 3]};
      continue;
    }
    if (il >= p.rows) continue;
    const DxRowTerms row(p, il);
#pragma unroll
    for (int a = 0; a < 4; ++a) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int j = jbase + a * 32 + 8 * q;
        if (j >= p.d) continue;                       // d is a multiple of 4, so j..j+3 are in range together
        row.store4<T>(p, dx + (int64_t)il * p.dx_ld + j, j, acc[a][b][4 * q + 0], acc[a][b][4 * q + 1], acc[a][b][4 * q + 2],
                      acc[a][b][4 * q + 3]);
      }
    }
  }
}

// A column that is the target of at least long_seg (LONG_SEG or LONG_SEG_PARTS) rows has its segment of the sorted list cut into
// nch = ceil(L / LONG_CHUNK) equal chunks (the last one may be shorter); chunk c starts at sorted
// position s0 + c * ceil(L / nch).
__device__ __forceinline__ void long_chunks(int L, int& nch, int& len) {
  nch = (L + LONG_CHUNK - 1) / LONG_CHUNK;
  len = (L + nch - 1) / nch;
}

// The chunk sums of the columns of several chunks are added up, in order, into the first one's place, where everything after finds a
// long column's sum.  One block of 256 rows of dW of one column at a time, all its loads but for every eighth in flight together.  A
// few microseconds of work that only the kernels storing dW wait for: it rides in the grid of bwd_dx_finish_kernel where there is
// one before them.  (Left to its readers it was a walk at the latency of memory, one wave to a SIMD: with Zipf targets the
// tiles of the first columns took 100 us longer than the rest, which a dW of one or two rounds of tiles waits for whole.
// 24064 rows of three offsets, d = 416, V = 27712: bwd_dw_out_kernel 406 us, now
// 306; 29184 rows of three, d = 2512, V = 9664: 512, now 356 and 8 for the fold.)
struct FoldParams {
  const int32_t *longlist, *longbase, *segoff;
  float* longsum;
  int64_t dq;
  int slots;
};
__device__ __forceinline__ void fold_chunks(const FoldParams& f, int block, int nblocks) {
  const int ny = (int)(f.dq / 256), items = f.longlist[2] * ny;
  for (int item = block; item < items; item += nblocks) {
    const int v = f.longlist[3 + f.slots + item / ny];
    int nch, len;
    long_chunks(f.segoff[v + 1] - f.segoff[v], nch, len);
    float* s = f.longsum + (int64_t)f.longbase[v] * f.dq + (item % ny) * 256 + threadIdx.x;
    float sum = 0.f;
    for (int c0 = 0; c0 < nch; c0 += 8) {
      float x[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) x[u] = c0 + u < nch ? s[(int64_t)(c0 + u) * f.dq] : 0.f;
#pragma unroll
      for (int u = 0; u < 8; ++u) sum += x[u];
    }
    *s = sum;
  }
}
__global__ __launch_bounds__(256) void bwd_dw_fold_kernel(FoldParams f) { fold_chunks(f, blockIdx.x, gridDim.x); }

// One-hot part of dW for the long columns: longsum[slot][:] = sum over the column's (or the chunk's) rows of h_i X_q[i, :], 256 rows
// of dW at a time (by).  What bounds it is the latency of the gathered rows, of which 16 lanes read 256 bytes: a
// wave has four rows' worth of lanes and eight loads in flight in each.  A chunk is a workgroup's, folded in LDS in a fixed order; a
// column of up to LONG_WAVE rows is one wave's, without a barrier (a workgroup each, with most of its lanes idle, took the many
// columns of 8 to 15 rows of a mid-sized vocabulary 138 us at 50000 rows of three offsets, d = 1024, V = 16384: now 53; LONG_WAVE = 64
// is faster there and at 48 rows a column, 16 for 22 us, but a wave's second round of loads is 2 us of a small step).  The grid is a
// fixed one that walks the lists, whose lengths the host does not know.  The result does not depend on scheduling.
constexpr int LONG_GRID = 1024, FOLD_GRID = 512;
struct LongParams {
  const int32_t* longlist;
  int slots;
  const int32_t *segoff, *srow;
  const float* sh;
  const uint8_t* xq;
  int64_t ldx, dq;
  const int32_t* longbase;
  float* longsum;
  int gx;                      // workgroups that walk the lists, for each 256 rows of dW
};
typedef float LongShared[16][256];
__device__ __forceinline__ void dw_long(LongShared& red, int bx, int by, const LongParams& p) {
  const auto &longlist = p.longlist, &segoff = p.segoff, &srow = p.srow, &longbase = p.longbase;
  const auto& sh = p.sh;
  const int slots = p.slots;
  const int64_t ldx = p.ldx, dq = p.dq;
  float* longsum = p.longsum;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6, c = t & 15, rl = t >> 4, q = lane >> 4;
  const int64_t jb = (int64_t)by * 256;
  const uint8_t* xcol = p.xq + jb + c * 16;
  // a[m] = sum over entries first, first + stride, ... of the L from s0 on, in that order, of the lane's 16 rows of dW
  auto rows = [&](int s0, int L, int first, int stride, float (&a)[16]) {
#pragma unroll
    for (int m = 0; m < 16; ++m) a[m] = 0.f;
    for (int n0 = first; n0 < L; n0 += stride * 8) {
      v4i raw[8];
      float h[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int n = n0 + stride * u;
        h[u] = n < L ? sh[s0 + n] : 0.f;
        raw[u] = *reinterpret_cast<const v4i*>(xcol + (int64_t)srow[n < L ? s0 + n : s0] * ldx);
      }
#pragma unroll
      for (int u = 0; u < 8; ++u) {        // rows in ascending order within a row-lane
#pragma unroll
        for (int m = 0; m < 4; ++m) {
          const uint32_t w = (uint32_t)raw[u][m];
          a[4 * m + 0] = fmaf(h[u], e4m3_to_float<0>(w), a[4 * m + 0]);
          a[4 * m + 1] = fmaf(h[u], e4m3_to_float<1>(w), a[4 * m + 1]);
          a[4 * m + 2] = fmaf(h[u], e4m3_to_float<2>(w), a[4 * m + 2]);
          a[4 * m + 3] = fmaf(h[u], e4m3_to_float<3>(w), a[4 * m + 3]);
        }
      }
    }
  };
  float a[16];
  const int nwave = longlist[0], nchunk = longlist[1];
  for (int i = bx; i < nchunk; i += p.gx) {
    const int slot = slots - 1 - i, v = longlist[3 + slot], ch = slot - longbase[v];
    int nch, len;
    const int seg0 = segoff[v], seg1 = segoff[v + 1];
    long_chunks(seg1 - seg0, nch, len);
    const int s0 = seg0 + ch * len;
    rows(s0, min(seg1 - s0, len), rl, 16, a);
#pragma unroll
    for (int m = 0; m < 16; ++m) red[rl][c * 16 + m] = a[m];
    __syncthreads();
    float sfold = 0.f;
#pragma unroll
    for (int k = 0; k < 16; ++k) sfold += red[k][t];
    longsum[(int64_t)slot * dq + jb + t] = sfold;
    __syncthreads();                       // `red` is written again for the next chunk
  }
  // (from the other end of the grid: while there are workgroups without a chunk, none has both to do one behind the other)
  for (int slot = (p.gx - 1 - bx) * 4 + wave; slot < nwave; slot += p.gx * 4) {
    const int v = longlist[3 + slot], s0 = segoff[v];
    rows(s0, segoff[v + 1] - s0, q, 4, a);
#pragma unroll
    for (int m = 0; m < 16; ++m) {         // over the four row lanes, pairwise; all of them get it
      a[m] += __shfl_xor(a[m], 16);
      a[m] += __shfl_xor(a[m], 32);
    }
    v4f mine;
#pragma unroll
    for (int m = 0; m < 4; ++m) mine[m] = q == 0 ? a[m] : q == 1 ? a[4 + m] : q == 2 ? a[8 + m] : a[12 + m];
    *reinterpret_cast<v4f*>(longsum + (int64_t)slot * dq + jb + c * 16 + q * 4) = mine;
  }
}
__global__ __launch_bounds__(256, 5) void bwd_dw_long_kernel(LongParams p) {
  __shared__ LongShared red;
  dw_long(red, blockIdx.x, blockIdx.y, p);
}

// Sum of the K-split partials, row scale, one-hot term, cast: a workgroup per 32 rows x 128 columns, a wave per 32 of the
// columns.  A thread's values are four quads of one row; they go out through LDS as whole pieces of rows.
// The first `riders` workgroups do work that only the kernels storing dW wait for, beside a kernel that is bound by the
// bandwidth of its partial sums: the sums of the long columns themselves (lng.gx > 0: a call of few entries), or, of a larger call, the folding
// of those of several chunks.  Two micro-batches of 2048 rows of Zipf targets, d = 1024: the sums in a launch of their own 18.8 and this kernel
// 29.9 us, together 39.2; 4096 rows, d = 1600 10.5 + 18.1, 24.0; 1000 rows, d = 256, V = 4096 3.9 + 6.3, 6.1; 2048 rows of uniform targets, which
// have no long columns, d = 768 4.2 + 14.1, 17.2.  (More than RANK_MAX entries make more chunks to a column than the kernels storing dW
// should walk, one wave to a SIMD, so there the sums come first and only the folding rides.)
template <typename T>
__global__ __launch_bounds__(256) void bwd_dx_finish_kernel(DxParams p_in, FoldParams f, LongParams lng, int riders) {
  __shared__ __attribute__((aligned(16))) union { LongShared red; uint8_t stage[32 * (128 * sizeof(T) + 16)]; } shared;
  if ((int)blockIdx.x < riders) {
    if (lng.gx > 0) return dw_long(shared.red, blockIdx.x % lng.gx, blockIdx.x / lng.gx, lng);
    return fold_chunks(f, blockIdx.x, riders);
  }
  DxParams p = p_in;
  if (p.dc) p.w_s = p.dc->w_s;
  constexpr int RB = 128 * (int)sizeof(T), PITCH = RB + 16, CH = RB / 16;
  uint8_t* stage = shared.stage;
  const int bid = blockIdx.x - riders;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6, wa = bid & 1, b = (bid >> 1) & 3, wb = (bid >> 3) & 1;
  const int tile = bid >> 4, rt = tile / p.CT, ct = tile - rt * p.CT, i0 = rt * 256 + wb * 128 + b * 32, j0 = ct * 256 + wa * 128;
  if (i0 >= p.rows || j0 >= p.d) return;
  v4f sum[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) sum[q] = (v4f){0.f, 0.f, 0.f, 0.f};
  const float* src = p.part + dx_part_offset(tile, wb, b, wa) + wave * 1024 + lane * 4;
  const int64_t step = (int64_t)p.RT * p.CT * 65536;
  for (int k0 = 0; k0 < p.ksplit; k0 += 4) {              // fixed order, the loads of four parts in flight together
    v4f x[4][4];
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int q = 0; q < 4; ++q) x[u][q] = k0 + u < p.ksplit ? *reinterpret_cast<const v4f*>(src + (k0 + u) * step + q * 256) : (v4f){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int q = 0; q < 4; ++q) sum[q] += x[u][q];
  }
  const int il = i0 + (lane & 31);
  if (il < p.rows) {
    const DxRowTerms row(p, il);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int c = wave * 32 + 8 * q + 4 * (lane >> 5);
      row.store4<T>(p, reinterpret_cast<T*>(stage + (lane & 31) * PITCH) + c, j0 + c, sum[q][0], sum[q][1], sum[q][2], sum[q][3]);
    }
  }
  __syncthreads();
  T* dx = reinterpret_cast<T*>(p.dx);
  const bool vec = ((reinterpret_cast<uintptr_t>(p.dx) | (uintptr_t)(p.dx_ld * (int64_t)sizeof(T))) & 15) == 0;
#pragma unroll
  for (int n = 0; n < 32 * CH / 256; ++n) {
    const int e = t + 256 * n, r = e / CH, k = e % CH, col = j0 + k * (16 / (int)sizeof(T));
    if (i0 + r >= p.rows || col >= p.d) continue;          // (d is a multiple of 16: a piece is in range as a whole)
    T* dst = dx + (int64_t)(i0 + r) * p.dx_ld + col;
    const T* from = reinterpret_cast<const T*>(stage + r * PITCH + k * 16);
    if (vec) *reinterpret_cast<v4i*>(dst) = *reinterpret_cast<const v4i*>(from);
    else
#pragma unroll
      for (int m = 0; m < 16 / (int)sizeof(T); ++m) dst[m] = from[m];
  }
}

struct DwParams {
  const uint8_t* xt;      // dq rows, K = Np, blocked                             A side (rows j)
  const uint8_t* ghat_t;  // G, tile by tile (rows i, K = v), already at the tile of this launch's first row      B side (rows v, through the transposing read)
  const uint32_t* gexp;   // its block exponents [Vp / 128][kbw], likewise
  float* dwacc;           // [dq][Vp] fp32
  int64_t kbn, kbw, kb0, Vp;   // K blocks per tile of xt; blocks of 128 rows that gexp counts; first K block of xt in this launch; row length of dwacc
  int64_t kbv;                 // blocks of 128 columns per tile of 256 rows of G
  int RT, CT, KT;
};

// ACC: add to what the partial holds (only when there are more dW launches than partial buffers)
template <bool ACC>
__global__ __launch_bounds__(256) void bwd_dw_kernel(DwParams p) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  int rt, ct;
  if (!map_tile_rr(blockIdx.x, p.RT, p.CT, rt, ct)) return;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6, wa = wave >> 1, wb = wave & 1;
  // the block exponents of this tile's K loop wait in LDS behind the two K slots: [v half][K block]
  uint32_t* lsc = reinterpret_cast<uint32_t*>(smem + SMEM_BYTES);
  for (int e = t; e < 2 * p.KT; e += NTHREADS) {
    const int w = e >= p.KT, kb = e - w * p.KT;
    lsc[e] = p.gexp[(int64_t)(2 * ct + w) * p.kbw + kb];
  }
  __syncthreads();
  v16f acc[4][4];
  // B = G with K (rows i) as the slow index: the 128 rows of a K block are half a tile of G, the 256 columns of this dW
  // tile its column blocks 2 ct and 2 ct + 1 (BLOCKED_KSTEP apart); from one tile of G to the next kbv blocks
  mfma_mainloop<false, NoHook, BLOCKED_KSTEP, true, 2>(p.xt + ((int64_t)rt * p.kbn + p.kb0) * BLOCKED_KSTEP, BK, p.ghat_t + (int64_t)(2 * ct) * BLOCKED_KSTEP, BLOCKED_KSTEP, p.KT,
                                                       smem, acc, ct & 7, 2 * (rt & 3), __builtin_amdgcn_readfirstlane(wave), NoHook(), 128 * BK, p.kbv * BLOCKED_KSTEP,
                                                       lsc + __builtin_amdgcn_readfirstlane(wb) * p.KT);
  const int jbase = rt * 256 + wa * 128 + 4 * (lane >> 5);
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    const int v = ct * 256 + wb * 128 + b * 32 + (lane & 31);
#pragma unroll
    for (int a = 0; a < 4; ++a) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int j = jbase + a * 32 + 8 * (r >> 2) + (r & 3);
        float* dst = p.dwacc + (int64_t)j * p.Vp + v;
        *dst = ACC ? (*dst + acc[a][b][r]) : acc[a][b][r];
      }
    }
  }
}

// The tiles of the last, partly filled round of dW (tile0 .. tile0 + ntail - 1 of the round-robin order), shared out
// along K: a tile's K loop is kp pairs of K blocks long, all of them together W = ntail * kp pairs, and workgroup g takes
// pairs [g share, (g + 1) share) of that line -- the end of one tile and the beginning of the next, when its range
// straddles them.  Piece (g, t) of tile t goes to buf[g + t] as plain stores (g + t grows by one from each piece to the
// next along the line, so no two pieces meet); bwd_dw_final_kernel adds up a tile's pieces in the order of g.
struct DwTail {
  float* buf;
  int tile0, ntail, kp, share;      // tile0 < 0: no tail (every tile is in the fp32 partial)
};
// (grid: workgroups x 2.  A workgroup's range is at most half a tile's K loop long, so it lies in one tile or straddles
// two: blockIdx.y = 0 takes the part in the first tile, blockIdx.y = 1 the part in the second, if there is one.  One piece
// per workgroup, with no loop around the main loop: looping over the pieces, the compiler spilled the accumulators.)
__global__ __launch_bounds__(256) void bwd_dw_tail_kernel(DwParams p, DwTail tl) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  const int g = blockIdx.x;
  const int pos0 = g * tl.share, end = min(tl.ntail * tl.kp, pos0 + tl.share);
  if (pos0 >= end) return;
  int tt = pos0 / tl.kp, pos = pos0;
  if (blockIdx.y == 1) {
    ++tt; pos = tt * tl.kp;
    if (pos >= end) return;
  }
  // (everything here is uniform, but the divisions leave their results in vector registers: the main loop wants
  // its addresses in scalar ones)
  tt = __builtin_amdgcn_readfirstlane(tt);
  const int k0 = __builtin_amdgcn_readfirstlane(pos - tt * tl.kp), k1 = min(tl.kp, k0 + (end - pos)), KD = __builtin_amdgcn_readfirstlane(2 * (k1 - k0));
  int rt, ct;
  tile_from_index(tl.tile0 + tt, p.RT, p.CT, rt, ct);
  rt = __builtin_amdgcn_readfirstlane(rt); ct = __builtin_amdgcn_readfirstlane(ct);
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6, wa = wave >> 1, wb = wave & 1;
  uint32_t* lsc = reinterpret_cast<uint32_t*>(smem + SMEM_BYTES);
  for (int e = t; e < 2 * KD; e += NTHREADS) {
    const int w = e >= KD, kb = e - w * KD;
    lsc[e] = p.gexp[(int64_t)(2 * ct + w) * p.kbw + 2 * k0 + kb];
  }
  __syncthreads();
  v16f acc[4][4];
  mfma_mainloop<false, NoHook, BLOCKED_KSTEP, true, 2>(uniform_ptr(p.xt + ((int64_t)rt * p.kbn + p.kb0 + 2 * k0) * BLOCKED_KSTEP), BK,
                                                       uniform_ptr(p.ghat_t + ((int64_t)k0 * p.kbv + 2 * ct) * BLOCKED_KSTEP), BLOCKED_KSTEP,
                                                       KD, smem, acc, ct & 7, 2 * (rt & 3), __builtin_amdgcn_readfirstlane(wave), NoHook(), 128 * BK, p.kbv * BLOCKED_KSTEP,
                                                       lsc + __builtin_amdgcn_readfirstlane(wb) * KD);
  float* dst0 = tl.buf + (size_t)(g + tt) * 65536 + (wa * 2 + wb) * 16384 + lane * 4;       // as the accumulators lie: [wa][wb][a][b][quad][lane]
#pragma unroll
  for (int b = 0; b < 4; ++b)
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        *reinterpret_cast<v4f*>(dst0 + (4 * a + b) * 1024 + q * 256) = (v4f){acc[a][b][4 * q], acc[a][b][4 * q + 1], acc[a][b][4 * q + 2], acc[a][b][4 * q + 3]};
}

// From the sorted keys: segoff[v] = first position whose key is at least v, v = 0 .. V, and the long columns (order
// irrelevant: each is handled on its own).  A long column has a slot for its sum, or one for each of its chunks if it has more
// than LONG_WAVE rows; longbase[v] is its first.  longlist[0] counts the slots of the former, which are given out from the
// first on, [1] those of the latter, from the last one down; behind the counters stands the column of every slot, and behind
// those, longlist[2] of them, the columns of several chunks once more.  One column per thread, by bisection: first among every stride-th key (in LDS), then within one
// stride.  (A thread per key that fills the gap up to the next key runs as long as the widest gap: with Zipf targets the
// rare end of the vocabulary holds gaps of thousands of columns, and 2048 rows took 63 us; this takes 4.7.)
// Also: row and coefficient of every sorted entry (srow, sh), so that the kernels that walk a segment load them side by
// side instead of one behind the other: at most SEG_ENTRIES to a block, with blocks beyond the columns' if need be (three
// offsets of 65536 rows over a vocabulary of 512 took the columns' 3 blocks 135 us, with 384 it is 17; V = 4096 39 -> 18).
constexpr int SEG_ENTRIES = 512;
static inline int segment_blocks(int64_t n, int64_t V) { return (int)std::max<int64_t>(V / 256 + 1, (n + SEG_ENTRIES - 1) / SEG_ENTRIES); }
struct SegShared { int32_t top[256], seg[257]; };
__device__ __forceinline__ void column_segments(SegShared& shared, int block, int nblocks, const int32_t* __restrict__ skeys, const int32_t* __restrict__ perm,
                                                const float* __restrict__ hcoef, int n, int Np, int V, int long_seg, int slots, int32_t* __restrict__ segoff,
                                                int32_t* __restrict__ longlist, int32_t* __restrict__ longbase,
                                                int32_t* __restrict__ srow, float* __restrict__ sh) {
  auto& top = shared.top;
  auto& seg = shared.seg;
  const int t = threadIdx.x, v0 = block * 256, stride = (n + 255) / 256;
  for (int q = v0 + t; q < n; q += nblocks * 256) {
    const int e = perm[q];             // entry id k * Np + i
    srow[q] = e % Np; sh[q] = hcoef[e];
  }
  if (v0 > V) return;                  // a block beyond the columns': entries only
  top[t] = t * stride < n ? skeys[t * stride] : 0x7fffffff;
  __syncthreads();
  auto lower_bound = [&](int v) {
    int lo = 0, hi = 256;              // top[lo - 1] < v <= top[hi]
    while (lo < hi) {
      const int m = (lo + hi) >> 1;
      if (top[m] < v) lo = m + 1; else hi = m;
    }
    if (lo == 0) return 0;
    int a = (lo - 1) * stride + 1, b = min(lo * stride, n);      // skeys[a - 1] < v; skeys[b] >= v or b = n
    while (a < b) {
      const int m = (a + b) >> 1;
      if (skeys[m] < v) a = m + 1; else b = m;
    }
    return a;
  };
  seg[t] = lower_bound(v0 + t);
  if (t == 255) seg[256] = lower_bound(v0 + 256);
  __syncthreads();
  const int v = v0 + t;
  if (v > V) return;
  segoff[v] = seg[t];
  if (v == V) return;
  const int L = seg[t + 1] - seg[t];
  if (L < long_seg) return;
  int nch = 1, len;
  if (L > LONG_WAVE) long_chunks(L, nch, len);
  const int at = L > LONG_WAVE ? slots - nch - atomicAdd(&longlist[1], nch) : atomicAdd(&longlist[0], 1);
  longbase[v] = at;
  for (int c = 0; c < nch; ++c) longlist[3 + at + c] = v;
  if (nch > 1) longlist[3 + slots + atomicAdd(&longlist[2], 1)] = v;
}

// The two in one launch, blocks [0, nxt) the tiles of X~ and the rest the segments: neither needs the other, and on few rows
// a launch of its own costs more than the work (2 x 4.8 us at 2048 rows, 5.8 together; 34 us, 27 together, at 32768 of three offsets).
struct XtSegParams {
  const uint8_t* xq;
  int64_t dp, ldx, kbn;
  const float *rho, *blockmax, *hcoef;
  float* xi;
  uint8_t* xt;
  const int32_t *skeys, *perm;
  int32_t *segoff, *longlist, *longbase, *srow;
  float* sh;
  int nblk, nxt, nx, n, Np, V, long_seg, slots;
};
__global__ __launch_bounds__(256) void bwd_xt_segments_kernel(XtSegParams p) {
  __shared__ union { XtShared x; SegShared s; } shared;
  const int bid = blockIdx.x;
  if (bid < p.nxt) xt_tile(shared.x, bid % p.nx, bid / p.nx, p.xq, p.dp, p.ldx, p.kbn, p.rho, p.blockmax, p.nblk, p.xi, p.xt);
  else column_segments(shared.s, bid - p.nxt, gridDim.x - p.nxt, p.skeys, p.perm, p.hcoef, p.n, p.Np, p.V, p.long_seg, p.slots, p.segoff, p.longlist, p.longbase, p.srow, p.sh);
}

// Where the one-hot part of dW comes from and where dW goes (bwd_dw_out_kernel, bwd_dw_final_kernel).
struct DwOut {
  void* dw;                    // [d][dw_ld], columns [0, V)
  int64_t dw_ld;
  const int32_t* segoff;       // entries [segoff[v], segoff[v + 1]) of the sorted list belong to column v
  const int32_t* srow;         // row i of a sorted entry
  const float* sh;             // its coefficient h
  const uint8_t* xq;           // [Np], row stride ldx
  const float* longsum;        // [slot][dq]: sums of the long columns
  const int32_t* longbase;     // slot of a long column
  const float* xi;
  const DevConsts* dc;         // non-NULL: x_s comes from here
  int64_t ldx, dq;
  float x_s;
  int d, V, long_seg;          // long_seg: LONG_SEG wherever bwd_dw_out_kernel runs
  bool chunks;                 // the chunk sums of a long column are not folded into the first
};
__device__ __forceinline__ int long_parts(const DwOut& o, int L) {
  int nch = 1, len;
  if (o.chunks && L > LONG_WAVE) long_chunks(L, nch, len);
  return nch;
}

// dW straight from the main loop: dW = x_s (xi (X~^T G) - sum over the column's target entries of h_i X_q[i, :]), cast and
// stored by the workgroup that has the tile in its accumulators.  Used whenever one launch covers all rows: up to 131072 with
// the dlogits kept; formed again, as many whole dX panels as fit in 131072 rows, and a workspace of the default size.  What
// the separate pass over an fp32 partial cost was its traffic: 8 bytes an element written and read again (1 GB at
// d = 2560, V = 50304) around 2 bytes of result, 65 us of a 560 us step at N = 2048, d = 768 and 172 us at N = 30011,
// d = 2560, whatever the number of rows.
//
// The epilogue must not wait on memory: one wave per SIMD has nothing to hide a load behind (gathering the one-hot rows
// with dependent loads was measured at +0.5 ms of a 20 ms step).  So the rows X_q[i] of the tile's target entries -- the
// short columns' only; columns with LONG_SEG or more entries have their sums ready -- go to LDS with direct loads:
// before the main loop, into what the K slots and the block exponents leave free (100 to 112 entries of 256 bytes; of a half tile an entry
// is 128 bytes, everywhere), if they fit there -- all tiles' do of 16384 rows with uniform targets over 50257 columns, four fifths of the tiles' of 65536
// rows with Zipf targets, next to none of 26400 uniform ones -- and otherwise into the K slots after it, as many row blocks at a
// time as fit (a row block's 64 columns have at most 64 (LONG_SEG - 1) = 448 entries).  Each lane then walks the entries of its own
// column.  A 16-byte chunk c of an entry's 256 bytes lies at position c ^ (entry & 15): the lanes of a wave read the same
// columns j of neighbouring entries, which would all lie in the same banks.
// On the way out a bf16 quadrant is turned in LDS, 32 columns x 64 rows at a time, by the transposing read, so that a lane
// stores 16 bytes of one row of dW and a wave 64 consecutive bytes of 16 rows.
constexpr int DWO_AUX = 2 * 260 * 4;                         // entry offsets and segment starts of the tile's 256 columns
constexpr int DWO_STAGE_PITCH = 64 * 2 + 16, DWO_STAGE = 32 * DWO_STAGE_PITCH;      // per wave
constexpr int DWO_GROUP = 480;                               // entries that the K slots hold (256 bytes of X_q, row and coefficient each)
static_assert(DWO_GROUP * (256 + 8) <= SMEM_BYTES && DWO_GROUP >= 64 * (LONG_SEG - 1), "a row block's entries must fit the K slots");
constexpr int DWO_MAX_KT = 131072 / BK;
static_assert(SMEM_MAX - SMEM_BYTES - 8 * DWO_MAX_KT - DWO_AUX >= 4 * DWO_STAGE, "no room for the staging tiles beside the K slots");

// NA = 2: 128 rows of dW (rt counts those), the half tiles of bwd_dw_out_kernel.
template <typename T, int NA>
__device__ __forceinline__ void dw_out_tile(const DwParams& p, const DwOut& o, uint8_t* smem, int rt, int ct) {
  constexpr int TROWS = 64 * NA, EB = TROWS, CHUNKS = EB / 16;               // rows of dW in the tile = bytes of X_q of an entry
  static_assert(DWO_GROUP % (64 / CHUNKS) == 0, "load_rows fills up its last load: beyond the group lie the entries' rows and coefficients");
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wa = wave >> 1, wb = wave & 1;
  const int KT = p.KT;
  uint32_t* lsc = reinterpret_cast<uint32_t*>(smem + SMEM_BYTES);            // block exponents of the K loop: [v half][K block]
  int* ioff = reinterpret_cast<int*>(smem + SMEM_BYTES + 8 * KT);            // [257]: first short entry of column c, counted over the tile
  int* spos = ioff + 260;                                                    // [257]: segoff of the tile's columns
  uint8_t* area = reinterpret_cast<uint8_t*>(spos + 260);                    // the rest of LDS
  const int room = ((SMEM_MAX - SMEM_BYTES - DWO_AUX - 8 * KT) / (EB + 8)) & ~(64 / CHUNKS - 1);
  // entry q's row and coefficient; its EB bytes of X_q (columns rt * TROWS on) at x + q * EB
  struct Item { int row; float h; };
  auto load_rows = [&](const Item* items, int n, uint8_t* x) {
    const int lane = lane_id();
    const uint32_t lds0 = (uint32_t)(uintptr_t)((__attribute__((address_space(3))) void*)x);
    constexpr int PER = 64 / CHUNKS;                         // entries to one load: four (NA = 4); beyond the last one it is loaded again
    for (int q0 = PER * wave; q0 < n; q0 += 4 * PER) {
      const int q = q0 + lane / CHUNKS, c = (lane % CHUNKS) ^ (q & (CHUNKS - 1));
      lds_direct_16_far(__builtin_amdgcn_readfirstlane(lds0 + q0 * EB), o.xq + (int64_t)items[q < n ? q : n - 1].row * o.ldx + rt * TROWS + c * 16);
    }
  };
  bool pre;
  {
    const int t = threadIdx.x, v = ct * 256 + t;
    const int s0 = o.segoff[v < o.V ? v : o.V], s1 = o.segoff[v + 1 < o.V ? v + 1 : o.V];
    for (int e = t; e < 2 * KT; e += NTHREADS) {
      const int w = e >= KT, kb = e - w * KT;
      lsc[e] = p.gexp[(int64_t)(2 * ct + w) * p.kbw + kb];
    }
    const int cnt = s1 - s0 < LONG_SEG ? s1 - s0 : 0;
    int incl = cnt;
#pragma unroll
    for (int s = 1; s < 64; s <<= 1) {
      const int up = __shfl_up(incl, s);
      if ((t & 63) >= s) incl += up;
    }
    int* wtot = reinterpret_cast<int*>(area);
    if ((t & 63) == 63) wtot[wave] = incl;
    __syncthreads();
    for (int w = 0; w < wave; ++w) incl += wtot[w];
    ioff[t] = incl - cnt; spos[t] = s0;
    if (t == 255) { ioff[256] = incl; spos[256] = s1; }
    __syncthreads();
    const int E = __builtin_amdgcn_readfirstlane(ioff[256]);
    pre = E <= room;
    if (pre && E > 0) {
      Item* items = reinterpret_cast<Item*>(area + room * EB);
      for (int k = 0; k < cnt; ++k) items[incl - cnt + k].row = s0 + k;
      __syncthreads();
      for (int q = t; q < E; q += NTHREADS) {
        const int at = items[q].row;
        items[q].row = o.srow[at]; items[q].h = o.sh[at];
      }
      __syncthreads();
      load_rows(items, E, area);
    }
  }
  v16f acc[NA][4];
  // (128 rows: half a 256-row tile of X~, whose K blocks are 256 rows of BK bytes)
  const uint8_t* xt = p.xt + ((int64_t)(NA == 4 ? rt : rt >> 1) * p.kbn + p.kb0) * BLOCKED_KSTEP + (NA == 4 ? 0 : (rt & 1) * TROWS * BK);
  mfma_mainloop<false, NoHook, BLOCKED_KSTEP, true, 2, false, false, NA>(xt, BK, p.ghat_t + (int64_t)(2 * ct) * BLOCKED_KSTEP, BLOCKED_KSTEP, p.KT,
                                                       smem, acc, ct & 7, 2 * (rt & 3), wave, NoHook(), 128 * BK, p.kbv * BLOCKED_KSTEP, lsc + wb * p.KT);
  const float x_s = o.dc ? o.dc->x_s : o.x_s, scale = x_s * o.xi[0];
  T* dw = reinterpret_cast<T*>(o.dw);
  const bool vec = sizeof(T) == 2 && ((reinterpret_cast<uintptr_t>(o.dw) | (uintptr_t)(o.dw_ld * (int64_t)sizeof(T))) & 15) == 0 && (o.V % 8 == 0 || ct * 256 + 256 <= o.V);
  uint8_t* stage = (pre ? smem : area) + wave * DWO_STAGE;
  const uint8_t* xrows = pre ? area : smem;
  const Item* items = reinterpret_cast<const Item*>(pre ? area + room * EB : smem + DWO_GROUP * EB);
  int bend = pre ? 4 : 0, qsub = 0;            // row blocks whose entries are in LDS; what to take off an entry's number for its place there
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    if (b >= bend) {
      // the entries of as many row blocks from b on as fit, of both halves of the columns: first those of the lower half
      auto upto = [&](int e) { return ioff[32 * e] - ioff[32 * b] + ioff[128 + 32 * e] - ioff[128 + 32 * b]; };
      bend = b + 1;
      while (bend < 4 && upto(bend + 1) <= DWO_GROUP) ++bend;
      bend = __builtin_amdgcn_readfirstlane(bend);
      const int total = __builtin_amdgcn_readfirstlane(upto(bend)), base0 = ioff[32 * b], sub1 = ioff[128 + 32 * b] - (ioff[32 * bend] - base0);
      Item* list = reinterpret_cast<Item*>(smem + DWO_GROUP * EB);
      __syncthreads();                         // every wave is done with the entries that were there
      const int t = wave * 64 + lane_id(), tb = (t & 127) >> 5;
      if (tb >= b && tb < bend) {
        const int first = ioff[t] - (t < 128 ? base0 : sub1), cnt = ioff[t + 1] - ioff[t];
        for (int k = 0; k < cnt; ++k) list[first + k].row = spos[t] + k;
      }
      __syncthreads();
      for (int q = t; q < total; q += NTHREADS) {
        const int at = list[q].row;
        list[q].row = o.srow[at]; list[q].h = o.sh[at];
      }
      __syncthreads();
      load_rows(list, total, smem);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      qsub = __builtin_amdgcn_readfirstlane(wb ? sub1 : base0);
    }
#pragma unroll
    for (int ah = 0; ah < NA / 2; ++ah) {      // rows 64 ah .. + 63 of the quadrant
      const int lane = lane_id(), h = lane >> 5, c = wb * 128 + b * 32 + (lane & 31), v = ct * 256 + c;
      float val[32];
#pragma unroll
      for (int m = 0; m < 32; ++m) val[m] = acc[2 * ah + (m >> 4)][b][m & 15] * scale;
      const int q0 = ioff[c] - qsub, n = ioff[c + 1] - ioff[c];
      for (int k = 0; __builtin_amdgcn_ballot_w64(k < n) != 0; ++k) {
        if (k < n) {
          const int q = q0 + k;
          const float hx = items[q].h * x_s;
          const uint8_t* xr = xrows + q * EB + 4 * h;
          const int sw = (2 * NA * wa + 4 * ah) ^ (q & (CHUNKS - 1));
#pragma unroll
          for (int g = 0; g < 8; ++g) {        // four rows each: 32 (g / 4) + 8 (g % 4) + 4 h on
            const uint32_t w = *reinterpret_cast<const uint32_t*>(xr + ((sw ^ (g >> 1)) << 4) + 8 * (g & 1));
            val[4 * g + 0] -= hx * e4m3_to_float<0>(w);
            val[4 * g + 1] -= hx * e4m3_to_float<1>(w);
            val[4 * g + 2] -= hx * e4m3_to_float<2>(w);
            val[4 * g + 3] -= hx * e4m3_to_float<3>(w);
          }
        }
      }
      const int L = spos[c + 1] - spos[c];
      if (__builtin_amdgcn_ballot_w64(L >= LONG_SEG) != 0) {
        if (L >= LONG_SEG) {
          const float* ls = o.longsum + (int64_t)o.longbase[v] * o.dq + rt * TROWS + wa * 32 * NA + ah * 64 + 4 * h;
          for (int c2 = long_parts(o, L); c2 > 0; --c2, ls += o.dq)
#pragma unroll
            for (int g = 0; g < 8; ++g) {
              const v4f s = *reinterpret_cast<const v4f*>(ls + 32 * (g >> 2) + 8 * (g & 3));
#pragma unroll
              for (int m = 0; m < 4; ++m) val[4 * g + m] -= s[m] * x_s;
            }
        }
      }
      const int j0 = rt * TROWS + wa * 32 * NA + ah * 64;
      if (vec) {
#pragma unroll
        for (int g = 0; g < 8; ++g) {
          typedef __bf16 v4bf __attribute__((ext_vector_type(4)));
          const v4bf e = {(__bf16)val[4 * g], (__bf16)val[4 * g + 1], (__bf16)val[4 * g + 2], (__bf16)val[4 * g + 3]};
          *reinterpret_cast<v2i*>(stage + (lane & 31) * DWO_STAGE_PITCH + 2 * (32 * (g >> 2) + 8 * (g & 3) + 4 * h)) = __builtin_bit_cast(v2i, e);
        }
        asm volatile("" ::: "memory");         // (a wave's own LDS operations complete in order)
        // ds_read_b64_tr_b16: of the 4 x 16 matrix that 16 lanes point at, 8 bytes each, lane i gets column i
        typedef short v4s __attribute__((ext_vector_type(4)));
        typedef __attribute__((address_space(3))) v4s lds_v4s;
        const int i = lane & 15, v8 = 8 * (lane >> 4);
        const uint8_t* src = stage + (v8 + (i >> 2)) * DWO_STAGE_PITCH + 8 * (i & 3);
        T* dst = dw + (int64_t)(j0 + i) * o.dw_ld + ct * 256 + wb * 128 + b * 32 + v8;
        const bool in = ct * 256 + wb * 128 + b * 32 + v8 < o.V;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          const v2i lo = __builtin_bit_cast(v2i, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s*)(src + 32 * s)));
          const v2i hi = __builtin_bit_cast(v2i, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s*)(src + 32 * s + 4 * DWO_STAGE_PITCH)));
          if (in && j0 + 16 * s + i < o.d) *reinterpret_cast<v4i*>(dst + (int64_t)(16 * s) * o.dw_ld) = (v4i){lo[0], lo[1], hi[0], hi[1]};
        }
        asm volatile("" ::: "memory");
      } else if (v < o.V) {
#pragma unroll
        for (int m = 0; m < 32; ++m) {
          const int j = j0 + 32 * (m >> 4) + 8 * ((m & 15) >> 2) + 4 * h + (m & 3);
          if (j < o.d) Elem<T>::store(dw + (int64_t)j * o.dw_ld + v, val[m]);
        }
      }
      __builtin_amdgcn_sched_barrier(0);       // one half at a time: the accumulators of all of them, moved up front, do not fit the registers
    }
  }
}

// The first half_grid workgroups take the tiles tile0 .. of a last round that would leave more than half of the CUs idle, 128 rows each, two
// neighbours on one XCD to a tile (their columns of G are the same): nhalf of them.  No partial sums and no launch to add them up,
// but a K loop as long as a whole tile's with half its MFMAs.  They go first, so that the CUs fall out of step: when all of them
// store their tiles at the same time, the matrix pipes stand idle, and the stores are the whole of 19 us of a tile's 43 at 2048 rows in fp32.
// Measured, d = 768 (79 tiles in the last round), 2048 rows, fp32: full rounds, tail kernel and its sum 98 + 27 + 17 us; half tiles in a
// launch of their own 98 + 28; like this 108.  d = 1024 (20 tiles), bf16: 2048 rows 114 + 13 + 10, 114 + 23, 115; 4096 rows 192 + 17 + 10
// and 200; 8192 rows 302 + 24 + 12 for 345; 32768 rows 1128 + 61 + 20 for 1379.  d = 1600 (99 tiles), 4096 rows 281 + 45 + 16 and 309.
// So it is a matter of kp, the pairs of K blocks, and of n, the tiles of the last round, which the K-split cuts into 256 / n
// parts: as lines, tail kernel and sum 18 + n / 4 + kp (0.25 + n / 70), this 1.3 kp and next to nothing (dw_tail_plan).
template <typename T>
__global__ __launch_bounds__(256) void bwd_dw_out_kernel(DwParams p, DwOut o, int tile0, int nhalf, int half_grid) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  int rt, ct;
  if ((int)blockIdx.x < half_grid) {
    int lin, none;
    if (!map_tile(blockIdx.x, 1, nhalf, none, lin)) return;
    tile_from_index(tile0 + (lin >> 1), p.RT, p.CT, rt, ct);
    rt = __builtin_amdgcn_readfirstlane(rt); ct = __builtin_amdgcn_readfirstlane(ct);
    dw_out_tile<T, 2>(p, o, smem, 2 * rt + (lin & 1), ct);
    return;
  }
  if (!map_tile_rr(blockIdx.x - half_grid, p.RT, p.CT, rt, ct)) return;
  dw_out_tile<T, 4>(p, o, smem, rt, ct);
}

// The same from fp32 partials: what is left are the tiles of a K-split last round (tl.tile0 >= 0: grid.y = tl.ntail tiles of
// 16 blocks of 64 x 64 elements), and every tile where dW took more than one launch (grid = blocks of 64 columns x 64
// rows of dW).  A thread owns one column v and four groups of four rows j: 16 consecutive rows, or, of the pieces of a K-split
// tile, the rows that one lane's accumulators of a 32 x 32 block are.  The segment sum is formed here for short segments
// and read from the sums of the long columns for the others.
template <typename T>
__global__ __launch_bounds__(256) void bwd_dw_final_kernel(const float* __restrict__ dwacc, int nparts, int64_t part_stride, int64_t Vp, DwOut o, DwTail tl, int RT,
                                                          int CT) {
  const float x_s = o.dc ? o.dc->x_s : o.x_s;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const bool pieces = tl.tile0 >= 0;
  int v = blockIdx.x * 64 + lane, j0 = blockIdx.y * 64 + wave * 16;
  int wa = 0, wb = 0, a = 0, b = 0;
  if (pieces) {
    int rt, ct;
    tile_from_index(tl.tile0 + blockIdx.y, RT, CT, rt, ct);
    const int by = blockIdx.x >> 2, bx = blockIdx.x & 3;            // 64 rows and 64 columns of the tile
    wa = by >> 1; a = 2 * (by & 1) + (wave >> 1); wb = bx >> 1; b = 2 * (bx & 1) + (wave & 1);
    v = ct * 256 + wb * 128 + b * 32 + (lane & 31);
    j0 = rt * 256 + wa * 128 + a * 32 + 4 * (lane >> 5);
  }
  const int step = pieces ? 8 : 4;                                  // rows from one group of four to the next
  if (v >= o.V || j0 >= o.d) return;
  const float scale = x_s * o.xi[0];
  v4f val[4];
  if (pieces) {
    const int tt = blockIdx.y, g0 = (tt * tl.kp) / tl.share, g1 = ((tt + 1) * tl.kp - 1) / tl.share;
    const float* src = tl.buf + (size_t)tt * 65536 + (wa * 2 + wb) * 16384 + (4 * a + b) * 1024 + lane * 4;
#pragma unroll
    for (int q = 0; q < 4; ++q) val[q] = (v4f){0.f, 0.f, 0.f, 0.f};
    for (int g = g0; g <= g1; ++g) {                      // fixed order; the loads of a piece are in flight together
#pragma unroll
      for (int q = 0; q < 4; ++q) val[q] += *reinterpret_cast<const v4f*>(src + (size_t)g * 65536 + q * 256);
    }
  } else {
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        const float* src = dwacc + (int64_t)(j0 + 4 * q + m) * Vp + v;
        float sum = src[0];
        for (int n = 1; n < nparts; ++n) sum += src[n * part_stride];                                   // fixed order
        val[q][m] = sum;
      }
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) val[q] *= scale;
  const int s0 = o.segoff[v], L = o.segoff[v + 1] - s0;
  if (L >= o.long_seg) {
    const float* ls = o.longsum + (int64_t)o.longbase[v] * o.dq + j0;
    for (int c = long_parts(o, L); c > 0; --c, ls += o.dq)
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int m = 0; m < 4; ++m) val[q][m] -= ls[q * step + m] * x_s;
  } else if (L >= LONG_SEG) {
    // where dW took several launches: the entries' sum first and then x_s, in the order in which a wave of bwd_dw_long_kernel adds
    // them (four row lanes, then the lanes pairwise)
#pragma unroll 1
    for (int q = 0; q < 4; ++q) {
      v4f sum = (v4f){0.f, 0.f, 0.f, 0.f}, even = sum;
#pragma unroll 1
      for (int u = 0; u < 4; ++u) {
        v4f a = (v4f){0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
        for (int n = u; n < L; n += 4) {
          const float h = o.sh[s0 + n];
          const uint32_t w = *reinterpret_cast<const uint32_t*>(o.xq + (int64_t)o.srow[s0 + n] * o.ldx + j0 + q * step);
          a[0] = fmaf(h, e4m3_to_float<0>(w), a[0]);
          a[1] = fmaf(h, e4m3_to_float<1>(w), a[1]);
          a[2] = fmaf(h, e4m3_to_float<2>(w), a[2]);
          a[3] = fmaf(h, e4m3_to_float<3>(w), a[3]);
        }
        if (u & 1) { even += a; sum = u == 1 ? even : sum + even; }
        else even = a;
      }
#pragma unroll
      for (int k = 0; k < 4; ++k)                         // (registers are not indexed)
        if (k == q)
#pragma unroll
          for (int m = 0; m < 4; ++m) val[k][m] -= sum[m] * x_s;
    }
  } else if (L > 0) {
    for (int n = 0; n < L; ++n) {
      const float h = o.sh[s0 + n] * x_s;
      const uint8_t* row = o.xq + (int64_t)o.srow[s0 + n] * o.ldx + j0;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const uint32_t w = *reinterpret_cast<const uint32_t*>(row + q * step);
        val[q][0] -= h * e4m3_to_float<0>(w);
        val[q][1] -= h * e4m3_to_float<1>(w);
        val[q][2] -= h * e4m3_to_float<2>(w);
        val[q][3] -= h * e4m3_to_float<3>(w);
      }
    }
  }
  T* dw = reinterpret_cast<T*>(o.dw);
#pragma unroll
  for (int q = 0; q < 4; ++q)
#pragma unroll
    for (int m = 0; m < 4; ++m)
      if (j0 + q * step + m < o.d) Elem<T>::store(dw + (int64_t)(j0 + q * step + m) * o.dw_ld + v, val[q][m]);
}

}  // namespace sce
