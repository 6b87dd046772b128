// Forward kernels: row-boost sample, the logit-tile walk with its epilogues, combination of the vocabulary splits,
// mean reduction (internal header).
// Part of the one translation unit sce_kernels.hip, which includes it after the headers it builds on.
#pragma once

namespace sce {

// ------------------------------------------------------------------------------------------
// forward
// ------------------------------------------------------------------------------------------
struct FwdParams {
  const uint8_t* xq;       // [Np][dp]
  const uint8_t* wqt;      // [Vp][dp]
  float4* partials;        // [S][Np]: sum exp(z - cap), max u, argmax u (bits), unused
  const int64_t* targets;  // (N,)
  float* s_uy;             // [n_predict][Np]: raw logit u at the target of (offset, row): from fwd_sample_kernel (PRE), else written by the workgroup that meets it
  uint8_t* ghat_t;         // EMIT: G, all Np rows, tile by tile (kbv blocks of 128 columns per tile of 256 rows)
  uint32_t* gexp;          // EMIT: its block exponents [Vp / 128][kbw]
  float *lam, *lam2;       // EMIT: the two numbers of every row's exponent boost (row_boost), from the sample kernels
  int64_t ignore_index;
  int64_t dp, ldx;         // K extent and row stride of xq / wqt
  int64_t kbw, kbv;        // blocks of 128 rows (the exponents' row stride) and of 128 columns
  int N, V, Np, RT, CT, S, n_predict;      // V: columns that take part; CT: column tiles walked (EMIT: all of Vp / 256)
  float sc;                // x_s * w_s
  float k1;                // x_s * w_s * 2 log2(e) / cap : exp2(acc * k1) = e^{2u/cap}
  float ic2;               // 1 / c2, c2 = -2 cap log2(e): e^{z - cap} = exp2(c2 / (1 + e^{2u/cap}))
  float c2;
  float em2cap;            // e^{-2 cap}: what a logit of -inf adds to the sum of e^{z - cap}
  const DevConsts* dc;     // non-NULL: sc and k1 come from here (a scale lives on the device)
  uint8_t* hdr;            // header of the saved state
  int halves;              // EMIT and PRE: this many tiles of every row tile, whole ones of the vocabulary, are shared out in halves (fwd_halves)
  int want_argmax;         // the caller asks for the rows' argmax: the column of the running maximum is tracked
};

// What a forward call was asked for, as far as the matching backward call must have been asked the same: left in the header
// of the saved state (HDR_MODE_OFF bytes in) by fwd_combine_kernel and compared by bwd_prep_kernel.  A backward call whose
// flags differ would read dlogits that were never written, or mask other columns: it gets NaN gradients instead.
struct CallMode {
  int32_t emit, vocab_limit, n_predict, cap_bits;
};
constexpr int HDR_MODE_OFF = 64;
static inline CallMode call_mode(bool emit, int vocab_limit, int n_predict, float cap) {
  CallMode m;
  m.emit = emit ? 1 : 0; m.vocab_limit = vocab_limit; m.n_predict = n_predict;
  memcpy(&m.cap_bits, &cap, 4);
  return m;
}

// ... and HDR_COUNT_OFF bytes in, how many blocks of fwd_combine_kernel are done: set to zero by the forward kernel before it.
constexpr int HDR_COUNT_OFF = 128;
__device__ __forceinline__ uint32_t* done_count(const FwdParams& p) { return reinterpret_cast<uint32_t*>(p.hdr + HDR_COUNT_OFF); }

// Per 256 x 256 tile and per row a lane owns: add up e^{z - cap} over its 64 columns and keep the
// largest raw accumulator.  z is bounded by +-cap, so no running maximum is needed for the sum:
//   t = tanh(u/cap) = 1 - 2/(E + 1), E = e^{2u/cap};   e^{z - cap} = exp2(c2 / (E + 1)).
// The column of the maximum is looked up only on the (rare, after the first tiles) occasion that
// a tile raises a row's running maximum.
//
// Row block b of the tile.  hook(b, k), k = 0..31: called between the stages of the arithmetic, as in form_dlogits.  The order of the sum is that of
// the columns a lane owns.
template <int b, bool BF16, class Hook = NoHook>
__device__ __forceinline__ void fwd_epilogue(v16f (&acc)[4][4], const FwdParams& p, int col0, float* wave_stat, Hook&& hook = NoHook()) {
  constexpr bool HOOKED = !std::is_same<typename std::decay<Hook>::type, NoHook>::value;
  __builtin_amdgcn_sched_barrier(0);
  auto stage_end = [&](int k) {
    __builtin_amdgcn_sched_barrier(0);
    if (HOOKED) { hook(b, k); __builtin_amdgcn_sched_barrier(0); }
  };
  float tmax = -INFINITY, s = 0.f;
#pragma unroll
  for (int a = 0; a < 4; ++a) {
#pragma unroll
    for (int g0 = 0; g0 < 16; g0 += 8) {
      float pt[16];
      // the GEMM of the eager head returns bf16: the logits are rounded once, in place, and everything after sees the rounded values
      if (BF16) {
#pragma unroll
        for (int r = g0; r < g0 + 8; ++r) acc[a][b][r] = round_to_bf16_hw(acc[a][b][r]);
      }
#pragma unroll
      for (int r = g0; r < g0 + 8; ++r) pt[r] = fast_exp2(acc[a][b][r] * p.k1);
      stage_end(4 * (2 * a + g0 / 8));
      // z - cap = c2 / (1 + e^{2u/cap}) in units of log2: the reciprocal of (1 + e) / c2 gives it in one step
#pragma unroll
      for (int r = g0; r < g0 + 8; ++r) pt[r] = fast_rcp(fmaf(pt[r], p.ic2, p.ic2));
      stage_end(4 * (2 * a + g0 / 8) + 1);
#pragma unroll
      for (int r = g0; r < g0 + 8; ++r) pt[r] = fast_exp2(pt[r]);
      stage_end(4 * (2 * a + g0 / 8) + 2);
#pragma unroll
      for (int r = g0; r < g0 + 8; ++r) {
        s += pt[r];
        tmax = fmaxf(tmax, acc[a][b][r]);
      }
      stage_end(4 * (2 * a + g0 / 8) + 3);
    }
  }
  float* stat = wave_stat + lane_id();      // (taken anew, as the columns are below: nothing of them stays live across the arithmetic)
  stat[(0 + b) * NTHREADS] += s;
  const float amax = stat[(4 + b) * NTHREADS];
  if (p.want_argmax && __builtin_amdgcn_ballot_w64(tmax > amax) != 0) {
    if (tmax > amax) {
      int targ = 0x7fffffff;
#pragma unroll
      for (int a = 3; a >= 0; --a) {
#pragma unroll
        for (int r = 15; r >= 0; --r) {
          const int vo = a * 32 + 8 * (r >> 2) + (r & 3);
          if (acc[a][b][r] == tmax) targ = vo;   // descending scan: lowest column wins
        }
      }
      stat[(4 + b) * NTHREADS] = tmax;
      stat[(8 + b) * NTHREADS] = __int_as_float(col0 + 4 * (lane_id() >> 5) + targ);
    }
  }
}

// The sums of the four row blocks again, on top of the ones before this tile (stat[12 ..]), over the columns that exist (the
// others are -inf).  They are kept out by a factor of 0 or 1: 64 comparisons would be kept in scalar registers from block to block, and spilled.
__device__ __forceinline__ void sums_of_existing_columns(const v16f (&acc)[4][4], const FwdParams& p, int col0, float* wave_stat) {
  float* stat = wave_stat + lane_id();
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    int left = p.V - col0 - 4 * (lane_id() >> 5);
    asm volatile("" : "+v"(left));
    float s = 0.f;
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        s = fmaf((float)min(max(left - (a * 32 + 8 * (r >> 2) + (r & 3)), 0), 1), fast_exp2(fast_rcp(fmaf(fast_exp2(acc[a][b][r] * p.k1), p.ic2, p.ic2))), s);
    stat[(0 + b) * NTHREADS] = stat[(12 + b) * NTHREADS] + s;
  }
}

__device__ __forceinline__ bool target_valid(const int64_t* __restrict__ targets, int64_t ignore_index, int i, int N, int V) {
  if (i >= N) return false;
  const int64_t y = targets[i];
  return (y != ignore_index) && y >= 0 && y < V;
}

// The raw logit at a row's targets, taken from the accumulators of the tile that holds the target column, so that z_y
// and lse come from the same numbers: the fp8 matrix instruction sums with less than fp32 care (it aligns its 64 products
// to the largest and drops what falls below about 2^-12 of it: about 2e-5 low on a sum of like-signed terms at K = 2560), and a z_y from a separate fp32 dot product would leave that bias in z_y - lse, i.e. in
// 1 - p_y, where rows the model is sure of cannot afford it.  tgt (LDS): [4 offsets][TGT_STRIDE rows] target column or
// -1, already at the wave's first row.  A lane looks at its four rows; the 64-way select runs only when some lane of
// the wave has a hit (a few per cent of the tiles) -- but the compiler moves the row block's 64 accumulators out of the
// accumulation registers around every offset's lookup, hit or not, which is why the fp8 kernels take their target
// logits from fwd_sample_kernel where they can (PRE) and this function serves the rest: the bf16 kernel, and W_q^T
// beyond that kernel's reach.
// STORE: the logit goes to s_uy_tile[offset][row] (global).
// KNOCK: the accumulator of the target is then set to -inf, for the dlogits epilogue that follows: the target takes
//        no part in the stored dlogits (its column is handled in fp32, see bwd_prep_kernel) and must not set the
//        exponent of its block either -- a row the model is sure of would push its own other columns, and its
//        neighbours', out of the 8 bits.
// B0, B1: the row blocks [B0, B1) only.
// STATS: with KNOCK, the row statistics (stat, as in form_dlogits) take the target's share here: e^{z_y - cap} into the
//        sum, and the running maximum / argmax.
template <bool STORE, bool KNOCK, bool STATS, int TGT_STRIDE, int B0 = 0, int B1 = 4>
__device__ __forceinline__ void take_target_logits(v16f (&acc)[4][4], const int* tgt, int n_predict, int col0, int rowbase,
                                                   float sc, float* s_uy_tile, int Np, float* stat, float k1, float ic2, float em2cap) {
  const int lane = lane_id(), half = lane >> 5;
#pragma unroll
  for (int b = B0; b < B1; ++b) {
    const int row = b * 32 + (lane & 31);
    float xk[4] = {0.f, 0.f, 0.f, 0.f};
    for (int k = 0; k < n_predict; ++k) {
      const int y = tgt[k * TGT_STRIDE + row];
      const int rel = y - col0;                        // column within the wave's 128
      const bool hit = (unsigned)rel < 128u && ((rel >> 2) & 1) == half;
      if (__builtin_amdgcn_ballot_w64(hit) != 0) {
        if (hit) {
          const int idx = (rel >> 5) * 16 + ((rel >> 3) & 3) * 4 + (rel & 3);
          float x = 0.f;
          bool again = false;                          // an earlier offset of this row has the same target
          if (KNOCK) {
            for (int k2 = 0; k2 < k; ++k2)
              if (tgt[k2 * TGT_STRIDE + row] == y) { again = true; x = xk[k2]; }
          }
          if (!again) {
#pragma unroll
            for (int a = 0; a < 4; ++a)
#pragma unroll
              for (int r = 0; r < 16; ++r) {
                x = (idx == a * 16 + r) ? acc[a][b][r] : x;
                if (KNOCK) acc[a][b][r] = (idx == a * 16 + r) ? -INFINITY : acc[a][b][r];
              }
            if (KNOCK && STATS) {
              // (the -inf left behind reads as z = -cap to the epilogue that follows, which will add e^{-2 cap} for it)
              stat[(0 + b) * NTHREADS] += fast_exp2(fast_rcp(fmaf(fast_exp2(x * k1), ic2, ic2))) - em2cap;
              const float amax = stat[(4 + b) * NTHREADS];
              if (x > amax || (x == amax && y < __float_as_int(stat[(8 + b) * NTHREADS]))) {
                stat[(4 + b) * NTHREADS] = x;
                stat[(8 + b) * NTHREADS] = __int_as_float(y);
              }
            }
          }
          xk[k] = x;
          // (the lane index is taken anew: an address kept from outside the branch stays live across the main loop and is spilled)
          if (STORE) s_uy_tile[(int64_t)k * Np + rowbase + b * 32 + (lane_id() & 31)] = x * sc;
        }
      }
    }
  }
}

// A row's boost from the two numbers that were left for it (see sample_rows; fwd_sample_kernel leaves its one number twice).
__device__ __forceinline__ float row_boost(const float* __restrict__ lam, const float* __restrict__ lam2, int64_t i) {
  const float l = fminf(lam[i], lam2[i]);
  return l > -64.f ? (l < 120.f ? l : 120.f) : -64.f;            // (NaN: -64)
}

// The exponent boost of every row: lam_i = floor(-log2 Z^_i), Z^_i an estimate of the row's softmax sum Z_i = sum_v e^{z_iv - cap}
// made before the forward kernel starts, so that the stored value D 2^lam is close to the row's probabilities
// (times 1 - t^2) whatever the level of its logits.  Two tiles of logits go into it (one workgroup per row tile):
//   * 256 columns from the middle of the vocabulary, for the level of the row's bulk: V times m_i, the smallest of the
//     means of e^{z - cap} over 16 groups of 16 columns (the smallest, so that a few peaks inside the sample do not
//     pass for the level of the row);
//   * the 256 columns that are the targets of the tile's own rows (the rows of W^T gathered by the tile loader): the
//     row's own target -- where a confident row that is right has most of its sum -- and the tokens around it in the
//     text, where a language model's rows tend to have their other peaks.
// Every single e^{z - cap} is a lower bound of the sum, so Z^_i = max(V m_i, largest value seen in either tile).  What
// the estimate cannot see is a peak in a column that is in neither tile: such a row is boosted too far by the share
// of that peak in its sum (see form_dlogits for what that costs the rows that share its blocks).
// A row that has no valid target at all takes no part in the backward pass (its weight is zero): it gets the lowest
// boost, so that whatever its logits hold cannot set the exponent of a block.
//
// GATHER = false: the first tile only (the gathered rows' offsets would not fit the loader's 32 bits: W_q^T of 4 GiB or more).
// GATHER = true also leaves the target logits of the tile's rows in s_uy, for the forward kernel that follows: u[i, y_{i+k}]
// is element (i, i + k) of the gathered tile, computed by the same instructions in the same order as the forward
// kernel will compute it (bit for bit: that kernel recognises the entry by its value).  The offsets k >= 1 of the
// tile's last rows point at targets of the next tile's rows: those (at most three) ride as the last columns of the
// first tile, in place of the sampled columns there.
constexpr int SMEM_SAMPLE = SMEM_BYTES + 2 * 256 * 4 + 8 * 256 * 4;      // the K slots, the gathered rows, the rows without a target, the first tile's results
// BOOST = false (with GATHER): the target logits only, for a forward pass that emits nothing (the first tile is then
// computed only for the sake of its last columns, i.e. with more than one offset).
template <bool GATHER, bool BOOST = true>
__global__ __launch_bounds__(256) void fwd_sample_kernel(FwdParams p_in, int ct) {
  static_assert(GATHER || BOOST, "nothing to do");
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  FwdParams p = p_in;
  if (p.dc) { p.sc = p.dc->sc; p.k1 = p.dc->k1; }
  const int rt = blockIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wa = wave >> 1, wb = wave & 1;
  int* rows = reinterpret_cast<int*>(smem + SMEM_BYTES);         // [256]: the row of W^T that column j of a tile is
  int* dead = rows + 256;                                        // [256]: row j has no valid target
  const int ntail = GATHER ? p.n_predict - 1 : 0;                // columns 256 - ntail .. 255 of the first tile: the next rows' targets
  auto column_of = [&](int64_t y) { return (y != p.ignore_index && y >= 0 && y < p.V) ? (int)y : 0; };
  if (GATHER) {
    // (a row without a target stands in with column 0: any column of the vocabulary gives a valid lower bound of the sum)
    const int t = threadIdx.x, j = t - (256 - ntail), row = rt * 256 + 256 + j;
    rows[t] = j < 0 ? ct * 256 + t : column_of(row < p.N ? p.targets[row] : p.ignore_index);
    __syncthreads();
  }
  // the targets of the thread's row are fetched before the first main loop, which hides the wait
  int64_t yraw[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int row = rt * 256 + (int)threadIdx.x;
    yraw[k] = (k < p.n_predict && row + k < p.N && row < p.N) ? p.targets[row + k] : p.ignore_index;
  }
  v16f acc[4][4];
  const bool first_tile = BOOST || ntail > 0;
  if (first_tile) {
    if (GATHER) mfma_mainloop(p.wqt, p.ldx, p.xq + (int64_t)rt * 256 * p.ldx, p.ldx, (int)(p.dp / BK), smem, acc, 0, 0, wave, NoHook(), 0, 0, nullptr, rows);
    else mfma_mainloop(p.wqt + (int64_t)ct * 256 * p.ldx, p.ldx, p.xq + (int64_t)rt * 256 * p.ldx, p.ldx, (int)(p.dp / BK), smem, acc, 0, 0, wave);
  }
  {
    bool any = false;
#pragma unroll
    for (int k = 0; k < 4; ++k) any = any || (yraw[k] != p.ignore_index && yraw[k] >= 0 && yraw[k] < p.V);
    rows[threadIdx.x] = column_of(yraw[0]);
    dead[threadIdx.x] = !any;
  }
  const int lane = lane_id();
  if (GATHER && first_tile) {
    // columns 252 .. 255 are registers 12 .. 15 of A block 3 in the upper half-wave of the waves with wa = 1; rows 224 .. 255
    // are B block 3 of the waves with wb = 1
    const int i = 224 + (lane & 31);
    const bool mine = wave == 3 && lane >= 32;
#pragma unroll
    for (int r = 12; r < 16; ++r) {
      const int k = 256 + (252 + (r & 3) - (256 - ntail)) - i;       // the offset of row i that this column serves
      if (mine && 252 + (r & 3) >= 256 - ntail && k >= 1 && k < p.n_predict) p.s_uy[(int64_t)k * p.Np + rt * 256 + i] = acc[3][3][r] * p.sc;
    }
  }
  const int vlim = min(p.V - ct * 256, 256 - ntail), vloc0 = wa * 128 + 4 * (lane >> 5);
  float gmin[4], top[4];                                         // top: the largest logit seen (in the accumulator's units)
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    gmin[b] = INFINITY; top[b] = -INFINITY;
    if (!BOOST) continue;
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      float sum = 0.f, cnt = 0.f;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float pt = fast_exp2(fast_rcp(fmaf(fast_exp2(acc[a][b][r] * p.k1), p.ic2, p.ic2)));
        const bool live = vloc0 + a * 32 + 8 * (r >> 2) + (r & 3) < vlim;
        sum += live ? pt : 0.f;
        cnt += live ? 1.f : 0.f;
        top[b] = live ? fmaxf(top[b], acc[a][b][r]) : top[b];
      }
      if (cnt > 0.f) gmin[b] = fminf(gmin[b], sum / cnt);
    }
  }
  if (GATHER && p.n_predict > 0) {      // (a condition the compiler cannot decide: merged into one block, the code of the two main loops is spilled)
    // the first tile's results wait in LDS: there is no register for them in the main loop
    float* keep = reinterpret_cast<float*>(smem + SMEM_BYTES + 2048) + threadIdx.x;
#pragma unroll
    for (int b = 0; b < 4; ++b) { keep[b * 256] = gmin[b]; keep[(4 + b) * 256] = top[b]; }
    __syncthreads();
    mfma_mainloop(p.wqt, p.ldx, p.xq + (int64_t)rt * 256 * p.ldx, p.ldx, (int)(p.dp / BK), smem, acc, 0, 0, wave, NoHook(), 0, 0, nullptr, rows);
    keep = reinterpret_cast<float*>(smem + SMEM_BYTES + 2048) + wave * 64 + lane_id();
#pragma unroll
    for (int b = 0; b < 4; ++b) { gmin[b] = keep[b * 256]; top[b] = keep[(4 + b) * 256]; }
    if (BOOST) {
#pragma unroll
      for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int a = 0; a < 4; ++a)
#pragma unroll
          for (int r = 0; r < 16; ++r) top[b] = fmaxf(top[b], acc[a][b][r]);
    }
    // The band 0 <= column - row < n_predict lies in the 32 x 32 blocks on the diagonal and right of it: blocks (a, b) with
    // a - b = 0 or 1 of the waves with wa = wb, block (0, 3) of the wave with wa = 1, wb = 0.  (Stores under a lane
    // condition, no branches around the accumulators.)
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
      for (int a = b; a < 5; ++a) {
        if (a > b + 1 && !(a == 4 && b == 3)) continue;
        const int aa = a & 3;                                    // (a = 4: A block 0 of the waves one to the right)
        const bool mine = a < 4 ? wa == wb : (wa == 1 && wb == 0);
        const int i = wb * 128 + b * 32 + (lane_id() & 31);      // (the lane index taken anew: what is prepared before the main loop is spilled across it)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int k = wa * 128 + aa * 32 + 8 * (r >> 2) + 4 * (lane_id() >> 5) + (r & 3) - i;
          if (mine && k >= 0 && k < p.n_predict) p.s_uy[(int64_t)k * p.Np + rt * 256 + i] = acc[aa][b][r] * p.sc;
        }
        __builtin_amdgcn_sched_barrier(0);      // (one block's accumulators at a time: all of them moved up front do not fit the registers)
      }
  }
  if (!BOOST) return;
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    gmin[b] = fminf(gmin[b], __shfl_xor(gmin[b], 32));
    top[b] = fmaxf(top[b], __shfl_xor(top[b], 32));
  }
  float* red = reinterpret_cast<float*>(smem);          // free: the main loop has ended in every wave
  if (wa == 1 && lane < 32) {
#pragma unroll
    for (int b = 0; b < 4; ++b) { red[wb * 128 + b * 32 + lane] = gmin[b]; red[256 + wb * 128 + b * 32 + lane] = top[b]; }
  }
  __syncthreads();
  if (wa == 0 && lane < 32) {
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const float m = fminf(gmin[b], red[wb * 128 + b * 32 + lane]), u = fmaxf(top[b], red[256 + wb * 128 + b * 32 + lane]);
      const float peak = fast_exp2(fast_rcp(fmaf(fast_exp2(u * p.k1), p.ic2, p.ic2)));       // (u = -inf: e^{-2 cap})
      float l = floorf(-log2f(fmaxf((float)p.V * m, peak)));
      l = l > -64.f ? (l < 120.f ? l : 120.f) : -64.f;
      l = dead[wb * 128 + b * 32 + lane] ? -64.f : (l == l ? l : 0.f);
      const int i = rt * 256 + wb * 128 + b * 32 + lane;
      p.lam[i] = l; p.lam2[i] = l;
    }
  }
}

// The same numbers, bit for bit, with 32 RB rows and one of the two tiles to a workgroup instead of 256 rows and both: there
// are 16 / RB workgroups to a row tile, and the two K loops do not run one behind the other.  The eight waves of a workgroup take 32 of
// the tile's 256 columns each.  A 128-byte K block of the 256 rows of W_q^T and of the workgroup's own rows comes by direct loads,
// whole 128-byte pieces of rows, into a ring of STAGES LDS slots, STAGES - 1 blocks ahead; the swizzle, the bytes of a fragment
// and the order in which an accumulator block adds up are those of mfma_mainloop.  What bounds it is the path from L2 (32 + 4 RB KB a K
// block, 64 bytes a clock).  Before, each lane fetched its own 32 bytes of a row straight into registers, 64 pieces of 16
// bytes of 32 rows to an instruction, and the address unit took a clock for each.  Measured, V = 50304 unless said, that kernel or
// (over 8192 rows) fwd_sample_kernel against this: 1000 rows, d = 256, V = 4096 10.8 -> 5.7 us; 2048 rows, d = 768 21 -> 8.4, d = 1024
// 26 -> 9.9; 4096, d = 1600 45 -> 15; 8192, d = 1024 28 -> 13.7, d = 2560 61 -> 23; 16384, d = 1024 47 -> 18, d = 4096 and V = 131072 108 -> 45;
// 30011, d = 2560 85 -> 61; 32768, d = 1024 50 -> 35; 65536, d = 1024 58 for its 73, d = 2560 106 for 121.  So up to SAMPLE_RING_TILES row
// tiles, two rounds of workgroups with RB = 4 (three take as long as fwd_sample_kernel).  RB: the least with which one round of
// workgroups, one to a CU, is enough (8192 rows, d = 1024: 20, 13.7 and 18 us with 1, 2 and 4; 2048 rows: 9.9, 11.3, 14.9).
// What the two tiles say of a row stays apart -- lam[i] from the first, lam2[i] from the second, floor(-log2 of its
// estimate) each -- and row_boost takes the smaller: the floor of the larger estimate's.
constexpr int SAMPLE_THREADS = 512, SAMPLE_RING_TILES = 128;
static inline int sample_row_blocks(int RT) { return RT <= 16 ? 1 : RT <= 32 ? 2 : 4; }
template <int RB>
struct SampleRing {
  static constexpr int X_BYTES = 32 * RB * BK, STAGE = 256 * BK + X_BYTES, STAGES = RB == 4 ? 3 : 4;
  static constexpr int XL = RB == 4 ? 2 : 1, LOADS = 4 + XL;      // direct loads of a wave per K block (RB = 1: the second four waves load x again)
  static constexpr int SMEM = STAGES * STAGE;
  static_assert(SMEM <= SMEM_MAX && 2 * 8 * 32 * RB * 4 <= SMEM, "LDS: the ring, and after it the results of the waves");
};
template <int RB>
__device__ __forceinline__ void sample_rows(const FwdParams& p, int ct, uint8_t* smem) {
  using R = SampleRing<RB>;
  constexpr int GROUPS = 8 / RB;                                 // workgroups to the 256 rows of a tile
  // neighbours in this order run on one XCD: those of a row tile, whose gathered rows of W_q^T are the same
  const int total = p.RT * 2 * GROUPS, per = (total + 7) >> 3, idx = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per || idx >= total) return;
  const int rt = idx / (2 * GROUPS), rest = idx - rt * (2 * GROUPS);
  const bool second = rest >= GROUPS;                            // this workgroup's columns are the targets
  const int r0 = (second ? rest - GROUPS : rest) * 32 * RB;      // its first row in the row tile
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = lane_id(), h = lane >> 5;
  const int ntail = p.n_predict - 1;
  auto target_of = [&](int row) { return row < p.N ? p.targets[row] : p.ignore_index; };
  auto column_of = [&](int64_t y) { return (y != p.ignore_index && y >= 0 && y < p.V) ? (int)y : 0; };
  auto row_of_w = [&](int j) {                                   // the row of W^T that column j of the tile is
    const int q = j - (256 - ntail);
    if (second) return column_of(target_of(rt * 256 + j));
    return q < 0 ? ct * 256 + j : column_of(target_of(rt * 256 + 256 + q));
  };
  const uint32_t lds0 = (uint32_t)(uintptr_t)((__attribute__((address_space(3))) void*)smem);
  // one load: 8 rows of 128 bytes; a wave loads the W rows of its own 32 columns
  const int lr = lane >> 3, pc = lane & 7;
  auto swizzled = [&](int row) { return (uint32_t)((pc ^ ((row & 7) ^ ((row >> 3) & 1))) * 16); };
  auto xload = [&](int n) { return RB == 1 ? wave & 3 : wave * R::XL + n; };
  uint32_t wo[4], xo[R::XL];
#pragma unroll
  for (int n = 0; n < 4; ++n) wo[n] = (uint32_t)(row_of_w(wave * 32 + n * 8 + lr) * p.ldx) + swizzled(n * 8 + lr);
#pragma unroll
  for (int n = 0; n < R::XL; ++n) { const int row = xload(n) * 8 + lr; xo[n] = (uint32_t)(row * p.ldx) + swizzled(row); }
  const uint8_t* xbase = uniform_ptr(p.xq + (int64_t)(rt * 256 + r0) * p.ldx);
  const int nk = (int)(p.dp / BK);
  int ik = 0, islot = 0;                                         // the K block that is loaded next
  auto issue = [&]() {
    const uint32_t l = lds0 + islot * R::STAGE;
    const uint8_t* wb = p.wqt + (int64_t)ik * BK;
    const uint8_t* xb = xbase + (int64_t)ik * BK;
    lds_direct_16<0>(l + wave * 4096, wo[0], wb);
    lds_direct_16<1024>(l + wave * 4096, wo[1], wb);
    lds_direct_16<2048>(l + wave * 4096, wo[2], wb);
    lds_direct_16<3072>(l + wave * 4096, wo[3], wb);
#pragma unroll
    for (int n = 0; n < R::XL; ++n) lds_direct_16<256 * BK>(l + xload(n) * 1024, xo[n], xb);
    ++ik;
    if (++islot == R::STAGES) islot = 0;
  };
#pragma unroll 1
  for (int g = 0; g < R::STAGES - 1 && g < nk; ++g) issue();
  v16f acc[RB];
#pragma unroll
  for (int q = 0; q < RB; ++q)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[q][r] = 0.f;
  const int fr = lane & 31, fsw = (fr & 7) ^ ((fr >> 3) & 1);
  int slot = 0;
#pragma unroll 1
  for (int k = 0; k < nk; ++k) {
    // this wave's loads of the block have landed and its reads of the one before are complete; after the barrier that holds for
    // every wave, and the slot of the block before is free
    if (k + R::STAGES - 1 <= nk) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((R::STAGES - 2) * R::LOADS) : "memory");
    else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (k + R::STAGES - 1 < nk) issue();
    const uint8_t* ws = smem + slot * R::STAGE;
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      const int c0 = ((4 * half + 2 * h) ^ fsw) * 16;
      auto fragment = [&](const uint8_t* rows) {
        const v4i lo = *reinterpret_cast<const v4i*>(rows + fr * BK + c0), hi = *reinterpret_cast<const v4i*>(rows + fr * BK + (c0 ^ 16));
        return (v8i){lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      };
      const v8i fw = fragment(ws + wave * 4096);
      v8i fx[RB];
#pragma unroll
      for (int q = 0; q < RB; ++q) fx[q] = fragment(ws + 256 * BK + q * 4096);
#pragma unroll
      for (int q = 0; q < RB; ++q) acc[q] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(fw, fx[q], acc[q], 0, 0, 0, 0, 0, 0);
    }
    if (++slot == R::STAGES) slot = 0;
  }
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");      // the ring is free for the waves' results
  float* gmins = reinterpret_cast<float*>(smem);                 // [8 waves][32 RB]
  float* tops = gmins + 8 * 32 * RB;
  // element (row i, column j) of the tile is in register r: j = 32 wave + 8 (r / 4) + 4 h + r % 4
  const int vlim = second ? 256 : min(p.V - ct * 256, 256 - ntail);
#pragma unroll
  for (int q = 0; q < RB; ++q) {
    const int rb = r0 / 32 + q, i = rb * 32 + (lane & 31);       // block of 32 rows, the lane's row in the row tile
    if (second) {
      if (wave == rb || wave == rb + 1)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int k = 32 * wave + 8 * (r >> 2) + 4 * h + (r & 3) - i;
          if (k >= 0 && k < p.n_predict) p.s_uy[(int64_t)k * p.Np + rt * 256 + i] = acc[q][r] * p.sc;
        }
    } else if (rb == 7 && wave == 7) {                           // the next row tile's targets: columns 256 - ntail on of the first tile
#pragma unroll
      for (int r = 12; r < 16; ++r) {
        const int j = 252 + (r & 3), k = 256 + (j - (256 - ntail)) - i;
        if (h == 1 && j >= 256 - ntail && k >= 1 && k < p.n_predict) p.s_uy[(int64_t)k * p.Np + rt * 256 + i] = acc[q][r] * p.sc;
      }
    }
    float gmin = INFINITY, top = -INFINITY, sum = 0.f, cnt = 0.f;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const bool live = 32 * wave + 8 * (r >> 2) + 4 * h + (r & 3) < vlim;
      if (!second) {
        const float pt = fast_exp2(fast_rcp(fmaf(fast_exp2(acc[q][r] * p.k1), p.ic2, p.ic2)));
        sum += live ? pt : 0.f;
        cnt += live ? 1.f : 0.f;
      }
      top = live ? fmaxf(top, acc[q][r]) : top;
    }
    if (cnt > 0.f) gmin = sum / cnt;
    gmin = fminf(gmin, __shfl_xor(gmin, 32));
    top = fmaxf(top, __shfl_xor(top, 32));
    if (h == 0) { gmins[(wave * RB + q) * 32 + lane] = gmin; tops[(wave * RB + q) * 32 + lane] = top; }
  }
  __syncthreads();
  const int t = threadIdx.x;
  if (t >= 32 * RB) return;
  float gmin = INFINITY, top = -INFINITY;
#pragma unroll
  for (int w = 0; w < 8; ++w) { gmin = fminf(gmin, gmins[w * 32 * RB + t]); top = fmaxf(top, tops[w * 32 * RB + t]); }
  const float peak = fast_exp2(fast_rcp(fmaf(fast_exp2(top * p.k1), p.ic2, p.ic2)));
  const int row = rt * 256 + r0 + t;
  float l = floorf(-log2f(second ? peak : fmaxf((float)p.V * gmin, peak)));
  bool dead = true;
  for (int k = 0; k < p.n_predict; ++k) dead = dead && !(row < p.N && target_valid(p.targets, p.ignore_index, row + k, p.N, p.V));
  (second ? p.lam2 : p.lam)[row] = dead ? -64.f : l;
}

// BOOST = false: the target logits only, for a forward pass that emits nothing: 32 rows to a workgroup, fragments
// straight from memory to registers, four steps ahead; wave 0 computes the blocks on the diagonal and right of it, wave 1
// (a second wave only if there are several offsets) the last block of the first tile for the last rows of a row tile.  8192 rows of d = 2560
// 18 us for the 41 of fwd_sample_kernel; used up to SAMPLE_FEW_TILES row tiles.
constexpr int SAMPLE_FEW_TILES = 32;
template <bool BOOST>
__global__ __launch_bounds__(SAMPLE_THREADS) void fwd_sample_few_kernel(FwdParams p_in, int ct, int row_blocks) {
  FwdParams p = p_in;
  if (p.dc) { p.sc = p.dc->sc; p.k1 = p.dc->k1; }
  if constexpr (BOOST) {
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    if (row_blocks == 1) sample_rows<1>(p, ct, smem);
    else if (row_blocks == 2) sample_rows<2>(p, ct, smem);
    else sample_rows<4>(p, ct, smem);
    return;
  }
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = lane_id(), h = lane >> 5;
  const int rt = blockIdx.x >> 3, rb = blockIdx.x & 7;          // row tile, block of 32 rows in it
  const int ntail = p.n_predict - 1;
  const bool second = wave == 0;                                // this wave's columns are the targets
  const int ab[2] = {second ? rb : 6, second ? min(rb + 1, 7) : 7};
  if (!second && rb != 7) return;
  auto target_of = [&](int row) { return row < p.N ? p.targets[row] : p.ignore_index; };
  auto column_of = [&](int64_t y) { return (y != p.ignore_index && y >= 0 && y < p.V) ? (int)y : 0; };
  auto row_of_w = [&](int j) {                                   // the row of W^T that column j of the wave's tile is
    const int q = j - (256 - ntail);
    if (second) return column_of(target_of(rt * 256 + j));
    return q < 0 ? ct * 256 + j : column_of(target_of(rt * 256 + 256 + q));
  };
  const int i = rb * 32 + (lane & 31);                           // the lane's row in the row tile
  const uint8_t* xr = p.xq + (int64_t)(rt * 256 + i) * p.ldx + 32 * h;
  const uint8_t* wr0 = p.wqt + (int64_t)row_of_w(ab[0] * 32 + (lane & 31)) * p.ldx + 32 * h;
  const uint8_t* wr1 = p.wqt + (int64_t)row_of_w(ab[1] * 32 + (lane & 31)) * p.ldx + 32 * h;
  typedef int v8i_16 __attribute__((ext_vector_type(8), aligned(16)));
  constexpr int AHEAD = 4;                                       // steps of 64 bytes; the K extent is a multiple of 256
  v8i fx[AHEAD], fw[AHEAD][2];
  auto load = [&](int u, int64_t k) {
    fx[u] = *reinterpret_cast<const v8i_16*>(xr + k);
    fw[u][0] = *reinterpret_cast<const v8i_16*>(wr0 + k);
    fw[u][1] = *reinterpret_cast<const v8i_16*>(wr1 + k);
  };
#pragma unroll
  for (int u = 0; u < AHEAD; ++u) load(u, 64 * u);
  v16f acc[2];
#pragma unroll
  for (int r = 0; r < 16; ++r) { acc[0][r] = 0.f; acc[1][r] = 0.f; }
  for (int64_t k = 0; k < p.dp; k += 64 * AHEAD) {
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) {
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int a = 0; a < 2; ++a) acc[a] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(fw[u][a], fx[u], acc[a], 0, 0, 0, 0, 0, 0);
      if (k + 64 * AHEAD < p.dp) load(u, k + 64 * (AHEAD + u));
    }
  }
  // element (row i, column j) of the wave's tile is in register r of block a: j = 32 ab[a] + 8 (r / 4) + 4 h + r % 4
  if (second) {
#pragma unroll
    for (int a = 0; a < 2; ++a)
      if (ab[a] == rb || ab[a] == rb + 1)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int k = 32 * ab[a] + 8 * (r >> 2) + 4 * h + (r & 3) - i;
          if (k >= 0 && k < p.n_predict) p.s_uy[(int64_t)k * p.Np + rt * 256 + i] = acc[a][r] * p.sc;
        }
  } else if (rb == 7 && ab[1] == 7) {                            // the next row tile's targets: columns 256 - ntail on of the first tile
#pragma unroll
    for (int r = 12; r < 16; ++r) {
      const int j = 252 + (r & 3), k = 256 + (j - (256 - ntail)) - i;
      if (h == 1 && j >= 256 - ntail && k >= 1 && k < p.n_predict) p.s_uy[(int64_t)k * p.Np + rt * 256 + i] = acc[1][r] * p.sc;
    }
  }
}

// The target entries of the dlogits that a forward pass has emitted are set to zero (fwd_combine_kernel, which looks at every
// row's targets anyway; in backward, of dlogits formed again, fwd_knock_kernel, one thread per row): they take no part in D
// (their share goes into the one-hot coefficient in fp32, see bwd_prep_kernel).
__device__ __forceinline__ void knock_target(uint8_t* __restrict__ ghat, int64_t kbv, int i, int64_t y) {
  ghat[((int64_t)(i >> 8) * kbv + (y >> 7)) * BLOCKED_KSTEP + (i & 255) * BK + (y & 127)] = 0;
}
__global__ __launch_bounds__(256) void fwd_knock_kernel(uint8_t* __restrict__ ghat, int64_t kbv, const int64_t* __restrict__ targets,
                                                       int64_t ignore_index, int N, int V, int n_predict) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= N) return;
  for (int k = 0; k < n_predict; ++k) {
    if (!target_valid(targets, ignore_index, i + k, N, V)) continue;
    knock_target(ghat, kbv, i, targets[i + k]);
  }
}

// LDS of the forward kernel: the two K slots; the row statistics of the workgroup's walk (12 values per lane, and the boosts of
// its rows: kept in registers they are spilled around the main loop, and the reload -- a vector memory load -- makes the
// epilogue wait for the tile loads that were just put in flight for the next tile); the targets of the workgroup's 256 rows.
constexpr int FWD_STAT_OFF = SMEM_MAX - 4096 - 16 * 4 * NTHREADS;      // 12 statistics and the boosts of the lane's 4 rows
constexpr int FWD_TGT_OFF = SMEM_MAX - 4096;
constexpr int FWD_UY_OFF = FWD_STAT_OFF - 4096;                        // PRE: the target logits of the rows, laid out like the targets
constexpr int SMEM_FWD = SMEM_MAX;
static_assert(SMEM_BYTES <= FWD_UY_OFF, "K slots and row data overlap");

// PRE: which of the lane's values in the row block at row0 is a target of its row (one is looked for: two targets of a row in one
// lane's 64 columns are the same column, or rare enough that the second may set an exponent): its known value.
__device__ __forceinline__ float target_value(const uint8_t* smem, int n_predict, int col0, int row0) {
  const int* tgt = reinterpret_cast<const int*>(smem + FWD_TGT_OFF) + row0;
  const float* tuy = reinterpret_cast<const float*>(smem + FWD_UY_OFF) + row0;
  float v = __builtin_nanf("");
  for (int k = 0; k < n_predict; ++k) {
    const int rel = tgt[k * 256 + (lane_id() & 31)] - col0;
    if ((unsigned)rel < 128u && ((rel >> 2) & 1) == (lane_id() >> 5)) v = tuy[k * 256 + (lane_id() & 31)];
  }
  return v;
}

// EMIT: the epilogue also leaves the block-scaled dlogits of the tile in G (see form_dlogits), for a backward pass
// that does not compute the logits again.
// BF16 (without EMIT): bf16 operands, logits rounded to bf16 as the eager head's GEMM returns them (forward only).
// PRE: the target logits are in s_uy already (fwd_sample_kernel<true, .>) and this kernel does not look for them in
// its accumulators.  With EMIT the target entries go through the epilogue like any other, except that they are kept out
// of the block exponents (form_dlogits, EXCL), and fwd_combine_kernel clears their bytes of G afterwards.
template <bool EMIT, bool BF16 = false, bool PRE = false>
__global__ __launch_bounds__(256) void fwd_kernel(FwdParams p_in) {
  static_assert(!PRE || !BF16, "PRE is for the fp8 kernels");
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  FwdParams p = p_in;
  if (p.dc) { p.sc = p.dc->sc; p.k1 = p.dc->k1; }
  int rt, s;
  if (!map_tile(blockIdx.x, p.RT, p.S, rt, s)) return;
  if (blockIdx.x == 0 && threadIdx.x == 0) *done_count(p) = 0;
  const int cth = EMIT && PRE ? p.halves : 0;      // tiles [0, cth) as halves, one to a workgroup behind its whole tiles
  const int ct0 = cth + (int)((int64_t)(p.CT - cth) * s / p.S), ct1 = cth + (int)((int64_t)(p.CT - cth) * (s + 1) / p.S);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wa = wave >> 1, wb = wave & 1;
  {
    float* stat = reinterpret_cast<float*>(smem + FWD_STAT_OFF) + wave * 64 + lane_id();   // [12][256]: sum, amax, uarg of the 4 row blocks
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      stat[(0 + b) * NTHREADS] = 0.f;
      stat[(4 + b) * NTHREADS] = -INFINITY;
      stat[(8 + b) * NTHREADS] = __int_as_float(0x7fffffff);
      if (EMIT) stat[(12 + b) * NTHREADS] = row_boost(p.lam, p.lam2, rt * 256 + wb * 128 + b * 32 + (lane_id() & 31));
    }
    int* tgt = reinterpret_cast<int*>(smem + FWD_TGT_OFF);
    for (int e = threadIdx.x; e < p.n_predict * 256; e += NTHREADS) {
      const int i = rt * 256 + (e & 255) + (e >> 8);
      tgt[e] = ((e & 255) + rt * 256 < p.N && target_valid(p.targets, p.ignore_index, i, p.N, p.V)) ? (int)p.targets[i] : -1;
      if (PRE && EMIT) reinterpret_cast<float*>(smem + FWD_UY_OFF)[e] = p.s_uy[(int64_t)(e >> 8) * p.Np + rt * 256 + (e & 255)];
    }
  }
  __syncthreads();
  v16f acc[4][4];
  const uint8_t* Bg = p.xq + (int64_t)rt * 256 * p.ldx;
  const int KT = (int)(p.dp / BK);
  // of the workgroups that start together on this XCD, those with the same split share the W tiles, those with the same rt the X rows
  const int rot_a = 2 * (rt & 3), rot_b = s & 7;
  // the first K blocks of the next tile travel while the epilogue of this one runs (it does not touch the K slots)
  if (ct0 < ct1) mfma_prefetch(p.wqt + (int64_t)ct0 * 256 * p.ldx, p.ldx, Bg, p.ldx, smem, rot_a, rot_b, wave);
  for (int ct = ct0; ct < ct1; ++ct) {
    mfma_mainloop<true, NoHook, BK, false, 0, BF16, true>(p.wqt + (int64_t)ct * 256 * p.ldx, p.ldx, Bg, p.ldx, KT, smem, acc, rot_a, rot_b, wave);
    auto prefetch = [&]() {
      const int next = ct + 1 < ct1 ? ct + 1 : s < 2 * cth ? s >> 1 : -1;
      if (next >= 0) mfma_prefetch(p.wqt + (int64_t)next * 256 * p.ldx, p.ldx, Bg, p.ldx, smem, rot_a, rot_b, wave);
    };
    const int* tgt = reinterpret_cast<const int*>(smem + FWD_TGT_OFF) + wb * 128;
    DeferredTail<BF16> deferred(smem, wa, wb);
    auto tail = [&](int b, int k) { deferred(acc, b, k); };
    if (EMIT) {
      // The main loop has left 48 of the 64 MFMAs of its last pair of K blocks undone, those of row blocks 1 - 3; the pair
      // is still in LDS.  They are issued one at a time between the stages of the epilogues of row blocks 0 and 1, where
      // the matrix pipe would stand idle: during block 0's the 32 of blocks 1 and 2 (one at each of its 32 stage
      // boundaries), during block 1's the 16 of block 3.  Only then are the slots free for the next tile's first K blocks.
      float* stat = reinterpret_cast<float*>(smem + FWD_STAT_OFF) + wave * 64 + lane_id();
      const int vbase = ct * 256 + wa * 128 + 4 * (lane_id() >> 5);
      const int vlim = p.V - ct * 256;
      // the wave's quadrant of G: tile of rows rt, block of columns 2 ct + wa, rows 128 wb on
      uint8_t* gq = p.ghat_t + ((int64_t)rt * p.kbv + 2 * ct + wa) * BLOCKED_KSTEP + wb * 128 * BK;
      const float* lam = reinterpret_cast<const float*>(smem + FWD_STAT_OFF) + 12 * NTHREADS + wave * 64;
      const int col0 = ct * 256 + wa * 128, row0 = rt * 256 + wb * 128;
      // (one code path for the epilogue: with a second one for the last tile of the vocabulary, each with its MFMAs, the
      // accumulators are spilled; columns that do not exist are struck out of the finished accumulators instead)
      const bool ragged = vlim < 256;
      uint32_t ew;
      if (PRE) {
        auto target = [&](int b) { return target_value(smem, p.n_predict, col0, wb * 128 + b * 32); };
        float xc[4];                                   // (looked up a row block ahead of their use: the LDS reads have time)
        if (ragged) strike_columns_beyond<0, 1>(acc, vlim, wa, stat, p.em2cap);
        xc[0] = target(0); xc[1] = target(1);
        ew = form_dlogits<true, NTHREADS, 64, 0, 1, decltype(tail)&, true>(acc, p.k1, p.c2, vbase, gq, wa, wb, stat, lam, p.want_argmax != 0, tail, xc, p.sc);
        if (ragged) strike_columns_beyond<1, 2>(acc, vlim, wa, stat, p.em2cap);
        xc[2] = target(2); xc[3] = target(3);
        ew |= form_dlogits<true, NTHREADS, 64, 1, 2, decltype(tail)&, true>(acc, p.k1, p.c2, vbase, gq, wa, wb, stat, lam, p.want_argmax != 0, tail, xc, p.sc);
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");      // every wave has read its last fragment
        prefetch();
        if (ragged) strike_columns_beyond<2, 4>(acc, vlim, wa, stat, p.em2cap);
        NoHook none;
        ew |= form_dlogits<true, NTHREADS, 64, 2, 4, NoHook&, true>(acc, p.k1, p.c2, vbase, gq, wa, wb, stat, lam, p.want_argmax != 0, none, xc, p.sc);
      } else {
        if (ragged) strike_columns_beyond<0, 1>(acc, vlim, wa, stat, p.em2cap);
        take_target_logits<true, true, true, 256, 0, 1>(acc, tgt, p.n_predict, col0, row0, p.sc, p.s_uy, p.Np, stat, p.k1, p.ic2, p.em2cap);
        ew = form_dlogits<true, NTHREADS, 64, 0, 1>(acc, p.k1, p.c2, vbase, gq, wa, wb, stat, lam, p.want_argmax != 0, tail);
        if (ragged) strike_columns_beyond<1, 2>(acc, vlim, wa, stat, p.em2cap);
        take_target_logits<true, true, true, 256, 1, 2>(acc, tgt, p.n_predict, col0, row0, p.sc, p.s_uy, p.Np, stat, p.k1, p.ic2, p.em2cap);
        ew |= form_dlogits<true, NTHREADS, 64, 1, 2>(acc, p.k1, p.c2, vbase, gq, wa, wb, stat, lam, p.want_argmax != 0, tail);
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");      // every wave has read its last fragment
        prefetch();
        if (ragged) strike_columns_beyond<2, 4>(acc, vlim, wa, stat, p.em2cap);
        take_target_logits<true, true, true, 256, 2, 4>(acc, tgt, p.n_predict, col0, row0, p.sc, p.s_uy, p.Np, stat, p.k1, p.ic2, p.em2cap);
        ew |= form_dlogits<true, NTHREADS, 64, 2, 4>(acc, p.k1, p.c2, vbase, gq, wa, wb, stat, lam, p.want_argmax != 0);
      }
      if (lane_id() == 0) p.gexp[(int64_t)(2 * ct + wa) * p.kbw + 2 * rt + wb] = ew;
    } else {
      // The same, with the epilogue that forms no dlogits: 16384 rows, d = 1024, V = 50304 with bf16 operands, where the epilogue is a third of a tile's
      // time, a pass of 1567 us takes 1518; 8192 rows, d = 2560 in e4m3, which the card's power bounds, the same either way.  Of a tile that reaches beyond the
      // vocabulary the columns that do not exist are struck out here too, and the sums are then formed again without them: what they add, e^{-2 cap} apiece, cannot be taken off exactly
      const bool ragged = ct * 256 + 256 > p.V;
      const int col0 = ct * 256 + wa * 128;
      float* wave_stat = reinterpret_cast<float*>(smem + FWD_STAT_OFF) + wave * 64;
      if (ragged) {
        float* stat = wave_stat + lane_id();
#pragma unroll
        for (int b = 0; b < 4; ++b) stat[(12 + b) * NTHREADS] = stat[(0 + b) * NTHREADS];
        strike_columns_beyond<0, 1>(acc, p.V - ct * 256, wa);
      }
      fwd_epilogue<0, BF16>(acc, p, col0, wave_stat, tail);
      if (!PRE) take_target_logits<true, false, false, 256, 0, 1>(acc, tgt, p.n_predict, col0, rt * 256 + wb * 128, p.sc, p.s_uy, p.Np, nullptr, 0.f, 0.f, 0.f);
      if (ragged) strike_columns_beyond<1, 2>(acc, p.V - ct * 256, wa);
      fwd_epilogue<1, BF16>(acc, p, col0, wave_stat, tail);
      if (!PRE) take_target_logits<true, false, false, 256, 1, 2>(acc, tgt, p.n_predict, col0, rt * 256 + wb * 128, p.sc, p.s_uy, p.Np, nullptr, 0.f, 0.f, 0.f);
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");      // every wave has read its last fragment
      prefetch();
      if (ragged) strike_columns_beyond<2, 4>(acc, p.V - ct * 256, wa);
      fwd_epilogue<2, BF16>(acc, p, col0, wave_stat);
      if (!PRE) take_target_logits<true, false, false, 256, 2, 3>(acc, tgt, p.n_predict, col0, rt * 256 + wb * 128, p.sc, p.s_uy, p.Np, nullptr, 0.f, 0.f, 0.f);
      fwd_epilogue<3, BF16>(acc, p, col0, wave_stat);
      if (!PRE) take_target_logits<true, false, false, 256, 3, 4>(acc, tgt, p.n_predict, col0, rt * 256 + wb * 128, p.sc, p.s_uy, p.Np, nullptr, 0.f, 0.f, 0.f);
      if (ragged) sums_of_existing_columns(acc, p, col0, wave_stat);
    }
  }
  if constexpr (EMIT && PRE) {
    if (s < 2 * cth) {
      // half of tile s / 2: row blocks 2 hb and 2 hb + 1 of every wave, which are blocks 0 and 1 to everything here
      const int ct = s >> 1, hb = s & 1;
      mfma_mainloop<true, NoHook, BK, false, 0, false, false, 4, 2>(p.wqt + (int64_t)ct * 256 * p.ldx, p.ldx, Bg, p.ldx, KT, smem, acc, rot_a, rot_b, wave, NoHook(), 0, 0,
                                                                    nullptr, nullptr, 64 * hb);
      float* stat = reinterpret_cast<float*>(smem + FWD_STAT_OFF) + 2 * hb * NTHREADS + wave * 64 + lane_id();
      const float* lam = reinterpret_cast<const float*>(smem + FWD_STAT_OFF) + (12 + 2 * hb) * NTHREADS + wave * 64;
      const int col0 = ct * 256 + wa * 128, vbase = col0 + 4 * (lane_id() >> 5), r0 = wb * 128 + hb * 64;
      uint8_t* gq = p.ghat_t + ((int64_t)rt * p.kbv + 2 * ct + wa) * BLOCKED_KSTEP + r0 * BK;
      float xc[2];
#pragma unroll
      for (int b = 0; b < 2; ++b) xc[b] = target_value(smem, p.n_predict, col0, r0 + b * 32);
      NoHook none;
      const uint32_t ew = form_dlogits<true, NTHREADS, 64, 0, 2, NoHook&, true>(acc, p.k1, p.c2, vbase, gq, wa, wb, stat, lam, p.want_argmax != 0, none, xc, p.sc);
      if (lane_id() == 0) reinterpret_cast<uint16_t*>(p.gexp + (int64_t)(2 * ct + wa) * p.kbw + 2 * rt + wb)[hb] = (uint16_t)ew;
    }
  }
  float sum[4], amax[4];
  int uarg[4];
  const int lane = lane_id();
  float* stat = reinterpret_cast<float*>(smem + FWD_STAT_OFF) + wave * 64 + lane;
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    sum[b] = stat[(0 + b) * NTHREADS]; amax[b] = stat[(4 + b) * NTHREADS]; uarg[b] = __float_as_int(stat[(8 + b) * NTHREADS]);
  }
  // the two half-waves hold different columns of the same rows
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    const float s2 = __shfl_xor(sum[b], 32), um2 = __shfl_xor(amax[b], 32);
    const int ua2 = __shfl_xor(uarg[b], 32);
    sum[b] += s2;
    if (um2 > amax[b] || (um2 == amax[b] && ua2 < uarg[b])) { amax[b] = um2; uarg[b] = ua2; }
  }
  // waves wa = 0 and wa = 1 hold different columns of the same rows
  float4* red = reinterpret_cast<float4*>(smem);
  if (wa == 1 && lane < 32) {
#pragma unroll
    for (int b = 0; b < 4; ++b) red[wb * 128 + b * 32 + lane] = make_float4(sum[b], amax[b], __int_as_float(uarg[b]), 0.f);
  }
  __syncthreads();
  if (wa == 0 && lane < 32) {
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const float4 o = red[wb * 128 + b * 32 + lane];
      const int ua2 = __float_as_int(o.z);
      sum[b] += o.x;
      if (o.y > amax[b] || (o.y == amax[b] && ua2 < uarg[b])) { amax[b] = o.y; uarg[b] = ua2; }
      p.partials[(int64_t)s * p.Np + rt * 256 + wb * 128 + b * 32 + lane] =
          make_float4(sum[b], amax[b] * p.sc, __int_as_float(uarg[b]), 0.f);
    }
  }
}

// The bf16 forward pass of few rows (scoring one short text): W (d, V) read as it lies, once, without the transposed copy.
// What bounds it is that read (2 bytes an element); the copy costs as many bytes again in each direction and a second
// read.  One workgroup to 256 columns (the split of fwd_splits), each of its eight waves to 32 of them and all 32 NB rows.
// The whole LDS is a ring of FEW_K-deep slices of W and x, filled by direct loads up to STAGES - 1 slices ahead, with one barrier a slice.  K runs along the rows of W, so the A fragments come through the transposing read: ds_read_b64_tr_b16 gives lane i
// of 16 column i of the 4 x 16 matrix that the 16 lanes point at, four K values, and two reads the eight of an instruction.
// d is a multiple of 16, the K of one instruction: the last slice may be half a one, and nothing is padded.
// In a slice the pair of 16-byte chunks c / 2 of W's row k lies at position (c / 2) ^ (k & 3), chunk c of a row of x at
// c ^ (row / 2 & 3): the rows that one read touches would otherwise lie in the same banks.
// 61 rows, d = 2560, V = 50304: copy 88 us and general kernel 86, now 44.7 with the weight just
// read before (5.8 TB/s: part of its 257 MB is still in the 256 MB memory-side cache) and 92 right
// after a 1 GiB fill (whose lines are then still on their way out; the copy 225 and the general kernel 811 there, with 16
// splits).  The whole pass, copy and general kernel
// against this: 200 us against 51 (64 rows), 66 (128) and 101 (256); d = 4096, V = 4096, where 16 workgroups do it all:
// 95 against 64 and 81, but 97 against 125 for 256 rows (a CU's LDS reads are the bound then): beyond 128 rows only with
// FEW_TILES column tiles, half as many as there are CUs; d = 512, V = 8192: 36 against 18 and 23.
// With so few column tiles that their workgroups' K loops are all there is, 128 rows go the general way from FEW_DEEP on, where its loop
// is the shorter one and the copy small beside it (128 rows, cold weight: d = 32768, V = 256 510 us against 570, V = 1024 563 and
// 575, V = 2048 750 and 572; d = 8192 160 and 158); 64 rows never (507 and 459 there).
constexpr int FEW_K = 32;
constexpr int FEW_MAX_ROWS = 256, FEW_TILES = 128, FEW_THREADS = 512, FEW_DEEP = 8192, FEW_DEEP_TILES = 8;
template <int NB>
struct FewRows {
  static constexpr int W_BYTES = FEW_K * 512, STAGE = W_BYTES + NB * 2048, STAGES = NB == 2 ? 7 : NB == 4 ? 6 : 4;
  static constexpr int XL = NB == 8 ? 2 : 1, LOADS = 2 + XL;      // direct loads of a wave per slice (NB = 2: the second four waves load x again)
  static constexpr int TGT_OFF = STAGES * STAGE, SMEM = TGT_OFF + 4 * 32 * NB * 4;
  static_assert(SMEM <= SMEM_MAX && (STAGES - 2) * LOADS < 64, "LDS, and what s_waitcnt can count");
};
struct FewParams {
  const uint8_t* x;        // bf16, row stride x_ldb bytes
  const uint8_t* w;        // bf16 (d, Vw), row stride w_ldb bytes; 16-byte aligned rows, Vw a multiple of 8
  int64_t x_ldb, w_ldb;
  int d, Vw;
};

template <int NB>
__global__ __launch_bounds__(FEW_THREADS) void fwd_few_rows_kernel(FwdParams p, FewParams f) {
  using F = FewRows<NB>;
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = lane_id(), h = lane >> 5;
  const int ct0 = (int)((int64_t)p.CT * blockIdx.x / p.S), ct1 = (int)((int64_t)p.CT * (blockIdx.x + 1) / p.S);
  if (blockIdx.x == 0 && threadIdx.x == 0) *done_count(p) = 0;
  int* tgt = reinterpret_cast<int*>(smem + F::TGT_OFF);           // [4 offsets][32 NB]
  for (int e = threadIdx.x; e < p.n_predict * 32 * NB; e += FEW_THREADS) {
    const int row = e % (32 * NB), i = row + e / (32 * NB);
    tgt[e] = (row < p.N && target_valid(p.targets, p.ignore_index, i, p.N, p.V)) ? (int)p.targets[i] : -1;
  }
  __syncthreads();
  const uint32_t lds0 = (uint32_t)(uintptr_t)((__attribute__((address_space(3))) void*)smem);
  // W: load n of a wave is rows 4 wave + 2 n and + 1 of the slice, 32 chunks each; x: load q is 16 rows of 4 chunks
  auto xload = [&](int n) { return NB == 2 ? wave & 3 : wave * F::XL + n; };
  uint32_t xo[F::XL];
  const int xc = (lane & 3) ^ ((lane >> 3) & 3);
#pragma unroll
  for (int n = 0; n < F::XL; ++n) xo[n] = (uint32_t)(min(xload(n) * 16 + (lane >> 2), p.N - 1) * f.x_ldb + xc * 16);
  const uint32_t xhalf = (xc & 2) ? 32u : 0u;                     // the last slice's second half does not exist: its first half again
  uint32_t wo[2];
  auto columns = [&](int ct) {                                    // (the last tile may reach beyond W: its last chunk again)
#pragma unroll
    for (int n = 0; n < 2; ++n) {
      const int pc = lane & 31, c = (((pc >> 1) ^ ((2 * n + h) & 3)) << 1) | (pc & 1);
      wo[n] = (uint32_t)((wave * 4 + 2 * n + h) * f.w_ldb + 2 * min(ct * 256 + c * 8, f.Vw - 8));
    }
  };
  const int nk = (f.d + FEW_K - 1) / FEW_K, total = (ct1 - ct0) * nk;
  const bool half_slice = f.d % FEW_K != 0;
  int ict = ct0, ik = 0, islot = 0;                               // the slice that is loaded next
  auto issue = [&]() {
    if (ik == 0) columns(ict);
    const bool tail = half_slice && ik == nk - 1;
    const uint8_t* wb = f.w + (int64_t)(ik * FEW_K - (tail && wave >= 4 ? 16 : 0)) * f.w_ldb;
    const uint8_t* xb = f.x + (int64_t)ik * (2 * FEW_K);
    const uint32_t l = lds0 + islot * F::STAGE;
    lds_direct_16<0>(l + wave * 2048, wo[0], wb);
    lds_direct_16<1024>(l + wave * 2048, wo[1], wb);
#pragma unroll
    for (int n = 0; n < F::XL; ++n) lds_direct_16<F::W_BYTES>(l + xload(n) * 1024, xo[n] - (tail ? xhalf : 0u), xb);
    if (++ik == nk) { ik = 0; ++ict; }
    if (++islot == F::STAGES) islot = 0;
  };
#pragma unroll 1
  for (int g = 0; g < F::STAGES - 1 && g < total; ++g) issue();
  float sum[NB], amax[NB];
  int uarg[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b) { sum[b] = 0.f; amax[b] = -INFINITY; uarg[b] = 0x7fffffff; }
  v16f acc[NB];
  typedef short v4s __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) v4s lds_v4s;
  const int i16 = lane & 15, g4 = lane >> 4;                      // group g4 of 16 lanes: columns 16 (g4 & 1) on, K values 8 (g4 / 2) on
  int slot = 0, done = 0;
#pragma unroll 1
  for (int ct = ct0; ct < ct1; ++ct) {
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[b][r] = 0.f;
#pragma unroll 1
    for (int k = 0; k < nk; ++k, ++done) {
      // this wave's loads of the slice have landed and its reads of the one before are complete; after the barrier that holds
      // for every wave, and the slot of the slice before is free
      if (done + F::STAGES - 1 <= total) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((F::STAGES - 2) * F::LOADS) : "memory");
      else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
      if (done + F::STAGES - 1 < total) issue();
      const uint8_t* ws = smem + slot * F::STAGE;
      const uint8_t* xs = ws + F::W_BYTES;
#pragma unroll
      for (int s = 0; s < 2; ++s) {                               // 16 K values
        v8bf fa, fb[NB];
        if (s == 1 && half_slice && k == nk - 1) {                // not there: products of zeros (a branch around the MFMAs would have the accumulators moved in every slice)
          fa = __builtin_bit_cast(v8bf, (v4i){0, 0, 0, 0});
#pragma unroll
          for (int b = 0; b < NB; ++b) fb[b] = fa;
        } else {
          const int kr = 16 * s + 8 * (g4 >> 1) + (i16 >> 2), pair = wave * 2 + (g4 & 1);      // (32 bytes of columns)
          const uint8_t* src = ws + kr * 512 + ((pair ^ (kr & 3)) << 5) + 8 * (i16 & 3);
          const v2i lo = __builtin_bit_cast(v2i, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s*)src));
          const v2i hi = __builtin_bit_cast(v2i, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s*)(src + 4 * 512)));
          fa = __builtin_bit_cast(v8bf, (v4i){lo[0], lo[1], hi[0], hi[1]});
#pragma unroll
          for (int b = 0; b < NB; ++b) {
            const int r = b * 32 + (lane & 31);
            fb[b] = __builtin_bit_cast(v8bf, *reinterpret_cast<const v4i*>(xs + r * 64 + (((2 * s + h) ^ ((r >> 1) & 3)) << 4)));
          }
        }
#pragma unroll
        for (int b = 0; b < NB; ++b) acc[b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa, fb[b], acc[b], 0, 0, 0);
      }
      if (++slot == F::STAGES) slot = 0;
    }
    // the lane's 16 columns of a row: v0 + 8 (r / 4) + r % 4; logits rounded to bf16 as the eager head's GEMM returns them
    const int v0 = ct * 256 + wave * 32 + 4 * h;
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      __builtin_amdgcn_sched_barrier(0);                          // one row block at a time
      const int row = b * 32 + (lane & 31);
      float s = 0.f;
      int arg = -1;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int v = 8 * (r >> 2) + (r & 3);
        float x = round_to_bf16_hw(acc[b][r]), pt = fast_exp2(fast_rcp(fmaf(fast_exp2(x * p.k1), p.ic2, p.ic2)));
        if (v >= p.V - v0) { pt = 0.f; x = -INFINITY; }
        s += pt;
        if (x > amax[b]) { amax[b] = x; arg = v; }                // ascending columns: the lowest wins
      }
      if (arg >= 0) uarg[b] = v0 + arg;
      sum[b] += s;
      for (int k = 0; k < p.n_predict; ++k) {
        const int rel = tgt[k * 32 * NB + row] - v0;
        if ((unsigned)rel < 32u && (rel & 4) == 0) {
          float x = 0.f;
#pragma unroll
          for (int r = 0; r < 16; ++r) x = rel == 8 * (r >> 2) + (r & 3) ? acc[b][r] : x;
          p.s_uy[(int64_t)k * p.Np + row] = round_to_bf16_hw(x) * p.sc;
        }
      }
    }
  }
  // fold the two half-waves and the eight waves: all hold different columns of the same rows
  __syncthreads();
  float4* red = reinterpret_cast<float4*>(smem);                  // [8 waves][32 NB]
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    const float s2 = __shfl_xor(sum[b], 32), um2 = __shfl_xor(amax[b], 32);
    const int ua2 = __shfl_xor(uarg[b], 32);
    sum[b] += s2;
    if (um2 > amax[b] || (um2 == amax[b] && ua2 < uarg[b])) { amax[b] = um2; uarg[b] = ua2; }
    if (h == 0) red[wave * 32 * NB + b * 32 + lane] = make_float4(sum[b], amax[b], __int_as_float(uarg[b]), 0.f);
  }
  __syncthreads();
  if (threadIdx.x < 32 * NB) {
    float4 o = red[threadIdx.x];
    for (int w = 1; w < 8; ++w) {
      const float4 q = red[w * 32 * NB + threadIdx.x];
      o.x += q.x;
      if (q.y > o.y || (q.y == o.y && __float_as_int(q.z) < __float_as_int(o.z))) { o.y = q.y; o.z = q.z; }
    }
    p.partials[(int64_t)blockIdx.x * p.Np + threadIdx.x] = make_float4(o.x, o.y * p.sc, o.z, 0.f);
  }
}

// What a block of COMBINE_ROWS rows contributes to the mean loss: left by fwd_combine_kernel in the first 16 bytes of the
// block's own rows of the partial records (which it has consumed by then), summed by its last block or by fwd_reduce_kernel:
//   8 bytes: sum of lse_i - z[i, y_i] over the valid rows (a double); 4: valid rows; 4: targets outside [0, V) other than ignore_index
constexpr int COMBINE_ROWS = 64, MERGE_BLOCKS = 256;

// n_valid, targets out of range and the mean from what the blocks left (of a single block: sum, cnt and bad as they are), in a fixed
// order; a workgroup of COMBINE_ROWS * G threads.
template <int G>
__device__ __forceinline__ void finish_mean(const float4* partials, int nblk, double sum, int cnt, int bad, uint8_t* __restrict__ hdr,
                                            float* __restrict__ loss_out, int32_t* __restrict__ nvalid_out, const CallMode& mode) {
  if (nblk > 1) {
    __shared__ double wsum[G];
    __shared__ int wcnt[G], wbad[G];
    const int r = threadIdx.x & 63, g = threadIdx.x >> 6;
    sum = 0.0; cnt = 0; bad = 0;
    for (int b = threadIdx.x; b < nblk; b += COMBINE_ROWS * G) {
      const uint64_t* slot = reinterpret_cast<const uint64_t*>(partials + (int64_t)b * COMBINE_ROWS);
      sum += __longlong_as_double((long long)__hip_atomic_load(slot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
      const uint64_t c = __hip_atomic_load(slot + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      cnt += (int)(uint32_t)c; bad += (int)(uint32_t)(c >> 32);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) { sum += __shfl_xor(sum, o); cnt += __shfl_xor(cnt, o); bad += __shfl_xor(bad, o); }
    if (r == 0) { wsum[g] = sum; wcnt[g] = cnt; wbad[g] = bad; }
    __syncthreads();
    if (threadIdx.x == 0)
      for (int w = 1; w < G; ++w) { sum += wsum[w]; cnt += wcnt[w]; bad += wbad[w]; }
  }
  if (threadIdx.x != 0) return;
  const float mean = (float)(sum / (double)cnt);                 // 0/0 = NaN, as F.cross_entropy gives
  int32_t* head = reinterpret_cast<int32_t*>(hdr);
  head[0] = cnt; head[1] = bad;
  reinterpret_cast<float*>(hdr)[2] = mean;
  *reinterpret_cast<CallMode*>(hdr + HDR_MODE_OFF) = mode;
  if (loss_out) *loss_out = mean;
  if (nvalid_out) { nvalid_out[0] = cnt; nvalid_out[1] = bad; }
}
__global__ __launch_bounds__(COMBINE_ROWS * 16) void fwd_reduce_kernel(const float4* __restrict__ partials, int nblk, uint8_t* __restrict__ hdr,
                                                                      float* __restrict__ loss_out, int32_t* __restrict__ nvalid_out, CallMode mode) {
  finish_mean<16>(partials, nblk, 0.0, 0, 0, hdr, loss_out, nvalid_out, mode);
}

// p(target) = exp(-loss), 0 for the rows without a target (fwd_combine_kernel forms it for sce_forward_probability).
__device__ __forceinline__ float row_probability(float loss, int64_t target, int64_t ignore_index) { return target == ignore_index ? 0.f : expf(-loss); }

// The same of losses from any call.  Bound by its launch: in place of five elementwise operations of
// torch's (compare, zeros, negate, exp, where) a call that scores 61 rows at d = 2560, V = 50304 takes 65.6 us for 73.6.
__global__ __launch_bounds__(256) void target_probability_kernel(const float* __restrict__ losses, const int64_t* __restrict__ targets, int64_t n,
                                                                int64_t ignore_index, float* __restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) out[i] = row_probability(losses[i], targets[i], ignore_index);
}

// Folds the V-splits of a row and writes lse / loss / argmax and the saved row statistics: COMBINE_ROWS rows to a
// workgroup, one wave to every G-th split (its 64 rows' records are 1 KB in a row), four records in flight per lane.
// What bounds it is the chain of loads, not their volume: with one thread per row the records of a call of 61 rows and
// 197 splits were 197 loads of one workgroup.  Rows beyond N have no records (fwd_few_rows_kernel writes none).  G = 4 for up to 16 splits, 16 beyond (rows too few to fill the chip
// without cutting the vocabulary finer); the order of the sums depends on G alone.
// Up to MERGE_BLOCKS blocks the one that is done last adds up what all of them left (finish_mean).  The blocks' sums and the count go past the
// L2 caches (agent scope: every XCD has its own), the sum before the count.  One counter takes its arrivals one at a time, some 15 ns each, and a
// block waits for its own stores before it arrives, so of more blocks the sum is a launch of one workgroup, fwd_reduce_kernel, which takes 4.7 us
// whatever their number.  From the end of the forward kernel to the end of the mean, emitting, d = 256, V = 16384, merged and with the launch:
// 64 blocks (4096 rows) 5.7 and 9.7 us, 192 7.9 and 9.8, 256 8.9 and 10.1, 320 10.6 and 10.9, 384 11.1 and 10.6, 512 12.9 and 11.2, 1024 21.7 and
// 14.0; without dlogits 256 7.9 and 9.4, 384 9.6 and 9.3, 1024 18.5 and 9.7.
// The probabilities of a caller that scores rows ride along (a launch of their own: 4 us).  A call of 64 rows at most that no
// backward call follows is one block, which has nobody to wait for.
template <int G>
__global__ __launch_bounds__(COMBINE_ROWS * G) void fwd_combine_kernel(float4* __restrict__ partials, int S, int N, int Np, int V,
                                                         const int64_t* __restrict__ targets, int64_t ignore_index, float cap,
                                                         const float* __restrict__ mtp_weights, int n_predict,
                                                         float* __restrict__ s_lse, float* __restrict__ s_zy, float* __restrict__ losses,
                                                         float* __restrict__ lse_out, int32_t* __restrict__ argmax_out,
                                                         uint8_t* __restrict__ ghat, int64_t kbv, float* __restrict__ probability, uint8_t* __restrict__ hdr,
                                                         float* __restrict__ loss_out, int32_t* __restrict__ nvalid_out, CallMode mode) {
  static_assert(G >= 4, "one wave per prediction offset");
  __shared__ float rsum[G][COMBINE_ROWS], rmax[G][COMBINE_ROWS], rl[4][COMBINE_ROWS];
  __shared__ int rarg[G][COMBINE_ROWS];
  __shared__ bool last;
  const int r = threadIdx.x & 63, g = threadIdx.x >> 6, i = blockIdx.x * COMBINE_ROWS + r;      // the grid covers Np rows exactly, or N alone if no backward call can follow
  {
    float sum = 0.f, umax = -INFINITY;
    int uarg = 0x7fffffff;
    for (int s0 = g; s0 < S; s0 += 4 * G) {
      float4 o[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int s = s0 + q * G;
        o[q] = s < S && i < N ? partials[(int64_t)s * Np + i] : make_float4(0.f, -INFINITY, __int_as_float(0x7fffffff), 0.f);
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int ua = __float_as_int(o[q].z);
        sum += o[q].x;
        if (o[q].y > umax || (o[q].y == umax && ua < uarg)) { umax = o[q].y; uarg = ua; }
      }
    }
    rsum[g][r] = sum; rmax[g][r] = umax; rarg[g][r] = uarg;
  }
  __syncthreads();               // also: every wave of this block has read its partial records
  float lse = 0.f;
  double sum = 0.0;                                              // of this block and in the end of all, in thread 0
  int cnt = 0, bad = 0;
  if (g < n_predict && i < N) {
    float sum = 0.f;
#pragma unroll
    for (int q = 0; q < G; ++q) sum += rsum[q][r];
    lse = cap + logf(sum);
  }
  // one wave per offset: the raw logit at each target that takes part is there; z_y = cap tanh(u_y / cap) replaces it (0 for the
  // others); loss_i = sum_k w_k (lse_i - z[i, y_{i+k}]) over the offsets that take part (tiny/cuda_kernels.py:226-240)
  if (g < n_predict) {
    float zy = 0.f, l = 0.f;
    if (i < N && target_valid(targets, ignore_index, i + g, N, V)) {
      if (ghat) knock_target(ghat, kbv, i, targets[i + g]);
      zy = cap * tanhf(s_zy[(int64_t)g * Np + i] / cap);
      l = (mtp_weights ? mtp_weights[g] : 1.0f) * (lse - zy);
    }
    s_zy[(int64_t)g * Np + i] = zy;
    rl[g][r] = l;
    if (g == 0) {
      s_lse[i] = lse;
      if (i < N) {
        if (lse_out) lse_out[i] = lse;
        if (argmax_out) {
          float umax = -INFINITY;
          int uarg = 0x7fffffff;
          for (int q = 0; q < G; ++q)
            if (rmax[q][r] > umax || (rmax[q][r] == umax && rarg[q][r] < uarg)) { umax = rmax[q][r]; uarg = rarg[q][r]; }
          argmax_out[i] = (uarg == 0x7fffffff) ? 0 : uarg;
        }
        const int64_t y = targets[i];
        if (y != ignore_index) {
          if (y < 0 || y >= V) bad = 1;
          else { sum = (double)(lse - zy); cnt = 1; }
        }
      }
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) { sum += __shfl_xor(sum, o); cnt += __shfl_xor(cnt, o); bad += __shfl_xor(bad, o); }
      if (r == 0) {
        last = gridDim.x == 1;
        if (!last) {
          uint64_t* slot = reinterpret_cast<uint64_t*>(partials + (int64_t)blockIdx.x * COMBINE_ROWS);
          const uint64_t counts = (uint64_t)(uint32_t)cnt | ((uint64_t)(uint32_t)bad << 32);
          __hip_atomic_store(slot, (uint64_t)__double_as_longlong(sum), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          __hip_atomic_store(slot + 1, counts, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          if (gridDim.x <= MERGE_BLOCKS) {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");     // both have arrived
            last = __hip_atomic_fetch_add(reinterpret_cast<uint32_t*>(hdr + HDR_COUNT_OFF), 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == gridDim.x - 1;
          }
        }
      }
    }
  }
  __syncthreads();
  if (losses && g == 0 && i < N) {
    float l = rl[0][r];
    for (int k = 1; k < n_predict; ++k) l += rl[k][r];
    losses[i] = l;
    if (probability) probability[i] = row_probability(l, targets[i], ignore_index);
  }
  if (last) finish_mean<G>(partials, gridDim.x, sum, cnt, bad, hdr, loss_out, nvalid_out, mode);
}

}  // namespace sce
