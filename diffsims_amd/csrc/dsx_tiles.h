// Sub-pixel patterns of long spot lists (more than the LDS spot table of the
// small kernels holds) and their adjoint, on the matrix cores.
//
// A spot's Gaussian is separable and its clip box is a product of a row range
// and a column range, so the pixels of a 16x16 tile are a matrix product over
// the tile's spots k,
//   P[y][x] = sum_k (amp_k gy_k(y)) gx_k(x),
// with gy, gx zero outside the box, and the gathered sums of its spots are two
// more (G = dL/dP):
//   T1[x][k] = sum_y G[y][x] gy_k(y),  T2[x][k] = sum_y G[y][x] dy gy_k(y),
//   A_k = sum_x T1 gx,  BX_k = sum_x T1 gx dx,  BY_k = sum_x T2 gx.
// v_mfma_f32_16x16x4_f32 takes one factor value per lane and operand: two
// exponentials per four spots and lane instead of one per pixel of every box,
// and no pixel atomics.  The tile's G stays in the registers the product left
// it in: contracting over y in the order 4 (lane / 16) + r makes register r of
// the result an operand of the next product.
//
// One 512-thread block per pattern, persistent over patterns:
//   count    every listed spot's pixel, clip box and tiles; entries per tile
//   scatter  one 16-byte record per (spot, tile) {x, y in the tile, amplitude,
//            row and column bits of the box} in tile order, into the block's
//            workspace; a pattern with more entries than that holds is taken
//            in ranges of tiles
//   maximum  (normalize) a tile whose bound (the sum of its spots' largest
//            values there) is below the largest value known is skipped; the
//            others are evaluated with the very products of the last step, so
//            the maximum is the written one
//   tiles    each wave takes tiles: product, then the scaled pixels, or the
//            loss, G and the gathered sums
// The strip kernel before it (bins by row strip, one exponential and one LDS
// atomic per pixel and box, pixels kept in HBM between the maximum and the
// read-out) took 19.6 ms for 4,096 patterns of 512 x 512 with 28,700 boxes
// (43,000 listed spots) and their gradients, 11.7 ms here; forward only 9.95
// and 6.4 ms then (6.54 since): count 1.1, scatter 1.8, maximum 0.2 (a few tiles in ten can
// hold it), tiles 3.2 ms, the gather 3.6 ms more.  Bound by VALU issue (78 % of
// the SIMDs' cycles forward, 74 % with the gather, which keeps 12 registers in
// scratch at 128): the factors of all 16 rows and columns of a tile are formed
// for boxes of 5.4; the scatter by its 16-byte writes.  Small frames of few spots
// in thin tiles (20 x 900, 480 spots) take up to 1.2 times as long as the strip
// kernel did.  Measured and not kept: four spots' loads in flight per lane in
// count and scatter (7.7 ms forward, registers), 1,024-thread blocks (7.2), the
// next tile's records loaded ahead (6.7 and 12.5), the gather's factors by
// recurrence along a lane's four rows (no faster).
#pragma once

#include "dsx_splat.h"

namespace dsx {

constexpr int kTileThreads = 512;
constexpr int kTileWaves = kTileThreads / kWave;
constexpr int kTileEdge = 16;
constexpr int kTilePixBits = 22;  // argmax key: value << 22 | (2^22 - 1 - pixel)
constexpr int kRecInts = 5;       // workspace ints per entry: the record and its spot's row

typedef float tile_f4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ void tile_wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
}

struct TileShared {
  float4 stage[kTileWaves][kWave];  // records of the wave's current 64 entries
  int row[kTileWaves][kWave];       // their rows of the gradient hand-over
  int ns, total, t1;
  float wf[kTileWaves], wv[kTileWaves];
  int wsum[kTileWaves];
  unsigned long long best;          // key of the largest pixel found
  double red[kTileWaves][2];
};

// One factor of a spot's Gaussian at offset d from its centre, zero where bit
// `bit` of the box mask is clear (c = log2(e) * -1 / (2 sigma^2)).
__device__ __forceinline__ float tile_factor(float d, float c, int mask, int bit) {
  const float e = __builtin_amdgcn_exp2f(d * d * c);
  const int keep = __builtin_amdgcn_sbfe(mask, bit, 1);  // 0 or -1
  return __int_as_float(__float_as_int(e) & keep);
}

// Stage entries [e, e + 64) of the tile (those below e_end) in the wave's LDS.
__device__ __forceinline__ void tile_stage(TileShared &sh, const float4 *rec, const int *erow, int e,
                                           int e_end, int lane, int wid) {
  float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  if (e + lane < e_end) {
    v = rec[e + lane];
    if (erow) sh.row[wid][lane] = erow[e + lane];
  }
  tile_wave_sync();  // the previous entries have been read
  sh.stage[wid][lane] = v;
  tile_wave_sync();
}

// Pixels of the tile: register r of lane l holds row 4 (l / 16) + r, column l % 16.
// Two FP32 accumulators take 64 entries (8 steps of four each), FP64 adds these
// sums.  One accumulator for all of a tile's entries left errors of 1.8e-7 of the
// maximum where hundreds of boxes overlap (512 x 512, sigma 6) and 1e-4 with 20,000
// boxes in one place; now 1.3e-7, as 32-bit fixed point has.  Fused step 11.73 ->
// 11.81 ms, forward 6.43 -> 6.54 ms; adding FP64 sums after 32 entries of one
// accumulator gives the same errors in 12.3 and 6.7 ms.
__device__ __forceinline__ tile_f4 tile_pixels(TileShared &sh, const float4 *rec, const int *erow,
                                               int e0, int e1, float c, int lane, int wid) {
  tile_f4 acc = {0.0f, 0.0f, 0.0f, 0.0f}, odd = acc;
  double sum[4] = {0.0, 0.0, 0.0, 0.0};
  const int pos = lane & 15, sub = lane >> 4;
  const float fp = static_cast<float>(pos);
  for (int e = e0; e < e1; e += kWave) {
    tile_stage(sh, rec, erow, e, e1, lane, wid);
    const int m = min(kWave, e1 - e);
    int k = 0;
#pragma unroll 2
    for (; k + 4 < m; k += 8) {  // records past m have zero amplitude and mask
      const float4 v = sh.stage[wid][k + sub], w = sh.stage[wid][k + 4 + sub];
      const int mv = __float_as_int(v.w), mw = __float_as_int(w.w);
      const float av = v.z * tile_factor(fp - v.y, c, mv, pos);
      const float bv = tile_factor(fp - v.x, c, mv, 16 + pos);
      const float aw = w.z * tile_factor(fp - w.y, c, mw, pos);
      const float bw = tile_factor(fp - w.x, c, mw, 16 + pos);
      acc = __builtin_amdgcn_mfma_f32_16x16x4f32(av, bv, acc, 0, 0, 0);
      odd = __builtin_amdgcn_mfma_f32_16x16x4f32(aw, bw, odd, 0, 0, 0);
    }
    if (k < m) {
      const float4 v = sh.stage[wid][k + sub];
      const int mv = __float_as_int(v.w);
      const float av = v.z * tile_factor(fp - v.y, c, mv, pos);
      acc = __builtin_amdgcn_mfma_f32_16x16x4f32(av, tile_factor(fp - v.x, c, mv, 16 + pos), acc, 0, 0, 0);
    }
    if (e1 - e0 > kWave) {  // uniform
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        sum[r] += static_cast<double>(acc[r] + odd[r]);
        acc[r] = e + kWave < e1 ? 0.0f : static_cast<float>(sum[r]);
        odd[r] = 0.0f;
      }
    }
  }
  acc += odd;
  return acc;
}

// Gathered sums of the staged entries (m of them) against the tile's G, added
// into their rows of the hand-over (one spot has one entry per tile, so float
// atomics meet only over the tiles a box spans).
__device__ __forceinline__ void tile_gather(TileShared &sh, const tile_f4 &G, float4 *gsum, int m,
                                            float c, float pref, int lane, int wid) {
  const int pos = lane & 15, sub = lane >> 4;
  for (int k = 0; k < m; k += 16) {
    const float4 v = sh.stage[wid][k + pos];  // this lane's spot (rows past m: mask 0)
    const int mask = __float_as_int(v.w);
    tile_f4 t1 = {0.0f, 0.0f, 0.0f, 0.0f}, t2 = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int y = 4 * sub + r;
      const float dy = static_cast<float>(y) - v.y;
      const float gy = tile_factor(dy, c, mask, y);
      t1 = __builtin_amdgcn_mfma_f32_16x16x4f32(G[r], gy, t1, 0, 0, 0);
      t2 = __builtin_amdgcn_mfma_f32_16x16x4f32(G[r], gy * dy, t2, 0, 0, 0);
    }
    float A = 0.0f, BX = 0.0f, BY = 0.0f;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int x = 4 * sub + r;
      const float dx = static_cast<float>(x) - v.x;
      const float gx = tile_factor(dx, c, mask, 16 + x);
      const float tg = t1[r] * gx;
      A += tg;
      BX = fmaf(tg, dx, BX);
      BY = fmaf(t2[r], gx, BY);
    }
#pragma unroll
    for (int off = 16; off <= 32; off <<= 1) {
      A += __shfl_xor(A, off, kWave);
      BX += __shfl_xor(BX, off, kWave);
      BY += __shfl_xor(BY, off, kWave);
    }
    if (sub < 3 && k + pos < m) {  // lanes 0..15 add A, 16..31 BX, 32..47 BY
      float *h = reinterpret_cast<float *>(gsum + sh.row[wid][k + pos]);
      unsafeAtomicAdd(h + sub, pref * (sub == 0 ? A : (sub == 1 ? BX : BY)));
    }
  }
}

// Bits lo..hi (clipped to 0..15) of a tile's rows or columns.
__device__ __forceinline__ int tile_bits(int lo, int hi) {
  lo = max(lo, 0);
  hi = min(hi, 15);
  return ((2 << hi) - 1) & ~((1 << lo) - 1);
}

// kFwd: patterns only.  Otherwise the loss against the target (or the given
// dL/dP), optionally the patterns and the gathered sums.  Args: AdjArgs.
template <bool kFwd, class Args>
__device__ __forceinline__ void tiles_body(const Args &a, int *s_tiles, TileShared &sh) {
  const int tid = threadIdx.x, lane = lane_id(), wid = tid / kWave;
  const int H = a.H, W = a.W;
  const size_t HW = static_cast<size_t>(H) * W;
  const int ntx = (W + kTileEdge - 1) / kTileEdge;
  const int n_tiles = ntx * ((H + kTileEdge - 1) / kTileEdge);
  // The list is split over the first `cw` waves in consecutive parts, each
  // with counters of its own, so that a tile's entries are in list order whatever
  // the waves' timing, and patterns and losses the same bits in every run (the
  // lanes of one LDS atomic are served in order, as on every run so far).  The
  // gathered sums meet in float atomics and vary in their last bits.
  const int cw = a.count_waves, last = (cw - 1) * n_tiles;
  int *s_start = s_tiles;                // [cw][n_tiles]: first entry of (tile, part), tile-major
  int *s_u = s_tiles + cw * n_tiles;     // [n_tiles] bounds
  // the block's workspace: records | their spots' rows | first row per 64 listed spots
  int *work = a.work + static_cast<size_t>(blockIdx.x) * a.work_per_block;
  const int E = a.work_entries;
  float4 *rec = reinterpret_cast<float4 *>(work);
  int *erow = work + 4 * static_cast<size_t>(E);
  int *chunk_row = erow + E;
  const float c = a.ep * 1.4426950408889634f;
  const int pos = lane & 15, sub = lane >> 4;
  const bool grad = !kFwd && a.want_grad;

  // no room: the pattern is reported in status and left as zeros
  auto refuse = [&](int p) {
    if (a.pattern)
      for (size_t i = tid; i < HW; i += kTileThreads) a.pattern[static_cast<size_t>(p) * HW + i] = 0.0f;
    if (tid == 0) {
      if (a.loss) a.loss[p] = 0.0f;
      if (a.status) a.status[p] = 1;
      if (grad) a.gcount[p] = 0;
    }
  };

  for (int p = blockIdx.x; p < a.n; p += gridDim.x) {
    if (!a.work) {
      refuse(p);
      continue;
    }
    const int n = min(a.count[p], a.cap);
    const float4 *spots = a.spots + static_cast<size_t>(p) * a.cap;
    float4 *gsum = grad ? a.gsum + static_cast<size_t>(p) * a.cap : nullptr;
    for (int t = tid; t < (cw + 1) * n_tiles; t += kTileThreads) s_tiles[t] = 0;
    if (tid == 0) {
      sh.ns = 0;
      sh.best = 0;
    }
    lds_sync();

    // f(spot j in frame with a box: amplitude, pixel, box, chunk's first row) over the list
    auto each_spot = [&](auto &&f) {
      if (wid >= cw) return;
      const int part = ((n + kWave - 1) / kWave + cw - 1) / cw * kWave;  // whole chunks of 64
      const int end = min(n, (wid + 1) * part);
      float4 next = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      if (wid * part + lane < end) next = spots[wid * part + lane];
      for (int j0 = wid * part; j0 < end; j0 += kWave) {
        const int j = j0 + lane;
        const float4 sp = next;
        if (j + kWave < end) next = spots[j + kWave];
        float X = 0.0f, Y = 0.0f;
        int lo = 1, hi = 0, xlo = 0, xhi = 0;
        const bool in = j < end && to_pixel(sp, a, X, Y) &&
                        subpixel_box_fast(sp.w, X, Y, a, lo, hi, xlo, xhi);
        f(j0, j, in, sp.w * a.pref, X, Y, lo, hi, xlo, xhi);
      }
    };

    // ---- count -----------------------------------------------------------
    float pm = 0.0f, vlow = 0.0f;
    each_spot([&](int j0, int j, bool in, float amp, float X, float Y, int lo, int hi, int xlo, int xhi) {
      const uint64_t m = __ballot(in);
      if (grad) {
        int q = 0;
        if (lane == 0) {
          q = m ? atomicAdd(&sh.ns, __popcll(m)) : 0;
          chunk_row[j0 / kWave] = q;
        }
        q = __shfl(q, 0, kWave);
        if (in) gsum[q + mask_rank(m)] = make_float4(0.0f, 0.0f, 0.0f, __int_as_float(j));
      }
      if (!in) return;
      pm = fmaxf(pm, amp);
      // a pixel of the box near the centre holds at least this much
      const float dx = rintf(fminf(fmaxf(X, static_cast<float>(xlo)), static_cast<float>(xhi))) - X;
      const float dy = rintf(fminf(fmaxf(Y, static_cast<float>(lo)), static_cast<float>(hi))) - Y;
      vlow = fmaxf(vlow, amp * __builtin_amdgcn_exp2f(c * (dx * dx + dy * dy)));
      const int tx0 = xlo / kTileEdge, tx1 = xhi / kTileEdge, ty0 = lo / kTileEdge, ty1 = hi / kTileEdge;
      int *cnt = s_start + wid * n_tiles;
      if (tx1 - tx0 <= 1 && ty1 - ty0 <= 1) {  // at most 2 x 2 tiles: no loops
        int *at = cnt + ty0 * ntx + tx0;
        atomicAdd(at, 1);
        if (tx1 > tx0) atomicAdd(at + 1, 1);
        if (ty1 > ty0) {
          atomicAdd(at + ntx, 1);
          if (tx1 > tx0) atomicAdd(at + ntx + 1, 1);
        }
      } else {
        for (int ty = ty0; ty <= ty1; ++ty)
          for (int tx = tx0; tx <= tx1; ++tx) atomicAdd(cnt + ty * ntx + tx, 1);
      }
    });
    pm = wave_max(pm);
    vlow = wave_max(vlow);
    if (lane == 0) {
      sh.wf[wid] = pm;
      sh.wv[wid] = vlow;
    }
    lds_sync();
    float pmax = 0.0f;
    vlow = 0.0f;
    for (int w = 0; w < kTileWaves; ++w) {
      pmax = fmaxf(pmax, sh.wf[w]);
      vlow = fmaxf(vlow, sh.wv[w]);
    }
    vlow *= 0.9999f;
    // ---- starts: exclusive scan over the tiles -----------------------------
    const int per = (n_tiles + kTileThreads - 1) / kTileThreads;
    const int i0 = min(n_tiles, tid * per), i1 = min(n_tiles, i0 + per);
    // entries are numbered in 32 bits: lists with more of them (131,100 boxes
    // over all of a 256 x 16,384 pattern's tiles) are not taken
    if (static_cast<long long>(n) * n_tiles > 0x7fffffffll) {
      double all = 0.0;
      for (int t = i0; t < i1; ++t)
        for (int w = 0; w < cw; ++w) all += s_start[w * n_tiles + t];
#pragma unroll
      for (int off = 32; off >= 1; off >>= 1) all += __shfl_xor(all, off, kWave);
      if (lane == 0) sh.red[wid][0] = all;
      lds_sync();
      all = 0.0;
      for (int w = 0; w < kTileWaves; ++w) all += sh.red[w][0];
      if (all > 2147483647.0) {
        refuse(p);
        __syncthreads();
        continue;
      }
    }
    {
      int sum = 0;
      for (int t = i0; t < i1; ++t)
        for (int w = 0; w < cw; ++w) sum += s_start[w * n_tiles + t];
      const int incl = wave_inclusive_scan(sum);
      if (lane == kWave - 1) sh.wsum[wid] = incl;
      lds_sync();
      int run = incl - sum;
      for (int w = 0; w < wid; ++w) run += sh.wsum[w];
      for (int t = i0; t < i1; ++t)
        for (int w = 0; w < cw; ++w) {
          const int k = s_start[w * n_tiles + t];
          s_start[w * n_tiles + t] = run;
          run += k;
        }
      if (tid == kTileThreads - 1) sh.total = run;  // its tiles end at n_tiles
      lds_sync();
    }
    const int total = sh.total;
    if (tid == 0 && a.status) a.status[p] = 0;

    // Records of tiles [t0, t1) to the workspace.  The starts of the range
    // move on by one part: tile t then ends at s_start[last + t] and starts
    // where tile t - 1 ends.
    bool bounded = false;
    auto scatter = [&](int t0, int t1) {
      const int first = s_start[t0];
      // later ranges only visit the tile rows they hold
      const int row0 = bounded ? t0 / ntx : 0, row1 = bounded ? (t1 - 1) / ntx : n_tiles;
      const float inv_p = pmax > 0.0f ? a.bound_units / pmax : 0.0f;
      lds_sync();
      each_spot([&](int j0, int j, bool in, float amp, float X, float Y, int lo, int hi, int xlo, int xhi) {
        int q = 0;
        if (grad) q = chunk_row[j0 / kWave] + mask_rank(__ballot(in));
        if (!in) return;
        const int tx0 = xlo / kTileEdge, tx1 = xhi / kTileEdge, ty0 = lo / kTileEdge, ty1 = hi / kTileEdge;
        // one entry: offset (x, y) of the spot in tile t, box bits, and the
        // largest value it has there (from the distance to the tile), rounded up
        auto entry = [&](int t, float x, float y, int bits, float gx, float gy) {
          if (!bounded) {
            const float u = amp * __builtin_amdgcn_exp2f(c * (gx * gx + gy * gy)) * inv_p;
            atomicAdd(&s_u[t], static_cast<int>(u) + 1);
          }
          if (t < t0 || t >= t1) return;
          const int at = atomicAdd(&s_start[wid * n_tiles + t], 1) - first;
          rec[at] = make_float4(x, y, amp, __int_as_float(bits));
          if (grad) erow[at] = q;
        };
        if (tx1 - tx0 <= 1 && ty1 - ty0 <= 1) {  // at most 2 x 2 tiles: no loops
          const float x = X - static_cast<float>(tx0 * kTileEdge), y = Y - static_cast<float>(ty0 * kTileEdge);
          // 32 rows and columns from the first tile's; a box ends in its second tile at most
          const unsigned yb = (~0u >> (31 - (hi - ty0 * kTileEdge))) & (~0u << (lo - ty0 * kTileEdge));
          const unsigned xb = (~0u >> (31 - (xhi - tx0 * kTileEdge))) & (~0u << (xlo - tx0 * kTileEdge));
          const int t = ty0 * ntx + tx0;
          // the centre lies in the box's first or second tile along each axis
          const float gx0 = fmaxf(x - 15.0f, 0.0f), gy0 = fmaxf(y - 15.0f, 0.0f);
          const float gx1 = fmaxf(16.0f - x, 0.0f), gy1 = fmaxf(16.0f - y, 0.0f);
          const int ylow = yb & 0xffff, yhigh = yb >> 16, xlow = xb << 16, xhigh = xb & 0xffff0000u;
          entry(t, x, y, ylow | xlow, gx0, gy0);
          if (tx1 > tx0) entry(t + 1, x - 16.0f, y, ylow | xhigh, gx1, gy0);
          if (ty1 > ty0) {
            entry(t + ntx, x, y - 16.0f, yhigh | xlow, gx0, gy1);
            if (tx1 > tx0) entry(t + ntx + 1, x - 16.0f, y - 16.0f, yhigh | xhigh, gx1, gy1);
          }
        } else {
          for (int ty = max(ty0, row0); ty <= min(ty1, row1); ++ty)
            for (int tx = tx0; tx <= tx1; ++tx) {
              const float x = X - static_cast<float>(tx * kTileEdge), y = Y - static_cast<float>(ty * kTileEdge);
              const int bits = tile_bits(lo - ty * kTileEdge, hi - ty * kTileEdge) |
                               (tile_bits(xlo - tx * kTileEdge, xhi - tx * kTileEdge) << 16);
              entry(ty * ntx + tx, x, y, bits, fmaxf(0.0f, fmaxf(-x, x - 15.0f)),
                    fmaxf(0.0f, fmaxf(-y, y - 15.0f)));
            }
        }
      });
      bounded = true;
      __syncthreads();  // the records in global memory, block-visible
      return first;
    };
    auto unscatter = [&](int t0, int t1, int first) {  // the starts as they were
      lds_sync();
      const int a0 = max(i0, t0), a1 = min(i1, t1);
      const int before = a0 < a1 && a0 > t0 ? s_start[last + a0 - 1] : first;
      lds_sync();
      for (int t = a1 - 1; t >= a0; --t) {
        for (int w = cw - 1; w > 0; --w) s_start[w * n_tiles + t] = s_start[(w - 1) * n_tiles + t];
        s_start[t] = t > a0 ? s_start[last + t - 1] : before;
      }
      lds_sync();
    };
    // end of the range of tiles from t0 whose entries fit the workspace (a
    // tile alone always does: E >= cap)
    auto range_end = [&](int t0) {
      if (total - s_start[t0] <= E) return n_tiles;
      lds_sync();
      if (tid == 0) sh.t1 = t0 + 1;
      lds_sync();
      int mine = t0 + 1;
      for (int t = max(i0, t0) + 1; t <= i1; ++t)
        if ((t < n_tiles ? s_start[t] : total) - s_start[t0] <= E) mine = t;
      atomicMax(&sh.t1, mine);
      lds_sync();
      return sh.t1;
    };
    // ---- maximum, tiles, max term: each over the tiles of a range, the range's
    // records scattered once when the whole pattern's fit the workspace ----------
    const bool whole = total <= E;
    bool scattered = false;
    double lsum = 0.0, csum = 0.0;
    const float *tgt = kFwd ? nullptr : a.target + static_cast<size_t>(p) * a.target_stride;
    float *pat = a.pattern ? a.pattern + static_cast<size_t>(p) * HW : nullptr;
    const bool l2 = a.mode == DSX_ADJ_L2;
    const float unit = pmax / a.bound_units * 1.0001f;
    bool norm = false;
    float out_scale = 1.0f, corr = 0.0f;
    int px = 0, py = 0;  // the maximum's pixel
    enum { kMaximum, kTiles, kMaxTerm };
    for (int phase = a.normalize && total > 0 ? kMaximum : kTiles; phase <= kMaxTerm; ++phase) {
      int t0 = 0, t_end = n_tiles;
      if (phase == kTiles) {
        lds_sync();  // every wave's maximum
        const unsigned long long best = sh.best;
        const float vmax = __uint_as_float(static_cast<unsigned>(best >> kTilePixBits));
        const int pstar = (1 << kTilePixBits) - 1 - static_cast<int>(best & ((1ull << kTilePixBits) - 1));
        // a zero maximum leaves the pattern unnormalised (the reference returns
        // the zeros as they are)
        norm = a.normalize && vmax > 0.0f;
        out_scale = norm ? 1.0f / vmax : 1.0f;
        py = pstar / W;
        px = pstar - py * W;
      }
      if (phase == kMaxTerm) {
        if (kFwd) break;
        auto sum_d = [](double v) {
#pragma unroll
          for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, kWave);
          return v;
        };
        lsum = sum_d(lsum);
        csum = sum_d(csum);
        if (lane == 0) {
          sh.red[wid][0] = lsum;
          sh.red[wid][1] = csum;
        }
        __syncthreads();  // the gathered sums too
        double ltot = 0.0, ctot = 0.0;
        for (int w = 0; w < kTileWaves; ++w) {
          ltot += sh.red[w][0];
          ctot += sh.red[w][1];
        }
        if (tid == 0 && a.loss) a.loss[p] = static_cast<float>(ltot);
        if (tid == 0 && grad) a.gcount[p] = sh.ns;
        if (!grad || !norm) break;
        corr = static_cast<float>(ctot) * out_scale;
        t0 = (py / kTileEdge) * ntx + px / kTileEdge;
        t_end = t0 + 1;
      }
      while (t0 < t_end) {
        const int r0 = whole ? 0 : t0;  // first tile of the scattered range
        const int t1 = whole || phase == kMaxTerm ? t_end : range_end(t0);
        int first = 0;
        if (total > 0 && !(whole && scattered)) {
          first = scatter(r0, whole ? n_tiles : t1);
          scattered = true;
        }
        auto entries = [&](int t, int &e0, int &e1) {
          e0 = (t > r0 ? s_start[last + t - 1] : first) - first;
          e1 = s_start[last + t] - first;
        };
        if (phase == kMaxTerm) {
          // the max term of the normalisation, -(sum G P)/m at the maximum's
          // pixel, for the spots whose box holds it (the entries of its tile)
          int e0, e1;
          entries(t0, e0, e1);
          const int by = py % kTileEdge, bx = px % kTileEdge;
          for (int e = e0 + tid; e < e1; e += kTileThreads) {
            const float4 v = rec[e];
            const int mask = __float_as_int(v.w);
            if (!((mask >> by) & 1) || !((mask >> (16 + bx)) & 1)) continue;
            const float dx = static_cast<float>(bx) - v.x, dy = static_cast<float>(by) - v.y;
            const float kc = corr * a.pref * expf(a.ep * (dx * dx + dy * dy));
            float *g = reinterpret_cast<float *>(gsum + erow[e]);
            unsafeAtomicAdd(g, -kc);
            unsafeAtomicAdd(g + 1, -kc * dx);
            unsafeAtomicAdd(g + 2, -kc * dy);
          }
        } else {
          // the waves take the range's tiles in turn, a fixed share each, so the
          // loss is summed in one order (turning by one per eight tiles, so that
          // no wave keeps to a column of the pattern)
          for (int g = 0; t0 + g * kTileWaves < t1; ++g) {
            const int t = t0 + g * kTileWaves + ((wid + g) & (kTileWaves - 1));
            if (t >= t1) continue;
            int e0, e1;
            entries(t, e0, e1);
            const int ty = t / ntx, tx = t - ty * ntx;
            const int x = tx * kTileEdge + pos, y = ty * kTileEdge + 4 * sub;
            if (phase == kMaximum) {
              if (e0 == e1) continue;
              const float known = fmaxf(vlow, __uint_as_float(static_cast<unsigned>(
                                                  *const_cast<volatile unsigned long long *>(&sh.best) >> kTilePixBits)));
              if (static_cast<float>(s_u[t]) * unit < known) continue;
            }
            const size_t at = static_cast<size_t>(y) * W + x;
            tile_f4 G = {0.0f, 0.0f, 0.0f, 0.0f};  // the target until the products are done
            if (!kFwd && phase == kTiles) {
#pragma unroll
              for (int r = 0; r < 4; ++r)
                if (x < W && y + r < H) G[r] = tgt[at + static_cast<size_t>(r) * W];
            }
            tile_f4 P = tile_pixels(sh, rec, grad && phase == kTiles ? erow : nullptr, e0, e1, c, lane, wid);
            if (phase == kMaximum) {
              unsigned long long key = 0;
#pragma unroll
              for (int r = 0; r < 4; ++r) {
                if (y + r >= H || x >= W) continue;
                const unsigned long long k =
                    (static_cast<unsigned long long>(__float_as_uint(fmaxf(P[r], 0.0f))) << kTilePixBits) |
                    static_cast<unsigned long long>((1 << kTilePixBits) - 1 - ((y + r) * W + x));
                key = k > key ? k : key;
              }
              key = static_cast<unsigned long long>(wave_max_acc(static_cast<long long>(key)));
              if (lane == 0) atomicMax(&sh.best, key);
              continue;
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              P[r] *= out_scale;
              if (x >= W || y + r >= H) continue;
              if (pat) pat[at + static_cast<size_t>(r) * W] = P[r];
              if (kFwd) continue;
              float gr = G[r];
              if (l2) {
                const float d = P[r] - gr;
                lsum += static_cast<double>(d * d);
                gr = 2.0f * d;
              }
              csum += static_cast<double>(gr * P[r]);
              G[r] = gr * out_scale;
            }
            if (!grad || e0 == e1) continue;
            // the entries of a tile with at most 64 are still staged
            for (int e = e0; e < e1; e += kWave) {
              if (e1 - e0 > kWave) tile_stage(sh, rec, erow, e, e1, lane, wid);
              tile_gather(sh, G, gsum, min(kWave, e1 - e), c, a.pref, lane, wid);
            }
          }
        }
        if (!whole) unscatter(t0, t1, first);
        t0 = t1;
      }
    }
    __syncthreads();  // LDS and workspace state of this pattern is dead before the next one
  }
}

}  // namespace dsx
