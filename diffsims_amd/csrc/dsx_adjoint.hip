// Adjoint of the pattern path: gradients of a loss on the rendered sub-pixel
// patterns with respect to the orientation matrices, the reciprocal basis
// (hence the lattice parameters), the fractional atom positions and the
// Debye-Waller factors.  diffsims has no gradients; this is the reverse mode
// of dsx_simulate + dsx_render_subpixel + dsx_structure_factor.
//
// render_adjoint_kernel (one block per pattern, persistent over patterns)
//   recomputes the pattern as render_kernel<subpixel> does (same spots and
//   clip boxes; 32-bit fixed-point LDS strips), so it needs no stored pattern:
//     pass A  pattern maximum m and its first pixel p* (normalize): exact
//             evaluation of the few 16x16 tiles whose bound can reach the
//             value at the brightest spot (a full pass when too many remain);
//     pass B  per strip: P = Q/m, then the upstream gradient G = dL/dP
//             (2 (P - T) for the L2 loss, or given), kept in LDS as G/m;
//             each spot gathers A = sum G/m K, B = sum G/m K (x - X) over its
//             box (the transpose of the splat: no atomics on pixels);
//     then    the max term of the normalisation, -(sum_q G P)/m at p*, and
//             the per-spot sums go to a workspace.
// spot_chain_kernel (one wave per pattern)
//   per spot the chain through pixel position, intensity I = |F|^2 f(s, r)
//   and the excitation error (recomputed in FP64 from the integer hkl, the
//   orientation and the reciprocal basis): dL/dRt of the pattern, dL/d|F|^2
//   per reflection (atomics) and dL/drec through g (block partials, summed by
//   sum_partials_kernel in a fixed order).
// render_tiles_kernel (dsx_tiles.h): the same for spot lists longer than the
//   LDS spot table, on the matrix cores; its gsum rows go through the same
//   spot_chain_kernel.
// structure_factor_adjoint_kernel (one thread per reflection)
//   recomputes F(hkl) and reduces dL/d|F|^2 into dL/dxyz and dL/dB per atom
//   and into dL/d(rec) through |g|.
#include <algorithm>
#include <mutex>

#include "dsx_internal.h"
#include "dsx_physics.h"
#include "dsx_sf.h"
#include "dsx_splat.h"
#include "dsx_tiles.h"

namespace dsx {

constexpr int kAdjThreads = 512;
constexpr int kAdjWaves = kAdjThreads / kWave;
constexpr int kAdjMaxSpots = 1024;   // longest spot list of the two-blocks-per-CU kernel
constexpr int kAdjMaxStrips = 256;
constexpr int kAdjBinCap = 4096;
constexpr int kPixBits = 22;  // argmax key: value << 22 | (2^22 - 1 - pixel)
constexpr int kNRed = 20;     // block sums: loss, sum G P, dRt[9], dL/drec[9]
constexpr int kAdjTile = 16;      // tile edge of the fixed-point bound
constexpr int kAdjMaxTiles = 1024;
constexpr int kAdjMaxCand = 16;    // candidate tiles of the maximum search
constexpr int kAdjCandSpots = 64;  // spots touching one candidate tile
// float4 target values each thread of the two-blocks-per-CU kernel prefetches
// for one strip of at most kAdjSmallStripBytes / 8 pixels
constexpr int kAdjPre = 4;
constexpr int kAdjSmallStripBytes = kAdjPre * 4 * kAdjThreads * 8;
constexpr float kAdjRange = 2040109465.6f;  // 1.9 * 2^30 units per bound
constexpr float kAdjBoundUnits = 1048576.0f;  // 2^20 bound units per largest spot

// 32-bit fixed-point strip words: the largest per-tile sum U of the spots'
// peak values bounds every pixel, so one unit = U / (1.9 * 2^30) cannot
// overflow (the bound is an integer sum, independent of the atomics' order).
typedef int aacc_t;

struct AdjArgs {
  const int *idx;
  const float4 *spots;
  const int *count;
  int cap;
  int n;
  const int4 *hkl;
  const float *F2;
  int n_refl;
  const double *Rt;
  double rec[9];
  // physics (fill_physics)
  double k, k2, me, width, sigma, fac;
  int model, precession;
  double phi, Pz, Pt;
  // detector
  int H, W;
  float cal, cx, cy, ca, sa;
  int mirrored, normalize;
  float pref, ep, inv_s2, clip;
  float log2_clip, two_s2_ln2, tiny_box, box_margin;  // subpixel_box_fast
  float bound_units;        // long lists: tile-bound units of the largest spot
  int count_waves;          // long lists: waves that count and scatter the spots
  float e2ep;  // exp(2 ep): ratio of consecutive row ratios of the Gaussian
  int strip_rows, n_strips, acc_words;
  int slots, bin_cap;       // LDS spot slots and strip-bin entries
  int mode;
  int want_grad;
  long long target_stride;  // elements between targets (0: one target for every pattern)
  int *work;                // long lists: per-block entries (may be NULL)
  long long work_per_block; // ints
  int work_entries;         // entries per block
  float4 *gsum;             // per pattern and slot: A, BX, BY, list position (chain kernel input)
  int *gcount;              // per pattern: slots used
  const float *target;
  float *pattern;
  float *loss;
  double *dRt;
  float *dF2;    // [n_refl] dL/d|F|^2, accumulated (may be NULL)
  double *drec;  // [9] sum dL/dg (x) hkl, accumulated (may be NULL)
  double *dpart; // chain kernel: per-block partial sums of drec
  int *status;
};

struct AdjShared {
  int bin_start[kAdjMaxStrips + 1];
  int bin_fill[kAdjMaxStrips];
  int ns, cols_max;
  float wmaxf[kAdjWaves];
  long long wkey[kAdjWaves];
  int wu[kAdjWaves];
  int qstar, n_cand, fail;
  long long lkey;
  int cand_tile[kAdjMaxCand], cand_n[kAdjMaxCand];
  double red[kAdjWaves][kNRed];
};

// The spot table lives in dynamic LDS after the two strip buffers (acc_words
// fixed-point words, acc_words gradient floats), sized by the host: `slots`
// entries of each field, then `bin_cap` strip-bin entries.
struct SpotTab {
  float *I, *X, *Y, *A, *BX, *BY;
  int *xb;    // (xlo << 16) | xhi
  int *jpos;  // position in the pattern's spot list
  short *ylo, *yhi, *bin;
};

constexpr int kSpotTabBytes = 6 * 4 + 2 * 4 + 2 * 2;  // per slot

__device__ __forceinline__ SpotTab spot_tab(aacc_t *s_acc, size_t strip_words, int slots) {
  float *f = reinterpret_cast<float *>(s_acc + strip_words);
  SpotTab t;
  t.I = f;
  t.X = f + slots;
  t.Y = f + 2 * slots;
  t.A = f + 3 * slots;
  t.BX = f + 4 * slots;
  t.BY = f + 5 * slots;
  int *iv = reinterpret_cast<int *>(f + 6 * slots);
  t.xb = iv;
  t.jpos = iv + slots;
  short *sv = reinterpret_cast<short *>(iv + 2 * slots);
  t.ylo = sv;
  t.yhi = sv + slots;
  t.bin = sv + 2 * slots;
  return t;
}

// Reflection-side constants of the chain rule, staged in LDS once per block so
// the kernels do not hold them in scalar registers throughout.
struct ChainConsts {
  double rec[9];
  double k, k2, me, width, sigma, fac;
  int model, precession;
  double phi, Pz, Pt;
};

__device__ __forceinline__ void stage_chain_consts(const AdjArgs &a, ChainConsts &c) {
  for (int i = 0; i < 9; ++i) c.rec[i] = a.rec[i];
  c.k = a.k;
  c.k2 = a.k2;
  c.me = a.me;
  c.width = a.width;
  c.sigma = a.sigma;
  c.fac = a.fac;
  c.model = a.model;
  c.precession = a.precession;
  c.phi = a.phi;
  c.Pz = a.Pz;
  c.Pt = a.Pt;
}

__device__ __forceinline__ double wave_sum_d(double v) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, kWave);
  return v;
}

// Fixed-point value of one Gaussian term amp exp(ep r^2) at offset (dx, dy),
// written once so the splat and the maximum search round it identically.
__device__ __forceinline__ int gauss_term(float amp, float dx, float dy, float ep, float scale) {
  return __float2int_rn(amp * fast_exp(ep * fmaf(dy, dy, dx * dx)) * scale);
}

// it / ncols, a shift for powers of two (ncols is uniform)
__device__ __forceinline__ int item_spot(int it, int ncols) {
  return (ncols & (ncols - 1)) == 0 ? it >> __builtin_ctz(ncols) : it / ncols;
}
// Column count of a gather pass: the next power of two up to a wave, so a
// spot's run of items never straddles two waves and its first lane ends up
// with the whole sum (no LDS float atomics, which run far slower than
// integer ones)
__device__ __forceinline__ int gather_cols(int w) {
  return w <= 1 ? 1 : (w <= kWave ? 1 << (32 - __builtin_clz(w - 1)) : w);
}

// Splat (kGather = false) or gather (true) of every binned spot footprint
// inside strip rows [y0, y1).  Work item = (spot, footprint column) so a wave
// touches consecutive LDS columns.
template <bool kGather>
__device__ __forceinline__ void strip_pass(const AdjArgs &a, const SpotTab &t, int cols_max,
                                           aacc_t *acc, const float *G, int b0, int nb,
                                           bool binned, int y0, int y1, float scale, int tid) {
  // unbinned: LDS slots b0 .. b0 + nb - 1
  const int W = a.W;
  const int ncols = cols_max;
  const int n_items = nb * ncols;
  if (!kGather) {
    for (int it = tid; it < n_items; it += kAdjThreads) {
      const int bi = item_spot(it, ncols);
      const int c = it - bi * ncols;
      const int q = binned ? t.bin[b0 + bi] : b0 + bi;
      const int ya = max(static_cast<int>(t.ylo[q]), y0);
      const int yb = min(static_cast<int>(t.yhi[q]), y1 - 1);
      if (ya > yb) continue;
      const int xlo = t.xb[q] >> 16, xhi = t.xb[q] & 0xffff;
      const int x = xlo + c;
      if (x > xhi) continue;
      const float dx = static_cast<float>(x) - t.X[q];
      const float cy = t.Y[q];
      const float amp = t.I[q] * a.pref;
      aacc_t *col = acc + x;
      lds_reads_done();
      for (int y = ya; y <= yb; ++y) {
        const float dy = static_cast<float>(y) - cy;
        atomicAdd(col + (y - y0) * W, gauss_term(amp, dx, dy, a.ep, scale));
      }
    }
    return;
  }
  // Gather: the ncols consecutive items of a spot sit in consecutive lanes,
  // so their column sums are combined across lanes first (segmented shuffle
  // reduction) and only the first lane of each spot's run adds them to LDS:
  // LDS float atomics to one address serialise, and a spot's columns would
  // otherwise all hit the same three words.
  const int lane = lane_id();
  for (int base = tid - lane; base < n_items; base += kAdjThreads) {
    const int it = base + lane;
    const int bi = item_spot(it, ncols);
    const int c = it - bi * ncols;
    int q = -1;
    float sa = 0.0f, sx = 0.0f, sy = 0.0f;
    if (it < n_items) {
      q = binned ? t.bin[b0 + bi] : b0 + bi;
      const int ya = max(static_cast<int>(t.ylo[q]), y0);
      const int yb = min(static_cast<int>(t.yhi[q]), y1 - 1);
      const int xlo = t.xb[q] >> 16, xhi = t.xb[q] & 0xffff;
      const int x = xlo + c;
      if (ya <= yb && x <= xhi) {
        // down the column the Gaussian follows K(y + 1) = K(y) r(y) with
        // r(y + 1) = r(y) exp(2 ep): two products per row instead of an exp
        // (a few ulps over a box; the splat keeps its exact per-pixel terms)
        const float dx = static_cast<float>(x) - t.X[q];
        float dy = static_cast<float>(ya) - t.Y[q];
        float k = a.pref * fast_exp(a.ep * (dy * dy + dx * dx));
        float r = fast_exp(a.ep * (2.0f * dy + 1.0f));
        const float *g = G + (ya - y0) * W + x;
        auto row = [&](float gv) {
          const float kg = k * gv;
          sa += kg;
          sy = fmaf(kg, dy, sy);
          k *= r;
          r *= a.e2ep;
          dy += 1.0f;
        };
        // four rows' G words are read together, so one LDS round trip
        // serves four rows
        int y = ya;
        for (; y + 3 <= yb; y += 4, g += 4 * W) {
          const float g0 = g[0], g1 = g[W], g2 = g[2 * W], g3 = g[3 * W];
          row(g0);
          row(g1);
          row(g2);
          row(g3);
        }
        for (; y <= yb; ++y, g += W) row(*g);
        sx = sa * dx;
      }
    }
    // lane L takes lane L + d while both lie in the same spot's run; after
    // the steps the first lane of each run (in this wave) holds its sums
    for (int d = 1; d < ncols && d < kWave; d <<= 1) {
      const float oa = __shfl_down(sa, d, kWave);
      const float ox = __shfl_down(sx, d, kWave);
      const float oy = __shfl_down(sy, d, kWave);
      if (c + d < ncols && lane + d < kWave) {
        sa += oa;
        sx += ox;
        sy += oy;
      }
    }
    if (q >= 0 && (c == 0 || lane == 0) && (sa != 0.0f || sx != 0.0f || sy != 0.0f)) {
      if ((ncols & (ncols - 1)) == 0 && ncols <= kWave) {
        // the run lies in this wave and this lane (c == 0) holds its sum;
        // a spot has one run per pass
        t.A[q] += sa;
        t.BX[q] += sx;
        t.BY[q] += sy;
      } else {
        atomicAdd(&t.A[q], sa);
        atomicAdd(&t.BX[q], sx);
        atomicAdd(&t.BY[q], sy);
      }
    }
  }
}

// Chain rule of one spot: (dL/dI, dL/dX, dL/dY) -> dL/dRt of the pattern (dR,
// accumulated), dL/dg (x) hkl of its reflection (dG, accumulated when a.drec)
// and dL/d|F|^2 of its reflection (a global atomic when a.dF2).
__device__ __forceinline__ void spot_chain(const AdjArgs &a, const ChainConsts &c, const double *R,
                                           int row, double I, double dI, double BX, double BY,
                                           double *dR, double *dG) {
  const double dX = I * BX * a.inv_s2;
  const double dY = I * BY * a.inv_s2;
  if (dI == 0.0 && dX == 0.0 && dY == 0.0) return;
  const double ca = a.ca, sa = a.sa, ic = 1.0 / static_cast<double>(a.cal);
  double dx, dy;  // d/d(lab x, lab y)
  if (a.mirrored) {
    dx = (dX * ca + dY * sa) * ic;
    dy = (dX * sa - dY * ca) * ic;
  } else {
    dx = (dX * ca + dY * sa) * ic;
    dy = (-dX * sa + dY * ca) * ic;
  }
  const int4 h = a.hkl[row];
  const double hx = h.x, hy = h.y, hz = h.z;
  const double g0 = c.rec[0] * hx + c.rec[1] * hy + c.rec[2] * hz;
  const double g1 = c.rec[3] * hx + c.rec[4] * hy + c.rec[5] * hz;
  const double g2 = c.rec[6] * hx + c.rec[7] * hy + c.rec[8] * hz;
  const double x = R[0] * g0 + R[1] * g1 + R[2] * g2;
  const double y = R[3] * g0 + R[4] * g1 + R[5] * g2;
  const double z = R[6] * g0 + R[7] * g1 + R[8] * g2;
  const double r2 = x * x + y * y;
  const double r = fsqrt_pos(r2);
  const double qk = fsqrt_pos(fmax(c.k2 - r2, 0.0));
  const double sv = fdiv(r2, c.k + qk) - z;
  double fs, fr;
  const double f = shape_factor_grad(sv, r, c, fs, fr);
  const double F2 = a.F2[row];
  const double dF2 = dI * f;
  const double ds = dI * F2 * fs;
  const double dr = dI * F2 * fr;
  double gx = dx, gy = dy, gz = -ds;
  double radial = 0.0;  // along (x, y)
  if (c.k2 > r2) radial = ds * frcp(qk);
  if (r2 > 0.0 && dr != 0.0) radial += dr * frcp(r);
  gx += radial * x;
  gy += radial * y;
  // g_lab = Rt g: dL/dRt[i][c] = dL/dg_lab[i] g[c]; dL/dg = Rt^T dL/dg_lab
  dR[0] += gx * g0; dR[1] += gx * g1; dR[2] += gx * g2;
  dR[3] += gy * g0; dR[4] += gy * g1; dR[5] += gy * g2;
  dR[6] += gz * g0; dR[7] += gz * g1; dR[8] += gz * g2;
  if (a.drec) {
    // dL/dg (crystal frame) = Rt^T dL/dg_lab; g = rec hkl: dL/drec += dL/dg hkl^T
    const double d0 = R[0] * gx + R[3] * gy + R[6] * gz;
    const double d1 = R[1] * gx + R[4] * gy + R[7] * gz;
    const double d2 = R[2] * gx + R[5] * gy + R[8] * gz;
    dG[0] += d0 * hx; dG[1] += d0 * hy; dG[2] += d0 * hz;
    dG[3] += d1 * hx; dG[4] += d1 * hy; dG[5] += d1 * hz;
    dG[6] += d2 * hx; dG[7] += d2 * hy; dG[8] += d2 * hz;
  }
  if (a.dF2) unsafeAtomicAdd(a.dF2 + row, static_cast<float>(dF2));
}

// The max term of the normalisation (-(sum G P)/m at the maximum's pixel p*)
// for a spot whose box holds p*, added to its gathered sums.
__device__ __forceinline__ void max_term(const AdjArgs &a, float corr, int px, int py, float X,
                                         float Y, int xlo, int xhi, int lo, int hi, float &A,
                                         float &BX, float &BY) {
  if (px < xlo || px > xhi || py < lo || py > hi) return;
  const float dx = static_cast<float>(px) - X, dy = static_cast<float>(py) - Y;
  const float kc = corr * a.pref * expf(a.ep * (dx * dx + dy * dy));
  A -= kc;
  BX -= kc * dx;
  BY -= kc * dy;
}

// Fixed-point value at pixel (x, y) of LDS spot q (0 outside its clip box).
__device__ __forceinline__ int spot_at(const AdjArgs &a, const SpotTab &t, int q, int x, int y,
                                       float scale) {
  if (y < t.ylo[q] || y > t.yhi[q] || x < (t.xb[q] >> 16) || x > (t.xb[q] & 0xffff)) return 0;
  return gauss_term(t.I[q] * a.pref, static_cast<float>(x) - t.X[q],
                    static_cast<float>(y) - t.Y[q], a.ep, scale);
}

// Pattern maximum and its first pixel, as the key value << kPixBits |
// (2^kPixBits - 1 - pixel), without rendering the whole pattern: a tile whose
// bound (the per-tile sums tile_u of the spots' peak values, in units of
// `unit`) stays below the exact value at the brightest spot's nearest pixel
// cannot hold the maximum, and the few remaining tiles are evaluated pixel by
// pixel with the splat's own fixed-point terms (integer sums: the result equals
// a full pass bit for bit).  Every pixel holding the maximum lies in a
// remaining tile, so the first of them is found.  Returns false (uniformly)
// when too many tiles or spots remain; the caller then runs the full pass.
// tile_u is overwritten (candidate slots); cand_q borrows the gradient buffer.
template <class Shared>
__device__ bool bounded_max_key(const AdjArgs &a, Shared &sh, const SpotTab &t, int *tile_u,
                                short (*cand_q)[kAdjCandSpots], int ntx, int n_tiles, int ns,
                                float scale, float unit, int tid, int lane, int wid,
                                long long &key_out) {
  const int H = a.H, W = a.W;
  if (tid == 0) {
    sh.n_cand = 0;
    sh.fail = 0;
  }
  if (wid == 0) {
    const int qs = sh.qstar;
    const int xs = min(max(static_cast<int>(rintf(t.X[qs])), t.xb[qs] >> 16), t.xb[qs] & 0xffff);
    const int ys = min(max(static_cast<int>(rintf(t.Y[qs])), static_cast<int>(t.ylo[qs])),
                       static_cast<int>(t.yhi[qs]));
    long long acc = 0;
    for (int q = lane; q < ns; q += kWave) acc += spot_at(a, t, q, xs, ys, scale);
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) acc += __shfl_xor(acc, off, kWave);
    if (lane == 0)
      sh.lkey = (max(acc, 0ll) << kPixBits) |
                static_cast<long long>((1 << kPixBits) - 1 - (ys * W + xs));
  }
  lds_sync();
  const long long lkey = sh.lkey;
  const float lfix = static_cast<float>(lkey >> kPixBits);
  // per term: the float product is within 1e-5 of the bound's share and the
  // rounding adds at most one half
  const float margin = 0.5f * static_cast<float>(ns) + 1.0f;
  int *slot_of = tile_u;
  for (int ti = tid; ti < n_tiles; ti += kAdjThreads) {
    const float bound = static_cast<float>(tile_u[ti]) * unit * scale * 1.00001f + margin;
    int slot = -1;
    if (bound >= lfix) {
      slot = atomicAdd(&sh.n_cand, 1);
      if (slot < kAdjMaxCand) {
        sh.cand_tile[slot] = ti;
        sh.cand_n[slot] = 0;
      } else {
        slot = -1;
        sh.fail = 1;
      }
    }
    slot_of[ti] = slot;
  }
  lds_sync();
  if (sh.fail) return false;
  const int n_cand = sh.n_cand;
  for (int q = tid; q < ns; q += kAdjThreads) {
    const int tx0 = (t.xb[q] >> 16) / kAdjTile, tx1 = (t.xb[q] & 0xffff) / kAdjTile;
    const int ty0 = t.ylo[q] / kAdjTile, ty1 = t.yhi[q] / kAdjTile;
    for (int ty = ty0; ty <= ty1; ++ty)
      for (int tx = tx0; tx <= tx1; ++tx) {
        const int sl = slot_of[ty * ntx + tx];
        if (sl < 0) continue;
        const int pos = atomicAdd(&sh.cand_n[sl], 1);
        if (pos < kAdjCandSpots)
          cand_q[sl][pos] = static_cast<short>(q);
        else
          sh.fail = 1;
      }
  }
  lds_sync();
  if (sh.fail) return false;
  long long key = lkey;
  for (int i = tid; i < n_cand * kAdjTile * kAdjTile; i += kAdjThreads) {
    const int sl = i / (kAdjTile * kAdjTile);
    const int ti = sh.cand_tile[sl];
    const int x = (ti % ntx) * kAdjTile + (i % kAdjTile);
    const int y = (ti / ntx) * kAdjTile + (i / kAdjTile) % kAdjTile;
    if (x >= W || y >= H) continue;
    long long acc = 0;
    const int nq = sh.cand_n[sl];
    for (int k = 0; k < nq; ++k) acc += spot_at(a, t, cand_q[sl][k], x, y, scale);
    const long long kv =
        (max(acc, 0ll) << kPixBits) | static_cast<long long>((1 << kPixBits) - 1 - (y * W + x));
    key = kv > key ? kv : key;
  }
  key = wave_max_acc(key);
  if (lane == 0) sh.wkey[wid] = key;
  lds_sync();
  key = 0;
  for (int w = 0; w < kAdjWaves; ++w) key = sh.wkey[w] > key ? sh.wkey[w] : key;
  key_out = key;
  lds_sync();  // wkey and the candidate state are reused
  return true;
}

// One pattern per block iteration: every in-frame spot fits the LDS slots (the
// host guarantees slots >= cap) and the per-spot sums go to gsum for
// spot_chain_kernel, which keeps the FP64 chain rule (and its registers) out
// of this kernel.
__device__ __forceinline__ void adjoint_body(const AdjArgs &a, aacc_t *s_acc,
                                             AdjShared &sh) {
  float *s_G = reinterpret_cast<float *>(s_acc + a.acc_words);
  const SpotTab t = spot_tab(s_acc, 2 * static_cast<size_t>(a.acc_words), a.slots);
  const int tid = threadIdx.x;
  const int lane = lane_id();
  const int wid = tid / kWave;
  const int H = a.H, W = a.W;
  const size_t HW = static_cast<size_t>(H) * W;
  for (int i = tid; i < a.acc_words; i += kAdjThreads) s_acc[i] = 0;
  lds_sync();

  for (int p = blockIdx.x; p < a.n; p += gridDim.x) {
    const int n = min(a.count[p], a.cap);
    const float4 *spots = a.spots + (size_t)p * a.cap;
    if (tid == 0) {
      sh.ns = 0;
      sh.cols_max = 1;
      sh.qstar = 0;
    }
    for (int b = tid; b <= kAdjMaxStrips; b += kAdjThreads) sh.bin_start[b] = 0;
    lds_sync();

    // ---- 1. spots in frame with their clip boxes --------------------------
    float tmax = 0.0f;
    for (int j = tid; j < n; j += kAdjThreads) {
      const float4 sp = spots[j];
      float X = 0.0f, Y = 0.0f;
      int lo = 1, hi = 0, xlo = 0, xhi = 0;
      const bool in = to_pixel(sp, a, X, Y) &&
                      subpixel_box_fast(sp.w, X, Y, a, lo, hi, xlo, xhi);
      if (!in) continue;
      tmax = fmaxf(tmax, fabsf(sp.w) * a.pref);
      atomicMax(&sh.cols_max, xhi - xlo + 1);
      for (int s = lo / a.strip_rows; s <= hi / a.strip_rows; ++s)
        atomicAdd(&sh.bin_start[s + 1], 1);
      const int q = atomicAdd(&sh.ns, 1);
      t.I[q] = sp.w;
      t.X[q] = X;
      t.Y[q] = Y;
      t.A[q] = 0.0f;
      t.BX[q] = 0.0f;
      t.BY[q] = 0.0f;
      t.xb[q] = (xlo << 16) | xhi;
      t.jpos[q] = j;
      t.ylo[q] = static_cast<short>(lo);
      t.yhi[q] = static_cast<short>(hi);
    }
    tmax = wave_max(tmax);
    if (lane == 0) sh.wmaxf[wid] = tmax;
    lds_sync();
    const int ns = sh.ns;
    float pmax = 0.0f;
    for (int w = 0; w < kAdjWaves; ++w) pmax = fmaxf(pmax, sh.wmaxf[w]);
    float scale = 1.0f;  // set from the tile bounds below

    // ---- 2. strip bins ----------------------------------------------------
    const int n_bins = a.n_strips;
    if (tid == 0) {
      int acc = 0;
      for (int b = 0; b < n_bins; ++b) {
        acc += sh.bin_start[b + 1];
        sh.bin_start[b + 1] = acc;
      }
    }
    lds_sync();
    const int entries = sh.bin_start[n_bins];
    if (tid == 0 && a.status) a.status[p] = 0;
    const bool binned = entries <= a.bin_cap;
    for (int b = tid; b < n_bins; b += kAdjThreads) sh.bin_fill[b] = sh.bin_start[b];
    lds_sync();
    if (binned) {
      for (int q = tid; q < ns; q += kAdjThreads) {
        for (int s = t.ylo[q] / a.strip_rows; s <= t.yhi[q] / a.strip_rows; ++s) {
          const int pos = atomicAdd(&sh.bin_fill[s], 1);
          t.bin[pos] = static_cast<short>(q);
        }
      }
    }
    lds_sync();
    const int cols_max = sh.cols_max;

    // ---- 2b. fixed-point scale: per-tile sums of the spots' peak values ------
    const int ntx = (W + kAdjTile - 1) / kAdjTile;
    const int n_tiles = ntx * ((H + kAdjTile - 1) / kAdjTile);
    const bool tiles = n_tiles <= kAdjMaxTiles && n_tiles <= a.acc_words;
    int *tile_u = s_acc;  // the strip buffer is zero here and zeroed again below
    const float unit = pmax / kAdjBoundUnits;  // value of one bound unit
    {
      const float inv_p = pmax > 0.0f ? kAdjBoundUnits / pmax : 0.0f;
      int usum = 0;
      auto add_bound = [&](float I, int lo, int hi, int xlo, int xhi) {
        const int u = min(static_cast<int>(ceilf(fabsf(I) * a.pref * inv_p)) + 1,
                          static_cast<int>(kAdjBoundUnits) + 1);
        usum += u;
        if (!tiles) return;
        for (int ty = lo / kAdjTile; ty <= hi / kAdjTile; ++ty)
          for (int tx = xlo / kAdjTile; tx <= xhi / kAdjTile; ++tx) atomicAdd(&tile_u[ty * ntx + tx], u);
      };
      for (int q = tid; q < ns; q += kAdjThreads) {
        if (fabsf(t.I[q]) * a.pref == pmax) sh.qstar = q;  // the brightest spot (any of a tie)
        add_bound(t.I[q], t.ylo[q], t.yhi[q], t.xb[q] >> 16, t.xb[q] & 0xffff);
      }
      int lu = 0;
      if (tiles) {
        lds_sync();
        for (int ti = tid; ti < n_tiles; ti += kAdjThreads) lu = max(lu, tile_u[ti]);
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) lu = max(lu, __shfl_xor(lu, off, kWave));
      } else {
        lu = wave_sum(usum);
      }
      if (lane == 0) sh.wu[wid] = lu;
      lds_sync();
      int Ui = 0;
      for (int w = 0; w < kAdjWaves; ++w) Ui = tiles ? max(Ui, sh.wu[w]) : Ui + sh.wu[w];
      const float U = static_cast<float>(Ui) * unit;
      scale = U > 0.0f ? kAdjRange / (U * 1.00001f) : 1.0f;
    }

    // splat (or gather) strip s: every spot of its bin
    auto strip_spots = [&](int s, bool gather, int y0, int y1) {
      const int b0 = binned ? sh.bin_start[s] : 0;
      const int nb = binned ? sh.bin_start[s + 1] - b0 : ns;
      if (nb <= 0) return;
      if (gather)
        strip_pass<true>(a, t, gather_cols(cols_max), s_acc, s_G, b0, nb, binned, y0, y1, scale, tid);
      else
        strip_pass<false>(a, t, cols_max, s_acc, nullptr, b0, nb, binned, y0, y1, scale, tid);
    };

    // ---- 3. pass A: maximum and its first pixel -----------------------------
    long long key = 0;
    bool have_key = false;
    if (a.normalize && ns > 0 && tiles &&
        a.acc_words * sizeof(float) >= sizeof(short) * kAdjMaxCand * kAdjCandSpots) {
      have_key = bounded_max_key(a, sh, t, tile_u, reinterpret_cast<short(*)[kAdjCandSpots]>(s_G),
                                 ntx, n_tiles, ns, scale, unit, tid, lane, wid, key);
    }
    if (tiles) {  // hand the borrowed words back zeroed
      for (int ti = tid; ti < n_tiles; ti += kAdjThreads) tile_u[ti] = 0;
      lds_sync();
    }
    if (a.normalize && ns > 0 && !have_key) {
      for (int s = 0; s < a.n_strips; ++s) {
        const int y0 = s * a.strip_rows;
        const int y1 = min(H, y0 + a.strip_rows);
        if (sh.bin_start[s + 1] == sh.bin_start[s]) continue;
        strip_spots(s, false, y0, y1);
        lds_sync();
        const int cnt = (y1 - y0) * W;
        const int pix0 = y0 * W;
        for (int i = tid; i < cnt; i += kAdjThreads) {
          const aacc_t v = s_acc[i];
          s_acc[i] = 0;
          const long long kv = (static_cast<long long>(max(v, 0)) << kPixBits) |
                               static_cast<long long>((1 << kPixBits) - 1 - (pix0 + i));
          key = kv > key ? kv : key;
        }
        lds_sync();
      }
      key = wave_max_acc(key);
      if (lane == 0) sh.wkey[wid] = key;
      lds_sync();
      key = 0;
      for (int w = 0; w < kAdjWaves; ++w) key = sh.wkey[w] > key ? sh.wkey[w] : key;
    }
    const long long m_fixed = key >> kPixBits;
    const int pstar = (1 << kPixBits) - 1 - static_cast<int>(key & ((1 << kPixBits) - 1));
    // a zero maximum leaves the pattern unnormalised (the reference returns the
    // zeros as they are)
    const bool norm = a.normalize && m_fixed > 0;
    const float out_scale = norm ? 1.0f / static_cast<float>(m_fixed) : 1.0f / scale;
    const float gscale = scale * out_scale;  // dL/dQ = G / m  (1 without normalisation)

    // ---- 4. pass B: pattern, loss, upstream gradient, gather ----------------
    double lsum = 0.0, csum = 0.0;
    const float *tgt = a.target ? a.target + (size_t)p * a.target_stride : nullptr;
    float *pat = a.pattern ? a.pattern + (size_t)p * HW : nullptr;
    const bool l2 = a.mode == DSX_ADJ_L2;
    const bool fwd_only = a.mode == DSX_ADJ_FORWARD;
    // the target of strip s + 1 is loaded into registers while strip s is
    // gathered and strip s + 1 splatted, so its HBM latency is hidden
    constexpr int kPre = kAdjPre;
    native_float4 tp[kPre];
    auto prefetch = [&](int s) {
      if (fwd_only || (W & 3) != 0 || s >= a.n_strips) return;
      const int y0 = s * a.strip_rows;
      const int cnt4 = (min(H, y0 + a.strip_rows) - y0) * W / 4;
      const native_float4 *src = reinterpret_cast<const native_float4 *>(tgt + (size_t)y0 * W);
#pragma unroll
      for (int k = 0; k < kPre; ++k) {
        const int i = tid + k * kAdjThreads;
        if (i < cnt4) tp[k] = __builtin_nontemporal_load(src + i);
      }
    };
    prefetch(0);
    for (int s = 0; s < a.n_strips; ++s) {
      const int y0 = s * a.strip_rows;
      const int y1 = min(H, y0 + a.strip_rows);
      const int cnt = (y1 - y0) * W;
      const bool any = sh.bin_start[s + 1] > sh.bin_start[s];
      if (any) {
        strip_spots(s, false, y0, y1);
        lds_sync();
      }
      const size_t off = (size_t)y0 * W;
      if ((W & 3) == 0) {
        // four pixels i: pattern, loss and G / m from the target values tv
        auto readout4 = [&](int i, const native_float4 &tv) {
          int4 *pv = reinterpret_cast<int4 *>(s_acc) + i;
          const int4 u = *pv;
          if (any) *pv = make_int4(0, 0, 0, 0);
          const float4 P = make_float4(static_cast<float>(u.x) * out_scale, static_cast<float>(u.y) * out_scale,
                                       static_cast<float>(u.z) * out_scale, static_cast<float>(u.w) * out_scale);
          if (pat) store_nt(P, reinterpret_cast<float4 *>(pat + off) + i);
          if (fwd_only) return;
          float4 g;
          if (l2) {
            const float4 d = make_float4(P.x - tv.x, P.y - tv.y, P.z - tv.z, P.w - tv.w);
            lsum += static_cast<double>(d.x * d.x + d.y * d.y + d.z * d.z + d.w * d.w);
            g = make_float4(2.0f * d.x, 2.0f * d.y, 2.0f * d.z, 2.0f * d.w);
          } else {
            g = make_float4(tv.x, tv.y, tv.z, tv.w);
          }
          csum += static_cast<double>(g.x * P.x + g.y * P.y + g.z * P.z + g.w * P.w);
          reinterpret_cast<float4 *>(s_G)[i] =
              make_float4(g.x * gscale, g.y * gscale, g.z * gscale, g.w * gscale);
        };
        const int n4 = cnt / 4;
        if (fwd_only) {
          const native_float4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
          for (int i = tid; i < n4; i += kAdjThreads) readout4(i, zero);
        } else {
#pragma unroll
          for (int k = 0; k < kPre; ++k) {
            const int i = tid + k * kAdjThreads;
            if (i < n4) readout4(i, tp[k]);
          }
        }
      } else {
        for (int i = tid; i < cnt; i += kAdjThreads) {
          const aacc_t v = s_acc[i];
          if (any) s_acc[i] = 0;
          const float P = static_cast<float>(v) * out_scale;
          if (pat) __builtin_nontemporal_store(P, pat + off + i);
          if (fwd_only) continue;
          const float tv = tgt[off + i];
          float g;
          if (l2) {
            const float d = P - tv;
            lsum += static_cast<double>(d * d);
            g = 2.0f * d;
          } else {
            g = tv;
          }
          csum += static_cast<double>(g * P);
          s_G[i] = g * gscale;
        }
      }
      prefetch(s + 1);
      lds_sync();
      if (a.want_grad && any) strip_spots(s, true, y0, y1);
      lds_sync();
    }
    lsum = wave_sum_d(lsum);
    csum = wave_sum_d(csum);
    if (lane == 0) {
      sh.red[wid][0] = lsum;
      sh.red[wid][1] = csum;
    }
    lds_sync();
    double ctot = 0.0, ltot = 0.0;
    for (int w = 0; w < kAdjWaves; ++w) {
      ltot += sh.red[w][0];
      ctot += sh.red[w][1];
    }

    if (a.want_grad) {
      // ---- 5. per spot: the normalisation's max term, then the chain rule ----
      const float corr = norm ? static_cast<float>(ctot) * gscale : 0.0f;
      const int px = pstar % W, py = pstar / W;
      // sums with the max term to gsum; spot_chain_kernel does the rest
      float4 *gs = a.gsum + (size_t)p * a.slots;
      for (int q = tid; q < ns; q += kAdjThreads) {
        float A = t.A[q], BX = t.BX[q], BY = t.BY[q];
        if (norm)
          max_term(a, corr, px, py, t.X[q], t.Y[q], t.xb[q] >> 16, t.xb[q] & 0xffff, t.ylo[q],
                   t.yhi[q], A, BX, BY);
        gs[q] = make_float4(A, BX, BY, __int_as_float(t.jpos[q]));
      }
      if (tid == 0) a.gcount[p] = ns;
    }
    if (tid == 0 && a.loss) a.loss[p] = static_cast<float>(ltot);
    lds_sync();  // LDS state of this pattern is dead before the next one
  }
}

// Two blocks per CU: at most 128 VGPRs (four waves per SIMD).
__global__ __launch_bounds__(kAdjThreads, 4) void render_adjoint_kernel(AdjArgs a) {
  extern __shared__ __align__(16) aacc_t s_acc[];  // 16-byte aligned for the 16-byte read-out
  __shared__ AdjShared sh;
  adjoint_body(a, s_acc, sh);
}

__global__ __launch_bounds__(kTileThreads, 4) void render_tiles_kernel(AdjArgs a) {
  extern __shared__ int s_tiles[];
  __shared__ TileShared sh;
  tiles_body<false>(a, s_tiles, sh);
}

__global__ __launch_bounds__(kTileThreads, 4) void render_tiles_fwd_kernel(AdjArgs a) {
  extern __shared__ int s_tiles[];
  __shared__ TileShared sh;
  tiles_body<true>(a, s_tiles, sh);
}

// Chain rule of every spot gathered by the render adjoint: one block per
// pattern (grid-stride), its spots spread over the block's threads; dL/dRt of
// the pattern is a block sum, dL/d|F|^2 of the reflections global atomics,
// dL/drec a per-block partial summed later in a fixed order.  Bound by latency:
// at 253 registers two waves per SIMD, 82 % of the time waiting, for the rows
// (15 % of it), the atomics (20 %) and FP64 results, VALU busy 27 %.
// 4,096 patterns of the 500-atom cell under precession 3.50 ms with the
// library's roots and quotients, 3.08 with those of dsx_physics.h.  Reading the
// rows a spot ahead (3.28) and more waves per SIMD (10.9, spills) are slower.
constexpr int kChainThreads = 256;
constexpr int kChainWaves = kChainThreads / kWave;

__global__ __launch_bounds__(kChainThreads) void spot_chain_kernel(AdjArgs a) {
  __shared__ ChainConsts s_cc;
  __shared__ double s_R[9];
  __shared__ double s_part[kChainWaves][9];
  if (threadIdx.x == 0) stage_chain_consts(a, s_cc);
  const int lane = lane_id();
  const int wid = threadIdx.x / kWave;
  double dG[9];  // dL/drec over this thread's spots
#pragma unroll
  for (int i = 0; i < 9; ++i) dG[i] = 0.0;
  for (int p = blockIdx.x; p < a.n; p += gridDim.x) {
    if (threadIdx.x < 9) s_R[threadIdx.x] = a.Rt[(size_t)p * 9 + threadIdx.x];
    __syncthreads();
    double R[9];
#pragma unroll
    for (int i = 0; i < 9; ++i) R[i] = s_R[i];
    double dR[9];
#pragma unroll
    for (int i = 0; i < 9; ++i) dR[i] = 0.0;
    const int ns = a.gcount[p];
    const float4 *gs = a.gsum + (size_t)p * a.slots;
    const int *idx = a.idx + (size_t)p * a.cap;
    const float4 *spots = a.spots + (size_t)p * a.cap;
    for (int q = threadIdx.x; q < ns; q += kChainThreads) {
      const float4 v = gs[q];
      const int j = __float_as_int(v.w);
      spot_chain(a, s_cc, R, idx[j], spots[j].w, v.x, v.y, v.z, dR, dG);
    }
#pragma unroll
    for (int i = 0; i < 9; ++i) dR[i] = wave_sum_d(dR[i]);
    if (lane == 0) {
#pragma unroll
      for (int i = 0; i < 9; ++i) s_part[wid][i] = dR[i];
    }
    __syncthreads();
    if (threadIdx.x < 9) {
      double v = 0.0;
      for (int w = 0; w < kChainWaves; ++w) v += s_part[w][threadIdx.x];
      a.dRt[(size_t)p * 9 + threadIdx.x] = v;
    }
    __syncthreads();  // s_R and s_part are rewritten for the next pattern
  }
  if (!a.drec) return;  // uniform
  // this block's partial dL/drec (summed in a fixed order by sum_partials_kernel)
#pragma unroll
  for (int i = 0; i < 9; ++i) dG[i] = wave_sum_d(dG[i]);
  if (lane == 0) {
#pragma unroll
    for (int i = 0; i < 9; ++i) s_part[wid][i] = dG[i];
  }
  __syncthreads();
  if (threadIdx.x < 9) {
    double v = 0.0;
    for (int w = 0; w < kChainWaves; ++w) v += s_part[w][threadIdx.x];
    a.dpart[(size_t)blockIdx.x * 9 + threadIdx.x] = v;
  }
}

// drec[i] += sum over blocks of part[b][i]; one wave per entry.
__global__ __launch_bounds__(9 * kWave) void sum_partials_kernel(const double *part, int nb,
                                                                 double *drec) {
  const int i = threadIdx.x / kWave, lane = lane_id();
  double v = 0.0;
  for (int b = lane; b < nb; b += kWave) v += part[(size_t)b * 9 + i];
  v = wave_sum_d(v);
  if (lane == 0) drec[i] += v;
}

// ---------------------------------------------------------------------------
// structure factor adjoint
// ---------------------------------------------------------------------------

constexpr int kSfaThreads = 256;
constexpr int kSfaWaves = kSfaThreads / kWave;

struct SfAdjArgs {
  const int4 *hkl;
  int n;
  double rec[9];
  const uint4 *xyz_fx;
  const int *elem;
  const float *occ;
  const float *B;
  int n_atoms;
  const double *coeff;
  int n_elem;
  int scatter;
  const float *dF2;
  float *dxyz;
  float *dB;
  double *drec;
};

__device__ __forceinline__ float turns_of(uint32_t uh, uint32_t uk, uint32_t ul, const uint4 &x) {
  const uint32_t t = uh * x.x + uk * x.y + ul * x.z;
  return static_cast<float>(static_cast<int32_t>(t)) * 2.3283064365386963e-10f;
}

__global__ __launch_bounds__(kSfaThreads) void structure_factor_adjoint_kernel(SfAdjArgs a) {
  __shared__ uint4 s_xyz[kSfaThreads];
  __shared__ float s_occ[kSfaThreads];
  __shared__ float s_B[kSfaThreads];
  __shared__ int s_el[kSfaThreads];
  __shared__ float s_g[4][kSfaThreads];  // per-atom sums of the chunk: dx, dy, dz, dB
  __shared__ double s_rec[kSfaWaves][9];

  const int tid = threadIdx.x;
  const int lane = lane_id();
  const int wid = tid / kWave;
  const int i = blockIdx.x * kSfaThreads + tid;
  const bool valid = i < a.n;
  const int4 hkl = valid ? a.hkl[i] : make_int4(0, 0, 0, 0);
  const double w = valid ? static_cast<double>(a.dF2[i]) : 0.0;
  const double hx = hkl.x, hy = hkl.y, hz = hkl.z;
  const double gx = a.rec[0] * hx + a.rec[1] * hy + a.rec[2] * hz;
  const double gy = a.rec[3] * hx + a.rec[4] * hy + a.rec[5] * hz;
  const double gz = a.rec[6] * hx + a.rec[7] * hy + a.rec[8] * hz;
  const double g2 = gx * gx + gy * gy + gz * gz;
  const float mq = -0.25f * static_cast<float>(g2);
  const uint32_t uh = static_cast<uint32_t>(hkl.x), uk = static_cast<uint32_t>(hkl.y),
                 ul = static_cast<uint32_t>(hkl.z);

  // pass 1: F and dF/d(g^2)
  double Fr = 0.0, Fi = 0.0, Qr = 0.0, Qi = 0.0;
  int cur_el = -1;
  double f = 0.0, df = 0.0;
  for (int base = 0; base < a.n_atoms; base += kSfaThreads) {
    __syncthreads();
    const int j = base + tid;
    if (j < a.n_atoms) {
      s_xyz[tid] = a.xyz_fx[j];
      s_occ[tid] = a.occ[j];
      s_B[tid] = a.B[j];
      s_el[tid] = a.elem[j];
    }
    __syncthreads();
    const int m = min(kSfaThreads, a.n_atoms - base);
    for (int jj = 0; jj < m; ++jj) {
      const int el = min(max(s_el[jj], 0), a.n_elem - 1);
      if (el != cur_el) {
        f = atomic_f_grad(a.coeff + 10 * el, g2, a.scatter, df);
        cur_el = el;
      }
      float sn, cs;
      sincospif(2.0f * turns_of(uh, uk, ul, s_xyz[jj]), &sn, &cs);
      const double od = static_cast<double>(s_occ[jj] * expf(mq * s_B[jj]));
      const double amp = f * od;
      // d/dq [f occ exp(-B q/4)] = (f' - f B/4) occ exp(-B q/4)
      const double damp = (df - 0.25 * f * static_cast<double>(s_B[jj])) * od;
      Fr = fma(amp, static_cast<double>(cs), Fr);
      Fi = fma(amp, static_cast<double>(sn), Fi);
      Qr = fma(damp, static_cast<double>(cs), Qr);
      Qi = fma(damp, static_cast<double>(sn), Qi);
    }
  }
  // through |F|^2: dL/dg = 2 g dL/d(g^2), dL/d(g^2) = w 2 Re(conj(F) dF/dq)
  const double dq = w * 2.0 * (Fr * Qr + Fi * Qi);
  const double dgx = 2.0 * gx * dq;
  const double dgy = 2.0 * gy * dq;
  const double dgz = 2.0 * gz * dq;
  double dr[9] = {dgx * hx, dgx * hy, dgx * hz, dgy * hx, dgy * hy, dgy * hz,
                  dgz * hx, dgz * hy, dgz * hz};
#pragma unroll
  for (int t = 0; t < 9; ++t) dr[t] = wave_sum_d(dr[t]);
  if (lane == 0) {
#pragma unroll
    for (int t = 0; t < 9; ++t) s_rec[wid][t] = dr[t];
  }

  // pass 2: per-atom terms, dF2/dx_a = -4 pi h Im(conj(F) t_a),
  // dF2/dB_a = -(g^2/2) Re(conj(F) t_a)
  const bool any = __ballot(w != 0.0) != 0;
  cur_el = -1;
  for (int base = 0; base < a.n_atoms; base += kSfaThreads) {
    __syncthreads();
    const int j = base + tid;
    if (j < a.n_atoms) {
      s_xyz[tid] = a.xyz_fx[j];
      s_occ[tid] = a.occ[j];
      s_B[tid] = a.B[j];
      s_el[tid] = a.elem[j];
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) s_g[c][tid] = 0.0f;
    __syncthreads();
    const int m = min(kSfaThreads, a.n_atoms - base);
    if (any) {
      for (int jj = 0; jj < m; ++jj) {
        const int el = min(max(s_el[jj], 0), a.n_elem - 1);
        if (el != cur_el) {
          f = atomic_f(a.coeff + 10 * el, g2, a.scatter);
          cur_el = el;
        }
        float sn, cs;
        sincospif(2.0f * turns_of(uh, uk, ul, s_xyz[jj]), &sn, &cs);
        const double amp = f * static_cast<double>(s_occ[jj] * expf(mq * s_B[jj]));
        const double tr = amp * cs, ti = amp * sn;
        const double im = Fr * ti - Fi * tr;
        const double re = Fr * tr + Fi * ti;
        const float ci = static_cast<float>(-4.0 * M_PI * w * im);
        float vx = ci * static_cast<float>(hx), vy = ci * static_cast<float>(hy),
              vz = ci * static_cast<float>(hz);
        float vb = static_cast<float>(-0.5 * g2 * w * re);
        vx = wave_sum_f(vx);
        vy = wave_sum_f(vy);
        vz = wave_sum_f(vz);
        vb = wave_sum_f(vb);
        if (lane == 0) {
          atomicAdd(&s_g[0][jj], vx);
          atomicAdd(&s_g[1][jj], vy);
          atomicAdd(&s_g[2][jj], vz);
          atomicAdd(&s_g[3][jj], vb);
        }
      }
    }
    __syncthreads();
    if (tid < m) {
      const int atom = base + tid;
      if (s_g[0][tid] != 0.0f) unsafeAtomicAdd(&a.dxyz[3 * atom + 0], s_g[0][tid]);
      if (s_g[1][tid] != 0.0f) unsafeAtomicAdd(&a.dxyz[3 * atom + 1], s_g[1][tid]);
      if (s_g[2][tid] != 0.0f) unsafeAtomicAdd(&a.dxyz[3 * atom + 2], s_g[2][tid]);
      if (s_g[3][tid] != 0.0f) unsafeAtomicAdd(&a.dB[atom], s_g[3][tid]);
    }
  }
  __syncthreads();
  if (tid < 9) {
    double v = 0.0;
    for (int ww = 0; ww < kSfaWaves; ++ww) v += s_rec[ww][tid];
    if (v != 0.0) unsafeAtomicAdd(&a.drec[tid], v);
  }
}

// The same with a lane per atom (dsx_sf.h): runs of 4 rows.  Pass 1 forms F
// and dF/dq of the run's rows, pass 2 adds every atom's terms in its own lane.
// 1.56 million reflections of the 500-atom cell: 4.39 ms with a thread per
// reflection (whose per-atom sums cross the wave 24 times), 2.56 here, VALU busy
// 90 % (five of its registers are in scratch at 128).
constexpr int kSfaRun = 4;

// FP32 sums of the blocks meet in float atomics, whose rounding grows with the
// number of blocks: with 64 rows a block the gradients' error was 1.1 to 2 times
// that of the thread-per-reflection kernel (256 rows a block) up to 64 k rows.
// 60,000 rows x 48 atoms: 2.9e-7 of the norm there, 5.1e-7 with 64 rows and 2.9e-7
// with 256, as many waves as the block's LDS holds; 84 -> 44 us, 17,332 x 48 35 -> 29.
// Small tables take fewer rows, where the error stays below that kernel's and
// more CUs work: 4,614 x 24 1.35e-7 with a thread per reflection; 1.12e-7 with 256
// rows in 25.5 us, 1.25e-7 with 192 in 21.7, 1.40e-7 with 128 in 18.7; 3,000 x 24
// 1.38e-7; 1.11e-7, 1.13e-7 and 1.22e-7; 8,000 x 24 1.60e-7; 1.38e-7, 1.49e-7, 1.64e-7.
static int sfa_atom_rows(int n) { return n <= 4096 ? 128 : n <= 8192 ? 192 : 256; }

template <int kWaves>
__global__ __launch_bounds__(kWaves *kWave, 4) void structure_factor_adjoint_atoms_kernel(SfAdjArgs a,
                                                                                          int rows) {
  // the atoms | their sums [4][n_atoms] | per wave: f and df/dq [n_elem][kAtomRows + 1]
  extern __shared__ double s_dyn[];
  __shared__ int4 s_hkl[kWaves][kAtomRows];
  __shared__ double s_g2[kWaves][kAtomRows], s_w[kWaves][kAtomRows];
  __shared__ double s_F[kWaves][kSfaRun][4];  // of the run: Fr, Fi, then w Fr, w Fi
  __shared__ double s_rec[kWaves][9];
  const int tid = threadIdx.x, lane = lane_id(), wid = tid / kWave;
  const AtomTable tab = atom_table(s_dyn, a.n_atoms);
  double *s_g = s_dyn + atom_table_doubles(a.n_atoms);
  double *s_f = s_g + 4 * a.n_atoms + wid * 2 * a.n_elem * (kAtomRows + 1);
  double *s_df = s_f + a.n_elem * (kAtomRows + 1);
  stage_atoms(a, tab);
  for (int i = tid; i < 4 * a.n_atoms; i += kWaves * kWave) s_g[i] = 0.0;
  __syncthreads();
  double dr[9];  // lanes below kSfaRun: dL/drec over their rows
#pragma unroll
  for (int i = 0; i < 9; ++i) dr[i] = 0.0;
  const int end = min(a.n, (static_cast<int>(blockIdx.x) + 1) * rows);
  for (int r0 = blockIdx.x * rows + wid * kAtomRows; r0 < end; r0 += kWaves * kAtomRows) {
    int4 h = make_int4(0, 0, 0, 0);
    bool anew = true;
    double w = 0.0;
    if (lane < kAtomRows) {
      const int i = r0 + lane;
      if (i < a.n) {
        h = a.hkl[i];
        w = static_cast<double>(a.dF2[i]);
        if (lane % kSfaRun > 0) anew = !line_goes_on(a.hkl[i - 1], h);
      }
      const double gx = a.rec[0] * h.x + a.rec[1] * h.y + a.rec[2] * h.z;
      const double gy = a.rec[3] * h.x + a.rec[4] * h.y + a.rec[5] * h.z;
      const double gz = a.rec[6] * h.x + a.rec[7] * h.y + a.rec[8] * h.z;
      s_hkl[wid][lane] = h;
      s_g2[wid][lane] = gx * gx + gy * gy + gz * gz;
      s_w[wid][lane] = w;
    }
    const unsigned fresh = static_cast<unsigned>(__ballot(anew));
    const unsigned used = static_cast<unsigned>(__ballot(w != 0.0));
    if (used == 0) continue;  // nothing reaches these rows
    atom_wave_sync();
    for (int q = lane; q < kAtomRows * a.n_elem; q += kWave) {
      const int el = q / kAtomRows, r = q - el * kAtomRows;
      double df;
      s_f[el * (kAtomRows + 1) + r] = atomic_f_grad(a.coeff + 10 * el, s_g2[wid][r], a.scatter, df);
      s_df[el * (kAtomRows + 1) + r] = df;
    }
    atom_wave_sync();
#pragma unroll 1
    for (int b = 0; b < kAtomRows; b += kSfaRun) {
      if (((used >> b) & ((1u << kSfaRun) - 1)) == 0) continue;  // uniform
      // ---- pass 1: F and Q = dF/d(g^2) of the run's rows --------------------
      double v[4 * kSfaRun];
#pragma unroll
      for (int k = 0; k < 4 * kSfaRun; ++k) v[k] = 0.0;
#pragma unroll 1
      for (int a0 = 0; a0 < a.n_atoms; a0 += kWave) {
        AtomLane t = load_atom(tab, a0 + lane, a.n_atoms);
        const double *f = s_f + t.el * (kAtomRows + 1) + b, *df = s_df + t.el * (kAtomRows + 1) + b;
        const double b4 = 0.25 * static_cast<double>(t.B);
#pragma unroll
        for (int r = 0; r < kSfaRun; ++r) {
          row_phase<false>(t, (fresh >> (b + r)) & 1, s_hkl[wid][b + r]);
          const float mq = -0.25f * static_cast<float>(s_g2[wid][b + r]);
          const double od = static_cast<double>(t.occ * expf(mq * t.B));
          const double amp = f[r] * od;
          const double damp = fma(-b4, f[r], df[r]) * od;  // d/dq [f occ exp(-B q/4)]
          v[4 * r] = fma(amp, t.c, v[4 * r]);
          v[4 * r + 1] = fma(amp, t.s, v[4 * r + 1]);
          v[4 * r + 2] = fma(damp, t.c, v[4 * r + 2]);
          v[4 * r + 3] = fma(damp, t.s, v[4 * r + 3]);
        }
      }
      const double mine = fold(v, lane);  // lane 4 r + {0, 1, 2, 3}: Fr, Fi, Qr, Qi of row r
      if (lane < 4 * kSfaRun) s_F[wid][lane >> 2][lane & 3] = mine;
      atom_wave_sync();
      if (lane < kSfaRun) {
        const double Fr = s_F[wid][lane][0], Fi = s_F[wid][lane][1];
        const double wr = s_w[wid][b + lane];
        const int4 hr = s_hkl[wid][b + lane];
        const double gx = a.rec[0] * hr.x + a.rec[1] * hr.y + a.rec[2] * hr.z;
        const double gy = a.rec[3] * hr.x + a.rec[4] * hr.y + a.rec[5] * hr.z;
        const double gz = a.rec[6] * hr.x + a.rec[7] * hr.y + a.rec[8] * hr.z;
        // through |F|^2: dL/dg = 2 g dL/d(g^2), dL/d(g^2) = w 2 Re(conj(F) dF/dq)
        const double dq = wr * 2.0 * (Fr * s_F[wid][lane][2] + Fi * s_F[wid][lane][3]);
        const double dx = 2.0 * gx * dq, dy = 2.0 * gy * dq, dz = 2.0 * gz * dq;
        dr[0] += dx * hr.x; dr[1] += dx * hr.y; dr[2] += dx * hr.z;
        dr[3] += dy * hr.x; dr[4] += dy * hr.y; dr[5] += dy * hr.z;
        dr[6] += dz * hr.x; dr[7] += dz * hr.y; dr[8] += dz * hr.z;
        s_F[wid][lane][2] = wr * Fr;
        s_F[wid][lane][3] = wr * Fi;
      }
      atom_wave_sync();
      // ---- pass 2: dF2/dx_a = -4 pi h Im(conj(F) t_a), dF2/dB_a = -(g^2/2) Re(conj(F) t_a)
#pragma unroll 1
      for (int a0 = 0; a0 < a.n_atoms; a0 += kWave) {
        AtomLane t = load_atom(tab, a0 + lane, a.n_atoms);
        const double *f = s_f + t.el * (kAtomRows + 1) + b;
        double sx = 0.0, sy = 0.0, sz = 0.0, sb = 0.0;
#pragma unroll
        for (int r = 0; r < kSfaRun; ++r) {
          const int4 hr = s_hkl[wid][b + r];
          row_phase<false>(t, (fresh >> (b + r)) & 1, hr);
          const double g2r = s_g2[wid][b + r];
          const double amp = f[r] * static_cast<double>(t.occ * expf(-0.25f * static_cast<float>(g2r) * t.B));
          const double wr = s_F[wid][r][2], wi = s_F[wid][r][3];
          const double im = amp * fma(wr, t.s, -(wi * t.c));
          const double re = amp * fma(wr, t.c, wi * t.s);
          sx = fma(im, static_cast<double>(hr.x), sx);
          sy = fma(im, static_cast<double>(hr.y), sy);
          sz = fma(im, static_cast<double>(hr.z), sz);
          sb = fma(re, g2r, sb);
        }
        if (a0 + lane < a.n_atoms) {  // the block's waves share the sums
          unsafeAtomicAdd(&s_g[a0 + lane], sx);
          unsafeAtomicAdd(&s_g[a.n_atoms + a0 + lane], sy);
          unsafeAtomicAdd(&s_g[2 * a.n_atoms + a0 + lane], sz);
          unsafeAtomicAdd(&s_g[3 * a.n_atoms + a0 + lane], sb);
        }
      }
      atom_wave_sync();  // the next run overwrites s_F
    }
  }
#pragma unroll
  for (int i = 0; i < 9; ++i) dr[i] = wave_sum_d(dr[i]);
  if (lane == 0) {
#pragma unroll
    for (int i = 0; i < 9; ++i) s_rec[wid][i] = dr[i];
  }
  __syncthreads();
  for (int i = tid; i < a.n_atoms; i += kWaves * kWave) {
    const float v[3] = {static_cast<float>(-4.0 * M_PI * s_g[i]),
                        static_cast<float>(-4.0 * M_PI * s_g[a.n_atoms + i]),
                        static_cast<float>(-4.0 * M_PI * s_g[2 * a.n_atoms + i])};
#pragma unroll
    for (int k = 0; k < 3; ++k)
      if (v[k] != 0.0f) unsafeAtomicAdd(&a.dxyz[3 * i + k], v[k]);
    const float vb = static_cast<float>(-0.5 * s_g[3 * a.n_atoms + i]);
    if (vb != 0.0f) unsafeAtomicAdd(&a.dB[i], vb);
  }
  if (tid < 9) {
    double v = 0.0;
    for (int ww = 0; ww < kWaves; ++ww) v += s_rec[ww][tid];
    if (v != 0.0) unsafeAtomicAdd(&a.drec[tid], v);
  }
}

// Dynamic LDS of the kernel with this many waves, and whether it fits beside the static part.
static size_t sfa_atoms_lds(int n_atoms, int n_elem, int waves) {
  return 8 * (static_cast<size_t>(atom_table_doubles(n_atoms)) + 4 * n_atoms +
              2 * static_cast<size_t>(waves) * n_elem * (kAtomRows + 1));
}

static bool sfa_atoms_fit(int n_atoms, int n_elem, int waves) {
  return sfa_atoms_lds(n_atoms, n_elem, waves) + 712 * static_cast<size_t>(waves) <= 64 * 1024;
}

template <int kWaves>
static void launch_sfa_atoms(const SfAdjArgs &a, hipStream_t s) {
  const int rows = atom_rows_per_block(a.n, kWaves, sfa_atom_rows(a.n));
  hipLaunchKernelGGL(structure_factor_adjoint_atoms_kernel<kWaves>, dim3((a.n + rows - 1) / rows),
                     dim3(kWaves * kWave), sfa_atoms_lds(a.n_atoms, a.n_elem, kWaves), s, a, rows);
}

}  // namespace dsx

using namespace dsx;

// Workspace of the long lists' kernel, per block: large_block_ints(cap, H W)
// ints, filled with the first row of every 64 listed spots and as many entries'
// records and rows as the rest holds (dsx_tiles.h): at least one tile's, and with
// a pattern's pixels besides enough for wide boxes to be taken in few ranges;
// with gradients the chain-rule hand-over follows the
// blocks.  Chain-rule hand-over (the small-pattern kernel's whole workspace):
// float4 gsum[n * cap] | int gcount[n] | (8-byte aligned) double
// dpart[chain blocks][9].
constexpr int kWorkEntriesPerSpot = 4;
constexpr int kAdjLdsBytes = 160 * 1024;

static bool adjoint_large(int cap) { return cap > kAdjMaxSpots; }
static int chain_blocks_max() { return cu_count() * 8; }
static long long small_work_ints(int cap, int n) {
  return 4ll * n * cap + n + 1 + 18ll * chain_blocks_max();
}
static long long large_block_ints(int cap, long long hw) {
  const long long e = kWorkEntriesPerSpot * static_cast<long long>(cap);
  return ((e + 3) & ~3ll) + ((2ll * cap + 3) & ~3ll) + ((cap + 3ll) & ~3ll) + ((hw + 3) & ~3ll);
}
// blocks of the long lists' kernel: two per CU
static int large_blocks(int n) { return std::min(n, 2 * cu_count()); }

extern "C" long long dsx_render_adjoint_workspace_ints(int cap, int n, int height, int width,
                                                       int gradients) {
  if (cap < 1 || n < 0 || height < 1 || width < 1) return 0;
  if (adjoint_large(cap))
    return static_cast<long long>(large_blocks(n)) *
               large_block_ints(cap, static_cast<long long>(height) * width) +
           (gradients ? small_work_ints(cap, n) : 0);
  return small_work_ints(cap, n);
}

// Static LDS of a kernel (queried once) and its dynamic LDS limit raised to
// what is left of the CU's 160 KB.
static int adjoint_static_lds(const void *kernel, int *cache, int *raised) {
  if (*cache < 0) {
    hipFuncAttributes attr;
    if (hipFuncGetAttributes(&attr, kernel) != hipSuccess) {
      (void)hipGetLastError();
      return -1;
    }
    *cache = static_cast<int>(attr.sharedSizeBytes);
  }
  if (!*raised) {
    if (hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                            kAdjLdsBytes - *cache) != hipSuccess) {
      (void)hipGetLastError();
      return -1;
    }
    *raised = 1;
  }
  return *cache;
}

// Chain rule of the gathered sums (rows of `slots` entries).
static int launch_chain(const AdjArgs &a, hipStream_t s) {
  const int cblocks = std::min(a.n, chain_blocks_max());
  hipLaunchKernelGGL(spot_chain_kernel, dim3(cblocks), dim3(kChainThreads), 0, s, a);
  if (a.drec)
    hipLaunchKernelGGL(sum_partials_kernel, dim3(1), dim3(9 * kWave), 0, s, a.dpart, cblocks, a.drec);
  return check_launch("dsx_render_adjoint (chain)");
}

// Long lists: two blocks per CU (one when the tiles' LDS needs it), each with
// its part of the workspace.
static int launch_tiles(AdjArgs &a, int *work_d, long long work_ints, hipStream_t s) {
  const bool fwd = a.mode == DSX_ADJ_FORWARD;
  const long long n_tiles = static_cast<long long>((a.W + kTileEdge - 1) / kTileEdge) *
                            ((a.H + kTileEdge - 1) / kTileEdge);
  // counters of as many waves as leave room for two blocks per CU
  a.count_waves = 8;
  while (a.count_waves > 1 && 4 * (a.count_waves + 1) * n_tiles > 64 * 1024) a.count_waves /= 2;
  const long long lds = (4 * (a.count_waves + 1) * n_tiles + 15) & ~15ll;
  static int static_grad = -1, static_fwd = -1, raised_grad = 0, raised_fwd = 0;
  const int st = fwd ? adjoint_static_lds(reinterpret_cast<const void *>(&render_tiles_fwd_kernel),
                                          &static_fwd, &raised_fwd)
                     : adjoint_static_lds(reinterpret_cast<const void *>(&render_tiles_kernel),
                                          &static_grad, &raised_grad);
  if (st < 0) {
    set_error("dsx_render_adjoint: cannot query or reserve the kernel's LDS");
    return DSX_ELAUNCH;
  }
  if (st + lds > kAdjLdsBytes) {
    set_error("dsx_render_adjoint: %lld tiles of a %dx%d pattern exceed the LDS", n_tiles, a.H, a.W);
    return DSX_EINVAL;
  }
  // The shapes that are taken: 256 strips of 8,192 pixels (16,384 for rows above
  // 8,192).  With sides of at most 32,767 and 2^22 pixels that is at most 16,384
  // tiles, whose counters always fit above.
  const int strip_rows = std::min(a.H, (a.W <= 8192 ? 8192 : 16384) / a.W);
  if (strip_rows < 1 || (a.H + strip_rows - 1) / strip_rows > kAdjMaxStrips) {
    set_error("dsx_render_adjoint: a %dx%d pattern exceeds the sides taken", a.H, a.W);
    return DSX_EINVAL;
  }
  const int blocks = large_blocks(a.n);
  const long long per_block = large_block_ints(a.cap, static_cast<long long>(a.H) * a.W);
  const long long need = per_block * blocks + (a.want_grad ? small_work_ints(a.cap, a.n) : 0);
  if (work_d ? work_ints < need || reinterpret_cast<uintptr_t>(work_d) % 16 != 0 : a.want_grad != 0) {
    set_error("dsx_render_adjoint: workspace of %lld ints is smaller than %lld or not 16-byte "
              "aligned (dsx_render_adjoint_workspace_ints)", work_d ? work_ints : 0ll, need);
    return DSX_EINVAL;
  }
  a.work = work_d;
  a.work_per_block = per_block;
  // records and rows fill a block's part after the first rows per 64 listed spots
  const long long entries = (per_block - (a.cap + kWave - 1) / kWave) / kRecInts;
  a.work_entries = static_cast<int>(std::min<long long>(entries, 1ll << 28));
  if (a.want_grad) {
    int *hand = work_d + per_block * blocks;  // a multiple of 4 ints: 16-byte aligned
    a.gsum = reinterpret_cast<float4 *>(hand);
    a.gcount = hand + static_cast<size_t>(a.n) * 4 * a.cap;
    const size_t off = (static_cast<size_t>(a.n) * (4ull * a.cap + 1) + 1) & ~static_cast<size_t>(1);
    a.dpart = reinterpret_cast<double *>(hand + off);
  }
  if (fwd)
    hipLaunchKernelGGL(render_tiles_fwd_kernel, dim3(blocks), dim3(kTileThreads), static_cast<size_t>(lds), s, a);
  else
    hipLaunchKernelGGL(render_tiles_kernel, dim3(blocks), dim3(kTileThreads), static_cast<size_t>(lds), s, a);
  const int rc = check_launch("dsx_render_adjoint");
  if (rc != DSX_OK || !a.want_grad) return rc;
  a.slots = a.cap;
  return launch_chain(a, s);
}

extern "C" int dsx_render_adjoint(const int *idx_d, const float *spot_d, const int *count_d, int cap,
                                  int n, const int *hkl_d, const float *F2_d, int n_refl,
                                  const double *Rt_d, const dsx_sim_params *sim,
                                  const dsx_render_params *rp, int mode, const float *target_d,
                                  long long target_stride, float *pattern_d, float *loss_d,
                                  double *dRt_d, float *dF2_d, double *drec_d, int *work_d,
                                  long long work_ints,
                                  int *status_d, void *stream) {
  clear_error();
  if (!sim || !rp || n < 0 || cap < 1 || n_refl < 0 || work_ints < 0 || target_stride < 0) {
    set_error("dsx_render_adjoint: bad arguments (n=%d cap=%d n_refl=%d)", n, cap, n_refl);
    return DSX_EINVAL;
  }
  if (mode != DSX_ADJ_L2 && mode != DSX_ADJ_PATTERN_GRAD && mode != DSX_ADJ_FORWARD) {
    set_error("dsx_render_adjoint: unknown mode %d", mode);
    return DSX_EINVAL;
  }
  if (n == 0) return DSX_OK;
  const bool want_grad = dRt_d != nullptr;
  if (!want_grad && (dF2_d || drec_d)) {
    set_error("dsx_render_adjoint: dF2_d and drec_d need dRt_d");
    return DSX_EINVAL;
  }
  if (mode == DSX_ADJ_FORWARD && (want_grad || !pattern_d)) {
    set_error("dsx_render_adjoint: forward mode writes patterns and no gradients");
    return DSX_EINVAL;
  }
  if (!spot_d || !count_d || (mode != DSX_ADJ_FORWARD && !target_d) ||
      (want_grad && (!idx_d || !Rt_d)) || (want_grad && n_refl > 0 && (!hkl_d || !F2_d))) {
    set_error("dsx_render_adjoint: null device pointer");
    return DSX_EINVAL;
  }
  if (rp->height < 1 || rp->width < 1 || rp->height > 32767 || rp->width > 32767 ||
      static_cast<long long>(rp->height) * rp->width > (1ll << kPixBits) ||
      !(rp->calibration > 0.0f) || !(rp->sigma > 0.0f) || !(rp->clip_threshold > 0.0f)) {
    set_error("dsx_render_adjoint: bad pattern shape %dx%d (at most 2^22 pixels), calibration, "
              "sigma or clip_threshold", rp->height, rp->width);
    return DSX_EINVAL;
  }
  if (sim->shape_model < DSX_SF_LINEAR || sim->shape_model > DSX_SF_LORENTZIAN_PRECESSION ||
      !(sim->k > 0.0) || sim->shape_width == 0.0) {
    set_error("dsx_render_adjoint: bad physical parameters");
    return DSX_EINVAL;
  }
  AdjArgs a;
  a.idx = idx_d;
  a.spots = reinterpret_cast<const float4 *>(spot_d);
  a.count = count_d;
  a.cap = cap;
  a.n = n;
  a.hkl = reinterpret_cast<const int4 *>(hkl_d);
  a.F2 = F2_d;
  a.n_refl = n_refl;
  a.Rt = Rt_d;
  for (int i = 0; i < 9; ++i) a.rec[i] = sim->rec[i];
  fill_physics(a, sim);
  a.H = rp->height;
  a.W = rp->width;
  a.cal = rp->calibration;
  a.cx = rp->center_x;
  a.cy = rp->center_y;
  a.ca = rp->cos_angle;
  a.sa = rp->sin_angle;
  a.mirrored = rp->mirrored;
  a.normalize = rp->normalize;
  const double sg = rp->sigma;
  a.pref = static_cast<float>(1.0 / (2.0 * M_PI * sg * sg));
  a.ep = static_cast<float>(-1.0 / (2.0 * sg * sg));
  a.inv_s2 = static_cast<float>(1.0 / (sg * sg));
  a.e2ep = static_cast<float>(exp(-1.0 / (sg * sg)));
  a.clip = rp->clip_threshold;
  a.log2_clip = static_cast<float>(log2(static_cast<double>(rp->clip_threshold)));
  a.two_s2_ln2 = static_cast<float>(2.0 * sg * sg * M_LN2);
  a.tiny_box = static_cast<float>(0.04 * sg * sg);
  a.box_margin = static_cast<float>(2e-4 * std::max(1.0, sg) + 1e-6 * std::max(rp->height, rp->width));
  // every spot of the list on one tile stays below 2^31 units
  a.bound_units = static_cast<float>((1 << 30) / std::max(cap, 1024));
  a.mode = mode;
  a.want_grad = want_grad ? 1 : 0;
  a.target = target_d;
  a.target_stride = target_stride;
  a.pattern = pattern_d;
  a.loss = loss_d;
  a.dRt = dRt_d;
  a.dF2 = dF2_d;
  a.drec = drec_d;
  a.dpart = nullptr;
  a.status = status_d;
  a.work = nullptr;
  a.work_per_block = 0;
  a.work_entries = 0;
  a.gsum = nullptr;
  a.gcount = nullptr;

  if (adjoint_large(cap)) return launch_tiles(a, work_d, work_ints, as_stream(stream));

  // LDS per block: the static part, the spot table (slots entries; bins) and
  // two strip buffers of rows x W words; two blocks per CU when their strips
  // hold at least 8 rows (or the whole pattern).
  static int static_small = -1, raised_small = 0;
  const int st = adjoint_static_lds(reinterpret_cast<const void *>(&render_adjoint_kernel), &static_small,
                                    &raised_small);
  if (st < 0) {
    set_error("dsx_render_adjoint: cannot query or reserve the kernel's LDS");
    return DSX_ELAUNCH;
  }
  int bpc = 2;
  a.slots = cap;
  a.bin_cap = std::min(kAdjBinCap, 4 * cap + 256);
  const long long table = static_cast<long long>(kSpotTabBytes) * a.slots + 2ll * a.bin_cap + 16;
  auto rows_for = [&](int per_block) {
    const long long strip = std::min<long long>(kAdjSmallStripBytes, per_block - st - table);
    return strip < 8ll * a.W ? 0 : static_cast<int>(std::min<long long>(a.H, strip / (8ll * a.W)));
  };
  int rows = rows_for(kAdjLdsBytes / bpc);
  if (rows < std::min(a.H, 8)) {
    bpc = 1;
    rows = rows_for(kAdjLdsBytes);
  }
  if (rows < 1) {
    set_error("dsx_render_adjoint: pattern width %d exceeds the LDS strip budget", a.W);
    return DSX_EINVAL;
  }
  const int n_strips = (a.H + rows - 1) / rows;
  if (n_strips > kAdjMaxStrips) {
    set_error("dsx_render_adjoint: pattern height %d needs %d strips (> %d)", a.H, n_strips,
              kAdjMaxStrips);
    return DSX_EINVAL;
  }
  a.strip_rows = rows;
  a.n_strips = n_strips;
  a.acc_words = rows * a.W;
  const int blocks = std::min(n, cu_count() * bpc);
  if (want_grad) {
    const long long need = small_work_ints(cap, n);
    if (!work_d || work_ints < need) {
      set_error("dsx_render_adjoint: gradients need a workspace of %lld ints, got %lld "
                "(dsx_render_adjoint_workspace_ints)", need, work_d ? work_ints : 0ll);
      return DSX_EINVAL;
    }
    if (reinterpret_cast<uintptr_t>(work_d) % 16 != 0) {
      set_error("dsx_render_adjoint: workspace must be 16-byte aligned");
      return DSX_EINVAL;
    }
    a.gsum = reinterpret_cast<float4 *>(work_d);
    a.gcount = work_d + static_cast<size_t>(n) * 4 * cap;
    const size_t off = (static_cast<size_t>(n) * (4ull * cap + 1) + 1) & ~static_cast<size_t>(1);
    a.dpart = reinterpret_cast<double *>(work_d + off);
  }
  const size_t lds = (2ull * a.acc_words * 4 + static_cast<size_t>(table) + 15) & ~static_cast<size_t>(15);
  hipStream_t s = as_stream(stream);
  hipLaunchKernelGGL(render_adjoint_kernel, dim3(blocks), dim3(kAdjThreads), lds, s, a);
  const int rc = check_launch("dsx_render_adjoint");
  if (rc != DSX_OK || !want_grad) return rc;
  return launch_chain(a, s);
}

// ---------------------------------------------------------------------------
// Allocation-free form of dsx_render_adjoint: the workspace is a file-scope
// device array (one copy per GPU, held until the process ends).  Host code
// never passes the array's name to a kernel (on the host it is only a
// stand-in); its device address is looked up once per device with
// hipGetSymbolAddress and kept here.
// ---------------------------------------------------------------------------

constexpr long long kNoallocScratchInts = 16ll << 20;  // 64 MiB
static __device__ __align__(256) int scratch[kNoallocScratchInts];

static std::mutex g_scratch_mu;
static int *g_scratch_ptr[64] = {};

// Device address of this device's scratch (looked up on the first call).
static int scratch_address(int **out) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) {
    (void)hipGetLastError();
    set_error("dsx_render_adjoint_noalloc: no current device (or device id >= 64)");
    return DSX_ELAUNCH;
  }
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void *ptr = nullptr;
    const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr) {
      (void)hipGetLastError();
      set_error("dsx_render_adjoint_noalloc: hipGetSymbolAddress(scratch) failed: %s",
                hipGetErrorString(e));
      return DSX_ELAUNCH;
    }
    g_scratch_ptr[dev] = static_cast<int *>(ptr);
  }
  *out = g_scratch_ptr[dev];
  return DSX_OK;
}

extern "C" long long dsx_render_adjoint_noalloc_max_ints(void) { return kNoallocScratchInts; }

extern "C" int dsx_render_adjoint_noalloc(const int *idx_d, const float *spot_d, const int *count_d,
                                          int cap, int n, const int *hkl_d, const float *F2_d,
                                          int n_refl, const double *Rt_d, const dsx_sim_params *sim,
                                          const dsx_render_params *rp, int mode,
                                          const float *target_d, long long target_stride,
                                          float *pattern_d, float *loss_d, double *dRt_d,
                                          float *dF2_d, double *drec_d, int *status_d,
                                          void *stream) {
  clear_error();
  if (cap < 1 || n < 0 || !rp) {
    set_error("dsx_render_adjoint_noalloc: bad arguments (n=%d cap=%d)", n, cap);
    return DSX_EINVAL;
  }
  const long long need =
      dsx_render_adjoint_workspace_ints(cap, n, rp->height, rp->width, dRt_d != nullptr);
  if (need > kNoallocScratchInts) {
    set_error("dsx_render_adjoint_noalloc: %d patterns with capacity %d need %lld ints of "
              "scratch; the static scratch holds %lld (use dsx_render_adjoint with a workspace, "
              "or fewer patterns per call)", n, cap, need, kNoallocScratchInts);
    return DSX_EINVAL;
  }
  int *work = nullptr;
  const int rc = scratch_address(&work);
  if (rc != DSX_OK) return rc;
  return dsx_render_adjoint(idx_d, spot_d, count_d, cap, n, hkl_d, F2_d, n_refl, Rt_d, sim, rp, mode,
                            target_d, target_stride, pattern_d, loss_d, dRt_d, dF2_d, drec_d, work,
                            kNoallocScratchInts, status_d, stream);
}

extern "C" int dsx_structure_factor_adjoint(const int *hkl_d, int n, const double rec[9],
                                            const uint32_t *xyz_fx_d, const int *elem_d,
                                            const float *occ_d, const float *B_d, int n_atoms,
                                            const double *coeff_d, int n_elem, int scatter,
                                            const float *dF2_d, float *dxyz_d, float *dB_d,
                                            double *drec_d, void *stream) {
  clear_error();
  if (n < 0 || n_atoms < 0 || n_elem < 0 || !rec) {
    set_error("dsx_structure_factor_adjoint: bad sizes n=%d n_atoms=%d n_elem=%d", n, n_atoms, n_elem);
    return DSX_EINVAL;
  }
  if (scatter != DSX_SCATTER_NONE && scatter != DSX_SCATTER_LOBATO && scatter != DSX_SCATTER_XTABLES) {
    set_error("dsx_structure_factor_adjoint: unknown scattering parameterisation %d", scatter);
    return DSX_EINVAL;
  }
  if (n == 0) return DSX_OK;
  if (n_atoms > 0 && n_elem == 0) {
    set_error("dsx_structure_factor_adjoint: atoms given but no element coefficients");
    return DSX_EINVAL;
  }
  if (!hkl_d || !dF2_d || !drec_d ||
      (n_atoms > 0 && (!xyz_fx_d || !elem_d || !occ_d || !B_d || !dxyz_d || !dB_d)) ||
      (n_elem > 0 && !coeff_d)) {
    set_error("dsx_structure_factor_adjoint: null device pointer");
    return DSX_EINVAL;
  }
  SfAdjArgs a;
  a.hkl = reinterpret_cast<const int4 *>(hkl_d);
  a.n = n;
  for (int i = 0; i < 9; ++i) a.rec[i] = rec[i];
  a.xyz_fx = reinterpret_cast<const uint4 *>(xyz_fx_d);
  a.elem = elem_d;
  a.occ = occ_d;
  a.B = B_d;
  a.n_atoms = n_atoms;
  a.coeff = coeff_d;
  a.n_elem = n_elem;
  a.scatter = scatter;
  a.dF2 = dF2_d;
  a.dxyz = dxyz_d;
  a.dB = dB_d;
  a.drec = drec_d;
  if (atoms_per_lane_adjoint(n, n_atoms, n_elem)) {
    const int waves = sfa_atom_rows(n) / kAtomRows;  // 8, 12 or 16: a turn of the block's rows
    if (waves >= 16 && sfa_atoms_fit(n_atoms, n_elem, 16))
      launch_sfa_atoms<16>(a, as_stream(stream));
    else if (waves >= 12 && sfa_atoms_fit(n_atoms, n_elem, 12))
      launch_sfa_atoms<12>(a, as_stream(stream));
    else if (sfa_atoms_fit(n_atoms, n_elem, 8))
      launch_sfa_atoms<8>(a, as_stream(stream));
    else
      launch_sfa_atoms<4>(a, as_stream(stream));
  } else {
    hipLaunchKernelGGL(structure_factor_adjoint_kernel, dim3((n + kSfaThreads - 1) / kSfaThreads),
                       dim3(kSfaThreads), 0, as_stream(stream), a);
  }
  return check_launch("dsx_structure_factor_adjoint");
}
