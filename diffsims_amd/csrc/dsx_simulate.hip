// (b) Persistent per-orientation kernel: rotate g, excitation error against the
// Ewald sphere, shape factor, intensity, relative cut, ordered compaction.
//
// Follows calculate_diffraction2d's orientation loop and
// get_intersecting_reflections (diffsims/generators/simulation_generator.py:
// 211-241, :319-412) and the models of diffsims/utils/shape_factor_models.py.
//
// Mapping: one wave64 owns a tile of kOT orientations; its lanes sweep the
// reflection table 64 rows at a time.  A cheap rotation-invariant FP32 pretest
// (|g|^2 - 2 k z, one dot product) rejects almost all rows; rows that pass are
// re-evaluated in FP64 from their integer hkl (g = rec hkl, g_lab = R g) with
// the reference's arithmetic made cancellation-free, and survivors are
// appended in reflection order with a wave ballot + mbcnt prefix.  The relative intensity cut needs the maximum over the whole
// intersecting set, so survivors are written first and, only if some fall
// below the cut, re-compacted in place by the same wave.
//
// With a line index (dsx_hkl_lines) the sweep visits only rows that can pass
// the pretest: a row passes only if its beam coordinate z lies in a slab
// [(wmin - thr) / 2k, (wmax + thr) / 2k] (w = |g|^2 over the row's line), and
// along a line z is linear in l, so each line contributes one interval of
// rows per orientation.  The intervals of 64 lines are flattened across the
// wave (prefix sum, per-lane binary search) in row order, so the pretest sees
// exactly the rows it would pass in a full sweep, in the same order, and the
// outputs are identical.
#include <algorithm>

#include "dsx_internal.h"
#include "dsx_physics.h"

namespace dsx {

// Orientations per wave: one 16-byte table load feeds kOT dot products
// (measured on the 40-atom library: 2.25 ms with 4, 2.82 ms with 2, 5.88 ms
// with 8, which spills).
constexpr int kOT = 4;
constexpr int kSlotBits = 2;      // bits of an orientation slot in a queue entry
static_assert((1 << kSlotBits) == kOT, "orientation slot bits");
// one wave per block: the waves share nothing, and single-wave blocks let the
// dispatcher refill a finished wave's slot at once (the library's spot kernel
// 1.46 -> 1.43 ms, the 64-phase batch's 18.5 -> 18.2 ms against four waves)
constexpr int kSimThreads = 64;
// The line sweep pays once lines average this many rows.  Measured with the
// intervals of a group formed for all orientations at once: the 40-atom
// library table (14.6 rows per line) 2.19 ms full sweep against 1.55 ms line
// sweep for 200,000 orientations; thresholds of 6 or 3 gain nothing more on
// the 64-phase ragged batch.
constexpr int kMinLineRows = DSX_LINE_SWEEP_MIN_ROWS;

__host__ __device__ __forceinline__ bool lines_pay(int n_refl, int n_lines) {
  return n_lines > 0 && static_cast<long long>(n_refl) >= static_cast<long long>(kMinLineRows) * n_lines;
}

struct SimArgs {
  double k, k2;
  double me;         // max_excitation_error
  double width;      // shape width
  double sigma;      // pi / width
  double fac;        // pi * minima_number / width (|width| for atanc)
  int model;
  int precession;
  double phi, Pz, Pt;  // precession angle (rad), k cos(phi), k sin(phi)
  double sin_phi;
  float min_I;
  float k_f;
  int n_items;                  // tiles of kOT orientations
  dsx_phase_desc single;        // plain launch: the one phase
  const dsx_phase_desc *phases; // ragged launch: device array of phases
  const int2 *items;            // ragged launch: {phase, first orientation} per tile
};

// Pretest bound: e = |g|^2 - 2 k z = s (2k - z_sphere - z), and |s| <= me
// (+ r sin(phi) with precession); the slack covers FP32 rounding of e.
__host__ __device__ __forceinline__ float pretest_threshold(double me, double k, double gmax,
                                                            double sin_phi) {
  const double me_eff = me + (sin_phi > 0.0 ? 1.1 * gmax * sin_phi : 0.0);
  return static_cast<float>(1.05 * me_eff * (2.0 * k + gmax) + 1e-3 +
                            1e-6 * (2.0 * k * gmax + gmax * gmax));
}

// One candidate in FP64: lab position of row `row` in the orientation Rd, its
// membership and its intensity.  Sums are written as fma chains, so every
// kernel rounds them alike.
template <bool kAvg>
__device__ __forceinline__ bool eval_candidate(const SimArgs &a, const int4 *hkl, const float *F2,
                                               const double *rec, const double *Rd, int row,
                                               float4 &spot) {
  const int4 h = hkl[row];
  const double hx = h.x, hy = h.y, hz = h.z;
  const double gx = fma(rec[2], hz, fma(rec[1], hy, rec[0] * hx));
  const double gy = fma(rec[5], hz, fma(rec[4], hy, rec[3] * hx));
  const double gz = fma(rec[8], hz, fma(rec[7], hy, rec[6] * hx));
  const double x = fma(Rd[2], gz, fma(Rd[1], gy, Rd[0] * gx));
  const double y = fma(Rd[5], gz, fma(Rd[4], gy, Rd[3] * gx));
  const double z = fma(Rd[8], gz, fma(Rd[7], gy, Rd[6] * gx));
  double s, r;
  const bool in = intersects(x, y, z, a, s, r);
  spot = make_float4(static_cast<float>(x), static_cast<float>(y), static_cast<float>(z), 0.0f);
  if (in) spot.w = static_cast<float>(shape_factor<kAvg>(s, r, a) * static_cast<double>(F2[row]));
  return in;
}

// Candidate queue per wave: (reflection row << kSlotBits) | orientation slot, in the
// order the sweep produced them (row-major, so per orientation ascending rows).
// Ring of at least one batch plus one worst-case step (64 + kOT * 64
// entries), a power of two so that positions wrap with a mask: candidates
// are spread thinly over the rows, so nearly every step queues a few for
// every orientation, and a modulo by a non-power of two there cost more
// than the pretest itself.
constexpr int kQueue = 512;
static_assert(kQueue >= 64 + kOT * kWave && (kQueue & (kQueue - 1)) == 0, "queue ring size");
__device__ __forceinline__ int qpos(int i) { return i & (kQueue - 1); }
constexpr int kWavesPerBlock = kSimThreads / kWave;

// Register budgets (waves per SIMD), measured: the full sweep at 5 (96 VGPRs)
// and the line sweep at 4 (128 VGPRs) are 5-6 % faster than the compiler's own
// choice (111 and 151-165 VGPRs) despite a few spilled registers; the
// averaged-precession models keep theirs.
constexpr int sim_min_waves(bool avg, bool lines) { return avg ? 1 : (lines ? 4 : 5); }

template <bool kRagged, bool kAvg, bool kLines>
__global__ __launch_bounds__(kSimThreads, sim_min_waves(kAvg, kLines)) void simulate_kernel(SimArgs a) {
  __shared__ int s_queue[kWavesPerBlock][kQueue];
  __shared__ double s_R[kWavesPerBlock][kOT][9];
  __shared__ double s_abc[kWavesPerBlock][kOT][4];  // beam . (a*, b*, c*), 1 / (beam . c*)
  // FP32 beam rows of the full-sweep pretest: in the line-sweep kernels, which
  // run the full sweep only for short-line phases, they wait in LDS instead
  // of holding 12 VGPRs through the line machinery
  __shared__ float s_Rf[kWavesPerBlock][kOT][3];
  // line sweep: the current group's intervals per orientation and lane
  constexpr int kLO = kLines ? kOT : 1, kLW = kLines ? kWave : 1;
  __shared__ int s_P[kWavesPerBlock][kLO][kLW];
  __shared__ int s_rb[kWavesPerBlock][kLO][kLW];
  __shared__ float s_eA[kWavesPerBlock][kLO][kLW];
  __shared__ float s_eB[kWavesPerBlock][kLO][kLW];
  __shared__ int s_tot[kWavesPerBlock][kLO];
  const int lane = lane_id();
  const int wib = threadIdx.x / kWave;
  int *queue = s_queue[wib];
  const int wave = blockIdx.x * kWavesPerBlock + wib;
  const int n_waves = gridDim.x * kWavesPerBlock;
  const float two_k = 2.0f * a.k_f;

  for (int tile = wave; tile < a.n_items; tile += n_waves) {
    const dsx_phase_desc *d;
    int o0;
    if (kRagged) {
      const int2 it = a.items[tile];
      d = a.phases + it.x;
      o0 = it.y;
    } else {
      d = &a.single;
      o0 = tile * kOT;
    }
    const int n_here = min(kOT, d->n_orient - o0);
    const int4 *hkl = reinterpret_cast<const int4 *>(d->hkl);
    const float4 *g4 = reinterpret_cast<const float4 *>(d->g4);
    const float *F2 = d->F2;
    const double *Rt = d->Rt;
    const double *rec = d->rec;
    const int n_refl = d->n_refl;
    const int cap = d->cap;
    int *idx_out = d->idx;
    float4 *spot_out = reinterpret_cast<float4 *>(d->spots);
    const float pre_thr = pretest_threshold(a.me, a.k, d->g_max, a.sin_phi);
    float R[kLines ? 1 : kOT][3];  // third rows (beam direction) for the FP32 pretest
    int cnt[kOT];
    float lmax[kOT], lmin[kOT];
    for (int e = lane; e < kOT * 9; e += kWave) {
      const int o = e / 9, j = e - o * 9;
      s_R[wib][o][j] = o < n_here ? Rt[(size_t)(o0 + o) * 9 + j] : 0.0;
    }
#pragma unroll
    for (int o = 0; o < kOT; ++o) {
      const bool ok = o < n_here;
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        const float v = ok ? static_cast<float>(Rt[(size_t)(o0 + o) * 9 + 6 + j]) : 0.0f;
        if (kLines)
          s_Rf[wib][o][j] = v;
        else
          R[o][j] = v;
      }
      cnt[o] = 0;
      lmax[o] = 0.0f;
      lmin[o] = __builtin_huge_valf();
    }
    int head = 0, qn = 0;  // ring buffer state (uniform)

    // Evaluate one batch of up to 64 queued candidates in FP64, all lanes busy.
    auto drain = [&](int nb) {
      bool in = false;
      int row = 0, slot = 0;
      float4 spot = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      if (lane < nb) {
        const int e = queue[qpos(head + lane)];
        row = e >> kSlotBits;
        slot = e & (kOT - 1);
        in = eval_candidate<kAvg>(a, hkl, F2, rec, s_R[wib][slot], row, spot);
      }
#pragma unroll
      for (int o = 0; o < kOT; ++o) {
        const bool mine = in && slot == o;
        const uint64_t m = __ballot(mine);
        if (m == 0) continue;
        if (mine) {
          const int pos = cnt[o] + mask_rank(m);
          lmax[o] = fmaxf(lmax[o], spot.w);
          lmin[o] = fminf(lmin[o], spot.w);
          if (pos < cap) {
            const size_t off = (size_t)(o0 + o) * cap + pos;
            idx_out[off] = row;
            spot_out[off] = spot;
          }
        }
        cnt[o] += __popcll(m);
      }
      head = qpos(head + nb);
      qn -= nb;
    };

    // Queue the rows of this lane that pass the pretest of orientation o
    // (beam direction r0, r1, r2 in FP32).
    auto pretest = [&](bool v, int row, const float4 &g, float r0, float r1, float r2, int o) {
      const float zf = fmaf(r0, g.x, fmaf(r1, g.y, r2 * g.z));
      const bool pre = v && fabsf(fmaf(-two_k, zf, g.w)) < pre_thr;
      const uint64_t pm = __ballot(pre);
      if (pm == 0) return;
      if (pre) queue[qpos(head + qn + mask_rank(pm))] = (row << kSlotBits) | o;
      qn += __popcll(pm);
    };

    // Line sweep state: the current group of 64 lines (lb), orientation (lo)
    // and window (win).  When a group loads, the row interval of every line
    // (one per lane) is formed for all kOT orientations at once -- four
    // independent chains of FP64 arithmetic and prefix sums instead of one
    // chain per orientation -- and parked in LDS (per orientation and lane:
    // first candidate P, first row rb, pretest coefficients eA, eB; the
    // orientation's candidate total in s_tot), so the line data is dead while
    // the windows and drains run.
    const bool use_lines = kLines && d->lines != nullptr && lines_pay(n_refl, d->n_lines);
    const int4 *lines = reinterpret_cast<const int4 *>(d->lines);
    const int n_lines = use_lines ? d->n_lines : 0;
    int lb = -kWave, lo = kOT - 1, win = 0, total = 0;
    // along a line (hkl = (h, k, l0 - t)) the pretest value is a quadratic in
    // t: e(t) = |g0 - t c*|^2 - 2k (zt - t ga) = A + B t + c2 t^2, so a window
    // forms it from its line's coefficients (eA, eB at the interval's first
    // row) instead of loading the row's g4; w0 = |g0|^2, cd = g0 . c* (FP32:
    // their rounding, ~1e-6 of e, is far inside the pretest's slack)
    const double c2 = rec[2] * rec[2] + rec[5] * rec[5] + rec[8] * rec[8];
    const float c2f = static_cast<float>(c2);
    // pretest pass => |w - 2k zf| < thr (1 + 2^-24); zf (FP32 R and g, two
    // fmaf) is within 1e-6 |g| of the FP64 beam coordinate, ten times inside
    // the margin zm = 1e-5 (1 + max |g| of the line) below
    const double two_kd = static_cast<double>(two_k);
    const double thr = static_cast<double>(pre_thr) * (1.0 + 1e-6);
    if (use_lines) {
      // beam direction (third row of R) against the reciprocal axes, FP64
      if (lane < kOT * 4) {
        const int o = lane / 4, c = lane - 4 * o, cc = c < 3 ? c : 2;
        double v = 0.0;
        if (o < n_here) {
          const double *b = Rt + (size_t)(o0 + o) * 9 + 6;
          v = b[0] * rec[cc] + b[1] * rec[3 + cc] + b[2] * rec[6 + cc];
          // 1 / (beam . c*); 0 marks a line direction perpendicular to the beam
          if (c == 3) v = fabs(v) < 1e-200 ? 0.0 : 1.0 / v;
        }
        s_abc[wib][o][c] = v;
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
    }
    // Next group of lines: false once the lines are exhausted.
    auto load_group = [&]() -> bool {
      lb += kWave;
      if (lb >= n_lines) return false;
      const int j = lb + lane;
      int first = 0, nrow = 0, lh = 0, lk = 0, l0 = 0;
      double zlo = 0.0, zhi = -1.0;
      float w0 = 0.0f, cd = 0.0f;
      if (j < n_lines) {
        const int4 e0 = lines[2 * (size_t)j], e1 = lines[2 * (size_t)j + 1];
        first = e0.x;
        nrow = e0.y;
        lh = e0.z;
        lk = e0.w;
        l0 = e1.x;
        const double wmin = __int_as_float(e1.y), wmax = __int_as_float(e1.z);
        const double zm = 1e-5 * (1.0 + sqrt(wmax));
        zlo = (wmin - thr) / two_kd - zm;
        zhi = (wmax + thr) / two_kd + zm;
        const double hx = lh, hy = lk, hz = l0;
        const double gx = rec[0] * hx + rec[1] * hy + rec[2] * hz;
        const double gy = rec[3] * hx + rec[4] * hy + rec[5] * hz;
        const double gz = rec[6] * hx + rec[7] * hy + rec[8] * hz;
        w0 = static_cast<float>(gx * gx + gy * gy + gz * gz);
        cd = static_cast<float>(gx * rec[2] + gy * rec[5] + gz * rec[8]);
      }
      int t0[kOT], len[kOT], incl[kOT];
#pragma unroll
      for (int o = 0; o < kOT; ++o) {
        // z of row first + t is zt - t ga (l = l0 - t): the rows with z in [zlo, zhi]
        const double al = s_abc[wib][o][0], be = s_abc[wib][o][1], ga = s_abc[wib][o][2];
        const double inv = s_abc[wib][o][3];
        const double zt = static_cast<double>(lh) * al + static_cast<double>(lk) * be +
                          static_cast<double>(l0) * ga;
        t0[o] = 0;
        len[o] = 0;
        if (o >= n_here || nrow <= 0) {
          // no rows (an orientation past the tile's end, or no line)
        } else if (inv == 0.0) {  // line perpendicular to the beam: all rows or none
          if (zt >= zlo && zt <= zhi) len[o] = nrow;
        } else {
          const double q1 = (zt - zhi) * inv, q2 = (zt - zlo) * inv;
          const double tlo = fmax(ceil(fmin(q1, q2)), 0.0);
          const double thi = fmin(floor(fmax(q1, q2)), static_cast<double>(nrow - 1));
          if (thi >= tlo) {
            t0[o] = static_cast<int>(tlo);
            len[o] = static_cast<int>(thi - tlo) + 1;
          }
        }
        const double tt = static_cast<double>(t0[o]);
        const double eb = two_kd * ga - 2.0 * static_cast<double>(cd);
        s_eA[wib][o][lane] =
            static_cast<float>((static_cast<double>(w0) - two_kd * zt) + tt * (eb + c2 * tt));
        s_eB[wib][o][lane] = static_cast<float>(eb + 2.0 * c2 * tt);
        s_rb[wib][o][lane] = first + t0[o];
        incl[o] = len[o];  // inclusive prefix over the lanes (lines in row order)
      }
#pragma unroll
      for (int off = 1; off < kWave; off <<= 1) {
#pragma unroll
        for (int o = 0; o < kOT; ++o) {
          const int v = __shfl_up(incl[o], off);
          if (lane >= off) incl[o] += v;
        }
      }
#pragma unroll
      for (int o = 0; o < kOT; ++o) {
        s_P[wib][o][lane] = incl[o] - len[o];  // first candidate of this lane's line
        if (lane == kWave - 1) s_tot[wib][o] = incl[o];
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
      return true;
    };

    // One step per iteration: a window of 64 line candidates of one
    // orientation, or 64 table rows for every orientation; full batches are
    // drained as they fill, everything after the last step.
    for (int base = 0;; base += kWave) {
      bool done;
      if (use_lines) {
        done = false;
        win += kWave;
        while (win >= total) {
          if (++lo >= n_here) {  // next group of lines
            lo = 0;
            if (!load_group()) {
              done = true;
              break;
            }
          }
          total = s_tot[wib][lo];
          win = 0;
        }
        if (!done) {
          const int c = win + lane;
          // the last lane whose line starts at or before candidate c holds it
          const int *Pw = s_P[wib][lo];
          int src = 0;
#pragma unroll
          for (int step = kWave / 2; step > 0; step >>= 1)
            if (Pw[src + step] <= c) src += step;
          const int u = c - Pw[src];
          const int row = s_rb[wib][lo][src] + u;
          const bool v = c < total && static_cast<unsigned>(row) < static_cast<unsigned>(n_refl);
          const float uf = static_cast<float>(u);
          const float e = fmaf(fmaf(c2f, uf, s_eB[wib][lo][src]), uf, s_eA[wib][lo][src]);
          const bool pre = v && fabsf(e) < pre_thr;
          const uint64_t pm = __ballot(pre);
          if (pm != 0) {
            if (pre) queue[qpos(head + qn + mask_rank(pm))] = (row << kSlotBits) | lo;
            qn += __popcll(pm);
          }
        }
      } else {
        done = base >= n_refl;
        if (!done) {
          const int i = base + lane;
          const bool v = i < n_refl;
          const float4 g = v ? g4[i] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll
          for (int o = 0; o < kOT; ++o) {
            if (o >= n_here) break;  // uniform
            if (kLines)
              pretest(v, i, g, s_Rf[wib][o][0], s_Rf[wib][o][1], s_Rf[wib][o][2], o);
            else
              pretest(v, i, g, R[o][0], R[o][1], R[o][2], o);
          }
        }
      }
      const int need = done ? 1 : kWave;
      if (qn >= need) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
        while (qn >= need) drain(min(qn, kWave));
      }
      if (done) break;
    }

#pragma unroll
    for (int o = 0; o < kOT; ++o) {
      const int orient = o0 + o;
      if (o >= n_here) break;
      const float mx = wave_max(lmax[o]);
      const float mn = wave_min(lmin[o]);
      const int n = cnt[o];
      const int nw = min(n, cap);
      int final_count = nw;
      const float thr = mx * a.min_I;
      // mx == 0 with n > 0: every intersecting reflection is kinematically
      // forbidden (|F| exactly 0); the reference keeps them all (its FP64
      // round-off passes the relative cut), so they are kept with I = 0.
      if (n > 0 && mx > 0.0f && !(mn > thr)) {
        __threadfence_block();
        const size_t off = (size_t)orient * cap;
        int w = 0;
        for (int b = 0; b < nw; b += kWave) {
          const int j = b + lane;
          float4 sp = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
          int id = 0;
          bool keep = false;
          if (j < nw) {
            sp = spot_out[off + j];
            id = idx_out[off + j];
            keep = sp.w > thr;
          }
          const uint64_t km = __ballot(keep);
          if (keep) {
            const int pos = w + mask_rank(km);
            spot_out[off + pos] = sp;
            idx_out[off + pos] = id;
          }
          w += __popcll(km);
        }
        final_count = w;
      }
      if (lane == 0) {
        d->count[orient] = final_count;
        d->ncand[orient] = n;
        d->maxI[orient] = mx;
      }
    }
    // the next tile rewrites s_R and the queue
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
  }
}

// ---------------------------------------------------------------------------
// Few orientations: a block of 1, 2, 4 or 8 waves per orientation.
//
// With a wave per four orientations, 4,096 orientations are 1,024 waves, one
// per SIMD with nothing to hide its latencies, and 64 are 16 waves.  Here the
// waves of a block take consecutive parts of one orientation's rows: a step
// is 256 candidates per wave in row order, pretested into the wave's queue,
// evaluated in FP64 up to 64 at a time, the survivors kept in registers until
// one barrier has published every wave's count, then written at their place.
// With a line index a chunk is a line per thread (row interval, block prefix
// sum), and its candidates are taken in steps.
// The rows tested, their order and every value are those of simulate_kernel.
// Held to 128 registers (four waves per SIMD) the line form keeps 9 of them in
// scratch with 8 or 4 waves, 8 with 2 and 3 with 1; VALU busy 74 % on 4,096
// orientations of 14,306 lines.
// ---------------------------------------------------------------------------

constexpr int kCoopPer = 4;                      // candidates per lane and step
constexpr int kCoopWaveStep = kCoopPer * kWave;  // candidates per wave and step

template <bool kLines, int kCoopWaves>
__global__ __launch_bounds__(kCoopWaves *kWave, 4) void simulate_coop_kernel(SimArgs a) {
  constexpr int kCoopThreads = kCoopWaves * kWave;
  constexpr int kCoopStep = kCoopWaves * kCoopWaveStep;
  constexpr int kLW = kLines ? kCoopThreads : 1;
  __shared__ int s_queue[kCoopWaves][kCoopWaveStep];
  __shared__ int s_P[kLW], s_rb[kLW];
  __shared__ float s_eA[kLW], s_eB[kLW], s_wA[kLW], s_wB[kLW];
  __shared__ int s_sum[kCoopWaves];
  __shared__ int s_cnt[2][kCoopWaves];
  __shared__ double s_R[9], s_abc[4];
  __shared__ float s_mx[kCoopWaves], s_mn[kCoopWaves];
  const int tid = threadIdx.x, lane = lane_id(), wid = tid / kWave;
  const dsx_phase_desc &d = a.single;
  const int4 *hkl = reinterpret_cast<const int4 *>(d.hkl);
  const float4 *g4 = reinterpret_cast<const float4 *>(d.g4);
  const float *F2 = d.F2;
  const double *rec = d.rec;
  const int n_refl = d.n_refl, cap = d.cap, n_lines = d.n_lines;
  const int4 *lines = reinterpret_cast<const int4 *>(d.lines);
  const float two_k = 2.0f * a.k_f;
  const double two_kd = static_cast<double>(two_k);
  const float pre_thr = pretest_threshold(a.me, a.k, d.g_max, a.sin_phi);
  // Under precession the band of a row widens with its own |g| (|e| <= 2 k
  // (me + r sin(phi)), r <= |g|), not with the table's largest: a row's
  // threshold is pre0 + pre1 |g|, at most pre_thr.  64,000 -> 48,000 FP64
  // candidates per orientation of the 500-atom cell at 1 degree.
  const float pre0 = pretest_threshold(a.me, a.k, d.g_max, 0.0);
  const float pre1 = static_cast<float>(1.05 * 1.1 * a.sin_phi * (2.0 * a.k + d.g_max));
  auto passes = [&](float e, float w) {  // w = |g|^2
    const float t = pre1 > 0.0f ? fmaf(pre1, __builtin_amdgcn_sqrtf(fmaxf(w, 0.0f)), pre0) : pre_thr;
    return fabsf(e) < t;
  };
  const double thr = static_cast<double>(pre_thr) * (1.0 + 1e-6);
  const double c2 = rec[2] * rec[2] + rec[5] * rec[5] + rec[8] * rec[8];
  const float c2f = static_cast<float>(c2);
  int *queue = s_queue[wid];

  for (long long o = blockIdx.x; o < d.n_orient; o += gridDim.x) {
    const double *b = d.Rt + static_cast<size_t>(o) * 9;
    if (tid < 9) s_R[tid] = b[tid];
    if (kLines && tid < 4) {
      const int cc = tid < 3 ? tid : 2;
      double v = b[6] * rec[cc] + b[7] * rec[3 + cc] + b[8] * rec[6 + cc];
      if (tid == 3) v = fabs(v) < 1e-200 ? 0.0 : 1.0 / v;
      s_abc[tid] = v;
    }
    lds_sync();
    const float r0 = static_cast<float>(s_R[6]), r1 = static_cast<float>(s_R[7]),
                r2 = static_cast<float>(s_R[8]);
    int *idx_out = d.idx + static_cast<size_t>(o) * cap;
    float4 *spot_out = reinterpret_cast<float4 *>(d.spots) + static_cast<size_t>(o) * cap;
    int base = 0, buf = 0;
    float lmax = 0.0f, lmin = __builtin_huge_valf();

    // Evaluate the wave's queue of q candidates, publish the count, and write
    // the survivors at their place in the list (one block barrier).
    auto finish_step = [&](int q) {
      float4 spot[kCoopPer];
      int row[kCoopPer], rank[kCoopPer];
      int cnt = 0;
#pragma unroll
      for (int k = 0; k < kCoopPer; ++k) {
        rank[k] = -1;
        if (k * kWave >= q) continue;  // uniform
        bool in = false;
        if (k * kWave + lane < q) {
          row[k] = queue[k * kWave + lane];
          in = eval_candidate<false>(a, hkl, F2, rec, s_R, row[k], spot[k]);
        }
        const uint64_t m = __ballot(in);
        if (in) {
          rank[k] = cnt + mask_rank(m);
          lmax = fmaxf(lmax, spot[k].w);
          lmin = fminf(lmin, spot[k].w);
        }
        cnt += __popcll(m);
      }
      if (lane == 0) s_cnt[buf][wid] = cnt;
      lds_sync();
      int at = base;
#pragma unroll
      for (int w = 0; w < kCoopWaves; ++w) {
        const int c = s_cnt[buf][w];
        if (w < wid) at += c;
        base += c;
      }
      buf ^= 1;  // rewritten two steps on, after every wave has read it
#pragma unroll
      for (int k = 0; k < kCoopPer; ++k) {
        const int pos = at + rank[k];
        if (rank[k] >= 0 && pos < cap) {
          idx_out[pos] = row[k];
          spot_out[pos] = spot[k];
        }
      }
    };
    auto wave_sync = [&]() {
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
    };

    if (kLines) {
      const double al = s_abc[0], be = s_abc[1], ga = s_abc[2], inv = s_abc[3];
      for (int l0 = 0; l0 < n_lines; l0 += kCoopThreads) {
        // the rows of this thread's line that can pass the pretest (as
        // load_group of simulate_kernel)
        const int j = l0 + tid;
        int first = 0, len = 0, t0 = 0;
        double eA = 0.0, eB = 0.0, wA = 0.0, wB = 0.0;
        if (j < n_lines) {
          const int4 e0 = lines[2 * static_cast<size_t>(j)], e1 = lines[2 * static_cast<size_t>(j) + 1];
          first = e0.x;
          const int nrow = e0.y;
          const double hx = e0.z, hy = e0.w, hz = e1.x;
          const double wmin = __int_as_float(e1.y), wmax = __int_as_float(e1.z);
          const double zm = 1e-5 * (1.0 + sqrt(wmax));
          const double zlo = (wmin - thr) / two_kd - zm, zhi = (wmax + thr) / two_kd + zm;
          const double gx = rec[0] * hx + rec[1] * hy + rec[2] * hz;
          const double gy = rec[3] * hx + rec[4] * hy + rec[5] * hz;
          const double gz = rec[6] * hx + rec[7] * hy + rec[8] * hz;
          const float w0 = static_cast<float>(gx * gx + gy * gy + gz * gz);
          const float cd = static_cast<float>(gx * rec[2] + gy * rec[5] + gz * rec[8]);
          const double zt = hx * al + hy * be + hz * ga;
          if (inv == 0.0) {  // line perpendicular to the beam: all rows or none
            if (zt >= zlo && zt <= zhi) len = nrow;
          } else {
            const double q1 = (zt - zhi) * inv, q2 = (zt - zlo) * inv;
            const double tlo = fmax(ceil(fmin(q1, q2)), 0.0);
            const double thi = fmin(floor(fmax(q1, q2)), static_cast<double>(nrow - 1));
            if (thi >= tlo) {
              t0 = static_cast<int>(tlo);
              len = static_cast<int>(thi - tlo) + 1;
            }
          }
          const double tt = static_cast<double>(t0);
          const double eb = two_kd * ga - 2.0 * static_cast<double>(cd);
          eA = (static_cast<double>(w0) - two_kd * zt) + tt * (eb + c2 * tt);
          eB = eb + 2.0 * c2 * tt;
          wB = -2.0 * static_cast<double>(cd) + 2.0 * c2 * tt;
          wA = static_cast<double>(w0) + tt * (c2 * tt - 2.0 * static_cast<double>(cd));
        }
        const int incl = wave_inclusive_scan(len);
        if (lane == kWave - 1) s_sum[wid] = incl;
        lds_sync();
        int before = 0, total = 0;
#pragma unroll
        for (int w = 0; w < kCoopWaves; ++w) {
          const int c = s_sum[w];
          if (w < wid) before += c;
          total += c;
        }
        s_P[tid] = before + incl - len;
        s_rb[tid] = first + t0;
        s_eA[tid] = static_cast<float>(eA);
        s_eB[tid] = static_cast<float>(eB);
        s_wA[tid] = static_cast<float>(wA);
        s_wB[tid] = static_cast<float>(wB);
        lds_sync();
        for (int s0 = 0; s0 < total; s0 += kCoopStep) {
          int q = 0;
#pragma unroll
          for (int k = 0; k < kCoopPer; ++k) {
            const int w0 = s0 + wid * kCoopWaveStep + k * kWave;
            if (w0 >= total) break;  // uniform
            const int c = w0 + lane;
            int src = 0;  // the last line that starts at or before candidate c holds it
#pragma unroll
            for (int step = kCoopThreads / 2; step > 0; step >>= 1)
              if (s_P[src + step] <= c) src += step;
            const int u = c - s_P[src];
            const int row = s_rb[src] + u;
            const bool v = c < total && static_cast<unsigned>(row) < static_cast<unsigned>(n_refl);
            const float uf = static_cast<float>(u);
            const float e = fmaf(fmaf(c2f, uf, s_eB[src]), uf, s_eA[src]);
            const float w = pre1 > 0.0f ? fmaf(fmaf(c2f, uf, s_wB[src]), uf, s_wA[src]) : 0.0f;
            const bool pre = v && passes(e, w);
            const uint64_t m = __ballot(pre);
            if (pre) queue[q + mask_rank(m)] = row;
            q += __popcll(m);
          }
          wave_sync();
          finish_step(q);
        }
      }
    } else {
      for (int s0 = 0; s0 < n_refl; s0 += kCoopStep) {
        const int w0 = s0 + wid * kCoopWaveStep;
        float4 g[kCoopPer];
#pragma unroll
        for (int k = 0; k < kCoopPer; ++k) {
          const int i = w0 + k * kWave + lane;
          g[k] = i < n_refl ? g4[i] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        }
        int q = 0;
#pragma unroll
        for (int k = 0; k < kCoopPer; ++k) {
          const int i = w0 + k * kWave + lane;
          const float zf = fmaf(r0, g[k].x, fmaf(r1, g[k].y, r2 * g[k].z));
          const bool pre = i < n_refl && passes(fmaf(-two_k, zf, g[k].w), g[k].w);
          const uint64_t m = __ballot(pre);
          if (pre) queue[q + mask_rank(m)] = i;
          q += __popcll(m);
        }
        wave_sync();
        finish_step(q);
      }
    }

    // ---- relative cut (as simulate_kernel), the whole block compacting -------
    lmax = wave_max(lmax);
    lmin = wave_min(lmin);
    if (lane == 0) {
      s_mx[wid] = lmax;
      s_mn[wid] = lmin;
    }
    __syncthreads();  // the list in global memory too
    float mx = s_mx[0], mn = s_mn[0];
#pragma unroll
    for (int w = 1; w < kCoopWaves; ++w) {
      mx = fmaxf(mx, s_mx[w]);
      mn = fminf(mn, s_mn[w]);
    }
    const int nw = min(base, cap);
    int final_count = nw;
    const float cut = mx * a.min_I;
    if (base > 0 && mx > 0.0f && !(mn > cut)) {
      int kept = 0;
      for (int c0 = 0; c0 < nw; c0 += kCoopThreads) {
        const int j = c0 + tid;
        float4 sp = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        int id = 0;
        if (j < nw) {
          sp = spot_out[j];
          id = idx_out[j];
        }
        const bool keep = j < nw && sp.w > cut;
        const uint64_t m = __ballot(keep);
        if (lane == 0) s_cnt[buf][wid] = __popcll(m);
        __syncthreads();  // every entry of the chunk is read before any is written
        int at = kept;
#pragma unroll
        for (int w = 0; w < kCoopWaves; ++w) {
          const int c = s_cnt[buf][w];
          if (w < wid) at += c;
          kept += c;
        }
        buf ^= 1;
        if (keep) {
          const int pos = at + mask_rank(m);
          spot_out[pos] = sp;
          idx_out[pos] = id;
        }
      }
      final_count = kept;
    }
    if (tid == 0) {
      d.count[o] = final_count;
      d.ncand[o] = base;
      d.maxI[o] = mx;
    }
    __syncthreads();  // s_R, s_mx and the counts are rewritten for the next orientation
  }
}

// Waves per orientation of simulate_coop_kernel, 0: simulate_kernel's wave per
// four orientations (which shares each row or line among them).  As many
// waves as fill four per SIMD, in us, by waves (wave per four: last):
//   500-atom precession (14,306 lines)  16: 451 (8) 776 (4) 2,287 (1) 8,647
//     1,024: 1,139 (8) 1,164 (4) 1,563 (2) 8,519   2,048: 2,029 (2) 2,640 (1)
//     4,096: 4,308 (2) 3,669 (1) 9,134   16,384: 13,031 (1) 13,557
//     (before the per-row threshold: with it 3,334 (1) and 12,015 (1))
//   40-atom library (1,186 lines)  64: 18 (8) 41 (1) 87   2,000: 68 (8) 38 (2)
//     51 (1) 93   4,096: 67 (1) 97   8,192: 122 (1) 104
//   17 A cell (3,482 lines)  8,000: 381 (1) 460   20,000: 877 (1) 866
//   24-atom cell, full sweep of 4,614 rows  512: 11 (8) 29 (1) 45   2,048: 23
//     (2) 31 (1) 45   4,096: 40 (1) 48   8,192: 76 (1) 52
//   256 rows  500: 12 (8) 9 (2) 11   4,000: 10 (1) 11   20,000: 21 (1) 16
// How many orientations a wave each stays ahead for, time over the wave per
// four, non-precessed tables of 282 to 7,798 lines: it repeats the work per line
// that the other shares, so it depends on the candidates per line, c = rows per
// line (1.5 max_excitation_error / g_max + sin phi).  They cross at 4,600 to 5,000
// orientations for c <= 0.12, 5,200-6,200 at 0.16, 6,500 at 0.22, 7,800-8,700 at
// 0.32, 10,500 at 0.46, 11,300-12,000 at 0.54-0.66 and 12,500-14,000 above; 16,384
// take 1.7-1.9 times as long at 0.12 and 1.1 at 1.  Where precession gives most
// of the candidates (rows per line times sin phi of 0.3 and more) the per-row
// threshold saves a quarter of them and one wave is ahead at any number (20,000:
// 0.66-0.91; 500-atom cell 14,622 us against 20,271).  The full sweep shares each row:
// they cross at 3,900-4,200 with 6,212 to 28,800 rows, at 5,000-6,100 with 484 and
// beyond 6,144 with 250 (9.4 us | 12.8 there).
static int coop_waves(int n_orient, int n_refl, int n_lines, double me, double g_max, double sin_phi) {
  double limit = n_refl < 384 ? 6144 : n_refl < 1024 ? 5120 : 4096;
  if (n_lines > 0) {
    const double rows = static_cast<double>(n_refl) / n_lines;
    const double c = g_max > 0.0 ? rows * (1.5 * me / g_max + sin_phi) : 0.0;
    limit = rows * sin_phi >= 0.3 ? 1e10 : std::min(std::max(3000.0 + 15500.0 * c, 4500.0), 12288.0);
    if (n_lines < 2048) limit = std::min(limit, 6144.0);
  }
  if (n_orient > limit) return 0;
  int w = n_orient <= 512 ? 8 : (n_orient <= 1280 ? 4 : (n_orient <= 2560 ? 2 : 1));
  while (w > 1 && n_refl < w * 2 * kWave) w /= 2;  // at least two rows per lane
  return w;
}

// Blocks of a launch; beyond them the kernel's loop takes the remaining
// orientations (a launch holds less than 2^32 threads).
constexpr int kCoopBlocks = 1 << 23;

template <bool kLines>
static void launch_coop(int waves, const SimArgs &a, hipStream_t s) {
  const dim3 blocks(static_cast<unsigned>(std::min(a.single.n_orient, kCoopBlocks))),
      threads(static_cast<unsigned>(waves * kWave));
  switch (waves) {
    case 8: hipLaunchKernelGGL((simulate_coop_kernel<kLines, 8>), blocks, threads, 0, s, a); break;
    case 4: hipLaunchKernelGGL((simulate_coop_kernel<kLines, 4>), blocks, threads, 0, s, a); break;
    case 2: hipLaunchKernelGGL((simulate_coop_kernel<kLines, 2>), blocks, threads, 0, s, a); break;
    default: hipLaunchKernelGGL((simulate_coop_kernel<kLines, 1>), blocks, threads, 0, s, a);
  }
}

static int check_physics(const dsx_sim_params *p, const char *name) {
  const bool averaged = p->shape_model >= DSX_SF_PRECESSION_AVG + DSX_SF_LINEAR &&
                        p->shape_model <= DSX_SF_PRECESSION_AVG + DSX_SF_BINARY;
  if (!averaged && (p->shape_model < DSX_SF_LINEAR || p->shape_model > DSX_SF_LORENTZIAN_PRECESSION)) {
    set_error("%s: unknown shape model %d", name, p->shape_model);
    return DSX_EINVAL;
  }
  if (averaged && !(p->precession_angle > 0.0)) {
    set_error("%s: the full precession average needs a positive precession angle", name);
    return DSX_EINVAL;
  }
  if (!(p->k > 0.0) || !(p->max_excitation_error > 0.0) || p->shape_width == 0.0 ||
      !(p->precession_angle >= 0.0) || !(p->g_max >= 0.0)) {
    set_error("%s: bad physical parameters", name);
    return DSX_EINVAL;
  }
  if (p->shape_model == DSX_SF_LORENTZIAN_PRECESSION && !(p->precession_angle > 0.0)) {
    set_error("%s: the precession shape factor needs a positive precession angle", name);
    return DSX_EINVAL;
  }
  return DSX_OK;
}

static void fill_args(SimArgs &a, const dsx_sim_params *p) {
  fill_physics(a, p);
  a.k_f = static_cast<float>(p->k);
  a.sin_phi = p->precession_angle > 0.0 ? sin(p->precession_angle) : 0.0;
  a.min_I = static_cast<float>(p->minimum_intensity);
  a.phases = nullptr;
  a.items = nullptr;
}

// Blocks of the spot kernel's launch: each wave takes every n_waves-th tile.
// Far more waves than stay resident (default 128 one-wave blocks per CU, one
// or two tiles per wave on the library) let the dispatcher hand the slots of
// waves that finish early to the next ones, which balances tiles of unequal
// cost; a launch of only the resident waves leaves each a fixed share.  The
// library's 50,000 tiles, in waves per CU (four-wave blocks): 1.60 ms with 16,
// 1.55 with 32, 1.52 with 48, 1.50 with 64, 1.45-1.46 with 128 or 256.
static int launch_blocks(int n_items, int blocks_per_cu) {
  const int waves_per_block = kSimThreads / kWave;
  const int blocks = (n_items + waves_per_block - 1) / waves_per_block;
  return std::max(1, std::min(blocks, cu_count() * (blocks_per_cu > 0 ? blocks_per_cu : 128)));
}

}  // namespace dsx

using namespace dsx;

extern "C" int dsx_simulate(const int *hkl_d, const float *g4_d, const float *F2_d, int n_refl,
                            const int *lines_d, int n_lines, const double *Rt_d, int n_orient,
                            const dsx_sim_params *p, int cap, int *idx_d, float *spot_d,
                            int *count_d, int *ncand_d, float *maxI_d, void *stream) {
  clear_error();
  if (!p || n_refl < 0 || n_orient < 0 || cap < 1 || n_lines < 0 || (n_lines > 0 && !lines_d)) {
    set_error("dsx_simulate: bad arguments (n_refl=%d n_orient=%d cap=%d)", n_refl, n_orient, cap);
    return DSX_EINVAL;
  }
  if (n_orient == 0) return DSX_OK;
  if (!Rt_d || !idx_d || !spot_d || !count_d || !ncand_d || !maxI_d ||
      (n_refl > 0 && (!hkl_d || !g4_d || !F2_d))) {
    set_error("dsx_simulate: null device pointer");
    return DSX_EINVAL;
  }
  const int st = check_physics(p, "dsx_simulate");
  if (st != DSX_OK) return st;
  if ((size_t)n_orient * (size_t)cap > (size_t)1 << 40) {
    set_error("dsx_simulate: n_orient*cap too large");
    return DSX_EINVAL;
  }
  SimArgs a;
  fill_args(a, p);
  dsx_phase_desc &d = a.single;
  d.hkl = hkl_d;
  d.g4 = g4_d;
  d.F2 = F2_d;
  d.n_refl = n_refl;
  d.cap = cap;
  for (int i = 0; i < 9; ++i) d.rec[i] = p->rec[i];
  d.g_max = p->g_max;
  d.Rt = Rt_d;
  d.n_orient = n_orient;
  d.n_lines = lines_d ? n_lines : 0;
  d.idx = idx_d;
  d.spots = spot_d;
  d.count = count_d;
  d.ncand = ncand_d;
  d.maxI = maxI_d;
  d.lines = lines_d;
  a.n_items = (n_orient + kOT - 1) / kOT;
  const dim3 grid(launch_blocks(a.n_items, 0));
  hipStream_t s = as_stream(stream);
  // the averaged-precession model keeps the full sweep: its FP64 evaluation
  // dominates, and the line state would cost it occupancy
  const bool avg = p->shape_model >= DSX_SF_PRECESSION_AVG;
  const bool use_lines = lines_d && !avg && lines_pay(n_refl, n_lines);
  const int coop = avg ? 0 : coop_waves(n_orient, n_refl, use_lines ? n_lines : 0, p->max_excitation_error,
                                        p->g_max, a.precession ? a.sin_phi : 0.0);
  if (coop > 0) {
    if (use_lines)
      launch_coop<true>(coop, a, s);
    else
      launch_coop<false>(coop, a, s);
  } else if (use_lines)
    hipLaunchKernelGGL((simulate_kernel<false, false, true>), grid, dim3(kSimThreads), 0, s, a);
  else if (avg)
    hipLaunchKernelGGL((simulate_kernel<false, true, false>), grid, dim3(kSimThreads), 0, s, a);
  else
    hipLaunchKernelGGL((simulate_kernel<false, false, false>), grid, dim3(kSimThreads), 0, s, a);
  return check_launch("dsx_simulate");
}

extern "C" int dsx_simulate_tile_size(void) { return kOT; }

extern "C" int dsx_simulate_ragged(const dsx_phase_desc *phases_d, int n_phases, const int *items_d,
                                   int n_items, const dsx_sim_params *p, int blocks_per_cu,
                                   void *stream) {
  clear_error();
  if (!p || n_phases < 0 || n_items < 0 || blocks_per_cu < 0) {
    set_error("dsx_simulate_ragged: bad arguments (n_phases=%d n_items=%d)", n_phases, n_items);
    return DSX_EINVAL;
  }
  if (n_items == 0) return DSX_OK;
  if (!phases_d || !items_d || n_phases == 0) {
    set_error("dsx_simulate_ragged: null device pointer or no phases");
    return DSX_EINVAL;
  }
  const int st = check_physics(p, "dsx_simulate_ragged");
  if (st != DSX_OK) return st;
  SimArgs a;
  fill_args(a, p);
  a.phases = phases_d;
  a.items = reinterpret_cast<const int2 *>(items_d);
  a.n_items = n_items;
  // each phase uses its line index when it has one (lines != NULL) and its
  // lines are long enough, except under the averaged-precession model
  if (p->shape_model >= DSX_SF_PRECESSION_AVG)
    hipLaunchKernelGGL((simulate_kernel<true, true, false>), dim3(launch_blocks(n_items, blocks_per_cu)),
                       dim3(kSimThreads), 0, as_stream(stream), a);
  else
    hipLaunchKernelGGL((simulate_kernel<true, false, true>), dim3(launch_blocks(n_items, blocks_per_cu)),
                       dim3(kSimThreads), 0, as_stream(stream), a);
  return check_launch("dsx_simulate_ragged");
}
