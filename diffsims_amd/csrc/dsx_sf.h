// Structure factors of many atoms and their adjoint with one atom per lane.
//
// F(h) = sum_a f_a(|g|) occ_a exp(-B_a |g|^2 / 4) e^(2 pi i h.x_a).  The kernels
// of dsx_tables.hip / dsx_adjoint.hip give every reflection a thread and form
// each atom's phase anew: an integer phase, a sine and cosine, an exponential
// (about 85 instructions per reflection and atom, and another 48 cross-lane
// steps in the adjoint).  Here a lane keeps an atom and a wave walks down
// consecutive rows of the table: along a line (equal h and k, l falling by
// one) the phase turns by -2 pi z_a, two FP64 products and two fmas, and only
// a row that starts a line (the same for all lanes) forms it anew.  The sums
// over atoms collect in registers, one set per row of a short run of rows, and
// are folded over the lanes once per run; the adjoint's sums over reflections
// stay with the atom's lane.
#pragma once

#include "dsx_internal.h"
#include "dsx_physics.h"

namespace dsx {

constexpr int kAtomThreads = 256;
constexpr int kAtomWaves = kAtomThreads / kWave;
constexpr int kAtomRows = 16;     // rows a wave stages at a time
// atoms and elements whose tables fit the 64 KB of LDS that a block has without
// further ado; larger cells keep a thread per reflection
constexpr int kAtomMax = 512;
constexpr int kAtomElems = 20;

// Sum over the lanes of each of 16 values, v[i] -> lanes i mod 16.  Every step
// halves the values: a lane keeps those with its bit of the index and hands
// the others to its partner.
template <int w>
__device__ __forceinline__ void fold_step(double *v, int lane) {
  const bool high = (lane & w) != 0;
#pragma unroll
  for (int i = 0; i < w; ++i) {
    const double keep = high ? v[i + w] : v[i];
    const double give = high ? v[i] : v[i + w];
    v[i] = keep + __shfl_xor(give, w, kWave);
  }
}

// (a loop over the widths is not unrolled and would index v at run time)
__device__ __forceinline__ double fold(double (&v)[16], int lane) {
  fold_step<8>(v, lane);
  fold_step<4>(v, lane);
  fold_step<2>(v, lane);
  fold_step<1>(v, lane);
  const double s = v[0] + __shfl_xor(v[0], 16, kWave);
  return s + __shfl_xor(s, 32, kWave);
}

struct AtomLane {
  uint4 x;        // fixed-point fractional position
  float B, occ;   // occ = 0 past the last atom
  int el;
  double ct, st;  // one row down a line: cos(2 pi z), -sin(2 pi z)
  double c, s;    // the current row's phase
};

// The block's atoms in LDS, 44 B each, with e^(-2 pi i z).
struct AtomTable {
  double2 *turn;
  uint4 *x;
  float2 *Bo;  // B, occ
  int *el;
};

__host__ __device__ __forceinline__ int atom_table_doubles(int n) { return (44 * n + 15) / 16 * 2; }

__device__ __forceinline__ AtomTable atom_table(double *s, int n) {
  AtomTable t;
  t.turn = reinterpret_cast<double2 *>(s);
  t.x = reinterpret_cast<uint4 *>(t.turn + n);
  t.Bo = reinterpret_cast<float2 *>(t.x + n);
  t.el = reinterpret_cast<int *>(t.Bo + n);
  return t;
}

template <class Args>
__device__ __forceinline__ void stage_atoms(const Args &a, const AtomTable &t) {
  for (int i = threadIdx.x; i < a.n_atoms; i += blockDim.x) {
    const uint4 x = a.xyz_fx[i];
    double sn, cs;
    sincospi(static_cast<double>(static_cast<int32_t>(x.z)) * (2.0 / 4294967296.0), &sn, &cs);
    t.turn[i] = make_double2(cs, -sn);
    t.x[i] = x;
    t.Bo[i] = make_float2(a.B[i], a.occ[i]);
    t.el[i] = min(max(a.elem[i], 0), a.n_elem - 1);
  }
}

__device__ __forceinline__ AtomLane load_atom(const AtomTable &tab, int atom, int n) {
  AtomLane t;
  const int i = atom < n ? atom : 0;
  t.x = tab.x[i];
  const float2 bo = tab.Bo[i];
  t.B = bo.x;
  t.occ = atom < n ? bo.y : 0.0f;
  t.el = tab.el[i];
  const double2 turn = tab.turn[i];
  t.ct = turn.x;
  t.st = turn.y;
  t.c = t.s = 0.0;
  return t;
}

// cos and sin of u / 2^32 turns in FP64: the nearest quarter turn is taken off
// in integers, the rest (at most an eighth) goes through the Taylor series to
// 2e-18 (cos) and 5e-17 (sin); multiples of a quarter are exact.
__device__ __forceinline__ void turn_sincos(uint32_t u, double &c, double &s) {
  const uint32_t q = (u + (1u << 29)) >> 30;
  const double x = static_cast<double>(static_cast<int32_t>(u - (q << 30))) * (2.0 * M_PI / 4294967296.0);
  const double y = x * x;
  constexpr double f2 = 2, f4 = 24, f6 = 720, f8 = 40320, f10 = 3628800, f12 = 479001600,
                   f14 = 87178291200.0, f16 = 20922789888000.0;
  const double cs = fma(y, fma(y, fma(y, fma(y, fma(y, fma(y, fma(y, fma(y, 1 / f16, -1 / f14), 1 / f12),
                    -1 / f10), 1 / f8), -1 / f6), 1 / f4), -1 / f2), 1.0);
  const double sn = x * fma(y, fma(y, fma(y, fma(y, fma(y, fma(y, fma(y, -1 / (f14 * 15), 1 / (f12 * 13)),
                    -1 / (f10 * 11)), 1 / (f8 * 9)), -1 / (f6 * 7)), 1 / (f4 * 5)), -1 / (f2 * 3)), 1.0);
  const double p = (q & 1) ? sn : cs, r = (q & 1) ? cs : sn;
  c = ((q + 1) & 2) ? -p : p;
  s = (q & 2) ? -r : r;
}

// Phase of the row h: turned on from the row before it in its line, or anew.
// The tables form it in FP64 (kExact): where atoms cancel, the turned phases and
// the newly formed ones have to agree to rounding, or extinct reflections come
// out at 1e-16 of the strongest |F|^2 (FP32 phases, atoms at eighths of the
// cell) instead of 1e-32 and pass the relative cut.  The adjoint sees only
// reflections that passed and takes sincospif.
template <bool kExact>
__device__ __forceinline__ void row_phase(AtomLane &t, bool anew, const int4 &h) {
  if (anew) {  // uniform
    const uint32_t u = static_cast<uint32_t>(h.x) * t.x.x + static_cast<uint32_t>(h.y) * t.x.y +
                       static_cast<uint32_t>(h.z) * t.x.z;
    if (kExact) {
      turn_sincos(u, t.c, t.s);
    } else {
      float sn, cs;
      sincospif(2.0f * (static_cast<float>(static_cast<int32_t>(u)) * 2.3283064365386963e-10f), &sn, &cs);
      t.c = cs;
      t.s = sn;
    }
  } else {
    const double c = fma(t.c, t.ct, -(t.s * t.st));
    t.s = fma(t.s, t.ct, t.c * t.st);
    t.c = c;
  }
}

__device__ __forceinline__ bool line_goes_on(const int4 &before, const int4 &h) {
  return before.x == h.x && before.y == h.y && before.z == h.z + 1;
}

__device__ __forceinline__ void atom_wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
}

// Rows per block, a whole number of its waves' rows: enough to pay for the staged
// turns, few enough to fill the chip.
static inline int atom_rows_per_block(int n, int waves, int least) {
  const int unit = kAtomRows * waves, most = 512;
  const int rows = (n / 1024 + unit - 1) / unit * unit;
  return rows < least ? least : (rows > most ? most : rows);
}

// Which tables take these kernels.  A lane per atom costs a pass per 64 atoms,
// full or not, a thread per reflection costs in proportion to the atoms but needs
// many rows to fill the chip.  Measured in us, thread per reflection | atom per
// lane (lines of 17 to 40 rows, 4 elements):
//   rows       24 atoms   32        48        64        65        80        100
//   1,000,000  55 | 128   65 | 128  87 | 127  108 | 128 107 | 179 128 | 178 156 | 178
//              341 | 341  376 | 341 390 | 341 427 | 341 440 | 482 496 | 481 606 | 480
//   400,000    27 | 64    32 | 64   43 | 64   53 | 64   53 | 89   63 | 89   76 | 89
//              159 | 174  178 | 175 200 | 176 232 | 177 215 | 244 251 | 245 299 | 246
//   195,590    15 | 30    18 | 30   24 | 30   30 | 30   30 | 41   36 | 41   43 | 41
//              95 | 92    106 | 92  124 | 92  147 | 94  147 | 118 167 | 119 196 | 119
//   100,000    12 | 21    15 | 21   20 | 21   25 | 21   25 | 28   30 | 28   36 | 28
//              62 | 64    70 | 64   88 | 65   105 | 65 106 | 82  122 | 82  144 | 82
//   58,076     11 | 12    13 | 12   18 | 12   22 | 12   22 | 16   26 | 16   32 | 16
//              50 | 40    59 | 40   76 | 40   94 | 40   95 | 49   112 | 50  133 | 49
//   17,332     11 | 8     13 | 8    17 | 8    22 | 8    22 | 12   26 | 12   31 | 12
//              38 | 28    47 | 28   65 | 28   82 | 28   83 | 37   100 | 37  122 | 37
//   4,614      10 | 7     12 | 7    17 | 7    21 | 7    22 | 9    26 | 9    31 | 9
//              35 | 22    44 | 22   62 | 22   80 | 22   81 | 30   98 | 30   120 | 30
// (first line forward, second adjoint; at 400,000 rows forward 129 atoms 96 | 113,
// 160 116 | 114, 193 138 | 138, 500 346 | 240, at 195,590 96 atoms 41 | 41 and 129
// 53 | 52; adjoint 129 atoms 375 | 319 and 500 1,398 | 634.)
static inline bool atoms_fit(int n_atoms, int n_elem) {
  return n_atoms <= kAtomMax && n_elem >= 1 && n_elem <= kAtomElems;
}

static inline bool atoms_per_lane(int n, int n_atoms, int n_elem) {
  const int least = n <= 24 * 1024 ? 24 : n <= 64 * 1024 ? 32 : n <= 128 * 1024 ? 76 : n <= 256 * 1024 ? 96 : 160;
  return atoms_fit(n_atoms, n_elem) && n_atoms >= least;
}

static inline bool atoms_per_lane_adjoint(int n, int n_atoms, int n_elem) {
  const int passes = (n_atoms + kWave - 1) / kWave;
  const int least = n <= 64 * 1024 ? 24 : n <= 256 * 1024 ? 32 : 40 * passes;
  return atoms_fit(n_atoms, n_elem) && n_atoms >= least;
}

}  // namespace dsx
