// Device code shared by the stage kernels (stage_kernel.hip: the column-chunk
// global path; stage_tile.hip, stage_tile3.hip: tiles): pair inputs, the
// global path's stencil walk with acceptance masks and pair loop, the
// per-target SSPRK update, the per-wave reductions and the chunk queue.  Every
// path visits a target's candidates in the same order and rounds
// identically, so all schedules produce the same bits.
#pragma once

#include <algorithm>
#include <type_traits>

#include "pair_math.hpp"
#include "sph_kernels.hpp"
#include "stencil.hpp"

namespace tit_amd {

namespace {

constexpr int kWordsG = 24;    // 32-candidate masks held per lane (column chunks)

// Positions from global memory (any dimension), WORDS acceptance masks per
// lane between two pair loops.
template <int DIM, int WORDS = kWordsG>
struct GlobalPos {
  const DevTank& T;
  const DevState& S;
  const uint32_t* coff;
  int cx, cy;    // target column
  uint32_t* wm;  // this wave's [WORDS][64] 32-candidate acceptance masks
  uint32_t* wj;  // global index of each mask's bit 0

  __device__ __forceinline__ bool range(int k, int w0, int w1, uint32_t& b,
                                        uint32_t& e) const {
    constexpr int L = DIM - 1;
    int ix, iy = 0;
    if constexpr (DIM == 2) {
      ix = cx - kStencil + k;
    } else {
      ix = cx - kStencil + k / kCols2;
      iy = cy - kStencil + k % kCols2;
      if (iy < 0 || iy >= T.nc[1]) return false;
    }
    if (ix < 0 || ix >= T.nc[0]) return false;
    const int nz = T.nc[L];
    const int z0 = max(w0, 0), z1 = min(w1, nz - 1);
    if (z0 > z1) return false;
    uint32_t row;
    if constexpr (DIM == 2) {
      row = T.cell_off + static_cast<uint32_t>(ix) * nz;
    } else {
      row = T.cell_off +
            (static_cast<uint32_t>(ix) * T.nc[1] + static_cast<uint32_t>(iy)) * nz;
    }
    b = coff[row + z0];
    e = coff[row + z1 + 1];
    return true;
  }
};

template <int DIM>
struct PairIn {
  double x[DIM];
  float4 pv;
  float2 aux;
  float vol;  // 3D with per-particle masses: m / rho
};

template <int DIM, int KERNEL, int FLAVOUR>
__device__ __forceinline__ void term_of(const DevParams& P, const Target<DIM>& a,
                                        const PairIn<DIM>& p, float& c, float* f) {
  double d[DIM];
#pragma unroll
  for (int q = 0; q < DIM; ++q) d[q] = p.x[q] - a.x[q];
  pair_term<DIM, KERNEL, FLAVOUR>(P, a, d, p.pv, p.aux.x, p.aux.y, p.vol, c, f);
}

template <int DIM, int KERNEL, int FLAVOUR>
__device__ __forceinline__ void sum_pair(const DevParams& P, const Target<DIM>& a,
                                         const PairIn<DIM>& p, Sums<DIM>& acc) {
  float c, f[DIM];
  term_of<DIM, KERNEL, FLAVOUR>(P, a, p, c, f);
  acc.add(c, f);
}

template <int DIM>
__device__ __forceinline__ bool within(const DevParams& P, const double* xb,
                                       const double* xa) {
  const double d0 = xb[0] - xa[0];
  double s = d0 * d0;
#pragma unroll
  for (int q = 1; q < DIM; ++q) {
    const double dq = xb[q] - xa[q];
    s = s + dq * dq;
  }
  return s <= P.R2;
}

// Candidate order, the same on every path so that all schedules produce the
// same bits: stencil columns in order, within a column ascending index; the
// accepted candidates' terms enter the compensated sums two at a time.
//
// Global-memory path, the same scheme with 32-candidate masks (the 3D stencil
// has 25 short column ranges): all columns' accepted candidates are summed
// in one loop per lane, in the common candidate order.
template <int DIM, int KERNEL, int FLAVOUR, int WORDS>
__device__ __forceinline__ void sum_words_g(const DevParams& P, const GlobalPos<DIM, WORDS>& ps,
                                            const DevState& S, const Target<DIM>& a,
                                            uint32_t n_acc, Sums<DIM>& acc) {
  const int lane = threadIdx.x & 63;
  int w = 0;
  uint32_t m = 0, m_next = ps.wm[lane], j0 = 0, j_next = ps.wj[lane];
  // the next of the n_acc accepted candidates (stored masks are never empty)
  auto take = [&](PairIn<DIM>& p) {
    if (m == 0) {
      m = m_next;
      j0 = j_next;
      w = min(w + 1, WORDS - 1);
      m_next = ps.wm[w * 64 + lane];
      j_next = ps.wj[w * 64 + lane];
    }
    const uint32_t j = j0 + static_cast<uint32_t>(__builtin_ctz(m));
    m &= m - 1u;
#pragma unroll
    for (int k = 0; k < DIM; ++k) p.x[k] = S.x[k][j];
    p.pv = S.pv[j];
    p.aux = S.aux[j];
    p.vol = (DIM == 3 && mass_flavour(FLAVOUR)) ? S.vol[j] : 0.0f;
  };
  uint32_t rem = n_acc;
  PairIn<DIM> A, B;
  if (rem == 0) return;
  if (acc.pend) {  // an odd term of an earlier batch of masks waits for its partner
    take(A);
    sum_pair<DIM, KERNEL, FLAVOUR>(P, a, A, acc);
    if (--rem == 0) return;
  }
  take(A);
  --rem;
  while (true) {
    const bool hb = rem > 0;
    if (hb) {
      take(B);
      --rem;
    }
    float ca, fa[DIM];
    term_of<DIM, KERNEL, FLAVOUR>(P, a, A, ca, fa);
    if (!hb) {
      acc.add(ca, fa);
      break;
    }
    const bool ha = rem > 0;
    if (ha) {
      take(A);
      --rem;
    }
    float cb, fb[DIM];
    term_of<DIM, KERNEL, FLAVOUR>(P, a, B, cb, fb);
    acc.add2(ca, fa, cb, fb);
    if (!ha) break;
  }
}

template <int DIM, int KERNEL, int FLAVOUR, int NCOL, int WORDS>
__device__ __forceinline__ void gather_words_g(const DevParams& P,
                                               const GlobalPos<DIM, WORDS>& ps, const DevState& S, const Target<DIM>& a,
                                               uint32_t i, int zc, const Windows<DIM, NCOL>& W,
                                               Sums<DIM>& acc, uint32_t& count) {
  const int lane = threadIdx.x & 63;
  int k = 0;
  uint32_t c0 = 0, e = 0;
  bool more = true;
  while (more) {
    int nw = 0;
    uint32_t n_acc = 0;
    while (nw < WORDS) {
      if (c0 >= e) {  // next non-empty column range
        bool found = false;
        for (; k < NCOL && !found; ++k) {
          const uint32_t v = W.get(k);
          if ((v & 7u) == 7u) continue;
          const int w0 = zc - kStencil + static_cast<int>(v & 7u);
          const int w1 = zc - kStencil + static_cast<int>(v >> 3);
          uint32_t b, eb;
          if (ps.range(k, w0, w1, b, eb) && b < eb) {
            found = true;
            c0 = b;
            e = eb;
          }
        }
        if (!found) {
          more = false;
          break;
        }
      }
      const uint32_t len = min(e - c0, 32u);
      uint32_t mask = 0;
      uint32_t t = 0;
      for (; t + 4 <= len; t += 4) {
        double x0[DIM], x1[DIM], x2[DIM], x3[DIM];
#pragma unroll
        for (int q = 0; q < DIM; ++q) {
          x0[q] = S.x[q][c0 + t];
          x1[q] = S.x[q][c0 + t + 1];
          x2[q] = S.x[q][c0 + t + 2];
          x3[q] = S.x[q][c0 + t + 3];
        }
        const uint32_t mm = (within<DIM>(P, x0, a.x) ? 1u : 0u) |
                            (within<DIM>(P, x1, a.x) ? 2u : 0u) |
                            (within<DIM>(P, x2, a.x) ? 4u : 0u) |
                            (within<DIM>(P, x3, a.x) ? 8u : 0u);
        mask |= mm << t;
      }
      for (; t < len; ++t) {
        double x0[DIM];
#pragma unroll
        for (int q = 0; q < DIM; ++q) x0[q] = S.x[q][c0 + t];
        if (within<DIM>(P, x0, a.x)) mask |= 1u << t;
      }
      if (i >= c0 && i < c0 + len) mask &= ~(1u << (i - c0));  // not self
      const uint32_t na = static_cast<uint32_t>(__builtin_popcount(mask));
      count += na;
      n_acc += na;
      if (mask) {
        ps.wm[nw * 64 + lane] = mask;
        ps.wj[nw * 64 + lane] = c0;
        ++nw;
      }
      c0 += len;
    }
    sum_words_g<DIM, KERNEL, FLAVOUR>(P, ps, S, a, n_acc, acc);
  }
}

__device__ __forceinline__ float wave_max_f32(float v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off));
  return v;
}

__device__ __forceinline__ unsigned long long wave_min_u64(unsigned long long v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const unsigned long long o = __shfl_xor(v, off);
    v = o < v ? o : v;
  }
  return v;
}

// Per-wave running reductions of a persistent loop: the chunks a wave takes
// in turn mostly belong to one tank, so the tank's slots are updated once per
// change of tank (and at the end) instead of once per chunk.
struct WaveReduce {
  uint32_t t = ~0u;
  float vmax = 0.0f;
  unsigned long long dtmin = ~0ull;
  __device__ __forceinline__ void flush(const StageArgs& A) {
    if (t == ~0u) return;
    if ((threadIdx.x & 63) == 0) {
      if (vmax > 0.0f) atomicMax(red_slot(A.vmax, t), __float_as_uint(vmax));
      if (dtmin != ~0ull) atomicMin(red_slot(A.dt_min, t), dtmin);
    }
    vmax = 0.0f;
    dtmin = ~0ull;
  }
  __device__ __forceinline__ void add(const StageArgs& A, uint32_t tank, float vm,
                                      unsigned long long dm) {
    if (tank != t) {
      flush(A);
      t = tank;
    }
    vmax = fmaxf(vmax, vm);
    dtmin = dm < dtmin ? dm : dtmin;
  }
};

struct ChunkInfo {
  uint32_t t, col_row, t0, t1;
  int cx, cy, nz;
  DevTank T;
};

template <int DIM>
__device__ __forceinline__ ChunkInfo chunk_info(const StageArgs& A, uint32_t q) {
  ChunkInfo c;
  const uint4 ch = A.chunks[q];
  const uint4 col = A.cols[ch.x];
  c.t = col.x;
  c.T = A.tanks[c.t];
  c.cx = static_cast<int>(col.y);
  c.cy = static_cast<int>(col.z);
  c.col_row = col.w;
  c.nz = c.T.nc[DIM - 1];
  c.t0 = ch.y;
  c.t1 = ch.z;
  return c;
}

// What finish_target reads of particle i, loaded together (loaded where each
// value is used, the 2M-particle 2D launch takes 295 us instead of 285).
template <int DIM>
struct TargetState {
  double x[DIM], v[DIM], rho;
  double ox[DIM], ov[DIM], orho;  // the step's start (combination stages)
  double dt;
};

template <int DIM, int KIND>
__device__ __forceinline__ void load_target(const StageArgs& A, uint32_t tank, uint32_t i,
                                            TargetState<DIM>& t) {
#pragma unroll
  for (int k = 0; k < DIM; ++k) {
    t.x[k] = A.in.x[k][i];
    t.v[k] = A.in.v[k][i];
    if constexpr (KIND == kCombine) {
      t.ox[k] = A.old.x[k][i];
      t.ov[k] = A.old.v[k][i];
    }
  }
  t.rho = A.in.rho[i];
  if constexpr (KIND == kCombine) t.orho = A.old.rho[i];
  if constexpr (KIND != kRhsOnly) t.dt = A.dt[tank];
}

// After the pair sums of one target (one lane): particle i's right-hand side
// (KIND kRhsOnly), or the SSPRK substep / combination of
// time_integrator.hpp:188-223 in FP64 and, on the last stage, the next step's
// CFL candidate.  Fixed particles keep their state.  The lane's speed and CFL
// candidate come back in vmax and dtmin for the per-wave reductions.
template <int DIM, int FLAVOUR, int KIND, bool FINAL>
__device__ __forceinline__ void finish_target(const StageArgs& A,
                                              const TargetState<DIM>& t, uint32_t i,
                                              bool in_range, bool fluid, const Sums<DIM>& acc,
                                              uint32_t count, float& vmax,
                                              unsigned long long& dtmin) {
  const DevParams& P = A.P;
  vmax = 0.0f;
  dtmin = ~0ull;
  if (in_range && !fluid) {
    if constexpr (KIND == kRhsOnly) {
      A.rhs_drho[i] = 0.0;
#pragma unroll
      for (int k = 0; k < DIM; ++k) A.rhs_dv[k][i] = 0.0;
      if (A.rhs_count) A.rhs_count[i] = 0u;
    } else {
#pragma unroll
      for (int k = 0; k < DIM; ++k) {
        A.out.x[k][i] = A.in.x[k][i];
        A.out.v[k][i] = 0.0;
      }
      A.out.rho[i] = A.in.rho[i];
      A.out.aux[i] = A.in.aux[i];
      A.out.pv[i] = A.in.pv[i];
      if constexpr (DIM == 3 && mass_flavour(FLAVOUR)) A.out.vol[i] = A.in.vol[i];
    }
  }
  if (fluid) {
    const double *xa = t.x, *va = t.v;
    const double rho_a = t.rho;
    if constexpr (KIND == kRhsOnly) {
      if (A.rhs_count) A.rhs_count[i] = count;
    }
    double drho = static_cast<double>(acc.rho.value());
    double dv[DIM];
#pragma unroll
    for (int k = 0; k < DIM; ++k) dv[k] = static_cast<double>(acc.v[k].value());
    if constexpr (FLAVOUR == kFlavourWall) {
      // face terms (already divided by gamma_a) + pair sums / gamma_a; none
      // without walls (per-particle masses alone)
      if (A.wall) {
        const double* wt = A.wall + 4 * static_cast<size_t>(i);
        const double ig = 1.0 / wt[3];
        drho = wt[0] + drho * ig;
#pragma unroll
        for (int k = 0; k < DIM; ++k) dv[k] = wt[1 + k] + dv[k] * ig;
      }
    }
    dv[1] = dv[1] - P.g;
    if constexpr (KIND == kRhsOnly) {
      A.rhs_drho[i] = drho;
#pragma unroll
      for (int k = 0; k < DIM; ++k) A.rhs_dv[k][i] = dv[k];
    } else {
      double v2 = 0.0;
#pragma unroll
      for (int k = 0; k < DIM; ++k) v2 = v2 + va[k] * va[k];
      vmax = static_cast<float>(sqrt(v2));
      const double h = t.dt;
      double rn[DIM], vn[DIM];
#pragma unroll
      for (int k = 0; k < DIM; ++k) {
        rn[k] = xa[k] + h * va[k];
        vn[k] = va[k] + h * dv[k];
      }
      double rhon = rho_a + h * drho;
      if constexpr (KIND == kCombine) {
        const double wn = A.w, wo = 1.0 - A.w;
#pragma unroll
        for (int k = 0; k < DIM; ++k) {
          rn[k] = wo * t.ox[k] + wn * rn[k];
          vn[k] = wo * t.ov[k] + wn * vn[k];
        }
        rhon = wo * t.orho + wn * rhon;
      }
#pragma unroll
      for (int k = 0; k < DIM; ++k) {
        A.out.x[k][i] = rn[k];
        A.out.v[k][i] = vn[k];
      }
      A.out.rho[i] = rhon;
      write_pair_data<DIM>(P, A.out, i, vn, rhon, P.mass ? P.mass[A.id[i]] : P.m);
      if constexpr (FINAL) {
        dtmin = dbl_bits(particle_time_step<DIM>(P, rhon, vn, dv));
        if (A.dv_last[0]) {  // kept for the time step after post-integration
#pragma unroll
          for (int k = 0; k < DIM; ++k) A.dv_last[k][i] = dv[k];
        }
      }
    }
  }
}

// Pair sums of one fluid target (one lane), particle i of cell column (cx, cy)
// (col_row: the global index of the column's first cell), every candidate from
// global memory.
template <int DIM, int KERNEL, int FLAVOUR, int WORDS>
__device__ __forceinline__ void sum_from_global(const StageArgs& A, const DevTank& T, int cx,
                                                int cy, uint32_t col_row, uint32_t i,
                                                const GlobalPos<DIM, WORDS>& ps, Sums<DIM>& acc,
                                                uint32_t& count) {
  constexpr int NCOL = DIM == 2 ? kCols2 : kCols2 * kCols2;
  const DevParams& P = A.P;
  double xa[DIM], va[DIM];
#pragma unroll
  for (int k = 0; k < DIM; ++k) {
    xa[k] = A.in.x[k][i];
    va[k] = A.in.v[k][i];
  }
  Target<DIM> a;
  make_target<DIM, FLAVOUR>(P, xa, va, A.in.rho[i], A.in.aux[i], a);
  const int zc = static_cast<int>(A.key[i] - col_row);
  const Windows<DIM, NCOL> W = stencil_windows<DIM, NCOL>(P, T, xa, cx, cy, zc);
  gather_words_g<DIM, KERNEL, FLAVOUR, NCOL>(P, ps, A.in, a, i, zc, W, acc, count);
  acc.finish();
}

// The per-wave reductions of one chunk's targets (all of one tank).
template <int KIND, bool FINAL>
__device__ __forceinline__ void reduce_chunk(const StageArgs& A, uint32_t tank, float vmax,
                                             unsigned long long dtmin, WaveReduce& red) {
  if constexpr (KIND != kRhsOnly) {
    const float vm = wave_max_f32(vmax);
    unsigned long long dm = ~0ull;
    if constexpr (FINAL) dm = wave_min_u64(dtmin);
    red.add(A, tank, vm, dm);
  }
}

// Targets of one column chunk, one per lane.
template <int DIM, int KERNEL, int FLAVOUR, int KIND, bool FINAL, int WORDS>
__device__ __forceinline__ void chunk_targets(const StageArgs& A, const ChunkInfo& c,
                                              const GlobalPos<DIM, WORDS>& ps, WaveReduce& red) {
  const uint32_t i = c.t0 + threadIdx.x;
  const bool in_range = i < c.t1;
  const uint32_t tag = in_range ? A.tag[i] : 1u;
  const bool fluid = in_range && !(tag & 1u);
  Sums<DIM> acc;
  acc.init();
  uint32_t count = 0;
  TargetState<DIM> ts;
  if (fluid) {
    sum_from_global<DIM, KERNEL, FLAVOUR>(A, c.T, c.cx, c.cy, c.col_row, i, ps, acc, count);
    load_target<DIM, KIND>(A, c.t, i, ts);
  }
  float vmax;
  unsigned long long dtmin;
  finish_target<DIM, FLAVOUR, KIND, FINAL>(A, ts, i, in_range, fluid, acc, count, vmax, dtmin);
  reduce_chunk<KIND, FINAL>(A, c.t, vmax, dtmin, red);
}

// Chunk indices handed out to a persistent grid.  Launch index b runs on XCD
// b % 8, whose eighth of the list is its band (so each XCD's L2 holds a
// contiguous band of columns): a workgroup starts on its own slot of the band
// and then draws from the band's counter, and when the band is finished from
// the other bands'.  A fixed share per workgroup left the 2M-particle 2D
// launch waiting: workgroups ended between 209 and 329 us.  The counters
// (kWorkStride apart, one cache line each) are cleared before the launch.
struct ChunkQueue {
  uint32_t n, slots, q;
  uint32_t k;  // bands given up so far (the own one first)
  __device__ __forceinline__ uint32_t band_end(uint32_t x) const {
    return static_cast<uint32_t>((static_cast<uint64_t>(n) * (x + 1)) / 8);
  }
  __device__ __forceinline__ uint32_t band_begin(uint32_t x) const {
    return static_cast<uint32_t>((static_cast<uint64_t>(n) * x) / 8);
  }
  // The workgroup's first chunk, ~0 if there is none (then no other band
  // has chunks left to draw either: every band is as long, to within one).
  __device__ __forceinline__ void init(uint32_t n_chunks) {
    n = n_chunks;
    slots = gridDim.x >> 3;
    k = 0;
    const uint32_t x = blockIdx.x & 7u;
    q = band_begin(x) + (blockIdx.x >> 3);
    if (q >= band_end(x)) q = ~0u;
  }
  // One thread draws: take() asks the current band's counter, before a
  // chunk's last part, so that the answer arrives during it (asked at the
  // chunk's start, every workgroup would hold a chunk it cannot begin, and
  // where a launch has few rounds the idle ones would find none left); next()
  // turns the answer into the next chunk, ~0 when every band is finished.  A
  // finished band is not asked again: 768 workgroups asking it for every
  // chunk wait for each other (11.5 ns per atomic on one address).
  __device__ __forceinline__ uint32_t take(uint32_t* work) const {
    const uint32_t x = (blockIdx.x + k) & 7u;
    if (k >= 8 || band_begin(x) + slots >= band_end(x)) return ~0u;  // no second round
    return atomicAdd(work + x * kWorkStride, 1u);
  }
  __device__ __forceinline__ uint32_t next(uint32_t* work, uint32_t r) {
    for (bool asked = true; k < 8; ++k, asked = false) {
      const uint32_t x = (blockIdx.x + k) & 7u;
      const uint32_t b = band_begin(x) + slots, e = band_end(x);
      if (b >= e) continue;
      if (!asked) r = atomicAdd(work + x * kWorkStride, 1u);
      if (r < e - b) return b + r;
    }
    return ~0u;
  }
};

struct Band {
  uint32_t lo, hi, step;
};
__device__ __forceinline__ Band xcd_band(uint32_t n) {
  const uint32_t x = blockIdx.x & 7u, slot = blockIdx.x >> 3;
  Band b;
  b.lo = static_cast<uint32_t>((static_cast<uint64_t>(n) * x) / 8) + slot;
  b.hi = static_cast<uint32_t>((static_cast<uint64_t>(n) * (x + 1)) / 8);
  b.step = gridDim.x >> 3;
  return b;
}

}  // namespace

}  // namespace tit_amd
