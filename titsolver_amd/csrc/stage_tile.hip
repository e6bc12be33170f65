// 2D stage kernel over tiles: continuity + momentum pair sums, EOS, update.
//
// Work unit: a chunk holds the particles of a block of kBlk2 adjacent cell
// columns over a few rows (at most kTileThreads of them, one per lane).  Its
// window, the block grown by the stencil on every side, is staged in LDS
// whole: FP64 positions and the FP32 pair records, 40 B per candidate, so the
// pair loop reads nothing from global memory.  A block of columns rather than
// a strip of one column because the window is what costs LDS: a 128-particle
// strip stages 5.9 candidates per target, a tile of 4 columns 2.7, which
// leaves room for the records and for three waves per SIMD.
//
// Each lane walks its own trimmed 5 x 5 stencil with the exact FP64 predicate
// and appends the accepted candidates' LDS indices to its list in LDS; then
// the FP32 pair terms run over the list, two at a time, the next entry's data
// loading while the current one is summed.  The list is emptied where the
// next column might not fit, between columns, so the lanes of a wave are at
// the same place.  Candidate order and rounding are those of the
// global-memory path (stage_common.hpp), so every schedule gives the same
// bits.
//
// Bound: VALU issue (96 % of the cycles at 2M particles: 1.55e8 wave
// instructions per launch; the compiled pair loop takes 43 per pair, the
// predicate 10.5 per candidate); the LDS is busy for 56 % of them, a third of
// that in bank conflicts.  The 2M-particle dam break's launch takes 281 us; strips of one column with
// acceptance masks in registers and the records gathered from L2 took 361 us
// and 1.71e8 (95 per pair).  Of that, drawing chunks from a queue instead of
// fixed shares gave 50 us.
#include "chunk_build.hpp"
#include "stage_common.hpp"

namespace tit_amd {

namespace {

constexpr int kWinC = kBlk2 + 2 * kStencil;    // window columns
constexpr int kRows2 = kChunkRows2 + 2 * kStencil;
constexpr int NT = kTileThreads;
// Entries after each window column's candidates that fail the predicate, so
// that a lane can test four candidates at a time past its range's end (past
// it in the same column lie rows beyond the stencil, which fail it too).
constexpr uint32_t kPad = kTilePad;
// Chunks that do not fit (h from 3.8 spacings on, and dense clumps) take their
// candidates from global memory, one lane per target, with the acceptance
// masks where the lists are: the column chunks' walk, trimmed stencils and
// four candidates' loads in flight.  us per launch at h = 4 and 5 spacings,
// with one candidate at a time of the whole stencil and one row per chunk,
// and now: 6,218 particles 312, 680 and 121, 207; 131,030 particles 391, 580
// and 249, 414.
constexpr int kOverWords = 11;
constexpr int kListLds = (kTileList + 2) * NT;
static_assert(kOverWords * 64 * 2 * (NT / 64) * sizeof(uint32_t) <= kListLds * sizeof(uint16_t),
              "masks fit the lists");

// Pair records as plain vectors (arrays of the HIP vector classes go to
// scratch memory here).
typedef __attribute__((ext_vector_type(4))) float Rec4;
typedef __attribute__((ext_vector_type(2))) float Rec2;

struct TileChunk {
  uint32_t tank;
  const DevTank* T;
  int bx;        // first cell column of the block
  int zs, ze;    // rows [zs, ze)
  bool over;     // the window or the targets exceed what the kernel holds
};

__device__ __forceinline__ TileChunk tile_chunk(const StageArgs& A, uint32_t q) {
  const uint4 ch = A.bchunks[q];
  TileChunk c;
  c.tank = ch.x & 0x7fffffffu;
  c.T = A.tanks + c.tank;
  c.bx = static_cast<int>(ch.y);
  c.zs = static_cast<int>(ch.z);
  c.ze = static_cast<int>(ch.w);
  c.over = (ch.x >> 31) != 0u;
  return c;
}

// The per-target values of the pair terms from the particle's own pair record
// (written with its state, so equal to make_target's).
template <int FLAVOUR>
__device__ __forceinline__ void target_of_record(const DevParams& P, double2 x, float4 pv,
                                                 float2 aux, Target<2>& a) {
  a.x[0] = x.x;
  a.x[1] = x.y;
  a.v[0] = pv.x;
  a.v[1] = pv.y;
  const float drho = pv.w;
  a.kd = P.kd * drho;
  if constexpr (FLAVOUR == kFlavourCfg || FLAVOUR == kFlavourCfgM) {
    a.rb = 0.5f * (P.rho0_f + drho) + 0.5f * P.rho0_f;
    a.cv = P.kv * aux.y;
  } else {
    a.rb = P.rho0_f + drho;
    a.cv = aux.y;
  }
  a.pa = mass_flavour(FLAVOUR) ? aux.x : P.mg * aux.x;
}

// Row windows of the five stencil columns of a target at cell (cx, zc): the
// rows whose cells, grown by skin/2, can hold a particle within R (in units
// of the cell size; the trimming of stencil.hpp in FP32, bounds widened by
// 1e-5 of a cell, from the position's fraction within its cell).  Windows
// that touch a border cell, which holds the particles clamped into it, are
// kept whole.
struct RowSpans {
  float g2x[2 * kStencil + 1];  // squared column gaps
  float tm2, tm1, tp1, tp2, t0; // column gap bounds of the rows zc - 2 .. zc + 2
};

__device__ __forceinline__ RowSpans row_spans(const DevParams& P, const DevTank& T, double2 x,
                                              int cx, int zc) {
  RowSpans s;
  const bool inner = cx - kStencil > 0 && cx + kStencil < T.nc[0] - 1 && zc - kStencil > 0 &&
                     zc + kStencil < T.nc[1] - 1;
  const float fx = static_cast<float>((x.x - T.lo[0]) * T.inv_c[0] - cx);
  const float fz = static_cast<float>((x.y - T.lo[1]) * T.inv_c[1] - zc);
  const float sx = static_cast<float>(P.skin_half * T.inv_c[0]) + 1e-5f;
  const float sz = static_cast<float>(P.skin_half * T.inv_c[1]) + 1e-5f;
  const float R = inner ? static_cast<float>(P.R2 * T.inv_c[0] * T.inv_c[0]) * (1.0f + 1e-5f)
                        : 1e30f;
  auto sq = [](float g) {
    g = fmaxf(g, 0.0f);
    return g * g;
  };
  s.g2x[0] = sq(fx + 1.0f - sx);
  s.g2x[1] = sq(fx - sx);
  s.g2x[2] = 0.0f;
  s.g2x[3] = sq(1.0f - fx - sx);
  s.g2x[4] = sq(2.0f - fx - sx);
  s.t0 = R;
  s.tm2 = R - sq(fz + 1.0f - sz);
  s.tm1 = R - sq(fz - sz);
  s.tp1 = R - sq(1.0f - fz - sz);
  s.tp2 = R - sq(2.0f - fz - sz);
  return s;
}

// Positions and pair records of the window, and the lane's list.
struct Tile {
  const double2* xy;
  const float4* pv;
  const float2* aux;
  uint16_t* list;  // this lane's entries: LDS index x 8, stride NT
};

__device__ __forceinline__ void tile_take(const Tile& t, uint32_t e, PairIn<2>& p) {
  const double2 x = *reinterpret_cast<const double2*>(reinterpret_cast<const char*>(t.xy) + 2 * e);
  p.x[0] = x.x;
  p.x[1] = x.y;
  p.pv = *reinterpret_cast<const float4*>(reinterpret_cast<const char*>(t.pv) + 2 * e);
  p.aux = *reinterpret_cast<const float2*>(reinterpret_cast<const char*>(t.aux) + e);
  p.vol = 0.0f;
}

// Sums the listed candidates, in twos; an odd last entry is kept for the next
// batch, or (last) enters as its sum with zero.  Entries cnt and cnt + 1 are
// set to a valid index first: the loop loads one entry ahead.  The scheduling
// barriers keep each entry's loads ahead of the other's arithmetic (left to
// itself the compiler gathers all of them at the loop's top and waits there).
template <int KERNEL, int FLAVOUR, bool LAST>
__device__ __forceinline__ void tile_flush(const DevParams& P, const Tile& t, const Target<2>& a,
                                           uint32_t self8, uint32_t& cnt, Sums<2>& acc) {
  t.list[cnt * NT] = static_cast<uint16_t>(self8);
  t.list[(cnt + 1) * NT] = static_cast<uint16_t>(self8);
  const uint32_t ne = cnt & ~1u;
  const uint16_t* p = t.list;
  PairIn<2> A, B;
  uint32_t ea = p[0], eb = p[NT];
  tile_take(t, ea, A);
  for (uint32_t k = 0; k < ne; k += 2) {
    p += 2 * NT;
    tile_take(t, eb, B);
    ea = p[0];
    eb = p[NT];
    __builtin_amdgcn_sched_barrier(0);
    float ca, fa[2], cb, fb[2];
    term_of<2, KERNEL, FLAVOUR>(P, a, A, ca, fa);
    __builtin_amdgcn_sched_barrier(0);
    tile_take(t, ea, A);
    __builtin_amdgcn_sched_barrier(0);
    term_of<2, KERNEL, FLAVOUR>(P, a, B, cb, fb);
    acc.add2(ca, fa, cb, fb);
  }
  if constexpr (LAST) {
    if (cnt & 1u) {
      float ca, fa[2];
      const float z[2] = {};
      term_of<2, KERNEL, FLAVOUR>(P, a, A, ca, fa);
      acc.add2(ca, fa, 0.0f, z);
    }
  } else {
    t.list[0] = static_cast<uint16_t>(ea);  // entry ne, when cnt is odd
    cnt &= 1u;
  }
}

// ---- four lanes per target ---------------------------------------------------
// A set too small to fill the chip is one latency chain per lane: about 100
// candidates tested and 25 term pairs summed in turn, 24.5 us a launch whatever
// the chunk length, 18.1 with this (kQuadN has the sizes).  There a target has
// the four lanes of a quad: each tests a
// contiguous quarter of a pass of 4 kQuadPart candidates (so that the quad's
// list keeps the candidate order), evaluates every fourth pair of terms, and
// all four add the pairs in order, taking each other's by DPP.  Same bits.
constexpr uint32_t kQuadPart = 6;
constexpr uint32_t kQuadStride = 174;  // entries per target (87 words: spreads the banks)
constexpr uint32_t kQuadList = kQuadStride - 2;
static_assert(kQuadStride * (NT / 4) <= (kTileList + 2) * NT && kQuadStride % 2 == 0,
              "lists of the quads fit those of the lanes, pairs word-aligned");

// Value of lane S of this lane's quad.
template <int S>
__device__ __forceinline__ uint32_t quad_lane(uint32_t v) {
  return static_cast<uint32_t>(
      __builtin_amdgcn_mov_dpp(static_cast<int>(v), S * 0x55, 0xf, 0xf, true));
}
template <int S>
__device__ __forceinline__ float quad_lane(float v) {
  return __uint_as_float(quad_lane<S>(__float_as_uint(v)));
}

// Adds lane S's pair sums if the quad has that pair.
template <int S>
__device__ __forceinline__ void quad_add(Sums<2>& acc, bool has, float c, float f0, float f1) {
  const float cs = quad_lane<S>(c), s0 = quad_lane<S>(f0), s1 = quad_lane<S>(f1);
  if (has) {
    acc.rho.add(cs);
    acc.v[0].add(s0);
    acc.v[1].add(s1);
  }
}

// tile_flush of a quad's list (t.list: its first entry; cnt the same in all
// four lanes).
template <int KERNEL, int FLAVOUR, bool LAST>
__device__ __forceinline__ void quad_flush(const DevParams& P, const Tile& t, const Target<2>& a,
                                           uint32_t& cnt, Sums<2>& acc) {
  wave_lds_sync();  // entries of the other lanes
  const uint32_t j = threadIdx.x & 3u, np = cnt >> 1;
  for (uint32_t p = 0; p < np; p += 4) {  // uniform in the quad
    const uint32_t w =
        reinterpret_cast<const uint32_t*>(t.list)[min(p + j, np - 1)];
    PairIn<2> A, B;
    tile_take(t, w & 0xffffu, A);
    tile_take(t, w >> 16, B);
    float ca, fa[2], cb, fb[2];
    term_of<2, KERNEL, FLAVOUR>(P, a, A, ca, fa);
    term_of<2, KERNEL, FLAVOUR>(P, a, B, cb, fb);
    const float c = ca + cb, f0 = fa[0] + fb[0], f1 = fa[1] + fb[1];
    quad_add<0>(acc, true, c, f0, f1);
    quad_add<1>(acc, p + 1 < np, c, f0, f1);
    quad_add<2>(acc, p + 2 < np, c, f0, f1);
    quad_add<3>(acc, p + 3 < np, c, f0, f1);
  }
  if (cnt & 1u) {
    const uint32_t e = t.list[cnt - 1];
    if constexpr (LAST) {
      PairIn<2> A;
      tile_take(t, e, A);
      float ca, fa[2];
      const float z[2] = {};
      term_of<2, KERNEL, FLAVOUR>(P, a, A, ca, fa);
      acc.add2(ca, fa, 0.0f, z);
    } else {
      wave_lds_sync();
      t.list[0] = static_cast<uint16_t>(e);  // all four lanes write the same
    }
  }
  if constexpr (!LAST) cnt &= 1u;
  wave_lds_sync();
}

// One column's range [l, le) (uniform in the quad).
template <int KERNEL, int FLAVOUR>
__device__ __forceinline__ void quad_column(const DevParams& P, const Tile& t,
                                            const Target<2>& a, uint32_t self, uint32_t l,
                                            uint32_t le, uint32_t& cnt, uint32_t& count,
                                            Sums<2>& acc) {
  const uint32_t j = threadIdx.x & 3u;
  while (__any(l < le)) {
    if (__any(cnt + 4 * kQuadPart > kQuadList)) {
      count += cnt & ~1u;
      quad_flush<KERNEL, FLAVOUR, false>(P, t, a, cnt, acc);
    }
    const uint32_t c0 = l + kQuadPart * j;
    double2 x[kQuadPart];
#pragma unroll
    for (uint32_t u = 0; u < kQuadPart; ++u) x[u] = t.xy[c0 + u < le ? c0 + u : self];
    uint32_t mask = 0;
#pragma unroll
    for (uint32_t u = 0; u < kQuadPart; ++u) {
      const double xb[2] = {x[u].x, x[u].y};
      // (a candidate past the range's end stands for the target itself)
      const bool ok = within<2>(P, xb, a.x) && c0 + u < le && c0 + u != self;
      mask |= ok ? 1u << u : 0u;
    }
    const uint32_t n = static_cast<uint32_t>(__builtin_popcount(mask));
    const uint32_t n0 = quad_lane<0>(n), n1 = quad_lane<1>(n), n2 = quad_lane<2>(n),
                   n3 = quad_lane<3>(n);
    uint32_t pos = cnt + (j > 0 ? n0 : 0u) + (j > 1 ? n1 : 0u) + (j > 2 ? n2 : 0u);
#pragma unroll
    for (uint32_t u = 0; u < kQuadPart; ++u) {  // the others go to the spare entry
      const bool ok = (mask >> u) & 1u;
      t.list[ok ? pos : kQuadStride - 1] = static_cast<uint16_t>((c0 + u) * 8);
      pos += ok ? 1u : 0u;
    }
    cnt += n0 + n1 + n2 + n3;
    l += 4 * kQuadPart;
  }
}

// Q: lanes per target, 1 or 4.
template <int KERNEL, int FLAVOUR, int KIND, bool FINAL, int Q>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(kTileWaves, kTileWaves))) void
k_stage_tile(StageArgs A) {
  __shared__ double2 s_xy[kTileCap + 8];  // a lane loads up to 8 past its range
  __shared__ float4 s_pv[kTileCap];
  __shared__ float2 s_aux[kTileCap];
  __shared__ __attribute__((aligned(4))) uint16_t s_list[kListLds];
  __shared__ uint16_t s_row[kWinC][kRows2 + 1];  // LDS index of each row's first candidate
  __shared__ uint32_t s_lb[kWinC + 1], s_d[kWinC];  // LDS index of each column; + d = global
  __shared__ uint32_t s_tb[kBlk2 + 1], s_first[kBlk2];  // targets before column; its first
  const DevParams& P = A.P;
  const int tid = threadIdx.x;
  __shared__ uint32_t s_next;
  ChunkQueue queue;
  queue.init(A.counts[1]);
  WaveReduce red;
  for (uint32_t q = queue.q; q != ~0u;) {
    const TileChunk c = tile_chunk(A, q);
    const DevTank& T = *c.T;
    const int nz = T.nc[1];
    const int zlo = max(c.zs - kStencil, 0), zhi = min(c.ze - 1 + kStencil, nz - 1);
    const int nrows = zhi - zlo + 1;
    const uint32_t per = c.over ? NT : NT / Q;            // targets of a round
    const uint32_t slot = c.over ? tid : tid / Q;         // this lane's
    const bool lead = Q == 1 || c.over || tid % Q == 0;   // the lane that updates it
    uint32_t drawn = ~0u;
    // target t of the chunk: its particle, column in the block, tag and row
    auto target_of = [&](uint32_t t, uint32_t& i, int& b, uint32_t& tag, int& zc) {
      i = 0;
      b = 0;
      tag = 1u;
      zc = zlo;
      if (t >= s_tb[kBlk2]) return;
#pragma unroll
      for (int u = 1; u < kBlk2; ++u) b += t >= s_tb[u] ? 1 : 0;
      i = s_first[b] + (t - s_tb[b]);
      tag = A.tag[i];
      zc = static_cast<int>(A.key[i] - T.cell_off - static_cast<uint32_t>(c.bx + b) * nz);
    };
    uint32_t i = 0, tag = 1u;
    int b = 0, zc = zlo;
    if (!c.over) {
      // wave 0, lane = window column: LDS offsets by a shuffle scan
      if (tid < 64) {
        uint32_t g0 = 0, len = 0, nb = 0, first = 0;
        const int ix = c.bx - kStencil + tid;
        if (tid < kWinC && ix >= 0 && ix < T.nc[0]) {
          const uint32_t* co = A.cell_off + T.cell_off + static_cast<uint32_t>(ix) * nz;
          g0 = co[zlo];
          len = co[zhi + 1] - g0 + kPad;
          if (tid >= kStencil && tid < kStencil + kBlk2) {
            first = co[c.zs];
            nb = co[c.ze] - first;
          }
        }
        uint32_t sl = len, sb = nb;
#pragma unroll
        for (int off = 1; off < kWinC; off <<= 1) {
          const uint32_t yl = __shfl_up(sl, off), yb = __shfl_up(sb, off);
          if (tid >= off) {
            sl += yl;
            sb += yb;
          }
        }
        if (tid < kWinC) {
          s_lb[tid] = sl - len;
          s_d[tid] = g0 - (sl - len);
          if (tid == kWinC - 1) s_lb[kWinC] = sl;
          if (tid >= kStencil && tid <= kStencil + kBlk2) s_tb[tid - kStencil] = sb - nb;
          if (tid >= kStencil && tid < kStencil + kBlk2) s_first[tid - kStencil] = first;
        }
      }
      __syncthreads();
      target_of(slot, i, b, tag, zc);  // its loads overlap the staging's
      for (int r = tid; r < kWinC * (nrows + 1); r += NT) {
        const int k = r / (nrows + 1), row = r % (nrows + 1);
        const int ix = c.bx - kStencil + k;
        uint32_t l = s_lb[k];
        if (ix >= 0 && ix < T.nc[0]) {
          l = A.cell_off[T.cell_off + static_cast<uint32_t>(ix) * nz + zlo + row] - s_d[k];
        }
        s_row[k][row] = static_cast<uint16_t>(l);
      }
      const uint32_t total = s_lb[kWinC];
      // every load of the window in flight before the first LDS write
      constexpr int kPer = (kTileCap + NT - 1) / NT;
      double2 gx[kPer];
      Rec4 gp[kPer];
      Rec2 ga[kPer];
      bool real[kPer];
#pragma unroll
      for (int v = 0; v < kPer; ++v) {
        const uint32_t l = tid + v * NT;
        int k = 0;
#pragma unroll
        for (int u = 1; u < kWinC; ++u) k += l >= s_lb[u] ? 1 : 0;
        real[v] = l + kPad < s_lb[k + 1];
        const uint32_t j = real[v] ? l + s_d[k] : 0u;  // (idle: any particle)
        gx[v] = make_double2(A.in.x[0][j], A.in.x[1][j]);
        gp[v] = reinterpret_cast<const Rec4*>(A.in.pv)[j];
        ga[v] = reinterpret_cast<const Rec2*>(A.in.aux)[j];
      }
#pragma unroll
      for (int v = 0; v < kPer; ++v) {
        const uint32_t l = tid + v * NT;
        if (real[v]) {
          s_xy[l] = gx[v];
          reinterpret_cast<Rec4*>(s_pv)[l] = gp[v];
          reinterpret_cast<Rec2*>(s_aux)[l] = ga[v];
        } else if (l < total) {
          s_xy[l] = make_double2(1e300, 1e300);
        }
      }
      __syncthreads();
    } else {
      if (tid == 0) {
        uint32_t nt = 0;
        for (int b = 0; b < kBlk2; ++b) {
          s_tb[b] = nt;
          s_first[b] = 0u;
          if (c.bx + b < T.nc[0]) {
            const uint32_t* co = A.cell_off + T.cell_off + static_cast<uint32_t>(c.bx + b) * nz;
            s_first[b] = co[c.zs];
            nt += co[c.ze] - co[c.zs];
          }
        }
        s_tb[kBlk2] = nt;
      }
      __syncthreads();
    }
    // targets, one per lane (a chunk that does not fit may need more rounds)
    const uint32_t n_t = s_tb[kBlk2];
    for (uint32_t base = 0; base < n_t; base += per) {
      if (c.over) target_of(base + slot, i, b, tag, zc);
      const bool in_range = base + slot < n_t, fluid = !(tag & 1u);
      const int cx = c.bx + b;
      Sums<2> acc;
      acc.init();
      uint32_t count = 0;
      if (!c.over && __any(fluid)) {
        Target<2> a;
        // its LDS index, in its row's range (a valid one for an idle lane)
        const uint32_t self = in_range ? i - s_d[b + kStencil] : s_lb[kStencil];
        const double2 xa = s_xy[self];
        target_of_record<FLAVOUR>(P, xa, s_pv[self], s_aux[self], a);
        const Tile tile{s_xy, s_pv, s_aux, Q == 1 ? s_list + tid : s_list + slot * kQuadStride};
        const RowSpans W = row_spans(P, T, xa, cx, zc);
        const uint32_t self8 = self * 8;
        uint32_t cnt = 0;
        // the five columns' ranges in order
#pragma unroll
        for (int k = 0; k < kCols2; ++k) {
          const float g2 = W.g2x[k];
          int f = zc - (g2 <= W.tm1 ? 1 : 0) - (g2 <= W.tm2 ? 1 : 0);
          int e = zc + 1 + (g2 <= W.tp1 ? 1 : 0) + (g2 <= W.tp2 ? 1 : 0);
          f = max(f, zlo);
          e = min(e, zhi + 1);
          uint32_t l = s_row[b + k][f - zlo], le = s_row[b + k][e - zlo];
          if (!fluid || !(g2 <= W.t0)) le = l;
          if constexpr (Q == 4) {
            quad_column<KERNEL, FLAVOUR>(P, tile, a, self, l, le, cnt, count, acc);
            continue;
          }
          do {
            // a range longer than the list in pieces (never on a lattice)
            const uint32_t lp = min(le, l + static_cast<uint32_t>(kTileList - 8));
            if (__any(cnt + ((lp - l + 3u) & ~3u) > static_cast<uint32_t>(kTileList))) {
              count += cnt & ~1u;
              tile_flush<KERNEL, FLAVOUR, false>(P, tile, a, self8, cnt, acc);
            }
            // two sets of four candidates in turn, the next one loading while
            // the current one is tested
            auto load = [&](double2* x, uint32_t l0) {
#pragma unroll
              for (int u = 0; u < 4; ++u) x[u] = s_xy[l0 + u];
              __builtin_amdgcn_sched_barrier(0);
            };
            auto test = [&](const double2* x) {
#pragma unroll
              for (int u = 0; u < 4; ++u) {
                const double xb[2] = {x[u].x, x[u].y};
                bool ok = within<2>(P, xb, a.x);
                if (k == kStencil) ok = ok && l + u != self;
                tile.list[cnt * NT] = static_cast<uint16_t>((l + u) * 8);
                cnt += ok ? 1u : 0u;
              }
              l += 4;
            };
            if (l < lp) {
              double2 x[4], y[4];
              load(x, l);
              while (true) {
                load(y, l + 4);
                test(x);
                if (l >= lp) break;
                load(x, l + 4);
                test(y);
                if (l >= lp) break;
              }
            }
          } while (__any(l < le));
        }
        count += cnt;
        if constexpr (Q == 4) {
          quad_flush<KERNEL, FLAVOUR, true>(P, tile, a, cnt, acc);
        } else {
          tile_flush<KERNEL, FLAVOUR, true>(P, tile, a, self8, cnt, acc);
        }
      } else if (c.over && fluid) {
        uint32_t* words = reinterpret_cast<uint32_t*>(s_list) + (tid >> 6) * kOverWords * 128;
        const GlobalPos<2, kOverWords> ps{T,  A.in, A.cell_off, cx, 0, words,
                                          words + kOverWords * 64};
        sum_from_global<2, KERNEL, FLAVOUR>(
            A, T, cx, 0, T.cell_off + static_cast<uint32_t>(cx) * nz, i, ps, acc, count);
      }
      float vmax;
      unsigned long long dtmin;
      if (tid == 0 && base + per >= n_t) drawn = queue.take(A.work);
      TargetState<2> ts;
      load_target<2, KIND>(A, c.tank, i, ts);
      finish_target<2, FLAVOUR, KIND, FINAL>(A, ts, i, in_range && lead, fluid && lead, acc,
                                             count, vmax, dtmin);
      reduce_chunk<KIND, FINAL>(A, c.tank, vmax, dtmin, red);
    }
    if (tid == 0) s_next = queue.next(A.work, drawn);
    __syncthreads();  // this chunk's LDS reads are done
    q = s_next;
  }
  red.flush(A);
}

template <int KERNEL, int FLAVOUR, int KIND, bool FINAL>
void launch_lanes(hipStream_t s, const StageArgs& a) {
  if (a.quad) {
    k_stage_tile<KERNEL, FLAVOUR, KIND, FINAL, 4><<<a.grid_tile, NT, 0, s>>>(a);
  } else {
    k_stage_tile<KERNEL, FLAVOUR, KIND, FINAL, 1><<<a.grid_tile, NT, 0, s>>>(a);
  }
}

template <int KERNEL, int FLAVOUR>
void launch_flavour(hipStream_t s, const StageArgs& a, int kind, bool final) {
  if (kind == kRhsOnly) {
    launch_lanes<KERNEL, FLAVOUR, kRhsOnly, false>(s, a);
  } else if (kind == kEuler) {
    launch_lanes<KERNEL, FLAVOUR, kEuler, false>(s, a);
  } else if (final) {
    launch_lanes<KERNEL, FLAVOUR, kCombine, true>(s, a);
  } else {
    launch_lanes<KERNEL, FLAVOUR, kCombine, false>(s, a);
  }
}

template <int KERNEL>
void launch_kernel(hipStream_t s, const StageArgs& a, int kind, bool final) {
  if (a.P.flavour == kFlavourCfg) {
    launch_flavour<KERNEL, kFlavourCfg>(s, a, kind, final);
  } else if (a.P.flavour == kFlavourWall) {
    launch_flavour<KERNEL, kFlavourWall>(s, a, kind, final);
  } else if (a.P.flavour == kFlavourCfgM) {
    launch_flavour<KERNEL, kFlavourCfgM>(s, a, kind, final);
  } else {
    launch_flavour<KERNEL, kFlavourRef>(s, a, kind, final);
  }
}

}  // namespace

int tile_groups_per_cu() {
  int n = 0;
  (void)hipOccupancyMaxActiveBlocksPerMultiprocessor(
      &n, reinterpret_cast<const void*>(k_stage_tile<kKernelC2, kFlavourCfg, kCombine, false, 1>), NT,
      0);
  return std::max(n, 1);
}

void launch_stage_tile(hipStream_t s, const StageArgs& a, int kind, bool final) {
  if (a.P.kernel == kKernelC4) {
    launch_kernel<kKernelC4>(s, a, kind, final);
  } else {
    launch_kernel<kKernelC2>(s, a, kind, final);
  }
}

}  // namespace tit_amd
