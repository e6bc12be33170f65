// 3D stage kernel over tiles: continuity + momentum pair sums, EOS, update.
//
// Work unit: a chunk holds the particles of a block of kBlk3 x kBlk3 cell
// columns over a few rows (at most kStage3Threads of them, one per lane); the
// FP64 positions of its window (the block grown by the stencil on every side)
// are staged in LDS.  Each lane walks its own trimmed 5^3 stencil column by
// column with the exact FP64 predicate and appends the accepted candidates to
// its list in LDS; when the next column might not fit, the FP32 pair terms run
// over the list, two at a time, the pair records coming from L2 one pair
// ahead.  (With the records in LDS too, as in 2D, a window would take 110 KB and
// leave one workgroup per CU.)  Candidate order and rounding are those of
// the global-memory path (stage_common.hpp), so every schedule gives the same
// bits.
//
// Bound: latency at two waves per SIMD (VALU issue takes 61 % of the cycles at
// 7.0e8 wave instructions per launch, the LDS 41 %, two fifths of that bank
// conflicts).  2M fluid particles at h = 1.3 spacings: 1,905 us per launch; with
// acceptance masks queued in registers, three workgroups per CU and fixed
// shares of the chunk list it took 2,610 us.  Tried: three workgroups with
// lists of 18 entries (2,430 us: the windows that fit cut chunks to 160
// targets on average), six waves per workgroup (2,775 us: the second
// workgroup does not fit beside the first on every SIMD).
//
// A list entry is the window column and the place in it (6 + 10 bits); the
// column's LDS and global bases come from a 64-entry table, so an entry gives
// both the position's and the records' address.
#include "stage_common.hpp"

namespace tit_amd {

namespace {

constexpr int NT = kStage3Threads;
constexpr int NW = kWin3 * kWin3;
constexpr int NB = kBlk3 * kBlk3;
static_assert(NW == 64, "one lane of a wave per window column");
static_assert(kTile3Cap <= 2040, "an LDS index takes 11 bits");
// Chunks that do not fit take their candidates from global memory (the column
// chunks' walk), with the acceptance masks where the lists are.  At h = 2
// spacings every interior window is one (about 3,400 candidates in one row):
// 1.5M particles take 5,750 us per launch, as many with one candidate at a
// time of the untrimmed stencil 7,610, column chunks 11,000 (their workgroups
// read one column's neighbourhood each).
constexpr int kOverWords = 16;
constexpr int kListLds = (kTile3List + 2) * NT;
static_assert(kOverWords * 64 * 2 * (NT / 64) * sizeof(uint32_t) <= kListLds * sizeof(uint16_t),
              "masks fit the lists");
constexpr uint32_t kColMax = 255;   // candidates of one window column at most
constexpr uint32_t kSpanMax = 1u << 27;  // global-index span of a window

struct Tile3 {
  const double *x, *y, *z;
  const uint2* base;   // per window column: LDS index, index in the records
  const float4* pv;    // records from the window's first particle on
  const float2* aux;
  const float* vol;
  uint16_t* list;      // this lane's entries, stride NT
};

template <int FLAVOUR>
__device__ __forceinline__ void tile_take3(const Tile3& t, uint32_t e, PairIn<3>& p) {
  const uint2 b = t.base[e >> 10];
  const uint32_t off = e & 1023u;
  const uint32_t l = b.x + off, j = b.y + off;
  p.x[0] = t.x[l];
  p.x[1] = t.y[l];
  p.x[2] = t.z[l];
  // 32-bit byte offsets from uniform bases
  p.pv = *reinterpret_cast<const float4*>(reinterpret_cast<const char*>(t.pv) + (j << 4));
  p.aux = *reinterpret_cast<const float2*>(reinterpret_cast<const char*>(t.aux) + (j << 3));
  p.vol = mass_flavour(FLAVOUR)
              ? *reinterpret_cast<const float*>(reinterpret_cast<const char*>(t.vol) + (j << 2))
              : 0.0f;
}

// The listed candidates in twos, the next entry's data loading while the
// current one is summed; an odd last entry is kept for the next batch, or
// (last) enters as its sum with zero.  Entries cnt and cnt + 1 are set to a
// valid one first.
template <int KERNEL, int FLAVOUR, bool LAST>
__device__ __forceinline__ void tile_flush3(const DevParams& P, const Tile3& t,
                                            const Target<3>& a, uint32_t self, uint32_t& cnt,
                                            Sums<3>& acc) {
  t.list[cnt * NT] = static_cast<uint16_t>(self);
  t.list[(cnt + 1) * NT] = static_cast<uint16_t>(self);
  const uint32_t ne = cnt & ~1u;
  const uint16_t* p = t.list;
  PairIn<3> A, B;
  uint32_t ea = p[0], eb = p[NT];
  tile_take3<FLAVOUR>(t, ea, A);
  for (uint32_t k = 0; k < ne; k += 2) {
    p += 2 * NT;
    tile_take3<FLAVOUR>(t, eb, B);
    ea = p[0];
    eb = p[NT];
    __builtin_amdgcn_sched_barrier(0);
    float ca, fa[3], cb, fb[3];
    term_of<3, KERNEL, FLAVOUR>(P, a, A, ca, fa);
    __builtin_amdgcn_sched_barrier(0);
    tile_take3<FLAVOUR>(t, ea, A);
    __builtin_amdgcn_sched_barrier(0);
    term_of<3, KERNEL, FLAVOUR>(P, a, B, cb, fb);
    acc.add2(ca, fa, cb, fb);
  }
  if constexpr (LAST) {
    if (cnt & 1u) {
      float ca, fa[3];
      const float z[3] = {};
      term_of<3, KERNEL, FLAVOUR>(P, a, A, ca, fa);
      acc.add2(ca, fa, 0.0f, z);
    }
  } else {
    t.list[0] = static_cast<uint16_t>(ea);  // entry ne, when cnt is odd
    cnt &= 1u;
  }
}

template <int KERNEL, int FLAVOUR, int KIND, bool FINAL>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(2, 2))) void k_stage_tile3(
    StageArgs A) {
  __shared__ double s_x[kTile3Cap + 8], s_y[kTile3Cap + 8], s_z[kTile3Cap + 8];
  __shared__ __attribute__((aligned(4))) uint16_t s_list[kListLds];
  __shared__ uint16_t s_row[NW][kRows3 + 1];  // LDS index of each row's first candidate
  __shared__ uint2 s_base[NW];
  __shared__ uint32_t s_lb[NW + 1], s_d[NW];  // LDS index of each column; + d = global
  __shared__ uint32_t s_tb[NB + 1], s_first[NB];  // targets before column; its first
  __shared__ uint32_t s_g0, s_next;
  __shared__ int s_fits;
  const DevParams& P = A.P;
  const int tid = threadIdx.x;
  ChunkQueue queue;
  queue.init(A.counts[1]);
  WaveReduce red;
  for (uint32_t q = queue.q; q != ~0u;) {
    const uint4 ch = A.bchunks[q];
    const uint4 blk = A.blocks[ch.x];
    const uint32_t tank = blk.x;
    const DevTank& T = A.tanks[tank];
    const int bx = static_cast<int>(blk.y), by = static_cast<int>(blk.z);
    const int zs = static_cast<int>(ch.y), ze = static_cast<int>(ch.z);
    const int nz = T.nc[2];
    const int zlo = max(zs - kStencil, 0), zhi = min(ze - 1 + kStencil, nz - 1);
    const int nrows = zhi - zlo + 1;
    uint32_t drawn = ~0u;
    // global index of the first particle of window column kw's row z
    auto column = [&](int kw) {
      const int ix = bx - kStencil + kw / kWin3, iy = by - kStencil + kw % kWin3;
      const bool in = ix >= 0 && ix < T.nc[0] && iy >= 0 && iy < T.nc[1];
      return in ? A.cell_off + T.cell_off +
                      (static_cast<uint32_t>(ix) * T.nc[1] + static_cast<uint32_t>(iy)) * nz
                : nullptr;
    };
    if (tid < 64) {
      // wave 0: LDS offsets of the window columns (lane = column) and the
      // targets of the block's columns, by shuffle scans
      uint32_t g0 = 0, len = 0, nb = 0, first = 0;
      const uint32_t* co = column(tid);
      if (co) {
        g0 = co[zlo];
        len = co[zhi + 1] - g0;
      }
      if (tid < NB) {
        const uint32_t* cb = column((kStencil + tid / kBlk3) * kWin3 + kStencil + tid % kBlk3);
        if (cb) {
          first = cb[zs];
          nb = cb[ze] - first;
        }
      }
      uint32_t sl = len, sb = nb, lo = len ? g0 : ~0u, hi = g0 + len, longest = len;
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) {
        const uint32_t yl = __shfl_up(sl, off), yb = __shfl_up(sb, off);
        if (tid >= off) {
          sl += yl;
          sb += yb;
        }
        lo = min(lo, __shfl_xor(lo, off));
        hi = max(hi, __shfl_xor(hi, off));
        longest = max(longest, __shfl_xor(longest, off));
      }
      s_lb[tid] = sl - len;
      s_d[tid] = g0 - (sl - len);
      // (an empty column: any record, an idle lane's entry may name it)
      s_base[tid] = make_uint2(sl - len, len ? g0 - lo : 0u);
      if (tid < NB) {
        s_tb[tid] = sb - nb;
        s_first[tid] = first;
      }
      if (tid == 63) {
        s_lb[NW] = sl;
        s_tb[NB] = sb;
        s_g0 = lo;
        s_fits = ch.w == 0u && nrows <= kRows3 && sl <= static_cast<uint32_t>(kTile3Cap) &&
                 sb <= static_cast<uint32_t>(NT) && longest <= kColMax && hi - lo < kSpanMax;
      }
    }
    __syncthreads();
    const bool fits = s_fits;
    const uint32_t n_t = s_tb[NB];
    // target t of the chunk: its particle, column in the block, tag and row
    uint32_t i = 0, tag = 1u;
    int b = 0, zc = zlo;
    auto target_of = [&](uint32_t t) {
      i = 0;
      b = 0;
      tag = 1u;
      zc = zlo;
      if (t >= n_t) return;
#pragma unroll
      for (int u = 1; u < NB; ++u) b += t >= s_tb[u] ? 1 : 0;
      i = s_first[b] + (t - s_tb[b]);
      tag = A.tag[i];
      zc = static_cast<int>(
          A.key[i] - T.cell_off -
          (static_cast<uint32_t>(bx + b / kBlk3) * T.nc[1] + static_cast<uint32_t>(by + b % kBlk3)) *
              nz);
    };
    if (fits) {
      target_of(tid);  // its loads overlap the staging's
      for (int r = tid; r < NW * (nrows + 1); r += NT) {
        const int kw = r & (NW - 1), row = r / NW;
        const uint32_t* co = column(kw);
        s_row[kw][row] = static_cast<uint16_t>(co ? co[zlo + row] - s_d[kw] : s_lb[kw]);
      }
      // each window column's candidates by 32 lanes (a column holds about 30)
      for (int r = tid; r < NW * 32; r += NT) {
        const int kw = r >> 5;
        const uint32_t e = s_lb[kw + 1], d = s_d[kw];
        for (uint32_t l = s_lb[kw] + (r & 31); l < e; l += 32) {
          const uint32_t j = l + d;
          s_x[l] = A.in.x[0][j];
          s_y[l] = A.in.x[1][j];
          s_z[l] = A.in.x[2][j];
        }
      }
    }
    __syncthreads();
    // targets, one per lane (a chunk that does not fit may need more rounds)
    for (uint32_t base = 0; base < n_t; base += NT) {
      if (!fits) target_of(base + tid);
      const bool in_range = base + tid < n_t, fluid = !(tag & 1u);
      Sums<3> acc;
      acc.init();
      uint32_t count = 0;
      if (fits && __any(fluid)) {
        const int bxq = b / kBlk3, byq = b % kBlk3;
        const int kself = (bxq + kStencil) * kWin3 + byq + kStencil;
        // its LDS index and list entry (a valid one for an idle lane)
        const uint32_t self = in_range ? i - s_d[kself] : s_lb[kself];
        const uint32_t self_e = static_cast<uint32_t>(kself) << 10 | (self - s_lb[kself]);
        Target<3> a;
        a.x[0] = s_x[self];
        a.x[1] = s_y[self];
        a.x[2] = s_z[self];
        {
          // make_target's values from the particle's own pair record
          const float4 pv = A.in.pv[i];
          const float2 aux = A.in.aux[i];
          a.v[0] = pv.x;
          a.v[1] = pv.y;
          a.v[2] = pv.z;
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
        const Tile3 tile{s_x, s_y, s_z, s_base, A.in.pv + s_g0, A.in.aux + s_g0,
                         mass_flavour(FLAVOUR) ? A.in.vol + s_g0 : nullptr, s_list + tid};
        // the rows that can hold a neighbour, from squared gaps in cells
        // (stencil.hpp in FP32, bounds widened by 1e-5 of a cell); windows
        // that touch a border cell are kept whole
        const int cx = bx + bxq, cy = by + byq;
        const bool inner = cx - kStencil > 0 && cx + kStencil < T.nc[0] - 1 &&
                           cy - kStencil > 0 && cy + kStencil < T.nc[1] - 1 &&
                           zc - kStencil > 0 && zc + kStencil < nz - 1;
        const float fx = static_cast<float>((a.x[0] - T.lo[0]) * T.inv_c[0] - cx);
        const float fy = static_cast<float>((a.x[1] - T.lo[1]) * T.inv_c[1] - cy);
        const float fz = static_cast<float>((a.x[2] - T.lo[2]) * T.inv_c[2] - zc);
        const float sk = static_cast<float>(P.skin_half * T.inv_c[0]) + 1e-5f;
        const float R =
            inner ? static_cast<float>(P.R2 * T.inv_c[0] * T.inv_c[0]) * (1.0f + 1e-5f) : 1e30f;
        auto sq = [](float g) {
          g = fmaxf(g, 0.0f);
          return g * g;
        };
        // squared gap to the cells d away along an axis, at fraction f
        auto gap2 = [&](int d, float f) {
          const float dd = static_cast<float>(d);
          return d == 0 ? 0.0f : sq((d < 0 ? f - 1.0f - dd : dd - f) - sk);
        };
        const float tm2 = R - gap2(-2, fz), tm1 = R - gap2(-1, fz), tp1 = R - gap2(1, fz),
                    tp2 = R - gap2(2, fz);
        uint32_t cnt = 0;
        // The 25 columns in order, the target's own in two parts around it.
        // A cell is 1.43 spacings wide at h = 1.3 spacings, so a column holds
        // 1, 2 or 4 lattice lines and the lanes' ranges of one column differ
        // up to fourfold; over the five columns of a plane they even out.  So
        // the ranges of a plane are queued in registers and each lane goes
        // through its own queue (180 -> 105 passes of four candidates).
#pragma unroll 1
        for (int dx = 0; dx < kCols2; ++dx) {
          const float g2x = gap2(dx - kStencil, fx);
          uint32_t rq[kCols2 + 1] = {};  // LDS index | length << 11 | window column << 19
          auto push = [&](bool on, uint32_t v) {
#pragma unroll
            for (int u = kCols2; u > 0; --u) rq[u] = on ? rq[u - 1] : rq[u];
            rq[0] = on ? v : rq[0];
          };
#pragma unroll
          for (int dy = kCols2 - 1; dy >= 0; --dy) {  // the last is the first out
            const float g2 = g2x + gap2(dy - kStencil, fy);
            const int kw = (bxq + dx) * kWin3 + byq + dy;
            int f = zc - (g2 <= tm1 ? 1 : 0) - (g2 <= tm2 ? 1 : 0);
            int e = zc + 1 + (g2 <= tp1 ? 1 : 0) + (g2 <= tp2 ? 1 : 0);
            f = max(f, zlo);
            e = min(e, zhi + 1);
            const uint32_t l = s_row[kw][f - zlo], le = s_row[kw][e - zlo];
            const uint32_t tagk = static_cast<uint32_t>(kw) << 19;
            const bool on = fluid && g2 <= R;
            if (dy == kStencil && dx == kStencil) {
              push(on && self + 1 < le, (self + 1) | (le - self - 1) << 11 | tagk);
              push(on && l < self, l | (self - l) << 11 | tagk);
            } else {
              push(on && l < le, l | (le - l) << 11 | tagk);
            }
          }
          uint32_t l = 0, le = 0, et = 0;  // et: list entry of LDS index 0
          while (true) {
            if (l >= le) {  // the next range, an empty one when none is left
              const uint32_t r = rq[0];
#pragma unroll
              for (int u = 0; u < kCols2; ++u) rq[u] = rq[u + 1];
              rq[kCols2] = 0u;
              const uint32_t kw = r >> 19;
              l = r & 2047u;
              le = l + ((r >> 11) & 255u);
              et = (kw << 10) - s_lb[kw];
            }
            if (!__any(l < le)) break;
            if (__any(cnt > static_cast<uint32_t>(kTile3List - 4))) {
              count += cnt & ~1u;
              tile_flush3<KERNEL, FLAVOUR, false>(P, tile, a, self_e, cnt, acc);
            }
            double x[4], y[4], z[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
              x[u] = s_x[l + u];
              y[u] = s_y[l + u];
              z[u] = s_z[l + u];
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) {
              const double xb[3] = {x[u], y[u], z[u]};
              tile.list[cnt * NT] = static_cast<uint16_t>(et + l + u);
              cnt += within<3>(P, xb, a.x) && l + u < le ? 1u : 0u;
            }
            l += 4;
          }
        }
        count += cnt;
        tile_flush3<KERNEL, FLAVOUR, true>(P, tile, a, self_e, cnt, acc);
      } else if (!fits && fluid) {
        const int cx = bx + b / kBlk3, cy = by + b % kBlk3;
        uint32_t* words = reinterpret_cast<uint32_t*>(s_list) + (tid >> 6) * kOverWords * 128;
        const GlobalPos<3, kOverWords> ps{T,  A.in, A.cell_off, cx, cy, words,
                                          words + kOverWords * 64};
        sum_from_global<3, KERNEL, FLAVOUR>(
            A, T, cx, cy,
            T.cell_off + (static_cast<uint32_t>(cx) * T.nc[1] + static_cast<uint32_t>(cy)) * nz, i,
            ps, acc, count);
      }
      if (tid == 0 && base + NT >= n_t) drawn = queue.take(A.work);
      TargetState<3> ts;
      load_target<3, KIND>(A, tank, i, ts);
      float vmax;
      unsigned long long dtmin;
      finish_target<3, FLAVOUR, KIND, FINAL>(A, ts, i, in_range, fluid, acc, count, vmax, dtmin);
      reduce_chunk<KIND, FINAL>(A, tank, vmax, dtmin, red);
    }
    if (tid == 0) s_next = queue.next(A.work, drawn);
    __syncthreads();  // this chunk's LDS reads are done
    q = s_next;
  }
  red.flush(A);
}

template <int KERNEL, int FLAVOUR>
void launch_flavour(hipStream_t s, const StageArgs& a, int kind, bool final) {
  if (kind == kRhsOnly) {
    k_stage_tile3<KERNEL, FLAVOUR, kRhsOnly, false><<<a.grid_tile, NT, 0, s>>>(a);
  } else if (kind == kEuler) {
    k_stage_tile3<KERNEL, FLAVOUR, kEuler, false><<<a.grid_tile, NT, 0, s>>>(a);
  } else if (final) {
    k_stage_tile3<KERNEL, FLAVOUR, kCombine, true><<<a.grid_tile, NT, 0, s>>>(a);
  } else {
    k_stage_tile3<KERNEL, FLAVOUR, kCombine, false><<<a.grid_tile, NT, 0, s>>>(a);
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

int tile3_groups_per_cu() {
  int n = 0;
  (void)hipOccupancyMaxActiveBlocksPerMultiprocessor(
      &n, reinterpret_cast<const void*>(k_stage_tile3<kKernelC2, kFlavourCfg, kCombine, false>),
      NT, 0);
  return std::max(n, 1);
}

void launch_stage_tile3(hipStream_t s, const StageArgs& a, int kind, bool final) {
  if (a.P.kernel == kKernelC4) {
    launch_kernel<kKernelC4>(s, a, kind, final);
  } else {
    launch_kernel<kKernelC2>(s, a, kind, final);
  }
}

}  // namespace tit_amd
