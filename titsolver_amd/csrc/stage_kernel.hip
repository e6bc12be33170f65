// Fused SSPRK stage kernel: continuity + momentum pair sums, EOS, update.
//
// Two families of work units, both recut on the device after every cell
// rebuild and taken by a persistent grid in XCD-major bands (launch index b
// runs on XCD b % 8 and takes chunks from that XCD's eighth of the list, so
// each XCD's L2 holds a contiguous band of columns):
//  - block chunks (schedules with LDS): the particles of a block of cell
//    columns over a few rows, the block's window staged in LDS: the tile
//    kernels of stage_tile.hip (2D) and stage_tile3.hip (3D), which draw
//    chunks from their band's queue and then from the others';
//  - column chunks (schedules without LDS): at most chunk_targets consecutive
//    (cell-sorted) particles of one cell column, positions from global memory,
//    a fixed share of the band for each workgroup.
// Every path visits a target's candidates in the same order and rounds
// identically, so all schedules produce the same bits.
#include "chunk_build.hpp"
#include "stage_common.hpp"

namespace tit_amd {

namespace {

// Column chunks with positions from global memory (schedules without LDS).
template <int DIM, int KERNEL, int FLAVOUR, int KIND, bool FINAL, int NT>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(3, 3))) void k_stage_global(
    StageArgs A) {
  __shared__ uint32_t s_wm[NT / 64][kWordsG * 64];
  __shared__ uint32_t s_wj[NT / 64][kWordsG * 64];
  const Band band = xcd_band(A.counts[0]);
  WaveReduce red;
  for (uint32_t q = band.lo; q < band.hi; q += band.step) {
    const ChunkInfo c = chunk_info<DIM>(A, q);
    const GlobalPos<DIM> ps{c.T,  A.in, A.cell_off, c.cx, c.cy, s_wm[threadIdx.x >> 6],
                            s_wj[threadIdx.x >> 6]};
    chunk_targets<DIM, KERNEL, FLAVOUR, KIND, FINAL>(A, c, ps, red);
  }
  red.flush(A);
}

// Chunks of the blocks, one workgroup each, and their counts.
template <int DIM, int LANES, int ROWS>
__global__ __launch_bounds__(LANES) void k_block_chunks(StageArgs A, const uint32_t* ctl) {
  if (!ctl[0]) return;
  __shared__ ChunkScratch<ROWS> sc;
  const uint32_t n = block_chunks<DIM, LANES>(A, blockIdx.x, sc);
  if (threadIdx.x == 0) A.bcount[blockIdx.x] = n;
}

// The blocks' chunks into one list (counts scanned), one wave per block.
constexpr int kEmitBlocks = 4;
template <int DIM>
__global__ __launch_bounds__(64 * kEmitBlocks) void k_block_emit(StageArgs A,
                                                                 const uint32_t* ctl) {
  if (!ctl[0]) return;
  const uint32_t b = blockIdx.x * kEmitBlocks + (threadIdx.x >> 6);
  if (b >= A.n_blocks) return;
  emit_block_chunks<DIM>(A, b, b + 1 < A.n_blocks ? A.bcount[b + 1] : A.counts[1]);
}

// ---- chunk list (after every cell rebuild) ----------------------------------

constexpr int kScanBlock = 1024;

// The chunks of a column, in order: the column's particles in
// ceil(n / chunk_targets) equal parts.
struct ColumnParts {
  uint32_t beg, n, nch;
};

__device__ __forceinline__ ColumnParts column_parts(const StageArgs& A, uint32_t col_i) {
  const uint4 col = A.cols[col_i];
  const DevTank& T = A.tanks[col.x];
  const int nz = T.nc[A.P.dim - 1];
  ColumnParts cp;
  cp.beg = A.cell_off[col.w];
  cp.n = A.cell_off[col.w + nz] - cp.beg;
  cp.nch = (cp.n + A.chunk_targets - 1) / A.chunk_targets;
  return cp;
}

// Exclusive scan over a 1024-thread block: wave shuffles, then the 16 wave
// totals.
__device__ __forceinline__ uint32_t block_excl_scan(uint32_t v, uint32_t* wsum,
                                                    uint32_t* total) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  uint32_t x = v;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const uint32_t y = __shfl_up(x, off);
    if (lane >= off) x += y;
  }
  if (lane == 63) wsum[wave] = x;
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t s = 0;
    for (int w = 0; w < kScanBlock / 64; ++w) {
      const uint32_t t = wsum[w];
      wsum[w] = s;
      s += t;
    }
    wsum[kScanBlock / 64] = s;
  }
  __syncthreads();
  const uint32_t r = wsum[wave] + x - v;
  *total = wsum[kScanBlock / 64];
  __syncthreads();
  return r;
}

// Chunk list in column order, in three passes, one wave per column: chunks
// per workgroup of columns; an exclusive scan of those (one workgroup, also
// writes the chunk count); each column's chunks at its scanned offset.
constexpr uint32_t kColsPerBlock = kScanBlock / 64;

__global__ __launch_bounds__(kScanBlock) void k_chunk_count(StageArgs A, uint32_t* block_tot,
                                                           const uint32_t* ctl) {
  if (!ctl[0]) return;
  __shared__ uint32_t wtot[kColsPerBlock];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint32_t c = blockIdx.x * kColsPerBlock + wave;
  if (lane == 0) wtot[wave] = c < A.n_cols ? column_parts(A, c).nch : 0u;
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t t = 0;
    for (uint32_t w = 0; w < kColsPerBlock; ++w) t += wtot[w];
    block_tot[blockIdx.x] = t;
  }
}

// Exclusive scan of n_blocks counts in place (one workgroup); *out = the total.
__global__ __launch_bounds__(kScanBlock) void k_chunk_base(uint32_t* block_tot, uint32_t n_blocks,
                                                          uint32_t* out, const uint32_t* ctl) {
  if (!ctl[0]) return;
  __shared__ uint32_t wsum[kScanBlock / 64 + 1];
  uint32_t base_off = 0;
  for (uint32_t base = 0; base < n_blocks; base += kScanBlock) {
    const uint32_t b = base + threadIdx.x;
    const uint32_t v = b < n_blocks ? block_tot[b] : 0u;
    uint32_t tot;
    const uint32_t off = base_off + block_excl_scan(v, wsum, &tot);
    if (b < n_blocks) block_tot[b] = off;
    base_off += tot;
  }
  if (threadIdx.x == 0) *out = base_off;
}

__global__ __launch_bounds__(kScanBlock) void k_chunk_emit(StageArgs A,
                                                          const uint32_t* block_tot,
                                                          const uint32_t* ctl) {
  if (!ctl[0]) return;
  __shared__ uint32_t wtot[kColsPerBlock];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint32_t c = blockIdx.x * kColsPerBlock + wave;
  // the counts again (the offsets need every earlier column's)
  const ColumnParts cp = c < A.n_cols ? column_parts(A, c) : ColumnParts{0u, 0u, 0u};
  if (lane == 0) wtot[wave] = cp.nch;
  __syncthreads();
  uint32_t off = block_tot[blockIdx.x];
  for (int w = 0; w < wave; ++w) off += wtot[w];
  for (uint32_t k = lane; k < cp.nch; k += 64) {
    auto part = [&](uint32_t q) {
      return cp.beg + static_cast<uint32_t>((static_cast<uint64_t>(cp.n) * q) / cp.nch);
    };
    A.chunks[off + k] = make_uint4(c, part(k), part(k + 1), 0u);
  }
}

// ---- dispatch -------------------------------------------------------------------

constexpr int kThreads = kChunkMax;

template <int DIM, int KERNEL, int FLAVOUR, int KIND, bool FINAL>
void launch_kind(hipStream_t s, const StageArgs& a) {
  k_stage_global<DIM, KERNEL, FLAVOUR, KIND, FINAL, kThreads><<<a.grid_global, kThreads, 0, s>>>(a);
}

template <int DIM, int KERNEL, int FLAVOUR>
void dispatch_kind(hipStream_t s, const StageArgs& a, int kind, bool final) {
  if (kind == kRhsOnly) {
    launch_kind<DIM, KERNEL, FLAVOUR, kRhsOnly, false>(s, a);
  } else if (kind == kEuler) {
    launch_kind<DIM, KERNEL, FLAVOUR, kEuler, false>(s, a);
  } else {
    if (final) {
      launch_kind<DIM, KERNEL, FLAVOUR, kCombine, true>(s, a);
    } else {
      launch_kind<DIM, KERNEL, FLAVOUR, kCombine, false>(s, a);
    }
  }
}

template <int DIM, int KERNEL>
void dispatch_flavour(hipStream_t s, const StageArgs& a, int kind, bool final) {
  if (a.P.flavour == kFlavourCfg) {
    dispatch_kind<DIM, KERNEL, kFlavourCfg>(s, a, kind, final);
  } else if (a.P.flavour == kFlavourWall) {
    dispatch_kind<DIM, KERNEL, kFlavourWall>(s, a, kind, final);
  } else if (a.P.flavour == kFlavourCfgM) {
    dispatch_kind<DIM, KERNEL, kFlavourCfgM>(s, a, kind, final);
  } else {
    dispatch_kind<DIM, KERNEL, kFlavourRef>(s, a, kind, final);
  }
}

template <int DIM>
void dispatch_kernel(hipStream_t s, const StageArgs& a, int kind, bool final) {
  if (a.P.kernel == kKernelC4) {
    dispatch_flavour<DIM, kKernelC4>(s, a, kind, final);
  } else {
    dispatch_flavour<DIM, kKernelC2>(s, a, kind, final);
  }
}

template <class F>
int occupancy(F* f, int threads = kThreads) {
  int n = 0;
  (void)hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, reinterpret_cast<const void*>(f),
                                                     threads, 0);
  return std::max(n, 1);
}

}  // namespace

uint32_t stage_lds_capacity(int dim) { return dim == 2 ? kStageLdsCap : kStage3LdsCap; }

void stage_grids(const DevParams& P, int n_cu, StageGrids* g) {
  int bt, bg;
  if (P.dim == 2) {
    bt = tile_groups_per_cu();
    bg = occupancy(k_stage_global<2, kKernelC2, kFlavourCfg, kCombine, false, kThreads>);
  } else {
    bt = tile3_groups_per_cu();
    bg = occupancy(k_stage_global<3, kKernelC2, kFlavourCfg, kCombine, false, kThreads>);
  }
  // multiples of 8: every XCD owns the same number of slots
  auto grid = [&](int per_cu) { return 8u * static_cast<uint32_t>((per_cu * n_cu + 7) / 8); };
  g->tile = grid(bt);
  g->global = grid(bg);
}

// 2D blocks of more rows than a wave holds at once get a wide workgroup where
// they are too few to fill the chip.  The whole list, a wave and a wide
// workgroup per block: 131,030 particles (92 blocks of 273 rows) 26 and 17 us,
// 2.0M (366 of 1,090) 69 and 24, 8.0M (732 of 2,180) 128 and 43.  Thousands of
// blocks fill it with a wave each.
constexpr uint32_t kWideBlocks = 1024;
constexpr int kWaveRows = 256;

void launch_build_chunks(hipStream_t s, const StageArgs& a, uint32_t* block_tot,
                         const uint32_t* ctl) {
  if (a.n_cols == 0) return;
  if (a.lds_cap > 0) {
    const uint32_t ne = (a.n_blocks + kEmitBlocks - 1) / kEmitBlocks;
    if (a.P.dim == 3) {
      k_block_chunks<3, 256, 1024><<<a.n_blocks, 256, 0, s>>>(a, ctl);
    } else if (a.block_rows > kWaveRows && a.n_blocks <= kWideBlocks) {
      k_block_chunks<2, 1024, 2048><<<a.n_blocks, 1024, 0, s>>>(a, ctl);
    } else {
      k_block_chunks<2, 64, kWaveRows><<<a.n_blocks, 64, 0, s>>>(a, ctl);
    }
    k_chunk_base<<<1, kScanBlock, 0, s>>>(a.bcount, a.n_blocks, a.counts + 1, ctl);
    if (a.P.dim == 2) {
      k_block_emit<2><<<ne, 64 * kEmitBlocks, 0, s>>>(a, ctl);
    } else {
      k_block_emit<3><<<ne, 64 * kEmitBlocks, 0, s>>>(a, ctl);
    }
  } else {
    const uint32_t nb = (a.n_cols + kColsPerBlock - 1) / kColsPerBlock;
    k_chunk_count<<<nb, kScanBlock, 0, s>>>(a, block_tot, ctl);
    k_chunk_base<<<1, kScanBlock, 0, s>>>(block_tot, nb, a.counts, ctl);
    k_chunk_emit<<<nb, kScanBlock, 0, s>>>(a, block_tot, ctl);
  }
}

// A chunk ends because the next row with targets would pass a limit.  By the
// target limit at most 2 n / targets times (two neighbouring chunks together
// pass it); by the row limit nz / rows times per block; by the window limit at
// most 14 n / window times: a particle is in the windows of at most two blocks
// per blocked axis and, along the rows, of at most seven chunks with their
// next row (those that begin within a stencil of it).  One more chunk per
// block.
size_t block_chunk_bound(int dim, size_t n, size_t n_blocks, size_t nz, uint32_t chunk_targets,
                         uint32_t lds_cap) {
  if (dim == 3) return std::min(n, n_blocks * nz) + 1;  // a row or more each
  const ChunkLimits l = chunk_limits<2>(chunk_targets, std::max(lds_cap, 1u));
  return std::min(n, 2 * n / l.targets + 14 * n / l.window +
                         n_blocks * (nz / static_cast<size_t>(l.rows) + 2)) + 1;
}

void launch_stage(hipStream_t s, const StageArgs& a, int kind, bool final) {
  if (a.n == 0 || a.n_cols == 0) return;
  if (a.lds_cap > 0) {
    if (a.P.dim == 2) {
      launch_stage_tile(s, a, kind, final);
    } else {
      launch_stage_tile3(s, a, kind, final);
    }
  } else if (a.P.dim == 2) {
    dispatch_kernel<2>(s, a, kind, final);
  } else {
    dispatch_kernel<3>(s, a, kind, final);
  }
}

}  // namespace tit_amd
