// Chunk lists of the tile kernels: one block's chunks.
#pragma once

#include "sph_kernels.hpp"

namespace tit_amd {

struct ChunkLimits {
  uint32_t targets, window;
  int rows;
};

template <int DIM>
__host__ __device__ __forceinline__ ChunkLimits chunk_limits(uint32_t chunk_targets,
                                                             uint32_t lds_cap) {
  if (DIM == 2) {
    // chunk_targets scales the tile from its full size at kChunkMax
    const uint32_t t = chunk_targets * kTileThreads / kChunkMax;
    // of the LDS entries, those between the window's columns hold no candidate
    constexpr uint32_t pad = kTilePad * (kBlk2 + 2 * kStencil);
    const uint32_t cap = lds_cap < kTileCap ? lds_cap : kTileCap;
    return ChunkLimits{t > 1u ? t : 1u, cap > pad ? cap - pad : 1u, kChunkRows2};
  }
  return ChunkLimits{kStage3Threads, lds_cap * kTile3Cap / kStage3LdsCap, kChunkRows3};
}

// Targets of a chunk that does not fit (several rows of it): one per lane.
constexpr uint32_t kOverTargets = kTileThreads;
static_assert(kStage3Threads == kTileThreads, "one limit for both tiles");

// LDS written by other lanes of this wave is visible after it.
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Scratch of the lanes that cut a block's chunks, for a segment of ROWS rows:
// T(z) and W(z), and per row that a chunk could begin at its end and the next
// one's start.
template <int ROWS>
struct ChunkScratch {
  static constexpr int kRows = ROWS;
  uint32_t T[kRows + 2 * kStencil + 1], W[kRows + 2 * kStencil + 1], cut[kRows];
  uint32_t z, count;
};

// Block chunks of block b (all LANES lanes: a wave, or a whole workgroup).
// Greedy from the block's first row: a chunk takes as many rows as keep its
// targets, its window's candidates and its rows within their limits; rows
// without targets are skipped at both ends.  A row beyond a limit by itself
// does not fit the LDS; consecutive such rows of at most kOverTargets targets
// together (one at least) form a chunk that takes its candidates from global
// memory, so that its lanes are busy.  T(z) and W(z): particles of the
// block's and of the window's columns below row z, each a sum of cell offsets
// (differences are the counts).  The lanes find, for every row a chunk could
// begin at, where it would end and the next one begin (T and W ascend, so by
// bisection), and one lane then follows the chain, one LDS read per chunk.
// The chunks go to the block's place in A.bcuts (a chunk per row at most);
// returns their number.
//
// Bound by latency: the list of 2M particles (366 blocks of 1,090 rows, 70
// chunks in a full one) takes 24 us; with a wave per block that found every
// chunk's end by ballots in turn, once to count and once to write, 114.
template <int DIM, int LANES, int ROWS>
__device__ __forceinline__ uint32_t block_chunks(const StageArgs& A, uint32_t b,
                                                 ChunkScratch<ROWS>& sc) {
  constexpr int BX = DIM == 2 ? kBlk2 : kBlk3, BY = DIM == 2 ? 1 : kBlk3;
  constexpr int S = kStencil, SY = DIM == 2 ? 0 : kStencil;
  constexpr int kRows = ROWS, kAhead = 64;
  static_assert(kRows < 65536 && kChunkRows2 <= kAhead && kChunkRows3 <= kAhead, "cut packs");
  auto sync = [] {
    if constexpr (LANES == 64) {
      wave_lds_sync();
    } else {
      __syncthreads();
    }
  };
  const ChunkLimits lim = chunk_limits<DIM>(A.chunk_targets, A.lds_cap);
  const uint4 blk = A.blocks[b];
  const DevTank T = A.tanks[blk.x];
  const int nz = T.nc[DIM - 1], ny = DIM == 2 ? 1 : T.nc[1];
  const int bx = static_cast<int>(blk.y), by = static_cast<int>(blk.z);
  const int lane = threadIdx.x & (LANES - 1);
  uint32_t count = 0;
  for (int seg = 0; seg < nz;) {  // uniform; every chunk before row seg is cut
    // sc.T[k], sc.W[k]: row seg - S + k, clamped to [0, nz]
    const int n_k = min(kRows + 2 * S, nz - seg + S) + 1;
    sync();
    for (int k = lane; k < n_k; k += LANES) {
      const uint32_t row = static_cast<uint32_t>(min(max(seg - S + k, 0), nz));
      uint32_t t = 0, w = 0;
#pragma unroll 2
      for (int dx = -S; dx < BX + S; ++dx) {
#pragma unroll
        for (int dy = -SY; dy < BY + SY; ++dy) {
          // a column outside the tank: any inside, as zero (all loads in flight)
          const int ix = bx + dx, iy = by + dy;
          const bool in = ix >= 0 && ix < T.nc[0] && iy >= 0 && iy < ny;
          const uint32_t col = in ? static_cast<uint32_t>(ix) * ny + iy : 0u;
          const uint32_t c = A.cell_off[T.cell_off + col * nz + row];
          const uint32_t v = in ? c : 0u;
          w += v;
          if (dx >= 0 && dx < BX && dy >= 0 && dy < BY) t += v;
        }
      }
      sc.T[k] = t;
      sc.W[k] = w;
    }
    sync();
    auto Tz = [&](int z) { return sc.T[min(z, nz) - seg + S]; };
    auto Wz = [&](int z) { return sc.W[min(max(z, 0), nz) - seg + S]; };
    // rows [seg, zl): a chunk's end, kAhead rows on at most, is in the segment
    const int zl = min(seg + kRows - kAhead + 1, nz);
    // the first row from z on that holds targets, zl if there is none before
    auto next_row = [&](int z) {
      const uint32_t t = Tz(z);
      if (Tz(z + 1) != t) return z;
      int lo = z, hi = zl;  // T(lo) == t; T(hi + 1) != t or hi == zl
      while (lo < hi) {
        const int mid = (lo + hi) / 2;
        if (Tz(mid + 1) != t) {
          hi = mid;
        } else {
          lo = mid + 1;
        }
      }
      return lo;
    };
    for (int z = seg + lane; z < zl; z += LANES) {
      const uint32_t t0 = Tz(z), w0 = Wz(z - S);
      if (Tz(z + 1) == t0) continue;
      // the last end row within the limits
      int lo = z, hi = min(z + lim.rows, nz);
      while (lo < hi) {
        const int mid = (lo + hi + 1) / 2;
        if (Tz(mid) - t0 <= lim.targets && Wz(mid + S) - w0 <= lim.window) {
          lo = mid;
        } else {
          hi = mid - 1;
        }
      }
      int end = lo;
      const bool over = end == z;
      if (over) {
        // and the rows after it that do not fit by themselves either
        ++end;
        while (end < min(z + kAhead, nz) && Tz(end + 1) - t0 <= kOverTargets &&
               (Tz(end + 1) - Tz(end) > lim.targets ||
                Wz(end + 1 + S) - Wz(end - S) > lim.window)) {
          ++end;
        }
      }
      while (Tz(end - 1) == Tz(end)) --end;  // (row z holds targets)
      const int next = end < zl ? next_row(end) : end;
      sc.cut[z - seg] = static_cast<uint32_t>(next - seg) |
                        static_cast<uint32_t>(end - z) << 16 | (over ? 1u : 0u) << 31;
    }
    const int z0 = next_row(seg);
    sync();
    if (lane == 0) {
      int z = z0;
      while (z < zl) {
        const uint32_t c = sc.cut[z - seg];
        const uint32_t end = static_cast<uint32_t>(z) + ((c >> 16) & 127u);
        A.bcuts[blk.w + count] = make_uint2(z, end | (c & (1u << 31)));
        ++count;
        z = seg + static_cast<int>(c & 0xffffu);
      }
      sc.z = static_cast<uint32_t>(z);
      sc.count = count;
    }
    sync();
    seg = static_cast<int>(sc.z);
    count = sc.count;
  }
  return count;
}

// Block b's chunks from A.bcuts to the list, from A.bcount[b] on (scanned; next:
// the following block's), by all lanes of a wave.
template <int DIM>
__device__ __forceinline__ void emit_block_chunks(const StageArgs& A, uint32_t b, uint32_t next) {
  const uint4 blk = A.blocks[b];
  const uint32_t base = A.bcount[b];
  for (uint32_t k = threadIdx.x & 63; base + k < next; k += 64) {
    const uint2 c = A.bcuts[blk.w + k];
    const uint32_t over = c.y >> 31, end = c.y & 0x7fffffffu;
    A.bchunks[base + k] = DIM == 2 ? make_uint4(blk.x | over << 31, blk.y, c.x, end)
                                   : make_uint4(b, c.x, end, over);
  }
}

}  // namespace tit_amd
