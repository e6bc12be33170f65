// Chunk lists of the tile kernels: one block's chunks, cut by one wave.
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
constexpr int kSegRows = 256;

// One wave's scratch: T(z) and W(z) of a segment of rows.
struct ChunkScratch {
  uint32_t T[kSegRows + 2 * kStencil + 1], W[kSegRows + 2 * kStencil + 1];
};

// LDS written by other lanes of this wave is visible after it.
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Block chunks of block b (all 64 lanes of a wave).  Greedy from the block's
// first row: a chunk takes as many rows as keep its targets, its window's
// candidates and its rows within their limits, the lanes testing the possible
// end rows at once; rows without targets are skipped at both ends.  A row
// beyond a limit by itself does not fit the LDS; consecutive such rows of at
// most kOverTargets targets together (one at least) form a chunk that takes
// its candidates from global memory, so that its lanes are busy.  T(z) and
// W(z): particles of the block's and of the window's columns below row z, each
// a sum of cell offsets (differences are the counts), for a segment of rows in
// LDS.  With emit, the chunks are
// written from `base` on.  Returns their number.
template <int DIM>
__device__ __forceinline__ uint32_t block_chunks(const StageArgs& A, uint32_t b, bool emit,
                                                 uint32_t base, ChunkScratch& sc) {
  constexpr int BX = DIM == 2 ? kBlk2 : kBlk3, BY = DIM == 2 ? 1 : kBlk3;
  constexpr int S = kStencil, SY = DIM == 2 ? 0 : kStencil;
  const ChunkLimits lim = chunk_limits<DIM>(A.chunk_targets, A.lds_cap);
  const uint4 blk = A.blocks[b];
  const DevTank T = A.tanks[blk.x];
  const int nz = T.nc[DIM - 1], ny = DIM == 2 ? 1 : T.nc[1];
  const int bx = static_cast<int>(blk.y), by = static_cast<int>(blk.z);
  const int lane = threadIdx.x & 63;
  int seg = 0;  // sc.T[k], sc.W[k]: row seg - S + k, clamped to [0, nz]
  auto load = [&](int z) {
    seg = z;
    wave_lds_sync();
    for (int k = lane; k < kSegRows + 2 * S + 1; k += 64) {
      const uint32_t row = static_cast<uint32_t>(min(max(seg - S + k, 0), nz));
      uint32_t t = 0, w = 0;
      for (int dx = -S; dx < BX + S; ++dx) {
        for (int dy = -SY; dy < BY + SY; ++dy) {
          const int ix = bx + dx, iy = by + dy;
          if (ix < 0 || ix >= T.nc[0] || iy < 0 || iy >= ny) continue;
          const uint32_t v =
              A.cell_off[T.cell_off + (static_cast<uint32_t>(ix) * ny + iy) * nz + row];
          w += v;
          if (dx >= 0 && dx < BX && dy >= 0 && dy < BY) t += v;
        }
      }
      sc.T[k] = t;
      sc.W[k] = w;
    }
    wave_lds_sync();
  };
  auto Tz = [&](int z) { return sc.T[min(z, nz) - seg + S]; };
  auto Wz = [&](int z) { return sc.W[min(max(z, 0), nz) - seg + S]; };
  load(0);
  uint32_t count = 0;
  int z = 0;
  while (z < nz) {  // uniform over the wave
    if (z + 64 > seg + kSegRows) load(z);
    // rows z .. z + 63 with targets
    uint64_t m = __ballot(Tz(z + lane + 1) != Tz(z + lane));
    if (m == 0) {
      z += 64;
      continue;
    }
    const int skip = __builtin_ctzll(m);
    if (skip > 0) {
      z += skip;
      continue;
    }
    // end rows z + 1 .. z + 64; the tests hold up to the chunk's end
    const int e = z + 1 + lane;
    const bool ok = lane < lim.rows && e <= nz && Tz(e) - Tz(z) <= lim.targets &&
                    Wz(e + S) - Wz(z - S) <= lim.window;
    uint64_t fit = ~__ballot(ok);
    const uint32_t over = (fit & 1ull) ? 1u : 0u;
    if (over) {
      // and the rows after it that do not fit by themselves either
      const bool with = e <= nz && Tz(e) - Tz(z) <= kOverTargets &&
                        (Tz(e) - Tz(e - 1) > lim.targets || Wz(e + S) - Wz(e - 1 - S) > lim.window);
      fit = ~__ballot(with);
    }
    const int rows = fit == 0 ? 64 : max(1, static_cast<int>(__builtin_ctzll(fit)));
    m &= rows < 64 ? (1ull << rows) - 1ull : ~0ull;
    const int end = z + 64 - __builtin_clzll(m);
    if (emit && lane == 0) {
      A.bchunks[base + count] = DIM == 2 ? make_uint4(blk.x | over << 31, blk.y, z, end)
                                         : make_uint4(b, z, end, over);
    }
    ++count;
    z = end;
  }
  return count;
}

}  // namespace tit_amd
