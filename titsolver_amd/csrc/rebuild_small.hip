// Cell-index rebuild of a small particle set in one launch.
//
// A step holds its rebuild unconditionally, and most steps do not need it, so
// what the rebuild costs there is its launches: the large form's chain of 17
// to 20 (keys, three per radix pass, gather, copy back, cell offsets, listing,
// chunks) takes about 2 us each in a replayed graph even when every kernel
// returns at once, 40 us of a 150 us step at 5,000 particles.  One workgroup
// of 16 waves does the whole sequence for up to kSmallN particles and
// kSmallCells cells, with the keys sorted in LDS (key and source slot packed
// in 32 bits).  One CU's latency costs more per rebuild than the chain's:
// beyond that, and where many steps rebuild, the chain runs (sph_kernels.hpp
// has the figures).
//
// Same results as the large form: the same keys, a stable sort by cell, the
// same offsets, lists (in another order where the order is irrelevant) and
// chunks.
#include "chunk_build.hpp"
#include "index_common.hpp"

namespace tit_amd {

namespace {

constexpr int NT = 1024;
constexpr int kWaves = NT / 64;
constexpr int kRadix = 256;
static_assert(kSmallN <= 65536 && kSmallCells <= 65536, "key and slot pack into 32 bits");

struct SortScratchLds {
  uint32_t item[kSmallN];         // key << 16 | source slot
  uint32_t cnt[kWaves][kRadix];
};

// The lanes of the wave (among `valid`) whose digit equals this lane's.
__device__ __forceinline__ uint64_t match8(uint32_t d, uint64_t valid) {
  uint64_t peers = valid;
#pragma unroll
  for (int b = 0; b < 8; ++b) {
    const bool bit = (d >> b) & 1u;
    const uint64_t bal = __ballot(bit);
    peers &= bit ? bal : ~bal;
  }
  return peers;
}

// Exclusive scan over the workgroup; *total the sum.
__device__ __forceinline__ uint32_t group_scan(uint32_t v, uint32_t* wsum, uint32_t* total) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  uint32_t x = v;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const uint32_t y = __shfl_up(x, off);
    if (lane >= off) x += y;
  }
  __syncthreads();
  if (lane == 63) wsum[wave] = x;
  __syncthreads();
  uint32_t before = 0, sum = 0;
  for (int w = 0; w < kWaves; ++w) {
    before += w < wave ? wsum[w] : 0u;
    sum += wsum[w];
  }
  *total = sum;
  return before + x - v;
}

// One stable pass by the 8 bits at `shift`: digit counts per wave, each
// digit's first place per wave, then the items to their places.
__device__ __forceinline__ void sort_pass(SortScratchLds& S, uint32_t* wsum, const uint32_t* src,
                                          uint32_t* dst, uint32_t n, uint32_t rounds, int shift) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const uint32_t first = wave * rounds * 64 + lane;
  __syncthreads();
  for (int d = tid; d < kWaves * kRadix; d += NT) S.cnt[d / kRadix][d % kRadix] = 0u;
  __syncthreads();
  for (uint32_t r = 0; r < rounds; ++r) {
    const bool ok = first + r * 64 < n;
    const uint32_t d = ok ? (src[first + r * 64] >> shift) & (kRadix - 1) : 0u;
    const uint64_t peers = match8(d, __ballot(ok));
    if (ok && (peers & ((1ull << lane) - 1ull)) == 0) {
      atomicAdd(&S.cnt[wave][d], static_cast<uint32_t>(__popcll(peers)));
    }
  }
  __syncthreads();
  uint32_t sum = 0, total;
  if (tid < kRadix) {
    for (int w = 0; w < kWaves; ++w) sum += S.cnt[w][tid];
  }
  uint32_t at = group_scan(sum, wsum, &total);
  if (tid < kRadix) {
    for (int w = 0; w < kWaves; ++w) {
      const uint32_t t = S.cnt[w][tid];
      S.cnt[w][tid] = at;
      at += t;
    }
  }
  __syncthreads();
  for (uint32_t r = 0; r < rounds; ++r) {
    const bool ok = first + r * 64 < n;
    const uint32_t it = ok ? src[first + r * 64] : 0u;
    const uint32_t d = (it >> shift) & (kRadix - 1);
    const uint64_t peers = match8(d, __ballot(ok));
    const uint64_t below = peers & ((1ull << lane) - 1ull);
    const uint32_t place = S.cnt[wave][d];
    if (ok) dst[place + static_cast<uint32_t>(__popcll(below))] = it;
    wave_lds_sync();
    if (ok && below == 0) S.cnt[wave][d] = place + static_cast<uint32_t>(__popcll(peers));
    wave_lds_sync();
  }
  __syncthreads();
}

template <int DIM>
__global__ __launch_bounds__(NT) void k_rebuild_small(SmallRebuildArgs R) {
  if (!R.rc.ctl[0]) return;
  __shared__ __attribute__((aligned(16))) unsigned char raw[sizeof(SortScratchLds)];
  __shared__ uint32_t s_wsum[kWaves], s_fixed, s_active;
  SortScratchLds& S = *reinterpret_cast<SortScratchLds*>(raw);
  using WaveScratch = ChunkScratch<256>;
  WaveScratch* chunk_scratch = reinterpret_cast<WaveScratch*>(raw);
  static_assert(sizeof(WaveScratch) * kWaves <= sizeof(SortScratchLds), "scratch overlay");
  const DevParams& P = R.b.P;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const uint32_t n = R.n;
  // a wave's items are contiguous, `rounds` times 64 of them
  const uint32_t rounds = (n + NT - 1) / NT;

  // keys (a tank that is not re-sorted keeps its own, hence its order)
  for (uint32_t i = tid; i < n; i += NT) {
    const uint32_t t = R.tag[i] >> 1;
    uint32_t k = R.key[i];
    if (R.rc.need[t]) {
      bool bad = false;
      k = cell_key<DIM>(R.b.tanks[t], [&](int q) { return R.st.x[q][i]; }, bad);
      if (bad) atomicOr(R.flags, 2u);
    }
    R.item[i] = k << 16 | i;
  }
  if (tid == 0) s_fixed = s_active = 0u;

  // stable LSD passes of 8 bits, from global memory into LDS and (a second
  // one) back; the order within the workgroup is wave, round, lane, which is
  // the slots' order
  const bool two = R.key_bits > 8;
  sort_pass(S, s_wsum, R.item, S.item, n, rounds, 16);
  if (two) {
    sort_pass(S, s_wsum, S.item, R.item, n, rounds, 24);
    for (uint32_t i = tid; i < n; i += NT) S.item[i] = R.item[i];
  }

  // the state in the new order into the scratch state, then back
  __syncthreads();
  for (uint32_t i = tid; i < n; i += NT) {
    const uint32_t it = S.item[i], src = it & 0xffffu;
    R.key[i] = it >> 16;
    if (src == i) continue;
#pragma unroll
    for (int k = 0; k < DIM; ++k) {
      R.tmp.x[k][i] = R.st.x[k][src];
      R.tmp.v[k][i] = R.st.v[k][src];
    }
    R.tmp.rho[i] = R.st.rho[src];
    R.id_tmp[i] = R.id[src];
    R.tag_tmp[i] = R.tag[src];
  }
  __syncthreads();
  for (uint32_t i = tid; i < n; i += NT) {
    if ((S.item[i] & 0xffffu) == i) continue;
    double v[DIM];
#pragma unroll
    for (int k = 0; k < DIM; ++k) {
      R.st.x[k][i] = R.tmp.x[k][i];
      v[k] = R.tmp.v[k][i];
      R.st.v[k][i] = v[k];
    }
    const double rho = R.tmp.rho[i];
    const uint32_t id = R.id_tmp[i];
    R.st.rho[i] = rho;
    R.id[i] = id;
    R.tag[i] = R.tag_tmp[i];
    write_pair_data<DIM>(P, R.st, i, v, rho, particle_mass(P, id));
  }

  // cell offsets: the first sorted slot whose key is at least c
  for (uint32_t c = tid; c <= R.n_cells; c += NT) {
    uint32_t lo = 0, hi = n;
    while (lo < hi) {
      const uint32_t mid = (lo + hi) / 2;
      if ((S.item[mid] >> 16) < c) {
        lo = mid + 1;
      } else {
        hi = mid;
      }
    }
    R.cell_off[c] = lo;
    if (c < R.n_cells) R.cell_fluid[c] = 0;
  }
  __syncthreads();
  // cells holding fluid, and the fixed particles
  for (uint32_t i = tid; i < n; i += NT) {
    if (R.tag[i] & 1u) {
      R.fixed_list[atomicAdd(&s_fixed, 1u)] = i;
    } else {
      R.cell_fluid[S.item[i] >> 16] = 1;
    }
  }
  __syncthreads();
  // fixed particles with fluid in their stencil are listed, the others'
  // state is written (k_fixed_active)
  for (uint32_t q = tid; q < s_fixed; q += NT) {
    const uint32_t i = R.fixed_list[q];
    const DevTank T = R.b.tanks[R.tag[i] >> 1];
    int c[3];
    cell_coords<DIM>(R.b, T, i, c);
    constexpr int L = DIM - 1;
    const int z0 = max(c[L] - kStencil, 0), z1 = min(c[L] + kStencil, T.nc[L] - 1);
    const int y0 = DIM == 3 ? max(c[1] - kStencil, 0) : 0;
    const int y1 = DIM == 3 ? min(c[1] + kStencil, T.nc[1] - 1) : 0;
    const int ny = DIM == 3 ? T.nc[1] : 1;
    uint32_t any = 0;
    for (int ix = max(c[0] - kStencil, 0); ix <= min(c[0] + kStencil, T.nc[0] - 1); ++ix) {
      for (int iy = y0; iy <= y1; ++iy) {
        const uint32_t row = T.cell_off + (static_cast<uint32_t>(ix) * ny + iy) * T.nc[L];
        for (int z = z0; z <= z1; ++z) any |= R.cell_fluid[row + z];
      }
    }
    if (any) {
      R.b.active[atomicAdd(&s_active, 1u)] = i;
    } else {
      write_fixed<DIM>(R.b, i, 0.0, 0.0);
    }
  }
  __syncthreads();
  // block chunks: counts, their scan, the chunks
  const StageArgs& A = R.s;
  if (A.lds_cap > 0) {
    for (uint32_t b = wave; b < A.n_blocks; b += kWaves) {
      const uint32_t c = block_chunks<DIM, 64>(A, b, chunk_scratch[wave]);
      if (lane == 0) A.bcount[b] = c;
    }
    __syncthreads();
    uint32_t before = 0;
    for (uint32_t b0 = 0; b0 < A.n_blocks; b0 += NT) {
      const uint32_t b = b0 + tid;
      uint32_t total;
      const uint32_t off = group_scan(b < A.n_blocks ? A.bcount[b] : 0u, s_wsum, &total);
      if (b < A.n_blocks) A.bcount[b] = before + off;
      before += total;
      __syncthreads();
    }
    for (uint32_t b = wave; b < A.n_blocks; b += kWaves) {
      emit_block_chunks<DIM>(A, b, b + 1 < A.n_blocks ? A.bcount[b + 1] : before);
    }
    if (tid == 0) A.counts[1] = before;
  }
  for (int t = tid; t < R.n_tanks; t += NT) {
    if (R.rc.need[t]) R.disp[t] = 0.0;
  }
  if (tid == 0) {
    R.counter[0] = s_fixed;
    R.counter[2] = s_active;
    R.rc.ctl[1] = 0u;  // no forced rebuild pending
    R.rc.ctl[2] = 1u;  // the cell index is valid
    *R.rc.count += 1ull;
  }
}

}  // namespace

void launch_rebuild_small(hipStream_t s, const SmallRebuildArgs& a) {
  if (a.b.P.dim == 2) {
    k_rebuild_small<2><<<1, NT, 0, s>>>(a);
  } else {
    k_rebuild_small<3><<<1, NT, 0, s>>>(a);
  }
}

}  // namespace tit_amd
