// The prefill GEMM's tile list (device code shared by its own kernel and the
// dispatch's block that writes the descriptors).
#pragma once

#include "dsk_internal.h"

namespace dsk {

constexpr int kPfToksMx = 128;   // dispatch rows of an MX tile

// The DMA loads read 16-byte pieces at 16-byte steps from the given bases.
__device__ __forceinline__ bool aligned16(const void* a, const void* b) {
  return ((reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(b)) & 15u) == 0;
}

// Every FP4 array of an expert at 16-byte alignment.
__device__ __forceinline__ bool slot_aligned16(const SlotDesc& d) {
  return aligned16(d.p[0], d.p[1]) && aligned16(d.p[3], d.p[4]) && aligned16(d.p[6], d.p[7]);
}

// Tile list of the active slots (one block of 1024 threads; a thread has at most
// one slot, of `rows` rows, slots ascending with the threads; rows 0: none): routed
// tiles, then the shared expert's tiles of kPfToks tokens.  The routed tiles run on the MX kernels
// (kPfToksMx rows each) when the layer allows it (mx) and every active
// slot's six FP4 arrays are 16-byte aligned (`ok`; the LDS DMA's pieces), else on
// the 8-wave kernels (kPfToks rows each).  Slots of at most `narrow` rows are
// the wide kernels' (of FP4 layers: with the MX kernels) when at least min_narrow
// slots are that small.  with_shared: the shared expert's tiles (2: only if the
// narrow slots stay here; it is the wide kernels' else).
// tiles[2 + 2 max_tiles]: the switch word.
__device__ __forceinline__ void prefill_tiles_block(const PrefillTiles& o, int slot, int rows, bool ok) {
  int32_t* tiles = o.tiles;
  const int max_tiles = o.max_tiles;
  __shared__ int32_t wsum[16];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const bool on = o.mx && __syncthreads_and(rows == 0 || ok ? 1 : 0);
  const int rtoks = on ? kPfToksMx : kPfToks;
  const bool few = __syncthreads_count(rows > 0 && rows <= o.narrow) < o.min_narrow;
  const bool wide = o.narrow > 0 && !few && (on || !o.mx);
  const int cnt = wide && rows <= o.narrow ? 0 : (rows + rtoks - 1) / rtoks;
  const int small = __syncthreads_count(cnt > 0 && rows - (cnt - 1) * rtoks <= 64);   // tiles of at most 64 rows
  int incl = cnt;
#pragma unroll
  for (int s = 1; s < 64; s <<= 1) {
    const int v = __shfl_up(incl, s, 64);
    if (lane >= s) incl += v;
  }
  if (lane == 63) wsum[wave] = incl;
  __syncthreads();
  int base = 0, total = 0;
  for (int w = 0; w < 16; ++w) {
    base += w < wave ? wsum[w] : 0;
    total += wsum[w];
  }
  const int off = base + incl - cnt;
  for (int j = 0; j < cnt; ++j) {
    tiles[2 + off + j] = slot;
    tiles[2 + max_tiles + off + j] = j * rtoks;
  }
  const int sh = o.with_shared == 1 || (o.with_shared && !wide) ? (o.T + kPfToks - 1) / kPfToks : 0;
  for (int j = t; j < sh; j += 1024) {
    tiles[2 + total + j] = -1;
    tiles[2 + max_tiles + total + j] = j * kPfToks;
  }
  if (t == 0) {
    tiles[0] = total + sh;
    tiles[1] = total;
    tiles[2 + 2 * max_tiles] = (on ? kTilesMx : 0) | (wide ? kTilesWide : 0) | (2 * small < total ? kTilesFull : 0);
  }
}

}  // namespace dsk
