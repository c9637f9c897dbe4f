// Grouped expert products for medium batches (a few to a few dozen tokens).
//
// Replaces the per-expert gate/up and w2 products of the reference's
// moe_layer (src/deepseeker/mlx_forward.py:388-406) and its shared expert
// (src/deepseeker/mlx_runner.py:765-783) when each active expert sees only a
// handful of tokens: every expert's weights must be streamed from HBM once,
// and the MFMA B operand (16 columns) is mostly empty.
//
// The wide kernels (k_up_wide, k_down_wide and their float32 and q3 forms)
// take most shapes: a block's waves walk all of K of one slot together with the
// weights straight in registers and all of the slot's rows of a pass staged.
// The others (k_up_grouped, k_down_grouped: FP4 with H out of the wide kernels'
// range, of little work, or whose rows leave in float32; q3 below one superblock or
// 24 tokens; the decode pipeline's down at three tokens; the shared expert of up to
// eight tokens) are column tiles: a block takes one slot (an active expert, or the
// shared expert as a pseudo-slot over all T tokens) and a group of row tiles; it
// walks the slot's dispatch rows in column tiles of kGNC.  For each column tile the
// block gathers only that tile's activation rows into LDS (x for gate/up, the h planes for down), the
// waves issue their first weight batches behind those loads (not in front of
// them, where the LDS stores would wait for the weights too), and each wave
// then multiplies its K range; K ranges are added in a fixed
// order through LDS.  Gate/up writes h = SwiGLU(gate, up) * route weight by
// dispatch row (hs by token for the shared expert); down writes one float32
// output row per dispatch row (ys per token for the shared expert), which
// the combine kernel adds in ascending expert id.
#include "mx.h"

namespace dsk {
namespace {

constexpr int kGI = 2;              // gate/up: row tiles of a block
constexpr int kGKS = 4;             // gate/up: K ranges of a row tile (one wave each)
constexpr int kGW = kGI * kGKS;     // waves of a gate/up block
constexpr int kDI = 8;              // down: row tiles of a block
constexpr int kDKS = 1;             // down: K ranges of a row tile
constexpr int kDW = kDI * kDKS;     // waves of a down block
constexpr int kGNC = 8;             // dispatch rows (B columns) of a column tile
constexpr int kDnRingFP4 = 4;       // down: FP4 weight batches in flight per wave

static_assert(kGW == kDW, "both kernels use the same block size");

struct GroupedArgs {
  int T, H, I, Is, k;
  float limit;
  const SlotDesc* desc; const int32_t* active;   // active[0] = number of descriptors
  const int32_t* xrow; const float* wrow;        // per dispatch row: token, route weight
  const uint16_t* x;                             // [T][H] bf16 (float32 x: its hi part)
  const uint16_t* x_lo;                          // float32 x: its lo part
  const uint16_t* ws1; const uint16_t* ws3;      // shared [Is][H] bf16
  const uint16_t* ws2;                           // shared [H][Is] bf16
  uint16_t* h_hi; uint16_t* h_lo;                // [T*k][I] by dispatch row
  uint16_t* hs_hi; uint16_t* hs_lo;              // [T][Is]
  float* y;                                      // [T*k][H]
  float* ys;                                     // [T][H]
  int up_groups, up_shared;                      // gate/up: row-tile groups per slot, shared blocks
  int dn_groups, dn_shared;                      // down: the same
  int q3f;                                       // q3 gate/up in the factored form (up_block_q3f)
  int q3fd;                                      // q3 down in the factored form (down_block_q3f)
  uint8_t* xp;                                   // q3f: x scaled, [T][H] bf16, then its 64-group sums
  // wide kernels: x (in xp) and h as FP8 planes in stage rows
  uint8_t* hp;                                   // [T*k][planes I]
  const uint8_t* xe; uint8_t* he;                // their E8M0 bytes [T][H/32], [T*k][I/32]
  int max_rows;                                  // slots with more rows are another kernel's
  const int32_t* on;                             // device switch of the FP4 slots' blocks, or null (on)
  int few;                                       // wide: slots of up to this many rows may run on wide_mul_few
  int y_bf16;                                    // routed rows rounded to bf16
  int slot_step;                                 // wide q3: a block takes every slot_step-th slot
  int sh_on;                                     // shared blocks under the switch too, ys rounded to bf16
  int sh_tiles;                                  // shared expert in column tiles (up_block, down_block)
  int sh_tg;                                     // shared expert: groups of kGsCols tokens in blocks of their own
};

// K blocks per weight batch, two batches in flight per wave, within the
// register budget of four waves per SIMD: one for bf16 rows (64 bytes per
// lane and K block) and for q3 (20 bytes, but its dequantisation needs many
// temporaries), two for FP4 (20 bytes).
template <typename Raw>
constexpr int batch_blocks() { return std::is_same_v<Raw, RawFP4> ? 2 : 1; }
// Weight batches in flight per wave in the down kernel.
template <typename Raw>
constexpr int down_ring() { return std::is_same_v<Raw, RawFP4> ? kDnRingFP4 : 2; }

// Rows [c0, c0 + cols) of the slot's activations (row r comes from source row
// src(r) of `base`, row stride `ld` elements, K elements) into LDS rows of
// stride K + 8, Q chunks per thread in flight per pass.
template <int Q, typename Src>
__device__ __forceinline__ void stage_rows_q(uint16_t* dst, const uint16_t* base, int ld, int K, int cols,
                                             Src src) {
  const int cpr = K / 8, chunks = cols * cpr, nt = blockDim.x;
  for (int c = threadIdx.x; c < chunks; c += Q * nt) {
    u32x4 v[Q];
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const int cc = min(c + q * nt, chunks - 1);   // no condition on the load (see load_raw_nc)
      v[q] = ldg16(base + static_cast<int64_t>(src(cc / cpr)) * ld + (cc % cpr) * 8);
    }
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const int cc = c + q * nt;
      if (cc < chunks) *reinterpret_cast<u32x4*>(dst + (cc / cpr) * (K + 8) + (cc % cpr) * 8) = v[q];
    }
  }
}

// Up to two chunks per thread: one pass of two; more: passes of four (a pass
// is a round trip; four chunks where two would do cost their issue slots).
template <typename Src>
__device__ __forceinline__ void stage_rows(uint16_t* dst, const uint16_t* base, int ld, int K, int cols,
                                           Src src) {
  if (cols * (K / 8) <= 2 * static_cast<int>(blockDim.x)) stage_rows_q<2>(dst, base, ld, K, cols, src);
  else stage_rows_q<4>(dst, base, ld, K, cols, src);
}

// Gate/up of one block: row tile rt (rows 16 rt ..) of w1 and w3 for the n
// dispatch rows base .. base + n - 1 (shared: tokens 0 .. n - 1).
template <typename Raw, typename LoadW, typename WPtr>
__device__ __forceinline__ void up_block(const GroupedArgs& p, LoadW load_w, WPtr wptr, int rt, bool rok, int n,
                                         int base, bool shared, uint16_t* lds) {
  constexpr int G = batch_blocks<Raw>();
  const int lane = __lane_id(), wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r16 = lane & 15, g4 = lane >> 4;
  const int item = wave / kGKS, ks = wave % kGKS;
  const int K = p.H, nblk = K / 128;
  const int per = (nblk + kGKS - 1) / kGKS;
  const int k0 = min(ks * per, nblk), k1 = min(k0 + per, nblk);
  const int xs = K + 8;
  const uint32_t row = static_cast<uint32_t>(rt * 16 + r16);
  float (*red)[kGKS][2][64][4] = reinterpret_cast<float (*)[kGKS][2][64][4]>(lds);   // over the x tile
  for (int c0 = 0; c0 < n; c0 += kGNC) {
    const int cols = min(kGNC, n - c0);
    Raw a1[G], a3[G], b1[G], b3[G];
    // FP4: each role's scales of a batch's 2 blocks (all lane groups) as one
    // 8-byte window instead of one byte per lane and block (picked at use)
    u32x2 wa1{}, wa3{}, wb1{}, wb3{};
    // no condition on the loads (see load_raw_nc): rows past the tile read
    // row 0, blocks past the range the range's last block (not computed)
    auto ld = [&](Raw (&r1)[G], Raw (&r3)[G], u32x2& w1, u32x2& w3, int kb) {
      const uint32_t rw = rok ? row : 0u;
      if constexpr (std::is_same_v<Raw, RawFP4> && G == 2) {
        const int kbc = min(kb, k1 - 2);   // every range has an even number of blocks
        const uint32_t co = rw * static_cast<uint32_t>(K / 2) + g4 * 16, so = rw * static_cast<uint32_t>(K / 32) + kbc * 4;
#pragma unroll
        for (int i = 0; i < G; ++i) {
          r1[i].c = ldg16(static_cast<const uint8_t*>(wptr(0)) + co + (kbc + i) * 64);
          r3[i].c = ldg16(static_cast<const uint8_t*>(wptr(3)) + co + (kbc + i) * 64);
        }
        w1 = ldg<u32x2>(static_cast<const uint8_t*>(wptr(1)) + so);
        w3 = ldg<u32x2>(static_cast<const uint8_t*>(wptr(4)) + so);
      } else {
#pragma unroll
        for (int i = 0; i < G; ++i) {
          const int kc = min(kb + i, k1 - 1) * 128 + g4 * 32;
          load_w(r1[i], 0, rw, kc);
          load_w(r3[i], 1, rw, kc);
        }
      }
    };
    // the tile's activation rows first: their loads are then not queued behind the
    // weights', so the LDS stores and the barrier do not wait for the weights
    if (shared) stage_rows(lds, p.x, K, K, cols, [&](int r) { return c0 + r; });
    else stage_rows(lds, p.x, K, K, cols, [&](int r) { return p.xrow[base + c0 + r]; });
    ld(a1, a3, wa1, wa3, k0);
    ld(b1, b3, wb1, wb3, k0 + G);
    __syncthreads();
    const bool tv = r16 < cols;
    const uint16_t* brow = lds + (tv ? r16 : 0) * xs;
    f32x4 ag = {0.f, 0.f, 0.f, 0.f}, au = ag;
    auto mm = [&](Raw (&r1)[G], Raw (&r3)[G], const u32x2& w1, const u32x2& w3, int kb) {
#pragma unroll
      for (int i = 0; i < G; ++i) {
        const int kc = (kb + i) * 128 + g4 * 32;
        if constexpr (std::is_same_v<Raw, RawFP4> && G == 2) {
          r1[i].s = ((i == 0 ? w1.x : w1.y) >> (8 * g4)) & 0xffu;
          r3[i].s = ((i == 0 ? w3.x : w3.y) >> (8 * g4)) & 0xffu;
        }
        mma_block2(r1[i], r3[i], brow, kc, tv && kb + i < k1, ag, au);
      }
    };
    // batches a, b alternate; pairs whose reloads both lie in the range run
    // without conditions (exact waits, see down_block), the last pair reloads
    // only what remains
    const int nb = (k1 - k0 + G - 1) / G;
    int j0 = 0;
    for (; j0 + 4 <= nb; j0 += 2) {
      mm(a1, a3, wa1, wa3, k0 + j0 * G);
      ld(a1, a3, wa1, wa3, k0 + (j0 + 2) * G);
      mm(b1, b3, wb1, wb3, k0 + (j0 + 1) * G);
      ld(b1, b3, wb1, wb3, k0 + (j0 + 3) * G);
    }
    for (; j0 < nb; j0 += 2) {
      mm(a1, a3, wa1, wa3, k0 + j0 * G);
      if (j0 + 2 < nb) ld(a1, a3, wa1, wa3, k0 + (j0 + 2) * G);
      if (j0 + 1 < nb) mm(b1, b3, wb1, wb3, k0 + (j0 + 1) * G);
      if (j0 + 3 < nb) ld(b1, b3, wb1, wb3, k0 + (j0 + 3) * G);
    }
    if constexpr (kGKS > 1) {
      __syncthreads();   // every wave is done with the x tile
      *reinterpret_cast<f32x4*>(&red[item][ks][0][lane][0]) = ag;
      *reinterpret_cast<f32x4*>(&red[item][ks][1][lane][0]) = au;
      __syncthreads();
    }
    if (ks == 0 && rok && tv) {
#pragma unroll
      for (int w = 1; w < kGKS; ++w) {
        ag += *reinterpret_cast<const f32x4*>(&red[item][w][0][lane][0]);
        au += *reinterpret_cast<const f32x4*>(&red[item][w][1][lane][0]);
      }
      const int r = base + c0 + r16;              // dispatch row (shared: token)
      const float wr = shared ? 1.0f : p.wrow[r];
      uint16_t hh[4], hl[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) split_bf16(silu_clamped(ag[q], au[q], p.limit) * wr, hh[q], hl[q]);
      const int ldh = shared ? p.Is : p.I;
      const int64_t off = static_cast<int64_t>(r) * ldh + rt * 16 + 4 * g4;
      uint16_t* dh = shared ? p.hs_hi : p.h_hi;
      uint16_t* dl = shared ? p.hs_lo : p.h_lo;
      *reinterpret_cast<uint2*>(dh + off) = uint2{hh[0] | (uint32_t(hh[1]) << 16), hh[2] | (uint32_t(hh[3]) << 16)};
      *reinterpret_cast<uint2*>(dl + off) = uint2{hl[0] | (uint32_t(hl[1]) << 16), hl[2] | (uint32_t(hl[3]) << 16)};
    }
    __syncthreads();   // the next column tile reuses the LDS
  }
}

// Gate/up of one q3 block in the factored form (x . W = s * sum(q x) + b *
// sum(x) per 64-group, see q3m_pair): row tile rt of w1 / w3 for the n
// dispatch rows base .. in column tiles of kGNC; the A operand is the
// activations (row 2t + h: dispatch row c0 + t of the tile on the K block's
// h-th 64-group), the B operand the raw codes.  Block = one row tile x kQ3gKS
// K ranges (one wave each); every wave's range is whole 512-code superblocks
// (hidden % (kQ3gKS * 512) == 0), one batch (superblock) in flight.  The
// tile's x rows (divided by 8 at the 8q positions, k_x_q3) and their group
// sums are copied into LDS first; then the weights are issued.
constexpr int kQ3gKS = kGW;
constexpr int kQ3gMaxGroups = 128;   // 64-groups of a row: hidden up to 8192
__device__ __forceinline__ void up_block_q3f(const GroupedArgs& p, const void* const* wp, int rt, bool rok, int n,
                                             int base, uint16_t* lds) {
  constexpr int G = 4;                       // K blocks per batch: one superblock
  constexpr int NT = kGW * 64;
  constexpr int kSumRegs = kQ3gMaxGroups * kGNC / NT;   // group sums per thread
  static_assert(kSumRegs * NT == kQ3gMaxGroups * kGNC, "whole passes of group sums");
  const int tid = threadIdx.x, lane = __lane_id(), wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, g4 = lane >> 4;
  const int ks = wave;
  const int K = p.H, nblk = K / 128, ng = K / 64;
  const uint16_t* xq = reinterpret_cast<const uint16_t*>(p.xp);
  const float* xg = reinterpret_cast<const float*>(p.xp + static_cast<size_t>(p.T) * K * 2);
  const int per = nblk / kQ3gKS;
  const int k0 = ks * per, k1 = k0 + per;
  const int xs = K + 8;
  uint16_t* xh = lds;                                                        // [kGNC][K + 8]
  float* xsum = reinterpret_cast<float*>(lds + kGNC * xs);                   // [nblk][8][2][2]
  u32x4* zero4 = reinterpret_cast<u32x4*>(xsum + nblk * kQ3fMaxTokens * 4);  // 64 zero bytes
  const uint16_t* zero = reinterpret_cast<const uint16_t*>(zero4);
  float (*red)[2][64][2] = reinterpret_cast<float (*)[2][64][2]>(lds);       // [wave][role], over the x tile
  if (tid < 4) zero4[tid] = u32x4{0u, 0u, 0u, 0u};
  const uint32_t rowc = rok ? static_cast<uint32_t>(rt * 16 + r16) : 0u;   // rows past the tile: row 0, not stored
  const uint32_t code_row = rowc * static_cast<uint32_t>(K / 8 * 3);
  const uint32_t sb_row = rowc * static_cast<uint32_t>(K / 64) * 2;        // bytes
  const uint8_t* W1 = static_cast<const uint8_t*>(wp[0]);
  const uint8_t* W3 = static_cast<const uint8_t*>(wp[3]);
  const uint8_t* SB[4] = {static_cast<const uint8_t*>(wp[1]), static_cast<const uint8_t*>(wp[2]),
                          static_cast<const uint8_t*>(wp[4]), static_cast<const uint8_t*>(wp[5])};
  // loads without conditions (see load_raw_nc): a batch past the range re-reads its last superblock
  auto ld = [&](Q3Batch<G>& b, int kb0) {
    const int kbc = min(kb0, k1 - G);
    const uint32_t off = code_row + (kbc >> 2) * 192 + 48 * g4;
    const auto c1 = gptr<u32x4>(W1 + off);
    const auto c3 = gptr<u32x4>(W3 + off);
#pragma unroll
    for (int v = 0; v < 3; ++v) {
      const u32x4 a = c1[v];
      const u32x4 e = c3[v];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        b.c1[(4 * v + j) / 3][(4 * v + j) % 3] = a[j];
        b.c3[(4 * v + j) / 3][(4 * v + j) % 3] = e[j];
      }
    }
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      const u32x4 w = ldg16(SB[a] + sb_row + kbc * 4);
#pragma unroll
      for (int i = 0; i < G; ++i) b.sb[a][i] = w[i];
    }
  };
  const int ta = r16 >> 1;
  const Q3Masks km = q3_masks();
  for (int c0 = 0; c0 < n; c0 += kGNC) {
    const int cols = min(kGNC, n - c0);
    // the tile's x rows and group sums first (written once per call by
    // k_x_q3; their registers are free again before the weights land): the
    // sums' loads go out ahead of the rows', both stored once the rows land
    {
      const int nsum = cols * ng;
      u32x2 sv[kSumRegs];   // {sum x, sum x / m} as loaded
#pragma unroll
      for (int j = 0; j < kSumRegs; ++j) {
        const int i = min(tid + j * NT, nsum - 1);
        const int r = i / ng, gi = i - r * ng;
        sv[j] = ldg<u32x2>(xg + (static_cast<int64_t>(p.xrow[base + c0 + r]) * ng + gi) * 2);
      }
      stage_rows(xh, xq, K, K, cols, [&](int r) { return p.xrow[base + c0 + r]; });
#pragma unroll
      for (int j = 0; j < kSumRegs; ++j) {
        const int i = tid + j * NT;
        if (i < nsum) {
          const int r = i / ng, gi = i - r * ng;
          *reinterpret_cast<u32x2*>(xsum + (((gi >> 1) * kQ3fMaxTokens + r) * 2 + (gi & 1)) * 2) = sv[j];
        }
      }
    }
    Q3Batch<G> A;
    ld(A, k0);
    __syncthreads();
    const bool av = ta < cols && (r16 & 1) == (g4 >> 1);
    const int t0 = 2 * g4;
    float acc1[2] = {0.0f, 0.0f}, acc3[2] = {0.0f, 0.0f};
    auto mm = [&](const Q3Batch<G>& b, int kb0) {
#pragma unroll
      for (int i = 0; i < G; ++i) {
        const int kb = kb0 + i;
        const uint16_t* ah = av ? xh + ta * xs + kb * 128 + 32 * g4 : zero;
        f32x4 d1 = {0.0f, 0.0f, 0.0f, 0.0f}, d3 = d1;
#define DSK_Q3G_STEP(M)                                                              \
        {                                                                            \
          const bf16x8 xa = as_bf16x8(*reinterpret_cast<const u32x4*>(ah + 8 * M)); \
          d1 = mfma16(xa, q3m_operand<M>(b.c1[i], km), d1);                          \
          d3 = mfma16(xa, q3m_operand<M>(b.c3[i], km), d3);                          \
        }
        DSK_Q3G_STEP(0) DSK_Q3G_STEP(1) DSK_Q3G_STEP(2) DSK_Q3G_STEP(3)
#undef DSK_Q3G_STEP
        const float* xg = xsum + (kb * kQ3fMaxTokens + t0) * 4;
        const f32x4 xa = *reinterpret_cast<const f32x4*>(xg);
        const f32x4 xb = *reinterpret_cast<const f32x4*>(xg + 4);
        q3_factor(d1, b.sb[0][i], b.sb[1][i], xa, xb, acc1);
        q3_factor(d3, b.sb[2][i], b.sb[3][i], xa, xb, acc3);
      }
    };
    for (int kb = k0; kb < k1; kb += G) {   // one batch at hidden 4096
      if (kb > k0) ld(A, kb);
      mm(A, kb);
    }
    // K ranges added in order, through LDS over the x tile
    __syncthreads();
    *reinterpret_cast<float2*>(&red[ks][0][lane][0]) = float2{acc1[0], acc1[1]};
    *reinterpret_cast<float2*>(&red[ks][1][lane][0]) = float2{acc3[0], acc3[1]};
    __syncthreads();
    if (ks == 0 && rok && t0 < cols) {
#pragma unroll
      for (int w = 1; w < kQ3gKS; ++w) {
        const float2 g = *reinterpret_cast<const float2*>(&red[w][0][lane][0]);
        const float2 u = *reinterpret_cast<const float2*>(&red[w][1][lane][0]);
        acc1[0] += g.x; acc1[1] += g.y;
        acc3[0] += u.x; acc3[1] += u.y;
      }
      const int n16 = rt * 16 + r16;
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        if (t0 + q < cols) {
          const int r = base + c0 + t0 + q;   // dispatch row
          uint16_t hh, hl;
          split_bf16(silu_clamped(acc1[q], acc3[q], p.limit) * p.wrow[r], hh, hl);
          p.h_hi[static_cast<int64_t>(r) * p.I + n16] = hh;
          p.h_lo[static_cast<int64_t>(r) * p.I + n16] = hl;
        }
      }
    }
    __syncthreads();   // the next column tile reuses the LDS
  }
}

// x for the factored q3 gate/up (up_block_q3f), once per call instead of once
// per block (x_q3_chunk); the blocks copy the rows and sums of their column tile.
__global__ __launch_bounds__(256) void k_x_q3(const uint16_t* __restrict__ x, int T, int H,
                                              uint16_t* __restrict__ xq, float* __restrict__ xg) {
  const int n = T * (H / 8);
  const int c = static_cast<int>(blockIdx.x) * 256 + static_cast<int>(threadIdx.x);
  x_q3_chunk(x, H, min(c, n - 1), c < n, xq, xg);   // every lane takes part in the group's sums
}

// The shared expert over more than kGNC tokens.  Its weights are 50 MB of
// bf16 at hidden 4096 / inter 2048, which the column-tile walk above would
// stream once per kGNC tokens (8x at 64 tokens).  Here a block's waves each
// take one row tile (16 rows of one weight matrix) over the whole of K and
// step through K together: at step s every wave multiplies K block s of its
// rows against the same activation block (up to kGsCols tokens x 128 of K,
// four 16-column MFMA tiles) staged in LDS.  The activations are
// L2-resident and small next to the weights; they go through registers into
// two LDS buffers, one barrier per step (gs_walk).  Weights stream once per
// kGsCols tokens.
constexpr int kGsCols = 64;              // tokens of a wide shared column group
constexpr int kGsCT = kGsCols / 16;      // its 16-column MFMA tiles
constexpr int kGsStride = 128 + 8;       // LDS row stride (elements) of a staged K block
constexpr int kGsPlane = kGsCols * kGsStride;

__host__ __device__ constexpr size_t gs_up_lds_bytes() { return 2 * size_t{kGsPlane} * 2; }
__host__ __device__ constexpr size_t gs_down_lds_bytes() { return 2 * 2 * size_t{kGsPlane} * 2; }

// K block kb of the group's rows g0 .. g0 + ncol - 1 of a [rows][ld] bf16
// matrix: thread t's 16-byte chunks t and t + 512 (row c / 16, 8 elements
// c % 16); rows past the group read its last row (never stored).
__device__ __forceinline__ void gs_load(u32x4 (&v)[2], const uint16_t* m, int ld, int g0, int ncol, int kb) {
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int c = static_cast<int>(threadIdx.x) + q * kGW * 64;
    const int r = min(c >> 4, ncol - 1);
    v[q] = ldg16(m + static_cast<int64_t>(g0 + r) * ld + kb * 128 + (c & 15) * 8);
  }
}

__device__ __forceinline__ void gs_store(const u32x4 (&v)[2], uint16_t* buf) {
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int c = static_cast<int>(threadIdx.x) + q * kGW * 64;
    *reinterpret_cast<u32x4*>(buf + (c >> 4) * kGsStride + (c & 15) * 8) = v[q];
  }
}

static_assert(kGW * 64 * 2 * 8 == kGsCols * 128, "two chunks per thread stage one K block of the group");

// Steps 0 .. nb - 1 of a wide shared walk with rings of NB weight batches
// and NB activation register slots, and two LDS buffers: mm(i, buf)
// multiplies batch i against buffer buf, ldw(i, kb) reloads batch i with K
// block kb, ldx(i, kb) loads K block kb's activations into slot i, stx(i,
// buf) copies slot i into buffer buf.  Block t's activations are loaded NB
// steps ahead, before the weights of block t, so copying them into LDS at
// step t - 1 waits only for weights already used.  Loads past the end
// re-read block nb - 1 (unused), so no load in the main loop sits under a
// condition; the last steps load only what remains.  mid() runs once the
// first steps' loads are out.
template <int NB, typename MM, typename LW, typename LX, typename SX, typename Mid>
__device__ __forceinline__ void gs_walk(int nb, MM mm, LW ldw, LX ldx, SX stx, Mid mid) {
  constexpr int U = NB % 2 == 0 ? NB : 2 * NB;   // steps per pass: slots and buffers back in phase
#pragma unroll
  for (int i = 0; i < NB; ++i) ldx(i, min(i, nb - 1));
#pragma unroll
  for (int i = 0; i < NB; ++i) ldw(i, min(i, nb - 1));
  mid();
  stx(0, 0);
  __syncthreads();
  int s = 0;
  for (; s + U <= nb; s += U) {
#pragma unroll
    for (int i = 0; i < U; ++i) {
      mm(i % NB, i & 1);
      ldx(i % NB, min(s + i + NB, nb - 1));
      ldw(i % NB, min(s + i + NB, nb - 1));
      stx((i + 1) % NB, (i + 1) & 1);
      __syncthreads();
    }
  }
  // the last nb - s < U steps
#pragma unroll
  for (int i = 0; i < U - 1; ++i) {
    if (s + i < nb) {
      mm(i % NB, i & 1);
      if (s + i + NB < nb) {
        ldx(i % NB, s + i + NB);
        ldw(i % NB, s + i + NB);
      }
      if (s + i + 1 < nb) stx((i + 1) % NB, (i + 1) & 1);
      __syncthreads();
    }
  }
}

// Gate/up of the shared expert over more than kGNC tokens: waves 2i and
// 2i + 1 take row tile 4b + i of w1 (gate) and of w3 (up), so that a wave
// holds one role's accumulators and a ring of four weight batches; the up
// wave hands its sums to the gate wave through LDS for SwiGLU.
// kPair: x as a bf16 hi / lo pair (two planes staged and multiplied, as in the down),
// a step's products in a sum of their own (see wide_mul_pair: one chain over K cost
// float32 layers 0.3 to 0.8 % of their error: 20 tokens at H 4096 4.309e-6, 4.284e-6
// so, 4.289e-6 in the general kernels).
template <bool kPair>
__device__ __forceinline__ void up_shared_wide(const GroupedArgs& p, int b, int first, int step, uint16_t* lds) {
  constexpr int NB = kPair ? 2 : 3, NX = kPair ? 2 : 1;
  const int lane = __lane_id(), wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r16 = lane & 15, g4 = lane >> 4;
  const int role = wave & 1, pair = wave >> 1;
  const int rt = b * (kGW / 2) + pair;
  const bool rok = rt < p.Is / 16;
  const uint32_t row = rok ? static_cast<uint32_t>(rt * 16 + r16) : 0u;
  const uint16_t* W = role ? p.ws3 : p.ws1;
  const int K = p.H, nb = K / 128;
  f32x4 (*xch)[kGsCT][64] = reinterpret_cast<f32x4 (*)[kGsCT][64]>(lds);   // [pair][tile][lane], after the walk
  for (int g0 = first; g0 < p.T; g0 += step) {
    const int ncol = min(kGsCols, p.T - g0);
    const int nct = (ncol + 15) / 16;
    RawBF16 w[NB];
    u32x4 xv[NB][NX][2];
    f32x4 acc[kGsCT];
#pragma unroll
    for (int c = 0; c < kGsCT; ++c) acc[c] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto mm = [&](int i, int buf) {
#pragma unroll
      for (int c = 0; c < kGsCT; ++c)
        if (c < nct) {
          const uint16_t* x = lds + buf * NX * kGsPlane + (c * 16 + r16) * kGsStride;
          if constexpr (kPair) {
            f32x4 st = {0.f, 0.f, 0.f, 0.f};
            mma_block(w[i], x, g4 * 32, true, st);
            mma_block(w[i], x + kGsPlane, g4 * 32, true, st);
            acc[c] += st;
          } else {
            mma_block(w[i], x, g4 * 32, true, acc[c]);
          }
        }
    };
    auto ldw = [&](int i, int kb) { load_raw_nc(w[i], W, row, K, kb * 128 + g4 * 32); };
    auto ldx = [&](int slot, int kb) {
      gs_load(xv[slot][0], p.x, K, g0, ncol, kb);
      if constexpr (kPair) gs_load(xv[slot][NX - 1], p.x_lo, K, g0, ncol, kb);
    };
    auto stx = [&](int slot, int buf) {
#pragma unroll
      for (int i = 0; i < NX; ++i) gs_store(xv[slot][i], lds + (buf * NX + i) * kGsPlane);
    };
    gs_walk<NB>(nb, mm, ldw, ldx, stx, [] {});   // ends with a barrier: the buffers are free
    if (role) {
#pragma unroll
      for (int c = 0; c < kGsCT; ++c) xch[pair][c][lane] = acc[c];
    }
    __syncthreads();
    if (!role && rok) {
#pragma unroll
      for (int c = 0; c < kGsCT; ++c) {
        const int t = c * 16 + r16;
        if (t < ncol) {
          const f32x4 au = xch[pair][c][lane];
          uint16_t hh[4], hl[4];
#pragma unroll
          for (int q = 0; q < 4; ++q) split_bf16(silu_clamped(acc[c][q], au[q], p.limit), hh[q], hl[q]);
          const int64_t off = static_cast<int64_t>(g0 + t) * p.Is + rt * 16 + 4 * g4;
          *reinterpret_cast<uint2*>(p.hs_hi + off) =
              uint2{hh[0] | (uint32_t(hh[1]) << 16), hh[2] | (uint32_t(hh[3]) << 16)};
          *reinterpret_cast<uint2*>(p.hs_lo + off) =
              uint2{hl[0] | (uint32_t(hl[1]) << 16), hl[2] | (uint32_t(hl[3]) << 16)};
        }
      }
    }
    __syncthreads();   // the exchange is read before the next group restages the buffers
  }
}

static_assert(size_t{kGW / 2} * kGsCT * 64 * 16 <= gs_up_lds_bytes(), "the SwiGLU exchange fits the buffers");

// Gate/up of the shared expert, block b: column tiles of a few row tiles (up to kGNC
// tokens: the wide walk takes as long however few they are: experts' kernels of two
// tokens at H 4096, I 2048, top-8 104 us with it, 82 with the tiles), or the wide walk over group
// b % sh_tg of kGsCols tokens and every sh_tg-th after it.
__device__ __forceinline__ void up_shared(const GroupedArgs& p, int b, uint16_t* lds) {
  if (!p.sh_tiles) {
    up_shared_wide<false>(p, b / p.sh_tg, (b % p.sh_tg) * kGsCols, p.sh_tg * kGsCols, lds);
    return;
  }
  const int rt = b * kGI + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) / kGKS;
  auto load_w = [&](RawBF16& r, int role, uint32_t row, int kc) { load_raw_nc(r, role ? p.ws3 : p.ws1, row, p.H, kc); };
  up_block<RawBF16>(p, load_w, [&](int) -> const void* { return p.ws1; }, rt, rt < p.Is / 16, p.T, 0, true, lds);
}

// Down of the shared expert over more than kGNC tokens, as up_shared_wide:
// block b's eight waves each take one row tile of w2 (16 output rows) over
// K = Is, the h planes (hi, lo) of up to kGsCols tokens staged per K block.
// kPair: as there.
template <bool kPair>
__device__ __forceinline__ void down_shared_wide(const GroupedArgs& p, int b, int first, int step, uint16_t* lds) {
  constexpr int NB = 2;
  const int lane = __lane_id(), wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r16 = lane & 15, g4 = lane >> 4;
  const int rt = b * kDW + wave;
  const uint32_t row = static_cast<uint32_t>(rt * 16 + r16);
  const int K = p.Is, nb = K / 128;
  for (int g0 = first; g0 < p.T; g0 += step) {
    const int ncol = min(kGsCols, p.T - g0);
    const int nct = (ncol + 15) / 16;
    RawBF16 w[NB];
    u32x4 xh[NB][2], xl[NB][2];
    f32x4 acc[kGsCT];
#pragma unroll
    for (int c = 0; c < kGsCT; ++c) acc[c] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto mm = [&](int i, int buf) {
      const uint16_t* hi = lds + buf * 2 * kGsPlane;
#pragma unroll
      for (int c = 0; c < kGsCT; ++c) {
        if (c < nct) {
          const int o = (c * 16 + r16) * kGsStride;
          f32x4 st = kPair ? f32x4{0.f, 0.f, 0.f, 0.f} : acc[c];
          mma_block(w[i], hi + o, g4 * 32, true, st);
          mma_block(w[i], hi + kGsPlane + o, g4 * 32, true, st);
          acc[c] = kPair ? acc[c] + st : st;
        }
      }
    };
    auto ldw = [&](int i, int kb) { load_raw_nc(w[i], p.ws2, row, K, kb * 128 + g4 * 32); };
    auto ldx = [&](int slot, int kb) {
      gs_load(xh[slot], p.hs_hi, K, g0, ncol, kb);
      gs_load(xl[slot], p.hs_lo, K, g0, ncol, kb);
    };
    auto stx = [&](int slot, int buf) {
      gs_store(xh[slot], lds + buf * 2 * kGsPlane);
      gs_store(xl[slot], lds + buf * 2 * kGsPlane + kGsPlane);
    };
    gs_walk<NB>(nb, mm, ldw, ldx, stx, [] {});
#pragma unroll
    for (int c = 0; c < kGsCT; ++c) {
      const int t = c * 16 + r16;
      const int64_t at = static_cast<int64_t>(g0 + t) * p.H + rt * 16 + 4 * g4;
      if (t < ncol && p.sh_on) {
        ushort4 b;
        b.x = f32_to_bf16_bits(acc[c][0]);
        b.y = f32_to_bf16_bits(acc[c][1]);
        b.z = f32_to_bf16_bits(acc[c][2]);
        b.w = f32_to_bf16_bits(acc[c][3]);
        *reinterpret_cast<ushort4*>(reinterpret_cast<uint16_t*>(p.ys) + at) = b;
      } else if (t < ncol) {
        *reinterpret_cast<f32x4*>(p.ys + at) = acc[c];
      }
    }
    __syncthreads();   // the next group restages buffer 0
  }
}

// Down of one block: row tile rt (output rows 16 rt ..) of w2 for the n
// dispatch rows base .. base + n - 1 (shared: tokens 0 .. n - 1), K = I (Is).
template <typename Raw, typename LoadW, typename WPtr>
__device__ __forceinline__ void down_block(const GroupedArgs& p, LoadW load_w, WPtr wptr, int rt, int n, int base,
                                           bool shared, uint16_t* lds) {
  constexpr int G = batch_blocks<Raw>();
  const int lane = __lane_id(), wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r16 = lane & 15, g4 = lane >> 4;
  const int item = wave / kDKS, ks = wave % kDKS;
  const int K = shared ? p.Is : p.I, nblk = K / 128;
  const int per = (nblk + kDKS - 1) / kDKS;
  const int k0 = min(ks * per, nblk), k1 = min(k0 + per, nblk);
  const int hs = K + 8;
  const uint32_t row = static_cast<uint32_t>(rt * 16 + r16);
  const uint16_t* src_hi = shared ? p.hs_hi : p.h_hi;
  const uint16_t* src_lo = shared ? p.hs_lo : p.h_lo;
  uint16_t* thi = lds;                      // [kGNC][K + 8] hi plane
  uint16_t* tlo = lds + kGNC * hs;          // [kGNC][K + 8] lo plane
  float (*red)[kDKS][64][4] = reinterpret_cast<float (*)[kDKS][64][4]>(lds);   // over the h tile
  constexpr int NB = down_ring<Raw>();
  for (int c0 = 0; c0 < n; c0 += kGNC) {
    const int cols = min(kGNC, n - c0);
    Raw a[NB][G];
    // FP4: the scales of a batch's 2 blocks (all lane groups) as one 8-byte
    // window instead of one byte per lane and block; the byte is picked at use
    u32x2 wa[NB] = {};
    // no condition on the loads (see load_raw_nc): blocks past the range
    // re-read its last block (not computed)
    auto ld = [&](Raw (&r)[G], u32x2& w, int kb) {
      if constexpr (std::is_same_v<Raw, RawFP4> && G == 2) {
        const int kbc = min(kb, k1 - 2);   // the range has an even number of blocks
#pragma unroll
        for (int i = 0; i < G; ++i) r[i].c = ldg16(static_cast<const uint8_t*>(wptr(0)) + row * static_cast<uint32_t>(K / 2) + (kbc + i) * 64 + g4 * 16);
        w = ldg<u32x2>(static_cast<const uint8_t*>(wptr(1)) + row * static_cast<uint32_t>(K / 32) + kbc * 4);
      } else {
#pragma unroll
        for (int i = 0; i < G; ++i) load_w(r[i], row, min(kb + i, k1 - 1) * 128 + g4 * 32);
      }
    };
    // the h rows first (see up_block)
    stage_rows(thi, src_hi, K, K, cols, [&](int r) { return base + c0 + r; });
    stage_rows(tlo, src_lo, K, K, cols, [&](int r) { return base + c0 + r; });
#pragma unroll
    for (int i = 0; i < NB; ++i) ld(a[i], wa[i], k0 + i * G);
    __syncthreads();
    const bool tv = r16 < cols;
    const uint16_t* bh = thi + (tv ? r16 : 0) * hs;
    const uint16_t* bl = tlo + (tv ? r16 : 0) * hs;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    auto mm = [&](Raw (&r)[G], const u32x2& w, int kb) {
#pragma unroll
      for (int i = 0; i < G; ++i) {
        const int kc = (kb + i) * 128 + g4 * 32;
        const bool ok = tv && kb + i < k1;
        if constexpr (std::is_same_v<Raw, RawFP4> && G == 2) r[i].s = ((i == 0 ? w.x : w.y) >> (8 * g4)) & 0xffu;
        mma_block(r[i], bh, kc, ok, acc);
        mma_block(r[i], bl, kc, ok, acc);
      }
    };
    // NB batches in a ring: each is multiplied, then reloaded NB batches ahead.
    // Groups whose reloads all lie in the range run without conditions (a load
    // under a condition makes the next use of an older batch wait for every
    // load, as at a branch merge the wait counter cannot tell which were
    // issued); the last groups reload only what remains.
    const int nb = (k1 - k0 + G - 1) / G;
    int j0 = 0;
    for (; j0 + 2 * NB <= nb; j0 += NB) {
#pragma unroll
      for (int i = 0; i < NB; ++i) {
        mm(a[i], wa[i], k0 + (j0 + i) * G);
        ld(a[i], wa[i], k0 + (j0 + i + NB) * G);
      }
    }
    for (; j0 < nb; j0 += NB) {
#pragma unroll
      for (int i = 0; i < NB; ++i) {
        if (j0 + i < nb) {
          mm(a[i], wa[i], k0 + (j0 + i) * G);
          if (j0 + i + NB < nb) ld(a[i], wa[i], k0 + (j0 + i + NB) * G);
        }
      }
    }
    if constexpr (kDKS > 1) {
      __syncthreads();   // every wave is done with the h tile
      *reinterpret_cast<f32x4*>(&red[item][ks][lane][0]) = acc;
      __syncthreads();
    }
    if (ks == 0 && tv) {
#pragma unroll
      for (int w = 1; w < kDKS; ++w) acc += *reinterpret_cast<const f32x4*>(&red[item][w][lane][0]);
      float* out = shared ? p.ys : p.y;
      *reinterpret_cast<f32x4*>(out + static_cast<int64_t>(base + c0 + r16) * p.H + rt * 16 + 4 * g4) = acc;
    }
    __syncthreads();   // the next column tile reuses the LDS
  }
}

// Down of the shared expert, block b (up_shared).
__device__ __forceinline__ void down_shared(const GroupedArgs& p, int b, uint16_t* lds) {
  if (!p.sh_tiles) {
    down_shared_wide<false>(p, b / p.sh_tg, (b % p.sh_tg) * kGsCols, p.sh_tg * kGsCols, lds);
    return;
  }
  const int rt = b * kDI + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) / kDKS;
  auto load_w = [&](RawBF16& r, uint32_t row, int kc) { load_raw_nc(r, p.ws2, row, p.Is, kc); };
  down_block<RawBF16>(p, load_w, [&](int) -> const void* { return p.ws2; }, rt, p.T, 0, true, lds);
}

// ---------------------------------------------------------------- wide FP4 slots
// FP4 slots on v_mfma_scale_f32_16x16x128_f8f6f4 with the block's eight waves
// walking all of K together (gs_walk), 256 of K a step: each wave multiplies
// two weight row tiles (gate/up: the same 16 rows of w1 and w3; down: 32 rows
// of w2), whose codes go from memory straight into its registers, by up to
// 16 NCT dispatch rows, whose planes the block stages in LDS, one barrier a
// step.  A dispatch row is one B column and its planes are products of their
// own into the same accumulators (plane p's scale is plane 0's times 2^-4p),
// so 16 rows share a column tile.
//
// WidePlanes ("stage rows"): row r of K values in NP FP8 planes takes NP K
// bytes, NP x 64 per 64-value stage (plane by plane, plain K order), and one
// E8M0 byte (plane 0's) per 32 values in an array of its own.
//
// What bounds it: the weight stream (16 waves of two blocks a CU, NB steps of
// 4 KB each in flight).  A step is 256 of K so that a row's 128-byte cache line
// is asked for in one go: with steps of 128 (the line's halves about 2 us
// apart, when many lines had left the L2 again) the gate/up took 402 us at 200
// tokens (H 4096, top-8 of 256: 1.8 GB of w1 / w3) against 346 (5.3 TB/s), and
// 363 at H 5120 and 24 tokens (top-6 of 384) against 306.  The kernels these
// replace: blocks of one row tile pair whose waves held four K ranges whole
// and took eight rows a pass (same box, 20 / 64 / 96 tokens at H 4096: gate/up
// 168 / 345 / 367 -> 161 / 259 / 294 us, down 84 / 176 / 218 -> 88 / 158 / 170;
// H 5120 had bf16 products there: 407 -> 306 and 162 -> 142 us at 24 tokens),
// and, from 128 tokens, GEMM tiles of 128 rows (200 tokens: 573 -> 346 and 290
// -> 204 us, the shared expert included).
constexpr int kWdWaves = 8;
constexpr int kWdStep = 256;         // K of a step
constexpr int kWdScales = 8;         // 8-byte pieces of the weights' scales a lane holds (K up to 4096 at once)

// LDS of a wide block: two buffers of a step's planes (rows padded by 16
// bytes: 16 rows at one chunk then fall on distinct banks), the dispatch rows'
// exponents and the weight rows' E8M0 bytes for all of K (rows padded by a
// word for the same reason).
constexpr int wd_row(int NP) { return NP * kWdStep + 16; }
__host__ __device__ constexpr int wd_scale_row(int K) { return K / 32 + 4; }
constexpr size_t wd_lds_bytes(int NCT, int NP, int K) {
  return size_t{2} * (16 * NCT) * wd_row(NP) + size_t(16 * NCT + 32 * kWdWaves) * wd_scale_row(K);
}

// n rows of K / 32 scale bytes each (row r at src(r)) into LDS rows of
// wd_scale_row(K) by `threads` threads from thread `t`, in pieces of 8 bytes
// (K % 256 == 0): load() issues the first Q pieces a thread, store() puts them
// away and copies what is left.
template <int Q>
struct WideScales {
  u32x2 v[Q];
  // piece c's row: c / (K / 256) through a 16-bit reciprocal (exact: c < 2^11, K / 256 < 2^5)
  static __device__ __forceinline__ int row(int c, int inv) { return static_cast<int>(__umul24(c, inv) >> 16); }
  static __device__ __forceinline__ void put(uint8_t* dst, int K, int c, int r, const u32x2& x) {
    uint32_t* d = reinterpret_cast<uint32_t*>(dst + r * wd_scale_row(K) + 8 * (c - r * (K / 256)));
    d[0] = x.x;
    d[1] = x.y;
  }
  template <typename Src>
  static __device__ __forceinline__ u32x2 get(int K, int c, int r, Src src) {
    return ldg<u32x2>(src(r) + 8 * (c - r * (K / 256)));
  }
  template <typename Src>
  __device__ __forceinline__ void load(int n, int K, int inv, int t, int threads, Src src) {
    const int last = n * (K / 256) - 1;
#pragma unroll
    for (int i = 0; i < Q; ++i) {
      const int c = min(t + i * threads, last);   // no condition on the load
      v[i] = get(K, c, row(c, inv), src);
    }
  }
  template <typename Src>
  __device__ __forceinline__ void store(uint8_t* dst, int n, int K, int inv, int t, int threads, Src src) {
    const int total = n * (K / 256);
#pragma unroll
    for (int i = 0; i < Q; ++i) {
      const int c = t + i * threads;
      if (c < total) put(dst, K, c, row(c, inv), v[i]);
    }
    for (int c = t + Q * threads; c < total; c += threads) {
      const int r = row(c, inv);
      put(dst, K, c, r, get(K, c, r, src));
    }
  }
};

// acc[a][c] = row tile a of this wave (16 weight rows, this lane's at W[a] +
// co[a], their scales at row a of S) by the tile's rows 16 c + [0, 16): n rows
// from source row src(r) of the planes q / exponents e.
template <int NCT, int NP, int NB, typename Src>
__device__ __forceinline__ void wide_mul(const uint8_t* const (&W)[2], const uint8_t* const (&S)[2],
                                         const uint32_t (&co)[2], const uint32_t (&so)[2], const uint8_t* q,
                                         const uint8_t* e, int K, int n, Src src, uint8_t* lds,
                                         f32x4 (&acc)[2][NCT]) {
  constexpr int kThreads = kWdWaves * 64, kRow = wd_row(NP), kBuf = 16 * NCT * kRow;
  constexpr int kPer = NP * (kWdStep / 16), kChunks = 16 * NCT * kPer;   // 16-byte pieces of a row, of a step
  constexpr int Q = (kChunks + kThreads - 1) / kThreads;
  // (from a copy of the thread id made here: addresses hoisted out of a loop over a
  // slot's rows would be spilled)
  int tid = threadIdx.x;
  asm volatile("" : "+v"(tid));
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, g4 = lane >> 4;
  const int es = wd_scale_row(K);
  uint8_t* xe = lds + 2 * kBuf;
  uint8_t* ws = xe + 16 * NCT * es + wave * 32 * es;
  // this thread's pieces: row c / kPer, piece c % kPer; rows past n repeat the last
  uint32_t xs[Q];   // (offsets from q: the planes are below 4 GB, wide_shapes)
  int xo[Q];
#pragma unroll
  for (int i = 0; i < Q; ++i) {
    const int c = min(tid + i * kThreads, kChunks - 1);
    const int r = c / kPer, j = c - r * kPer;
    xs[i] = static_cast<uint32_t>(src(min(r, n - 1))) * static_cast<uint32_t>(NP * K) + 16 * j;
    xo[i] = r * kRow + 16 * j;
  }
  const int inv = (65536 + K / 256 - 1) / (K / 256);
  auto esrc = [&](int r) { return e + static_cast<uint32_t>(src(r)) * static_cast<uint32_t>(K / 32); };
  auto wsrc = [&](int r) { return (r < 16 ? S[0] + so[0] : S[1] + so[1]) + (r & 15) * (K / 32); };
  WideScales<NCT> esc;
  WideScales<kWdScales> wsc;
  wsc.load(32, K, inv, lane, 64, wsrc);
  esc.load(n, K, inv, tid, kThreads, esrc);
  u32x4 w[NB][2][2];   // [slot][row tile][K block]: a row's 128 bytes in one go (whole cache lines)
  u32x4 xv[NB][Q];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int c = 0; c < NCT; ++c) acc[a][c] = f32x4{0.f, 0.f, 0.f, 0.f};
  const uint8_t* wsl = ws + r16 * es + g4;                    // + 8 per step
  const uint8_t* xel = xe + min(r16, n - 1) * es + g4;
  const int xn = max(n - 1 - r16, 0);                         // column tile c reads row min(16 c, xn) further
  auto mm = [&](int i, int buf) {
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const uint8_t* xb = lds + buf * kBuf + r16 * kRow + 16 * g4 + b * 128 * NP;
      const uint32_t s0 = wsl[4 * b], s1 = wsl[16 * es + 4 * b];
#pragma unroll
      for (int c = 0; c < NCT; ++c) {
        // the operands of one column tile at a time, its products here (left to the
        // compiler they sink to the end of a pass of steps, all operands live, and spill)
        asm volatile("" : "+v"(acc[0][c]), "+v"(acc[1][c])::"memory");
        const uint32_t bs = xel[min(16 * c, xn) * es + 4 * b];
#pragma unroll
        for (int p = 0; p < NP; ++p) {
          const uint8_t* x = xb + c * 16 * kRow + 64 * p;
          const u32x4 lo = *reinterpret_cast<const u32x4*>(x), hi = *reinterpret_cast<const u32x4*>(x + 64 * NP);
          acc[0][c] = mx_mfma(w[i][0][b], s0, lo, hi, bs - 4u * p, acc[0][c]);
          acc[1][c] = mx_mfma(w[i][1][b], s1, lo, hi, bs - 4u * p, acc[1][c]);
        }
      }
    }
#pragma unroll
    for (int c = 0; c < NCT; ++c) asm volatile("" : "+v"(acc[0][c]), "+v"(acc[1][c])::"memory");
    wsl += 8;
    xel += 8;
  };
  auto ldw = [&](int i, int kb) {
#pragma unroll
    for (int a = 0; a < 2; ++a) {
      w[i][a][0] = ldg16(W[a] + kb * (kWdStep / 2) + co[a]);
      w[i][a][1] = ldg16(W[a] + kb * (kWdStep / 2) + co[a] + 64);
    }
  };
  auto ldx = [&](int i, int kb) {
#pragma unroll
    for (int j = 0; j < Q; ++j) xv[i][j] = ldg16(q + kb * (NP * kWdStep) + xs[j]);
  };
  auto stx = [&](int i, int buf) {
#pragma unroll
    for (int j = 0; j < Q; ++j)
      if (kChunks % kThreads == 0 || tid + j * kThreads < kChunks)
        *reinterpret_cast<u32x4*>(lds + buf * kBuf + xo[j]) = xv[i][j];
  };
  // the scales' loads go out ahead of the first steps' and are put away behind them
  gs_walk<NB>(K / kWdStep, mm, ldw, ldx, stx, [&] {
    asm volatile("" ::: "memory");
    wsc.store(ws, 32, K, inv, lane, 64, wsrc);
    esc.store(xe, n, K, inv, tid, kThreads, esrc);
  });   // ends with a barrier: the buffers are free
}

// h of row tile rt, `tile` of its block, in NPH planes (two: of h rounded to bf16, as
// the prefill GEMM rounds it) for dispatch rows base + [0, n), by the waves that
// hold the tile's gate and up sums (`mine`); tiles 2j and 2j + 1 of a block share
// their rows' exponents.
template <int NCT, int NPH>
__device__ __forceinline__ void wide_store_h(const GroupedArgs& p, const f32x4 (&gate)[NCT], const f32x4 (&up)[NCT],
                                             bool mine, int tile, int rt, int n, int base, uint8_t* lds) {
  const int lane = __lane_id(), r16 = lane & 15, g4 = lane >> 4;
  float (*gmx)[NCT][16] = reinterpret_cast<float (*)[NCT][16]>(lds);   // [tile][row]: largest of its 16 features
  float hv[NCT][4];
  if (mine) {
#pragma unroll
    for (int c = 0; c < NCT; ++c) {
      const float wr = p.wrow[base + min(16 * c + r16, n - 1)];
      float m = 0.0f;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        float v = silu_clamped(gate[c][q], up[c][q], p.limit) * wr;
        if constexpr (NPH == 2) v = bf16_bits_to_f32(f32_to_bf16_bits(v));
        hv[c][q] = v;
        m = fmaxf(m, fabsf(v));
      }
      m = max_over_rows(m);
      if (g4 == 0) gmx[tile][c][r16] = m;
    }
  }
  __syncthreads();
  if (mine) {
    const int i0 = rt * 16 + 4 * g4;
#pragma unroll
    for (int c = 0; c < NCT; ++c) {
      const int ex = fp8_plane_exp(fmaxf(gmx[tile][c][r16], gmx[tile ^ 1][c][r16]));
      uint32_t pl[NPH];
      fp8_planes4<NPH>(hv[c], ex, pl);
      if (16 * c + r16 < n) {
        const int64_t r = base + 16 * c + r16;
        uint8_t* dst = p.hp + r * (NPH * p.I) + (i0 >> 6) * (64 * NPH) + (i0 & 63);
#pragma unroll
        for (int i = 0; i < NPH; ++i) *reinterpret_cast<uint32_t*>(dst + 64 * i) = pl[i];
        if ((tile & 1) == 0 && g4 == 0) p.he[r * (p.I / 32) + (i0 >> 5)] = static_cast<uint8_t>(e8m0_byte(ex));
      }
    }
  }
}

// Gate/up of one FP4 slot: rows 128 grp + [0, 128) of w1 and w3 for dispatch
// rows base + [0, n), n <= 16 NCT; h in NPH planes.
template <int NCT, int NB, int NPH>
__device__ __forceinline__ void up_wide_tile(const GroupedArgs& p, const void* const* wp, int grp, int n, int base,
                                             uint8_t* lds) {
  const int lane = __lane_id(), wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r16 = lane & 15, g4 = lane >> 4;
  const int rt = grp * kWdWaves + wave;
  const int K = p.H;
  const uint32_t row = static_cast<uint32_t>(rt * 16 + r16);
  const uint8_t* const W[2] = {static_cast<const uint8_t*>(wp[0]), static_cast<const uint8_t*>(wp[2])};
  const uint8_t* const S[2] = {static_cast<const uint8_t*>(wp[1]), static_cast<const uint8_t*>(wp[3])};
  const uint32_t c0 = row * static_cast<uint32_t>(K / 2) + static_cast<uint32_t>(g4 * 16);
  const uint32_t s0 = static_cast<uint32_t>(rt * 16) * static_cast<uint32_t>(K / 32);   // (the tile's first row)
  const uint32_t co[2] = {c0, c0}, so[2] = {s0, s0};
  f32x4 acc[2][NCT];
  wide_mul<NCT, 2, NB>(W, S, co, so, p.xp, p.xe, K, n, [&](int r) { return p.xrow[base + r]; }, lds, acc);
  wide_store_h<NCT, NPH>(p, acc[0], acc[1], true, wave, rt, n, base, lds);
  __syncthreads();   // the next rows reuse the LDS
}

// Down of one FP4 slot: output rows 256 grp + [0, 256) of w2 for n dispatch
// rows from base; h in NPH planes.
template <int NCT, int NB, int NPH>
__device__ __forceinline__ void down_wide_tile(const GroupedArgs& p, int slot, int grp, int n, int base,
                                               uint8_t* lds) {
  const int lane = __lane_id(), wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r16 = lane & 15, g4 = lane >> 4;
  const int rt = (grp * kWdWaves + wave) * 2;
  const int K = p.I;
  const uint8_t* W2 = static_cast<const uint8_t*>(desc_ptr(p.desc, slot, 6));
  const uint8_t* S2 = static_cast<const uint8_t*>(desc_ptr(p.desc, slot, 7));
  const uint8_t* const W[2] = {W2, W2};
  const uint8_t* const S[2] = {S2, S2};
  const uint32_t row = static_cast<uint32_t>(rt * 16 + r16);
  const uint32_t c0 = row * static_cast<uint32_t>(K / 2) + static_cast<uint32_t>(g4 * 16);
  const uint32_t s0 = static_cast<uint32_t>(rt * 16) * static_cast<uint32_t>(K / 32);
  const uint32_t co[2] = {c0, c0 + static_cast<uint32_t>(8 * K)}, so[2] = {s0, s0 + static_cast<uint32_t>(K / 2)};
  f32x4 acc[2][NCT];
  wide_mul<NCT, NPH, NB>(W, S, co, so, p.hp, p.he, K, n, [&](int r) { return base + r; }, lds, acc);
#pragma unroll
  for (int c = 0; c < NCT; ++c) {
    if (16 * c + r16 >= n) continue;
    const int64_t o = static_cast<int64_t>(base + 16 * c + r16) * p.H + rt * 16 + 4 * g4;
#pragma unroll
    for (int a = 0; a < 2; ++a) {
      if (p.y_bf16) {
        uint16_t b[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) b[q] = f32_to_bf16_bits(acc[a][c][q]);
        *reinterpret_cast<uint2*>(reinterpret_cast<uint16_t*>(p.y) + o + 16 * a) =
            uint2{b[0] | (uint32_t(b[1]) << 16), b[2] | (uint32_t(b[3]) << 16)};
      } else {
        *reinterpret_cast<f32x4*>(p.y + o + 16 * a) = acc[a][c];
      }
    }
  }
}

// ---------------------------------------------------------------- FP4 slots of few rows
// Slots of up to kWfRows rows where the slots are many for the batch's rows
// (wide_few_mode): their planes fit the LDS for all of K, so the waves walk without
// barriers, and a block's rows are half as many with the K range split between two
// waves of a row tile pair, so that blocks are half as long and the launch's last
// ones leave less of the chip idle.  H 4096, top-8 of 256, even routing, gate/up and
// down against the passes above: 8 tokens 93 -> 88 and 57 -> 49 us (layer 157 -> 148;
// 10 tokens 198 -> 183, 16 243 -> 240), at H 5120, top-6 of 384, 8 tokens' experts
// 186 -> 165.  Split in four: 8 tokens 165 (planes staged by twice the blocks).
// Weights ahead of the planes in a block's first loads: 3-8 us slower (the planes'
// waits then cover them).
constexpr int kWfRows = 3;
constexpr int kWfKS = 2;                       // K ranges of a row tile pair, one wave each
constexpr int kWfTiles = kWdWaves / kWfKS;     // row tile pairs of a block
constexpr int kWfNB = 4;                       // steps in flight (two: the same; five spill)
__host__ __device__ constexpr int wf_row(int NP, int K) { return NP * K + 64; }   // rows on distinct banks
__host__ __device__ constexpr int wf_steps(int K) { return (K / kWdStep + kWfKS - 1) / kWfKS; }   // of a K range
constexpr size_t wf_lds_bytes(int rows, int NP, int K) {
  return size_t(rows) * (wf_row(NP, K) + wd_scale_row(K)) + size_t(32 * kWdWaves) * wd_scale_row(wf_steps(K) * kWdStep);
}

// Blocks of a slot are kWfKS times as many with this on.  Where the passes' blocks and
// the shared expert's would fill between half the CUs and all of them once, the passes
// keep their longer walk (one block a CU; 8 tokens' experts 31 us and 36 at H 2048, I
// 1024, one token with a shared expert 48 and 64 at H 4096), and where a slot has more
// than one and a half rows on average, few of them are small (skewed routing, 8 tokens:
// layer 64 us and 85).
__device__ __forceinline__ bool wide_few_mode(int slots, int blocks, int positions) {
  return 2 * positions <= 3 * slots && (blocks <= 128 || blocks > 256);
}

// acc[a], in the waves of K range 0: row tile a of this wave by the slot's n rows (row
// r from source row src(r) of the planes q / exponents e; columns past them repeat the
// last).  The caller may reuse the LDS past the first wf_red_bytes of it.
constexpr int wf_red_bytes = (kWfKS - 1) * kWfTiles * 2 * 64 * 16;
template <int NP, typename Src>
__device__ __forceinline__ void wide_mul_few(const uint8_t* const (&W)[2], const uint8_t* const (&S)[2],
                                             const uint32_t (&co)[2], const uint32_t (&so)[2], const uint8_t* q,
                                             const uint8_t* e, int K, int n, Src src, uint8_t* lds, f32x4 (&acc)[2]) {
  constexpr int kThreads = kWdWaves * 64, Q = 4, NB = kWfNB;
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, g4 = lane >> 4, ks = wave % kWfKS, tile = wave / kWfKS;
  const int es = wd_scale_row(K), row = wf_row(NP, K), per = NP * K / 16;   // per: 16-byte pieces of a row
  // this wave's steps (none where the ranges before it cover K: st0 is then the last)
  const int ns = max(min(wf_steps(K), K / kWdStep - ks * wf_steps(K)), 0);
  const int st0 = min(ks * wf_steps(K), K / kWdStep - 1);
  const int kw = max(ns, 1) * kWdStep, ew = wd_scale_row(kw);
  uint8_t* xe = lds + n * row;
  uint8_t* ws = xe + n * es + wave * (32 * wd_scale_row(wf_steps(K) * kWdStep));
  const int inv = (65536 + K / 256 - 1) / (K / 256), invw = (65536 + kw / 256 - 1) / (kw / 256);
  auto esrc = [&](int r) { return e + static_cast<uint32_t>(src(r)) * static_cast<uint32_t>(K / 32); };
  auto wsrc = [&](int r) { return (r < 16 ? S[0] + so[0] : S[1] + so[1]) + (r & 15) * (K / 32) + 8 * st0; };
  auto at = [&](int c) { return static_cast<uint32_t>(src(c / per)) * static_cast<uint32_t>(NP * K) + 16u * (c % per); };
  WideScales<1> esc;
  WideScales<kWdScales / kWfKS> wsc;
  u32x4 xv[Q], w[NB][2][2];
  const int total = n * per;
#pragma unroll
  for (int j = 0; j < Q; ++j) xv[j] = ldg16(q + at(min(tid + j * kThreads, total - 1)));   // no condition on the load
  wsc.load(32, kw, invw, lane, 64, wsrc);
  esc.load(n, K, inv, tid, kThreads, esrc);
  asm volatile("" ::: "memory");
  auto ldw = [&](int i, int kb) {
#pragma unroll
    for (int a = 0; a < 2; ++a) {
      w[i][a][0] = ldg16(W[a] + kb * (kWdStep / 2) + co[a]);
      w[i][a][1] = ldg16(W[a] + kb * (kWdStep / 2) + co[a] + 64);
    }
  };
#pragma unroll
  for (int i = 0; i < NB; ++i) ldw(i, st0 + max(min(i, ns - 1), 0));
  asm volatile("" ::: "memory");
#pragma unroll
  for (int j = 0; j < Q; ++j) {
    const int c = tid + j * kThreads;
    if (c < total) *reinterpret_cast<u32x4*>(lds + (c / per) * row + 16 * (c % per)) = xv[j];
  }
  for (int c = tid + Q * kThreads; c < total; c += kThreads)
    *reinterpret_cast<u32x4*>(lds + (c / per) * row + 16 * (c % per)) = ldg16(q + at(c));
  wsc.store(ws, 32, kw, invw, lane, 64, wsrc);
  esc.store(xe, n, K, inv, tid, kThreads, esrc);
  acc[0] = f32x4{0.f, 0.f, 0.f, 0.f};
  acc[1] = acc[0];
  const int br = min(r16, n - 1);
  const uint8_t* wsl = ws + r16 * ew + g4;                    // + 8 per step
  const uint8_t* xel = xe + br * es + g4 + 8 * st0;
  const uint8_t* xb = lds + br * row + 16 * g4 + NP * kWdStep * st0;
  __syncthreads();
  auto mm = [&](int i) {
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const uint32_t s0 = wsl[4 * b], s1 = wsl[16 * ew + 4 * b], bs = xel[4 * b];
#pragma unroll
      for (int p = 0; p < NP; ++p) {
        const uint8_t* x = xb + b * 128 * NP + 64 * p;
        const u32x4 lo = *reinterpret_cast<const u32x4*>(x), hi = *reinterpret_cast<const u32x4*>(x + 64 * NP);
        acc[0] = mx_mfma(w[i][0][b], s0, lo, hi, bs - 4u * p, acc[0]);
        acc[1] = mx_mfma(w[i][1][b], s1, lo, hi, bs - 4u * p, acc[1]);
      }
    }
    asm volatile("" : "+v"(acc[0]), "+v"(acc[1])::"memory");   // (see wide_mul)
    wsl += 8;
    xel += 8;
    xb += NP * kWdStep;
  };
  int st = 0;
  for (; st + 2 * NB <= ns; st += NB) {
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      mm(i);
      ldw(i, st0 + st + i + NB);
    }
  }
  for (; st < ns; st += NB) {
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      if (st + i < ns) {
        mm(i);
        if (st + i + NB < ns) ldw(i, st0 + st + i + NB);
      }
    }
  }
  __syncthreads();   // every wave is done with the planes
  f32x4 (*red)[kWfTiles][2][64] = reinterpret_cast<f32x4 (*)[kWfTiles][2][64]>(lds);   // [range - 1][tile][a][lane]
  if (ks) {
    red[ks - 1][tile][0][lane] = acc[0];
    red[ks - 1][tile][1][lane] = acc[1];
  }
  __syncthreads();
  if (!ks) {
#pragma unroll
    for (int r = 0; r < kWfKS - 1; ++r) {
      acc[0] += red[r][tile][0][lane];
      acc[1] += red[r][tile][1][lane];
    }
  }
}

// Gate/up of one slot of few rows: rows 16 kWfTiles grp + [0, 16 kWfTiles) of w1 and w3.
template <int NPH>
__device__ __forceinline__ void up_wide_few(const GroupedArgs& p, const void* const* wp, int grp, int n, int base,
                                            uint8_t* lds) {
  const int lane = __lane_id(), wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r16 = lane & 15, g4 = lane >> 4, tile = wave / kWfKS;
  const int rt = grp * kWfTiles + tile, K = p.H;
  const uint8_t* const W[2] = {static_cast<const uint8_t*>(wp[0]), static_cast<const uint8_t*>(wp[2])};
  const uint8_t* const S[2] = {static_cast<const uint8_t*>(wp[1]), static_cast<const uint8_t*>(wp[3])};
  const uint32_t c0 = static_cast<uint32_t>(rt * 16 + r16) * static_cast<uint32_t>(K / 2) + static_cast<uint32_t>(g4 * 16);
  const uint32_t s0 = static_cast<uint32_t>(rt * 16) * static_cast<uint32_t>(K / 32);
  const uint32_t co[2] = {c0, c0}, so[2] = {s0, s0};
  f32x4 acc[2];
  wide_mul_few<2>(W, S, co, so, p.xp, p.xe, K, n, [&](int r) { return p.xrow[base + r]; }, lds, acc);
  const f32x4 g[1] = {acc[0]}, u[1] = {acc[1]};
  wide_store_h<1, NPH>(p, g, u, wave % kWfKS == 0, tile, rt, n, base, lds + wf_red_bytes);
}

// Down of one slot of few rows: output rows 32 kWfTiles grp + [0, 32 kWfTiles) of w2.
template <int NPH>
__device__ __forceinline__ void down_wide_few(const GroupedArgs& p, int slot, int grp, int n, int base, uint8_t* lds) {
  const int lane = __lane_id(), wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r16 = lane & 15, g4 = lane >> 4;
  const int rt = (grp * kWfTiles + wave / kWfKS) * 2, K = p.I;
  const uint8_t* W2 = static_cast<const uint8_t*>(desc_ptr(p.desc, slot, 6));
  const uint8_t* S2 = static_cast<const uint8_t*>(desc_ptr(p.desc, slot, 7));
  const uint8_t* const W[2] = {W2, W2};
  const uint8_t* const S[2] = {S2, S2};
  const uint32_t c0 = static_cast<uint32_t>(rt * 16 + r16) * static_cast<uint32_t>(K / 2) + static_cast<uint32_t>(g4 * 16);
  const uint32_t s0 = static_cast<uint32_t>(rt * 16) * static_cast<uint32_t>(K / 32);
  const uint32_t co[2] = {c0, c0 + static_cast<uint32_t>(8 * K)}, so[2] = {s0, s0 + static_cast<uint32_t>(K / 2)};
  f32x4 acc[2];
  wide_mul_few<NPH>(W, S, co, so, p.hp, p.he, K, n, [&](int r) { return base + r; }, lds, acc);
  if (wave % kWfKS == 0 && r16 < n) {
    const int64_t o = static_cast<int64_t>(base + r16) * p.H + rt * 16 + 4 * g4;
    *reinterpret_cast<f32x4*>(p.y + o) = acc[0];
    *reinterpret_cast<f32x4*>(p.y + o + 16) = acc[1];
  }
}

// ---------------------------------------------------------------- the wide FP4 kernels
// Column tiles of a pass and steps in flight.  Of one column tile three steps:
// two took 289 us of gate/up at 64 tokens (H 4096, top-8 of 256) against 259,
// four 307 (16 KB in flight per wave then overrun the XCD's L2: a 128-byte row
// piece is two loads).  Two column tiles leave registers for two steps; four
// spill.
constexpr int kWdMaxCT = 2;
constexpr int kWdNB1 = 3, kWdNB2 = 2;

// Blocks [0, up_shared): the shared expert; the others: up_groups blocks per slot
// (or kWfKS times as many), which walk its rows in passes of up to CT column tiles.
// (A slot has more rows than the call has tokens where a caller's routing names an
// expert twice in a row.)
template <int NPH, int CT>
__global__ __launch_bounds__(kWdWaves * 64) __attribute__((amdgpu_waves_per_eu(4))) void k_up_wide(GroupedArgs p) {
  extern __shared__ __align__(16) uint16_t lds_g[];
  uint8_t* lds = reinterpret_cast<uint8_t*>(lds_g);
  const int b = static_cast<int>(blockIdx.x);
  if (b < p.up_shared) {
    up_shared(p, b, lds_g);
    return;
  }
  if (p.on && !(*p.on & kTilesWide)) return;   // (first: an empty launch is as long as its loads)
  const int rb = b - p.up_shared, n_act = p.active[0];
  const bool few = CT == 1 && p.few > 0 && wide_few_mode(n_act, n_act * p.up_groups + p.up_shared, p.T * p.k);
  const int groups = few ? kWfKS * p.up_groups : p.up_groups;
  const int slot = rb / groups, grp = rb % groups;
  if (slot >= n_act) return;
  const SlotDesc* d = p.desc + slot;
  const int n = d->n_tok, base = d->tok_base;
  if (n > p.max_rows) return;
  const void* const wp[4] = {desc_ptr(p.desc, slot, 0), desc_ptr(p.desc, slot, 1), desc_ptr(p.desc, slot, 3),
                             desc_ptr(p.desc, slot, 4)};
  if constexpr (CT == 1) {
    if (few && n <= p.few) {
      up_wide_few<NPH>(p, wp, grp, n, base, lds);
      return;
    }
    if (grp >= p.up_groups) return;
  }
  int r = 0;
  if (CT == 2 || n > 16)
    for (; n - r > 16 * (CT - 1); r += 16 * CT)
      up_wide_tile<CT, kWdNB2, NPH>(p, wp, grp, min(n - r, 16 * CT), base + r, lds);
  if (n > r) up_wide_tile<1, kWdNB1, NPH>(p, wp, grp, n - r, base + r, lds);
}

template <int NPH, int CT>
__global__ __launch_bounds__(kWdWaves * 64) __attribute__((amdgpu_waves_per_eu(4))) void k_down_wide(GroupedArgs p) {
  extern __shared__ __align__(16) uint16_t lds_g[];
  uint8_t* lds = reinterpret_cast<uint8_t*>(lds_g);
  const int b = static_cast<int>(blockIdx.x);
  if (b < p.dn_shared) {
    down_shared(p, b, lds_g);
    return;
  }
  if (p.on && !(*p.on & kTilesWide)) return;   // (first: an empty launch is as long as its loads)
  const int rb = b - p.dn_shared, n_act = p.active[0];
  const bool few = CT == 1 && p.few > 0 && wide_few_mode(n_act, n_act * p.dn_groups + p.dn_shared, p.T * p.k);
  const int groups = few ? kWfKS * p.dn_groups : p.dn_groups;
  const int slot = rb / groups, grp = rb % groups;
  if (slot >= n_act) return;
  const SlotDesc* d = p.desc + slot;
  const int n = d->n_tok, base = d->tok_base;
  if (n > p.max_rows) return;
  if constexpr (CT == 1) {
    if (few && n <= p.few) {
      down_wide_few<NPH>(p, slot, grp, n, base, lds);
      return;
    }
    if (grp >= p.dn_groups) return;
  }
  int r = 0;
  if (CT == 2 || n > 16)
    for (; n - r > 16 * (CT - 1); r += 16 * CT)
      down_wide_tile<CT, kWdNB2, NPH>(p, slot, grp, min(n - r, 16 * CT), base + r, lds);
  if (n > r) down_wide_tile<1, kWdNB1, NPH>(p, slot, grp, n - r, base + r, lds);
}

// ---------------------------------------------------------------- wide FP4 slots, float32 x
// The same walk for activations as bf16 hi / lo pairs (float32 x, whose products
// keep 2^-17 and float32 sums: the scaled MFMA would sum to 2^-14): per 128-code
// block, row tile and plane four v_mfma_f32_16x16x32_bf16, the codes converted
// to bf16 with their scale once for both planes; 16 dispatch rows a pass.  Bound
// by the weight stream.  H 4096, top-8 of 256, 20 tokens: gate/up
// 490 -> 177 us, down 230 -> 100 against tiles of 16 rows by 16 tokens that read
// their activations from memory per wave; 60 tokens 1011 -> 302 and 460 -> 168;
// H 5120, top-6 of 384, 30 tokens 1080 -> 386 and 457 -> 191.  Three steps in
// flight spill (209 and 119 at 20 tokens).
constexpr int kWpNB = 2;                              // steps in flight
constexpr int kWpRow = 2 * kWdStep * 2 + 16;          // LDS bytes of a row's step: hi, lo, padding
constexpr size_t wp_lds_bytes(int K) { return size_t{2} * 16 * kWpRow + size_t(32 * kWdWaves) * wd_scale_row(K); }

template <typename Src>
__device__ __forceinline__ void wide_mul_pair(const uint8_t* const (&W)[2], const uint8_t* const (&S)[2],
                                              const uint32_t (&co)[2], const uint32_t (&so)[2], const uint16_t* hi,
                                              const uint16_t* lo, int K, int n, Src src, uint8_t* lds,
                                              f32x4 (&acc)[2]) {
  constexpr int kThreads = kWdWaves * 64, kBuf = 16 * kWpRow, NB = kWpNB;
  constexpr int Q = 16 * 64 / kThreads;               // 16-byte pieces a thread stages (64 a row)
  static_assert(Q == 2, "piece i of a thread: plane i");
  int tid = threadIdx.x;
  asm volatile("" : "+v"(tid));   // (see wide_mul)
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, g4 = lane >> 4;
  const int es = wd_scale_row(K);
  uint8_t* ws = lds + 2 * kBuf + wave * 32 * es;
  // this thread's pieces: row tid / 32, piece tid % 32 of each plane
  const uint32_t xs = static_cast<uint32_t>(src(min(tid >> 5, n - 1))) * static_cast<uint32_t>(K) + 8 * (tid & 31);
  const int xo = (tid >> 5) * kWpRow + 16 * (tid & 31);
  const int inv = (65536 + K / 256 - 1) / (K / 256);
  auto wsrc = [&](int r) { return (r < 16 ? S[0] + so[0] : S[1] + so[1]) + (r & 15) * (K / 32); };
  WideScales<kWdScales> wsc;
  wsc.load(32, K, inv, lane, 64, wsrc);
  u32x4 w[NB][2][2];   // [slot][row tile][K block]
  u32x4 xv[NB][Q];
  acc[0] = f32x4{0.f, 0.f, 0.f, 0.f};
  acc[1] = acc[0];
  const uint8_t* wsl = ws + r16 * es + g4;
  auto mm = [&](int i, int buf) {
    // a step's products in a sum of their own: chains as short as the K splits of
    // the general path's kernels (one chain over all of K was 1.5 % less exact)
    f32x4 st[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const uint8_t* xb = lds + buf * kBuf + r16 * kWpRow + b * 256 + g4 * 64;
      const float s0 = e8m0_to_f32(wsl[4 * b]), s1 = e8m0_to_f32(wsl[16 * es + 4 * b]);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        asm volatile("" : "+v"(st[0]), "+v"(st[1])::"memory");   // (see wide_mul)
        const bf16x8 xh = as_bf16x8(*reinterpret_cast<const u32x4*>(xb + 16 * j));
        const bf16x8 xl = as_bf16x8(*reinterpret_cast<const u32x4*>(xb + 2 * kWdStep + 16 * j));
        const bf16x8 a0 = fp4_word_to_bf16x8(w[i][0][b][j], s0), a1 = fp4_word_to_bf16x8(w[i][1][b][j], s1);
        st[0] = mfma16(a0, xh, st[0]);
        st[1] = mfma16(a1, xh, st[1]);
        st[0] = mfma16(a0, xl, st[0]);
        st[1] = mfma16(a1, xl, st[1]);
      }
    }
    acc[0] += st[0];
    acc[1] += st[1];
    asm volatile("" : "+v"(acc[0]), "+v"(acc[1])::"memory");
    wsl += 8;
  };
  auto ldw = [&](int i, int kb) {
#pragma unroll
    for (int a = 0; a < 2; ++a) {
      w[i][a][0] = ldg16(W[a] + kb * (kWdStep / 2) + co[a]);
      w[i][a][1] = ldg16(W[a] + kb * (kWdStep / 2) + co[a] + 64);
    }
  };
  auto ldx = [&](int i, int kb) {
    xv[i][0] = ldg16(hi + kb * kWdStep + xs);
    xv[i][1] = ldg16(lo + kb * kWdStep + xs);
  };
  auto stx = [&](int i, int buf) {
    *reinterpret_cast<u32x4*>(lds + buf * kBuf + xo) = xv[i][0];
    *reinterpret_cast<u32x4*>(lds + buf * kBuf + xo + 2 * kWdStep) = xv[i][1];
  };
  gs_walk<NB>(K / kWdStep, mm, ldw, ldx, stx, [&] {
    asm volatile("" ::: "memory");
    wsc.store(ws, 32, K, inv, lane, 64, wsrc);
  });
}

// Blocks as in k_up_wide; h as the bf16 hi / lo pair by dispatch row.
__global__ __launch_bounds__(kWdWaves * 64) __attribute__((amdgpu_waves_per_eu(4))) void k_up_wide_pair(GroupedArgs p) {
  extern __shared__ __align__(16) uint16_t lds_g[];
  uint8_t* lds = reinterpret_cast<uint8_t*>(lds_g);
  const int b = static_cast<int>(blockIdx.x);
  if (b < p.up_shared) {
    up_shared_wide<true>(p, b / p.sh_tg, (b % p.sh_tg) * kGsCols, p.sh_tg * kGsCols, lds_g);
    return;
  }
  const int rb = b - p.up_shared, slot = rb / p.up_groups, grp = rb % p.up_groups;
  if (slot >= p.active[0]) return;
  const SlotDesc* d = p.desc + slot;
  const int n = d->n_tok, base = d->tok_base;
  const int lane = __lane_id(), wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r16 = lane & 15, g4 = lane >> 4;
  const int rt = grp * kWdWaves + wave, K = p.H;
  const uint8_t* const W[2] = {static_cast<const uint8_t*>(desc_ptr(p.desc, slot, 0)),
                               static_cast<const uint8_t*>(desc_ptr(p.desc, slot, 3))};
  const uint8_t* const S[2] = {static_cast<const uint8_t*>(desc_ptr(p.desc, slot, 1)),
                               static_cast<const uint8_t*>(desc_ptr(p.desc, slot, 4))};
  const uint32_t row0 = static_cast<uint32_t>(rt * 16);
  const uint32_t c0 = (row0 + r16) * static_cast<uint32_t>(K / 2) + static_cast<uint32_t>(g4 * 16);
  const uint32_t s0 = row0 * static_cast<uint32_t>(K / 32);
  const uint32_t co[2] = {c0, c0}, so[2] = {s0, s0};
  for (int r = 0; r < n; r += 16) {
    const int m = min(n - r, 16);
    f32x4 acc[2];
    wide_mul_pair(W, S, co, so, p.x, p.x_lo, K, m, [&](int i) { return p.xrow[base + r + i]; }, lds, acc);
    if (r16 < m) {
      const int64_t row = base + r + r16;
      const float wr = p.wrow[row];
      uint16_t hh[4], hl[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) split_bf16(silu_clamped(acc[0][q], acc[1][q], p.limit) * wr, hh[q], hl[q]);
      const int64_t off = row * p.I + rt * 16 + 4 * g4;
      *reinterpret_cast<uint2*>(p.h_hi + off) = uint2{hh[0] | (uint32_t(hh[1]) << 16), hh[2] | (uint32_t(hh[3]) << 16)};
      *reinterpret_cast<uint2*>(p.h_lo + off) = uint2{hl[0] | (uint32_t(hl[1]) << 16), hl[2] | (uint32_t(hl[3]) << 16)};
    }
  }
}

__global__ __launch_bounds__(kWdWaves * 64) __attribute__((amdgpu_waves_per_eu(4))) void k_down_wide_pair(GroupedArgs p) {
  extern __shared__ __align__(16) uint16_t lds_g[];
  uint8_t* lds = reinterpret_cast<uint8_t*>(lds_g);
  const int b = static_cast<int>(blockIdx.x);
  if (b < p.dn_shared) {
    down_shared_wide<true>(p, b / p.sh_tg, (b % p.sh_tg) * kGsCols, p.sh_tg * kGsCols, lds_g);
    return;
  }
  const int rb = b - p.dn_shared, slot = rb / p.dn_groups, grp = rb % p.dn_groups;
  if (slot >= p.active[0]) return;
  const SlotDesc* d = p.desc + slot;
  const int n = d->n_tok, base = d->tok_base;
  const int lane = __lane_id(), wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r16 = lane & 15, g4 = lane >> 4;
  const int rt = (grp * kWdWaves + wave) * 2, K = p.I;
  const uint8_t* W2 = static_cast<const uint8_t*>(desc_ptr(p.desc, slot, 6));
  const uint8_t* S2 = static_cast<const uint8_t*>(desc_ptr(p.desc, slot, 7));
  const uint8_t* const W[2] = {W2, W2};
  const uint8_t* const S[2] = {S2, S2};
  const uint32_t c0 = static_cast<uint32_t>(rt * 16 + r16) * static_cast<uint32_t>(K / 2) + static_cast<uint32_t>(g4 * 16);
  const uint32_t s0 = static_cast<uint32_t>(rt * 16) * static_cast<uint32_t>(K / 32);
  const uint32_t co[2] = {c0, c0 + static_cast<uint32_t>(8 * K)}, so[2] = {s0, s0 + static_cast<uint32_t>(K / 2)};
  for (int r = 0; r < n; r += 16) {
    const int m = min(n - r, 16);
    f32x4 acc[2];
    wide_mul_pair(W, S, co, so, p.h_hi, p.h_lo, K, m, [&](int i) { return base + r + i; }, lds, acc);
    if (r16 < m) {
#pragma unroll
      for (int a = 0; a < 2; ++a)
        *reinterpret_cast<f32x4*>(p.y + static_cast<int64_t>(base + r + r16) * p.H + (rt + a) * 16 + 4 * g4) = acc[a];
    }
  }
}

// ---------------------------------------------------------------- wide q3 slots
// The walk for q3 experts in the factored form (x . W = s sum(q x) + b sum(x) per
// 64-group), 512 of K a step, one row tile a wave: the A operand is the
// activations (row 2t + h: dispatch row t of eight on a block's h-th 64-group;
// the other half's lanes read a row of zeros), the B operand the codes as 128 +
// q, and a product with ones gives the group sums where the kernels of
// up_block_q3f read prepared ones, so x and h are staged as they lie (h as its
// hi / lo pair).  All codes are shifted down to bits 0..2 for that: six shifts
// a block more than the 128 + 8q form.  Up to 16 dispatch rows a pass.
//
// Bound by the weight stream and, near it, by the masking.  Gate/up and down at H 4096, top-8 of 256
// (against blocks of eight K ranges and eight rows a pass): 64 tokens 416 -> 371 and
// 212 -> 210 us, 100 tokens 507 -> 426 and 262 -> 256 (at 16 tokens, 226 -> 220 and 121 ->
// 124 with even routing, skewed routing lost 3 %: q3_tiles).  At H 5120, I 2304, top-6 of 384, where the other kernels dequantise every
// weight: 24 tokens 696 -> 361 and 369 -> 199, 6 tokens 367 -> 108 and 121 -> 72.
constexpr int kWqStep = 512;                                // K of a step: a superblock
constexpr int kWqNB = 2;                                    // steps in flight
constexpr int kWqUpTiles = 4;                               // gate/up: row tiles of a block (w1 and w3 in waves 2i, 2i + 1)
constexpr int wq_row(int NPL) { return NPL * kWqStep * 2 + 16; }
constexpr int wq_buf(int NPL) { return 17 * wq_row(NPL); }  // 16 rows and one of zeros
constexpr size_t wq_lds_bytes(int NPL) { return size_t{2} * wq_buf(NPL); }

// Pair P of a lane's 32 codes as two bf16 128 + q (see q3m_pair).
template <int P>
__device__ __forceinline__ uint32_t q3_pair128(const uint32_t (&w)[3], const Q3Masks& k) {
  if constexpr (P < 15) return ((w[P / 5] >> (3 * (P % 5))) & k.m7) | k.magic;
  else return q3m_pair<15>(w, k);
}

template <int M>
__device__ __forceinline__ bf16x8 q3_operand128(const uint32_t (&w)[3], const Q3Masks& k) {
  return as_bf16x8(u32x4{q3_pair128<4 * M>(w, k), q3_pair128<4 * M + 1>(w, k), q3_pair128<4 * M + 2>(w, k),
                         q3_pair128<4 * M + 3>(w, k)});
}

// acc[s][i]: dispatch row 8 s + 2 g4 + i of the n rows (row r from source row
// src(r) of the NPL planes) by this lane's weight row (codes W + co, scales and
// biases S / B + so), K in whole 128-code blocks.
template <int NS, int NPL, typename Src>
__device__ __forceinline__ void wide_mul_q3(const uint8_t* W, const uint8_t* S, const uint8_t* B, uint32_t co,
                                            uint32_t so, const uint16_t* hi, const uint16_t* lo, int K, int n, Src src,
                                            uint8_t* lds, float (&acc)[NS][2]) {
  constexpr int kRow = wq_row(NPL), kBuf = wq_buf(NPL), NB = kWqNB;
  int tid = threadIdx.x;
  asm volatile("" : "+v"(tid));   // (see wide_mul)
  const int lane = tid & 63;
  const int r16 = lane & 15, g4 = lane >> 4;
  const int nsb = K / kWqStep, tb = (K / 128) & 3;   // superblocks, blocks after them
  // this thread's pieces: rows tid / 64 + 8 i, piece tid % 64 of each plane
  uint32_t xs[NS];
#pragma unroll
  for (int i = 0; i < NS; ++i)
    xs[i] = static_cast<uint32_t>(src(min((tid >> 6) + 8 * i, n - 1))) * static_cast<uint32_t>(K);
  const int xp = tid & 63, xo = (tid >> 6) * kRow + 16 * xp;
  if (tid < kRow / 16) {   // the zero rows
    *reinterpret_cast<u32x4*>(lds + 16 * kRow + 16 * tid) = u32x4{0u, 0u, 0u, 0u};
    *reinterpret_cast<u32x4*>(lds + kBuf + 16 * kRow + 16 * tid) = u32x4{0u, 0u, 0u, 0u};
  }
  struct Sb { uint32_t c[4][3]; u32x4 s, b; } w[NB];
  u32x4 xv[NB][NS][NPL];
#pragma unroll
  for (int s2 = 0; s2 < NS; ++s2) acc[s2][0] = acc[s2][1] = 0.0f;
  const Q3Masks km = q3_masks();
  const bf16x8 ones = as_bf16x8(u32x4{0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u});
  const bool av = (r16 & 1) == (g4 >> 1);
  // one block: codes c, scale / bias words, activations at byte offset `at` of a row
  auto block = [&](const uint32_t (&c)[3], uint32_t sw, uint32_t bw, const uint8_t* xb, int at) {
#pragma unroll
    for (int s2 = 0; s2 < NS; ++s2) {
      asm volatile("" : "+v"(acc[s2][0]), "+v"(acc[s2][1])::"memory");   // (see wide_mul)
      const uint8_t* x = xb + (av ? 8 * s2 + (r16 >> 1) : 16) * kRow + at + 64 * g4;
      f32x4 d = {0.f, 0.f, 0.f, 0.f}, sum = d;
#define DSK_WQ3_STEP(M)                                                                             \
      {                                                                                             \
        const bf16x8 q = q3_operand128<M>(c, km);                                                   \
        _Pragma("unroll") for (int pl = 0; pl < NPL; ++pl) {                                        \
          const bf16x8 xa = as_bf16x8(*reinterpret_cast<const u32x4*>(x + pl * 2 * kWqStep + 16 * M)); \
          d = mfma16(xa, q, d);                                                                     \
          sum = mfma16(xa, ones, sum);                                                              \
        }                                                                                           \
      }
      DSK_WQ3_STEP(0) DSK_WQ3_STEP(1) DSK_WQ3_STEP(2) DSK_WQ3_STEP(3)
#undef DSK_WQ3_STEP
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        acc[s2][i] = fmaf(f16_half<0>(sw), fmaf(-128.0f, sum[2 * i], d[2 * i]), acc[s2][i]);
        acc[s2][i] = fmaf(f16_half<0>(bw), sum[2 * i], acc[s2][i]);
        acc[s2][i] = fmaf(f16_half<1>(sw), fmaf(-128.0f, sum[2 * i + 1], d[2 * i + 1]), acc[s2][i]);
        acc[s2][i] = fmaf(f16_half<1>(bw), sum[2 * i + 1], acc[s2][i]);
      }
    }
  };
  auto mm = [&](int i, int buf) {
    const uint32_t sw[4] = {w[i].s.x, w[i].s.y, w[i].s.z, w[i].s.w}, bw[4] = {w[i].b.x, w[i].b.y, w[i].b.z, w[i].b.w};
#pragma unroll
    for (int b = 0; b < 4; ++b) block(w[i].c[b], sw[b], bw[b], lds + buf * kBuf, b * 256);
#pragma unroll
    for (int s2 = 0; s2 < NS; ++s2) asm volatile("" : "+v"(acc[s2][0]), "+v"(acc[s2][1])::"memory");
  };
  auto ldw = [&](int i, int sb) {
    const auto c = gptr<u32x4>(W + sb * 192 + co + 48 * g4);
#pragma unroll
    for (int v = 0; v < 3; ++v) {
      const u32x4 a = c[v];
#pragma unroll
      for (int j = 0; j < 4; ++j) w[i].c[(4 * v + j) / 3][(4 * v + j) % 3] = a[j];
    }
    w[i].s = ldg16(S + sb * 16 + so);
    w[i].b = ldg16(B + sb * 16 + so);
  };
  auto ldx_at = [&](int i, int k0, int piece) {
#pragma unroll
    for (int r = 0; r < NS; ++r) {
      xv[i][r][0] = ldg16(hi + k0 + 8 * piece + xs[r]);
      if constexpr (NPL == 2) xv[i][r][NPL - 1] = ldg16(lo + k0 + 8 * piece + xs[r]);
    }
  };
  auto stx = [&](int i, int buf) {
#pragma unroll
    for (int r = 0; r < NS; ++r)
#pragma unroll
      for (int pl = 0; pl < NPL; ++pl)
        *reinterpret_cast<u32x4*>(lds + buf * kBuf + 8 * r * kRow + xo + pl * 2 * kWqStep) = xv[i][r][pl];
  };
  gs_walk<NB>(nsb, mm, ldw, [&](int i, int sb) { ldx_at(i, sb * kWqStep, xp); }, stx, [] {});
  if (tb) {
    // the blocks after the last superblock (plain 48-byte blocks)
    uint32_t tw[3][3], ts[3], tbi[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const int kb = min(nsb * 4 + i, K / 128 - 1);
      const auto c = gptr<uint32_t>(W + kb * 48 + co + 12 * g4);
#pragma unroll
      for (int j = 0; j < 3; ++j) tw[i][j] = c[j];
      ts[i] = ldg<uint32_t>(S + kb * 4 + so);
      tbi[i] = ldg<uint32_t>(B + kb * 4 + so);
    }
    // (pieces past the blocks repeat the last one; nothing reads them)
    ldx_at(0, nsb * kWqStep, min(xp, tb * 16 - 1));
    stx(0, 0);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 3; ++i)
      if (i < tb) block(tw[i], ts[i], tbi[i], lds, i * 256);
    __syncthreads();
  }
}

// Gate/up of one q3 slot, NS sets of eight dispatch rows: row tile 4 grp + wave / 2
// of w1 (even waves) and w3 (odd); h as the hi / lo pair by dispatch row.
template <int NS>
__device__ __forceinline__ void up_wide_q3(const GroupedArgs& p, int slot, int grp, int n, int base, uint8_t* lds) {
  const int lane = __lane_id(), wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r16 = lane & 15, g4 = lane >> 4;
  const int role = wave & 1, pair = wave >> 1, rt = grp * kWqUpTiles + pair, K = p.H;
  const uint32_t row = static_cast<uint32_t>(rt * 16 + r16);
  const uint8_t* W = static_cast<const uint8_t*>(desc_ptr(p.desc, slot, 3 * role));
  const uint8_t* S = static_cast<const uint8_t*>(desc_ptr(p.desc, slot, 3 * role + 1));
  const uint8_t* B = static_cast<const uint8_t*>(desc_ptr(p.desc, slot, 3 * role + 2));
  float acc[NS][2];
  wide_mul_q3<NS, 1>(W, S, B, row * static_cast<uint32_t>(K / 8 * 3), row * static_cast<uint32_t>(K / 32), p.x, p.x, K, n,
                     [&](int r) { return p.xrow[base + r]; }, lds, acc);
  float (*xch)[NS][2][64] = reinterpret_cast<float (*)[NS][2][64]>(lds);   // [pair]: the up sums
  if (role) {
#pragma unroll
    for (int s2 = 0; s2 < NS; ++s2)
#pragma unroll
      for (int i = 0; i < 2; ++i) xch[pair][s2][i][lane] = acc[s2][i];
  }
  __syncthreads();
  if (!role) {
#pragma unroll
    for (int s2 = 0; s2 < NS; ++s2)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int t = 8 * s2 + 2 * g4 + i;
        if (t < n) {
          const int64_t r = base + t;
          uint16_t hh, hl;
          split_bf16(silu_clamped(acc[s2][i], xch[pair][s2][i][lane], p.limit) * p.wrow[r], hh, hl);
          p.h_hi[r * p.I + rt * 16 + r16] = hh;
          p.h_lo[r * p.I + rt * 16 + r16] = hl;
        }
      }
  }
  __syncthreads();   // the next rows reuse the LDS
}

template <int NS>
__device__ __forceinline__ void down_wide_q3(const GroupedArgs& p, int slot, int grp, int n, int base, uint8_t* lds) {
  const int lane = __lane_id(), wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r16 = lane & 15, g4 = lane >> 4;
  const int rt = grp * kWdWaves + wave, K = p.I;
  const uint32_t row = static_cast<uint32_t>(rt * 16 + r16);
  const uint8_t* W = static_cast<const uint8_t*>(desc_ptr(p.desc, slot, 6));
  const uint8_t* S = static_cast<const uint8_t*>(desc_ptr(p.desc, slot, 7));
  const uint8_t* B = static_cast<const uint8_t*>(desc_ptr(p.desc, slot, 8));
  float acc[NS][2];
  wide_mul_q3<NS, 2>(W, S, B, row * static_cast<uint32_t>(K / 8 * 3), row * static_cast<uint32_t>(K / 32), p.h_hi, p.h_lo,
                     K, n, [&](int r) { return base + r; }, lds, acc);
#pragma unroll
  for (int s2 = 0; s2 < NS; ++s2)
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int t = 8 * s2 + 2 * g4 + i;
      if (t < n) p.y[static_cast<int64_t>(base + t) * p.H + rt * 16 + r16] = acc[s2][i];
    }
}

__global__ __launch_bounds__(kWdWaves * 64) __attribute__((amdgpu_waves_per_eu(4))) void k_up_wide_q3(GroupedArgs p) {
  extern __shared__ __align__(16) uint16_t lds_g[];
  uint8_t* lds = reinterpret_cast<uint8_t*>(lds_g);
  const int b = static_cast<int>(blockIdx.x);
  if (b < p.up_shared) {
    if (p.sh_on && !(*p.on & kTilesWide)) return;
    up_shared(p, b, lds_g);
    return;
  }
  if (p.on && !(*p.on & kTilesWide)) return;
  const int rb = b - p.up_shared, first = rb / p.up_groups, grp = rb % p.up_groups;
  const int n_act = p.active[0];
  for (int slot = first; slot < n_act; slot += p.slot_step) {
    const SlotDesc* d = p.desc + slot;
    const int n = d->n_tok, base = d->tok_base;
    if (n > p.max_rows) continue;
    int r = 0;
    for (; n - r > 8; r += 16) up_wide_q3<2>(p, slot, grp, min(n - r, 16), base + r, lds);
    if (n > r) up_wide_q3<1>(p, slot, grp, n - r, base + r, lds);
  }
}

__global__ __launch_bounds__(kWdWaves * 64) __attribute__((amdgpu_waves_per_eu(4))) void k_down_wide_q3(GroupedArgs p) {
  extern __shared__ __align__(16) uint16_t lds_g[];
  uint8_t* lds = reinterpret_cast<uint8_t*>(lds_g);
  const int b = static_cast<int>(blockIdx.x);
  if (b < p.dn_shared) {
    if (p.sh_on && !(*p.on & kTilesWide)) return;
    down_shared(p, b, lds_g);
    return;
  }
  if (p.on && !(*p.on & kTilesWide)) return;
  const int rb = b - p.dn_shared, first = rb / p.dn_groups, grp = rb % p.dn_groups;
  const int n_act = p.active[0];
  for (int slot = first; slot < n_act; slot += p.slot_step) {
    const SlotDesc* d = p.desc + slot;
    const int n = d->n_tok, base = d->tok_base;
    if (n > p.max_rows) continue;
    int r = 0;
    for (; n - r > 8; r += 16) down_wide_q3<2>(p, slot, grp, min(n - r, 16), base + r, lds);
    if (n > r) down_wide_q3<1>(p, slot, grp, n - r, base + r, lds);
  }
}

// Blocks [0, up_shared): the shared expert (bf16 w1/w3, all T tokens); the
// others: up_groups blocks per slot.
template <typename Raw>
__global__ __launch_bounds__(kGW * 64) __attribute__((amdgpu_waves_per_eu(4))) void k_up_grouped(GroupedArgs p) {
  extern __shared__ __align__(16) uint16_t lds_g[];
  const int b = static_cast<int>(blockIdx.x);
  const int item = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) / kGKS;
  if (b < p.up_shared) {
    up_shared(p, b, lds_g);
    return;
  }
  const int rb = b - p.up_shared;
  const int slot = rb / p.up_groups;
  if (slot >= p.active[0]) return;
  const SlotDesc* d = p.desc + slot;
  const int rt = (rb % p.up_groups) * kGI + item;
  const void* const wp[6] = {desc_ptr(p.desc, slot, 0), desc_ptr(p.desc, slot, 1), desc_ptr(p.desc, slot, 2),
                             desc_ptr(p.desc, slot, 3), desc_ptr(p.desc, slot, 4), desc_ptr(p.desc, slot, 5)};
  if constexpr (std::is_same_v<Raw, RawQ3>) {
    if (p.q3f) {   // one row tile per block (up_groups = I / 16)
      const int rt1 = rb % p.up_groups;
      up_block_q3f(p, wp, rt1, rt1 < p.I / 16, d->n_tok, d->tok_base, lds_g);
      return;
    }
  }
  auto load_w = [&](Raw& r, int role, uint32_t row, int kc) { load_role_nc(r, wp, role, row, p.H, kc); };
  up_block<Raw>(p, load_w, [&](int i) { return wp[i]; }, rt, rt < p.I / 16, d->n_tok, d->tok_base, false, lds_g);
}

// Down of one q3 block in the factored form (as up_block_q3f): output row
// tile rt (one wave) over all of K = I in 512-code superblocks (I % 512 ==
// 0), two in flight; A operand row 2t + h on the hi plane and then the lo
// plane of dispatch row c0 + t's h (both into one accumulator), B operand the
// raw w2 codes; the tile's h rows are staged divided by 8 at the 8q positions
// with the group sums of hi + lo.  Writes one float32 row per dispatch row.
struct Q3Sb { uint32_t c[4][3]; u32x4 s, b; };   // one superblock of a lane's w2 row: codes, windows

__device__ __forceinline__ void down_block_q3f(const GroupedArgs& p, int slot, int rt, int n, int base,
                                               uint16_t* lds) {
  constexpr int kStg = 2;                    // h chunks per thread in flight while staging
  constexpr int NT = kDW * 64;
  const int tid = threadIdx.x, lane = __lane_id();
  const int r16 = lane & 15, g4 = lane >> 4;
  const int K = p.I, nblk = K / 128, nsb = K / 512, cpr = K / 8;
  const int hs = K + 8;
  uint16_t* thi = lds;                                                       // [kGNC][K + 8]
  uint16_t* tlo = lds + kGNC * hs;                                           // [kGNC][K + 8]
  float* hsum = reinterpret_cast<float*>(lds + 2 * kGNC * hs);               // [nblk][8][2][2]
  u32x4* zero4 = reinterpret_cast<u32x4*>(hsum + nblk * kQ3fMaxTokens * 4);  // 64 zero bytes
  const uint16_t* zero = reinterpret_cast<const uint16_t*>(zero4);
  if (tid < 4) zero4[tid] = u32x4{0u, 0u, 0u, 0u};
  const uint32_t row = static_cast<uint32_t>(rt * 16 + r16);
  const uint8_t* W = static_cast<const uint8_t*>(desc_ptr(p.desc, slot, 6));
  const uint8_t* S = static_cast<const uint8_t*>(desc_ptr(p.desc, slot, 7));
  const uint8_t* B = static_cast<const uint8_t*>(desc_ptr(p.desc, slot, 8));
  const uint32_t code_row = row * static_cast<uint32_t>(K / 8 * 3), sb_row = row * static_cast<uint32_t>(K / 64) * 2;
  // no condition on the loads (see load_raw_nc): past the last superblock, the last again (not computed)
  auto ld = [&](Q3Sb& r, int sb) {
    const int sbc = min(sb, nsb - 1);
    const auto c = gptr<u32x4>(W + code_row + sbc * 192 + 48 * g4);
#pragma unroll
    for (int v = 0; v < 3; ++v) {
      const u32x4 a = c[v];
#pragma unroll
      for (int j = 0; j < 4; ++j) r.c[(4 * v + j) / 3][(4 * v + j) % 3] = a[j];
    }
    r.s = ldg16(S + sb_row + sbc * 16);
    r.b = ldg16(B + sb_row + sbc * 16);
  };
  const int ta = r16 >> 1;
  const Q3Masks km = q3_masks();
  for (int c0 = 0; c0 < n; c0 += kGNC) {
    const int cols = min(kGNC, n - c0);
    // the tile's h rows (hi + lo), kStg chunks per thread in flight (whole lane groups)
    const int xch = cols * cpr;
    for (int cb = 0; cb < xch; cb += kStg * NT) {
      u32x4 vh[kStg], vl[kStg];
#pragma unroll
      for (int j = 0; j < kStg; ++j) {
        const int c = min(cb + j * NT + tid, xch - 1);
        const int64_t e = static_cast<int64_t>(base + c0 + c / cpr) * K + (c % cpr) * 8;
        vh[j] = ldg16(p.h_hi + e);
        vl[j] = ldg16(p.h_lo + e);
      }
#pragma unroll
      for (int j = 0; j < kStg; ++j) {
        const int c = cb + j * NT + tid;
        if (c < xch) {
          // hi + lo is exact in float32; staged again as a (hi, lo) pair of the scaled value
          const uint32_t wh[4] = {vh[j].x, vh[j].y, vh[j].z, vh[j].w}, wl[4] = {vl[j].x, vl[j].y, vl[j].z, vl[j].w};
          uint32_t f[8];
#pragma unroll
          for (int e2 = 0; e2 < 8; ++e2) {
            const uint32_t sh = (e2 & 1) ? 0u : 16u;
            const float v = __uint_as_float(((wh[e2 >> 1] << sh) & 0xffff0000u)) +
                            __uint_as_float(((wl[e2 >> 1] << sh) & 0xffff0000u));
            f[e2] = __float_as_uint(v);
          }
          stage_chunk_q3<true>(thi, tlo, hsum, hs, cpr, c, u32x4{f[0], f[1], f[2], f[3]}, u32x4{f[4], f[5], f[6], f[7]});
        }
      }
    }
    // keep the weight loads below the staging (their registers would overlap)
    __builtin_amdgcn_sched_barrier(0);
    Q3Sb ra, rb;
    ld(ra, 0);
    ld(rb, 1);
    __syncthreads();
    const bool av = ta < cols && (r16 & 1) == (g4 >> 1);
    const int t0 = 2 * g4;
    float acc[2] = {0.0f, 0.0f};
    auto mm = [&](const Q3Sb& r, int sb) {
      const uint32_t sw[4] = {r.s.x, r.s.y, r.s.z, r.s.w}, bw[4] = {r.b.x, r.b.y, r.b.z, r.b.w};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int kb = 4 * sb + i;
        const int ao = ta * hs + kb * 128 + 32 * g4;
        const uint16_t* ah = av ? thi + ao : zero;
        const uint16_t* al = av ? tlo + ao : zero;
        f32x4 d = {0.0f, 0.0f, 0.0f, 0.0f};
#define DSK_Q3D_STEP(M)                                                                                \
        d = mfma16(as_bf16x8(*reinterpret_cast<const u32x4*>(ah + 8 * M)), q3m_operand<M>(r.c[i], km), d); \
        d = mfma16(as_bf16x8(*reinterpret_cast<const u32x4*>(al + 8 * M)), q3m_operand<M>(r.c[i], km), d);
        DSK_Q3D_STEP(0) DSK_Q3D_STEP(1) DSK_Q3D_STEP(2) DSK_Q3D_STEP(3)
#undef DSK_Q3D_STEP
        const float* xg = hsum + (kb * kQ3fMaxTokens + t0) * 4;
        q3_factor(d, sw[i], bw[i], *reinterpret_cast<const f32x4*>(xg), *reinterpret_cast<const f32x4*>(xg + 4), acc);
      }
    };
    for (int sb = 0; sb < nsb; sb += 2) {
      mm(ra, sb);
      if (sb + 2 < nsb) ld(ra, sb + 2);
      if (sb + 1 < nsb) mm(rb, sb + 1);
      if (sb + 3 < nsb) ld(rb, sb + 3);
    }
#pragma unroll
    for (int q = 0; q < 2; ++q)
      if (t0 + q < cols) p.y[static_cast<int64_t>(base + c0 + t0 + q) * p.H + rt * 16 + r16] = acc[q];
    __syncthreads();   // the next column tile reuses the LDS
  }
}

// Blocks [0, dn_shared): the shared expert's w2 (bf16, all T tokens); the
// others: dn_groups blocks per slot.
// q3: three waves per SIMD (the factored product keeps two superblocks of w2
// in flight per wave)
template <typename Raw>
__global__ __launch_bounds__(kDW * 64) __attribute__((amdgpu_waves_per_eu(std::is_same_v<Raw, RawQ3> ? 3 : 4))) void
k_down_grouped(GroupedArgs p) {
  extern __shared__ __align__(16) uint16_t lds_g[];
  const int b = static_cast<int>(blockIdx.x);
  const int item = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) / kDKS;
  if (b < p.dn_shared) {
    down_shared(p, b, lds_g);
    return;
  }
  const int rb = b - p.dn_shared;
  const int slot = rb / p.dn_groups;
  if (slot >= p.active[0]) return;
  const SlotDesc* d = p.desc + slot;
  const int rt = (rb % p.dn_groups) * kDI + item;
  if constexpr (std::is_same_v<Raw, RawQ3>) {
    if (p.q3fd) {
      down_block_q3f(p, slot, rt, d->n_tok, d->tok_base, lds_g);
      return;
    }
  }
  auto load_w = [&](Raw& r, uint32_t row, int kc) { load_w2_nc(r, p.desc, slot, row, p.I, kc); };
  auto wptr = [&](int i) { return desc_ptr(p.desc, slot, 6 + i); };   // 0: w2 codes, 1: w2 scales
  down_block<Raw>(p, load_w, wptr, rt, d->n_tok, d->tok_base, false, lds_g);
}

// The factored q3 gate/up: every wave's K range whole superblocks.
bool up_q3f(const dsk_moe_desc& d) {
  return d.quant == DSK_QUANT_Q3 && d.hidden % (kQ3gKS * 512) == 0 && d.hidden <= kQ3gMaxGroups * 64;
}

}  // namespace

bool grouped_x_q3(const dsk_moe_desc& d) { return up_q3f(d); }

namespace {

size_t up_lds(const dsk_moe_desc& d) {
  const size_t x_tile = static_cast<size_t>(kGNC) * (d.hidden + 8) * 2;
  const size_t red = static_cast<size_t>(kGI) * kGKS * 2 * 64 * 4 * sizeof(float);
  // factored q3: the x tile, its group sums [H/128][8][2][2] f32, 64 zero bytes
  const size_t q3f = x_tile + static_cast<size_t>(d.hidden / 128) * kQ3fMaxTokens * 16 + 64;
  size_t base = x_tile > red ? x_tile : red;
  if (d.tokens > kGNC && d.inter_shared > 0 && gs_up_lds_bytes() > base) base = gs_up_lds_bytes();
  return up_q3f(d) && q3f > base ? q3f : base;
}

hipError_t launch_x_q3(const dsk_moe_desc& d, const GroupedArgs& p, hipStream_t s) {
  const int64_t n = static_cast<int64_t>(d.tokens) * (d.hidden / 8);
  uint16_t* xq = reinterpret_cast<uint16_t*>(p.xp);
  float* xg = reinterpret_cast<float*>(p.xp + static_cast<size_t>(d.tokens) * d.hidden * 2);
  launch_kernel(k_x_q3, static_cast<unsigned>((n + 255) / 256), 256, 0, s, p.x, d.tokens, d.hidden, xq, xg);
  return hipGetLastError();
}

// The factored q3 down: K = I whole superblocks.
bool down_q3f(const dsk_moe_desc& d) { return d.quant == DSK_QUANT_Q3 && d.inter % 512 == 0; }

size_t down_lds(const dsk_moe_desc& d) {
  const int K = d.inter > d.inter_shared ? d.inter : d.inter_shared;
  const size_t h_tile = 2 * static_cast<size_t>(kGNC) * (K + 8) * 2;
  const size_t red = static_cast<size_t>(kDI) * kDKS * 64 * 4 * sizeof(float);
  const size_t base = h_tile > red ? h_tile : red;
  // factored q3: the h tile of I, its group sums [I/128][8][2][2] f32, 64 zero bytes
  const size_t q3f = 2 * static_cast<size_t>(kGNC) * (d.inter + 8) * 2 +
                     static_cast<size_t>(d.inter / 128) * kQ3fMaxTokens * 16 + 64;
  size_t b2 = base;
  if (d.tokens > kGNC && d.inter_shared > 0 && gs_down_lds_bytes() > b2) b2 = gs_down_lds_bytes();
  return down_q3f(d) && q3f > b2 ? q3f : b2;
}

}  // namespace

bool grouped_path(const dsk_moe_desc& d) {
  // FP4 reads 2-block scale windows: an even number of K blocks in every
  // wave's range (down: I % 256 == 0; gate/up, 4 ranges: H % 1024 == 0)
  return d.x_dtype == DSK_DTYPE_BF16 && d.hidden % (kGI * 16) == 0 && d.hidden % (kDI * 16) == 0 &&
         (d.quant != DSK_QUANT_FP4 || (d.inter % 256 == 0 && d.hidden % (kGKS * 256) == 0)) &&
         d.hidden % 128 == 0 && d.inter % 128 == 0 && d.inter % (kGI * 16) == 0 &&
         d.inter_shared % 128 == 0 && d.inter_shared % (kGI * 16) == 0 &&
         up_lds(d) <= kMaxLds && down_lds(d) <= kMaxLds;
}

namespace {

GroupedArgs grouped_args(const dsk_moe_desc& d, const Workspace& L, const ExpertsArgs& a, const SlotDesc* desc,
                         const int32_t* xrow, const float* wrow) {
  GroupedArgs p{};
  p.T = d.tokens; p.H = d.hidden; p.I = d.inter; p.Is = d.inter_shared; p.k = d.top_k; p.limit = d.limit;
  p.desc = desc; p.active = a.active; p.xrow = xrow; p.wrow = wrow;
  p.x = static_cast<const uint16_t*>(a.x);
  p.ws1 = static_cast<const uint16_t*>(a.ws1);
  p.ws3 = static_cast<const uint16_t*>(a.ws3);
  p.ws2 = static_cast<const uint16_t*>(a.ws2);
  p.h_hi = reinterpret_cast<uint16_t*>(a.ws + L.h_hi);
  p.h_lo = reinterpret_cast<uint16_t*>(a.ws + L.h_lo);
  p.hs_hi = reinterpret_cast<uint16_t*>(a.ws + L.hs_hi);
  p.hs_lo = reinterpret_cast<uint16_t*>(a.ws + L.hs_lo);
  p.y = rows_buffer(a.rows_out, a.ws, L);
  p.ys = reinterpret_cast<float*>(a.ws + L.ys);
  p.q3f = up_q3f(d) ? 1 : 0;
  p.q3fd = down_q3f(d) ? 1 : 0;
  p.xp = reinterpret_cast<uint8_t*>(a.ws + L.xp);
  p.hp = reinterpret_cast<uint8_t*>(a.ws + L.hp);
  p.up_groups = p.q3f ? d.inter / 16 : d.inter / 16 / kGI;   // factored q3: one row tile per block
  // shared gate/up: past kGNC tokens, four row tiles per block (up_shared_wide)
  p.sh_tiles = d.tokens <= kGNC ? 1 : 0;
  p.sh_tg = 1;
  p.up_shared = p.sh_tiles ? d.inter_shared / 16 / kGI : (d.inter_shared / 16 + kGW / 2 - 1) / (kGW / 2);
  p.dn_groups = d.hidden / 16 / kDI;
  p.dn_shared = d.inter_shared > 0 ? p.dn_groups : 0;
  return p;
}

int max_slots(const dsk_moe_desc& d) { return d.n_experts < d.tokens * d.top_k ? d.n_experts : d.tokens * d.top_k; }

hipError_t grouped_down(const dsk_moe_desc& d, const GroupedArgs& p, hipStream_t s, int repeat) {
  const unsigned blocks = static_cast<unsigned>(p.dn_shared + max_slots(d) * p.dn_groups);
  const size_t lds = down_lds(d);
  for (int r = 0; r < repeat; ++r) {
    if (d.quant == DSK_QUANT_Q3) launch_kernel(k_down_grouped<RawQ3>, blocks, kDW * 64, lds, s, p);
    else launch_kernel(k_down_grouped<RawFP4>, blocks, kDW * 64, lds, s, p);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

}  // namespace

// Rows handed to the caller stay float32, so they keep what the column tiles hold: bf16
// products with float32 sums and h as a pair (FP4: 2.5e-6 of the rows, against 2.6e-5 on
// the scaled MFMAs, whose sums and planes hold 2^-14), the factored q3 products (8.4e-6
// against 1.1e-5).  Where h's planes have space of their own, the rows are the planes'.
// H 5120, I 2304, top-6, tiles and wide: 20 tokens 424 and 331 us; H 4096, I 2048,
// top-8, 127 tokens 761 and 593.
static bool rows_on_tiles(const dsk_moe_desc& d) {
  return d.quant == DSK_QUANT_FP4 ? !wide_own_space(d) : d.hidden % 4096 == 0 && d.inter % 512 == 0;
}

// The factored q3 down keeps its column tiles to 27 tokens, the gate/up beside it only
// below 24 (q3_tiles): at H 4096, I 2048, top-8 of 256 and 24 tokens the gate/up takes
// 281 and 277 us (skewed routing 90 and 66) in tiles and wide, the down 142 and 170 (52
// and 44).  Layers with tiles, wide and so: 24 tokens 415, 418 and 402 us (skewed 152,
// 133 and 134), 26 tokens 432, 435 and 419; 28 tokens, 459 and 455, are faster wide.
static bool q3_down_tiles(const dsk_moe_desc& d) {
  return d.quant == DSK_QUANT_Q3 && d.hidden % 4096 == 0 && down_q3f(d) && d.tokens < 28;
}

hipError_t launch_experts_grouped(const dsk_moe_desc& d, const Workspace& L, const ExpertsArgs& a,
                                  const SlotDesc* desc, const int32_t* xrow, const float* wrow, hipStream_t s,
                                  int repeat) {
  hipError_t e;
  if ((grouped_wide(d) || grouped_wide_q3(d)) && !(a.rows_out && rows_on_tiles(d))) {
    const bool planes = d.quant == DSK_QUANT_FP4;
    const WideCall w{3, kAllRows, nullptr, 0, d.inter_shared > 0};
    if ((e = stage_open(kStageUp)) != hipSuccess) return e;
    for (int r = 0; r < repeat; ++r) {
      if (planes && !a.x_planes_ready && (e = launch_pf_planes(d, L, a, s)) != hipSuccess) return e;
      if ((e = launch_wide_up(d, L, a, desc, xrow, wrow, w, s)) != hipSuccess) return e;
    }
    if ((e = stage_open(kStageDown)) != hipSuccess) return e;
    if (q3_down_tiles(d)) return grouped_down(d, grouped_args(d, L, a, desc, xrow, wrow), s, repeat);
    for (int r = 0; r < repeat; ++r)
      if ((e = launch_wide_down(d, L, a, desc, w, s)) != hipSuccess) return e;
    return e;
  }
  GroupedArgs p = grouped_args(d, L, a, desc, xrow, wrow);
  const unsigned up_blocks = static_cast<unsigned>(p.up_shared + max_slots(d) * p.up_groups);
  const size_t ul = up_lds(d);
  if ((e = stage_open(kStageUp)) != hipSuccess) return e;
  for (int r = 0; r < repeat; ++r) {
    if (p.q3f && !a.x_planes_ready && (e = launch_x_q3(d, p, s)) != hipSuccess) return e;
    if (d.quant == DSK_QUANT_Q3) launch_kernel(k_up_grouped<RawQ3>, up_blocks, kGW * 64, ul, s, p);
    else launch_kernel(k_up_grouped<RawFP4>, up_blocks, kGW * 64, ul, s, p);
    if ((e = hipGetLastError()) != hipSuccess) return e;
  }
  if ((e = stage_open(kStageDown)) != hipSuccess) return e;
  return grouped_down(d, p, s, repeat);
}

// The wide kernels from four tokens (gate/up + down: H 4096, top-8 of 256 at three
// tokens 88 us against 81 on the streaming kernels, at five 114 and 118, H 5120,
// top-6 of 384 at six 155 and 225), the
// others of the grouped path from eight.
int decode_grouped_up_min(const dsk_moe_desc& d) {
  // q3 shapes without the factored decode kernels: k_up_q3 with one superblock a wave (H
  // a multiple of 4096), k_down_q3 (I 2048).  Gate/up + down of one token at H 5120, I
  // 2304: 151 -> 63 us; layer at H 2048, I 1024: 53.5 -> 39.5 us; at H 4096, I 512 one
  // token is faster on k_up_q3 (41.3 against 45.5), two are not (61.1, 47.9)
  if (grouped_wide_q3(d)) return d.hidden % 4096 != 0 ? 1 : 2;
  return grouped_wide(d) ? 4 : kDecodeGroupedUpMin;
}

// Little work: a wide block walks all of K however few blocks there are, so up to half
// a block a CU (from H 4096 a quarter) stays with the column tiles: experts' kernels
// with a shared expert, tiles and wide: H 3072, I 512, top-2: one token 27 and 33 us; H
// 1024, I 768, top-4: one 23 and 26, 8 tokens (192 blocks) 29 and 28; layer of 4 tokens
// at H 4096, I 1024, top-2 (64 blocks) 33 and 37.  So do two tokens with a shared
// expert (H 4096, I 2048, top-8: one 58 and 48, two 69 and 83, three 94 and 89; H 5120,
// I 2304, top-6: 63 and 54, 91 and 100, 121 and 110).
static bool little_work(const dsk_moe_desc& d) {
  if (d.tokens == 2 && d.inter_shared > 0) return true;
  return int64_t{d.tokens} * d.top_k * d.inter <= int64_t{d.hidden < 4096 ? 128 : 64} * 128;
}

bool grouped_wide(const dsk_moe_desc& d) {
  return wide_shapes(d) && grouped_path(d) && !prefill_gemm(d) && !little_work(d);
}

// Below 24 tokens the column tiles' factored products (H a multiple of 4096, I of
// 512) keep their shapes: a layer of H 4096, I 2048, top-8 of 256 takes 8 / 12 / 16
// tokens in 215 / 280 / 340 us there and 218 / 284 / 329 in the wide kernels, but 86 /
// 114 / 127 and 95 / 120 / 130 when the routing is skewed (Zipf, 15 experts: few blocks,
// each with all of K to walk); 32 tokens skewed 196 and 154.  So does the decode
// pipeline's factored gate/up (4 tokens 140 and 141, skewed 75 and 92).
static bool q3_tiles(const dsk_moe_desc& d) {
  return d.hidden % 4096 == 0 && d.inter % 512 == 0 && d.tokens < 24 && (d.tokens >= 3 || d.inter == 2048);
}

bool grouped_wide_q3(const dsk_moe_desc& d) {
  return wide_q3(d) && grouped_path(d) && !prefill_gemm(d) && !q3_tiles(d);
}

bool wide_shapes(const dsk_moe_desc& d) {
  return d.quant == DSK_QUANT_FP4 && d.x_dtype == DSK_DTYPE_BF16 && d.hidden % kWdStep == 0 &&
         d.inter % kWdStep == 0 && d.inter_shared % 128 == 0 && d.hidden < 8192 && d.inter < 8192 &&
         int64_t{d.tokens} * d.top_k * 3 * d.inter < (int64_t{1} << 32) &&
         int64_t{d.tokens} * 2 * d.hidden < (int64_t{1} << 32) && wd_lds_bytes(kWdMaxCT, 3, d.inter) <= kMaxLds &&
         wd_lds_bytes(kWdMaxCT, 2, d.hidden) <= kMaxLds;
}

namespace {

int wide_col_tiles(const dsk_moe_desc& d) { return d.tokens <= 16 ? 1 : kWdMaxCT; }

// The shared expert's column tiles (T rows of x, or of h's pair) in a wide launch: as
// much LDS as two blocks a CU leave each.
size_t shared_tile_lds(const dsk_moe_desc& d) {
  const size_t x = static_cast<size_t>(d.tokens) * (d.hidden + 8) * 2, h = static_cast<size_t>(kGNC + d.tokens) * (d.inter_shared + 8) * 2;
  const size_t red = static_cast<size_t>(kGI) * kGKS * 2 * 64 * 4 * sizeof(float);
  return x > h ? (x > red ? x : red) : (h > red ? h : red);
}
bool wide_shared_tiles(const dsk_moe_desc& d) { return d.tokens <= kGNC && shared_tile_lds(d) <= kMaxLds / 2; }

GroupedArgs wide_args(const dsk_moe_desc& d, const Workspace& L, const ExpertsArgs& a, const SlotDesc* desc,
                      const int32_t* xrow, const float* wrow, const WideCall& w) {
  GroupedArgs p = grouped_args(d, L, a, desc, xrow, wrow);
  p.xe = p.xp + static_cast<size_t>(d.tokens) * 2 * d.hidden;
  p.he = p.hp + static_cast<size_t>(d.tokens) * d.top_k * w.h_planes * d.inter;
  p.max_rows = w.max_rows;
  p.on = w.on;
  p.sh_on = w.on && w.sh_on ? 1 : 0;
  p.y_bf16 = w.y_bf16;
  p.sh_tiles = wide_shared_tiles(d) && d.x_dtype == DSK_DTYPE_BF16 ? 1 : 0;
  p.sh_tg = (d.tokens + kGsCols - 1) / kGsCols;
  p.up_groups = d.inter / 16 / kWdWaves;
  p.dn_groups = d.hidden / 256;
  if (d.quant == DSK_QUANT_Q3) {
    p.up_groups = d.inter / 16 / kWqUpTiles;
    p.dn_groups = d.hidden / 128;
  }
  // q3 under the device switch: blocks for 64 slots, each walking every 64th.  Skewed
  // routing switches them off, and a block per slot then costs what it takes to launch
  // 8192 that only look (layer of 300 tokens, top-8 of 256: 406 us, 395 so, 390
  // without the wide kernels; even routing 200 tokens: 982 and 1029, without 1801)
  p.slot_step = max_slots(d);
  if (d.quant == DSK_QUANT_Q3 && w.on && p.slot_step > 64) p.slot_step = 64;
  p.up_shared = !w.shared    ? 0
                : p.sh_tiles ? d.inter_shared / 16 / kGI
                             : (d.inter_shared / 16 + kGW / 2 - 1) / (kGW / 2) * p.sh_tg;
  p.dn_shared = w.shared && d.inter_shared > 0 ? d.hidden / 128 * p.sh_tg : 0;
  return p;
}

// Rows up to which a slot may run on wide_mul_few, with LDS for two blocks a CU.
int wide_few_rows(const dsk_moe_desc& d, int planes, int K) {
  if (wide_col_tiles(d) != 1 || d.quant != DSK_QUANT_FP4) return 0;
  int rows = kWfRows;
  while (rows > 0 && wf_lds_bytes(rows, planes, K) > kMaxLds / 2) --rows;
  return rows;
}

// LDS of a wide launch of the FP4 or q3 kernels: the slots' passes or few rows over K,
// and the shared expert's form (if any of its blocks are there).
size_t wide_lds(const dsk_moe_desc& d, const GroupedArgs& p, int planes, int K, int shared_blocks, size_t shared_walk) {
  size_t lds = d.quant == DSK_QUANT_Q3 ? wq_lds_bytes(planes) : wd_lds_bytes(wide_col_tiles(d), planes, K);
  if (p.few > 0 && wf_lds_bytes(p.few, planes, K) > lds) lds = wf_lds_bytes(p.few, planes, K);
  const size_t sh = shared_blocks == 0 ? 0 : p.sh_tiles ? shared_tile_lds(d) : shared_walk;
  return sh > lds ? sh : lds;
}

}  // namespace

hipError_t launch_wide_up(const dsk_moe_desc& d, const Workspace& L, const ExpertsArgs& a, const SlotDesc* desc,
                          const int32_t* xrow, const float* wrow, const WideCall& w, hipStream_t s) {
  GroupedArgs p = wide_args(d, L, a, desc, xrow, wrow, w);
  const bool q3 = d.quant == DSK_QUANT_Q3;
  const int ct = wide_col_tiles(d), planes = q3 ? 1 : 2;
  p.few = wide_few_rows(d, planes, d.hidden);
  const unsigned blocks = static_cast<unsigned>(p.up_shared + p.slot_step * p.up_groups * (p.few > 0 ? kWfKS : 1));
  const size_t lds = wide_lds(d, p, planes, d.hidden, p.up_shared, gs_up_lds_bytes());
  if (q3) launch_kernel(k_up_wide_q3, blocks, kWdWaves * 64, lds, s, p);
  else if (w.h_planes == 2) launch_kernel(k_up_wide<2, kWdMaxCT>, blocks, kWdWaves * 64, lds, s, p);
  else if (ct == 1) launch_kernel(k_up_wide<3, 1>, blocks, kWdWaves * 64, lds, s, p);
  else launch_kernel(k_up_wide<3, kWdMaxCT>, blocks, kWdWaves * 64, lds, s, p);
  return hipGetLastError();
}

hipError_t launch_wide_down(const dsk_moe_desc& d, const Workspace& L, const ExpertsArgs& a, const SlotDesc* desc,
                            const WideCall& w, hipStream_t s) {
  GroupedArgs p = wide_args(d, L, a, desc, nullptr, nullptr, w);
  const bool q3 = d.quant == DSK_QUANT_Q3;
  const int ct = wide_col_tiles(d), planes = q3 ? 2 : w.h_planes;
  p.few = wide_few_rows(d, planes, d.inter);
  const unsigned blocks = static_cast<unsigned>(p.dn_shared + p.slot_step * p.dn_groups * (p.few > 0 ? kWfKS : 1));
  const size_t lds = wide_lds(d, p, planes, d.inter, p.dn_shared, gs_down_lds_bytes());
  if (q3) launch_kernel(k_down_wide_q3, blocks, kWdWaves * 64, lds, s, p);
  else if (w.h_planes == 2) launch_kernel(k_down_wide<2, kWdMaxCT>, blocks, kWdWaves * 64, lds, s, p);
  else if (ct == 1) launch_kernel(k_down_wide<3, 1>, blocks, kWdWaves * 64, lds, s, p);
  else launch_kernel(k_down_wide<3, kWdMaxCT>, blocks, kWdWaves * 64, lds, s, p);
  return hipGetLastError();
}

bool wide_q3(const dsk_moe_desc& d) {
  return d.quant == DSK_QUANT_Q3 && d.x_dtype == DSK_DTYPE_BF16 && d.hidden >= kWqStep && d.inter >= kWqStep &&
         d.inter_shared % 128 == 0 && int64_t{d.tokens} * d.top_k * d.inter < (int64_t{1} << 31) &&
         int64_t{d.tokens} * d.hidden < (int64_t{1} << 31);
}

bool wide_pair(const dsk_moe_desc& d) {
  return d.quant == DSK_QUANT_FP4 && d.x_dtype == DSK_DTYPE_F32 && d.tokens < kPrefillMinTokens &&
         d.hidden % kWdStep == 0 && d.inter % kWdStep == 0 && d.inter_shared % 128 == 0 && d.hidden < 8192 &&
         d.inter < 8192 && wp_lds_bytes(d.hidden) <= kMaxLds && wp_lds_bytes(d.inter) <= kMaxLds;
}

hipError_t launch_experts_wide_pair(const dsk_moe_desc& d, const Workspace& L, const ExpertsArgs& a,
                                    const SlotDesc* desc, const int32_t* xrow, const float* wrow, hipStream_t s,
                                    int repeat, bool hs_ready) {
  GroupedArgs p = wide_args(d, L, a, desc, xrow, wrow, WideCall{3, kAllRows, nullptr, 0, d.inter_shared > 0});
  if (hs_ready) p.up_shared = 0;
  p.x = reinterpret_cast<const uint16_t*>(a.ws + L.xb_hi);
  p.x_lo = reinterpret_cast<const uint16_t*>(a.ws + L.xb_lo);
  const size_t sh = d.inter_shared > 0 ? gs_down_lds_bytes() : 0;
  const size_t ul = wp_lds_bytes(d.hidden) > sh ? wp_lds_bytes(d.hidden) : sh;
  const size_t dl = wp_lds_bytes(d.inter) > sh ? wp_lds_bytes(d.inter) : sh;
  hipError_t e;
  for (int r = 0; r < repeat; ++r) {
    launch_kernel(k_up_wide_pair, static_cast<unsigned>(p.up_shared + max_slots(d) * p.up_groups), kWdWaves * 64, ul, s, p);
    if ((e = hipGetLastError()) != hipSuccess) return e;
  }
  if ((e = stage_open(kStageDown)) != hipSuccess) return e;
  for (int r = 0; r < repeat; ++r) {
    launch_kernel(k_down_wide_pair, static_cast<unsigned>(p.dn_shared + max_slots(d) * p.dn_groups), kWdWaves * 64, dl, s, p);
    if ((e = hipGetLastError()) != hipSuccess) return e;
  }
  return hipSuccess;
}

hipError_t launch_grouped_up_routed(const dsk_moe_desc& d, const Workspace& L, const ExpertsArgs& a,
                                    const SlotDesc* desc, const int32_t* xrow, const float* wrow, hipStream_t s,
                                    int repeat, bool x_planes_ready) {
  const bool wide = grouped_wide(d) || grouped_wide_q3(d);
  GroupedArgs p = grouped_args(d, L, a, desc, xrow, wrow);
  p.up_shared = 0;
  const unsigned blocks = static_cast<unsigned>(max_slots(d) * p.up_groups);
  const size_t lds = up_lds(d);
  for (int r = 0; r < repeat; ++r) {
    hipError_t e = hipSuccess;
    if (wide) {
      if (d.quant == DSK_QUANT_FP4 && !x_planes_ready && (e = launch_pf_planes(d, L, a, s)) != hipSuccess) return e;
      if ((e = launch_wide_up(d, L, a, desc, xrow, wrow, WideCall{3, kAllRows, nullptr, 0, false}, s)) != hipSuccess)
        return e;
      continue;
    }
    if (p.q3f && (e = launch_x_q3(d, p, s)) != hipSuccess) return e;
    if (d.quant == DSK_QUANT_Q3) launch_kernel(k_up_grouped<RawQ3>, blocks, kGW * 64, lds, s, p);
    else launch_kernel(k_up_grouped<RawFP4>, blocks, kGW * 64, lds, s, p);
    if ((e = hipGetLastError()) != hipSuccess) return e;
  }
  return hipSuccess;
}

hipError_t launch_grouped_down(const dsk_moe_desc& d, const Workspace& L, const ExpertsArgs& a,
                               const SlotDesc* desc, hipStream_t s, int repeat, bool h_planes) {
  if (h_planes) {
    for (int r = 0; r < repeat; ++r) {
      const hipError_t e = launch_wide_down(d, L, a, desc, WideCall{3, kAllRows, nullptr, 0, d.inter_shared > 0}, s);
      if (e != hipSuccess) return e;
    }
    return hipSuccess;
  }
  const GroupedArgs p = grouped_args(d, L, a, desc, nullptr, nullptr);
  return grouped_down(d, p, s, repeat);
}

}  // namespace dsk
