// General bf16 "NT" GEMM on the LDS-DMA pipeline of the triangle contraction:
// for every batch b
//     C[i][j] = epilogue( sum_k A[i][k] * B[j][k] )
// with both operands k-contiguous (B a PyTorch [out, in] weight), the epilogue
// of gemm_nt_kernel (fjx_contract.hip): + bias[j], sigmoid or SiLU on the
// columns from act_col0, * gate[i][j], + residual[i][j], rows whose row_gate
// is 0 written as 0. It serves the projections of the general-width paths,
// whose row counts are the pair grid's (B N^2) and whose K is a layer width.
//
// Tiling as contract_dma_kernel: a 256 x 256 output tile per 512-thread
// workgroup (8 waves of 128 x 64) or 128 x 128 per 256 threads (4 waves of 64 x
// 64, two workgroups a CU), k in stages of 64 copied global -> LDS by DMA
// (buffer_load ... lds: no registers, no LDS write instructions), two stages in
// 128 or 64 KB of LDS, chunk c of row r in slot 8 r + (c ^ ((r / 2) % 8)) so the
// fragment reads of 16 consecutive rows hit 16 bank groups. The DMA goes
// through buffer resources sized to the operands, and a lane whose chunk lies
// past K gets an offset past the resource's end: rows past M or N and the k
// tail read as zero, so any M, N and K (K a multiple of 8) work. A lane's whole
// row offset is in its vector offset: the raw-buffer range check covers the
// vector and instruction offsets, not the scalar one, which carries only the k
// offset.
//
// Persistent: the resident workgroups walk their XCD's contiguous share of the
// tiles, n-tiles fastest, so an A row block is reused from that XCD's L2 by its
// consecutive n-tiles; the next tile's first stage goes out during the last
// k-step. Accumulators are transposed (A operand = B rows), and the B rows of a
// wave's 64 columns sit in LDS in a permuted order (the DMA of B writes LDS row
// 16 j + r of a 64-row block from B row pcol(j, r) = 32 (j / 2) + 8 (r / 4) +
// 4 (j % 2) + r % 4), so that a lane's accumulators of column tiles 2s and 2s+1
// are 8 consecutive output columns: 16-byte epilogue accesses, half the store
// instructions of 4-column pieces. The fragment reads and their swizzle are
// those of consecutive LDS rows.
//
// The paired forms read two weights, 32 rows of each in turn, so a wave holds
// both products of its units in the same lanes and combines them without LDS.
// kPairPlanes writes the gated product as the triangle contraction reads it,
// channel by channel with rows padded to 64 columns (accumulators not
// transposed and A's rows permuted instead: a lane's 8 consecutive values are
// positions of one channel): the product, the position-major copy and the two
// passes that turned it took 131 + 90 us of a 384-channel tri-mul at n = 245,
// this form takes 115 us. Here the kernel is bound by its k-steps being short (6
// of 64): a third of the time goes into epilogues that one workgroup a CU can
// not overlap with matrix work.
#include <algorithm>
#include <type_traits>

#include "fjx_common.hpp"
#include "fjx_kernels.hpp"
#include "fjx_tile.hpp"

namespace fjx {
namespace {

constexpr int kGDK = 64;         // k per stage
constexpr int kGCH = kGDK / 8;   // 16-byte chunks per tile row in a stage
constexpr int kGRPI = 64 / kGCH; // tile rows per DMA instruction (1 KB)
constexpr int kGNI = kGCH / 2;   // DMA instructions per wave per operand per stage (32 rows)
constexpr int kGXcd = 8;
constexpr uint32_t kGOob = 0x80000000u;  // a lane offset past every resource's end
// fewer 256 x 256 tiles than this go to gemm_nt_kernel's 128- or 64-wide tiles
constexpr int64_t kMinTiles = 64;

enum GemmMode { kRows, kPair, kPairPlanes };

__device__ __forceinline__ int gswz(int r) { return (r / (16 / kGCH)) % kGCH; }
__device__ __forceinline__ int gslot(int r, int c) { return kGCH * r + (c ^ gswz(r)); }

// raw buffer resource over `bytes` bytes from `base` (at most 2^31 - 1: the
// tiles address their operands from a per-tile base)
__device__ __forceinline__ __amdgpu_buffer_rsrc_t grsrc(const void* base, int64_t bytes) {
  const int64_t b = bytes < 0 ? 0 : (bytes > 0x7FFFFFFF ? 0x7FFFFFFF : bytes);
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, (int)b, 0x00020000);
}

__device__ __forceinline__ void gopaque(int& v) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("" : "+s"(v));
#endif
}

// the paired forms' value of one unit, both products rounded to bf16 first
__device__ __forceinline__ float pair_value(int kind, float x, float y) {
  const float a = round_to<bf16>(x), b = round_to<bf16>(y);
  return kind == 1 ? a * fast_sigmoid(a) * b : a * round_to<bf16>(fast_sigmoid(b));
}

// kPairPlanes: row m of the product is column s of row r of item b of a grid
// whose rows are `pitch` apart (a multiple of 64, so the 32 or 64 rows a wave
// moves or stores at a time are of one grid row)
struct GridBlock {
  int b, r, s;
};
// x / d as (x * inverse(d)) >> 32, exact while x * d < 2^32 (gemm_dma_ok): a
// division by a run-time value is some 25 vector instructions, eight of them a tile
uint64_t inverse(int64_t d) { return ((uint64_t)1 << 32) / (uint64_t)d + 1; }
struct GridInverse {
  uint64_t blocks, n;  // of the 64-column blocks of a row, and of n
};
__device__ __forceinline__ GridBlock grid_block(int64_t m, int n, int pitch, const GridInverse& inv) {
  const uint32_t blk = (uint32_t)(m >> 6);
  const uint32_t row = (uint32_t)((blk * inv.blocks) >> 32);
  GridBlock g;
  g.s = (int)((uint32_t)m - row * (uint32_t)pitch);
  g.b = (int)((row * inv.n) >> 32);
  g.r = (int)(row - (uint32_t)g.b * (uint32_t)n);
  return g;
}

template <int BT, GemmMode MODE>
__device__ __forceinline__ void gemm_dma_body(const GemmParams<bf16, bf16>& P, const GridInverse& inv = {}) {
  constexpr int MI = BT / 32;  // 16-row tiles per wave (waves: 2 along the rows)
  constexpr int WN = BT / 64;  // waves along the columns
  constexpr bool kPaired = MODE != kRows;
  constexpr int kStores = MI;  // output stores per lane per tile of the paired forms
  __shared__ __attribute__((aligned(16))) bf16 S[2][2][BT * kGDK];  // [stage][A, B][BT rows x 64]
  __shared__ float Mk[MODE == kPairPlanes ? BT : 1];                // the tile rows' mask

  const int64_t M = P.m, N = P.n;
  const int K = (int)P.k;
  const int tn = (int)((N + BT - 1) / BT);
  const int64_t total = ((M + BT - 1) / BT) * tn;
  const int per_xcd = (int)gridDim.x / kGXcd;  // the grid is a multiple of 8
  const int64_t xcd = blockIdx.x % kGXcd;
  const int64_t hi = (xcd + 1) * total / kGXcd;

  const int t = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);  // uniform: wave offsets in SGPRs
  const int lane = t & 63;
  const int li = lane & 15;
  const int lg = lane >> 4;
  const int wm = (wave / WN) * 16 * MI;
  const int wn = (wave % WN) * 64;

  // this lane's DMA rows and chunks: instruction j writes LDS row
  // r = 32 wave + 8 j + lane / 8, chunk c (k = 8 c), of a consecutive operand
  // from row 8 j + lane / 8 of the wave's 32, of a permuted one from row
  // 16 (j % 2) + 4 (j / 2) + 8 (lane bit 5) + (lane / 8) % 4. The swizzle of r
  // depends on j only through j % 2, so two per-lane offsets per operand serve
  // all four instructions, plus a uniform step (16 consecutive or 4 permuted
  // rows per two instructions) added to the lane's offset. B is permuted, and
  // A too where the accumulators are not transposed (kPairPlanes).
  const int64_t arow = MODE == kPairPlanes && P.grid_t ? P.grid_n * P.lda : P.lda;
  uint32_t aoff[2], boff[2];
  int kc[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int c = (lane % kGCH) ^ gswz(32 * wave + kGRPI * j + lane / kGCH);
    kc[j] = 8 * c;
    const int rc = kGRPI * j + lane / kGCH;
    const int rp = 16 * j + 8 * ((lane >> 5) & 1) + ((lane >> 3) & 3);
    aoff[j] = (uint32_t)((MODE == kPairPlanes ? rp : rc) * arow * 2 + 16 * c);
    boff[j] = (uint32_t)(rp * P.ldb * 2 + 16 * c);
  }
  const uint32_t astep = (uint32_t)((MODE == kPairPlanes ? 4 : 2 * kGRPI) * arow * 2), bstep = (uint32_t)(4 * P.ldb * 2);

  struct Tile {
    int64_t m0;
    int n0;
    __amdgpu_buffer_rsrc_t ra, rb;  // from this wave's 32 rows of A and of B
  };
  auto tile_at = [&](int ti, int tj) {
    Tile tl;
    tl.m0 = (int64_t)ti * BT;
    tl.n0 = tj * BT;
    const int64_t ar = tl.m0 + 32 * wave;
    if constexpr (MODE == kPairPlanes) {
      const int n = (int)P.grid_n;
      const GridBlock g = grid_block(ar, n, (int)P.grid_pitch, inv);
      const int64_t row0 = (int64_t)g.b * n * n + (P.grid_t ? (int64_t)g.s * n + g.r : (int64_t)g.r * n + g.s);
      tl.ra = grsrc(P.a + row0 * P.lda, ar < M && g.s < n ? ((n - g.s - 1) * arow + P.lda) * 2 : 0);
    } else {
      tl.ra = grsrc(P.a + ar * P.lda, (M - ar) * P.lda * 2);
    }
    if constexpr (kPaired) {
      // LDS rows alternate between 32 rows of the first weight and the same
      // 32 of the second: a wave's 64 columns are both halves of 32 units
      const int64_t u = tl.n0 / 2 + 32 * (wave >> 1);
      tl.rb = grsrc((wave & 1 ? P.b2 : P.b) + u * P.ldb, (N / 2 - u) * P.ldb * 2);
    } else {
      const int64_t br = tl.n0 + 32 * wave;
      tl.rb = grsrc(P.b + br * P.ldb, (N - br) * P.ldb * 2);
    }
    return tl;
  };
  // stage st <- k-tile kt of tile tl (st a compile-time constant at every call)
  auto issue = [&](const Tile& tl, int kt, int st) {
    const int k0 = kt * kGDK;
    // opaque here, so the sums and compares below are formed per call rather
    // than hoisted into loop-invariant registers, which spilled: the reload of
    // a spilled 64-bit k offset waited (vmcnt counts in issue order) for the
    // next stage's DMA issued just before it, in every k-step
#pragma unroll
    for (int j = 0; j < 2; ++j) asm volatile("" : "+v"(aoff[j]), "+v"(boff[j]), "+v"(kc[j]));
    // the k offset goes in the scalar offset; a lane whose chunk lies past K
    // reads from past the resource's end
    const int krem = K - k0;
    const bool in0 = kc[0] < krem, in1 = kc[1] < krem;
#pragma unroll
    for (int j = 0; j < kGNI; ++j) {
      const bool kin = (j & 1) ? in1 : in0;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          tl.ra, (__attribute__((address_space(3))) void*)(&S[st][0][(32 * wave + kGRPI * j) * kGDK]), 16,
          kin ? aoff[j & 1] + (uint32_t)(j >> 1) * astep : kGOob, (uint32_t)(2 * k0), 0, 0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          tl.rb, (__attribute__((address_space(3))) void*)(&S[st][1][(32 * wave + kGRPI * j) * kGDK]), 16,
          kin ? boff[j & 1] + (uint32_t)(j >> 1) * bstep : kGOob, (uint32_t)(2 * k0), 0, 0);
    }
  };

  const int ktiles = (K + kGDK - 1) / kGDK;
  int64_t lid = xcd * total / kGXcd + blockIdx.x / kGXcd;
  if (lid >= hi) return;
  // a workgroup's tiles are lid, lid + per_xcd, ...: the next one's coordinates
  // come from fixed carries
  const int step_i = per_xcd / tn, step_j = per_xcd % tn;
  int ci = (int)(lid / tn), cj = (int)(lid % tn);
  Tile cur = tile_at(ci, cj);
  issue(cur, 0, 0);
  int pend = 0;  // the previous tile's stores may be in flight (opaque: or the compiler peels a k-step per case)
  for (;;) {
    const bool has_next = lid + per_xcd < hi;
    int ni = ci + step_i, nj = cj + step_j;
    if (nj >= tn) {
      nj -= tn;
      ++ni;
    }
    const Tile nxt = has_next ? tile_at(ni, nj) : cur;

    float mk = 0.f;
    if constexpr (MODE == kPairPlanes) {
      // the mask of tile row t: 0 past the grid row's n
      if (wave < BT / 64) {
        const int64_t m = cur.m0 + 64 * wave;
        const int n = (int)P.grid_n;
        const GridBlock g = grid_block(m, n, (int)P.grid_pitch, inv);
        if (m < M && g.s + lane < n) {
          const int64_t at = (int64_t)g.b * n * n + (P.grid_t ? (int64_t)(g.s + lane) * n + g.r
                                                              : (int64_t)g.r * n + g.s + lane);
          mk = P.grid_mask ? to_f32(P.grid_mask[at]) : 1.f;
        }
      }
    }

    f32x4 acc[4][MI];
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int i = 0; i < MI; ++i) acc[j][i] = f32x4{0.f, 0.f, 0.f, 0.f};

    // k-tile kt uses stage kt % 2; every tile starts in stage 0, so the
    // next tile's first stage goes to the stage after the last k-tile's
    for (int kb = 0; kb < ktiles; kb += 2) {
#pragma unroll
      for (int st = 0; st < 2; ++st) {
        const int kt = kb + st;
        if (st == 1 && kt >= ktiles) break;  // an odd number of k-tiles ends in stage 0
        // this wave's DMA of stage st is complete; on a tile's first k-step
        // the previous tile's stores, issued after that DMA, may still run
        if (kPaired && st == 0 && pend) lds_wait<kStores>();
        else lds_wait<0>();
        pend = 0;
        gopaque(pend);
        lds_barrier();
        if (kt + 1 < ktiles) issue(cur, kt + 1, st ^ 1);
        else if (has_next && st == 1) issue(nxt, 0, 0);
        const bf16* As_ = &S[st][0][0];
        const bf16* Bs_ = &S[st][1][0];
#pragma unroll
        for (int ks = 0; ks < kGDK / 32; ++ks) {
          bf16x8 af[MI], bfr[4];
#pragma unroll
          for (int i = 0; i < MI; ++i)
            af[i] = *reinterpret_cast<const bf16x8*>(As_ + 8 * gslot(wm + 16 * i + li, 4 * ks + lg));
#pragma unroll
          for (int j = 0; j < 4; ++j)
            bfr[j] = *reinterpret_cast<const bf16x8*>(Bs_ + 8 * gslot(wn + 16 * j + li, 4 * ks + lg));
#pragma unroll
          for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int i = 0; i < MI; ++i) {
              if constexpr (MODE == kPairPlanes) mma(acc[j][i], af[i], bfr[j]);
              else mma(acc[j][i], bfr[j], af[i]);
            }
        }
      }
    }
    if (ktiles & 1) {
      // an odd number of k-tiles: the last one is in stage 0, where the next
      // tile's first stage goes once every wave is past its reads
      lds_wait<63>();
      lds_barrier();
      if (has_next) issue(nxt, 0, 0);
    }

    // lane coordinates, opaque here: the epilogue's offsets are then formed
    // after the k-loop instead of being hoisted above it (and the paired forms'
    // stores stay behind the next tile's DMA, as its wait counts on)
    int lrow = li, lcol = 8 * lg;
    asm volatile("" : "+v"(lrow), "+v"(lcol) : : "memory");

    if constexpr (MODE == kPair) {
      // tiles 0, 1 hold units u0 + lcol .. +7 of a, tiles 2, 3 of b
      const int64_t u0 = cur.n0 / 2 + wn / 2;
      const __amdgpu_buffer_rsrc_t ro =
          grsrc(P.c + cur.m0 * P.ldc + u0, u0 < N / 2 ? ((M - cur.m0 - 1) * P.ldc + 32) * 2 : 0);
#pragma unroll
      for (int i = 0; i < MI; ++i) {
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e)
          v[e] = pair_value(P.swiglu, acc[e >> 2][i][e & 3], acc[2 + (e >> 2)][i][e & 3]);
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, pack8<bf16>(v)), ro,
                                               (uint32_t)((wm + 16 * i + lrow) * (int)P.ldc + lcol) * 2, 0, 0);
      }
    } else if constexpr (MODE == kPairPlanes) {
      // tiles i = 2s, 2s + 1 hold columns 32 s + lcol .. +7 of a grid row, of
      // unit u0 + 8 (li / 4) + 4 j + li % 4 (j: 0, 1)
      if (wave < BT / 64) Mk[64 * wave + lane] = mk;
      lds_wait<63>();
      lds_barrier();
      const int n = (int)P.grid_n, pitch = (int)P.grid_pitch;
      const int64_t half = P.grid_units, plane = (int64_t)n * pitch;
      const int u0 = cur.n0 / 2 + wn / 2;
      const bool second = u0 >= half;
#pragma unroll
      for (int h = 0; h < MI / 4; ++h) {
        const int64_t m = cur.m0 + wm + 64 * h;
        const GridBlock g = grid_block(m, n, pitch, inv);
        bf16* O = (second ? P.c2 : P.c) + ((int64_t)g.b * half + u0 - (second ? half : 0)) * plane +
                  (int64_t)g.r * pitch + g.s;
        // every unit of the wave lies in a plane, and its 64 columns within
        // the pitch, or none is stored
        const __amdgpu_buffer_rsrc_t ro = grsrc(O, m < M && u0 < N / 2 ? (31 * plane + 64) * 2 : 0);
        const uint32_t ulane = (uint32_t)((8 * (lrow >> 2) + (lrow & 3)) * plane);
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          float mv[8];
#pragma unroll
          for (int e = 0; e < 8; ++e) mv[e] = Mk[wm + 64 * h + 32 * s + lcol + e];
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            float v[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
              const int i = 4 * h + 2 * s + (e >> 2);
              v[e] = round_to<bf16>(pair_value(2, acc[j][i][e & 3], acc[2 + j][i][e & 3])) * mv[e];
            }
            if (g.s + 64 > n) {  // the padding stays zero whatever the weights hold
#pragma unroll
              for (int e = 0; e < 8; ++e) v[e] = g.s + 32 * s + lcol + e < n ? v[e] : 0.f;
            }
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, pack8<bf16>(v)), ro,
                                                   (ulane + (uint32_t)(4 * j * plane) + 32 * s + lcol) * 2, 0, 0);
          }
        }
      }
    } else {
      // this lane holds row m0 + wm + 16 i + lrow, columns n0 + wn + 32 s + lcol
      // .. +7 in acc[2s][i] (the first 4) and acc[2s+1][i]. What the epilogue
      // reads is loaded for 4 rows before the first is used: one
      // row at a time, every load's latency was in line (with the selects
      // below 64 -> 54 us for 60025 x 384 x 384 with a gate and a residual)
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const int64_t col = cur.n0 + wn + 32 * s + lcol;
        if (col >= N) continue;  // N is a multiple of 8 (checked by the launcher)
        const int act0 = (int)max<int64_t>(P.act_col0 - col, -1);  // of this lane's 8 columns, the activated ones
        float bias[8];
#pragma unroll
        for (int e = 0; e < 8; ++e)
          bias[e] = P.bias && (P.bias_n == 0 || col + e < P.bias_n) ? to_f32(P.bias[col + e]) : 0.f;
#pragma unroll
        for (int i0 = 0; i0 < MI; i0 += 4) {
          int64_t off[4];
          u32x4 gate[4], res[4];
          float zero[4], scale[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int64_t row = cur.m0 + wm + 16 * (i0 + i) + lrow;
            off[i] = row < M ? grid_row(row, P.map_n, P.map_t) : -1;
          }
          if (P.gate) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
              gate[i] = *reinterpret_cast<const u32x4*>(P.gate + (off[i] < 0 ? 0 : off[i]) * P.ldc + col);
          }
          if (P.residual) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
              res[i] = *reinterpret_cast<const u32x4*>(P.residual + (off[i] < 0 ? 0 : off[i]) * P.ldc + col);
          }
#pragma unroll
          for (int i = 0; i < 4; ++i) zero[i] = scale[i] = 1.f;
          if (P.row_gate) {
#pragma unroll
            for (int i = 0; i < 4; ++i) zero[i] = to_f32(P.row_gate[off[i] < 0 ? 0 : off[i]]);
          }
          if (P.proj_round && P.row_scale) {
#pragma unroll
            for (int i = 0; i < 4; ++i) scale[i] = to_f32(P.row_scale[off[i] < 0 ? 0 : off[i]]);
          }
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            float v[8];
#pragma unroll
            for (int e = 0; e < 8; ++e)
              v[e] = (e < 4 ? acc[2 * s][i0 + i][e] : acc[2 * s + 1][i0 + i][e - 4]) + bias[e];
            // one uniform branch per 8 values and selects within them: a branch
            // per value kept the exponentials from overlapping
            if (P.act == 1) {
#pragma unroll
              for (int e = 0; e < 8; ++e) {
                const float y = fast_sigmoid(v[e]);
                v[e] = e >= act0 ? y : v[e];
              }
            } else if (P.act == 2) {
#pragma unroll
              for (int e = 0; e < 8; ++e) {
                const float y = v[e] * fast_sigmoid(v[e]);  // silu
                v[e] = e >= act0 ? y : v[e];
              }
            }
            if (P.gate) {
              float g[8];
              to_f32x8(__builtin_bit_cast(bf16x8, gate[i]), g);
#pragma unroll
              for (int e = 0; e < 8; ++e) v[e] *= g[e];
            }
            if (P.proj_round) {
#pragma unroll
              for (int e = 0; e < 8; ++e) v[e] = round_to<bf16>(round_to<bf16>(v[e]) * scale[i]);
            }
            if (P.residual) {
              float r[8];
              to_f32x8(__builtin_bit_cast(bf16x8, res[i]), r);
#pragma unroll
              for (int e = 0; e < 8; ++e) v[e] += r[e];
            }
            if (P.row_gate && zero[i] == 0.f) {
#pragma unroll
              for (int e = 0; e < 8; ++e) v[e] *= 0.f;
            }
            if (off[i] >= 0) store8(P.c + off[i] * P.ldc + col, pack8<bf16>(v));
          }
        }
      }
    }
    if (!has_next) break;
    lid += per_xcd;
    ci = ni;
    cj = nj;
    cur = nxt;
    pend = 1;
    gopaque(pend);
  }
  // no DMA is in flight here: the prefetch of a next tile is issued only if there is one
}

}  // namespace

// plain kernels around the body: a __global__ template that uses the buffer
// builtins loses its host stub
#define FJX_GEMM_DMA(BT)                                                                                        \
  __global__ __launch_bounds__(2 * BT) void gemm_dma_kernel_##BT(GemmParams<bf16, bf16> P) {                      \
    gemm_dma_body<BT, kRows>(P);                                                                                  \
  }                                                                                                               \
  __global__ __launch_bounds__(2 * BT) void gemm_dma_pair_kernel_##BT(GemmParams<bf16, bf16> P) {                 \
    gemm_dma_body<BT, kPair>(P);                                                                                  \
  }                                                                                                               \
  __global__ __launch_bounds__(2 * BT) void gemm_dma_planes_kernel_##BT(GemmParams<bf16, bf16> P, GridInverse inv) { \
    gemm_dma_body<BT, kPairPlanes>(P, inv);                                                                       \
  }
FJX_GEMM_DMA(256)
FJX_GEMM_DMA(128)
#undef FJX_GEMM_DMA

bool gemm_dma_ok(const GemmParams<bf16, bf16>& p) {
  // 16-byte rows for the DMA, 16-byte output groups, and enough rows to fill
  // the device with 256 x 256 tiles
  auto al16 = [](const void* q) { return (reinterpret_cast<uintptr_t>(q) & 15) == 0; };
  constexpr int64_t T = 256;
  const bool ok = p.batches == 1 && p.k % 8 == 0 && p.lda % 8 == 0 && p.ldb % 8 == 0 && p.n % 8 == 0 &&
                  p.ldc % 8 == 0 && al16(p.a) && al16(p.b) && al16(p.b2) && al16(p.c) && al16(p.c2) &&
                  al16(p.gate) && al16(p.residual) && p.lda * 2 * T < (int64_t)kGOob &&
                  p.ldb * 2 * T < (int64_t)kGOob && p.ldc * 2 * T < (int64_t)kGOob;
  const int64_t total = ((p.m + T - 1) / T) * ((p.n + T - 1) / T);
  // at least half a tile of columns: narrower products (a triangle bias of a
  // few heads) would waste most of every tile
  if (!ok || total < kMinTiles || total >= ((int64_t)1 << 28) || p.n < T / 2) return false;
  if (p.swiglu && (p.n % T || p.gate || p.residual || p.proj_round || p.map_t)) return false;
  // planes: a wave's 32 units in one of the two outputs, its DMA rows and its
  // output planes within the 32-bit offsets
  return !p.grid_pitch || (p.grid_units % 32 == 0 && p.grid_pitch % 64 == 0 && p.m < ((int64_t)1 << 31) - T &&
                           32 * p.grid_n * p.lda * 2 < (int64_t)kGOob &&
                           32 * p.grid_n * p.grid_pitch * 2 < (int64_t)kGOob &&
                           p.m / 64 * (p.grid_pitch / 64) < ((int64_t)1 << 32) &&
                           p.m / p.grid_pitch * p.grid_n < ((int64_t)1 << 32));
}

template <int BT>
static void launch_gemm_dma_bt(const GemmParams<bf16, bf16>& p, hipStream_t st) {
  const void* k = p.grid_pitch ? reinterpret_cast<const void*>(BT == 256 ? gemm_dma_planes_kernel_256 : gemm_dma_planes_kernel_128)
                  : p.swiglu   ? reinterpret_cast<const void*>(BT == 256 ? gemm_dma_pair_kernel_256 : gemm_dma_pair_kernel_128)
                               : reinterpret_cast<const void*>(BT == 256 ? gemm_dma_kernel_256 : gemm_dma_kernel_128);
  const int64_t total = ((p.m + BT - 1) / BT) * ((p.n + BT - 1) / BT);
  const int64_t cap = std::max<int64_t>(kGXcd, tile::resident_blocks(k, 2 * BT) / kGXcd * kGXcd);
  const dim3 grid((unsigned)std::min<int64_t>(cap, (total + kGXcd - 1) / kGXcd * kGXcd)), block(2 * BT);
  if (p.grid_pitch)
    hipLaunchKernelGGL((BT == 256 ? gemm_dma_planes_kernel_256 : gemm_dma_planes_kernel_128), grid, block, 0, st, p,
                       GridInverse{inverse(p.grid_pitch / 64), inverse(p.grid_n)});
  else if (p.swiglu)
    hipLaunchKernelGGL((BT == 256 ? gemm_dma_pair_kernel_256 : gemm_dma_pair_kernel_128), grid, block, 0, st, p);
  else
    hipLaunchKernelGGL((BT == 256 ? gemm_dma_kernel_256 : gemm_dma_kernel_128), grid, block, 0, st, p);
}

bool launch_gemm_dma(const GemmParams<bf16, bf16>& p, hipStream_t st) {
  if (!gemm_dma_ok(p)) return false;
  // 128-wide tiles, two workgroups a CU, where they take fewer rounds over the
  // 256 CUs (a round of 256-wide tiles counted as two of theirs) by more than
  // their operands' second reading costs: 1161 against 1056 us for a transition
  // of 200000 x 384, where neither has a last round to lose, and 1775 against
  // 1738 us for the one-weight products of a tri-attn at n = 512. Saved rounds:
  // tri-mul of 384 channels at n = 90, 86 against 110 us, at 110, 95 against
  // 112; transition of 8300 x 384, 65 against 85 us
  auto rounds = [&](int64_t bt, int64_t per_cu) {
    return (((p.m + bt - 1) / bt) * ((p.n + bt - 1) / bt) + 256 * per_cu - 1) / (256 * per_cu) * (bt == 256 ? 2 : 1);
  };
  if ((p.swiglu ? 6 : 17) * rounds(128, 2) < (p.swiglu ? 5 : 16) * rounds(256, 1))
    launch_gemm_dma_bt<128>(p, st);
  else
    launch_gemm_dma_bt<256>(p, st);
  return true;
}

}  // namespace fjx
