// The float32 forms of the row kernels (fjx_rowproj.hip) and of the pair
// transition (fjx_transition.hip) at 128 channels, on the bf16 matrix cores:
// every product runs as six bf16 MFMAs on three-plane splits of its operands
// (Split8, fjx_common.hpp), 2.7 times the rate of the fp32 MFMAs that bounded
// the fp32 instances of those kernels (trimul prologue at N = 256: the fp32
// matrix pipe was busy 64 % of its 87 us) at no larger error (relative to
// float64, whole tri-mul at N = 256: 4.8e-7 before, 3.8e-7 now). At N = 245:
// tri-mul prologue 100 -> 57 us, epilogue 70 -> 47; tri-attn prologue 69 -> 52,
// epilogue 60 -> 49; transition 248 -> 210. What bounds them now is the sum of
// MFMA, LDS reads, LayerNorm and splits: one workgroup fits a CU, and its two
// waves per SIMD mostly run the same phase.
//
// Common shape: tiles of 64 positions, 512 threads. LayerNorm takes 8 threads a
// position; its output is split once and stored as three [position][channel]
// bf16 planes in LDS (55 KB). Wave w owns 16 output channels of each product
// and holds their weights, split, in registers for the whole launch (48 VGPRs
// per 128-wide weight column tile), so that a workgroup works on two
// 128-channel products at a time; the prologues, which have four, run two
// kinds of workgroups over the same tiles. The virtual grid, masks and layouts
// are those of the bf16 kernels.
#include "fjx_common.hpp"
#include "fjx_kernels.hpp"
#include "fjx_tile.hpp"

namespace fjx {

using namespace tile;

namespace {

constexpr int kTS = 64;  // positions per tile
typedef bf16 Planes[3][kTS][kLd];

// channels of part j = t % 8 of a position: 8j .. 8j+7 and 64 + 8j .. +7
__device__ __forceinline__ int part_chunk(int q) { return 64 * q + 8 * (threadIdx.x & 7); }
struct Part {
  f32x8 f[2];
};
__device__ __forceinline__ void load_part(const float* src, Part& r) {
#pragma unroll
  for (int q = 0; q < 2; ++q) r.f[q] = src ? load8(src + part_chunk(q)) : f32x8{};
}
// the sum over the 8 lanes of a position: the quads' sums, then the half-row mirror
__device__ __forceinline__ float part_sum(float v) {
  v = quad_sum(v);
  return v + __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x141, 0xF, 0xF, false));
}
__device__ __forceinline__ void put_planes(Planes& xs, int row, int c, const f32x8& o, bool plain) {
  const Split8 s = split8(o, plain);
#pragma unroll
  for (int u = 0; u < 3; ++u) store8(&xs[u][row][c], s.p[u]);
}
// whether this LayerNorm's outputs (the affine of values within sqrt(127)) stay
// far from what split8_plain does not take; wave-uniform
__device__ __forceinline__ bool ln_plain(const LnAffine& l) {
  const int c = threadIdx.x & 63;
  const float big = fmaxf(fmaxf(fabsf(l.w[c]), fabsf(l.w[c + 64])), fmaxf(fabsf(l.b[c]), fabsf(l.b[c + 64])));
  return __builtin_amdgcn_ballot_w64(!(big < 0x1p120f)) == 0;
}
// LayerNorm (two-pass statistics) of the position t / 8 into row t / 8
__device__ __forceinline__ void ln_planes(const Part& r, const LnAffine& l, float eps, Planes& xs, bool plain) {
  float s = 0.f, q2 = 0.f;
#pragma unroll
  for (int q = 0; q < 2; ++q)
#pragma unroll
    for (int e = 0; e < 8; ++e) s += r.f[q][e];
  const float mean = part_sum(s) * (1.0f / kC);
#pragma unroll
  for (int q = 0; q < 2; ++q)
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float d = r.f[q][e] - mean;
      q2 += d * d;
    }
  const float rstd = __builtin_amdgcn_rsqf(part_sum(q2) * (1.0f / kC) + eps);
  const float shift = -mean * rstd;
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int c = part_chunk(q);
    const f32x8 w = load8(&l.w[c]), b = load8(&l.b[c]);
    f32x8 o;
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = fmaf(fmaf(r.f[q][e], rstd, shift), w[e], b[e]);
    put_planes(xs, threadIdx.x >> 3, c, o, plain);
  }
}

// one 16-channel column tile of a weight over K = 128, as loaded and split (all
// of a kernel's tiles are loaded before the first is split: the rare branch of
// a split would otherwise keep the next loads behind it)
struct RawTile {
  f32x8 f[4];
};
struct WTile {
  Split8 f[4];
};
__device__ __forceinline__ void load_raw(const float* w, int64_t ldw, int row, int64_t k0, RawTile& r) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) r.f[ks] = load8(w + row * ldw + k0 + 32 * ks + 8 * (lane >> 4));
}
__device__ __forceinline__ void split_tile(const RawTile& r, WTile& wt) {
  const bool plain = split_plain(r.f);
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) wt.f[ks] = split8(r.f[ks], plain);
}
__device__ __forceinline__ Split8 xfrag(const Planes& xs, int row, int ks) {
  Split8 x;
#pragma unroll
  for (int u = 0; u < 3; ++u) x.p[u] = load8(&xs[u][row][32 * ks + 8 * ((threadIdx.x >> 4) & 3)]);
  return x;
}
// 4 consecutive values -> the three planes (8-byte stores)
__device__ __forceinline__ void put_planes4(Planes& xs, int row, int c, const float* v) {
  const Split8 s = split8(f32x8{v[0], v[1], v[2], v[3], 0.f, 0.f, 0.f, 0.f});
#pragma unroll
  for (int u = 0; u < 3; ++u)
    *reinterpret_cast<bf16x4*>(&xs[u][row][c]) = bf16x4{s.p[u][0], s.p[u][1], s.p[u][2], s.p[u][3]};
}

}  // namespace

// ---------------------------------------------------------------------------
// Tri-mul prologue. Even workgroups produce a, odd ones b: wave w channels
// 16w .. 16w+15, written as three planes, `plane` elements apart, for the split
// contraction. Two LDS tiles: the next tile's LayerNorm runs halfway through
// this tile's products.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(512) void trimul_prologue_split_kernel(TriMulPrologueParams<float> P, bf16* a, bf16* b,
                                                                    int64_t plane, int64_t ntiles) {
  __shared__ __attribute__((aligned(16))) Planes xs[2];
  __shared__ __attribute__((aligned(16))) float mrow[2][kTS];
  __shared__ __attribute__((aligned(16))) LnAffine ln;

  const int64_t n = P.n, nn = n * n, pitch = P.pitch, chplane = n * pitch;
  const int64_t ntx = pitch / kTS;
  const int t = threadIdx.x;
  const int wave = t >> 6;
  const int lane = t & 63;
  const int li = lane & 15;
  const int lg = lane >> 4;
  const int p = t >> 3;
  const int half = blockIdx.x & 1;
  const int ch = 16 * wave + li;
  const int64_t stride = gridDim.x >> 1;

  WTile wp, wg;
  RawTile rp, rg;
  load_raw(P.w_p, kC, half * kC + ch, 0, rp);
  load_raw(P.w_g, kC, half * kC + ch, 0, rg);
  split_tile(rp, wp);
  split_tile(rg, wg);
  stage_ln<float>(P.ln_w, P.ln_b, ln);

  Part xr;
  float mraw = 0.f;
  bool mvalid = false;
  auto fetch = [&](int64_t tile) {
    const TileRS tl = tile_at(tile, ntx, n, kTS);
    const int s = tl.s0 + p;
    mvalid = s < n;
    const int ss = mvalid ? s : tl.s0;
    const int64_t pos = tl.b * nn + (P.transpose ? ss * n + tl.r : tl.r * n + ss);
    load_part(P.x + pos * kC, xr);  // columns past n repeat the tile's first one (trimul_prologue_kernel)
    if (P.mask) mraw = P.mask[pos];
  };
  bool plain;
  auto ln_tile = [&](int buf) {
    ln_planes(xr, ln, P.eps, xs[buf], plain);
    if ((t & 7) == 0) mrow[buf][p] = mvalid ? (P.mask ? mraw : 1.0f) : 0.f;
  };
  int64_t tile = blockIdx.x >> 1;
  if (tile < ntiles) fetch(tile);
  __syncthreads();  // LayerNorm affine staged
  plain = ln_plain(ln);
  if (tile < ntiles) {
    ln_tile(0);
    if (tile + stride < ntiles) fetch(tile + stride);
  }
  __syncthreads();
  for (int cur = 0; tile < ntiles; tile += stride, cur ^= 1) {
    const TileRS tl = tile_at(tile, ntx, n, kTS);
    bf16* dst = (half == 0 ? a : b) + (tl.b * kC + ch) * chplane + tl.r * pitch + tl.s0;
    auto pair = [&](int j) {
      f32x4 ap[2], ag[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        ap[h] = ag[h] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
          const Split8 x = xfrag(xs[cur], paired_row(j, h, li), ks);
          mma(ap[h], x, wp.f[ks]);
          mma(ag[h], x, wg.f[ks]);
        }
      }
      const int p0 = 32 * j + 8 * lg;  // this lane's 8 positions of channel ch
      const f32x8 m = load8(&mrow[cur][p0]);
      f32x8 v;
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = m[e] * fast_sigmoid(ag[e >> 2][e & 3]) * ap[e >> 2][e & 3];
      const Split8 s = split8(v);
#pragma unroll
      for (int u = 0; u < 3; ++u) store8(dst + u * plane + p0, s.p[u]);
    };
    pair(0);
    if (tile + stride < ntiles) {
      ln_tile(cur ^ 1);
      if (tile + 2 * stride < ntiles) fetch(tile + 2 * stride);
    }
    pair(1);
    __syncthreads();  // the next tile's rows are in LDS; this tile's buffer is free
  }
}

// ---------------------------------------------------------------------------
// Tri-mul epilogue: out = LN_out(o) p_out^T * sigmoid(LN_in(x) g_out^T)
// [+ residual], o tile-blocked ([128 channels][64 positions] per tile). Wave w
// LayerNorms channels 16w .. +15 of o, a position per lane, its statistics
// summed over the waves through LDS, and owns output channels 16w .. +15.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(512) void trimul_epilogue_split_kernel(TriMulEpilogueParams<float> P, int64_t ntiles) {
  __shared__ __attribute__((aligned(16))) Planes xg;  // LN_in(x)
  __shared__ __attribute__((aligned(16))) Planes xp;  // LN_out(o)
  __shared__ __attribute__((aligned(16))) float red[2][8][kTS];
  __shared__ __attribute__((aligned(16))) LnAffine ln_in, ln_out;

  const int64_t n = P.n, nn = n * n, pitch = P.pitch;
  const int64_t ntx = pitch / kTS;
  const int t = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int lane = t & 63;
  const int li = lane & 15;
  const int lg = lane >> 4;
  const int p = t >> 3;

  WTile wg, wp;
  RawTile rg, rp;
  load_raw(P.w_gout, kC, 16 * wave + li, 0, rg);
  load_raw(P.w_pout, kC, 16 * wave + li, 0, rp);
  split_tile(rg, wg);
  split_tile(rp, wp);
  stage_ln<float>(P.ln_in_w, P.ln_in_b, ln_in);
  stage_ln<float>(P.ln_out_w, P.ln_out_b, ln_out);

  Part xr;
  float ov[16];
  auto fetch = [&](int64_t tile) {
    const TileRS tl = tile_at(tile, ntx, n, kTS);
    const int64_t row = tl.b * n + tl.r;
    load_part(tl.s0 + p < n ? P.x + (row * n + tl.s0 + p) * kC : nullptr, xr);
    const float* src = P.o + (row * pitch + tl.s0) * kC + 16 * wave * kTS + lane;
#pragma unroll
    for (int c = 0; c < 16; ++c) ov[c] = src[c * kTS];
  };
  int64_t tile = blockIdx.x;
  if (tile < ntiles) fetch(tile);
  __syncthreads();
  const bool plain_in = ln_plain(ln_in), plain_out = ln_plain(ln_out);
  for (; tile < ntiles; tile += gridDim.x) {
    const TileRS tl = tile_at(tile, ntx, n, kTS);
    const int nvalid = (int)min<int64_t>(kTS, n - tl.s0);
    const int64_t pos0 = tl.b * nn + tl.r * n + tl.s0;
    float s = 0.f;
#pragma unroll
    for (int c = 0; c < 16; ++c) s += ov[c];
    red[0][wave][lane] = s;
    ln_planes(xr, ln_in, P.eps, xg, plain_in);
    __syncthreads();
    float mean = 0.f;
#pragma unroll
    for (int w = 0; w < 8; ++w) mean += red[0][w][lane];
    mean *= 1.0f / kC;
    float q2 = 0.f;
#pragma unroll
    for (int c = 0; c < 16; ++c) q2 += (ov[c] - mean) * (ov[c] - mean);
    red[1][wave][lane] = q2;
    __syncthreads();
    float var = 0.f;
#pragma unroll
    for (int w = 0; w < 8; ++w) var += red[1][w][lane];
    const float rstd = __builtin_amdgcn_rsqf(var * (1.0f / kC) + P.eps);
    const float shift = -mean * rstd;
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      f32x8 o;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int c = 16 * wave + 8 * q + e;
        o[e] = fmaf(fmaf(ov[8 * q + e], rstd, shift), ln_out.w[c], ln_out.b[c]);
      }
      put_planes(xp, lane, 16 * wave + 8 * q, o, plain_out);
    }
    if (tile + gridDim.x < ntiles) fetch(tile + gridDim.x);
    __syncthreads();
#pragma unroll 2
    for (int rt = 0; rt < kTS / 16; ++rt) {
      f32x4 ag = f32x4{0.f, 0.f, 0.f, 0.f}, ap = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        mma(ag, wg.f[ks], xfrag(xg, 16 * rt + li, ks));
        mma(ap, wp.f[ks], xfrag(xp, 16 * rt + li, ks));
      }
      // transposed: this lane holds channels 16 wave + 4 lg .. +3 of position pp
      const int pp = 16 * rt + li;
      if (pp < nvalid) {
        const int64_t off = (pos0 + pp) * kC + 16 * wave + 4 * lg;
        float y[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) y[q] = ap[q] * fast_sigmoid(ag[q]);
        if (P.residual) {
          float rv[4];
          load4f(P.residual + off, rv);
#pragma unroll
          for (int q = 0; q < 4; ++q) y[q] += rv[q];
        }
        if (P.out_mask) {
          const float g = P.out_mask[pos0 + pp] != 0.f ? 1.f : 0.f;
#pragma unroll
          for (int q = 0; q < 4; ++q) y[q] *= g;
        }
        store4f(P.out + off, y);
      }
    }
    __syncthreads();  // the LDS tiles are free for the next tile
  }
}

// ---------------------------------------------------------------------------
// Tri-attn prologue (layouts of triattn_prologue_kernel). Even workgroups
// produce q and k, odd ones v, the triangle bias (waves 0-3, a row tile each)
// and the mask bias.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(512) void triattn_prologue_split_kernel(TriAttnPrologueParams<float> P, int64_t ntiles) {
  __shared__ __attribute__((aligned(16))) Planes xs[2];
  __shared__ __attribute__((aligned(16))) LnAffine ln;
  constexpr int D = 32;
  constexpr int H = 4;

  const int64_t n = P.n, np = P.np, nn = n * n;
  const int64_t ntx = np / kTS;
  const int t = threadIdx.x;
  const int wave = t >> 6;
  const int lane = t & 63;
  const int li = lane & 15;
  const int lg = lane >> 4;
  const int p = t >> 3;
  const int role = blockIdx.x & 1;
  const int64_t stride = gridDim.x >> 1;

  // role 0: q and k; role 1: v and the bias weight (rows past the 4 heads are
  // computed on head 0's and dropped)
  WTile w1, w2;
  RawTile r1, r2;
  load_raw(role == 0 ? P.w_q : P.w_v, kC, 16 * wave + li, 0, r1);
  load_raw(role == 0 ? P.w_k : P.w_bias, kC, role == 0 ? 16 * wave + li : (li < H ? li : 0), 0, r2);
  split_tile(r1, w1);
  split_tile(r2, w2);
  stage_ln<float>(P.ln_w, P.ln_b, ln);

  Part xr;
  float mraw = 0.f;
  bool mvalid = false;
  auto fetch = [&](int64_t tile) {
    const TileRS tl = tile_at(tile, ntx, n, kTS);
    const int s = tl.s0 + p;
    mvalid = s < n;
    const int ss = mvalid ? s : tl.s0;
    const int64_t pos = tl.b * nn + (P.transpose ? ss * n + tl.r : tl.r * n + ss);
    load_part(mvalid ? P.x + pos * kC : nullptr, xr);
    if (P.mask) mraw = P.mask[pos];
  };
  bool plain;
  auto ln_tile = [&](int64_t tile, int buf) {
    ln_planes(xr, ln, P.eps, xs[buf], plain);
    if (role == 1 && (t & 7) == 0) {
      const TileRS tl = tile_at(tile, ntx, n, kTS);
      P.mb[(tl.b * n + tl.r) * np + tl.s0 + p] =
          mvalid ? P.inf * ((P.mask ? mraw : 1.0f) - 1.0f) * kLog2e : -INFINITY;
    }
  };
  int64_t tile = blockIdx.x >> 1;
  if (tile < ntiles) fetch(tile);
  __syncthreads();
  plain = ln_plain(ln);
  if (tile < ntiles) {
    ln_tile(tile, 0);
    if (tile + stride < ntiles) fetch(tile + stride);
  }
  __syncthreads();
  for (int cur = 0; tile < ntiles; tile += stride, cur ^= 1) {
    const TileRS tl = tile_at(tile, ntx, n, kTS);
    const int nreal = (int)min<int64_t>(kTS, n - tl.s0);
    auto next_ln = [&] {
      if (tile + stride < ntiles) {
        ln_tile(tile + stride, cur ^ 1);
        if (tile + 2 * stride < ntiles) fetch(tile + 2 * stride);
      }
    };
    if (role == 0) {
      // transposed: lane li of row tile rt holds head dims (16 wave + 4 lg) % 32 .. +3
      const int64_t head_off = (((int64_t)tl.b * n + tl.r) * H + (wave >> 1)) * np * D;
      const int d0 = 16 * (wave & 1) + 4 * lg;
      auto rows = [&](int rt) {
        f32x4 aq = f32x4{0.f, 0.f, 0.f, 0.f}, ak = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
          const Split8 x = xfrag(xs[cur], 16 * rt + li, ks);
          mma(aq, w1.f[ks], x);
          mma(ak, w2.f[ks], x);
        }
        const int pp = 16 * rt + li;
        const bool real = pp < nreal;
        float vq[4], vk[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          vq[q] = real ? aq[q] * P.q_scale : 0.f;
          vk[q] = real ? ak[q] : 0.f;
        }
        const int64_t off = head_off + (int64_t)(tl.s0 + pp) * D + d0;
        store4f(P.q + off, vq);
        store4f(P.k + off, vk);
      };
      rows(0);
      rows(1);
      next_ln();
      rows(2);
      rows(3);
    } else {
      // v, channel-major: lane group lg holds positions 32j + 8lg .. +7 of its channel
      float* vdst = P.vt + (((int64_t)tl.b * n + tl.r) * kC + 16 * wave + li) * np + tl.s0;
      auto pair = [&](int j) {
        f32x4 av[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          av[h] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int ks = 0; ks < 4; ++ks) mma(av[h], xfrag(xs[cur], paired_row(j, h, li), ks), w1.f[ks]);
        }
        const int p0 = 32 * j + 8 * lg;
        f32x8 v;
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = p0 + e < nreal ? av[e >> 2][e & 3] : 0.f;
        store8(vdst + p0, v);
      };
      pair(0);
      next_ln();
      pair(1);
      if (wave < 4) {
        f32x4 ab = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) mma(ab, xfrag(xs[cur], 16 * wave + li, ks), w2.f[ks]);
        const int p0 = 16 * wave + 4 * lg;  // this lane's 4 positions of head li
        if (li < H) {
          float v[4], zero[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = p0 + e < nreal ? ab[e] * kLog2e : 0.f;
          float* brow = P.bias + (((int64_t)tl.b * H + li) * np + tl.r) * np + tl.s0 + p0;
          store4f(brow, v);
          // the bias rows of the padded queries n .. np-1 are zeros
          for (int64_t rz = n + tl.r; rz < np; rz += n) store4f(brow + (rz - tl.r) * np, zero);
        }
      }
    }
    __syncthreads();  // the next tile's rows are in LDS; this tile's buffer is free
  }
}

// ---------------------------------------------------------------------------
// Tri-attn epilogue (gated): out[orig] = (o * sigmoid(LN(x[orig]) w_g^T)) w_o^T
// [+ residual[orig]], o head-major [B][N rows][4][N][32]
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(512) void triattn_epilogue_split_kernel(TriAttnEpilogueParams<float> P, int64_t ntiles) {
  __shared__ __attribute__((aligned(16))) Planes xs;  // LN(x)
  __shared__ __attribute__((aligned(16))) Planes xo;  // gated o
  __shared__ __attribute__((aligned(16))) LnAffine ln;

  const int64_t n = P.n, nn = n * n;
  const int64_t ntx = (n + kTS - 1) / kTS;
  const int t = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int lane = t & 63;
  const int li = lane & 15;
  const int lg = lane >> 4;
  const int p = t >> 3;

  WTile wg, wo;
  RawTile rg, ro;
  load_raw(P.w_g, kC, 16 * wave + li, 0, rg);
  load_raw(P.w_o, kC, 16 * wave + li, 0, ro);
  split_tile(rg, wg);
  split_tile(ro, wo);
  stage_ln<float>(P.ln_w, P.ln_b, ln);

  auto orig_of = [&](const TileRS& tl, int pp) -> int64_t {
    const int64_t s = tl.s0 + pp;
    return (int64_t)tl.b * nn + (P.transpose ? s * n + tl.r : (int64_t)tl.r * n + s);
  };
  Part xr;
  f32x4 ov[kTS / 16];  // o of this lane's positions 16rt + li, channels 16 wave + 4 lg .. +3
  auto fetch = [&](int64_t tile) {
    const TileRS tl = tile_at(tile, ntx, n, kTS);
    const int nvalid = (int)min<int64_t>(kTS, n - tl.s0);
    load_part(p < nvalid ? P.x + orig_of(tl, p) * kC : nullptr, xr);
    const float* src = P.o + ((((int64_t)tl.b * n + tl.r) * 4 + (wave >> 1)) * n + tl.s0) * 32 + 16 * (wave & 1) + 4 * lg;
#pragma unroll
    for (int rt = 0; rt < kTS / 16; ++rt) {
      const int pp = 16 * rt + li;
      ov[rt] = pp < nvalid ? *reinterpret_cast<const f32x4*>(src + pp * 32) : f32x4{0.f, 0.f, 0.f, 0.f};
    }
  };
  int64_t tile = blockIdx.x;
  if (tile < ntiles) fetch(tile);
  __syncthreads();
  const bool plain = ln_plain(ln);
  for (; tile < ntiles; tile += gridDim.x) {
    const TileRS tl = tile_at(tile, ntx, n, kTS);
    const int nvalid = (int)min<int64_t>(kTS, n - tl.s0);
    ln_planes(xr, ln, P.eps, xs, plain);
    __syncthreads();
#pragma unroll 2
    for (int rt = 0; rt < kTS / 16; ++rt) {
      f32x4 ag = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) mma(ag, wg.f[ks], xfrag(xs, 16 * rt + li, ks));
      float v[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) v[q] = ov[rt][q] * fast_sigmoid(ag[q]);
      put_planes4(xo, 16 * rt + li, 16 * wave + 4 * lg, v);
    }
    if (tile + gridDim.x < ntiles) fetch(tile + gridDim.x);
    __syncthreads();
#pragma unroll 2
    for (int rt = 0; rt < kTS / 16; ++rt) {
      f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) mma(acc, wo.f[ks], xfrag(xo, 16 * rt + li, ks));
      const int pp = 16 * rt + li;
      if (pp < nvalid) {
        const int64_t pos = orig_of(tl, pp), off = pos * kC + 16 * wave + 4 * lg;
        float y[4] = {acc[0], acc[1], acc[2], acc[3]};
        if (P.residual) {
          float rv[4];
          load4f(P.residual + off, rv);
#pragma unroll
          for (int q = 0; q < 4; ++q) y[q] += rv[q];
        }
        if (P.out_mask) {
          const float g = P.out_mask[pos] != 0.f ? 1.f : 0.f;
#pragma unroll
          for (int q = 0; q < 4; ++q) y[q] *= g;
        }
        store4f(P.out + off, y);
      }
    }
    // xs is rewritten only after the next tile's loads, behind this barrier;
    // xo after the one that follows
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// Pair transition (transition128_body): per 128-wide hidden chunk wave w forms
// hidden columns 16w .. +15 of a and b, writes silu(a) * b as planes, and
// accumulates the chunk into its output channels. The weights (1.2 MB as
// planes) do not fit the registers: they are loaded and split per chunk.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(512) void transition_split_kernel(TransitionParams<float> P) {
  __shared__ __attribute__((aligned(16))) Planes xs;  // LN(x)
  __shared__ __attribute__((aligned(16))) Planes hs;  // silu(a) * b, one hidden chunk
  __shared__ __attribute__((aligned(16))) LnAffine ln;
  __shared__ __attribute__((aligned(16))) LnAffine pb_ln;

  const int64_t m0 = (int64_t)blockIdx.x * kTS;
  const int nvalid = (int)min<int64_t>(kTS, P.rows - m0);
  const int t = threadIdx.x;
  const int wave = t >> 6;
  const int lane = t & 63;
  const int li = lane & 15;
  const int lg = lane >> 4;
  const int p = t >> 3;
  const int col = 16 * wave;
  {
    Part xr;
    load_part(p < nvalid ? P.x + (m0 + p) * kC : nullptr, xr);
    stage_ln<float>(P.ln_w, P.ln_b, ln);
    if (P.pb_out) stage_ln<float>(P.pb_ln_w, P.pb_ln_b, pb_ln);
    __syncthreads();
    ln_planes(xr, ln, P.eps, xs, ln_plain(ln));
  }
  __syncthreads();
  f32x4 out[kTS / 16];
#pragma unroll
  for (int rt = 0; rt < kTS / 16; ++rt) out[rt] = f32x4{0.f, 0.f, 0.f, 0.f};
  // a 16-channel column tile of a weight as loaded, split a fragment at a time
  // right before its products: splitting and products of the two waves of a
  // SIMD then interleave, and the next tile's loads are in flight meanwhile
  RawTile ra, rb, ro;
  load_raw(P.w_a, kC, col + li, 0, ra);
  load_raw(P.w_b, kC, col + li, 0, rb);
#pragma unroll 1
  for (int chk = 0; chk < 4; ++chk) {
    load_raw(P.w_o, 4 * kC, col + li, chk * kC, ro);
    const bool plain_a = split_plain(ra.f), plain_b = split_plain(rb.f);
    f32x4 av[kTS / 16], bv[kTS / 16];
#pragma unroll
    for (int rt = 0; rt < kTS / 16; ++rt) av[rt] = bv[rt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      const Split8 wa = split8(ra.f[ks], plain_a), wb = split8(rb.f[ks], plain_b);
#pragma unroll
      for (int rt = 0; rt < kTS / 16; ++rt) {
        const Split8 x = xfrag(xs, 16 * rt + li, ks);
        mma(av[rt], wa, x);
        mma(bv[rt], wb, x);
      }
    }
    if (chk < 3) {
      load_raw(P.w_a, kC, (chk + 1) * kC + col + li, 0, ra);
      load_raw(P.w_b, kC, (chk + 1) * kC + col + li, 0, rb);
    }
#pragma unroll
    for (int rt = 0; rt < kTS / 16; ++rt) {
      float h[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) h[q] = av[rt][q] * fast_sigmoid(av[rt][q]) * bv[rt][q];
      put_planes4(hs, 16 * rt + li, col + 4 * lg, h);
    }
    __syncthreads();
    const bool plain_o = split_plain(ro.f);
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      const Split8 wo = split8(ro.f[ks], plain_o);
#pragma unroll
      for (int rt = 0; rt < kTS / 16; ++rt) mma(out[rt], wo, xfrag(hs, 16 * rt + li, ks));
    }
    __syncthreads();  // hs is rewritten by the next chunk
  }

  // the output rows, kept in LDS (over hs, free now) for the pair bias
  float(*ys)[kC + 4] = reinterpret_cast<float(*)[kC + 4]>(&hs[0][0][0]);
  static_assert(sizeof(float) * kTS * (kC + 4) <= sizeof(Planes), "the output tile fits the hidden planes");
#pragma unroll
  for (int rt = 0; rt < kTS / 16; ++rt) {
    const int row = 16 * rt + li;
    if (row < nvalid) {
      const int64_t off = (m0 + row) * kC + col + 4 * lg;
      float y[4];
      const float msk = P.row_mask ? P.row_mask[m0 + row] : 1.0f;
#pragma unroll
      for (int q = 0; q < 4; ++q) y[q] = out[rt][q] * msk;
      if (P.residual) {
        float rv[4];
        load4f(P.residual + off, rv);
#pragma unroll
        for (int q = 0; q < 4; ++q) y[q] += rv[q];
      }
      if (P.out_mask) {
        const float g = P.out_mask[m0 + row] != 0.f ? 1.f : 0.f;
#pragma unroll
        for (int q = 0; q < 4; ++q) y[q] *= g;
      }
      store4f(P.out + off, y);
      if (P.pb_out) store4f(&ys[row][col + 4 * lg], y);
    }
  }
  if (!P.pb_out) return;
  // the single attention's pair bias LN_pb(out row) w^T, as pair_bias_epilogue
  WTile wz;
  RawTile rz;
  load_raw(P.pb_w, kC, min(li, P.pb_heads - 1), 0, rz);
  split_tile(rz, wz);
  __syncthreads();
  Part yr;
  load_part(&ys[p][0], yr);
  ln_planes(yr, pb_ln, P.pb_eps, xs, ln_plain(pb_ln));
  __syncthreads();
  if (wave >= kTS / 16) return;
  f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) mma(acc, xfrag(xs, 16 * wave + li, ks), wz.f[ks]);
  const int pos0 = 16 * wave + 4 * lg;  // this lane's 4 rows of head li
  if (li >= P.pb_heads || pos0 >= nvalid) return;
  const int64_t n = P.pb_n, nn = n * n, np = P.pb_np;
  float v[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) v[q] = acc[q] * kLog2e;
  const int64_t m = m0 + pos0;
  int64_t b = m / nn, rem = m - b * nn, r = rem / n, c = rem - r * n;
  if ((n & 3) == 0) {
    // nvalid is a multiple of 16 and the 4 rows share (b, r), c a multiple of 4
    store4f(P.pb_out + ((b * P.pb_heads + li) * np + r) * np + c, v);
    return;
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    if (pos0 + q >= nvalid) break;
    P.pb_out[((b * P.pb_heads + li) * np + r) * np + c] = v[q];
    if (++c == n) {
      c = 0;
      if (++r == n) {
        r = 0;
        ++b;
      }
    }
  }
}

// ---------------------------------------------------------------------------
// host-side launchers
// ---------------------------------------------------------------------------
namespace {
// a persistent grid of two kinds of workgroups over the same tiles
unsigned two_kinds_grid(const void* k, int64_t ntiles) {
  return (persistent_grid(k, 512, 2 * ntiles) + 1) / 2 * 2;
}
}  // namespace

void launch_trimul_prologue_split(const TriMulPrologueParams<float>& p, bf16* a, bf16* b, int64_t plane, int64_t batch,
                                  hipStream_t st) {
  const int64_t ntiles = p.pitch / kTS * p.n * batch;
  hipLaunchKernelGGL(trimul_prologue_split_kernel,
                     dim3(two_kinds_grid(reinterpret_cast<const void*>(trimul_prologue_split_kernel), ntiles)),
                     dim3(512), 0, st, p, a, b, plane, ntiles);
}
void launch_trimul_epilogue_split(const TriMulEpilogueParams<float>& p, int64_t batch, hipStream_t st) {
  const int64_t ntiles = p.pitch / kTS * p.n * batch;
  hipLaunchKernelGGL(trimul_epilogue_split_kernel,
                     dim3(persistent_grid(reinterpret_cast<const void*>(trimul_epilogue_split_kernel), 512, ntiles)),
                     dim3(512), 0, st, p, ntiles);
}
void launch_triattn_prologue_split(const TriAttnPrologueParams<float>& p, int64_t batch, hipStream_t st) {
  const int64_t ntiles = p.np / kTS * p.n * batch;
  hipLaunchKernelGGL(triattn_prologue_split_kernel,
                     dim3(two_kinds_grid(reinterpret_cast<const void*>(triattn_prologue_split_kernel), ntiles)),
                     dim3(512), 0, st, p, ntiles);
}
void launch_triattn_epilogue_split(const TriAttnEpilogueParams<float>& p, int64_t batch, hipStream_t st) {
  const int64_t ntiles = (p.n + kTS - 1) / kTS * p.n * batch;
  hipLaunchKernelGGL(triattn_epilogue_split_kernel,
                     dim3(persistent_grid(reinterpret_cast<const void*>(triattn_epilogue_split_kernel), 512, ntiles)),
                     dim3(512), 0, st, p, ntiles);
}
void launch_transition_split(const TransitionParams<float>& p, hipStream_t st) {
  hipLaunchKernelGGL(transition_split_kernel, dim3((unsigned)((p.rows + kTS - 1) / kTS)), dim3(512), 0, st, p);
}

}  // namespace fjx
