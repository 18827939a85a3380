// Single-track helpers for the attention with pair bias of a Pairformer block
// (Boltz-2 attention_pair_bias_forward): row LayerNorm, head split into the
// padded flash layout with the key mask bias, and the pair-bias projection
// LN(z) W_z^T.
#include "fjx_common.hpp"
#include "fjx_kernels.hpp"
#include "fjx_tile.hpp"

namespace fjx {

namespace {

// one wave per row, C <= 1024, C % 64 == 0 or handled by the stride loop
template <typename T>
__global__ __launch_bounds__(256) void layernorm_rows_kernel(const T* __restrict__ x, const T* __restrict__ w,
                                                             const T* __restrict__ b, T* __restrict__ y,
                                                             int64_t rows, int c, float eps) {
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (row >= rows) return;
  const T* xr = x + row * c;
  float v[16];
  float s = 0.f;
#pragma unroll
  for (int u = 0; u < 16; ++u) {
    const int ch = lane + 64 * u;
    v[u] = ch < c ? to_f32(xr[ch]) : 0.f;
    s += v[u];
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) s += shfl_xor(s, o);
  const float mean = s / c;
  float q2 = 0.f;
#pragma unroll
  for (int u = 0; u < 16; ++u) {
    const int ch = lane + 64 * u;
    if (ch < c) q2 += (v[u] - mean) * (v[u] - mean);
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) q2 += shfl_xor(q2, o);
  const float rstd = __builtin_amdgcn_rsqf(q2 / c + eps);
#pragma unroll
  for (int u = 0; u < 16; ++u) {
    const int ch = lane + 64 * u;
    if (ch < c) y[row * c + ch] = from_f32<T>((v[u] - mean) * rstd * to_f32(w[ch]) + to_f32(b[ch]));
  }
}

// the same for c <= 512 channels, a multiple of 8 (ln_row8)
template <typename T>
__global__ __launch_bounds__(256) void layernorm_rows8_kernel(const T* __restrict__ x, const T* __restrict__ w,
                                                              const T* __restrict__ b, T* __restrict__ y,
                                                              int64_t rows, int c, float eps) {
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;
  ln_row8<T>(x + row * c, w, b, y + row * c, c, eps, threadIdx.x & 63);
}

// qkv rows [B*N][ld] holding q | k | v (each heads*dh wide) ->
//   q, k: [B][H][Np][32] (q times q_mul), vt: [B][H*32][Np]; zero padding in d and keys
// and the key mask mb[b][k] = log2(e) * (1 - mask[b,k]) * (-inf_const), -inf for padded keys
template <typename T>
__global__ void split_heads_kernel(const T* __restrict__ qkv, int64_t ld, int64_t batch, int64_t n, int64_t np,
                                   int heads, int dh, float q_mul, T* __restrict__ q, T* __restrict__ k,
                                   T* __restrict__ vt, const T* __restrict__ mask, float* __restrict__ mb, float inf) {
  const int64_t total = batch * heads * np * 32;
  const int64_t hd = (int64_t)heads * dh;
  for (int64_t idx = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; idx < total;
       idx += (int64_t)gridDim.x * blockDim.x) {
    const int d = idx % 32;
    const int64_t s = (idx / 32) % np;
    const int64_t h = (idx / (32 * np)) % heads;
    const int64_t b = idx / (32 * np * heads);
    float qv = 0.f, kv = 0.f, vv = 0.f;
    if (s < n && d < dh) {
      const T* r = qkv + (b * n + s) * ld + h * dh + d;
      qv = to_f32(r[0]) * q_mul;
      kv = to_f32(r[hd]);
      vv = to_f32(r[2 * hd]);
    }
    q[idx] = from_f32<T>(qv);
    k[idx] = from_f32<T>(kv);
    vt[((b * heads + h) * 32 + d) * np + s] = from_f32<T>(vv);
    if (idx < batch * np) {
      const int64_t mk = idx % np, bm = idx / np;
      mb[idx] = mk < n ? (mask ? (1.0f - to_f32(mask[bm * n + mk])) * (-inf) * kLog2e : 0.f) : -INFINITY;
    }
  }
}

// bias[b][h][q][k] = log2(e) * LN(z[b,q,k,:]) . w[h,:] over the padded
// [np, np] grid, zeros outside [n, n] (the attention never reads
// uninitialised memory next to a -inf key mask).
//
// Waves work alone, each walking 16-key tiles of a query row: the 4 lanes of a
// key (16 apart) load its 128 channels as the MFMA fragments they are needed
// as, LayerNorm them in registers and multiply by the [heads][128] weight, 16
// heads per MFMA column tile; a lane stores 4 consecutive keys of one head.
// No tile goes through LDS and no wave waits for another; the next tile's rows
// are in flight meanwhile. Bound by HBM: 257 MB of z read and 67 MB of fp32
// bias written at n = 1003 take 116 us with the tile LayerNormed into LDS by
// the workgroup (two barriers a tile), 75 us so
// (three waves per SIMD where z is bf16; two, 79 us).
// z may be narrower than the bias (TZ = bf16, T = float: the fp32 single
// track of Boltz-2 over a bf16 pair tensor); the LayerNorm runs in fp32 and
// its output is rounded to T, so the projection then runs at T's precision.
template <typename TZ, typename T>
__global__ __launch_bounds__(256, (sizeof(TZ) == 2 ? 3 : 2)) void pair_bias_kernel(const TZ* __restrict__ z, const T* __restrict__ ln_w,
                                                        const T* __restrict__ ln_b, const T* __restrict__ w,
                                                        T* __restrict__ bias, int64_t n, int64_t np, int heads,
                                                        float eps, int64_t ntiles) {
  using namespace tile;
  __shared__ __attribute__((aligned(16))) LnAffine ln;

  const int lane = threadIdx.x & 63;
  const int li = lane & 15;
  const int lg = lane >> 4;
  const int nht = (heads + 15) / 16;
  stage_ln<T>(ln_w, ln_b, ln);

  auto load_heads = [&](int ht, typename Frag<T>::type (&wf)[4]) {
    const float zero[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    const int h = 16 * ht + li;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) wf[ks] = h < heads ? load8(w + (int64_t)h * kC + 32 * ks + 8 * lg) : pack8<T>(zero);
  };
  typename Frag<T>::type w0[4];
  load_heads(0, w0);

  // tile -> (batch, query row, key tile), advanced by fixed carries
  const int64_t kt_row = np / 16;
  const int64_t nw = (int64_t)gridDim.x * 4;
  int64_t tile = (int64_t)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  struct At {
    int64_t b, r, k;
  };
  const At step = {nw / kt_row / np, nw / kt_row % np, nw % kt_row};
  At cur = {tile / kt_row / np, tile / kt_row % np, tile % kt_row};
  auto next = [&](const At& a) {
    At o = {a.b + step.b, a.r + step.r, a.k + step.k};
    if (o.k >= kt_row) {
      o.k -= kt_row;
      ++o.r;
    }
    if (o.r >= np) {
      o.r -= np;
      ++o.b;
    }
    return o;
  };
  RowPart<TZ> xr;
  auto fetch = [&](const At& a) {
    const int64_t kk = 16 * a.k + li;
    const bool valid = a.r < n && kk < n;
    load_row_part<TZ, true>(valid ? z + ((a.b * n + a.r) * n + kk) * kC : nullptr, xr);
  };
  if (tile < ntiles) fetch(cur);
  __syncthreads();  // LayerNorm affine staged
  for (; tile < ntiles; tile += nw) {
    const bool some = cur.r < n && 16 * cur.k < n;  // wave-uniform
    typename Frag<T>::type xf[4];
    ln_frag<TZ, T>(xr, ln, eps, xf);
    const At nxt = next(cur);
    if (tile + nw < ntiles) fetch(nxt);
    const int64_t p0 = 16 * cur.k + 4 * lg;  // this lane's 4 keys
    T* dst = bias + ((cur.b * heads + li) * np + cur.r) * np + p0;
    for (int ht = 0; ht < nht; ++ht) {
      f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
      if (some) {
        typename Frag<T>::type wf[4];
        if (ht == 0) {
#pragma unroll
          for (int ks = 0; ks < 4; ++ks) wf[ks] = w0[ks];
        } else {
          load_heads(ht, wf);
        }
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) mma(acc, xf[ks], wf[ks]);
      }
      if (16 * ht + li < heads) {
        float v[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) v[q] = cur.r < n && p0 + q < n ? acc[q] * kLog2e : 0.f;
        store4f(dst + 16 * ht * np * np, v);
      }
    }
    cur = nxt;
  }
}

// zeros of a prepared pair bias outside the [n, n] block of each padded
// [np, np] plane: rows r < n, columns n .. np-1, then rows n .. np-1 whole
// (the transition's fused epilogue writes only the real positions)
template <typename T>
__global__ void pair_bias_border_kernel(T* __restrict__ bias, int64_t planes, int64_t n, int64_t np) {
  const int64_t w = np - n;
  const int64_t per = n * w + w * np;
  const int64_t total = planes * per;
  for (int64_t idx = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; idx < total;
       idx += (int64_t)gridDim.x * blockDim.x) {
    const int64_t plane = idx / per;
    int64_t j = idx - plane * per;
    int64_t r, c;
    if (j < n * w) {
      r = j / w;
      c = n + (j - r * w);
    } else {
      j -= n * w;
      r = n + j / np;
      c = j - (r - n) * np;
    }
    bias[(plane * np + r) * np + c] = from_f32<T>(0.f);
  }
}

// an additive attention bias given by the caller (Protenix's extra_attn_bias),
// broadcast over batch (sb = 0) and heads (sh = 0), added in fp32 to the
// projected bias: bias = src + log2(e) * extra over the real [n, n] block.
// src is a prepared bias (read-only) or bias itself.
template <typename T>
__global__ void add_extra_bias_kernel(const T* __restrict__ src, T* __restrict__ bias, const T* __restrict__ extra,
                                      int64_t sb, int64_t sh, int64_t batch, int heads, int64_t n, int64_t np) {
  const int64_t total = batch * heads * n * n;
  for (int64_t idx = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; idx < total;
       idx += (int64_t)gridDim.x * blockDim.x) {
    const int64_t k = idx % n;
    const int64_t q = (idx / n) % n;
    const int64_t h = (idx / (n * n)) % heads;
    const int64_t b = idx / (n * n * heads);
    const int64_t at = ((b * heads + h) * np + q) * np + k;
    const float e = to_f32(extra[b * sb + h * sh + q * n + k]);
    bias[at] = from_f32<T>(to_f32(src[at]) + e * kLog2e);
  }
}

dim3 grid_stride(int64_t total) {
  int64_t blocks = (total + 255) / 256;
  if (blocks > 65536) blocks = 65536;
  if (blocks < 1) blocks = 1;
  return dim3((unsigned)blocks);
}

}  // namespace

template <typename T>
void launch_layernorm_rows(const T* x, const T* w, const T* b, T* y, int64_t rows, int c, float eps, hipStream_t st) {
  auto al16 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
  const bool vec = c % 8 == 0 && c <= 512 && al16(x) && al16(w) && al16(b) && al16(y);
  for_pieces((rows + 3) / 4, [&](int64_t first, unsigned count) {
    hipLaunchKernelGGL(vec ? layernorm_rows8_kernel<T> : layernorm_rows_kernel<T>, dim3(count), dim3(256), 0, st,
                       x + 4 * first * c, w, b, y + 4 * first * c, rows - 4 * first, c, eps);
  });
}
template <typename T>
void launch_split_heads(const T* qkv, int64_t ld, int64_t batch, int64_t n, int64_t np, int heads, int dh,
                        float q_mul, T* q, T* k, T* vt, const T* mask, float* mb, float inf, hipStream_t st) {
  hipLaunchKernelGGL(split_heads_kernel<T>, grid_stride(batch * heads * np * 32), dim3(256), 0, st, qkv, ld, batch, n,
                     np, heads, dh, q_mul, q, k, vt, mask, mb, inf);
}
template <typename TZ, typename T>
void launch_pair_bias(const TZ* z, const T* ln_w, const T* ln_b, const T* w, T* bias, int64_t batch, int64_t n,
                      int64_t np, int heads, float eps, hipStream_t st) {
  const int64_t ntiles = np / 16 * np * batch;
  const unsigned grid =
      tile::persistent_grid(reinterpret_cast<const void*>(&pair_bias_kernel<TZ, T>), 256, (ntiles + 3) / 4);
  hipLaunchKernelGGL((pair_bias_kernel<TZ, T>), dim3(grid), dim3(256), 0, st, z, ln_w, ln_b, w, bias, n, np, heads,
                     eps, ntiles);
}
template <typename T>
void launch_add_extra_bias(const T* src, T* bias, const T* extra, int64_t sb, int64_t sh, int64_t batch, int heads,
                           int64_t n, int64_t np, hipStream_t st) {
  hipLaunchKernelGGL(add_extra_bias_kernel<T>, grid_stride(batch * heads * n * n), dim3(256), 0, st, src ? src : bias,
                     bias, extra, sb, sh, batch, heads, n, np);
}
template <typename T>
void launch_pair_bias_border(T* bias, int64_t planes, int64_t n, int64_t np, hipStream_t st) {
  if (np == n) return;
  hipLaunchKernelGGL(pair_bias_border_kernel<T>, grid_stride(planes * (n * (np - n) + (np - n) * np)), dim3(256), 0,
                     st, bias, planes, n, np);
}
#define FJX_INST(T)                                                                                              \
  template void launch_layernorm_rows<T>(const T*, const T*, const T*, T*, int64_t, int, float, hipStream_t);   \
  template void launch_split_heads<T>(const T*, int64_t, int64_t, int64_t, int64_t, int, int, float, T*, T*, T*, \
                                      const T*, float*, float, hipStream_t);                                     \
  template void launch_pair_bias<T, T>(const T*, const T*, const T*, const T*, T*, int64_t, int64_t, int64_t, int, \
                                       float, hipStream_t);                                                      \
  template void launch_add_extra_bias<T>(const T*, T*, const T*, int64_t, int64_t, int64_t, int, int64_t, int64_t,  \
                                         hipStream_t);                                                           \
  template void launch_pair_bias_border<T>(T*, int64_t, int64_t, int64_t, hipStream_t);
FJX_INST(bf16)
FJX_INST(float)
#undef FJX_INST
template void launch_pair_bias<bf16, float>(const bf16*, const float*, const float*, const float*, float*, int64_t,
                                            int64_t, int64_t, int, float, hipStream_t);
template void launch_pair_bias<float, bf16>(const float*, const bf16*, const bf16*, const bf16*, bf16*, int64_t,
                                            int64_t, int64_t, int, float, hipStream_t);

}  // namespace fjx
