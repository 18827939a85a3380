// Layout and elementwise kernels of the general-width paths: the triangle
// ops and the transition for channel widths the fused kernels do not take
// (the fused ones are built for c_z = c_h = 128, H*D = 128). The C ABI layer
// composes these with the row LayerNorm, the generic GEMM, the contraction
// and the flash attention core into the same computation:
//
//   tri-mul:  xn = LN_in(x) -> G = sigmoid(xn g_in^T), P = (xn p_in^T) * G
//             -> a, b = mask * P, channel-major in the virtual grid
//             -> o[c] = a[c] b[c]^T -> LN_out(o) -> (.. p_out^T) * sigmoid(xn g_out^T)
//   tri-attn: xn = LN(x) in the virtual grid -> q|k|v|g and the bias by GEMM
//             -> padded head layouts -> flash core -> o * sigmoid(g) -> o w_o^T
//   transition: LN -> silu(xn a^T) * (xn b^T) -> (..) o^T [* row mask]
//
// Positions of the virtual grid are v = r*n + s; for the incoming direction
// and the ending node they read the original grid at s*n + r.
#include "fjx_common.hpp"
#include "fjx_kernels.hpp"

namespace fjx {

namespace {

__device__ __forceinline__ int64_t orig_pos(int64_t v, int64_t n, int t) {
  if (!t) return v;
  const int64_t r = v / n;
  return (v - r * n) * n + r;
}

dim3 stride_grid(int64_t total) {
  int64_t blocks = (total + 255) / 256;
  if (blocks > 65536) blocks = 65536;
  if (blocks < 1) blocks = 1;
  return dim3((unsigned)blocks);
}

// one wave per position: y[b][v][:] = LN(x[b][orig(v)][:]), c <= 1024
template <typename T>
__global__ __launch_bounds__(256) void ln_grid_kernel(const T* __restrict__ x, const T* __restrict__ w,
                                                      const T* __restrict__ b, T* __restrict__ y, int64_t rows,
                                                      int64_t n, int c, float eps, int t, int64_t first) {
  const int64_t row = (first + blockIdx.x) * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (row >= rows) return;
  const int64_t nn = n * n;
  const int64_t bb = row / nn;
  const T* xr = x + (bb * nn + orig_pos(row - bb * nn, n, t)) * c;
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

// For products the paired GEMM does not write as planes itself.
// a and b as planes (launch_to_planes), through LDS tiles of 64 columns of one
// grid row x 64 channels, so that both sides move whole rows: 16-byte accesses
// where the widths (vs) and the pitch (vd) allow, elements otherwise
template <typename T>
__global__ __launch_bounds__(256) void to_planes_kernel(const T* __restrict__ src, int64_t ld, int C,
                                                        const T* __restrict__ mask, T* __restrict__ A,
                                                        T* __restrict__ B, int64_t n, int64_t pitch, int t, bool vs,
                                                        bool vd, int64_t first) {
  __shared__ float tile[64][65];
  const int ctiles = (2 * C + 63) / 64;
  const int64_t stiles = (pitch + 63) / 64;
  int64_t id = first + blockIdx.x;
  const int cb = (int)(id % ctiles) * 64;
  id /= ctiles;
  const int64_t s0 = id % stiles * 64;
  id /= stiles;
  const int64_t r = id % n, bb = id / n;
  const int tx = threadIdx.x;
  if (vs) {
    for (int e = tx; e < 512; e += 256) {
      const int ps = e >> 3, c = cb + 8 * (e & 7);
      const int64_t s = s0 + ps;
      float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
      if (s < n && c < 2 * C) {
        const int64_t o = bb * n * n + (t ? s * n + r : r * n + s);
        to_f32x8(load8(src + o * ld + c), v);
        const float m = mask ? to_f32(mask[o]) : 1.f;
#pragma unroll
        for (int k = 0; k < 8; ++k) v[k] *= m;
      }
#pragma unroll
      for (int k = 0; k < 8; ++k) tile[ps][8 * (e & 7) + k] = v[k];
    }
  } else {
    for (int e = tx; e < 4096; e += 256) {
      const int ps = e >> 6, c = cb + (e & 63);
      const int64_t s = s0 + ps;
      float v = 0.f;
      if (s < n && c < 2 * C) {
        const int64_t o = bb * n * n + (t ? s * n + r : r * n + s);
        v = to_f32(src[o * ld + c]);
        if (mask) v *= to_f32(mask[o]);
      }
      tile[ps][e & 63] = v;
    }
  }
  __syncthreads();
  auto row_of = [&](int c) { return (c < C ? A + (bb * C + c) * n * pitch : B + (bb * C + c - C) * n * pitch) + r * pitch; };
  if (vd) {
    for (int e = tx; e < 512; e += 256) {
      const int pc = e >> 3, vv = 8 * (e & 7);
      if (s0 + vv >= pitch || cb + pc >= 2 * C) continue;
      float o8[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) o8[k] = tile[vv + k][pc];
      store8(row_of(cb + pc) + s0 + vv, pack8<T>(o8));
    }
  } else {
    for (int e = tx; e < 4096; e += 256) {
      const int pc = e >> 6, ps = e & 63;
      if (s0 + ps < pitch && cb + pc < 2 * C) row_of(cb + pc)[s0 + ps] = from_f32<T>(tile[ps][pc]);
    }
  }
}

// positions per tile of planes_layernorm_kernel: one 128-byte piece of a plane
template <typename T>
constexpr int kLnCols = 128 / (int)sizeof(T);

// position-major rows from planes, with the LayerNorm over the channels
// (w null: none; channels blockIdx.y * 512 .. of more than 512; `written` of a
// row's columns hold values, n at least). A workgroup
// takes kLnCols columns of one grid row: the planes' 128-byte pieces go to LDS
// as they are, chunk q (16 bytes) of channel c in slot q ^ (c / 8) % 8, so that
// 8 lanes reading the same position of channels 8 apart hit different banks; a
// position's channels are then in the registers of 8 lanes, 8 consecutive ones
// each at a time, and leave as 16-byte stores.
// Bound by latency, a workgroup's loads, LDS pass and reductions being one chain
// (three workgroups a CU at 384 channels): 33 us at n = 245 and 384 channels, 94
// MB, where a transpose (33) and a LayerNorm (19) took 52; four chunks a thread
// in flight measured 31.
template <typename T>
__global__ __launch_bounds__(256) void planes_layernorm_kernel(const T* __restrict__ src, int C,
                                                               const T* __restrict__ w, const T* __restrict__ b,
                                                               T* __restrict__ dst, int64_t n, int64_t pitch,
                                                               int64_t written, bool blocked, bool vec, float eps,
                                                               int64_t first) {
  constexpr int PB = kLnCols<T>, E = 16 / (int)sizeof(T);  // columns per tile, elements per chunk
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  T* S = reinterpret_cast<T*>(smem);
  const int64_t stiles = (n + PB - 1) / PB;
  const int64_t id = first + blockIdx.x;
  const int64_t s0 = id % stiles * PB;
  const int64_t br = id / stiles, r = br % n, bb = br / n;
  const int c0 = blockIdx.y * 512, cn = C - c0 < 512 ? C - c0 : 512;
  // channel c of the item at (p / 128) gs + (p % 128) cs, p = item C + c
  const int64_t cs = blocked ? 64 : n * pitch, gs = 128 * n * pitch;
  const T* base = src + (blocked ? r * pitch * 128 + s0 / 64 * 64 * 128 + s0 % 64 : r * pitch + s0);
  for (int e = threadIdx.x; e < cn * 8; e += 256) {
    const int c = e >> 3, q = e & 7;
    const int64_t p = bb * C + c0 + c;
    const T* g = base + (p >> 7) * gs + (p & 127) * cs + q * E;
    T* d = S + c * PB + (q ^ ((c >> 3) & 7)) * E;
    if (vec && s0 + q * E + E <= written) {
      *reinterpret_cast<u32x4*>(d) = *reinterpret_cast<const u32x4*>(g);
    } else {
#pragma unroll
      for (int k = 0; k < E; ++k) d[k] = s0 + q * E + k < n ? g[k] : from_f32<T>(0.f);
    }
  }
  __syncthreads();
  const int lane = threadIdx.x & 63, l8 = lane & 7;
  for (int ps = (threadIdx.x >> 6) * 8 + (lane >> 3); ps < PB; ps += 32) {
    float v[8][8], sum = 0.f;
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int c = 64 * u + 8 * l8;
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        v[u][k] = c < cn ? to_f32(S[(c + k) * PB + ((ps / E) ^ l8) * E + ps % E]) : 0.f;
        sum += v[u][k];
      }
    }
    float mean = 0.f, rstd = 1.f;
    if (w) {
#pragma unroll
      for (int o = 4; o >= 1; o >>= 1) sum += shfl_xor(sum, o);
      mean = sum / C;
      float q2 = 0.f;
#pragma unroll
      for (int u = 0; u < 8; ++u)
#pragma unroll
        for (int k = 0; k < 8; ++k)
          if (64 * u + 8 * l8 < cn) q2 += (v[u][k] - mean) * (v[u][k] - mean);
#pragma unroll
      for (int o = 4; o >= 1; o >>= 1) q2 += shfl_xor(q2, o);
      rstd = __builtin_amdgcn_rsqf(q2 / C + eps);
    }
    if (s0 + ps >= n) continue;
    T* out = dst + ((bb * n + r) * n + s0 + ps) * C + c0;
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int c = 64 * u + 8 * l8;
      if (c >= cn) continue;
      if (w) {
        float wv[8], bv[8];
        to_f32x8(load8(w + c), wv);
        to_f32x8(load8(b + c), bv);
#pragma unroll
        for (int k = 0; k < 8; ++k) v[u][k] = (v[u][k] - mean) * rstd * wv[k] + bv[k];
      }
      store8(out + c, pack8<T>(v[u]));
    }
  }
}

// q/k of the flash core: dst[br][h][s][d] (s < np) = src[br*n + s][c0 + 32h + d] * mul, zero padded keys
template <typename T>
__global__ void split_qk_kernel(const T* __restrict__ src, int64_t ld, int64_t c0, T* __restrict__ dst, int64_t rows,
                                int64_t n, int64_t np, int heads, float mul) {
  const int64_t total = rows * heads * np * 32;
  for (int64_t idx = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; idx < total;
       idx += (int64_t)gridDim.x * blockDim.x) {
    const int d = (int)(idx % 32);
    const int64_t s = (idx / 32) % np;
    const int h = (int)((idx / (32 * np)) % heads);
    const int64_t br = idx / (32 * np * heads);
    dst[idx] = s < n ? from_f32<T>(to_f32(src[(br * n + s) * ld + c0 + 32 * h + d]) * mul) : from_f32<T>(0.f);
  }
}

// triangle bias planes: dst[b][h][q][k] (np x np) = src[b][q*n + k][c0 + h] * log2 e, zeros outside
template <typename T>
__global__ void bias_planes_kernel(const T* __restrict__ src, int64_t ld, int64_t c0, T* __restrict__ dst,
                                   int64_t batch, int64_t n, int64_t np, int heads) {
  const int64_t total = batch * heads * np * np;
  for (int64_t idx = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; idx < total;
       idx += (int64_t)gridDim.x * blockDim.x) {
    const int64_t k = idx % np;
    const int64_t q = (idx / np) % np;
    const int h = (int)((idx / (np * np)) % heads);
    const int64_t bb = idx / (np * np * heads);
    dst[idx] = (q < n && k < n) ? from_f32<T>(to_f32(src[(bb * n * n + q * n + k) * ld + c0 + h]) * kLog2e)
                                : from_f32<T>(0.f);
  }
}

// mask bias of row r: mb[b][r][k] = inf * (mask[b][orig(r*n + k)] - 1) * log2 e (0 without a mask),
// -inf for the padded keys
template <typename T>
__global__ void grid_mask_bias_kernel(const T* __restrict__ mask, float* __restrict__ mb, int64_t batch, int64_t n,
                                      int64_t np, float inf, int t) {
  const int64_t total = batch * n * np;
  for (int64_t idx = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; idx < total;
       idx += (int64_t)gridDim.x * blockDim.x) {
    const int64_t k = idx % np;
    const int64_t r = (idx / np) % n;
    const int64_t bb = idx / (np * n);
    float v = -INFINITY;
    if (k < n) v = mask ? inf * (to_f32(mask[bb * n * n + orig_pos(r * n + k, n, t)]) - 1.0f) * kLog2e : 0.f;
    mb[idx] = v;
  }
}

// o[i][j] *= g[i*ldg + c0 + j] for rows x width
template <typename T>
__global__ void gate_rows_kernel(T* __restrict__ o, const T* __restrict__ g, int64_t ldg, int64_t c0, int64_t rows,
                                 int width) {
  const int64_t total = rows * width;
  for (int64_t idx = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; idx < total;
       idx += (int64_t)gridDim.x * blockDim.x) {
    const int64_t i = idx / width;
    const int j = (int)(idx - i * width);
    o[idx] = from_f32<T>(to_f32(o[idx]) * to_f32(g[i * ldg + c0 + j]));
  }
}


// ---- vectorized forms (8 contiguous elements, 16-byte accesses for bf16),
// used when the widths and offsets are multiples of 8

template <typename T>
__global__ __launch_bounds__(256) void ln_grid8_kernel(const T* __restrict__ x, const T* __restrict__ w,
                                                       const T* __restrict__ b, T* __restrict__ y, int64_t rows,
                                                       int64_t n, int c, float eps, int t, int64_t first) {
  const int64_t row = (first + blockIdx.x) * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;
  const int64_t nn = n * n;
  const int64_t bb = row / nn;
  ln_row8<T>(x + (bb * nn + orig_pos(row - bb * nn, n, t)) * c, w, b, y + row * c, c, eps, threadIdx.x & 63);
}

// split_qk_kernel, 8 head dims per thread
template <typename T>
__global__ void split_qk8_kernel(const T* __restrict__ src, int64_t ld, int64_t c0, T* __restrict__ dst, int64_t rows,
                                 int64_t n, int64_t np, int heads, float mul) {
  const int64_t total = rows * heads * np * 4;
  for (int64_t i8 = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i8 < total;
       i8 += (int64_t)gridDim.x * blockDim.x) {
    const int d0 = (int)(i8 & 3) * 8;
    int64_t r = i8 >> 2;
    const int64_t s = r % np;
    r /= np;
    const int h = (int)(r % heads);
    const int64_t br = r / heads;
    float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (s < n) {
      to_f32x8(load8(src + (br * n + s) * ld + c0 + 32 * h + d0), v);
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] *= mul;
    }
    store8(dst + i8 * 8, pack8<T>(v));
  }
}

// v of the flash core, keys innermost: dst[br][hd][s] = src[br*n + s][c0 + hd] (zero for
// s >= n), through 64 x 64 LDS tiles so that both sides move whole rows
template <typename T>
__global__ __launch_bounds__(256) void split_vt_tiled_kernel(const T* __restrict__ src, int64_t ld, int64_t c0,
                                                             T* __restrict__ dst, int64_t n, int64_t np,
                                                             int hd_total) {
  __shared__ T tile[64][66];
  const int htiles = (hd_total + 63) / 64;
  const int64_t stiles = (np + 63) / 64;
  int64_t id = blockIdx.x;
  const int ht = (int)(id % htiles);
  id /= htiles;
  const int64_t st = id % stiles;
  const int64_t br = id / stiles;
  const int64_t s0 = st * 64;
  const int h0 = ht * 64;
  for (int e = threadIdx.x; e < 64 * 64; e += 256) {
    const int sl = e >> 6, hl = e & 63;
    const int64_t s = s0 + sl;
    const int hd = h0 + hl;
    tile[sl][hl] = (s < n && hd < hd_total) ? src[(br * n + s) * ld + c0 + hd] : from_f32<T>(0.f);
  }
  __syncthreads();
  for (int e = threadIdx.x; e < 64 * 64; e += 256) {
    const int hl = e >> 6, sl = e & 63;
    const int64_t s = s0 + sl;
    const int hd = h0 + hl;
    if (s < np && hd < hd_total) dst[(br * hd_total + hd) * np + s] = tile[sl][hl];
  }
}

// gate_rows_kernel, 8 columns per thread
template <typename T>
__global__ void gate_rows8_kernel(T* __restrict__ o, const T* __restrict__ g, int64_t ldg, int64_t c0, int64_t rows,
                                  int width) {
  const int w8 = width / 8;
  const int64_t total = rows * w8;
  for (int64_t i8 = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i8 < total;
       i8 += (int64_t)gridDim.x * blockDim.x) {
    const int64_t i = i8 / w8;
    const int j = (int)(i8 - i * w8) * 8;
    float ov[8], gv[8];
    to_f32x8(load8(o + i * width + j), ov);
    to_f32x8(load8(g + i * ldg + c0 + j), gv);
#pragma unroll
    for (int e = 0; e < 8; ++e) ov[e] *= gv[e];
    store8(o + i * width + j, pack8<T>(ov));
  }
}

// out[b][orig(v)][c] = (T(y[b][v][c] * m) + residual[b][orig(v)][c]) * (g != 0),
// with m the row mask and g the output mask at the output position (1 without);
// y the sum of `splits` partial products ss elements apart
template <typename T>
__global__ void scatter_add_kernel(const T* __restrict__ y, const T* __restrict__ row_mask,
                                   const T* __restrict__ residual, const T* __restrict__ out_mask,
                                   T* __restrict__ out, int64_t rows, int64_t n, int c, int t, int splits, int64_t ss) {
  const int64_t total = rows * c;
  const int64_t nn = n * n;
  for (int64_t idx = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; idx < total;
       idx += (int64_t)gridDim.x * blockDim.x) {
    const int64_t row = idx / c;
    const int ch = (int)(idx - row * c);
    const int64_t bb = row / nn;
    const int64_t o = bb * nn + orig_pos(row - bb * nn, n, t);
    float v = to_f32(y[idx]);
    for (int s = 1; s < splits; ++s) v += to_f32(y[s * ss + idx]);
    if (row_mask) v *= to_f32(row_mask[o]);
    v = round_to<T>(v);
    if (residual) v += to_f32(residual[o * c + ch]);
    if (out_mask && to_f32(out_mask[o]) == 0.f) v *= 0.f;
    out[o * c + ch] = from_f32<T>(v);
  }
}

// scatter_add_kernel, 8 channels per thread
template <typename T>
__global__ void scatter_add8_kernel(const T* __restrict__ y, const T* __restrict__ row_mask,
                                    const T* __restrict__ residual, const T* __restrict__ out_mask,
                                    T* __restrict__ out, int64_t rows, int64_t n, int c, int t, int splits,
                                    int64_t ss) {
  const int c8 = c / 8;
  const int64_t total = rows * c8;
  const int64_t nn = n * n;
  for (int64_t i8 = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i8 < total;
       i8 += (int64_t)gridDim.x * blockDim.x) {
    const int64_t row = i8 / c8;
    const int ch = (int)(i8 - row * c8) * 8;
    const int64_t bb = row / nn;
    const int64_t o = bb * nn + orig_pos(row - bb * nn, n, t);
    float v[8];
    to_f32x8(load8(y + row * c + ch), v);
    for (int s = 1; s < splits; ++s) {
      float w[8];
      to_f32x8(load8(y + s * ss + row * c + ch), w);
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] += w[e];
    }
    const float m = row_mask ? to_f32(row_mask[o]) : 1.f;
    const float g = out_mask && to_f32(out_mask[o]) == 0.f ? 0.f : 1.f;
    float r[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (residual) to_f32x8(load8(residual + o * c + ch), r);
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = (round_to<T>(v[e] * m) + r[e]) * g;
    store8(out + o * c + ch, pack8<T>(v));
  }
}

bool al16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

}  // namespace

template <typename T>
void launch_ln_grid(const T* x, const T* w, const T* b, T* y, int64_t batch, int64_t n, int c, float eps, int t,
                    hipStream_t st) {
  const int64_t rows = batch * n * n;
  const bool vec = c % 8 == 0 && c <= 512 && al16(x) && al16(w) && al16(b) && al16(y);
  for_pieces((rows + 3) / 4, [&](int64_t first, unsigned count) {
    hipLaunchKernelGGL(vec ? ln_grid8_kernel<T> : ln_grid_kernel<T>, dim3(count), dim3(256), 0, st, x, w, b, y, rows, n,
                       c, eps, t, first);
  });
}
template <typename T>
void launch_to_planes(const T* src, int64_t ld, int C, const T* mask, T* a, T* b, int64_t batch, int64_t n,
                      int64_t pitch, int t, hipStream_t st) {
  const int64_t blocks = batch * n * ((pitch + 63) / 64) * ((2 * C + 63) / 64);
  const bool vs = C % 8 == 0 && ld % 8 == 0 && al16(src), vd = pitch % 8 == 0 && al16(a) && al16(b);
  for_pieces(blocks, [&](int64_t first, unsigned count) {
    hipLaunchKernelGGL(to_planes_kernel<T>, dim3(count), dim3(256), 0, st, src, ld, C, mask, a, b, n, pitch, t, vs, vd,
                       first);
  });
}
template <typename T>
void launch_planes_layernorm(const T* src, int C, const T* w, const T* b, T* dst, T* tmp, int64_t batch, int64_t n,
                             int64_t pitch, bool blocked, float eps, hipStream_t st) {
  // C is a multiple of 8 (checked at the entry point); a row of more than 512
  // channels is moved 512 at a time and normalized afterwards
  const bool fused = C <= 512;
  const int64_t blocks = batch * n * ((n + kLnCols<T> - 1) / kLnCols<T>);
  const size_t lds = (size_t)(C < 512 ? C : 512) * 128;
  // columns of a plane's row that the contraction wrote: the DMA one's all, zeros past n
  const int64_t written = std::is_same<T, bf16>::value && pitch % 64 == 0 ? pitch : n;
  for_pieces(blocks, [&](int64_t first, unsigned count) {
    hipLaunchKernelGGL(planes_layernorm_kernel<T>, dim3(count, (unsigned)((C + 511) / 512)), dim3(256), lds, st, src, C,
                       fused ? w : nullptr, b, fused ? dst : tmp, n, pitch, written, blocked,
                       pitch % 8 == 0 && al16(src), eps, first);
  });
  if (!fused) launch_layernorm_rows<T>(tmp, w, b, dst, batch * n * n, C, eps, st);
}
template <typename T>
void launch_split_qk(const T* src, int64_t ld, int64_t c0, T* dst, int64_t rows, int64_t n, int64_t np, int heads,
                     float mul, hipStream_t st) {
  if (ld % 8 == 0 && c0 % 8 == 0 && al16(src) && al16(dst))
    hipLaunchKernelGGL(split_qk8_kernel<T>, stride_grid(rows * heads * np * 4), dim3(256), 0, st, src, ld, c0, dst,
                       rows, n, np, heads, mul);
  else
    hipLaunchKernelGGL(split_qk_kernel<T>, stride_grid(rows * heads * np * 32), dim3(256), 0, st, src, ld, c0, dst,
                       rows, n, np, heads, mul);
}
template <typename T>
void launch_split_vt(const T* src, int64_t ld, int64_t c0, T* dst, int64_t rows, int64_t n, int64_t np, int hd_total,
                     hipStream_t st) {
  const int64_t blocks = rows * ((np + 63) / 64) * ((hd_total + 63) / 64);
  hipLaunchKernelGGL(split_vt_tiled_kernel<T>, dim3((unsigned)blocks), dim3(256), 0, st, src, ld, c0, dst, n, np,
                     hd_total);
}
template <typename T>
void launch_bias_planes(const T* src, int64_t ld, int64_t c0, T* dst, int64_t batch, int64_t n, int64_t np, int heads,
                        hipStream_t st) {
  hipLaunchKernelGGL(bias_planes_kernel<T>, stride_grid(batch * heads * np * np), dim3(256), 0, st, src, ld, c0, dst,
                     batch, n, np, heads);
}
template <typename T>
void launch_grid_mask_bias(const T* mask, float* mb, int64_t batch, int64_t n, int64_t np, float inf, int t,
                           hipStream_t st) {
  hipLaunchKernelGGL(grid_mask_bias_kernel<T>, stride_grid(batch * n * np), dim3(256), 0, st, mask, mb, batch, n, np,
                     inf, t);
}
template <typename T>
void launch_gate_rows(T* o, const T* g, int64_t ldg, int64_t c0, int64_t rows, int width, hipStream_t st) {
  if (width % 8 == 0 && ldg % 8 == 0 && c0 % 8 == 0 && al16(o) && al16(g))
    hipLaunchKernelGGL(gate_rows8_kernel<T>, stride_grid(rows * width / 8), dim3(256), 0, st, o, g, ldg, c0, rows,
                       width);
  else
    hipLaunchKernelGGL(gate_rows_kernel<T>, stride_grid(rows * width), dim3(256), 0, st, o, g, ldg, c0, rows, width);
}
template <typename T>
void launch_scatter_add(const T* y, const T* row_mask, const T* residual, const T* out_mask, T* out, int64_t rows,
                        int64_t n, int c, int t, hipStream_t st, int splits, int64_t split_stride) {
  if (c % 8 == 0 && split_stride % 8 == 0 && al16(y) && al16(out) && (!residual || al16(residual)))
    hipLaunchKernelGGL(scatter_add8_kernel<T>, stride_grid(rows * c / 8), dim3(256), 0, st, y, row_mask, residual,
                       out_mask, out, rows, n, c, t, splits, split_stride);
  else
    hipLaunchKernelGGL(scatter_add_kernel<T>, stride_grid(rows * c), dim3(256), 0, st, y, row_mask, residual, out_mask,
                       out, rows, n, c, t, splits, split_stride);
}

#define FJX_INST(T)                                                                                                \
  template void launch_ln_grid<T>(const T*, const T*, const T*, T*, int64_t, int64_t, int, float, int, hipStream_t); \
  template void launch_to_planes<T>(const T*, int64_t, int, const T*, T*, T*, int64_t, int64_t, int64_t, int,        \
                                    hipStream_t);                                                                   \
  template void launch_planes_layernorm<T>(const T*, int, const T*, const T*, T*, T*, int64_t, int64_t, int64_t,   \
                                           bool, float, hipStream_t);                                                     \
  template void launch_split_qk<T>(const T*, int64_t, int64_t, T*, int64_t, int64_t, int64_t, int, float,           \
                                   hipStream_t);                                                                   \
  template void launch_split_vt<T>(const T*, int64_t, int64_t, T*, int64_t, int64_t, int64_t, int, hipStream_t);   \
  template void launch_bias_planes<T>(const T*, int64_t, int64_t, T*, int64_t, int64_t, int64_t, int, hipStream_t); \
  template void launch_grid_mask_bias<T>(const T*, float*, int64_t, int64_t, int64_t, float, int, hipStream_t);     \
  template void launch_gate_rows<T>(T*, const T*, int64_t, int64_t, int64_t, int, hipStream_t);                      \
  template void launch_scatter_add<T>(const T*, const T*, const T*, const T*, T*, int64_t, int64_t, int, int,     \
                                      hipStream_t, int, int64_t);
FJX_INST(float)
FJX_INST(bf16)
#undef FJX_INST

}  // namespace fjx
