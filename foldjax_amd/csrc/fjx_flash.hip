// Flash triangle attention on MFMA with a softmax offset: the fp32 kernel, and
// the bf16 fallback of the pipelined offset-free pass (fjx_flash_pipe.hip).
//
// One wave owns one attention row i of the pair grid and 64 queries of
// one head; the ROWS waves of a workgroup own ROWS consecutive rows with the same
// head and query tile, so the [queries x 64] tile of the triangle bias -- shared by
// every row -- is staged once in LDS per key block (double-buffered, the next
// tile prefetched into registers while the current one is consumed) and read
// by all of them. Each row's mask bias for the block travels the same way.
//
// Memory pipeline per key block: at its top the wave issues the loads of the
// next block's V (into a second register set), bias tile and mask bias; after
// the last query tile has used K it issues the next block's K. Every prefetch
// is unconditional (the last block re-reads itself), so no path through the
// loop leaves a load outstanding at its top, and the in-order memory counter
// never makes a product wait for a prefetch issued after its own operands. Q
// lives in LDS (fragment order, conflict-free) to leave registers for V.
//
// Everything is computed transposed so that each lane keeps one query:
//   S^T[key][q] = K[key][:] . Q[q][:]   (A = K fragment, B = Q fragment)
//   lane l holds S^T[key_of(kt, 4g + r)][16qt + l%16], g = l/16
// with the accumulator initialised to the bias tile (plus the mask bias when
// the block holds masked keys). The K rows of a block are loaded in a
// permuted order (key_of below) so that lane group g ends up holding the 8
// consecutive keys 32c + 8g .. +7 of each 32-key chunk c: the probabilities
// then feed the second product directly as the B operand,
//   O^T[d][q] += V^T[d][keys] . P^T[keys][q]
// and each V^T fragment is one contiguous 16-byte load (an unpermuted order
// needs two 8-byte pieces per lane, twice the load instructions and cache-line
// touches, and the memory pipeline bounds this kernel). The
// online-softmax max lives in the lane of its query. The softmax
// denominator is a third product with an all-ones A operand, so the running
// sums cost MFMA cycles instead of VALU adds. The softmax offset of each query
// is lazy: it moves (rescaling O and the sums, behind a wave-uniform test)
// only when some score of the block exceeds it by more than 2^8 in
// probability.
// Scores are in log2 units: q carries scale*log2(e), and the bias and mask
// bias arrive multiplied by log2(e).
#include <type_traits>

#include "fjx_common.hpp"
#include "fjx_kernels.hpp"
#include "fjx_tile.hpp"

namespace fjx {

constexpr int kQT = 64;   // queries per wave
constexpr int kKB = 64;   // keys per block
constexpr int kD = 32;    // head dim
constexpr int kNumXcdF = 8;
constexpr int kBiasLd = kKB + 4;  // padded LDS row (floats)
constexpr float kLazy = 8.0f;     // running-max slack before a rescale (log2 units)

__device__ __forceinline__ int64_t xcd_remap_f(int64_t w, int64_t total) {
  const int64_t per = total / kNumXcdF;
  if (w >= per * kNumXcdF) return w;
  return (w % kNumXcdF) * per + w / kNumXcdF;
}

// Key order inside a 64-key block. Row i of the K tile kt holds key
//   key_of(kt, i) = 32 (kt/2) + 8 (i/4) + 4 (kt%2) + i%4,
// so accumulator row 4g + r of tile kt is key 32 (kt/2) + 8g + 4 (kt%2) + r:
// lane group g holds, for the 32-key chunk c = kt/2, the 8 consecutive keys
// 32c + 8g .. +7 -- one contiguous 16-byte V^T fragment per lane -- and its
// 4 bias / mask values of tile kt are 4 consecutive columns.
__device__ __forceinline__ int key_of(int kt, int i) { return 32 * (kt >> 1) + 8 * (i >> 2) + 4 * (kt & 1) + (i & 3); }
__device__ __forceinline__ int col_of(int kt, int g) { return 32 * (kt >> 1) + 8 * g + 4 * (kt & 1); }

// max over the 4 lanes {l%16 + 16g}
__device__ __forceinline__ float max_over_groups(float x) {
  const unsigned u = __float_as_uint(x);
  const auto a = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  const float y = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const unsigned v = __float_as_uint(y);
  const auto b = __builtin_amdgcn_permlane32_swap(v, v, false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}

template <typename T> __device__ __forceinline__ typename Frag<T>::type ones8() {
  const T o = from_f32<T>(1.0f);
  return typename Frag<T>::type{o, o, o, o, o, o, o, o};
}

// the workgroup of rows ROWS rg .. of item b and queries q0 .. q0 + 63 of head h
template <typename T, int ROWS>
__device__ __forceinline__ void flash_tri_body(const FlashParams<T>& P, int64_t b, int64_t h, int64_t rg, int64_t q0) {
  typedef typename Frag<T>::type FragT;
  constexpr int NQT = 4;  // query tiles of 16
  constexpr int QTL = 16 * NQT;
  __shared__ __attribute__((aligned(16))) float bias_s[2][QTL][kBiasLd];
  __shared__ __attribute__((aligned(16))) FragT q_s[ROWS][4][64];  // [wave][qt][lane]: B fragments of Q
  __shared__ __attribute__((aligned(16))) float mb_s[2][ROWS][kKB];  // each row's mask bias, one key block

  const int64_t n = P.n;
  const int64_t np = P.np;
  const int64_t H = P.heads;

  const int t = threadIdx.x;
  const int wave = t >> 6;
  const int lane = t & 63;
  const int li = lane & 15;
  const int lg = lane >> 4;
  const int64_t row = rg * ROWS + wave;
  const bool row_ok = row < P.rows;
  const int64_t i = row_ok ? row : P.rows - 1;

  const int64_t head_off = ((b * P.rows + i) * H + h) * P.qk_rows;  // in rows of length kD
  const int last = (int)P.qk_rows - 1;  // keys past it repeat it (their mask bias is -inf); queries are zeros
  const T* Q = P.q + head_off * kD;
  const T* K = P.k + head_off * kD;
  const T* VT = P.vt + ((b * P.rows + i) * H * kD + h * kD) * np;
  const float* MB = P.mb + (b * P.rows + i) * np;
  const T* BIAS = P.bias + b * P.bias_stride_b + h * np * np;

  const int64_t nblk = np / kKB;

  // Q stays in LDS (in fragment order: conflict-free 16-byte reads) and is
  // re-read per key block, which leaves registers for a second V buffer
#pragma unroll
  for (int qt = 0; qt < NQT; ++qt) {
    const int q = (int)q0 + 16 * qt + li;
    FragT f = load8(Q + min(q, last) * kD + 8 * lg);
    if (q > last) f = FragT{};
    if (P.q_mul != 1.f) {
#pragma unroll
      for (int e = 0; e < 8; ++e) f[e] = from_f32<T>(to_f32(f[e]) * P.q_mul);
    }
    q_s[wave][qt][lane] = f;
  }

  float m[NQT];
  f32x4 o[2][NQT], lsum[NQT];  // a query tile has sums of its own: what a NaN score spoils is its query alone
#pragma unroll
  for (int qt = 0; qt < NQT; ++qt) {
    m[qt] = -1.0e30f;
    o[0][qt] = f32x4{0.f, 0.f, 0.f, 0.f};
    o[1][qt] = f32x4{0.f, 0.f, 0.f, 0.f};
    lsum[qt] = f32x4{0.f, 0.f, 0.f, 0.f};
  }

  // bias tile fill: 8 threads cover one 64-key row (a whole cache line in
  // bf16), 64*ROWS/8 rows per pass
  constexpr int NT = 64 * ROWS;
  constexpr int RPP = NT / 8;             // rows per pass
  constexpr int PASSES = QTL / RPP;
  static_assert(PASSES * RPP == QTL, "bias tile fill");
  const int br = t >> 3;
  const int bc = 8 * (t & 7);
  const T* bsrc = BIAS + (q0 + br) * np + bc;
  // the next key block's bias tile and mask bias travel in registers and are
  // written to the other LDS buffer at the end of the current block; the
  // mask flag (any non-zero mask bias in this row's block) is wave-uniform
  typename Frag<T>::type breg[PASSES];
  float mbn;
  auto fetch_tile = [&](int64_t k0) {
#pragma unroll
    for (int c = 0; c < PASSES; ++c) breg[c] = load8(bsrc + (int64_t)RPP * c * np + k0);
    mbn = MB[k0 + lane];
  };
  auto put_tile = [&](int buf) {
#pragma unroll
    for (int c = 0; c < PASSES; ++c) {
      float f[8];
      to_f32x8(breg[c], f);
      *reinterpret_cast<f32x4*>(&bias_s[buf][br + RPP * c][bc]) = f32x4{f[0], f[1], f[2], f[3]};
      *reinterpret_cast<f32x4*>(&bias_s[buf][br + RPP * c][bc + 4]) = f32x4{f[4], f[5], f[6], f[7]};
    }
    mb_s[buf][wave][lane] = mbn;
    return __builtin_amdgcn_ballot_w64(mbn != 0.f) != 0;
  };
  fetch_tile(0);
  bool masked_blk = put_tile(0);

  FragT kf[4];
  auto load_k = [&](int64_t k0) {
#pragma unroll
    for (int kt = 0; kt < 4; ++kt) kf[kt] = load8(K + min((int)k0 + key_of(kt, li), last) * kD + 8 * lg);
  };
  load_k(0);
  // V of the current block in vf, the next block's arriving in vn
  FragT vf[2][2], vn[2][2];  // [dt][c]
  auto load_v = [&](FragT (&v)[2][2], int64_t k0) {
#pragma unroll
    for (int dt = 0; dt < 2; ++dt)
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        v[dt][c] = load8(VT + (int64_t)(16 * dt + li) * np + k0 + 32 * c + 8 * lg);
      }
  };
  load_v(vf, 0);
  // drain every counter once here: the loop's own waits then see nothing
  // pending from before it (an outstanding pre-loop load would be waited on,
  // in issue order, behind the next block's prefetch)
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();

  // one key block; V of this block in vc, the next block's loaded into vx
  auto key_block = [&](int64_t blk, FragT (&vc)[2][2], FragT (&vx)[2][2]) {
    const int buf = blk & 1;
    const int64_t k0 = blk * kKB;
    // prefetches run unconditionally (the last block re-reads itself), so
    // that no path through the loop leaves a load outstanding at its top
    const int64_t kn = blk + 1 < nblk ? k0 + kKB : k0;
    load_v(vx, kn);
    fetch_tile(kn);

#pragma unroll
    for (int qt = 0; qt < NQT; ++qt) {
      const FragT qf = q_s[wave][qt][lane];
      f32x4 s[4];
#pragma unroll
      for (int kt = 0; kt < 4; ++kt) s[kt] = *reinterpret_cast<const f32x4*>(&bias_s[buf][16 * qt + li][col_of(kt, lg)]);
      // blocks holding masked or padded keys add the mask bias (re-read per
      // query tile, a cache hit, so that it is not live across the block);
      // the test is wave-uniform, a scalar branch
      if (masked_blk) {
#pragma unroll
        for (int kt = 0; kt < 4; ++kt) {
          s[kt] += *reinterpret_cast<const f32x4*>(&mb_s[buf][wave][col_of(kt, lg)]);
        }
      }
#pragma unroll
      for (int kt = 0; kt < 4; ++kt) mma(s[kt], kf[kt], qf);
      if (qt == NQT - 1) {
        // K of this block is consumed: fetch the next block's into the same registers
        load_k(kn);
      }
      float pv[4][4];
      // this lane's 16 scores: a max3 tree (5 + 2 + 1)
      const float t0 = fmaxf(fmaxf(s[0][0], s[0][1]), s[0][2]);
      const float t1 = fmaxf(fmaxf(s[0][3], s[1][0]), s[1][1]);
      const float t2 = fmaxf(fmaxf(s[1][2], s[1][3]), s[2][0]);
      const float t3 = fmaxf(fmaxf(s[2][1], s[2][2]), s[2][3]);
      const float t4 = fmaxf(fmaxf(s[3][0], s[3][1]), s[3][2]);
      const float u0 = fmaxf(fmaxf(t0, t1), t2);
      const float u1 = fmaxf(fmaxf(t3, t4), s[3][3]);
      const float lmx = fmaxf(u0, u1);
      // lazy offset: m moves only when some score of the block exceeds it by
      // more than kLazy (log2 units), so exp2(s - m) <= 2^kLazy; the test
      // needs no cross-lane reduction, and the rescale (a wave-uniform
      // branch, rare after the first block) takes the exact block max of
      // each query over its 4 lane groups
      if (__builtin_amdgcn_ballot_w64(lmx > m[qt] + kLazy) != 0) {
        const float mnew = fmaxf(m[qt], max_over_groups(lmx));
        const float alpha = __builtin_amdgcn_exp2f(m[qt] - mnew);
        o[0][qt] *= alpha;
        o[1][qt] *= alpha;
        lsum[qt] *= alpha;
        m[qt] = mnew;
      }
      const float mnew = m[qt];
#pragma unroll
      for (int kt = 0; kt < 4; ++kt)
#pragma unroll
        for (int r = 0; r < 4; ++r) pv[kt][r] = __builtin_amdgcn_exp2f(s[kt][r] - mnew);
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const float f[8] = {pv[2 * c][0], pv[2 * c][1], pv[2 * c][2], pv[2 * c][3],
                            pv[2 * c + 1][0], pv[2 * c + 1][1], pv[2 * c + 1][2], pv[2 * c + 1][3]};
        const FragT pf = pack8<T>(f);
        mma(o[0][qt], vc[0][c], pf);
        mma(o[1][qt], vc[1][c], pf);
        mma(lsum[qt], ones8<T>(), pf);
      }
    }

    masked_blk = put_tile(buf ^ 1);
    __syncthreads();
  };
  // unrolled by two so that the V register sets alternate instead of being copied
  for (int64_t blk = 0;;) {
    key_block(blk, vf, vn);
    if (++blk >= nblk) break;
    key_block(blk, vn, vf);
    if (++blk >= nblk) break;
  }

  if (!row_ok) return;
  T* OUT = P.out + b * P.o_stride_b + i * P.o_stride_row + h * P.o_stride_head;
#pragma unroll
  for (int qt = 0; qt < NQT; ++qt) {
    const float inv = 1.0f / lsum[qt][0];
    const int64_t q = q0 + 16 * qt + li;
    if (q >= n) continue;
#pragma unroll
    for (int dt = 0; dt < 2; ++dt) {
      float v[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = o[dt][qt][r] * inv;
      // 4 consecutive head dims; every o_stride_* is a multiple of 4
      store4f(OUT + q * P.o_stride_q + 16 * dt + 4 * lg, v);
    }
  }
}

constexpr int kRows = 4;

// workgroup vb of a grid of `total`, of `queries` queries each
template <typename T>
struct FlashTile {
  int64_t b, h, rg, q0;
  __device__ __forceinline__ FlashTile(const FlashParams<T>& P, int64_t vb, int64_t total, int queries) {
    const int64_t QT = (P.np + queries - 1) / queries;
    const int64_t RG = (P.rows + kRows - 1) / kRows;
    int64_t lid = xcd_remap_f(vb, total);
    q0 = lid % QT * queries;
    lid /= QT;
    rg = lid % RG;
    lid /= RG;
    h = lid % P.heads;
    b = lid / P.heads;
  }
};

// The bf16 fallback of the pipelined offset-free pass (fjx_flash_pipe.hip),
// over that pass's grid of `total` workgroups of `queries` queries: workgroup w
// reads the flags of `per` consecutive ones (64 a load) and recomputes the
// flagged ones with a softmax offset, 64 queries at a time (128 would need
// their sums to share accumulators, through which a NaN of one query reached
// three others, and spilled). At most four workgroups per resident one: fewer
// when nothing is flagged, yet flags that lie together still spread. The core
// on 4 heads, 128 queries and one workgroup per resident one against this, us:
// nothing flagged 154 / 150 at n = 499, 920 / 916 at 1024; everything 324 / 301
// and 2100 / 2055; one row in 50 at n = 952 1678 / 1008.
__global__ __launch_bounds__(64 * kRows) __attribute__((amdgpu_waves_per_eu(2, 2)))
void flash_tri_redo_kernel_bf16(FlashParams<bf16> P, int queries, int64_t total, int64_t per) {
  const int64_t base = (int64_t)blockIdx.x * per;
  const int lane = threadIdx.x & 63;
  for (int64_t c0 = 0; c0 < per; c0 += 64) {
    const int64_t vb = base + c0 + lane;
    const bool f = c0 + lane < per && vb < total && P.fallback[vb] != 0u;
    uint64_t m = __builtin_amdgcn_ballot_w64(f);  // the same in every wave
    while (m != 0) {
      const int k = __builtin_ctzll(m);
      m &= m - 1;
      const FlashTile<bf16> tl(P, base + c0 + k, total, queries);
      for (int64_t q0 = tl.q0; q0 < tl.q0 + queries && q0 < P.np; q0 += 64) {
        flash_tri_body<bf16, kRows>(P, tl.b, tl.h, tl.rg, q0);
        __syncthreads();  // LDS is reused by the next queries or workgroup
      }
    }
  }
}

__global__ __launch_bounds__(64 * kRows) void flash_tri_kernel_f32(FlashParams<float> P) {
  const FlashTile<float> tl(P, blockIdx.x, gridDim.x, kQT);
  flash_tri_body<float, kRows>(P, tl.b, tl.h, tl.rg, tl.q0);
}

template <typename T>
void launch_flash(const FlashParams<T>& p, int64_t batch, hipStream_t st) {
  // one row (the single-track attention, a bias per head): the keys are split
  // over the waves of a workgroup instead (fjx_single_flash.hip)
  if (p.rows == 1) {
    launch_flash_single<T>(p, batch, st);
    return;
  }
  const int64_t groups = batch * p.heads * ((p.rows + kRows - 1) / kRows);
  if constexpr (std::is_same<T, bf16>::value) {
    // the pipelined pass writes every flag of its grid; the offset kernel then
    // redoes the flagged workgroups
    // 128 queries a workgroup (each K and V load serves twice the queries)
    // unless that leaves the GPU mostly without workgroups: whole tri-attn,
    // 64 against 128 queries: 36.2 / 38.0 us at n = 77, 49.8 / 54.3 at 150 (304
    // workgroups of 128), 55.3 / 55.3 at 180 (360), 64.8 / 62.8 at 200, 267.7 /
    // 237.7 at 499
    const int queries = groups * ((p.np + 127) / 128) < 320 ? 64 : 128;
    const int64_t total = groups * ((p.np + queries - 1) / queries);
    launch_flash_pipe(p, groups, queries, st);
    const int64_t cap =
        tile::resident_blocks(reinterpret_cast<const void*>(flash_tri_redo_kernel_bf16), 64 * kRows);
    const int64_t per = (total + 4 * cap - 1) / (4 * cap);  // flags a workgroup
    hipLaunchKernelGGL(flash_tri_redo_kernel_bf16, dim3((unsigned)((total + per - 1) / per)), dim3(64 * kRows), 0, st,
                       p, queries, total, per);
  } else {
    hipLaunchKernelGGL(flash_tri_kernel_f32, dim3((unsigned)(groups * (p.np / kQT))), dim3(64 * kRows), 0, st, p);
  }
}

template void launch_flash<bf16>(const FlashParams<bf16>&, int64_t, hipStream_t);
template void launch_flash<float>(const FlashParams<float>&, int64_t, hipStream_t);

}  // namespace fjx
