// Kernel parameter blocks and launchers shared between the HIP translation
// units and the C ABI layer (fjx_capi.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace fjx {

// A launch takes fewer than 2^32 threads; past them its block count wraps, with
// no error. Launches of up to 2^23 blocks of 256 threads, from block `first` on
template <typename F>
void for_pieces(int64_t blocks, F launch) {
  constexpr int64_t kMax = (int64_t)1 << 23;
  for (int64_t first = 0; first < blocks; first += kMax)
    launch(first, (unsigned)(blocks - first < kMax ? blocks - first : kMax));
}

template <typename T>
struct TriMulPrologueParams {
  const T* x;     // [B][N][N][128]
  const T* mask;  // [B][N][N] or null
  const T* ln_w;
  const T* ln_b;
  const T* w_p;     // [256][128]: rows 0..127 -> a, 128..255 -> b
  const T* w_g;     // [256][128]
  T* a_cm;          // [B][128][N][pitch] virtual grid; columns N .. pitch-1 are written as zeros
  T* b_cm;
  int64_t n;
  int64_t pitch;    // elements per row of a and b: N rounded up to 64, or N (tight)
  float eps;
  int transpose;    // 1 for the incoming direction
  int cw;           // channels of x (and rows of w_p/w_g) when below 128 (a multiple of 32); 0: 128
};

template <typename T>
struct TriAttnPrologueParams {
  const T* x;
  const T* mask;
  const T* ln_w;
  const T* ln_b;
  const T* w_bias;  // [4][128]
  const T* w_q;     // [128][128]
  const T* w_k;
  const T* w_v;
  T* q;             // [B][N][4][Np][32]
  T* k;
  T* vt;            // [B][N][128][Np]
  T* bias;          // [B][4][Np][Np]
  float* mb;        // [B][N][Np]
  int64_t n;
  int64_t np;
  float eps;
  float inf;
  float q_scale;    // head_dim^-0.5 * log2(e)
  int transpose;    // 1 for the ending node
  int cw;           // channels of x (the k of every weight) when below 128 (a multiple of 32); 0: 128
};

template <typename T>
struct TriMulEpilogueParams {
  const T* o;         // contraction output, channel-major [B][128][N][pitch], or tile-blocked (o_blocked)
  const T* x;         // the op's input [B][N][N][128] (for the output gate)
  const T* ln_in_w;   // LN_in, recomputed for the gate
  const T* ln_in_b;
  const T* ln_out_w;  // LN over the contraction output
  const T* ln_out_b;
  const T* w_pout;    // [128][128]
  const T* w_gout;    // [128][128]
  const T* residual;  // [B][N][N][128] or null (may alias out)
  const T* out_mask;  // [B][N][N] or null: positions where it is 0 are written as 0
  T* out;
  int64_t n;
  float eps;
  int64_t pitch;      // elements per row of o: N rounded up to 64, or N (tight)
  // o tile-blocked (the LDS-DMA contraction's output): a row's columns in
  // blocks of 64, [B][N rows][pitch / 64 blocks][128 channels][64]
  bool o_blocked;
  int cw;             // channels of x / out (k of w_gout, rows of both weights) when below 128; 0: 128
};

template <typename T>
struct TriAttnEpilogueParams {
  const T* o;         // attention output, head-major [B][N rows][4 heads][N][32] in the virtual grid
  const T* x;         // the op's input [B][N][N][128] (for the gate)
  const T* ln_w;
  const T* ln_b;
  const T* w_g;       // [128][128] or null (ungated)
  const T* w_o;       // [128][128]
  const T* residual;  // original grid, or null (may alias out)
  const T* out_mask;  // original grid [B][N][N], or null: positions where it is 0 are written as 0
  T* out;             // original grid
  int64_t n;
  float eps;
  int transpose;      // 1 for the ending node
  int cw;             // channels of x / out (k of w_g, rows of w_o) when below 128; 0: 128
};

template <typename T, typename TO>
struct GemmParams {
  const T* a;       // [batches][m][lda], k-contiguous rows
  const T* b;       // [batches][n][ldb], k-contiguous rows (a PyTorch [out, in] weight)
  TO* c;            // [batches][m][ldc]
  int64_t m, n, k;
  int64_t lda, ldb, ldc;
  int64_t sa, sb, sc;  // batch strides in elements (0 = shared)
  int64_t batches;
  const T* bias;       // [n] or null
  int64_t bias_n;      // the bias covers columns < bias_n (0: all n)
  int act;             // 0 none, 1 sigmoid, 2 silu
  int64_t act_col0;    // the activation applies to columns >= act_col0
  const TO* gate;      // indexed like c, or null
  const TO* residual;  // indexed like c, or null (may alias c)
  const TO* row_gate;  // [m] per output row, or null: rows where it is 0 are written as 0 (after the residual)
  // proj_round: the product is a projection output -- rounded to TO, times
  // row_scale[row] when set, rounded again -- before the residual is added
  // (the order of a transition's row mask and residual)
  int proj_round;
  const TO* row_scale;  // [m] or null (with proj_round)
  // map_t: row r of the product is stored at, and reads its residual and
  // row gate from, the transposed pair-grid position: with N = map_n,
  // r = b N^2 + i N + j goes to b N^2 + j N + i (the ending node's grid)
  int map_t;
  int64_t map_n;
  // pair mode (launch_gemm_dma only): b and b2 are two weights of `units`
  // rows, n = 2 units, and C[i][u] combines a = A b^T and b = A b2^T (both
  // rounded to TO first): 1 = silu(a) * b (SwiGLU), 2 = a * sigmoid(b) (a gated
  // projection); C has `units` columns
  int swiglu;
  const T* b2;
  // with swiglu 2 and grid_pitch > 0: the product goes out channel by channel,
  // the layout of the triangle contraction. A is a pair grid [item][grid_n]
  // [grid_n] of rows, m counts the rows of the padded grid [item][r][grid_pitch],
  // whose column s of row r is A's position (r, s), or (s, r) with grid_t. Unit
  // u times the position's mask goes to c, or from grid_units on to c2, at
  // [item][u % grid_units][r][s]; zeros past grid_n
  int64_t grid_n, grid_pitch, grid_units;
  int grid_t;
  const T* grid_mask;  // [item][grid_n][grid_n] or null
  TO* c2;
};

template <typename T>
struct TransitionParams {
  const T* x;         // [rows][C]
  const T* ln_w;
  const T* ln_b;
  const T* w_a;       // [4C][C] (silu branch)
  const T* w_b;       // [4C][C]
  const T* w_o;       // [C][4C]
  const T* row_mask;  // [rows] or null
  const T* residual;  // [rows][C] or null (may alias out)
  const T* out_mask;  // [rows] or null: rows where it is 0 are written as 0 (after the residual)
  T* out;             // [rows][C]
  int64_t rows;
  float eps;
  // optional pair-bias epilogue (pb_out null: off): rows are the positions
  // (b, r, s) of [B, pb_n, pb_n]; pb_out[b][h][r][s] = log2(e) *
  // LN_pb(out row) . pb_w[h] in the padded [B, pb_heads, pb_np, pb_np]
  // layout the flash kernel reads; pb_heads <= 16
  const T* pb_ln_w;
  const T* pb_ln_b;
  const T* pb_w;      // [pb_heads][C]
  T* pb_out;
  int64_t pb_n;
  int64_t pb_np;
  int pb_heads;
  float pb_eps;
  // the same epilogue with the norm, weight and bias in fp32 over a bf16
  // transition (the Boltz-2 single track's precision); pbf_out null: off
  const float* pbf_ln_w;
  const float* pbf_ln_b;
  const float* pbf_w;  // [pb_heads][C]
  float* pbf_out;
  // channels of x / out when below 128 (a multiple of 32, hidden 4 cw): the
  // narrow form of the kernel; 0 or 128: the full form
  int cw;
};

template <typename T>
struct FlashParams {
  const T* q;        // [B][N][H][qk_rows][32], times q_mul on load: scale*log2 e (or 1, pre-scaled)
  const T* k;        // [B][N][H][qk_rows][32]
  const T* vt;       // [B][N][H*32][Np]
  const T* bias;     // [B][H][Np][Np], already times log2 e
  const float* mb;   // [B][N][Np], already times log2 e; -inf for padded keys
  T* out;            // out[b][i][q][h*32+d] via the strides below
  int64_t n;
  int64_t np;
  int64_t heads;
  int64_t rows;      // number of attention rows i (== n for the fused module)
  int64_t qk_rows;   // q and k rows per head: np, zeros past n; or n (rows > 1 only), nothing read past them
  float q_mul;
  int64_t o_stride_b;
  int64_t o_stride_row;
  int64_t o_stride_head;
  int64_t o_stride_q;
  int64_t bias_stride_b;  // 0 when one bias is shared by all batches
  // bf16, rows > 1: a flag per workgroup of the offset-free pass, written by
  // it (fjx_flash_pipe.hip) and read by the offset kernel (fjx_flash.hip)
  unsigned* fallback;
  // rows == 1 only: out is [B][n][heads * gate_dh], the first gate_dh (<= 32)
  // dims of each head times gate[B n][ld]'s same columns; null: o_stride_*
  const T* gate;
  int64_t gate_ld;
  int gate_dh;
};

template <typename T>
void launch_trimul_prologue(const TriMulPrologueParams<T>& p, int64_t batch, hipStream_t st);
// float: below 128 channels (launch_triattn_prologue_split takes 128)
template <typename T>
void launch_triattn_prologue(const TriAttnPrologueParams<T>& p, int64_t batch, hipStream_t st);
template <typename T>
void launch_trimul_epilogue(const TriMulEpilogueParams<T>& p, int64_t batch, hipStream_t st);
template <typename T>
void launch_triattn_epilogue(const TriAttnEpilogueParams<T>& p, int64_t batch, hipStream_t st);
template <typename T, typename TO>
void launch_gemm(const GemmParams<T, TO>& p, hipStream_t st);
// the bf16 GEMM on the LDS-DMA pipeline (fjx_gemm_dma.hip); false when the
// shape or alignment does not suit it (the caller then runs gemm_nt_kernel)
bool launch_gemm_dma(const GemmParams<bf16, bf16>& p, hipStream_t st);
// whether launch_gemm_dma takes p (shape, alignment and size)
bool gemm_dma_ok(const GemmParams<bf16, bf16>& p);
// triangle contraction, bf16: o[c] = a[c] b[c]^T for c < batches, each n rows
// of n elements, rows `pitch` apart in a, b and o. A pitch that is a multiple
// of 64 (with zeros past n in a and b) runs the LDS-DMA kernel, which writes
// whole rows of o, any other the register-staged one, which writes n columns.
// o comes tile-blocked (TriMulEpilogueParams::o_blocked) from the former where
// batches is a multiple of 128, else as [batches][n][pitch]; returns whether it
// is blocked
bool launch_contract(const bf16* a, const bf16* b, bf16* o, int64_t n, int64_t pitch, int64_t batches, hipStream_t st);
// the same in fp32 from bf16 planes (Split8) of a and b, `plane` elements
// apart; pitch a multiple of 64, batches of 128, o tile-blocked
void launch_contract_split(const bf16* a, const bf16* b, float* o, int64_t n, int64_t pitch, int64_t plane,
                           int64_t batches, hipStream_t st);
// float: below 128 channels (launch_transition_split takes 128)
template <typename T>
void launch_transition(const TransitionParams<T>& p, int c, hipStream_t st);
// fp32 on the bf16 matrix cores (fjx_rowproj_f32.hip), c_z = 128: a and b of
// the prologue as three bf16 planes `plane` elements apart, o tile-blocked
void launch_trimul_prologue_split(const TriMulPrologueParams<float>& p, bf16* a, bf16* b, int64_t plane, int64_t batch,
                                  hipStream_t st);
void launch_trimul_epilogue_split(const TriMulEpilogueParams<float>& p, int64_t batch, hipStream_t st);
void launch_triattn_prologue_split(const TriAttnPrologueParams<float>& p, int64_t batch, hipStream_t st);
// gated only
void launch_triattn_epilogue_split(const TriAttnEpilogueParams<float>& p, int64_t batch, hipStream_t st);
void launch_transition_split(const TransitionParams<float>& p, hipStream_t st);

// single-track helpers (fjx_single.hip)
template <typename T>
void launch_layernorm_rows(const T* x, const T* w, const T* b, T* y, int64_t rows, int c, float eps, hipStream_t st);
template <typename T>
void launch_split_heads(const T* qkv, int64_t ld, int64_t batch, int64_t n, int64_t np, int heads, int dh,
                        float q_mul, T* q, T* k, T* vt, const T* mask, float* mb, float inf, hipStream_t st);
// z (and its norm and weight) in TZ, the bias in T: the Boltz-2 single track
// runs in fp32 over a bf16 pair tensor
template <typename TZ, typename T>
void launch_pair_bias(const TZ* z, const T* ln_w, const T* ln_b, const T* w, T* bias, int64_t batch, int64_t n,
                      int64_t np, int heads, float eps, hipStream_t st);
// bias[b][h][q][k] (+)= log2(e) * extra[b * sb + h * sh + q * n + k] for q, k < n;
// src (a prepared bias of the same layout) is read when given, else bias itself
template <typename T>
void launch_add_extra_bias(const T* src, T* bias, const T* extra, int64_t sb, int64_t sh, int64_t batch, int heads,
                           int64_t n, int64_t np, hipStream_t st);
template <typename T>
void launch_pair_bias_border(T* bias, int64_t planes, int64_t n, int64_t np, hipStream_t st);
template <typename T>
void launch_flash(const FlashParams<T>& p, int64_t batch, hipStream_t st);
// rows == 1, a bias per head: keys split over the waves of a workgroup
// (fjx_single_flash.hip); launch_flash routes such calls here
template <typename T>
void launch_flash_single(const FlashParams<T>& p, int64_t batch, hipStream_t st);
// the pipelined offset-free pass (fjx_flash_pipe.hip): `groups` (batch x heads
// x row groups of 4) times np / queries workgroups (64 or 128 queries each),
// each writing its fallback flag
void launch_flash_pipe(const FlashParams<bf16>& p, int64_t groups, int queries, hipStream_t st);
// the flash tile's instruction mix alone (fjx_probe.hip): kernel ms, or -1 on a HIP error
int probe_issue_mix(int mix, int waves_per_simd, int iters, float* ms, hipStream_t st);
int probe_hbm_stream(int mode, int wgs_per_cu, int64_t bytes, float* ms, hipStream_t st);

// general-width paths (fjx_generic.hip); positions v = r*n + s of the virtual
// grid read the original grid at s*n + r when t = 1
template <typename T>
void launch_ln_grid(const T* x, const T* w, const T* b, T* y, int64_t batch, int64_t n, int c, float eps, int t,
                    hipStream_t st);
// a and b of a triangle product, channel by channel with rows `pitch` apart:
// dst[item][c][r][s] = src[item][(r, s) or, with t, (s, r)][c] * mask, zeros for
// n <= s < pitch; channels 0 .. C-1 go to a, C .. 2C-1 to b
template <typename T>
void launch_to_planes(const T* src, int64_t ld, int C, const T* mask, T* a, T* b, int64_t batch, int64_t n,
                      int64_t pitch, int t, hipStream_t st);
// dst[item][(r, s)][c] = LayerNorm over c of the planes [item][c][r][pitch], or
// with `blocked` [128 planes][r][64-column block][plane][64]; tmp: as large as
// dst, used from 513 channels on
template <typename T>
void launch_planes_layernorm(const T* src, int C, const T* w, const T* b, T* dst, T* tmp, int64_t batch, int64_t n,
                             int64_t pitch, bool blocked, float eps, hipStream_t st);
template <typename T>
void launch_split_qk(const T* src, int64_t ld, int64_t c0, T* dst, int64_t rows, int64_t n, int64_t np, int heads,
                     float mul, hipStream_t st);
template <typename T>
void launch_split_vt(const T* src, int64_t ld, int64_t c0, T* dst, int64_t rows, int64_t n, int64_t np, int hd_total,
                     hipStream_t st);
template <typename T>
void launch_bias_planes(const T* src, int64_t ld, int64_t c0, T* dst, int64_t batch, int64_t n, int64_t np, int heads,
                        hipStream_t st);
template <typename T>
void launch_grid_mask_bias(const T* mask, float* mb, int64_t batch, int64_t n, int64_t np, float inf, int t,
                           hipStream_t st);
template <typename T>
void launch_gate_rows(T* o, const T* g, int64_t ldg, int64_t c0, int64_t rows, int width, hipStream_t st);
// out[orig(v)] = (T(y[v] * row_mask) + residual[orig(v)]) * (out_mask != 0),
// for a product the DMA GEMM does not take (its epilogue does this itself);
// y may be `splits` partial products (split K), `split_stride` elements
// apart, summed here
template <typename T>
void launch_scatter_add(const T* y, const T* row_mask, const T* residual, const T* out_mask, T* out, int64_t rows,
                        int64_t n, int c, int t, hipStream_t st, int splits = 1, int64_t split_stride = 0);

}  // namespace fjx
