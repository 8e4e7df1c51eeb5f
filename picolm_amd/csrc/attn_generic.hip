// attn_generic.hip -- decode and prefill attention for head dims without a
// tuned kernel (every even head_dim up to 256 but 64 and 128), and small
// prefill launches of these two (few_tiles_pay, attn_prefill.hip).
//
// Replaces the same reference code as the tuned kernels: model.c:807-892
// (decode: QK-norm, RoPE, fp16 append at row pos, online-softmax GQA
// attention over rows 0..pos) and model.c:1019-1089 (prefill: the same per
// prompt token, causal).  The reference accepts any even head_dim up to 256
// (model.c:408 sets head_dim = n_embd / n_heads; its accumulator is
// acc[256], model.c:856); the tuned kernels are built around 32-wide d blocks
// and one rope pair per lane, so other head dims run here.
//
// generic_attn_kernel  a wave takes 16 columns (a column is one token and q head
//     of a kv head) and 32 keys at a time; KS waves of a workgroup share a
//     column tile's keys and merge in LDS.  Both products run on
//     v_mfma_f32_16x16x32_f16 with fp32 sums: K and V are fp16 already, and q
//     (scaled by a power of two per column) and the weights go in as three
//     fp16 parts, the lower ones scaled up (split3): all 24 bits of weights and
//     q elements down to 2^-36 of the column's largest.  q's QK-norm sums over a
//     column's 16 lanes (not the reference's AVX2 order, which only the cached k
//     rows need).  S = K q^T with the K rows
//     straight from the cache, O^T += V^T P^T with V^T through a wave's own
//     LDS tile and ds_read_b64_tr_b16.  The S accumulators hold keys 4 g + v
//     and 16 + 4 g + v of column c in lane (g, c), which is the PV operand if
//     its k index runs over them in that order: P stays in its registers.
//     Launches with few workgroups split the keys over several of them; the
//     last to finish merges their partials.  Decode (one token) appends in the
//     same launch: the workgroup whose range holds row pos rotates and rounds
//     it and takes it from LDS.
// generic_rows_kernel  few keys of wide heads (few_keys): a workgroup per (layer,
//     token, q head) on the VALU.
// generic_append_kernel, generic_append_rows_kernel  the rows, elsewhere: RoPE
//     with the reference's four-product rotation and its fp16 rounding, a
//     thread per rope pair; with QK-norm (rmsnorm in the reference's AVX2 order),
//     and for a single token, one workgroup per row.
// Cache rows are bit-identical to the reference's (and optionally mirrored
// into caller row buffers); the softmax is exp2-based and per tile, so outputs
// agree with the reference's within the attention tolerance.
//
// What bounds it: a workgroup's serial chain (arguments, q's rotation and
// parts, the first tile, the merge: 11 to 13 thousand cycles however few keys),
// and at prompts of several hundred tokens the softmax's VALU work beside the
// MFMAs.  One workgroup per token and q head on the VALU, which this replaced,
// against this, us a layer of 8 launched one by one, with the appends: decode at
// head_dim 80, 32 heads, pos 1499: 132 -> 11.4; 300-token prompt at head_dim 96, 32
// q and 8 kv heads: 78 -> 16.1 (8 layers in one launch: 67 -> 8.2 each).  With plain
// parts (see split3) 11.0, 16.0 and 8.1; on v_mfma_f32_16x16x4_f32 without parts 1.1,
// 1.7 and 1.65 times as long.  Relative error against 64 bits, before -> now: 2.4e-7
// -> 2.0e-7 and 1.6e-7 -> 1.3e-7.
#include <algorithm>
#include <type_traits>

#include "picolm_hip.h"
#include "attn_common.h"
#include "plh_internal.h"

namespace plh {
namespace {

constexpr int kGThreads = 256;
constexpr int kGMaxD = 256;
constexpr int kGChunk = kGThreads;  // generic_rows_kernel: positions, one per thread
constexpr int kGSq = 8 * ((kGMaxD / 8 + 3) / 4 * 4 + 4);  // rms_sq_pitch(256) rows of 8
constexpr int kGMaxSplit = 16;
constexpr int kGCtrPitch = 32;  // counters on 128-byte lines of their own

struct GenericArgs {
  const float* q;  // [n_launch_layers][n_tokens][n_heads*D]
  const float* k;  // [n_launch_layers][n_tokens][kv_dim]
  const float* v;
  uint16_t* kc;    // [n_layers][S][kv_dim] fp16 bits
  uint16_t* vc;
  const float* cos_t;  // [S][D/2]
  const float* sin_t;
  float* out;      // [n_launch_layers][n_tokens][out_stride]
  const float* qn;  // QK-norm weights [n_launch_layers][D], or null
  const float* kn;
  float norm_eps;
  uint16_t* k_rows;  // appended rows also here [n_launch_layers][n_tokens][kv_dim], or null
  uint16_t* v_rows;
  int layer0, n_launch_layers, n_heads, n_kv_heads, D, max_seq_len, rope_type;
  int start_pos, n_tokens, out_stride;
  int col_tiles;                   // 16-column tiles per kv head
  int n_split, split_len;          // key ranges per tile (split_len a multiple of 32)
  int n_chunk;                     // append: workgroups per (layer, token)
  FastDiv fd_chunk, fd_tok, fd_half;   // n_chunk, n_tokens, D / 2
  FastDiv fd_split, fd_tiles, fd_kvh, fd_g;  // n_split, col_tiles, n_kv_heads, heads per kv head
  float* part;                     // [unit] GShape::kPart floats (n_split > 1)
  unsigned* ctr;                   // [group * kGCtrPitch], zero between launches
};

// Rope pair i of a head: (2i, 2i+1) for LLAMA, (i, i + D/2) for QWEN
// (tensor.c:583-601).
__device__ __forceinline__ void pair_of(int rope_type, int D, int i, int& i0, int& i1) {
  i0 = rope_type == PLH_ROPE_QWEN ? i : 2 * i;
  i1 = rope_type == PLH_ROPE_QWEN ? i + D / 2 : 2 * i + 1;
}

// x (global, D floats) into xs (LDS): rmsnorm(x, w) with the reference's
// rounding when w is given ((x * scale) * w, tensor.c:425-492), else a copy.
// Every thread must call it.
__device__ __forceinline__ void load_normed(const float* x, const float* w, int D, float eps,
                                            float* xs, float* sq, float* red) {
  float scale = 1.0f;
  if (w) scale = rms_scale_block<kGThreads>(x, D, eps, sq, red);
  for (int i = threadIdx.x; i < D; i += kGThreads) xs[i] = w ? (x[i] * scale) * w[i] : x[i];
  __syncthreads();
}

// A thread per rope pair of a (layer, token)'s kv heads, `fd_chunk` workgroups
// a token (no QK-norm).
__global__ __launch_bounds__(kGThreads) void generic_append_kernel(GenericArgs a) {
  const int D = a.D, half = D / 2, kv_dim = a.n_kv_heads * D;
  const int lt = (int)fdiv(blockIdx.x, a.fd_chunk);
  const int pair = (int)(blockIdx.x - lt * a.n_chunk) * kGThreads + threadIdx.x;
  if (pair >= kv_dim / 2) return;
  const int li = (int)fdiv(lt, a.fd_tok), t = lt - li * a.n_tokens;
  const int kvh = (int)fdiv(pair, a.fd_half), i = pair - kvh * half;
  const int pos = a.start_pos + t;
  const size_t src = (size_t)lt * kv_dim + kvh * D;
  const size_t dst = ((size_t)(a.layer0 + li) * a.max_seq_len + pos) * kv_dim + kvh * D;
  int i0, i1;
  pair_of(a.rope_type, D, i, i0, i1);
  float x0 = a.k[src + i0], x1 = a.k[src + i1];
  const float v0 = a.v[src + i0], v1 = a.v[src + i1];
  rope_rotate(x0, x1, a.cos_t[(size_t)pos * half + i], a.sin_t[(size_t)pos * half + i]);
  const uint16_t kb0 = f16_bits_rha(x0), kb1 = f16_bits_rha(x1);
  const uint16_t vb0 = f16_bits_rha(v0), vb1 = f16_bits_rha(v1);
  a.kc[dst + i0] = kb0, a.kc[dst + i1] = kb1;
  a.vc[dst + i0] = vb0, a.vc[dst + i1] = vb1;
  if (a.k_rows) {
    a.k_rows[src + i0] = kb0, a.k_rows[src + i1] = kb1;
    a.v_rows[src + i0] = vb0, a.v_rows[src + i1] = vb1;
  }
}

__global__ __launch_bounds__(kGThreads) void generic_append_rows_kernel(GenericArgs a) {
  __shared__ __align__(16) float sq[kGSq];
  __shared__ float red[8];
  __shared__ float kr[kGMaxD];
  const int D = a.D, kv_dim = a.n_kv_heads * D;
  const int kvh = blockIdx.x % a.n_kv_heads;
  const int t = (blockIdx.x / a.n_kv_heads) % a.n_tokens;
  const int li = blockIdx.x / (a.n_kv_heads * a.n_tokens);
  const int pos = a.start_pos + t;
  const size_t src = ((size_t)li * a.n_tokens + t) * kv_dim + (size_t)kvh * D;
  load_normed(a.k + src, a.kn ? a.kn + (size_t)li * D : nullptr, D, a.norm_eps, kr, sq, red);
  const float* cr = a.cos_t + (size_t)pos * (D / 2);
  const float* sr = a.sin_t + (size_t)pos * (D / 2);
  const size_t dst =
      ((size_t)(a.layer0 + li) * a.max_seq_len + pos) * kv_dim + (size_t)kvh * D;
  for (int i = threadIdx.x; i < D / 2; i += kGThreads) {
    int i0, i1;
    pair_of(a.rope_type, D, i, i0, i1);
    float x0 = kr[i0], x1 = kr[i1];
    rope_rotate(x0, x1, cr[i], sr[i]);
    const uint16_t b0 = f16_bits_rha(x0), b1 = f16_bits_rha(x1);
    a.kc[dst + i0] = b0;
    a.kc[dst + i1] = b1;
    if (a.k_rows) {
      a.k_rows[src + i0] = b0;
      a.k_rows[src + i1] = b1;
    }
  }
  for (int i = threadIdx.x; i < D; i += kGThreads) {
    const uint16_t b = f16_bits_rha(a.v[src + i]);
    a.vc[dst + i] = b;
    if (a.v_rows) a.v_rows[src + i] = b;
  }
}

// The appended row of one kv head (decode), D <= 2 * kGThreads: this thread's
// rope pair, loaded before the workgroup's other loads, and its fp16 bits into
// LDS.  With QK-norm every thread must call finish.
struct NewRow {
  float k0, k1, v0, v1, c, s;
  int i0, i1;
  __device__ __forceinline__ void load(const GenericArgs& a, size_t src) {
    const int i = min((int)threadIdx.x, a.D / 2 - 1);
    pair_of(a.rope_type, a.D, i, i0, i1);
    k0 = a.k[src + i0], k1 = a.k[src + i1];
    v0 = a.v[src + i0], v1 = a.v[src + i1];
    c = a.cos_t[(size_t)a.start_pos * (a.D / 2) + i];
    s = a.sin_t[(size_t)a.start_pos * (a.D / 2) + i];
  }
  __device__ __forceinline__ void finish(const GenericArgs& a, size_t src, int li, uint16_t* kb,
                                         uint16_t* vb, float* kr, float* sq, float* red) {
    if (a.kn) {
      load_normed(a.k + src, a.kn + (size_t)li * a.D, a.D, a.norm_eps, kr, sq, red);
      k0 = kr[i0], k1 = kr[i1];
    }
    if ((int)threadIdx.x >= a.D / 2) return;
    rope_rotate(k0, k1, c, s);
    kb[i0] = f16_bits_rha(k0), kb[i1] = f16_bits_rha(k1);
    vb[i0] = f16_bits_rha(v0), vb[i1] = f16_bits_rha(v1);
  }
};

__device__ __forceinline__ float4_t mfma_f32(float x, float y, float4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(x, y, c, 0, 0, 0);
}

// A pair of fp32 values of at most 2^14 as three fp16 parts each, every remainder
// exact: x = hi + 2^-11 (mid + lo) keeps all 24 bits of values from 2^-11 up and
// stops at 2^-35; DEEP, x = hi + 2^-11 (mid + 2^-11 lo), from 2^-22 up and 2^-46.
// (Unscaled parts: from 1 up and 2^-24.)
constexpr float kPartUp = 2048.0f, kPartDown = 1.0f / kPartUp;
template <bool DEEP>
__device__ __forceinline__ void split3(float x0, float x1, half2_t& hi, half2_t& mid,
                                       half2_t& lo) {
  const auto h = __builtin_amdgcn_cvt_pkrtz(x0, x1);
  hi = __builtin_bit_cast(half2_t, h);
  const float r0 = __builtin_fmaf((float)hi[0], -kPartUp, x0 * kPartUp);
  const float r1 = __builtin_fmaf((float)hi[1], -kPartUp, x1 * kPartUp);
  split_pair_rtz(r0, r1, mid, lo);
  if constexpr (DEEP) {
    const float l0 = __builtin_fmaf((float)mid[0], -kPartUp, r0 * kPartUp);
    const float l1 = __builtin_fmaf((float)mid[1], -kPartUp, r1 * kPartUp);
    lo = __builtin_bit_cast(half2_t, __builtin_amdgcn_cvt_pkrtz(l0, l1));
  }
}

// Shapes for DT 16-wide tiles of d (D rounded up).  LDS: q's parts and the
// waves' V tiles, then the waves' results over them.
template <int DT, int KS>
struct GShape {
  static constexpr int CW = 4 / KS;        // column tiles of a workgroup, KS waves each
  static constexpr int DP = 16 * DT;
  static constexpr int DK = (DT + 1) / 2;  // 32-wide steps of the QK product
  static constexpr int QP = 32 * DK + 8;   // halves per q row: 16 rows' 16-byte reads and
  static constexpr int VP = 32 * DK + 16;  // per V row: 16 rows' transposing reads, all banks
  static constexpr int OP = DP + 4;        // floats per result column
  static constexpr int kQ = 3 * 16 * QP;   // halves of a column tile's three parts
  static constexpr int kQV = (CW * kQ + 4 * 32 * VP) / 2;
  static constexpr int kOut = 4 * 16 * OP + 4 * 2 * 16;
  static constexpr int kFloats = kQV > kOut ? kQV : kOut;
  static constexpr int kPart = 16 * (DP + 2);  // a unit's partial: O [16][DP], (max, sum) [16]
};

constexpr int kDeviceScope = 16;  // buffer cache policy sc1

// Eight halves 32 j + 8 g .. + 7 of a row, per 32-wide step j: one 16-byte
// load where every row starts on 16 bytes (D8), else
// four of 4 bytes.  Past D the row's first halves (see clear_past).
template <int DK, bool D8>
__device__ __forceinline__ void load_row(const uint16_t* p, int D, int g, u32x4_t (&r)[DK]) {
#pragma unroll
  for (int j = 0; j < DK; ++j) {
    const int d0 = 32 * j + 8 * g;
    if constexpr (D8) {
      r[j] = *(const u32x4_t*)(p + (d0 < D ? d0 : 0));
    } else {
      r[j][0] = *(const uint32_t*)(p + (d0 < D ? d0 : 0));
      r[j][1] = *(const uint32_t*)(p + (d0 + 2 < D ? d0 + 2 : 0));
      r[j][2] = *(const uint32_t*)(p + (d0 + 4 < D ? d0 + 4 : 0));
      r[j][3] = *(const uint32_t*)(p + (d0 + 6 < D ? d0 + 6 : 0));
    }
  }
}
// Zeros past D (K: the padding meets a zero of q, but must be finite).  Apart
// from the loads, so that these stay in flight.
template <int DK>
__device__ __forceinline__ void clear_past(int D, int g, u32x4_t (&r)[DK]) {
#pragma unroll
  for (int j = 0; j < DK; ++j) {
    if (32 * j + 32 <= D) continue;  // uniform
    const int d0 = 32 * j + 8 * g;
    if (d0 >= D) r[j][0] = 0u;
    if (d0 + 2 >= D) r[j][1] = 0u;
    if (d0 + 4 >= D) r[j][2] = 0u;
    if (d0 + 6 >= D) r[j][3] = 0u;
  }
}

// ONE: a single token, whose row is appended here (KS 4).  Prompts at head dims
// 65 to 96 ask for registers for three workgroups a CU: 300 tokens at head_dim
// 96, 32 q and 8 kv heads, 17.5 -> 16.4 us with the append (at 64 the compiler
// gets there by itself, at 128 it cannot; a decode's few workgroups lose 2%).
template <int DT, int KS, bool D8, bool ONE>
__global__ __launch_bounds__(kGThreads, !ONE && D8 && (DT == 5 || DT == 6) ? 3 : 1) void
generic_attn_kernel(GenericArgs a) {
  static_assert(!ONE || KS == 4, "NewRow::finish has barriers: one column tile a workgroup");
  using Sh = GShape<DT, KS>;
  constexpr int DK = Sh::DK, CW = Sh::CW, NC = 16 * CW;
  extern __shared__ __align__(16) float lds[];
  __shared__ __align__(16) float sq[kGSq];
  __shared__ float red[8], ups[NC];
  __shared__ float kr[kGMaxD];
  __shared__ __align__(16) uint16_t knew[kGMaxD], vnew[kGMaxD];
  __shared__ int s_last;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 15, g = lane >> 4;
  const int cw = wave / KS, ks = wave % KS;  // this wave's column tile and its share of the keys
  PLH_ARGS_NOW("s"(a.q), "s"(a.k), "s"(a.v), "s"(a.kc), "s"(a.vc), "s"(a.cos_t), "s"(a.sin_t),
               "s"(a.qn), "s"(a.kn), "s"(a.layer0), "s"(a.n_heads), "s"(a.n_kv_heads), "s"(a.D),
               "s"(a.max_seq_len), "s"(a.rope_type), "s"(a.start_pos), "s"(a.n_tokens),
               "s"(a.col_tiles), "s"(a.n_split), "s"(a.split_len),
               "s"(a.fd_split.m), "s"(a.fd_split.sh), "s"(a.fd_tiles.m));
  const int D = a.D, kv_dim = a.n_kv_heads * D;
  const int G = (int)fdiv(a.n_heads, a.fd_kvh);
  // workgroup -> kv head, split, column tile (the tiles with the most keys
  // first), layer.  Workgroup b runs on XCD b % 8: with 8 kv heads or a multiple
  // an XCD's L2 holds its own heads' rows only (300 tokens, head_dim 80, 32 heads:
  // 23.1 us with the column tile fastest, 19.2 so).
  const int bh = (int)fdiv(blockIdx.x, a.fd_kvh), kvh = blockIdx.x - bh * a.n_kv_heads;
  const int bs = (int)fdiv(bh, a.fd_split), split = bh - bs * a.n_split;
  const int li = (int)fdiv(bs, a.fd_tiles);
  const int tile = a.col_tiles - 1 - (bs - li * a.col_tiles);
  const int group = bs * a.n_kv_heads + kvh;
  const int cols = a.n_tokens * G;
  const int w0 = NC * tile;                                   // the workgroup's first column
  const int c0 = min(w0 + 16 * cw, cols - 1);                 // this wave's
  const int nc = min(16, cols - (w0 + 16 * cw));              // and how many (none: below 1)
  const int kmax =
      nc > 0 ? a.start_pos + (int)fdiv(c0 + nc - 1, a.fd_g) + 1 : 0;  // last column's keys
  const int t0 = split * a.split_len, te = min(t0 + a.split_len, kmax);
  const size_t layer_off = (size_t)(a.layer0 + li) * a.max_seq_len * kv_dim + (size_t)kvh * D;
  const uint16_t* kl = a.kc + layer_off;
  const uint16_t* vl = a.vc + layer_off;
  const bool own = ONE && t0 < te && te == kmax;  // appends row start_pos
  // rows this workgroup reads from the cache: below te, and below the new row
  const int rmax = max((ONE ? min(te, a.start_pos) : te) - 1, 0);

  // ---- loads: the new row's inputs, q, then the first tile --------------------
  const size_t nsrc = (size_t)li * kv_dim + (size_t)kvh * D;
  NewRow nr;
  if (own) nr.load(a, nsrc);
  // q: 16 lanes a column, rope pairs j, j + 16, ... of its token and head
  constexpr int QK = (DT + 1) / 2;
  const int qj = tid & 15;
  float x0[CW][QK], x1[CW][QK], qcos[CW][QK], qsin[CW][QK];
#pragma unroll
  for (int w = 0; w < CW; ++w) {
    const int qi = min(w0 + 16 * w + (tid >> 4), cols - 1), qtok = (int)fdiv(qi, a.fd_g);
    const float* qx = a.q + ((size_t)li * a.n_tokens + qtok) * a.n_heads * D +
                      (size_t)(kvh * G + qi - qtok * G) * D;
    const size_t qpos = (size_t)(a.start_pos + qtok) * (D / 2);
#pragma unroll
    for (int k = 0; k < QK; ++k) {
      const int i = min(qj + 16 * k, D / 2 - 1);
      int i0, i1;
      pair_of(a.rope_type, D, i, i0, i1);
      x0[w][k] = qx[i0], x1[w][k] = qx[i1];
      qcos[w][k] = a.cos_t[qpos + i], qsin[w][k] = a.sin_t[qpos + i];
    }
  }
  // a wave's tiles are 32 keys: rows t + c and t + 16 + c of each lane
  u32x4_t ka[DK], kb[DK], va[DK], vb[DK];
  auto load_rows = [&](const uint16_t* base, int t, u32x4_t(&r0)[DK], u32x4_t(&r1)[DK]) {
    load_row<DK, D8>(base + (size_t)max(min(t + c, rmax), 0) * kv_dim, D, g, r0);
    load_row<DK, D8>(base + (size_t)max(min(t + 16 + c, rmax), 0) * kv_dim, D, g, r1);
  };
  const int tw = t0 + 32 * ks;
  load_rows(kl, tw, ka, kb);
  load_rows(vl, tw, va, vb);
  _Float16* qs = (_Float16*)lds;
  const float fold = kLog2e / sqrtf((float)D);  // scores in log2 units
#pragma unroll
  for (int w = 0; w < CW; ++w) {
    float scale = 1.0f, ss = 0.0f;
    if (a.qn) {
#pragma unroll
      for (int k = 0; k < QK; ++k)
        if (qj + 16 * k < D / 2) ss += x0[w][k] * x0[w][k] + x1[w][k] * x1[w][k];
#pragma unroll
      for (int m = 1; m < 16; m *= 2) ss += __shfl_xor(ss, m);
      scale = 1.0f / sqrtf(ss / (float)D + a.norm_eps);
    }
    float amax = 0.0f;
#pragma unroll
    for (int k = 0; k < QK; ++k) {
      // lanes past the last pair repeat it (same values to the same place)
      float &y0 = x0[w][k], &y1 = x1[w][k];
      if (a.qn) {
        int i0, i1;
        pair_of(a.rope_type, D, min(qj + 16 * k, D / 2 - 1), i0, i1);
        y0 = (y0 * scale) * a.qn[(size_t)li * D + i0];
        y1 = (y1 * scale) * a.qn[(size_t)li * D + i1];
      }
      rope_rotate(y0, y1, qcos[w][k], qsin[w][k]);
      y0 *= fold, y1 *= fold;
      amax = vmax(amax, vmax(fabsf(y0), fabsf(y1)));
    }
#pragma unroll
    for (int m = 1; m < 16; m *= 2) amax = vmax(amax, __shfl_xor(amax, m));
    // the column by a power of two to [2^13, 2^14): its three parts keep all 24
    // bits of elements down to 2^-36 of the largest; 2^up goes to the scores
    const int ex = max((int)((__float_as_uint(amax) >> 23) & 0xFFu) - 127, -100);
    const float down = __uint_as_float((uint32_t)(127 + 13 - ex) << 23);
    if (qj == 0) ups[16 * w + (tid >> 4)] = __uint_as_float((uint32_t)(127 + ex - 13) << 23);
    _Float16* qrow = qs + w * Sh::kQ + (tid >> 4) * Sh::QP;
#pragma unroll
    for (int k = 0; k < QK; ++k) {
      int i0, i1;
      pair_of(a.rope_type, D, min(qj + 16 * k, D / 2 - 1), i0, i1);
      half2_t hi, mid, lo;
      split3<true>(x0[w][k] * down, x1[w][k] * down, hi, mid, lo);
      qrow[i0] = hi[0], qrow[i1] = hi[1];
      qrow[16 * Sh::QP + i0] = mid[0], qrow[16 * Sh::QP + i1] = mid[1];
      qrow[32 * Sh::QP + i0] = lo[0], qrow[32 * Sh::QP + i1] = lo[1];
    }
    for (int d = D + qj; d < 32 * DK; d += 16)
      qrow[d] = qrow[16 * Sh::QP + d] = qrow[32 * Sh::QP + d] = (_Float16)0.0f;
  }
  if (own) nr.finish(a, nsrc, li, knew, vnew, kr, sq, red);
  __syncthreads();
  if (own && tile == 0) {  // G > 16: the first column tile's workgroup stores it
    const size_t dst = layer_off + (size_t)a.start_pos * kv_dim;
    for (int i = tid; i < D; i += kGThreads) {
      a.kc[dst + i] = knew[i];
      a.vc[dst + i] = vnew[i];
      if (a.k_rows) {
        a.k_rows[nsrc + i] = knew[i];
        a.v_rows[nsrc + i] = vnew[i];
      }
    }
  }
  // the last key of column c and of the first column
  const int lim = a.start_pos + (int)fdiv(c0 + max(min(c, nc - 1), 0), a.fd_g);
  const int lim0 = a.start_pos + (int)fdiv(c0, a.fd_g);
  const float up = ups[16 * cw + c];
  qs += cw * Sh::kQ;

  // ---- the tiles ---------------------------------------------------------------
  // Fast: fp16 MFMAs over the three parts of q and of P.  The wave takes its
  // tiles again as fp32 products that skip masked keys, which is what the rows'
  // own values give, where
  // - an infinity or a NaN among the rows made a result infinite or NaN (inf
  //   times a zero part), or
  // - some weight was below 2^-36 of the largest (the parts stop at 2^-60 of it)
  //   and a column's result is so small that its bits could count: all of it
  //   below 2^-16 of the largest weight, the heavier keys' V zero or nearly.
  _Float16* vt = (_Float16*)lds + CW * Sh::kQ + wave * 32 * Sh::VP;
  float4_t o[DT];
  float m, l;
  bool lost = false;
  for (int slow = 0; slow < 2; ++slow) {
#pragma unroll
    for (int j = 0; j < DT; ++j) o[j] = float4_t{0.f, 0.f, 0.f, 0.f};
    m = kNegBig, l = 0.0f;
    if (slow) {
      load_rows(kl, tw, ka, kb);
      load_rows(vl, tw, va, vb);
    }
    for (int t = tw; t < te; t += 32 * KS) {
      if (own && t + 31 >= a.start_pos) {
        if (t + c == a.start_pos) {
          load_row<DK, D8>(knew, D, g, ka);
          load_row<DK, D8>(vnew, D, g, va);
        }
        if (t + 16 + c == a.start_pos) {
          load_row<DK, D8>(knew, D, g, kb);
          load_row<DK, D8>(vnew, D, g, vb);
        }
      }
      // V rows into the wave's tile (padding columns: whatever, not stored later)
#pragma unroll
      for (int j = 0; j < DK; ++j) {
        *(u32x4_t*)(vt + c * Sh::VP + 32 * j + 8 * g) = va[j];
        *(u32x4_t*)(vt + (16 + c) * Sh::VP + 32 * j + 8 * g) = vb[j];
      }
      // rows past the range re-read its last one (not used)
      load_rows(vl, t + 32 * KS, va, vb);
      clear_past<DK>(D, g, ka);
      clear_past<DK>(D, g, kb);
      // S = K q^T: keys 16 h + 4 g + v of column c
      float4_t s[2] = {};
      if (!slow) {
#pragma unroll
        for (int part = 2; part >= 0; --part) {
          if (part < 2) s[0] = s[0] * kPartDown, s[1] = s[1] * kPartDown;
#pragma unroll
          for (int j = 0; j < DK; ++j) {
            const half8_t qf =
                *(const half8_t*)(qs + (16 * part + c) * Sh::QP + 32 * j + 8 * g);
            s[0] = mfma16x16x32(__builtin_bit_cast(half8_t, ka[j]), qf, s[0]);
            s[1] = mfma16x16x32(__builtin_bit_cast(half8_t, kb[j]), qf, s[1]);
          }
        }
      } else {
#pragma unroll
        for (int j = 0; j < DK; ++j) {
          const _Float16* qp = qs + c * Sh::QP + 32 * j + 8 * g;
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const float q =
                (float)qp[e] + ((float)qp[16 * Sh::QP + e] +
                                (float)qp[32 * Sh::QP + e] * kPartDown) * kPartDown;
            s[0] = mfma_f32((float)__builtin_bit_cast(half8_t, ka[j])[e], q, s[0]);
            s[1] = mfma_f32((float)__builtin_bit_cast(half8_t, kb[j])[e], q, s[1]);
          }
        }
      }
      load_rows(kl, t + 32 * KS, ka, kb);
      float p[8];
      float mx = kNegBig, least = -kNegBig;  // least: masked keys' too
      const bool cross = t + 31 > lim0;  // uniform: some key is past some column's last
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        p[i] = s[i / 4][i % 4] * up;
        least = vmin(least, p[i]);
        if (cross && t + 16 * (i / 4) + 4 * g + i % 4 > lim) p[i] = kNegBig;
      }
      mx = vmax(vmax(vmax(p[0], p[1]), vmax(p[2], p[3])), vmax(vmax(p[4], p[5]), vmax(p[6], p[7])));
      const float mn = vmax(m, max_xor32(max_xor16(mx)));
      if (__any(!(mn <= m))) {
        const float corr = fast_exp2(m - mn);
        l *= corr;
#pragma unroll
        for (int j = 0; j < DT; ++j) o[j] = o[j] * corr;
        m = mn;
      }
      // weights times 2^14 (the sums too): their parts keep all 24 bits of
      // weights down to 2^-25, the deeper ones (more VALU work) down to 2^-36
      const bool deep = __any(least < m - 25.0f);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        p[i] = fast_exp2(p[i] - m) * 16384.0f;
        if (cross && t + 16 * (i / 4) + 4 * g + i % 4 > lim) p[i] = 0.0f;
      }
      l += ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
      __builtin_amdgcn_wave_barrier();
      auto pv = [&](auto deeper) {  // O^T += V^T P^T
        constexpr bool DEEP = decltype(deeper)::value;
        half2_t ph[4], pm[4], pl[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) split3<DEEP>(p[2 * i], p[2 * i + 1], ph[i], pm[i], pl[i]);
        auto cat = [](const half2_t (&x)[4]) {
          return half8_t{x[0][0], x[0][1], x[1][0], x[1][1], x[2][0], x[2][1], x[3][0], x[3][1]};
        };
        const half8_t bh = cat(ph), bm = cat(pm), bl = cat(pl);
        // keys 4 g + v and 16 + 4 g + v of 16 d's: the order of P's registers
        const _Float16* vr = vt + (4 * g + (c >> 2)) * Sh::VP + 4 * (c & 3);
        constexpr int H = 3;  // d tiles whose V operands are in registers together
#pragma unroll
        for (int j0 = 0; j0 < DT; j0 += H) {
          half8_t vv[H];
#pragma unroll
          for (int j = j0; j < j0 + H && j < DT; ++j) {
            const half4_t v0 = lds_read_tr4(vr + 16 * j);
            const half4_t v1 = lds_read_tr4(vr + 16 * Sh::VP + 16 * j);
            vv[j - j0] = __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7);
          }
#pragma unroll
          for (int j = j0; j < j0 + H && j < DT; ++j) {
            float4_t x = {0.f, 0.f, 0.f, 0.f};
            x = mfma16x16x32(vv[j - j0], bl, x);
            if constexpr (DEEP) x = x * kPartDown;
            x = mfma16x16x32(vv[j - j0], bm, x);
            x = mfma16x16x32(vv[j - j0], bh, x * kPartDown);
            o[j] = o[j] + x;
          }
          asm volatile("" ::: "memory");
        }
      };
      if (!slow && !deep) {
        pv(std::false_type{});
      } else if (!slow) {
        lost |= __any(least < m - 36.0f);
        pv(std::true_type{});
      } else {
#pragma unroll 1
        for (int key = 0; key < 32; ++key) {
          const int from = c + 16 * (key % 16 / 4);
          float w = 0.0f;
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            const float xa = __shfl(p[v], from), xb = __shfl(p[4 + v], from);
            if (key % 4 == v) w = key < 16 ? xa : xb;
          }
          if (t + key > lim) continue;
#pragma unroll
          for (int j = 0; j < DT; ++j)
#pragma unroll
            for (int v = 0; v < 4; ++v)
              o[j][v] = __builtin_fmaf(w, (float)vt[key * Sh::VP + 16 * j + 4 * g + v], o[j][v]);
        }
      }
      __builtin_amdgcn_wave_barrier();
    }
    if (slow) break;
    // infinite or NaN if any result is (d past D: not looked at)
    float4_t sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < DT; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v)
        if (16 * j + 16 <= D || 16 * j + 4 * g + v < D) sum[v] += fabsf(o[j][v]);
    const float os = (sum[0] + sum[1]) + (sum[2] + sum[3]);
    if (__any(!(l + os <= 3.4028235e38f))) continue;
    if (!lost) break;
    const float lc = add_xor32(add_xor16(l)), oc = add_xor32(add_xor16(os));
    if (!__any(c < nc && lc > 0.0f && oc < 0.25f)) break;  // 2^-16 times 2^14
  }
  l = add_xor32(add_xor16(l));

  const size_t row0 = (size_t)li * a.n_tokens;
  auto out_at = [&](int ci) {  // the output row of column ci
    const int tok = (int)fdiv(ci, a.fd_g);
    return a.out + (row0 + tok) * a.out_stride + (size_t)(kvh * G + ci - tok * G) * D;
  };
  // ---- the waves' results together: each scaled to the column's maximum, then
  // summed four elements at a time ---------------------------------------------
  float* ml = lds + 4 * 16 * Sh::OP;  // [wave][max, sum][column]
  __syncthreads();                    // q and the V tiles are dead
  if (g == 0) ml[wave * 32 + c] = m;
  __syncthreads();
  float M = kNegBig;
#pragma unroll
  for (int w = 0; w < KS; ++w) M = fmaxf(M, ml[(cw * KS + w) * 32 + c]);
  const float e = fast_exp2(m - M);
  if (g == 0) ml[wave * 32 + 16 + c] = l * e;
  float* ow = lds + (wave * 16 + c) * Sh::OP + 4 * g;
#pragma unroll
  for (int j = 0; j < DT; ++j) *(float4_t*)(ow + 16 * j) = o[j] * e;
  __syncthreads();
  const int wcols = min(NC, cols - w0);
  for (int idx = tid; idx < wcols * (Sh::DP / 4); idx += kGThreads) {
    const int col = idx / (Sh::DP / 4), d = 4 * (idx % (Sh::DP / 4));
    const int w1 = col / 16 * KS, cc = col % 16;  // the column's first wave
    float4_t O = {0.f, 0.f, 0.f, 0.f};
    float L = 0.0f, mx = kNegBig;
#pragma unroll
    for (int w = 0; w < KS; ++w) {
      O = O + *(const float4_t*)(lds + ((w1 + w) * 16 + cc) * Sh::OP + d);
      mx = fmaxf(mx, ml[(w1 + w) * 32 + cc]);
      L += ml[(w1 + w) * 32 + 16 + cc];
    }
    if (a.n_split == 1) {
      float* ot = out_at(w0 + col) + d;
      const float inv = 1.0f / L;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (d + i < D) ot[i] = O[i] * inv;
    } else {  // KS 4: one column tile
      const __amdgpu_buffer_rsrc_t prs = __builtin_amdgcn_make_buffer_rsrc(
          a.part + ((size_t)group * a.n_split + split) * Sh::kPart, 0, Sh::kPart * 4, 0x00020000);
      __builtin_amdgcn_raw_buffer_store_b128(O, prs, (col * Sh::DP + d) * 4, 0, kDeviceScope);
      if (d == 0) {
        const int at = (16 * Sh::DP + 2 * col) * 4;
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(mx), prs, at, 0, kDeviceScope);
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(L), prs, at + 4, 0, kDeviceScope);
      }
    }
  }
  if (KS != 4 || a.n_split == 1) return;
  // ---- the group's last split to finish merges: the partials' device-scope
  // stores are complete before the count goes up; it resets the count -------
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  unsigned* ctr = a.ctr + group * kGCtrPitch;
  if (tid == 0)
    s_last = __hip_atomic_fetch_add(ctr, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
             (unsigned)(a.n_split - 1);
  __syncthreads();
  if (!s_last) return;
  if (tid == 0) __hip_atomic_store(ctr, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const __amdgpu_buffer_rsrc_t grs = __builtin_amdgcn_make_buffer_rsrc(
      a.part + (size_t)group * a.n_split * Sh::kPart, 0, a.n_split * Sh::kPart * 4, 0x00020000);
  for (int idx = tid; idx < wcols * (Sh::DP / 4); idx += kGThreads) {
    const int col = idx / (Sh::DP / 4), d = 4 * (idx % (Sh::DP / 4));
    float Mg = kNegBig, L = 0.0f;
    float4_t O = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
    for (int s0 = 0; s0 < a.n_split; s0 += 8) {
      float4_t oi[8];
      float mi[8], lw[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        // splits past the last re-read it (not used)
        const int u = min(s0 + i, a.n_split - 1) * Sh::kPart;
        const int at = (u + 16 * Sh::DP + 2 * col) * 4;
        oi[i] = __builtin_amdgcn_raw_buffer_load_b128(grs, (u + col * Sh::DP + d) * 4, 0,
                                                      kDeviceScope);
        mi[i] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(grs, at, 0, kDeviceScope));
        lw[i] =
            __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(grs, at + 4, 0, kDeviceScope));
      }
      float Mn = Mg;
#pragma unroll
      for (int i = 0; i < 8; ++i) Mn = fmaxf(Mn, mi[i]);
      const float r = fast_exp2(Mg - Mn);
      L *= r;
      O = O * r;
#pragma unroll
      for (int i = 0; i < 8; ++i)
        if (s0 + i < a.n_split) {
          const float w = fast_exp2(mi[i] - Mn);
          L += lw[i] * w;
          O = O + oi[i] * w;
        }
      Mg = Mn;
    }
    float* ot = out_at(w0 + col) + d;
    const float inv = 1.0f / L;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (d + i < D) ot[i] = O[i] * inv;
  }
}

// Maximum (MAX) or sum of v over the workgroup; every thread gets it.
template <bool MAX>
__device__ __forceinline__ float block_reduce(float v, float* wred) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const float w = __shfl_xor(v, o);
    v = MAX ? fmaxf(v, w) : v + w;
  }
  __syncthreads();  // the previous reduction's readers are done with wred
  if ((threadIdx.x & 63) == 0) wred[threadIdx.x >> 6] = v;
  __syncthreads();
  float r = wred[0];
#pragma unroll
  for (int i = 1; i < kGThreads / 64; ++i) r = MAX ? fmaxf(r, wred[i]) : r + wred[i];
  return r;
}

// dot(q, k row) over D elements (q in LDS, the row fp16 bits in HBM): 16-byte
// loads when D is a multiple of 8 (every row offset then is too), 4-byte ones
// otherwise (D is even); four partial sums.
__device__ __forceinline__ float row_dot(const float* qs, const uint16_t* kr, int D) {
  float d4[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  if (D % 8 == 0) {
    const uint4* kp = (const uint4*)kr;
    const int nw = D / 8;
    for (int j = 0; j < nw; j += 4) {  // four 16-byte loads issued together
      uint4 w[4];
#pragma unroll
      for (int b = 0; b < 4; ++b) w[b] = j + b < nw ? kp[j + b] : make_uint4(0u, 0u, 0u, 0u);
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        const uint32_t ws[4] = {w[b].x, w[b].y, w[b].z, w[b].w};
        const float* qq = qs + 8 * (j + b);
        if (j + b < nw) {
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            d4[u] = d4[u] + qq[2 * u] * f16_bits_to_f32((uint16_t)(ws[u] & 0xFFFFu));
            d4[u] = d4[u] + qq[2 * u + 1] * f16_bits_to_f32((uint16_t)(ws[u] >> 16));
          }
        }
      }
    }
  } else {
    const uint32_t* kp = (const uint32_t*)kr;
    for (int j = 0; j < D / 2; ++j) {
      const uint32_t w = kp[j];
      float& d = d4[j & 3];
      d = d + qs[2 * j] * f16_bits_to_f32((uint16_t)(w & 0xFFFFu));
      d = d + qs[2 * j + 1] * f16_bits_to_f32((uint16_t)(w >> 16));
    }
  }
  return (d4[0] + d4[1]) + (d4[2] + d4[3]);
}

// Few keys of a wide head (few_keys): one workgroup per (layer, token, q head) on
// the VALU, after the append.  The positions in chunks of 256, one per thread:
// scores, the chunk's maximum, exp weights and the rescaled sums of the online
// softmax, v accumulated by one thread per d.
__global__ __launch_bounds__(kGThreads) void generic_rows_kernel(GenericArgs a) {
  __shared__ float qs[kGMaxD];
  __shared__ float ps[kGChunk];
  __shared__ __align__(16) float sq[kGSq];
  __shared__ float red[8];
  __shared__ float wred[kGThreads / 64];
  const int tid = threadIdx.x;
  const int D = a.D, kv_dim = a.n_kv_heads * D, G = a.n_heads / a.n_kv_heads;
  const int h = blockIdx.x % a.n_heads;
  const int t = (blockIdx.x / a.n_heads) % a.n_tokens;
  const int li = blockIdx.x / (a.n_heads * a.n_tokens);
  const int pos = a.start_pos + t, kvh = h / G;
  const size_t row = (size_t)li * a.n_tokens + t;
  load_normed(a.q + row * a.n_heads * D + (size_t)h * D, a.qn ? a.qn + (size_t)li * D : nullptr,
              D, a.norm_eps, qs, sq, red);
  const float* cr = a.cos_t + (size_t)pos * (D / 2);
  const float* sr = a.sin_t + (size_t)pos * (D / 2);
  for (int i = tid; i < D / 2; i += kGThreads) {
    int i0, i1;
    pair_of(a.rope_type, D, i, i0, i1);
    float x0 = qs[i0], x1 = qs[i1];
    rope_rotate(x0, x1, cr[i], sr[i]);
    qs[i0] = x0;
    qs[i1] = x1;
  }
  __syncthreads();
  const size_t layer_off = (size_t)(a.layer0 + li) * a.max_seq_len * kv_dim + (size_t)kvh * D;
  const uint16_t* kl = a.kc + layer_off;
  const uint16_t* vl = a.vc + layer_off;
  const float root = sqrtf((float)D);
  float m = kNegBig, l = 0.0f, acc = 0.0f;  // acc: element d = tid of the output
  for (int c0 = 0; c0 <= pos; c0 += kGChunk) {
    const int p = c0 + tid;
    float s = kNegBig;
    if (p <= pos) s = row_dot(qs, kl + (size_t)p * kv_dim, D) / root;
    const float mn = fmaxf(m, block_reduce<true>(s, wred));
    const float e = p <= pos ? expf(s - mn) : 0.0f;
    ps[tid] = e;
    const float esum = block_reduce<false>(e, wred);  // its barriers publish ps
    const float corr = expf(m - mn);
    l = l * corr + esum;
    if (tid < D) {
      const int np = min(kGChunk, pos + 1 - c0);
      const uint16_t* vp = vl + (size_t)c0 * kv_dim + tid;
      // eight v loads in flight, four independent partial sums
      float s4[4] = {0.0f, 0.0f, 0.0f, 0.0f};
      int j = 0;
      for (; j + 8 <= np; j += 8) {
        uint16_t vb[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) vb[u] = vp[(size_t)(j + u) * kv_dim];
#pragma unroll
        for (int u = 0; u < 8; ++u) s4[u & 3] = s4[u & 3] + ps[j + u] * f16_bits_to_f32(vb[u]);
      }
      for (; j < np; ++j) s4[0] = s4[0] + ps[j] * f16_bits_to_f32(vp[(size_t)j * kv_dim]);
      acc = acc * corr + ((s4[0] + s4[1]) + (s4[2] + s4[3]));
    }
    m = mn;
    __syncthreads();  // ps is rewritten by the next chunk
  }
  if (tid < D) a.out[row * a.out_stride + (size_t)h * D + tid] = acc / l;
}

// d tiles for which two column tiles a workgroup are built (from 10 on, 77 KB and
// more of LDS, a second workgroup would no longer fit a CU).
constexpr bool two_tiles(int dt) { return dt > 4 && dt <= 8; }

// 16-wide tiles of d that head_dim runs on: the next built number.
int built_tiles(int head_dim) {
  const int t = (head_dim + 15) / 16;
  return t <= 6 ? t : t <= 8 ? 8 : t <= 10 ? 10 : t <= 12 ? 12 : 16;
}

// Whether generic_rows_kernel is the faster one: few keys at head dims whose
// tiles a CU holds once (10 d tiles and more; 4-byte loads from 5 on).  There a
// launch costs 10 to 12 us however few the keys, and as much again where the
// tiles exceed the CUs (head_dim 160, 12 layers of 32 kv heads, 64 q heads, 1 key:
// 15.5 us, 10.9 here; 85 keys and 128 q heads 16.7, 25.6).  us, tiles / rows:
// head_dim 256, one token of up to 256 heads, 1.10 in the median to 32 keys, 1.03 to
// 64; prompts of 2 to 8 tokens 1.25 to 16 keys, 1.15 to 192; 192 from 2 tokens on
// 1.1 to 32 keys; 100 (4-byte loads) 1.1 to 192; 160 1.05 to 16.
bool few_keys(int n_layers, int n_heads, int n_kv_heads, int head_dim, int start_pos,
              int n_tokens, int cus) {
  const int dt = built_tiles(head_dim), keys = start_pos + n_tokens;
  if (dt < 10 && (head_dim % 8 == 0 || dt < 5)) return false;
  const long rows = (long)n_layers * n_tokens * n_heads;
  const long cols = (long)n_tokens * (n_heads / n_kv_heads);
  if ((long)n_layers * n_kv_heads * ((cols + 15) / 16) > cus)
    return rows <= 6L * cus && rows * keys <= (dt >= 12 ? 256L : 128L) * cus;
  if (n_tokens == 1) return dt == 16 && keys <= 64 && rows <= cus;
  if (rows <= cus && keys <= 192 && (dt == 16 || dt < 10)) return true;
  return keys <= (dt == 16 ? 128 : dt == 12 ? 32 : 16) && rows <= (dt >= 12 ? 4L : 1L) * cus;
}

template <int DT, int KS, bool ONE>
void launch_attn_ks(const GenericArgs& a, unsigned grid, hipStream_t st) {
  constexpr size_t lds = sizeof(float) * GShape<DT, KS>::kFloats;
  // 16-byte loads where every row starts on 16 bytes
  if (a.D % 8 == 0 && ((uintptr_t)a.kc | (uintptr_t)a.vc) % 16 == 0)
    hipLaunchKernelGGL((generic_attn_kernel<DT, KS, true, ONE>), dim3(grid), dim3(kGThreads), lds,
                       st, a);
  else
    hipLaunchKernelGGL((generic_attn_kernel<DT, KS, false, ONE>), dim3(grid), dim3(kGThreads), lds,
                       st, a);
}
template <int DT>
void launch_attn(const GenericArgs& a, bool one, int ks, unsigned grid, hipStream_t st) {
  if (one) return launch_attn_ks<DT, 4, true>(a, grid, st);
  if constexpr (two_tiles(DT)) {
    if (ks == 2) return launch_attn_ks<DT, 2, false>(a, grid, st);
  }
  launch_attn_ks<DT, 4, false>(a, grid, st);
}

void launch_attn(const GenericArgs& a, bool one, int ks, unsigned grid, hipStream_t st) {
  switch (built_tiles(a.D)) {
    case 1: launch_attn<1>(a, one, ks, grid, st); break;
    case 2: launch_attn<2>(a, one, ks, grid, st); break;
    case 3: launch_attn<3>(a, one, ks, grid, st); break;
    case 4: launch_attn<4>(a, one, ks, grid, st); break;
    case 5: launch_attn<5>(a, one, ks, grid, st); break;
    case 6: launch_attn<6>(a, one, ks, grid, st); break;
    case 8: launch_attn<8>(a, one, ks, grid, st); break;
    case 10: launch_attn<10>(a, one, ks, grid, st); break;
    case 12: launch_attn<12>(a, one, ks, grid, st); break;
    default: launch_attn<16>(a, one, ks, grid, st); break;
  }
}

}  // namespace

int attn_generic(int n_heads, int n_kv_heads, int head_dim, int max_seq_len, int rope_type,
                 int layer0, int n_launch_layers, int start_pos, int n_tokens, const float* q,
                 const float* k, const float* v, uint16_t* key_cache, uint16_t* val_cache,
                 const float* rope_cos, const float* rope_sin, float* out, int out_stride,
                 const float* q_norm, const float* k_norm, float norm_eps, uint16_t* k_rows,
                 uint16_t* v_rows, bool append) {
  if (head_dim < 2 || head_dim > kGMaxD || head_dim % 2) {
    set_error("attention: head_dim %d must be even and at most %d", head_dim, kGMaxD);
    return -1;
  }
  if (n_tokens == 0) return 0;
  // A launch holds at most 2^32 - 1 threads.  First: the counts below are ints.
  const long max_wg = 0xFFFFFFFFL / kGThreads;
  if ((long)n_tokens * n_heads > max_wg) {
    set_error("attention: %d tokens x %d heads exceed one launch's %ld workgroups", n_tokens,
              n_heads, max_wg);
    return -1;
  }
  GenericArgs a{};
  a.q = q, a.k = k, a.v = v, a.kc = key_cache, a.vc = val_cache;
  a.cos_t = rope_cos, a.sin_t = rope_sin, a.out = out;
  a.qn = q_norm, a.kn = k_norm, a.norm_eps = norm_eps;
  a.k_rows = k_rows, a.v_rows = v_rows;
  a.layer0 = layer0, a.n_launch_layers = n_launch_layers, a.n_heads = n_heads;
  a.n_kv_heads = n_kv_heads, a.D = head_dim, a.max_seq_len = max_seq_len;
  a.rope_type = rope_type, a.start_pos = start_pos, a.n_tokens = n_tokens;
  a.out_stride = out_stride;
  // Keys split over several workgroups where the launch would fill less than
  // one per CU (head_dim 80, 32 heads, pos 1499, us a layer for 128 / 256 / 384 /
  // 512 workgroups: 15.5 / 11.3 / 13.5 / 12.6), as far as every wave keeps a
  // tile, the partials fit the static scratch and the merges its counters.  Up to
  // 256 keys, two tiles a wave, the merge costs more than the second tile where
  // two workgroups share a CU (129 to 256 keys in two splits: 1.09 times as long in
  // the median of 480 prompt launches, 1.22 from 128 groups on, 1.02 for single
  // tokens; 257 to 384 keys 0.93), the second tile more in the wider forms (head_dim
  // 224 and 256 0.85, 100 0.86).
  const int G = n_heads / n_kv_heads, cus = ctx().num_cus > 0 ? ctx().num_cus : 256;
  const bool rows = few_keys(n_launch_layers, n_heads, n_kv_heads, head_dim, start_pos,
                             n_tokens, cus);
  const bool one = append && n_tokens == 1 && !rows;
  const int dt = built_tiles(head_dim), kmax = start_pos + n_tokens;
  const long tiles = (long)n_kv_heads * ((n_tokens * G + 15) / 16) * n_launch_layers;
  // Two column tiles a workgroup halve its fixed chain per column but give a
  // wave twice the tiles: faster with many workgroups and few keys (32 q and 8
  // kv heads, 8 layers in a launch, KS 2 / 4, us: head_dim 96, 128 tokens 26.2 /
  // 28.2, 300 64.8 / 69.2, 500 130 / 138, head_dim 112, 300 tokens 85.7 / 100.4; one
  // layer of 300 tokens 16.8 / 15.6, of 1500 116 / 115).  Up to head_dim 64 both
  // take the same.
  const int ks = !one && two_tiles(dt) && tiles >= 4L * cus && kmax <= 512 ? 2 : 4;
  a.col_tiles = (n_tokens * G + 64 / ks - 1) / (64 / ks);
  const long groups_layer = (long)n_kv_heads * a.col_tiles;
  unsigned* ctr = nullptr;
  float* part = nullptr;
  size_t part_bytes = 0;
  decode_scratch(&ctr, &part, &part_bytes);
  const bool paired = dt <= 8 && head_dim % 8 == 0;  // two workgroups a CU
  long want = (cus - 1 + groups_layer * n_launch_layers) / (groups_layer * n_launch_layers);
  if (ks != 4) want = 1;
  want = std::min<long>({want, paired && kmax <= 256 ? 1 : (kmax + 127) / 128, kGMaxSplit});
  a.split_len = ((kmax + (int)want - 1) / (int)want + 31) / 32 * 32;
  a.n_split = (kmax + a.split_len - 1) / a.split_len;
  const long groups = groups_layer * n_launch_layers;
  if (groups * kGCtrPitch > kDecodeCounters ||
      (size_t)groups * a.n_split * 16 * (16 * dt + 2) * sizeof(float) > part_bytes) {
    a.n_split = 1;
    a.split_len = (kmax + 31) / 32 * 32;
  }
  a.ctr = ctr, a.part = part;
  a.n_chunk = (n_kv_heads * (head_dim / 2) + kGThreads - 1) / kGThreads;
  a.fd_chunk = make_fastdiv((uint32_t)a.n_chunk);
  a.fd_tok = make_fastdiv((uint32_t)n_tokens);
  a.fd_half = make_fastdiv((uint32_t)head_dim / 2);
  a.fd_split = make_fastdiv((uint32_t)a.n_split);
  a.fd_tiles = make_fastdiv((uint32_t)a.col_tiles);
  a.fd_kvh = make_fastdiv((uint32_t)n_kv_heads);
  a.fd_g = make_fastdiv((uint32_t)G);
  // Layers go in as many launches as that takes (each is independent); one
  // fits: n_split is 1 unless the launch has fewer groups than CUs.
  const long per_layer =
      rows ? (long)n_tokens * n_heads
           : std::max<long>(groups_layer * a.n_split, (long)n_tokens * n_kv_heads);
  const int step = (int)std::min<long>(n_launch_layers, max_wg / per_layer);
  const size_t q_dim = (size_t)n_heads * head_dim, kv_dim = (size_t)n_kv_heads * head_dim;
  hipStream_t st = ctx().stream;
  for (int l = 0; l < n_launch_layers; l += step) {
    GenericArgs b = a;
    const size_t rows_before = (size_t)l * n_tokens;
    b.layer0 = layer0 + l;
    b.n_launch_layers = std::min(step, n_launch_layers - l);
    b.q = q + rows_before * q_dim;
    b.k = k + rows_before * kv_dim;
    b.v = v + rows_before * kv_dim;
    b.out = out + rows_before * out_stride;
    if (q_norm) b.qn = q_norm + (size_t)l * head_dim;
    if (k_norm) b.kn = k_norm + (size_t)l * head_dim;
    if (k_rows) b.k_rows = k_rows + rows_before * kv_dim;
    if (v_rows) b.v_rows = v_rows + rows_before * kv_dim;
    const long nl = b.n_launch_layers;
    if (append && !one) {
      const long kv_rows = nl * n_tokens * n_kv_heads;
      // a token's few rows: a workgroup each (head_dim 256, 32 heads, with the
      // attention: 10.9 us with a thread per rope pair, 9.6 so)
      if (b.kn || n_tokens == 1)
        hipLaunchKernelGGL(generic_append_rows_kernel, dim3((unsigned)kv_rows), dim3(kGThreads), 0,
                           st, b);
      else
        hipLaunchKernelGGL(generic_append_kernel, dim3((unsigned)(nl * n_tokens * a.n_chunk)),
                           dim3(kGThreads), 0, st, b);
      if (check_hip(hipGetLastError(), "generic_append_kernel")) return -1;
    }
    if (rows)
      hipLaunchKernelGGL(generic_rows_kernel, dim3((unsigned)(nl * per_layer)), dim3(kGThreads), 0,
                         st, b);
    else
      launch_attn(b, one, ks, (unsigned)(nl * groups_layer * a.n_split), st);
    if (check_hip(hipGetLastError(), "generic_attn_kernel")) return -1;
  }
  return 0;
}

}  // namespace plh
