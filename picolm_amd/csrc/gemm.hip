// gemm.hip -- the batched GEMV (matmul_batch, tensor.c:322-366) on the fp32
// matrix cores, bit-identical to the single-vector kernel's exact order.
//
// The reference's dot products keep eight running sums per block (one per
// AVX2 lane), each a chain of fused multiply-adds over the block's elements
// 8s + j, and add the eight as hsum_avx2 does.  v_mfma_f32_16x16x4_f32 is
// four such steps for 16 tokens x 16 rows at once: its K index is a chain of
// correctly rounded fused multiply-adds in increasing k, subnormals kept
// (checked on the device against fmaf on 0.5 M results per value range), so
// with k = s one instruction per j forms a Q4_K sub-block's running sum j
// from zero.  v_mfma_f32_16x16x1_4b_f32 (four independent 16 x 16 tiles, one
// step each) forms four of a Q6_K group's running sums in two steps, or the
// four rounded products of a Q8_0 block's lane.  A weight is then converted
// to fp32 once per 16 tokens instead of once per token, and only the
// adds between the running sums, the scales and the block chain stay on the
// VALU.
//
// What bounds it: the fp32 MFMA and the VALU share one pipe (measured: a
// 16x16x4 takes 32 cycles, and VALU instructions between them add their 4
// cycles each), so a 16 x 16 tile of a 64-element Q4_K unit costs 16 x 32
// MFMA cycles + ~120 x 4 VALU cycles (88 of them the exact order's own adds
// and products).  TinyLlama's 128-token prompt, us a launch before (the VALU
// kernel) and now: gate/up pair (5632 x 2048 Q4_K twice) 340 -> 93, down (2048 x
// 5632 Q6_K) 287 -> 76, o 70 -> 26, q, k and v 102 in three launches -> 34 in
// one; the whole prompt 18.1 -> 5.5 ms.  Set aside: x straight from the caches
// instead of LDS (Q4_K 11264 x 2048, 128 tokens: 136 us against 96, Q6_K 387
// against 130: the vector memory path handles the 16 tokens' lines one by
// one); two token tiles a wave (88 against 94 us on that shape, slower below it).
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "gemv_formats.h"
#include "plh_internal.h"

using namespace plh;

namespace {

constexpr int kMT = 16;         // tokens and rows of one MFMA tile
constexpr int kSubPitch = 36;   // staged floats per 32 elements of x (4 of padding)

// x is staged in chunks: a unit per wave of 8 (512 elements), else 256, or 128
// where the exchanged terms (KW 2) would otherwise take the LDS of a second
// workgroup.  Staged floats per
// token: a pitch of 4 mod 16 floats, so that 16 tokens' 16-byte reads hit
// different banks.
constexpr int waves_of(int kw) { return kw == 8 ? 8 : 4; }  // of a workgroup
template <int KW>
struct Chunk {
  static constexpr int K = KW == 8 ? 512 : KW == 2 ? 128 : 256, U = K / 64;
  static constexpr int kTokPitch = K / 32 * kSubPitch + 4;
  static constexpr int kXs = kMT * kTokPitch;   // floats of a buffer
  static constexpr int kSums = K / 32 * kMT;    // its sub-block sums [sub][token]
};

__device__ __forceinline__ float4_t mfma_f32_k4(float a, float b) {
  const float4_t z = {0.f, 0.f, 0.f, 0.f};
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, z, 0, 0, 0);
}
__device__ __forceinline__ f32x16_t mfma_f32_4b(float a, float b, f32x16_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x1f32(a, b, c, 0, 0, 0);
}

// Byte b of a word as a float (plain C, so that the compiler sees every
// operand the MFMAs read): v_cvt_f32_ubyte0..3.
__device__ __forceinline__ float byte_f(uint32_t w, int b) {
  return (float)((w >> (8 * b)) & 0xFFu);
}

// Keeps a masked word whole: without it the compiler extracts every nibble
// with its own shift and mask instead of converting the word's bytes.
__device__ __forceinline__ uint32_t whole(uint32_t w) {
  asm("" : "+v"(w));
  return w;
}

// 16 consecutive elements of x: one thread's share of a staged chunk, or a
// lane's operand of one unit (64 elements) and token tile.
struct XV {
  float4_t f[4];
};

__device__ __forceinline__ float4_t ld4v(const float* p) { return *(const float4_t*)p; }

// Makes the MFMAs that read x wait for v: without it the compiler starts
// every tile of a chunk at once and runs out of registers.
__device__ __forceinline__ void after(XV& x, float4_t& v) {
  asm("" : "+v"(x.f[0]), "+v"(x.f[1]), "+v"(x.f[2]), "+v"(x.f[3]), "+v"(v));
}

// The formats.  Lane l = 16 s + c of a wave holds weight row c of the tile and
// token c, the k = s (or tile s) operands; results are tokens 4 s .. 4 s + 3 of
// row c.  Raw, load: the packed weights of one unit; W, weights: its fp32
// operands and block scales; stage: 16 elements of x as the lanes read them;
// load_x: a lane's operand, xt the staged unit of its token; terms: the unit's
// kUnitTerms chained terms, sums the sub-block sums of x (kSums) at token 4 s
// of the unit's first sub-block, sp floats per sub-block.
struct Q4KM {
  static constexpr int kUnitTerms = 1;
  static constexpr bool kSums = true;
  static constexpr bool kHalf = false;
  struct Raw {
    uint4 hdr;
    uint2 q;  // bytes 8 s .. 8 s + 7 of the unit's 32
  };
  struct W {
    float lo[8], hi[8];
    float d1, m1, d2, m2;
  };
  static __device__ __forceinline__ void load(const GemvArgs& a, const uint8_t* w, int row, int s,
                                              int unit, Raw& r) {
    const uint32_t i = (uint32_t)row * a.nb * 4 + unit;
    r.hdr = ld<uint4>(w, a.off0 + (i >> 2) * 16);
    r.q = ld<uint2>(w, (s < 2 ? a.off1 : a.off2) + i * 16 + 8 * (s & 1));
  }
  static __device__ __forceinline__ void weights(const Raw& r, int u, int, W& w) {
    const uint32_t q[2] = {r.q.x, r.q.y};
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const uint32_t lo = whole(q[h] & 0x0F0F0F0Fu), hi = whole((q[h] >> 4) & 0x0F0F0F0Fu);
#pragma unroll
      for (int b = 0; b < 4; ++b) w.lo[4 * h + b] = byte_f(lo, b), w.hi[4 * h + b] = byte_f(hi, b);
    }
    // scales and mins of sub-blocks 2u, 2u + 1 (quant.c:82-91), u uniform
    uint32_t sc, mn;
    if (u < 2) {
      sc = r.hdr.y & 0x3F3F3F3Fu;
      mn = r.hdr.z & 0x3F3F3F3Fu;
    } else {
      sc = (r.hdr.w & 0x0F0F0F0Fu) | ((r.hdr.y >> 2) & 0x30303030u);
      mn = ((r.hdr.w >> 4) & 0x0F0F0F0Fu) | ((r.hdr.z >> 2) & 0x30303030u);
    }
    sc >>= 16 * (u & 1);
    mn >>= 16 * (u & 1);
    const float dd = f16_bits_to_f32((uint16_t)(r.hdr.x & 0xFFFFu));
    const float dmin = f16_bits_to_f32((uint16_t)(r.hdr.x >> 16));
    w.d1 = dd * byte_f(sc, 0), w.m1 = dmin * byte_f(mn, 0);
    w.d2 = dd * byte_f(sc, 1), w.m2 = dmin * byte_f(mn, 1);
  }
  static __device__ __forceinline__ void stage(const XV& x, float* dst) {
#pragma unroll
    for (int i = 0; i < 4; ++i) *(float4_t*)(dst + 4 * i) = x.f[i];
  }
  // x[8 s .. 8 s + 7] of both sub-blocks
  static __device__ __forceinline__ void load_x(const float* xt, int s, XV& x) {
#pragma unroll
    for (int i = 0; i < 4; ++i) x.f[i] = ld4v(xt + kSubPitch * (i >> 1) + 8 * s + 4 * (i & 1));
  }
  // the running sums of 32 elements, added as hsum_avx2 adds them
  static __device__ __forceinline__ float4_t dot32(const float4_t& x0, const float4_t& x1,
                                                   const float (&w)[8]) {
    const float xv[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
    float4_t v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = mfma_f32_k4(xv[j], w[j]);
    return ((v[0] + v[4]) + (v[2] + v[6])) + ((v[1] + v[5]) + (v[3] + v[7]));
  }
  static __device__ __forceinline__ void terms(const W& w, const XV& x, const float* sums, int sp,
                                               float4_t* t) {
    const float4_t x1 = *(const float4_t*)sums, x2 = *(const float4_t*)(sums + sp);
    const float4_t q1 = dot32(x.f[0], x.f[1], w.lo);
    const float4_t q2 = dot32(x.f[2], x.f[3], w.hi);
    t[0] = ((w.d1 * q1 - w.m1 * x1) + w.d2 * q2) - w.m2 * x2;
  }
};

struct Q6KM {
  static constexpr int kUnitTerms = 4;
  static constexpr bool kSums = false;
  static constexpr bool kHalf = false;
  struct Raw {
    uint4 q[3];   // L0, L1, H words of the unit's four groups
    uint32_t sc;  // their int8 scales
    uint32_t d;
  };
  struct W {
    float f[4][4];  // [group][element s + 4 e]
    float ds[4];
  };
  static __device__ __forceinline__ void load(const GemvArgs& a, const uint8_t* w, int row, int,
                                              int unit, Raw& r) {
    const uint32_t i = (uint32_t)row * a.nb * 4 + unit;
    const uint32_t offs[3] = {a.off0, a.off1, a.off2};
#pragma unroll
    for (int p = 0; p < 3; ++p) r.q[p] = ld<uint4>(w, offs[p] + i * 16);
    r.sc = ld<uint32_t>(w, a.scales_off + i * 4);
    r.d = ld<uint16_t>(w, a.d_off + (i >> 2) * 2);
  }
  // byte s of the four groups' words, group g in byte g
  static __device__ __forceinline__ uint32_t gather(const uint4& w, int s) {
    const uint32_t sel = 0x0C0C0400u + 0x0101u * (uint32_t)s;
    const uint32_t a = __builtin_amdgcn_perm(w.y, w.x, sel);
    const uint32_t b = __builtin_amdgcn_perm(w.w, w.z, sel);
    return a | (b << 16);
  }
  static __device__ __forceinline__ void weights(const Raw& r, int, int s, W& w) {
    const uint32_t m4 = 0x0F0F0F0Fu, m30 = 0x30303030u;
    const uint32_t L0 = gather(r.q[0], s), L1 = gather(r.q[1], s), H = gather(r.q[2], s);
    const uint32_t v[4] = {(L0 & m4) | ((H << 4) & m30), ((L0 >> 4) & m4) | ((H << 2) & m30),
                           (L1 & m4) | (H & m30), ((L1 >> 4) & m4) | ((H >> 2) & m30)};
    const float dd = f16_bits_to_f32((uint16_t)(r.d & 0xFFFFu));
#pragma unroll
    for (int g = 0; g < 4; ++g) {
#pragma unroll
      for (int e = 0; e < 4; ++e) w.f[g][e] = byte_f(v[e], g) - 32.0f;
      w.ds[g] = dd * sbyte(r.sc, g);
    }
  }
  // elements e, 4 + e, 8 + e, 12 + e of the group side by side: lane s reads
  // its four in one vector
  static __device__ __forceinline__ void stage(const XV& x, float* dst) {
    const float* e = (const float*)x.f;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      *(float4*)(dst + 4 * i) = make_float4(e[i], e[4 + i], e[8 + i], e[12 + i]);
  }
  static __device__ __forceinline__ void load_x(const float* xt, int s, XV& x) {
#pragma unroll
    for (int g = 0; g < 4; ++g)
      x.f[g] = ld4v(xt + kSubPitch * (g >> 1) + 16 * (g & 1) + 4 * s);
  }
  static __device__ __forceinline__ void terms(const W& w, const XV& x, const float*, int,
                                               float4_t* t) {
    const f32x16_t z = {};
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      // running sum j: element j fused onto the product of element 8 + j
      f32x16_t a = mfma_f32_4b(x.f[g].z, w.f[g][2], z), b = mfma_f32_4b(x.f[g].w, w.f[g][3], z);
      a = mfma_f32_4b(x.f[g].x, w.f[g][0], a);
      b = mfma_f32_4b(x.f[g].y, w.f[g][1], b);
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const float h = ((a[v] + b[v]) + (a[8 + v] + b[8 + v])) +
                        ((a[4 + v] + b[4 + v]) + (a[12 + v] + b[12 + v]));
        t[g][v] = w.ds[g] * h;
      }
    }
  }
};

struct Q80M {
  static constexpr int kUnitTerms = 2;
  static constexpr bool kSums = false;
  static constexpr bool kHalf = true;  // a row's last unit may be one block
  struct Raw {
    uint2 q[2];  // bytes 8 s .. 8 s + 7 of the unit's two blocks
    uint32_t d[2];
  };
  struct W {
    float f[2][8];
    float d[2];
  };
  static __device__ __forceinline__ void load(const GemvArgs& a, const uint8_t* w, int row, int s,
                                              int unit, Raw& r) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      // blocks past the row's end re-read its last one (their terms are not used)
      const uint32_t blk = (uint32_t)row * a.nb + min(2 * unit + h, a.nb - 1);
      r.q[h] = ld<uint2>(w, (s < 2 ? a.off0 : a.off1) + blk * 16 + 8 * (s & 1));
      r.d[h] = ld<uint16_t>(w, a.d_off + blk * 2);
    }
  }
  static __device__ __forceinline__ void weights(const Raw& r, int, int, W& w) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int b = 0; b < 4; ++b)
        w.f[h][b] = sbyte(r.q[h].x, b), w.f[h][4 + b] = sbyte(r.q[h].y, b);
      w.d[h] = f16_bits_to_f32((uint16_t)(r.d[h] & 0xFFFFu));
    }
  }
  static __device__ __forceinline__ void stage(const XV& x, float* dst) { Q4KM::stage(x, dst); }
  static __device__ __forceinline__ void load_x(const float* xt, int s, XV& x) {
    Q4KM::load_x(xt, s, x);
  }
  static __device__ __forceinline__ void terms(const W& w, const XV& x, const float*, int,
                                               float4_t* t) {
    const f32x16_t z = {};
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      float4_t x0 = x.f[2 * h], x1 = x.f[2 * h + 1];
      if (h) asm("" : "+v"(x0), "+v"(x1), "+v"(t[0]));  // as after()
      const float xv[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
      float4_t acc[8];
      f32x16_t p = mfma_f32_4b(xv[0], w.f[h][0], z);
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        // p: the rounded products of elements k, 8 + k, 16 + k, 24 + k; the
        // next four are multiplied while these are added
        f32x16_t n = p;
        if (k < 7) {
          n = mfma_f32_4b(xv[k + 1], w.f[h][k + 1], z);
          asm("" : "+v"(p), "+v"(n));
        }
#pragma unroll
        for (int v = 0; v < 4; ++v) acc[k][v] = (p[v] + p[4 + v]) + (p[8 + v] + p[12 + v]);
        p = n;
      }
      t[h] = w.d[h] *
             (((acc[0] + acc[4]) + (acc[2] + acc[6])) + ((acc[1] + acc[5]) + (acc[3] + acc[7])));
    }
  }
};

// sum_x of a 32-element sub-block (quant.c:433, as Q4K::load_x): running sum k
// is (x[k] + x[8+k]) + (x[16+k] + x[24+k]), the pairs in this lane (the even
// lane of a pair holds elements 0-15, the odd one 16-31).
__device__ __forceinline__ float sub_sum(const XV& x) {
  const float* e = (const float*)x.f;
  float t[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const float p = 0.0f + (e[k] + e[8 + k]);
    const int q = __builtin_amdgcn_mov_dpp(__float_as_int(p), 0xB1, 0xF, 0xF, true);  // lane ^ 1
    t[k] = p + __int_as_float(q);
  }
  return hsum8(t);
}

// LDS floats of a workgroup: two buffers of staged x and its sums, two of the
// terms that waves of one row tile exchange (KW > 1).
template <class F, int KW>
constexpr int x_floats() {
  return Chunk<KW>::kXs + (F::kSums ? Chunk<KW>::kSums : 0);
}
template <class F, int KW, int M>
constexpr int term_floats() {
  return KW == 1 ? 0 : waves_of(KW) / KW * Chunk<KW>::U * F::kUnitTerms * M * 4 * 64;
}
template <class F, int KW, bool PAIR>
constexpr size_t lds_bytes() {
  return sizeof(float) * 2 * (size_t)(x_floats<F, KW>() + term_floats<F, KW, PAIR ? 2 : 1>());
}

// One workgroup: 16 tokens x (4 / KW) * 16 rows (16 with KW 8; of two matrices
// for a gate/up pair).  The waves take row tiles of their own (KW 1), or KW
// waves share a row tile: each forms the terms of a KW-th of a chunk's units
// into LDS, then chains a KW-th of the tile's sums (KW 8: the first four waves a
// quarter) over the chunk's terms, in block order.  One barrier per chunk; the
// next chunk's x, the next unit's operand and the weights of the next two units
// are in flight meanwhile.
template <class F, int KW, bool PAIR>
__device__ __forceinline__ void gemm_body(const GemvArgs& a, const BatchShape& b, int r_tile,
                                          int t_tile, float* lds) {
  using C = Chunk<KW>;
  constexpr int RW = waves_of(KW) / KW, M = PAIR ? 2 : 1;
  constexpr int S = KW == 8 ? 1 : 4 / KW;  // sums per lane and matrix
  constexpr int TU = F::kUnitTerms, UW = C::U / KW;  // a wave's units of a chunk
  constexpr int XF = x_floats<F, KW>(), TF = term_floats<F, KW, M>();
  static_assert(UW * KW == C::U, "a chunk's units divide among the waves");
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 15, s = lane >> 4;
  const int kw = wave % KW, rw = wave / KW;
  const int r = (r_tile * RW + rw) * kMT + c;
  const int row = min(r, a.d - 1);
  const int tk0 = t_tile * kMT;
  const int units = (a.n + 63) / 64;  // the last may be half (Q8_0)
  const int chunks = (a.n + C::K - 1) / C::K;
  // staging: thread p takes 16-element piece p % PP of token p / PP; pieces
  // past the row's end re-read its last one, tokens past the prompt's its last
  // (not used)
  constexpr int PP = C::K / 16;
  const int stok = tid / PP, piece = tid % PP;
  const bool stager = tid < PP * kMT;
  const float* xsrc = a.x + (size_t)min(tk0 + stok, b.n_tok - 1) * b.x_stride;
  const int xdst = stok * C::kTokPitch + (piece >> 1) * kSubPitch + 16 * (piece & 1);
  XV xg;
  auto fetch_x = [&](int chunk) {
    if (!stager) return;
    const float* p = xsrc + min(chunk * C::K + 16 * piece, a.n - 16);
#pragma unroll
    for (int i = 0; i < 4; ++i) xg.f[i] = ld4v(p + 4 * i);
  };
  auto stage_x = [&](float* buf) {
    if (!stager) return;
    F::stage(xg, buf + xdst);
    if constexpr (F::kSums) {
      const float v = sub_sum(xg);
      if ((piece & 1) == 0) buf[C::kXs + (piece >> 1) * kMT + stok] = v;
    }
  };
  // KW 1: tokens 4 s .. 4 s + 3 of row c; else this wave's S of them
  float4_t sum[M];
#pragma unroll
  for (int m = 0; m < M; ++m) sum[m] = float4_t{0.f, 0.f, 0.f, 0.f};
  // unit k (0 .. 2 UW - 1) of this wave, counted from chunk on
  auto unit_at = [&](int chunk, int k) { return (chunk + k / UW) * C::U + kw * UW + k % UW; };
  typename F::Raw raw[2][M];
  auto load_w = [&](int unit, typename F::Raw(&w)[M]) {
    F::load(a, a.w, row, s, min(unit, units - 1), w[0]);
    if constexpr (PAIR) F::load(a, a.w2, row, s, min(unit, units - 1), w[1]);
  };
  // One chunk; with one unit a chunk its weights are in raw[P], else a wave's
  // even units' are in raw[0] and its odd ones' in raw[1].
  auto body = [&](int chunk, auto par) {
    constexpr int P = decltype(par)::value;
    float* xs = lds + (chunk & 1) * XF;
    float* xch = lds + 2 * XF + (chunk & 1) * TF;
    const bool more = chunk + 1 < chunks;
    if (more) fetch_x(chunk + 1);
    const float* xt = xs + c * C::kTokPitch + kw * UW * 2 * kSubPitch;
    XV xn;
    F::load_x(xt, s, xn);
    // unit k of the wave's UW, its weights in rk
    auto step = [&](int k, typename F::Raw(&rk)[M]) {
      const int ku = kw * UW + k, unit = chunk * C::U + ku;
      typename F::W w[M];
#pragma unroll
      for (int m = 0; m < M; ++m) F::weights(rk[m], unit & 3, s, w[m]);
      load_w(unit_at(chunk, k + 2), rk);
      XV x = xn;
      // after the chunk's last unit: read again, not used
      F::load_x(xt + min(k + 1, UW - 1) * 2 * kSubPitch, s, xn);
      const float* st = xs + C::kXs + 2 * ku * kMT + 4 * s;
#pragma unroll
      for (int m = 0; m < M; ++m) {
        float4_t t[TU];
        F::terms(w[m], x, st, kMT, t);
        if constexpr (KW == 1) {
#pragma unroll
          for (int g = 0; g < TU; ++g)
            if (!F::kHalf || unit * TU + g < a.terms) sum[m] = sum[m] + t[g];
          if constexpr (M > 1) after(m + 1 < M ? x : xn, sum[m]);
        } else {
          float* o = xch + ((rw * C::U + ku) * TU * M + m) * 256 + 4 * lane;
#pragma unroll
          for (int g = 0; g < TU; ++g) *(float4_t*)(o + g * M * 256) = t[g];
          if constexpr (M > 1) after(m + 1 < M ? x : xn, t[TU - 1]);
        }
      }
    };
    if constexpr (UW == 1) {
      step(0, raw[P]);
    } else {
#pragma unroll 1
      for (int k = 0; k < UW; k += 2) {
        step(k, raw[0]);
        step(k + 1, raw[1]);
      }
    }
    if (more) stage_x(lds + ((chunk + 1) & 1) * XF);
    __syncthreads();
    if (KW > 1 && kw * S < 4) {
      const int left = a.terms - chunk * C::U * TU;
#pragma unroll
      for (int m = 0; m < M; ++m) {
        const float* o = xch + (rw * C::U * TU * M + m) * 256 + 4 * lane + kw * S;
#pragma unroll
        for (int g = 0; g < C::U * TU; ++g) {
          if ((F::kHalf || C::K > 256) && g >= left) break;
          if constexpr (S == 1) {
            sum[m][0] = sum[m][0] + o[g * M * 256];
          } else {
            const float2 v = *(const float2*)(o + g * M * 256);
            sum[m][0] = sum[m][0] + v.x;
            sum[m][1] = sum[m][1] + v.y;
          }
        }
      }
    }
  };
  fetch_x(0);
  load_w(unit_at(0, 0), raw[0]);
  load_w(unit_at(0, 1), raw[1]);
  stage_x(lds);
  __syncthreads();
  if constexpr (UW == 1) {
#pragma unroll 1
    for (int chunk = 0; chunk < chunks; chunk += 2) {
      body(chunk, std::integral_constant<int, 0>{});
      if (chunk + 1 < chunks) body(chunk + 1, std::integral_constant<int, 1>{});
    }
  } else {
#pragma unroll 1
    for (int chunk = 0; chunk < chunks; ++chunk) body(chunk, std::integral_constant<int, 0>{});
  }
  if (kw * S >= 4) return;
#pragma unroll
  for (int i = 0; i < S; ++i) {
    const int tok = tk0 + 4 * s + kw * S + i;
    if (r >= a.d || tok >= b.n_tok) continue;
    const size_t o = (size_t)tok * b.out_stride + r;
    float v = sum[0][i];
    if constexpr (PAIR) {
      a.out[o] = silu(v) * sum[M - 1][i];
    } else {
      if (a.bias_mode == 1) v = v + a.bias[r];
      if (a.bias_mode == 2) v = v + 0.0f;
      if (a.gate) v = silu(a.gate[o]) * v;
      if (a.resid) v = a.resid[o] + v;
      a.out[o] = v;
    }
  }
}

// Workgroup id -> row tile and token tile: the token tiles of a row tile share
// an XCD (ids congruent mod 8) and its L2, so its weights come from HBM about
// once.  False past the last row tile.
__device__ __forceinline__ bool tile_of(int row_tiles, int tok_tiles, int& r_tile, int& t_tile) {
  const int kb = blockIdx.x >> 3;
  r_tile = (kb / tok_tiles) * 8 + (blockIdx.x & 7);
  t_tile = kb % tok_tiles;
  return r_tile < row_tiles;
}

template <class F, int KW, bool PAIR>
__global__ __launch_bounds__(64 * waves_of(KW)) void gemm_mfma_kernel(GemvArgs a, BatchShape b) {
  extern __shared__ __align__(16) float lds[];
  int r_tile, t_tile;
  if (tile_of(b.row_tiles, b.tok_tiles, r_tile, t_tile))
    gemm_body<F, KW, PAIR>(a, b, r_tile, t_tile, lds);
}

// Three matrices over the same x in one launch (q, k and v), the row tiles of
// each a range of the grid's: a small matrix alone leaves most CUs idle.  K
// quants and Q8_0 are built apart: with both, Q8_0's registers leave two
// workgroups a CU instead of three.
struct MultiBatch {
  GemvArgs seg[3];
  BatchShape shape[3];  // row_tiles: of the segment
  int qtype[3];
  int tile1, tile2, row_tiles;  // first tiles of segments 1 and 2, all tiles
};

template <int KW, bool Q8>
__global__ __launch_bounds__(64 * waves_of(KW)) void gemm_mfma_multi_kernel(MultiBatch m) {
  extern __shared__ __align__(16) float lds[];
  int r_tile, t_tile;
  if (!tile_of(m.row_tiles, m.shape[0].tok_tiles, r_tile, t_tile)) return;
  const int i = (r_tile >= m.tile1) + (r_tile >= m.tile2);
  r_tile -= i == 2 ? m.tile2 : i == 1 ? m.tile1 : 0;
  if constexpr (Q8)
    gemm_body<Q80M, KW, false>(m.seg[i], m.shape[i], r_tile, t_tile, lds);
  else if (m.qtype[i] == kTypeQ4K)
    gemm_body<Q4KM, KW, false>(m.seg[i], m.shape[i], r_tile, t_tile, lds);
  else
    gemm_body<Q6KM, KW, false>(m.seg[i], m.shape[i], r_tile, t_tile, lds);
}

constexpr size_t kLds = 160 << 10;  // of a CU

int cu_count() { return ctx().num_cus > 0 ? ctx().num_cus : 256; }

// Whether the eight-wave form of a launch is built: its LDS fits a CU (a Q6_K
// pair's exchanged terms don't).
bool eight_built(int qtype, bool pair) {
  if (!pair) return true;
  return (qtype == kTypeQ4K   ? lds_bytes<Q4KM, 8, true>()
          : qtype == kTypeQ6K ? lds_bytes<Q6KM, 8, true>()
                              : lds_bytes<Q80M, 8, true>()) <= kLds;
}
static_assert(std::max({lds_bytes<Q4KM, 8, false>(), lds_bytes<Q6KM, 8, false>(),
                        lds_bytes<Q80M, 8, false>()}) <= kLds, "plain launches: always built");

// Eight waves on a row tile: where the launch's tiles leave CUs idle, two waves
// a SIMD instead of one hide each other's MFMA and LDS waits; not for rows of
// a chunk or two.
// Measured, us for 8 / 4 waves: n = 2048, 128 tiles, Q4_K 9.4 / 11.5, Q6_K 11.9 /
// 13.7, Q8_0 12.0 / 14.5; n = 5632 20.1 / 27.9; n = 512 4.4 / 4.4 (Q6_K 5.7 / 5.4);
// 384 tiles of n = 2048 17.6 / 15.7.
bool eight_waves(const GemvArgs& a, long tiles, int qtype, bool pair) {
  return tiles <= cu_count() && a.n >= 1024 && eight_built(qtype, pair);
}

// Waves per row tile, from the launch's 16 x 16 tiles (a pair's count once):
// the most that still adds waves to idle SIMDs.  Measured, us at n = 2048,
// KW 4 / 2 / 1: Q4_K 256 tiles 11.2 / 18.6 / 23.9, 1024 26.8 / 25.7 / 25.4,
// 1408 35 / 32 / 37, 5632 114 / 95 / 94; Q6_K 256 13.6 / 21 / 28, 1024 36 /
// 32 / 30, 5632 179 / 142 / 137.  Q8_0's products keep four tiles of
// registers each and spill the unsplit form: 5632 tiles 179 / 156 / 213.
int waves_per_tile(const GemvArgs& a, long tiles, int qtype, bool pair) {
  if (eight_waves(a, tiles, qtype, pair)) return 8;
  const int cus = cu_count();
  if (tiles < 4L * cus) return 4;
  return tiles < 8L * cus || qtype == kTypeQ8_0 ? 2 : 1;
}

BatchShape shape_of(const GemvArgs& a, int n_tok, int x_stride, int out_stride, int kw) {
  BatchShape b{};
  b.n_tok = n_tok;
  b.x_stride = x_stride;
  b.out_stride = out_stride;
  const int rows = kMT * (waves_of(kw) / kw);
  b.row_tiles = (a.d + rows - 1) / rows;
  b.tok_tiles = (n_tok + kMT - 1) / kMT;
  return b;
}

unsigned grid_of(int row_tiles, int tok_tiles) {
  return 8u * (unsigned)((row_tiles + 7) / 8) * (unsigned)tok_tiles;
}

long tiles_of(const GemvArgs& a, int n_tok) {
  return (long)((a.d + kMT - 1) / kMT) * ((n_tok + kMT - 1) / kMT);
}

// A launch holds fewer than 2^32 threads, here 2^32 / 256 workgroups of 512 outputs
// (32 GiB) in the smallest case.  The VALU kernel's hold up to 2048 where rows
// are short.
bool launchable(int qtype, const GemvArgs& a, int n_tok, bool pair) {
  const int kw = waves_per_tile(a, tiles_of(a, n_tok), qtype, pair);
  const BatchShape b = shape_of(a, n_tok, 0, 0, kw);
  return 8LL * ((b.row_tiles + 7) / 8) * b.tok_tiles * 64 * waves_of(kw) < 1LL << 32;
}

// Which of the two batched kernels runs, by estimates in us fitted to both (34000 shapes
// of n 64 to 11000, d 64 to 12000, 2 to 256 tokens, warm) so that the choice is
// right rather than the estimate.  The VALU kernel: its latency, or its work per
// weight, token and group of four tokens, of which a workgroup's idle lanes (169
// units leave 87 of 256) waste a share.  Here: a wave's chain of units, longer with
// every further tile a CU (its workgroups share the SIMDs; from four on fewer waves
// share a tile), or, with the chip full, the work of the padded token tiles.
// VALU / here: 2048 x 2048 Q4_K, 2 / 4 / 16 / 128 tokens 8.7 / 12.2 / 19 / 70 and
// 9.4 / 9.4 / 9.4 / 25; Q8_0 5408 x 1581, 39 tokens 75 and 47; Q6_K 512 x 9343, 2
// tokens 7.7 and 10.8; the pair 2816 x 7936 Q4_K, 5 tokens 55 and 28.  Of these 33
// shapes run more than 2% longer than on the VALU kernel, 484 more than 10%
// longer than on the better one; of 8800 pairs 69 and (5%) 261.
struct Rule {
  double least[3], least_n;    // VALU latency: 2, 3, more tokens; per unit of a row
  double valu0, valu1, valu4;  // a launch; 10^6 weights times tokens, times fours
  double lanes;                // its power of the active lanes' share
  double mfma0, unit[5];       // here: a launch; units by tiles a CU (1, 2, 3, more;
  double work;                 // eight waves); 10^6 weights times padded tokens
  double pair;                 // a pair's chain and work
};
constexpr Rule kRule4K = {{8.8, 10.1, 12.4}, 0.0111, 7.3, 0.107, 0.0476, 0.74,
                          3.34, {0.283, 0.302, 0.4065, 0.614, 0.191}, 0.0508, 1.8};
constexpr Rule kRule6K = {{7.34, 8.2, 12.8}, 0.1, 7.16, 0.165, 0.107, 0.51,
                          3.713, {0.2958, 0.4896, 0.7191, 1.193, 0.2479}, 0.038, 1};
constexpr Rule kPair6K = {{10, 12, 12}, 0, 8, 0.22, 0, 0,
                          2.8, {0.35, 0.62, 0.89, 1.16, 0}, 0.046, 2};  // no eight waves
constexpr Rule kRule80 = {{5.77, 6.94, 7.58}, 0.0308, 5.79, 0.086, 0.169, 1.04,
                          3.47, {0.317, 0.538, 0.695, 0.908, 0.278}, 0.0569, 2.1};

const Rule& rule_of(int qtype, bool pair) {
  if (qtype == kTypeQ6K) return pair ? kPair6K : kRule6K;
  return qtype == kTypeQ4K ? kRule4K : kRule80;
}

int units64(const GemvArgs& a) { return (a.n + 63) / 64; }
double mega(const GemvArgs& a) { return 1e-6 * a.n * (double)a.d; }

double valu_us(int qtype, const GemvArgs& a, int n_tok, bool pair) {
  const Rule& r = rule_of(qtype, pair);
  const double lanes = (double)a.units * a.row_par / (a.unit_iters * (double)kThreads);
  const double work = mega(a) * (r.valu1 * n_tok + r.valu4 * ((n_tok + 3) / 4));
  return std::max(r.least[n_tok > 3 ? 2 : n_tok > 2] + r.least_n * units64(a),
                  r.valu0 + (pair ? 2 : 1) * work / std::pow(lanes, r.lanes));
}
// of a launch of so many tiles
double unit_us(int qtype, const GemvArgs& a, long tiles, bool pair) {
  const long past_first = std::min((tiles - 1) / cu_count(), 3L);
  return rule_of(qtype, pair).unit[eight_waves(a, tiles, qtype, pair) ? 4 : past_first];
}
double work_us(int qtype, const GemvArgs& a, int n_tok, bool pair) {
  return rule_of(qtype, pair).work * mega(a) * ((n_tok + kMT - 1) / kMT * kMT);
}

template <class F, int KW>
int launch_k(bool pair, const GemvArgs& a, const BatchShape& b, hipStream_t st) {
  const dim3 grid(grid_of(b.row_tiles, b.tok_tiles)), block(64 * waves_of(KW));
  if (!pair) {
    hipLaunchKernelGGL((gemm_mfma_kernel<F, KW, false>), grid, block, (lds_bytes<F, KW, false>()),
                       st, a, b);
  } else if constexpr (lds_bytes<F, KW, true>() <= kLds) {
    hipLaunchKernelGGL((gemm_mfma_kernel<F, KW, true>), grid, block, (lds_bytes<F, KW, true>()),
                       st, a, b);
  } else {
    set_error("gemm_mfma: no pair of %d waves a tile", KW);
    return -1;
  }
  return check_hip(hipGetLastError(), "gemm_mfma_kernel launch");
}
template <class F>
int launch_f(int kw, bool pair, const GemvArgs& a, const BatchShape& b, hipStream_t st) {
  if (kw == 8) return launch_k<F, 8>(pair, a, b, st);
  if (kw == 4) return launch_k<F, 4>(pair, a, b, st);
  if constexpr (!F::kHalf) {  // Q8_0: waves_per_tile has no 1
    if (kw == 1) return launch_k<F, 1>(pair, a, b, st);
  }
  return launch_k<F, 2>(pair, a, b, st);
}

template <int KW, bool Q8>
void launch_multi(const MultiBatch& m, hipStream_t st) {
  const size_t lds = Q8 ? lds_bytes<Q80M, KW, false>()
                        : std::max(lds_bytes<Q4KM, KW, false>(), lds_bytes<Q6KM, KW, false>());
  hipLaunchKernelGGL((gemm_mfma_multi_kernel<KW, Q8>),
                     dim3(grid_of(m.row_tiles, m.shape[0].tok_tiles)), dim3(64 * waves_of(KW)), lds,
                     st, m);
}

}  // namespace

namespace plh {

bool gemm_mfma_pays(int qtype, const GemvArgs& a, int n_tok, bool pair) {
  if (!launchable(qtype, a, n_tok, pair)) return false;
  const Rule& r = rule_of(qtype, pair);
  const double chain = unit_us(qtype, a, tiles_of(a, n_tok), pair) * units64(a);
  return r.mfma0 + (pair ? r.pair : 1) * std::max(chain, work_us(qtype, a, n_tok, pair)) <
         valu_us(qtype, a, n_tok, pair);
}

int gemm_mfma(int qtype, bool pair, const GemvArgs& a, int n_tok, int x_stride, int out_stride) {
  const int kw = waves_per_tile(a, tiles_of(a, n_tok), qtype, pair);
  const BatchShape b = shape_of(a, n_tok, x_stride, out_stride, kw);
  hipStream_t st = ctx().stream;
  if (qtype == kTypeQ4K) return launch_f<Q4KM>(kw, pair, a, b, st);
  if (qtype == kTypeQ8_0) return launch_f<Q80M>(kw, pair, a, b, st);
  return launch_f<Q6KM>(kw, pair, a, b, st);
}

// Nearly always: one launch beats three of the matrix cores, which small
// matrices leave idle, and three of the VALU kernel but for two or three tokens of long
// rows (Q8_0 n = 4096, 4096 + 2 x 512 rows: 34 us against 26; 128 tokens of
// TinyLlama's 2048 + 2 x 256: 34 against 102).  Of 6950 shapes 12 lose more than 2%.
bool gemm_mfma_multi_pays(const int* qtype, const GemvArgs* a, int n_tok) {
  const int q8 = (qtype[0] == kTypeQ8_0) + (qtype[1] == kTypeQ8_0) + (qtype[2] == kTypeQ8_0);
  if (q8 != 0 && q8 != 3) return false;
  long tiles = 0, threads = 0;
  for (int i = 0; i < 3; ++i) tiles += tiles_of(a[i], n_tok);
  double apart = 0, first = 0, unit = 0, work = 0;
  for (int i = 0; i < 3; ++i) {
    apart += valu_us(qtype[i], a[i], n_tok, false);
    first = std::max(first, rule_of(qtype[i], false).mfma0);
    unit += unit_us(qtype[i], a[i], tiles, false) * tiles_of(a[i], n_tok) / tiles;
    work += work_us(qtype[i], a[i], n_tok, false);
    threads += tiles_of(a[i], n_tok) * 512;  // at most, but for the last tiles
  }
  return threads < 1LL << 31 && first + std::max(unit * units64(a[0]), work) < apart;
}

int gemm_mfma_multi(const int* qtype, const GemvArgs* a, int n_tok, int x_stride,
                    const int* out_stride) {
  MultiBatch m{};
  long tiles = 0;
  for (int i = 0; i < 3; ++i) tiles += tiles_of(a[i], n_tok);
  const bool q8 = qtype[0] == kTypeQ8_0;
  const int kw = waves_per_tile(a[0], tiles, qtype[0], false);
  for (int i = 0; i < 3; ++i) {
    m.seg[i] = a[i];
    m.qtype[i] = qtype[i];
    m.shape[i] = shape_of(a[i], n_tok, x_stride, out_stride[i], kw);
  }
  m.tile1 = m.shape[0].row_tiles;
  m.tile2 = m.tile1 + m.shape[1].row_tiles;
  m.row_tiles = m.tile2 + m.shape[2].row_tiles;
  hipStream_t st = ctx().stream;
  if (q8) {  // never with one wave (waves_per_tile)
    if (kw == 8)
      launch_multi<8, true>(m, st);
    else if (kw == 2)
      launch_multi<2, true>(m, st);
    else
      launch_multi<4, true>(m, st);
  } else if (kw == 1) {
    launch_multi<1, false>(m, st);
  } else if (kw == 8) {
    launch_multi<8, false>(m, st);
  } else if (kw == 2) {
    launch_multi<2, false>(m, st);
  } else {
    launch_multi<4, false>(m, st);
  }
  return check_hip(hipGetLastError(), "gemm_mfma_multi_kernel launch");
}

}  // namespace plh
