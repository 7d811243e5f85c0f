// Reference-semantics decode attention for gfx950, for what the MFMA kernels
// of attn.hip do not take:
//   - fp32 queries and caches, and bf16 ones off a 16-byte boundary
//     (dense_kernel.py:21-67 and sparse_kernel.py:67-102 load q, k, v in
//     whatever dtype they are given, compute in fp32 and store o in q's dtype);
//   - KIVI caches of any code width and group size (quant_kernel.py:436-548,
//     whose BITS and GROUP_SIZE are kernel parameters: QMAX = 2^BITS - 1,
//     8 / BITS codes per byte).
// Everything is fp32: every K and V element is loaded (or dequantized as
// scale * (code - zero), quant_kernel.py:263-266, 308-311) as a float, the
// logits are fp32 dot products, the softmax runs online in the log2 domain
// and the output is rounded once to q's dtype.
//
// Both contractions run on the fp32 matrix instruction (16x16x4, fp32 operands
// and sums): scalar dot products of every query head with every row, which
// stood here before, took 1.2 to 1.9 TB/s of fp32 K and V.  One workgroup of 8
// waves per (KV head, split); a wave takes every eighth 16-token tile, two in
// flight, straight from memory into operand order, with no LDS: lane (i, g),
// i = lane % 16, g = lane / 16, loads channels 16c + 4g .. + 3 of token i (K,
// c = 0..7: 64 contiguous bytes of a fp32 row per load) and channels
// 64h + 4i .. + 3 of token 4g + r (V, h = 0..1, r = 0..3: 256 contiguous
// bytes).  The logits come out with lane (n, g) holding head n of tokens
// 4g + r, which is the operand order of the probabilities against those V
// loads, so the softmax runs online between the two in registers and each wave
// keeps its own; the waves' states meet in LDS at the end.  A 16-token tile is
// 64 matrix instructions of 32 cycles for 16 KB of fp32 rows, 3 times the
// memory's rate over the chip.  Several splits per KV head leave (m, l, acc)
// partials in the workspace, combined by generic_merge_kernel.
// Per call, scalar products -> this: fp32 dense B=1 of 8 KV heads, L=16505
// 86.0 -> 33.1 us (4.1 TB/s), B=26 of 2, L=3141 90.5 -> 54.9; fp32 sparse B=15,
// W=1815 90.8 -> 56.5, B=3, W=61 13.6 -> 7.5; 8-bit bf16 KIVI B=27, W=928
// 200.8 -> 48.7; 4-bit fp32 KIVI B=1, W=2048 414.8 -> 90.5 (one workgroup per KV
// head: the call brings no workspace).
//
// KIVI slot mapping (the regime composition of quant_kernel.py:358-401):
// slot s < sink is sink token s, slot s < sink + win_tok window-old token
// s - sink, later slots residual row s - sink - win_tok.  (The reference's
// tile dequantizer positions a tile's codes relative to the tile start,
// quant_kernel.py:238-245, which agrees with this mapping whenever the sink
// is a multiple of 8 / BITS, as the default sink of 4 is for BITS >= 2.)

#include "generic.h"

#include "kvdec.h"

#include <algorithm>

namespace kvdec {
namespace {

constexpr int kGWaves = 8;
constexpr int kGT = 64 * kGWaves;   // threads per workgroup
constexpr int kGTile = 16;          // tokens of a tile

// Element types of the rows: four adjacent values as loaded (from any address
// of the type's own alignment), and as floats.
template <int DT>
struct GElt;
template <>
struct GElt<KVDEC_F16> {
  typedef _Float16 T;
};
template <>
struct GElt<KVDEC_BF16> {
  typedef uint16_t T;
};
template <>
struct GElt<KVDEC_F32> {
  typedef float T;
};
typedef _Float16 half4v __attribute__((ext_vector_type(4)));

template <class T>
struct Four {
  T x[4];
};
template <class T>
__device__ __forceinline__ Four<T> load4(const T* p) {
  Four<T> f;
  __builtin_memcpy(&f, p, sizeof f);
  return f;
}
__device__ __forceinline__ float4v floats(const Four<float>& f) { return float4v{f.x[0], f.x[1], f.x[2], f.x[3]}; }
__device__ __forceinline__ float4v floats(const Four<_Float16>& f) {
  return float4v{(float)f.x[0], (float)f.x[1], (float)f.x[2], (float)f.x[3]};
}
__device__ __forceinline__ float4v floats(const Four<uint16_t>& f) {   // bf16
  float4v v;
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = __builtin_bit_cast(float, (uint32_t)f.x[e] << 16);
  return v;
}

// Four adjacent values of q and o, whose type is an argument.
__device__ __forceinline__ float4v load_q4(const void* q, int dt, size_t i) {
  if (dt == KVDEC_F32) return floats(load4(static_cast<const float*>(q) + i));
  if (dt == KVDEC_F16) return floats(load4(static_cast<const _Float16*>(q) + i));
  return floats(load4(static_cast<const uint16_t*>(q) + i));
}
__device__ __forceinline__ void store_o(void* o, int dt, size_t i, float v) {
  if (dt == KVDEC_F32) static_cast<float*>(o)[i] = v;
  else if (dt == KVDEC_F16) static_cast<_Float16*>(o)[i] = (_Float16)v;
  else static_cast<uint16_t*>(o)[i] = __builtin_bit_cast(uint16_t, (__bf16)v);
}

// Slot validity of sequence b.
struct GRange {
  SlotRanges R;
  const int32_t* lens;   // null: R for every sequence
  bool sparse;
  int32_t window, sink, layout;
  int64_t rows;
  __device__ SlotRanges at(int64_t b) const {
    if (!lens) return R;
    int64_t len = lens[b];
    len = len < 0 ? 0 : len;
    if (sparse) return sparse_ranges(len, window, sink, layout);
    return SlotRanges{(int)(len < rows ? len : rows), 0, 0};
  }
};

struct GArgs {
  const void* q;
  void* o;
  int dt;                 // element type of q and o
  float* ws;              // split partials: acc [units][128], then m [units], then l [units]
  int64_t pairs;
  int32_t H, KVH, G;
  int n_tiles, per_split, n_splits;
  float scale_log2;
  GRange range;
};

// A wave's online softmax over its tiles, lane (n, g): head n; l and O are sums
// over the lane's own tokens; O[h][e][r] is channel 64h + 16g + 4r + e.
struct GState {
  float4v O[2][4];
  float m, l;
};

// One tile.  k(c): K[token i][16c + 4g ..]; v(r, h): V[token 4g + r][64h + 4i
// ..]; bit r of `valid`: whether token 4g + r is attended (masked K values take
// part in no valid logit, masked V values are replaced by zeros, so neither
// need be finite).  Heads >= G have a zero query and are not stored.
template <class K, class V>
__device__ __forceinline__ void generic_tile(K&& k, V&& v, uint32_t valid, const float4v (&q)[8], float scale_log2,
                                             GState& st) {
  // A logit's 128 products in 8 sums of 16: the length of the chains is most of
  // the result's error against 64 bits (fp32 sparse W=61: 3.5e-7 with 2 sums of
  // 64, 2.0e-7 with 8; the scalar products' 4 of 32 had 2.3e-7), and the time is
  // the same.
  constexpr int kChains = 8;
  float4v s[kChains];
#pragma unroll
  for (int c = 0; c < kChains; ++c) s[c] = float4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int c = 0; c < 8; ++c) {
    const float4v a = k(c);
#pragma unroll
    for (int e = 0; e < 4; ++e)
      s[c % kChains] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], q[c][e], s[c % kChains], 0, 0, 0);
  }
#pragma unroll
  for (int d = kChains / 2; d >= 1; d /= 2)
#pragma unroll
    for (int c = 0; c < d; ++c) s[c] += s[c + d];
  float x[4], lmax = -INFINITY;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    x[r] = (valid >> r) & 1u ? s[0][r] * scale_log2 : -INFINITY;
    lmax = fmaxf(lmax, x[r]);
  }
  if (__ballot(lmax > st.m)) {
    const float mnew = fmaxf(st.m, group_max(lmax));
    const float alpha = st.m == -INFINITY ? 0.f : exp2f(st.m - mnew);
    st.l *= alpha;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int e = 0; e < 4; ++e) st.O[h][e] *= alpha;
    st.m = mnew;
  }
  // m = -inf: every logit so far is masked, whose exp2 is 0, or NaN, which has
  // to reach the output also where a tile holds nothing else.
  const float m = st.m == -INFINITY ? 0.f : st.m;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const float p = exp2f(x[r] - m);
    st.l += p;
    const bool ok = (valid >> r) & 1u;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const float4v a = v(r, h);
#pragma unroll
      for (int e = 0; e < 4; ++e)
        st.O[h][e] = __builtin_amdgcn_mfma_f32_16x16x4f32(ok ? a[e] : 0.f, p, st.O[h][e], 0, 0, 0);
    }
  }
}

// `n` rows of element type DT of one KV head, the first at slot `slot0`.
template <int DT>
struct GRowTiles {
  typedef typename GElt<DT>::T T;
  struct Raw {
    Four<T> k[8], v[4][2];
  };
  const T* kb;
  const T* vb;
  int n, slot0;
  __device__ __forceinline__ void load(int t0, Raw& X, int i, int g) const {
    const T* kr = kb + (size_t)min(t0 + i, n - 1) * kHeadDim + 4 * g;   // rows past n: masked
#pragma unroll
    for (int c = 0; c < 8; ++c) X.k[c] = load4(kr + 16 * c);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const T* vr = vb + (size_t)min(t0 + 4 * g + r, n - 1) * kHeadDim + 4 * i;
#pragma unroll
      for (int h = 0; h < 2; ++h) X.v[r][h] = load4(vr + 64 * h);
    }
  }
  __device__ __forceinline__ void step(int, const Raw& X, uint32_t valid, int, int, const float4v (&q)[8],
                                       float scale_log2, GState& st) const {
    generic_tile([&](int c) { return floats(X.k[c]); }, [&](int r, int h) { return floats(X.v[r][h]); }, valid, q,
                 scale_log2, st);
  }
};

// `n` quantized tokens of one KV head, the first at slot `slot0`: PF codes of
// `bits` bits per byte, K per channel over groups of `group` tokens, V per token
// over `group` channels.  SMALL: groups of fewer than 4 channels, whose V scales
// are read where they are used (four times as many would not fit two tiles).
template <int PF, bool SMALL>
struct GQuantTiles {
  static constexpr int kVBytes = PF >= 4 ? 1 : 4 / PF;   // of 4 channels' codes
  struct Raw {
    uint32_t kc[8], vc[4][2];
    half4v ks[8], kz[8];
    _Float16 vs[4][2], vz[4][2];
  };
  const uint8_t* kp;
  const uint8_t* vp;
  const _Float16 *ks, *kz, *vs, *vz;
  int n, slot0, group, bits;

  __device__ __forceinline__ void load(int t0, Raw& X, int i, int g) const {
    // K: byte row t / PF, scale and zero of group t / group (quant_kernel.py:236-266)
    const int t = min(t0 + i, n - 1);   // tokens past n: masked
    const uint8_t* kb = kp + (size_t)(t / PF) * kHeadDim + 4 * g;
    const size_t km = (size_t)(t / group) * kHeadDim + 4 * g;
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      __builtin_memcpy(&X.kc[c], kb + 16 * c, 4);
      __builtin_memcpy(&X.ks[c], ks + km + 16 * c, 8);
      __builtin_memcpy(&X.kz[c], kz + km + 16 * c, 8);
    }
    // V: byte channel / PF of row t, scale and zero of group channel / group
    // (quant_kernel.py:281-311)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const size_t tv = (size_t)min(t0 + 4 * g + r, n - 1);
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int ch = 64 * h + 4 * i;
        X.vc[r][h] = 0;
        __builtin_memcpy(&X.vc[r][h], vp + tv * (kHeadDim / PF) + ch / PF, kVBytes);
        if (!SMALL) {
          const size_t m = tv * (kHeadDim / group) + ch / group;
          X.vs[r][h] = vs[m];
          X.vz[r][h] = vz[m];
        }
      }
    }
  }
  __device__ __forceinline__ void step(int t0, const Raw& X, uint32_t valid, int i, int g, const float4v (&q)[8],
                                       float scale_log2, GState& st) const {
    const uint32_t qmax = (1u << bits) - 1u;
    const uint32_t ksh = (uint32_t)(((t0 + i) % PF) * bits);
    generic_tile(
        [&](int c) {
          float4v a;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float code = (float)((((X.kc[c] >> (8 * e)) & 0xffu) >> ksh) & qmax);
            a[e] = (float)X.ks[c][e] * (code - (float)X.kz[c][e]);
          }
          return a;
        },
        [&](int r, int h) {
          float4v a;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            // channel 4i + e: with 8 codes a byte, the byte's half i % 2
            const uint32_t byte = (X.vc[r][h] >> (8 * (e / PF))) & 0xffu;
            const uint32_t at = (uint32_t)(((PF == 8 ? 4 * (i & 1) : 0) + e) % PF) * (uint32_t)bits;
            const size_t m = (size_t)min(t0 + 4 * g + r, n - 1) * (kHeadDim / group) + (64 * h + 4 * i + e) / group;
            const float s = (float)(SMALL ? vs[m] : X.vs[r][h]), z = (float)(SMALL ? vz[m] : X.vz[r][h]);
            a[e] = s * ((float)((byte >> at) & qmax) - z);
          }
          return a;
        },
        valid, q, scale_log2, st);
  }
};

// Tiles first, first + step, .. < end of one region for this wave, two in
// flight; tiles with no attended token are skipped.
template <class Tiles>
__device__ __forceinline__ void generic_run(const Tiles& S, int first, int end, const SlotRanges& R, int i, int g,
                                            const float4v (&q)[8], float scale_log2, GState& st) {
  typename Tiles::Raw A, B;
  auto live = [&](int t) {
    if (t >= end) return false;
    const int s0 = S.slot0 + kGTile * t, s1 = S.slot0 + min(kGTile * (t + 1), S.n);
    return s0 < R.va || (s1 > R.vb && s0 < R.vc);
  };
  auto load = [&](int t, typename Tiles::Raw& X) {
    if (live(t)) S.load(kGTile * t, X, i, g);
  };
  auto step = [&](int t, const typename Tiles::Raw& X) {
    if (!live(t)) return;
    uint32_t valid = 0;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int tok = kGTile * t + 4 * g + r;
      valid |= (tok < S.n && slot_valid(R, S.slot0 + tok) ? 1u : 0u) << r;
    }
    S.step(kGTile * t, X, valid, i, g, q, scale_log2, st);
  };
  load(first, A);
  load(first + kGWaves, B);
  for (int t = first; t < end; t += 2 * kGWaves) {
    step(t, A);
    load(t + 2 * kGWaves, A);
    step(t + kGWaves, B);
    load(t + 3 * kGWaves, B);
  }
}

// Rows of element type DT: [pairs][rows][128].
template <int DT>
struct GRowsSrc {
  typedef typename GElt<DT>::T T;
  const T* k;
  const T* v;
  int rows;
  template <class Run>
  __device__ __forceinline__ void regions(int64_t pair, Run&& run) const {
    const size_t at = (size_t)pair * rows * kHeadDim;
    run(GRowTiles<DT>{k + at, v + at, rows, 0});
  }
};

// A KIVI cache of any width: the quantized window-old (win_tok tokens) and sink
// (one group, `sink` real tokens) regions and residual rows of element type RT.
template <int RT, int PF, bool SMALL>
struct GKiviSrc {
  typedef typename GElt<RT>::T T;
  const T* kres;
  const T* vres;
  const uint8_t* kp[2];     // sink, window-old
  const _Float16* ks[2];
  const _Float16* kz[2];
  const uint8_t* vp[2];
  const _Float16* vs[2];
  const _Float16* vz[2];
  int32_t sink, win_tok, res_rows, group, bits;

  __device__ __forceinline__ GQuantTiles<PF, SMALL> part(int64_t pair, int r, int ntok, int n, int slot0) const {
    const size_t p = (size_t)pair, kg = p * (size_t)(ntok / group) * kHeadDim,
                 vg = p * (size_t)ntok * (size_t)(kHeadDim / group);
    return GQuantTiles<PF, SMALL>{kp[r] + p * (size_t)(ntok / PF) * kHeadDim, vp[r] + p * (size_t)ntok * (kHeadDim / PF),
                                  ks[r] + kg, kz[r] + kg, vs[r] + vg, vz[r] + vg, n, slot0, group, bits};
  }
  template <class Run>
  __device__ __forceinline__ void regions(int64_t pair, Run&& run) const {
    if (win_tok > 0) run(part(pair, 1, win_tok, win_tok, sink));
    run(part(pair, 0, group, sink, 0));
    const size_t at = (size_t)pair * res_rows * kHeadDim;
    run(GRowTiles<RT>{kres + at, vres + at, res_rows, sink + win_tok});
  }
};

// LDS: every wave's maxima and sums (16 heads), then its output rows
// [head][128], 16-byte chunks XOR-swizzled by head.
constexpr int kGLdsL = kGWaves * kMaxGroup * 4;
constexpr int kGLdsO = 2 * kGLdsL;
constexpr int kGLdsBytes = kGLdsO + kGWaves * kMaxGroup * kHeadDim * 4;
__device__ __forceinline__ float4v* g_row(char* lds, int wave, int head, int chunk) {
  return reinterpret_cast<float4v*>(lds + kGLdsO) + (wave * kMaxGroup + head) * (kHeadDim / 4) + (chunk ^ head);
}

template <class Src>
__global__ __launch_bounds__(kGT, 1) void generic_attn_kernel(GArgs A, Src S) {
  extern __shared__ __align__(16) char lds[];
  const int lane = threadIdx.x & 63, i = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t pair = blockIdx.x;
  const int split = blockIdx.y;
  const int64_t b = pair / A.KVH;
  const int kvh = (int)(pair % A.KVH);
  const int G = A.G;
  const size_t row0 = (size_t)b * A.H + (size_t)kvh * G;
  float4v q[8];
#pragma unroll
  for (int c = 0; c < 8; ++c)
    q[c] = i < G ? load_q4(A.q, A.dt, (row0 + i) * kHeadDim + 16 * c + 4 * g) : float4v{0.f, 0.f, 0.f, 0.f};
  const SlotRanges R = A.range.at(b);
  GState st;
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int e = 0; e < 4; ++e) st.O[h][e] = float4v{0.f, 0.f, 0.f, 0.f};
  st.m = -INFINITY;
  st.l = 0.f;
  // the split's tiles lo .. hi - 1, counted through the regions; this wave's
  // are lo + wave, + 8, ..
  const int lo = split * A.per_split, hi = min(lo + A.per_split, A.n_tiles);
  int base = 0;   // tiles of the regions before
  S.regions(pair, [&](const auto& tiles) {
    const int nt = (tiles.n + kGTile - 1) / kGTile;
    int first = lo + wave;
    if (first < base) first += (base - first + kGWaves - 1) / kGWaves * kGWaves;
    if (first < min(hi, base + nt))
      generic_run(tiles, first - base, min(hi - base, nt), R, i, g, q, A.scale_log2, st);
    base += nt;
  });
  float* sm = reinterpret_cast<float*>(lds);
  float* sl = reinterpret_cast<float*>(lds + kGLdsL);
  st.l = group_sum(st.l);
  if (g == 0) {
    sm[wave * kMaxGroup + i] = st.m;
    sl[wave * kMaxGroup + i] = st.l;
  }
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      *g_row(lds, wave, i, 16 * h + 4 * g + r) = float4v{st.O[h][0][r], st.O[h][1][r], st.O[h][2][r], st.O[h][3][r]};
  __syncthreads();
  const int hn = threadIdx.x >> 5, ch = threadIdx.x & 31;
  if (hn >= G) return;
  float M = -INFINITY, L = 0.f;
  float4v acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int w = 0; w < kGWaves; ++w) M = fmaxf(M, sm[w * kMaxGroup + hn]);
#pragma unroll
  for (int w = 0; w < kGWaves; ++w) {
    const float mw = sm[w * kMaxGroup + hn];
    const float f = mw == -INFINITY ? 0.f : exp2f(mw - M);
    L = fmaf(sl[w * kMaxGroup + hn], f, L);
    acc += *g_row(lds, w, hn, ch) * f;
  }
  if (A.n_splits == 1) {
    const float inv = L > 0.f ? 1.0f / L : 0.f;   // no valid slot: zeros
#pragma unroll
    for (int e = 0; e < 4; ++e) store_o(A.o, A.dt, (row0 + hn) * kHeadDim + 4 * ch + e, acc[e] * inv);
  } else {
    const size_t units = (size_t)A.pairs * A.n_splits * G;
    const size_t u = ((size_t)pair * A.n_splits + split) * G + hn;
    *reinterpret_cast<float4v*>(A.ws + u * kHeadDim + 4 * ch) = acc;
    if (ch == 0) {
      A.ws[units * kHeadDim + u] = M;
      A.ws[units * kHeadDim + units + u] = L;
    }
  }
}

// One workgroup per output row, whose four waves share its splits (each lane
// two channels): the partials combined in the log2 domain.
constexpr int kGMergeWaves = 4;
__global__ __launch_bounds__(64 * kGMergeWaves) void generic_merge_kernel(GArgs A) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const size_t row = blockIdx.x, pair = row / A.G, h = row - pair * A.G;
  const size_t units = (size_t)A.pairs * A.n_splits * A.G, base = pair * A.n_splits * A.G + h;
  const float* wm = A.ws + units * kHeadDim;
  float M = -INFINITY;
  for (int sp = lane; sp < A.n_splits; sp += 64) M = fmaxf(M, wm[base + (size_t)sp * A.G]);
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) M = fmaxf(M, __shfl_xor(M, off));
  float L = 0.f;
  float2v acc = {0.f, 0.f};
  for (int sp = wave; sp < A.n_splits; sp += kGMergeWaves) {
    const size_t u = base + (size_t)sp * A.G;
    const float mu = wm[u], f = mu == -INFINITY ? 0.f : exp2f(mu - M);
    L = fmaf(wm[units + u], f, L);
    acc += *reinterpret_cast<const float2v*>(A.ws + u * kHeadDim + 2 * lane) * f;
  }
  __shared__ float2v part[kGMergeWaves][64];
  __shared__ float part_l[kGMergeWaves];
  part[wave][lane] = acc;
  if (lane == 0) part_l[wave] = L;
  __syncthreads();
  if (wave != 0) return;
#pragma unroll
  for (int w = 1; w < kGMergeWaves; ++w) {
    acc += part[w][lane];
    L += part_l[w];
  }
  // row = b * H + head; no valid slot: zeros (L may be NaN)
  store_o(A.o, A.dt, row * kHeadDim + 2 * lane, L == 0.f ? 0.f : acc[0] / L);
  store_o(A.o, A.dt, row * kHeadDim + 2 * lane + 1, L == 0.f ? 0.f : acc[1] / L);
}

int gstatus() {
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? KVDEC_OK : (int)e;
}

template <class Src>
int launch_generic(const GArgs& A, const Src& S, hipStream_t st) {
  const dim3 grid((unsigned)A.pairs, (unsigned)A.n_splits);
  hipLaunchKernelGGL(generic_attn_kernel<Src>, grid, dim3(kGT), kGLdsBytes, st, A, S);
  const int rc = gstatus();
  if (rc != KVDEC_OK || A.n_splits == 1) return rc;
  hipLaunchKernelGGL(generic_merge_kernel, dim3((unsigned)(A.pairs * A.G)), dim3(64 * kGMergeWaves), 0, st, A);
  return gstatus();
}

// Splits: a workgroup per CU (they fill it), each with at least two tiles a
// wave, as many as the workspace holds.
constexpr int64_t kGUnits = 256, kGMinTiles = 2 * kGWaves;
void plan_splits(GArgs& A, size_t ws_bytes) {
  const int64_t tiles = A.n_tiles;
  int64_t sp = std::min<int64_t>((kGUnits + A.pairs - 1) / A.pairs, tiles / kGMinTiles);
  const size_t per_unit = (size_t)A.pairs * A.G * (kHeadDim + 2) * sizeof(float);
  sp = std::min<int64_t>(sp, A.ws ? (int64_t)(ws_bytes / per_unit) : 1);
  sp = std::max<int64_t>(sp, 1);
  A.per_split = (int)((tiles + sp - 1) / sp);
  A.n_splits = (int)((tiles + A.per_split - 1) / A.per_split);
}

int64_t tiles_of(int64_t n) { return (n + kGTile - 1) / kGTile; }

GArgs generic_args(const void* q, void* o, int dt, int64_t B, int32_t H, int32_t KVH, float sm_scale, void* ws) {
  GArgs A{};
  A.q = q;
  A.o = o;
  A.dt = dt;
  A.ws = static_cast<float*>(ws);
  A.pairs = B * KVH;
  A.H = H;
  A.KVH = KVH;
  A.G = H / KVH;
  A.scale_log2 = (float)((double)sm_scale * 1.4426950408889634);
  return A;
}

template <int DT>
int launch_rows(const GArgs& A, const void* k, const void* v, int64_t rows, hipStream_t st) {
  typedef typename GElt<DT>::T T;
  return launch_generic(A, GRowsSrc<DT>{static_cast<const T*>(k), static_cast<const T*>(v), (int)rows}, st);
}

template <int RT, int PF, bool SMALL>
int launch_kivi(const GArgs& A, const void* k_res, const void* v_res, const void* const* kivi, int32_t sink,
                int32_t res_rows, int32_t win_tok, int32_t group, int32_t bits, hipStream_t st) {
  GKiviSrc<RT, PF, SMALL> S{};
  S.kres = static_cast<const typename GElt<RT>::T*>(k_res);
  S.vres = static_cast<const typename GElt<RT>::T*>(v_res);
  for (int r = 0; r < 2; ++r) {
    const int base = 6 * r;
    S.kp[r] = static_cast<const uint8_t*>(kivi[base]);
    S.ks[r] = static_cast<const _Float16*>(kivi[base + 1]);
    S.kz[r] = static_cast<const _Float16*>(kivi[base + 2]);
    S.vp[r] = static_cast<const uint8_t*>(kivi[base + 3]);
    S.vs[r] = static_cast<const _Float16*>(kivi[base + 4]);
    S.vz[r] = static_cast<const _Float16*>(kivi[base + 5]);
  }
  S.sink = sink;
  S.win_tok = win_tok;
  S.res_rows = res_rows;
  S.group = group;
  S.bits = bits;
  return launch_generic(A, S, st);
}

template <int RT>
int launch_kivi_width(const GArgs& A, const void* k_res, const void* v_res, const void* const* kivi, int32_t sink,
                      int32_t res_rows, int32_t win_tok, int32_t group, int32_t bits, hipStream_t st) {
  auto run = [&](auto launch) {
    return launch(A, k_res, v_res, kivi, sink, res_rows, win_tok, group, bits, st);
  };
  switch (8 / bits) {   // codes per byte; a group holds whole bytes
    case 8: return run(launch_kivi<RT, 8, false>);
    case 4: return run(launch_kivi<RT, 4, false>);
    case 2: return group < 4 ? run(launch_kivi<RT, 2, true>) : run(launch_kivi<RT, 2, false>);
    default: return group < 4 ? run(launch_kivi<RT, 1, true>) : run(launch_kivi<RT, 1, false>);
  }
}

}  // namespace

int generic_rows_decode(const void* q, const void* k, const void* v, void* o, int dtype, int64_t B,
                        int32_t H, int32_t KVH, int64_t rows, SlotRanges R, const int32_t* lens,
                        bool sparse, int32_t window, int32_t sink, int32_t layout, float sm_scale,
                        void* ws, size_t ws_bytes, hipStream_t stream) {
  GArgs A = generic_args(q, o, dtype, B, H, KVH, sm_scale, ws);
  A.n_tiles = (int)tiles_of(rows);
  A.range = GRange{R, lens, sparse, window, sink, layout, rows};
  plan_splits(A, ws_bytes);
  switch (dtype) {
    case KVDEC_F32: return launch_rows<KVDEC_F32>(A, k, v, rows, stream);
    case KVDEC_BF16: return launch_rows<KVDEC_BF16>(A, k, v, rows, stream);
    case KVDEC_F16: return launch_rows<KVDEC_F16>(A, k, v, rows, stream);
    default: return KVDEC_E_DTYPE;
  }
}

int generic_kivi_decode(const void* q, const void* k_res, const void* v_res, const void* const* kivi,
                        void* o, int q_dtype, int res_dtype, const int32_t* lens, int64_t B, int32_t H,
                        int32_t KVH, int64_t seq_len, int32_t window, int32_t sink, int32_t res_rows,
                        int32_t win_tok, int32_t group, int32_t bits, float sm_scale, void* ws,
                        size_t ws_bytes, hipStream_t stream) {
  GArgs A = generic_args(q, o, q_dtype, B, H, KVH, sm_scale, ws);
  A.n_tiles = (int)(tiles_of(win_tok) + tiles_of(sink) + tiles_of(res_rows));
  A.range = GRange{sparse_ranges(seq_len, window, sink, KVDEC_LAYOUT_LINEAR), lens, true, window, sink,
                   KVDEC_LAYOUT_LINEAR, (int64_t)sink + window};
  plan_splits(A, ws_bytes);
  auto run = [&](auto launch) {
    return launch(A, k_res, v_res, kivi, sink, res_rows, win_tok, group, bits, stream);
  };
  switch (res_dtype) {
    case KVDEC_F16: return run(launch_kivi_width<KVDEC_F16>);
    case KVDEC_BF16: return run(launch_kivi_width<KVDEC_BF16>);
    case KVDEC_F32: return run(launch_kivi_width<KVDEC_F32>);
    default: return KVDEC_E_DTYPE;
  }
}

}  // namespace kvdec
