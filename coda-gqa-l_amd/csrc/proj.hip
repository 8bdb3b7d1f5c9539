// Projection front end of the bounded layer on gfx950: one GEMM of the
// token rows against the packed [q | k | v | lambda | write-gate] weights
// (bf16 MFMA, fp32 accumulation), with the epilogues of the reference's
// eager ops fused into the tile's store (attention.py:396-410, 592-608):
//   q, v    (+ bias) rounded to bf16;
//   k       (+ bias) rounded to bf16, then RoPE with the tables of the row's
//           position, one bf16 rounding per op (primitives.py:83-113);
//   lambda  sigmoid(bf16(acc + bias)) in bf16;
//   gate    sigmoid(bf16(acc + bias)) in bf16, stored as float32.
// The tile computes C^T = W X^T: MFMA A operand = weight rows (features), B
// operand = token rows, so each lane holds 4 consecutive features of one
// token (the RoPE pairs of a head sit in one lane; the half-split layout
// is packed with each pair (i, i + Dh/2) on adjacent weight rows).
#include "common.h"

#include <climits>
#include <type_traits>

namespace coda {

typedef __bf16 pbf16x8_t __attribute__((ext_vector_type(8)));
typedef float pf32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t pu32x4 __attribute__((ext_vector_type(4)));

// dword 3 of a raw buffer resource on gfx9 (32-bit data format, no swizzle)
static constexpr int kProjBufWord3 = 0x00020000;
static constexpr int kProjKT = 64;        // D of coda_project: whole multiples

__device__ __forceinline__ float proj_sigmoid(float x) { return 1.f / (1.f + expf(-x)); }

// Four consecutive elements to memory: one 8-byte (bf16) or 16-byte (fp32,
// any 4-byte address) store
typedef float pf4u __attribute__((ext_vector_type(4), aligned(4)));
__device__ __forceinline__ void proj_put4(bf16_t* p, const pf32x4& v) {
  using E = Elt<bf16_t>;
  uint2 w;
  w.x = (uint32_t)E::st(v[0]) | ((uint32_t)E::st(v[1]) << 16);
  w.y = (uint32_t)E::st(v[2]) | ((uint32_t)E::st(v[3]) << 16);
  *reinterpret_cast<uint2*>(p) = w;
}
__device__ __forceinline__ void proj_put4(float* p, const pf32x4& v) { *reinterpret_cast<pf4u*>(p) = v; }

// The layer's own parameters (coda_proj_params) as sections of the packed
// feature order: q, k, v, lambda, gate
template <typename T>
struct ParamRows {
  const T* w[5];
  const T* b[5];
  int64_t sm[5];
  int start[5];  // first feature of a section; INT_MAX: not there
  int Dh;
  int halves;  // k rows of a head in the order (0, half, 1, half + 1, ..): half-split RoPE
  __device__ __forceinline__ int section(int f) const {
    int s = 0;
#pragma unroll
    for (int i = 1; i < 5; ++i) s = f >= start[i] ? i : s;
    return s;
  }
  // a[s], from registers
  template <typename V>
  __device__ __forceinline__ V pick(const V (&a)[5], int s) const {
    V v = a[0];
#pragma unroll
    for (int i = 1; i < 5; ++i) v = s == i ? a[i] : v;
    return v;
  }
  // row of section s that feature f is
  __device__ __forceinline__ int row_in(int s, int f) const {
    int r = f - pick(start, s);
    if (halves && s == 1) {
      const int c = r % Dh;
      r = r - c + (c >> 1) + (c & 1) * (Dh / 2);
    }
    return r;
  }
  // row of feature f0 + r16, at most last; f0, last the same in every lane:
  // in most blocks of 16 the section is too (200 vector instructions before
  // the first load cost 0.4 us)
  __device__ __forceinline__ const T* row16(int f0, int r16, int last) const {
    const int s0 = section(min(f0, last)), f = min(f0 + r16, last);
    if (s0 == section(min(f0 + 15, last))) return pick(w, s0) + row_in(s0, f) * pick(sm, s0);
    const int s = section(f);
    return pick(w, s) + row_in(s, f) * pick(sm, s);
  }
  __device__ __forceinline__ float bias1(int f) const {
    const int s = section(f);
    const T* p = pick(b, s);
    return p ? Elt<T>::ld(p[row_in(s, f)]) : 0.f;
  }
  // biases of features f .. f + 3 (f a multiple of 4; past the last: any)
  __device__ __forceinline__ pf32x4 bias4(int f, int last) const {
    const int s = section(f);
    pf32x4 v{0.f, 0.f, 0.f, 0.f};
    if (s < 3) {
      const T* p = pick(b, s);
      if (!p) return v;
      const int r = row_in(s, f), hs = halves && s == 1 ? Dh / 2 : 0;
      const int o1 = hs ? hs : 1, o2 = hs ? 1 : 2, o3 = hs ? hs + 1 : 3;
      return pf32x4{Elt<T>::ld(p[r]), Elt<T>::ld(p[r + o1]), Elt<T>::ld(p[r + o2]), Elt<T>::ld(p[r + o3])};
    }
    const T* lb = b[3];
    const T* gb = b[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int ff = min(f + e, last);
      const bool gate = ff >= start[4];
      const T* p = gate ? gb : lb;
      if (p) v[e] = Elt<T>::ld(p[ff - (gate ? start[4] : start[3])]);
    }
    return v;
  }
};
// Angle tables made by the launch itself (pointers null: given in the
// descriptor, or not asked for)
struct FrontTables {
  const void* inv_freq;
  int inv_dtype;
  int64_t p0;
  void* rope_cos;
  void* rope_sin;
  const void* theta;
  int theta_dtype, n_theta;
  void* theta_cos;
  void* theta_sin;
};

// Epilogue of features f .. f + 3 (f a multiple of 4) of token row m:
// the fp32 accumulators plus bias, rounded and routed to q / k (RoPE) / v /
// lambda / gate
// PARAMS: biases from the parameters, the launch's own tables; else one
// packed fp32 bias vector (zero where a linear has none) and given tables
template <typename T, bool PARAMS>
struct FrontEpilogue {
  coda_proj_desc d;
  FrontTables tab;
  template <typename Src>
  __device__ __forceinline__ pf32x4 bias4(const Src& W, int f, int last) const {
    if constexpr (PARAMS) {
      return W.bias4(f, last);
    } else {
      if (f + 3 <= last) {
        const float4 v = *reinterpret_cast<const float4*>(d.bias + f);
        return pf32x4{v.x, v.y, v.z, v.w};
      }
      return pf32x4{d.bias[f], d.bias[min(f + 1, last)], d.bias[min(f + 2, last)], d.bias[min(f + 3, last)]};
    }
  }
  template <typename Src>
  __device__ __forceinline__ void operator()(const Src& W, int f, int m, pf32x4 v) const {
    using E = Elt<T>;
    const int Fq = d.H * d.Dh, Fk = d.Hkv * d.Dh, half = d.Dh / 2;
    const int o_k = Fq, o_v = Fq + Fk, o_l = Fq + 2 * Fk, o_g = o_l + d.H;
    v += bias4(W, f, o_g - (d.gate ? 0 : 1));
    if (f + 3 < o_k) {  // q
      proj_put4((T*)d.q + (int64_t)m * d.q_sm + f, v);
    } else if (f >= o_k && f + 3 < o_v) {  // k: two RoPE pairs
      const int kf = f - o_k, hk = kf / d.Dh, c = kf % d.Dh, prow = m % d.L;
      const bool inter = d.rope_interleaved != 0;
      const T* cs = (const T*)d.rope_cos;
      const T* sn = (const T*)d.rope_sin;
      T* krow = (T*)d.k + (int64_t)m * d.k_sm + (int64_t)hk * d.Dh;
      float r[4];
#pragma unroll
      for (int pp = 0; pp < 2; ++pp) {
        const int p = c / 2 + pp;  // pair index
        float cc, ss;
        if constexpr (!PARAMS) {
          cc = E::ld(cs[(int64_t)prow * half + p]);
          ss = E::ld(sn[(int64_t)prow * half + p]);
        } else if (tab.inv_freq) {
          const float2 t = rope_angle<T>(tab.inv_freq, tab.inv_dtype, tab.p0 + prow, p);
          cc = t.x;
          ss = t.y;
        } else {
          cc = E::ld(cs[(int64_t)prow * half + p]);
          ss = E::ld(sn[(int64_t)prow * half + p]);
        }
        rope_pair_t<T>(E::rnd(v[2 * pp]), E::rnd(v[2 * pp + 1]), cc, ss, inter, r[2 * pp], r[2 * pp + 1]);
      }
      if (inter) {
        proj_put4(krow + c, pf32x4{r[0], r[1], r[2], r[3]});
      } else {  // packed pairs (p, p + half): channels c/2, c/2 + 1 and the same + half
        const int p = c / 2;
        krow[p] = E::st(r[0]);
        krow[p + 1] = E::st(r[2]);
        krow[p + half] = E::st(r[1]);
        krow[p + half + 1] = E::st(r[3]);
      }
    } else if (f >= o_v && f + 3 < o_l) {  // v
      proj_put4((T*)d.v + (int64_t)m * d.v_sm + (f - o_v), v);
    } else {  // lambda / write gate, one feature at a time
#pragma unroll
      for (int rr = 0; rr < 4; ++rr) {
        const int ff = f + rr;
        if (ff < o_l || ff >= o_g + (d.gate ? 1 : 0)) continue;
        const float lin = E::rnd(v[rr]);
        const float sg = E::rnd(proj_sigmoid(lin));
        if (ff < o_g) ((T*)d.lam)[(int64_t)m * d.lam_sm + (ff - o_l)] = E::st(sg);
        else d.g[m] = sg;
      }
    }
  }
  // no gate column: the gate is 1; the tables that the launch leaves
  __device__ __forceinline__ void once(int t) const {
    if (!d.gate && t < d.M) d.g[t] = 1.f;
    if constexpr (PARAMS) {
      const int half = d.Dh / 2;
      if (tab.inv_freq)
        for (int i = t; i < d.L * half; i += 512) {
          const float2 a = rope_angle<T>(tab.inv_freq, tab.inv_dtype, tab.p0 + i / half, i % half);
          ((T*)tab.rope_cos)[i] = Elt<T>::st(a.x);
          ((T*)tab.rope_sin)[i] = Elt<T>::st(a.y);
        }
      if (tab.theta)
        for (int i = t; i < tab.n_theta; i += 512) {
          const float2 a = cos_sin_of<T>(angle_ld(tab.theta, tab.theta_dtype, i), tab.theta_dtype);
          ((T*)tab.theta_cos)[i] = Elt<T>::st(a.x);
          ((T*)tab.theta_sin)[i] = Elt<T>::st(a.y);
        }
    }
  }
};

// Epilogue of a plain linear layer: out = acc + bias, one rounding
template <typename T, typename BT>
struct LinearEpilogue {
  T* out;
  const BT* bias;  // or null
  int64_t o_sm;
  int n_feat;
  template <typename Src>
  __device__ __forceinline__ void operator()(const Src&, int f, int m, pf32x4 v) const {
    T* row = out + (int64_t)m * o_sm;
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] += bias && f + e < n_feat ? Elt<BT>::ld(bias[f + e]) : 0.f;
    if (f + 3 < n_feat) {
      proj_put4(row + f, v);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (f + e < n_feat) row[f + e] = Elt<T>::st(v[e]);
    }
  }
  __device__ __forceinline__ void once(int) const {}
};

// Few token rows (M <= 128): the weights are the traffic.  A workgroup owns
// 16 RB features over all of K: its 8 waves split K and stream their weight
// rows and the token rows of that range straight from memory into MFMA
// fragments, one 16 x 16 accumulator per 16 features and 16 tokens; the
// partials meet in LDS and are summed in wave order (deterministic), then
// the epilogue.  No workspace, no cross-workgroup exchange.  Weights cross
// HBM once; the token rows are read by every workgroup from L2.
// K goes in pairs of 64-byte steps: a lane's two 16-byte pieces of a row
// come from the two halves of one 128-byte line, requested back to back.
// Measured (bf16, tiles, weights not in cache): 6177 x 4096 M = 1 12.2 us, M
// = 16 13.3 us (4.1 / 3.8 TB/s), 10305 x 8192 M = 1 31.3 us (5.4 TB/s).
// The weights: in fragment tiles (TileRows; coda_project_pack), where the
// operand of row block fb at k-step ks is the KiB at (fb D/32 + ks) 512
// elements (bf16), lane l's 16 bytes at 16 l; or rows as they lie (MatRows:
// one matrix; ParamRows: the layer's own parameters), at any element address.
// A load of tiles is a KiB in one piece, one of rows 16 pieces of 64 bytes:
// 6177 x 4096 M = 1 13.3 us (tiles 12.2), M = 64 22.3 (18.2), 10305 x 8192 M =
// 128 63.3 (53.7), 4096 x 4096 M = 1 8.7 (7.9; the library 14.9).
template <typename T>
struct TileRows {
  static constexpr bool kTiles = true;
  const T* w;
};
template <typename T>
struct MatRows {
  const T* w;
  int64_t sm;
  __device__ __forceinline__ const T* row16(int f0, int r16, int last) const { return w + min(f0 + r16, last) * sm; }
};
template <typename Src>
struct IsTiles : std::false_type {};
template <typename T>
struct IsTiles<TileRows<T>> : std::true_type {};
// a row's 16 bytes at any element address
typedef uint32_t pu32x4u __attribute__((ext_vector_type(4), aligned(2)));
template <typename T>
__device__ __forceinline__ pf32x4 rows_mfma(const pu32x4& a, const pu32x4& b, pf32x4 c) {
  if constexpr (sizeof(T) == 2) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(pbf16x8_t, a), __builtin_bit_cast(pbf16x8_t, b),
                                                   c, 0, 0, 0);
  } else {
    const pf32x4 x = __builtin_bit_cast(pf32x4, a), y = __builtin_bit_cast(pf32x4, b);
#pragma unroll
    for (int e = 0; e < 4; ++e) c = __builtin_amdgcn_mfma_f32_16x16x4f32(x[e], y[e], c, 0, 0, 0);
    return c;
  }
}
// waves whose partials meet in LDS at once: all 8, or 4 after the upper 4
// have handed theirs to the lower 4
template <int MT, int RB>
struct RowsLds {
  static constexpr int kWaves = RB * MT <= 8 ? 8 : 4;
  static constexpr size_t kBytes = (size_t)kWaves * RB * MT * 64 * sizeof(pf32x4);
};
// One dword of each 64 bytes of the epilogue's arguments, read before the
// products: the compiler loads them where they are used, after the products,
// in several dependent rounds, each a miss of the scalar cache then
template <typename V>
__device__ __forceinline__ void touch_args(const V& v) {
  const int* p = reinterpret_cast<const int*>(&v);
#pragma unroll
  for (int i = 0; i < (int)(sizeof(V) / 4); i += 16) asm volatile("" ::"s"(p[i]));
}
// The waves' partials (accumulators of 16 features x 16 tokens each), summed in
// wave order, and the epilogue
template <int MT, int RB, typename Src, typename Epi>
__device__ __forceinline__ void rows_finish(pf32x4 (&acc)[RB][MT], char* smem, int n_feat, int M, const Src& W,
                                            const Epi& epi) {
  pf32x4* part = reinterpret_cast<pf32x4*>(smem);
  const int t = threadIdx.x, lane = t & 63, wv = __builtin_amdgcn_readfirstlane(t >> 6), f0 = blockIdx.x * 16 * RB;
  constexpr int NWv = RowsLds<MT, RB>::kWaves;
  if constexpr (NWv == 4) {
    if (wv >= 4)
#pragma unroll
      for (int i = 0; i < RB; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j) part[(((wv - 4) * RB + i) * MT + j) * 64 + lane] = acc[i][j];
    __syncthreads();
    if (wv < 4)
#pragma unroll
      for (int i = 0; i < RB; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j) acc[i][j] += part[((wv * RB + i) * MT + j) * 64 + lane];
    __syncthreads();
  }
  if (wv < NWv)
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
      for (int j = 0; j < MT; ++j) part[((wv * RB + i) * MT + j) * 64 + lane] = acc[i][j];
  __syncthreads();
  if (blockIdx.x == 0) epi.once(t);
  // item 64 (MT i + j) + l: features f0 + 16 i + 4 (l / 16) .. + 3 of token
  // 16 j + l % 16
  for (int item = t; item < 64 * MT * RB; item += 512) {
    const int ij = item >> 6, l = item & 63;
    pf32x4 sum = part[ij * 64 + l];
#pragma unroll
    for (int w = 1; w < NWv; ++w) sum += part[(w * RB * MT + ij) * 64 + l];
    const int m = 16 * (ij % MT) + (l & 15), f = f0 + 16 * (ij / MT) + 4 * (l >> 4);
    if (m < M && f < n_feat) epi(W, f, m, sum);
  }
}

template <typename T, int MT, int RB, typename Src, typename Epi>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2))) void proj_rows(
    const Src W, int n_feat, int D, const T* __restrict__ X, int64_t x_sm, int M, const Epi epi) {
  constexpr bool TILED = IsTiles<Src>::value;
  extern __shared__ __attribute__((aligned(16))) char rows_smem[];
  // pairs of k-steps in flight ahead of the products
  constexpr int LP = RB * MT <= 3 ? 4 : RB * MT <= 12 ? 2 : 1;
  const int f0 = blockIdx.x * 16 * RB;
  const int t = threadIdx.x, lane = t & 63, wv = __builtin_amdgcn_readfirstlane(t >> 6), r16 = lane & 15, kq = lane >> 4;
  const int pairs = D * (int)sizeof(T) / 128, p0 = pairs * wv / 8, np = pairs * (wv + 1) / 8 - p0;
  // byte addresses of this lane's first piece of pair 0; WP / WH: bytes from
  // a pair to the next, from its first half to its second
  constexpr int WP = TILED ? 2048 : 128, WH = TILED ? 1024 : 64;
  const char* wr[RB];
#pragma unroll
  for (int i = 0; i < RB; ++i)
    if constexpr (TILED)
      wr[i] = (const char*)W.w + ((int64_t)min(f0 / 16 + i, (n_feat + 15) / 16 - 1) * pairs + p0) * 2048 + 16 * lane;
    else
      wr[i] = (const char*)W.row16(f0 + 16 * i, r16, n_feat - 1) + 128 * p0 + 16 * kq;
  const char* xr[MT];
#pragma unroll
  for (int j = 0; j < MT; ++j) xr[j] = (const char*)(X + (int64_t)min(16 * j + r16, M - 1) * x_sm) + 128 * p0 + 16 * kq;
  pu32x4 a[LP][RB][2], b[LP][MT][2];
  auto load = [&](int u, int p) {
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        a[u][i][h] = *reinterpret_cast<const typename std::conditional<TILED, pu32x4, pu32x4u>::type*>(wr[i] + WP * p + WH * h);
#pragma unroll
    for (int j = 0; j < MT; ++j)
#pragma unroll
      for (int h = 0; h < 2; ++h) b[u][j][h] = *reinterpret_cast<const pu32x4*>(xr[j] + 128 * p + 64 * h);
  };
  pf32x4 acc[RB][MT];
#pragma unroll
  for (int i = 0; i < RB; ++i)
#pragma unroll
    for (int j = 0; j < MT; ++j) acc[i][j] = pf32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int u = 0; u < LP; ++u)
    if (u < np) load(u, u);
  touch_args(epi);
  auto products = [&](const pu32x4 (&as)[RB][2], const pu32x4 (&bs)[MT][2]) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int i = 0; i < RB; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j) acc[i][j] = rows_mfma<T>(as[i][h], bs[j][h], acc[i][j]);
  };
  int p = 0;
  for (; p + 2 * LP <= np; p += LP) {
#pragma unroll
    for (int u = 0; u < LP; ++u) {
      products(a[u], b[u]);
      load(u, p + u + LP);
    }
  }
#pragma unroll
  for (int u = 0; u < 2 * LP; ++u) {
    if (p + u >= np) break;
    products(a[u % LP], b[u % LP]);
    if (p + u + LP < np) load(u % LP, p + u + LP);
  }
  rows_finish<MT, RB>(acc, rows_smem, n_feat, M, W, epi);
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rows_rsrc(const char* p, int nbytes) {
  const uint64_t v = (uint64_t)p;
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
  return __builtin_amdgcn_make_buffer_rsrc((void*)(((uint64_t)hi << 32) | lo), (short)0,
                                           __builtin_amdgcn_readfirstlane(nbytes), kProjBufWord3);
}
// The same for 17 .. 128 rows and K in whole chunks (8 waves x CS steps of 64
// bytes): the token rows pass through LDS.  Operand loads straight from
// memory take 16 rows' 64-byte pieces at a power-of-two stride, a quarter of
// the rate of contiguous ones, and with 64 rows they outweigh the weights
// (6184 x 4096, M = 64: 23.7 us with them, 18.8 us here; 10305 x 8192, M =
// 128: 83 against 52.7 us; 4096 x 4096, M = 32: 12.1 against 11.1 us).  Per chunk and 16
// tokens a wave loads its own part of the rows as CS * 64 contiguous bytes a
// row into registers (two such slabs in flight), writes it to its LDS slab
// and reads the operands back; 16-byte pieces are swizzled by the row, so
// writes and reads spread over the banks.  The slab is the wave's alone and
// LDS serves a wave in order: no barrier.  The next chunk's weights load
// while this chunk's products run.  Same sums in the same order as proj_rows.
template <typename T, int MT, int RB, int CS, typename Src, typename Epi>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2))) void proj_rows_lds(
    const Src W, int n_feat, int D, const T* __restrict__ X, int64_t x_sm, int M, const Epi epi) {
  constexpr bool TILED = IsTiles<Src>::value;
  extern __shared__ __attribute__((aligned(16))) char rows_smem[];
  constexpr int RBY = CS * 64, PCS = RBY / 16, NI = 16 * PCS / 64, RPI = 64 / PCS;  // row bytes, pieces; loads a slab, rows a load
  const int f0 = blockIdx.x * 16 * RB;
  const int t = threadIdx.x, lane = t & 63, wv = __builtin_amdgcn_readfirstlane(t >> 6), r16 = lane & 15, kq = lane >> 4;
  const int steps = D * (int)sizeof(T) / 64, nc = steps / (8 * CS), s0 = nc * CS * wv;
  char* slab = rows_smem + wv * 16 * RBY;
  // tiles and token rows through raw buffer resources: 32-bit offsets, and
  // token rows past the last read 0 without touching memory
  const int nfb = (n_feat + 15) / 16;
  const __amdgpu_buffer_rsrc_t rx = rows_rsrc((const char*)X, (int)(((M - 1) * x_sm + D) * (int)sizeof(T)));
  __amdgpu_buffer_rsrc_t rw;
  int wo[RB];
  const char* wr[RB];
  if constexpr (TILED) {
    rw = rows_rsrc((const char*)W.w + (int64_t)(f0 / 16) * steps * 1024, RB * steps * 1024);
#pragma unroll
    for (int i = 0; i < RB; ++i) wo[i] = (min(f0 / 16 + i, nfb - 1) - f0 / 16) * steps * 1024 + s0 * 1024;
  } else {
#pragma unroll
    for (int i = 0; i < RB; ++i)
      wr[i] = (const char*)W.row16(f0 + 16 * i, r16, n_feat - 1) + 64 * s0 + 16 * kq;
  }
  const int lr = lane / PCS, lp = lane % PCS, xrow = (int)x_sm * (int)sizeof(T);
  const int xo = 64 * s0 + 16 * lp + lr * xrow;
  pu32x4 a0[CS][RB], a1[CS][RB], x0[NI], x1[NI];
  auto load_w = [&](pu32x4 (&w)[CS][RB], int c) {
#pragma unroll
    for (int s = 0; s < CS; ++s)
#pragma unroll
      for (int i = 0; i < RB; ++i) {
        if constexpr (TILED) w[s][i] = __builtin_amdgcn_raw_buffer_load_b128(rw, 16 * lane, wo[i] + (c * CS + s) * 1024, 0);
        else w[s][i] = *reinterpret_cast<const pu32x4u*>(wr[i] + c * RBY + 64 * s);
      }
  };
  // slab (chunk c, tokens 16 j ..)
  auto load_x = [&](pu32x4 (&v)[NI], int c, int j) {
    const int cb = xo + c * RBY;
#pragma unroll
    for (int i = 0; i < NI; ++i) v[i] = __builtin_amdgcn_raw_buffer_load_b128(rx, cb + (16 * j + RPI * i) * xrow, 0, 0);
  };
  pf32x4 acc[RB][MT];
#pragma unroll
  for (int i = 0; i < RB; ++i)
#pragma unroll
    for (int j = 0; j < MT; ++j) acc[i][j] = pf32x4{0.f, 0.f, 0.f, 0.f};
  auto tokens = [&](int c, int j, pu32x4 (&v)[NI], const pu32x4 (&w)[CS][RB], pf32x4 (&ac)[RB][MT]) {
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int row = RPI * i + lr;
      *reinterpret_cast<pu32x4*>(slab + row * RBY + ((lp ^ row) & (PCS - 1)) * 16) = v[i];
    }
    // slab j + 2 of the walk over (chunk, tokens); past the end: the last again
    load_x(v, j + 2 < MT ? c : min(c + 1, nc - 1), (j + 2) % MT);
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int s = 0; s < CS; ++s) {
      const pu32x4 b = *reinterpret_cast<const pu32x4*>(slab + r16 * RBY + (((4 * s + kq) ^ r16) & (PCS - 1)) * 16);
#pragma unroll
      for (int i = 0; i < RB; ++i) ac[i][j] = rows_mfma<T>(w[s][i], b, ac[i][j]);
    }
    __builtin_amdgcn_wave_barrier();
  };
  auto chunk = [&](int c, pu32x4 (&w)[CS][RB], pu32x4 (&wn)[CS][RB]) {
    load_w(wn, min(c + 1, nc - 1));
#pragma unroll
    for (int j = 0; j < MT; j += 2) {
      tokens(c, j, x0, w, acc);
      tokens(c, j + 1, x1, w, acc);
    }
  };
  static_assert(MT % 2 == 0, "slabs alternate between two register sets");
  load_w(a0, 0);
  load_x(x0, 0, 0);
  load_x(x1, 0, 1);
  touch_args(epi);
  int c = 0;
  for (; c + 1 < nc; c += 2) {
    chunk(c, a0, a1);
    chunk(c + 1, a1, a0);
  }
  if (c < nc) chunk(c, a0, a1);
  __syncthreads();
  rows_finish<MT, RB>(acc, rows_smem, n_feat, M, W, epi);
}

template <typename T, int MT, int RB, typename Src, typename Epi>
static int launch_rows_k(const Src& W, int n_feat, int D, const T* X, int64_t x_sm, int M, const Epi& epi,
                         hipStream_t st, const char* who) {
  constexpr size_t lds = RowsLds<MT, RB>::kBytes;
  const int rc = lds_limit<proj_rows<T, MT, RB, Src, Epi>>(lds, who);
  if (rc) return rc;
  hipLaunchKernelGGL((proj_rows<T, MT, RB, Src, Epi>), dim3((n_feat + 16 * RB - 1) / (16 * RB)), dim3(512), lds, st, W,
                     n_feat, D, X, x_sm, M, epi);
  return check_launch("proj_rows");
}
// Features a workgroup: the RB (1 .. 3) of the fewest 16-feature turns, ceil
// (workgroups / CUs) * RB, and of these the largest (it reads the token rows
// least often)
static int rows_rb(int n_feat) {
  const int cus = device_cus(), fb = (n_feat + 15) / 16;
  int best = 1, turns = INT_MAX;
  for (int rb = 1; rb <= 3; ++rb) {
    const int n = ((fb + rb - 1) / rb + cus - 1) / cus * rb;
    if (n <= turns) {
      turns = n;
      best = rb;
    }
  }
  return best;
}
template <typename T, int MT, int RB, typename Src, typename Epi>
static int launch_rows_lds(const Src& W, int n_feat, int D, const T* X, int64_t x_sm, int M, const Epi& epi,
                           hipStream_t st, const char* who) {
  // steps a chunk: as many as the accumulators (and the row addresses of
  // weights that are not tiles) leave registers for
  constexpr int CS = RB * MT <= (IsTiles<Src>::value ? 4 : 3) || RB == 1 && MT == 4 ? 8 : RB * MT <= 16 ? 4 : 2;
  constexpr size_t slabs = (size_t)8 * 16 * CS * 64;
  constexpr size_t lds = slabs > RowsLds<MT, RB>::kBytes ? slabs : RowsLds<MT, RB>::kBytes;
  const int rc = lds_limit<proj_rows_lds<T, MT, RB, CS, Src, Epi>>(lds, who);
  if (rc) return rc;
  hipLaunchKernelGGL((proj_rows_lds<T, MT, RB, CS, Src, Epi>), dim3((n_feat + 16 * RB - 1) / (16 * RB)), dim3(512), lds,
                     st, W, n_feat, D, X, x_sm, M, epi);
  return check_launch("proj_rows_lds");
}
template <typename T, int MT, typename Src, typename Epi>
static int launch_rows_mt(const Src& W, int n_feat, int D, const T* X, int64_t x_sm, int M, const Epi& epi,
                          hipStream_t st, const char* who) {
  if constexpr (MT > 1) {
    // (token rows within a 31-bit offset)
    if (D * sizeof(T) % 4096 == 0 && x_sm >= 0 && (M * x_sm + D) * (int64_t)sizeof(T) < INT_MAX) {
      switch (rows_rb(n_feat)) {
        case 1: return launch_rows_lds<T, MT, 1>(W, n_feat, D, X, x_sm, M, epi, st, who);
        case 2: return launch_rows_lds<T, MT, 2>(W, n_feat, D, X, x_sm, M, epi, st, who);
        default: return launch_rows_lds<T, MT, 3>(W, n_feat, D, X, x_sm, M, epi, st, who);
      }
    }
  }
  switch (rows_rb(n_feat)) {
    case 1: return launch_rows_k<T, MT, 1>(W, n_feat, D, X, x_sm, M, epi, st, who);
    case 2: return launch_rows_k<T, MT, 2>(W, n_feat, D, X, x_sm, M, epi, st, who);
    default: return launch_rows_k<T, MT, 3>(W, n_feat, D, X, x_sm, M, epi, st, who);
  }
}
template <typename T, typename Src, typename Epi>
static int launch_rows(const Src& W, int n_feat, int D, const T* X, int64_t x_sm, int M, const Epi& epi,
                       hipStream_t st, const char* who) {
  if (M <= 16) return launch_rows_mt<T, 1>(W, n_feat, D, X, x_sm, M, epi, st, who);
  if (M <= 32) return launch_rows_mt<T, 2>(W, n_feat, D, X, x_sm, M, epi, st, who);
  if (M <= 64) return launch_rows_mt<T, 4>(W, n_feat, D, X, x_sm, M, epi, st, who);
  return launch_rows_mt<T, 8>(W, n_feat, D, X, x_sm, M, epi, st, who);
}
// one thread per 16-byte piece of the tiled copy; row_pieces: 16-byte pieces
// of a row
__global__ __launch_bounds__(256) void proj_pack_kernel(const char* __restrict__ w, int n_feat, int row_pieces,
                                                        int64_t row_bytes, uint4* __restrict__ out, int64_t n_pieces) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n_pieces) return;
  const int l = (int)(i & 63), r = l & 15, q = l >> 4;
  const int64_t tile = i >> 6;
  const int ksteps = row_pieces / 4;
  const int64_t fb = tile / ksteps;
  const int ks = (int)(tile % ksteps);
  const int64_t f = fb * 16 + r;
  uint4 v = make_uint4(0u, 0u, 0u, 0u);
  if (f < n_feat) v = *reinterpret_cast<const uint4*>(w + f * row_bytes + 64 * ks + 16 * q);
  out[i] = v;
}
static int launch_pack(int esz, const void* w, int n_feat, int D, int64_t w_sm, void* out, hipStream_t st) {
  // (rows padded to a multiple of 64)
  const int row_pieces = D * esz / 16;
  const int64_t n_pieces = (int64_t)((n_feat + 63) / 64) * 64 * row_pieces;
  hipLaunchKernelGGL(proj_pack_kernel, dim3((unsigned)((n_pieces + 255) / 256)), dim3(256), 0, st, (const char*)w, n_feat,
                     row_pieces, w_sm * esz, (uint4*)out, n_pieces);
  return check_launch("proj_pack_kernel");
}

// D of the tiled weights that coda_project_pack makes
static bool rows_path(int D) {
  return D >= 512 && D <= 8192 && D % 256 == 0 && ((D / 256) & (D / 256 - 1)) == 0;
}

// What the front-end entries ask of a descriptor (packed: of its w and bias too)
static int check_project(const coda_proj_desc* d, const char* who, bool packed) {
  CODA_REQUIRE(d->D > 0 && d->D % kProjKT == 0, "%s: D=%d must be a positive multiple of %d", who, d->D, kProjKT);
  CODA_REQUIRE(d->H > 0 && d->Hkv > 0 && d->Dh > 0 && d->Dh % 4 == 0 && d->L > 0,
               "%s: bad sizes H=%d Hkv=%d Dh=%d L=%d", who, d->H, d->Hkv, d->Dh, d->L);
  CODA_REQUIRE(d->x && d->q && d->k && d->v && d->lam && d->g, "%s: pointer missing", who);
  CODA_REQUIRE(!packed || (d->w && d->bias && d->rope_cos && d->rope_sin), "%s: pointer missing", who);
  CODA_REQUIRE(!packed || ((uintptr_t)d->bias % 16) == 0, "%s: bias must be 16-byte aligned", who);
  const int pc = d->dtype == CODA_BF16 ? 8 : 4;  // elements of a 16-byte piece
  CODA_REQUIRE(d->x_sm % pc == 0 && ((uintptr_t)d->x % 16) == 0 && (!packed || ((uintptr_t)d->w % 16) == 0),
               "%s: x / w rows must be 16-byte aligned", who);
  CODA_REQUIRE(d->q_sm % 4 == 0 && d->k_sm % 4 == 0 && d->v_sm % 4 == 0 && ((uintptr_t)d->q % 8) == 0 &&
                   ((uintptr_t)d->k % 8) == 0 && ((uintptr_t)d->v % 8) == 0,
               "%s: q / k / v rows must be 8-byte aligned", who);
  return CODA_OK;
}
static int front_features(const coda_proj_desc* d) {
  return d->H * d->Dh + 2 * d->Hkv * d->Dh + d->H + (d->gate ? 1 : 0);
}
template <typename T>
static int run_project(const coda_proj_desc* d, hipStream_t st, const char* who) {
  const FrontEpilogue<T, false> epi{*d, FrontTables{}};
  const T *w = (const T*)d->w, *x = (const T*)d->x;
  const int n = front_features(d);
  return d->w_layout ? launch_rows<T>(TileRows<T>{w}, n, d->D, x, d->x_sm, d->M, epi, st, who)
                     : launch_rows<T>(MatRows<T>{w, d->D}, n, d->D, x, d->x_sm, d->M, epi, st, who);
}
template <typename T>
static ParamRows<T> param_rows(const coda_proj_desc* d, const coda_proj_params* p) {
  ParamRows<T> r;
  const int sizes[5] = {d->H * d->Dh, d->Hkv * d->Dh, d->Hkv * d->Dh, d->H, d->gate ? 1 : 0};
  int f = 0;
  for (int i = 0; i < 5; ++i) {
    r.w[i] = (const T*)p->w[i];
    r.b[i] = (const T*)p->b[i];
    r.sm[i] = p->w_sm[i];
    r.start[i] = sizes[i] ? f : INT_MAX;
    f += sizes[i];
  }
  r.Dh = d->Dh;
  r.halves = !d->rope_interleaved;
  return r;
}
template <typename T>
static int run_project_params(const coda_proj_desc* d, const coda_proj_params* p, hipStream_t st, const char* who) {
  const ParamRows<T> r = param_rows<T>(d, p);
  const FrontTables t{p->inv_freq,  p->inv_dtype, p->p0,        p->rope_cos, p->rope_sin,
                      p->theta, p->theta_dtype, d->H * (d->Dh / 2), p->theta_cos, p->theta_sin};
  return launch_rows<T>(r, front_features(d), d->D, (const T*)d->x, d->x_sm, d->M, FrontEpilogue<T, true>{*d, t}, st,
                        who);
}
// The packed form of a layer's parameters, tiles and fp32 biases, in one
// launch: one thread per 16-byte piece of the tiles (a concatenation and its
// packing moved the weights twice and took a dozen launches of a layer's
// first token)
template <typename T>
__global__ __launch_bounds__(256) void proj_pack_params_kernel(const ParamRows<T> W, int n_feat, int row_pieces,
                                                               uint4* __restrict__ out, int64_t n_pieces,
                                                               float* __restrict__ bias) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < (n_feat + 3) / 4 * 4) bias[i] = i < n_feat ? W.bias1((int)i) : 0.f;
  if (i >= n_pieces) return;
  const int l = (int)(i & 63), ksteps = row_pieces / 4;
  const int64_t tile = i >> 6, fb = tile / ksteps;
  const int ks = (int)(tile % ksteps);
  pu32x4 v{0u, 0u, 0u, 0u};
  if (fb * 16 + (l & 15) < n_feat)
    v = *reinterpret_cast<const pu32x4u*>((const char*)W.row16((int)fb * 16, l & 15, n_feat - 1) + 64 * ks + 16 * (l >> 4));
  out[i] = make_uint4(v[0], v[1], v[2], v[3]);
}
template <typename T>
static int run_pack_params(const coda_proj_desc* d, const coda_proj_params* p, void* out, float* bias, hipStream_t st) {
  const int n = front_features(d), row_pieces = d->D * (int)sizeof(T) / 16;
  const int64_t n_pieces = (int64_t)((n + 63) / 64) * 64 * row_pieces;
  hipLaunchKernelGGL(proj_pack_params_kernel<T>, dim3((unsigned)((n_pieces + 255) / 256)), dim3(256), 0, st,
                     param_rows<T>(d, p), n, row_pieces, (uint4*)out, n_pieces, bias);
  return check_launch("proj_pack_params_kernel");
}

}  // namespace coda

using namespace coda;

extern "C" int coda_project(const coda_proj_desc* d, void* stream) {
  CODA_REQUIRE(d != nullptr, "coda_project: null descriptor");
  CODA_REQUIRE(d->dtype == CODA_BF16, "coda_project: bf16 only");
  CODA_REQUIRE(d->M >= 0 && d->M <= 64, "coda_project: %d token rows; the front end serves decode-shaped inputs "
               "(at most 64 rows), many rows are library GEMMs", d->M);
  const int rc = check_project(d, "coda_project", true);
  if (rc) return rc;
  if (d->M == 0) return CODA_OK;
  CODA_REQUIRE(d->w_layout == 0 || (d->w_layout == 1 && rows_path(d->D)),
               "coda_project: weight layout %d with D=%d (tiles serve the row kernel's D only)", d->w_layout, d->D);
  return run_project<bf16_t>(d, (hipStream_t)stream, "coda_project");
}

extern "C" int coda_project_rows(const coda_proj_desc* d, void* stream) {
  CODA_REQUIRE(d != nullptr, "coda_project_rows: null descriptor");
  CODA_REQUIRE(d->dtype == CODA_BF16 || d->dtype == CODA_F32, "coda_project_rows: dtype must be CODA_F32 or CODA_BF16");
  CODA_REQUIRE(d->M >= 0 && d->M <= 128, "coda_project_rows: %d token rows (at most 128)", d->M);
  const int rc = check_project(d, "coda_project_rows", true);
  if (rc) return rc;
  if (d->M == 0) return CODA_OK;
  CODA_REQUIRE(d->w_layout == 0 || d->w_layout == 1, "coda_project_rows: weight layout %d", d->w_layout);
  return d->dtype == CODA_BF16 ? run_project<bf16_t>(d, (hipStream_t)stream, "coda_project_rows")
                               : run_project<float>(d, (hipStream_t)stream, "coda_project_rows");
}

// What both entries on parameters ask of them
static int check_params(const coda_proj_desc* d, const coda_proj_params* p, const char* who) {
  const size_t esz = d->dtype == CODA_BF16 ? 2 : 4;
  for (int i = 0; i < (d->gate ? 5 : 4); ++i) {
    CODA_REQUIRE(p->w[i] && p->w_sm[i] >= d->D, "%s: weight %d missing or its rows shorter than D", who, i);
    CODA_REQUIRE((uintptr_t)p->w[i] % esz == 0 && (uintptr_t)p->b[i] % esz == 0, "%s: weight or bias %d off its type",
                 who, i);
  }
  return CODA_OK;
}

extern "C" int coda_project_pack_params(const coda_proj_desc* d, const coda_proj_params* p, void* out, float* bias,
                                        void* stream) {
  const char* who = "coda_project_pack_params";
  CODA_REQUIRE(d != nullptr && p != nullptr && out && bias, "%s: null pointer", who);
  CODA_REQUIRE(d->dtype == CODA_BF16 || d->dtype == CODA_F32, "%s: dtype must be CODA_F32 or CODA_BF16", who);
  CODA_REQUIRE(d->D > 0 && d->D % kProjKT == 0 && d->H > 0 && d->Hkv > 0 && d->Dh > 0 && d->Dh % 4 == 0,
               "%s: bad sizes D=%d H=%d Hkv=%d Dh=%d", who, d->D, d->H, d->Hkv, d->Dh);
  CODA_REQUIRE((uintptr_t)out % 16 == 0 && (uintptr_t)bias % 16 == 0, "%s: outputs must be 16-byte aligned", who);
  const int rc = check_params(d, p, who);
  if (rc) return rc;
  return d->dtype == CODA_BF16 ? run_pack_params<bf16_t>(d, p, out, bias, (hipStream_t)stream)
                               : run_pack_params<float>(d, p, out, bias, (hipStream_t)stream);
}

extern "C" int coda_project_params(const coda_proj_desc* d, const coda_proj_params* p, void* stream) {
  const char* who = "coda_project_params";
  CODA_REQUIRE(d != nullptr && p != nullptr, "%s: null descriptor", who);
  CODA_REQUIRE(d->dtype == CODA_BF16 || d->dtype == CODA_F32, "%s: dtype must be CODA_F32 or CODA_BF16", who);
  CODA_REQUIRE(d->M >= 0 && d->M <= 128, "%s: %d token rows (at most 128)", who, d->M);
  int rc = check_project(d, who, false);
  if (!rc) rc = check_params(d, p, who);
  if (rc) return rc;
  const auto angle = [](int t) { return t == CODA_F32 || t == CODA_BF16; };
  CODA_REQUIRE(p->inv_freq ? p->rope_cos && p->rope_sin && angle(p->inv_dtype) && p->p0 >= 0 && p->p0 + d->L <= 1 << 24
                           : d->rope_cos && d->rope_sin,
               "%s: RoPE tables missing, or positions past 2^24", who);
  CODA_REQUIRE(!p->theta || (p->theta_cos && p->theta_sin && angle(p->theta_dtype)), "%s: theta tables missing", who);
  if (d->M == 0) return CODA_OK;
  return d->dtype == CODA_BF16 ? run_project_params<bf16_t>(d, p, (hipStream_t)stream, who)
                               : run_project_params<float>(d, p, (hipStream_t)stream, who);
}

static int check_linear(int dtype, const void* x, int64_t x_sm, int M, const void* w, int n_feat, int D, const void* out,
                        int64_t o_sm, const char* who) {
  CODA_REQUIRE(dtype == CODA_BF16 || dtype == CODA_F32, "%s: dtype must be CODA_F32 or CODA_BF16", who);
  CODA_REQUIRE(M >= 0 && M <= 128 && n_feat > 0 && D > 0 && D % kProjKT == 0,
               "%s: bad sizes M=%d n_feat=%d D=%d (at most 128 rows, D a multiple of %d)", who, M, n_feat, D, kProjKT);
  CODA_REQUIRE(x && w && out, "%s: null pointer", who);
  const int pc = dtype == CODA_BF16 ? 8 : 4;
  CODA_REQUIRE(x_sm % pc == 0 && ((uintptr_t)x % 16) == 0, "%s: x / w rows must be 16-byte aligned", who);
  CODA_REQUIRE(o_sm % 4 == 0 && ((uintptr_t)out % 8) == 0, "%s: out rows must be 8-byte aligned", who);
  return CODA_OK;
}
template <typename T, typename BT, typename Src>
static int run_linear(const Src& w, const void* x, int64_t x_sm, int M, int n_feat, int D, const void* bias, void* out,
                      int64_t o_sm, void* stream, const char* who) {
  return launch_rows<T>(w, n_feat, D, (const T*)x, x_sm, M,
                        LinearEpilogue<T, BT>{(T*)out, (const BT*)bias, o_sm, n_feat}, (hipStream_t)stream, who);
}

extern "C" int coda_linear_rows(int dtype, const void* x, int64_t x_sm, int M, const void* w, int n_feat, int D,
                                const float* bias, void* out, int64_t o_sm, void* stream) {
  const char* who = "coda_linear_rows";
  const int rc = check_linear(dtype, x, x_sm, M, w, n_feat, D, out, o_sm, who);
  if (rc) return rc;
  CODA_REQUIRE(((uintptr_t)w % 16) == 0, "%s: x / w rows must be 16-byte aligned", who);
  if (M == 0) return CODA_OK;
  return dtype == CODA_BF16
             ? run_linear<bf16_t, float>(TileRows<bf16_t>{(const bf16_t*)w}, x, x_sm, M, n_feat, D, bias, out, o_sm, stream, who)
             : run_linear<float, float>(TileRows<float>{(const float*)w}, x, x_sm, M, n_feat, D, bias, out, o_sm, stream, who);
}

extern "C" int coda_linear_params(int dtype, const void* x, int64_t x_sm, int M, const void* w, int64_t w_sm, int n_feat,
                                  int D, const void* bias, void* out, int64_t o_sm, void* stream) {
  const char* who = "coda_linear_params";
  const int rc = check_linear(dtype, x, x_sm, M, w, n_feat, D, out, o_sm, who);
  if (rc) return rc;
  const size_t esz = dtype == CODA_BF16 ? 2 : 4;
  CODA_REQUIRE(w_sm >= D && (uintptr_t)w % esz == 0 && (uintptr_t)bias % esz == 0,
               "%s: weight rows shorter than D, or off their type", who);
  if (M == 0) return CODA_OK;
  return dtype == CODA_BF16
             ? run_linear<bf16_t, bf16_t>(MatRows<bf16_t>{(const bf16_t*)w, w_sm}, x, x_sm, M, n_feat, D, bias, out, o_sm, stream, who)
             : run_linear<float, float>(MatRows<float>{(const float*)w, w_sm}, x, x_sm, M, n_feat, D, bias, out, o_sm, stream, who);
}

extern "C" int coda_rows_pack(int dtype, const void* w, int n_feat, int D, int64_t w_sm, void* out, void* stream) {
  CODA_REQUIRE(dtype == CODA_BF16 || dtype == CODA_F32, "coda_rows_pack: dtype must be CODA_F32 or CODA_BF16");
  CODA_REQUIRE(w && out && n_feat > 0 && D > 0 && D % kProjKT == 0 && w_sm >= D, "coda_rows_pack: bad arguments");
  const int esz = dtype == CODA_BF16 ? 2 : 4;
  CODA_REQUIRE(w_sm * esz % 16 == 0 && ((uintptr_t)w % 16) == 0 && ((uintptr_t)out % 16) == 0,
               "coda_rows_pack: rows must be 16-byte aligned");
  return launch_pack(esz, w, n_feat, D, w_sm, out, (hipStream_t)stream);
}

extern "C" int coda_project_pack(const void* w, int n_feat, int D, int64_t w_sm, void* out, void* stream) {
  CODA_REQUIRE(w && out && n_feat > 0 && D > 0 && w_sm >= D, "coda_project_pack: bad arguments");
  if (!rows_path(D)) return fail(CODA_EUNSUP, "coda_project_pack: D=%d does not take the tiled weights", D);
  CODA_REQUIRE(w_sm % 8 == 0 && ((uintptr_t)w % 16) == 0 && ((uintptr_t)out % 16) == 0,
               "coda_project_pack: rows must be 16-byte aligned");
  return launch_pack(2, w, n_feat, D, w_sm, out, (hipStream_t)stream);
}

extern "C" int coda_project_workspace_bytes(const coda_proj_desc* d, size_t* bytes) {
  CODA_REQUIRE(d != nullptr && bytes != nullptr, "coda_project_workspace_bytes: null pointer");
  *bytes = 0;
  return CODA_OK;
}
