// Skinny GEMM (batched decode, 4 < M <= 64, and larger M in blocks of 64 rows):
// Y[M,N] = X[M,K] . W[N,K]^T (+ bias) on the 16x16x32 MFMA, every weight byte streamed from
// HBM once per block of rows.
//
// Each weight is dequantized once in registers (the routines of qgemm_wdequant.h, the ones
// the prefill GEMM and mlxr_qgemm_dequant use) and the rows of X ride along in the MFMA: the
// weights are its first operand in tiles of 16 rows of N, the activations the second in
// blocks of 16 rows of M.
//
// Work split: a workgroup of NG x KG wavefronts owns a slab of NG * RT * 16 weight rows, for
// every K.  Wavefront (ng, kg) owns RT tiles of the slab and every KG-th super-block (256 of
// K), walked in steps of 128: lane (r, j) = (lane % 16, lane / 16) owns sub-block j of the
// step for row r of each tile, and MFMA kk takes word kk of every lane's sub-block (K
// positions 32j + 8kk .. +7 of the step, for both operands).  The partial tiles of the KG
// wavefronts meet in LDS at the end and are added in wavefront order.  The K split depends on
// K alone, so an output's sum does not depend on how many rows or weights a launch holds.
//
// The activations go through LDS, read with whole 256-byte row segments.  (Read straight
// into the operand layout, one load instruction touches 64 different 64-byte segments and
// uses a quarter of each, four times the first-level cache's work: the kernel that did so
// spent 30 us of 105 us on it at [13] x (2 x 28672) x 8192 and 9 us of 23 us at [24] x 14336
// x 4096.)
#include <stdlib.h>

#include <algorithm>
#include <atomic>
#include <type_traits>
#include <utility>

#include "qgemm_device.h"
#include "qgemm_internal.h"
#include "qgemm_vmem.h"
#include "qgemm_wdequant.h"

namespace mlxr {

std::atomic<int> g_skinny_stage{1};

namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(8))) _Float16 f16x8_t;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;

constexpr int MAX_SG = 4;
// One weight of a launch (its planes follow from the packed base, N and K).
struct SkinnyGroup {
  const uint8_t* packed;
  void* y;
  const void* bias;
  int N;
  int slab0;  // first slab of this weight in the launch
  int y_dtype, bias_dtype;
};
struct SkinnyParams {
  const void* x;
  int M, K;
  int mblocks;  // blocks of XR rows of M
  uint32_t mdiv;  // ceil(2^32 / mblocks): item / mblocks by a multiplication (mblocks > 1)
  int per, rem; // items (slab, block of M) of a workgroup; the first rem workgroups have one more
  int ngroups;
  int swiglu;  // g[0] gate, g[1] up: half of a wavefront's tiles are rows of gate, half the same rows of up
  SkinnyGroup g[MAX_SG];
};

// Compile-time loop: fn(integral_constant<int, i>) for i = 0 .. N-1, fully expanded.
template <typename Fn, int... I>
__device__ __forceinline__ void sfor_impl(Fn&& fn, std::integer_sequence<int, I...>) {
  (fn(std::integral_constant<int, I>()), ...);
}
template <int N, typename Fn>
__device__ __forceinline__ void sfor(Fn&& fn) {
  sfor_impl(fn, std::make_integer_sequence<int, N>());
}

template <int XT>
__device__ __forceinline__ f32x4_t mfma16(const uint4& a, const u32x4_t& b, const f32x4_t& c) {
  if constexpr (XT == X_BF16)
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c,
                                                   0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c,
                                                  0, 0, 0);
}

// Factors of sub-block 4 half + j of a super-block, in slot 0 of Scales: header entry e sits
// in word e / 2, half e % 2 (the layout decode_hdr reads); sel picks entry j of a pair of words
// (bytes 2j, 2j + 1).
template <int QT, int half>
__device__ __forceinline__ void decode_hdr1(const Hdr<QT>& h, uint32_t sel, Scales<QT>& s) {
  const uint32_t e = __builtin_amdgcn_perm(h.h[2 * half + 1], h.h[2 * half], sel);
  if constexpr (QT == QT_Q4_K || QT == QT_Q5_K) {
    const uint32_t dd = q4k_dd(make_uint4(h.h[0], h.h[1], h.h[2], h.h[3]));
    s.a[0] = f16_bits_to_f32(dd & 0xffffu) * SUB24 * (float)(e & 63u);
    s.b[0] = -f16_bits_to_f32(dd >> 16) * (float)((e >> 6) & 63u);
  } else if constexpr (QT == QT_Q6_K) {
    const float d = f16_bits_to_f32(h.d & 0xffffu) * SUB24;
    s.a[0] = d * (float)(int8_t)(e & 0xffu);
    s.b[0] = d * (float)(int8_t)((e >> 8) & 0xffu);
  }
}

// Four consecutive outputs of one row.
__device__ __forceinline__ void store4(void* y, int y_dtype, size_t rowbase, int nn, int N, const f32x4_t& v) {
  const uint2 h = y_dtype == DT_BF16 ? make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]))
                                     : make_uint2(pack2<X_F16>(v[0], v[1]), pack2<X_F16>(v[2], v[3]));
  const size_t at = rowbase + nn;
  if ((N & 3) == 0 && nn + 3 < N) {
    if (y_dtype == DT_F32) *(f32x4_t*)((float*)y + at) = v;
    else *(uint2*)((uint16_t*)y + at) = h;
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (nn + e < N) {
        if (y_dtype == DT_F32) ((float*)y)[at + e] = v[e];
        else ((uint16_t*)y)[at + e] = (uint16_t)((e < 2 ? h.x : h.y) >> (16 * (e & 1)));
      }
  }
}

// Buffer resources of a weight's planes.
template <int QT>
__device__ __forceinline__ void plane_rsrc(const uint8_t* packed, int N, int K, rsrc_t* R) {
  PackedLayout L;
  make_layout(QT, N, K, &L);
#pragma unroll
  for (int i = 0; i < 4; ++i) R[i] = make_rsrc(packed + L.off[i], (uint32_t)L.size[i]);
}

// A tile's bytes of one step, in LDS: the 16-byte nibble pieces (Q8_0: 32), then the high bits
// or scales.
template <int QT>
constexpr int tile_lds() {
  return QT == QT_Q8_0 ? 2048 + 128 : QT == QT_Q6_K ? 1024 + 512 : QT == QT_Q4_K ? 1024 : QT == QT_Q4_0 ? 1024 + 128 : 1024 + 256;
}
// Header bytes of a super-block for RT tiles.
template <int QT, int RT>
constexpr int hdr_lds() {
  return QT == QT_Q6_K ? RT * 16 * 18 : is_kquant(QT) ? RT * 256 : 0;
}
constexpr int align16(int v) { return (v + 15) / 16 * 16; }

// Sub-block loads with the row's part of the offset in a scalar: the lane offset vs is fixed
// for the whole kernel.
template <int QT>
__device__ __forceinline__ void load_raw_s(const rsrc_t* R, uint32_t vs, uint32_t ss, bool ok, Raw<QT>& r) {
  if constexpr (QT == QT_Q6_K) {
    r.ql = bload16(R[0], ok ? vs * 16u : OOB, ss * 16u);
    r.qh = __builtin_amdgcn_raw_buffer_load_b64(R[1], ok ? vs * 8u : OOB, ss * 8u, 0);
  } else if constexpr (QT == QT_Q8_0) {
    r.a = bload16(R[0], ok ? vs * 32u : OOB, ss * 32u);
    r.b = bload16(R[0], ok ? vs * 32u + 16u : OOB, ss * 32u);
    r.d = __builtin_amdgcn_raw_buffer_load_b16(R[1], ok ? vs * 2u : OOB, ss * 2u, 0);
  } else {
    r.q = bload16(R[0], ok ? vs * 16u : OOB, ss * 16u);
    if constexpr (QT == QT_Q5_K) r.qh = __builtin_amdgcn_raw_buffer_load_b32(R[1], ok ? vs * 4u : OOB, ss * 4u, 0);
    if constexpr (QT == QT_Q4_0) r.d = __builtin_amdgcn_raw_buffer_load_b16(R[1], ok ? vs * 2u : OOB, ss * 2u, 0);
    if constexpr (QT == QT_Q4_1) r.d = __builtin_amdgcn_raw_buffer_load_b32(R[1], ok ? vs * 4u : OOB, ss * 4u, 0);
  }
}
// The tile's pieces to LDS in load order (slot i of 64), and back from slot i.
template <int QT>
__device__ __forceinline__ void put_raw(uint8_t* l, int i, const Raw<QT>& r) {
  if constexpr (QT == QT_Q6_K) {
    *(u32x4_t*)(l + i * 16) = r.ql;
    *(u32x2_t*)(l + 1024 + i * 8) = r.qh;
  } else if constexpr (QT == QT_Q8_0) {
    *(u32x4_t*)(l + i * 16) = r.a;
    *(u32x4_t*)(l + 1024 + i * 16) = r.b;
    *(uint16_t*)(l + 2048 + i * 2) = (uint16_t)r.d;
  } else {
    *(u32x4_t*)(l + i * 16) = r.q;
    if constexpr (QT == QT_Q5_K) *(uint32_t*)(l + 1024 + i * 4) = r.qh;
    if constexpr (QT == QT_Q4_0) *(uint16_t*)(l + 1024 + i * 2) = (uint16_t)r.d;
    if constexpr (QT == QT_Q4_1) *(uint32_t*)(l + 1024 + i * 4) = r.d;
  }
}
template <int QT>
__device__ __forceinline__ void get_raw(const uint8_t* l, int i, Raw<QT>& r) {
  if constexpr (QT == QT_Q6_K) {
    r.ql = *(const u32x4_t*)(l + i * 16);
    r.qh = *(const u32x2_t*)(l + 1024 + i * 8);
  } else if constexpr (QT == QT_Q8_0) {
    r.a = *(const u32x4_t*)(l + i * 16);
    r.b = *(const u32x4_t*)(l + 1024 + i * 16);
    r.d = *(const uint16_t*)(l + 2048 + i * 2);
  } else {
    r.q = *(const u32x4_t*)(l + i * 16);
    if constexpr (QT == QT_Q5_K) r.qh = *(const uint32_t*)(l + 1024 + i * 4);
    if constexpr (QT == QT_Q4_0) r.d = *(const uint16_t*)(l + 1024 + i * 2);
    if constexpr (QT == QT_Q4_1) r.d = *(const uint32_t*)(l + 1024 + i * 4);
  }
}

// LDS of a wavefront: activations, two tile slots, headers; the partial tiles reuse it.
template <int QT, int XR, int RT>
constexpr int wave_lds() {
  return std::max(XR * 256 + 2 * tile_lds<QT>() + align16(hdr_lds<QT, RT>()), RT * ((XR + 15) / 16) * 1024);
}

// Wavefronts per SIMD the registers are bounded for: 4 (two workgroups on a CU) where that takes
// no more than a handful of spills, else 2.
template <int QT, int XR, int RT>
constexpr int skinny_occ() {
  return XR > 16 || QT == QT_Q6_K || QT == QT_Q8_0 || (QT == QT_Q5_K && XR == 16 && RT == 4) ? 2 : 4;
}

template <int QT, int XT, int XR, int RT, int D, int KG, bool SW>
__global__ __launch_bounds__(64 * KG, (skinny_occ<QT, XR, RT>())) void qgemm_skinny_kernel(SkinnyParams p) {
  static_assert(D == 1 || D == 2, "weights one or two steps ahead");
  static_assert(RT <= 4 && (!SW || RT >= 2), "tiles of a wavefront");
  constexpr bool KQ = is_kquant(QT);
  constexpr int NB = (XR + 15) / 16;  // 16-row blocks of activations
  constexpr int XN = XR / 4;          // activation loads of a step
  constexpr int HT = SW ? RT / 2 : RT;  // tiles of one weight
  constexpr int TL = tile_lds<QT>();
  constexpr int WLDS = wave_lds<QT, XR, RT>();
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int kg = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int M = p.M, K = p.K, mblocks = p.mblocks;
  const int nsub = K >> 5, nsb = K >> 8;
  // each XCD (workgroup id % 8) takes a contiguous run of (slab, block of M) items
  const int nwg = (int)gridDim.x;
  const int f = (nwg & 7) == 0 ? ((int)blockIdx.x & 7) * (nwg >> 3) + ((int)blockIdx.x >> 3) : (int)blockIdx.x;
  const int item0 = f * p.per + min(f, p.rem), item1 = item0 + p.per + (f < p.rem ? 1 : 0);
  const int r = lane & 15, j = lane >> 4;
  auto slab_of = [&](int item) { return mblocks == 1 ? item : (int)__umulhi((uint32_t)item, p.mdiv); };
  const int nit = 2 * ((((K + 255) >> 8) + KG - 1) / KG);  // steps per item, even

  // LDS of this wavefront: activations, two tile slots, headers
  uint8_t* const xl = lds + kg * WLDS;
  uint8_t* const tl = xl + XR * 256;
  uint8_t* const hl = tl + 2 * TL;

  // ---- activations: 256 bytes (K of one step) of four rows per load; row m's 16-byte chunk c
  // goes to m * 256 + 16 (c ^ (m % 16)), so the 16 rows an operand read takes from one chunk
  // column lie in 16 different bank groups.  Rows past the last repeat it: they only reach
  // outputs that are never stored.
  const rsrc_t RX = make_rsrc(p.x, (uint32_t)M * (uint32_t)K * 2u);
  uint32_t xrow[XN];
  u32x4_t xs[XN];
  int x_mb = 0, x_it = 0;  // next step whose activations are loaded
  auto open_x = [&](int mb) {
    x_mb = mb;
#pragma unroll
    for (int q = 0; q < XN; ++q) xrow[q] = (uint32_t)(min(mb * XR + 4 * q + j, M - 1) * K + 8 * r) * 2u;
  };
  auto issue_x = [&]() {
    const uint32_t k0 = (uint32_t)(256 * (KG * (x_it >> 1) + kg) + 128 * (x_it & 1));
    const bool in = k0 + 8 * r < (uint32_t)K;
    const uint32_t so = k0 < (uint32_t)K ? k0 * 2u : 0u;  // scalar offsets stay inside the buffer
#pragma unroll
    for (int q = 0; q < XN; ++q) xs[q] = __builtin_amdgcn_raw_buffer_load_b128(RX, in ? xrow[q] : OOB, so, 0);
    if (++x_it == nit) {
      x_it = 0;
      if (mblocks > 1) open_x(x_mb + 1 == mblocks ? 0 : x_mb + 1);
    }
  };
  uint32_t xw = (uint32_t)(j * 256 + ((r ^ j) << 4));  // where chunk r of row j goes
  const int fr = XR < 16 ? (r & (XR - 1)) : r;
  uint32_t fo = (uint32_t)(fr * 256 + (((4 * j) ^ fr) << 4));  // chunk 4j of operand row r
  // Four tiles of a 16-row block just fit the registers of four wavefronts per SIMD when the
  // addresses derived from these two are formed at every step instead of kept: [13] x (2 x
  // 28672) x 8192 Q4_K SwiGLU 86.8 -> 81.9 us.
  auto unhoist = [&]() {
    if constexpr (RT == 4 && XR == 16) asm volatile("" : "+v"(xw), "+v"(fo));
  };
  auto write_x = [&]() {
#pragma unroll
    for (int q = 0; q < XN; ++q) *(u32x4_t*)(xl + q * 1024 + (xw ^ (64u * (q & 3)))) = xs[q];
  };

  open_x(item0 - slab_of(item0) * mblocks);
  issue_x();

  // ---- weights, D steps ahead of the products, with their own item and step.  Loaded in
  // memory order, lane 4 row + piece (a quarter of the wavefront then takes four whole 64-byte
  // segments; in operand order, lane row + 16 piece, it would touch sixteen and the first-level
  // cache would work four times as long), and turned to operand order through LDS: slot 4 row +
  // i holds piece i ^ (row / 4), so the 16 rows of one operand piece lie in 16 bank groups.
  rsrc_t R[2][4];  // [1]: SwiGLU's up weight
  int wn0 = 0, wN = 0;  // first row of this wavefront's tiles, rows of the weight
  auto group_of = [&](int slab) {
    int gi = 0;
    if constexpr (!SW) {
#pragma unroll
      for (int g = 1; g < MAX_SG; ++g) gi = (g < p.ngroups && slab >= p.g[g].slab0) ? g : gi;
    }
    return gi;
  };
  auto open_w = [&](int item) {
    const int slab = slab_of(item);
    const SkinnyGroup& G = p.g[group_of(slab)];
    wN = G.N;
    wn0 = (slab - G.slab0) * 16 * HT;
    plane_rsrc<QT>(G.packed, wN, K, R[0]);
    if constexpr (SW) plane_rsrc<QT>(p.g[1].packed, wN, K, R[1]);
  };
  const int lr = lane >> 2, lp = (lane & 3) ^ (lane >> 4);  // row and piece this lane loads
  const int slot = 4 * r + (j ^ (r >> 2));                  // where operand (r, j) is found
  const uint32_t vs = (uint32_t)lr * (uint32_t)nsub + 8u * kg + lp;
  int w_item = item0, w_it = 0;  // next step whose weights are loaded
  Raw<QT> raw[D][RT];
  Hdr<QT> hdr[SW ? 2 : 1];  // lane 16 t + row: tile t's super-block header of that row
  // tile t of step it of an item, this wavefront: half it % 2 of super-block KG * (it / 2) + kg
  auto issue_w = [&](int t, auto HALF) {
    constexpr int half = decltype(HALF)::value;
    const uint32_t s0 = 8 * KG * (w_it >> 1) + 4 * half;
    const int n = wn0 + 16 * (t % HT);
    const bool any = w_item < item1 && (int)s0 < nsub && n < wN;  // of the whole tile
    const bool in = any && (int)s0 + 8 * kg + lp < nsub && n + lr < wN;
    load_raw_s<QT>(R[SW && t >= HT ? 1 : 0], vs, any ? (uint32_t)n * (uint32_t)nsub + s0 : 0u, in, raw[half % D][t]);
  };
  auto issue_h = [&]() {  // the super-block the next even step starts
    if constexpr (KQ) {
      const int g = KG * (w_it >> 1) + kg;
#pragma unroll
      for (int w = 0; w < (SW ? 2 : 1); ++w) {
        const int n = wn0 + (SW ? lane - 16 * HT * w : lane);
        const bool in = w_item < item1 && g < nsb && n < wN && lane >= 16 * HT * w && lane < 16 * HT * (w + 1);
        load_hdr<QT>(R[w], (uint32_t)n * (uint32_t)nsb, g, in, hdr[w]);
      }
    }
  };
  auto write_h = [&]() {
    if constexpr (KQ) {
      u32x4_t h = hdr[0].h;
      if constexpr (SW) h |= hdr[1].h;  // lanes outside a weight's tiles hold zeros
      if (lane < 16 * RT) *(u32x4_t*)(hl + lane * 16) = h;
      if constexpr (QT == QT_Q6_K) {
        uint32_t d = hdr[0].d;
        if constexpr (SW) d |= hdr[1].d;
        if (lane < 16 * RT) *(uint16_t*)(hl + RT * 256 + lane * 2) = (uint16_t)d;
      }
    }
  };
  auto next_w = [&](auto HALF) {
    ++w_it;
    if constexpr (decltype(HALF)::value == 1) {
      if (w_it == nit) {
        w_it = 0;
        if (++w_item < item1) open_w(w_item);
      }
    }
  };

  // The products of a super-block (8 MFMAs) are summed in acc and added to tot, so the fp32
  // rounding of a long K stays that of a sum of few terms: over K = 14336 the largest relative
  // error of an output (above 1% of the largest) is 6e-6 against 2.3e-5 for one chain of MFMAs.
  f32x4_t acc[RT][NB], tot[RT][NB];
  auto clear = [&](f32x4_t (&v)[RT][NB]) {
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
      for (int b = 0; b < NB; ++b) v[t][b] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  };
  clear(tot);
  const uint32_t hsel = (uint32_t)(2 * j) | (uint32_t)(2 * j + 1) << 8 | 0x0c0c0000u;

  // The KG partial tiles of an item meet in LDS (each wavefront's in its own part, between
  // two barriers): accumulator tile (t, q): lane holds Y[m][n .. n+3] for m = m0 + 16q + lane
  // % 16, n = n0 + 16t + 4 (lane / 16) (SwiGLU: tiles 0 .. HT-1 gate, HT .. 2HT-1 up).
  auto part = [&](int w, int u) { return *(const f32x4_t*)(lds + w * WLDS + (u * 64 + lane) * 16); };
  auto finish = [&](int item) {
    const int slab = slab_of(item), m0 = (item - slab * mblocks) * XR;
    const SkinnyGroup& G = p.g[group_of(slab)];
    const int N = G.N, n0 = (slab - G.slab0) * 16 * HT;
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
      for (int q = 0; q < NB; ++q) *(f32x4_t*)(xl + ((t * NB + q) * 64 + lane) * 16) = tot[t][q];
    clear(tot);
    __syncthreads();
    for (int u = kg; u < HT * NB; u += KG) {
      const int t = u / NB, q = u - t * NB;
      const int m = m0 + q * 16 + r, nn = n0 + 16 * t + 4 * j;
      f32x4_t sum = part(0, u);
#pragma unroll
      for (int w = 1; w < KG; ++w) sum += part(w, u);
      if constexpr (SW) {
        f32x4_t up = part(0, HT * NB + u);
#pragma unroll
        for (int w = 1; w < KG; ++w) up += part(w, HT * NB + u);
#pragma unroll
        for (int e = 0; e < 4; ++e) sum[e] = swiglu1(sum[e], up[e]);
      } else if (G.bias) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (nn + e < N) sum[e] += load_scalar(G.bias, G.bias_dtype, nn + e);
      }
      if (m < M) store4(G.y, G.y_dtype, (size_t)m * N, nn, N, sum);
    }
  };

  open_w(item0);
  issue_h();
  sfor<D>([&](auto S_) {
#pragma unroll
    for (int t = 0; t < RT; ++t) issue_w(t, S_);
    next_w(S_);
  });

  // A step: its activations to LDS and the next step's loaded; per tile its weights to LDS, the
  // ones D steps on loaded into the registers just freed, the products of the tile before.
  // Nothing here is shared between wavefronts, whose LDS accesses are carried out in order;
  // order() keeps the compiler from moving one lane's reads past its writes for other lanes.
  auto order = [] { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local"); };
  auto step = [&](auto U) {
    constexpr int u = decltype(U)::value;
    using NH = std::integral_constant<int, (u + D) % 2>;  // half of the step D steps on
    unhoist();
    write_x();
    issue_x();
    if constexpr (u == 0) write_h();
    order();
    // D = 1: the next even step's weights start at the odd step; D = 2: at the even one
    if constexpr (NH::value == 0) issue_h();
    auto move = [&](int t) {
      put_raw<QT>(tl + (t & 1) * TL, lane, raw[u % D][t]);
      order();
      issue_w(t, NH());
    };
    Raw<QT> cur[2];
    move(0);
    get_raw<QT>(tl, slot, cur[0]);
    u32x4_t xf[4][NB];
#pragma unroll
    for (int kk = 0; kk < 4; ++kk)
#pragma unroll
      for (int q = 0; q < NB; ++q) xf[kk][q] = *(const u32x4_t*)(xl + q * 4096 + (fo ^ (16u * kk)));
    sfor<RT>([&](auto T_) {
      constexpr int t = decltype(T_)::value;
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (t + 1 < RT) {
        move(t + 1);
        get_raw<QT>(tl + ((t + 1) & 1) * TL, slot, cur[(t + 1) & 1]);
      }
      Scales<QT> sc;
      if constexpr (KQ) {
        Hdr<QT> h;
        h.h = *(const u32x4_t*)(hl + (16 * t + r) * 16);
        if constexpr (QT == QT_Q6_K) h.d = *(const uint16_t*)(hl + RT * 256 + (16 * t + r) * 2);
        decode_hdr1<QT, u>(h, hsel, sc);
      }
      sfor<4>([&](auto KK) {
        constexpr int kk = decltype(KK)::value;
        const uint4 w = dequant_word<QT, XT, kk, true>(cur[t & 1], sc, 0);
#pragma unroll
        for (int q = 0; q < NB; ++q) acc[t][q] = mfma16<XT>(w, xf[kk][q], acc[t][q]);
      });
    });
    order();
    next_w(NH());
  };
  int item = item0, it = 0;
  for (;;) {
    clear(acc);
    step(std::integral_constant<int, 0>());
    step(std::integral_constant<int, 1>());
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
      for (int q = 0; q < NB; ++q) tot[t][q] += acc[t][q];
    it += 2;
    if (it == nit) {
      finish(item);
      it = 0;
      if (++item >= item1) break;
      __syncthreads();  // the partial tiles have been read
    }
  }
}

// Dispatch over (rows of a block, tiles per wavefront).
template <int QT, int XT, int XR, int RT, int D, int KG, bool SW>
hipError_t launch_k(SkinnyParams sp, hipStream_t s) {
  constexpr size_t lds = (size_t)KG * wave_lds<QT, XR, RT>();
  constexpr int rows = SW ? 8 * RT : 16 * RT;
  int slabs = 0;
  for (int i = 0; i < sp.ngroups; ++i) {
    sp.g[i].slab0 = slabs;
    if (i == 0 || !SW) slabs += (sp.g[i].N + rows - 1) / rows;
  }
  sp.mblocks = (sp.M + XR - 1) / XR;
  const int nitems = slabs * sp.mblocks;
  sp.mdiv = sp.mblocks > 1 ? (uint32_t)(((1ull << 32) + sp.mblocks - 1) / sp.mblocks) : 0u;
  const void* const fn = (const void*)qgemm_skinny_kernel<QT, XT, XR, RT, D, KG, SW>;
  // workgroups a CU holds, once per device (with the LDS limit raised)
  static std::atomic<int> occ_cache[64];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) dev = 0;
  int occ = occ_cache[dev].load(std::memory_order_acquire);
  if (occ == 0) {
    if (lds > 65536) {
      const hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
      if (e != hipSuccess) return e;
    }
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, fn, 64 * KG, lds) != hipSuccess || occ <= 0) occ = 1;
    occ_cache[dev].store(occ, std::memory_order_release);
  }
  const int grid = std::min(nitems, occ * device_cu_count());
  sp.per = nitems / grid;
  sp.rem = nitems % grid;
  qgemm_skinny_kernel<QT, XT, XR, RT, D, KG, SW><<<dim3((unsigned)grid), dim3(64 * KG), lds, s>>>(sp);
  return hipGetLastError();
}

template <int QT, int XT, int RT, int D, bool SW>
hipError_t launch_rt(const SkinnyParams& sp, hipStream_t s) {
  if (sp.M <= 8) return launch_k<QT, XT, 8, RT, D, 8, SW>(sp, s);
  if (sp.M <= 16) return launch_k<QT, XT, 16, RT, D, 8, SW>(sp, s);
  return launch_k<QT, XT, 32, RT, D, 8, SW>(sp, s);
}

// Tiles per wavefront: as many as leave items (slabs x blocks of M) for three quarters of the
// CUs.  More tiles share each activation read and its LDS traffic; fewer fill the chip where
// the weight has few rows.  Measured on MI355X (us at one, two, four tiles; Q4_K): 14336 x
// 4096 at M = 8 14.2 / 13.5 / 12.6, at M = 24 22.2 / 18.3 / 15.3; 8192 x 8192 at M = 13 16.5 /
// 14.9 / 19.6; 4096 x 4096 at M = 8 6.0 / 7.9 / 10.8; 2 x 28672 x 8192 SwiGLU at M = 13 86 (two)
// / 78 (four).
// Items of n weights (SwiGLU: gate's rows) at rt tiles per wavefront.
long items_of(const int* N, int n, int M, bool swiglu, int rt) {
  const int rows = swiglu ? 8 * rt : 16 * rt;
  long slabs = 0;
  for (int i = 0; i < n; ++i) slabs += (N[i] + rows - 1) / rows;
  return slabs * ((M + 31) / 32);
}
int tiles_for(const int* N, int n, int M, bool swiglu) {
  const int mode = g_skinny_stage.load(std::memory_order_relaxed);  // 1: by shape; 0, 2, 4: one, two, four tiles
  const long want = (long)device_cu_count() * 3 / 4;
  if (swiglu) return mode == 4 || (mode == 1 && items_of(N, n, M, true, 4) >= want) ? 4 : 2;
  if (mode != 1) return mode == 0 ? 1 : mode;
  return items_of(N, n, M, false, 4) >= want ? 4 : items_of(N, n, M, false, 2) >= want ? 2 : 1;
}

template <int QT, int XT>
hipError_t launch_s(const SkinnyParams& sp, hipStream_t s) {
  int N[MAX_SG];
  for (int i = 0; i < sp.ngroups; ++i) N[i] = sp.g[i].N;
  const int rt = tiles_for(N, sp.swiglu ? 1 : sp.ngroups, sp.M, sp.swiglu != 0);
  if (sp.swiglu) return rt == 4 ? launch_rt<QT, XT, 4, 1, true>(sp, s) : launch_rt<QT, XT, 2, 2, true>(sp, s);
  return rt == 4   ? launch_rt<QT, XT, 4, 1, false>(sp, s)
         : rt == 2 ? launch_rt<QT, XT, 2, 2, false>(sp, s)
                   : launch_rt<QT, XT, 1, 2, false>(sp, s);
}

hipError_t launch_any(const RunArgs* const* items, int n, bool swiglu, hipStream_t s) {
  SkinnyParams sp;
  const RunArgs& a = *items[0];
  sp.x = a.x;
  sp.M = a.M;
  sp.K = a.L.K;
  sp.mblocks = sp.per = 1;
  sp.rem = 0;
  sp.ngroups = n;
  sp.swiglu = swiglu ? 1 : 0;
  for (int i = 0; i < MAX_SG; ++i) {
    const RunArgs& b = *items[i < n ? i : 0];
    SkinnyGroup& g = sp.g[i];
    g.packed = b.packed;
    g.y = b.y;
    g.bias = b.bias;
    g.N = b.L.N;
    g.slab0 = 0;
    g.y_dtype = b.y_dtype;
    g.bias_dtype = b.bias_dtype;
  }
  const bool f16 = a.x_dtype == DT_F16;
  switch (a.L.qtype) {
    case QT_Q4_K: return f16 ? launch_s<QT_Q4_K, X_F16>(sp, s) : launch_s<QT_Q4_K, X_BF16>(sp, s);
    case QT_Q6_K: return f16 ? launch_s<QT_Q6_K, X_F16>(sp, s) : launch_s<QT_Q6_K, X_BF16>(sp, s);
    case QT_Q5_K: return f16 ? launch_s<QT_Q5_K, X_F16>(sp, s) : launch_s<QT_Q5_K, X_BF16>(sp, s);
    case QT_Q4_0: return f16 ? launch_s<QT_Q4_0, X_F16>(sp, s) : launch_s<QT_Q4_0, X_BF16>(sp, s);
    case QT_Q4_1: return f16 ? launch_s<QT_Q4_1, X_F16>(sp, s) : launch_s<QT_Q4_1, X_BF16>(sp, s);
    default: return f16 ? launch_s<QT_Q8_0, X_F16>(sp, s) : launch_s<QT_Q8_0, X_BF16>(sp, s);
  }
}

// The workspace sizes the library reports for these calls (skinny_workspace_bytes): the
// partial planes of a K split over workgroups.  The kernel splits K inside a workgroup and
// leaves the workspace untouched; the sizes stay what callers have been told, as they decide
// which calls mlxr_qgemm_run_noalloc takes.
constexpr int TK = 64, TK16 = 128;  // K of a step (M > 32, M <= 32)
constexpr int MAXW = 8;             // wavefronts of a workgroup
constexpr int UNROLL16 = 4;         // steps per trip
struct SkinnyPlan {
  int ks, spg, w, spw;
};
SkinnyPlan skinny_plan(int N, int K, int ring, bool allow_split, int mblocks = 1) {
  constexpr int wpc = 8;  // wavefronts per CU aimed for
  const int cus = device_cu_count();
  const int slabs = (N + 31) / 32 * mblocks;  // workgroups per K split
  const int nkt = (K + TK - 1) / TK;
  SkinnyPlan pl;
  pl.ks = allow_split && slabs < cus ? std::max(1, std::min(cus / slabs, nkt / ring)) : 1;
  pl.spg = (((nkt + pl.ks - 1) / pl.ks) + ring - 1) / ring * ring;
  pl.ks = (nkt + pl.spg - 1) / pl.spg;
  const long want = (long)wpc * cus;
  pl.w = (int)std::min<long>(MAXW, std::max<long>(1, (want + (long)slabs * pl.ks - 1) / ((long)slabs * pl.ks)));
  pl.spw = (((pl.spg + pl.w - 1) / pl.w) + ring - 1) / ring * ring;
  pl.w = (pl.spg + pl.spw - 1) / pl.spw;
  return pl;
}

// The narrow kernels' geometry: as skinny_plan, in 128-wide steps (whole multiples of
// `unroll` per wavefront), at most `wcap` wavefronts per workgroup, the K split over
// workgroups sized for about `wpc` wavefronts per CU.
SkinnyPlan skinny16_plan(int N, int K, bool allow_split, int unroll, int wcap, int wpc) {
  const int maxw = std::max(1, std::min(wcap, MAXW));
  const int cus = device_cu_count();
  const int slabs = (N + 31) / 32;
  const int nkt = (K + TK16 - 1) / TK16;
  const long want = (long)wpc * cus;
  SkinnyPlan pl;
  pl.ks = 1;
  // split K over workgroups (partials + a reduce launch, a few us) only when the slabs
  // alone would fill less than half the target
  if (allow_split && 2L * slabs * maxw <= want)
    pl.ks = (int)std::max<long>(1, std::min<long>((want + (long)slabs * maxw - 1) / ((long)slabs * maxw),
                                                  nkt / unroll));
  pl.spg = (((nkt + pl.ks - 1) / pl.ks) + unroll - 1) / unroll * unroll;
  pl.ks = (nkt + pl.spg - 1) / pl.spg;
  pl.w = (int)std::min<long>(maxw, std::max<long>(1, (want + (long)slabs * pl.ks - 1) / ((long)slabs * pl.ks)));
  pl.spw = (((pl.spg + pl.w - 1) / pl.w) + unroll - 1) / unroll * unroll;
  pl.w = (pl.spg + pl.spw - 1) / pl.spw;
  return pl;
}

bool narrow_plan(int M) { return M <= 32; }

}  // namespace

hipError_t launch_skinny(const RunArgs& a, hipStream_t s) {
  const RunArgs* items[1] = {&a};
  return launch_any(items, 1, false, s);
}
hipError_t launch_skinny_grouped(const RunArgs* const* items, int n, hipStream_t s) {
  return launch_any(items, n, false, s);
}
hipError_t launch_skinny_swiglu(const RunArgs& gate, const RunArgs& up, hipStream_t s) {
  RunArgs u = up;
  u.y = gate.y;
  const RunArgs* items[2] = {&gate, &u};
  return launch_any(items, 2, true, s);
}

// Rounds of items over the CUs (one workgroup each at 32 rows), each as long as its K (ns per
// element at one, two, four tiles; measured on MI355X, Q4_K, us, estimate / time: 8192 x 8192 at
// M = 64 24.5 / 24.9, at M = 96 45.0 / 45.0; 14336 x 4096 at M = 96 34.7 / 36.3; 4096 x 14336 at
// M = 128 39.8 / 37.5; 4096 x 4096 at M = 33 10.6 / 10.2, at M = 256 24.5 / 24.6), the other types
// by their dequantization (4096 x 14336 Q6_K at M = 64 33.8 / 33.6).
double skinny_est_us(const RunArgs* const* items, int n) {
  const RunArgs& a = *items[0];
  int N[MAX_SG];
  for (int i = 0; i < n; ++i) N[i] = items[i]->L.N;
  const int rt = tiles_for(N, n, a.M, false);
  const int cus = device_cu_count();
  const long rounds = (items_of(N, n, a.M, false, rt) + cus - 1) / cus;
  const double qf = a.L.qtype == QT_Q6_K ? 1.3 : a.L.qtype == QT_Q5_K ? 1.16 : a.L.qtype == QT_Q8_0 ? 1.08 : 1.0;
  const int k = (a.L.K + 2047) / 2048 * 2048;  // the 8 wavefronts' super-blocks: a rest takes as long
  return 4.0 + (double)rounds * k * qf * (rt == 4 ? 2.5e-3 : rt == 2 ? 1.6e-3 : 0.8e-3);
}

size_t skinny_swiglu_workspace_bytes(int M, int N, int K) {
  const SkinnyPlan pl = skinny16_plan(32 * ((N + 15) / 16), K, true, UNROLL16, MAXW, 8);
  return pl.ks > 1 ? (size_t)pl.ks * (size_t)M * (size_t)N * 8u : 0;
}

namespace {
// The kernel divides an item by the blocks of M with a multiplication (mdiv), which is exact while
// items x blocks is below 2^32; one tile per wavefront has the most items.
bool items_fit(int64_t slabs, int M) {
  const uint64_t mb = ((uint64_t)M + 31) / 32;
  return (uint64_t)slabs * mb * mb < (1ull << 32);
}
}  // namespace

bool skinny_fits(const RunArgs& a) {
  const size_t lim = operand_limit();
  if ((size_t)a.M * (size_t)a.L.K * 2u >= lim) return false;
  for (int i = 0; i < a.L.nplanes; ++i)
    if (a.L.size[i] >= lim) return false;
  return items_fit((a.L.N + 15) / 16, a.M);
}

bool skinny_group_fits(const RunArgs* const* items, int n) {
  int64_t slabs = 0;
  for (int i = 0; i < n; ++i) {
    if (!skinny_fits(*items[i])) return false;
    slabs += (items[i]->L.N + 15) / 16;
  }
  return items_fit(slabs, items[0]->M);
}

double skinny_mb_est_us(int M, int N, int K) {
  // each 32-row slab reads its 64-row blocks of X from L2 (~7.5 TB/s device-wide), plus
  // ~8 us of launch, prologue and epilogue (measured on MI355X, Llama-3-8B shapes)
  return 8.0 + (double)((N + 31) / 32) * M * K * 2.0 / 7.5e6;
}

size_t skinny_workspace_bytes(int M, int N, int K, int qtype) {
  const SkinnyPlan pl = narrow_plan(M) ? skinny16_plan(N, K, true, UNROLL16, MAXW, 8)
                                         : skinny_plan(N, K, qtype == QT_Q8_0 ? 4 : 8, true, (M + 63) / 64);
  return pl.ks > 1 ? (size_t)pl.ks * (size_t)M * (size_t)N * 4u : 0;
}

}  // namespace mlxr
