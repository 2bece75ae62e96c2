// Skinny GEMM (batched decode, and larger M in blocks of 32 rows for narrow weights):
// Y[M,N] = X[M,K] . W[N,K]^T (+ bias) on the 16x16x32 MFMA, the weights streamed once per block of
// rows (memory traffic counted against weights and activations: 1.03-1.15 at M <= 32, 1.48 for [13]
// x (2 x 28672) x 8192, whose half lines of a step are partly evicted before the next; two blocks
// of rows, M = 64, 1.26-1.39).
//
// Each weight is dequantized once in registers (the routines of qgemm_wdequant.h, the ones
// the prefill GEMM and mlxr_qgemm_dequant use) and the rows of X ride along in the MFMA: the
// weights are its first operand in tiles of 16 rows of N, the activations the second in
// blocks of 16 rows of M.
//
// Work split: a workgroup of KG wavefronts owns a slab of RT * 16 weight rows.  Wavefront kg takes
// every KG-th super-block (256 of K) of its RT tiles, walked in steps of 128: lane (r, j) = (lane %
// 16, lane / 16) owns sub-block j of the step for row r of each tile, and MFMA kk takes word kk of
// every lane's sub-block (K positions 32j + 8kk .. +7 of the step, for both operands).  The partial
// tiles of the KG wavefronts meet in LDS at the end and are added in wavefront order.  KG is 8; a
// lone wavefront (KG = 1, K <= 1024, where the eight have a super-block or less) adds the same
// super-blocks in the same order and has neither barrier nor exchange.  So an output's sum does not
// depend on how many rows or weights a launch holds, unless K is split over workgroups (SPLIT):
// then each item has some turns (KG super-blocks) of K, and a second launch adds their fp32 partial
// sums.
//
// The activations go through LDS, read with whole 256-byte row segments.  (Read straight
// into the operand layout, one load instruction touches 64 different 64-byte segments and
// uses a quarter of each, four times the first-level cache's work: the kernel that did so
// spent 30 us of 105 us on it at [13] x (2 x 28672) x 8192 and 9 us of 23 us at [24] x 14336
// x 4096.)
#pragma once
#include <algorithm>
#include <atomic>
#include <type_traits>
#include <utility>

#include "qgemm_device.h"
#include "qgemm_internal.h"
#include "qgemm_vmem.h"
#include "qgemm_wdequant.h"

namespace mlxr {

namespace skinny {

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
  int wide;  // y's address (split: ws's) and rows are aligned to four outputs
};
struct SkinnyParams {
  const void* x;
  int M, K;
  int parts;      // items of a slab: blocks of XR rows of M, times splits of K
  uint32_t mdiv;  // ceil(2^32 / parts): item / parts by a multiplication (parts > 1)
  int per, rem;   // items of a workgroup; the first rem workgroups have one more
  int ks, tps;    // split: splits of K, turns (KG super-blocks) of K of an item
  uint32_t kdiv;  // ceil(2^32 / ks)
  float* ws;      // split: fp32 partials, split s at ws + s * ws_split, rows of ws_ld (SwiGLU: gate, up)
  size_t ws_split;
  int ws_ld;
  int ngroups;
  // SwiGLU: g[0] gate, g[1] up; half of a wavefront's tiles are rows of gate, half the same rows of up
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

// Four consecutive outputs of one row, in one store where they are aligned to it.
__device__ __forceinline__ void store4(void* y, int y_dtype, bool wide, size_t rowbase, int nn, int N, const f32x4_t& v) {
  const uint2 h = y_dtype == DT_BF16 ? make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]))
                                     : make_uint2(pack2<X_F16>(v[0], v[1]), pack2<X_F16>(v[2], v[3]));
  const size_t at = rowbase + nn;
  if (wide && nn + 3 < N) {
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
template <int QT, int XR, int RT, int KG>
constexpr int wave_lds() {
  constexpr int stage = XR * 256 + 2 * tile_lds<QT>() + align16(hdr_lds<QT, RT>());
  return KG == 1 ? stage : std::max(stage, RT * ((XR + 15) / 16) * 1024);
}

// Wavefronts per SIMD the registers are bounded for: 4 (two workgroups on a CU) where that takes
// no more than a handful of spills, else 2 (lone wavefronts: 3).
template <int QT, int XR, int RT, int KG, bool SPLIT>
constexpr int skinny_occ() {
  if (SPLIT) return 2;  // no more than a workgroup per CU
  if (KG == 1 && RT == 4 && XR <= 16) return 3;
  return XR > 16 || QT == QT_Q6_K || QT == QT_Q8_0 || (QT == QT_Q5_K && XR == 16 && RT == 4) ? 2 : 4;
}

template <int QT, int XT, int XR, int RT, int D, int KG, bool SW, bool SPLIT>
__global__ __launch_bounds__(64 * KG, (skinny_occ<QT, XR, RT, KG, SPLIT>())) void qgemm_skinny_kernel(SkinnyParams p) {
  static_assert(D == 1 || D == 2, "weights one or two steps ahead");
  static_assert(RT <= 4 && (!SW || RT >= 2), "tiles of a wavefront");
  constexpr bool KQ = is_kquant(QT);
  constexpr int NB = (XR + 15) / 16;  // 16-row blocks of activations
  constexpr int XN = XR / 4;          // activation loads of a step
  constexpr int HT = SW ? RT / 2 : RT;  // tiles of one weight
  constexpr int TL = tile_lds<QT>();
  constexpr int WLDS = wave_lds<QT, XR, RT, KG>();
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int kg = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int M = p.M, K = p.K, parts = p.parts;
  const int nsub = K >> 5, nsb = K >> 8;
  // each XCD (workgroup id % 8) takes a contiguous run of (slab, block of M) items
  const int nwg = (int)gridDim.x;
  const int f = (nwg & 7) == 0 ? ((int)blockIdx.x & 7) * (nwg >> 3) + ((int)blockIdx.x >> 3) : (int)blockIdx.x;
  const int item0 = f * p.per + min(f, p.rem), item1 = item0 + p.per + (f < p.rem ? 1 : 0);
  const int r = lane & 15, j = lane >> 4;
  auto slab_of = [&](int item) { return parts == 1 ? item : (int)__umulhi((uint32_t)item, p.mdiv); };
  const int nit = SPLIT ? 2 * p.tps : 2 * ((((K + 255) >> 8) + KG - 1) / KG);  // steps per item, even

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
  int x_part = 0, x_it = 0;  // next step whose activations are loaded
  auto block_of = [&](int part) { return SPLIT ? (int)__umulhi((uint32_t)part, p.kdiv) : part; };  // of M
  auto split_of = [&](int part) { return part - block_of(part) * p.ks; };
  auto open_x = [&](int part) {
    x_part = part;
    x_it = SPLIT ? split_of(part) * nit : 0;
    const int m0 = block_of(part) * XR;
#pragma unroll
    for (int q = 0; q < XN; ++q) xrow[q] = (uint32_t)(min(m0 + 4 * q + j, M - 1) * K + 8 * r) * 2u;
  };
  auto issue_x = [&]() {
    const uint32_t k0 = (uint32_t)(256 * (KG * (x_it >> 1) + kg) + 128 * (x_it & 1));
    const bool in = k0 + 8 * r < (uint32_t)K;
    const uint32_t so = k0 < (uint32_t)K ? k0 * 2u : 0u;  // scalar offsets stay inside the buffer
#pragma unroll
    for (int q = 0; q < XN; ++q) xs[q] = __builtin_amdgcn_raw_buffer_load_b128(RX, in ? xrow[q] : OOB, so, 0);
    if (++x_it == (SPLIT ? (split_of(x_part) + 1) * nit : nit)) {
      x_it = 0;
      if (parts > 1) open_x(x_part + 1 == parts ? 0 : x_part + 1);
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

  open_x(item0 - slab_of(item0) * parts);
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
  int w_item = item0, w_it = 0, w_end = nit;  // next step whose weights are loaded
  auto open_w = [&](int item) {
    const int slab = slab_of(item);
    if constexpr (SPLIT) {
      w_it = split_of(item - slab * parts) * nit;
      w_end = w_it + nit;
    }
    const SkinnyGroup& G = p.g[group_of(slab)];
    wN = G.N;
    wn0 = (slab - G.slab0) * 16 * HT;
    plane_rsrc<QT>(G.packed, wN, K, R[0]);
    if constexpr (SW) plane_rsrc<QT>(p.g[1].packed, wN, K, R[1]);
  };
  const int lr = lane >> 2, lp = (lane & 3) ^ (lane >> 4);  // row and piece this lane loads
  const int slot = 4 * r + (j ^ (r >> 2));                  // where operand (r, j) is found
  const uint32_t vs = (uint32_t)lr * (uint32_t)nsub + 8u * kg + lp;
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
      if (w_it == (SPLIT ? w_end : nit)) {
        if constexpr (!SPLIT) w_it = 0;
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

  // Accumulator tile (t, q): lane holds Y[m][n .. n+3] for m = m0 + 16q + lane % 16, n = n0 + 16t
  // + 4 (lane / 16) (SwiGLU: tiles 0 .. HT-1 gate, HT .. 2HT-1 up).  The KG partial tiles of an
  // item meet in LDS (each wavefront's in its own part, between two barriers); a lone wavefront
  // has the sums in its registers.
  auto part = [&](int w, int u) { return *(const f32x4_t*)(lds + w * WLDS + (u * 64 + lane) * 16); };
  auto finish = [&](int item) {
    const int slab = slab_of(item), sub = item - slab * parts, m0 = block_of(sub) * XR;
    const SkinnyGroup& G = p.g[group_of(slab)];
    const int N = G.N, n0 = (slab - G.slab0) * 16 * HT;
    // sums of tile t, block q of X (and of up's)
    auto put = [&](int t, int q, f32x4_t sum, const f32x4_t& up) {
      const int m = m0 + q * 16 + r, nn = n0 + 16 * t + 4 * j;
      if constexpr (SPLIT) {  // this split's partial sums, no bias
        float* const w = p.ws + (size_t)split_of(sub) * p.ws_split + (size_t)m * p.ws_ld;
        if (m < M) {
          store4(w, DT_F32, G.wide, 0, nn, N, sum);
          if constexpr (SW) store4(w + N, DT_F32, G.wide, 0, nn, N, up);
        }
        return;
      }
      if constexpr (SW) {
#pragma unroll
        for (int e = 0; e < 4; ++e) sum[e] = swiglu1(sum[e], up[e]);
      } else if (G.bias) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (nn + e < N) sum[e] += load_scalar(G.bias, G.bias_dtype, nn + e);
      }
      if (m < M) store4(G.y, G.y_dtype, G.wide, (size_t)m * N, nn, N, sum);
    };
    if constexpr (KG == 1) {
      sfor<HT * NB>([&](auto U_) {
        constexpr int t = decltype(U_)::value / NB, q = decltype(U_)::value % NB;
        put(t, q, tot[t][q], tot[SW ? HT + t : t][q]);
      });
      clear(tot);
      return;
    }
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
      for (int q = 0; q < NB; ++q) *(f32x4_t*)(xl + ((t * NB + q) * 64 + lane) * 16) = tot[t][q];
    clear(tot);
    __syncthreads();
    for (int u = kg; u < HT * NB; u += KG) {
      f32x4_t sum = part(0, u), up = sum;
#pragma unroll
      for (int w = 1; w < KG; ++w) sum += part(w, u);
      if constexpr (SW) {
        up = part(0, HT * NB + u);
#pragma unroll
        for (int w = 1; w < KG; ++w) up += part(w, HT * NB + u);
      }
      put(u / NB, u % NB, sum, up);
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
      if constexpr (KG > 1) __syncthreads();  // the partial tiles have been read
    }
  }
}

// A kernel as the host launches it.  residents: workgroups a CU holds, per device (0: not asked yet).
struct SkinnyKern {
  const void* fn;
  int lds, threads;
  std::atomic<int>* residents;
};

template <int QT, int XT, int XR, int RT, int KG, bool SW, bool SPLIT>
const SkinnyKern& kern() {
  static std::atomic<int> residents[64];
  static const SkinnyKern k{(const void*)qgemm_skinny_kernel<QT, XT, XR, RT, RT == 4 ? 1 : 2, KG, SW, SPLIT>,
                            KG * wave_lds<QT, XR, RT, KG>(), 64 * KG, residents};
  return k;
}
template <int QT, int XT, int XR>
const SkinnyKern& kern_of(int rt, int kg, bool sw, bool split) {
  if (split) return sw ? kern<QT, XT, XR, 2, 8, true, true>() : kern<QT, XT, XR, 1, 8, false, true>();
  if (kg == 1) {
    if (sw) return rt == 4 ? kern<QT, XT, XR, 4, 1, true, false>() : kern<QT, XT, XR, 2, 1, true, false>();
    return rt == 4   ? kern<QT, XT, XR, 4, 1, false, false>()
           : rt == 2 ? kern<QT, XT, XR, 2, 1, false, false>()
                     : kern<QT, XT, XR, 1, 1, false, false>();
  }
  if (sw) return rt == 4 ? kern<QT, XT, XR, 4, 8, true, false>() : kern<QT, XT, XR, 2, 8, true, false>();
  return rt == 4   ? kern<QT, XT, XR, 4, 8, false, false>()
         : rt == 2 ? kern<QT, XT, XR, 2, 8, false, false>()
                   : kern<QT, XT, XR, 1, 8, false, false>();
}
template <int QT, int XT>
const SkinnyKern& kern_of(int xr, int rt, int kg, bool sw, bool split) {
  return xr == 8    ? kern_of<QT, XT, 8>(rt, kg, sw, split)
         : xr == 16 ? kern_of<QT, XT, 16>(rt, kg, sw, split)
                    : kern_of<QT, XT, 32>(rt, kg, sw, split);
}

// One translation unit per quant type instantiates the kernels (qgemm_skinny_<type>.hip).  xr: rows
// of a block of M (8, 16, 32); rt: tiles per wavefront (1, 2, 4; SwiGLU 2, 4); kg: wavefronts (8, or
// 1 for K <= 1024); split: K split over workgroups (kg = 8 and the fewest tiles).
const SkinnyKern& kern_q4k(bool f16, int xr, int rt, int kg, bool sw, bool split);
const SkinnyKern& kern_q6k(bool f16, int xr, int rt, int kg, bool sw, bool split);
const SkinnyKern& kern_q5k(bool f16, int xr, int rt, int kg, bool sw, bool split);
const SkinnyKern& kern_q40(bool f16, int xr, int rt, int kg, bool sw, bool split);
const SkinnyKern& kern_q41(bool f16, int xr, int rt, int kg, bool sw, bool split);
const SkinnyKern& kern_q80(bool f16, int xr, int rt, int kg, bool sw, bool split);

}  // namespace skinny
}  // namespace mlxr
