// Causal prefill-chunk attention at fp32-class precision on the gfx950 matrix
// cores: fp32, INT8 and FP8 K/V, and the bf16 shapes PrefillMfmaBf16 does not
// cover.
//
// Semantics: kernels::PrefillAttentionVarlenF32 (src/kernels/attention.h:221-227):
// chunk row t sits at position P + t and attends keys [0, P + t]. K/V are read
// through the block table (or an identity table over a contiguous cache); INT8
// and FP8 K/V carry per-(block, kv head) scales.
//
// Arithmetic: operands are cut into bf16 planes whose sum is the value (plane
// i the RNE bf16 of what the earlier ones leave), and the products of planes
// whose indices sum to at most 2 run on v_mfma_f32_16x16x32_bf16, smallest
// first. fp32 K and V take three planes, int8, E4M3 and bf16 values are one
// plane exactly; q takes three (two over FP8 K/V, the split its decode kernel
// uses), the probabilities three. What is left out is below 2^-24 of the
// factors' magnitudes (over FP8 K/V below 2^-18, q's third plane), so a row
// agrees with the decode kernels' result. Scales multiply the finished scores (K) and the probabilities (V).
//
// Work: one workgroup of 4 wavefronts (8 over fp32 K/V) per (chunk, kv head,
// up to 64 or 128 query vectors). A vector is one (row, query head) pair; a kv
// head's g heads of consecutive rows are consecutive vectors, so any g fills
// the 16-vector MFMA blocks, and each wavefront owns HB of those. K/V go
// through registers (two tiles of loads ahead), are converted once per
// workgroup and stored in LDS as planes that all its wavefronts read.
//
// Bound by instruction issue: about 170 (one-plane K/V) to 225 (fp32) VALU
// instructions and 40 to 48 MFMAs per wavefront and tile, where one wavefront
// alone issues an instruction every ~8 cycles (measured: 12 independent FMAs
// take 40 ns with one wavefront on a SIMD, 43 ns with two, 65 ns with four).
// Hence the packed pair splits, the conversions shared by the workgroup, and
// key splits down to 4 tiles, which spread a small step over the chip.
// Measured, chunks' share of a layer before (rows on the decode kernels,
// joint over up to four of them) and now: FP8, d = 128, g = 4, four chunks of
// 256-1024 rows: ~420 -> 78 us (MFMA busy 28%, VALU 43%); fp32, d = 64, g = 7,
// two chunks of 128-768 rows: ~40 -> 19 us.
//
// S^T = K Q^T and O^T = V^T P^T as in PrefillMfmaBf16: a lane's scores, its
// probabilities and its output columns all belong to its own query vector.
//
// The planes of a non-finite V value cannot go through the matrix cores: the
// zero probability of a masked key would turn it into NaN in rows that do not
// attend it. A tile holding one takes a VALU pass that adds each row's
// attended keys only. Nor can those of a non-finite fp32 or bf16 K value,
// whose products with q's planes can be infinities of both signs: a tile
// holding one forms its scores by fp32 multiply-adds of the whole values.
#include <climits>

#include "decode_common.h"
#include "device_util.h"
#include "kernels.h"

namespace ehip {
namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4_t;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2_t;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;
typedef __attribute__((ext_vector_type(2))) float f32x2_t;
// 16 bytes at any alignment (one global load or store: unaligned access is on).
struct __attribute__((packed)) Vec16 {
  uint32_t x[4];
};
// A global (not flat) load from a computed address.
__device__ __forceinline__ Vec16 LoadGlobal(uint64_t at) {
  typedef uint32_t __attribute__((ext_vector_type(4), aligned(1))) u32x4_t;
  const u32x4_t v = *reinterpret_cast<const __attribute__((address_space(1))) u32x4_t*>(at);
  return Vec16{{v.x, v.y, v.z, v.w}};
}

constexpr int kTile = 32;  // keys per tile
constexpr float kRefSlack = 8.f;
// Softmax references below this size take the exponents as one fused
// multiply-add; a larger one rounds further from its score than an exponent's
// unit, so there the score is rounded first, as the reference was.
constexpr float kFusedRef = 16777216.f;
constexpr int kPP = 3;  // planes of the probabilities

template <int KV>
struct KvTraits;
template <>
struct KvTraits<EHIP_KV_F32> {
  static constexpr int ES = 4, KP = 3, QP = 3;
};
template <>
struct KvTraits<EHIP_KV_BF16> {
  static constexpr int ES = 2, KP = 1, QP = 3;
};
template <>
struct KvTraits<EHIP_KV_INT8> {
  static constexpr int ES = 1, KP = 1, QP = 3;
};
template <>
struct KvTraits<EHIP_KV_FP8> {
  static constexpr int ES = 1, KP = 1, QP = 2;
};

__device__ __forceinline__ bf16x4_t TransposedRead(const unsigned char* p) {
  typedef __attribute__((ext_vector_type(4))) short s16x4_t;
  const s16x4_t r = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (__attribute__((address_space(3))) s16x4_t*)(p));
  return __builtin_bit_cast(bf16x4_t, r);
}

// Sum or maximum over the 4 lanes of a query vector (l, l ^ 16, l ^ 32, l ^ 48).
template <typename Op>
__device__ __forceinline__ float RowReduce(float x, Op op) {
  const auto h = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false,
                                                  false);
  x = op(__uint_as_float(h[0]), __uint_as_float(h[1]));
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false,
                                                  false);
  return op(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

// a * b rounded by itself (not fused into a sum it enters).
__device__ __forceinline__ float Product(float a, float b) {
#pragma clang fp contract(off)
  return a * b;
}

// The pair (x, y) as N bf16 planes, one packed word each: a packed RNE
// conversion per plane, and the remainder x - bf16(x) as one v_dot2 (the
// packed pair times (-1, 0) or (0, -1), plus x: exact, checked against the
// subtraction over 2^20 log-uniform values) instead of a widening and a
// subtraction. The factors come in registers: as a literal, (0, -1) is the
// bits of -1.0f, which the assembler turns into a constant of another meaning.
struct PairFactors {
  uint32_t first, second;
};
__device__ __forceinline__ PairFactors MakePairFactors() {
  PairFactors f{0x0000BF80u, 0xBF800000u};
  asm("" : "+s"(f.first));
  asm("" : "+s"(f.second));
  return f;
}
template <int N>
__device__ __forceinline__ void SplitPair(float x, float y, PairFactors f, uint32_t (&out)[N]) {
#pragma unroll
  for (int a = 0; a < N; ++a) {
    const f32x2_t v = {x, y};
    const bf16x2_t h = __builtin_convertvector(v, bf16x2_t);
    out[a] = __builtin_bit_cast(uint32_t, h);
    if (a + 1 < N) {
      x = __builtin_amdgcn_fdot2_f32_bf16(h, __builtin_bit_cast(bf16x2_t, f.first), x, false);
      y = __builtin_amdgcn_fdot2_f32_bf16(h, __builtin_bit_cast(bf16x2_t, f.second), y, false);
    }
  }
}

// Bits of |v| from which the RNE bf16 is not finite.
constexpr uint32_t kBf16Overflow = 0x7F7F8000u;

template <int KV, int D, int WAVES, int HB>
__global__ __launch_bounds__(WAVES * 64) __attribute__((amdgpu_waves_per_eu(2)))
void PrefillSplitMfma(PrefillParams p) {
  constexpr int kThreads = WAVES * 64;
  using KT = KvTraits<KV>;
  constexpr int KP = KT::KP, QP = KT::QP;
  constexpr bool kScaled = KV == EHIP_KV_INT8 || KV == EHIP_KV_FP8;
  constexpr int NC = D / 32;  // MFMA k-chunks over head_dim (QK^T)
  constexpr int NB = D / 16;  // 16-wide output column blocks (PV)
  // LDS rows of a plane: 32 bytes past the row, so that the 16-byte K reads
  // of 16 rows and the transposed V reads of 8 rows hit distinct banks.
  constexpr int PITCH = D * 2 + 32;
  constexpr int PLANE = kTile * PITCH;
  constexpr int VPR = D * KT::ES / 16;           // 16-byte vectors per K or V row
  constexpr int NV = 2 * kTile * VPR / kThreads;  // vectors per thread and tile
  constexpr int NID = NV > 1 ? NV / 2 : 1;        // distinct rows per thread
  static_assert(NV >= 1 && NV * kThreads == 2 * kTile * VPR, "tile / block shape");

  __shared__ __align__(16) unsigned char tiles[2][2 * KP * PLANE];
  __shared__ __align__(16) float tile_scale[2][4];  // K, V scales of the tile's halves
  __shared__ __align__(16) int tile_odd[2][WAVES];  // non-finite V (1), K (2) a wavefront saw

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int n = lane & 15;
  const int kq = lane >> 4;

  const PrefillItem it = p.items[blockIdx.x];
  const int hk = UnpackHk(it.hk_split);
  const int split = UnpackSplit(it.hk_split);
  const int g = p.group;
  const int P = it.past;
  const int rows = p.rows_per_item;              // chunk rows of a full item
  const int q0 = it.q0;
  const int qn = min(rows, it.chunk - q0);       // live rows of this one
  const int nvec = qn * g;                       // live query vectors
  const int kend = P + q0 + qn;
  const int key0 = it.key_begin;
  const int key1 = it.key_end;
  const bool whole = key0 == 0 && key1 >= kend;  // else: partials for the split merge

  const int w0 = wave * 16 * HB;                 // this wavefront's first vector
  const int wn = min(16 * HB, nvec - w0);        // its live vectors (<= 0: none)
  const int wend = wn > 0 ? min(P + q0 + (w0 + wn - 1) / g + 1, key1) : 0;
  const int wlo = P + q0 + (wn > 0 ? w0 : 0) / g;  // position of its first vector
  int vrow[HB], vhead[HB], lim[HB];  // chunk row past q0, head in the group, last key
#pragma unroll
  for (int hh = 0; hh < HB; ++hh) {
    const int v = min(w0 + 16 * hh + n, nvec - 1);
    vrow[hh] = v / g;
    vhead[hh] = v - vrow[hh] * g;
    lim[hh] = min(P + q0 + vrow[hh], key1 - 1);
  }

  const int bs = p.bs;
  const int bsh = __builtin_ctz(bs), bmask = bs - 1;
  const int32_t* const table = p.table + it.table_off;
  // Block strides below 4 GiB (the host checks): one 32 x 32 + 64-bit
  // multiply-add per loaded row; V sits at K's address plus a uniform distance.
  const uint32_t stride_b = static_cast<uint32_t>(p.block_stride * KT::ES);
  const uint32_t nblk = static_cast<uint32_t>(min(p.slab_blocks, int64_t{INT32_MAX}));
  uint64_t kbase = reinterpret_cast<uint64_t>(p.k_slab);
  uint64_t v_from_k = reinterpret_cast<uint64_t>(p.v_slab) - kbase;
  int64_t head_bytes = p.head_stride * KT::ES;
  if constexpr (KV == EHIP_KV_F32) {
    if (p.seqs != nullptr) {  // separate per-sequence caches
      const SeqBase sb = p.seqs[it.seq];
      kbase = sb.k;
      v_from_k = sb.v - sb.k;
      head_bytes = sb.head_bytes;
    }
  }
  kbase += hk * head_bytes;
  const PairFactors pf = MakePairFactors();
  bool bad = false;

  // Vector i of this thread: row (tid / VPR + i * (256 / VPR)) mod 32 of K,
  // then of V, at 16-byte column tid % VPR.
  const int vc = tid & (VPR - 1);
  const uint64_t kcol = kbase + vc * 16;
  auto vrow_of = [&](int i) { return (tid / VPR + i * (kThreads / VPR)) & (kTile - 1); };
  auto is_v = [&](int i) { return NV > 1 ? i >= NV / 2 : tid >= kTile * VPR; };
  struct Stage {
    Vec16 x[NV];
    float sc[kScaled ? 2 : 1];
  };
  auto load_ids = [&](int k0, int (&id)[NID]) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NID; ++i) id[i] = table[min(k0 + vrow_of(i), key1 - 1) >> bsh];
  };
  auto load_tile = [&](int k0, const int (&ids)[NID], Stage& st) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NID; ++i) {
      const int pos = min(k0 + vrow_of(i), key1 - 1);
      const bool ok = static_cast<uint32_t>(ids[i]) < nblk;
      const uint32_t id = ok ? static_cast<uint32_t>(ids[i]) : 0u;
      bad = bad | !ok;
      const uint64_t at = uint64_t{id} * stride_b + kcol +
                          static_cast<uint32_t>((pos & bmask) * (D * KT::ES));
      if constexpr (NV == 1) {
        st.x[0] = LoadGlobal(at + (is_v(0) ? v_from_k : 0));
      } else {
        st.x[i] = LoadGlobal(at);
        st.x[i + NID] = LoadGlobal(at + v_from_k);
      }
      // The scales of the tile's two 16-key halves (each inside one block):
      // every thread reads its first row's (a branch here would make the
      // compiler wait for all loads), the ones with a half's first vector
      // store them.
      if constexpr (kScaled) {
        if (i == 0) {
          const uint32_t so = id * static_cast<uint32_t>(p.kv_heads) + hk;
          if constexpr (NV == 1) {
            st.sc[0] = (is_v(0) ? p.v_scale : p.k_scale)[so];
          } else {
            st.sc[0] = p.k_scale[so];
            st.sc[1] = p.v_scale[so];
          }
        }
      }
    }
  };
  // Convert a loaded tile into planes in LDS; notes non-finite values.
  auto store_tile = [&](const Stage& st, int buf) __attribute__((always_inline)) {
    bool odd = false, oddk = false;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const bool isv = is_v(i);
      unsigned char* const dst = tiles[buf] + (isv ? KP * PLANE : 0) + vrow_of(i) * PITCH;
      const uint32_t(&x)[4] = st.x[i].x;
      if constexpr (KV == EHIP_KV_F32) {
        uint32_t lo[KP], hi[KP];
        SplitPair(__uint_as_float(x[0]), __uint_as_float(x[1]), pf, lo);
        SplitPair(__uint_as_float(x[2]), __uint_as_float(x[3]), pf, hi);
        uint32_t top = 0;
#pragma unroll
        for (int e = 0; e < 4; ++e) top = max(top, x[e] & 0x7FFFFFFFu);
        if (top >= kBf16Overflow) {
          // Non-finite values whole in plane 0 (a NaN's payload quieted),
          // finite ones cut towards zero, which cannot overflow.
          odd = odd | isv;
          oddk = oddk | !isv;
          uint32_t cut[4][KP];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const bool fin = (x[e] & 0x7FFFFFFFu) < 0x7F800000u;
            float r = __uint_as_float(x[e]);
#pragma unroll
            for (int a = 0; a < KP; ++a) {
              cut[e][a] = a == 0 && !fin ? Fp32ToBf16Bits(r) : __float_as_uint(r) >> 16;
              r = fin ? r - __uint_as_float(cut[e][a] << 16) : 0.f;
            }
          }
#pragma unroll
          for (int a = 0; a < KP; ++a) {
            lo[a] = cut[0][a] | cut[1][a] << 16;
            hi[a] = cut[2][a] | cut[3][a] << 16;
          }
        }
#pragma unroll
        for (int a = 0; a < KP; ++a)
          *reinterpret_cast<uint2*>(dst + a * PLANE + vc * 8) = make_uint2(lo[a], hi[a]);
      } else if constexpr (KV == EHIP_KV_BF16) {
        *reinterpret_cast<uint4*>(dst + vc * 16) = make_uint4(x[0], x[1], x[2], x[3]);
        bool over = false;
#pragma unroll
        for (int e = 0; e < 4; ++e)
          over = over | ((((x[e] & 0x7FFF7FFFu) + 0x00800080u) & 0x80008000u) != 0);
        odd = odd | (over & isv);
        oddk = oddk | (over & !isv);
      } else {
        uint32_t w[8];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if constexpr (KV == EHIP_KV_INT8) {
            f32x2_t f[2];
#pragma unroll
            for (int b = 0; b < 4; ++b)
              f[b >> 1][b & 1] = static_cast<float>(static_cast<int8_t>(x[e] >> (8 * b)));
#pragma unroll
            for (int b = 0; b < 2; ++b)
              w[2 * e + b] = __builtin_bit_cast(uint32_t, __builtin_convertvector(f[b], bf16x2_t));
          } else {
            // Two E4M3 codes per instruction; every E4M3 value is a bf16 value.
            w[2 * e] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(
                                                        static_cast<int>(x[e]), 1.0f, false));
            w[2 * e + 1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(
                                                            static_cast<int>(x[e]), 1.0f, true));
            if (isv) odd = odd | ((((x[e] & 0x7F7F7F7Fu) + 0x01010101u) & 0x80808080u) != 0);
          }
        }
        *reinterpret_cast<uint4*>(dst + vc * 32) = make_uint4(w[0], w[1], w[2], w[3]);
        *reinterpret_cast<uint4*>(dst + vc * 32 + 16) = make_uint4(w[4], w[5], w[6], w[7]);
      }
    }
    if constexpr (kScaled) {
      if (vc == 0 && (vrow_of(0) & 15) == 0) {
        const int half = vrow_of(0) >> 4;
        if constexpr (NV == 1) {
          tile_scale[buf][(is_v(0) ? 2 : 0) + half] = st.sc[0];
          odd = odd | (is_v(0) && !(fabsf(st.sc[0]) < INFINITY));
        } else {
          tile_scale[buf][half] = st.sc[0];
          tile_scale[buf][2 + half] = st.sc[1];
          odd = odd | !(fabsf(st.sc[1]) < INFINITY);
        }
      }
    }
    const int any = (__any(odd) ? 1 : 0) | (__any(oddk) ? 2 : 0);
    if (lane == 0) tile_odd[buf][wave] = any;
  };

  // q as MFMA B operands: lane l holds vector w0 + 16 hh + l % 16 at elements
  // 32 c + 8 (l / 16) .. +8, cut into QP planes.
  bf16x8_t qreg[HB][NC][QP];
  f32x4_t o[HB][NB];
  float ref[HB], l[HB];
#pragma unroll
  for (int hh = 0; hh < HB; ++hh) {
    ref[hh] = -INFINITY;
    l[hh] = 0.f;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) o[hh][nb] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  }
  Vec16 qraw[HB][NC][2];
  auto load_q = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int hh = 0; hh < HB; ++hh) {
      const float* qp = p.q + (int64_t{it.row_base + q0 + vrow[hh]} * p.heads + hk * g +
                               vhead[hh]) * D + kq * 8;
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        qraw[hh][c][0] = *reinterpret_cast<const Vec16*>(qp + c * 32);
        qraw[hh][c][1] = *reinterpret_cast<const Vec16*>(qp + c * 32 + 4);
      }
    }
  };
  auto convert_q = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int hh = 0; hh < HB; ++hh)
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        uint32_t w[4][QP];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const Vec16& x = qraw[hh][c][i >> 1];
          SplitPair(__uint_as_float(x.x[2 * (i & 1)]), __uint_as_float(x.x[2 * (i & 1) + 1]), pf,
                    w[i]);
        }
#pragma unroll
        for (int a = 0; a < QP; ++a)
          qreg[hh][c][a] =
              __builtin_bit_cast(bf16x8_t, make_uint4(w[0][a], w[1][a], w[2][a], w[3][a]));
      }
  };

  auto compute_tile = [&](int tile, int buf) __attribute__((always_inline)) {
    const int k0 = key0 + tile * kTile;
    if (k0 >= wend) return;  // wavefront-uniform: past its last row
    const unsigned char* const kb = tiles[buf];
    const unsigned char* const vb = tiles[buf] + KP * PLANE;
    const bool diag = k0 + kTile > wlo + 1 || k0 + kTile > key1;

    f32x4_t s[HB][2];
#pragma unroll
    for (int hh = 0; hh < HB; ++hh) s[hh][0] = s[hh][1] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    // Smallest products of every chunk first: the accumulator rounds at the
    // score's magnitude only for the NC leading ones. With one plane per key
    // the two halves' chains of dependent MFMAs alternate (78.4 against 80.5 us
    // on an FP8 step's chunks); three planes of both would cost the registers.
    constexpr int kHalves = KP == 1 ? 2 : 1;
#pragma unroll
    for (int h0 = 0; h0 < 2; h0 += kHalves) {
      bf16x8_t ka[kHalves][NC][KP];
#pragma unroll
      for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int h = 0; h < kHalves; ++h)
#pragma unroll
          for (int a = 0; a < KP; ++a)
            ka[h][c][a] = *reinterpret_cast<const bf16x8_t*>(
                kb + a * PLANE + (16 * (h0 + h) + n) * PITCH + (4 * c + kq) * 16);
#pragma unroll
      for (int sum = QP - 1; sum >= 0; --sum)
#pragma unroll
        for (int c = 0; c < NC; ++c)
#pragma unroll
          for (int a = 0; a < KP; ++a) {
            const int b = sum - a;
            if (b < 0 || b >= QP) continue;
#pragma unroll
            for (int hh = 0; hh < HB; ++hh)
#pragma unroll
              for (int h = 0; h < kHalves; ++h)
                s[hh][h0 + h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                    ka[h][c][a], qreg[hh][c][b], s[hh][h0 + h], 0, 0, 0);
          }
    }
    float ks[2] = {p.scale_log2, p.scale_log2}, vs[2] = {1.f, 1.f};
    if constexpr (kScaled) {
      const float4 sc = *reinterpret_cast<const float4*>(tile_scale[buf]);
      ks[0] *= sc.x;
      ks[1] *= sc.y;
      vs[0] = sc.z;
      vs[1] = sc.w;
    }
    int oddw = 0;
#pragma unroll
    for (int i = 0; i < WAVES; i += 4) {
      const int4 x = *reinterpret_cast<const int4*>(&tile_odd[buf][i]);
      oddw |= x.x | x.y | x.z | x.w;
    }
    const int oddf = __builtin_amdgcn_readfirstlane(oddw);
    const bool odd = (oddf & 1) != 0;
    if constexpr (!kScaled) {
      if (oddf & 2) {
        // Non-finite K in the tile: each key's products over this lane's
        // elements of q (read again: the loop keeps few registers), added over
        // the vector's four lanes.
#pragma unroll 1
        for (int tok = 0; tok < kTile; ++tok) {
          float sum[HB];
#pragma unroll
          for (int hh = 0; hh < HB; ++hh) sum[hh] = 0.f;
#pragma unroll 1
          for (int e = 8 * kq; e < D; e += e % 8 == 7 ? 25 : 1) {
            float kv = 0.f;
#pragma unroll
            for (int a = KP - 1; a >= 0; --a)
              kv += static_cast<float>(
                  *reinterpret_cast<const __bf16*>(kb + a * PLANE + tok * PITCH + 2 * e));
#pragma unroll
            for (int hh = 0; hh < HB; ++hh)
              sum[hh] = fmaf(p.q[(int64_t{it.row_base + q0 + vrow[hh]} * p.heads + hk * g +
                                  vhead[hh]) * D + e],
                             kv, sum[hh]);
          }
#pragma unroll
          for (int hh = 0; hh < HB; ++hh) {
            const float x = RowReduce(sum[hh], [](float a, float b) { return a + b; });
#pragma unroll
            for (int j = 0; j < 8; ++j)
              if (tok == 16 * (j >> 2) + 4 * kq + (j & 3)) s[hh][j >> 2][j & 3] = x;
          }
        }
      }
    }

    // The operand of lane (n, kq) is V[token][16 nb + n] over the tokens its
    // probabilities cover: two transposed reads per plane. A group of column
    // blocks is requested ahead of the softmax, the next ahead of its MFMAs.
    const unsigned char* const vl = vb + (4 * kq + (n >> 2)) * PITCH + 8 * (n & 3);
    bf16x8_t va[NB][KP];
    auto read_v = [&](int nb) __attribute__((always_inline)) {
#pragma unroll
      for (int a = 0; a < KP; ++a) {
        const bf16x4_t v0 = TransposedRead(vl + a * PLANE + 32 * nb);
        const bf16x4_t v1 = TransposedRead(vl + a * PLANE + 16 * PITCH + 32 * nb);
        va[nb][a] = __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7);
      }
    };
    constexpr int kGroup = KP == 1 ? 4 : 2;
#pragma unroll
    for (int nb = 0; nb < kGroup; ++nb) read_v(nb);

    // t[hh][j]: exponent of key k0 + 16 (j / 4) + 4 kq + j % 4, relative to the
    // row's reference; masked keys are -inf. The reference moves only past a
    // slack of 2^8 (lazy rescaling), so most tiles need no row reduction.
    float t[HB][8];
    bool need = false;
#pragma unroll
    for (int hh = 0; hh < HB; ++hh) {
      const float r = ref[hh] == -INFINITY ? 0.f : ref[hh];
#pragma unroll
      for (int j = 0; j < 8; ++j) t[hh][j] = fmaf(s[hh][j >> 2][j & 3], ks[j >> 2], -r);
      if (diag) {
#pragma unroll
        for (int j = 0; j < 8; ++j)
          if (k0 + 16 * (j >> 2) + 4 * kq + (j & 3) > lim[hh]) t[hh][j] = -INFINITY;
      }
      float tm = -INFINITY;
#pragma unroll
      for (int j = 0; j < 8; ++j) tm = fmaxf(tm, t[hh][j]);
      need = need || !(fabsf(ref[hh]) < kFusedRef) || tm > kRefSlack;
    }
    if (__any(need)) {
      // The reference moves to the row's largest score, and the exponents are
      // formed from the scores again: the first ones would keep the rounding
      // at the jump's size.
      bool moved = false;
      float alpha[HB];
#pragma unroll
      for (int hh = 0; hh < HB; ++hh) {
        float x[8], top = -INFINITY;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          x[j] = Product(s[hh][j >> 2][j & 3], ks[j >> 2]);
          top = fmaxf(top, t[hh][j] == -INFINITY ? -INFINITY : x[j]);
        }
        top = RowReduce(top, [](float a, float b) { return fmaxf(a, b); });
        const bool mv = top > ref[hh] + kRefSlack;
        alpha[hh] = mv && ref[hh] != -INFINITY ? Exp2(ref[hh] - top) : 1.f;
        ref[hh] = mv ? top : ref[hh];
        moved = moved || mv;
        const bool fused = fabsf(ref[hh]) < kFusedRef;
#pragma unroll
        for (int j = 0; j < 8; ++j)
          if (t[hh][j] != -INFINITY)
            t[hh][j] = fused ? fmaf(s[hh][j >> 2][j & 3], ks[j >> 2], -ref[hh]) : x[j] - ref[hh];
        l[hh] *= alpha[hh];
      }
      if (__any(moved)) {
#pragma unroll
        for (int hh = 0; hh < HB; ++hh)
#pragma unroll
          for (int nb = 0; nb < NB; ++nb)
#pragma unroll
            for (int i = 0; i < 4; ++i) o[hh][nb][i] *= alpha[hh];
      }
    }
    bf16x8_t pb[HB][kPP];
#pragma unroll
    for (int hh = 0; hh < HB; ++hh) {
#pragma unroll
      for (int j = 0; j < 8; ++j) t[hh][j] = Exp2(t[hh][j]);
      l[hh] += ((t[hh][0] + t[hh][1]) + (t[hh][2] + t[hh][3])) +
               ((t[hh][4] + t[hh][5]) + (t[hh][6] + t[hh][7]));
      uint32_t w[4][kPP];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float sc = vs[i >> 1];
        SplitPair(kScaled ? t[hh][2 * i] * sc : t[hh][2 * i],
                  kScaled ? t[hh][2 * i + 1] * sc : t[hh][2 * i + 1], pf, w[i]);
      }
#pragma unroll
      for (int a = 0; a < kPP; ++a)
        pb[hh][a] =
            __builtin_bit_cast(bf16x8_t, make_uint4(w[0][a], w[1][a], w[2][a], w[3][a]));
    }
    // The tile's P V on its own (smallest products first), then one fp32 add
    // into the output, kGroup column blocks at a time.
#pragma unroll
    for (int n0 = 0; n0 < NB; n0 += kGroup) {
      f32x4_t part[HB][kGroup];
#pragma unroll
      for (int hh = 0; hh < HB; ++hh)
#pragma unroll
        for (int nb = 0; nb < kGroup; ++nb) part[hh][nb] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      if (!odd) {
#pragma unroll
        for (int nb = 0; nb < kGroup; ++nb)
          if (n0 + nb + kGroup < NB) read_v(n0 + nb + kGroup);
#pragma unroll
        for (int sum = kPP - 1; sum >= 0; --sum)
#pragma unroll
          for (int a = 0; a < KP; ++a) {
            const int b = sum - a;
            if (b < 0 || b >= kPP) continue;
#pragma unroll
            for (int nb = 0; nb < kGroup; ++nb)
#pragma unroll
              for (int hh = 0; hh < HB; ++hh)
                part[hh][nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(va[n0 + nb][a], pb[hh][b],
                                                                       part[hh][nb], 0, 0, 0);
          }
      } else {
        // Non-finite V in the tile: each vector adds its attended keys one by
        // one. Column 16 nb + 4 kq + i of vector n is this lane's element i.
#pragma unroll 1
        for (int tok = 0; tok < kTile; ++tok) {
          const unsigned char* const vt = vb + tok * PITCH + 8 * kq;
          float pj[HB];
#pragma unroll
          for (int hh = 0; hh < HB; ++hh) {
            float x = 0.f;
#pragma unroll
            for (int j = 0; j < 8; ++j)
              x = 4 * (tok >> 4) + (tok & 3) == j ? t[hh][j] * vs[j >> 2] : x;
            pj[hh] = __shfl(x, ((tok & 15) >> 2) * 16 + n);
          }
#pragma unroll
          for (int nb = 0; nb < kGroup; ++nb) {
            f32x4_t v = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int a = KP - 1; a >= 0; --a) {
              const bf16x4_t x =
                  *reinterpret_cast<const bf16x4_t*>(vt + a * PLANE + 32 * (n0 + nb));
#pragma unroll
              for (int i = 0; i < 4; ++i) v[i] += static_cast<float>(x[i]);
            }
#pragma unroll
            for (int hh = 0; hh < HB; ++hh)
              if (k0 + tok <= lim[hh]) {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                  part[hh][nb][i] = fmaf(pj[hh], v[i], part[hh][nb][i]);
              }
          }
        }
      }
#pragma unroll
      for (int hh = 0; hh < HB; ++hh)
#pragma unroll
        for (int nb = 0; nb < kGroup; ++nb)
#pragma unroll
          for (int i = 0; i < 4; ++i) o[hh][n0 + nb][i] += part[hh][nb][i];
    }
  };

  // Step t: convert tile t (its loads were issued two steps before) into LDS,
  // then issue the block ids of tile t + 3 and the loads of tile t + 2, whose
  // ids were issued a step before, so that waiting for ids never waits for
  // the newest tile loads (they retire in issue order); then compute tile t.
  // Loads past the item's last tile read its last row again.
  const int ntiles = (key1 - key0 + kTile - 1) / kTile;
  Stage st0, st1;
  int id0[NID], id1[NID];
#define EHIP_PS_FENCE() asm volatile("" ::: "memory")
#define EHIP_PS_BARRIER()                                   \
  do {                                                      \
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local"); \
    __builtin_amdgcn_s_barrier();                           \
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local"); \
  } while (0)
  {
    // The same issue order as the loop's (tile, ids, tile), so that its first
    // pass waits for no more than its later ones.
    int ida[NID], idb[NID];
    load_ids(key0, ida);
    load_ids(key0 + kTile, idb);
    EHIP_PS_FENCE();
    load_q();
    EHIP_PS_FENCE();
    load_tile(key0, ida, st0);
    EHIP_PS_FENCE();
    load_ids(key0 + 2 * kTile, id0);
    EHIP_PS_FENCE();
    load_tile(key0 + kTile, idb, st1);
    EHIP_PS_FENCE();
    convert_q();
  }
#define EHIP_PS_STEP(T, ST, IDC, IDN)                            \
  do {                                                           \
    const int buf = (T) & 1;                                      \
    store_tile(ST, buf);                                          \
    EHIP_PS_FENCE();                                              \
    load_ids(key0 + ((T) + 3) * kTile, IDN);                      \
    EHIP_PS_FENCE();                                              \
    load_tile(key0 + ((T) + 2) * kTile, IDC, ST);                 \
    EHIP_PS_BARRIER();                                            \
    compute_tile((T), buf);                                       \
  } while (0)
  // Two steps per pass without an exit between them (with one, the compiler
  // waits at the loop's head for the loads of the newest tile too). The second
  // step of an odd count computes nothing: its keys lie past every row.
  for (int tile = 0; tile < ntiles; tile += 2) {
    EHIP_PS_STEP(tile, st0, id0, id1);
    EHIP_PS_STEP(tile + 1, st1, id1, id0);
  }
#undef EHIP_PS_STEP
#undef EHIP_PS_BARRIER
#undef EHIP_PS_FENCE

#pragma unroll
  for (int hh = 0; hh < HB; ++hh) {
    const float lt = RowReduce(l[hh], [](float a, float b) { return a + b; });
    if (w0 + 16 * hh + n >= nvec) continue;
    const int row = it.row_base + q0 + vrow[hh];
    if (whole) {
      const float inv = 1.0f / lt;
      float* po = p.out + (int64_t{row} * p.heads + hk * g + vhead[hh]) * D + 4 * kq;
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        Vec16 v;
#pragma unroll
        for (int i = 0; i < 4; ++i) v.x[i] = __float_as_uint(o[hh][nb][i] * inv);
        *reinterpret_cast<Vec16*>(po + 16 * nb) = v;
      }
    } else {
      const RowDesc rd = p.rows[row];
      const int64_t pi = PartialIndex(rd, p.kv_heads, hk, split) * g + vhead[hh];
      float* po = p.part_o + pi * D + 4 * kq;
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
        *reinterpret_cast<float4*>(po + 16 * nb) =
            make_float4(o[hh][nb][0], o[hh][nb][1], o[hh][nb][2], o[hh][nb][3]);
      if (kq == 0) *reinterpret_cast<float2*>(p.part_ml + pi * 2) = make_float2(ref[hh], lt);
    }
  }
  if (__any(bad) && lane == 0) atomicOr(p.err, kErrBlockRange);
}

// Wavefronts per item and 16-vector blocks per wavefront.
constexpr int SplitWaves(int kv_dtype) { return kv_dtype == EHIP_KV_F32 ? 8 : 4; }
constexpr int SplitBlocks(int kv_dtype, int d) { return kv_dtype != EHIP_KV_F32 && d == 64 ? 2 : 1; }

}  // namespace

namespace {

// Steps of few rows that the decode kernels take in one launch and finish
// before this kernel, whose chunks past four tiles need the split merge too.
// us a layer, decode kernels / this kernel, by the step's longest context:
//   fp32, d = 64: g = 1 (24 rows, 8 kv heads) 7.4/8.3 at 24 keys, 12.7/14.9 at
//     760, 13.4/14.6 at 800, 15.4/15.0 at 1100; g = 4 (32 rows) 8.3/9.6 at 32, 16.8/18.0 at 760,
//     19.4/17.5 at 900; g = 7 (32 rows, 2 kv heads) 11.2/10.3 at 64, 12.0/13.4
//     at 128, 12.4/16.3 at 200, 16.4/17.3 at 500, 19.1/17.6 at 600; g = 8 (32
//     rows, 2) 10.8/10.3 at 64, 11.1/12.5 at 80, 14.5/16.7 at 200, 17.2/17.0 at
//     300.
//   fp32, d = 128: g = 2 (24 rows, 8) 8.1/10.7 at 24, 19.1/19.6 at 700, 22.5/19.2
//     at 900; g = 7 (32 rows, 2) 17.0/14.5 at 64, 15.5/18.3 at 80, 17.4/22.5 at
//     200, 24.2/22.9 at 300; g = 8 (24 rows, 8) 12.2/13.1 at 24, 18.9/22.3 at
//     200, 23.8/24.6 at 300, 28.4/25.1 at 400. (g = 4 has no workgroup per row
//     there: 15.3/13.8 at 48, 68/24 at 200.)
//   FP8, 8 kv heads: d = 64, g = 4 8.5/9.5 at 24, 9.3/10.2 at 64, 10.4/11.6 at 96
//     (32 rows); g = 8 9.0/9.9 at 16, 10.4/10.5 at 48; d = 128, g = 4 8.4/9.2 at
//     16, 10.1/9.5 at 36. INT8, d = 64, g = 4: 9.0/9.7 at 32, 11.1/11.7 at 80;
//     d = 128: 9.7/9.5 at 24. Past about 350 units or below 128 (2 kv heads) the
//     two are within 5%, this kernel ahead.
void SetFewRows(int kv_dtype, int d, int group, PrefillShape* s) {
  const bool d64 = d == 64, fp8 = kv_dtype == EHIP_KV_FP8;
  if (kv_dtype == EHIP_KV_F32) {
    s->few_lo = 1;
    s->few_hi = kWgMaxUnits;
    if (group == 1 || group == 2 || (group == 4 && d64))
      s->few_keys_hi = group == 1 && d64 ? 896 : 768;
    else if (group == 7)
      s->few_keys_lo = 64, s->few_keys_hi = d64 ? 512 : 256;
    else if (group == 8)
      s->few_keys_lo = d64 ? 64 : 0, s->few_keys_hi = d64 ? 256 : 384;
  } else if (kv_dtype != EHIP_KV_BF16) {
    s->few_lo = 128;
    s->few_hi = 352;
    if (group <= 4)
      s->few_keys_hi = d64 ? 128 : fp8 ? 32 : 0;
    else
      s->few_keys_hi = d64 && fp8 ? 32 : 0;
  }
}

}  // namespace

PrefillShape PrefillSplitShape(int kv_dtype, int d, int group, int64_t block_stride) {
  PrefillShape s;
  if ((d != 64 && d != 128) || group < 1 || group > 64) return s;
  if (block_stride > int64_t{0xFFFFFFFF} / 4) return s;  // 32-bit byte strides
  s.rows = SplitWaves(kv_dtype) * 16 * SplitBlocks(kv_dtype, d) / group;
  s.slots = 256 * 8 / SplitWaves(kv_dtype);  // two wavefronts per SIMD
  s.min_tiles = 4;
  s.split = 1.0;
  // Beside decode rows the chunks cost a launch of their own (~6 us a layer),
  // which little work does not earn back. Measured over 8,438 random steps (12
  // layers; 1-64 decode rows, 1-3 chunks of 16-400 rows after 0-1500 keys; g 1
  // to 8; steps of few rows apart), this kernel's time over the decode kernels',
  // median (10th to 90th percentile), by pairs x kv heads x d, a kv head's heads
  // sharing an item on the decode kernels:
  //   fp32, g <= 4: 2-4M 1.26 (1.04-1.47), 4-9M 1.10 (0.71-1.44), 9-18M 0.87
  //     (0.62-1.13), 18-36M 0.72; g > 4: 3-6M 1.11, 6-13M 1.03 (0.83-1.19),
  //     13-26M 0.85 (0.69-1.03)
  //   bf16, d = 64: g = 1 4-9M 1.13, 9-18M 1.04, 18-36M 0.86; g = 4 2-4M 1.21, 4-9M
  //     0.96, 9-18M 0.85; g = 8 4-9M 1.09, 9-18M 1.00, 18-36M 0.84
  //   INT8 and FP8: 5-9M 1.18 (1.07-1.33), 9-18M 1.10 (0.94-1.24), 18-36M 0.93
  //     (0.77-1.12), 36-72M 0.77
  // and by the chunk's context: past 130 keys its rows share 128 and more, which
  // puts the whole decode launch on the joint items of two or four rows. At d =
  // 128, g >= 4 that gives 0.46 (0.22-0.70) over fp32, 0.71 (0.42-0.94) over INT8
  // and FP8 and 0.61 over bf16 whatever the work, 1.21 (1.06-1.34) up to there;
  // bf16 at d = 64 0.62 to 0.75 (0.78 and 1.03 at g = 1 and 8). Outside bf16 the
  // rule is within 15% of the faster side in 98 of 100 steps. The worst lose 1.24
  // times (fp32, d = 64, g = 1, a 67-row chunk over 424 keys) where it takes this
  // kernel and 1.66 (g = 4, three 110-row chunks) where it does not.
  const bool scaled = kv_dtype != EHIP_KV_F32 && kv_dtype != EHIP_KV_BF16;
  s.min_work = scaled ? 18'000'000 : group > 4 ? 13'000'000 : 10'000'000;
  if (kv_dtype == EHIP_KV_BF16 ? d == 128 || (group != 1 && group != 8) : d == 128 && group >= 4)
    s.any_work_keys = 130;
  SetFewRows(kv_dtype, d, group, &s);
  return s;
}

bool LaunchPrefillSplit(const PrefillParams& p, int kv_dtype, hipStream_t stream,
                        hipError_t* err) {
  if (p.n_items == 0) {
    *err = hipSuccess;
    return true;
  }
  const dim3 grid(p.n_items);
#define EHIP_PREFILL_SPLIT_CASE(KK, DD)                                                       \
  if (kv_dtype == KK && p.d == DD) {                                                          \
    hipLaunchKernelGGL((PrefillSplitMfma<KK, DD, SplitWaves(KK), SplitBlocks(KK, DD)>), grid, \
                       dim3(SplitWaves(KK) * 64), 0, stream, p);                              \
    *err = hipGetLastError();                                                                 \
    return true;                                                                              \
  }
  EHIP_PREFILL_SPLIT_CASE(EHIP_KV_F32, 64)
  EHIP_PREFILL_SPLIT_CASE(EHIP_KV_F32, 128)
  EHIP_PREFILL_SPLIT_CASE(EHIP_KV_BF16, 64)
  EHIP_PREFILL_SPLIT_CASE(EHIP_KV_BF16, 128)
  EHIP_PREFILL_SPLIT_CASE(EHIP_KV_INT8, 64)
  EHIP_PREFILL_SPLIT_CASE(EHIP_KV_INT8, 128)
  EHIP_PREFILL_SPLIT_CASE(EHIP_KV_FP8, 64)
  EHIP_PREFILL_SPLIT_CASE(EHIP_KV_FP8, 128)
#undef EHIP_PREFILL_SPLIT_CASE
  return false;
}

}  // namespace ehip
