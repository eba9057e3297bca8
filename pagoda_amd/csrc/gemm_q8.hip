// gemm_q8.hip — candle's CPU quantized matmul (gemv_q8.hip describes the
// arithmetic) for many activation rows of Q4_K / Q6_K matrices on the f16
// matrix cores, bit-equal to the per-row kernels.
//
// Why the matrix cores give the same bits: per 256-weight block and residue
// class l (element index mod 8, GGML's aux32[8] lanes) the CPU code needs the
// integer sum over the class's 32 elements of scale * code * x_q. That is one
// v_mfma_f32_16x16x32_f16 per 16 x 16 outputs: scale * code (Q4_K: at most
// 63 * 15) and x_q (8 bits) are exact in f16, the products and every partial
// sum are integers of at most 2^24, exact in the f32 accumulator. Q6_K's
// scale * code needs 12 bits and goes as two operands, (scale & 15) * code and
// (scale - (scale & 15)) * code, into one accumulator. The Q4_K mins times the
// 16-element activation sums (at most 2048) are one more 16x16x16 product.
// The float part stays on the vector ALUs in GGML's order: sums[l] += d * aux
// with separate roundings, block after block, the eight sums added last.
//
// Two launches. q8k_prep_kernel quantizes 16 rows x 256 elements per
// workgroup to Q8_K and writes them as matrix-core operands, class by class
// (kStageBytes per 16-row tile and block). q8_mm_kernel: a wave owns 16
// weight rows, a workgroup of NW waves shares MT 16-row activation tiles,
// double-buffered through LDS, and walks the K blocks in order; weights go
// from HBM straight into registers, two blocks ahead (one with two tiles).
//
// Bound: the vector ALUs, 64 multiplies and adds per 16 x 16 outputs and
// block for the ordered sums (32 cycles per MFMA of 16) plus the unpacking,
// which MT tiles share; at few tiles, the K chain of one wave (about 1 us per
// block). Measured against 16 rows per launch on the vector ALUs: 4864 x 896
// Q4_K 81 rows 138 -> 11.5 us, 333 rows 547 -> 22.5 us, 1000 rows 1643 ->
// 47 us; 896 x 4864 Q6_K 81 rows 632 -> 27 us, 1000 rows 7786 -> 54 us.
#include <mutex>

#include "common.h"
#include "gemv_impl.h"
#include "quant.h"

namespace pgd {
namespace gemv {

namespace {

typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef _Float16 h4 __attribute__((ext_vector_type(4)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef uint32_t u2v __attribute__((ext_vector_type(2)));
typedef uint32_t u4v __attribute__((ext_vector_type(4)));

// One 16-row tile x 256-element block of prepared activations: the operands
// of the eight classes (1 KiB each, lane (kq, row) holding slots 0..7), the
// sums of each 16 elements as the mins operand, and the rows' d. Slot mm of
// lane kq = 2u + kk holds element 128 u + 16 mm + 8 kk + l of class l, the
// order in which a lane's bytes of the Q6_K planes hold a class.
constexpr int kSumOff = 8192, kDOff = kSumOff + 512, kStageBytes = kDOff + 64;
constexpr int kTailUnits = (kStageBytes - kSumOff) / 16;
// activation rows prepared at a time: bounds the scratch (9.0 MB at K 4096)
constexpr int kRowChunk = 1024;

__device__ inline h2 as_h2(uint32_t v) { return __builtin_bit_cast(h2, v); }
__device__ inline h2 splat(_Float16 v) { return h2{v, v}; }
// f16 1024 + c for c < 1024 in the low bits of a half
constexpr uint32_t kMagic = 0x64006400u;
// the masked bits of v, kMagic elsewhere, in one instruction (the compiler
// would fold the constants into an and plus an or)
__device__ inline h2 magic_bits(uint32_t mask, uint32_t v, uint32_t magic) {
  uint32_t r;
  asm("v_bfi_b32 %0, %1, %2, %3" : "=v"(r) : "s"(mask), "v"(v), "v"(magic));
  return as_h2(r);
}
// byte b of lo and of hi, each alone in a 16-bit half
template <int B>
__device__ inline uint32_t pair_bytes(uint32_t lo, uint32_t hi) {
  return __builtin_amdgcn_perm(hi, lo, 0x0c000c00u | ((4u + B) << 16) | B);
}

__global__ __launch_bounds__(256) void q8k_prep_kernel(const float* __restrict__ x, int ldx, int rows, int n_in,
                                                       int nsb, char* __restrict__ out) {
  __shared__ __attribute__((aligned(16))) char st[kStageBytes];
  const int sb = blockIdx.x, bt = blockIdx.y;
  const int r = threadIdx.x >> 4, s = threadIdx.x & 15;  // 16 lanes of 16 elements per row
  const int row = bt * 16 + r, e0 = sb * 256 + 16 * s;
  float v[16];
  const float* xr = x + (size_t)row * ldx + e0;
  if (row < rows && e0 + 16 <= n_in && (((uintptr_t)xr) & 15) == 0) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float4 t = reinterpret_cast<const float4*>(xr)[i];
      v[4 * i] = t.x;
      v[4 * i + 1] = t.y;
      v[4 * i + 2] = t.z;
      v[4 * i + 3] = t.w;
    }
  } else {
#pragma unroll
    for (int i = 0; i < 16; ++i) v[i] = (row < rows && e0 + i < n_in) ? xr[i] : 0.0f;
  }
  // the first element of largest magnitude (BlockQ8K::from_float)
  float amax = 0.0f, mx = 0.0f;
  int idx = 0x7fffffff;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const float ax = fabsf(v[i]);
    if (ax > amax) {
      amax = ax;
      mx = v[i];
      idx = e0 + i;
    }
  }
#pragma unroll
  for (int o = 1; o < 16; o <<= 1) {
    const float oa = __shfl_xor(amax, o, 64), om = __shfl_xor(mx, o, 64);
    const int oi = __shfl_xor(idx, o, 64);
    if (oa > amax || (oa == amax && oi < idx)) {
      amax = oa;
      mx = om;
      idx = oi;
    }
  }
  const float iscale = -128.0f / mx;
  int sum = 0;
  _Float16* q = reinterpret_cast<_Float16*>(st);
  const int u = s >> 3, mm = s & 7;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const float t = roundf(iscale * v[i]);
    const int qi = amax == 0.0f ? 0 : (int)(int8_t)(int)(t < 127.0f ? t : 127.0f);
    sum += qi;
    q[(i & 7) * 512 + ((2 * u + (i >> 3)) * 16 + r) * 8 + mm] = (_Float16)qi;
  }
  reinterpret_cast<_Float16*>(st + kSumOff)[((s >> 2) * 16 + r) * 4 + (s & 3)] = (_Float16)sum;
  if (s == 0) reinterpret_cast<float*>(st + kDOff)[r] = amax == 0.0f ? 0.0f : 1.0f / iscale;
  __syncthreads();
  u4v* dst = reinterpret_cast<u4v*>(out + ((size_t)bt * nsb + sb) * kStageBytes);
  const u4v* src = reinterpret_cast<const u4v*>(st);
  for (int i = threadIdx.x; i < kStageBytes / 16; i += 256) dst[i] = src[i];
}

// One lane's weights of one block: row sub * 16 + (lane & 15), slots of
// kq = lane >> 4.
template <int FMT>
struct Raw;

template <>
struct Raw<FMT_Q4K> {
  u2v a0, a1, b0, b1;  // bytes 8 kk.. and 16 + 8 kk.. of 64-chunks 2u and 2u + 1
  u4v hdr;
  __device__ void load(const uint8_t* p0, const uint8_t* p1, const uint8_t*, const uint8_t*, int row, int sb, int nsb) {
    const int kq = (threadIdx.x & 63) >> 4, u = kq >> 1, kk = kq & 1;
    const uint8_t* q = p0 + q4k_qs_off(row, 32 * (4 * sb + 2 * u) + 8 * kk, nsb);
    a0 = *reinterpret_cast<const u2v*>(q);
    a1 = *reinterpret_cast<const u2v*>(q + 16);
    b0 = *reinterpret_cast<const u2v*>(q + 1024);
    b1 = *reinterpret_cast<const u2v*>(q + 1040);
    hdr = *reinterpret_cast<const u4v*>(p1 + q4k_hdr_off(row, sb, nsb));
  }
};

template <>
struct Raw<FMT_Q6K> {
  u4v ql[2];  // dword 2 kk + p of the four 16-byte runs of half u, p = 0, 1
  u2v qh[2], sc;
  uint32_t d;
  __device__ void load(const uint8_t* p0, const uint8_t* p1, const uint8_t* p2, const uint8_t* p3, int row, int sb,
                       int nsb) {
    const int kq = (threadIdx.x & 63) >> 4, u = kq >> 1, kk = kq & 1;
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      const int i = 4 * (2 * kk + p);
      ql[p] = *reinterpret_cast<const u4v*>(p0 + q6k_ql_off(row, 64 * (2 * sb + u) + i, nsb));
      qh[p] = *reinterpret_cast<const u2v*>(p1 + q6k_qh_off(row, 32 * (2 * sb + u) + i, nsb));
    }
    sc = *reinterpret_cast<const u2v*>(p2 + q6k_sc_off(row, 16 * sb + 8 * u, nsb));
    d = reinterpret_cast<const uint16_t*>(p3)[q6k_d_off(row, sb, nsb)];
  }
};

template <int MT>
struct Acc {
  float s[MT][8][4];  // GGML's sums[8] of the lane's 4 rows of each tile
  float m[MT][4];     // minus the Q4_K min terms
};

// one residue class of one block: aux from the matrix cores, then the ordered sum
template <int MT, int L, bool TWO>
__device__ inline void add_class(const char* st, h8 b, h8 b2, const float (&d)[MT][4], Acc<MT>& acc) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    const h8 x = *reinterpret_cast<const h8*>(st + t * kStageBytes + L * 1024 + lane * 16);
    f4 c = __builtin_amdgcn_mfma_f32_16x16x32_f16(x, b, f4{0, 0, 0, 0}, 0, 0, 0);
    if constexpr (TWO) c = __builtin_amdgcn_mfma_f32_16x16x32_f16(x, b2, c, 0, 0, 0);
#pragma unroll
    for (int i = 0; i < 4; ++i) acc.s[t][L][i] += d[t][i] * c[i];
  }
  // keep the scheduler from holding every class's operands and products at once
  if constexpr ((L & 1) != 0) __builtin_amdgcn_sched_barrier(0);
}

template <int MT>
__device__ inline void scales(const char* st, float dw, float (&d)[MT][4]) {
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    const f4 dx = *reinterpret_cast<const f4*>(st + t * kStageBytes + kDOff + ((threadIdx.x & 63) >> 4) * 16);
#pragma unroll
    for (int i = 0; i < 4; ++i) d[t][i] = dw * dx[i];
  }
}

template <int MT, int L>
__device__ inline void class_q4k(const char* st, const Raw<FMT_Q4K>& w, const h2 (&s)[4], const h2 (&o)[4],
                                 const float (&d)[MT][4], Acc<MT>& acc) {
  constexpr int D = L >> 2, B = L & 3;
  const uint32_t magic = kMagic;
  const uint32_t pa = pair_bytes<B>(w.a0[D], w.a1[D]), pb = pair_bytes<B>(w.b0[D], w.b1[D]);
  // scale * code in one fused step: (1024 + code) s - 1024 s, and with the
  // high nibble in place (1024 + 16 code) s/16 - 64 s; both exact
  const h2 v[4] = {__builtin_elementwise_fma(magic_bits(0x000F000Fu, pa, magic), s[0], o[0]),
                   __builtin_elementwise_fma(magic_bits(0x00F000F0u, pa, magic), s[1], o[1]),
                   __builtin_elementwise_fma(magic_bits(0x000F000Fu, pb, magic), s[2], o[2]),
                   __builtin_elementwise_fma(magic_bits(0x00F000F0u, pb, magic), s[3], o[3])};
  const h8 b = {v[0][0], v[0][1], v[1][0], v[1][1], v[2][0], v[2][1], v[3][0], v[3][1]};
  add_class<MT, L, false>(st, b, b, d, acc);
}

template <int MT>
__device__ inline void block_q4k(const char* st, const Raw<FMT_Q4K>& w, Acc<MT>& acc) {
  const int lane = threadIdx.x & 63, kq = lane >> 4, u = kq >> 1, kk = kq & 1;
  // 6-bit scales and mins of sub-blocks 4u .. 4u + 3, one per byte
  const uint32_t sw = u ? (w.hdr[3] & 0x0F0F0F0Fu) | ((w.hdr[1] >> 2) & 0x30303030u) : w.hdr[1] & 0x3F3F3F3Fu;
  const uint32_t mw = u ? ((w.hdr[3] >> 4) & 0x0F0F0F0Fu) | ((w.hdr[2] >> 2) & 0x30303030u) : w.hdr[2] & 0x3F3F3F3Fu;
  h2 s[4], o[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const _Float16 f = (_Float16)(float)((sw >> (8 * j)) & 63u);
    s[j] = splat(j & 1 ? f * (_Float16)0.0625f : f);
    o[j] = s[j] * splat((_Float16)-1024.0f);
  }
  const float dw = (float)__builtin_bit_cast(_Float16, (uint16_t)(w.hdr[0] & 0xffffu));
  const float dmin = (float)__builtin_bit_cast(_Float16, (uint16_t)(w.hdr[0] >> 16));
  float d[MT][4];
  scales<MT>(st, dmin, d);
  const uint32_t m2 = mw >> (16 * kk);
  const _Float16 m0 = (_Float16)(float)(m2 & 63u), m1 = (_Float16)(float)((m2 >> 8) & 63u);
  const h4 mb = {m0, m0, m1, m1};
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    const h4 bs = *reinterpret_cast<const h4*>(st + t * kStageBytes + kSumOff + lane * 8);
    const f4 c = __builtin_amdgcn_mfma_f32_16x16x16f16(bs, mb, f4{0, 0, 0, 0}, 0, 0, 0);
#pragma unroll
    for (int i = 0; i < 4; ++i) acc.m[t][i] -= d[t][i] * c[i];
  }
  scales<MT>(st, dw, d);
  class_q4k<MT, 0>(st, w, s, o, d, acc);
  class_q4k<MT, 1>(st, w, s, o, d, acc);
  class_q4k<MT, 2>(st, w, s, o, d, acc);
  class_q4k<MT, 3>(st, w, s, o, d, acc);
  class_q4k<MT, 4>(st, w, s, o, d, acc);
  class_q4k<MT, 5>(st, w, s, o, d, acc);
  class_q4k<MT, 6>(st, w, s, o, d, acc);
  class_q4k<MT, 7>(st, w, s, o, d, acc);
}

template <int MT, int P, int B>
__device__ inline void class_q6k(const char* st, const uint32_t (&v)[8], const h2 (&lo)[4], const h2 (&hi)[4],
                                 const float (&d)[MT][4], Acc<MT>& acc) {
  h2 a[4], b[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const h2 q = as_h2(pair_bytes<B>(v[2 * i], v[2 * i + 1]) | kMagic) + splat((_Float16)-1056.0f);  // code - 32
    a[i] = q * lo[i];
    b[i] = q * hi[i];
  }
  const h8 x = {a[0][0], a[0][1], a[1][0], a[1][1], a[2][0], a[2][1], a[3][0], a[3][1]};
  const h8 y = {b[0][0], b[0][1], b[1][0], b[1][1], b[2][0], b[2][1], b[3][0], b[3][1]};
  add_class<MT, 4 * P + B, true>(st, x, y, d, acc);
}

template <int MT>
__device__ inline void block_q6k(const char* st, const Raw<FMT_Q6K>& w, Acc<MT>& acc) {
  // scale = lo + hi, lo = scale & 15, hi a multiple of 16 in [-128, 112]
  h2 lo[4], hi[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t sw = w.sc[i >> 1];
    const uint32_t s = i & 1 ? pair_bytes<2>(sw, sw >> 8) : pair_bytes<0>(sw, sw >> 8);
    lo[i] = as_h2((s & 0x000F000Fu) | kMagic) + splat((_Float16)-1024.0f);
    hi[i] = as_h2(((s ^ 0x00800080u) & 0x00F000F0u) | kMagic) + splat((_Float16)-1152.0f);
  }
  float d[MT][4];
  scales<MT>(st, (float)__builtin_bit_cast(_Float16, (uint16_t)w.d), d);
  auto half = [&](auto pc) {
    constexpr int P = decltype(pc)::value;
    uint32_t v[8];
#pragma unroll
    for (int mm = 0; mm < 8; ++mm) {
      const uint32_t n = (mm >= 4 ? w.ql[P][mm & 3] >> 4 : w.ql[P][mm & 3]) & 0x0F0F0F0Fu;
      const uint32_t hq = w.qh[P][mm & 1];
      const int sh = 4 - 2 * (mm >> 1);
      v[mm] = n | ((sh >= 0 ? hq << sh : hq >> -sh) & 0x30303030u);
    }
    class_q6k<MT, P, 0>(st, v, lo, hi, d, acc);
    class_q6k<MT, P, 1>(st, v, lo, hi, d, acc);
    class_q6k<MT, P, 2>(st, v, lo, hi, d, acc);
    class_q6k<MT, P, 3>(st, v, lo, hi, d, acc);
  };
  half(std::integral_constant<int, 0>{});
  half(std::integral_constant<int, 1>{});
}

// Planes of the matrix a wave works on.
struct Planes {
  const uint8_t *p0, *p1, *p2, *p3;
};

// The K loop of a workgroup: v[t][i] = output (weight row sub * 16 + (lane &
// 15), batch row 16 (bt0 + t) + 4 (lane >> 4) + i). Tiles past the last are
// computed on the last one's operands and dropped by the caller. lds: two
// stages; every wave of the workgroup calls it. Weights and activation
// operands are loaded into register rings D blocks deep, so a block's loads
// have D - 1 blocks of work to arrive under.
template <int FMT, int MT, int NW>
__device__ void mm_loop(const Planes& w, int nsb, int sub, const char* act, int bt0, int nbt, char* lds,
                        float (&v)[MT][4]) {
  constexpr int NT = 64 * NW, NU = MT * 512 / NT, D = MT == 1 ? 3 : 2;
  static_assert(NU * NT == MT * 512 && MT * kTailUnits <= NT, "units of a stage per thread");
  const int tid = threadIdx.x, row = sub * 16 + (tid & 15);
  const size_t ld_bt = (size_t)nsb * kStageBytes;
  // this thread's units of a stage: where they come from (block 0) and go to
  const char* src[NU];
  int dst[NU];
#pragma unroll
  for (int i = 0; i < NU; ++i) {
    const int un = tid + i * NT, t = un >> 9, off = (un & 511) * 16;
    src[i] = act + (size_t)min(bt0 + t, nbt - 1) * ld_bt + off;
    dst[i] = t * kStageBytes + off;
  }
  const bool tail = tid < MT * kTailUnits;
  const int tt = tail ? tid / kTailUnits : 0, toff = kSumOff + (tail ? tid % kTailUnits : 0) * 16;
  const char* tsrc = act + (size_t)min(bt0 + tt, nbt - 1) * ld_bt + toff;
  const int tdst = tt * kStageBytes + toff;
  u4v x[D][NU], xt[D];
  Raw<FMT> raw[D];
  auto fetch = [&](int sb, u4v (&xs)[NU], u4v& xe) {
    const size_t o = (size_t)sb * kStageBytes;
#pragma unroll
    for (int i = 0; i < NU; ++i) xs[i] = *reinterpret_cast<const u4v*>(src[i] + o);
    if (tail) xe = *reinterpret_cast<const u4v*>(tsrc + o);
  };
  auto publish = [&](char* st, const u4v (&xs)[NU], const u4v& xe) {
#pragma unroll
    for (int i = 0; i < NU; ++i) *reinterpret_cast<u4v*>(st + dst[i]) = xs[i];
    if (tail) *reinterpret_cast<u4v*>(st + tdst) = xe;
  };
  Acc<MT> acc;
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      acc.m[t][i] = 0.0f;
#pragma unroll
      for (int l = 0; l < 8; ++l) acc.s[t][l][i] = 0.0f;
    }
#pragma unroll
  for (int j = 0; j < D; ++j) {
    const int sb = min(j, nsb - 1);
    fetch(sb, x[j], xt[j]);
    raw[j].load(w.p0, w.p1, w.p2, w.p3, row, sb, nsb);
  }
  publish(lds, x[0], xt[0]);
  for (int s0 = 0; s0 < nsb; s0 += D) {
#pragma unroll
    for (int j = 0; j < D; ++j) {
      const int sb = s0 + j;
      if (sb >= nsb) break;
      __syncthreads();  // stage sb is whole; everyone is done with stage sb - 1
      // past the last block the ring refills with it: no branch around the loads
      const int nx = min(sb + D, nsb - 1);
      fetch(nx, x[j], xt[j]);
      const char* st = lds + (sb & 1) * MT * kStageBytes;
      if constexpr (FMT == FMT_Q4K) block_q4k<MT>(st, raw[j], acc);
      else block_q6k<MT>(st, raw[j], acc);
      raw[j].load(w.p0, w.p1, w.p2, w.p3, row, nx, nsb);
      publish(lds + ((sb + 1) & 1) * MT * kStageBytes, x[(j + 1) % D], xt[(j + 1) % D]);
    }
  }
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float f = acc.m[t][i];
#pragma unroll
      for (int l = 0; l < 8; ++l) f += acc.s[t][l][i];
      v[t][i] = f;
    }
}

template <int FMT, int MT, int NW, int EPI>
__device__ void mm_tile(const GemvArgs& a, const char* act, int group, int bt0, int rows, char* lds) {
  constexpr int NS = EPI == EPI_SWIGLU ? NW / 2 : NW;  // 16-row subtiles per workgroup
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const bool second = EPI == EPI_SWIGLU && wv >= NS;  // the up matrix
  const int nsub = (a.n_out + 15) >> 4;
  const int sub = group * NS + (second ? wv - NS : wv);
  const Planes w = second ? Planes{a.u0, a.u1, a.u2, a.u3} : Planes{a.p0, a.p1, a.p2, a.p3};
  const int nbt = (rows + 15) >> 4;
  float v[MT][4];
  mm_loop<FMT, MT, NW>(w, a.nsb, min(sub, nsub - 1), act, bt0, nbt, lds, v);
  const int n = sub * 16 + (lane & 15);
  if constexpr (EPI == EPI_SWIGLU) {
    f4* ex = reinterpret_cast<f4*>(lds) + (size_t)(second ? wv - NS : wv) * MT * 64 + lane;
    __syncthreads();
    if (second) {
#pragma unroll
      for (int t = 0; t < MT; ++t) ex[t * 64] = f4{v[t][0], v[t][1], v[t][2], v[t][3]};
    }
    __syncthreads();
    if (second) return;
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      const f4 up = ex[t * 64];
#pragma unroll
      for (int i = 0; i < 4; ++i) v[t][i] = silu_f(v[t][i]) * up[i];
    }
  }
  if (n >= a.n_out) return;
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int b = (bt0 + t) * 16 + 4 * (lane >> 4) + i;
      if (b >= rows) continue;
      if constexpr (EPI == EPI_RES) a.y[(size_t)b * a.ldy + n] = a.res[(size_t)b * a.ldres + n] + v[t][i];
      else a.y[(size_t)b * a.ldy + n] = v[t][i];
    }
}

template <int FMT, int MT, int NW, int EPI>
__global__ __launch_bounds__(64 * NW, 2) void q8_mm_kernel(GemvArgs a, const char* __restrict__ act, int rows) {
  extern __shared__ __attribute__((aligned(16))) char dsm[];
  mm_tile<FMT, MT, NW, EPI>(a, act, blockIdx.x, blockIdx.y * MT, rows, dsm);
}

// two matrices over the same rows: workgroups below split take groups of a, the rest of b
template <int FMT, int FMT2, int MT, int NW>
__global__ __launch_bounds__(64 * NW, 2) void q8_mm_pair_kernel(GemvArgs a, GemvArgs b, int split,
                                                             const char* __restrict__ act, int rows) {
  extern __shared__ __attribute__((aligned(16))) char dsm[];
  if ((int)blockIdx.x < split) mm_tile<FMT, MT, NW, EPI_STORE>(a, act, blockIdx.x, blockIdx.y * MT, rows, dsm);
  else mm_tile<FMT2, MT, NW, EPI_STORE>(b, act, blockIdx.x - split, blockIdx.y * MT, rows, dsm);
}

int groups_of(int n_out, int per) { return ((n_out + 15) / 16 + per - 1) / per; }

template <int FMT, int MT, int EPI>
void launch_mm(const GemvArgs& a, const char* act, int rows, hipStream_t s) {
  constexpr int NW = 4;
  constexpr size_t lds = 2 * MT * (size_t)kStageBytes;
  const int gx = groups_of(a.n_out, EPI == EPI_SWIGLU ? NW / 2 : NW), gy = ((rows + 15) / 16 + MT - 1) / MT;
  hipLaunchKernelGGL((q8_mm_kernel<FMT, MT, NW, EPI>), dim3(gx, gy), dim3(64 * NW), lds, s, a, act, rows);
  PGD_HIP(hipGetLastError());
}

template <int FMT, int FMT2, int MT>
void launch_mm_pair(const GemvArgs& a, const GemvArgs& b, const char* act, int rows, hipStream_t s) {
  constexpr int NW = 4;
  constexpr size_t lds = 2 * MT * (size_t)kStageBytes;
  const int ga = groups_of(a.n_out, NW), gb = groups_of(b.n_out, NW), gy = ((rows + 15) / 16 + MT - 1) / MT;
  hipLaunchKernelGGL((q8_mm_pair_kernel<FMT, FMT2, MT, NW>), dim3(ga + gb, gy), dim3(64 * NW), lds, s, a, b, ga, act,
                     rows);
  PGD_HIP(hipGetLastError());
}

// Activation tiles per workgroup (waves: the launch's 16-row weight subtiles).
// Two tiles share one unpacking of the weights, worth it once the launch has
// about a workgroup per CU that way: 896 x 4864 Q6_K at 1000 rows (441
// workgroups) 70.7 us with one tile, 53.8 with two; at 333 rows (154) two
// tiles would leave CUs idle. Four spill (144 accumulators).
int pick_mt(int waves, int rows) {
  const int nbt = (rows + 15) / 16;
  return nbt > 1 && (waves / 4) * ((nbt + 1) / 2) >= 200 ? 2 : 1;
}

const char* prep(const float* x, int ldx, int rows, int n_in, int nsb, hipStream_t s) {
  const int nbt = (rows + 15) / 16;
  char* act = static_cast<char*>(gemv_scratch(s, (size_t)nbt * nsb * kStageBytes, 2));
  hipLaunchKernelGGL(q8k_prep_kernel, dim3(nsb, nbt), dim3(256), 0, s, x, ldx, rows, n_in, nsb, act);
  PGD_HIP(hipGetLastError());
  return act;
}

template <int FMT, int EPI>
void run_mm(const GemvArgs& a, const char* act, int rows, hipStream_t s) {
  switch (pick_mt((EPI == EPI_SWIGLU ? 2 : 1) * ((a.n_out + 15) / 16), rows)) {
    case 2: return launch_mm<FMT, 2, EPI>(a, act, rows, s);
    default: return launch_mm<FMT, 1, EPI>(a, act, rows, s);
  }
}

template <int FMT>
void run_epi(const GemvArgs& a, const char* act, int rows, int epi, hipStream_t s) {
  if (epi == EPI_SWIGLU) run_mm<FMT, EPI_SWIGLU>(a, act, rows, s);
  else if (epi == EPI_RES) run_mm<FMT, EPI_RES>(a, act, rows, s);
  else run_mm<FMT, EPI_STORE>(a, act, rows, s);
}

template <int FMT, int FMT2>
void run_pair(const GemvArgs& a, const GemvArgs& b, const char* act, int rows, hipStream_t s) {
  switch (pick_mt((a.n_out + 15) / 16 + (b.n_out + 15) / 16, rows)) {
    case 2: return launch_mm_pair<FMT, FMT2, 2>(a, b, act, rows, s);
    default: return launch_mm_pair<FMT, FMT2, 1>(a, b, act, rows, s);
  }
}

void advance(GemvArgs& a, int rows) {
  a.x = reinterpret_cast<const float*>(a.x) + (size_t)rows * a.ldx;
  a.y += (size_t)rows * a.ldy;
  if (a.res) a.res += (size_t)rows * a.ldres;
}

// The operands lie in the stream's scratch between the two launches. Held over
// both, so that no other host thread's call on the stream is queued between
// them or replaces the buffer.
std::mutex g_operands;

}  // namespace

// Microseconds of up to 16 rows: both launches and the K chain, once per round
// of a workgroup on each CU (a second one of any size counts 0.6). Measured
// over the same shapes as q8k_us, within 10% up to 1024 tiles.
double q8_gemm_us(int fmt, int tiles16, int nsb) {
  const double rounds = tiles16 / 4 / 256.0;
  return 5.9 + (fmt == FMT_Q4K ? 0.76 : 1.1) * nsb * (rounds <= 1.0 ? 1.0 : std::max(1.6, 0.92 * rounds));
}

void run_q8_gemm(int fmt, GemvArgs a, int nrows, int epi, hipStream_t s) {
  for (int r0 = 0; r0 < nrows; r0 += kRowChunk) {
    const int rows = min(kRowChunk, nrows - r0);
    std::lock_guard<std::mutex> lock(g_operands);
    const char* act = prep(reinterpret_cast<const float*>(a.x), a.ldx, rows, a.n_in, a.nsb, s);
    if (fmt == FMT_Q4K) run_epi<FMT_Q4K>(a, act, rows, epi, s);
    else run_epi<FMT_Q6K>(a, act, rows, epi, s);
    advance(a, rows);
  }
}

void run_q8_gemm_pair(int fmt_a, GemvArgs a, int fmt_b, GemvArgs b, int nrows, hipStream_t s) {
  for (int r0 = 0; r0 < nrows; r0 += kRowChunk) {
    const int rows = min(kRowChunk, nrows - r0);
    std::lock_guard<std::mutex> lock(g_operands);
    const char* act = prep(reinterpret_cast<const float*>(a.x), a.ldx, rows, a.n_in, a.nsb, s);
    if (fmt_a == FMT_Q4K && fmt_b == FMT_Q4K) run_pair<FMT_Q4K, FMT_Q4K>(a, b, act, rows, s);
    else if (fmt_a == FMT_Q4K) run_pair<FMT_Q4K, FMT_Q6K>(a, b, act, rows, s);
    else if (fmt_b == FMT_Q4K) run_pair<FMT_Q6K, FMT_Q4K>(a, b, act, rows, s);
    else run_pair<FMT_Q6K, FMT_Q6K>(a, b, act, rows, s);
    advance(a, rows);
    advance(b, rows);
  }
}

}  // namespace gemv
}  // namespace pgd
