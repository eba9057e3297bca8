// gemv_q8k.hip — candle's CPU quantized matmul (gemv_q8.hip describes the
// arithmetic) for a few activation rows of Q4_K / Q6_K matrices: a decode
// step's projections, bit-equal to the CPU restatement.
//
// One workgroup per 16 weight rows (tiles of a grid-stride loop for tall
// matrices), one wave per 256-weight block at a time. Such a launch is all
// latency (28 to 300 workgroups of a few KB each), so the design is about the
// length of its chain:
//  - a wave's first block of weights is requested before anything else and
//    arrives under the quantization of the activation row;
//  - 32 lanes quantize a block (8 elements each), and leave x in LDS with the
//    four elements that one weight dword meets side by side;
//  - four lanes share a weight row of a block. A byte transpose in registers
//    (v_perm) gathers four codes of one residue class and one scale into a
//    dword, so one v_dot4 replaces four masked ones; scales multiply through
//    v_mad_i32_i24. Q6_K codes run as 4 (code - 32), the 6-bit code in the top
//    bits of a signed byte, and the exact sum is shifted back;
//  - the block terms meet in LDS and one lane per (row, class) adds them in
//    block order, then one lane per row the eight classes (GGML's order).
// Measured at one row against 32-row tiles with masked byte dots and weights
// loaded after the quantization: 4864 x 896 Q4_K 7.0 -> 4.6 us, 896 x 4864
// Q4_K 12.5 -> 6.6 us and Q6_K 15.1 -> 8.0 us, 151936 x 896 Q6_K (102 MB)
// 51.9 -> 31.6 us.
#include "common.h"
#include "gemv_impl.h"
#include "quant.h"

namespace pgd {
namespace gemv {

namespace {

typedef uint32_t u2v __attribute__((ext_vector_type(2)));
typedef uint32_t u4v __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));

constexpr int kRows = 16;       // weight rows per tile
constexpr int kMaxWaves = 16;

__device__ inline int dot4(uint32_t a, uint32_t b, int c) {
  return __builtin_amdgcn_sdot4((int)a, (int)b, c, false);
}
// the value of lane ^ 1 and lane ^ 2 of a quad
__device__ inline int quad_x1(int v) { return __builtin_amdgcn_mov_dpp(v, 0xB1, 0xF, 0xF, true); }
__device__ inline int quad_x2(int v) { return __builtin_amdgcn_mov_dpp(v, 0x4E, 0xF, 0xF, true); }
// [a.x, b.x, a.y, b.y] of bytes x = 0, y = 1 (lo) or x = 2, y = 3 (hi)
__device__ inline uint32_t zip_lo(uint32_t a, uint32_t b) { return __builtin_amdgcn_perm(b, a, 0x05010400u); }
__device__ inline uint32_t zip_hi(uint32_t a, uint32_t b) { return __builtin_amdgcn_perm(b, a, 0x07030602u); }
// the low / high halves of a and b
__device__ inline uint32_t cat_lo(uint32_t a, uint32_t b) { return __builtin_amdgcn_perm(b, a, 0x05040100u); }
__device__ inline uint32_t cat_hi(uint32_t a, uint32_t b) { return __builtin_amdgcn_perm(b, a, 0x07060302u); }

struct Planes {
  const uint8_t *p0, *p1, *p2, *p3;
};

// floats of one row's squares: whole rounds of 64 and one more that the last
// round's prefetch reads
__host__ __device__ inline int sq_stride(int n) { return ((n + 63) & ~63) + 64; }

// ((0 + q[0]) + q[1]) + ... over np (a multiple of 64) floats in LDS: the reads
// of 32 in flight under the additions of the 32 before (rmsnorm_ordered_kernel)
__device__ inline float ordered_sum(const float* q0, int np) {
  const f4* q = reinterpret_cast<const f4*>(q0);
  float ss = 0.0f;
  auto read = [&](f4 (&v)[8], int i) {
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = q[i + k];
  };
  auto add = [&](const f4 (&v)[8]) {
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      ss += v[k][0];
      ss += v[k][1];
      ss += v[k][2];
      ss += v[k][3];
    }
  };
  f4 a[8], b[8];
  read(a, 0);
  for (int i = 0; i < np / 4; i += 16) {
    read(b, i + 8);
    add(a);
    read(a, i + 16);
    add(b);
  }
  return ss;
}

// LDS: per row the quantized activation blocks (XB bytes each), Q4_K's sums of
// 32 elements and the blocks' d; the block terms [matrix][row][block][16][NT];
// the class sums [matrix][row][16][9]; with a norm, the squares of each row
// (sq_stride floats) and its rms
template <int FMT>
struct Lds {
  static constexpr int XB = FMT == FMT_Q4K ? 256 : 512;
  static constexpr int NS = FMT == FMT_Q4K ? 8 : 0;   // sums per block
  static constexpr int NT = FMT == FMT_Q4K ? 12 : 8;  // term stride: 9 (8) used, rows 16-byte aligned
  static constexpr int NC = FMT == FMT_Q4K ? 9 : 8;   // ordered sums per output
  int nb;
  char* x;
  int* bs;
  float *d, *t, *s, *sq, *rms;
  __device__ Lds(char* base, int nb_, int rb, int nm) : nb(nb_) {
    x = base;
    t = reinterpret_cast<float*>(x + (size_t)rb * nb * XB);
    s = t + (size_t)nm * rb * nb * kRows * NT;
    bs = reinterpret_cast<int*>(s + nm * rb * kRows * 9);
    d = reinterpret_cast<float*>(bs + (size_t)rb * nb * NS);
    rms = d + (size_t)rb * nb;
    sq = reinterpret_cast<float*>(((uintptr_t)(rms + rb) + 15) & ~(uintptr_t)15);
  }
  static size_t bytes(int nb, int rb, int nm, int norm_n = 0) {
    return (size_t)rb * nb * (XB + NS * 4 + 4) + (size_t)nm * rb * kRows * (nb * NT + 9) * 4 +
           (norm_n ? (size_t)rb * (sq_stride(norm_n) + 1) * 4 + 16 : 0);
  }
  __device__ float* term(int m, int rb, int r, int b, int row) const {
    return t + ((((size_t)m * rb + r) * nb + b) * kRows + row) * NT;
  }
};

// Eight consecutive elements of a row of n (zeros past its end).
__device__ inline void load8(const float* p, int left, float (&v)[8]) {
  if (left >= 8 && (((uintptr_t)p) & 15) == 0) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const f4 w = reinterpret_cast<const f4*>(p)[i];
#pragma unroll
      for (int k = 0; k < 4; ++k) v[4 * i + k] = w[k];
    }
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = i < left ? p[i] : 0.0f;
  }
}

// BlockQ8K::from_float of the launch's rows, the whole workgroup; half a wave
// per block. NORM: of x / rms * nw, rms from the squares' left-to-right sum
// (candle's rms_norm, as rmsnorm_ordered_kernel).
template <int FMT, bool NORM>
__device__ void quantize(const float* __restrict__ x, int ldx, int rows, int n_in, const float* __restrict__ nw,
                         float eps, const Lds<FMT>& L) {
  const int t = threadIdx.x & 31, hi = threadIdx.x & 32, units = rows * L.nb;
  float v[8], wv[8];
  auto fetch = [&](int un) {
    const int r = un / L.nb, e0 = (un - r * L.nb) * 256 + 8 * t;
    load8(x + (size_t)r * ldx + e0, n_in - e0, v);
    if constexpr (NORM) load8(nw + e0, n_in - e0, wv);
  };
  const int first = threadIdx.x >> 5, step = blockDim.x >> 5;
  if constexpr (NORM) {
    const int ld = sq_stride(n_in), np = ld - 64;
    for (int un = first; un < units; un += step) {
      const int r = un / L.nb, e = (un - r * L.nb) * 256 + 8 * t;
      fetch(un);
      if (e < np) {
        f4* q = reinterpret_cast<f4*>(L.sq + r * ld + e);
        q[0] = f4{v[0] * v[0], v[1] * v[1], v[2] * v[2], v[3] * v[3]};
        q[1] = f4{v[4] * v[4], v[5] * v[5], v[6] * v[6], v[7] * v[7]};
      }
    }
    __syncthreads();
    if ((int)threadIdx.x < rows)
      L.rms[threadIdx.x] = sqrtf(ordered_sum(L.sq + threadIdx.x * ld, np) / (float)n_in + eps);
    __syncthreads();
  }
  for (int un = first; un < units; un += step) {
    const int r = un / L.nb, b = un - r * L.nb;
    if (!NORM || units > step) fetch(un);  // else still in registers
    if constexpr (NORM) {
      const float m = L.rms[r];
#pragma unroll
      for (int i = 0; i < 8; ++i) v[i] = v[i] / m * wv[i];
    }
    float amax = 0.0f, mx = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (fabsf(v[i]) > amax) {
        amax = fabsf(v[i]);
        mx = v[i];
      }
    // the first element of largest magnitude: the lowest lane that holds it
    float top = amax;
#pragma unroll
    for (int o = 1; o < 32; o <<= 1) top = fmaxf(top, __shfl_xor(top, o, 64));
    const uint64_t holds = __ballot(amax == top);
    mx = __shfl(mx, hi + __builtin_ctz((uint32_t)(holds >> hi)), 64);
    const float iscale = -128.0f / mx;
    int q[8], sum = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float s = roundf(iscale * v[i]);
      q[i] = top == 0.0f ? 0 : (int)(int8_t)(int)(s < 127.0f ? s : 127.0f);
      sum += q[i];
    }
    char* xb = L.x + (size_t)un * Lds<FMT>::XB;
    if constexpr (FMT == FMT_Q4K) {
      // dword (sub-block t / 4, class l): elements 8 i + l, i = 0..3
#pragma unroll
      for (int l = 0; l < 8; ++l) xb[((t >> 2) * 8 + l) * 4 + (t & 3)] = (char)q[l];
      sum += quad_x1(sum);
      sum += quad_x2(sum);
      if ((t & 3) == 0) L.bs[un * 8 + (t >> 2)] = sum;
    } else {
      // dword (half u, class parity p, sub-block mm, class 4 p + c): elements
      // c and 8 + c of the sub-block, in the low half for even mm, else high
      const int u = t >> 4, mm = (t >> 1) & 7, sh = 16 * (mm & 1);
      u4v w[2];
#pragma unroll
      for (int l = 0; l < 8; ++l) w[l >> 2][l & 3] = ((uint32_t)(q[l] & 255) | (uint32_t)((quad_x1(q[l]) & 255) << 8)) << sh;
      if ((t & 1) == 0) {
#pragma unroll
        for (int p = 0; p < 2; ++p) *reinterpret_cast<u4v*>(xb + (((u * 2 + p) * 8 + mm) * 16)) = w[p];
      }
    }
    if (t == 0) L.d[un] = top == 0.0f ? 0.0f : 1.0f / iscale;
  }
}

template <int FMT>
struct Raw;

// Q4_K: lane 4 row + j holds 64-chunk j of its row
template <>
struct Raw<FMT_Q4K> {
  u4v q[2], hdr;
  __device__ void load(const Planes& w, int tile, int sb, int nsb) {
    const int lane = threadIdx.x & 63, row = tile * kRows + (lane >> 2), j = lane & 3;
    const u4v* p = reinterpret_cast<const u4v*>(w.p0 + q4k_qs_off(row, 32 * (4 * sb + j), nsb));
    q[0] = p[0];
    q[1] = p[1];
    hdr = *reinterpret_cast<const u4v*>(w.p1 + q4k_hdr_off(row, sb, nsb));
  }
  __device__ void terms(const Lds<FMT_Q4K>& L, int m, int rb, int rows, int sb) const {
    const int lane = threadIdx.x & 63, row = lane >> 2, j = lane & 3;
    // scales and mins of sub-blocks 2j and 2j + 1
    const int sh = 16 * (j & 1);
    const uint32_t a = hdr[1] >> sh, b = hdr[2] >> sh, c = hdr[3] >> sh;
    const uint32_t sc = j < 2 ? a & 0x3F3Fu : (c & 0x0F0Fu) | ((a >> 2) & 0x3030u);
    const uint32_t mn = j < 2 ? b & 0x3F3Fu : ((c >> 4) & 0x0F0Fu) | ((b >> 2) & 0x3030u);
    const int s0 = (int)(sc & 63u), s1 = (int)((sc >> 8) & 63u), m0 = (int)(mn & 63u), m1 = (int)((mn >> 8) & 63u);
    const float dw = (float)__builtin_bit_cast(_Float16, (uint16_t)(hdr[0] & 0xffffu));
    const float dmin = (float)__builtin_bit_cast(_Float16, (uint16_t)(hdr[0] >> 16));
    // byte i of dword l: code 8 i + l of the chunk's first (low nibble) and second 32 codes
    uint32_t w[8];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const uint32_t b0 = q[0][h], b1 = q[0][2 + h], b2 = q[1][h], b3 = q[1][2 + h];
      const uint32_t l01 = zip_lo(b0, b1), h01 = zip_hi(b0, b1), l23 = zip_lo(b2, b3), h23 = zip_hi(b2, b3);
      w[4 * h] = cat_lo(l01, l23);
      w[4 * h + 1] = cat_hi(l01, l23);
      w[4 * h + 2] = cat_lo(h01, h23);
      w[4 * h + 3] = cat_hi(h01, h23);
    }
    for (int r = 0; r < rows; ++r) {
      const int un = r * L.nb + sb;
      const u4v* xb = reinterpret_cast<const u4v*>(L.x + (size_t)un * Lds<FMT_Q4K>::XB) + 4 * j;
      const u4v xl[2] = {xb[0], xb[1]}, xh[2] = {xb[2], xb[3]};
      int aux[8];
#pragma unroll
      for (int l = 0; l < 8; ++l) {
        aux[l] = __mul24(s0, dot4(w[l] & 0x0F0F0F0Fu, xl[l >> 2][l & 3], 0));
        aux[l] += __mul24(s1, dot4((w[l] >> 4) & 0x0F0F0F0Fu, xh[l >> 2][l & 3], 0));
        aux[l] += quad_x1(aux[l]);
        aux[l] += quad_x2(aux[l]);
      }
      int ms = __mul24(m0, L.bs[un * 8 + 2 * j]) + __mul24(m1, L.bs[un * 8 + 2 * j + 1]);
      ms += quad_x1(ms);
      ms += quad_x2(ms);
      const float d8 = L.d[un], d = dw * d8;
      float* t = L.term(m, rb, r, sb, row);
      if (j == 0) {
        reinterpret_cast<f4*>(t)[0] = f4{d * (float)aux[0], d * (float)aux[1], d * (float)aux[2], d * (float)aux[3]};
        reinterpret_cast<f4*>(t)[1] = f4{d * (float)aux[4], d * (float)aux[5], d * (float)aux[6], d * (float)aux[7]};
        t[8] = dmin * d8 * (float)ms;
      }
    }
  }
};

// Q6_K: lane 4 row + 2 u + p holds half u's elements of classes 4 p .. 4 p + 3
template <>
struct Raw<FMT_Q6K> {
  u4v ql[2];  // elements 16 mm + 8 kk + 4 p + c: kk = 0, 1
  u2v qh[2], sc;
  uint32_t d;
  __device__ void load(const Planes& w, int tile, int sb, int nsb) {
    const int lane = threadIdx.x & 63, row = tile * kRows + (lane >> 2), u = (lane >> 1) & 1, p = lane & 1;
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      const int i = 4 * (2 * kk + p);
      ql[kk] = *reinterpret_cast<const u4v*>(w.p0 + q6k_ql_off(row, 64 * (2 * sb + u) + i, nsb));
      qh[kk] = *reinterpret_cast<const u2v*>(w.p1 + q6k_qh_off(row, 32 * (2 * sb + u) + i, nsb));
    }
    sc = *reinterpret_cast<const u2v*>(w.p2 + q6k_sc_off(row, 16 * sb + 8 * u, nsb));
    d = reinterpret_cast<const uint16_t*>(w.p3)[q6k_d_off(row, sb, nsb)];
  }
  // bytes 4 (code - 32) of sub-block mm
  __device__ uint32_t codes(int kk, int mm) const {
    const uint32_t n = ql[kk][mm & 3], h = qh[kk][mm & 1];
    return (((mm < 4 ? n << 2 : n >> 2) & 0x3C3C3C3Cu) | ((h << (6 - 2 * (mm >> 1))) & 0xC0C0C0C0u)) ^ 0x80808080u;
  }
  __device__ void terms(const Lds<FMT_Q6K>& L, int m, int rb, int rows, int sb) const {
    const int lane = threadIdx.x & 63, row = lane >> 2, up = lane & 3;
    const float dw = (float)__builtin_bit_cast(_Float16, (uint16_t)d);
    // byte order of w[i][c]: class 4 p + c of sub-blocks 2 i (kk 0, 1) and 2 i + 1
    uint32_t w[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t a0 = codes(0, 2 * i), b0 = codes(1, 2 * i), a1 = codes(0, 2 * i + 1), b1 = codes(1, 2 * i + 1);
      const uint32_t l0 = zip_lo(a0, b0), h0 = zip_hi(a0, b0), l1 = zip_lo(a1, b1), h1 = zip_hi(a1, b1);
      w[i][0] = cat_lo(l0, l1);
      w[i][1] = cat_hi(l0, l1);
      w[i][2] = cat_lo(h0, h1);
      w[i][3] = cat_hi(h0, h1);
    }
    for (int r = 0; r < rows; ++r) {
      const int un = r * L.nb + sb;
      const u4v* xb = reinterpret_cast<const u4v*>(L.x + (size_t)un * Lds<FMT_Q6K>::XB) + 8 * up;
      int aux[4] = {0, 0, 0, 0};
#pragma unroll
      for (int mm = 0; mm < 8; ++mm) {
        const u4v x = xb[mm];
        const int s = (int)(int8_t)((sc[mm >> 2] >> (8 * (mm & 3))) & 255u);
#pragma unroll
        for (int c = 0; c < 4; ++c) aux[c] += __mul24(s, dot4(w[mm >> 1][c], x[c], 0));
      }
#pragma unroll
      for (int c = 0; c < 4; ++c) aux[c] = (aux[c] + quad_x2(aux[c])) >> 2;
      const float dd = dw * L.d[un];
      if (up < 2)
        *reinterpret_cast<f4*>(L.term(m, rb, r, sb, row) + 4 * up) =
            f4{dd * (float)aux[0], dd * (float)aux[1], dd * (float)aux[2], dd * (float)aux[3]};
    }
  }
};

// The tiles of one matrix (two for SwiGLU) that this workgroup owns: block
// terms, the ordered sums, the epilogue. rb: row capacity of the LDS layout.
template <int FMT, int EPI, bool NORM>
__device__ void run_tiles(const GemvArgs& a, int first, int ntiles, int stride, int rows, int rb, char* lds) {
  constexpr int NM = EPI == EPI_SWIGLU ? 2 : 1, NC = Lds<FMT>::NC;
  const int nb = a.nsb, units = NM * nb, nw = blockDim.x >> 6, wv = threadIdx.x >> 6;
  const Lds<FMT> L(lds, nb, rb, NM);
  auto load = [&](Raw<FMT>& w, int tile, int unit) {
    const bool up = NM == 2 && unit >= nb;
    const Planes p = up ? Planes{a.u0, a.u1, a.u2, a.u3} : Planes{a.p0, a.p1, a.p2, a.p3};
    w.load(p, tile, up ? unit - nb : unit, nb);
  };
  // a wave without a block of its own loads (and drops) the last one
  Raw<FMT> cur, nxt;
  load(cur, first, min(wv, units - 1));
  quantize<FMT, NORM>(reinterpret_cast<const float*>(a.x), a.ldx, rows, a.n_in, a.nw, a.rss_eps, L);
  __syncthreads();
  for (int tile = first; tile < ntiles; tile += stride) {
    for (int unit = wv; unit < units; unit += nw) {
      // the next block (of this tile, or the wave's first of the next one) is on its way meanwhile
      const bool last = unit + nw >= units;
      load(nxt, last ? min(tile + stride, ntiles - 1) : tile, last ? wv : unit + nw);
      cur.terms(L, unit >= nb ? 1 : 0, rb, rows, unit >= nb ? unit - nb : unit);
      cur = nxt;
    }
    __syncthreads();
    for (int i = threadIdx.x; i < NM * rows * kRows * NC; i += blockDim.x) {
      const int c = i % NC, o = i / NC, row = o % kRows, mr = o / kRows, m = mr / rows, r = mr - m * rows;
      const float* t = L.term(m, rb, r, 0, row) + c;
      // class sums add block after block; the min terms are subtracted
      float s = 0.0f;
      int b = 0;
      for (; b + 4 <= nb; b += 4) {
        float v[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) v[k] = t[(size_t)(b + k) * kRows * Lds<FMT>::NT];
#pragma unroll
        for (int k = 0; k < 4; ++k) s = c == 8 ? s - v[k] : s + v[k];
      }
      for (; b < nb; ++b) {
        const float v = t[(size_t)b * kRows * Lds<FMT>::NT];
        s = c == 8 ? s - v : s + v;
      }
      L.s[o * 9 + c] = s;
    }
    __syncthreads();
    for (int o = threadIdx.x; o < rows * kRows; o += blockDim.x) {
      const int r = o / kRows, n = tile * kRows + o % kRows;
      float v[NM];
#pragma unroll
      for (int m = 0; m < NM; ++m) {
        const float* s = L.s + (m * rows * kRows + o) * 9;
        float f = NC == 9 ? s[8] : 0.0f;
#pragma unroll
        for (int l = 0; l < 8; ++l) f += s[l];
        v[m] = f;
      }
      if (n < a.n_out) {
        const size_t at = (size_t)r * a.ldy + n;
        if constexpr (EPI == EPI_STORE) a.y[at] = v[0];
        if constexpr (EPI == EPI_RES) a.y[at] = a.res[(size_t)r * a.ldres + n] + v[0];
        if constexpr (EPI == EPI_SWIGLU) a.y[at] = silu_f(v[0]) * v[NM - 1];
      }
    }
    // the next tile's terms do not touch L.s; its sums come after a barrier
  }
}

template <int FMT, int EPI, bool NORM>
__global__ __launch_bounds__(64 * kMaxWaves) void q8k_kernel(GemvArgs a, int ntiles, int rows, int rb) {
  extern __shared__ __attribute__((aligned(16))) char dsm[];
  run_tiles<FMT, EPI, NORM>(a, blockIdx.x, ntiles, gridDim.x, rows, rb, dsm);
}

// Two matrices of one input: workgroups below split take tiles of a, the rest
// of b, each quantizing the rows in its own format's layout.
template <int FMT, int FMT2, bool NORM>
__global__ __launch_bounds__(64 * kMaxWaves) void q8k_pair_kernel(GemvArgs a, GemvArgs b, int split, int rows, int rb) {
  extern __shared__ __attribute__((aligned(16))) char dsm[];
  const int id = blockIdx.x;
  if (id < split) run_tiles<FMT, EPI_STORE, NORM>(a, id, id + 1, 1, rows, rb, dsm);
  else run_tiles<FMT2, EPI_STORE, NORM>(b, id - split, id - split + 1, 1, rows, rb, dsm);
}

constexpr size_t kLdsMax = 160 * 1024;
// workgroups of a launch: past the chip's wave slots (2048 of 4 waves) a
// workgroup takes several tiles, so the row is quantized fewer times
constexpr int kMaxGroups = 2048;

int tiles_of(int n_out) { return (n_out + kRows - 1) / kRows; }

// waves per workgroup: one per block up to 16, else an even share
int waves_of(int units) {
  if (units <= kMaxWaves) return units < 4 ? 4 : units;
  const int each = (units + kMaxWaves - 1) / kMaxWaves;
  return (units + each - 1) / each;
}

template <class K>
void allow_lds(K kernel) {
  PGD_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                              (int)kLdsMax));
}

void advance(GemvArgs& a, int rows) {
  a.x = reinterpret_cast<const float*>(a.x) + (size_t)rows * a.ldx;
  a.y += (size_t)rows * a.ldy;
  if (a.res) a.res += (size_t)rows * a.ldres;
}

template <int FMT, int EPI, bool NORM>
void launch(GemvArgs a, int nrows, hipStream_t s) {
  constexpr int NM = EPI == EPI_SWIGLU ? 2 : 1;
  auto need = [&](int rb) { return Lds<FMT>::bytes(a.nsb, rb, NM, NORM ? a.n_in : 0); };
  // wide rows: one row per launch where the rows' terms do not fit together
  const int rb = need(nrows) <= kLdsMax ? nrows : 1;
  const size_t lds = need(rb);
  PGD_CHECK(lds <= kLdsMax, kErrShape, "activation rows too wide for the quantized-activation GEMV");
  if (lds > 64 * 1024) {
    static const bool ok = (allow_lds(&q8k_kernel<FMT, EPI, NORM>), true);
    (void)ok;
  }
  const int tiles = tiles_of(a.n_out), nw = waves_of(NM * a.nsb);
  for (int r0 = 0; r0 < nrows; r0 += rb) {
    const int rows = min(rb, nrows - r0);
    hipLaunchKernelGGL((q8k_kernel<FMT, EPI, NORM>), dim3(min(tiles, kMaxGroups)), dim3(64 * nw), lds, s, a, tiles,
                       rows, rb);
    PGD_HIP(hipGetLastError());
    advance(a, rows);
  }
}

template <int FMT, int FMT2, bool NORM>
void launch_pair(GemvArgs a, GemvArgs b, int nrows, hipStream_t s) {
  auto need = [&](int rb) {
    const int n = NORM ? a.n_in : 0;
    return std::max(Lds<FMT>::bytes(a.nsb, rb, 1, n), Lds<FMT2>::bytes(a.nsb, rb, 1, n));
  };
  const int rb = need(nrows) <= kLdsMax ? nrows : 1;
  const size_t lds = need(rb);
  PGD_CHECK(lds <= kLdsMax, kErrShape, "activation rows too wide for the quantized-activation GEMV");
  if (lds > 64 * 1024) {
    static const bool ok = (allow_lds(&q8k_pair_kernel<FMT, FMT2, NORM>), true);
    (void)ok;
  }
  const int ta = tiles_of(a.n_out), tb = tiles_of(b.n_out), nw = waves_of(a.nsb);
  for (int r0 = 0; r0 < nrows; r0 += rb) {
    const int rows = min(rb, nrows - r0);
    hipLaunchKernelGGL((q8k_pair_kernel<FMT, FMT2, NORM>), dim3(ta + tb), dim3(64 * nw), lds, s, a, b, ta, rows, rb);
    PGD_HIP(hipGetLastError());
    advance(a, rows);
    advance(b, rows);
  }
}

template <int FMT>
void run_epi(const GemvArgs& a, int nrows, int epi, hipStream_t s) {
  if (epi == EPI_SWIGLU) {
    if (a.nw) launch<FMT, EPI_SWIGLU, true>(a, nrows, s);
    else launch<FMT, EPI_SWIGLU, false>(a, nrows, s);
  } else if (epi == EPI_RES) {
    launch<FMT, EPI_RES, false>(a, nrows, s);
  } else {
    launch<FMT, EPI_STORE, false>(a, nrows, s);
  }
}

template <int FMT, int FMT2>
void run_pair(const GemvArgs& a, const GemvArgs& b, int nrows, hipStream_t s) {
  if (a.nw) launch_pair<FMT, FMT2, true>(a, b, nrows, s);
  else launch_pair<FMT, FMT2, false>(a, b, nrows, s);
}

}  // namespace

void run_q8k_gemv(int fmt, const GemvArgs& a, int nrows, int epi, hipStream_t s) {
  if (fmt == FMT_Q4K) run_epi<FMT_Q4K>(a, nrows, epi, s);
  else run_epi<FMT_Q6K>(a, nrows, epi, s);
}

void run_q8k_gemv_pair(int fmt_a, const GemvArgs& a, int fmt_b, const GemvArgs& b, int nrows, hipStream_t s) {
  if (fmt_a == FMT_Q4K && fmt_b == FMT_Q4K) run_pair<FMT_Q4K, FMT_Q4K>(a, b, nrows, s);
  else if (fmt_a == FMT_Q4K) run_pair<FMT_Q4K, FMT_Q6K>(a, b, nrows, s);
  else if (fmt_b == FMT_Q4K) run_pair<FMT_Q6K, FMT_Q4K>(a, b, nrows, s);
  else run_pair<FMT_Q6K, FMT_Q6K>(a, b, nrows, s);
}

// Microseconds of run_q8k_gemv. The workgroups of a CU share its issue slots (24
// waves of these kernels fit, by 80 registers; one of 14 waves or more, or one
// that fills the LDS, has the CU to itself), a row costs about as much per K
// block in each; rows that do not fit the LDS together run one launch each.
// Fitted to 33 shapes of 256..152064 x 896..18944 in both formats at 1..8 rows:
// 3% off in the median. What q8act_few_rows chooses by it is 0.1% slower than
// the faster of both on average, 8% at most but for 152064 x 896 (21%, 2 rows).
double q8k_us(int fmt, int tiles16, int nsb, int nrows, int nm) {
  auto need = [&](int rb) {
    return fmt == FMT_Q4K ? Lds<FMT_Q4K>::bytes(nsb, rb, nm) : Lds<FMT_Q6K>::bytes(nsb, rb, nm);
  };
  if (nrows > 1 && need(nrows) > kLdsMax) return nrows * q8k_us(fmt, tiles16, nsb, 1, nm);
  const int nw = waves_of(nm * nsb);
  const int per_cu = std::max(1, std::min((int)(kLdsMax / need(nrows)), 24 / nw));
  const double blocks = (fmt == FMT_Q4K ? 1.0 : 1.3) * nm * nsb;
  const double one = 2.4 + 0.07 * blocks + nrows * ((nm * nsb <= kMaxWaves ? 0.55 : 1.15) + 0.065 * blocks);
  return 1.0 + one * (1.0 + std::max(0.93 / per_cu, nw / 17.5) * ((tiles16 + 255) / 256 - 1));
}

// Every workgroup of a launch with the norm repeats the chain of n_in additions,
// so the norm goes in only where all of them are resident at once: per CU the
// LDS, and 16 waves (the kernels' 128 registers), at most two. A second round
// repeats the chain. us per layer of a decode step, norm inside / in its own
// launch: 4608 x 3584 (288 workgroups of 14 waves) 1 row 139.5 / 134.1, 5 rows
// 142 / 133; gate/up 8192 x 2048 (512 of 16 waves) 76.1 / 71.2; in one round
// (1152 x 896 and gate/up 4864 x 896) 47.5 / 51.1.
bool q8k_norm_ok(int tiles16, int nsb, int n_in, int nrows, int nm) {
  const size_t lds =
      std::max(Lds<FMT_Q4K>::bytes(nsb, nrows, nm, n_in), Lds<FMT_Q6K>::bytes(nsb, nrows, nm, n_in));
  if (n_in > 8192 || lds > kLdsMax) return false;
  const int per_cu = std::min(std::min((int)(kLdsMax / lds), kMaxWaves / waves_of(nm * nsb)), 2);
  return tiles16 <= 256 * per_cu;
}

}  // namespace gemv
}  // namespace pgd
