// gemv_q8.hip — GGML-format GEMV with the arithmetic of candle's CPU
// quantized matmul (the reference's CPU path keeps QMatMul for the Qwen2 GGUF
// weights, pagoda-hf/src/qwen2_gguf.rs:280-289): every activation row is
// quantized to the weight type's vec_dot_type and each output is an integer
// block dot scaled in f32.
//
//   Q4_K, Q6_K  x  Q8_K  (256-element blocks: f32 d, 256 i8, 16 i16 sums)
//   Q8_0, Q5_0  x  Q8_0  (32-element blocks: f16 d, 32 i8)
//
// Activation quantization (BlockQ8K / BlockQ8_0 ::from_float): Q8_K takes the
// first element of largest magnitude as max, iscale = -128 / max,
// q = min(127, round(iscale x)) (round half away from zero), d = 1 / iscale,
// and the sums of each 16 q; Q8_0 takes d = amax / 127, q = round(x / d)
// with d rounded to f16. Every workgroup quantizes the launch's rows into LDS
// itself (no separate launch); all of them compute the same bytes.
//
// Block dots: integer products through v_dot4 (exact), per weight block
//   Q4_K: d_w d_x sum_j sc_j dot_j - dmin_w d_x sum_j m_j bsum_j
//   Q6_K: d_w d_x sum_j sc_j (dot_j(q) - 32 bsum_j)       (q = 6-bit code)
//   Q8_0: sumi d_w d_x;  Q5_0: (dot(q) - 16 sum(x_q)) d_w d_x   (q = 5-bit code)
// The float arithmetic is GGML's scalar one, term for term and in its order,
// so every output is bit-equal to the CPU restatement: the integer products
// of a 256-block are kept in eight residue classes (element index mod 8,
// GGML's aux32[8] lanes), each scaled by d = d_w d_x and added into its own
// running sum block after block, the Q4_K min terms into a ninth, and the
// eight sums are added at the end; 32-blocks add (sumi d_w) d_x block after
// block. Waves compute their blocks' terms in parallel (exact integers, one
// rounding per product) and leave them in LDS; one lane per output then adds
// them in block order. The per-row arithmetic does not depend on the number
// of rows, so batched rows are bitwise equal to single-row launches.
//
// This file holds the choice of kernel and the Q8_0 / Q5_0 kernels; Q4_K /
// Q6_K run in gemv_q8k.hip (a few rows) and gemm_q8.hip (more, on the matrix
// cores), with the same bits. Work split here: one workgroup of NW waves (4
// or 8, from the number of K blocks) per 32-row tile of the weight matrix;
// wave w takes K blocks w, w + NW, ... Weights are read once per launch of up
// to RB activation rows.
#include <type_traits>

#include "common.h"
#include "gemv_impl.h"
#include "quant.h"

namespace pgd {
namespace gemv {

namespace {


typedef uint32_t u2v __attribute__((ext_vector_type(2)));

__device__ inline int dot4(uint32_t a, uint32_t b, int c) {
  return __builtin_amdgcn_sdot4((int)a, (int)b, c, false);
}

// activations in LDS: q [RB][n_in] i8 | d [RB][nb] f32 | sums [RB][nb] i32,
// then the block terms [NM][RB][nb][32 outputs] f32
template <int RB>
struct ActLds {
  int n_in, nb;
  int8_t* q;
  float* d;
  int* s;
  float* t;
  __host__ __device__ static size_t act_bytes(int nbh) { return ((size_t)RB * nbh * 40 + 15) & ~(size_t)15; }
  __device__ ActLds(char* base, int k) : n_in(k), nb(k / 32) {
    q = reinterpret_cast<int8_t*>(base);
    d = reinterpret_cast<float*>(base + (size_t)RB * n_in);
    s = reinterpret_cast<int*>(d + RB * nb);
    t = reinterpret_cast<float*>(base + act_bytes(nb));
  }
  // term of matrix m, row r, block b, tile output n
  __device__ float& term(int m, int r, int b, int n) const { return t[(((size_t)m * RB + r) * nb + b) * 32 + n]; }
  static size_t bytes(int n_in, int nm) {
    const int nbh = n_in / 32;
    return act_bytes(nbh) + (size_t)nm * RB * nbh * 32 * 4;
  }
};

// Quantize rows [0, rows) of x (the launch's chunk) into LDS; the whole
// workgroup calls it.
template <int RB>
__device__ void quantize_rows(const float* __restrict__ x, int ldx, int rows, const ActLds<RB>& L) {
  // one lane per 32-element block
  const int units = rows * L.nb;
  for (int u = threadIdx.x; u < units; u += blockDim.x) {
    const int r = u / L.nb, b = u % L.nb;
    const float* xr = x + (size_t)r * ldx + b * 32;
    float v[32];
    float amax = 0.0f;
#pragma unroll
    for (int i = 0; i < 32; ++i) {
      v[i] = xr[i];
      amax = fmaxf(amax, fabsf(v[i]));
    }
    const float d = amax / 127.0f;
    const float id = d != 0.0f ? 1.0f / d : 0.0f;
    int8_t* q = L.q + (size_t)r * L.n_in + b * 32;
    int sum = 0;
#pragma unroll
    for (int i = 0; i < 32; ++i) {
      const int qi = (int)roundf(v[i] * id);
      q[i] = (int8_t)qi;
      sum += qi;
    }
    L.s[u] = sum;
    L.d[u] = (float)(_Float16)d;  // the f16 d of block_q8_0
  }
}

// Q8_0 / Q5_0 (row-major planes, no row padding): lane l = output row l >> 1,
// half h = l & 1 of each block.
template <int FMT, int RB, int NW, int NM>
__device__ void dots_q32(const GemvArgs& a, int tile, int rows, const ActLds<RB>& L) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int h = lane & 1;
  const int row = min(tile * 32 + (lane >> 1), a.n_out - 1);
  const int nb = a.n_in / 32;
  for (int b = w; b < nb; b += NW) {
#pragma unroll
    for (int m = 0; m < NM; ++m) {
      const uint8_t* p0 = m ? a.u0 : a.p0;
      const uint8_t* p1 = m ? a.u1 : a.p1;
      const uint8_t* p2 = m ? a.u2 : a.p2;
      uint32_t v[4];
      float dw;
      if constexpr (FMT == FMT_Q8_0) {
        const uint4 q = *reinterpret_cast<const uint4*>(p0 + (size_t)row * a.n_in + 32 * b + 16 * h);
        v[0] = q.x;
        v[1] = q.y;
        v[2] = q.z;
        v[3] = q.w;
        dw = f16_to_f32(reinterpret_cast<const uint16_t*>(p1)[(size_t)row * nb + b]);
      } else {
        // bytes 8h..8h+7 of the block's 16: low nibbles are weights 8h + i,
        // high nibbles weights 16 + 8h + i; qh bit j is weight j's fifth bit
        const u2v q = *reinterpret_cast<const u2v*>(p0 + (size_t)row * (a.n_in / 2) + 16 * b + 8 * h);
        const uint32_t qh = reinterpret_cast<const uint32_t*>(p1)[(size_t)row * nb + b];
        auto spread = [](uint32_t bits4) {  // 4 bits -> bit 4 of 4 bytes
          return ((bits4 & 1u) | ((bits4 & 2u) << 7) | ((bits4 & 4u) << 14) | ((bits4 & 8u) << 21)) << 4;
        };
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const uint32_t wd = i ? q.y : q.x;
          const int j0 = 8 * h + 4 * i;
          v[i] = (wd & 0x0F0F0F0Fu) | spread((qh >> j0) & 15u);
          v[2 + i] = ((wd >> 4) & 0x0F0F0F0Fu) | spread((qh >> (16 + j0)) & 15u);
        }
        dw = f16_to_f32(reinterpret_cast<const uint16_t*>(p2)[(size_t)row * nb + b]);
      }
#pragma unroll
      for (int r = 0; r < RB; ++r) {
        if (r >= rows) break;
        const int8_t* xq = L.q + (size_t)r * L.n_in + 32 * b;
        int sumi = 0;
        if constexpr (FMT == FMT_Q8_0) {
          const uint4 xv = *reinterpret_cast<const uint4*>(xq + 16 * h);
          sumi = dot4(v[0], xv.x, sumi);
          sumi = dot4(v[1], xv.y, sumi);
          sumi = dot4(v[2], xv.z, sumi);
          sumi = dot4(v[3], xv.w, sumi);
          sumi += __shfl_xor(sumi, 1, 64);
        } else {
          const u2v xl = *reinterpret_cast<const u2v*>(xq + 8 * h);
          const u2v xh = *reinterpret_cast<const u2v*>(xq + 16 + 8 * h);
          sumi = dot4(v[0], xl.x, sumi);
          sumi = dot4(v[1], xl.y, sumi);
          sumi = dot4(v[2], xh.x, sumi);
          sumi = dot4(v[3], xh.y, sumi);
          sumi += __shfl_xor(sumi, 1, 64);
          sumi -= 16 * L.s[r * L.nb + b];
        }
        if (h == 0) L.term(m, r, b, lane >> 1) = (float)sumi * dw * L.d[r * L.nb + b];
      }
    }
  }
}

// Touch one dword of every 128-byte line of [base, base + bytes) across the
// workgroup: the tile's weights are on their way into the cache while the
// activations are quantized (the loads' values only feed `sink`).
__device__ inline void touch(const uint8_t* base, size_t bytes, int nthreads, uint32_t& sink) {
  for (size_t off = (size_t)threadIdx.x * 128; off + 4 <= bytes; off += (size_t)nthreads * 128)
    sink ^= *reinterpret_cast<const uint32_t*>(base + off);
}

template <int FMT>
__device__ inline void prefetch_tile(const GemvArgs& a, bool second, int tile, int nthreads, uint32_t& sink) {
  const uint8_t* p0 = second ? a.u0 : a.p0;
  const uint8_t* p1 = second ? a.u1 : a.p1;
  const uint8_t* p2 = second ? a.u2 : a.p2;
  // row-major planes: the tile's rows
  const size_t r0 = (size_t)tile * 32, nr = (size_t)min(32, a.n_out - tile * 32), nb = (size_t)(a.n_in / 32);
  if constexpr (FMT == FMT_Q8_0) {
    touch(p0 + r0 * a.n_in, nr * a.n_in, nthreads, sink);
    touch(p1 + r0 * nb * 2, nr * nb * 2, nthreads, sink);
  } else {
    touch(p0 + r0 * (a.n_in / 2), nr * (a.n_in / 2), nthreads, sink);
    touch(p1 + r0 * nb * 4, nr * nb * 4, nthreads, sink);
    touch(p2 + r0 * nb * 2, nr * nb * 2, nthreads, sink);
  }
}

// One 32-row weight tile of a launch: block terms over the activations
// already quantized in L, then one lane per (row, output) adds them in block
// order (GGML's scalar sums) and applies the epilogue.
template <int FMT, int RB, int NW, int EPI>
__device__ void q8_tile(const GemvArgs& a, int tile, int rows, const ActLds<RB>& L) {
  constexpr int NM = EPI == EPI_SWIGLU ? 2 : 1;
  dots_q32<FMT, RB, NW, NM>(a, tile, rows, L);
  __syncthreads();
  for (int t = threadIdx.x; t < rows * 32; t += blockDim.x) {
    const int r = t >> 5, j = t & 31, n = tile * 32 + j;
    if (n >= a.n_out) continue;
    float v[NM];
#pragma unroll
    for (int m = 0; m < NM; ++m) {
      float sumf = 0.0f;
      for (int b = 0; b < L.nb; ++b) sumf += L.term(m, r, b, j);
      v[m] = sumf;
    }
    const size_t o = (size_t)r * a.ldy + n;
    if constexpr (EPI == EPI_STORE) a.y[o] = v[0];
    if constexpr (EPI == EPI_RES) a.y[o] = a.res[(size_t)r * a.ldres + n] + v[0];
    if constexpr (EPI == EPI_SWIGLU) a.y[o] = silu_f(v[0]) * v[NM - 1];
  }
}

// the prefetch loads' values are never used: a store no launch can reach keeps them
__device__ inline void keep(const GemvArgs& a, int rows, uint32_t sink) {
  if (rows < 0 && sink == 0x9e3779b9u) a.y[0] = 0.0f;
}

// Rows of 36 blocks or more prefetch: a wave of 8 then walks five or more. One
// row of 896 x 4864 Q8_0 17.3 -> 13.6 us and Q5_0 19.3 -> 15.5, 3584 x 3584 13.9
// -> 11.1 and 15.2 -> 13.0. Short of that it gives nothing (896 x 2048 Q8_0 7.2
// and 7.2, Q5_0 8.4 -> 9.1), and 8 rows too wide to share a launch pay it in
// each (4096 x 12288 Q8_0 251 -> 287).
__device__ inline bool prefetches(const GemvArgs& a) { return a.n_in / 32 >= 36; }

template <int FMT, int RB, int NW, int EPI>
__global__ __launch_bounds__(64 * NW) void q8_gemv_kernel(GemvArgs a, int rows) {
  extern __shared__ __attribute__((aligned(16))) char dsm[];
  // long rows: the tile's later blocks are in the cache by the time a wave
  // reaches them
  uint32_t sink = 0;
  if (NW == 8 && prefetches(a)) {
    prefetch_tile<FMT>(a, false, blockIdx.x, 64 * NW, sink);
    if constexpr (EPI == EPI_SWIGLU) prefetch_tile<FMT>(a, true, blockIdx.x, 64 * NW, sink);
  }
  const ActLds<RB> L(dsm, a.n_in);
  quantize_rows<RB>(reinterpret_cast<const float*>(a.x), a.ldx, rows, L);
  __syncthreads();
  q8_tile<FMT, RB, NW, EPI>(a, blockIdx.x, rows, L);
  keep(a, rows, sink);
}

// Two matrices of one input (the attention's stacked q|k and v, whose formats
// may differ) in one launch: both formats take the same
// activation type, quantized once per workgroup; workgroups [0, split) run
// tiles of a, the rest tiles of b. Every tile's arithmetic is that of its own
// single-matrix launch.
template <int FMT, int FMT2, int RB, int NW>
__global__ __launch_bounds__(64 * NW) void q8_pair_kernel(GemvArgs a, GemvArgs b, int split, int rows) {
  extern __shared__ __attribute__((aligned(16))) char dsm[];
  const bool first = (int)blockIdx.x < split;
  uint32_t sink = 0;
  if (NW == 8 && prefetches(a)) {
    if (first) prefetch_tile<FMT>(a, false, blockIdx.x, 64 * NW, sink);
    else prefetch_tile<FMT2>(b, false, blockIdx.x - split, 64 * NW, sink);
  }
  const ActLds<RB> L(dsm, a.n_in);
  quantize_rows<RB>(reinterpret_cast<const float*>(a.x), a.ldx, rows, L);
  __syncthreads();
  if (first) {
    q8_tile<FMT, RB, NW, EPI_STORE>(a, blockIdx.x, rows, L);
  } else {
    q8_tile<FMT2, RB, NW, EPI_STORE>(b, blockIdx.x - split, rows, L);
  }
  keep(a, rows, sink);
}

template <int FMT, int RB, int NW, int EPI>
void launch_q8(GemvArgs a, int nrows, hipStream_t s) {
  const size_t lds = ActLds<RB>::bytes(a.n_in, EPI == EPI_SWIGLU ? 2 : 1);
  PGD_CHECK(lds <= 160 * 1024, kErrShape, "activation rows too wide for the quantized-activation GEMV");
  if (lds > 64 * 1024) {
    static bool set = false;  // per kernel instance: the largest LDS it may be launched with
    if (!set) {
      PGD_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&q8_gemv_kernel<FMT, RB, NW, EPI>),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
      set = true;
    }
  }
  const int tiles = (a.n_out + 31) / 32;
  for (int r0 = 0; r0 < nrows; r0 += RB) {
    const int rows = min(RB, nrows - r0);
    hipLaunchKernelGGL((q8_gemv_kernel<FMT, RB, NW, EPI>), dim3(tiles), dim3(64 * NW), lds, s, a, rows);
    PGD_HIP(hipGetLastError());
    a.x = reinterpret_cast<const float*>(a.x) + (size_t)rows * a.ldx;
    a.y += (size_t)rows * a.ldy;
    if (a.res) a.res += (size_t)rows * a.ldres;
  }
}

// waves per workgroup from the K blocks of a row (the sums do not depend on
// it: every block's terms are added in block order by one lane): four walk at
// most five blocks each, from 20 blocks on eight
constexpr int kEightWaveBlocks = 20;

template <int FMT, int RB, int EPI>
void launch_waves(const GemvArgs& a, int nrows, hipStream_t s) {
  if (a.n_in / 32 < kEightWaveBlocks) return launch_q8<FMT, RB, 4, EPI>(a, nrows, s);
  launch_q8<FMT, RB, 8, EPI>(a, nrows, s);
}

// rows per launch: decode steps take 1..8; prefills 16 at a time (weights
// read once per 16 rows). Wide rows whose RB quantized rows do not fit the
// 160 KiB of LDS take fewer rows per launch (the per-row arithmetic does not
// depend on RB, so the results are the same).
template <int FMT, int EPI>
void launch_rows(const GemvArgs& a, int nrows, hipStream_t s) {
  const int nm = EPI == EPI_SWIGLU ? 2 : 1;
  const size_t cap = 160 * 1024;
  if (nrows > 8 && ActLds<16>::bytes(a.n_in, nm) <= cap) return launch_waves<FMT, 16, EPI>(a, nrows, s);
  if (nrows > 4 && ActLds<8>::bytes(a.n_in, nm) <= cap) return launch_waves<FMT, 8, EPI>(a, nrows, s);
  if (nrows > 1 && ActLds<4>::bytes(a.n_in, nm) <= cap) return launch_waves<FMT, 4, EPI>(a, nrows, s);
  launch_waves<FMT, 1, EPI>(a, nrows, s);
}

// The most rows a Q4_K / Q6_K launch runs in gemv_q8k.hip.
constexpr int kFewRows = 6;

// The widest rows Q4_K / Q6_K launches take, the same for every row count: one
// quantized row and the block terms of 32 outputs in 160 KiB.
bool k256_fits(int fmt, int nsb, int nm) {
  const size_t act = ((size_t)nsb * (256 + 4 + 64) + 15) & ~(size_t)15;
  return act + (size_t)nm * nsb * 32 * (fmt == FMT_Q4K ? 9 : 8) * 4 <= 160 * 1024;
}

template <int EPI>
void dispatch(int fmt, const GemvArgs& a, int nrows, hipStream_t s) {
  switch (fmt) {
    case FMT_Q4K:
    case FMT_Q6K:
      PGD_CHECK(k256_fits(fmt, a.nsb, EPI == EPI_SWIGLU ? 2 : 1), kErrShape,
                "activation rows too wide for the quantized-activation GEMV");
      if (a.nw || q8act_few_rows(fmt, (a.n_out + 15) / 16, a.nsb, nrows, EPI == EPI_SWIGLU ? 2 : 1))
        return run_q8k_gemv(fmt, a, nrows, EPI, s);
      return run_q8_gemm(fmt, a, nrows, EPI, s);
    case FMT_Q8_0: return launch_rows<FMT_Q8_0, EPI>(a, nrows, s);
    case FMT_Q5_0: return launch_rows<FMT_Q5_0, EPI>(a, nrows, s);
  }
  throw Error{kErrFormat, "quantized-activation GEMV takes Q4_K, Q6_K, Q8_0 or Q5_0 matrices"};
}

template <int FMT, int FMT2, int RB, int NW>
void launch_pair_q8(GemvArgs a, GemvArgs b, int nrows, hipStream_t s) {
  const size_t lds = ActLds<RB>::bytes(a.n_in, 1);
  PGD_CHECK(lds <= 160 * 1024, kErrShape, "activation rows too wide for the quantized-activation GEMV");
  if (lds > 64 * 1024) {
    static bool set = false;
    if (!set) {
      PGD_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&q8_pair_kernel<FMT, FMT2, RB, NW>),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
      set = true;
    }
  }
  const int ta = (a.n_out + 31) / 32, tb = (b.n_out + 31) / 32;
  for (int r0 = 0; r0 < nrows; r0 += RB) {
    const int rows = min(RB, nrows - r0);
    hipLaunchKernelGGL((q8_pair_kernel<FMT, FMT2, RB, NW>), dim3(ta + tb), dim3(64 * NW), lds, s, a, b, ta, rows);
    PGD_HIP(hipGetLastError());
    a.x = reinterpret_cast<const float*>(a.x) + (size_t)rows * a.ldx;
    a.y += (size_t)rows * a.ldy;
    b.y += (size_t)rows * b.ldy;
  }
}

// the waves and rows per launch of launch_waves / launch_rows (shared by both
// matrices: they have the same K)
template <int FMT, int FMT2>
void pair_rows(const GemvArgs& a, const GemvArgs& b, int nrows, hipStream_t s) {
  auto go = [&](auto rb) {
    constexpr int RB = decltype(rb)::value;
    if (a.n_in / 32 < kEightWaveBlocks) return launch_pair_q8<FMT, FMT2, RB, 4>(a, b, nrows, s);
    launch_pair_q8<FMT, FMT2, RB, 8>(a, b, nrows, s);
  };
  const size_t cap = 160 * 1024;
  if (nrows > 8 && ActLds<16>::bytes(a.n_in, 1) <= cap) return go(std::integral_constant<int, 16>{});
  if (nrows > 4 && ActLds<8>::bytes(a.n_in, 1) <= cap) return go(std::integral_constant<int, 8>{});
  if (nrows > 1 && ActLds<4>::bytes(a.n_in, 1) <= cap) return go(std::integral_constant<int, 4>{});
  go(std::integral_constant<int, 1>{});
}

}  // namespace

bool q8act_pair_ok(int fmt_a, int fmt_b) {
  auto k256 = [](int f) { return f == FMT_Q4K || f == FMT_Q6K; };
  auto b32 = [](int f) { return f == FMT_Q8_0 || f == FMT_Q5_0; };
  return (k256(fmt_a) && k256(fmt_b)) || (b32(fmt_a) && b32(fmt_b));
}

// Same bits either way; the estimates of both say which is faster. us, few-row
// kernel / matrix cores: 5120 x 5120 Q4_K 2 rows 13.8 / 20.9, 4 rows 26.1 / 20.9
// (two workgroups no longer fit a CU's LDS); 3840 x 5120 6 rows 18.9 / 21.0;
// 2048 x 11008 2 rows 14.4 / 38.1, 5 rows 48.4 / 38.2 (rows one at a time);
// 18944 x 3584 2 rows 29.8 / 21.1; 4864 x 896 4 rows 7.6 / 8.8.
bool q8act_few_rows(int fmt, int tiles16, int nsb, int nrows, int nm, double slack) {
  if (nrows <= 1) return true;
  return nrows <= kFewRows && q8k_us(fmt, tiles16, nsb, nrows, nm) <= q8_gemm_us(fmt, nm * tiles16, nsb) + slack;
}

// An RMSNorm launch of one 896-wide row takes 6.0 us, of which the GEMV launch
// repeats about 4.5 (q|k + v 5.2 -> 9.5 us, gate/up 7.5 -> 12.8 us with the
// norm inside); a decode step of the 0.5B model 1271 -> 1139 us. So the fused
// launch may be slower than the matrix cores by 2.7: gate/up 4864 x 896 4 rows
// 15.0 us against 16.1 with a norm launch, 5 rows 17.6 against 16.1.
bool q8act_norm_fused(int fmt, int tiles16, int nsb, int n_in, int nrows, int nm) {
  return (fmt == FMT_Q4K || fmt == FMT_Q6K) && k256_fits(fmt, nsb, nm) &&
         q8act_few_rows(fmt, tiles16, nsb, nrows, nm, 2.7) && q8k_norm_ok(tiles16, nsb, n_in, nrows, nm);
}

void run_q8act_pair(int fmt_a, const GemvArgs& a, int fmt_b, const GemvArgs& b, int nrows, hipStream_t s) {
  PGD_CHECK(a.n_in == b.n_in, kErrShape, "paired GEMVs need one input width");
  PGD_CHECK(q8act_pair_ok(fmt_a, fmt_b), kErrFormat, "paired GEMVs need one activation type");
  if (fmt_a == FMT_Q4K || fmt_a == FMT_Q6K) {
    PGD_CHECK(k256_fits(fmt_a, a.nsb, 1) && k256_fits(fmt_b, b.nsb, 1), kErrShape,
              "activation rows too wide for the quantized-activation GEMV");
    if (a.nw || q8act_few_rows(fmt_a, (a.n_out + 15) / 16 + (b.n_out + 15) / 16, a.nsb, nrows, 1))
      return run_q8k_gemv_pair(fmt_a, a, fmt_b, b, nrows, s);
    return run_q8_gemm_pair(fmt_a, a, fmt_b, b, nrows, s);
  }
#define PGD_PAIR(F1, F2) \
  if (fmt_a == F1 && fmt_b == F2) return pair_rows<F1, F2>(a, b, nrows, s);
  PGD_PAIR(FMT_Q8_0, FMT_Q8_0)
  PGD_PAIR(FMT_Q8_0, FMT_Q5_0)
  PGD_PAIR(FMT_Q5_0, FMT_Q8_0)
  PGD_PAIR(FMT_Q5_0, FMT_Q5_0)
#undef PGD_PAIR
}

void run_q8act(int fmt, const GemvArgs& a, int nrows, int epi, hipStream_t s) {
  if (epi == EPI_SWIGLU) dispatch<EPI_SWIGLU>(fmt, a, nrows, s);
  else if (epi == EPI_RES) dispatch<EPI_RES>(fmt, a, nrows, s);
  else dispatch<EPI_STORE>(fmt, a, nrows, s);
}

}  // namespace gemv
}  // namespace pgd
