// gemm_a8.hip — MLX affine-8 (group 64) GEMM for prefill: batches of >= 256
// activation rows, every weight byte read once per 64 rows.
//
// Same per-group products as the GEMV kernels (gemv_mma.hip): with the
// prepared activations (xh + xl f16 operands, a8_act.h) and codes as the f16
// 1024 + c,
//   P[b, n] = -1024 XSP[b, g] + sum_k (1024 + c[n, k]) (xh + xl)[b, k]   4 x v_mfma_f32_16x16x32_f16
//   Y[b, n] += s[n, g] P[b, n] + bias[n, g] XS[b, g]
// but the groups of a row are summed in order 0..G-1 by one wave (no split-K,
// no partial sums in memory).
//
// Tiling: a workgroup of 4 waves computes 64 NS weight rows (NS 16-row
// subtiles per wave, 4 or 3; the SwiGLU pair: half gate, half up) x 64 batch
// rows (2 activation chunks): 4 x 4 accumulators of 16 x 16 per wave. Per group
// it stages in LDS the codes (16 KiB), scale/bias (1 KiB), operands (16 KiB)
// and constants (1 KiB) by direct global->LDS loads, two stages deep: group
// g + 1 loads while g computes. Two such workgroups share a CU, so that one
// reads LDS, folds or waits at its barrier while the other feeds the matrix
// cores (one workgroup of 8 waves on 128 rows went through those phases in
// step). A batch tile's products are folded into Y under the next one's MFMAs.
//
// Bound: matrix cores, four MFMAs per useful 16 x 16 x 64 (hi and lo operands).
// Measured at 2048 rows against the 8-wave form on the same card: gate/up 2 x
// 17408 x 5120 1761 -> 1537 us (475 TFLOP/s useful, 950 issued; a large f16
// library product reaches 1250), down 5120 x 17408 1148 -> 890 us, 12352 x 5120
// 697 -> 593 us. One constant instead of two (the bias on XSP) was 5% faster
// and 4% further from float64.
//
// Workgroups are numbered so that one XCD works on 8 batch blocks x 8 weight
// blocks at a time: both operands are re-read from its L2 (all batch blocks of
// a weight block first: gate/up 5% slower).
#include "a8_act.h"
#include "common.h"
#include "gemv_impl.h"
#include "quant.h"

namespace pgd {
namespace gemv {

namespace {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void lds_void;
typedef __attribute__((address_space(1))) void glb_void;

constexpr int kGW = 4;            // waves per workgroup
constexpr int kBC = 2;            // batch chunks (32 rows) per workgroup
constexpr int kStX = kBC * 8192;  // operands per stage
constexpr int kStC = kBC * 512;   // constants per stage
// NS: 16-row weight subtiles per wave
template <int NS>
struct Stage {
  static constexpr int WT = 2 * NS;                             // weight tiles (32 rows) per workgroup
  static constexpr int W = WT * 2048;                           // codes
  static constexpr int S = (WT * 128 + 1023) / 1024 * 1024;     // scale/bias
  static constexpr int BYTES = W + S + kStX + kStC;
  static constexpr int LOADS = BYTES / 1024;                    // 1 KiB wave loads
  static_assert(BYTES % 1024 == 0 && 2 * BYTES <= 80 * 1024, "two workgroups of two stages per CU");
};

__device__ __forceinline__ void dma16(const void* g, void* l) {
  __builtin_amdgcn_global_load_lds((glb_void*)g, (lds_void*)l, 16, 0, 0);
}

// v plus lane ^ 1's v
__device__ inline f4 add_neighbour(f4 v) {
  f4 r;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float e = v[i];  // (a bit cast of the element itself reads element 0)
    r[i] = e + __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, e), 0xB1, 0xF, 0xF, true));
  }
  return r;
}

__device__ inline h8 codes8(uint32_t w0, uint32_t w1) {
  const uint32_t c0 = __builtin_amdgcn_perm(0x64646464u, w0, 0x04010400u);
  const uint32_t c1 = __builtin_amdgcn_perm(0x64646464u, w0, 0x04030402u);
  const uint32_t c2 = __builtin_amdgcn_perm(0x64646464u, w1, 0x04010400u);
  const uint32_t c3 = __builtin_amdgcn_perm(0x64646464u, w1, 0x04030402u);
  return __builtin_bit_cast(h8, make_uint4(c0, c1, c2, c3));
}

// global source of wave load j of group g for this lane: the stage is [codes:
// tile t, 2 KiB] [sb: tile t, 128 B] [operands: chunk c, bt, 4 KiB]
// [constants: chunk c, bt, 256 B]; the SwiGLU pair's first NS tiles are the
// gate's, the others the up matrix's
template <bool DUAL, int NS>
__device__ inline const void* load_src(const GemvArgs& a, const uint4* XA, const float* CA, int wblk, int cblk, int G,
                                       int ntiles, int nchunks, int j, int lane) {
  constexpr int WT = Stage<NS>::WT;
  auto tile = [&](int t) { return min(DUAL ? wblk * NS + t % NS : wblk * WT + t, ntiles - 1); };
  if (j < WT * 2) {  // codes: tile j / 2, half j % 2
    const int t = j >> 1;
    return (DUAL && t >= NS ? a.u0 : a.p0) + (((size_t)tile(t) * G) << 11) + (j & 1) * 1024 + lane * 16;
  }
  j -= WT * 2;
  if (j < Stage<NS>::S / 1024) {  // scale/bias: tile j 8 + lane / 8, 16 B (l % 8); past the last into the padding
    const int t = min(j * 8 + (lane >> 3), WT - 1);
    return (DUAL && t >= NS ? a.u1 : a.p1) + (((size_t)tile(t) * G) << 7) + (lane & 7) * 16;
  }
  j -= Stage<NS>::S / 1024;
  if (j < kBC * 8) {  // operands: chunk j / 8, tile (j / 4) % 2, operand j % 4
    const int c = min(cblk * kBC + (j >> 3), nchunks - 1), bt = (j >> 2) & 1, i = j & 3;
    const size_t item = (size_t)c * G * 2 + bt;
    return XA + item * 256 + i * 64 + lane;
  }
  // constants: lane l -> item (chunk, bt) = l / 16
  const int it = lane >> 4;
  const int c = min(cblk * kBC + (it >> 1), nchunks - 1), bt = it & 1;
  const size_t item = (size_t)c * G * 2 + bt;
  return CA + item * 64 + (lane & 15) * 4;
}

template <int EPI, int NS>
__global__ __launch_bounds__(64 * kGW, 2) void a8_gemm_kernel(GemvArgs a, const uint4* __restrict__ XA,
                                                              const float* __restrict__ CA, int rows, int nwblk,
                                                              int ncblk, int per_xcd) {
  constexpr bool DUAL = EPI == EPI_SWIGLU;
  using St = Stage<NS>;
  static_assert(!DUAL || NS % 2 == 0, "a wave's subtiles are gate and up halves");
  extern __shared__ __attribute__((aligned(16))) char smem[];
  // XCD-aware numbering: workgroups are dealt to the 8 XCDs in turn; XCD x
  // takes the contiguous range [x per_xcd, (x + 1) per_xcd) of pairs: batch
  // blocks in groups of 8, in a group weight block by weight block
  const int id = blockIdx.x, xcd = id & 7;
  const int gi = xcd * per_xcd + (id >> 3);
  if (gi >= nwblk * ncblk || (id >> 3) >= per_xcd) return;
  const int c0 = gi / (8 * nwblk) * 8, cw = min(8, ncblk - c0), in_group = gi - c0 * nwblk;
  const int wblk = in_group / cw, cblk = c0 + in_group % cw;
  const int G = a.n_in / 64;
  const int ntiles = (a.n_out + 31) / 32, nchunks = (rows + 31) / 32;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int j16 = lane & 15, q = lane >> 4;

  // this wave's loads: j = wave + 4 k; sources of group 0 and the per-group
  // stride of each (codes 2 KiB, scale/bias 128 B, operands 8 KiB, constants
  // 512 B). A wave with fewer repeats the stage's last load: same bytes to the
  // same place.
  constexpr int NK = (St::LOADS + kGW - 1) / kGW;
  const char* src[NK];
  uint32_t step[NK];
#pragma unroll
  for (int k = 0; k < NK; ++k) {
    const int j = min(wave + k * kGW, St::LOADS - 1);
    src[k] = static_cast<const char*>(load_src<DUAL, NS>(a, XA, CA, wblk, cblk, G, ntiles, nchunks, j, lane));
    step[k] = j < St::WT * 2 ? 2048u : j < (St::W + St::S) / 1024 ? 128u : j < (St::W + St::S + kStX) / 1024 ? 8192u : 512u;
  }
  auto issue = [&](int g, int stage) {
    char* base = smem + stage * St::BYTES;
#pragma unroll
    for (int k = 0; k < NK; ++k) {
      const int j = min(wave + k * kGW, St::LOADS - 1);
      dma16(src[k] + (size_t)g * step[k], base + j * 1024);
    }
  };
  // stage tile and row half of the wave's subtile st: NS consecutive ones, or
  // NS / 2 of the gate and the same of up
  auto sub_of = [&](int st) { return DUAL ? (st % (NS / 2)) + wave * (NS / 2) + (st >= NS / 2 ? 2 * NS : 0) : wave * NS + st; };

  f4 Y[NS][4];  // [subtile][batch tile]
#pragma unroll
  for (int st = 0; st < NS; ++st)
#pragma unroll
    for (int bt = 0; bt < 4; ++bt) Y[st][bt] = (f4){0.f, 0.f, 0.f, 0.f};

  const uint32_t woff = (q >> 1) * 1024 + j16 * 32 + (q & 1) * 16;
  // Two stages: group g + 1 loads while g computes. All of a group's LDS reads
  // come first, before the next group's direct-to-LDS loads are issued: the
  // compiler would wait for loads in flight before any LDS read after them.
  const char* w_lane = smem + woff;
  const char* s_lane = smem + St::W + j16 * 4;
  const char* x_lane = smem + St::W + St::S + lane * 16;
  // constants of the lane's 4 rows: even lanes read -1024 XSP and XS of
  // quarters 0-1, odd lanes of quarters 2-3, and neighbours add (half the LDS
  // reads of every lane reading both)
  const char* c_lane = smem + St::W + St::S + kStX + q * 16 + (j16 & 1) * 64;
  // products of the batch tile before the current one, folded into Y under the
  // current one's MFMAs
  f4 P[NS], xs = {0.f, 0.f, 0.f, 0.f};
  float S[NS], Bi[NS];
#pragma unroll
  for (int st = 0; st < NS; ++st) {
    P[st] = xs;
    S[st] = Bi[st] = 0.f;
  }
  auto fold = [&](int bt) {
#pragma unroll
    for (int st = 0; st < NS; ++st)
#pragma unroll
      for (int rr = 0; rr < 4; ++rr) Y[st][bt][rr] = fmaf(Bi[st], xs[rr], fmaf(S[st], P[st][rr], Y[st][bt][rr]));
  };
  issue(0, 0);
  for (int g = 0; g < G; ++g) {
    // group g landed, and every wave is done with the other stage
    __builtin_amdgcn_s_waitcnt(0 | (7 << 4) | (15 << 8));  // vmcnt(0)
    __builtin_amdgcn_s_barrier();
    const int so = (g & 1) * St::BYTES;
    // codes of the subtiles and their scale/bias, and the 4 batch tiles'
    // operands and constants
    uint4 W[NS], XR[4][4];
    uint32_t SV[NS];
    f4 C[4][2];
#pragma unroll
    for (int st = 0; st < NS; ++st) {
      const int u = sub_of(st);
      W[st] = *reinterpret_cast<const uint4*>(w_lane + so + (u >> 1) * 2048 + (u & 1) * 512);
      SV[st] = *reinterpret_cast<const uint32_t*>(s_lane + so + u * 64);
    }
    auto read_x = [&](int bt) {
#pragma unroll
      for (int i = 0; i < 4; ++i) XR[bt][i] = *reinterpret_cast<const uint4*>(x_lane + so + bt * 4096 + i * 1024);
#pragma unroll
      for (int i = 0; i < 2; ++i) C[bt][i] = *reinterpret_cast<const f4*>(c_lane + so + bt * 256 + i * 128);
    };
    read_x(0);
    read_x(1);
    // the last batch tile of the group before, while these reads arrive
    fold(3);
    h8 B0[NS], B1[NS];
#pragma unroll
    for (int st = 0; st < NS; ++st) {
      B0[st] = codes8(W[st].x, W[st].y);
      B1[st] = codes8(W[st].z, W[st].w);
      S[st] = bf16_to_f32(SV[st] & 0xffffu);
      Bi[st] = bf16_to_f32(SV[st] >> 16);
    }
#pragma unroll
    for (int bt = 0; bt < 4; ++bt) {
      if (bt < 2) read_x(bt + 2);
      if (bt == 1) issue(min(g + 1, G - 1), (g + 1) & 1);
      f4 N[NS];
      const f4 cn = add_neighbour(C[bt][0]), xn = add_neighbour(C[bt][1]);  // -1024 XSP, XS
#pragma unroll
      for (int st = 0; st < NS; ++st)
        N[st] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8, XR[bt][0]), B0[st], cn, 0, 0, 0);
#pragma unroll
      for (int st = 0; st < NS; ++st)
        N[st] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8, XR[bt][1]), B1[st], N[st], 0, 0, 0);
#pragma unroll
      for (int st = 0; st < NS; ++st)
        N[st] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8, XR[bt][2]), B0[st], N[st], 0, 0, 0);
#pragma unroll
      for (int st = 0; st < NS; ++st)
        N[st] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8, XR[bt][3]), B1[st], N[st], 0, 0, 0);
      if (bt > 0) fold(bt - 1);
#pragma unroll
      for (int st = 0; st < NS; ++st) P[st] = N[st];
      xs = xn;
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  fold(3);
  __builtin_amdgcn_s_waitcnt(0);  // the re-read loads of the last iterations

  // deferred RMSNorm of the input: 1/rms of each batch row
  if (a.inv) {
#pragma unroll
    for (int bt = 0; bt < 4; ++bt) {
      const int b = (cblk * kBC + (bt >> 1)) * 32 + 16 * (bt & 1) + 4 * q;
#pragma unroll
      for (int rr = 0; rr < 4; ++rr) {
        const float f = b + rr < rows ? a.inv[b + rr] : 1.0f;
#pragma unroll
        for (int st = 0; st < NS; ++st) Y[st][bt][rr] *= f;
      }
    }
  }
  // epilogue: lane (j16, q) holds weight row 16 h + j16 of its subtiles and
  // batch rows 16 bh + 4 q + rr of each batch tile
#pragma unroll
  for (int bt = 0; bt < 4; ++bt) {
    const int c = cblk * kBC + (bt >> 1);
#pragma unroll
    for (int rr = 0; rr < 4; ++rr) {
      const int b = c * 32 + 16 * (bt & 1) + 4 * q + rr;
      if (b >= rows) continue;
#pragma unroll
      for (int st = 0; st < (DUAL ? NS / 2 : NS); ++st) {
        const int n = (wblk * (DUAL ? 2 * NS : 4 * NS) + sub_of(st)) * 16 + j16;
        if (n >= a.n_out) continue;
        const size_t o = (size_t)b * a.ldy + n;
        if constexpr (DUAL) a.y[o] = silu_f(Y[st][bt][rr]) * Y[NS / 2 + st][bt][rr];
        else if constexpr (EPI == EPI_RES) a.y[o] = a.res[(size_t)b * a.ldres + n] + Y[st][bt][rr];
        else a.y[o] = Y[st][bt][rr];
      }
    }
  }
}

// 1/rms of each row from its partial sums of squares, one wave per row: once
// per launch, not by every workgroup for its rows (64 dependent reductions in
// the epilogue of each: gate/up at 1266 rows 1227 -> 951 us).
__global__ __launch_bounds__(256) void a8_inv_kernel(const float* __restrict__ rss, int nh, int n, float eps, int rows,
                                                     float* __restrict__ inv) {
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;
  const float f = rss_inv(rss + (size_t)row * nh, nh, n, eps);
  if ((threadIdx.x & 63) == 0) inv[row] = f;
}

int wblocks(int n_out, int ns, int epi) {
  const int subs = (n_out + 15) / 16, per = epi == EPI_SWIGLU ? 2 * ns : 4 * ns;
  return (subs + per - 1) / per;
}
int cblocks(int rows) { return ((rows + 31) / 32 + kBC - 1) / kBC; }

// Weight subtiles per wave: 4, or 3 where that fills the last round of the
// chip's 2 x 256 workgroups better. A round costs its NS subtiles (a subtile of
// 3 about 1.13 of one of 4, whose operands serve more products), a last round
// of at most one workgroup per CU about 0.6 of a full one. 5120 x 17408 at
// 1152 rows (360 or 486 workgroups) 3 is 7% faster; at 2048 rows
// (640 or 864) 4 is the better. 2 and 5 lost everywhere (5 spills).
int pick_ns(int n_out, int rows, int epi) {
  if (epi == EPI_SWIGLU) return 4;
  auto cost = [&](int ns) {
    const int wg = wblocks(n_out, ns, epi) * cblocks(rows), rest = wg % 512;
    return (wg / 512 + (rest == 0 ? 0.0 : rest <= 256 ? 0.6 : 1.0)) * ns * (ns == 3 ? 1.13 : 1.0);
  };
  return cost(3) < cost(4) ? 3 : 4;
}

template <int EPI, int NS>
void launch_gemm(const GemvArgs& a, const uint4* XA, const float* CA, int rows, hipStream_t s) {
  const int nwblk = wblocks(a.n_out, NS, EPI), ncblk = cblocks(rows);
  const int total = nwblk * ncblk, per_xcd = (total + 7) / 8;
  constexpr int lds = 2 * Stage<NS>::BYTES;
  static const bool ok = [] {
    PGD_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(a8_gemm_kernel<EPI, NS>),
                                hipFuncAttributeMaxDynamicSharedMemorySize, lds));
    return true;
  }();
  (void)ok;
  hipLaunchKernelGGL((a8_gemm_kernel<EPI, NS>), dim3(8 * per_xcd), dim3(64 * kGW), lds, s, a, XA, CA, rows, nwblk,
                     ncblk, per_xcd);
  PGD_HIP(hipGetLastError());
}

template <int EPI>
void launch_ns(const GemvArgs& a, const uint4* XA, const float* CA, int rows, hipStream_t s) {
  if constexpr (EPI != EPI_SWIGLU)
    if (pick_ns(a.n_out, rows, EPI) == 3) return launch_gemm<EPI, 3>(a, XA, CA, rows, s);
  launch_gemm<EPI, 4>(a, XA, CA, rows, s);
}

}  // namespace

int a8_gemm_workgroups(int n_out, int rows, int epi) {
  return wblocks(n_out, pick_ns(n_out, rows, epi), epi) * cblocks(rows);
}

// Microseconds of the GEMM, to compare with the GEMV kernels: a round of 512
// workgroups takes 33 ns per weight column with four subtiles per wave and 28
// with three, one of at most 256 half of that (0.42 behind whole rounds), in
// between linear. Measured within 10% for 4096..17408 columns and 256..2048
// rows of 2048..17408 outputs and SwiGLU pairs.
double a8_gemm_us(int n_out, int n_in, int rows, int epi) {
  const int ns = pick_ns(n_out, rows, epi), wg = wblocks(n_out, ns, epi) * cblocks(rows);
  const int whole = wg / 512, rest = wg % 512;
  const double round = ns == 4 ? 1.0 : 0.85;
  const double part = rest == 0 ? 0.0 : rest > 256 ? (0.57 + 0.43 * (rest - 256) / 256) * round : whole ? 0.42 : 0.5;
  return 5.0 + 0.0332 * n_in * (whole * round + part);
}

void run_a8_gemm(GemvArgs a, const uint4* XA, const float* CA, int rows, int epi, hipStream_t s) {
  PGD_CHECK(rows > 0 && (rows % 32 == 0 || rows % 32 > 4), kErrShape,
            "the A8 GEMM takes activation chunks in the full (not compact) layout");
  PGD_CHECK(a.n_in % 64 == 0, kErrShape, "A8 GEMM width");
  a.inv = nullptr;
  if (a.rss) {
    a.inv = static_cast<float*>(gemv_scratch(s, (size_t)rows * sizeof(float), 5));
    hipLaunchKernelGGL(a8_inv_kernel, dim3((rows + 3) / 4), dim3(256), 0, s, a.rss, a.rss_nh, a.rss_n, a.rss_eps, rows,
                       a.inv);
    PGD_HIP(hipGetLastError());
  }
  if (epi == EPI_SWIGLU) launch_ns<EPI_SWIGLU>(a, XA, CA, rows, s);
  else if (epi == EPI_RES) launch_ns<EPI_RES>(a, XA, CA, rows, s);
  else launch_ns<EPI_STORE>(a, XA, CA, rows, s);
}

}  // namespace gemv
}  // namespace pgd
