// ops.hip — RMSNorm, causal conv step, Gated-DeltaNet recurrence, q/k/v
// preparation with paged KV writes and argmax (attention: attn.hip).
#include <climits>

#include "common.h"
#include "ops.h"
#include "gemv_impl.h"

namespace pgd {

namespace {

typedef float f4 __attribute__((ext_vector_type(4)));

// ---------------------------------------------------------------------------
// block reductions (256 threads = 4 waves)
// ---------------------------------------------------------------------------
__device__ inline float block_sum256(float v, float* red4) {
  v = wave_sum(v);
  const int w = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) red4[w] = v;
  __syncthreads();
  float t = red4[0] + red4[1] + red4[2] + red4[3];
  __syncthreads();
  return t;
}

// ---------------------------------------------------------------------------
// RMSNorm
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void rmsnorm_kernel(const float* __restrict__ x, int ldx, const int* rows_idx,
                                                      int n, const float* __restrict__ w, float eps, int mode,
                                                      float* __restrict__ y, int ldy) {
  __shared__ float red[4];
  const int r = blockIdx.x;
  const int src = rows_idx ? rows_idx[r] : r;
  const float* xr = x + (size_t)src * ldx;
  float ss = 0.0f;
  for (int i = threadIdx.x; i < n; i += 256) ss += xr[i] * xr[i];
  ss = block_sum256(ss, red);
  float* yr = y + (size_t)r * ldy;
  if (mode == 0) {
    float inv = 1.0f / sqrtf(ss / (float)n + eps);
    for (int i = threadIdx.x; i < n; i += 256) yr[i] = xr[i] * inv * w[i];
  } else {
    float m = sqrtf(ss / (float)n + eps);
    for (int i = threadIdx.x; i < n; i += 256) yr[i] = xr[i] / m * w[i];
  }
}

// candle's CPU rms_norm sums the squares left to right in f32; the same order
// makes the normed values (and so their Q8 quantization, where an embedding
// row's grid values can sit exactly on a rounding tie) agree bit for bit. The
// squares are formed in parallel (each rounds the same wherever it is
// computed) and staged in LDS, padded with zeros (s + 0 = s) to whole rounds
// of 64; one lane adds them in order, the LDS reads of 32 in flight under the
// additions of the 32 before, so the chain of n dependent additions is all
// that is left. Rows of up to 8 * 256 elements stay in registers. One row of
// 896: 7.7 -> 6.0 us (four values per LDS round trip before), about 3 us of it
// the chain.
__global__ __launch_bounds__(256) void rmsnorm_ordered_kernel(const float* __restrict__ x, int ldx, const int* rows_idx,
                                                              int n, const float* __restrict__ w, float eps,
                                                              float* __restrict__ y, int ldy) {
  __shared__ __attribute__((aligned(16))) float sq[8192 + 64];
  __shared__ float sum;
  const int r = blockIdx.x, tid = threadIdx.x;
  const float* xr = x + (size_t)(rows_idx ? rows_idx[r] : r) * ldx;
  const int np = (n + 63) & ~63;
  constexpr int KEEP = 8;
  float xv[KEEP], wv[KEEP];
#pragma unroll
  for (int k = 0; k < KEEP; ++k) {
    const int i = tid + k * 256;
    xv[k] = i < n ? xr[i] : 0.0f;
    wv[k] = i < n ? w[i] : 0.0f;
  }
#pragma unroll
  for (int k = 0; k < KEEP; ++k) {
    const int i = tid + k * 256;
    if (i < np) sq[i] = xv[k] * xv[k];
  }
  for (int i = tid + KEEP * 256; i < np; i += 256) {
    const float v = i < n ? xr[i] : 0.0f;
    sq[i] = v * v;
  }
  __syncthreads();
  if (tid == 0) {
    const f4* q = reinterpret_cast<const f4*>(sq);
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
      read(a, i + 16);  // past the last round: behind the pad, dropped
      add(b);
    }
    sum = ss;
  }
  __syncthreads();
  const float m = sqrtf(sum / (float)n + eps);
  float* yr = y + (size_t)r * ldy;
#pragma unroll
  for (int k = 0; k < KEEP; ++k) {
    const int i = tid + k * 256;
    if (i < n) yr[i] = xv[k] / m * wv[k];
  }
  for (int i = tid + KEEP * 256; i < n; i += 256) yr[i] = xr[i] / m * w[i];
}

// ---------------------------------------------------------------------------
// causal conv step (sequential over a sequence's rows)
// ---------------------------------------------------------------------------
// The output of row t reads inputs t-k+1..t only (earlier rows' inputs come
// from the state), so a sequence is cut into segments of kConvSeg rows along
// grid z; each thread runs one channel through one segment. Segment 0 alone
// reads the old state and alone writes the new one (the last k-1 inputs of
// old state ++ x), so no segment reads a state another has rewritten.
constexpr int kConvSeg = 64;

// KW: the conv kernel length (a compile-time constant, so the window lives in
// registers rather than in per-lane scratch memory)
template <int KW>
__global__ __launch_bounds__(256) void conv_step_kernel(const float* __restrict__ x, int ldx, float* __restrict__ out,
                                                        int ldo, int channels, const float* __restrict__ weight,
                                                        float* const* state_base, size_t state_off,
                                                        const int* row_start, const int* row_count) {
  constexpr int kernel = KW;
  const int c = blockIdx.x * 256 + threadIdx.x;
  const int s = blockIdx.y;
  if (c >= channels) return;
  const int r0 = row_start[s], n = row_count[s];
  const int t_beg = blockIdx.z * kConvSeg;
  if (t_beg >= n && (blockIdx.z > 0 || n > 0)) return;
  const int t_end = gridDim.z == 1 ? n : min(n, t_beg + kConvSeg);
  constexpr int hist = kernel - 1, HA = hist > 0 ? hist : 1;
  float* st = state_base[s] + state_off + (size_t)c * hist;
  float win[HA];
  float wt[kernel];
  float old[HA];
#pragma unroll
  for (int k = 0; k < hist; ++k) {
    // window before row t_beg: inputs t_beg-hist..t_beg-1, from the state before row 0
    const int t = t_beg - hist + k;
    win[k] = t < 0 ? st[hist + t] : x[(size_t)(r0 + t) * ldx + c];
  }
  const bool whole = gridDim.z == 1;  // this thread runs every row: the last window is the new state
  if (!whole)
#pragma unroll
    for (int k = 0; k < hist; ++k) old[k] = win[k];
#pragma unroll
  for (int k = 0; k < kernel; ++k) wt[k] = weight[(size_t)c * kernel + k];
  // inputs loaded eight rows ahead (the steps are sequential; the loads are not)
  constexpr int PF = 8;
  float xr[PF];
#pragma unroll
  for (int k = 0; k < PF; ++k) xr[k] = t_beg + k < t_end ? x[(size_t)(r0 + t_beg + k) * ldx + c] : 0.0f;
  for (int t = t_beg; t < t_end; ++t) {
    const float xv = xr[0];
#pragma unroll
    for (int k = 0; k + 1 < PF; ++k) xr[k] = xr[k + 1];
    xr[PF - 1] = t + PF < t_end ? x[(size_t)(r0 + t + PF) * ldx + c] : 0.0f;
    float acc = 0.0f;
#pragma unroll
    for (int k = 0; k < hist; ++k) acc += win[k] * wt[k];
    acc += xv * wt[hist];
    out[(size_t)(r0 + t) * ldo + c] = acc / (1.0f + expf(-acc));
#pragma unroll
    for (int k = 0; k + 1 < hist; ++k) win[k] = win[k + 1];
    if constexpr (hist > 0) win[hist - 1] = xv;
  }
  if (whole) {
#pragma unroll
    for (int k = 0; k < hist; ++k) st[k] = win[k];
    return;
  }
  if (blockIdx.z != 0) return;
#pragma unroll
  for (int k = 0; k < hist; ++k) {
    // new state: inputs n-hist..n-1 of old state ++ x (old[] picked with
    // compile-time indices, so it stays in registers)
    const int t = n - hist + k;
    float v = 0.0f;
    if (t < 0) {
#pragma unroll
      for (int jj = 0; jj < hist; ++jj)
        if (jj == hist + t) v = old[jj];
    } else {
      v = x[(size_t)(r0 + t) * ldx + c];
    }
    st[k] = v;
  }
}

// ---------------------------------------------------------------------------
// Gated-DeltaNet
// ---------------------------------------------------------------------------
// One workgroup per (value head, sequence) of 32 RG threads. Thread (rg, cg)
// holds state rows RPT rg .. RPT rg + RPT - 1 (RPT = 128 / RG), columns
// 4cg..4cg+3 in registers for the whole sequence chunk. Column sums over rows
// (S^T k, S^T q) are folded through LDS across the RG row groups, in order.
// RG = 16 (512 threads, 32 state registers each) measured ~3% faster than 8
// at 1..64 sequences and 32 much slower from 32 sequences on (16 waves per
// workgroup, one workgroup per compute unit).
__device__ inline float softplus_f(float x) {
  if (x > 20.0f) return x;
  if (x < -20.0f) return expf(x);
  return logf(1.0f + expf(x));
}

__device__ inline int gdn_chunks(int n) { return n < kGdnLongRows ? 0 : (n + kGdnChunk - 1) / kGdnChunk; }

// Chunks of the long sequences are numbered in sequence order. The number of
// sequence s's first one, or -1 when its chunks do not all fit below cap (a
// caller's rows bound was too small for its counts: gdn_kernel's then). Whole
// waves call it.
__device__ inline int gdn_chunk_base(const int* row_count, int s, int cap) {
  int base = 0;
  for (int j0 = 0; j0 < s; j0 += 64) {
    const int j = j0 + (threadIdx.x & 63);
    int c = j < s ? gdn_chunks(row_count[j]) : 0;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) c += __shfl_xor(c, o, 64);
    base += c;
  }
  return base + gdn_chunks(row_count[s]) <= cap ? base : -1;
}

constexpr int kGdnRowGroups = 16;

template <int RG>
__global__ __launch_bounds__(32 * RG) void gdn_kernel(GdnParams p, const int* row_start, const int* row_count) {
  constexpr int D = 128, RPT = D / RG;  // row groups, rows per thread
  __shared__ float qs[D], ks[D], delta[D];
  __shared__ float red[RG][D];
  __shared__ float part[4];
  __shared__ float obuf[D];
  const int h = blockIdx.x, s = blockIdx.y, tid = threadIdx.x;
  const int cg = tid & 31, rg = tid >> 5;
  const int repeat = p.v_heads / p.k_heads;
  const int kh = h / repeat;
  const int key_dim = p.k_heads * D;
  const int r0 = row_start[s], n = row_count[s];
  // the chunkwise kernels' (unless their scratch does not hold the sequence)
  if (p.o_raw && n >= kGdnLongRows && gdn_chunk_base(row_count, s, p.chunk_cap) >= 0) return;
  const int row_end = p.o_raw ? p.o_rows : INT_MAX;  // a prefill's rows past its bound are not written
  float* st = p.state_base[s] + p.state_off + (size_t)h * D * D;
  float S[RPT][4];
#pragma unroll
  for (int ii = 0; ii < RPT; ++ii) {
    float4 v = *reinterpret_cast<const float4*>(st + (size_t)(RPT * rg + ii) * D + 4 * cg);
    S[ii][0] = v.x;
    S[ii][1] = v.y;
    S[ii][2] = v.z;
    S[ii][3] = v.w;
  }
  const float a_log = p.a_log[h], dtb = p.dt_bias[h];
  const float qscale = sqrtf((float)D);
  // the gate input z and the norm weight are loaded with the step's other
  // inputs, not after the reductions that need them
  const float nw = tid < D ? p.norm[tid] : 0.0f;
  // a step's inputs (gate z, v, this thread's q or k element, the a / b gate
  // inputs) are loaded one step ahead, so a prefill's sequential steps do
  // not wait for memory each
  struct In {
    float zg, vv, v, ar, br;
  };
  auto load_in = [&](int row) {
    const float* cv = p.conv_out + (size_t)row * p.ld_conv;
    In x;
    x.zg = tid < D ? p.z[(size_t)row * p.ld_z + h * D + tid] : 0.0f;
    x.vv = tid < D ? cv[2 * key_dim + h * D + tid] : 0.0f;
    x.v = tid < D ? cv[kh * D + tid] : tid < 2 * D ? cv[key_dim + kh * D + (tid - D)] : 0.0f;
    x.ar = p.a[(size_t)row * p.ld_ab + h];
    x.br = p.b[(size_t)row * p.ld_ab + h];
    return x;
  };
  In nxt = load_in(r0);
  for (int t = 0; t < n; ++t) {
    const int row = r0 + t;
    const In cur = nxt;
    if (t + 1 < n) nxt = load_in(row + 1);
    const float zg = cur.zg, vv = cur.vv;
    // q (threads 0..127) and k (128..255), L2-normalized per head
    float v = cur.v;
    float ss = wave_sum(v * v);
    if ((tid & 63) == 0 && tid < 2 * D) part[tid >> 6] = ss;
    __syncthreads();
    if (tid < D) {
      float inv = 1.0f / sqrtf(part[0] + part[1] + 1e-6f);
      qs[tid] = (v * inv) / qscale;
    } else if (tid < 2 * D) {
      float inv = 1.0f / sqrtf(part[2] + part[3] + 1e-6f);
      ks[tid - D] = v * inv;
    }
    const float g = -expf(a_log) * softplus_f(cur.ar + dtb);
    const float decay = expf(g);
    const float beta = 1.0f / (1.0f + expf(-cur.br));
    __syncthreads();
    // S *= decay; mem = S^T k (partial over this thread's 16 rows)
    float m4[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int ii = 0; ii < RPT; ++ii) {
      const float kv = ks[RPT * rg + ii];
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        S[ii][c] = S[ii][c] * decay;
        m4[c] += S[ii][c] * kv;
      }
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) red[rg][4 * cg + c] = m4[c];
    __syncthreads();
    if (tid < D) {
      float mem = 0.0f;
#pragma unroll
      for (int q = 0; q < RG; ++q) mem += red[q][tid];
      delta[tid] = (vv - mem) * beta;
    }
    __syncthreads();
    // S += k delta^T ; o = S^T q (partial)
    float o4[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    float dl[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) dl[c] = delta[4 * cg + c];
#pragma unroll
    for (int ii = 0; ii < RPT; ++ii) {
      const float kv = ks[RPT * rg + ii], qv = qs[RPT * rg + ii];
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        S[ii][c] = S[ii][c] + kv * dl[c];
        o4[c] += S[ii][c] * qv;
      }
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) red[rg][4 * cg + c] = o4[c];
    __syncthreads();
    // gated RMSNorm over the head (qwen3_5.rs:1747-1756)
    float o = 0.0f;
    if (tid < D) {
#pragma unroll
      for (int q = 0; q < RG; ++q) o += red[q][tid];
    }
    float oss = wave_sum(tid < D ? o * o : 0.0f);
    if ((tid & 63) == 0) part[tid >> 6] = oss;
    __syncthreads();
    if (tid < D) {
      const float inv = 1.0f / sqrtf((part[0] + part[1]) / (float)D + 1e-6f);
      const float val = o * inv * nw * (zg / (1.0f + expf(-zg)));
      if (p.out && row < row_end) p.out[(size_t)row * p.ld_out + h * D + tid] = val;
      obuf[tid] = val;
    }
    __syncthreads();
    if (p.act.XA && tid < D / 16 && row < row_end) {
      // the head's 128 outputs are two whole groups of the out projection's input
      float v[16];
#pragma unroll
      for (int e = 0; e < 16; ++e) v[e] = obuf[16 * tid + e];
      a8act::emit_slice(p.act, row, (h * D + 16 * tid) >> 6, tid & 3, v, true);
    }
    __syncthreads();
  }
#pragma unroll
  for (int ii = 0; ii < RPT; ++ii)
    *reinterpret_cast<float4*>(st + (size_t)(RPT * rg + ii) * D + 4 * cg) = make_float4(S[ii][0], S[ii][1], S[ii][2], S[ii][3]);
}

// Prefill form of the recurrence, chunkwise (the published chunked form of
// the gated delta rule, in exact arithmetic the same recurrence). Over a
// chunk of m tokens from state S0, with G_t the running sum of the log decay
// g from the chunk start, gamma_t = exp(G_t), and the sequential recurrence
// S_t = a_t S_{t-1} + k_t d_t^T, d_t = beta_t (v_t - (a_t S_{t-1})^T k_t):
//   d = T U,  T = (I + L)^-1,  U_t = beta_t (v_t - gamma_t S0^T k_t),
//                              L_ti = beta_t exp(G_t - G_i) (k_t . k_i), i < t
//   o_t = gamma_t S0^T q_t + sum_{i<=t} B_ti d_i,  B_ti = exp(G_t - G_i) (q_t . k_i)
//   S_m = gamma_m S0 + sum_i exp(G_m - G_i) k_i d_i^T
// (every decay factor exp(G_t - G_i) with t >= i is at most 1). T and B do not
// depend on the state, so the chunks of a sequence are only serial in the
// products with S. Two kernels:
//   gdn_prep_kernel, one workgroup per (chunk, key head), every chunk at once:
//     the token norms, K K^T and Q K^T, and per value head of the key head the
//     decays, B and T (16 x 16 diagonal blocks by forward substitution);
//   gdn_scan_kernel, one workgroup per (value head, 16 columns of S, sequence),
//     serial over the chunks. A column of S evolves on its own. Wave w keeps S
//     rows 32 w .. 32 w + 31 in registers (8 per lane): a 16x16 tile of the
//     fp32 MFMA's result is laid out exactly as the next one's B operand, so S,
//     W = K S0, U and d never leave them. Per chunk: each wave's part of K S0
//     and Q S0 over its 32 rows (32 MFMAs), one exchange of the parts through
//     LDS (the only barrier), then d = T U on every wave (12 MFMAs), B d on two
//     of them, and the wave's S rows (16 MFMAs); q, k and v of the next chunk
//     load meanwhile, k passes through wave-private LDS for its transpose.
// The outputs go to o_raw; gdn_norm_kernel applies the gated RMSNorm. Bound:
// the chain of one chunk, 68 fp32 MFMAs (0.9 us) and the exchange between
// them. Measured for one sequence of 1500 rows and 32 value heads: prep 17 us,
// scan 120 us (2.6 us a chunk; 180 us for two such sequences), norm 16 us; for
// prompts of 211, 562 and 1500 rows 790 -> 205 us against one kernel that
// repeated the token products and the triangular solve in every column group,
// inside the serial loop (15.5 us a chunk).
constexpr int kGdnScanCols = 16;
constexpr int kGdnHeadFloats = 2 * kGdnChunk * kGdnChunk + 4 * kGdnChunk;  // T | B | beta | gamma | exp(G_m - G) | gamma_m
constexpr int kGdnKeyFloats = 2 * kGdnChunk;                              // 1 / |k| | 1 / (|q| sqrt(128))

// The sequence and place in it of chunk g; false past the last.
__device__ inline bool gdn_find_chunk(const int* row_count, int nseq, int cap, int g, int& s, int& c) {
  const int lane = threadIdx.x & 63;
  int base = 0;
  for (int j0 = 0; j0 < nseq; j0 += 64) {
    const int own = j0 + lane < nseq ? gdn_chunks(row_count[j0 + lane]) : 0;
    int incl = own;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int y = __shfl_up(incl, o, 64);
      if (lane >= o) incl += y;
    }
    const uint64_t hit = __ballot(base + incl > g);
    if (hit) {
      const int l = __builtin_ctzll(hit);
      const int end = base + __shfl(incl, l, 64);
      s = j0 + l;
      c = g - (end - __shfl(own, l, 64));
      return end <= cap;
    }
    base += __shfl(incl, 63, 64);
  }
  return false;
}

__global__ __launch_bounds__(256, 4) void gdn_prep_kernel(GdnParams p, const int* row_start, const int* row_count,
                                                       int nseq, int cap, float* __restrict__ head_out,
                                                       float* __restrict__ key_out) {
  constexpr int D = 128, C = kGdnChunk, LD = C + 4;
  static_assert(C == 32, "two 16-token tiles");
  __shared__ __attribute__((aligned(16))) f4 part[4 * 6 * 64];  // K K^T and Q K^T tiles of each wave's k range; then L
  __shared__ float kk[C * LD], qk[C * LD];
  __shared__ float red[4][2][C];
  const int g = blockIdx.x, kh = blockIdx.y, tid = threadIdx.x;
  const int lane = tid & 63, w = tid >> 6, lr = lane & 15, lk = lane >> 4;
  int s, ci;
  if (!gdn_find_chunk(row_count, nseq, cap, g, s, ci)) return;
  const int t0 = ci * C, m = min(C, row_count[s] - t0), r0 = row_start[s] + t0;
  // token 16 tb + lr, elements 32 w + 16 j + 4 lk ..: both MFMA operands
  f4 K[2][2], Q[2][2];
  float sk[2] = {0.f, 0.f}, sq[2] = {0.f, 0.f};
#pragma unroll
  for (int tb = 0; tb < 2; ++tb) {
    const int t = 16 * tb + lr;
    const float* cv = p.conv_out + (size_t)(r0 + t) * p.ld_conv + kh * D + 32 * w + 4 * lk;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      K[tb][j] = Q[tb][j] = f4{0.f, 0.f, 0.f, 0.f};
      if (t < m) {
        Q[tb][j] = *reinterpret_cast<const f4*>(cv + 16 * j);
        K[tb][j] = *reinterpret_cast<const f4*>(cv + p.k_heads * D + 16 * j);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        sk[tb] += K[tb][j][e] * K[tb][j][e];
        sq[tb] += Q[tb][j][e] * Q[tb][j][e];
      }
    }
#pragma unroll
    for (int o = 16; o < 64; o <<= 1) {
      sk[tb] += __shfl_xor(sk[tb], o, 64);
      sq[tb] += __shfl_xor(sq[tb], o, 64);
    }
    if (lk == 0) {
      red[w][0][t] = sk[tb];
      red[w][1][t] = sq[tb];
    }
  }
  __syncthreads();
  const float qscale = sqrtf((float)D);
#pragma unroll
  for (int tb = 0; tb < 2; ++tb) {
    const int t = 16 * tb + lr;
    const float ik = 1.0f / sqrtf(((red[0][0][t] + red[1][0][t]) + (red[2][0][t] + red[3][0][t])) + 1e-6f);
    const float iq = 1.0f / sqrtf(((red[0][1][t] + red[1][1][t]) + (red[2][1][t] + red[3][1][t])) + 1e-6f) / qscale;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      K[tb][j] *= ik;
      Q[tb][j] *= iq;
    }
    if (w == 0 && lk == 0) {
      float* ko = key_out + ((size_t)g * p.k_heads + kh) * kGdnKeyFloats;
      ko[t] = ik;
      ko[C + t] = iq;
    }
  }
  // tiles (0, 0), (1, 0), (1, 1) of both products (the fourth is above the diagonal)
#pragma unroll
  for (int x = 0; x < 3; ++x) {
    const int tb = x > 0, ib = x > 1;
    f4 a = {0.f, 0.f, 0.f, 0.f}, b = a;
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        a = __builtin_amdgcn_mfma_f32_16x16x4f32(K[tb][j][e], K[ib][j][e], a, 0, 0, 0);
        b = __builtin_amdgcn_mfma_f32_16x16x4f32(Q[tb][j][e], K[ib][j][e], b, 0, 0, 0);
      }
    part[(w * 6 + x) * 64 + lane] = a;
    part[(w * 6 + 3 + x) * 64 + lane] = b;
  }
  __syncthreads();
  for (int i = tid; i < 6 * 64; i += 256) {
    const f4 v = (part[i] + part[384 + i]) + (part[768 + i] + part[1152 + i]);
    const int x = (i >> 6) % 3, l = i & 63;
    float* o = (i < 192 ? kk : qk) + (16 * (x > 0) + 4 * (l >> 4)) * LD + 16 * (x > 1) + (l & 15);
#pragma unroll
    for (int r = 0; r < 4; ++r) o[r * LD] = v[r];
  }
  __syncthreads();
  // one wave per value head: lanes (half, i) take column i, tokens 16 half ..
  const int repeat = p.v_heads / p.k_heads, i = lane & 31, half = lane >> 5;
  float* Lm = reinterpret_cast<float*>(part) + w * C * LD;
  for (int hh = w; hh < repeat; hh += 4) {
    const int h = kh * repeat + hh;
    float G = 0.f, beta = 0.f;
    if (i < m) {
      const size_t row = (size_t)(r0 + i) * p.ld_ab + h;
      G = -expf(p.a_log[h]) * softplus_f(p.a[row] + p.dt_bias[h]);
      beta = 1.0f / (1.0f + expf(-p.b[row]));
    }
#pragma unroll
    for (int o = 1; o < 32; o <<= 1) {
      const float y = __shfl_up(G, o, 32);
      if (i >= o) G += y;
    }
    float* out = head_out + ((size_t)g * p.v_heads + h) * kGdnHeadFloats;
#pragma unroll 4
    for (int k = 0; k < 16; ++k) {
      const int t = 16 * half + k;
      const float gt = __shfl(G, t, 64), bt = __shfl(beta, t, 64);
      float vl = 0.f, vb = 0.f;
      if (t < m && i <= t) {
        const float wd = expf(gt - G);
        vb = wd * qk[t * LD + i];
        if (i < t) vl = bt * (wd * kk[t * LD + i]);
      }
      Lm[t * LD + i] = vl;
      out[C * C + t * C + i] = vb;
    }
    const float gl = __shfl(G, m - 1, 64);
    if (half == 0) {
      float* v = out + 2 * C * C;
      v[i] = beta;
      v[C + i] = expf(G);
      v[2 * C + i] = i < m ? expf(gl - G) : 0.f;
      v[3 * C + i] = expf(gl);
    }
    // T = [[X, 0], [-Y L10 X, Y]], X and Y the inverses of the two diagonal
    // blocks of I + L: lanes 16 b + j take column j of block b, forward
    // substitution against the unit vector
    const int bo = 16 * ((lane >> 4) & 1);
    float x[16];
#pragma unroll
    for (int t = 0; t < 16; ++t) {
      float acc = t == lr ? 1.0f : 0.0f;
#pragma unroll
      for (int u = 0; u < t; u += 4) {
        const f4 l4 = *reinterpret_cast<const f4*>(Lm + (bo + t) * LD + bo + u);
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (u + e < t) acc = fmaf(-l4[e], x[u + e], acc);
      }
      x[t] = acc;
    }
    f4 pr = {0.f, 0.f, 0.f, 0.f}, lo = pr;
    if (half == 0) {
      // the diagonal blocks replace L's in LDS
#pragma unroll
      for (int t = 0; t < 16; ++t) {
        Lm[(bo + t) * LD + bo + lr] = x[t];
        out[(bo + t) * C + bo + lr] = x[t];
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    const f4 l10 = *reinterpret_cast<const f4*>(Lm + (16 + lr) * LD + 4 * lk);
    const f4 yt = *reinterpret_cast<const f4*>(Lm + (16 + lr) * LD + 16 + 4 * lk);
#pragma unroll
    for (int e = 0; e < 4; ++e)
      pr = __builtin_amdgcn_mfma_f32_16x16x4f32(l10[e], Lm[(4 * lk + e) * LD + lr], pr, 0, 0, 0);
#pragma unroll
    for (int e = 0; e < 4; ++e) lo = __builtin_amdgcn_mfma_f32_16x16x4f32(yt[e], pr[e], lo, 0, 0, 0);
#pragma unroll
    for (int r = 0; r < 4; ++r) out[(16 + 4 * lk + r) * C + lr] = -lo[r];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  }
}

__global__ __launch_bounds__(256, 3) void gdn_scan_kernel(GdnParams p, const int* row_start, const int* row_count,
                                                       int cap, const float* __restrict__ head_in,
                                                       const float* __restrict__ key_in) {
  constexpr int D = 128, C = kGdnChunk, LD = C + 4, NG = D / kGdnScanCols;
  __shared__ __attribute__((aligned(16))) f4 part[2][4][4][64];  // [chunk parity][wave][W tiles, Z tiles]
  __shared__ __attribute__((aligned(16))) float kl[4][C * LD];   // each wave's 32 columns of k
  // workgroups go to the 8 XCDs round robin: give each XCD whole heads, whose
  // column groups read the same q and k
  const int per = p.v_heads * NG / 8, id = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  const int h = id / NG, col0 = (id % NG) * kGdnScanCols, s = blockIdx.y;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, lr = lane & 15, lk = lane >> 4;
  const int n = row_count[s];
  if (n < kGdnLongRows) return;
  const int base = gdn_chunk_base(row_count, s, cap);
  if (base < 0) return;
  const int r0 = row_start[s], kh = h / (p.v_heads / p.k_heads), ldo = p.v_heads * D;
  float* st = p.state_base[s] + p.state_off + (size_t)h * D * D + col0 + lr;
  // S[j][r]: row 32 w + 16 j + 4 lk + r, column col0 + lr
  f4 S[2];
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int r = 0; r < 4; ++r) S[j][r] = st[(size_t)(32 * w + 16 * j + 4 * lk + r) * D];
  // A chunk's inputs. Each is loaded for the next chunk as soon as this one is
  // done with its registers (one set: three workgroups fit a CU); tokens past
  // the sequence re-read its last row, and their T, B, beta and decay entries
  // drop them.
  const int nc = gdn_chunks(n);
  f4 q[2][2], k[2][2], v[2];  // q, k: token 16 tb + lr; v: token 16 tb + 4 lk + r
  float iq[2], ik[2];
  f4 T00, T10, T11, be[2], ga[2], wd[2];
  float gm;
  auto head = [&](int c) { return head_in + ((size_t)(base + c) * p.v_heads + h) * kGdnHeadFloats; };
  // tile (tb, ib) of T or B: row 16 tb + lr, columns 16 ib + 4 lk ..
  auto tile = [&](const float* a, int tb, int ib) {
    return *reinterpret_cast<const f4*>(a + (16 * tb + lr) * C + 16 * ib + 4 * lk);
  };
  const float* qp = p.conv_out + kh * D + 32 * w + 4 * lk;
  const float* vp = p.conv_out + 2 * p.k_heads * D + h * D + col0 + lr;
  auto load_qk = [&](int c) {
    const float* kd = key_in + ((size_t)(base + c) * p.k_heads + kh) * kGdnKeyFloats + lr;
#pragma unroll
    for (int tb = 0; tb < 2; ++tb) {
      const float* row = qp + (size_t)(r0 + min(c * C + 16 * tb + lr, n - 1)) * p.ld_conv;
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        q[tb][j] = *reinterpret_cast<const f4*>(row + 16 * j);
        k[tb][j] = *reinterpret_cast<const f4*>(row + p.k_heads * D + 16 * j);
      }
      ik[tb] = kd[16 * tb];
      iq[tb] = kd[C + 16 * tb];
    }
  };
  auto load_v = [&](int c) {
#pragma unroll
    for (int tb = 0; tb < 2; ++tb)
#pragma unroll
      for (int r = 0; r < 4; ++r) v[tb][r] = vp[(size_t)(r0 + min(c * C + 16 * tb + 4 * lk + r, n - 1)) * p.ld_conv];
  };
  auto load_head = [&](int c) {
    const float* hd = head(c);
    T00 = tile(hd, 0, 0);
    T10 = tile(hd, 1, 0);
    T11 = tile(hd, 1, 1);
    const float* vec = hd + 2 * C * C + 4 * lk;
#pragma unroll
    for (int tb = 0; tb < 2; ++tb) {
      be[tb] = *reinterpret_cast<const f4*>(vec + 16 * tb);
      ga[tb] = *reinterpret_cast<const f4*>(vec + C + 16 * tb);
      wd[tb] = *reinterpret_cast<const f4*>(vec + 2 * C + 16 * tb);
    }
    gm = hd[2 * C * C + 3 * C];
  };
  const f4 zero = {0.f, 0.f, 0.f, 0.f};
  load_qk(0);
  load_v(0);
  load_head(0);
  auto chunk = [&](int c, auto more) {  // more: another chunk follows
    const int m = min(C, n - c * C), next = c + 1;
    f4 b0, b1;
    if (w < 2) {
      b0 = tile(head(c) + C * C, w, 0);
      b1 = tile(head(c) + C * C, 1, 1);
    }
    f4 W[2] = {zero, zero}, Z[2] = {zero, zero};
#pragma unroll
    for (int j = 0; j < 2; ++j) {
#pragma unroll
      for (int tb = 0; tb < 2; ++tb) {
        k[tb][j] *= ik[tb];
        q[tb][j] *= iq[tb];
        *reinterpret_cast<f4*>(&kl[w][(16 * tb + lr) * LD + 16 * j + 4 * lk]) = k[tb][j];
      }
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int tb = 0; tb < 2; ++tb) {
          W[tb] = __builtin_amdgcn_mfma_f32_16x16x4f32(k[tb][j][e], S[j][e], W[tb], 0, 0, 0);
          Z[tb] = __builtin_amdgcn_mfma_f32_16x16x4f32(q[tb][j][e], S[j][e], Z[tb], 0, 0, 0);
        }
    }
    if constexpr (more) load_qk(next);
    __builtin_amdgcn_sched_barrier(0);
    f4(*pc)[4][64] = part[c & 1];
#pragma unroll
    for (int tb = 0; tb < 2; ++tb) {
      pc[w][tb][lane] = W[tb];
      pc[w][2 + tb][lane] = Z[tb];
    }
    __syncthreads();  // (the other parity's parts were read before the previous one)
    auto whole = [&](int x) { return (pc[0][x][lane] + pc[1][x][lane]) + (pc[2][x][lane] + pc[3][x][lane]); };
    f4 U[2], d[2] = {zero, zero};
#pragma unroll
    for (int tb = 0; tb < 2; ++tb) U[tb] = be[tb] * (v[tb] - ga[tb] * whole(tb));
    if constexpr (more) load_v(next);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      d[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(T00[e], U[0][e], d[0], 0, 0, 0);
      d[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(T10[e], U[0][e], d[1], 0, 0, 0);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) d[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(T11[e], U[1][e], d[1], 0, 0, 0);
    if (w < 2) {
      // outputs of tokens 16 w ..
      f4 o = (w ? ga[1] : ga[0]) * whole(2 + w);
#pragma unroll
      for (int e = 0; e < 4; ++e) o = __builtin_amdgcn_mfma_f32_16x16x4f32(b0[e], d[0][e], o, 0, 0, 0);
      if (w)
#pragma unroll
        for (int e = 0; e < 4; ++e) o = __builtin_amdgcn_mfma_f32_16x16x4f32(b1[e], d[1][e], o, 0, 0, 0);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int t = 16 * w + 4 * lk + r, row = r0 + c * C + t;
        if (t < m && row < p.o_rows) p.o_raw[(size_t)row * ldo + h * D + col0 + lr] = o[r];
      }
    }
    // S = gamma_m S0 + K^T (weighted d)
#pragma unroll
    for (int tb = 0; tb < 2; ++tb) d[tb] *= wd[tb];
#pragma unroll
    for (int j = 0; j < 2; ++j) S[j] *= gm;
    if constexpr (more) load_head(next);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int tb = 0; tb < 2; ++tb)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          S[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(kl[w][(16 * tb + 4 * lk + e) * LD + 16 * j + lr], d[tb][e], S[j],
                                                      0, 0, 0);
  };
  // The last chunk is a copy of the loop's body without the loads of a next one:
  // the CU's address units take about 16 cycles for each of a wave's loads, so
  // what the last chunk loads again is time where chunks are few (whole call at
  // 4, 16 and 64 sequences of 32 rows 34.4 -> 30.5, 81 -> 65, 277 -> 221 us).
  // Branches around the loads instead make the loop 8% slower.
  for (int c = 0; c + 1 < nc; ++c) chunk(c, std::true_type{});
  chunk(nc - 1, std::false_type{});
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int r = 0; r < 4; ++r) st[(size_t)(32 * w + 16 * j + 4 * lk + r) * D] = S[j][r];
}

// Gated RMSNorm of the chunkwise outputs (rows of long sequences only), the
// step kernel's tail: out and / or the prepared activations. grid (row blocks,
// sequences, groups of four value heads), one wave per head, two elements per
// lane; a workgroup strides over its sequence's rows, kGdnNormRows loaded at a
// time. Bound: HBM.
constexpr int kGdnNormRows = 4;
__global__ __launch_bounds__(256) void gdn_norm_kernel(GdnParams p, const int* row_start, const int* row_count,
                                                       int cap) {
  constexpr int D = 128;
  __shared__ __attribute__((aligned(16))) float obuf[4][D];
  const int s = blockIdx.y, w = threadIdx.x >> 6, h = blockIdx.z * 4 + w, lane = threadIdx.x & 63;
  const int n = row_count[s];
  if (h >= p.v_heads || n < kGdnLongRows || gdn_chunk_base(row_count, s, cap) < 0) return;
  const float n0 = p.norm[2 * lane], n1 = p.norm[2 * lane + 1];
  // (rows at or past o_rows were never staged: a caller's rows bound was too small)
  const int r0 = row_start[s], t_end = min(n, p.o_rows - r0);
  for (int t0 = blockIdx.x * kGdnNormRows; t0 < t_end; t0 += gridDim.x * kGdnNormRows) {
    float2 o[kGdnNormRows];
    float z0[kGdnNormRows], z1[kGdnNormRows];
#pragma unroll
    for (int k = 0; k < kGdnNormRows; ++k) {
      const size_t row = r0 + min(t0 + k, t_end - 1);
      o[k] = *reinterpret_cast<const float2*>(p.o_raw + row * p.v_heads * D + h * D + 2 * lane);
      z0[k] = p.z[row * p.ld_z + h * D + 2 * lane];
      z1[k] = p.z[row * p.ld_z + h * D + 2 * lane + 1];
    }
#pragma unroll
    for (int k = 0; k < kGdnNormRows; ++k) {
      if (t0 + k >= t_end) break;
      const int row = r0 + t0 + k;
      const float inv = 1.0f / sqrtf(wave_sum(o[k].x * o[k].x + o[k].y * o[k].y) / (float)D + 1e-6f);
      const float v0 = o[k].x * inv * n0 * (z0[k] / (1.0f + expf(-z0[k])));
      const float v1 = o[k].y * inv * n1 * (z1[k] / (1.0f + expf(-z1[k])));
      if (p.out) {
        p.out[(size_t)row * p.ld_out + h * D + 2 * lane] = v0;
        p.out[(size_t)row * p.ld_out + h * D + 2 * lane + 1] = v1;
      }
      if (p.act.XA) {
        obuf[w][2 * lane] = v0;
        obuf[w][2 * lane + 1] = v1;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        if (lane < D / 16) {
          float v[16];
#pragma unroll
          for (int e = 0; e < 16; ++e) v[e] = obuf[w][16 * lane + e];
          a8act::emit_slice(p.act, row, (h * D + 16 * lane) >> 6, lane & 3, v, true);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      }
    }
  }
}

// ---------------------------------------------------------------------------
// q/k/v preparation + paged KV write; one wave per (head or kv head, row)
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(64) void qkv_prep_kernel(QkvPrep p, AttnLayout L, RowMeta m) {
  __shared__ float buf[512];
  const int r = blockIdx.y;
  const int hidx = blockIdx.x;
  const int lane = threadIdx.x;
  const int hd = L.head_dim, rd = L.rotary_dim, half = rd / 2;
  const int E = hd / 64;
  const bool is_q = hidx < L.heads;
  const int h = is_q ? hidx : hidx - L.heads;
  const float* src;
  const float* bias = nullptr;
  const float* nw = nullptr;
  if (is_q) {
    src = p.q_raw + (size_t)r * p.ld_q + (size_t)h * hd * (p.variant == 0 ? 2 : 1);
    bias = p.variant == 1 ? p.q_bias + (size_t)h * hd : nullptr;
    nw = p.variant == 0 ? p.q_norm : nullptr;
  } else {
    src = p.k_raw + (size_t)r * p.ld_kv + (size_t)h * hd;
    bias = p.variant == 1 ? p.k_bias + (size_t)h * hd : nullptr;
    nw = p.variant == 0 ? p.k_norm : nullptr;
  }
  float v[4], cs_v[4], sn_v[4];
  float ss = 0.0f;
  // the RoPE table entries are loaded with the row (one round trip)
  const float* cs = m.cos + (size_t)r * rd;
  const float* sn = m.sin + (size_t)r * rd;
  for (int e = 0; e < E; ++e) {
    const int d = lane + 64 * e;
    v[e] = src[d];
    cs_v[e] = d < rd ? cs[d] : 0.0f;
    sn_v[e] = d < rd ? sn[d] : 0.0f;
    if (bias) v[e] = v[e] + bias[d];
    ss += v[e] * v[e];
  }
  if (nw) {
    ss = wave_sum(ss);
    const float inv = 1.0f / sqrtf(ss / (float)hd + 1e-6f);
    for (int e = 0; e < E; ++e) v[e] = v[e] * inv * nw[lane + 64 * e];
  }
  for (int e = 0; e < E; ++e) buf[lane + 64 * e] = v[e];
  __syncthreads();
  for (int e = 0; e < E; ++e) {
    const int d = lane + 64 * e;
    if (d < rd) {
      const float rot = d < half ? -buf[d + half] : buf[d - half];
      v[e] = buf[d] * cs_v[e] + rot * sn_v[e];
    }
  }
  if (is_q) {
    float* qd = p.q + ((size_t)r * L.heads + h) * hd;
    for (int e = 0; e < E; ++e) qd[lane + 64 * e] = v[e];
    if (p.variant == 0) {
      float* gd = p.gate + ((size_t)r * L.heads + h) * hd;
      for (int e = 0; e < E; ++e) gd[lane + 64 * e] = src[hd + lane + 64 * e];
    }
  } else {
    const int seq = m.seq_of_row[r], pos = m.pos_of_row[r];
    const int blk = m.block_tables[(size_t)seq * m.max_blocks + pos / L.block];
    const size_t off = (((size_t)blk * L.kv_heads + h) * L.block + (pos % L.block)) * hd;
    const float* vs = p.v_raw + (size_t)r * p.ld_kv + (size_t)h * hd;
    const float* vb = p.variant == 1 ? p.v_bias + (size_t)h * hd : nullptr;
    for (int e = 0; e < E; ++e) {
      const int d = lane + 64 * e;
      L.k_pool[off + d] = v[e];
      L.v_pool[off + d] = vb ? vs[d] + vb[d] : vs[d];
    }
  }
}


// ---------------------------------------------------------------------------
// argmax
// ---------------------------------------------------------------------------
__device__ inline bool better(float v, int i, float bv, int bi, int last_max) {
  if (bi < 0) return true;
  if (v > bv) return true;
  if (v < bv) return false;
  return last_max ? i > bi : i < bi;
}

// Row argmax in two passes: kArgChunks workgroups per row each reduce one
// contiguous chunk, then one wave per row merges the chunk winners. better()
// is a total order on (value, index), so the merge order does not matter.
constexpr int kArgChunks = 64;
struct ArgPart {
  float v;
  int i, nf;
};

__device__ inline void arg_merge(float& bv, int& bi, int& nf, float v, int i, int n2, int last_max) {
  if (i >= 0 && better(v, i, bv, bi, last_max)) {
    bv = v;
    bi = i;
  }
  nf += n2;
}

__global__ __launch_bounds__(256) void argmax_part_kernel(const float* __restrict__ x, int ld, int n, int last_max,
                                                          ArgPart* __restrict__ part) {
  __shared__ ArgPart sp[4];
  const int r = blockIdx.y, b = blockIdx.x, tid = threadIdx.x;
  const int len = (n + kArgChunks - 1) / kArgChunks;
  const int lo = b * len, hi = min(n, lo + len);
  const float* xr = x + (size_t)r * ld;
  float bv = -INFINITY;
  int bi = -1, nf = 0;
  for (int i = lo + tid; i < hi; i += 256) {
    const float v = xr[i];
    if (!isfinite(v)) nf++;
    else if (better(v, i, bv, bi, last_max)) {
      bv = v;
      bi = i;
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const float v = __shfl_xor(bv, o, 64);
    const int i = __shfl_xor(bi, o, 64);
    const int f = __shfl_xor(nf, o, 64);
    arg_merge(bv, bi, nf, v, i, f, last_max);
  }
  if ((tid & 63) == 0) sp[tid >> 6] = ArgPart{bv, bi, nf};
  __syncthreads();
  if (tid == 0) {
    for (int w = 1; w < 4; ++w) arg_merge(bv, bi, nf, sp[w].v, sp[w].i, sp[w].nf, last_max);
    part[(size_t)r * kArgChunks + b] = ArgPart{bv, bi, nf};
  }
}

__global__ __launch_bounds__(64) void argmax_final_kernel(const ArgPart* __restrict__ part, int last_max,
                                                          uint32_t* ids, float* vals, int* nonfinite) {
  const int r = blockIdx.x, lane = threadIdx.x;
  ArgPart p = part[(size_t)r * kArgChunks + lane];
  float bv = p.v;
  int bi = p.i, nf = p.nf;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const float v = __shfl_xor(bv, o, 64);
    const int i = __shfl_xor(bi, o, 64);
    const int f = __shfl_xor(nf, o, 64);
    arg_merge(bv, bi, nf, v, i, f, last_max);
  }
  if (lane == 0) {
    ids[r] = bi < 0 ? 0xFFFFFFFFu : (uint32_t)bi;
    if (vals) vals[r] = bv;
    if (nonfinite) nonfinite[r] = nf;
  }
}

__global__ void gather_kernel(const float* src, int lds, const int* idx, int n, float* dst, int ldd) {
  const int r = blockIdx.y;
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) dst[(size_t)r * ldd + i] = src[(size_t)idx[r] * lds + i];
}

}  // namespace

// ---------------------------------------------------------------------------
void rmsnorm_rows(const float* x, int ldx, const int* rows_idx, int rows, int n, const float* w, float eps, int mode,
                  float* y, int ldy, hipStream_t s) {
  if (rows <= 0) return;
  PGD_CHECK(mode != 2 || n <= 8192, kErrShape, "ordered-sum RMSNorm rows are at most 8192 wide");
  if (mode == 2) hipLaunchKernelGGL(rmsnorm_ordered_kernel, dim3(rows), dim3(256), 0, s, x, ldx, rows_idx, n, w, eps, y, ldy);
  else hipLaunchKernelGGL(rmsnorm_kernel, dim3(rows), dim3(256), 0, s, x, ldx, rows_idx, n, w, eps, mode, y, ldy);
  PGD_HIP(hipGetLastError());
}

void conv_step(const float* x, int ldx, float* out, int ldo, int channels, int kernel, const float* weight,
               float* const* state_base, size_t state_off, SeqMeta meta, int nseq, int max_rows, hipStream_t s) {
  PGD_CHECK(kernel >= 1 && kernel <= 8, kErrShape, "conv kernel must be in 1..8");
  if (nseq <= 0) return;
  const int segs = max_rows > kConvSeg ? (max_rows + kConvSeg - 1) / kConvSeg : 1;
  const dim3 grid((channels + 255) / 256, nseq, segs);
#define PGD_CONV_CASE(K)                                                                                            \
  case K:                                                                                                          \
    hipLaunchKernelGGL(conv_step_kernel<K>, grid, dim3(256), 0, s, x, ldx, out, ldo, channels, weight, state_base, \
                       state_off, meta.row_start, meta.row_count);                                                 \
    break;
  switch (kernel) {
    PGD_CONV_CASE(1)
    PGD_CONV_CASE(2)
    PGD_CONV_CASE(3)
    PGD_CONV_CASE(4)
    PGD_CONV_CASE(5)
    PGD_CONV_CASE(6)
    PGD_CONV_CASE(7)
    PGD_CONV_CASE(8)
  }
#undef PGD_CONV_CASE
  PGD_HIP(hipGetLastError());
}

void gdn_step(const GdnParams& p, SeqMeta meta, int nseq, int rows, int max_rows, hipStream_t s) {
  PGD_CHECK(p.k_dim == 128 && p.v_dim == 128, kErrShape, "gated delta kernel needs k_dim == v_dim == 128");
  PGD_CHECK(p.k_heads > 0 && p.v_heads % p.k_heads == 0, kErrShape, "v_heads must be a multiple of k_heads");
  if (nseq <= 0) return;
  const bool chunked = rows > 0 && max_rows >= kGdnLongRows;
  GdnParams q = p;
  q.o_raw = nullptr;
  q.o_rows = q.chunk_cap = 0;
  float *head_ws = nullptr, *key_ws = nullptr;
  if (chunked) {
    // every long sequence's chunks: at most rows / 32 whole ones and a ragged one each
    q.o_rows = rows;
    q.chunk_cap = rows / kGdnChunk + nseq;
    const size_t o_floats = (size_t)rows * p.v_heads * 128, head_floats = (size_t)q.chunk_cap * p.v_heads * kGdnHeadFloats;
    const size_t key_floats = (size_t)q.chunk_cap * p.k_heads * kGdnKeyFloats;
    q.o_raw = static_cast<float*>(gemv::gemv_scratch(s, (o_floats + head_floats + key_floats) * sizeof(float), 7));
    head_ws = q.o_raw + o_floats;
    key_ws = head_ws + head_floats;
  }
  hipLaunchKernelGGL(gdn_kernel<kGdnRowGroups>, dim3(p.v_heads, nseq), dim3(32 * kGdnRowGroups), 0, s, q,
                     meta.row_start, meta.row_count);
  PGD_HIP(hipGetLastError());
  if (!chunked) return;
  PGD_CHECK(p.ld_conv % 4 == 0, kErrShape, "chunked gated delta kernel needs 16-byte aligned conv rows");
  hipLaunchKernelGGL(gdn_prep_kernel, dim3(q.chunk_cap, p.k_heads), dim3(256), 0, s, q, meta.row_start, meta.row_count,
                     nseq, q.chunk_cap, head_ws, key_ws);
  PGD_HIP(hipGetLastError());
  hipLaunchKernelGGL(gdn_scan_kernel, dim3(p.v_heads * (128 / kGdnScanCols), nseq), dim3(256), 0, s, q, meta.row_start,
                     meta.row_count, q.chunk_cap, head_ws, key_ws);
  PGD_HIP(hipGetLastError());
  hipLaunchKernelGGL(gdn_norm_kernel, dim3(std::min((max_rows + kGdnNormRows - 1) / kGdnNormRows, 4096), nseq, (p.v_heads + 3) / 4), dim3(256), 0, s, q,
                     meta.row_start, meta.row_count, q.chunk_cap);
  PGD_HIP(hipGetLastError());
}

void qkv_prep(const QkvPrep& p, const AttnLayout& L, const RowMeta& m, int rows, hipStream_t s) {
  PGD_CHECK(L.head_dim % 64 == 0 && L.head_dim <= 256, kErrShape, "head_dim must be 64, 128, 192 or 256");
  PGD_CHECK(L.rotary_dim % 2 == 0 && L.rotary_dim <= L.head_dim, kErrShape, "rotary_dim");
  if (rows <= 0) return;
  hipLaunchKernelGGL(qkv_prep_kernel, dim3(L.heads + L.kv_heads, rows), dim3(64), 0, s, p, L, m);
  PGD_HIP(hipGetLastError());
}

void argmax_rows(const float* x, int ld, int rows, int n, int last_max, uint32_t* ids, float* vals, int* nonfinite,
                 hipStream_t s) {
  if (rows <= 0) return;
  static_assert(kArgChunks == 64, "one wave merges the chunks");
  auto* part = static_cast<ArgPart*>(gemv::gemv_scratch(s, (size_t)rows * kArgChunks * sizeof(ArgPart)));
  hipLaunchKernelGGL(argmax_part_kernel, dim3(kArgChunks, rows), dim3(256), 0, s, x, ld, n, last_max, part);
  hipLaunchKernelGGL(argmax_final_kernel, dim3(rows), dim3(64), 0, s, part, last_max, ids, vals, nonfinite);
  PGD_HIP(hipGetLastError());
}

void gather_rows(const float* src, int lds, const int* idx, int rows, int n, float* dst, int ldd, hipStream_t s) {
  if (rows <= 0) return;
  hipLaunchKernelGGL(gather_kernel, dim3((n + 255) / 256, rows), dim3(256), 0, s, src, lds, idx, n, dst, ldd);
  PGD_HIP(hipGetLastError());
}

}  // namespace pgd
