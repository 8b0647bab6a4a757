// The fc products of rows that choose no slopes -- the spec backward, the
// alpha / beta loops and their gradient sweep -- on the bf16 matrix cores
// (vc_split.h), each with the elementwise step before it:
//   backward       e = pos(x) lo_s + neg(x) up_s [+ beta], out = e W,
//                  acc += neg(x) . up_t + e . bias
//   gradient step  e = x (pos(P) lo_s + neg(P) up_s) + neg(P) up_t,
//                  out = e W^T + bias
//   gradient input e = xl [x >= 0] + xh [x <= 0], out = e W^T + bias
// (verify_zono_bnb.py:4366-4407 and 4409-4453; the autograd of both).
//
// Two passes.  k_fc_rows forms e and writes its three parts in operand order
// (HBM bound: 4 bytes read and 6 written per value, slopes from the caches;
// 73,728 x 256 rows 45 us).  k_fc_gemm multiplies: four waves take 16 MT rows x
// 128 columns, 32 columns each; a step's rows go through LDS (two buffers, one
// barrier a step), the weights' parts, packed once by vc_fc_split_pack, straight
// from L2 into registers, since no two waves share a column.  Forming e in the
// product's loads instead costs as many vector instructions as the products and
// holds the registers that hide the loads' latency (113 TFLOP/s).
// Of the six part products the five small ones run on in the matrix core's
// accumulator (2^-8 of the result: what it cuts there is below the result's
// last bit); the largest starts from zero each step of 64 products and is added
// in fp32, and what rounding takes from that sum goes to the small ones.  (Steps
// of 32, one barrier and one such addition each: 136 TFLOP/s, not 155.)
//
// Measured, both passes, against the relaxation pass and fp32 product before
// (the gradient's: 64-bit folds of fp32 matrix steps): 1024 x 1024 at 4,608 rows
// 130 -> 88 us and 204 -> 87, at 73,728 rows 1193 -> 999 and 2743 -> 1047 (155
// TFLOP/s of the product); 256 x 256 at 73,728 rows 157 -> 114 and 197 -> 127.
// Relative to 64 bits 5.2e-8 in the 2-norm (2.5e-7 to 5e-7 before; the
// gradient's 4.6e-8, 7.2e-8 before).
#include "vc_gemm_core.h"
#include "vc_mlp_common.h"
#include "vc_split.h"

namespace {

using namespace vcs;
using vcg::FastDiv;

constexpr int FNT = 256;   // threads
constexpr int FBK = 32;    // one matrix step of a row's values
constexpr int FBN = 128;   // columns of a workgroup
constexpr int kTileU = 3 * 64;  // 16-byte units of 16 rows x 32 values, three parts

typedef uint32_t u4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ v4f mfma_bf16(u4 a, u4 b, v4f acc) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, a),
                                                 __builtin_bit_cast(v8bf, b), acc, 0, 0, 0);
}

enum Form { kRelax, kGradStep, kGradInput };

struct RowArgs {
  const float* x;   // rows (M, K); shared: (R, K), row m reads m mod R
  const float* P;   // gradient step: the rows before the relu, shared or not
  const float *s0, *s1, *s2;  // lo_s, up_s, up_t (M / R, K), or xl, xh
  const float* beta;
  const float* bias;  // backward: (K)
  uint4* parts;
  float* acc;
  int64_t M;
  int R, K, shared, nkc;
  FastDiv f_R;
};

// Values k .. k + 7 of K; past the end zero.
template <bool VEC>
__device__ __forceinline__ void ld8(const float* p, int k, int K, float* o) {
  if (VEC) {  // K a multiple of 4: a quad is inside or past the end
#pragma unroll
    for (int q = 0; q < 8; q += 4) {
      const float4 v = *reinterpret_cast<const float4*>(p + min(k + q, K - 4));
      const bool in = k + q < K;
      o[q] = in ? v.x : 0.f;
      o[q + 1] = in ? v.y : 0.f;
      o[q + 2] = in ? v.z : 0.f;
      o[q + 3] = in ? v.w : 0.f;
    }
  } else {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float v = p[min(k + j, K - 1)];
      o[j] = k + j < K ? v : 0.f;
    }
  }
}

// split8 that keeps every value: one that rounds to infinity is cut instead,
// and an infinity or NaN stands in the first part alone, so that the parts'
// sum is the value.
__device__ __forceinline__ void split8_all(const float* x, uint4& h, uint4& m, uint4& l) {
  split8(x, h, m, l);
  bool big = false;
#pragma unroll
  for (int j = 0; j < 8; ++j) big = big || !(fabsf(x[j]) < 3.38e38f);
  if (big) {
    uint32_t* const o[3] = {&h.x, &m.x, &l.x};
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      float v = x[j];
      uint32_t b[3];
#pragma unroll
      for (int p = 0; p < 3; ++p) {
        b[p] = __builtin_bit_cast(uint32_t, v) & 0xffff0000u;
        if (v != v) b[p] |= 0x400000u;
        v = finite(x[j]) ? v - __builtin_bit_cast(float, b[p]) : 0.f;
      }
#pragma unroll
      for (int p = 0; p < 3; ++p)
        o[p][j / 2] = (j & 1) ? (o[p][j / 2] & 0xffffu) | b[p] : (o[p][j / 2] & 0xffff0000u) | b[p] >> 16;
    }
  }
}

// The value that enters the product.
template <int FORM>
__device__ __forceinline__ float value(float x, float a, float b, float c, float d) {
  if (FORM == kRelax) return (fmaxf(x, 0.f) * a + fminf(x, 0.f) * b);
  if (FORM == kGradStep) {
    const bool mp = d >= 0.f, mn = d <= 0.f;
    float e = x * ((mp ? a : 0.f) + (mn ? b : 0.f));
    if (mn) e += c;
    return e;
  }
  float e = 0.f;
  if (x >= 0.f) e += a;
  if (x <= 0.f) e += b;
  return e;
}

// parts[row tile][32-deep step][part][lane][8]: the value of row
// 16 tile + lane % 16 at k = 32 step + 8 (lane / 16) + j; rows past M repeat
// the last one, values past K are zero.  A workgroup takes 16 rows, its waves
// every fourth step: 128 bytes of each row at a time, 1 KB stores.
template <int FORM, bool VEC>
__global__ __launch_bounds__(FNT) void k_fc_rows(RowArgs a) {
  __shared__ double red[4][16];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, g = lane >> 4, r = lane & 15;
  const int64_t m0 = (int64_t)blockIdx.x * 16;
  const int64_t m = m0 + r < a.M ? m0 + r : a.M - 1;
  const int64_t dom = a.f_R.div((uint32_t)m), row = a.shared ? m - dom * a.R : m;
  const float* x = a.x + (FORM == kGradStep ? m : row) * a.K;
  const float* P = FORM == kGradStep ? a.P + row * a.K : nullptr;
  const int64_t di = dom * a.K;
  uint4* out = a.parts + (int64_t)blockIdx.x * a.nkc * kTileU + lane;
  double part = 0.0;
  for (int kc = wv; kc < a.nkc; kc += 4) {
    const int k = kc * FBK + 8 * g;
    float xv[8], av[8], bv[8], cv[8], dv[8], e[8];
    ld8<VEC>(x, k, a.K, xv);
    ld8<VEC>(a.s0 + di, k, a.K, av);
    ld8<VEC>(a.s1 + di, k, a.K, bv);
    if (FORM != kGradInput) ld8<VEC>(a.s2 + di, k, a.K, cv);
    if (FORM == kGradStep) ld8<VEC>(P, k, a.K, dv);
#pragma unroll
    for (int j = 0; j < 8; ++j) e[j] = value<FORM>(xv[j], av[j], bv[j], cv[j], dv[j]);
    if (FORM == kRelax) {
      if (a.beta) {
        ld8<VEC>(a.beta + di, k, a.K, dv);
#pragma unroll
        for (int j = 0; j < 8; ++j) e[j] = e[j] + dv[j];
      }
      float bi[8] = {};
      if (a.bias) ld8<VEC>(a.bias, k, a.K, bi);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        float p = fminf(xv[j], 0.f) * cv[j];
        if (a.bias) p += e[j] * bi[j];
        part += (double)p;
      }
    }
    if (FORM == kGradStep) {  // P's zeros past the end would let up_t's in
#pragma unroll
      for (int j = 0; j < 8; ++j) e[j] = k + j < a.K ? e[j] : 0.f;
    }
    uint4 h, md, l;
    split8_all(e, h, md, l);
    uint4* const o = out + (int64_t)kc * kTileU;
    o[0] = h;
    o[64] = md;
    o[128] = l;
  }
  if (FORM == kRelax) {
    part += __shfl_xor(part, 16, 64);
    part += __shfl_xor(part, 32, 64);
    if (g == 0) red[wv][r] = part;
    __syncthreads();
    if (threadIdx.x < 16 && m0 + r < a.M)
      a.acc[m] = (float)((double)a.acc[m] + ((red[0][r] + red[1][r]) + (red[2][r] + red[3][r])));
  }
}

struct GemmArgs {
  const uint4 *Ap, *Bp;
  const float* bias;  // (N) or null
  float* out;         // (M, N)
  int64_t M;
  int N, nkc, ntn, mt16;
  int64_t tiles;
  FastDiv f_ntn;
};

// Value j of lane's eight in a packed tile: the sum of its three parts.
__device__ float part_sum(const uint4* p, int j) {
  float s = 0.f;
  for (int i = 2; i >= 0; --i)
    s += __builtin_bit_cast(float,
                            (uint32_t) reinterpret_cast<const uint16_t*>(p + 64 * i)[j] << 16);
  return s;
}

// One output as the plain sum in 64 bits.
__device__ float plain_sum(const GemmArgs& a, int64_t m, int n) {
  const uint4* A = a.Ap + (m >> 4) * a.nkc * kTileU + (m & 15);
  const uint4* B = a.Bp + (int64_t)(n >> 4) * a.nkc * kTileU + (n & 15);
  double s = 0.0;
  for (int kc = 0; kc < a.nkc; ++kc)
    for (int k = 0; k < FBK; ++k) {
      const int64_t o = (int64_t)kc * kTileU + 16 * (k >> 3);
      s += (double)part_sum(A + o, k & 7) * (double)part_sum(B + o, k & 7);
    }
  return (float)s;
}

template <int MT>
__global__ __launch_bounds__(FNT, 2) void k_fc_gemm(GemmArgs a) {
  constexpr int AU = MT * 2 * kTileU;       // 16-byte units of a double step's rows
  constexpr int NL = (AU + FNT - 1) / FNT;  // of them per thread
  constexpr int Q = MT >= 2 ? 2 : 1;        // row tiles at a time
  constexpr int NG = MT / Q;
  __shared__ __align__(16) u4 lds[2][NL * FNT];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int64_t w = vcg::xcd_tile(blockIdx.x, a.tiles);
  const int tm = (int)a.f_ntn.div((uint32_t)w);
  const int tn = (int)(w - (int64_t)tm * a.ntn);

  // this thread's units of each double step's rows (a row tile's two steps lie
  // together); past the last row tile the last one again, not stored
  const u4* A[NL];
#pragma unroll
  for (int i = 0; i < NL; ++i) {
    const int u = min(tid + i * FNT, AU - 1);
    const int t = min(tm * MT + u / (2 * kTileU), a.mt16 - 1);
    A[i] = reinterpret_cast<const u4*>(a.Ap) + (int64_t)t * a.nkc * kTileU + u % (2 * kTileU);
  }
  // this wave's two column tiles, likewise
  const int c0 = tn * 8 + wv * 2, nt16 = (a.N + 15) >> 4;
  const u4* B[2];
#pragma unroll
  for (int j = 0; j < 2; ++j)
    B[j] = reinterpret_cast<const u4*>(a.Bp) + (int64_t)min(c0 + j, nt16 - 1) * a.nkc * kTileU +
           lane;

  v4f acc[MT][2], small[MT][2], z[MT][2];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = small[i][j] = v4f{0.f, 0.f, 0.f, 0.f};

  // past the last step the last again: no branch, nothing waits for it
  const int steps = a.nkc >> 1;
  const auto load_rows = [&](int s, u4(&v)[NL]) {
    const int64_t o = (int64_t)min(s, steps - 1) * (2 * kTileU);
#pragma unroll
    for (int i = 0; i < NL; ++i) v[i] = A[i][o];
  };
  const auto load_cols = [&](int kc, u4(&v)[2][3]) {
    const int64_t o = (int64_t)min(kc, a.nkc - 1) * kTileU;
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int p = 0; p < 3; ++p) v[j][p] = B[j][o + 64 * p];
  };
  u4 rn[NL], b[2][2][3];
  load_rows(0, rn);
  load_cols(0, b[0]);
#pragma unroll
  for (int i = 0; i < NL; ++i) lds[0][tid + i * FNT] = rn[i];

#pragma unroll 1
  for (int s = 0; s < steps; ++s) {
    __syncthreads();  // this step's rows are laid down, the ones before are read
    load_cols(2 * s + 1, b[1]);
    load_rows(s + 1, rn);
    __builtin_amdgcn_sched_barrier(0);  // requested before the products, not where they are used
    const u4* from = lds[s & 1] + lane;
    u4 av[2][Q][3];
    const auto read = [&](int t, u4(&v)[Q][3]) {  // half t / NG, row tiles Q (t mod NG) ..
#pragma unroll
      for (int i = 0; i < Q; ++i)
#pragma unroll
        for (int p = 0; p < 3; ++p)
          v[i][p] = from[((t % NG * Q + i) * 2 + t / NG) * kTileU + 64 * p];
    };
    read(0, av[0]);
#pragma unroll
    for (int t = 0; t < 2 * NG; ++t) {
      const int hf = t / NG, i0 = t % NG * Q;
      if (t == NG) {
        __builtin_amdgcn_sched_barrier(0);
        load_cols(2 * s + 2, b[0]);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (t + 1 < 2 * NG) read(t + 1, av[(t + 1) & 1]);
      __builtin_amdgcn_sched_barrier(0xe);  // loads stay here, arithmetic may pass
#pragma unroll
      for (int p = 0; p < 6; ++p)
#pragma unroll
        for (int i = 0; i < Q; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            v4f& d = p == 5 ? z[i0 + i][j] : small[i0 + i][j];
            d = mfma_bf16(av[t & 1][i][kPartA[p]], b[hf][j][kPartB[p]],
                          p == 5 && hf == 0 ? v4f{0.f, 0.f, 0.f, 0.f} : d);
          }
      if (hf == 1) {
#pragma unroll
        for (int i = i0; i < i0 + Q; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            const v4f t2 = acc[i][j] + z[i][j];
            small[i][j] += z[i][j] - (t2 - acc[i][j]);
            acc[i][j] = t2;
          }
      }
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < NL; ++i) lds[(s & 1) ^ 1][tid + i * FNT] = rn[i];
  }

  const int g = lane >> 4, r = lane & 15;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int n = (c0 + j) * 16 + r;
    if (n >= a.N) continue;
    const float b = a.bias ? a.bias[n] : 0.f;
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int64_t m = (int64_t)tm * MT * 16 + 16 * i + 4 * g + q;
        if (m >= a.M) continue;
        float v = acc[i][j][q] + small[i][j][q];
        // an infinity or NaN among the values: the plain sum
        if (!finite(v)) v = plain_sum(a, m, n);
        a.out[m * a.N + n] = a.bias ? v + b : v;
      }
  }
}

// Wp[column tile][32-deep step][part][lane][8]: part of B[k][n] for
// k = 32 step + 8 (lane / 16) + j, n = 16 tile + lane % 16; zero past the ends.
__global__ void k_fc_split_pack(const float* W, int K, int N, int trans, int nkc, int64_t total,
                                uint4* out) {
  for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < total;
       t += (int64_t)gridDim.x * blockDim.x) {
    const int lane = (int)(t & 63);
    const int64_t q = t >> 6;
    const int kc = (int)(q % nkc), n = (int)(q / nkc) * 16 + (lane & 15);
    const int k0 = kc * FBK + 8 * (lane >> 4);
    float v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j)
      v[j] = n < N && k0 + j < K
                 ? (trans ? W[(int64_t)n * K + k0 + j] : W[(int64_t)(k0 + j) * N + n])
                 : 0.f;
    uint4 h, m, l;
    split8_all(v, h, m, l);
    uint4* o = out + q * kTileU + lane;
    o[0] = h;
    o[64] = m;
    o[128] = l;
  }
}

template <int FORM>
int launch_fc(RowArgs a, const void* packed, int N, const float* bias, float* out, hipStream_t st) {
  if (a.M == 0) return VC_OK;
  GemmArgs b{};
  const int64_t mt16 = (a.M + 15) / 16;
  a.nkc = b.nkc = 2 * ((a.K + 2 * FBK - 1) / (2 * FBK));
  a.f_R = FastDiv::make((uint32_t)a.R);
  b.Ap = a.parts;
  b.Bp = (const uint4*)packed;
  b.bias = bias;
  b.out = out;
  b.M = a.M;
  b.N = N;
  b.mt16 = (int)mt16;
  b.ntn = (N + FBN - 1) / FBN;
  b.f_ntn = FastDiv::make((uint32_t)b.ntn);
  // the tallest row block that still gives every CU a tile
  const int64_t cus = vcm::cu_count();
  int mt = 4;
  while (mt > 1 && (mt16 + mt - 1) / mt * b.ntn < cus) mt >>= 1;
  b.tiles = (mt16 + mt - 1) / mt * b.ntn;
  if (a.M >= (int64_t(1) << 31) || b.tiles >= (int64_t(1) << 31)) return VC_ERR_UNSUPPORTED;
  bool vec = a.K % 4 == 0;
  for (const float* p : {a.x, a.P, a.s0, a.s1, a.s2, a.beta, a.bias}) vec = vec && aligned16(p);
  if (vec)
    hipLaunchKernelGGL((k_fc_rows<FORM, true>), dim3((unsigned)mt16), dim3(FNT), 0, st, a);
  else
    hipLaunchKernelGGL((k_fc_rows<FORM, false>), dim3((unsigned)mt16), dim3(FNT), 0, st, a);
  VC_LAUNCH_CHECK();
  const dim3 grid((unsigned)b.tiles);
  if (mt == 4) hipLaunchKernelGGL(k_fc_gemm<4>, grid, dim3(FNT), 0, st, b);
  if (mt == 2) hipLaunchKernelGGL(k_fc_gemm<2>, grid, dim3(FNT), 0, st, b);
  if (mt == 1) hipLaunchKernelGGL(k_fc_gemm<1>, grid, dim3(FNT), 0, st, b);
  VC_LAUNCH_CHECK();
  return VC_OK;
}

bool bad_args(int64_t M, int R, int K, int N, const void* packed, const void* work) {
  return M < 0 || R <= 0 || K <= 0 || N <= 0 || M % R != 0 || !packed || !work ||
         !aligned16(packed) || !aligned16(work);
}

}  // namespace

extern "C" int64_t vc_fc_split_pack_bytes(int64_t K, int64_t N) {
  if (K <= 0 || N <= 0) return 0;
  return (N + 15) / 16 * (2 * ((K + 2 * FBK - 1) / (2 * FBK))) * kTileU * 16;
}

extern "C" int vc_fc_split_pack(const float* W, int K, int N, int trans, void* out,
                                vc_stream_t stream) {
  if (!W || !out || K <= 0 || N <= 0 || !aligned16(out)) return VC_ERR_ARG;
  const int nkc = 2 * ((K + 2 * FBK - 1) / (2 * FBK));
  const int64_t total = (int64_t)((N + 15) / 16) * nkc * 64;
  hipLaunchKernelGGL(k_fc_split_pack, dim3(vc_blocks(total, 256)), dim3(256), 0,
                     (hipStream_t)stream, W, K, N, trans, nkc, total, (uint4*)out);
  VC_LAUNCH_CHECK();
  return VC_OK;
}

extern "C" int vc_backward_fc_split(const float* ew_in, int64_t M, int R, int ew_shared, int n_out,
                                    const float* lo_s, const float* up_s, const float* up_t,
                                    const float* beta, const void* packed, const float* bias,
                                    int n_in, float* ew_out, float* acc, void* work,
                                    vc_stream_t stream) {
  if (!ew_in || !lo_s || !up_s || !up_t || !ew_out || !acc ||
      bad_args(M, R, n_out, n_in, packed, work))
    return VC_ERR_ARG;
  RowArgs a{};
  a.x = ew_in;
  a.s0 = lo_s;
  a.s1 = up_s;
  a.s2 = up_t;
  a.beta = beta;
  a.bias = bias;
  a.parts = (uint4*)work;
  a.acc = acc;
  a.M = M;
  a.R = R;
  a.K = n_out;
  a.shared = ew_shared;
  return launch_fc<kRelax>(a, packed, n_in, nullptr, ew_out, (hipStream_t)stream);
}

extern "C" int vc_alpha_grad_step_split(const float* gE, const float* P, int64_t M, int R, int n,
                                        const float* lo_s, const float* up_s, const float* up_t,
                                        int p_shared, const void* packed_t,
                                        const float* bias_next, int n_next, float* g_out,
                                        void* work, vc_stream_t stream) {
  if (!gE || !P || !lo_s || !up_s || !up_t || !g_out || bad_args(M, R, n, n_next, packed_t, work))
    return VC_ERR_ARG;
  RowArgs a{};
  a.x = gE;
  a.P = P;
  a.s0 = lo_s;
  a.s1 = up_s;
  a.s2 = up_t;
  a.parts = (uint4*)work;
  a.M = M;
  a.R = R;
  a.K = n;
  a.shared = p_shared;
  return launch_fc<kGradStep>(a, packed_t, n_next, bias_next, g_out, (hipStream_t)stream);
}

extern "C" int vc_alpha_grad_input_split(const float* A, const float* xl, const float* xh,
                                         int64_t M, int R, int n_in, const void* packed_t,
                                         const float* bias0, int n1, float* g_out, void* work,
                                         vc_stream_t stream) {
  if (!A || !xl || !xh || !g_out || bad_args(M, R, n_in, n1, packed_t, work)) return VC_ERR_ARG;
  RowArgs a{};
  a.x = A;
  a.s0 = xl;
  a.s1 = xh;
  a.parts = (uint4*)work;
  a.M = M;
  a.R = R;
  a.K = n_in;
  return launch_fc<kGradInput>(a, packed_t, n1, bias0, g_out, (hipStream_t)stream);
}
