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
  float* out;         // (M, N); domains: (domains, N, ld), M of its columns
  int64_t M;          // rows; domains: of each
  int N, nkc, ntn, mt16;  // mt16: row tiles; domains: of each
  int64_t tiles;
  FastDiv f_ntn;
  int64_t ld;
  FastDiv f_dom;  // domains: row blocks of each; images: pixels
  float* out2;    // images: the upper bounds
};

// Where the rows' results go: (M, N); many domains' rows, each stored
// transposed; the pixels of images, stored by channel, the intervals' centres
// or, onto those, their radii.
enum Mode { kRows, kDomains, kCentres, kRadii };

// Value j of lane's eight in a packed tile: the sum of its three parts.
__device__ float part_sum(const uint4* p, int j) {
  float s = 0.f;
  for (int i = 2; i >= 0; --i)
    s += __builtin_bit_cast(float,
                            (uint32_t) reinterpret_cast<const uint16_t*>(p + 64 * i)[j] << 16);
  return s;
}

// One output, row r of row tile t, as the plain sum in 64 bits.
__device__ float plain_sum(const GemmArgs& a, int64_t t, int r, int n) {
  const uint4* A = a.Ap + t * a.nkc * kTileU + r;
  const uint4* B = a.Bp + (int64_t)(n >> 4) * a.nkc * kTileU + (n & 15);
  double s = 0.0;
  for (int kc = 0; kc < a.nkc; ++kc)
    for (int k = 0; k < FBK; ++k) {
      const int64_t o = (int64_t)kc * kTileU + 16 * (k >> 3);
      s += (double)part_sum(A + o, k & 7) * (double)part_sum(B + o, k & 7);
    }
  return (float)s;
}

// NJ: column tiles of a wave.
template <int MT, int MODE, int NJ = 2>
__global__ __launch_bounds__(FNT, 2) void k_fc_gemm(GemmArgs a) {
  constexpr int AU = MT * 2 * kTileU;       // 16-byte units of a double step's rows
  constexpr int NL = (AU + FNT - 1) / FNT;  // of them per thread
  constexpr int Q = MT >= 2 ? 2 : 1;        // row tiles at a time
  constexpr int NG = MT / Q;
  __shared__ __align__(16) u4 lds[2][NL * FNT];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int64_t w = vcg::xcd_tile(blockIdx.x, a.tiles);
  const int tb = (int)a.f_ntn.div((uint32_t)w);
  const int tn = (int)(w - (int64_t)tb * a.ntn);
  const int dom = MODE == kDomains ? (int)a.f_dom.div((uint32_t)tb) : 0;
  const int tm = MODE == kDomains ? tb - dom * (int)a.f_dom.d : tb;
  const int64_t t0 = MODE == kDomains ? (int64_t)dom * a.mt16 : 0;  // the domain's first row tile

  // this thread's units of each double step's rows (a row tile's two steps lie
  // together); past the last row tile the last one again, not stored
  const u4* A[NL];
#pragma unroll
  for (int i = 0; i < NL; ++i) {
    const int u = min(tid + i * FNT, AU - 1);
    const int t = min(tm * MT + u / (2 * kTileU), a.mt16 - 1);
    A[i] = reinterpret_cast<const u4*>(a.Ap) + (t0 + t) * a.nkc * kTileU + u % (2 * kTileU);
  }
  // this wave's column tiles, likewise
  const int c0 = (tn * 4 + wv) * NJ, nt16 = (a.N + 15) >> 4;
  const u4* B[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j)
    B[j] = reinterpret_cast<const u4*>(a.Bp) + (int64_t)min(c0 + j, nt16 - 1) * a.nkc * kTileU +
           lane;

  v4f acc[MT][NJ], small[MT][NJ], z[MT][NJ];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[i][j] = small[i][j] = v4f{0.f, 0.f, 0.f, 0.f};

  // past the last step the last again: no branch, nothing waits for it
  const int steps = a.nkc >> 1;
  const auto load_rows = [&](int s, u4(&v)[NL]) {
    const int64_t o = (int64_t)min(s, steps - 1) * (2 * kTileU);
#pragma unroll
    for (int i = 0; i < NL; ++i) v[i] = A[i][o];
  };
  const auto load_cols = [&](int kc, u4(&v)[NJ][3]) {
    const int64_t o = (int64_t)min(kc, a.nkc - 1) * kTileU;
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int p = 0; p < 3; ++p) v[j][p] = B[j][o + 64 * p];
  };
  u4 rn[NL], b[2][NJ][3];
  load_rows(0, rn);
  load_cols(0, b[0]);
#pragma unroll
  for (int i = 0; i < NL; ++i) lds[0][tid + i * FNT] = rn[i];

  const auto step = [&](int s, int buf) {
    __syncthreads();  // this step's rows are laid down, the ones before are read
    load_cols(2 * s + 1, b[1]);
    load_rows(s + 1, rn);
    __builtin_amdgcn_sched_barrier(0);  // requested before the products, not where they are used
    const u4* from = lds[buf] + lane;
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
          for (int j = 0; j < NJ; ++j) {
            v4f& d = p == 5 ? z[i0 + i][j] : small[i0 + i][j];
            d = mfma_bf16(av[t & 1][i][kPartA[p]], b[hf][j][kPartB[p]],
                          p == 5 && hf == 0 ? v4f{0.f, 0.f, 0.f, 0.f} : d);
          }
      if (hf == 1) {
#pragma unroll
        for (int i = i0; i < i0 + Q; ++i)
#pragma unroll
          for (int j = 0; j < NJ; ++j) {
            const v4f t2 = acc[i][j] + z[i][j];
            small[i][j] += z[i][j] - (t2 - acc[i][j]);
            acc[i][j] = t2;
          }
      }
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < NL; ++i) lds[buf ^ 1][tid + i * FNT] = rn[i];
  };
  // two at a time: one's sums would be copied back at the loop's end
#pragma unroll 1
  for (int s = 0;; s += 2) {
    step(s, 0);
    if (s + 1 == steps) break;
    step(s + 1, 1);
    if (s + 2 == steps) break;
  }

  const int g = lane >> 4, r = lane & 15;
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const int n = (c0 + j) * 16 + r;
    if (n >= a.N) continue;
    const float b = a.bias ? a.bias[n] : 0.f;
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const int64_t m0 = (int64_t)tm * MT * 16 + 16 * i + 4 * g;
      float v[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        v[q] = acc[i][j][q] + small[i][j][q];
        // an infinity or NaN among the values: the plain sum
        if (!finite(v[q]) && m0 + q < a.M)
          v[q] = plain_sum(a, t0 + tm * MT + i, 4 * g + q, n);
        if (a.bias) v[q] = v[q] + b;
      }
      typedef float v4u __attribute__((ext_vector_type(4), aligned(4)));
      if (MODE == kDomains) {
        float* o = a.out + ((int64_t)dom * a.N + n) * a.ld + m0;
        if (m0 + 4 <= a.M) {
          *reinterpret_cast<v4u*>(o) = v4u{v[0], v[1], v[2], v[3]};
          continue;
        }
#pragma unroll
        for (int q = 0; q < 4; ++q)
          if (m0 + q < a.M) o[q] = v[q];
        continue;
      }
      if (MODE == kCentres || MODE == kRadii) {
        const uint32_t npx = a.f_dom.d;
        const int64_t img = a.f_dom.div((uint32_t)m0);
        const int64_t at = (img * a.N + n) * npx + (m0 - img * npx);
        if (m0 + 4 <= a.M && m0 - img * npx + 4 <= npx) {
          v4u* const o = reinterpret_cast<v4u*>(a.out + at);
          v4u x = v4u{v[0], v[1], v[2], v[3]};
          if (MODE == kRadii) {
            const v4u c = *o;
            *reinterpret_cast<v4u*>(a.out2 + at) = c + x;
            x = c - x;
          }
          *o = x;
          continue;
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          if (m0 + q >= a.M) continue;
          const int64_t im = a.f_dom.div((uint32_t)(m0 + q));
          const int64_t o = (im * a.N + n) * npx + (m0 + q - im * npx);
          if (MODE == kRadii) {
            const float c = a.out[o];
            a.out2[o] = c + v[q];
            v[q] = c - v[q];
          }
          a.out[o] = v[q];
        }
        continue;
      }
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (m0 + q < a.M) a.out[(m0 + q) * a.N + n] = v[q];
    }
  }
}

// The interval forward of a conv (verify_zono_bnb.py:1114-1123): centres and
// radii of the pixels it reads, as rows of its products with the kernel and its
// magnitudes.  Row = output pixel m, value k = (channel, tap) of the kernel.  A
// wave forms 16 pixels' parts, both kinds from one load of the bounds (HBM
// bound, by the parts written: 1.2 GB in 385 us).  Three convs of 512 32x32
// images to 64 channels, the whole forward 1465 -> 1141 us (32 -> 64 and 64 ->
// 64, 4x4: the gathering product 1017 us, now 680).
struct ConvRows {
  const float *l, *h;
  int C_in, H, W, kh, kw, sh, sw, ph, pw, Wo, K, nkc;
  int64_t M;
  FastDiv f_px, f_wo, f_taps, f_kw;
  uint4 *mid, *rad;
};
__global__ __launch_bounds__(FNT) void k_conv_rows(ConvRows a) {
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, g = lane >> 4, r = lane & 15;
  const int64_t m0 = (int64_t)blockIdx.x * 16;
  const uint32_t m = (uint32_t)(m0 + r < a.M ? m0 + r : a.M - 1);
  const int64_t img = a.f_px.div(m);
  const int px = (int)(m - img * a.f_px.d);
  const int oy = (int)a.f_wo.div((uint32_t)px), ox = px - oy * a.Wo;
  const int y0 = oy * a.sh - a.ph, x0 = ox * a.sw - a.pw;
  const float* const pl = a.l + img * a.C_in * a.H * a.W;
  const float* const ph = a.h + img * a.C_in * a.H * a.W;
  const int64_t out = (int64_t)blockIdx.x * a.nkc * kTileU + lane;
  for (int kc = wv; kc < a.nkc; kc += 4) {
    float mid[8], rad[8];
    int k = kc * FBK + 8 * g;
    int ci = (int)a.f_taps.div((uint32_t)k), t = k - ci * (int)a.f_taps.d;
    int ky = (int)a.f_kw.div((uint32_t)t), kx = t - ky * a.kw;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int y = y0 + ky, x = x0 + kx;
      const bool in = k + j < a.K && (unsigned)y < (unsigned)a.H && (unsigned)x < (unsigned)a.W;
      const int o = in ? (ci * a.H + y) * a.W + x : 0;
      const float l = pl[o], h = ph[o];
      mid[j] = in ? (l + h) / 2.f : 0.f;
      rad[j] = in ? (h - l) / 2.f : 0.f;
      // the next tap
      const bool row = ++kx == a.kw;
      kx = row ? 0 : kx;
      ky += row ? 1 : 0;
      const bool chan = ky == a.kh;
      ky = chan ? 0 : ky;
      ci += chan ? 1 : 0;
    }
    uint4 p[3];
    uint4* o = a.mid + out + (int64_t)kc * kTileU;
    split8_all(mid, p[0], p[1], p[2]);
    o[0] = p[0];
    o[64] = p[1];
    o[128] = p[2];
    o = a.rad + out + (int64_t)kc * kTileU;
    split8_all(rad, p[0], p[1], p[2]);
    o[0] = p[0];
    o[64] = p[1];
    o[128] = p[2];
  }
}

// The zonotope's relu and the fc after it (verify_zono_bnb.py:3120-3211): the
// relu's slope scales the generators' rows, here in the pass that forms their
// parts, and its new generators are one neuron's each, so through the fc they
// are scaled columns of W and need no product.  784-1024x4-10, 512 boxes: the
// relu's pass over (B, n, K) and the fp32 product of all columns 83 ms, now 37
// (28 of them k_fc_gemm, at 150 TFLOP/s); 784-256x6-10, 64 boxes, the whole
// forward 1.76 -> 1.25 ms.
//
// Parts of the generators as rows: row = generator column j < cols of domain b,
// its values G[b][k][j] lam[b][k] over the neurons k, K of a neuron's values
// apart.  Four waves take 64 columns, each 16 of them: 256 bytes of a neuron's
// row at a time.
__global__ __launch_bounds__(FNT) void k_zono_rows(const float* G, const float* lam, int n, int K,
                                                   int cols, int mt16, int nkc, FastDiv f_blk,
                                                   uint4* parts) {
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, g = lane >> 4, r = lane & 15;
  const int64_t dom = f_blk.div((uint32_t)blockIdx.x);
  const int t = ((int)(blockIdx.x - dom * f_blk.d)) * 4 + wv;
  if (t >= mt16) return;
  const float* x = G + dom * n * (int64_t)K + min(16 * t + r, cols - 1);
  const float* l = lam ? lam + dom * n : nullptr;
  uint4* out = parts + (dom * mt16 + t) * nkc * kTileU + lane;
  for (int kc = blockIdx.y; kc < nkc; kc += gridDim.y) {
    const int k0 = kc * FBK + 8 * g;
    float e[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int k = min(k0 + j, n - 1);
      e[j] = x[(int64_t)k * K];
      if (l) e[j] = e[j] * l[k];
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) e[j] = k0 + j < n ? e[j] : 0.f;
    uint4 h, m, lo;
    split8_all(e, h, m, lo);
    uint4* const o = out + (int64_t)kc * kTileU;
    o[0] = h;
    o[64] = m;
    o[128] = lo;
  }
}

// A zonotope relu's slope and centre per neuron, and its new generators as a
// list per domain: neuron and size of each, in order (the operations of
// vc_zono_relu_apply).
__global__ void k_zono_lists(const float* c, const float* lo, const float* hi,
                             const int32_t* rank, int64_t rows, int n, int k_new, float* c_out,
                             float* lam_out, int32_t* idx, float* mu_out) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < rows;
       i += (int64_t)gridDim.x * blockDim.x) {
    const float l = lo[i], h = hi[i];
    const bool ust = l < 0.f && h > 0.f;
    const float lam = ust ? h / (h - l) : (h <= 0.f ? 0.f : 1.f);
    const float mu = ust ? (-h * l) / (2.f * (h - l)) : 0.f;
    lam_out[i] = lam;
    c_out[i] = lam * c[i] + mu;
    if (ust) {
      const int64_t b = i / n, o = b * k_new + rank[i];
      idx[o] = (int)(i - b * n);
      mu_out[o] = mu;
    }
  }
}

// Generators that are one neuron's, through an fc: scaled columns of W.
// G_out[b][o][k0 + j] = W[o][idx[j]] mu[j] for j < cnt[b], else zero.
constexpr int kColRows = 16;
__global__ __launch_bounds__(FNT) void k_zono_cols(const float* W, int n_out, int n, int k,
                                                   const int32_t* idx, int64_t idx_ld,
                                                   const float* mu, const float* xl,
                                                   const float* xh, const int32_t* cnt,
                                                   int64_t blocks, FastDiv f_j, FastDiv f_o,
                                                   float* out, int64_t ld) {
  for (int64_t blk = blockIdx.x; blk < blocks; blk += gridDim.x) {
    const uint32_t q = f_j.div((uint32_t)blk);
    const int64_t b = f_o.div(q);
    const int j = (int)(blk - (int64_t)q * f_j.d) * FNT + threadIdx.x;
    const int o0 = (int)(q - b * f_o.d) * kColRows;
    if (j >= k) continue;
    int i = 0;
    float m = 0.f;
    if (!cnt || j < cnt[b]) {
      i = idx[b * idx_ld + j];
      m = mu ? mu[b * idx_ld + j] : (xh[b * n + i] - xl[b * n + i]) / 2.f;
    }
    const bool has = !cnt || j < cnt[b];
    float* o = out + (b * n_out + o0) * ld + j;
    for (int r = 0; r < kColRows && o0 + r < n_out; ++r)
      o[r * ld] = has ? W[(int64_t)(o0 + r) * n + i] * m : 0.f;
  }
}

// One matrix' parts; and as many as a launch's arguments hold.
struct Pack {
  const float* W;
  uint4 *out, *out_abs;
  int K, N, trans, nkc;
  uint32_t block0;  // its first workgroup
};
constexpr int kPacks = 16;
struct Packs {
  Pack p[kPacks];
  int count;
};

// out[column tile][32-deep step][part][lane][8]: part of B[k][n] for
// k = 32 step + 8 (lane / 16) + j, n = 16 tile + lane % 16; zero past the ends.
// out_abs (or null): the same of |B|.  A launch takes 5 us whatever it packs up
// to a million weights, so a call's matrices go together (five of 256 x 256: 22
// us apart, 6 together).
__global__ __launch_bounds__(256) void k_fc_split_pack(Packs a) {
  int i = 0;
  while (i + 1 < a.count && blockIdx.x >= a.p[i + 1].block0) ++i;
  const Pack& m = a.p[i];
  const int64_t t = (int64_t)(blockIdx.x - m.block0) * 256 + threadIdx.x;
  const int64_t q = t >> 6;
  if (q >= (int64_t)((m.N + 15) >> 4) * m.nkc) return;
  const int lane = (int)(t & 63);
  const int kc = (int)(q % m.nkc), n = (int)(q / m.nkc) * 16 + (lane & 15);
  const int k0 = kc * FBK + 8 * (lane >> 4);
  float v[8];
#pragma unroll
  for (int j = 0; j < 8; ++j)
    v[j] = n < m.N && k0 + j < m.K
               ? (m.trans ? m.W[(int64_t)n * m.K + k0 + j] : m.W[(int64_t)(k0 + j) * m.N + n])
               : 0.f;
  uint4 h, md, l;
  split8_all(v, h, md, l);
  uint4* o = m.out + q * kTileU + lane;
  o[0] = h;
  o[64] = md;
  o[128] = l;
  if (!m.out_abs) return;
#pragma unroll
  for (int j = 0; j < 8; ++j) v[j] = fabsf(v[j]);
  split8_all(v, h, md, l);
  o = m.out_abs + q * kTileU + lane;
  o[0] = h;
  o[64] = md;
  o[128] = l;
}

int launch_pack(Packs& a, hipStream_t st) {
  int64_t blocks = 0;
  for (int i = 0; i < a.count; ++i) {
    Pack& m = a.p[i];
    m.nkc = 2 * ((m.K + 2 * FBK - 1) / (2 * FBK));
    m.block0 = (uint32_t)blocks;
    blocks += ((int64_t)((m.N + 15) / 16) * m.nkc * 64 + 255) / 256;
    if (blocks >= (int64_t(1) << 31)) return VC_ERR_UNSUPPORTED;
  }
  hipLaunchKernelGGL(k_fc_split_pack, dim3((unsigned)blocks), dim3(256), 0, st, a);
  VC_LAUNCH_CHECK();
  return VC_OK;
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
  // The tallest row block that gives every CU a tile, or four of them: two fit
  // a CU, and a third round half empty costs more than the weights read twice
  // (64 and 32 rows: 4,608 x 1024 x 1024, 576 tiles, 84 and 78 us, 18,432 x 256 x
  // 256 38 and 34; 18,432 x 1024 x 1024, 2,304 tiles, 251 and 276).
  const int64_t cus = vcm::cu_count();
  const auto blocks = [&](int mt) { return (mt16 + mt - 1) / mt * b.ntn; };
  const int mt = blocks(4) >= 4 * cus ? 4 : (blocks(2) >= cus ? 2 : 1);
  b.tiles = blocks(mt);
  if (a.M >= (int64_t(1) << 31) || b.tiles >= (int64_t(1) << 31)) return VC_ERR_UNSUPPORTED;
  bool vec = a.K % 4 == 0;
  for (const float* p : {a.x, a.P, a.s0, a.s1, a.s2, a.beta, a.bias}) vec = vec && aligned16(p);
  if (vec)
    hipLaunchKernelGGL((k_fc_rows<FORM, true>), dim3((unsigned)mt16), dim3(FNT), 0, st, a);
  else
    hipLaunchKernelGGL((k_fc_rows<FORM, false>), dim3((unsigned)mt16), dim3(FNT), 0, st, a);
  VC_LAUNCH_CHECK();
  const dim3 grid((unsigned)b.tiles);
  if (mt == 4) hipLaunchKernelGGL((k_fc_gemm<4, kRows>), grid, dim3(FNT), 0, st, b);
  if (mt == 2) hipLaunchKernelGGL((k_fc_gemm<2, kRows>), grid, dim3(FNT), 0, st, b);
  if (mt == 1) hipLaunchKernelGGL((k_fc_gemm<1, kRows>), grid, dim3(FNT), 0, st, b);
  VC_LAUNCH_CHECK();
  return VC_OK;
}

template <int MODE>
void launch_conv(const GemmArgs& b, int mt, int nj, hipStream_t st) {
  const dim3 grid((unsigned)b.tiles);
  if (mt == 4 && nj == 1) hipLaunchKernelGGL((k_fc_gemm<4, MODE, 1>), grid, dim3(FNT), 0, st, b);
  if (mt == 4 && nj == 2) hipLaunchKernelGGL((k_fc_gemm<4, MODE, 2>), grid, dim3(FNT), 0, st, b);
  if (mt == 2 && nj == 1) hipLaunchKernelGGL((k_fc_gemm<2, MODE, 1>), grid, dim3(FNT), 0, st, b);
  if (mt == 2 && nj == 2) hipLaunchKernelGGL((k_fc_gemm<2, MODE, 2>), grid, dim3(FNT), 0, st, b);
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
  Packs a{{{W, (uint4*)out, nullptr, K, N, trans}}, 1};
  return launch_pack(a, (hipStream_t)stream);
}

extern "C" int vc_fc_split_pack_abs(const float* W, int K, int N, int trans, void* out,
                                    void* out_abs, vc_stream_t stream) {
  if (!W || !out || !out_abs || K <= 0 || N <= 0 || !aligned16(out) || !aligned16(out_abs))
    return VC_ERR_ARG;
  Packs a{{{W, (uint4*)out, (uint4*)out_abs, K, N, trans}}, 1};
  return launch_pack(a, (hipStream_t)stream);
}

extern "C" int vc_fc_split_pack_many(const float* const* W, const int32_t* K, const int32_t* N,
                                     const int32_t* trans, void* const* out, int count,
                                     vc_stream_t stream) {
  if (count < 0 || (count > 0 && (!W || !K || !N || !trans || !out))) return VC_ERR_ARG;
  for (int i = 0; i < count; ++i)
    if (!W[i] || !out[i] || K[i] <= 0 || N[i] <= 0 || !aligned16(out[i])) return VC_ERR_ARG;
  for (int i0 = 0; i0 < count; i0 += kPacks) {
    Packs a{};
    a.count = count - i0 < kPacks ? count - i0 : kPacks;
    for (int i = 0; i < a.count; ++i)
      a.p[i] =
          Pack{W[i0 + i], (uint4*)out[i0 + i], nullptr, K[i0 + i], N[i0 + i], trans[i0 + i]};
    const int rc = launch_pack(a, (hipStream_t)stream);
    if (rc != VC_OK) return rc;
  }
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

extern "C" int vc_zono_relu_lists(const float* c, const float* lo, const float* hi,
                                  const int32_t* rank, int64_t B, int n, int k_new, float* c_out,
                                  float* lam, int32_t* idx, float* mu, vc_stream_t stream) {
  if (!c || !lo || !hi || !rank || !c_out || !lam || B < 0 || n <= 0 || k_new < 0 ||
      (k_new > 0 && (!idx || !mu)))
    return VC_ERR_ARG;
  if (B == 0) return VC_OK;
  hipLaunchKernelGGL(k_zono_lists, dim3(vc_blocks(B * n, FNT)), dim3(FNT), 0, (hipStream_t)stream,
                     c, lo, hi, rank, B * n, n, k_new, c_out, lam, idx, mu);
  VC_LAUNCH_CHECK();
  return VC_OK;
}

extern "C" int vc_zono_fc_cols(const float* W, int n_out, int n, int64_t B, int k,
                               const int32_t* idx, int64_t idx_ld, const float* mu,
                               const float* xl, const float* xh, const int32_t* cnt, int k0,
                               int64_t ld, float* G_out, vc_stream_t stream) {
  if (B < 0 || n <= 0 || n_out <= 0 || k < 0 || k0 < 0 || ld < (int64_t)k0 + k) return VC_ERR_ARG;
  if (B == 0 || k == 0) return VC_OK;
  if (!W || !idx || !G_out || (!mu && (!xl || !xh))) return VC_ERR_ARG;
  const int nj = (k + FNT - 1) / FNT, no = (n_out + kColRows - 1) / kColRows;
  const int64_t blocks = B * nj * no;
  if (blocks >= (int64_t(1) << 31)) return VC_ERR_UNSUPPORTED;
  hipLaunchKernelGGL(k_zono_cols, dim3((unsigned)blocks), dim3(FNT), 0, (hipStream_t)stream, W,
                     n_out, n, k, idx, idx_ld, mu, xl, xh, cnt, blocks, FastDiv::make(nj),
                     FastDiv::make(no), G_out + k0, ld);
  VC_LAUNCH_CHECK();
  return VC_OK;
}

extern "C" int vc_zono_fc_split(const float* G, const float* lam, int64_t B, int n, int K,
                                const void* packed_t, int n_out, int64_t ld, float* G_out,
                                void* work, int64_t work_bytes, vc_stream_t stream) {
  if (B < 0 || n <= 0 || n_out <= 0 || K < 0 || ld < K) return VC_ERR_ARG;
  if (B == 0 || K == 0) return VC_OK;
  if (!G || !packed_t || !G_out || !work || !aligned16(packed_t) || !aligned16(work))
    return VC_ERR_ARG;
  const hipStream_t st = (hipStream_t)stream;
  GemmArgs b{};
  b.nkc = 2 * ((n + 2 * FBK - 1) / (2 * FBK));
  b.Ap = (const uint4*)work;
  b.Bp = (const uint4*)packed_t;
  b.N = n_out;
  b.ld = ld;
  b.ntn = (n_out + FBN - 1) / FBN;
  b.f_ntn = FastDiv::make((uint32_t)b.ntn);
  const int ny = b.nkc < 4 ? b.nkc : 4;
  // domains whose parts the buffer holds, or columns of one
  int64_t step = work_bytes / vc_fc_split_pack_bytes(n, K), cols = K;
  if (step < 1) {
    step = 1;
    cols = work_bytes / vc_fc_split_pack_bytes(n, 16) / 4 * 64;
    if (cols < 64) return VC_ERR_ARG;
  }
  for (int64_t j0 = 0; j0 < K; j0 += cols) {
    const int kc = (int)(K - j0 < cols ? K - j0 : cols);
    b.M = kc;
    b.mt16 = (kc + 15) / 16;
    const int blk = (b.mt16 + 3) / 4;
    b.f_dom = FastDiv::make((uint32_t)blk);
    // domains whose tiles a launch counts
    const int64_t most = (((int64_t)1 << 31) - 1) / ((int64_t)blk * b.ntn);
    if (most < 1) return VC_ERR_ARG;
    if (step > most) step = most;
    for (int64_t b0 = 0; b0 < B; b0 += step) {
      const int64_t cnt = B - b0 < step ? B - b0 : step;
      hipLaunchKernelGGL(k_zono_rows, dim3((unsigned)(cnt * blk), ny), dim3(FNT), 0, st,
                         G + b0 * n * K + j0, lam ? lam + b0 * n : nullptr, n, K, kc, b.mt16,
                         b.nkc, b.f_dom, (uint4*)work);
      VC_LAUNCH_CHECK();
      b.out = G_out + b0 * n_out * ld + j0;
      b.tiles = cnt * blk * b.ntn;
      hipLaunchKernelGGL((k_fc_gemm<4, kDomains>), dim3((unsigned)b.tiles), dim3(FNT), 0, st, b);
      VC_LAUNCH_CHECK();
    }
  }
  return VC_OK;
}

extern "C" int vc_ibp_conv_split(const float* l, const float* h, int64_t B, int C_in, int H, int W,
                                 const void* packed_t, const void* packed_abs_t,
                                 const float* bias, int C_out, int kh, int kw, int sh, int sw,
                                 int ph, int pw, int H_out, int W_out, float* lo, float* hi,
                                 void* work, int64_t work_bytes, vc_stream_t stream) {
  if (B < 0 || C_in <= 0 || H <= 0 || W <= 0 || C_out <= 0 || kh <= 0 || kw <= 0 || sh <= 0 ||
      sw <= 0 || ph < 0 || pw < 0 || H_out <= 0 || W_out <= 0)
    return VC_ERR_ARG;
  if (B == 0) return VC_OK;
  if (!l || !h || !packed_t || !packed_abs_t || !lo || !hi || !work || !aligned16(packed_t) ||
      !aligned16(packed_abs_t) || !aligned16(work))
    return VC_ERR_ARG;
  const int64_t npx = (int64_t)H_out * W_out, K = (int64_t)C_in * kh * kw;
  if (npx >= 1 << 24 || K >= 1 << 24 || (int64_t)H * W >= 1 << 28 ||
      (int64_t)C_in * H * W >= (int64_t(1) << 31))
    return VC_ERR_UNSUPPORTED;
  const hipStream_t st = (hipStream_t)stream;
  ConvRows a{l, h, C_in, H, W, kh, kw, sh, sw, ph, pw, W_out, (int)K};
  a.nkc = 2 * (((int)K + 2 * FBK - 1) / (2 * FBK));
  a.f_px = FastDiv::make((uint32_t)npx);
  a.f_wo = FastDiv::make((uint32_t)W_out);
  a.f_taps = FastDiv::make((uint32_t)(kh * kw));
  a.f_kw = FastDiv::make((uint32_t)kw);
  // images whose parts the buffer holds, centres and radii, within 32-bit rows
  const int64_t per = vc_fc_split_pack_bytes(K, npx);
  int64_t step = work_bytes / (2 * per);
  const int64_t most = (((int64_t)1 << 31) - 64) / npx;
  if (step > most) step = most;
  if (step < 1) return VC_ERR_ARG;
  // one column tile a wave where two would leave half of the waves without
  const int nj = C_out <= 64 ? 1 : 2;
  const int64_t cus = vcm::cu_count();
  GemmArgs b{};
  b.nkc = a.nkc;
  b.N = C_out;
  b.ntn = (C_out + 64 * nj - 1) / (64 * nj);
  b.f_ntn = FastDiv::make((uint32_t)b.ntn);
  b.f_dom = a.f_px;
  for (int64_t b0 = 0; b0 < B; b0 += step) {
    const int64_t cnt = B - b0 < step ? B - b0 : step;
    a.l = l + b0 * C_in * H * W;
    a.h = h + b0 * C_in * H * W;
    a.M = b.M = cnt * npx;
    b.mt16 = (int)((a.M + 15) / 16);
    a.mid = (uint4*)work;
    a.rad = a.mid + (int64_t)b.mt16 * a.nkc * kTileU;
    hipLaunchKernelGGL(k_conv_rows, dim3((unsigned)b.mt16), dim3(FNT), 0, st, a);
    VC_LAUNCH_CHECK();
    // 32 pixels a row block where 64 give fewer than three tiles for two CUs
    // (two fit a CU).  Both kinds of tiles, us: 256 tiles of 64 (16,384 pixels)
    // of 32 and 64 channels, 5x5, onto 33 170 and 149, onto 64 170 and 154, 3x3
    // onto 64 58 and 56; 304 of 32, 5x5, onto 128 452 and 407; 448 of 64, 3x3,
    // onto 128 1,150 and 1,209; a few boxes of any of these 77 and 62.
    const auto blocks = [&](int mt) { return (int64_t)((b.mt16 + mt - 1) / mt) * b.ntn; };
    const int mt = 2 * blocks(4) >= 3 * cus ? 4 : 2;
    b.tiles = blocks(mt);
    if (b.tiles >= (int64_t(1) << 31)) return VC_ERR_UNSUPPORTED;
    b.out = lo + b0 * C_out * npx;
    b.out2 = hi + b0 * C_out * npx;
    b.Ap = a.mid;
    b.Bp = (const uint4*)packed_t;
    b.bias = bias;
    launch_conv<kCentres>(b, mt, nj, st);
    VC_LAUNCH_CHECK();
    b.Ap = a.rad;
    b.Bp = (const uint4*)packed_abs_t;
    b.bias = nullptr;
    launch_conv<kRadii>(b, mt, nj, st);
    VC_LAUNCH_CHECK();
  }
  return VC_OK;
}
