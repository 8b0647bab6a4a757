// The transposed convolution of a CROWN backward step on the bf16 matrix
// cores (vc_split.h), with the ReLU relaxation before it in its loads:
//   e = pos(x) lo_s + neg(x) up_s [+ beta], acc += neg(x) . up_t + e . bias,
//   out = conv_transpose2d(e)
// (verify_zono_bnb.py:4409-4453 and 4568-4593).
//
// A workgroup takes G source images (one image, or one band of its rows, where
// they are large) and 32 source channels at a time: it loads, relaxes and
// splits each value once and lays the three parts down pixel by pixel with the
// channels together, so that every kernel tap is the same LDS array read at
// another pixel offset.  (An implicit GEMM gathers and splits each value once
// per tap, sixteen times for a 4x4 kernel.)  Outputs run by output parity
// (y mod sh, x mod sw): a class takes the taps ky = k0 + sh ty only, from
// source row yy + c - ty, so no zero tap is multiplied; the four waves take
// the four classes of a stride-2 kernel, or quarters of a stride-1 one.  A
// wave holds MT x NTW tiles of 16 channels x 16 pixels; each tap's weights
// (packed in operand order by vc_conv_split_pack) are read from L2 once for
// all of its pixels.
//
// Measured at 16,384 rows of 64 domains, relaxation included, against the
// implicit fp32 GEMM after a relaxation pass: 64 -> 32 channels, 4x4 stride 2
// onto 32x32, 6.89 -> 2.03 ms (136 TFLOP/s of the convolution); 64 -> 64 onto
// 16x16, 2.66 -> 0.91 ms (150); at 9 rows 50 -> 47 us and 30 -> 27.  Relative to
// 64 bits the results are 6.7e-8 off in the 2-norm (the fp32 GEMM: 8.3e-8).
// The 3-channel first layer stays with the GEMM and fold (vc_conv.hip): its 16
// output rows here hold 3, and 16,384 rows take 2.3 ms against 0.9.
#include "vc_gemm_core.h"
#include "vc_mlp_common.h"
#include "vc_split.h"

namespace {

using namespace vcs;
using vcg::FastDiv;

constexpr int CNT = 256;       // threads
constexpr int CK = 32;         // channels per chunk: one MFMA step
constexpr int PTB = 2 * CK;        // LDS bytes per pixel and part
constexpr int PXB = 3 * PTB + 16;  // per pixel: 208, so that 16 consecutive pixels start
                                   // on 16 distinct groups of four banks
constexpr int kMaxLds = 78 * 1024;  // two workgroups per CU

struct SplitArgs {
  const float* ew;  // R rows (shared) or M rows of C_out Hs Ws
  int64_t M, R;
  int shared;
  const float *ls, *us, *ut, *beta;  // (M / R, C_out Hi Wi) or null
  const float* K;                    // (C_out, C_in, kh, kw): the exact form's
  const uint4* A;                    // packed parts
  const float* bias;
  float* out;  // (M, C_in, H, W)
  float* acc;
  int C_out, Hs, Ws, Hi, Wi, C_in, H, W, kh, kw, sh, sw, ph, pw;
  // plan
  int G, TI;               // images per workgroup, threads per image
  int NB, YB, Hb;          // bands, class rows per band, source rows in LDS
  int cminy, Ty, Tx;       // smallest row offset of a class, taps per class
  int P0, IMG, Wp;         // LDS pixel of (image 0, row 0, column 0), strides
  int npix;                // LDS pixels
  int nchunk, classes, NG, gs, passes, cib, MTp;
  int Hc, Wc, comp;
  int64_t n_tiles;
  FastDiv f_cw, f_wc, f_npx, f_ws, f_cib, f_R, f_sw, f_ng;
};

// The kernel's arguments read again, where a phase of it needs them: all of
// them held over the main loop would spill.
__device__ __forceinline__ const SplitArgs& reread() {
  typedef const __attribute__((address_space(4))) SplitArgs* Args;
  Args p = (Args)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  return *(const SplitArgs*)p;
}

// One output as the plain sum of relaxed values times taps, in 64 bits.
template <int RL>
__device__ __forceinline__ float plain_sum(const SplitArgs& a, int64_t m, int ci, int y, int x) {
  const int64_t d = m / a.R;
  const float* s = a.ew + (a.shared ? m - d * a.R : m) * a.C_out * a.Hs * a.Ws;
  double sum = 0.0;
  for (int ky = 0; ky < a.kh; ++ky) {
    const int ty = y + a.ph - ky, qy = ty / a.sh;
    if (ty < 0 || qy * a.sh != ty || qy >= a.Hs) continue;
    for (int kx = 0; kx < a.kw; ++kx) {
      const int tx = x + a.pw - kx, qx = tx / a.sw;
      if (tx < 0 || qx * a.sw != tx || qx >= a.Ws) continue;
      for (int co = 0; co < a.C_out; ++co) {
        const int64_t i = ((d * a.C_out + co) * a.Hi + qy) * a.Wi + qx;
        float e = s[((int64_t)co * a.Hs + qy) * a.Ws + qx];
        if (RL > 0) e = e * (e < 0.f ? a.us[i] : a.ls[i]);
        if (RL > 0 && a.beta) e = e + a.beta[i];
        sum += (double)e * (double)a.K[(((int64_t)co * a.C_in + ci) * a.kh + ky) * a.kw + kx];
      }
    }
  }
  return (float)sum;
}

template <int MT, int NTW, int RL, bool COMP>
__global__ __launch_bounds__(CNT, 2) void k_conv_split(SplitArgs a) {
  constexpr int NB = MT == 4 || NTW == 1 ? 1 : 2;  // column tiles at a time
  extern __shared__ __align__(16) char lds[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kg = lane >> 4, r = lane & 15;
  // the pixels around and between the images stay zero
  for (int i = tid; i < a.npix * (PXB / 16); i += CNT)
    reinterpret_cast<uint4*>(lds)[i] = uint4{0u, 0u, 0u, 0u};
  const int g = tid / a.TI, tl = tid - g * a.TI;

  for (int64_t blk = blockIdx.x; blk < a.n_tiles; blk += gridDim.x) {
    const uint32_t w = (uint32_t)vcg::xcd_tile(blk, a.n_tiles);
    const uint32_t ig = a.f_cib.div(w);
    const int cb = (int)(w - ig * a.cib);
    const int64_t m0 = (int64_t)ig * a.G;
    double part = 0.0;

    for (int band = 0; band < a.NB; ++band) {
      const int yy0 = band * a.YB;
      const int ycnt = min(a.YB, a.Hc - yy0);
      const int qa = a.NB > 1 ? yy0 + a.cminy - (a.Ty - 1) : 0;
      const int cols = a.G * ycnt * a.Wc;
      for (int pass = 0; pass < a.passes; ++pass) {
        const int item = pass * 4 + wv;
        const int cls0 = (int)a.f_ng.div((uint32_t)item);
        const bool live = cls0 < a.classes;
        const int cls = live ? cls0 : 0;
        const int py = (int)a.f_sw.div((uint32_t)cls), px = cls - py * a.sw;
        const int k0y = (py + a.ph) % a.sh, k0x = (px + a.pw) % a.sw;
        const int c0 = (item - cls0 * a.NG) * a.gs * 16;
        const int ntl = live && c0 < cols ? min(a.gs, (cols - c0 + 15) >> 4) : 0;
        int base[NTW];
        {
          const int cy = (py + a.ph - k0y) / a.sh, cx = (px + a.pw - k0x) / a.sw;
#pragma unroll
          for (int nt = 0; nt < NTW; ++nt) {
            const int c = min(c0 + 16 * nt + r, cols - 1);  // past the end: any pixel, not stored
            const int img = (int)a.f_cw.div((uint32_t)c);
            const int rem = c - img * a.Hc * a.Wc;
            const int yy = (int)a.f_wc.div((uint32_t)rem), xx = rem - yy * a.Wc;
            base[nt] = (a.P0 + img * a.IMG + (yy0 + yy + cy - qa) * a.Wp + xx + cx) * PXB + 16 * kg;
          }
        }
        v4f acc[MT][NTW];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
          for (int nt = 0; nt < NTW; ++nt) acc[mt][nt] = v4f{0.f, 0.f, 0.f, 0.f};
        // COMP: what rounding took from each sum, added to the next step's
        v4f lost[COMP ? MT : 1][COMP ? NTW : 1];
#pragma unroll
        for (int mt = 0; mt < (COMP ? MT : 1); ++mt)
#pragma unroll
          for (int nt = 0; nt < (COMP ? NTW : 1); ++nt) lost[mt][nt] = v4f{0.f, 0.f, 0.f, 0.f};

        const int nchunk = a.nchunk;
#pragma unroll 1
        for (int ch = 0; ch < nchunk; ++ch) {
          __syncthreads();  // the chunk before has been read
          if (pass == 0 || nchunk > 1) {
            const SplitArgs& b = reread();
            const int64_t m = m0 + g;
            const bool ok = m < b.M;
            const int npx = b.Hb * b.Ws, nu = 4 * npx, TI = b.TI;
            const int64_t n_e = (int64_t)b.C_out * b.Hs * b.Ws;
            const int64_t n_i = (int64_t)b.C_out * b.Hi * b.Wi;
            // buffers from the tile's first image (shared rows: from the first
            // row) and first domain on, this thread's image by its byte offset
            const uint32_t dom0 = b.f_R.div((uint32_t)m0);
            const uint32_t dom = ok ? b.f_R.div((uint32_t)m) : dom0;
            const int64_t xb = b.shared ? 0 : m0 * n_e, ib = (int64_t)dom0 * n_i;
            const uint32_t gx = 4 * (uint32_t)((b.shared ? (ok ? m - dom * b.R : 0) : g) * n_e);
            const uint32_t gi = 4 * (uint32_t)((dom - dom0) * n_i);
            const Buf bx = buffer(b.ew + xb, ((b.shared ? b.R : b.M) * n_e - xb) * 4);
            const int64_t left = (b.M / b.R * n_i - ib) * 4;
            const Buf bl = buffer(b.ls + ib, RL > 0 ? left : 0);
            const Buf bu = buffer(b.us + ib, RL > 0 ? left : 0);
            const Buf bt = buffer(b.ut + ib, RL > 0 ? left : 0);
            const Buf bb = buffer(b.beta + ib, RL > 0 && b.beta ? left : 0);
            const int sx = 4 * b.Hs * b.Ws, si = 4 * b.Hi * b.Wi;
            // source rows whose constant terms this band counts
            const bool count = pass == 0 && cb == 0;
            const int own0 = band == 0 ? 0 : yy0;
            const int own1 = band == b.NB - 1 ? b.Hs : yy0 + b.YB;
            char* const img = lds + (b.P0 + g * b.IMG) * PXB;
#pragma unroll 1
            for (int j = tl; j < nu; j += TI) {
              const int ukg = (int)b.f_npx.div((uint32_t)j), up = j - ukg * npx;
              const int rr = (int)b.f_ws.div((uint32_t)up), x = up - rr * b.Ws;
              const int q = qa + rr, co0 = ch * CK + 8 * ukg;
              const bool in = ok && (unsigned)q < (unsigned)b.Hs && co0 < b.C_out;
              // outside the image: past the buffer, which reads as zero
              const uint32_t xo = in ? gx + 4 * ((co0 * b.Hs + q) * b.Ws + x) : kOut;
              const uint32_t io = in ? gi + 4 * ((co0 * b.Hi + q) * b.Wi + x) : kOut;
              float e[8], lv[8], uv[8], tv[8], bv[8];
#pragma unroll
              for (int i = 0; i < 8; ++i) {
                const bool has = co0 + i < b.C_out;
                const uint32_t ioi = has ? io : kOut;
                e[i] = ldb(bx, has ? xo : kOut, i * sx);
                if (RL > 0) {
                  lv[i] = ldb(bl, ioi, i * si);
                  uv[i] = ldb(bu, ioi, i * si);
                  tv[i] = ldb(bt, ioi, i * si);
                }
              }
              if (RL > 0 && b.beta) {
#pragma unroll
                for (int i = 0; i < 8; ++i) bv[i] = ldb(bb, co0 + i < b.C_out ? io : kOut, i * si);
              } else {
#pragma unroll
                for (int i = 0; i < 8; ++i) bv[i] = 0.f;
              }
              double pd = 0.0;
#pragma unroll
              for (int i = 0; i < 8; ++i) {
                const bool has = co0 + i < b.C_out;
                float v = e[i], p = 0.f;
                if (RL > 0) {
                  // pos(x) lo_s + neg(x) up_s: one of the two parts is zero
                  const bool ng = v < 0.f;
                  p = (ng ? v : 0.f) * tv[i];
                  v = v * (ng ? uv[i] : lv[i]);
                  v = v + bv[i];
                }
                p += v * (b.bias && has ? b.bias[co0 + i] : 0.f);
                e[i] = has ? v : 0.f;
                pd += (double)(has ? p : 0.f);
              }
              if (count && q >= own0 && q < own1) part += pd;
              uint4 h, md, l;
              split8(e, h, md, l);
              char* const d = img + (rr * b.Wp + x) * PXB + 16 * ukg;
              *reinterpret_cast<uint4*>(d) = h;
              *reinterpret_cast<uint4*>(d + PTB) = md;
              *reinterpret_cast<uint4*>(d + 2 * PTB) = l;
            }
          }
          __syncthreads();
          const SplitArgs& b = reread();
          const int T = b.Ty * b.Tx, Tx = b.Tx, tap_y = b.Wp * PXB;
          const int64_t as = (int64_t)b.MTp * 3 * 64;
          const uint4* Ac = b.A + ((int64_t)(k0y * b.sw + k0x) * nchunk + ch) * T * as +
                            cb * MT * 3 * 64 + lane;
          int tx = 0;
          const char* lp = lds;
#pragma unroll 1
          for (int tap = 0; tap < T; ++tap) {
            uint4 av[MT][3];
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
              for (int p = 0; p < 3; ++p) av[mt][p] = Ac[(mt * 3 + p) * 64];
            Ac += as;
            // NB tiles of columns at a time, the next ones' parts requested
            // before this one's products; tiles past the last column repeat it
            // (a condition here would keep the loads from moving ahead)
            uint4 bv[NB][3], nx[NB][3];
#pragma unroll
            for (int k = 0; k < NB; ++k)
#pragma unroll
              for (int p = 0; p < 3; ++p)
                bv[k][p] = *reinterpret_cast<const uint4*>(lp + base[k] + p * PTB);
#pragma unroll
            for (int n0 = 0; n0 < NTW; n0 += NB) {
#pragma unroll
              for (int k = 0; k < NB; ++k)
                if (n0 + NB + k < NTW)
#pragma unroll
                  for (int p = 0; p < 3; ++p)
                    nx[k][p] =
                        *reinterpret_cast<const uint4*>(lp + base[n0 + NB + k] + p * PTB);
              __builtin_amdgcn_sched_barrier(0);
              v4f t[MT][NB], z[MT][NB];
#pragma unroll
              for (int p = 0; p < 6; ++p)
#pragma unroll
                for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                  for (int k = 0; k < NB; ++k)
                    if (n0 + k < NTW) {
                      const v4f zero = v4f{0.f, 0.f, 0.f, 0.f};
                      if (p < 5)
                        t[mt][k] = mfma_bf16(av[mt][kPartA[p]], bv[k][kPartB[p]], p ? t[mt][k] : zero);
                      else
                        z[mt][k] = mfma_bf16(av[mt][0], bv[k][0], zero);
                    }
#pragma unroll
              for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                for (int k = 0; k < NB; ++k)
                  if (n0 + k < NTW) {
                    if (COMP) {
                      v4f& c = lost[COMP ? mt : 0][COMP ? n0 + k : 0];
                      const v4f y = z[mt][k] + (t[mt][k] + c);
                      const v4f s = acc[mt][n0 + k] + y;
                      c = y - (s - acc[mt][n0 + k]);
                      acc[mt][n0 + k] = s;
                    } else {
                      acc[mt][n0 + k] += z[mt][k] + t[mt][k];
                    }
                    // summed here: sunk to the end, the parts of every tile would
                    // live at once
                    asm volatile("" : "+v"(acc[mt][n0 + k]));
                  }
#pragma unroll
              for (int k = 0; k < NB; ++k)
#pragma unroll
                for (int p = 0; p < 3; ++p) bv[k][p] = nx[k][p];
            }
            // the next tap's source pixel: one to the left, or the row above
            lp -= PXB;
            if (++tx == Tx) {
              tx = 0;
              lp += Tx * PXB - tap_y;
            }
          }
        }

        // channel ci0 + 16 mt + i of the column's pixel
        const SplitArgs& e = reread();
        const int64_t hw = (int64_t)e.H * e.W, n_o = e.C_in * hw;
        int rc = r;  // opaque, so that the columns' places are not kept over the main loop
        asm volatile("" : "+v"(rc));
        const int ci0 = 16 * cb * MT + 4 * kg;
        const auto place = [&](int nt, int64_t& mo, int& y, int& x) {
          const int c = c0 + 16 * nt + rc;
          if (nt >= ntl || c >= cols) return false;
          const int img = (int)e.f_cw.div((uint32_t)c);
          const int rem = c - img * e.Hc * e.Wc;
          const int yr = (int)e.f_wc.div((uint32_t)rem), xx = rem - yr * e.Wc;
          y = e.sh * (yy0 + yr) + py;
          x = e.sw * xx + px;
          mo = m0 + img;
          return mo < e.M && y < e.H && x < e.W;
        };
        const int64_t rest = (e.M - m0) * n_o * 4;
        const Buf bo = buffer(e.out + m0 * n_o, rest);
        const int hw4 = 4 * (int)hw;
        bool odd = false;
#pragma unroll
        for (int nt = 0; nt < NTW; ++nt) {
          __builtin_amdgcn_sched_barrier(0);
          int64_t mo;
          int y, x;
          uint32_t off = kOut;
          if (place(nt, mo, y, x))
            off = 4 * (uint32_t)((mo - m0) * n_o + ci0 * hw + (int64_t)y * e.W + x);
#pragma unroll
          for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const float v = acc[mt][nt][i];
              odd = odd || !finite(v);
              __builtin_amdgcn_raw_buffer_store_b32(
                  __builtin_bit_cast(uint32_t, v), bo,
                  ci0 + 16 * mt + i < e.C_in ? off : kOut, (16 * mt + i) * hw4, 0);
            }
        }
        if (odd) {
          // an infinity or NaN among the values: the plain sum, in 64 bits
          const SplitArgs& f = reread();
#pragma unroll 1
          for (int k = 0; k < NTW * MT * 4; ++k) {
            const int nt = k / (MT * 4), ci = ci0 + 16 * ((k >> 2) % MT) + (k & 3);
            int64_t mo;
            int y, x;
            if (!place(nt, mo, y, x) || ci >= f.C_in) continue;
            float* o = f.out + mo * n_o + ci * hw + (int64_t)y * f.W + x;
            if (!finite(*o)) *o = plain_sum<RL>(f, mo, ci, y, x);
          }
        }
      }
    }
    const SplitArgs& b = reread();
    if (b.acc && (RL > 0 || b.bias) && cb == 0) {
      const int TI = b.TI;
      for (int o = 1; o < TI && o < 64; o <<= 1) part += __shfl_xor(part, o, 64);
      if (TI > 64) {
        double* red = reinterpret_cast<double*>(lds + b.npix * PXB);
        if (lane == 0) red[wv] = part;
        __syncthreads();
        if (tl == 0) {
          part = red[wv] + red[wv + 1];
          if (TI == 256) part += red[wv + 2] + red[wv + 3];
        }
      }
      const int64_t m = m0 + g;
      if (tl == 0 && m < b.M) b.acc[m] = (float)((double)b.acc[m] + part);
    }
  }
}

// Kernels whose parts one launch makes (5 us whatever their size).
struct PackArgs {
  const float* K;
  uint4* out;
  int C_out, C_in, kh, kw, sh, sw, Ty, Tx, nchunk, MTp;
  uint32_t block0;  // its first workgroup
};
constexpr int kPacks = 16;
struct PackList {
  PackArgs p[kPacks];
  int count;
};

// A[class][chunk][tap][mt][part][lane][8]: part of K[co][ci][k0y + sh ty][k0x
// + sw tx] with ci = 16 mt + lane % 16, co = 32 chunk + 8 (lane / 16) + j;
// zero past the kernel and the channels.  class = k0y sw + k0x.
__global__ __launch_bounds__(CNT) void k_conv_split_pack(PackList list) {
  int i = 0;
  while (i + 1 < list.count && blockIdx.x >= list.p[i + 1].block0) ++i;
  const PackArgs& a = list.p[i];
  const int T = a.Ty * a.Tx;
  const int64_t t = (int64_t)(blockIdx.x - a.block0) * CNT + threadIdx.x;
  if (t >= (int64_t)a.sh * a.sw * a.nchunk * T * a.MTp * 64) return;
  const int lane = (int)(t & 63);
  int64_t q = t >> 6;
  const int mt = (int)(q % a.MTp);
  q /= a.MTp;
  const int tap = (int)(q % T);
  q /= T;
  const int ch = (int)(q % a.nchunk), cls = (int)(q / a.nchunk);
  const int ky = cls / a.sw + a.sh * (tap / a.Tx), kx = cls % a.sw + a.sw * (tap % a.Tx);
  const int ci = 16 * mt + (lane & 15), co0 = CK * ch + 8 * (lane >> 4);
  float v[8];
#pragma unroll
  for (int j = 0; j < 8; ++j)
    v[j] = (ci < a.C_in && co0 + j < a.C_out && ky < a.kh && kx < a.kw)
               ? a.K[(((int64_t)(co0 + j) * a.C_in + ci) * a.kh + ky) * a.kw + kx]
               : 0.f;
  uint4 h, m, l;
  split8(v, h, m, l);
  uint4* o = a.out + ((t >> 6) * 3) * 64 + lane;
  o[0] = h;
  o[64] = m;
  o[128] = l;
}

int ceil_div(int a, int b) { return (a + b - 1) / b; }

int split_mt(int C_in) { return C_in > 32 ? 4 : (C_in > 16 ? 2 : 1); }
int split_mtp(int C_in) {
  const int mt = split_mt(C_in);
  return ceil_div(ceil_div(C_in, 16), mt) * mt;
}

// Steps of 32 products that a sum runs over from which its rounding is
// carried along (COMP): relative to 64 bits, 64 -> 64 channels, 3x3 (18 steps)
// 9.2e-8 without, 5x5 stride 1 (50) 1.4e-7, where sums of 32 products folded
// in 64 bits are 8.2e-8; up to 9 steps 7.0e-8.  It holds a second register
// per sum, so a wave takes half of the tiles.
constexpr int kCompSteps = 9;

// The largest group of images (or, for one image, band of rows) whose parts
// fit the LDS share and whose output tiles the four waves' registers.
// False: outside the kernel's limits.
bool split_plan(SplitArgs& a, int64_t M, int cus) {
  const int MT = split_mt(a.C_in);
  a.MTp = split_mtp(a.C_in);
  a.cib = a.MTp / MT;
  a.nchunk = ceil_div(a.C_out, CK);
  a.classes = a.sh * a.sw;
  a.Ty = ceil_div(a.kh, a.sh);
  a.Tx = ceil_div(a.kw, a.sw);
  a.comp = a.nchunk * a.Ty * a.Tx > kCompSteps;
  const int ntw = a.comp ? (MT == 4 ? 4 : (MT == 2 ? 8 : 9)) : (MT == 4 ? 8 : 16);
  a.Hc = ceil_div(a.H, a.sh);
  a.Wc = ceil_div(a.W, a.sw);
  a.cminy = a.ph / a.sh;
  const int cmaxy = (a.sh - 1 + a.ph) / a.sh;
  const int cminx = a.pw / a.sw, cmaxx = (a.sw - 1 + a.pw) / a.sw;
  // every source row is some band's (its constant terms)
  if (a.cminy > a.Ty - 1 || a.Hc - 1 + cmaxy < a.Hs - 1) return false;
  const int top = a.Ty - 1 - a.cminy, bot = a.Hc - 1 + cmaxy - (a.Hs - 1);
  const int hl = a.Tx - 1 - cminx > 0 ? a.Tx - 1 - cminx : 0;
  const int hr0 = a.Wc - 1 + cmaxx - (a.Ws - 1), hr = hr0 > 0 ? hr0 : 0;
  a.Wp = a.Ws + (hl > hr ? hl : hr);
  const auto fits = [&](int G, int YB, bool band) {
    a.G = G;
    a.YB = YB;
    a.NB = band ? ceil_div(a.Hc, YB) : 1;
    a.Hb = band ? YB + cmaxy - a.cminy + a.Ty - 1 : a.Hs;
    a.IMG = (band ? a.Hb : a.Hs + (top > bot ? top : bot)) * a.Wp;
    a.P0 = hl + (band ? 0 : top * a.Wp);
    const int64_t px = a.P0 + (int64_t)(G - 1) * a.IMG +
                       (int64_t)(band ? a.Hb : a.Hs + bot) * a.Wp + hr;
    if (px * PXB + 64 > kMaxLds) return false;
    a.npix = (int)px;
    const int nt = ceil_div(G * (YB < a.Hc ? YB : a.Hc) * a.Wc, 16);
    a.NG = a.classes >= 4 ? 1 : 4 / a.classes;
    if (ceil_div(nt, a.NG) > ntw) a.NG = ceil_div(nt, ntw);
    a.gs = ceil_div(nt, a.NG);
    a.passes = ceil_div(a.classes * a.NG, 4);
    return true;
  };
  const int least = ceil_div(a.classes, 4);  // passes that one image cannot avoid
  for (int G = 16; G >= 1; G >>= 1) {
    if (G > 1 && (M + G - 1) / G < 2 * (int64_t)cus) continue;  // fewer tiles than places for them
    if (fits(G, a.Hc, false) && a.passes <= least) return true;
  }
  for (int nb = 2; nb <= a.Hc; ++nb)
    if (fits(1, ceil_div(a.Hc, nb), true) && a.passes <= least) return true;
  return false;
}

template <int MT, int NTW, bool COMP = false>
const void* inst(bool relu) {
  return relu ? (const void*)&k_conv_split<MT, NTW, 1, COMP>
              : (const void*)&k_conv_split<MT, NTW, 0, COMP>;
}

// The instance for gs column tiles per wave (a wave runs all of its NTW).
const void* pick_kernel(int MT, int gs, bool relu, bool comp) {
  if (comp) {
    if (MT == 1)
      return gs <= 2 ? inst<1, 2, true>(relu) : (gs <= 4 ? inst<1, 4, true> : inst<1, 9, true>)(relu);
    if (MT == 2)
      return gs <= 2 ? inst<2, 2, true>(relu) : (gs <= 4 ? inst<2, 4, true> : inst<2, 8, true>)(relu);
    return gs <= 2 ? inst<4, 2, true>(relu) : inst<4, 4, true>(relu);
  }
  if (MT == 1)
    return gs <= 2   ? inst<1, 2>(relu)
           : gs <= 4 ? inst<1, 4>(relu)
           : gs <= 6 ? inst<1, 6>(relu)
           : gs <= 9 ? inst<1, 9>(relu)
                     : inst<1, 16>(relu);
  if (MT == 2)
    return gs <= 2    ? inst<2, 2>(relu)
           : gs <= 4  ? inst<2, 4>(relu)
           : gs <= 7  ? inst<2, 7>(relu)
           : gs <= 10 ? inst<2, 10>(relu)
           : gs <= 13 ? inst<2, 13>(relu)
                      : inst<2, 16>(relu);
  return gs <= 2 ? inst<4, 2>(relu) : (gs <= 4 ? inst<4, 4> : inst<4, 8>)(relu);
}

// The plan for the rows at hand; false: outside the kernel's limits.
bool split_fits(SplitArgs& a) {
  if (!split_plan(a, a.M, vcm::cu_count())) return false;
  a.TI = CNT / a.G;
  a.n_tiles = (a.M + a.G - 1) / a.G * a.cib;
  if (a.M >= (int64_t(1) << 31) || a.n_tiles >= (int64_t(1) << 31)) return false;
  // the loads' byte offsets are 32-bit: one tile's images, or all shared rows
  const int64_t n_e = (int64_t)a.C_out * a.Hs * a.Ws, n_i = (int64_t)a.C_out * a.Hi * a.Wi;
  return (a.shared ? a.R : a.G) * n_e * 4 < 0xf0000000ll && (a.G + 1) * n_i * 4 < 0xf0000000ll &&
         (int64_t)a.G * a.MTp * 16 * a.H * a.W * 4 < 0x7fffffffll;
}

int launch_split(SplitArgs& a, hipStream_t st) {
  const int cus = vcm::cu_count();
  if (!split_fits(a)) return VC_ERR_UNSUPPORTED;
  a.f_cw = FastDiv::make((uint32_t)(a.Hc * a.Wc));
  a.f_wc = FastDiv::make((uint32_t)a.Wc);
  a.f_npx = FastDiv::make((uint32_t)(a.Hb * a.Ws));
  a.f_ws = FastDiv::make((uint32_t)a.Ws);
  a.f_cib = FastDiv::make((uint32_t)a.cib);
  a.f_R = FastDiv::make((uint32_t)a.R);
  a.f_sw = FastDiv::make((uint32_t)a.sw);
  a.f_ng = FastDiv::make((uint32_t)a.NG);
  const void* fn = pick_kernel(split_mt(a.C_in), a.gs, a.ls != nullptr, a.comp);
  const size_t lds = (size_t)a.npix * PXB + 64;
  if (!vcm::allow_max_lds(fn)) return VC_ERR_UNSUPPORTED;
  int64_t grid = 2 * (int64_t)cus;
  if (grid > a.n_tiles) grid = a.n_tiles;
  void* args[] = {&a};
  if (hipLaunchKernel(fn, dim3((unsigned)grid), dim3(CNT), args, lds, st) != hipSuccess)
    return VC_ERR_LAUNCH;
  VC_LAUNCH_CHECK();
  return VC_OK;
}

// Rows of a window: C x kh x kw values of each seeded neuron's own kernel and
// their place in the image, "+" rows then "-" rows, and the bias as their
// constant term (the conv backward of one-hot rows).
__global__ void k_patch_seed(const float* K, const float* bias, const int* idx, int k, int sp,
                             int Wo, int n, int sh, int sw, int ph, int pw, float* rows,
                             int* origin, float* acc) {
  const int64_t total = (int64_t)2 * k * n;
  for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < total;
       t += (int64_t)gridDim.x * blockDim.x) {
    const int r = (int)(t / n), i = (int)(t - (int64_t)r * n);
    const int j = idx[r < k ? r : r - k];
    const int c = j / sp, y = (j - c * sp) / Wo, x = (j - c * sp) - y * Wo;
    const float v = K[(int64_t)c * n + i];
    rows[t] = r < k ? v : -v;
    if (i == 0) {
      origin[2 * r] = y * sh - ph;
      origin[2 * r + 1] = x * sw - pw;
      const float b = bias ? bias[c] : 0.f;
      acc[r] = r < k ? b : -b;
    }
  }
}

// The image positions of a conv's output windows from those of its input's.
__global__ void k_patch_shift(const int* in, int n, int sh, int sw, int ph, int pw, int* out) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) {
    out[2 * t] = in[2 * t] * sh - ph;
    out[2 * t + 1] = in[2 * t + 1] * sw - pw;
  }
}

// Rows of windows relaxed by their domains' slopes at the windows' places in
// the image (RELU 0: copied), zero outside the image, and the intercepts added
// to acc in 64 bits: the separate relu step on windows.  One wave per row, lanes
// along it: each row is read and written once, coalesced; a lane's four loads
// go out together, outside the image from its first pixel, not used.
template <bool RELU>
__global__ __launch_bounds__(CNT) void k_patch_relax(const float* x, int shared, const float* ls,
                                                     const float* us, const float* ut,
                                                     const int* origin, int64_t M, int64_t R,
                                                     int C, int H, int W, int wh, int ww,
                                                     FastDiv f_ww, FastDiv f_wp, float* out,
                                                     float* acc) {
  const int wp = wh * ww, n = C * wp, lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  for (int64_t m = (int64_t)blockIdx.x * (CNT / 64) + wv; m < M;
       m += (int64_t)gridDim.x * (CNT / 64)) {
    const int64_t d = m / R, row = m - d * R, img = d * C * H * W;
    const float* a = x + (shared ? row : m) * n;
    const float *lm = ls + img, *um = us + img, *tm = ut + img;
    float* const om = out + m * n;
    const int oy = origin[2 * row], ox = origin[2 * row + 1];
    double s = 0.0;
    for (int i = lane; i < n; i += 64) {
      const int c = (int)f_wp.div((uint32_t)i), p = i - c * wp;
      const int dy = (int)f_ww.div((uint32_t)p), dx = p - dy * ww;
      const int y = oy + dy, xx = ox + dx;
      const bool in = (unsigned)y < (unsigned)H && (unsigned)xx < (unsigned)W;
      float e = a[(uint32_t)i];
      if (RELU) {
        const uint32_t o = in ? (c * H + y) * W + xx : 0;
        const float l = lm[o], u = um[o], t = tm[o];
        const float en = e > 0.f ? 0.f : e, ep = e < 0.f ? 0.f : e;
        s += in ? (double)(en * t) : 0.0;
        e = ep * l + en * u;
      }
      om[(uint32_t)i] = in ? e : 0.f;
    }
    if (RELU) {
      s = wave_sum_f64(s);
      if (lane == 0) acc[m] = (float)((double)acc[m] + s);
    }
  }
}

// lb[m] = acc[m] + sum over the window's pixels inside the image of
// pos(A) xl + neg(A) xh; 16 lanes per row, summed in 64 bits.
__global__ __launch_bounds__(CNT) void k_patch_concretize(const float* A, int shared,
                                                          const int* origin, const float* acc,
                                                          const float* xl, const float* xh,
                                                          int64_t M, int64_t R, int C, int H,
                                                          int W, int wh, int ww, FastDiv f_ww,
                                                          FastDiv f_wp, float* lb) {
  const int wp = wh * ww, n = C * wp;
  for (int64_t m0 = (int64_t)blockIdx.x * (CNT / 16); m0 < M;
       m0 += (int64_t)gridDim.x * (CNT / 16)) {
    const int64_t mm = m0 + (threadIdx.x >> 4);
    const int64_t m = mm < M ? mm : M - 1;  // past the end: recompute the last row, no store
    const int64_t d = m / R, row = m - d * R;
    const float* a = A + (shared ? row : m) * n;
    const float *l = xl + d * C * H * W, *h = xh + d * C * H * W;
    const int oy = origin[2 * row], ox = origin[2 * row + 1];
    double s = 0.0;
    for (int i = threadIdx.x & 15; i < n; i += 16) {
      const int c = (int)f_wp.div((uint32_t)i), p = i - c * wp;
      const int dy = (int)f_ww.div((uint32_t)p), dx = p - dy * ww;
      const int y = oy + dy, x = ox + dx;
      if ((unsigned)y < (unsigned)H && (unsigned)x < (unsigned)W) {
        const int o = (c * H + y) * W + x;
        const float v = a[i];
        s += (double)(v * (v < 0.f ? h[o] : l[o]));
      }
    }
    s = row_sum16(s);
    if ((threadIdx.x & 15) == 0 && mm < M) lb[mm] = (float)((double)acc[mm] + s);
  }
}

// Windows into whole images: rows (N, C, H, W), zero outside the window.
// Row n's window sits at origin[n mod R].
__global__ __launch_bounds__(CNT) void k_patch_dense(const float* A, const int* origin, int64_t N,
                                                     int64_t R, int C, int H, int W, int wh,
                                                     int ww, FastDiv f_w, FastDiv f_hw,
                                                     float* out) {
  const int hw = H * W;
  for (int64_t n = blockIdx.x; n < N; n += gridDim.x) {
    const int64_t row = n % R;
    const int oy = origin[2 * row], ox = origin[2 * row + 1];
    for (int i = threadIdx.x; i < C * hw; i += CNT) {
      const int c = (int)f_hw.div((uint32_t)i), p = i - c * hw;
      const int y = (int)f_w.div((uint32_t)p) - oy, x = p - (y + oy) * W - ox;
      const bool in = (unsigned)y < (unsigned)wh && (unsigned)x < (unsigned)ww;
      out[n * C * hw + i] = in ? A[((n * C + c) * wh + y) * ww + x] : 0.f;
    }
  }
}

bool geom_ok(int C_out, int Hs, int Ws, int C_in, int H, int W, int kh, int kw, int sh, int sw,
             int ph, int pw) {
  return C_out > 0 && Hs > 0 && Ws > 0 && C_in > 0 && H > 0 && W > 0 && kh > 0 && kw > 0 &&
         sh > 0 && sw > 0 && ph >= 0 && pw >= 0 && Hs == (H + 2 * ph - kh) / sh + 1 &&
         Ws == (W + 2 * pw - kw) / sw + 1;
}

}  // namespace

extern "C" int64_t vc_conv_split_pack_bytes(int C_out, int C_in, int kh, int kw, int sh, int sw) {
  if (C_out <= 0 || C_in <= 0 || kh <= 0 || kw <= 0 || sh <= 0 || sw <= 0) return -VC_ERR_ARG;
  return (int64_t)sh * sw * ceil_div(C_out, CK) * ceil_div(kh, sh) * ceil_div(kw, sw) *
         split_mtp(C_in) * 3 * 64 * 16;
}

extern "C" int vc_conv_split_pack_many(const float* const* kernel, const int32_t* geom,
                                       void* const* out, int count, vc_stream_t stream) {
  if (count < 0 || (count > 0 && (!kernel || !geom || !out))) return VC_ERR_ARG;
  for (int i = 0; i < count; ++i) {
    const int32_t* g = geom + 6 * i;
    if (!kernel[i] || !out[i] || !aligned16(out[i]) ||
        vc_conv_split_pack_bytes(g[0], g[1], g[2], g[3], g[4], g[5]) < 0)
      return VC_ERR_ARG;
  }
  for (int i0 = 0; i0 < count; i0 += kPacks) {
    PackList a{};
    a.count = count - i0 < kPacks ? count - i0 : kPacks;
    int64_t blocks = 0;
    for (int i = 0; i < a.count; ++i) {
      const int32_t* g = geom + 6 * (i0 + i);
      a.p[i] = PackArgs{kernel[i0 + i], (uint4*)out[i0 + i], g[0], g[1], g[2], g[3], g[4], g[5],
                        ceil_div(g[2], g[4]), ceil_div(g[3], g[5]), ceil_div(g[0], CK),
                        split_mtp(g[1]), (uint32_t)blocks};
      blocks += (vc_conv_split_pack_bytes(g[0], g[1], g[2], g[3], g[4], g[5]) / 48 + CNT - 1) / CNT;
      if (blocks >= (int64_t(1) << 31)) return VC_ERR_UNSUPPORTED;
    }
    hipLaunchKernelGGL(k_conv_split_pack, dim3((unsigned)blocks), dim3(CNT), 0,
                       (hipStream_t)stream, a);
    VC_LAUNCH_CHECK();
  }
  return VC_OK;
}

extern "C" int vc_conv_split_pack(const float* kernel, int C_out, int C_in, int kh, int kw, int sh,
                                  int sw, void* out, vc_stream_t stream) {
  const int32_t geom[6] = {C_out, C_in, kh, kw, sh, sw};
  return vc_conv_split_pack_many(&kernel, geom, &out, 1, stream);
}

extern "C" int vc_backward_conv_split_ok(int C_out, int H_out, int W_out, int C_in, int H, int W,
                                         int kh, int kw, int sh, int sw, int ph, int pw) {
  if (!geom_ok(C_out, H_out, W_out, C_in, H, W, kh, kw, sh, sw, ph, pw)) return 0;
  SplitArgs a{};
  a.C_out = C_out, a.Hs = H_out, a.Ws = W_out, a.C_in = C_in, a.H = H, a.W = W;
  a.kh = kh, a.kw = kw, a.sh = sh, a.sw = sw, a.ph = ph, a.pw = pw;
  return split_plan(a, 1, 1) ? 1 : 0;
}

extern "C" int vc_backward_conv_split_fits(int64_t M, int64_t R, int ew_shared, int C_out,
                                           int H_out, int W_out, int C_in, int H, int W, int kh,
                                           int kw, int sh, int sw, int ph, int pw) {
  if (!geom_ok(C_out, H_out, W_out, C_in, H, W, kh, kw, sh, sw, ph, pw) || M <= 0 || R <= 0)
    return 0;
  SplitArgs a{};
  a.M = M, a.R = R, a.shared = ew_shared ? 1 : 0;
  a.C_out = C_out, a.Hs = H_out, a.Ws = W_out, a.Hi = H_out, a.Wi = W_out;
  a.C_in = C_in, a.H = H, a.W = W;
  a.kh = kh, a.kw = kw, a.sh = sh, a.sw = sw, a.ph = ph, a.pw = pw;
  return split_fits(a) ? a.NB : 0;
}

extern "C" int vc_backward_conv_split(const float* ew_in, int64_t M, int64_t R, int ew_shared,
                                      const float* lo_s, const float* up_s, const float* up_t,
                                      const float* beta, const float* kernel, const void* packed,
                                      const float* bias, int C_out, int H_out, int W_out,
                                      int C_in, int H, int W, int kh, int kw, int sh, int sw,
                                      int ph, int pw, float* ew_out, float* acc, vc_stream_t stream) {
  if (!geom_ok(C_out, H_out, W_out, C_in, H, W, kh, kw, sh, sw, ph, pw) || !ew_in || !kernel ||
      !packed || !aligned16(packed) || !ew_out || M < 0 || R <= 0 || M % R)
    return VC_ERR_ARG;
  if ((lo_s == nullptr) != (up_s == nullptr) || (lo_s == nullptr) != (up_t == nullptr) ||
      (beta && !lo_s) || ((lo_s || bias) && !acc))
    return VC_ERR_ARG;
  if (M == 0) return VC_OK;
  SplitArgs a{};
  a.ew = ew_in, a.M = M, a.R = R, a.shared = ew_shared ? 1 : 0;
  a.ls = lo_s, a.us = up_s, a.ut = up_t, a.beta = beta;
  a.K = kernel, a.A = (const uint4*)packed, a.bias = bias, a.out = ew_out, a.acc = acc;
  a.C_out = C_out, a.Hs = H_out, a.Ws = W_out, a.Hi = H_out, a.Wi = W_out;
  a.C_in = C_in, a.H = H, a.W = W;
  a.kh = kh, a.kw = kw, a.sh = sh, a.sw = sw, a.ph = ph, a.pw = pw;
  return launch_split(a, (hipStream_t)stream);
}

extern "C" int vc_patch_seed(const float* kernel, const float* bias, const int32_t* idx, int k,
                             int C_out, int H_out, int W_out, int C_in, int kh, int kw, int sh,
                             int sw, int ph, int pw, float* rows, int32_t* origin, float* acc,
                             vc_stream_t stream) {
  if (!kernel || !idx || !rows || !origin || !acc || k < 0 || C_out <= 0 || H_out <= 0 ||
      W_out <= 0 || C_in <= 0 || kh <= 0 || kw <= 0 || sh <= 0 || sw <= 0 || ph < 0 || pw < 0)
    return VC_ERR_ARG;
  const int64_t n = (int64_t)C_in * kh * kw;
  if (n > (1 << 30) || (int64_t)C_out * H_out * W_out > (1 << 30)) return VC_ERR_UNSUPPORTED;
  if (k == 0) return VC_OK;
  hipLaunchKernelGGL(k_patch_seed, dim3(vc_blocks(2 * k * n, CNT)), dim3(CNT), 0,
                     (hipStream_t)stream, kernel, bias, idx, k, H_out * W_out, W_out, (int)n, sh,
                     sw, ph, pw, rows, origin, acc);
  VC_LAUNCH_CHECK();
  return VC_OK;
}

extern "C" int vc_patch_shift(const int32_t* origin_in, int R, int sh, int sw, int ph, int pw,
                              int32_t* origin_out, vc_stream_t stream) {
  if (!origin_in || !origin_out || R < 0 || sh <= 0 || sw <= 0 || ph < 0 || pw < 0)
    return VC_ERR_ARG;
  if (R == 0) return VC_OK;
  hipLaunchKernelGGL(k_patch_shift, dim3((R + CNT - 1) / CNT), dim3(CNT), 0, (hipStream_t)stream,
                     origin_in, R, sh, sw, ph, pw, origin_out);
  VC_LAUNCH_CHECK();
  return VC_OK;
}

extern "C" int vc_patch_relax(const float* ew_in, int64_t M, int64_t R, int ew_shared,
                              const float* lo_s, const float* up_s, const float* up_t,
                              const int32_t* origin, int C, int H, int W,
                              int wh, int ww, float* ew_out, float* acc, vc_stream_t stream) {
  if (!ew_in || !origin || !ew_out || M < 0 || R <= 0 || M % R || C <= 0 || H <= 0 || W <= 0 ||
      wh <= 0 || ww <= 0)
    return VC_ERR_ARG;
  if ((lo_s == nullptr) != (up_s == nullptr) || (lo_s == nullptr) != (up_t == nullptr) ||
      (lo_s && !acc))
    return VC_ERR_ARG;
  if ((int64_t)C * wh * ww > (1 << 30) || (int64_t)C * H * W > (1 << 30)) return VC_ERR_UNSUPPORTED;
  if (M == 0) return VC_OK;
  hipLaunchKernelGGL(lo_s ? k_patch_relax<true> : k_patch_relax<false>,
                     dim3(vc_blocks(64 * M, CNT)), dim3(CNT), 0, (hipStream_t)stream, ew_in,
                     ew_shared ? 1 : 0, lo_s, up_s, up_t, origin, M, R, C, H, W, wh, ww,
                     FastDiv::make((uint32_t)ww), FastDiv::make((uint32_t)(wh * ww)), ew_out, acc);
  VC_LAUNCH_CHECK();
  return VC_OK;
}

extern "C" int vc_patch_concretize(const float* A, int a_shared, const int32_t* origin,
                                   const float* acc, const float* xl, const float* xh, int64_t M,
                                   int64_t R, int C, int H, int W, int wh, int ww, float* lb,
                                   vc_stream_t stream) {
  if (!A || !origin || !acc || !xl || !xh || !lb || M < 0 || R <= 0 || M % R || C <= 0 ||
      H <= 0 || W <= 0 || wh <= 0 || ww <= 0)
    return VC_ERR_ARG;
  if ((int64_t)C * wh * ww > (1 << 30) || (int64_t)C * H * W > (1 << 30)) return VC_ERR_UNSUPPORTED;
  if (M == 0) return VC_OK;
  hipLaunchKernelGGL(k_patch_concretize, dim3(vc_blocks(16 * M, CNT)), dim3(CNT), 0,
                     (hipStream_t)stream, A, a_shared ? 1 : 0, origin, acc, xl, xh, M, R, C, H, W,
                     wh, ww, FastDiv::make((uint32_t)ww), FastDiv::make((uint32_t)(wh * ww)), lb);
  VC_LAUNCH_CHECK();
  return VC_OK;
}

extern "C" int vc_patch_dense(const float* A, const int32_t* origin, int64_t N, int64_t R, int C,
                              int H, int W, int wh, int ww, float* out, vc_stream_t stream) {
  if (!A || !origin || !out || N < 0 || R <= 0 || C <= 0 || H <= 0 || W <= 0 || wh <= 0 || ww <= 0)
    return VC_ERR_ARG;
  if ((int64_t)C * H * W > (1 << 30)) return VC_ERR_UNSUPPORTED;
  if (N == 0) return VC_OK;
  hipLaunchKernelGGL(k_patch_dense, dim3((unsigned)(N < vcg::kMaxGrid ? N : vcg::kMaxGrid)),
                     dim3(CNT), 0, (hipStream_t)stream, A, origin, N, R, C, H, W, wh, ww,
                     FastDiv::make((uint32_t)W), FastDiv::make((uint32_t)(H * W)), out);
  VC_LAUNCH_CHECK();
  return VC_OK;
}
