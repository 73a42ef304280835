// The Wan2.2 VAE encoder's first frame (the policy call's prologue) around the library's GEMM.
// Activations are channels-last rows, one row per pixel ([h*w, C] bf16), so a 1x1 convolution
// is a GEMM over the rows and a 3x3 one a GEMM over the pixels' 3x3 neighbourhoods, taps
// outermost ((kh*3 + kw)*C + c), zero-padded to a multiple of 64 columns: fam_conv3x3 gathers
// them itself, and below its 128 output pixels im2col3x3_kernel lays them out.  The kernels here are the non-GEMM steps, each one elementwise pass over the bytes
// it moves (the middle attention's softmax is one wave per row).
#include "fam_common.h"

namespace fam {

// conv1's operand straight from the image: the 2x2 patchify ('b c (h q) (w r) -> b (c r q) h w',
// patched channel c*4 + r*2 + q) fused into the 3x3 im2col of the patched grid (h2 x w2).
// A thread gathers 8 columns (its loads are 2 bytes apart in up to 8 places; eight in flight and
// one 16-byte store instead of one of each); columns past 9*12 are zero.
// 224 x 448 image: 12.0 -> 8.7 us.
__global__ __launch_bounds__(256) void vae_patch_im2col_kernel(const bf16* __restrict__ img, int H, int W,
                                                               bf16* __restrict__ out, int64_t ldo, int vec,
                                                               int64_t total) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= total) return;
  const int w2 = W / 2, p = (int)(i >> 4), col0 = (int)(i & 15) * 8;
  const int py = p / w2, px = p - py * w2;
  bf16x8 v = zero8();
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const int col = col0 + e;
    const int tap = col / 12, ch = col - tap * 12;
    const int kh = tap / 3, kw = tap - kh * 3;
    const int c = ch >> 2, r = (ch >> 1) & 1, q = ch & 1;
    const int y = py + kh - 1, x = px + kw - 1;
    if (col < 108 && y >= 0 && y < H / 2 && x >= 0 && x < w2) v[e] = img[((int64_t)c * H + 2 * y + q) * W + 2 * x + r];
  }
  bf16* o = out + p * ldo + col0;
  if (vec) {
    store8(o, v);
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = v[e];
  }
}

// 3x3 im2col of channels-last rows, 8 channels (16 bytes) per thread.  stride 1: 'same' zero
// padding; stride 2: zero padding on the bottom / right only (ZeroPad2d((0, 1, 0, 1)) before a
// stride-2 3x3 convolution), output (H/2) x (W/2).
__global__ __launch_bounds__(256) void im2col3x3_kernel(const bf16* __restrict__ x, int64_t ldx, int H, int W,
                                                        int C, int stride, bf16* __restrict__ out, int64_t ldo,
                                                        int kpad, int64_t total) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= total) return;
  const int Wo = stride == 1 ? W : W / 2;
  const int k8 = kpad / 8;
  const int64_t p = i / k8;
  const int col = (int)(i - p * k8) * 8;
  bf16x8 v = zero8();
  if (col < 9 * C) {
    const int tap = col / C, c = col - tap * C;
    const int kh = tap / 3, kw = tap - kh * 3;
    const int oy = (int)(p / Wo), ox = (int)(p % Wo);
    const int y = stride == 1 ? oy + kh - 1 : 2 * oy + kh, xx = stride == 1 ? ox + kw - 1 : 2 * ox + kw;
    if (y >= 0 && y < H && xx >= 0 && xx < W) v = load8(x + ((int64_t)y * W + xx) * ldx + c);
  }
  store8(out + p * ldo + col, v);
}

// RMS_norm over the channels of a row (F.normalize: x / max(||x||_2, 1e-12), times sqrt(C) and
// gamma), then the activation.  LPR lanes per row, 8 channels per lane and step: 16 lanes up to
// 128 channels and 32 up to 256, so that the encoder's 160-channel rows (20 lanes' worth) do not
// leave two thirds of a wave idle.  HELD: the row stays in registers between the two passes (up
// to HELD steps); 0: it is read twice (C > 1024).  Rows of 160 channels,
// 25088 of them: 10.8 us with a wave per row and two reads, 6.7 now (16 MB; 3.2 at copy rate).
template <int LPR, int HELD>
__global__ __launch_bounds__(256) void chan_rmsnorm_kernel(const bf16* __restrict__ x, int64_t ldx, int64_t rows,
                                                           int C, const bf16* __restrict__ gamma, int act,
                                                           bf16* __restrict__ y, int64_t ldy) {
  const int lane = threadIdx.x & (LPR - 1);
  const int64_t r = (int64_t)blockIdx.x * (256 / LPR) + threadIdx.x / LPR;
  if (r >= rows) return;   // whole groups of LPR lanes, which reduce among themselves
  const bf16* xr = x + r * ldx;
  bf16x8 held[HELD ? HELD : 1];
  float ss = 0.f;
  auto square = [&](bf16x8 v) {
#pragma unroll
    for (int e = 0; e < 8; ++e) ss += to_f(v[e]) * to_f(v[e]);
  };
  if constexpr (HELD > 0) {
#pragma unroll
    for (int k = 0; k < HELD; ++k) {
      const int c = (k * LPR + lane) * 8;
      held[k] = c < C ? load8(xr + c) : zero8();
    }
#pragma unroll
    for (int k = 0; k < HELD; ++k) square(held[k]);
  } else {
    for (int c = lane * 8; c < C; c += LPR * 8) square(load8(xr + c));
  }
#pragma unroll
  for (int o = LPR / 2; o >= 1; o >>= 1) ss += __shfl_xor(ss, o, kWave);
  const float rn = sqrtf((float)C) / fmaxf(sqrtf(ss), 1e-12f);
  auto finish = [&](int c, bf16x8 v) {
    const bf16x8 gv = load8(gamma + c);
    bf16x8 o;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      float t = to_f(v[e]) * rn * to_f(gv[e]);
      if (act == FAM_ACT_SILU) t = silu(t);
      o[e] = to_bf(t);
    }
    store8(y + r * ldy + c, o);
  };
  if constexpr (HELD > 0) {
#pragma unroll
    for (int k = 0; k < HELD; ++k) {
      const int c = (k * LPR + lane) * 8;
      if (c < C) finish(c, held[k]);
    }
  } else {
    for (int c = lane * 8; c < C; c += LPR * 8) finish(c, load8(xr + c));
  }
}

// AvgDown3D of one frame: the frame axis front-padded with ft - 1 zero frames, (t, i, j) blocks
// of ft x fs x fs folded into channels c*F + t*fs*fs + i*fs + j (F = ft*fs*fs), output channel o
// the mean of group [o*G, (o+1)*G), G = Cin*F/Cout; plus `add` (same layout as out) when given.
// One thread per output element.
__global__ __launch_bounds__(256) void vae_avgdown_kernel(const bf16* __restrict__ x, int64_t ldx, int H, int W,
                                                          int Cin, int Cout, int ft, int fs,
                                                          const bf16* __restrict__ add, int64_t ldadd,
                                                          bf16* __restrict__ out, int64_t ldo, int64_t total) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= total) return;
  const int Wo = W / fs, F = ft * fs * fs, G = Cin * F / Cout;
  const int64_t p = i / Cout;
  const int o = (int)(i - p * Cout);
  const int oy = (int)(p / Wo), ox = (int)(p % Wo);
  float s = 0.f;
  for (int e = o * G; e < (o + 1) * G; ++e) {
    const int c = e / F, rem = e - c * F;
    const int t = rem / (fs * fs), ij = rem - t * fs * fs, ii = ij / fs, jj = ij - ii * fs;
    if (t == ft - 1) s += to_f(x[((int64_t)(oy * fs + ii) * W + ox * fs + jj) * ldx + c]);
  }
  const float a = add ? to_f(add[p * ldadd + o]) : 0.f;
  out[p * ldo + o] = to_bf(s / (float)G + a);
}

// The same where every group is the whole fs x fs block of one (channel, frame) pair (Cout = Cin
// ft, the encoder's own), on aligned rows of 8 k outputs: 8 outputs per thread, 16-byte accesses.
// Output o is channel o / ft; with ft = 2 the even ones are the zero frame's.  The sums run in the
// same order.  The one-output form above is bound by its index arithmetic: 112 x 224 x
// 160 halved 14.0 us there, 5.0 here; 56 x 112 x 320, two frames 8.3 and 4.6.
template <int FT, int FS>
__global__ __launch_bounds__(256) void vae_avgdown_vec_kernel(const bf16* __restrict__ x, int64_t ldx, int W, int Cout,
                                                              const bf16* __restrict__ add, int64_t ldadd,
                                                              bf16* __restrict__ out, int64_t ldo, int64_t total) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= total) return;
  typedef __bf16 bfin __attribute__((ext_vector_type(8 / FT)));
  const int Wo = W / FS, c8 = Cout / 8;
  const int64_t p = i / c8;
  const int o = (int)(i - p * c8) * 8, oy = (int)(p / Wo), ox = (int)(p - (int64_t)oy * Wo);
  bfin v[FS * FS];
#pragma unroll
  for (int k = 0; k < FS * FS; ++k)
    v[k] = *reinterpret_cast<const bfin*>(x + ((int64_t)(oy * FS + k / FS) * W + ox * FS + k % FS) * ldx + o / FT);
  const bf16x8 a = add ? load8(add + p * ldadd + o) : zero8();
  bf16x8 r;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    float s = 0.f;
    if (e % FT == FT - 1) {
#pragma unroll
      for (int k = 0; k < FS * FS; ++k) s += to_f(v[k][e / FT]);
    }
    r[e] = to_bf(s / (float)(FS * FS) + (add ? to_f(a[e]) : 0.f));
  }
  store8(out + p * ldo + o, r);
}

// Row softmax of fp32 scores times `scale`, rounded to bf16 (the middle attention's P).
__global__ __launch_bounds__(256) void softmax_rows_kernel(const float* __restrict__ s, int64_t lds, int64_t rows,
                                                           int cols, float scale, bf16* __restrict__ p, int64_t ldp) {
  const int lane = threadIdx.x & 63;
  const int64_t r = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (r >= rows) return;
  const float* sr = s + r * lds;
  const float sl2 = scale * 1.4426950408889634f;
  float m = -INFINITY;
  for (int c = lane; c < cols; c += 64) m = fmaxf(m, sr[c]);
  m = wave_max(m) * sl2;
  float l = 0.f;
  for (int c = lane; c < cols; c += 64) l += __builtin_amdgcn_exp2f(sr[c] * sl2 - m);
  l = wave_sum(l);
  const float inv = 1.0f / l;
  for (int c = lane; c < cols; c += 64) p[r * ldp + c] = to_bf(__builtin_amdgcn_exp2f(sr[c] * sl2 - m) * inv);
}

// out[c, p] = (x[p, c] - mean[c]) * inv_std[c]: the latent normalisation, channels-last rows to
// the channel-first latent.
__global__ __launch_bounds__(256) void chan_affine_nchw_kernel(const bf16* __restrict__ x, int64_t ldx, int64_t P,
                                                               int C, const float* __restrict__ mean,
                                                               const float* __restrict__ inv_std,
                                                               bf16* __restrict__ out, int64_t total) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= total) return;
  const int c = (int)(i / P);
  const int64_t p = i - (int64_t)c * P;
  out[i] = to_bf((to_f(x[p * ldx + c]) - mean[c]) * inv_std[c]);
}

}  // namespace fam

using namespace fam;

static unsigned blocks_for(int64_t n, int64_t per) { return (unsigned)((n + per - 1) / per); }

extern "C" int fam_vae_patch_im2col(const void* img, int64_t H, int64_t W, void* out, int64_t ldo, void* stream) {
  FAM_REQUIRE(img && out, FAM_ERR_INVALID_ARG, "fam_vae_patch_im2col: null pointer");
  FAM_REQUIRE(H >= 2 && W >= 2 && H % 2 == 0 && W % 2 == 0 && H < (1 << 15) && W < (1 << 15) && ldo >= 128,
              FAM_ERR_INVALID_ARG, "fam_vae_patch_im2col: need even H, W (< 32768) and ldo >= 128");
  const int64_t total = (H / 2) * (W / 2) * 16;
  const int vec = ldo % 8 == 0 && fam_host::aligned16(out);
  FAM_LAUNCH(vae_patch_im2col_kernel, dim3(blocks_for(total, 256)), dim3(256), 0, (hipStream_t)stream,
             (const bf16*)img, (int)H, (int)W, (bf16*)out, ldo, vec, total);
  return fam_host::check_launch("fam_vae_patch_im2col");
}

extern "C" int fam_im2col3x3(const void* x, int64_t ldx, int64_t H, int64_t W, int64_t C, int64_t stride, void* out,
                             int64_t ldo, int64_t kpad, void* stream) {
  FAM_REQUIRE(x && out, FAM_ERR_INVALID_ARG, "fam_im2col3x3: null pointer");
  FAM_REQUIRE((stride == 1 || (stride == 2 && H % 2 == 0 && W % 2 == 0)) && H >= 1 && W >= 1 && H * W < (1LL << 31),
              FAM_ERR_INVALID_ARG, "fam_im2col3x3: stride 1, or 2 with even H and W");
  FAM_REQUIRE(C >= 8 && C % 8 == 0 && ldx >= C && ldx % 8 == 0 && kpad >= 9 * C && kpad % 8 == 0 && ldo >= kpad &&
                  ldo % 8 == 0 && fam_host::aligned16(x) && fam_host::aligned16(out),
              FAM_ERR_INVALID_ARG, "fam_im2col3x3: C, ldx, kpad (>= 9 C), ldo multiples of 8; 16-byte aligned rows");
  const int64_t P = stride == 1 ? H * W : (H / 2) * (W / 2);
  const int64_t total = P * (kpad / 8);
  FAM_LAUNCH(im2col3x3_kernel, dim3(blocks_for(total, 256)), dim3(256), 0, (hipStream_t)stream, (const bf16*)x, ldx,
             (int)H, (int)W, (int)C, (int)stride, (bf16*)out, ldo, (int)kpad, total);
  return fam_host::check_launch("fam_im2col3x3");
}

extern "C" int fam_chan_rmsnorm(const void* x, int64_t ldx, int64_t rows, int64_t C, const void* gamma, int act,
                                void* y, int64_t ldy, void* stream) {
  FAM_REQUIRE(x && gamma && y, FAM_ERR_INVALID_ARG, "fam_chan_rmsnorm: null pointer");
  FAM_REQUIRE(rows >= 0 && C >= 8 && C % 8 == 0 && ldx >= C && ldy >= C && ldx % 8 == 0 && ldy % 8 == 0 &&
                  fam_host::aligned16(x) && fam_host::aligned16(y) && fam_host::aligned16(gamma),
              FAM_ERR_INVALID_ARG, "fam_chan_rmsnorm: C and strides multiples of 8, 16-byte aligned rows");
  FAM_REQUIRE(act == FAM_ACT_NONE || act == FAM_ACT_SILU, FAM_ERR_INVALID_ARG, "fam_chan_rmsnorm: act none or SiLU");
  if (rows == 0) return FAM_OK;
  const auto go = [&](auto kernel, int lpr) {
    FAM_LAUNCH(kernel, dim3(blocks_for(rows, 256 / lpr)), dim3(256), 0, (hipStream_t)stream, (const bf16*)x, ldx, rows,
               (int)C, (const bf16*)gamma, act, (bf16*)y, ldy);
  };
  if (C <= 128) go(chan_rmsnorm_kernel<16, 1>, 16);
  else if (C <= 256) go(chan_rmsnorm_kernel<32, 1>, 32);
  else if (C <= 512) go(chan_rmsnorm_kernel<64, 1>, 64);
  else if (C <= 1024) go(chan_rmsnorm_kernel<64, 2>, 64);
  else go(chan_rmsnorm_kernel<64, 0>, 64);
  return fam_host::check_launch("fam_chan_rmsnorm");
}

extern "C" int fam_vae_avgdown(const void* x, int64_t ldx, int64_t H, int64_t W, int64_t Cin, int64_t Cout,
                               int64_t ft, int64_t fs, const void* add, int64_t ld_add, void* out, int64_t ldo,
                               void* stream) {
  FAM_REQUIRE(x && out, FAM_ERR_INVALID_ARG, "fam_vae_avgdown: null pointer");
  FAM_REQUIRE((ft == 1 || ft == 2) && (fs == 1 || fs == 2) && H % fs == 0 && W % fs == 0 && Cin >= 1 && Cout >= 1 &&
                  (Cin * ft * fs * fs) % Cout == 0 && ldx >= Cin && ldo >= Cout && (!add || ld_add >= Cout) &&
                  H * W < (1LL << 31),
              FAM_ERR_INVALID_ARG, "fam_vae_avgdown: factors 1 or 2 dividing H and W, Cout dividing Cin*ft*fs*fs");
  if (Cout == Cin * ft && Cout % 8 == 0 && ldx % 8 == 0 && ldo % 8 == 0 && fam_host::aligned16(x) &&
      fam_host::aligned16(out) && (!add || (ld_add % 8 == 0 && fam_host::aligned16(add)))) {
    const int64_t n = (H / fs) * (W / fs) * (Cout / 8);
    const auto go = [&](auto kernel) {
      FAM_LAUNCH(kernel, dim3(blocks_for(n, 256)), dim3(256), 0, (hipStream_t)stream, (const bf16*)x, ldx, (int)W,
                 (int)Cout, (const bf16*)add, ld_add, (bf16*)out, ldo, n);
    };
    if (ft == 1 && fs == 1) go(vae_avgdown_vec_kernel<1, 1>);
    else if (ft == 1) go(vae_avgdown_vec_kernel<1, 2>);
    else if (fs == 1) go(vae_avgdown_vec_kernel<2, 1>);
    else go(vae_avgdown_vec_kernel<2, 2>);
    return fam_host::check_launch("fam_vae_avgdown");
  }
  const int64_t total = (H / fs) * (W / fs) * Cout;
  FAM_LAUNCH(vae_avgdown_kernel, dim3(blocks_for(total, 256)), dim3(256), 0, (hipStream_t)stream, (const bf16*)x,
             ldx, (int)H, (int)W, (int)Cin, (int)Cout, (int)ft, (int)fs, (const bf16*)add, ld_add, (bf16*)out, ldo,
             total);
  return fam_host::check_launch("fam_vae_avgdown");
}

extern "C" int fam_softmax_rows(const float* s, int64_t lds, int64_t rows, int64_t cols, float scale, void* p,
                                int64_t ldp, void* stream) {
  FAM_REQUIRE(s && p, FAM_ERR_INVALID_ARG, "fam_softmax_rows: null pointer");
  FAM_REQUIRE(rows >= 0 && cols >= 1 && cols < (1 << 30) && lds >= cols && ldp >= cols && scale > 0.f,
              FAM_ERR_INVALID_ARG, "fam_softmax_rows: need cols >= 1, strides >= cols, scale > 0");
  if (rows == 0) return FAM_OK;
  FAM_LAUNCH(softmax_rows_kernel, dim3(blocks_for(rows, 4)), dim3(256), 0, (hipStream_t)stream, s, lds, rows,
             (int)cols, scale, (bf16*)p, ldp);
  return fam_host::check_launch("fam_softmax_rows");
}

extern "C" int fam_chan_affine_nchw(const void* x, int64_t ldx, int64_t P, int64_t C, const float* mean,
                                    const float* inv_std, void* out, void* stream) {
  FAM_REQUIRE(x && mean && inv_std && out, FAM_ERR_INVALID_ARG, "fam_chan_affine_nchw: null pointer");
  FAM_REQUIRE(P >= 1 && C >= 1 && ldx >= C && P * C < (1LL << 40), FAM_ERR_INVALID_ARG,
              "fam_chan_affine_nchw: need P, C >= 1 and ldx >= C");
  const int64_t total = P * C;
  FAM_LAUNCH(chan_affine_nchw_kernel, dim3(blocks_for(total, 256)), dim3(256), 0, (hipStream_t)stream, (const bf16*)x,
             ldx, P, (int)C, mean, inv_std, (bf16*)out, total);
  return fam_host::check_launch("fam_chan_affine_nchw");
}
