// The image stages either side of the two networks, on the GPU, each with
// the reference's CPU arithmetic so the bytes and floats are identical:
//  - OpenCV's 8-bit bilinear resize (src/image.rs:33-142);
//  - the detector's input tensor from a page (src/det.rs:195-289);
//  - the recogniser's input tensor from a crop (src/rec.rs:10-43);
//  - the perspective text crop with bicubic sampling (src/crop.rs:1-127).
// Inputs and outputs are device memory, HWC. Every table a thread needs (a
// resize tap, a normalisation) is computed in the thread from the same
// integer and IEEE f32 / f64 operations the CPU performs, so no call
// allocates or uploads anything beyond its arguments.
#include "kernels.hpp"

namespace ppocr {

struct Tap {
  int near_i, far_i, near_w, far_w;
};

// Output coordinate d of a src -> dst resize: OpenCV's source position
// (d + 0.5) * scale - 0.5 rounded to f32, each 1/2048 weight rounded on its
// own, taps past an edge on the edge.
__host__ __device__ inline double tap_scale(int src, int dst) { return 1.0 / ((double)dst / (double)src); }
__device__ __forceinline__ Tap tap_at(int src, double scale, int d) {
  const float f = (float)(((double)d + 0.5) * scale - 0.5);
  const float fl = floorf(f);
  const float a = f - fl;
  const int s = (int)fl, last = src - 1;
  Tap t;
  t.near_i = min(max(s, 0), last);
  t.far_i = min(max(s + 1, 0), last);
  t.near_w = (int)rintf((1.0f - a) * 2048.0f);
  t.far_w = (int)rintf(a * 2048.0f);
  return t;
}
__device__ __forceinline__ Tap tap_at(int src, int dst, int d) { return tap_at(src, tap_scale(src, dst), d); }

// One output value from its four source values (near / far row, near / far
// column): horizontal products kept whole, then 4 bits off each row before
// its weight, 16 after, the sum rounded by 2 bits.
__device__ __forceinline__ int resize_mix(int nn, int nf, int fn, int ff, const Tap &tx, const Tap &ty) {
  const int a = nn * tx.near_w + nf * tx.far_w;
  const int b = fn * tx.near_w + ff * tx.far_w;
  const int v = (((a >> 4) * ty.near_w) >> 16) + (((b >> 4) * ty.far_w) >> 16);
  return min(max((v + 2) >> 2, 0), 255);
}

// Channel c of output pixel (x, y) of a resize of `src`.
__device__ __forceinline__ int resize_at(const uint8_t *src, int sw, const Tap &tx, const Tap &ty, int c) {
  const uint8_t *rn = src + (long)ty.near_i * sw * 3, *rf = src + (long)ty.far_i * sw * 3;
  return resize_mix(rn[tx.near_i * 3 + c], rn[tx.far_i * 3 + c], rf[tx.near_i * 3 + c], rf[tx.far_i * 3 + c],
                    tx, ty);
}

__global__ __launch_bounds__(256) void resize_kernel(const uint8_t *src, int sw, int sh, uint8_t *dst, int dw,
                                                     int dh) {
  const long g = (long)blockIdx.x * 256 + threadIdx.x;
  if (g >= (long)dw * dh) return;
  const int y = (int)(g / dw), x = (int)(g - (long)y * dw);
  const Tap tx = tap_at(sw, dw, x), ty = tap_at(sh, dh, y);
#pragma unroll
  for (int c = 0; c < 3; c++) dst[g * 3 + c] = (uint8_t)resize_at(src, sw, tx, ty, c);
}

struct __attribute__((packed, aligned(1))) Bytes8 {
  uint32_t w[2];
};

// The detector input: resized, x = v * (1/255 as f32), (x - mean) / std in
// f64, rounded once to f32. A resized value is one of 256: the block first
// makes each one's three results, one value a thread, so that the f64
// divisions are paid once for its `per` pixels a thread. Two neighbouring
// source pixels of a row come by one eight-byte load (at any alignment)
// where that stays in the row. Bound by the integer work of a pixel.
// Measured, 2550 x 3300 to 1536 x 1984: 26.4 us with the divisions per pixel
// and byte loads, now 17.4; to 736 x 960 9.9 and 6.8; 1100 x 700 to 1024 x 512
// 6.5 and 5.6; 331 x 223 to 320 x 224 4.1 both.
__global__ __launch_bounds__(256) void det_input_kernel(const uint8_t *src, int sw, int sh, float *out, int dw,
                                                        int dh, int per, double xscale, double yscale, double m0,
                                                        double m1, double m2, double s0, double s1, double s2) {
  __shared__ float value[3][256];
  {
    const float v = (float)threadIdx.x * (float)(1.0 / 255.0);
    value[0][threadIdx.x] = (float)(((double)v - m0) / s0);
    value[1][threadIdx.x] = (float)(((double)v - m1) / s1);
    value[2][threadIdx.x] = (float)(((double)v - m2) / s2);
  }
  __syncthreads();
  const long total = (long)dw * dh;
  for (int k = 0; k < per; k++) {
    const long g = ((long)blockIdx.x * per + k) * 256 + threadIdx.x;
    if (g >= total) return;
    const int y = (int)(g / dw), x = (int)(g - (long)y * dw);
    const Tap tx = tap_at(sw, xscale, x), ty = tap_at(sh, yscale, y);
    if (tx.far_i == tx.near_i + 1 && tx.near_i + 2 < sw) {
      const Bytes8 n = *reinterpret_cast<const Bytes8 *>(src + ((long)ty.near_i * sw + tx.near_i) * 3);
      const Bytes8 f = *reinterpret_cast<const Bytes8 *>(src + ((long)ty.far_i * sw + tx.near_i) * 3);
      auto byte = [](const Bytes8 &b, int i) { return (int)(b.w[i / 4] >> (8 * (i % 4)) & 255u); };
#pragma unroll
      for (int c = 0; c < 3; c++)
        out[g * 3 + c] = value[c][resize_mix(byte(n, c), byte(n, 3 + c), byte(f, c), byte(f, 3 + c), tx, ty)];
    } else {
#pragma unroll
      for (int c = 0; c < 3; c++) out[g * 3 + c] = value[c][resize_at(src, sw, tx, ty, c)];
    }
  }
}

// The recogniser input: 48 rows of `width`; the crop resized to rw columns
// and scaled to [-1, 1] in f32, zeros right of it.
__global__ __launch_bounds__(256) void rec_input_kernel(const uint8_t *src, int sw, int sh, float *out, int width,
                                                        int rw) {
  const long g = (long)blockIdx.x * 256 + threadIdx.x;
  if (g >= 48L * width) return;
  const int y = (int)(g / width), x = (int)(g - (long)y * width);
  if (x >= rw) {
#pragma unroll
    for (int c = 0; c < 3; c++) out[g * 3 + c] = 0.0f;
    return;
  }
  const Tap tx = tap_at(sw, rw, x), ty = tap_at(sh, 48, y);
#pragma unroll
  for (int c = 0; c < 3; c++) out[g * 3 + c] = ((float)resize_at(src, sw, tx, ty, c) / 255.0f - 0.5f) / 0.5f;
}

// Keys' cubic weights, a = -0.75, in OpenCV's factoring.
__device__ __forceinline__ void cubic(float t, float *w) {
  const float A = -0.75f;
  w[0] = ((A * (t + 1.0f) - 5.0f * A) * (t + 1.0f) + 8.0f * A) * (t + 1.0f) - 4.0f * A;
  w[1] = ((A + 2.0f) * t - (A + 3.0f)) * t * t + 1.0f;
  w[2] = ((A + 2.0f) * (1.0f - t) - (A + 3.0f)) * (1.0f - t) * (1.0f - t) + 1.0f;
  w[3] = 1.0f - w[0] - w[1] - w[2];
}

struct __attribute__((packed, aligned(1))) Bytes12 {
  uint32_t w[3];
};

// Pixel (x, y) of a crop rectangle: its source point through the
// projective map m (f64, then f32), the 4 x 4 bicubic window with edge pixels
// repeated, each row of four summed before the rows, rounded to 8 bits.
__device__ __forceinline__ void crop_pixel(const uint8_t *img, int iw, int ih, const CropMap &m, int x, int y,
                                           int v[3]) {
  const double xf = x, yf = y;
  double w = m.v[6] * xf + m.v[7] * yf + m.v[8];
  w = w == 0.0 ? 0.0 : 1.0 / w;
  const float sx = (float)((m.v[0] * xf + m.v[1] * yf + m.v[2]) * w);
  const float sy = (float)((m.v[3] * xf + m.v[4] * yf + m.v[5]) * w);
  const float fx = floorf(sx), fy = floorf(sy);
  float wx[4], wy[4];
  cubic(sx - fx, wx);
  cubic(sy - fy, wy);
  // The window's corner as an integer: a NaN reads as 0 and anything far
  // outside the image lands on its edge, as a saturating conversion does.
  const float kFar = 1073741824.0f;
  const long ix = (long)(isnan(fx) ? 0.0f : fminf(fmaxf(fx, -kFar), kFar)) - 1;
  const long iy = (long)(isnan(fy) ? 0.0f : fminf(fmaxf(fy, -kFar), kFar)) - 1;
  float acc[3] = {0.0f, 0.0f, 0.0f};
  const bool inside = ix >= 0 && ix + 3 < iw && iy >= 0 && iy + 3 < ih;
  // A window inside the image: each row's four pixels are twelve bytes in a
  // row, one load (at any alignment) for twelve.
  Bytes12 rows[4];
  if (inside) {
#pragma unroll
    for (int j = 0; j < 4; j++) rows[j] = *reinterpret_cast<const Bytes12 *>(img + ((iy + j) * iw + ix) * 3);
  } else {
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const uint8_t *row = img + min(max(iy + j, 0L), (long)ih - 1) * iw * 3;
      rows[j] = Bytes12{{0, 0, 0}};
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const uint8_t *p = row + min(max(ix + i, 0L), (long)iw - 1) * 3;
#pragma unroll
        for (int c = 0; c < 3; c++) rows[j].w[(3 * i + c) / 4] |= (uint32_t)p[c] << (8 * ((3 * i + c) % 4));
      }
    }
  }
#pragma unroll
  for (int j = 0; j < 4; j++) {
    float line[3] = {0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
      for (int c = 0; c < 3; c++)
        line[c] += (float)(rows[j].w[(3 * i + c) / 4] >> (8 * ((3 * i + c) % 4)) & 255u) * wx[i];
#pragma unroll
    for (int c = 0; c < 3; c++) acc[c] += line[c] * wy[j];
  }
#pragma unroll
  for (int c = 0; c < 3; c++) v[c] = (int)fminf(fmaxf(rintf(acc[c]), 0.0f), 255.0f);
}

// One crop pixel (x, y) of the width x height rectangle, written turned a
// quarter counter-clockwise when `turn`.
__global__ __launch_bounds__(256) void crop_kernel(const uint8_t *img, int iw, int ih, CropMap m, uint8_t *out,
                                                   int width, int height, int turn) {
  const long g = (long)blockIdx.x * 256 + threadIdx.x;
  if (g >= (long)width * height) return;
  const int y = (int)(g / width), x = (int)(g - (long)y * width);
  int v[3];
  crop_pixel(img, iw, ih, m, x, y, v);
  const long at = turn ? ((long)(width - 1 - x) * height + y) : g;
#pragma unroll
  for (int c = 0; c < 3; c++) out[at * 3 + c] = (uint8_t)v[c];
}

// The recogniser inputs of up to kCropLines crops in one launch, without the
// crops in memory: tile (blockIdx.x, blockIdx.y) of line blockIdx.z, 16 x 8
// pixels of its 48 x width tensor. The block first computes the crop pixels
// that the tile's resize taps name, each once, as crop_kernel computes it
// (through the turn when the crop is turned), into LDS: the range the taps
// span, or, when the crop is over twice the tensor's size, each tap's own two
// columns or rows. Then the resize and the [-1, 1] scaling of
// rec_input_kernel: the same values as crop_text then rec_input.
//
// Bound by the bicubic sums' vector work. Measured on 16 tilted lines of
// about 580 x 42 pixels (615 K tensor pixels): 12.7 us (40.5
// with every tensor pixel computing its own four crop pixels byte by byte).
constexpr int kCropTX = 16, kCropTY = 8;

__global__ __launch_bounds__(256) void crop_rec_kernel(const uint8_t *img, int iw, int ih, CropLines b) {
  __shared__ Tap taps[kCropTX + kCropTY];
  __shared__ uint32_t px[4 * kCropTX * kCropTY];
  const CropLine &L = b.l[blockIdx.z];
  const int x0 = blockIdx.x * kCropTX, y0 = blockIdx.y * kCropTY, tid = threadIdx.x;
  if (x0 >= L.width) return;
  const int nx = min(kCropTX, L.rw - x0);  // columns that hold the crop
  const int sw = L.turn ? L.ch : L.cw, sh = L.turn ? L.cw : L.ch;  // the crop image's sides
  if (nx > 0) {
    if (tid < kCropTX + kCropTY)
      taps[tid] = tid < kCropTX ? tap_at(sw, L.rw, min(x0 + tid, L.rw - 1)) : tap_at(sh, 48, y0 + tid - kCropTX);
    __syncthreads();
    const Tap *tx = taps, *ty = taps + kCropTX;
    const int cx0 = tx[0].near_i, cy0 = ty[0].near_i;
    const int wide = tx[nx - 1].far_i - cx0 + 1, high = ty[kCropTY - 1].far_i - cy0 + 1;
    const bool run_x = wide <= 2 * nx, run_y = high <= 2 * kCropTY;
    const int nc = run_x ? wide : 2 * nx, nr = run_y ? high : 2 * kCropTY;
    for (int k = tid; k < nc * nr; k += 256) {
      const int r = k / nc, c = k - r * nc;
      const int cx = run_x ? cx0 + c : ((c & 1) ? tx[c >> 1].far_i : tx[c >> 1].near_i);
      const int cy = run_y ? cy0 + r : ((r & 1) ? ty[r >> 1].far_i : ty[r >> 1].near_i);
      int v[3];
      // Crop image pixel (cx, cy) is rectangle pixel (cw - 1 - cy, cx) when turned.
      crop_pixel(img, iw, ih, L.m, L.turn ? L.cw - 1 - cy : cx, L.turn ? cx : cy, v);
      px[k] = (uint32_t)v[0] | (uint32_t)v[1] << 8 | (uint32_t)v[2] << 16;
    }
    __syncthreads();
    const int i = tid % kCropTX, j = tid / kCropTX;
    if (j < kCropTY && i < nx) {
      const Tap ax = tx[i], ay = ty[j];
      const int c0 = run_x ? ax.near_i - cx0 : 2 * i, c1 = run_x ? ax.far_i - cx0 : 2 * i + 1;
      const int r0 = run_y ? ay.near_i - cy0 : 2 * j, r1 = run_y ? ay.far_i - cy0 : 2 * j + 1;
      const uint32_t nn = px[r0 * nc + c0], nf = px[r0 * nc + c1], fn = px[r1 * nc + c0], ff = px[r1 * nc + c1];
      float *o = L.out + ((long)(y0 + j) * L.width + x0 + i) * 3;
#pragma unroll
      for (int c = 0; c < 3; c++)
        o[c] = ((float)resize_mix(nn >> (8 * c) & 255, nf >> (8 * c) & 255, fn >> (8 * c) & 255, ff >> (8 * c) & 255,
                                  ax, ay) / 255.0f - 0.5f) / 0.5f;
    }
  }
  // Zeros right of the crop.
  const int i = tid % kCropTX, j = tid / kCropTX;
  if (j < kCropTY && i >= nx && x0 + i < L.width) {
    float *o = L.out + ((long)(y0 + j) * L.width + x0 + i) * 3;
#pragma unroll
    for (int c = 0; c < 3; c++) o[c] = 0.0f;
  }
}

static unsigned blocks(long n) { return (unsigned)((n + 255) / 256); }

hipError_t launch_resize(const uint8_t *src, int sw, int sh, uint8_t *dst, int dw, int dh, hipStream_t s) {
  hipLaunchKernelGGL(resize_kernel, dim3(blocks((long)dw * dh)), dim3(256), 0, s, src, sw, sh, dst, dw, dh);
  return hipGetLastError();
}

hipError_t launch_det_input(const uint8_t *src, int sw, int sh, float *out, int dw, int dh, const double *mean,
                            const double *sd, hipStream_t s) {
  // Two pixels a thread, four from 2^21 pixels on: the fewer, the more blocks
  // hide the loads; the more, the fewer tables. Eight left about a block a CU
  // at 2^19: 1100 x 700 to 1024 x 512 8.6 us, and 6.5 without tables.
  const long n = (long)dw * dh;
  const int per = n >= (1L << 21) ? 4 : 2;
  hipLaunchKernelGGL(det_input_kernel, dim3(blocks((n + per - 1) / per)), dim3(256), 0, s, src, sw, sh, out, dw, dh, per,
                     tap_scale(sw, dw), tap_scale(sh, dh), mean[0], mean[1], mean[2], sd[0], sd[1], sd[2]);
  return hipGetLastError();
}

hipError_t launch_rec_input(const uint8_t *src, int sw, int sh, float *out, int width, int rw, hipStream_t s) {
  hipLaunchKernelGGL(rec_input_kernel, dim3(blocks(48L * width)), dim3(256), 0, s, src, sw, sh, out, width, rw);
  return hipGetLastError();
}

hipError_t launch_crop_rec(const uint8_t *img, int iw, int ih, const CropLines &b, hipStream_t s) {
  if (b.n <= 0 || b.n > kCropLines) return hipErrorInvalidValue;
  int widest = 0;
  for (int i = 0; i < b.n; i++) widest = max(widest, b.l[i].width);
  hipLaunchKernelGGL(crop_rec_kernel, dim3((unsigned)((widest + kCropTX - 1) / kCropTX), 48 / kCropTY, (unsigned)b.n),
                     dim3(256), 0, s, img, iw, ih, b);
  return hipGetLastError();
}

hipError_t launch_crop(const uint8_t *img, int iw, int ih, const CropMap &m, uint8_t *out, int width, int height,
                       bool turn, hipStream_t s) {
  hipLaunchKernelGGL(crop_kernel, dim3(blocks((long)width * height)), dim3(256), 0, s, img, iw, ih, m, out, width,
                     height, turn ? 1 : 0);
  return hipGetLastError();
}

}  // namespace ppocr
