// Convolutions with groups > 1 at the int32 contract: exact products of the int32 values, nothing is narrowed.
#include "conv_mfma.h"

namespace cvmhip {

// Any grouping: direct convolution, what the reference does for grouped filters (ops.cc:333-366).
__global__ void __launch_bounds__(256)
k_conv_grouped(const int32_t* __restrict__ x, const int32_t* __restrict__ w, const int32_t* __restrict__ bias,
               int32_t* __restrict__ y, int64_t total, int ic, int h, int wd, int oc, int oh, int ow, int kh, int kw,
               int sh, int sw, int ph, int pw, int dh, int dw, int icg, int ocg) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += stride) {
    const int q = (int)(i % ow);
    const int p = (int)((i / ow) % oh);
    const int o = (int)((i / ((int64_t)ow * oh)) % oc);
    const int64_t b = i / ((int64_t)ow * oh * oc);
    const int cbase = (o / ocg) * icg;
    int32_t acc = 0;
    for (int c = 0; c < icg; ++c) {
      const int32_t* xc = x + ((int64_t)b * ic + cbase + c) * h * wd;
      const int32_t* wc = w + ((int64_t)o * icg + c) * kh * kw;
      for (int r = 0; r < kh; ++r) {
        const int ih = p * sh + r * dh - ph;
        if (ih < 0 || ih >= h) continue;
        for (int t = 0; t < kw; ++t) {
          const int iw = q * sw + t * dw - pw;
          if (iw < 0 || iw >= wd) continue;
          acc = wadd(acc, wmul(xc[(int64_t)ih * wd + iw], wc[r * kw + t]));
        }
      }
    }
    y[i] = wadd(acc, bias ? bias[o] : 0);
  }
}

// One input channel per group (depthwise, with or without a channel multiplier), filter rows of KW taps, any strides and
// dilation: four neighbouring outputs of a row per thread, so a row of the window is read once for four outputs, and the
// filter, which is the same for a whole workgroup (one output plane), comes through the scalar cache.
template <int KH, int KW, bool UNIT>
__global__ void __launch_bounds__(256)
k_conv_planes(const int32_t* __restrict__ x, const int32_t* __restrict__ w, const int32_t* __restrict__ bias, int32_t* __restrict__ y,
              int planes, int ic, int h, int wd, int oc, int oh, int ow, int sh, int sw, int ph, int pw, int dh, int dw, int ocg,
              FastDiv div_quads) {
  const int quads = (ow + 3) >> 2;
  for (int plane = blockIdx.y; plane < planes; plane += gridDim.y) {
    const int b = plane / oc, o = plane - b * oc;
    const int32_t* xc = x + ((int64_t)b * ic + o / ocg) * h * wd;
    const int32_t* wc = w + (int64_t)o * KH * KW;
    const int32_t b0 = bias ? bias[o] : 0;
    const int lin = blockIdx.x * 256 + threadIdx.x;
    if (lin >= oh * quads) continue;
    const int p = (int)fastdiv((unsigned)lin, div_quads), q = (lin - p * quads) * 4;
    // every load of the window is issued, from the nearest pixel inside, and masked afterwards; at stride 1 the windows
    // of the four outputs share their columns
    constexpr int COLS = UNIT ? KW + 3 : 4 * KW;
    int32_t v[KH][COLS];
#pragma unroll
    for (int r = 0; r < KH; ++r) {
      const int ih = p * sh + r * dh - ph;
      const int32_t* xr = xc + (int64_t)(ih < 0 ? 0 : (ih < h ? ih : h - 1)) * wd;
#pragma unroll
      for (int e = 0; e < COLS; ++e) {
        const int iw = UNIT ? q + e - pw : (q + e / KW) * sw + (e % KW) * dw - pw;
        v[r][e] = xr[iw < 0 ? 0 : (iw < wd ? iw : wd - 1)];
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    int32_t acc[4] = {b0, b0, b0, b0};
#pragma unroll
    for (int r = 0; r < KH; ++r) {
      const int ih = p * sh + r * dh - ph;
      const bool row = ih >= 0 && ih < h;
#pragma unroll
      for (int e = 0; e < COLS; ++e) {
        const int iw = UNIT ? q + e - pw : (q + e / KW) * sw + (e % KW) * dw - pw;
        v[r][e] = row && iw >= 0 && iw < wd ? v[r][e] : 0;
      }
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int t = 0; t < KW; ++t) acc[u] = wadd(acc[u], wmul(v[r][UNIT ? u + t : u * KW + t], wc[r * KW + t]));
    }
    int32_t* yr = y + (int64_t)plane * oh * ow + (int64_t)p * ow + q;
    typedef int v4i __attribute__((ext_vector_type(4), aligned(4)));   // rows need not start on 16 bytes
    if (q + 3 < ow) {
      *reinterpret_cast<v4i*>(yr) = v4i{acc[0], acc[1], acc[2], acc[3]};
    } else {
#pragma unroll
      for (int u = 0; u < 3; ++u)
        if (q + u < ow) yr[u] = acc[u];
    }
  }
}

// The same for a 3 x 3 filter without dilation whose strides are both S (every depthwise layer of a MobileNet): four columns of
// ROWS output rows per thread.  What bounded the form above on 4 x 96 x 75 x 75 (13.4 us, 17 MB) was its loads, 18 of
// four bytes per thread that each touched 16 lines for 64 lanes, then the 32-bit multiplies (a quarter of the rate of an
// add) and the masks.  Here an input row of the window is one or two 16-byte loads and a remainder, and serves up to three output rows;
// where all values of a wavefront and the filter fit in 24 bits the products are v_mad_i32_i24, which keep the low 32 bits of
// the product like the wrapping multiply and run at full rate.  4 x 96 x 75 x 75: 12.3 -> 6.1 us; 8 x 256 x 96 x 96: 76 -> 28 us (5.4 TB/s),
// with stride 2 80 -> 17 us; planes of 7 x 7 as before (2.7-2.8 us, a launch).
// Rows are read past their ends (the columns outside are masked), never past the tensor: a thread that would takes the clamped loads.
template <int S, int ROWS>
__global__ void __launch_bounds__(128)
k_conv_planes_rows(const int32_t* __restrict__ x, const int32_t* __restrict__ w, const int32_t* __restrict__ bias, int32_t* __restrict__ y,
                   int planes, int ic, int h, int wd, int oc, int oh, int ow, int ph, int pw, int ocg, int64_t elements,
                   FastDiv div_quads) {
  typedef int v4i __attribute__((ext_vector_type(4), aligned(4)));
  typedef int v2i __attribute__((ext_vector_type(2), aligned(4)));
  constexpr int COLS = 3 * S + 3, IN = (ROWS - 1) * S + 3;
  const int quads = (ow + 3) >> 2, groups = (oh + ROWS - 1) / ROWS;
  for (int plane = blockIdx.y; plane < planes; plane += gridDim.y) {
    const int b = plane / oc, o = plane - b * oc;
    const int64_t first = ((int64_t)b * ic + o / ocg) * h * wd;
    const int32_t* xc = x + first;
    const int32_t* wc = w + (int64_t)o * 9;
    const int32_t b0 = bias ? bias[o] : 0;
    const int lin = blockIdx.x * 128 + threadIdx.x;
    if (lin >= groups * quads) continue;
    const int g = (int)fastdiv((unsigned)lin, div_quads), q = (lin - g * quads) * 4, p = g * ROWS;
    const int iw0 = q * S - pw, ih0 = p * S - ph;
    int32_t v[IN][COLS];
    const int top = ih0 < 0 ? 0 : (ih0 < h ? ih0 : h - 1), bottom = ih0 + IN - 1 < 0 ? 0 : (ih0 + IN - 1 < h ? ih0 + IN - 1 : h - 1);
    if (first + (int64_t)top * wd + iw0 >= 0 && first + (int64_t)bottom * wd + iw0 + COLS <= elements) {
#pragma unroll
      for (int r = 0; r < IN; ++r) {
        const int ih = ih0 + r;
        const int32_t* xr = xc + ((ih < 0 ? 0 : (ih < h ? ih : h - 1)) * wd + iw0);
        const v4i a = *reinterpret_cast<const v4i*>(xr);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[r][e] = a[e];
        if constexpr (S == 1) {
          const v2i c = *reinterpret_cast<const v2i*>(xr + 4);
          v[r][4] = c[0];
          v[r][5] = c[1];
        } else {
          const v4i c = *reinterpret_cast<const v4i*>(xr + 4);
#pragma unroll
          for (int e = 0; e < 4; ++e) v[r][4 + e] = c[e];
          v[r][8] = xr[8];
        }
      }
    } else {
#pragma unroll
      for (int r = 0; r < IN; ++r) {
        const int ih = ih0 + r;
        const int32_t* xr = xc + (ih < 0 ? 0 : (ih < h ? ih : h - 1)) * wd;
#pragma unroll
        for (int e = 0; e < COLS; ++e) {
          const int iw = iw0 + e;
          v[r][e] = xr[iw < 0 ? 0 : (iw < wd ? iw : wd - 1)];
        }
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    int32_t column[COLS];
#pragma unroll
    for (int e = 0; e < COLS; ++e) column[e] = (unsigned)(iw0 + e) < (unsigned)wd ? -1 : 0;
    int32_t wide = 0;   // above 2^23 if some value does not fit in 24 bits
#pragma unroll
    for (int r = 0; r < IN; ++r) {
#pragma unroll
      for (int e = 0; e < COLS; ++e) v[r][e] &= column[e];
      if ((unsigned)(ih0 + r) >= (unsigned)h)
#pragma unroll
        for (int e = 0; e < COLS; ++e) v[r][e] = 0;
#pragma unroll
      for (int e = 0; e < COLS; ++e) wide |= v[r][e] ^ (v[r][e] >> 31);
    }
    int32_t wt[9], wwide = 0;
#pragma unroll
    for (int t = 0; t < 9; ++t) {
      wt[t] = wc[t];
      wwide |= wt[t] ^ (wt[t] >> 31);
    }
    int32_t acc[ROWS][4];
#pragma unroll
    for (int rr = 0; rr < ROWS; ++rr)
#pragma unroll
      for (int u = 0; u < 4; ++u) acc[rr][u] = b0;
    if (!__any((wide | wwide) >= (1 << 23))) {
#pragma unroll
      for (int rr = 0; rr < ROWS; ++rr)
#pragma unroll
        for (int t = 0; t < 9; ++t)
#pragma unroll
          for (int u = 0; u < 4; ++u) acc[rr][u] = wadd(acc[rr][u], __mul24(v[rr * S + t / 3][u * S + t % 3], wt[t]));
    } else {
#pragma unroll
      for (int rr = 0; rr < ROWS; ++rr)
#pragma unroll
        for (int t = 0; t < 9; ++t)
#pragma unroll
          for (int u = 0; u < 4; ++u) acc[rr][u] = wadd(acc[rr][u], wmul(v[rr * S + t / 3][u * S + t % 3], wt[t]));
    }
    int32_t* yp = y + (int64_t)plane * oh * ow + (int64_t)p * ow + q;
#pragma unroll
    for (int rr = 0; rr < ROWS; ++rr) {
      if (p + rr >= oh) break;
      int32_t* yr = yp + (int64_t)rr * ow;
      if (q + 3 < ow) {
        *reinterpret_cast<v4i*>(yr) = v4i{acc[rr][0], acc[rr][1], acc[rr][2], acc[rr][3]};
      } else {
#pragma unroll
        for (int u = 0; u < 3; ++u)
          if (q + u < ow) yr[u] = acc[rr][u];
      }
    }
  }
}

// Four rows to a thread read an input row 1.5 times instead of 3 and leave a quarter of the threads.  One row against four, us: 96 planes
// of 14 x 14 to 256 of 33 x 33 (0.3 M outputs) 2.8-3.4 against 3.6-3.7; 2.2 M outputs 7.4 against 6.1; 18.9 M 35.2 against 28.1.  With
// stride 2 one row is the better everywhere (18.9 M inputs: 16.6 against 17.2 for two): only one of three rows is shared.
constexpr int64_t CONV_PLANES_TALL = 1 << 20;

int conv_grouped_i32(const int32_t* x, const int32_t* w, const int32_t* bias, int32_t* y, int n, int ic, int h, int wd, int oc, int oh, int ow,
                     int kh, int kw, int stride_h, int stride_w, int pad_h, int pad_w, int dil_h, int dil_w, int groups, hipStream_t s) {
  const int64_t total = (int64_t)n * oc * oh * ow;
  const int64_t quads = (ow + 3) / 4, planes = (int64_t)n * oc;
  if (ic == groups && kh == 3 && kw == 3 && planes < INT32_MAX && oh * quads < INT32_MAX && (int64_t)h * wd < INT32_MAX) {
    const unsigned gy = (unsigned)(planes < 65535 ? planes : 65535);
    const FastDiv div_quads = make_fastdiv((uint32_t)quads);
    if (stride_h == stride_w && stride_w <= 2 && dil_h == 1 && dil_w == 1) {
      auto launch = [&](auto kernel, int rows) {
        const int64_t items = (oh + rows - 1) / rows * quads;
        kernel<<<dim3((unsigned)((items + 127) / 128), gy), 128, 0, s>>>(x, w, bias, y, (int)planes, ic, h, wd, oc, oh, ow, pad_h, pad_w, oc / groups,
                                                                       (int64_t)n * ic * h * wd, div_quads);
      };
      if (stride_w == 2) launch(k_conv_planes_rows<2, 1>, 1);
      else if (total >= CONV_PLANES_TALL) launch(k_conv_planes_rows<1, 4>, 4);
      else launch(k_conv_planes_rows<1, 1>, 1);
      return check_launch("conv_planes_rows");
    }
    const dim3 grid((unsigned)((oh * quads + 255) / 256), gy);
    if (stride_w == 1 && dil_w == 1)
      k_conv_planes<3, 3, true><<<grid, 256, 0, s>>>(x, w, bias, y, (int)planes, ic, h, wd, oc, oh, ow, stride_h, stride_w, pad_h, pad_w, dil_h,
                                                     dil_w, oc / groups, div_quads);
    else
      k_conv_planes<3, 3, false><<<grid, 256, 0, s>>>(x, w, bias, y, (int)planes, ic, h, wd, oc, oh, ow, stride_h, stride_w, pad_h, pad_w, dil_h,
                                                      dil_w, oc / groups, div_quads);
    return check_launch("conv_planes");
  }
  k_conv_grouped<<<grid_for(total, 256, 1 << 20), 256, 0, s>>>(x, w, bias, y, total, ic, h, wd, oc, oh, ow, kh, kw, stride_h, stride_w, pad_h, pad_w,
                                                             dil_h, dil_w, ic / groups, oc / groups);
  return check_launch("conv_grouped");
}

}  // namespace cvmhip
