// k_jpeg.hip -- baseline JPEG encoding on the GPU for the o-jpg sink
// (reference o-jpg/main.c:101-160, which hands rgb scanlines to libjpeg with
// optimised Huffman coding).  The steps are libjpeg's published ones (ITU-T
// T.81 baseline with IJG's choices), so the file's tables and entropy-coded
// data are those libjpeg writes for the same image and settings:
//   k_jpg_front   a strip of MCUs per work group: fixed-point YCbCr, 2:1 chroma
//                 boxes with the alternating bias, samples past the edges
//                 replicated, the islow, ifast or float DCT (rows in
//                 registers, columns through LDS) and its quantisation, the
//                 blocks of the last MCUs past a component's own extent
//                 (zero, with the DC of the block to the left / above), and
//                 the symbol counts of the four tables; coefficients stored
//                 in zigzag order
//   k_jpg_dc0     the DC symbols of the strips' first MCUs
//   k_jpg_coef, k_jpg_dummy, k_jpg_stats   the same one lane a block, for
//                 libjpeg's smoothing filter, which reads past its block
//   (host)        optimal code lengths per table (T.81 K.2, K.3)
//   k_jpg_code<0> bits per 256 blocks; k_jpg_scan their offsets
//   k_jpg_code<1> each work group's codes into LDS at their bit offsets, then
//                 to memory in whole words (most significant bit first)
//   k_stuff_*     a zero byte after every 0xFF: counts per chunk, offsets,
//                 scatter
#include "launch.h"

#include <algorithm>
#include <stdlib.h>
#include <string.h>
#include <type_traits>
#include <vector>

namespace {

static const uint8_t jz_host[64] = {
  0, 1, 8, 16, 9, 2, 3, 10, 17, 24, 32, 25, 18, 11, 4, 5, 12, 19, 26, 33, 40, 48, 41, 34, 27, 20, 13, 6, 7, 14, 21,
  28, 35, 42, 49, 56, 57, 50, 43, 36, 29, 22, 15, 23, 30, 37, 44, 51, 58, 59, 52, 45, 38, 31, 39, 46, 53, 60, 61, 54,
  47, 55, 62, 63 };

struct jpg_geom
{
  const uint8_t *rgba;       // device, 4 bytes a pixel
  int W, H, pitch;           // pitch in pixels
  int hs, vs, bpm;           // luma sampling, blocks per MCU
  int mx, my, nb;            // MCUs across, down; blocks
  int wib[3], hib[3];        // each component's own extent in blocks
  int smooth;                // libjpeg's smoothing_factor, 0..100
};

// block b -> component, block column and row
DEV void jpg_block(const jpg_geom &g, int b, int &c, int &bx, int &by, int &i)
{
  const int m = b / g.bpm, r = b - m * g.bpm, n0 = g.hs * g.vs;
  const int ux = m % g.mx, uy = m / g.mx;
  if(r < n0) { c = 0; i = r % g.hs; bx = ux * g.hs + i; by = uy * g.vs + r / g.hs; }
  else { c = r - n0 + 1; i = 0; bx = ux; by = uy; }
}

DEV void jpg_ycc(const jpg_geom &g, int x, int y, int &Y, int &cb, int &cr)
{
  x = x < 0 ? 0 : (x < g.W ? x : g.W - 1);
  y = y < 0 ? 0 : (y < g.H ? y : g.H - 1);
  const uchar4 p = *(const uchar4 *)(g.rgba + 4 * ((long)y * g.pitch + x));
  const int r = p.x, gg = p.y, b = p.z;
  // 16-bit fixed point: round(0.299 * 65536) etc.
  Y  = (19595 * r + 38470 * gg + 7471 * b + 32768) >> 16;
  cb = (-11059 * r - 21709 * gg + 32768 * b + (128 << 16) + 32767) >> 16;
  cr = (32768 * r - 27439 * gg - 5329 * b + (128 << 16) + 32767) >> 16;
}

DEV int jpg_comp(const jpg_geom &g, int c, int x, int y)
{ // full-resolution sample of component c, replicated past the edges
  int v[3];
  jpg_ycc(g, x, y, v[0], v[1], v[2]);
  return v[c];
}

// libjpeg's input smoothing (smoothing_factor sf): a full-size component
// mixes a sample with its 8 neighbours, weights 1 - 8 sf/1024 and sf/1024
// in 16-bit fixed point; 2x2 chroma forms an output from its 4 members
// ((1 - 5 sf/1024)/4 each), their 8 edge neighbours (sf/512) and 4 corner
// neighbours (sf/1024).  2x1 chroma is not smoothed.
DEV int jpg_sample_smooth(const jpg_geom &g, int c, int x, int y)
{
  const int sf = g.smooth;
  if(c == 0 || g.hs * g.vs == 1)
  {
    int n = 0;
#pragma unroll
    for(int j = -1; j <= 1; j++)
#pragma unroll
      for(int i = -1; i <= 1; i++)
        if(i || j) n += jpg_comp(g, c, x + i, y + j);
    return (jpg_comp(g, c, x, y) * (65536 - 512 * sf) + n * (64 * sf) + 32768) >> 16;
  }
  const int X = 2 * x, Y = 2 * y;
  int m = 0, e = 0, k = 0;
#pragma unroll
  for(int j = -1; j <= 2; j++)
#pragma unroll
    for(int i = -1; i <= 2; i++)
    {
      const int v = jpg_comp(g, c, X + i, Y + j);
      const bool ix = i == 0 || i == 1, iy = j == 0 || j == 1;
      if(ix && iy) m += v;
      else if(ix || iy) e += v;
      else k += v;
    }
  return (m * (16384 - 80 * sf) + (2 * e + k) * (16 * sf) + 32768) >> 16;
}

DEV int jpg_sample(const jpg_geom &g, int c, int x, int y)
{
  if(g.smooth && !(c > 0 && g.hs == 2 && g.vs == 1)) return jpg_sample_smooth(g, c, x, y);
  int Y, cb, cr;
  if(c == 0) { jpg_ycc(g, x, y, Y, cb, cr); return Y; }
  int s = 0;
  for(int j = 0; j < g.vs; j++)
    for(int i = 0; i < g.hs; i++)
    {
      jpg_ycc(g, g.hs * x + i, g.vs * y + j, Y, cb, cr);
      s += c == 1 ? cb : cr;
    }
  if(g.hs * g.vs == 1) return s;
  if(g.vs == 2) return (s + ((x & 1) ? 2 : 1)) >> 2;   // 2x2: bias 1, 2, 1, 2, ...
  return (s + (x & 1)) >> 1;                          // 2x1: bias 0, 1, 0, 1, ...
}

#define JC(x) ((int32_t)((x) * 8192.0 + 0.5))
#define JDESC(x, n) (((x) + (1 << ((n) - 1))) >> (n))

// islow forward DCT of 8 values a stride apart (pass 0 rows, 1 columns)
template<int PASS, int S>
DEV void jpg_fdct8(int32_t *p)
{
  const int32_t t0 = p[0] + p[7 * S], t7 = p[0] - p[7 * S], t1 = p[S] + p[6 * S], t6 = p[S] - p[6 * S];
  const int32_t t2 = p[2 * S] + p[5 * S], t5 = p[2 * S] - p[5 * S], t3 = p[3 * S] + p[4 * S], t4 = p[3 * S] - p[4 * S];
  const int32_t t10 = t0 + t3, t13 = t0 - t3, t11 = t1 + t2, t12 = t1 - t2;
  constexpr int sh = PASS == 0 ? 13 - 2 : 13 + 2;
  if(PASS == 0) { p[0] = (t10 + t11) << 2; p[4 * S] = (t10 - t11) << 2; }
  else { p[0] = JDESC(t10 + t11, 2); p[4 * S] = JDESC(t10 - t11, 2); }
  const int32_t z1 = (t12 + t13) * JC(0.541196100);
  p[2 * S] = JDESC(z1 + t13 * JC(0.765366865), sh);
  p[6 * S] = JDESC(z1 + t12 * (-JC(1.847759065)), sh);
  int32_t a1 = t4 + t7, a2 = t5 + t6, a3 = t4 + t6, a4 = t5 + t7;
  const int32_t z5 = (a3 + a4) * JC(1.175875602);
  const int32_t b4 = t4 * JC(0.298631336), b5 = t5 * JC(2.053119869), b6 = t6 * JC(3.072711026), b7 = t7 * JC(1.501321110);
  a1 *= -JC(0.899976223); a2 *= -JC(2.562915447); a3 *= -JC(1.961570560); a4 *= -JC(0.390180644);
  a3 += z5; a4 += z5;
  p[7 * S] = JDESC(b4 + a1 + a3, sh);
  p[5 * S] = JDESC(b5 + a2 + a4, sh);
  p[3 * S] = JDESC(b6 + a2 + a3, sh);
  p[S] = JDESC(b7 + a1 + a4, sh);
}

// the scaled DCT of Arai, Agui and Nakajima, libjpeg's "ifast" (integer,
// 8 fractional bits, products truncated) and "float": outputs carry the
// factors 8 s_u s_v (s_0 = 1, s_k = sqrt(2) cos(k pi/16)), which the
// divisors hold
#define AAN8(v, c) ((int32_t)(((v) * (c)) >> 8))
template<int S>
DEV void jpg_fdct8_ifast(int32_t *p)
{
  const int32_t a0 = p[0] + p[7 * S], a7 = p[0] - p[7 * S], a1 = p[S] + p[6 * S], a6 = p[S] - p[6 * S];
  const int32_t a2 = p[2 * S] + p[5 * S], a5 = p[2 * S] - p[5 * S], a3 = p[3 * S] + p[4 * S], a4 = p[3 * S] - p[4 * S];
  const int32_t e0 = a0 + a3, e3 = a0 - a3, e1 = a1 + a2, e2 = a1 - a2;
  p[0] = e0 + e1;
  p[4 * S] = e0 - e1;
  const int32_t r = AAN8(e2 + e3, 181);
  p[2 * S] = e3 + r;
  p[6 * S] = e3 - r;
  const int32_t o0 = a4 + a5, o1 = a5 + a6, o2 = a6 + a7;
  const int32_t rot = AAN8(o0 - o2, 98);
  const int32_t q2 = AAN8(o0, 139) + rot, q4 = AAN8(o2, 334) + rot, q3 = AAN8(o1, 181);
  const int32_t h1 = a7 + q3, h3 = a7 - q3;
  p[5 * S] = h3 + q2;
  p[3 * S] = h3 - q2;
  p[S] = h1 + q4;
  p[7 * S] = h1 - q4;
}

template<int S>
DEV void jpg_fdct8_float(float *p)
{
  const float a0 = p[0] + p[7 * S], a7 = p[0] - p[7 * S], a1 = p[S] + p[6 * S], a6 = p[S] - p[6 * S];
  const float a2 = p[2 * S] + p[5 * S], a5 = p[2 * S] - p[5 * S], a3 = p[3 * S] + p[4 * S], a4 = p[3 * S] - p[4 * S];
  const float e0 = a0 + a3, e3 = a0 - a3, e1 = a1 + a2, e2 = a1 - a2;
  p[0] = e0 + e1;
  p[4 * S] = e0 - e1;
  const float r = (e2 + e3) * 0.707106781f;
  p[2 * S] = e3 + r;
  p[6 * S] = e3 - r;
  const float o0 = a4 + a5, o1 = a5 + a6, o2 = a6 + a7;
  const float rot = (o0 - o2) * 0.382683433f;
  const float q2 = 0.541196100f * o0 + rot, q4 = 1.306562965f * o2 + rot, q3 = o1 * 0.707106781f;
  const float h1 = a7 + q3, h3 = a7 - q3;
  p[5 * S] = h3 + q2;
  p[3 * S] = h3 - q2;
  p[S] = h1 + q4;
  p[7 * S] = h1 - q4;
}

DEV int jpg_quant(int32_t v, int q8)
{ // v / q8 rounded half away from zero
  if(v < 0) { v = -v + (q8 >> 1); return -(v >= q8 ? v / q8 : 0); }
  v += q8 >> 1;
  return v >= q8 ? v / q8 : 0;
}

// a pixel's luma and chroma as jpg_ycc
DEV void jpg_ycc_px(uint32_t p, int &Y, int &cb, int &cr)
{
  const int r = p & 255, g = (p >> 8) & 255, b = (p >> 16) & 255;
  Y  = (19595 * r + 38470 * g + 7471 * b + 32768) >> 16;
  cb = (-11059 * r - 21709 * g + 32768 * b + (128 << 16) + 32767) >> 16;
  cr = (32768 * r - 27439 * g - 5329 * b + (128 << 16) + 32767) >> 16;
}

// the row transform of eight samples (level shifted); islow's and ifast's
// results stay below 2^13 (samples below 2^7, at most 8 of them times 4, or
// the scaled basis' 8 x 1.39), so LDS holds them in 16 bits
template<int DCT, typename T>
DEV void jpg_rows(int32_t *l, T *d)
{
  if(DCT == 2)
  {
    float f[8];
#pragma unroll
    for(int k = 0; k < 8; k++) f[k] = (float)l[k];
    jpg_fdct8_float<1>(f);
#pragma unroll
    for(int k = 0; k < 8; k++) d[k] = (T)f[k];
    return;
  }
  if(DCT == 1) jpg_fdct8_ifast<1>(l);
  else jpg_fdct8<0, 1>(l);
#pragma unroll
  for(int k = 0; k < 8; k++) d[k] = (T)l[k];
}

// eight row values into LDS in 16-byte stores
DEV void jpg_put8(int16_t __attribute__((may_alias)) *p, const int16_t __attribute__((may_alias)) *d)
{
  uint32_t w[4];
#pragma unroll
  for(int k = 0; k < 4; k++) w[k] = (uint32_t)(uint16_t)d[2 * k] | ((uint32_t)(uint16_t)d[2 * k + 1] << 16);
  typedef uint4 __attribute__((may_alias)) u4;
  *(u4 *)p = make_uint4(w[0], w[1], w[2], w[3]);
}
DEV void jpg_put8(float *p, const float *d)
{
  ((float4 *)p)[0] = make_float4(d[0], d[1], d[2], d[3]);
  ((float4 *)p)[1] = make_float4(d[4], d[5], d[6], d[7]);
}

// v / q rounded half away from zero, as jpg_quant, by the reciprocal
// m = ceil(2^32 / q): floor(x m / 2^32) = floor(x / q) while x (m q - 2^32)
// stays below 2^32, and here x < 2^19, q < 2^12; q = 1 has m = 0
DEV int32_t jpg_quant_m(int32_t v, int32_t q, uint32_t m)
{
  const uint32_t x = (uint32_t)(v < 0 ? -v : v) + ((uint32_t)q >> 1);
  const uint32_t d = m ? __umulhi(x, m) : x;
  return v < 0 ? -(int32_t)d : (int32_t)d;
}

// a block's column (elements 8 apart) transformed and quantised; q: the
// divisors of the column, their reciprocals 128 further
template<int DCT, typename T>
DEV void jpg_cols(const T *p, int32_t o[8], const int32_t *q)
{
  if(DCT == 2)
  {
    float f[8];
#pragma unroll
    for(int r = 0; r < 8; r++) f[r] = (float)p[8 * r];
    jpg_fdct8_float<1>(f);
#pragma unroll
    for(int r = 0; r < 8; r++) o[r] = (int32_t)rintf(f[r] * __int_as_float(q[8 * r]));
    return;
  }
  int32_t d[8];
#pragma unroll
  for(int r = 0; r < 8; r++) d[r] = (int32_t)p[8 * r];
  if(DCT == 1) jpg_fdct8_ifast<1>(d);
  else jpg_fdct8<1, 1>(d);
#pragma unroll
  for(int r = 0; r < 8; r++) o[r] = jpg_quant_m(d[r], q[8 * r], (uint32_t)q[128 + 8 * r]);
}

constexpr uint8_t jz_dev[64] = {
  0, 1, 8, 16, 9, 2, 3, 10, 17, 24, 32, 25, 18, 11, 4, 5, 12, 19, 26, 33, 40, 48, 41, 34, 27, 20, 13, 6, 7, 14, 21,
  28, 35, 42, 49, 56, 57, 50, 43, 36, 29, 22, 15, 23, 30, 37, 44, 51, 58, 59, 52, 45, 38, 31, 39, 46, 53, 60, 61, 54,
  47, 55, 62, 63 };

// One lane a block, for the smoothing filter only (its 3x3 and 4x4 windows
// reach past the block).  q8: the divisors, luma then chroma: 8 x
// quantiser (DCT 0, islow), 8 x quantiser x the AAN factors in integer
// (1, ifast), or the float reciprocal of that (2, float; its bits)
template<int DCT>
__global__ void __launch_bounds__(64) k_jpg_coef(jpg_geom g, const int32_t *q8, int16_t *coef, uint8_t *dummy)
{
  const int b = blockIdx.x * 64 + threadIdx.x;
  if(b >= g.nb) return;
  int c, bx, by, i;
  jpg_block(g, b, c, bx, by, i);
  int16_t *o = coef + (long)b * 64;
  const bool dm = bx >= g.wib[c] || by >= g.hib[c];
  dummy[b] = dm ? (by >= g.hib[c] ? 2 : 1) : 0;
  if(dm)
  {
    for(int k = 0; k < 64; k += 4) *(uint2 *)(o + k) = make_uint2(0, 0);
    return;
  }
  int32_t d[64];
#pragma unroll
  for(int k = 0; k < 64; k++) d[k] = jpg_sample(g, c, bx * 8 + (k & 7), by * 8 + (k >> 3)) - 128;
  const int32_t *q = q8 + (c ? 64 : 0);
  if(DCT == 2)
  { // float: multiply by the reciprocal, round to nearest even
    float f[64];
#pragma unroll
    for(int k = 0; k < 64; k++) f[k] = (float)d[k];
#pragma unroll
    for(int k = 0; k < 8; k++) jpg_fdct8_float<1>(f + 8 * k);
#pragma unroll
    for(int k = 0; k < 8; k++) jpg_fdct8_float<8>(f + k);
#pragma unroll
    for(int k = 0; k < 64; k++) d[k] = (int32_t)rintf(f[k] * __int_as_float(q[k]));
  }
  else if(DCT == 1)
  {
#pragma unroll
    for(int k = 0; k < 8; k++) jpg_fdct8_ifast<1>(d + 8 * k);
#pragma unroll
    for(int k = 0; k < 8; k++) jpg_fdct8_ifast<8>(d + k);
  }
  else
  {
#pragma unroll
    for(int k = 0; k < 8; k++) jpg_fdct8<0, 1>(d + 8 * k);
#pragma unroll
    for(int k = 0; k < 8; k++) jpg_fdct8<1, 8>(d + k);
  }
  // stored in zigzag order, the order the entropy coder walks them
#pragma unroll
  for(int k = 0; k < 64; k += 2)
  {
    const int a = DCT == 2 ? d[jz_dev[k]] : jpg_quant(d[jz_dev[k]], q[jz_dev[k]]);
    const int e = DCT == 2 ? d[jz_dev[k + 1]] : jpg_quant(d[jz_dev[k + 1]], q[jz_dev[k + 1]]);
    *(uint32_t *)(o + k) = (uint32_t)(uint16_t)a | ((uint32_t)(uint16_t)e << 16);
  }
}

// a block's 64 coefficients (zigzag order) in registers: eight 16-byte loads
struct jpg_blk
{
  uint4 w[8];
  __device__ __forceinline__ int at(int k) const
  {
    const uint4 &v = w[k >> 3];
    const int j = (k >> 1) & 3;
    const uint32_t u = j == 0 ? v.x : j == 1 ? v.y : j == 2 ? v.z : v.w;
    return (int)(int16_t)(uint16_t)(u >> (16 * (k & 1)));
  }
};

DEV void jpg_load(jpg_blk &z, const int16_t *coef, int b)
{
  const uint4 *p = (const uint4 *)(coef + (long)b * 64);
#pragma unroll
  for(int i = 0; i < 8; i++) z.w[i] = p[i];
}

// the dummy blocks' DC: pass 1 the right edge (block to the left), pass 2 the
// bottom rows (the last block of the row above in the MCU, itself patched)
__global__ void __launch_bounds__(256) k_jpg_dummy(jpg_geom g, int16_t *coef, const uint8_t *dummy, int pass)
{
  const int b = blockIdx.x * 256 + threadIdx.x;
  if(b >= g.nb || dummy[b] != pass) return;
  int c, bx, by, i;
  jpg_block(g, b, c, bx, by, i);
  coef[(long)b * 64] = pass == 1 ? coef[(long)(b - 1) * 64] : coef[(long)(b - i - 1) * 64];
}

// the previous block of the same component in scan order, -1 for the first
DEV int jpg_prev(const jpg_geom &g, int b)
{
  const int m = b / g.bpm, r = b - m * g.bpm, n0 = g.hs * g.vs;
  if(r > 0 && r < n0) return b - 1;
  if(m == 0) return -1;
  return r == 0 ? b - g.bpm + n0 - 1 : b - g.bpm;
}

DEV int jpg_nbits(int v)
{
  v = v < 0 ? -v : v;
  return v ? 32 - __clz(v) : 0;
}

__global__ void __launch_bounds__(256) k_jpg_stats(jpg_geom g, const int16_t *coef, uint32_t *freq)
{
  __shared__ uint32_t h[4 * 257];
  for(int k = threadIdx.x; k < 4 * 257; k += 256) h[k] = 0;
  __syncthreads();
  const int b = blockIdx.x * 256 + threadIdx.x;
  if(b < g.nb)
  {
    int c, bx, by, i;
    jpg_block(g, b, c, bx, by, i);
    const int t = c ? 1 : 0;
    jpg_blk z;
    jpg_load(z, coef, b);
    const int p = jpg_prev(g, b);
    const int last = p < 0 ? 0 : coef[(long)p * 64];
    atomicAdd(h + (2 * t) * 257 + jpg_nbits(z.at(0) - last), 1u);
    uint32_t *ac = h + (2 * t + 1) * 257;
    int run = 0;
#pragma unroll
    for(int k = 1; k < 64; k++)
    {
      const int v = z.at(k);
      if(!v) { run++; continue; }
      while(run > 15) { atomicAdd(ac + 0xf0, 1u); run -= 16; }
      atomicAdd(ac + ((run << 4) | jpg_nbits(v)), 1u);
      run = 0;
    }
    if(run) atomicAdd(ac, 1u);
  }
  __syncthreads();
  for(int k = threadIdx.x; k < 4 * 257; k += 256)
    if(h[k]) atomicAdd(freq + k, h[k]);
}

// nonzero flags of the eight coefficients of a 16-byte chunk, one bit each
DEV uint32_t jpg_nz8(uint4 u)
{
  const uint32_t w[4] = { u.x, u.y, u.z, u.w };
  uint32_t m = 0;
#pragma unroll
  for(int k = 0; k < 4; k++) m |= ((w[k] & 0xffffu) ? 1u << (2 * k) : 0u) | ((w[k] >> 16) ? 2u << (2 * k) : 0u);
  return m;
}

// ---- samples, DCT, quantisation and symbol counts ------------------------------
//
// A work group takes 32 MCUs of one MCU row.  Thread (r, i) loads the pixels
// of chroma row r of MCU i (8 HS x VS pixels, 16-byte loads where the image
// allows), forms the component samples in registers and transforms their rows;
// the columns go through LDS (8 lanes a block: its columns; the block stride of
// 72 keeps both directions free of bank conflicts), where the quantised
// coefficients land in zigzag order and leave in 16-byte stores.  One lane a
// block with its 64 samples in registers converted every pixel once per
// component and touched 64 cache lines an instruction: 707 us for 24 MP 4:4:4,
// and 101 us more to read the coefficients again for the counts; this takes
// 123 us.  The 144 MB written and 96 MB read take 48 us at 5 TB/s.
#define JF_N 32                       // MCUs a strip
#define JF_S 72                       // elements a block in LDS
#define JF_COPIES 4                   // LDS histograms, by lane
#define JF_FREQ 8                     // global histograms, by work group
#define JF_HIST (2 * 256 + 2 * 16)    // AC luma, AC chroma, DC luma, DC chroma
typedef int16_t __attribute__((may_alias)) jpg_i16;
typedef uint4 __attribute__((may_alias)) jpg_u4;

template<int DCT, int HS, int VS>
__global__ void __launch_bounds__(256) k_jpg_front(jpg_geom g, const int32_t *q8, const uint8_t *zinv, int16_t *coef,
                                                   uint32_t *freq, int ntx, int ntiles, int vec)
{
  constexpr int NL = HS * VS, BPM = NL + 2;
  typedef typename std::conditional<DCT == 2, float, jpg_i16>::type T;
  __shared__ __align__(16) T tmp[BPM * JF_N * JF_S];
  __shared__ __align__(8) uint8_t nz[BPM * JF_N * 8];
  __shared__ uint32_t hist[JF_COPIES][JF_HIST];
  constexpr int ZS = JF_S * sizeof(T) / 2;   // int16 elements a block
  jpg_i16 *zt = (jpg_i16 *)tmp;
  const int t = threadIdx.x, col = t % 8;
  for(int k = t; k < JF_COPIES * JF_HIST; k += 256) (&hist[0][0])[k] = 0;
  uint32_t zp[8];   // zigzag positions of this lane's column
#pragma unroll
  for(int r = 0; r < 8; r++) zp[r] = zinv[8 * r + col];
#pragma unroll 1
  for(int tile = blockIdx.x; tile < ntiles; tile += gridDim.x)
  {
    const int uy = tile / ntx, u0 = (tile - uy * ntx) * JF_N, nu = min(JF_N, g.mx - u0);
    {
      const int i = t % JF_N, r = t / JF_N, ux = min(u0 + i, g.mx - 1);
      int cb[8], cr[8];
#pragma unroll
      for(int k = 0; k < 8; k++) cb[k] = cr[k] = 0;
#pragma unroll
      for(int v = 0; v < VS; v++)
#pragma unroll
        for(int h = 0; h < HS; h++)
        {
          const int yy = VS * r + v, x0 = (ux * HS + h) * 8, y = min(uy * 8 * VS + yy, g.H - 1);
          const uint8_t *row = g.rgba + 4 * (long)y * g.pitch;
          uint32_t px[8];
          if(vec && x0 + 8 <= g.W)
          {
            const uint4 a = *(const uint4 *)(row + 4 * x0), b = *(const uint4 *)(row + 4 * x0 + 16);
            px[0] = a.x; px[1] = a.y; px[2] = a.z; px[3] = a.w;
            px[4] = b.x; px[5] = b.y; px[6] = b.z; px[7] = b.w;
          }
          else
#pragma unroll
            for(int k = 0; k < 8; k++) px[k] = *(const uint32_t *)(row + 4 * min(x0 + k, g.W - 1));
          T d[8];
          int32_t l[8];
#pragma unroll
          for(int k = 0; k < 8; k++)
          {
            int Y, b, c;
            jpg_ycc_px(px[k], Y, b, c);
            l[k] = Y - 128;
            cb[(h * 8 + k) / HS] += b;
            cr[(h * 8 + k) / HS] += c;
          }
          jpg_rows<DCT>(l, d);
          const int j = (yy / 8) * HS + h;
          jpg_put8(tmp + (j * JF_N + i) * JF_S + (yy % 8) * 8, d);
        }
#pragma unroll
      for(int c = 0; c < 2; c++)
      {
        int32_t l[8];
        T d[8];
#pragma unroll
        for(int k = 0; k < 8; k++)
        {
          const int sum = c ? cr[k] : cb[k];
          l[k] = (NL == 1 ? sum : VS == 2 ? (sum + ((k & 1) ? 2 : 1)) >> 2 : (sum + (k & 1)) >> 1) - 128;
        }
        jpg_rows<DCT>(l, d);
        jpg_put8(tmp + ((NL + c) * JF_N + i) * JF_S + r * 8, d);
      }
    }
    __syncthreads();
    const bool edge = (u0 + nu) * HS > g.wib[0] || (uy + 1) * VS > g.hib[0];
#pragma unroll
    for(int j = 0; j < BPM; j++)
    { // the columns of block j of 32 MCUs, 8 lanes a block; a block's lanes are
      // of one wave, so its coefficients may take the place of its rows
      const int i = t / 8;
      T *p = tmp + (j * JF_N + i) * JF_S + col;
      int32_t o[8];
      jpg_cols<DCT>(p, o, q8 + (j < NL ? 0 : 64) + col);
      if(edge && j < NL && ((u0 + i) * HS + j % HS >= g.wib[0] || uy * VS + j / HS >= g.hib[0]))
#pragma unroll
        for(int r = 0; r < 8; r++) o[r] = 0;
      __builtin_amdgcn_wave_barrier();
      jpg_i16 *z = zt + (j * JF_N + i) * ZS;
#pragma unroll
      for(int r = 0; r < 8; r++) z[zp[r]] = (int16_t)o[r];
    }
    __syncthreads();
    if(NL > 1 && edge)
    { // blocks past the extent take the DC of the block to the left or, in the
      // rows below, of the last block of the row above in the MCU
      if(t < nu)
        for(int j = 1; j < NL; j++)
        {
          const bool below = uy * VS + j / HS >= g.hib[0], right = (u0 + t) * HS + j % HS >= g.wib[0];
          if(below || right) zt[(j * JF_N + t) * ZS] = zt[((below ? j - j % HS - 1 : j - 1) * JF_N + t) * ZS];
        }
      __syncthreads();
    }
    int16_t *co = coef + ((long)uy * g.mx + u0) * BPM * 64;
    for(int e = t; e < nu * BPM * 8; e += 256)
    {
      const int b = e / 8, c = e % 8, i = b / BPM, j = b - i * BPM;
      const uint4 u = *(const jpg_u4 *)(zt + (j * JF_N + i) * ZS + 8 * c);
      *(uint4 *)(co + (long)e * 8) = u;
      nz[(j * JF_N + i) * 8 + c] = (uint8_t)jpg_nz8(u);
    }
    __syncthreads();
    if(t < BPM * JF_N && t % JF_N < nu)
    { // a thread a block: its symbols
      const int j = t / JF_N, i = t % JF_N, c = j < NL ? 0 : 1;
      const jpg_i16 *z = zt + t * ZS;
      uint32_t *h = hist[t % JF_COPIES];
      const bool first = j == 0 || j >= NL;     // its predecessor lies in the MCU before
      const bool have = !first || i > 0 || (uy == 0 && u0 == 0);
      const int last = !first ? zt[(t - JF_N) * ZS] : i > 0 ? zt[((j == 0 ? NL - 1 : j) * JF_N + i - 1) * ZS] : 0;
      if(have) atomicAdd(h + 512 + 16 * c + jpg_nbits(z[0] - last), 1u);
      uint64_t m = *(const uint64_t *)(nz + 8 * t) & ~1ull;
      int prev = 0;
      const int end = m ? 63 - __clzll(m) : 0;
      while(m)
      {
        const int k = __builtin_ctzll(m);
        m &= m - 1;
        int run = k - prev - 1;
        prev = k;
        if(run > 15) { atomicAdd(h + 256 * c + 0xf0, (uint32_t)(run >> 4)); run &= 15; }
        atomicAdd(h + 256 * c + ((run << 4) | jpg_nbits(z[k])), 1u);
      }
      if(end < 63) atomicAdd(h + 256 * c, 1u);
    }
    __syncthreads();
  }
  uint32_t *f = freq + (blockIdx.x % JF_FREQ) * 4 * 257;
  for(int k = t; k < JF_HIST; k += 256)
  {
    uint32_t n = 0;
#pragma unroll
    for(int c = 0; c < JF_COPIES; c++) n += hist[c][k];
    // the tables' order: DC luma, AC luma, DC chroma, AC chroma
    if(n) atomicAdd(f + (k < 512 ? (2 * (k / 256) + 1) * 257 + k % 256 : 2 * ((k - 512) / 16) * 257 + (k - 512) % 16), n);
  }
}

// the DC symbols of each strip's first MCU, whose predecessor another work
// group made: a thread per strip and component
__global__ void __launch_bounds__(256) k_jpg_dc0(jpg_geom g, const int16_t *coef, uint32_t *freq, int ntx, int ntiles)
{
  __shared__ uint32_t h[32];
  if(threadIdx.x < 32) h[threadIdx.x] = 0;
  __syncthreads();
  const int k = blockIdx.x * 256 + threadIdx.x;
  const int tile = k / 3, c = k % 3, n0 = g.hs * g.vs;
  const int uy = tile / ntx, u = uy * g.mx + (tile - uy * ntx) * JF_N;
  if(k < 3 * ntiles && u > 0)
  {
    const int b = u * g.bpm + (c ? n0 + c - 1 : 0), p = jpg_prev(g, b);
    atomicAdd(h + 16 * (c ? 1 : 0) + jpg_nbits(coef[(long)b * 64] - coef[(long)p * 64]), 1u);
  }
  __syncthreads();
  if(threadIdx.x < 32 && h[threadIdx.x])
    atomicAdd(freq + (blockIdx.x % JF_FREQ) * 4 * 257 + 2 * (threadIdx.x / 16) * 257 + threadIdx.x % 16, h[threadIdx.x]);
}

// ---- entropy coding --------------------------------------------------------------
//
// A work group codes 256 consecutive blocks, a thread a block: the blocks are
// staged in LDS (coalesced; reading a block by its own lane fetched 64 cache
// lines an instruction), each thread walks its nonzero coefficients by their
// mask, and the code tables lie in LDS too.  EMIT 0: each block's bits and the
// group's.  EMIT 1: the blocks' bits are scanned and their codes ORed into the group's
// words in LDS, which leave as whole words; only the first and the last, which
// the neighbours share, are ORed in memory.  A group of more than JC_WORDS
// words (over 256 bits a block) ORs its words in memory directly.
#define JC_WORDS 2048
struct jpg_codes { uint32_t v[4][256]; };   // code | length << 16

template<int EMIT>
__global__ void __launch_bounds__(256) k_jpg_code(jpg_geom g, const int16_t *coef, const jpg_codes *hc, uint16_t *blen,
                                                  uint64_t *gbits, uint32_t *words, uint64_t cap)
{
  __shared__ __align__(16) int16_t zt[256 * JF_S];
  __shared__ __align__(8) uint8_t nz[256 * 8];
  __shared__ uint32_t tab[4][256];
  __shared__ uint32_t lw[EMIT ? JC_WORDS : 1];
  __shared__ uint32_t wsum[4];
  const int t = threadIdx.x, b0 = blockIdx.x * 256, nb = min(256, g.nb - b0), b = b0 + t;
  // a stream larger than the buffer: the host sees the total and asks again
  if(EMIT && gbits[gridDim.x] > cap) return;
  for(int k = t; k < 1024; k += 256) (&tab[0][0])[k] = (&hc->v[0][0])[k];
  if(EMIT) for(int k = t; k < JC_WORDS; k += 256) lw[k] = 0;
#pragma unroll
  for(int e = t; e < 2048; e += 256)
  {
    const uint4 u = e < 8 * nb ? ((const uint4 *)(coef + (long)b0 * 64))[e] : make_uint4(0, 0, 0, 0);
    *(jpg_u4 *)(zt + (e / 8) * JF_S + 8 * (e % 8)) = u;
    nz[e] = (uint8_t)jpg_nz8(u);
  }
  __syncthreads();
  int c = 0, bx, by, ii, last = 0;
  if(t < nb)
  {
    jpg_block(g, b, c, bx, by, ii);
    const int p = jpg_prev(g, b);
    last = p < 0 ? 0 : p >= b0 ? zt[(p - b0) * JF_S] : coef[(long)p * 64];
  }
  const uint32_t *dct = tab[c ? 2 : 0], *act = tab[c ? 3 : 1];
  const int16_t *z = zt + t * JF_S;
  const int diff = z[0] - last, dn = jpg_nbits(diff);
  const uint64_t ac = *(const uint64_t *)(nz + 8 * t) & ~1ull;
  // every code with its extra bits, at most 16 + 11 together
  auto walk = [&](auto put) {
    if(t >= nb) return;
    const uint32_t d = dct[dn];
    put(((d & 0xffffu) << dn) | ((uint32_t)(diff < 0 ? diff - 1 : diff) & ((1u << dn) - 1)), (int)(d >> 16) + dn);
    uint64_t m = ac;
    int prev = 0;
    while(m)
    {
      const int k = __builtin_ctzll(m);
      m &= m - 1;
      int run = k - prev - 1;
      prev = k;
      for(; run > 15; run -= 16) { const uint32_t e = act[0xf0]; put(e & 0xffffu, (int)(e >> 16)); }
      const int v = z[k], s = jpg_nbits(v);
      const uint32_t e = act[(run << 4) | s];
      put(((e & 0xffffu) << s) | ((uint32_t)(v < 0 ? v - 1 : v) & ((1u << s) - 1)), (int)(e >> 16) + s);
    }
    if(prev < 63) { const uint32_t e = act[0]; put(e & 0xffffu, (int)(e >> 16)); }
  };
  uint32_t total = 0;     // at most 64 codes of 27 bits
  if(EMIT) total = t < nb ? blen[b] : 0u;
  else
  {
    walk([&](uint32_t, int n) { total += n; });
    if(t < nb) blen[b] = (uint16_t)total;
  }
  // inclusive scan of the blocks' bits over the group
  uint32_t inc = total;
  for(int o = 1; o < 64; o <<= 1)
  {
    const uint32_t y = __shfl_up(inc, o);
    if(t % 64 >= o) inc += y;
  }
  if(t % 64 == 63) wsum[t / 64] = inc;
  __syncthreads();
  uint32_t before = 0, all = 0;
#pragma unroll
  for(int k = 0; k < 4; k++)
  {
    if(k < t / 64) before += wsum[k];
    all += wsum[k];
  }
  if(!EMIT) { if(t == 0) gbits[blockIdx.x] = all; return; }
  const uint64_t g0 = gbits[blockIdx.x];
  // the free bits of the stream's last byte are ones
  const uint32_t pad = b0 + nb == g.nb ? (uint32_t)(-(g0 + all) & 7) : 0u;
  const uint32_t o0 = (uint32_t)(g0 & 31), nw = (o0 + all + pad + 31) / 32;
  uint32_t *gw = words + (g0 >> 5);
  const bool lds = nw <= JC_WORDS;
  uint32_t at = o0 + before + inc - total, w = at >> 5;
  int used = (int)(at & 31);
  uint64_t acc = 0;
  auto flush = [&](uint32_t x) {
    if(lds) atomicOr(lw + w, x);
    else atomicOr(gw + w, x);
  };
  auto put = [&](uint32_t v, int n) {
    if(!n) return;
    acc |= (uint64_t)v << (64 - used - n);
    used += n;
    if(used >= 32)
    {
      flush((uint32_t)(acc >> 32));
      acc <<= 32;
      used -= 32;
      w++;
    }
  };
  walk(put);
  if(pad && t == nb - 1) put((1u << pad) - 1u, (int)pad);
  if(t < nb && used) flush((uint32_t)(acc >> 32));
  if(!lds) return;
  __syncthreads();
  for(uint32_t k = t; k < nw; k += 256)
    if(k == 0 || k == nw - 1) { if(lw[k]) atomicOr(gw + k, lw[k]); }
    else gw[k] = lw[k];
}

// exclusive scan of n u64 values in place by one work group, the total after
// them: each thread a run of values
__global__ void __launch_bounds__(1024) k_jpg_scan(uint64_t *v, int n)
{
  __shared__ uint64_t ws[16];
  const int t = threadIdx.x, per = (n + 1023) / 1024, a = min(t * per, n), e = min(a + per, n);
  uint64_t sum = 0;
  for(int k = a; k < e; k++) sum += v[k];
  uint64_t inc = sum;
  for(int o = 1; o < 64; o <<= 1)
  {
    const uint64_t y = __shfl_up(inc, o);
    if(t % 64 >= o) inc += y;
  }
  if(t % 64 == 63) ws[t / 64] = inc;
  __syncthreads();
  uint64_t run = inc - sum;
  for(int k = 0; k < t / 64; k++) run += ws[k];
  for(int k = a; k < e; k++)
  {
    const uint64_t x = v[k];
    v[k] = run;
    run += x;
  }
  if(t == 1023) v[n] = run;
}

// ---- byte stuffing: a work group 4096 bytes, a thread 16 -------------------------
#define JS_BYTES 4096

// the bytes of this thread's four words, and which of them (bit k) are 0xFF;
// bytes past the stream count as none
DEV int jpg_bytes16(const uint32_t *words, uint64_t nbytes, uint8_t by[16], uint32_t &ff)
{
  const uint64_t i0 = (uint64_t)blockIdx.x * JS_BYTES + 16 * threadIdx.x;
  ff = 0;
  if(i0 >= nbytes) return 0;
  const int n = (int)min((uint64_t)16, nbytes - i0);
  const uint4 u = *(const uint4 *)(words + i0 / 4);     // the words are padded to whole groups of four
  const uint32_t w[4] = { u.x, u.y, u.z, u.w };
#pragma unroll
  for(int k = 0; k < 16; k++)
  {
    by[k] = (uint8_t)(w[k / 4] >> (24 - 8 * (k % 4)));
    if(k < n && by[k] == 0xffu) ff |= 1u << k;
  }
  return n;
}

// total: the stream's bits; cap: the bits the buffer holds
__global__ void __launch_bounds__(256) k_stuff_count(const uint32_t *words, const uint64_t *total, uint64_t cap, uint64_t *cnt)
{
  __shared__ uint32_t s;
  if(threadIdx.x == 0) s = 0;
  __syncthreads();
  uint8_t by[16];
  uint32_t ff = 0;
  if(*total <= cap) jpg_bytes16(words, (*total + 7) / 8, by, ff);
  if(ff) atomicAdd(&s, (uint32_t)__popc(ff));
  __syncthreads();
  if(threadIdx.x == 0) cnt[blockIdx.x] = s;
}

// the chunk with its zeros is formed in LDS, at the alignment of its place in
// the output, and leaves in whole words but for its ends
__global__ void __launch_bounds__(256) k_stuff_scatter(const uint32_t *words, const uint64_t *total, uint64_t cap,
                                                       const uint64_t *off, uint8_t *out)
{
  __shared__ __align__(4) uint8_t o[2 * JS_BYTES + 4];
  __shared__ uint32_t ws[4];
  if(*total > cap) return;
  const uint64_t nbytes = (*total + 7) / 8, c0 = (uint64_t)blockIdx.x * JS_BYTES;
  if(c0 >= nbytes) return;
  const int t = threadIdx.x;
  uint8_t by[16];
  uint32_t ff;
  const int n = jpg_bytes16(words, nbytes, by, ff);
  const uint32_t c = n + __popc(ff);
  uint32_t inc = c;
  for(int d = 1; d < 64; d <<= 1)
  {
    const uint32_t y = __shfl_up(inc, d);
    if(t % 64 >= d) inc += y;
  }
  if(t % 64 == 63) ws[t / 64] = inc;
  __syncthreads();
  uint32_t at = inc - c, all = 0;
#pragma unroll
  for(int k = 0; k < 4; k++)
  {
    if(k < t / 64) at += ws[k];
    all += ws[k];
  }
  const uint64_t dst = c0 + off[blockIdx.x];
  const uint32_t lead = (uint32_t)((uintptr_t)(out + dst) & 3);
  at += lead;
#pragma unroll
  for(int k = 0; k < 16; k++)
    if(k < n)
    {
      o[at++] = by[k];
      if(ff & (1u << k)) o[at++] = 0;
    }
  __syncthreads();
  uint8_t *base = out + dst - lead;
  const uint32_t end = lead + all;
  for(uint32_t k = 4 * t; k < end; k += 1024)
  {
    if(k >= lead && k + 4 <= end) *(uint32_t *)(base + k) = *(const uint32_t *)(o + k);
    else
      for(uint32_t q = max(k, lead); q < min(k + 4, end); q++) base[q] = o[q];
  }
}

__global__ void k_jpg_zero(uint32_t *p, long n)
{
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if(i < n) p[i] = 0;
}

// zeros for the stream's words (total bits, where they fit cap)
__global__ void __launch_bounds__(256) k_jpg_zero_words(uint4 *w, const uint64_t *total, uint64_t cap)
{
  if(*total > cap) return;
  const uint64_t n = (*total + 127) / 128;
  for(uint64_t k = (uint64_t)blockIdx.x * 256 + threadIdx.x; k < n; k += (uint64_t)gridDim.x * 256) w[k] = make_uint4(0, 0, 0, 0);
}

// ---- host ------------------------------------------------------------------

// the stream's room that is taken without knowing its length: 30 MP in 4:4:4
#define JPG_ROOM ((size_t)128 << 20)

// optimal code lengths (T.81 K.2: the two smallest frequencies merged, ties to
// the larger symbol, a reserved symbol 256; K.3: lengths limited to 16)
void jpg_huff(const uint32_t *freq_in, uint8_t bits[17], uint8_t val[256], int *nval)
{
  long freq[257];
  int codesize[257], others[257];
  for(int i = 0; i < 256; i++) freq[i] = freq_in[i];
  freq[256] = 1;
  for(int i = 0; i < 257; i++) { codesize[i] = 0; others[i] = -1; }
  for(;;)
  {
    int c1 = -1, c2 = -1;
    long v = 1000000000L;
    for(int i = 0; i <= 256; i++) if(freq[i] && freq[i] <= v) { v = freq[i]; c1 = i; }
    v = 1000000000L;
    for(int i = 0; i <= 256; i++) if(freq[i] && freq[i] <= v && i != c1) { v = freq[i]; c2 = i; }
    if(c2 < 0) break;
    freq[c1] += freq[c2];
    freq[c2] = 0;
    codesize[c1]++;
    while(others[c1] >= 0) { c1 = others[c1]; codesize[c1]++; }
    others[c1] = c2;
    codesize[c2]++;
    while(others[c2] >= 0) { c2 = others[c2]; codesize[c2]++; }
  }
  int cnt[33] = { 0 };
  for(int i = 0; i <= 256; i++) if(codesize[i]) cnt[codesize[i] > 32 ? 32 : codesize[i]]++;
  for(int i = 32; i > 16; i--)
    while(cnt[i] > 0)
    {
      int j = i - 2;
      while(cnt[j] == 0) j--;
      cnt[i] -= 2;
      cnt[i - 1]++;
      cnt[j + 1] += 2;
      cnt[j]--;
    }
  int i = 16;
  while(cnt[i] == 0) i--;
  cnt[i]--;
  bits[0] = 0;
  for(int k = 1; k <= 16; k++) bits[k] = (uint8_t)cnt[k];
  int p = 0;
  for(int len = 1; len <= 32; len++)
    for(int s = 0; s < 256; s++) if(codesize[s] == len) val[p++] = (uint8_t)s;
  *nval = p;
}

struct out_t
{
  std::vector<uint8_t> d;
  void b(int v) { d.push_back((uint8_t)v); }
  void w(int v) { b(v >> 8); b(v & 255); }
};

} // namespace

extern "C" void vkdt_jpg_quant_tables(int quality, uint8_t luma[64], uint8_t chroma[64])
{
  static const int sl[64] = {
    16, 11, 10, 16, 24, 40, 51, 61, 12, 12, 14, 19, 26, 58, 60, 55, 14, 13, 16, 24, 40, 57, 69, 56,
    14, 17, 22, 29, 51, 87, 80, 62, 18, 22, 37, 56, 68, 109, 103, 77, 24, 35, 55, 64, 81, 104, 113, 92,
    49, 64, 78, 87, 103, 121, 120, 101, 72, 92, 95, 98, 112, 100, 103, 99 };
  static const int sc[64] = {
    17, 18, 24, 47, 99, 99, 99, 99, 18, 21, 26, 66, 99, 99, 99, 99, 24, 26, 56, 99, 99, 99, 99, 99,
    47, 66, 99, 99, 99, 99, 99, 99, 99, 99, 99, 99, 99, 99, 99, 99, 99, 99, 99, 99, 99, 99, 99, 99,
    99, 99, 99, 99, 99, 99, 99, 99, 99, 99, 99, 99, 99, 99, 99, 99 };
  quality = quality < 1 ? 1 : (quality > 100 ? 100 : quality);
  const long scale = quality < 50 ? 5000 / quality : 200 - 2 * quality;   // IJG quality scaling
  for(int i = 0; i < 64; i++)
  {
    const long l = (sl[i] * scale + 50) / 100, c = (sc[i] * scale + 50) / 100;
    luma[i] = (uint8_t)(l < 1 ? 1 : (l > 255 ? 255 : l));
    chroma[i] = (uint8_t)(c < 1 ? 1 : (c > 255 ? 255 : c));
  }
}

extern "C" int vkdt_hip_jpg_encode(const void *rgba, uint32_t wd, uint32_t ht, uint32_t pitch, int quality, int hs,
                                   int vs, uint8_t **out, size_t *out_len, void *stream)
{
  return vkdt_hip_jpg_encode_ex(rgba, wd, ht, pitch, quality, hs, vs, VKDT_JPG_DCT_ISLOW, 0, nullptr, 0, out, out_len,
                                stream);
}

extern "C" int vkdt_hip_jpg_encode_ex(const void *rgba, uint32_t wd, uint32_t ht, uint32_t pitch, int quality, int hs,
                                      int vs, int dct, int smoothing, const uint8_t *icc, size_t icc_len, uint8_t **out,
                                      size_t *out_len, void *stream)
{
  *out = nullptr;
  *out_len = 0;
  if(!rgba || wd == 0 || ht == 0 || wd > 65535 || ht > 65535 || pitch < wd)
    return vkdt_set_error(VKDT_HIP_INCOMPLETE, "jpg: extent %ux%u (pitch %u)", wd, ht, pitch);
  if(!((hs == 1 && vs == 1) || (hs == 2 && vs == 1) || (hs == 2 && vs == 2)))
    return vkdt_set_error(VKDT_HIP_INCOMPLETE, "jpg: sampling %dx%d (4:4:4, 4:2:2 or 4:2:0)", hs, vs);
  if(dct < VKDT_JPG_DCT_ISLOW || dct > VKDT_JPG_DCT_FLOAT)
    return vkdt_set_error(VKDT_HIP_INCOMPLETE, "jpg: dct method %d (0 islow, 1 ifast, 2 float)", dct);
  if(smoothing < 0 || smoothing > 100)
    return vkdt_set_error(VKDT_HIP_INCOMPLETE, "jpg: smoothing factor %d (0..100)", smoothing);
  // ICC.1 Annex B.4: at most 255 APP2 markers of 65519 profile bytes
  const size_t icc_chunk = 65533 - 14;
  if(icc_len && (!icc || (icc_len + icc_chunk - 1) / icc_chunk > 255))
    return vkdt_set_error(VKDT_HIP_INCOMPLETE, "jpg: icc profile of %zu bytes", icc_len);
  jpg_geom g;
  g.rgba = (const uint8_t *)rgba;
  g.W = (int)wd; g.H = (int)ht; g.pitch = (int)pitch;
  g.hs = hs; g.vs = vs; g.bpm = hs * vs + 2;
  g.mx = (g.W + 8 * hs - 1) / (8 * hs);
  g.my = (g.H + 8 * vs - 1) / (8 * vs);
  const long nbl = (long)g.mx * g.my * g.bpm;
  if(nbl >= (1l << 31) / 64) return vkdt_set_error(VKDT_HIP_INCOMPLETE, "jpg: %ld blocks", nbl);
  g.nb = (int)nbl;
  g.wib[0] = (g.W + 7) / 8;
  g.hib[0] = (g.H + 7) / 8;
  g.wib[1] = g.wib[2] = ((g.W + hs - 1) / hs + 7) / 8;
  g.hib[1] = g.hib[2] = ((g.H + vs - 1) / vs + 7) / 8;
  g.smooth = smoothing;
  uint8_t ql[64], qc[64];
  vkdt_jpg_quant_tables(quality, ql, qc);
  // divisors by DCT method; the AAN factors s_0 = 1, s_k = sqrt(2) cos(k pi/16)
  static const double aan[8] = { 1.0, 1.387039845, 1.306562965, 1.175875602, 1.0, 0.785694958, 0.541196100,
                                 0.275899379 };
  int32_t q8[128];
  for(int t = 0; t < 2; t++)
    for(int k = 0; k < 64; k++)
    {
      const int q = t ? qc[k] : ql[k];
      const double f = aan[k / 8] * aan[k % 8];
      if(dct == VKDT_JPG_DCT_FLOAT)
      {
        const float r = (float)(1.0 / ((double)q * aan[k / 8] * aan[k % 8] * 8.0));
        memcpy(q8 + 64 * t + k, &r, 4);
      }
      else if(dct == VKDT_JPG_DCT_IFAST)
        q8[64 * t + k] = (int32_t)(((int64_t)q * (int32_t)(16384.0 * f + 0.5) + 1024) >> 11);
      else
        q8[64 * t + k] = q << 3;
    }

  // reciprocals of the integer divisors, and the zigzag positions
  int32_t tables[256 + 16];
  memcpy(tables, q8, sizeof(q8));
  for(int k = 0; k < 128; k++)
    tables[128 + k] = dct == VKDT_JPG_DCT_FLOAT || q8[k] == 1 ? 0 : (int32_t)(uint32_t)(((1ull << 32) + q8[k] - 1) / q8[k]);
  for(int k = 0; k < 64; k++) ((uint8_t *)(tables + 256))[jz_host[k]] = (uint8_t)k;

  // device: tables | codes | counts | coef | dummy flags | bits per 256 blocks, total | bits per block
  const int ngroups = (int)((nbl + 255) / 256);
  const size_t o_codes = 2048, o_freq = o_codes + sizeof(jpg_codes), nfreq = JF_FREQ * 4 * 257;
  const size_t o_coef = (o_freq + nfreq * 4 + 255) & ~(size_t)255;
  const size_t o_dummy = o_coef + (size_t)nbl * 128;
  const size_t o_bits = (o_dummy + (smoothing ? nbl : 0) + 255) & ~(size_t)255;
  const size_t o_blen = o_bits + (size_t)(ngroups + 1) * 8;
  const size_t total = o_blen + (size_t)nbl * 2;
  scratch_t sc, st = {};
  if(int e = scratch_get(sc, total, "jpg scratch", true)) return e;
  uint8_t *dev = sc.dev;
  hipStream_t s = (hipStream_t)stream;
  int16_t *coef = (int16_t *)(dev + o_coef);
  uint32_t *freq = (uint32_t *)(dev + o_freq);
  uint64_t *bits = (uint64_t *)(dev + o_bits);
  uint16_t *blen = (uint16_t *)(dev + o_blen);
  // pinned: tables, then codes | counts | the stream's bits and 0xFF bytes
  static_assert(sizeof(jpg_codes) + JF_FREQ * 4 * 257 * 4 + 16 <= SCRATCH_PINNED, "pinned staging");
  jpg_codes *hc = (jpg_codes *)sc.pin;
  uint32_t *fr = (uint32_t *)(sc.pin + sizeof(jpg_codes));
  uint64_t *sizes = (uint64_t *)(sc.pin + sizeof(jpg_codes) + JF_FREQ * 4 * 257 * 4);
  memcpy(sc.pin, tables, sizeof(tables));
  int err = hip_fail(hipMemcpyAsync(dev, sc.pin, sizeof(tables), hipMemcpyHostToDevice, s), "jpg tables");
  if(!err)
  {
    const int32_t *dq = (const int32_t *)dev;
    hipLaunchKernelGGL(k_jpg_zero, dim3((unsigned)((nfreq + 255) / 256)), dim3(256), 0, s, freq, (long)nfreq);
    if(smoothing)
    {
      const auto coef_kernel = dct == VKDT_JPG_DCT_FLOAT ? k_jpg_coef<2> : (dct == VKDT_JPG_DCT_IFAST ? k_jpg_coef<1> : k_jpg_coef<0>);
      hipLaunchKernelGGL(coef_kernel, dim3((g.nb + 63) / 64), dim3(64), 0, s, g, dq, coef, dev + o_dummy);
      hipLaunchKernelGGL(k_jpg_dummy, dim3((g.nb + 255) / 256), dim3(256), 0, s, g, coef, (const uint8_t *)(dev + o_dummy), 1);
      hipLaunchKernelGGL(k_jpg_dummy, dim3((g.nb + 255) / 256), dim3(256), 0, s, g, coef, (const uint8_t *)(dev + o_dummy), 2);
      hipLaunchKernelGGL(k_jpg_stats, dim3((g.nb + 255) / 256), dim3(256), 0, s, g, (const int16_t *)coef, freq);
    }
    else
    {
      const int ntx = (g.mx + JF_N - 1) / JF_N, ntiles = ntx * g.my;
      const int vec = (uintptr_t)rgba % 16 == 0 && pitch % 4 == 0;
      const auto front = [&](auto d) {
        constexpr int D = decltype(d)::value;
        // a few strips a work group, so that the counts reach memory rarely
        hipLaunchKernelGGL((hs == 1 ? k_jpg_front<D, 1, 1> : vs == 1 ? k_jpg_front<D, 2, 1> : k_jpg_front<D, 2, 2>),
                           dim3((unsigned)std::min(ntiles, 2048)), dim3(256), 0, s, g, dq, dev + 1024, coef, freq, ntx, ntiles, vec);
      };
      if(dct == VKDT_JPG_DCT_FLOAT) front(std::integral_constant<int, 2>());
      else if(dct == VKDT_JPG_DCT_IFAST) front(std::integral_constant<int, 1>());
      else front(std::integral_constant<int, 0>());
      hipLaunchKernelGGL(k_jpg_dc0, dim3((3 * ntiles + 255) / 256), dim3(256), 0, s, g, (const int16_t *)coef, freq, ntx, ntiles);
    }
    err = launch_post("jpg coefficients");
    if(!err) err = hip_fail(hipMemcpyAsync(fr, freq, nfreq * 4, hipMemcpyDeviceToHost, s), "jpg counts");
    if(!err) err = hip_fail(hipStreamSynchronize(s), "jpg sync");
  }
  uint8_t hb[4][17], hv[4][256];
  int nv[4] = { 0, 0, 0, 0 };
  const jpg_codes *dhc = (const jpg_codes *)(dev + o_codes);
  if(!err)
  {
    for(size_t k = 4 * 257; k < nfreq; k++) fr[k % (4 * 257)] += fr[k];
    memset(hc, 0, sizeof(*hc));
    for(int t = 0; t < 4; t++)
    {
      jpg_huff(fr + 257 * t, hb[t], hv[t], nv + t);
      int code = 0, k = 0;
      for(int len = 1; len <= 16; len++)
      {
        for(int j = 0; j < hb[t][len]; j++, k++) hc->v[t][hv[t][k]] = (uint32_t)code++ | ((uint32_t)len << 16);
        code <<= 1;
      }
    }
    err = hip_fail(hipMemcpyAsync(dev + o_codes, hc, sizeof(*hc), hipMemcpyHostToDevice, s), "jpg codes");
  }
  if(!err)
  {
    hipLaunchKernelGGL(k_jpg_code<0>, dim3((unsigned)ngroups), dim3(256), 0, s, g, (const int16_t *)coef, dhc, blen, bits,
                       (uint32_t *)nullptr, (uint64_t)0);
    hipLaunchKernelGGL(k_jpg_scan, dim3(1), dim3(1024), 0, s, bits, ngroups);
    err = launch_post("jpg lengths");
  }
  // The stream is written into room for 4 bits a coefficient, so that its
  // length need not come back first; the kernels leave a longer one alone, and
  // it is written again into room for its length.  Above JPG_ROOM bytes, where
  // the round trip (20 us) is little against the kernels, and where there is no
  // memory for that room, the length is asked for first
  const uint64_t *tot = bits + ngroups;
  uint64_t nbits = 0, nff = 0;
  uint8_t *stuffed = nullptr;
  size_t cap = (size_t)nbl * 32;
  bool known = false;   // cap is the length
  const auto length = [&]() {
    int e = hip_fail(hipMemcpyAsync(sizes, tot, 8, hipMemcpyDeviceToHost, s), "jpg total");
    if(!e) e = hip_fail(hipStreamSynchronize(s), "jpg sync");
    if(e) return e;
    cap = (size_t)((sizes[0] + 7) / 8);
    known = true;
    return e;
  };
  if(!err && 3 * cap > JPG_ROOM) err = length();
  while(!err)
  { // words | 0xFF bytes before each chunk, their total | stuffed bytes (at most twice)
    const long nwords = (long)((cap + 15) / 16 * 4), nchunks = (long)((cap + JS_BYTES - 1) / JS_BYTES);
    const size_t wbytes = ((size_t)nwords * 4 + 255) & ~(size_t)255, cbytes = ((size_t)(nchunks + 1) * 8 + 255) & ~(size_t)255;
    err = scratch_get(st, wbytes + cbytes + 2 * cap + 16, "jpg stream");
    if(err == VKDT_HIP_OOM && !known)
    {
      err = length();
      continue;
    }
    if(err) break;
    uint32_t *words = (uint32_t *)st.dev;
    uint64_t *cnt = (uint64_t *)(st.dev + wbytes);
    stuffed = st.dev + wbytes + cbytes;
    hipLaunchKernelGGL(k_jpg_zero_words, dim3((unsigned)std::min((nwords / 4 + 255) / 256, 2048l)), dim3(256), 0, s, (uint4 *)words, tot,
                       (uint64_t)cap * 8);
    hipLaunchKernelGGL(k_jpg_code<1>, dim3((unsigned)ngroups), dim3(256), 0, s, g, (const int16_t *)coef, dhc, blen, bits, words,
                       (uint64_t)cap * 8);
    hipLaunchKernelGGL(k_stuff_count, dim3((unsigned)nchunks), dim3(256), 0, s, (const uint32_t *)words, tot, (uint64_t)cap * 8, cnt);
    hipLaunchKernelGGL(k_jpg_scan, dim3(1), dim3(1024), 0, s, cnt, (int)nchunks);
    hipLaunchKernelGGL(k_stuff_scatter, dim3((unsigned)nchunks), dim3(256), 0, s, (const uint32_t *)words, tot, (uint64_t)cap * 8,
                       (const uint64_t *)cnt, stuffed);
    err = launch_post("jpg stuffing");
    if(!err) err = hip_fail(hipMemcpyAsync(sizes, tot, 8, hipMemcpyDeviceToHost, s), "jpg total");
    if(!err) err = hip_fail(hipMemcpyAsync(sizes + 1, cnt + nchunks, 8, hipMemcpyDeviceToHost, s), "jpg stuffed");
    if(!err) err = hip_fail(hipStreamSynchronize(s), "jpg sync");
    if(err) break;
    nbits = sizes[0];
    nff = sizes[1];
    if(known || nbits <= (uint64_t)cap * 8) break;
    scratch_put(st, true);
    cap = (size_t)((nbits + 7) / 8);
    known = true;
  }
  const size_t nbytes = (size_t)((nbits + 7) / 8);
  out_t o;
  if(!err)
  {
    o.w(0xffd8);
    o.w(0xffe0); o.w(16);                                     // JFIF, 300 dpi (o-jpg/main.c:157-159)
    o.b('J'); o.b('F'); o.b('I'); o.b('F'); o.b(0);
    o.b(1); o.b(1); o.b(1); o.w(300); o.w(300); o.b(0); o.b(0);
    // the ICC profile in APP2 markers: "ICC_PROFILE\0", sequence number
    // from 1, marker count, then up to 65519 profile bytes (ICC.1 B.4)
    const int nicc = (int)((icc_len + icc_chunk - 1) / icc_chunk);
    for(int m = 0; m < nicc; m++)
    {
      const size_t n = std::min(icc_chunk, icc_len - m * icc_chunk);
      o.w(0xffe2); o.w((int)(2 + 14 + n));
      for(const char *c = "ICC_PROFILE"; *c; c++) o.b(*c);
      o.b(0); o.b(m + 1); o.b(nicc);
      o.d.insert(o.d.end(), icc + m * icc_chunk, icc + m * icc_chunk + n);
    }
    for(int t = 0; t < 2; t++)
    {
      o.w(0xffdb); o.w(67); o.b(t);
      for(int k = 0; k < 64; k++) o.b((t ? qc : ql)[jz_host[k]]);
    }
    o.w(0xffc0); o.w(17); o.b(8); o.w(g.H); o.w(g.W); o.b(3);
    o.b(1); o.b((hs << 4) | vs); o.b(0);
    o.b(2); o.b(0x11); o.b(1);
    o.b(3); o.b(0x11); o.b(1);
    for(int t = 0; t < 4; t++)
    {
      o.w(0xffc4); o.w(2 + 1 + 16 + nv[t]); o.b(((t & 1) << 4) | (t >> 1));
      for(int k = 1; k <= 16; k++) o.b(hb[t][k]);
      for(int k = 0; k < nv[t]; k++) o.b(hv[t][k]);
    }
    o.w(0xffda); o.w(12); o.b(3);
    o.b(1); o.b(0x00); o.b(2); o.b(0x11); o.b(3); o.b(0x11);
    o.b(0); o.b(63); o.b(0);
    // the file in the caller's memory, the stream straight from the device
    const size_t head = o.d.size(), body = nbytes + (size_t)nff;
    uint8_t *f = (uint8_t *)malloc(head + body + 2);
    if(!f) err = vkdt_set_error(VKDT_HIP_OOM, "jpg: out of memory");
    else
    {
      memcpy(f, o.d.data(), head);
      if(body) err = hip_fail(hipMemcpyAsync(f + head, stuffed, body, hipMemcpyDeviceToHost, s), "jpg download");
      if(!err) err = hip_fail(hipStreamSynchronize(s), "jpg sync");
      f[head + body] = 0xff;
      f[head + body + 1] = 0xd9;
      if(err) free(f);
      else
      {
        *out = f;
        *out_len = head + body + 2;
      }
    }
  }
  scratch_put(sc, !err);
  scratch_put(st, !err);
  return err;
}

extern "C" void vkdt_jpg_free(uint8_t *p) { free(p); }
