// convnet.hip -- the learned early stop: a causal dilated 1-D convolution
// network trained and run on the device with hand-written kernels.
//
// No reference counterpart (the reference always runs to the end
// criterion). The network maps port traces observed over the first part
// of a run, plus the known source, to the whole trace; see
// include/ems_learn.h for its shape and the C ABI.
//
// Layout: parameters [out][in][tap] f32 (the optimizer's master copy), their
// bf16 values in the passes' own orders.
//
// Training and inference have kernels of their own. A weight rounds to bf16
// before every use, so a last-bit difference in one step's gradient moves
// some weights by a whole bf16 step in the next, and a training run's loss
// by 1e-4 after a few steps: the training kernels therefore keep one fixed
// order of every sum (channels then taps per output; per weight 256 strided
// partial sums and a tree), whatever their tiling. A prediction has no such
// feedback: it runs on the matrix cores.
//
// Prediction: an f32 activation is the exact sum of three bf16 values (its
// leading, middle and last 8 significant bits), and a product of two bf16
// values is exact in f32, so three bf16 matrix products with f32
// accumulation give the f32 result (256 sequences of 512 samples, 64
// channels: 2.0e-7 off f64, the sums in f32 5.2e-7). Activations [batch]
// [time][channel], channels padded with zeros to a multiple of 32 (the
// input to 16).
//
// Training: activations [batch][channel][time], lanes along time.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>
#include <algorithm>
#include <cstring>
#include <random>
#include <string>
#include <vector>

#include "../../include/ems_gpu.h"
#include "../../include/ems_learn.h"

// The network tolerates reassociation (its parity is a tolerance, not bit
// identity): let the compiler contract multiply-adds here.
#pragma clang fp contract(fast)

namespace {

constexpr int CN_K = 9;  // taps

// Round to nearest even (finite inputs), as the host does.
__device__ __forceinline__ uint16_t f32_to_bf16(float f) {
  const uint32_t u = __float_as_uint(f);
  const uint32_t r = ((u >> 16) & 1u) + 0x7FFFu;
  return (uint16_t)((u + r) >> 16);
}

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// x as three bf16 values whose sum is x: its bits in runs of 8 significant
// ones (infinities and NaN in the first alone).
__device__ __forceinline__ void split3(float x, uint32_t &hi, uint32_t &mid, uint32_t &lo) {
  const uint32_t u = __float_as_uint(x);
  hi = u >> 16;
  const float r = x - __uint_as_float(u & 0xFFFF0000u);
  const uint32_t v = __float_as_uint(r);
  mid = v >> 16;
  lo = __float_as_uint(r - __uint_as_float(v & 0xFFFF0000u)) >> 16;
  if ((u & 0x7F800000u) == 0x7F800000u) {
    if (u & 0x007FFFFFu) hi = 0x7FC0u;
    mid = lo = 0;
  }
}

// ---- prediction ----
//
// out[b][t][m] = sum_q sum_c W_q[m][c] src[b][t - dil (8 - q)][c] over nine
// taps q (zero before t = 0).
//
// A block takes 64 samples of one sequence and up to 64 output channels.
// Samples of one phase (t modulo the dilation) only meet their own phase, so
// a block takes ml consecutive samples of each of 64 / ml phases, and its
// taps reach (64 / ml) (ml + 8) source rows: 72 to 96 of 512 samples with
// dilations 1 to 32, where 64 consecutive samples would reach 64 + 8 dil
// (320; 89 against 65 us a layer of 256 sequences). Those rows are staged in
// LDS once, split into their three bf16 parts (rows of KC channels, 16 bytes
// apart in banks); the weights come packed in operand order, a coalesced
// 1 KiB load per wave and product. Wave w takes 32 of the samples (w & 1)
// and every fourth step of the (tap, 16 channels) sum (w >> 1), both
// 32-channel tiles, so that a staged operand is read once for two products;
// the quarters of the sum are added through LDS, each wave finishing a
// quarter of the outputs.
//
// Bound by the latencies of a block's phases (source rows, staged rows,
// weights, the exchange, tanh and the outputs), not by the products (29
// bf16 GFLOP, 12 us at the matrix peak): 50 us per layer of 256 sequences of
// 512 samples and 64 channels, 12 us of 32 sequences (one block per CU); a
// thread per output took 1100 and 150 us, four waves per block instead of
// eight 65 and 17.
//
// Hidden layers write h_out = h_in + tanh(z), the last layer the API's
// [b][channel][t].
enum { CN_HIDDEN, CN_OUT };
struct ConvArgs {
  const float *src;
  int cps;  // channels of a source row (a multiple of KC)
  int craw; // > 0: src is [b][craw][T] (the network's input as it came), cps channels padded
  const u32x4 *w;
  int mt;  // 32-channel tiles of the output
  int mc;  // output channels
  int T, dil;
  int ml;      // samples per phase of a block
  int pt, nt;  // blocks along the phases and along a phase
  unsigned blk0;  // the launch's first block
  const float *bias;
  const float *h_in;  // HIDDEN: the residual input, or null
  float *h_out;       // HIDDEN
  float *out;         // OUT
};

constexpr int CN_TT = 64;  // samples per block

__host__ __device__ __forceinline__ int cn_rows(int ml) {
  return CN_TT / ml * (ml + CN_K - 1);
}
__host__ __device__ __forceinline__ size_t cn_lds(int ml, int kc) {
  const size_t x = (size_t)cn_rows(ml) * (kc + 8) * 2 * 3;
  const size_t r = 2 * 4 * 2 * 16 * 64 * 4;  // the quarters' exchange
  return x > r ? x : r;
}

template <int MODE, int KC>
__global__ void __launch_bounds__(512) cn_conv(ConvArgs p) {
  extern __shared__ u32x4 cn_smem[];
  uint16_t *xs = (uint16_t *)cn_smem;
  constexpr int LD = KC + 8;
  const int rows = cn_rows(p.ml), pr = p.ml + CN_K - 1;  // pr: rows of a phase
  const int tiles = p.pt * p.nt, mt0 = 2 * blockIdx.y;
  const unsigned blk = p.blk0 + blockIdx.x;
  const int b = (int)(blk / (unsigned)tiles), tile = (int)(blk - (unsigned)b * (unsigned)tiles);
  const int ph0 = tile / p.nt * (CN_TT / p.ml), m0 = tile % p.nt * p.ml;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, nt = wv & 1, kh = wv >> 1;
  const bool two = mt0 + 1 < p.mt;
  const float *src = p.src + (size_t)b * p.T * p.cps;
  const int plane = rows * LD;  // (in bf16 values)
  const int n = nt * 32 + (lane & 31), phn = n / p.ml, row0 = phn * pr + (n - phn * p.ml);
  const int nch = p.cps / 16;
  f32x16 acc0, acc1;
#pragma unroll
  for (int i = 0; i < 16; i++) acc0[i] = acc1[i] = 0.0f;
  for (int c0 = 0; c0 < p.cps; c0 += KC) {
    if (c0) __syncthreads();
    if (p.craw) {  // (lanes along the rows: a channel's samples are one run)
      for (int e = threadIdx.x; e < rows * KC; e += 512) {
        const int c = e / rows, r = e - c * rows;
        const int ph = r / pr, ms = m0 - (CN_K - 1) + (r - ph * pr);
        const int64_t t = ph0 + ph + (int64_t)p.dil * ms;
        float v = 0.0f;
        if (c0 + c < p.craw && ph0 + ph < p.dil && ms >= 0 && t < p.T)
          v = p.src[((size_t)b * p.craw + c0 + c) * p.T + t];
        uint32_t h, m, l;
        split3(v, h, m, l);
        xs[r * LD + c] = (uint16_t)h;
        xs[plane + r * LD + c] = (uint16_t)m;
        xs[2 * plane + r * LD + c] = (uint16_t)l;
      }
    }
    for (int e = p.craw ? rows * (KC / 4) : (int)threadIdx.x; e < rows * (KC / 4); e += 512) {
      const int r = e / (KC / 4), c = 4 * (e % (KC / 4));
      const int ph = r / pr, ms = m0 - (CN_K - 1) + (r - ph * pr);
      const int64_t t = ph0 + ph + (int64_t)p.dil * ms;
      float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      if (ph0 + ph < p.dil && ms >= 0 && t < p.T) v = *(const float4 *)(src + (size_t)t * p.cps + c0 + c);
      uint32_t h[4], m[4], l[4];
      split3(v.x, h[0], m[0], l[0]);
      split3(v.y, h[1], m[1], l[1]);
      split3(v.z, h[2], m[2], l[2]);
      split3(v.w, h[3], m[3], l[3]);
      uint2 *d = (uint2 *)(xs + r * LD + c);
      d[0] = make_uint2(h[0] | h[1] << 16, h[2] | h[3] << 16);
      *(uint2 *)(xs + plane + r * LD + c) = make_uint2(m[0] | m[1] << 16, m[2] | m[3] << 16);
      *(uint2 *)(xs + 2 * plane + r * LD + c) = make_uint2(l[0] | l[1] << 16, l[2] | l[3] << 16);
    }
    __syncthreads();
    constexpr int NC = KC / 16;
    const uint16_t *xb = xs + row0 * LD + 8 * (lane >> 5);
    const u32x4 *wb = p.w + ((size_t)(c0 / 16) * p.mt + mt0) * 64 + lane;
    const size_t wq = (size_t)nch * p.mt * 64;
    const int one = two ? 64 : 0;
    for (int s = kh; s < CN_K * NC; s += 4) {
      const int q = s / NC, c = s % NC;
      const u32x4 *wp = wb + q * wq + (size_t)c * p.mt * 64;
      const bf16x8 w0 = __builtin_bit_cast(bf16x8, wp[0]);
      const bf16x8 w1 = __builtin_bit_cast(bf16x8, wp[one]);
      const uint16_t *xr = xb + q * LD + 16 * c;
      const bf16x8 xh = __builtin_bit_cast(bf16x8, *(const u32x4 *)xr);
      const bf16x8 xm = __builtin_bit_cast(bf16x8, *(const u32x4 *)(xr + plane));
      const bf16x8 xl = __builtin_bit_cast(bf16x8, *(const u32x4 *)(xr + 2 * plane));
      acc0 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w0, xl, acc0, 0, 0, 0);
      if (two) acc1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w1, xl, acc1, 0, 0, 0);
      acc0 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w0, xm, acc0, 0, 0, 0);
      if (two) acc1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w1, xm, acc1, 0, 0, 0);
      acc0 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w0, xh, acc0, 0, 0, 0);
      if (two) acc1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w1, xh, acc1, 0, 0, 0);
    }
  }
  // Wave kh finishes half kh & 1 (8 of a lane's 16 channels) of tile kh >> 1.
  __syncthreads();
  float *red = (float *)cn_smem + (size_t)nt * 4 * 2 * 16 * 64 + lane;
#pragma unroll
  for (int i = 0; i < 16; i++) {
    red[(kh * 32 + i) * 64] = acc0[i];
    if (two) red[(kh * 32 + 16 + i) * 64] = acc1[i];
  }
  __syncthreads();
  const int64_t tt = ph0 + phn + (int64_t)p.dil * (m0 + n - phn * p.ml);
  const int mtile = mt0 + (kh >> 1), half = 8 * (kh & 1);
  if (ph0 + phn >= p.dil || tt >= p.T || mtile >= p.mt) return;
  const int t = (int)tt;
  const float *o = red + ((kh >> 1) * 16 + half) * 64;
  float v[8];
#pragma unroll
  for (int i = 0; i < 8; i++)
    v[i] = (o[i * 64] + o[(32 + i) * 64]) + (o[(64 + i) * 64] + o[(96 + i) * 64]);
  // element i of a tile: channel 32 mtile + 8 (i / 4) + 4 (lane / 32) + i % 4
  const int mb = 32 * mtile + 2 * half + 4 * (lane >> 5);
  const size_t row = ((size_t)b * p.T + t) * (32 * (size_t)p.mt);
#pragma unroll
  for (int g = 0; g < 2; g++) {
    const int m = mb + 8 * g;
    if (MODE == CN_OUT) {
#pragma unroll
      for (int e = 0; e < 4; e++)
        if (m + e < p.mc)
          p.out[((size_t)b * p.mc + m + e) * p.T + t] = v[4 * g + e] + p.bias[m + e];
    } else {
      float4 hv = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      if (p.h_in) hv = *(const float4 *)(p.h_in + row + m);
      float *hh = (float *)&hv;
#pragma unroll
      for (int e = 0; e < 4; e++)
        hh[e] = m + e < p.mc ? hh[e] + tanhf(v[4 * g + e] + p.bias[m + e]) : 0.0f;
      *(float4 *)(p.h_out + row + m) = hv;
    }
  }
}

// ---- training ----

template <class T>
__device__ __forceinline__ T cn_uniform(const T *p, size_t i) {
#if defined(__HIP_DEVICE_COMPILE__)
  return ((const __attribute__((address_space(4))) T *)p)[i];
#else
  return p[i];
#endif
}

// A causal convolution's sums over `ns` source channels and nine taps for
// 64 samples and M output channels per wave (MW = 8, or 1 where that leaves
// SIMDs idle: launch_fma): out[m] = init[m] + sum_s
// sum_k w[s][k][m] src[s][t + off_k], channels and taps in order, one fused
// multiply-add each (samples outside the sequence count as zeros; the
// forward pass has off_k = -dil (8 - k), the input gradient +dil (8 - k)).
// The weights are wave-uniform: they come through the scalar unit, as f32,
// a source channel's 72 at once (a wait per channel), and the samples
// straight from memory, 256 bytes a tap, four channels ahead. No LDS, no
// barrier. Bound by the waits for the weights, two waves a SIMD: 64
// channels, 32 sequences of 512 samples take 37 us, of which the
// multiply-adds are 18 (a wait per tap: 68; samples one channel ahead: 46;
// a thread per output, which read its weights as bf16 from memory: 173).
constexpr int MW = 8;
constexpr int AHEAD = 4;  // source channels loaded ahead
template <int M>
__device__ __forceinline__ void cn_sums(const float *__restrict__ src, int ns,
                                        const float *__restrict__ w, int groups, int T, int dil,
                                        int dir, unsigned t0, unsigned t, float acc[M]) {
  // per tap: the lane's sample (clamped) and whether it is one; byte offsets
  // from the first sample that the wave may read, so that 32 bits hold them
  // for sequences of any length (and dilations below 2^27)
  const int64_t reach = (int64_t)t0 - (int64_t)dil * (CN_K - 1);
  const int64_t first = dir > 0 ? (int64_t)t0 : (reach > 0 ? reach : 0);
  src += first;
  unsigned at[CN_K];
  bool in[CN_K];
#pragma unroll
  for (int k = 0; k < CN_K; k++) {
    const int64_t s = (int64_t)t + (int64_t)dir * dil * (CN_K - 1 - k);
    in[k] = s >= 0 && s < T;
    at[k] = in[k] ? 4u * (unsigned)(s - first) : 0u;
  }
  float x[AHEAD][CN_K];
#pragma unroll
  for (int a = 0; a < AHEAD; a++) {
    const float *sc = src + (size_t)(a < ns ? a : 0) * T;
#pragma unroll
    for (int k = 0; k < CN_K; k++) x[a][k] = *(const float *)((const char *)sc + at[k]);
  }
  for (int c0 = 0; c0 < ns; c0 += AHEAD) {
#pragma unroll
    for (int a = 0; a < AHEAD; a++) {
      const int c = c0 + a;
      if (c < ns) {
        float wk[CN_K * M];
        const float *wc = w + (size_t)c * groups * (CN_K * MW);
#pragma unroll
        for (int q = 0; q < CN_K * M; q++) wk[q] = cn_uniform(wc, q / M * MW + q % M);
#pragma unroll
        for (int k = 0; k < CN_K; k++) {
          const float xv = in[k] ? x[a][k] : 0.0f;
#pragma unroll
          for (int m = 0; m < M; m++) acc[m] += wk[k * M + m] * xv;
        }
        const float *nx = src + (size_t)(c + AHEAD < ns ? c + AHEAD : c) * T;
#pragma unroll
        for (int k = 0; k < CN_K; k++) x[a][k] = *(const float *)((const char *)nx + at[k]);
      }
    }
  }
}

// Grid of cn_fwd and cn_bwd: waves of 64 samples (4 a block), then sequences
// and groups of M channels.
struct FmaArgs {
  const float *src;  // [b][ns][T]
  int ns;
  const float *w;  // [ns][groups of 8 output channels][9][8]
  int mc;          // output channels
  int T, dil, tiles;
  int groups, rows;    // groups of the grid's waves; of the weights (8 channels each)
  const float *bias;   // forward
  const float *h_in;   // forward: the residual input; gradient: gh of the layer above (or null)
  float *a, *out;      // forward: tanh, h (last layer: z); gradient: gh
  const float *a_below;  // gradient: a of the layer below
  float *dz;             // gradient: dz of the layer below
  int last;              // forward: the last layer
};
template <int M>
__device__ __forceinline__ void cn_place(const FmaArgs &p, int &b, int &m0, unsigned &t0) {
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const unsigned id = blockIdx.x * 4u + wv;
  const unsigned g = id % (unsigned)p.groups, q = id / (unsigned)p.groups;
  b = (int)(q / (unsigned)p.tiles);
  t0 = (q - (unsigned)b * (unsigned)p.tiles) * 64;
  m0 = (int)g * M;
}

template <int M>
__global__ void __launch_bounds__(256) cn_fwd(FmaArgs p, int B) {
  int b, m0;
  unsigned t0;
  cn_place<M>(p, b, m0, t0);
  if (b >= B) return;
  const unsigned t = t0 + (threadIdx.x & 63);
  float acc[M];
#pragma unroll
  for (int m = 0; m < M; m++) acc[m] = m0 + m < p.mc ? cn_uniform(p.bias, m0 + m) : 0.0f;
  cn_sums<M>(p.src + (size_t)b * p.ns * p.T, p.ns, p.w + m0 / MW * (MW * CN_K) + m0 % MW, p.rows,
             p.T, p.dil, -1, t0, t, acc);
  if (t >= (unsigned)p.T) return;
#pragma unroll
  for (int m = 0; m < M; m++) {
    if (m0 + m >= p.mc) continue;
    const size_t o = ((size_t)b * p.mc + m0 + m) * p.T + t;
    if (p.last) {
      p.out[o] = acc[m];
    } else {
      const float v = tanhf(acc[m]);
      p.a[o] = v;
      if (p.h_in)
        p.out[o] = p.h_in[o] + v;
      else
        p.out[o] = v;
    }
  }
}

// The gradient of a layer's input: gh = [gh +] sums, and dz = gh (1 - a^2)
// of the layer below.
template <int M>
__global__ void __launch_bounds__(256) cn_bwd(FmaArgs p, int B) {
  int b, m0;
  unsigned t0;
  cn_place<M>(p, b, m0, t0);
  if (b >= B) return;
  const unsigned t = t0 + (threadIdx.x & 63);
  float acc[M];
#pragma unroll
  for (int m = 0; m < M; m++) acc[m] = 0.0f;
  cn_sums<M>(p.src + (size_t)b * p.ns * p.T, p.ns, p.w + m0 / MW * (MW * CN_K) + m0 % MW, p.rows,
             p.T, p.dil, 1, t0, t, acc);
  if (t >= (unsigned)p.T) return;
#pragma unroll
  for (int m = 0; m < M; m++) {
    if (m0 + m >= p.mc) continue;
    const size_t o = ((size_t)b * p.mc + m0 + m) * p.T + t;
    const float g = p.h_in ? p.h_in[o] + acc[m] : acc[m], v = p.a_below[o];
    p.out[o] = g;
    p.dz[o] = g * (1.0f - v * v);
  }
}

// dw[co][ci][k] = sum_b sum_t dz[b][co][t] x[b][ci][t - dil (8 - k)] and
// db[co] = sum dz: 256 strided partial sums over the (b, t) in order, then
// a tree. A block takes CO x CI pairs, a thread one partial sum of each
// tap: CO (9 CI) accumulators against CO + 9 CI loads, D samples ahead.
// Bound by those loads' latency (each step of 256 samples is first touched
// by all blocks at once) over two waves a SIMD: 64 x 64 channels, 32
// sequences of 512 samples take 48 us with CO, CI, D = 8, 1, 2 (8, 1, 4:
// 49; 8, 2, 2: 64; 4, 2, 3: 53; 4, 1, 4: 59), of which the multiply-adds
// are 18 (a block per pair, which loaded two values a product: 167).
template <int CO, int CI, int D>
__global__ void __launch_bounds__(256, 1) cn_wgrad(const float *__restrict__ dz, int con,
                                                   const float *__restrict__ x, int cin, int B,
                                                   int T, int dil, float *__restrict__ dw,
                                                   float *__restrict__ dbias) {
  constexpr int NA = CO * CI * CN_K + CO, RB = 32;
  __shared__ float red[RB][256];
  const int tiles = (cin + CI - 1) / CI;
  const int co0 = (int)blockIdx.x / tiles * CO, ci0 = (int)blockIdx.x % tiles * CI;
  // this thread's samples: every 256th of the B T
  const int n = (int)(((int64_t)B * T - (int)threadIdx.x + 255) / 256);
  float acc[NA];  // [co][ci][k], then the bias sums
#pragma unroll
  for (int q = 0; q < NA; q++) acc[q] = 0.0f;
  int lags[CN_K];  // (from T on: no samples)
#pragma unroll
  for (int k = 0; k < CN_K; k++) lags[k] = (int)min((int64_t)T, (int64_t)dil * (CN_K - 1 - k));
  // Sample i of them has time t, and od and ox are the byte offsets of
  // (sequence, channel 0, t) in dz and x.
  // (Past the end the last is read again, channels past the last read the
  // last, and a lag past the start reads x at t: none of those is added.)
  int i = 0;
  int t = (int)(threadIdx.x % T);
  const size_t seq = threadIdx.x / T;
  size_t od = 4 * (seq * con * T + t), ox = 4 * (seq * cin * T + t);
  if (n == 0) od = ox = 0, t = 0;
  float d[D][CO], v[D][CI][CN_K];
  int ts[D];
  auto load = [&](int a) {
    ts[a] = t;
#pragma unroll
    for (int c = 0; c < CO; c++)
      d[a][c] = *(const float *)((const char *)(dz + (size_t)min(co0 + c, con - 1) * T) + od);
#pragma unroll
    for (int k = 0; k < CN_K; k++) {
      const size_t o = t >= lags[k] ? ox - 4 * (size_t)lags[k] : ox;
#pragma unroll
      for (int c = 0; c < CI; c++)
        v[a][c][k] = *(const float *)((const char *)(x + (size_t)min(ci0 + c, cin - 1) * T) + o);
    }
    if (++i < n) {
      od += 1024, ox += 1024;
      unsigned next = (unsigned)t + 256;
      while (next >= (unsigned)T) {  // into the next sequence
        next -= T;
        od += 4 * (size_t)(con - 1) * T, ox += 4 * (size_t)(cin - 1) * T;
      }
      t = (int)next;
    }
  };
#pragma unroll
  for (int a = 0; a < D; a++) load(a);
  for (int u = 0; u < n;) {
#pragma unroll
    for (int a = 0; a < D; a++, u++) {
      if (u < n) {
#pragma unroll
        for (int e = 0; e < CI; e++)
#pragma unroll
          for (int k = 0; k < CN_K; k++) {
            const float xv = ts[a] >= lags[k] ? v[a][e][k] : 0.0f;
#pragma unroll
            for (int c = 0; c < CO; c++) acc[(c * CI + e) * CN_K + k] += d[a][c] * xv;
          }
#pragma unroll
        for (int c = 0; c < CO; c++) acc[CO * CI * CN_K + c] += d[a][c];
      }
      load(a);
    }
  }
  // The tree (threads 128 apart, 64 apart, ... 1 apart), RB sums at a time,
  // a wave per sum.
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
#pragma unroll
  for (int q0 = 0; q0 < NA; q0 += RB) {
    __syncthreads();
#pragma unroll
    for (int q = 0; q < RB; q++)
      if (q0 + q < NA) red[q][threadIdx.x] = acc[q0 + q];
    __syncthreads();
    for (int q = wv; q < RB && q0 + q < NA; q += 4) {
      const float *r = red[q] + lane;
      float s = (r[0] + r[128]) + (r[64] + r[192]);
#pragma unroll
      for (int st = 32; st > 0; st >>= 1) s += __shfl_down(s, st);
      if (lane == 0) {
        const int a = q0 + q;
        if (a >= CO * CI * CN_K) {
          const int co = co0 + a - CO * CI * CN_K;
          if (ci0 == 0 && co < con) dbias[co] = s;
        } else {
          const int k = a % CN_K, e = a / CN_K % CI, c = a / (CN_K * CI);
          if (co0 + c < con && ci0 + e < cin)
            dw[((size_t)(co0 + c) * cin + ci0 + e) * CN_K + k] = s;
        }
      }
    }
  }
}

// Mean squared error over t >= t0 and its gradient; per-block partial sums.
__global__ void __launch_bounds__(256) cn_loss(const float *__restrict__ out,
                                               const float *__restrict__ y, float *__restrict__ g,
                                               size_t n, int T, int t0, float inv_count,
                                               float *__restrict__ partial) {
  __shared__ float red[256];
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  float s = 0.0f;
  if (i < n) {
    const int t = (int)(i % T);
    const float d = t >= t0 ? out[i] - y[i] : 0.0f;
    g[i] = 2.0f * d * inv_count;
    s = d * d;
  }
  red[threadIdx.x] = s;
  __syncthreads();
  for (int st = 128; st > 0; st >>= 1) {
    if ((int)threadIdx.x < st) red[threadIdx.x] += red[threadIdx.x + st];
    __syncthreads();
  }
  if (threadIdx.x == 0) partial[blockIdx.x] = red[0];
}

// The errors of the spectral term, [u][row] (rows padded with zeros to a
// multiple of 8), and K transposed, [u][t]: what cn_spec reads along its
// lanes and through the scalar unit.
__global__ void __launch_bounds__(256) cn_spec_err(const float *__restrict__ out,
                                                   const float *__restrict__ y,
                                                   float *__restrict__ d, int BC, int rs, int T,
                                                   int t0, int len) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (size_t)rs * len) return;
  const int r = (int)(i / len), u = (int)(i % len);  // (lanes along u)
  const size_t o = (size_t)r * T + t0 + u;
  d[(size_t)u * rs + r] = r < BC ? out[o] - y[o] : 0.0f;
}
__global__ void __launch_bounds__(256) cn_transpose(const float *__restrict__ a,
                                                    float *__restrict__ b, int n) {
  __shared__ float s[32][33];
  const int x = threadIdx.x & 31, i0 = blockIdx.x * 32, j0 = blockIdx.y * 32;
  for (int q = threadIdx.x >> 5; q < 32; q += 8)
    if (i0 + q < n && j0 + x < n) s[q][x] = a[(size_t)(i0 + q) * n + j0 + x];
  __syncthreads();
  for (int q = threadIdx.x >> 5; q < 32; q += 8)
    if (j0 + q < n && i0 + x < n) b[(size_t)(j0 + q) * n + i0 + x] = s[x][q];
}

// The spectral term: per sample and output channel (row), the error d over
// samples [t0, t0 + len) adds w d^T K d to the loss and 2 w K d to its
// gradient (K symmetric, len x len). A wave takes 64 outputs t and 8 rows,
// the sum over u in order: K's column u along the lanes, the rows' errors
// through the scalar unit (a thread per output, which read K across its
// rows: 59 us for 64 rows of 384 samples; now 33). Per-block sums of
// d_t (K d)_t.
__global__ void __launch_bounds__(64) cn_spec(const float *__restrict__ out,
                                              const float *__restrict__ y,
                                              const float *__restrict__ Kt,
                                              const float *__restrict__ d, float *__restrict__ g,
                                              int BC, int rs, int T, int t0, int len, float w,
                                              float *__restrict__ partial) {
  const int lane = threadIdx.x, t = blockIdx.y * 64 + lane, r0 = blockIdx.x * 8;
  const float *kp = Kt + min(t, len - 1);
  float acc[8];
#pragma unroll
  for (int r = 0; r < 8; r++) acc[r] = 0.0f;
#pragma unroll 8
  for (int u = 0; u < len; u++) {
    const float k = kp[(size_t)u * len];
#pragma unroll
    for (int r = 0; r < 8; r++) acc[r] += k * cn_uniform(d, (size_t)u * rs + r0 + r);
  }
  float s = 0.0f;
#pragma unroll
  for (int r = 0; r < 8; r++) {
    if (r0 + r >= BC || t >= len) continue;
    const size_t o = (size_t)(r0 + r) * T + t0 + t;
    g[o] += 2.0f * w * acc[r];
    s += (out[o] - y[o]) * acc[r];
  }
  for (int st = 32; st > 0; st >>= 1) s += __shfl_xor(s, st);
  if (lane == 0) partial[blockIdx.y * gridDim.x + blockIdx.x] = w * s;
}

// Per-block sums of g^2 (the gradient norm, for clipping).
__global__ void __launch_bounds__(256) cn_sqsum(const float *__restrict__ g, size_t n,
                                                float *__restrict__ partial) {
  __shared__ float red[256];
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const float x = i < n ? g[i] : 0.0f;
  red[threadIdx.x] = x * x;
  __syncthreads();
  for (int st = 128; st > 0; st >>= 1) {
    if ((int)threadIdx.x < st) red[threadIdx.x] += red[threadIdx.x + st];
    __syncthreads();
  }
  if (threadIdx.x == 0) partial[blockIdx.x] = red[0];
}

// Per-layer table of the weights' orders.
struct CnLayer {
  int ci, co, mt, kc;  // channels; prediction: 32-tiles and 16-chunks
  int gf, gb;          // training: groups of 8 output channels, forward and gradient
  size_t woff;         // into the parameters
  size_t p;            // prediction's operands (in units of 8 bf16 values)
  size_t f, b;         // training's rows
};

// The bf16 values of every layer's weights in prediction's operand order:
// element j of lane `lane`, tile mt, chunk c, tap q is
// w[32 mt + lane % 32][16 c + 8 (lane / 32) + j][q] (zero past the layer's
// channels). A thread per 8 values.
__global__ void __launch_bounds__(256) cn_pack(const float *__restrict__ p,
                                               const CnLayer *__restrict__ layers, int L,
                                               size_t total, u32x4 *__restrict__ w) {
  const size_t e = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (e >= total) return;
  int l = L - 1;
  while (l > 0 && layers[l].p > e) l--;
  const CnLayer y = layers[l];
  size_t i = e - y.p;
  const int lane = (int)(i % 64);
  i /= 64;
  const int tile = (int)(i % y.mt);
  i /= y.mt;
  const int c = (int)(i % y.kc), q = (int)(i / y.kc);
  const int m = 32 * tile + (lane & 31), k0 = 16 * c + 8 * (lane >> 5);
  uint32_t v[8];
#pragma unroll
  for (int j = 0; j < 8; j++) {
    const int k = k0 + j;
    v[j] = m < y.co && k < y.ci ? f32_to_bf16(p[y.woff + ((size_t)m * y.ci + k) * CN_K + q]) : 0u;
  }
  w[e] = u32x4{v[0] | v[1] << 16, v[2] | v[3] << 16, v[4] | v[5] << 16, v[6] | v[7] << 16};
}

// The same values as f32 in training's orders: [source][group of 8 output
// channels][tap][8], source and output ci and co (forward) or co and ci
// (gradient), the groups padded with zeros. A thread per value.
__global__ void __launch_bounds__(256) cn_rows(const float *__restrict__ p,
                                               const CnLayer *__restrict__ layers, int L,
                                               size_t total, float *__restrict__ w) {
  const size_t e = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (e >= total) return;
  int l = L - 1;
  while (l > 0 && layers[l].f > e) l--;
  const CnLayer y = layers[l];
  const bool grad = e >= y.b;
  const size_t i = e - (grad ? y.b : y.f);
  const int gr = grad ? y.gb : y.gf;
  const int k = (int)(i / MW % CN_K), c = (int)(i / (MW * CN_K) / gr);
  const int m = (int)(i / (MW * CN_K) % gr) * MW + (int)(i % MW);
  const int co = grad ? c : m, ci = grad ? m : c;
  w[e] = co < y.co && ci < y.ci
             ? __uint_as_float(
                   (uint32_t)f32_to_bf16(p[y.woff + ((size_t)co * y.ci + ci) * CN_K + k]) << 16)
             : 0.0f;
}

// The sum of n floats by one block, in double, in a fixed order.
__device__ __forceinline__ double cn_total(const float *x, int n, double *red) {
  double s = 0.0;
  for (int i = threadIdx.x; i < n; i += 256) s += (double)x[i];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int st = 128; st > 0; st >>= 1) {
    if ((int)threadIdx.x < st) red[threadIdx.x] += red[threadIdx.x + st];
    __syncthreads();
  }
  const double v = red[0];
  __syncthreads();
  return v;
}

// The loss and the gradient norm (f64 sums of the blocks' partial sums) for
// the host, in pinned memory: res[0], res[1].
__device__ __forceinline__ void cn_result(const float *part, int nb, const float *spart, int nsb,
                                          float inv, double norm2, double *red, float *res) {
  const double s = cn_total(part, nb, red), ss = cn_total(spart, nsb, red);
  if (threadIdx.x == 0) {
    res[0] = (float)(s * inv + ss);
    res[1] = (float)sqrt(norm2);
  }
}
__global__ void __launch_bounds__(256) cn_finish(const float *part, int nb, const float *spart,
                                                 int nsb, float inv, const float *sq, int nsq,
                                                 float *res) {
  __shared__ double red[256];
  const double n2 = cn_total(sq, nsq, red);
  cn_result(part, nb, spart, nsb, inv, n2, red, res);
}

// Adam on the f32 master parameters, the gradient scaled to the norm `clip`
// where it is longer (every block adds up the norm's partial sums itself);
// block 0 leaves the loss and the norm for the host. A weight's new bf16
// value goes to training's rows (cn_rows) at once: packing them afresh cost
// the next step 4 us and a launch.
__global__ void __launch_bounds__(256) cn_adam(float *__restrict__ p, const float *__restrict__ g,
                                               float *__restrict__ m, float *__restrict__ v,
                                               size_t n, float lr, float b1, float b2, float eps,
                                               float c1, float c2, float clip, const float *part,
                                               int nb, const float *spart, int nsb, float inv,
                                               const float *sq, int nsq, float *res,
                                               const CnLayer *__restrict__ layers, int L,
                                               float *__restrict__ rows) {
  __shared__ double red[256];
  const double n2 = cn_total(sq, nsq, red);
  const double gn = sqrt(n2);
  const float gscale = (clip > 0.0f && gn > (double)clip) ? (float)((double)clip / gn) : 1.0f;
  if (blockIdx.x == 0) cn_result(part, nb, spart, nsb, inv, n2, red, res);
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float gi = g[i] * gscale;
  const float mi = b1 * m[i] + (1.0f - b1) * gi;
  const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  const float pi = p[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
  p[i] = pi;
  int l = L - 1;
  while (l > 0 && layers[l].woff > i) l--;
  const CnLayer y = layers[l];
  const size_t w = i - y.woff;
  if (w >= (size_t)y.co * y.ci * CN_K) return;  // a bias
  const int k = (int)(w % CN_K), ci = (int)(w / CN_K % y.ci), co = (int)(w / CN_K / y.ci);
  const float q = __uint_as_float((uint32_t)f32_to_bf16(pi) << 16);
  rows[y.f + (((size_t)ci * y.gf + co / MW) * CN_K + k) * MW + co % MW] = q;
  rows[y.b + (((size_t)co * y.gb + ci / MW) * CN_K + k) * MW + ci % MW] = q;
}

// Samples idx[] of a dataset [n][c][T] into a batch.
__global__ void __launch_bounds__(256) cn_gather(const float *__restrict__ src,
                                                 const int32_t *__restrict__ idx,
                                                 float *__restrict__ dst, int c, int T, int B) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const size_t per = (size_t)c * T;
  if (i >= per * B) return;
  const int b = (int)(i / per);
  dst[i] = src[(size_t)idx[b] * per + (i % per)];
}

unsigned blocks(size_t n) { return (unsigned)((n + 255) / 256); }

}  // namespace

struct ems_cn {
  int cin = 0, cout = 0, C = 0, L = 0;
  std::vector<int> dil;
  std::vector<int> li, lo;          // per layer in/out channels
  std::vector<size_t> woff, boff;   // offsets into the parameter vector
  size_t np = 0;                    // parameters
  float *p = nullptr, *g = nullptr, *m = nullptr, *v = nullptr;
  // the weights' bf16 values as prediction (cn_pack) and training (cn_rows)
  // read them, each made when first needed after a change (training's rows
  // follow its steps), and their table
  std::vector<CnLayer> lay;
  CnLayer *dlay = nullptr;
  u32x4 *w = nullptr;
  float *wr = nullptr;
  size_t nw = 0, nr = 0;
  bool w_ok = false, wr_ok = false;
  int step = 0;
  hipStream_t stream = nullptr;
  // dataset
  float *dx = nullptr, *dy = nullptr;
  int dn = 0, dT = 0;
  // work buffers, each grown when a call needs more
  struct Buf {
    float *d = nullptr;
    size_t n = 0;
  };
  // prediction: input batch, per layer its input ([b][t][padded channels])
  Buf xin;
  std::vector<Buf> hp;
  // training, [b][channel][t]: input and target batches; per layer its
  // input (from layer 1 on) and its tanh; gradients
  Buf hx, hy;
  std::vector<Buf> h, a;
  Buf out, gout, gh, dz[2];
  Buf part, spart, sq, serr;        // partial sums: loss, spectral term, squared gradient; errors
  // spectral loss term (len x len kernel over samples [st0, st0 + slen))
  float *dK = nullptr;              // transposed
  int st0 = 0, slen = 0;
  float sw = 0.0f;
  Buf didx;
  float *res = nullptr;             // pinned: loss, gradient norm
  std::string err;
};

namespace {

int cfail(ems_cn *n, int code, const std::string &m) {
  n->err = m;
  return code;
}

#define CCK(n, x)                                                                       \
  do {                                                                                  \
    hipError_t e_ = (x);                                                                \
    if (e_ != hipSuccess) return cfail((n), EMS_E_DEVICE, std::string(#x ": ") + hipGetErrorString(e_)); \
  } while (0)

constexpr int pad16(int c) { return (c + 15) / 16 * 16; }
constexpr int pad32(int c) { return (c + 31) / 32 * 32; }
int xstride(const ems_cn *n, int l) { return l == 0 ? pad16(n->cin) : pad32(n->C); }

// The work of the stream ends before a buffer that it may use is replaced.
int grow(ems_cn *n, ems_cn::Buf &b, size_t need) {
  if (need <= b.n) return 0;
  CCK(n, hipStreamSynchronize(n->stream));
  if (b.d) CCK(n, hipFree(b.d));
  b.d = nullptr, b.n = 0;
  CCK(n, hipMalloc(&b.d, need * sizeof(float)));
  b.n = need;
  return 0;
}

int ensure_predict(ems_cn *n, int B, int T) {
  const size_t BT = (size_t)B * T;
  int rc;
  n->hp.resize(n->L);
  if ((rc = grow(n, n->xin, BT * n->cin))) return rc;
  for (int l = 1; l < n->L; l++)
    if ((rc = grow(n, n->hp[l], BT * xstride(n, l)))) return rc;
  return grow(n, n->out, BT * n->cout);
}

int ensure_train(ems_cn *n, int B, int T) {
  const size_t BT = (size_t)B * T;
  int rc;
  // (with the first training call: a network that only predicts has neither)
  if (!n->wr) CCK(n, hipMalloc(&n->wr, n->nr * sizeof(float)));
  if (!n->res)
    CCK(n, hipHostMalloc((void **)&n->res, 2 * sizeof(float), hipHostMallocDefault));
  n->h.resize(n->L), n->a.resize(n->L);
  if ((rc = grow(n, n->hx, BT * n->cin))) return rc;
  if ((rc = grow(n, n->hy, BT * n->cout))) return rc;
  if ((rc = grow(n, n->out, BT * n->cout))) return rc;
  if ((rc = grow(n, n->gout, BT * n->cout))) return rc;
  for (int l = 0; l < n->L; l++) {
    if (l > 0 && (rc = grow(n, n->h[l], BT * n->C))) return rc;
    if (l < n->L - 1 && (rc = grow(n, n->a[l], BT * n->C))) return rc;
  }
  if ((rc = grow(n, n->gh, BT * n->C))) return rc;
  for (auto &d : n->dz)
    if ((rc = grow(n, d, BT * n->C))) return rc;
  if ((rc = grow(n, n->part, blocks(BT * n->cout)))) return rc;
  if (n->sw != 0.0f) {  // the spectral term's errors and partial sums
    const size_t rs = ((size_t)B * n->cout + 7) / 8 * 8;
    if ((rc = grow(n, n->spart, (size_t)((n->slen + 63) / 64) * (rs / 8)))) return rc;
    if ((rc = grow(n, n->serr, rs * n->slen))) return rc;
  }
  if ((rc = grow(n, n->sq, blocks(n->np)))) return rc;
  return grow(n, n->didx, B);
}

template <int MODE, int KC>
int launch_conv_k(ems_cn *n, ConvArgs a, int B) {
  const size_t lds = cn_lds(a.ml, KC);
  if (lds > 64 * 1024)
    CCK(n, hipFuncSetAttribute((const void *)cn_conv<MODE, KC>,
                               hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  // (a launch holds fewer than 2^32 threads)
  constexpr uint64_t MOST = 1u << 22;
  const uint64_t nb = (uint64_t)a.pt * a.nt * B;
  for (uint64_t b0 = 0; b0 < nb; b0 += MOST) {
    a.blk0 = (unsigned)b0;
    hipLaunchKernelGGL((cn_conv<MODE, KC>),
                       dim3((unsigned)std::min(MOST, nb - b0), (unsigned)((a.mt + 1) / 2)),
                       dim3(512), lds, n->stream, a);
    CCK(n, hipGetLastError());
  }
  return 0;
}

// Samples per phase: the split into phases with the fewest blocks, of equal
// ones the longest runs (the fewest source rows). Channels staged at a
// time: 64 or 32 where the source's rows hold a multiple of them, else 16
// (at most 192 rows and 83 KB).
template <int MODE>
int launch_conv(ems_cn *n, ConvArgs a, int B) {
  const int S = (a.T - 1) / a.dil + 1;  // samples of the longest phase
  int64_t best = -1;
  for (int ml = CN_TT; ml >= 4; ml /= 2) {
    const int64_t pt = ((int64_t)std::min(a.dil, a.T) + CN_TT / ml - 1) / (CN_TT / ml);
    const int64_t nt = (S + ml - 1) / ml;
    if (best < 0 || pt * nt < best) best = pt * nt, a.ml = ml, a.pt = (int)pt, a.nt = (int)nt;
  }
  if (a.cps % 64 == 0) return launch_conv_k<MODE, 64>(n, a, B);
  if (a.cps % 32 == 0) return launch_conv_k<MODE, 32>(n, a, B);
  return launch_conv_k<MODE, 16>(n, a, B);
}

int weights_predict(ems_cn *n) {
  if (n->w_ok) return 0;
  hipLaunchKernelGGL(cn_pack, dim3(blocks(n->nw)), dim3(256), 0, n->stream, n->p, n->dlay, n->L,
                     n->nw, n->w);
  CCK(n, hipGetLastError());
  n->w_ok = true;
  return 0;
}
int weights_train(ems_cn *n) {
  if (n->wr_ok) return 0;
  hipLaunchKernelGGL(cn_rows, dim3(blocks(n->nr)), dim3(256), 0, n->stream, n->p, n->dlay, n->L,
                     n->nr, n->wr);
  CCK(n, hipGetLastError());
  n->wr_ok = true;
  return 0;
}

// Prediction of the batch in n->xin; output in n->out.
int predict(ems_cn *n, int B, int T) {
  int rc = weights_predict(n);
  if (rc) return rc;
  for (int l = 0; l < n->L; l++) {
    const CnLayer &y = n->lay[l];
    ConvArgs a{};
    a.src = l > 0 ? n->hp[l].d : n->xin.d;
    a.cps = xstride(n, l);
    if (l == 0) a.craw = n->cin;
    a.w = n->w + y.p, a.mt = y.mt, a.mc = n->lo[l];
    a.T = T, a.dil = n->dil[l];
    a.bias = n->p + n->boff[l];
    if (l == n->L - 1) {
      a.out = n->out.d;
      rc = launch_conv<CN_OUT>(n, a, B);
    } else {
      a.h_in = l > 0 ? n->hp[l].d : nullptr;
      a.h_out = n->hp[l + 1].d;
      rc = launch_conv<CN_HIDDEN>(n, a, B);
    }
    if (rc) return rc;
  }
  return 0;
}

template <bool FWD, int M>
void launch_fma_m(ems_cn *n, FmaArgs a, int B) {
  a.groups = (a.mc + M - 1) / M;
  const dim3 g((unsigned)(((size_t)B * a.tiles * a.groups + 3) / 4)), t(256);
  if (FWD) hipLaunchKernelGGL(cn_fwd<M>, g, t, 0, n->stream, a, B);
  else hipLaunchKernelGGL(cn_bwd<M>, g, t, 0, n->stream, a, B);
}

template <bool FWD>
int launch_fma(ems_cn *n, FmaArgs a, int B) {
  a.tiles = (a.T - 1) / 64 + 1;
  a.rows = (a.mc + MW - 1) / MW;
  // Fewer such waves than SIMDs: a wave per output channel, whose chain over
  // the source channels is shorter (64 channels, 8 sequences of 512 samples
  // 253 us a step against 335, 256 channels and one trace of 16 samples 769
  // against 1138; at 1024 waves 379 against 374, at 2048 601 against 447).
  if ((size_t)B * a.tiles * a.rows < 1024) launch_fma_m<FWD, 1>(n, a, B);
  else launch_fma_m<FWD, MW>(n, a, B);
  CCK(n, hipGetLastError());
  return 0;
}

// Training's forward pass of the batch in n->hx; output in n->out.
int forward(ems_cn *n, int B, int T) {
  int rc = weights_train(n);
  if (rc) return rc;
  for (int l = 0; l < n->L; l++) {
    const CnLayer &y = n->lay[l];
    FmaArgs a{};
    a.src = l == 0 ? n->hx.d : n->h[l].d;
    a.ns = n->li[l];
    a.w = n->wr + y.f, a.mc = n->lo[l];
    a.T = T, a.dil = n->dil[l];
    a.bias = n->p + n->boff[l];
    a.last = l == n->L - 1;
    a.out = a.last ? n->out.d : n->h[l + 1].d;
    a.a = a.last ? nullptr : n->a[l].d;
    a.h_in = l > 0 ? n->h[l].d : nullptr;
    if ((rc = launch_fma<true>(n, a, B))) return rc;
  }
  return 0;
}

// What the loss and norm kernels add up.
struct Sums {
  int nb = 0, nsb = 0, nsq = 0;
  float inv = 0.0f;
};

// Loss over t >= t0 against n->hy and the parameter gradient in n->g; the
// partial sums of the loss and the squared gradient stay on the device.
int backward(ems_cn *n, int B, int T, int t0, Sums *sums) {
  const size_t BT = (size_t)B * T;
  const size_t no = BT * n->cout;
  const int Tv = T - t0 > 0 ? T - t0 : 1;
  sums->inv = 1.0f / (float)((size_t)B * n->cout * Tv);
  sums->nb = (int)blocks(no);
  hipLaunchKernelGGL(cn_loss, dim3(sums->nb), dim3(256), 0, n->stream, n->out.d, n->hy.d, n->gout.d,
                     no, T, t0, sums->inv, n->part.d);
  CCK(n, hipGetLastError());
  sums->nsb = 0;
  if (n->sw != 0.0f) {
    if (n->st0 + n->slen > T) return cfail(n, EMS_E_INVALID, "spectral term past the sequence end");
    const int BC = B * n->cout, rs = (BC + 7) / 8 * 8;
    hipLaunchKernelGGL(cn_spec_err, dim3(blocks((size_t)rs * n->slen)), dim3(256), 0, n->stream,
                       n->out.d, n->hy.d, n->serr.d, BC, rs, T, n->st0, n->slen);
    CCK(n, hipGetLastError());
    const dim3 gr((unsigned)(rs / 8), (unsigned)((n->slen + 63) / 64));
    sums->nsb = (int)(gr.x * gr.y);
    hipLaunchKernelGGL(cn_spec, gr, dim3(64), 0, n->stream, n->out.d, n->hy.d, n->dK, n->serr.d,
                       n->gout.d, BC, rs, T, n->st0, n->slen, n->sw / (float)BC, n->spart.d);
    CCK(n, hipGetLastError());
  }
  for (int l = n->L - 1; l >= 0; l--) {
    const bool last = l == n->L - 1;
    const CnLayer &y = n->lay[l];
    const float *dz = last ? n->gout.d : n->dz[l & 1].d;
    const float *x = l == 0 ? n->hx.d : n->h[l].d;
    constexpr int CO = 8, CI = 1;
    const unsigned nb = (unsigned)((n->lo[l] + CO - 1) / CO) * (unsigned)((n->li[l] + CI - 1) / CI);
    hipLaunchKernelGGL((cn_wgrad<CO, CI, 2>), dim3(nb), dim3(256), 0, n->stream, dz, n->lo[l], x,
                       n->li[l], B, T, n->dil[l], n->g + n->woff[l], n->g + n->boff[l]);
    CCK(n, hipGetLastError());
    if (l > 0) {
      // gradient of h[l]: through the conv, plus the skip path of a
      // residual layer (h[l+1] = h[l] + a[l]); then dz of the layer below.
      FmaArgs a{};
      a.src = dz, a.ns = n->lo[l];
      a.w = n->wr + y.b, a.mc = n->li[l];
      a.T = T, a.dil = n->dil[l];
      a.h_in = last ? nullptr : n->gh.d;
      a.out = n->gh.d, a.a_below = n->a[l - 1].d, a.dz = n->dz[(l - 1) & 1].d;
      const int rc = launch_fma<false>(n, a, B);
      if (rc) return rc;
    }
  }
  sums->nsq = (int)blocks(n->np);
  hipLaunchKernelGGL(cn_sqsum, dim3(sums->nsq), dim3(256), 0, n->stream, n->g, n->np, n->sq.d);
  CCK(n, hipGetLastError());
  return 0;
}

}  // namespace

extern "C" {

int ems_cn_create(int cin, int cout, int channels, int layers, const int32_t *dilation,
                  uint64_t seed, ems_cn **out) {
  if (!out || cin < 1 || cout < 1 || channels < 1 || layers < 2 || !dilation) return EMS_E_INVALID;
  ems_cn *n = new ems_cn();
  n->cin = cin, n->cout = cout, n->C = channels, n->L = layers;
  for (int l = 0; l < layers; l++) {
    if (dilation[l] < 1) {
      delete n;
      return EMS_E_INVALID;
    }
    n->dil.push_back(dilation[l]);
    n->li.push_back(l == 0 ? cin : channels);
    n->lo.push_back(l == layers - 1 ? cout : channels);
  }
  for (int l = 0; l < layers; l++) {
    n->woff.push_back(n->np);
    n->np += (size_t)n->lo[l] * n->li[l] * CN_K;
    n->boff.push_back(n->np);
    n->np += n->lo[l];
  }
  // Initial weights: normal(0, 1/sqrt(fan_in)), the output layer 0.1 of
  // that; biases 0.
  std::vector<float> p(n->np, 0.0f);
  std::mt19937_64 rng(seed);
  std::normal_distribution<float> nd(0.0f, 1.0f);
  for (int l = 0; l < layers; l++) {
    const float sc = (l == layers - 1 ? 0.1f : 1.0f) / std::sqrt((float)(n->li[l] * CN_K));
    for (size_t q = 0; q < (size_t)n->lo[l] * n->li[l] * CN_K; q++) p[n->woff[l] + q] = nd(rng) * sc;
  }
  for (int l = 0; l < layers; l++) {
    CnLayer y;
    y.ci = n->li[l], y.co = n->lo[l];
    y.mt = pad32(y.co) / 32, y.kc = xstride(n, l) / 16;
    y.gf = (y.co + MW - 1) / MW, y.gb = (y.ci + MW - 1) / MW;
    y.woff = n->woff[l];
    y.p = n->nw;
    n->nw += (size_t)CN_K * y.kc * y.mt * 64;
    y.f = n->nr;
    n->nr += (size_t)y.ci * y.gf * CN_K * MW;
    y.b = n->nr;
    n->nr += (size_t)y.co * y.gb * CN_K * MW;
    n->lay.push_back(y);
  }
  if (hipStreamCreateWithFlags(&n->stream, hipStreamNonBlocking) != hipSuccess ||
      hipMalloc(&n->p, n->np * 4) != hipSuccess || hipMalloc(&n->g, n->np * 4) != hipSuccess ||
      hipMalloc(&n->m, n->np * 4) != hipSuccess || hipMalloc(&n->v, n->np * 4) != hipSuccess ||
      hipMalloc(&n->w, n->nw * sizeof(u32x4)) != hipSuccess ||
      hipMalloc(&n->dlay, n->lay.size() * sizeof(CnLayer)) != hipSuccess ||
      hipMemcpyAsync(n->dlay, n->lay.data(), n->lay.size() * sizeof(CnLayer),
                     hipMemcpyHostToDevice, n->stream) != hipSuccess) {
    ems_cn_destroy(n);
    return EMS_E_DEVICE;
  }
  *out = n;
  return ems_cn_set_params(n, p.data(), n->np);
}

void ems_cn_destroy(ems_cn *n) {
  if (!n) return;
  if (n->stream) (void)hipStreamSynchronize(n->stream);
  for (void *q : {(void *)n->p, (void *)n->g, (void *)n->m, (void *)n->v, (void *)n->w,
                  (void *)n->wr,
                  (void *)n->dlay, (void *)n->dx, (void *)n->dy, (void *)n->dK})
    if (q) (void)hipFree(q);
  for (auto *q : {&n->hx, &n->xin, &n->hy, &n->out, &n->gout, &n->gh, &n->dz[0], &n->dz[1],
                  &n->part, &n->spart, &n->sq, &n->serr, &n->didx})
    if (q->d) (void)hipFree(q->d);
  for (auto *v : {&n->h, &n->a, &n->hp})
    for (auto &q : *v)
      if (q.d) (void)hipFree(q.d);
  if (n->res) (void)hipHostFree(n->res);
  if (n->stream) (void)hipStreamDestroy(n->stream);
  delete n;
}

const char *ems_cn_last_error(const ems_cn *n) { return n ? n->err.c_str() : "null network"; }

uint64_t ems_cn_param_count(const ems_cn *n) { return n ? n->np : 0; }

int ems_cn_set_params(ems_cn *n, const float *p, uint64_t count) {
  if (!n || !p || count != n->np) return EMS_E_INVALID;
  CCK(n, hipMemcpyAsync(n->p, p, n->np * 4, hipMemcpyHostToDevice, n->stream));
  CCK(n, hipMemsetAsync(n->m, 0, n->np * 4, n->stream));
  CCK(n, hipMemsetAsync(n->v, 0, n->np * 4, n->stream));
  n->w_ok = n->wr_ok = false;
  CCK(n, hipStreamSynchronize(n->stream));
  n->step = 0;
  return EMS_OK;
}

int ems_cn_get_params(ems_cn *n, float *p, uint64_t count) {
  if (!n || !p || count != n->np) return EMS_E_INVALID;
  CCK(n, hipStreamSynchronize(n->stream));
  CCK(n, hipMemcpyAsync(p, n->p, n->np * 4, hipMemcpyDeviceToHost, n->stream));
  CCK(n, hipStreamSynchronize(n->stream));
  return EMS_OK;
}

int ems_cn_set_spectral(ems_cn *n, const float *K, int t0, int len, float weight) {
  if (!n || t0 < 0 || len < 0 || (weight != 0.0f && (!K || len < 1))) return EMS_E_INVALID;
  if (n->dK) CCK(n, hipFree(n->dK));
  n->dK = nullptr, n->sw = 0.0f, n->st0 = 0, n->slen = 0;
  if (weight == 0.0f) return EMS_OK;
  const size_t bytes = (size_t)len * len * sizeof(float);
  CCK(n, hipMalloc(&n->dK, bytes));
  float *rows = nullptr;
  CCK(n, hipMalloc(&rows, bytes));
  CCK(n, hipMemcpyAsync(rows, K, bytes, hipMemcpyHostToDevice, n->stream));
  const unsigned nt = (unsigned)((len + 31) / 32);
  hipLaunchKernelGGL(cn_transpose, dim3(nt, nt), dim3(256), 0, n->stream, rows, n->dK, len);
  CCK(n, hipGetLastError());
  CCK(n, hipStreamSynchronize(n->stream));
  CCK(n, hipFree(rows));
  n->sw = weight, n->st0 = t0, n->slen = len;
  return EMS_OK;
}

int ems_cn_set_data(ems_cn *n, const float *x, const float *y, int count, int T) {
  if (!n || !x || !y || count < 1 || T < 1) return EMS_E_INVALID;
  if (n->dx) CCK(n, hipFree(n->dx));
  if (n->dy) CCK(n, hipFree(n->dy));
  n->dx = n->dy = nullptr;
  const size_t nx = (size_t)count * n->cin * T, ny = (size_t)count * n->cout * T;
  CCK(n, hipMalloc(&n->dx, nx * 4));
  CCK(n, hipMalloc(&n->dy, ny * 4));
  CCK(n, hipMemcpyAsync(n->dx, x, nx * 4, hipMemcpyHostToDevice, n->stream));
  CCK(n, hipMemcpyAsync(n->dy, y, ny * 4, hipMemcpyHostToDevice, n->stream));
  CCK(n, hipStreamSynchronize(n->stream));
  n->dn = count, n->dT = T;
  return EMS_OK;
}

int ems_cn_train_batch(ems_cn *n, const int32_t *idx, int B, int t0, float lr, float clip,
                       float *loss, float *grad_norm) {
  if (!n || !idx || B < 1 || !n->dx) return EMS_E_INVALID;
  for (int b = 0; b < B; b++)
    if (idx[b] < 0 || idx[b] >= n->dn) return cfail(n, EMS_E_INVALID, "sample index out of range");
  const int T = n->dT;
  int rc = ensure_train(n, B, T);
  if (rc) return rc;
  int32_t *didx = (int32_t *)n->didx.d;
  CCK(n, hipMemcpyAsync(didx, idx, B * sizeof(int32_t), hipMemcpyHostToDevice, n->stream));
  hipLaunchKernelGGL(cn_gather, dim3(blocks((size_t)B * n->cin * T)), dim3(256), 0, n->stream,
                     n->dx, didx, n->hx.d, n->cin, T, B);
  hipLaunchKernelGGL(cn_gather, dim3(blocks((size_t)B * n->cout * T)), dim3(256), 0, n->stream,
                     n->dy, didx, n->hy.d, n->cout, T, B);
  CCK(n, hipGetLastError());
  if ((rc = forward(n, B, T))) return rc;
  Sums s;
  if ((rc = backward(n, B, T, t0, &s))) return rc;
  n->step++;
  const float b1 = 0.9f, b2 = 0.999f;
  const float c1 = 1.0f - std::pow(b1, (float)n->step), c2 = 1.0f - std::pow(b2, (float)n->step);
  hipLaunchKernelGGL(cn_adam, dim3(blocks(n->np)), dim3(256), 0, n->stream, n->p, n->g, n->m, n->v,
                     n->np, lr, b1, b2, 1e-8f, c1, c2, clip, n->part.d, s.nb, n->spart.d, s.nsb,
                     s.inv, n->sq.d, s.nsq, n->res, n->dlay, n->L, n->wr);
  CCK(n, hipGetLastError());
  n->w_ok = false;
  CCK(n, hipStreamSynchronize(n->stream));
  if (loss) *loss = n->res[0];
  if (grad_norm) *grad_norm = n->res[1];
  return EMS_OK;
}

int ems_cn_forward(ems_cn *n, const float *x, int B, int T, float *out) {
  if (!n || !x || !out || B < 1 || T < 1) return EMS_E_INVALID;
  int rc = ensure_predict(n, B, T);
  if (rc) return rc;
  CCK(n, hipMemcpyAsync(n->xin.d, x, (size_t)B * n->cin * T * 4, hipMemcpyHostToDevice, n->stream));
  if ((rc = predict(n, B, T))) return rc;
  CCK(n, hipMemcpyAsync(out, n->out.d, (size_t)B * n->cout * T * 4, hipMemcpyDeviceToHost,
                        n->stream));
  CCK(n, hipStreamSynchronize(n->stream));
  return EMS_OK;
}

int ems_cn_loss_grad(ems_cn *n, const float *x, const float *y, int B, int T, int t0, float *loss,
                     float *grad) {
  if (!n || !x || !y || B < 1 || T < 1) return EMS_E_INVALID;
  int rc = ensure_train(n, B, T);
  if (rc) return rc;
  CCK(n, hipMemcpyAsync(n->hx.d, x, (size_t)B * n->cin * T * 4, hipMemcpyHostToDevice, n->stream));
  CCK(n, hipMemcpyAsync(n->hy.d, y, (size_t)B * n->cout * T * 4, hipMemcpyHostToDevice, n->stream));
  if ((rc = forward(n, B, T))) return rc;
  Sums s;
  if ((rc = backward(n, B, T, t0, &s))) return rc;
  hipLaunchKernelGGL(cn_finish, dim3(1), dim3(256), 0, n->stream, n->part.d, s.nb, n->spart.d,
                     s.nsb, s.inv, n->sq.d, s.nsq, n->res);
  CCK(n, hipGetLastError());
  CCK(n, hipStreamSynchronize(n->stream));
  if (loss) *loss = n->res[0];
  if (grad) {
    CCK(n, hipMemcpyAsync(grad, n->g, n->np * 4, hipMemcpyDeviceToHost, n->stream));
    CCK(n, hipStreamSynchronize(n->stream));
  }
  return EMS_OK;
}

}  // extern "C"
