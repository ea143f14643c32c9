// Opcode 19 (model auxiliary f32 ops) on gfx950: the normalizations,
// modulation, activations, layout changes and gated MLP products that sit
// between the GEMMs of a DiT / text-encoder block.
//
// Semantics (reference src/dsp/ops/mat_mul.c:2356-2486, hvx_model_aux_f32
// :2488-2501; activation formulas :787-826):
//   modes 0/1/9  one row of `width` per task: mean (mode 1: 0), centered sum of
//                squares, inv = 1/sqrt(sumsq/width + eps), v = (x-mean)*inv, then
//                affine w[i]/b[i] (modes 0/1) or modulation v += v*w; v += b
//                (mode 9, per batch when other_count != width); optional SiLU
//   mode 2       group norm, one task per (batch, group) of spatial*channels/groups
//                contiguous values, per-channel affine
//   modes 3/4    x + w[i % other_count] / x * w[i % other_count]
//   modes 5/6/7  SiLU / GELU-tanh / QuickGELU
//   mode 8       per-batch transpose [width][spatial] -> [spatial][width]
//   mode 10      x[i] * w[batch-or-0][i % width] + b[i]
//   mode 11      rotary embedding with 2x2 matrices per (token, pair), written in
//                [batch][head][token][dim] order
//   modes 12/13  SiLU(gate) * up from [.., gate | up ..] rows (13 also copies
//                an attention row in front of each output row)
// Every float step is one IEEE binary32 operation in the reference's order;
// the row sums of the norms accumulate in double (the reference sums its 32
// lanes in double, mat_mul.c:2352-2355), so mean and inv match a double
// restatement except at rounding ties.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstdint>

#include "hb_internal.h"

namespace {

#include "hb_lds_ring.h"

constexpr int kAuxThreads = 256;

int device_cus() {
  int dev = 0, v = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || v <= 0)
    v = 256;
  return v;
}

// x * sigmoid(z), with the stable sigmoid e/(1+e) for z < 0, e = 2^max(-|z|*log2(e), -126).
// On these arguments the exponential instruction gives exp2f's bits (every
// float in [-126, 0]) and one Newton step from the reciprocal instruction
// gives those of the division (every float in [1, 2]); both checked for all
// of them.  The library function and the division sequence are about half of
// the instructions of an element.
__device__ inline float times_sigmoid(float x, float z) {
  const float neg = fmaxf(__fmul_rn(fabsf(z), -1.4426950408889634f), -126.0f);
  const float e = __builtin_amdgcn_exp2f(neg);
  const float d = __fadd_rn(e, 1.0f), r = __builtin_amdgcn_rcpf(d);
  const float inv = __fmaf_rn(__fmaf_rn(-d, r, 1.0f), r, r);
  return __fmul_rn(x, z < 0.0f ? __fmul_rn(e, inv) : inv);
}

// Activation ids of the reference epilogue: 1 GELU-tanh, 2 QuickGELU, 4 and 5 SiLU.
__device__ inline float activate(float x, int act) {
  if (act == 1) {
    const float cubic = __fmul_rn(__fmul_rn(x, x), x);
    const float inner = __fadd_rn(x, __fmul_rn(cubic, 0.044715f));
    return times_sigmoid(x, __fmul_rn(inner, 1.5957691216057308f));
  }
  if (act == 2) return times_sigmoid(x, __fmul_rn(x, 1.702f));
  if (act == 4 || act == 5) return times_sigmoid(x, x);
  return x;
}

template <int T = kAuxThreads>
__device__ inline double block_sum(double v, double *red) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  __syncthreads();  // red may still be read from the previous reduction
  if (lane == 0) red[wave] = v;
  __syncthreads();
  double t = 0.0;
#pragma unroll
  for (int w = 0; w < T / 64; ++w) t += red[w];
  return t;
}

// Affine / modulation step of the norms for element i of the task (MODE as in aux_norm).
// Mode 2: a task is one (batch, group) of channels/groups whole channels, so
// the channel of element i is pbase + i / spatial with pbase = (task % groups)
// * channels / groups (the reference's ((offset + i) / spatial) % channels).
template <int MODE>
__device__ inline float norm_affine(float v, int i, const float *w, const float *b, size_t pbase, int spatial) {
  if (MODE == 0 || MODE == 1) {
    if (w) v = __fmul_rn(v, w[i]);
    if (b) v = __fadd_rn(v, b[i]);
  } else if (MODE == 2) {
    const int ch = (int)pbase + (int)((unsigned)i / (unsigned)spatial);
    if (w) v = __fmul_rn(v, w[ch]);
    if (b) v = __fadd_rn(v, b[ch]);
  } else {
    v = __fadd_rn(v, __fmul_rn(v, w[pbase + i]));
    v = __fadd_rn(v, b[pbase + i]);
  }
  return v;
}

// Modes 0, 1, 2, 9 with the task held in registers: T threads x NV float4,
// len % 4 == 0 and 16-byte aligned rows; x is read once.
template <int MODE, int NV, int T>
__global__ __launch_bounds__(T) void aux_norm_reg(float *__restrict__ y, const float *__restrict__ x,
                                                  const float *__restrict__ w, const float *__restrict__ b, int len,
                                                  int width, int channels, int spatial, int groups, int other_count,
                                                  float eps, int act) {
  __shared__ double red[T / 64];
  const size_t offset = (size_t)blockIdx.x * (size_t)len;
  const float4 *xr = (const float4 *)(x + offset);
  const int nv4 = len / 4;
  float4 v[NV];
#pragma unroll
  for (int j = 0; j < NV; ++j) v[j] = xr[min((int)threadIdx.x + j * T, nv4 - 1)];
  float mean = 0.0f;
  if (MODE != 1) {
    double s = 0.0;
#pragma unroll
    for (int j = 0; j < NV; ++j)
      if ((int)threadIdx.x + j * T < nv4) s += (double)v[j].x + (double)v[j].y + (double)v[j].z + (double)v[j].w;
    mean = (float)(block_sum<T>(s, red) / (double)len);
  }
  double q = 0.0;
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    if ((int)threadIdx.x + j * T < nv4) {
      const double d0 = __fsub_rn(v[j].x, mean), d1 = __fsub_rn(v[j].y, mean), d2 = __fsub_rn(v[j].z, mean),
                   d3 = __fsub_rn(v[j].w, mean);
      q += d0 * d0 + d1 * d1 + d2 * d2 + d3 * d3;
    }
  }
  const float inv = __fdiv_rn(1.0f, __fsqrt_rn((float)(block_sum<T>(q, red) / (double)len + (double)eps)));
  const size_t pbase = MODE == 9 ? (other_count != width ? (size_t)(blockIdx.x / spatial) * (size_t)width : 0)
                      : MODE == 2 ? (size_t)(blockIdx.x % groups) * (size_t)(channels / groups)
                                  : 0;
  float4 *yr = (float4 *)(y + offset);
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    const int idx = (int)threadIdx.x + j * T;
    if (idx < nv4) {
      float o[4] = {v[j].x, v[j].y, v[j].z, v[j].w};
      if (MODE == 2) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float t = norm_affine<MODE>(__fmul_rn(__fsub_rn(o[e], mean), inv), 4 * idx + e, w, b, pbase, spatial);
          o[e] = act ? activate(t, 4) : t;
        }
      } else {
        // the row's parameters are 16-byte aligned quads (width % 4 == 0)
        const float4 wv = w ? ((const float4 *)(w + pbase))[idx] : make_float4(1.0f, 1.0f, 1.0f, 1.0f);
        const float4 bv = b ? ((const float4 *)(b + pbase))[idx] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        const float wq[4] = {wv.x, wv.y, wv.z, wv.w}, bq[4] = {bv.x, bv.y, bv.z, bv.w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          float t = __fmul_rn(__fsub_rn(o[e], mean), inv);
          if (MODE == 9) {
            t = __fadd_rn(t, __fmul_rn(t, wq[e]));
            t = __fadd_rn(t, bq[e]);
          } else {
            if (w) t = __fmul_rn(t, wq[e]);
            if (b) t = __fadd_rn(t, bq[e]);
          }
          o[e] = act ? activate(t, 4) : t;
        }
      }
      yr[idx] = make_float4(o[0], o[1], o[2], o[3]);
    }
  }
}

// Modes 0, 1, 2, 9, any task length: one workgroup of T threads per task of
// `len` contiguous values, three passes (the later ones mostly from cache).
template <int MODE, int T>
__global__ __launch_bounds__(T) void aux_norm(float *__restrict__ y, const float *__restrict__ x,
                                              const float *__restrict__ w, const float *__restrict__ b, int len,
                                              int width, int channels, int spatial, int groups, int other_count,
                                              float eps, int act) {
  __shared__ double red[T / 64];
  const size_t offset = (size_t)blockIdx.x * (size_t)len;
  const float *xr = x + offset;
  float *yr = y + offset;
  float mean = 0.0f;
  if (MODE != 1) {
    double s = 0.0;
    for (int i = threadIdx.x; i < len; i += T) s += (double)xr[i];
    mean = (float)(block_sum<T>(s, red) / (double)len);
  }
  double q = 0.0;
  for (int i = threadIdx.x; i < len; i += T) {
    const double v = (double)__fsub_rn(xr[i], mean);
    q += v * v;
  }
  const float inv = __fdiv_rn(1.0f, __fsqrt_rn((float)(block_sum<T>(q, red) / (double)len + (double)eps)));
  // mode 9: per-batch parameters unless they are shared by all batches; mode 2: the group's first channel
  const size_t pbase = MODE == 9 ? (other_count != width ? (size_t)(blockIdx.x / spatial) * (size_t)width : 0)
                      : MODE == 2 ? (size_t)(blockIdx.x % groups) * (size_t)(channels / groups)
                                  : 0;
  for (int i = threadIdx.x; i < len; i += T) {
    float v = __fmul_rn(__fsub_rn(xr[i], mean), inv);
    v = norm_affine<MODE>(v, i, w, b, pbase, spatial);
    if (act) v = activate(v, 4);
    yr[i] = v;
  }
}

// Group norm over few long groups: each group is split into `chunks` pieces
// of `chunk` values (a multiple of 4) handled by separate workgroups, in two
// launches.  The first reads x once for shifted sums per chunk: with s the
// group's first value and d = x - s (exact in double for floats within 2^29
// of each other, otherwise below 1e-16 relative), sum d and sum d^2.
// The second adds the chunk partials in chunk order (so every workgroup of a
// group derives the same mean and inv), takes the reference's float mean
// (float)(sum x / len) with sum x = sum d + len * s, and its centered sum of
// squares about that mean, sum (x - mean)^2 = sum d^2 - 2 e sum d + len e^2
// with e = mean - s (exact in double), then writes the output.  The
// reference's second pass rounds each x - mean to float before squaring;
// the two sums differ by about 1e-10 relative (1e-16 * len in the worst
// case, a shift far from every other value), so inv is the same float but
// at rounding ties.  Centering on a sample of the group keeps the
// cancellation bounded where |mean| >> standard deviation.
// ws: double sum[tasks][chunks], then double sq[tasks][chunks].
constexpr int kGnUnroll = 4;
constexpr int kGnMaxPieces = 64;  // workgroups per group of aux_group_norm_resident

__device__ inline void shifted_add(const float4 v, double shift, double &s, double &q) {
  const double d0 = (double)v.x - shift, d1 = (double)v.y - shift, d2 = (double)v.z - shift,
               d3 = (double)v.w - shift;
  s += (d0 + d1) + (d2 + d3);
  q = fma(d3, d3, fma(d2, d2, fma(d1, d1, fma(d0, d0, q))));
}

// n / d for quotients below 2^22: the float estimate n * (1/d) is within one
// of the quotient there (three roundings of 2^-24 each), and one step against
// the remainder makes it exact.
__device__ inline unsigned small_quotient(unsigned n, unsigned d, float rd) {
  int q = (int)__fmul_rn((float)n, rd);
  const int r = (int)n - q * (int)d;
  q += r < 0 ? -1 : (r >= (int)d ? 1 : 0);
  return (unsigned)q;
}

// The float mean of the reference and 1 / sqrt of its variance from the
// shifted sums of a whole group.
__device__ inline void gn_stats(double ts, double tq, int len, float shift, float eps, float *stats) {
  const double n = (double)len;
  const float mean = (float)((ts + n * (double)shift) / n);
  const double e = (double)mean - (double)shift;
  const double centered = (tq - 2.0 * e * ts) + n * e * e;
  stats[0] = mean;
  stats[1] = __fdiv_rn(1.0f, __fsqrt_rn((float)(centered / n + (double)eps)));
}

// Output of a group's float4s: normalized, affine per channel, activated.
struct GnOutput {
  const float *w, *b;
  float mean, inv, rsp;
  unsigned pbase, held;  // channels: below 2^31
  float hw, hb;
  int spatial, act;
  bool fast, quad_channel;

  // the same value in every lane, in a scalar register
  static __device__ inline float uniform(float v) {
    return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v)));
  }

  __device__ GnOutput(const float *w_, const float *b_, float mean_, float inv_, int task, int channels, int spatial_,
                      int groups, int act_)
      : w(w_), b(b_), mean(uniform(mean_)), inv(uniform(inv_)), held(~0u), hw(1.0f), hb(0.0f),
        spatial(spatial_), act(act_) {
    const int cpg = channels / groups;
    pbase = (unsigned)(task % groups) * (unsigned)cpg;
    rsp = __fdiv_rn(1.0f, (float)spatial);
    fast = cpg < (1 << 22);  // the channel within the group by small_quotient
    // spatial % 4 == 0: a quad lies in one channel, and a lane's channel changes
    // only every spatial / 4 quads, so its parameters stay in registers until then
    quad_channel = spatial % 4 == 0 && fast;
  }

  __device__ inline hb_f32x4 value(hb_f32x4 v, int idx) {
    float o[4] = {v[0], v[1], v[2], v[3]};
    if (quad_channel && (w || b)) {
      const unsigned ch = pbase + small_quotient(4u * (unsigned)idx, (unsigned)spatial, rsp);
      if (ch != held) {
        held = ch;
        hw = w ? w[ch] : 1.0f;
        hb = b ? b[ch] : 0.0f;
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float t = __fmul_rn(__fsub_rn(o[e], mean), inv);
        if (w) t = __fmul_rn(t, hw);
        if (b) t = __fadd_rn(t, hb);
        o[e] = act ? activate(t, 4) : t;
      }
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float t = __fmul_rn(__fsub_rn(o[e], mean), inv);
        if (w || b) {
          const unsigned i = 4u * (unsigned)idx + (unsigned)e;
          const unsigned ch = pbase + (fast ? small_quotient(i, (unsigned)spatial, rsp) : i / (unsigned)spatial);
          if (w) t = __fmul_rn(t, w[ch]);
          if (b) t = __fadd_rn(t, b[ch]);
        }
        o[e] = act ? activate(t, 4) : t;
      }
    }
    return hb_f32x4{o[0], o[1], o[2], o[3]};
  }
};

template <int PASS>
__global__ __launch_bounds__(kAuxThreads) void aux_group_norm_chunk(float *__restrict__ y, const float *__restrict__ x,
                                                                    const float *__restrict__ w,
                                                                    const float *__restrict__ b, double *ws, int len,
                                                                    int chunk, int chunks, int tasks, int channels,
                                                                    int spatial, int groups, float eps, int act) {
  __shared__ double red[kAuxThreads / 64];
  __shared__ float stats[2];
  constexpr int T = kAuxThreads;
  const int c = blockIdx.x, task = blockIdx.y;
  const size_t offset = (size_t)task * (size_t)len;
  const int v0 = c * (chunk / 4), v1 = min(c * chunk + chunk, len) / 4;  // the chunk's float4 range
  const float4 *xr = (const float4 *)(x + offset);
  double *sum = ws + (size_t)task * chunks, *sq = ws + (size_t)tasks * chunks + (size_t)task * chunks;
  const float shift = x[offset];
  if (PASS == 0) {
    double s = 0.0, q = 0.0;
    int i = v0 + (int)threadIdx.x;
    for (; i + (kGnUnroll - 1) * T < v1; i += kGnUnroll * T) {
      float4 v[kGnUnroll];
#pragma unroll
      for (int u = 0; u < kGnUnroll; ++u) v[u] = xr[i + u * T];
#pragma unroll
      for (int u = 0; u < kGnUnroll; ++u) shifted_add(v[u], (double)shift, s, q);
    }
    for (; i < v1; i += T) shifted_add(xr[i], (double)shift, s, q);
    s = block_sum(s, red);
    q = block_sum(q, red);
    if (threadIdx.x == 0) {
      sum[c] = s;
      sq[c] = q;
    }
    return;
  }
  if (threadIdx.x == 0) {
    double ts = 0.0, tq = 0.0;
    for (int k = 0; k < chunks; ++k) {
      ts += sum[k];
      tq += sq[k];
    }
    gn_stats(ts, tq, len, shift, eps, stats);
  }
  __syncthreads();
  GnOutput out(w, b, stats[0], stats[1], task, channels, spatial, groups, act);
  hb_f32x4 *yr = (hb_f32x4 *)(y + offset);
  const hb_f32x4 *xq = (const hb_f32x4 *)xr;
  int i = v0 + (int)threadIdx.x;
  for (; i + (kGnUnroll - 1) * T < v1; i += kGnUnroll * T) {
    hb_f32x4 v[kGnUnroll];
#pragma unroll
    for (int u = 0; u < kGnUnroll; ++u) v[u] = xq[i + u * T];
#pragma unroll
    for (int u = 0; u < kGnUnroll; ++u) __builtin_nontemporal_store(out.value(v[u], i + u * T), yr + i + u * T);
  }
  for (; i < v1; i += T) __builtin_nontemporal_store(out.value(xq[i], i), yr + i);
}

// Group norm over few long groups whose values fit on the chip: x is read
// once, each workgroup (one per CU) keeping its piece of a group in registers
// (NV float4 per thread) and LDS (NL float4 per thread) while the group's
// workgroups exchange the sums of their pieces, then writes the output from
// there.  Bound by HBM: a second read of x costs as much as the first even
// where the memory-side cache holds it (aux_group_norm_chunk at 128 channels
// of 512 x 512: 25 us for the statistics pass and 47 for the output pass, in
// either order), so 512 KB held per CU save a third of the traffic.  32 groups
// with parameters and SiLU, both passes -> this kernel, microseconds: 512 x
// 128^2 21.5 -> 18.9, 256 x 256^2 39.1 -> 30.1, 256 x 320^2 57.2 -> 43.7, 128 x
// 512^2 72.3 -> 55.3 (268 MB at 4.9 TB/s; a copy of that size reaches 5.1); x
// written by the launch before, 128 x 512^2 67.9 -> 50.5.  Rows of T float4s past
// a piece are skipped: a form holds up to twice the piece, and working them out
// unstored took it behind the two passes (256 x 33175: 29.5 us in two passes,
// 32.5 with them, 25.1 without).
//
// The exchange: parts holds one slot per (task, piece, sum) that a fill kernel
// set to kGnEmpty; every workgroup stores its two sums with device-scope
// atomics (no fence: a slot is its own flag) and waits for the others' slots.
// The wait is bounded: if a slot stays empty for spin_ticks of the 100 MHz
// clock (the other workgroup may not be resident while another kernel holds
// its CU), the workgroup computes that piece's sums from x itself, the same
// additions in the same order, so the result does not depend on it and no
// workgroup ever depends on another to end.  Workgroups of one group run on
// one XCD where the groups divide by 8 (bid % 8): each XCD then starts whole
// groups in order.
//
// Per thread the sums are added in the order of its pieces' float4s, then as
// block_sum adds them, then piece by piece in order: fixed for a shape.  The
// statistics are those of aux_group_norm_chunk.  x and y do not overlap.
constexpr int kGnThreads = 1024;
constexpr unsigned long long kGnEmpty = ~0ull;  // a NaN that no sum produces

__global__ void aux_group_norm_clear(unsigned long long *parts, int n) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) parts[i] = kGnEmpty;
}

__device__ __attribute__((unused)) inline unsigned long long gn_bits(double v) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(v);
  return b == kGnEmpty ? 0x7ff8000000000000ull : b;
}

// Sums over the workgroup, waves in order: thread 0 gets that of s, thread 1
// that of q.  All threads call it; starts with a barrier.
__device__ __attribute__((unused)) inline double gn_reduce(double s, double q, double (&red)[2][kGnThreads / 64]) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    s += __shfl_xor(s, off, 64);
    q += __shfl_xor(q, off, 64);
  }
  __syncthreads();  // red and the sums of an earlier call have been read
  if ((threadIdx.x & 63) == 0) {
    red[0][threadIdx.x >> 6] = s;
    red[1][threadIdx.x >> 6] = q;
  }
  __syncthreads();
  double total = 0.0;
  if (threadIdx.x < 2) {
#pragma unroll 1
    for (int w = 0; w < kGnThreads / 64; ++w) total += red[threadIdx.x][w];
  }
  return total;
}

template <int NV, int NL>
__global__ __launch_bounds__(kGnThreads) void aux_group_norm_resident(
    float *__restrict__ y, const float *__restrict__ x, const float *__restrict__ w, const float *__restrict__ b,
    unsigned long long *parts, int len, int piece, int pieces, int tasks, int channels, int spatial, int groups,
    float eps, int act, int spin_ticks) {
#if defined(__HIP_DEVICE_COMPILE__)  // the buffer resource type does not exist in the host pass
  constexpr int T = kGnThreads;
  __shared__ float4 held_lds[NL > 0 ? NL * T : 1];
  __shared__ double red[2][T / 64];
  __shared__ double sums[2 * kGnMaxPieces];
  __shared__ float stats[2];
  const int t = threadIdx.x;
  int task = blockIdx.x / pieces, mine = blockIdx.x % pieces;
  if (tasks % 8 == 0) {  // whole groups per XCD
    const int slot = blockIdx.x / 8;
    task = blockIdx.x % 8 + 8 * (slot / pieces);
    mine = slot % pieces;
  }
  const size_t offset = (size_t)task * (size_t)len;
  const float4 *xr = (const float4 *)(x + offset);
  const int quads = len / 4;
  const float shift = x[offset];
  const int v0 = mine * piece, v1 = min(v0 + piece, quads);  // this workgroup's float4s

  // Loads and stores through a buffer resource per row of T float4s (scalar
  // work): one offset register serves them all, and lanes past the piece read
  // zeros and store nothing.
  const int have = max(v1 - v0, 0);
  const uint32_t at = (uint32_t)t * 16u;
  auto row = [&](const void *base, int u) {
    return __builtin_amdgcn_make_buffer_rsrc((void *)((const float4 *)base + u * T), 0,
                                             (uint32_t)max(have - u * T, 0) * 16u, 0x00020000);
  };
  const void *xp = xr + v0, *yp = y + offset + 4 * (size_t)v0;
  // LDS's share straight into LDS, then the registers' (all loads in flight)
#pragma unroll
  for (int u = 0; u < NL; ++u)
    __builtin_amdgcn_raw_ptr_buffer_load_lds(row(xp, NV + u), HB_LDS_PTR(held_lds + u * T + (t & ~63)), 16, at, 0, 0,
                                             0);
  hb_f32x4 v[NV];
#pragma unroll
  for (int u = 0; u < NV; ++u)
    v[u] = __builtin_bit_cast(hb_f32x4, __builtin_amdgcn_raw_buffer_load_b128(row(xp, u), at, 0, 0));
  double s = 0.0, q = 0.0;
#pragma unroll
  for (int u = 0; u < NV; ++u) {
    if (u * T + t < have) shifted_add(make_float4(v[u][0], v[u][1], v[u][2], v[u][3]), (double)shift, s, q);
    __builtin_amdgcn_sched_barrier(0);  // one value's double arithmetic at a time: registers
  }
  if (NL > 0) wait_vmcnt<0>();  // this wave's own LDS share has landed
#pragma unroll
  for (int u = 0; u < NL; ++u)
    if ((NV + u) * T + t < have) shifted_add(held_lds[u * T + t], (double)shift, s, q);
  unsigned long long *slots = parts + (size_t)task * (size_t)pieces * 2u;
  const double own = gn_reduce(s, q, red);  // thread 0: the sum, thread 1: the squares
  if (t < 2) __hip_atomic_store(slots + 2 * mine + t, gn_bits(own), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  bool late = false;
  if (t < 2 * pieces) {
    unsigned long long bits = kGnEmpty;
    const uint64_t t0 = wall_clock64();
    while (bits == kGnEmpty) {
      bits = __hip_atomic_load(slots + t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (bits == kGnEmpty && wall_clock64() - t0 >= (uint64_t)spin_ticks) break;
      if (bits == kGnEmpty) __builtin_amdgcn_s_sleep(2);
    }
    late = bits == kGnEmpty;
    sums[t] = __longlong_as_double((long long)bits);
  }
  if (__syncthreads_or(late)) {
#pragma unroll 1
    for (int p = 0; p < pieces; ++p) {
      const bool missing = (unsigned long long)__double_as_longlong(sums[2 * p]) == kGnEmpty ||
                           (unsigned long long)__double_as_longlong(sums[2 * p + 1]) == kGnEmpty;
      if (!missing) continue;  // the same for every thread: sums changes only between the barriers below
      const int p0 = p * piece, p1 = min(p0 + piece, quads);
      double ps = 0.0, pq = 0.0;
#pragma unroll 1
      for (int i = p0 + t; i < p1; i += T) shifted_add(xr[i], (double)shift, ps, pq);
      const double total = gn_reduce(ps, pq, red);
      if (t < 2) sums[2 * p + t] = total;
      __syncthreads();
    }
  }
  if (t == 0) {
    double ts = 0.0, tq = 0.0;
    for (int p = 0; p < pieces; ++p) {
      ts += sums[2 * p];
      tq += sums[2 * p + 1];
    }
    gn_stats(ts, tq, len, shift, eps, stats);
  }
  __syncthreads();
  GnOutput out(w, b, stats[0], stats[1], task, channels, spatial, groups, act);
  const int last = quads - 1;  // lanes past the piece compute some value of the group
#pragma unroll
  for (int u = 0; u < NV; ++u) {
    if (u * T >= have) break;
    const hb_f32x4 o = out.value(v[u], min(v0 + u * T + t, last));
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(hb_u32x4, o), row(yp, u), at, 0, 2);
    __builtin_amdgcn_sched_barrier(0);
  }
#pragma unroll
  for (int u = 0; u < NL; ++u) {
    if ((NV + u) * T >= have) break;
    const float4 l = held_lds[u * T + t];
    const hb_f32x4 o = out.value(hb_f32x4{l.x, l.y, l.z, l.w}, min(v0 + (NV + u) * T + t, last));
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(hb_u32x4, o), row(yp, NV + u), at, 0, 2);
    __builtin_amdgcn_sched_barrier(0);
  }
#endif
}

// Quotients of indexes below 2^31 by a divisor fixed for the launch: with
// 2^(s-1) < d <= 2^s and mul = ceil(2^(31+s) / d), n * mul >> (31 + s) is
// n / d for every n < 2^31 (Granlund and Montgomery, 1994: mul * d exceeds
// 2^(31+s) by less than 2^s).  A 64-bit division by a kernel argument is
// about a hundred instructions.
struct IndexDivisor {
  uint32_t d, mul, shift;

  __device__ inline uint32_t quotient(uint32_t n) const { return __umulhi(2u * n, mul) >> shift; }
};

// Divisors past the largest index give 0 for every index, as they should.
IndexDivisor index_divisor(int64_t d) {
  IndexDivisor v{(uint32_t)std::min<int64_t>(std::max<int64_t>(d, 1), INT32_MAX), 0, 0};
  while (((uint64_t)1 << v.shift) < v.d) ++v.shift;
  v.mul = (uint32_t)((((uint64_t)1 << (31 + v.shift)) + v.d - 1) / v.d);
  return v;
}

// Where value i of a mode 3, 4, 10 or 12 finds its other operand: row is the
// period of w (modes 3, 4) or a row's width, batch the values of a batch.
struct ElementIndex {
  IndexDivisor row, batch;
  uint32_t stride;  // mode 12: values from one row of x to the next
  bool shared;      // mode 10: one set of parameters for all batches

  template <int MODE>
  __device__ inline size_t operand(uint32_t i) const {
    const uint32_t r = row.quotient(i), column = i - r * row.d;
    if (MODE == 12) return (size_t)r * stride + column;
    if (MODE == 10 && !shared) return (size_t)batch.quotient(i) * row.d + column;
    return column;
  }
};

// Modes 3, 4, 5, 6, 7, 10, 12: one thread per output value, grid-stride.
template <int MODE>
__global__ __launch_bounds__(kAuxThreads) void aux_elementwise(float *__restrict__ y, const float *__restrict__ x,
                                                               const float *__restrict__ w,
                                                               const float *__restrict__ b, int64_t count, int width,
                                                               ElementIndex at, int act) {
  const int64_t stride = (int64_t)gridDim.x * kAuxThreads;
  for (int64_t i = (int64_t)blockIdx.x * kAuxThreads + threadIdx.x; i < count; i += stride) {
    float v;
    if (MODE == 3) {
      v = __fadd_rn(x[i], w[at.operand<MODE>((uint32_t)i)]);
    } else if (MODE == 4) {
      v = __fmul_rn(x[i], w[at.operand<MODE>((uint32_t)i)]);
    } else if (MODE == 5 || MODE == 6 || MODE == 7) {
      v = activate(x[i], MODE == 5 ? 4 : MODE == 6 ? 1 : 2);
    } else if (MODE == 10) {
      v = __fadd_rn(__fmul_rn(x[i], w[at.operand<MODE>((uint32_t)i)]), b[i]);
    } else {  // 12
      const float *a = x + at.operand<MODE>((uint32_t)i);
      const float gate = a[act ? 0 : width], up = a[act ? width : 0];
      v = __fmul_rn(activate(gate, 5), up);
    }
    y[i] = v;
  }
}

// The same modes, a quad of consecutive values per thread with 16-byte loads
// and stores (count % 4 == 0, x and y 16-byte aligned; mode 12 also needs
// width and channels divisible by 4).  QUAD: the quad's other operand is one
// 16-byte load too (a row or period of whole quads, aligned), else value by
// value.  Bound by HBM: one quad per thread keeps the most waves in flight;
// two or four measured up to 8 % slower (4352 x 1536, mode 6: 11.1 / 12.0 / 12.5
// us).  Against 64-bit divisions for every value, us: mode 3 40.9 -> 37.8 and
// mode 10 56.3 -> 54.1 at 4352 x 6144 (5.7 and 5.9 TB/s), 12.7 -> 11.3 and
// 16.6 -> 15.7 at 4352 x 1536.
template <int MODE, bool QUAD>
__global__ __launch_bounds__(kAuxThreads) void aux_elementwise4(float *__restrict__ y, const float *__restrict__ x,
                                                                const float *__restrict__ w,
                                                                const float *__restrict__ b, uint32_t count4,
                                                                int width, ElementIndex at, int act) {
  const uint32_t q = blockIdx.x * kAuxThreads + threadIdx.x;
  if (q >= count4) return;
  constexpr bool kOperand = MODE == 3 || MODE == 4 || MODE == 10;
  const float *a = MODE == 12 ? x + at.operand<MODE>(4u * q) : x;
  const float4 xv = MODE == 12 ? *(const float4 *)(a + (act ? 0 : width)) : ((const float4 *)x)[q];
  const float4 bv = MODE == 10 ? ((const float4 *)b)[q] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  float4 wv = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  if (MODE == 12) {
    wv = *(const float4 *)(a + (act ? width : 0));
  } else if (kOperand && QUAD) {
    wv = *(const float4 *)(w + at.operand<MODE>(4u * q));
  } else if (kOperand) {
    wv = make_float4(w[at.operand<MODE>(4u * q)], w[at.operand<MODE>(4u * q + 1u)], w[at.operand<MODE>(4u * q + 2u)],
                     w[at.operand<MODE>(4u * q + 3u)]);
  }
  const float xi[4] = {xv.x, xv.y, xv.z, xv.w}, wi[4] = {wv.x, wv.y, wv.z, wv.w}, bi[4] = {bv.x, bv.y, bv.z, bv.w};
  float o[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    if (MODE == 3) o[e] = __fadd_rn(xi[e], wi[e]);
    else if (MODE == 4) o[e] = __fmul_rn(xi[e], wi[e]);
    else if (MODE == 10) o[e] = __fadd_rn(__fmul_rn(xi[e], wi[e]), bi[e]);
    else if (MODE == 12) o[e] = __fmul_rn(activate(xi[e], 5), wi[e]);
    else o[e] = activate(xi[e], MODE == 5 ? 4 : MODE == 6 ? 1 : 2);
  }
  ((float4 *)y)[q] = make_float4(o[0], o[1], o[2], o[3]);
}

// Mode 8: x[batch][width][spatial] -> y[batch][spatial][width], 32 x 32 tiles through LDS.
__global__ __launch_bounds__(kAuxThreads) void aux_transpose(float *__restrict__ y, const float *__restrict__ x,
                                                             int width, int spatial) {
  __shared__ float tile[32][33];
  const int batch = blockIdx.z, r0 = blockIdx.y * 32, c0 = blockIdx.x * 32;
  const float *xb = x + (size_t)batch * width * spatial;
  float *yb = y + (size_t)batch * width * spatial;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;  // 32 x 8
  for (int r = ty; r < 32; r += 8)
    if (r0 + r < width && c0 + tx < spatial) tile[r][tx] = xb[(size_t)(r0 + r) * spatial + c0 + tx];
  __syncthreads();
  for (int c = ty; c < 32; c += 8)
    if (c0 + c < spatial && r0 + tx < width) yb[(size_t)(c0 + c) * width + r0 + tx] = tile[tx][c];
}

// The same with 64 x 64 tiles and 16-byte loads and stores (width and spatial
// multiples of 4, x and y 16-byte aligned): four loads in flight per thread,
// rows of 256 bytes on either side.  Rows of 65 words: the four words of a
// quad and the 16 quads of a row or column fall into different banks.  us, 32
// x 32 tiles of single values -> this: 4352 x 6144 58.8 -> 42.1 (5.1 TB/s),
// 4096 x 3072 30.0 -> 21.2, 4352 x 1536 16.9 -> 11.8, 333 x 1280 4.2 either way.
__global__ __launch_bounds__(kAuxThreads) void aux_transpose4(float *__restrict__ y, const float *__restrict__ x,
                                                              int width, int spatial) {
  __shared__ float tile[64][65];
  const int batch = blockIdx.z, r0 = blockIdx.y * 64, c0 = blockIdx.x * 64;
  const float *xb = x + (size_t)batch * width * spatial;
  float *yb = y + (size_t)batch * width * spatial;
  const int t4 = 4 * (threadIdx.x & 15), row = threadIdx.x >> 4;  // 16 quads x 16 rows
  float4 v[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int r = min(r0 + row + 16 * u, width - 1), c = min(c0 + t4, spatial - 4);
    v[u] = *(const float4 *)(xb + (size_t)r * spatial + c);
  }
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    float *d = &tile[row + 16 * u][t4];
    d[0] = v[u].x;
    d[1] = v[u].y;
    d[2] = v[u].z;
    d[3] = v[u].w;
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int c = row + 16 * u;
    if (c0 + c < spatial && r0 + t4 < width)
      *(float4 *)(yb + (size_t)(c0 + c) * width + r0 + t4) =
          make_float4(tile[t4][c], tile[t4 + 1][c], tile[t4 + 2][c], tile[t4 + 3][c]);
  }
}

// Mode 11: one workgroup per (batch, token); threads over heads x pairs.
__global__ __launch_bounds__(kAuxThreads) void aux_rope(float *__restrict__ y, const float *__restrict__ x,
                                                        const float *__restrict__ pe, int dim, int heads,
                                                        int tokens, int groups) {
  const int task = blockIdx.x;
  const int token = task % tokens, batch = task / tokens;
  const float *m_base = pe + ((size_t)(groups == 1 ? 0 : batch) * tokens + token) * (size_t)dim * 2;
  const int pairs = dim / 2;
  for (int t = threadIdx.x; t < heads * pairs; t += kAuxThreads) {
    const int head = t / pairs, p = t % pairs;
    const float *m = m_base + 4 * p;
    const float *xs = x + (((size_t)batch * tokens + token) * heads + head) * dim + 2 * p;
    float *ys = y + (((size_t)batch * heads + head) * tokens + token) * dim + 2 * p;
    const float x0 = xs[0], x1 = xs[1];
    ys[0] = __fadd_rn(__fmul_rn(x0, m[0]), __fmul_rn(x1, m[1]));
    ys[1] = __fadd_rn(__fmul_rn(x1, m[3]), __fmul_rn(x0, m[2]));
  }
}

// The same, two pairs (16 bytes) per thread over all quads of x in order (dim
// % 4 == 0, all operands 16-byte aligned, below 2^31 values): full waves
// whatever the number of heads.  us, a workgroup per token -> this: 4352 x 6144
// 46.7 -> 38.5 (5.6 TB/s), 4096 x 3072 22.1 -> 19.9, 4352 x 1536 13.1 -> 11.8.
__global__ __launch_bounds__(kAuxThreads) void aux_rope4(float *__restrict__ y, const float *__restrict__ x,
                                                         const float *__restrict__ pe, uint32_t count4, int heads,
                                                         int tokens, int groups, IndexDivisor by_dim4,
                                                         IndexDivisor by_heads, IndexDivisor by_tokens) {
  const uint32_t q = blockIdx.x * kAuxThreads + threadIdx.x, dim4 = by_dim4.d;
  if (q >= count4) return;
  const uint32_t row = by_dim4.quotient(q), p = q - row * dim4;  // (batch, token, head), quad
  const uint32_t task = by_heads.quotient(row), head = row - task * (uint32_t)heads;
  const uint32_t batch = by_tokens.quotient(task), token = task - batch * (uint32_t)tokens;
  const float4 *m = (const float4 *)pe + ((size_t)(groups == 1 ? token : task) * dim4 + p) * 2;
  const float4 v = ((const float4 *)x)[q], a = m[0], c = m[1];
  ((float4 *)y)[(((size_t)batch * heads + head) * tokens + token) * dim4 + p] =
      make_float4(__fadd_rn(__fmul_rn(v.x, a.x), __fmul_rn(v.y, a.y)),
                  __fadd_rn(__fmul_rn(v.y, a.w), __fmul_rn(v.x, a.z)),
                  __fadd_rn(__fmul_rn(v.z, c.x), __fmul_rn(v.w, c.y)),
                  __fadd_rn(__fmul_rn(v.w, c.w), __fmul_rn(v.z, c.z)));
}

// Mode 13: output row r = [attention row r (groups values) | SiLU(gate) * up (width values)].
__global__ __launch_bounds__(kAuxThreads) void aux_swiglu_concat(float *__restrict__ y, const float *__restrict__ x,
                                                                 const float *__restrict__ attn, int width,
                                                                 int groups, int channels, int act) {
  const size_t r = blockIdx.x;
  float *dst = y + r * (size_t)(width + groups);
  const float *a = attn + r * (size_t)groups;
  for (int i = threadIdx.x; i < groups; i += kAuxThreads) dst[i] = a[i];
  const float *xr = x + r * (size_t)channels;
  for (int i = threadIdx.x; i < width; i += kAuxThreads) {
    const float gate = xr[i + (act ? 0 : width)], up = xr[i + (act ? width : 0)];
    dst[groups + i] = __fmul_rn(activate(gate, 5), up);
  }
}

bool aligned16(const void *p) { return ((uintptr_t)p & 15u) == 0; }

// Register-resident tasks when they fit (256 threads up to 8192 values, 1024
// threads up to 65536), else the three-pass kernel; few long tasks (group
// norm) take 1024-thread workgroups.
template <int MODE>
void launch_norm(float *y, const float *x, const float *w, const float *b, int tasks, int len, int width,
                 int channels, int spatial, int groups, int other_count, float eps, int act, bool vec,
                 hipStream_t st) {
  const dim3 grid(tasks);
  const int nv4 = len / 4;
  // Rows of 513-2048 values: two waves per row, where the 256-thread form
  // leaves a quarter to a half of its lanes idle (4096 rows: LayerNorm +
  // modulation 10.9 -> 9.6 us at 1536 values and 13.2 -> 11.8 at 2048,
  // RMSNorm 10.0 -> 9.3 and 13.1 -> 11.8; from 3072 values the 256-thread
  // form is as fast or faster).
  if (vec && nv4 > 128 && nv4 <= 128 * 4) {
    if (nv4 <= 128 * 2)
      hipLaunchKernelGGL((aux_norm_reg<MODE, 2, 128>), grid, dim3(128), 0, st, y, x, w, b, len, width, channels,
                         spatial, groups, other_count, eps, act);
    else if (nv4 <= 128 * 3)
      hipLaunchKernelGGL((aux_norm_reg<MODE, 3, 128>), grid, dim3(128), 0, st, y, x, w, b, len, width, channels,
                         spatial, groups, other_count, eps, act);
    else
      hipLaunchKernelGGL((aux_norm_reg<MODE, 4, 128>), grid, dim3(128), 0, st, y, x, w, b, len, width, channels,
                         spatial, groups, other_count, eps, act);
    return;
  }
  if (vec && nv4 <= 256 * 1) {
    hipLaunchKernelGGL((aux_norm_reg<MODE, 1, 256>), grid, dim3(256), 0, st, y, x, w, b, len, width, channels,
                       spatial, groups, other_count, eps, act);
  } else if (vec && nv4 <= 256 * 2) {
    hipLaunchKernelGGL((aux_norm_reg<MODE, 2, 256>), grid, dim3(256), 0, st, y, x, w, b, len, width, channels,
                       spatial, groups, other_count, eps, act);
  } else if (vec && nv4 <= 256 * 4) {
    hipLaunchKernelGGL((aux_norm_reg<MODE, 4, 256>), grid, dim3(256), 0, st, y, x, w, b, len, width, channels,
                       spatial, groups, other_count, eps, act);
  } else if (vec && nv4 <= 256 * 8) {
    hipLaunchKernelGGL((aux_norm_reg<MODE, 8, 256>), grid, dim3(256), 0, st, y, x, w, b, len, width, channels,
                       spatial, groups, other_count, eps, act);
  } else if (vec && nv4 <= 1024 * 16) {
    hipLaunchKernelGGL((aux_norm_reg<MODE, 16, 1024>), grid, dim3(1024), 0, st, y, x, w, b, len, width, channels,
                       spatial, groups, other_count, eps, act);
  } else if (tasks < 1024) {
    hipLaunchKernelGGL((aux_norm<MODE, 1024>), grid, dim3(1024), 0, st, y, x, w, b, len, width, channels, spatial,
                       groups, other_count, eps, act);
  } else {
    hipLaunchKernelGGL((aux_norm<MODE, 256>), grid, dim3(256), 0, st, y, x, w, b, len, width, channels, spatial,
                       groups, other_count, eps, act);
  }
}

// Chunked group-norm plan: used when the groups alone would leave most CUs
// idle and the values divide into float4 quads; 0 chunks means "not chunked".
struct GroupPlan {
  int chunks, chunk;
};

GroupPlan group_plan(int tasks, int len) {
  GroupPlan p{0, 0};
  if (tasks >= 512 || len % 4 || len < 8192) return p;
  int chunks = (1024 + tasks - 1) / tasks;  // aim for about 1024 workgroups
  if (chunks > len / 4096) chunks = len / 4096;
  if (chunks < 2) return p;
  int chunk = (len + chunks - 1) / chunks;
  chunk = (chunk + 3) / 4 * 4;
  p.chunks = (len + chunk - 1) / chunk;
  p.chunk = chunk;
  return p;
}

// The resident form (aux_group_norm_resident): pieces per group so that every
// group's run at once, one workgroup per CU, and the float4s per thread of a
// piece; 0 pieces where the values do not fit.
struct ResidentPlan {
  int pieces, piece, per_thread;
};
// Below 8 M values the two passes are as fast: the second read comes from the
// XCDs' own L2s, and the exchange costs about 3 us (320 x 128^2, 5.2 M values:
// 14.3 us in both forms; 512 x 128^2, 8.4 M: 21.5 in two passes, 18.9 here).
constexpr int64_t kGnResidentMin = 8 << 20;
constexpr int kGnHeld = 32;  // float4s per thread that registers and LDS hold

ResidentPlan resident_plan(int tasks, int len, int chunks) {
  ResidentPlan p{0, 0, 0};
  int pieces = std::min(std::min(device_cus() / tasks, kGnMaxPieces), chunks);
  if (pieces < 2 || (int64_t)tasks * len < kGnResidentMin) return p;
  const int quads = len / 4, piece = (quads + pieces - 1) / pieces;
  if (piece > kGnHeld * kGnThreads) return p;
  p.pieces = (quads + piece - 1) / piece;
  p.piece = piece;
  p.per_thread = (piece + kGnThreads - 1) / kGnThreads;
  return p;
}

// How long a workgroup of the resident form waits for another's sums before
// it computes them itself, in 100 MHz ticks (hb_group_norm_spin): 100 us, twice
// the longest launch, so that a call whose workgroups find no CU (another
// stream's kernel holds it, or a CU mask) is not held up for much longer than
// two passes take.  Beside 30 products of all CUs on another stream waits of 10,
// 100 and 2000 us take the same time, 100-119 us a call (two passes 205).
std::atomic<int> g_gn_spin{10000};

template <int NV, int NL>
void launch_resident(const ResidentPlan &p, float *y, const float *x, const float *w, const float *b, void *ws, int len,
                     int tasks, int channels, int spatial, int groups, float eps, int act, hipStream_t st) {
  hipLaunchKernelGGL((aux_group_norm_resident<NV, NL>), dim3(tasks * p.pieces), dim3(kGnThreads), 0, st, y, x, w, b,
                     (unsigned long long *)ws, len, p.piece, p.pieces, tasks, channels, spatial, groups, eps, act,
                     g_gn_spin.load(std::memory_order_relaxed));
}

int elementwise_grid(int64_t count) {
  const int64_t blocks = (count + kAuxThreads - 1) / kAuxThreads;
  return (int)(blocks < 65536 ? blocks : 65536);
}

template <int MODE>
void launch_elementwise(float *y, const float *x, const float *w, const float *b, int count, int width, int channels,
                        int spatial, int other_count, int act, hipStream_t st) {
  constexpr bool kPeriod = MODE == 3 || MODE == 4;
  const ElementIndex at{index_divisor(kPeriod ? other_count : width), index_divisor((int64_t)width * spatial),
                        (uint32_t)channels, other_count == width};
  bool vec = count % 4 == 0 && aligned16(x) && aligned16(y) && (MODE != 10 || aligned16(b));
  if (MODE == 12) vec = vec && width % 4 == 0 && channels % 4 == 0;
  if (vec) {
    const int count4 = count / 4;
    const dim3 grid((count4 + kAuxThreads - 1) / kAuxThreads);
    const bool quad = kPeriod ? other_count % 4 == 0 && aligned16(w) : MODE != 10 || (width % 4 == 0 && aligned16(w));
    if (quad)
      hipLaunchKernelGGL((aux_elementwise4<MODE, true>), grid, dim3(kAuxThreads), 0, st, y, x, w, b, (uint32_t)count4,
                         width, at, act);
    else
      hipLaunchKernelGGL((aux_elementwise4<MODE, false>), grid, dim3(kAuxThreads), 0, st, y, x, w, b,
                         (uint32_t)count4, width, at, act);
  } else {
    hipLaunchKernelGGL(aux_elementwise<MODE>, dim3(elementwise_grid(count)), dim3(kAuxThreads), 0, st, y, x, w, b,
                       (int64_t)count, width, at, act);
  }
}

}  // namespace

extern "C" int hb_group_norm_spin(int ticks) {
  if (ticks < 0) return hb_invalid("hb_group_norm_spin ticks");
  return g_gn_spin.exchange(ticks, std::memory_order_relaxed);
}

extern "C" size_t hb_model_aux_workspace_bytes(int mode, int channels, int spatial, int groups, int batch) {
  if (mode != 2 || groups <= 0 || channels <= 0 || spatial <= 0 || batch <= 0 || channels % groups) return 0;
  const int64_t len64 = (int64_t)spatial * (channels / groups), tasks64 = (int64_t)groups * batch;
  if (len64 > INT32_MAX || tasks64 > INT32_MAX) return 0;
  const GroupPlan p = group_plan((int)tasks64, (int)len64);
  return p.chunks ? (size_t)tasks64 * (size_t)p.chunks * 2u * sizeof(double) : 0;
}

extern "C" int hb_model_aux_ws(float *d_y, const float *d_x, const float *d_w, const float *d_b, int mode, int count,
                               int width, int channels, int spatial, int groups, int batch, int other_count,
                               int activation, float eps, void *d_workspace, size_t workspace_bytes, hb_stream s) {
  if (!d_y || !d_x) return hb_invalid("hb_model_aux null pointer");
  if (count <= 0 || width <= 0 || channels <= 0 || spatial <= 0 || batch <= 0)
    return hb_invalid("hb_model_aux shape");
  hipStream_t st = hb_resolve_stream(s);
  const dim3 block(kAuxThreads);
  switch (mode) {
    case 0:
    case 1:
    case 9: {
      if (mode == 9 && (!d_w || !d_b)) return hb_invalid("hb_model_aux mode 9 parameters");
      const int rows = count / width;
      if (rows < 1) return hb_invalid("hb_model_aux rows");
      const bool vec = width % 4 == 0 && aligned16(d_x) && aligned16(d_y) && aligned16(d_w) && aligned16(d_b);
      if (mode == 0)
        launch_norm<0>(d_y, d_x, d_w, d_b, rows, width, width, channels, spatial, 1, other_count, eps, activation,
                       vec, st);
      else if (mode == 1)
        launch_norm<1>(d_y, d_x, d_w, d_b, rows, width, width, channels, spatial, 1, other_count, eps, activation,
                       vec, st);
      else
        launch_norm<9>(d_y, d_x, d_w, d_b, rows, width, width, channels, spatial, 1, other_count, eps, activation,
                       vec, st);
      break;
    }
    case 2: {
      if (groups <= 0 || channels % groups) return hb_invalid("hb_model_aux groups");
      if ((int64_t)batch * channels * spatial > count) return hb_invalid("hb_model_aux group norm extent");
      const int len = spatial * (channels / groups);
      const bool vec = len % 4 == 0 && aligned16(d_x) && aligned16(d_y);
      const GroupPlan gp = group_plan(groups * batch, len);
      const size_t need = hb_model_aux_workspace_bytes(mode, channels, spatial, groups, batch);
      if (vec && gp.chunks && d_workspace && workspace_bytes >= need && ((uintptr_t)d_workspace & 7u) == 0) {
        const dim3 grid(gp.chunks, groups * batch);
        double *ws = (double *)d_workspace;
        const int tasks = groups * batch;
        const ResidentPlan rp = resident_plan(tasks, len, gp.chunks);
        const size_t bytes = (size_t)tasks * (size_t)len * 4u;
        const bool apart = (uintptr_t)d_x + bytes <= (uintptr_t)d_y || (uintptr_t)d_y + bytes <= (uintptr_t)d_x;
        if (rp.pieces && apart) {
          const int slots = 2 * tasks * rp.pieces;
          hipLaunchKernelGGL(aux_group_norm_clear, dim3((slots + 255) / 256), dim3(256), 0, st,
                             (unsigned long long *)d_workspace, slots);
          if (int rc = hb_check_launch("aux_group_norm_clear")) return rc;
          // The fewest registers and the least LDS that hold the piece: in
          // the largest form 12 float4s take 26.3 us instead of 24.3, 20 take
          // 38.0 instead of 36.5, 26 the same (256 channels).
          if (rp.per_thread <= 8)
            launch_resident<8, 0>(rp, d_y, d_x, d_w, d_b, ws, len, tasks, channels, spatial, groups, eps, activation, st);
          else if (rp.per_thread <= 16)
            launch_resident<16, 0>(rp, d_y, d_x, d_w, d_b, ws, len, tasks, channels, spatial, groups, eps, activation, st);
          else if (rp.per_thread <= 26)
            launch_resident<20, 6>(rp, d_y, d_x, d_w, d_b, ws, len, tasks, channels, spatial, groups, eps, activation, st);
          else
            launch_resident<23, 9>(rp, d_y, d_x, d_w, d_b, ws, len, tasks, channels, spatial, groups, eps, activation, st);
          break;
        }
        hipLaunchKernelGGL(aux_group_norm_chunk<0>, grid, block, 0, st, d_y, d_x, d_w, d_b, ws, len, gp.chunk,
                           gp.chunks, groups * batch, channels, spatial, groups, eps, activation);
        hipLaunchKernelGGL(aux_group_norm_chunk<1>, grid, block, 0, st, d_y, d_x, d_w, d_b, ws, len, gp.chunk,
                           gp.chunks, groups * batch, channels, spatial, groups, eps, activation);
        break;
      }
      launch_norm<2>(d_y, d_x, d_w, d_b, groups * batch, len, width, channels, spatial, groups, other_count, eps,
                     activation, vec, st);
      break;
    }
    case 3:
    case 4:
      if (!d_w || other_count <= 0) return hb_invalid("hb_model_aux broadcast operand");
      if (mode == 3)
        launch_elementwise<3>(d_y, d_x, d_w, d_b, count, width, channels, spatial, other_count, activation, st);
      else
        launch_elementwise<4>(d_y, d_x, d_w, d_b, count, width, channels, spatial, other_count, activation, st);
      break;
    case 5:
      launch_elementwise<5>(d_y, d_x, d_w, d_b, count, width, channels, spatial, other_count, activation, st);
      break;
    case 6:
      launch_elementwise<6>(d_y, d_x, d_w, d_b, count, width, channels, spatial, other_count, activation, st);
      break;
    case 7:
      launch_elementwise<7>(d_y, d_x, d_w, d_b, count, width, channels, spatial, other_count, activation, st);
      break;
    case 8: {
      if ((int64_t)width * spatial * batch != count) return hb_invalid("hb_model_aux transpose shape");
      if (width % 4 == 0 && spatial % 4 == 0 && aligned16(d_x) && aligned16(d_y)) {
        const dim3 grid4((spatial + 63) / 64, (width + 63) / 64, batch);
        hipLaunchKernelGGL(aux_transpose4, grid4, block, 0, st, d_y, d_x, width, spatial);
        break;
      }
      const dim3 grid((spatial + 31) / 32, (width + 31) / 32, batch);
      hipLaunchKernelGGL(aux_transpose, grid, block, 0, st, d_y, d_x, width, spatial);
      break;
    }
    case 10:
      if (!d_w || !d_b) return hb_invalid("hb_model_aux mode 10 parameters");
      launch_elementwise<10>(d_y, d_x, d_w, d_b, count, width, channels, spatial, other_count, activation, st);
      break;
    case 11: {
      if (!d_w || width % 2 || (groups != 1 && groups != batch)) return hb_invalid("hb_model_aux rope");
      const int64_t values = (int64_t)spatial * batch * channels * width;
      if (width % 4 == 0 && aligned16(d_x) && aligned16(d_y) && aligned16(d_w) && values <= INT32_MAX) {
        const int64_t count4 = values / 4;
        const IndexDivisor dim4 = index_divisor(width / 4), heads = index_divisor(channels),
                           tokens = index_divisor(spatial);
        hipLaunchKernelGGL(aux_rope4, dim3((uint32_t)((count4 + kAuxThreads - 1) / kAuxThreads)), block, 0, st, d_y, d_x,
                           d_w, (uint32_t)count4, channels, spatial, groups, dim4, heads, tokens);
        break;
      }
      hipLaunchKernelGGL(aux_rope, dim3(spatial * batch), block, 0, st, d_y, d_x, d_w, width, channels, spatial,
                         groups);
      break;
    }
    case 12:
      if (channels < 2 * width) return hb_invalid("hb_model_aux gated width");
      launch_elementwise<12>(d_y, d_x, d_w, d_b, count, width, channels, spatial, other_count, activation, st);
      break;
    case 13:
      if (!d_w || groups <= 0 || channels < 2 * width) return hb_invalid("hb_model_aux concat");
      hipLaunchKernelGGL(aux_swiglu_concat, dim3(spatial * batch), block, 0, st, d_y, d_x, d_w, width, groups,
                         channels, activation);
      break;
    default:
      return hb_invalid("hb_model_aux mode");
  }
  return hb_check_launch("hb_model_aux");
}

extern "C" int hb_model_aux(float *d_y, const float *d_x, const float *d_w, const float *d_b, int mode, int count,
                            int width, int channels, int spatial, int groups, int batch, int other_count,
                            int activation, float eps, hb_stream s) {
  return hb_model_aux_ws(d_y, d_x, d_w, d_b, mode, count, width, channels, spatial, groups, batch, other_count,
                         activation, eps, nullptr, 0, s);
}
