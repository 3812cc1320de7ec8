// Vectorised forms of the row kernels for the common case (widths that are
// multiples of 4, no pending bias in the norm, full-head rotary): same formulas and
// the same order of additions as elementwise.hip, 16 bytes per load where the
// general kernels load one element. The entry points in elementwise.hip try these
// first and fall back to the general kernels.
#include "pyre_common.h"
#include "pyre_vec.h"
#include "pyre_vec4.h"

using namespace pyre;

namespace {

// ---------------------------------------------------------------------------
// add + RMSNorm, one block per row, the row kept in registers between the passes.
// ---------------------------------------------------------------------------
constexpr int kNormMaxVec = 8;  // float4 per thread of 256

// THREADS = 256 keeps up to 8192 elements of a row in registers and suits many rows;
// THREADS = 1024 gives a short row one float4 per thread, so that all loads of a
// decode step's few rows are in flight at once.
//
// A step of few rows is a chain of trips through memory with next to no bytes: whatever is asked for is asked for at
// once, the gain among it, the reduction is exchanges between lanes and one trip through LDS, and what the first loads need
// comes with the launch (arguments in that order). In a graph, us at 10 parts: 1,536 elements 3.1 -> 2.7 at one row, 4.65 -> 3.3 at 190;
// 3,584 elements 3.8 -> 3.5 and 7.7 -> 4.9. Rows get 1024 threads up to one row a compute unit (190 rows with
// 256 threads 4.1 and 6.8; at 400 rows the two are alike). STREAM has the waves that hide the gain. FOUR: it asks for four parts at a
// time, for three parts and more of so few rows that a trip through memory for each part is not hidden: one at a time and four, us at 566
// rows and 10 parts 11.6 and 8.3, 26.2 and 19.8. Two parts gain nothing by it (566 rows of 1,536 elements 4.0 and 4.2, of 4,096 8.45 and 8.7),
// and where rows and parts are many it takes the caches' order from the reads: 2,048 rows of 2,048 in 10 parts 33.8 and
// 39.3, 1,300 of 4,096 46.7 and 49.5. The line (rows times parts below 12,000) is where the two are alike over seven widths.
//
// The sum of squares is added up in an order that the row's width alone fixes, whichever
// variant runs: a row wider than 1024 elements is summed as 1024 threads would (thread t
// adds its pieces t, t + 1024, ... in ascending order; every 64 consecutive threads are
// reduced by the butterfly of wave_sum; the 16 results are added in ascending order).
// The 256-thread variant then plays VIRT = 4 of those threads per thread: t = thread +
// 256 j. A position's result therefore does not depend on how many rows share the step.
template <typename TD, typename TG, typename TO, int THREADS, int VIRT, bool STREAM, bool FOUR = false>
__global__ __launch_bounds__(THREADS) void add_rmsnorm_vec_kernel(
    float* __restrict__ resid, const TD* __restrict__ delta, int n_partials, int hidden, size_t partial_stride, const int* __restrict__ rows,
    const TG* __restrict__ gain, TO* __restrict__ out, float eps, const float* __restrict__ bias) {
  __shared__ __attribute__((aligned(16))) float scratch[16];
  const int r_out = blockIdx.x, r_in = rows ? rows[r_out] : r_out;
  const size_t in_off = static_cast<size_t>(r_in) * hidden;
  const int nvec = hidden / 4;
  constexpr int ITEMS = kNormMaxVec * 256 / THREADS;
  float4 v[ITEMS], gn[ITEMS];
  float ss[VIRT];
#pragma unroll
  for (int j = 0; j < VIRT; ++j) ss[j] = 0.f;
#pragma unroll
  for (int i = 0; i < ITEMS; ++i) {
    const int c = threadIdx.x + i * THREADS;
    if (c >= nvec) break;
    float4 x = STREAM ? Stream4<float>::load(resid + in_off + 4 * c) : Vec4<float>::load(resid + in_off + 4 * c);
    if (delta) {
      float4 d;
      if (STREAM) {  // the same sums in the same order
        d = FOUR ? sum_many_partials4_stream(delta + in_off + 4 * c, partial_stride, n_partials)
                 : sum_partials4_stream(delta + in_off + 4 * c, partial_stride, n_partials);
      } else {
        PendingSum4<TD> pending;
        pending.ask(delta + in_off + 4 * c, partial_stride, n_partials);
        gn[i] = Vec4<TG>::load(gain + 4 * c);
        d = pending.sum(delta + in_off + 4 * c, partial_stride, n_partials);
      }
      if (bias) d = add4(d, Vec4<float>::load(bias + 4 * c));  // all partial sums, then the bias
      x = add4(x, d);
      if (!rows) {
        if (STREAM) Stream4<float>::store(resid + in_off + 4 * c, x);
        else Vec4<float>::store(resid + in_off + 4 * c, x);
      }
    } else if (!STREAM) {
      gn[i] = Vec4<TG>::load(gain + 4 * c);
    }
    v[i] = x;
    // explicit fused multiply-adds: the same roundings in every variant of the kernel
    ss[i % VIRT] = fmaf(x.w, x.w, fmaf(x.z, x.z, fmaf(x.y, x.y, fmaf(x.x, x.x, ss[i % VIRT]))));
  }
  // the waves of the threads this thread stands for are wave + (THREADS / 64) j
#pragma unroll
  for (int j = 0; j < VIRT; ++j) {
    const float s = full_wave_sum(ss[j]);
    if ((threadIdx.x & (kWave - 1)) == 0) scratch[threadIdx.x / kWave + (THREADS / kWave) * j] = s;
  }
  __syncthreads();
  const float total = waves_sum<VIRT * THREADS / kWave>(scratch);
  const float inv = rsqrtf(total / static_cast<float>(hidden) + eps);
  const size_t out_off = static_cast<size_t>(r_out) * hidden;
#pragma unroll
  for (int i = 0; i < ITEMS; ++i) {
    const int c = threadIdx.x + i * THREADS;
    if (c >= nvec) break;
    if (STREAM) gn[i] = Vec4<TG>::load(gain + 4 * c);
    const float4 x = v[i], g = gn[i];
    const float4 y{x.x * inv * g.x, x.y * inv * g.y, x.z * inv * g.z, x.w * inv * g.w};
    if (STREAM) Stream4<TO>::store(out + out_off + 4 * c, y);
    else Vec4<TO>::store(out + out_off + 4 * c, y);
  }
}

// ---------------------------------------------------------------------------
// rotary + cache write, four pairs per item; grid (tokens, ceil(items / 256)).
// ---------------------------------------------------------------------------
// (The arguments that the first loads need come first: those are in registers when the kernel starts.)
// How the product's parts are read; they are always added in one order. kTogether: both values' parts and all else is asked for before
// anything is waited for. That takes 124 registers (kEach 62), so it is for as many blocks as the compute units then hold, four each (two
// parts, us with kEach and kTogether: 28 query and 4 key/value heads, three blocks a row, 4.6 and 4.1 at 256 rows, 5.3 and 6.0 at 400; 12 and 2,
// two blocks, 4.9 and 4.7 at 400; 40 and 8, four blocks, 7.6 and 8.5 at 400). kEach: one value after the other. From 512 rows on past the caches,
// one part at a time (kStream) or four (kStreamFour), for three parts and more of less than 1,200 rows (12 and 2 heads, us: 7 parts of 700
// rows 13.5 and 9.9, 2 parts of 566 rows 4.9 and 5.4, 7 parts of 28 and 4 heads at 2,048 rows 54.9 and 57.0).
enum Read { kTogether, kEach, kStream, kStreamFour };
template <typename TI, typename TC, Read READ>
__global__ __launch_bounds__(256) void rope_kv_write_vec_kernel(
    const TI* __restrict__ qkv, size_t partial_stride, int n_partials, int nq, int nkv, int hd, const void* __restrict__ bias,
    const int* __restrict__ positions, const int* __restrict__ slots, const float* __restrict__ cos_t, const float* __restrict__ sin_t,
    int bias_dt, int page_size, TC* __restrict__ q_out, TC* __restrict__ k_cache, TC* __restrict__ v_cache) {
  const int n = blockIdx.x;
  const int half = hd / 2, hv = half / 4;            // vec4 pairs per head
  const int n_rot = (nq + nkv) * hv, n_items = n_rot + nkv * (hd / 4);
  const int it = blockIdx.y * 256 + threadIdx.x;
  if (it >= (slots ? n_items : nq * hv)) return;  // (no slots: the cache is another layer's)
  const int width = (nq + 2 * nkv) * hd;
  const size_t in_row = static_cast<size_t>(n) * width;
  const int slot = slots ? slots[n] : -1;

  // Whatever is asked for is asked for before anything is waited for (a step of few tokens is all waiting): the product's parts, the
  // bias, the tables' row.
  struct Value {
    PendingSum4<TI> parts;
    uint4 bias;
  };
  auto ask4 = [&](Value& v, int col) {
    const TI* const src = qkv + in_row + col;
    if (READ == kStreamFour) v.parts.v[0] = sum_many_partials4_stream(src, partial_stride, n_partials);
    else if (READ == kStream) v.parts.v[0] = sum_partials4_stream(src, partial_stride, n_partials);
    else if (READ == kEach) v.parts.v[0] = sum_partials4(src, partial_stride, n_partials);
    else v.parts.ask(src, partial_stride, n_partials);
    if (bias) {  // col is a multiple of 4: one load of four, as they are
      if (bias_dt == kF32) {
        v.bias = *reinterpret_cast<const uint4*>(static_cast<const float*>(bias) + col);
      } else {
        const uint2 u = *reinterpret_cast<const uint2*>(static_cast<const bf16*>(bias) + col);
        v.bias.x = u.x, v.bias.y = u.y;
      }
    }
  };
  auto value4 = [&](const Value& v, int col) {
    const float4 s = READ != kTogether ? v.parts.v[0] : v.parts.sum(qkv + in_row + col, partial_stride, n_partials);
    if (!bias) return s;
    const uint4 u = v.bias;
    return add4(s, bias_dt == kF32 ? float4{__uint_as_float(u.x), __uint_as_float(u.y), __uint_as_float(u.z), __uint_as_float(u.w)}
                                   : float4{__uint_as_float(u.x << 16), __uint_as_float(u.x & 0xffff0000u), __uint_as_float(u.y << 16),
                                            __uint_as_float(u.y & 0xffff0000u)});
  };

  int page = 0, off = 0;
  auto place = [&] {
    if (slot >= 0) page = slot / page_size, off = slot % page_size;
  };

  if (it < n_rot) {
    const int head = it / hv, j = 4 * (it % hv);
    const int base = head * hd;
    Value p1, p2;
    ask4(p1, base + j);
    ask4(p2, base + j + half);
    const size_t t = static_cast<size_t>(positions[n]) * half + j;
    const float4 c = Vec4<float>::load(cos_t + t), s = Vec4<float>::load(sin_t + t);
    if (READ != kTogether) place();
    const float4 x1 = value4(p1, base + j), x2 = value4(p2, base + j + half);
    if (READ == kTogether) place();
    if (head >= nq && slot < 0) return;
    float4 a, b;
    rotate_pair(x1.x, x2.x, c.x, s.x, a.x, b.x);
    rotate_pair(x1.y, x2.y, c.y, s.y, a.y, b.y);
    rotate_pair(x1.z, x2.z, c.z, s.z, a.z, b.z);
    rotate_pair(x1.w, x2.w, c.w, s.w, a.w, b.w);
    TC* dst = head < nq ? q_out + static_cast<size_t>(n) * nq * hd + base
                        : k_cache + ((static_cast<size_t>(page) * nkv + (head - nq)) * page_size + off) * hd;
    Vec4<TC>::store(dst + j, a);
    Vec4<TC>::store(dst + j + half, b);
  } else {
    const int e = 4 * (it - n_rot);
    const int kvh = e / hd, d = e % hd;
    Value pv;
    ask4(pv, (nq + nkv) * hd + e);
    if (READ != kTogether) place();
    const float4 v = value4(pv, (nq + nkv) * hd + e);
    if (READ == kTogether) place();
    if (slot < 0) return;
    TC* row = v_cache + ((static_cast<size_t>(page) * nkv + kvh) * hd + d) * page_size;
    row[off] = from_float<TC>(v.x);
    row[page_size + off] = from_float<TC>(v.y);
    row[2 * static_cast<size_t>(page_size) + off] = from_float<TC>(v.z);
    row[3 * static_cast<size_t>(page_size) + off] = from_float<TC>(v.w);
    // the step's last token of a page leaves nothing of the page's previous owner behind it
    if (ends_its_page_run(slots, n, gridDim.x, slot, page_size)) {
#pragma unroll
      for (int r = 0; r < 4; ++r) zero_tail(row + r * static_cast<size_t>(page_size), off + 1, page_size);
    }
  }
}

// ---------------------------------------------------------------------------
// SiLU-gate, four features per thread; eight, in 16-byte loads that go past the caches,
// for bfloat16 without partial sums (a prompt portion's gate/up product, read once).
// ---------------------------------------------------------------------------
__device__ inline float silu_gate(float g, float u) { return g / (1.f + expf(-g)) * u; }
// For results that are rounded to bfloat16: the hardware's exponential and reciprocal (errors of a
// few units in the last place of float32), as in the epilogue of the decode step's gate/up product.
__device__ inline float silu_gate_fast(float g, float u) { return g * __builtin_amdgcn_rcpf(1.f + __expf(-g)) * u; }

template <typename TI, typename TO>
__global__ __launch_bounds__(256) void silu_mul_vec_kernel(const TI* __restrict__ gu, int n_partials,
                                                           size_t partial_stride, TO* __restrict__ out,
                                                           size_t total4, int inter) {
  const size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= total4) return;
  const int per_row = inter / 4;
  const size_t n = i / per_row, c = 4 * (i % per_row);
  const size_t gi = n * 2 * inter + c, ui = gi + inter;
  float4 g = Vec4<TI>::load(gu + gi), u = Vec4<TI>::load(gu + ui);
  for (int p = 1; p < n_partials; ++p) {
    g = add4(g, Vec4<TI>::load(gu + p * partial_stride + gi));
    u = add4(u, Vec4<TI>::load(gu + p * partial_stride + ui));
  }
  Vec4<TO>::store(out + n * inter + c, float4{silu_gate(g.x, u.x), silu_gate(g.y, u.y), silu_gate(g.z, u.z),
                                              silu_gate(g.w, u.w)});
}

__global__ __launch_bounds__(256) void silu_mul_stream_kernel(const bf16* __restrict__ gu, bf16* __restrict__ out,
                                                              size_t total8, int inter) {
  typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
  const size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= total8) return;
  const int per_row = inter / 8;
  const size_t n = i / per_row, c = 8 * (i % per_row);
  const bf16* gp = gu + n * 2 * inter + c;
  const u32x4 g = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(gp));
  const u32x4 u = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(gp + inter));
  u32x4 y;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const float lo = silu_gate_fast(__uint_as_float(g[j] << 16), __uint_as_float(u[j] << 16));
    const float hi = silu_gate_fast(__uint_as_float(g[j] & 0xffff0000u), __uint_as_float(u[j] & 0xffff0000u));
    y[j] = pack_bf16x2(lo, hi);
  }
  *reinterpret_cast<u32x4*>(out + n * inter + c) = y;
}

}  // namespace

namespace pyre {

bool add_rmsnorm_vec(float* resid, const void* delta, int delta_dt, int n_partials, long partial_stride,
                     const float* bias, const void* gain, int gain_dt, void* out, int out_dt, const int* rows, int n,
                     int hidden, float eps, hipStream_t stream) {
  if (hidden % 4 || hidden > 4 * 256 * kNormMaxVec || (delta && partial_stride % 4)) return false;
  if (bias && (!delta || reinterpret_cast<uintptr_t>(bias) % 16)) return false;
  // Which variant runs depends on the number of rows; what it computes does not (see the kernel).
  const bool wide = hidden > 1024;
  const bool few = n <= compute_units() && wide;  // a row a unit: spread over more threads
#define PYRE_NORM_LAUNCH(THREADS, VIRT, ...)                                                                         \
  hipLaunchKernelGGL((add_rmsnorm_vec_kernel<TD, TG, TO, THREADS, VIRT, __VA_ARGS__>), dim3(n), dim3(THREADS), 0, stream, \
                     resid, static_cast<const TD*>(delta), n_partials, hidden, static_cast<size_t>(partial_stride), rows, \
                     static_cast<const TG*>(gain), static_cast<TO*>(out), eps, bias)
  PYRE_DISPATCH(delta_dt, TD, PYRE_DISPATCH(gain_dt, TG, PYRE_DISPATCH(out_dt, TO, {
    const bool many = n >= 512;  // more bytes than the caches keep for the next kernel
    const bool four = n_partials > 2 && static_cast<long>(n) * n_partials < 12000;
    if (few) PYRE_NORM_LAUNCH(1024, 1, false);
    else if (wide && many && four) PYRE_NORM_LAUNCH(256, 4, true, true);
    else if (many && four) PYRE_NORM_LAUNCH(256, 1, true, true);
    else if (wide && many) PYRE_NORM_LAUNCH(256, 4, true);
    else if (wide) PYRE_NORM_LAUNCH(256, 4, false);
    else if (many) PYRE_NORM_LAUNCH(256, 1, true);
    else PYRE_NORM_LAUNCH(256, 1, false);
  })));
#undef PYRE_NORM_LAUNCH
  return true;
}

bool rope_kv_write_vec(const void* qkv, int qkv_dt, int n_partials, long partial_stride, const void* bias,
                       int bias_dt, void* q_out, int q_dt, void* k_cache, void* v_cache, int cache_dt,
                       const float* cos_t, const float* sin_t, int rotary_dim, const int* positions,
                       const int* slots, int n, int nq, int nkv, int hd, int page_size, int write_kv,
                       hipStream_t stream) {
  if (rotary_dim != hd || hd % 8 || partial_stride % 4 || (write_kv && q_dt != cache_dt)) return false;
  const int items = (nq + nkv) * (hd / 8) + nkv * (hd / 4);
  const dim3 grid(n, (items + 255) / 256);
  if (grid.y > 65535) return false;
#define PYRE_ROPE_LAUNCH(READ)                                                                                   \
  PYRE_DISPATCH(qkv_dt, TI, PYRE_DISPATCH(q_dt, TC,                                                               \
      hipLaunchKernelGGL((rope_kv_write_vec_kernel<TI, TC, READ>), grid, dim3(256), 0, stream,                  \
                         static_cast<const TI*>(qkv), static_cast<size_t>(partial_stride), n_partials, nq, nkv, hd, bias,  \
                         positions, write_kv ? slots : nullptr, cos_t, sin_t, bias_dt, page_size, static_cast<TC*>(q_out), \
                         static_cast<TC*>(k_cache), static_cast<TC*>(v_cache))))
  if (n >= 512) {
    if (n_partials > 2 && n < 1200) PYRE_ROPE_LAUNCH(kStreamFour);
    else PYRE_ROPE_LAUNCH(kStream);
  } else if (static_cast<int>(n * grid.y) <= 4 * compute_units()) {
    PYRE_ROPE_LAUNCH(kTogether);
  } else {
    PYRE_ROPE_LAUNCH(kEach);
  }
#undef PYRE_ROPE_LAUNCH
  return true;
}

bool silu_mul_vec(const void* gu, int gu_dt, int n_partials, long partial_stride, void* out, int out_dt,
                  int n, int inter, hipStream_t stream) {
  if (inter % 4 || partial_stride % 4) return false;
  if (gu_dt == kBF16 && out_dt == kBF16 && n_partials == 1 && inter % 8 == 0 && n > 128 &&
      reinterpret_cast<uintptr_t>(gu) % 16 == 0 && reinterpret_cast<uintptr_t>(out) % 16 == 0) {
    const size_t total8 = static_cast<size_t>(n) * (inter / 8);
    hipLaunchKernelGGL(silu_mul_stream_kernel, dim3((total8 + 255) / 256), dim3(256), 0, stream,
                       static_cast<const bf16*>(gu), static_cast<bf16*>(out), total8, inter);
    return true;
  }
  const size_t total4 = static_cast<size_t>(n) * (inter / 4);
  PYRE_DISPATCH(gu_dt, TI, PYRE_DISPATCH(out_dt, TO,
      hipLaunchKernelGGL((silu_mul_vec_kernel<TI, TO>), dim3((total4 + 255) / 256), dim3(256), 0, stream,
                         static_cast<const TI*>(gu), n_partials, static_cast<size_t>(partial_stride),
                         static_cast<TO*>(out), total4, inter)));
  return true;
}

}  // namespace pyre
