// out[m, n] = sum_k A[m, k] * W[n, k] (+ bias[n]) with all three in float32. This is the product of the 32-bit path
// of the model (`pyre/model.py:92-94,125,139,201` are the products it stands for); operands
// of mixed element types stay with gemm_generic.hip.
//
// The matrix cores' float32 instruction has a sixteenth of the 16-bit instruction's rate, so the products are made of bfloat16
// pieces: a float32 is the sum of three, x = h + m + l with eight bits each, exactly (with the scale below), and a product of two
// bfloat16 is exact in float32 (G. Henry, P. Tang, A. Heinecke, "Leveraging the bfloat16 Artificial Intelligence Datatype For
// Higher-Precision Computations", 2019). Of the nine products of pieces the six largest are added, l h', h l', m m', m h', h m' and
// h h' in this order; what is left out (m l', l m', l l') is at most 2^-24 of the product, |m| being up to 2^-8 and |l| up to 2^-17 of
// x, and 2^-27.4 in root mean square. An instruction adds sixteen products of each kind at once, so that an element's sum is rounded six
// times for 16 k where a chain of fused multiply-adds rounds 16 times, and the sum is made in chains that are added in float32 (below).
//
// Measured distance from 64 bits, root mean square over that of the values, here and of the float32 instruction on the same numbers;
// "repeated" is one pair of numbers in [1, 2) a sum, whose roundings all go one way:
//   products            8          16          128         1,536       8,960     part of 640  part of 2,112  part of 4,608
//   random signs  3.1 5.4e-8  3.3 7.1e-8  1.6 2.0e-7  1.8 7.1e-7  2.4 17e-7   3.8 4.5e-7    7.1 8.2e-7     1.1 1.2e-6
//   positive      2.6 4.6e-8  3.3 6.2e-8  1.3 1.6e-7  0.7 5.8e-7  1.3 14e-7   2.8 3.9e-7    4.2 6.6e-7     0.6 1.0e-6
//   repeated      2.5 5.4e-8  3.3 11e-8   3.0 9.2e-7  3.1 113e-7  6.0 658e-7  1.7 4.7e-6    3.9 15.6e-6    8.1 34.0e-6
// The largest error of an element, over the sum of its products' sizes: 0.9e-7 and 2.3e-7 for 8 random products, 0.3e-6 and 2.6e-6
// for 1,536 positive ones. Sums of one or two products are the exception (3.4e-8 and 2.6e-8 for one, at most 1.5e-7 and 6e-8), also where
// all others of a longer sum are far smaller; fewer than eight k are left to the float32 instruction. Numbers that
// a bfloat16 cannot hold the pieces of (infinities and, with the scale below, those from 2^104 on) give a sum that is not finite: such an
// element is made again on the float32 instruction.
//
// As in the weight-streaming kernels the product is computed transposed, out^T = W A^T: the
// 32 rows of an MFMA tile are output columns n, its 32 columns are rows m, so that a lane
// holds runs of four consecutive n of one row m and stores them as one float4.
//
// All kernels below walk k in steps of 16, lanes 0..31 holding k 0..7 of a step and lanes 32..63 k 8..15, on
// v_mfma_f32_32x32x16_bf16, so that an element's value does not depend on the kernel or the tile,
// on the number of rows in the step or on where the row lies in it, bit for bit. Steps past the end of k add zeros.
//
// k may be split into `ksplit` parts (grid.z or tiles of their own), each writing a partial sum out[s] that the
// consumer adds in the order 0..ksplit-1: products with few output columns and a long k would
// otherwise leave most of the chip idle. The caller chooses ksplit from N and K alone. A part is one chain of
// instructions; a product in one part is made in chains of 128 k, added in float32.
#include "pyre_api.h"
#include "pyre_common.h"

using namespace pyre;

namespace {

typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef f32x4 f32x4_any __attribute__((aligned(4)));  // where rows may start on any float: one load all the same
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;

constexpr int BK = 16;        // k per step
constexpr int kChain = 8;     // steps of a chain of a product in one part

// Operands are split 2^kUp times as large, so that the last piece of the smallest float32 (a multiple of 2^-149) is still a normal
// bfloat16 (2^-126 and more); the sums come down again where a part ends. Below about 2^-110 the third piece would otherwise lose bits (an
// operand around 2^-118 1.5e-5 of it, one around 2^-126 4e-3). It is two vector instructions of thirteen in the split and costs two to
// four per cent of a product (us, the 7B shape's gate/up 2,805 -> 2,899 at 2,000 rows, 92 -> 96 at 8; the 1.5B shape's 28.3 -> 29.0 at 8).
// Numbers from 2^104 and sums from 2^80 on are not finite on the way and are made again (`finish`). (A residual as one
// v_dot2_f32_bf16 instead of a shift and a subtraction is exact too and slower: 2,849 -> 3,145.)
constexpr int kUp = 24;
__device__ inline float down(float sum) { return __builtin_amdgcn_ldexpf(sum, -2 * kUp); }

// Eight float32 as three times eight bfloat16 that sum to 2^kUp times them.
struct Pieces {
  u32x4 p[3];
};
// FUSED: the first residual straight from the operand, a shorter chain of larger instructions, for code that is not fetched anew
// by every launch (tiles).
template <bool FUSED = false>
__device__ inline Pieces split8(f32x4 lo, f32x4 hi) {
#pragma clang fp contract(off)
  float up = 1 << kUp;  // these two from scalar registers: half the bytes of instructions that hold a constant
  uint32_t high = 0xffff0000u;
  if (!FUSED) asm("" : "+s"(up), "+s"(high));
  Pieces r;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float a0 = i < 2 ? lo[2 * i] : hi[2 * i - 4], b0 = i < 2 ? lo[2 * i + 1] : hi[2 * i - 3];
    float a = a0 * up, b = b0 * up;
#pragma unroll
    for (int t = 0; t < 3; ++t) {
      const uint32_t w = pack_bf16x2(a, b);
      r.p[t][i] = w;
      const float wa = __uint_as_float(w << 16), wb = __uint_as_float(w & high);
      a = FUSED && t == 0 ? __builtin_fmaf(a0, up, -wa) : a - wa;
      b = FUSED && t == 0 ? __builtin_fmaf(b0, up, -wb) : b - wb;
    }
  }
  return r;
}

// The six products of pieces, the smallest first: piece of W, piece of A.
constexpr int kTerms = 6;
constexpr int kTermW[kTerms] = {2, 0, 1, 1, 0, 0}, kTermA[kTerms] = {0, 2, 1, 0, 1, 0};
__device__ inline f32x16 multiply(u32x4 w, u32x4 a, f32x16 acc) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, w), __builtin_bit_cast(bf16x8, a), acc, 0, 0, 0);
}

// Output columns n .. n + 3 of a row, their sums still `up`; whether one of them is not finite.
__device__ inline bool store4(f32x4 v, bool up, float* row, bool rows_of_16, int n, int N) {
  bool bad = false;
#pragma unroll
  for (int j = 0; j < 4; ++j) v[j] = up ? down(v[j]) : v[j];
#pragma unroll
  for (int j = 0; j < 4; ++j) bad |= !(fabsf(v[j]) < INFINITY);
  if (n + 3 < N && rows_of_16) {
    *reinterpret_cast<f32x4*>(row + n) = v;
  } else {
#pragma unroll 1
    for (int j = 0; j < 4 && n + j < N; ++j) row[n + j] = j == 0 ? v[0] : j == 1 ? v[1] : j == 2 ? v[2] : v[3];
  }
  return bad;
}

// What the usual product does not need: the sums that are not finite once more, and the bias, over a wave's tiles of 32 x 32 (this
// lane's are rows m + 32 q and column groups of four at n + 32 r + 8 i; `a` and `w` are the operands at the part's first k of `len`).
// Infinities, numbers that are not one and those beyond the pieces' range go through the float32 instruction as they are, the whole tile
// in the same steps and chains, of which the elements are kept that were not finite. A row with such a number costs its own tiles
// this much (us, a launch by itself without and with one such row: the 1.5B shape's gate/up 38 and 91 at 20 rows, the 7B shape's 97 and
// 294, 937 and 1,360 at 566; all rows 3,801). An element made by one lane, k by k, held the step up for 2,142, 6,140, 13,530 and 160,351.
// PARTS: a chain is a part of k, whose sums are what the part would be by itself, of pieces where that is finite.
template <bool PARTS = false>
__device__ inline void finish(bool bad, const float* a, size_t lda, const float* w, size_t ldw, const void* bias, int bias_dt, float* out,
                              size_t ldo, int m, int mtiles, int M, int n, int ntiles, int N, int len, int chain) {
  constexpr int kAgain = PARTS ? 1 : 4;  // steps whose operands are asked for together
  const int c = threadIdx.x & 31, half = threadIdx.x >> 5 & 1;
  if (__ballot(bad)) {
#pragma unroll 1
    for (int t = 0; t < mtiles * ntiles; ++t) {
      const int row = m + 32 * (t / ntiles), col = n + 32 * (t % ntiles);
      bool again = false;
#pragma unroll 1
      for (int e = 0; e < 16; ++e) {
        const int at = col + 8 * (e / 4) + e % 4;
        if (row < M && at < N) again |= !(fabsf(out[row * ldo + at]) < INFINITY);
      }
      if (!__ballot(again)) continue;
      // rows and columns past the end are the last one once more
      const float* const x = a + static_cast<size_t>(min(row, M - 1)) * lda + 8 * half;
      const float* const y = w + static_cast<size_t>(min(col - 4 * half + c, N - 1)) * ldw + 8 * half;
      f32x16 acc, sum, total;
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[i] = sum[i] = total[i] = 0.f;
      auto end_chain = [&]() {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const float of_pieces = down(sum[i]);
          total[i] += PARTS && fabsf(of_pieces) < INFINITY ? of_pieces : acc[i];
          acc[i] = sum[i] = 0.f;
        }
      };
      int left = chain;
#pragma unroll 1
      for (int k0 = 0; k0 < len; k0 += kAgain * BK) {
        f32x4 xs[kAgain][2], ys[kAgain][2];
#pragma unroll
        for (int u = 0; u < kAgain; ++u)
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const int k = k0 + BK * u + 4 * h, there = len - 8 * half - k;
            if (there >= 4) {
              xs[u][h] = *reinterpret_cast<const f32x4_any*>(x + k);
              ys[u][h] = *reinterpret_cast<const f32x4_any*>(y + k);
            } else {
#pragma unroll
              for (int j = 0; j < 4; ++j) xs[u][h][j] = j < there ? x[k + j] : 0.f, ys[u][h][j] = j < there ? y[k + j] : 0.f;
            }
          }
#pragma unroll
        for (int u = 0; u < kAgain; ++u) {
          if (u > 0 && k0 + BK * u >= len) continue;
#pragma unroll
          for (int j = 0; j < 8; ++j) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(ys[u][j >> 2][j & 3], xs[u][j >> 2][j & 3], acc, 0, 0, 0);
          if (PARTS) {
            const Pieces p = split8<true>(ys[u][0], ys[u][1]), q = split8<true>(xs[u][0], xs[u][1]);
#pragma unroll
            for (int s = 0; s < kTerms; ++s) sum = multiply(p.p[kTermW[s]], q.p[kTermA[s]], sum);
          }
          if (--left == 0) {
            left = chain;
            end_chain();
          }
        }
      }
      end_chain();  // a last, shorter one (or nothing)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int at = col + 8 * (i / 4) + i % 4;
        float* const p = out + row * ldo + at;
        if (row < M && at < N && !(fabsf(*p) < INFINITY)) *p = total[i];
      }
    }
  }
  if (!bias) return;
#pragma unroll 1
  for (int e = 0; e < 16 * mtiles * ntiles; ++e) {
    const int row = m + 32 * (e / (16 * ntiles)), col = n + 8 * (e / 4 % (4 * ntiles)) + e % 4;
    if (row < M && col < N) out[row * ldo + col] += load_as_float(bias, bias_dt, col);
  }
}

// Fewer than eight k, on the float32 instruction: a sum of one or two products of pieces is up to twice as far from 64 bits as one of
// fused multiply-adds. A wave has 32 rows and 32 columns, straight from memory.
constexpr int kShort = 8;
__global__ __launch_bounds__(256) void gemm_f32_short_kernel(const float* __restrict__ A, size_t lda, const float* __restrict__ W, size_t ldw,
                                                             const void* __restrict__ bias, int bias_dt, float* __restrict__ out, size_t ldo,
                                                             int M, int N, int K, int mt) {
  const int wave = threadIdx.x >> 6, half = threadIdx.x >> 5 & 1, c = threadIdx.x & 31;
  const int n0 = static_cast<int>(blockIdx.x / mt) * 128 + 32 * wave, m = static_cast<int>(blockIdx.x % mt) * 32 + c;
  // rows and columns past the end are the last one once more and are not stored
  const float *const a = A + min(m, M - 1) * lda, *const w = W + min(n0 + c, N - 1) * ldw;
  f32x16 acc;
#pragma unroll
  for (int i = 0; i < 16; ++i) acc[i] = 0.f;
#pragma unroll
  for (int j = 0; j < kShort; j += 2) {
    const int k = j + half;
    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(k < K ? w[k] : 0.f, k < K ? a[k] : 0.f, acc, 0, 0, 0);
  }
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int n = n0 + 8 * (i / 4) + 4 * half + i % 4;
    if (m < M && n < N) out[m * ldo + n] = acc[i] + (bias ? load_as_float(bias, bias_dt, n) : 0.f);
  }
}

// More than 32 rows, and fewer where they do not start on 16 bytes. A block of four waves keeps BM rows of A and BN rows of W; every
// thread brings eight k of some rows, two steps ahead in registers, splits them once for the whole block and writes the pieces into one
// of two buffers in LDS, while the pieces in the other are multiplied: one barrier a slot of SL steps. TAIL: k may end within a step
// (at least eight k in all); the last step's loads lie as far before the end as keeps them in their rows, and what they bring is
// moved to its place, zeros behind it, before it is split.
//
// What bounds it: a step of 128 x 128 is 768 cycles of the matrix cores a SIMD, 580 cycles of LDS (24 KB written, 48 KB read) and
// 410 of splitting; two blocks share a compute unit and fill each other's waits. At 2,000 rows of the 7B shape the gate/up product
// runs at 190 TFLOP/s, 1.14 PFLOP/s of the 16-bit instruction, what that reaches at the clocks the card's power leaves. Against the float32
// instruction (135 of its 157 TFLOP/s; us): gate/up 4,035 -> 2,860 there, 1,240 -> 905 at 566 rows, 318 -> 273 at 99; the 1.5B shape's
// 842 -> 600, 243 -> 207 and 80 -> 75, its way down 447 -> 320, 130 -> 110 and 38 -> 35.
// Rows that start on any float cost two per cent, k that ends within a step five to ten. Against the float32 instruction in tiles that
// went through registers, the 7B shape's gate/up with rows a float off: 713 -> 153 at one row, 1,132 -> 156 at 33, 2,357 -> 567 at 300; with
// four k more: 271 -> 197 at 33 (there against a stream of 64 rows), 523 -> 271 at 99, 1,050 -> 592 at 300.
// The eight k of a lane lie in arrays of their own, so that the lanes of a read are neighbours; each starts 64 bytes (32 of
// slots of two steps) off the banks of the one before, since a write's lanes go to all of them in turn.
//
// A chain of instructions ends after `chain` steps and is added to the total in float32. A block that walks all parts of k
// (where the rows alone fill the chip) ends its chains where the parts end: the bits of the consumer's sum of partial sums, which
// then do not go through memory (WHOLE: every part's sum comes down by itself, as in memory).
struct TileArgs {
  const float* A;
  long lda;
  const float* W;
  long ldw;
  const void* bias;
  int bias_dt;
  float* out;
  size_t ldo, part_stride;
  int M, N, K, kper, chain, nt;
};
template <int BM, int BN, int SL>
constexpr int tile_bytes() { return 2 * 3 * 2 * SL * (16 * (BM + BN) + 64 / SL); }

// Block `block` of `blocks`, whose tiles begin at row `row0` of A.
template <int BM, int BN, int WM, int WN, int SL, bool TAIL, bool WHOLE>
__device__ inline void gemm_f32_tile(unsigned char* const lds, const TileArgs& s, int row0, int mt, int block, int blocks) {
  constexpr int R = BM + BN, KP = 2 * SL, P = KP * R / 256, ROWS = 16 * R + 64 / SL, PLANE = KP * ROWS, BUF = 3 * PLANE;
  constexpr int CT = BM / WM / 32, RT = BN / WN / 32;
  static_assert(WM * WN == 4 && KP * R % 256 == 0 && 2 * BUF == tile_bytes<BM, BN, SL>(), "four waves, whose threads bring equally many pieces");
  const float *const A = s.A, *const W = s.W;
  const long lda = s.lda, ldw = s.ldw;
  const size_t ldo = s.ldo;
  const int M = s.M, N = s.N, chain = s.chain, nt = s.nt;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int c = lane & 31, half = lane >> 5, wm = wave % WM, wn = wave / WM;
  // Blocks are dealt to the eight dies in turn: a die's blocks are neighbours, eight tiles along m by some along n.
  const int die = block & 7, share = blocks >> 3, rest = blocks & 7;
  int t = die * share + min(die, rest) + (block >> 3);
  const int per = mt * nt, ks = t / per;
  t -= ks * per;
  const int group = t / (8 * nt), first = 8 * group, gm = min(8, mt - first);
  t -= 8 * nt * group;
  const int m0 = row0 + (first + t % gm) * BM, n0 = (t / gm) * BN;
  const int kbeg = ks * s.kper, kend = min(s.K, kbeg + s.kper), len = kend - kbeg, steps = (len + BK - 1) / BK;
  const int slots = (steps + SL - 1) / SL;
  float* const out = s.out + ks * s.part_stride;
  const void* const bias = ks ? nullptr : s.bias;  // the bias belongs to one part only

  const float* src[P];
  unsigned dst[P];
#pragma unroll
  for (int i = 0; i < P; ++i) {
    const int p = threadIdx.x + 256 * i, row = p / KP, h = p % KP;  // rows past the end are the last one once more, and are not stored
    src[i] = (row < BM ? A + static_cast<size_t>(min(m0 + row, M - 1)) * lda : W + static_cast<size_t>(min(n0 + row - BM, N - 1)) * ldw) +
             kbeg + 8 * h;
    dst[i] = h * ROWS + 16 * row;
  }
  f32x4 st[2][P][2];
  const bool short_end = SL > 1 && steps % SL;  // the last slot has fewer steps: what lies behind them is not multiplied
  auto last_k = [&](int i) { return len - 8 - 8 * static_cast<int>((threadIdx.x + 256 * i) % KP); };  // of a load in its row, from src[i] on
  auto fetch = [&](int buf, int slot) {
    const int at = min(slot, slots - 1);
#pragma unroll
    for (int i = 0; i < P; ++i) {
      const int k = TAIL ? min(BK * SL * at, last_k(i)) : BK * SL * at - (short_end && at == slots - 1 && (threadIdx.x + 256 * i) % KP >= 2 ? BK : 0);
      st[buf][i][0] = *reinterpret_cast<const f32x4_any*>(src[i] + k);
      st[buf][i][1] = *reinterpret_cast<const f32x4_any*>(src[i] + k + 4);
    }
  };
  auto convert = [&](int buf, int i, int slot) {
    f32x4 lo = st[buf][i][0], hi = st[buf][i][1];
    if (TAIL && slot == slots - 1) {
      const int by = BK * SL * slot - min(BK * SL * slot, last_k(i));  // places towards the front; from eight on nothing is left
#pragma unroll
      for (int b = 1; b < 8; b *= 2)
        if (by & b)
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            const float v = j + b < 4 ? lo[(j + b) & 3] : j + b < 8 ? hi[(j + b) & 3] : 0.f;
            if (j < 4) lo[j] = v;
            else hi[j - 4] = v;
          }
      if (by >= 8) lo = hi = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    const Pieces v = split8<true>(lo, hi);
#pragma unroll
    for (int s = 0; s < 3; ++s) *reinterpret_cast<u32x4*>(lds + buf * BUF + s * PLANE + dst[i]) = v.p[s];
  };
  const unsigned char* const arow = lds + half * ROWS + 16 * (wm * 32 * CT + c);
  const unsigned char* const wrow = lds + half * ROWS + 16 * (BM + wn * 32 * RT + c);
  f32x16 acc[RT][CT], total[RT][CT];
#pragma unroll
  for (int r = 0; r < RT; ++r)
#pragma unroll
    for (int q = 0; q < CT; ++q)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[r][q][i] = total[r][q][i] = 0.f;
  auto end_chain = [&]() {
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
      for (int q = 0; q < CT; ++q)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          total[r][q][i] += WHOLE ? down(acc[r][q][i]) : acc[r][q][i];
          acc[r][q][i] = 0.f;
        }
  };
  int left = chain;
  auto turn = [&](int buf, int slot) {
#pragma unroll
    for (int j = 0; j < SL; ++j) {
      if (j > 0 && SL * slot + j >= steps) break;
      u32x4 a[RT][3], b[CT][3];
      const int at = buf * BUF + 2 * j * ROWS;
#pragma unroll
      for (int s = 0; s < 3; ++s) {
#pragma unroll
        for (int r = 0; r < RT; ++r) a[r][2 - s] = *reinterpret_cast<const u32x4*>(wrow + at + (2 - s) * PLANE + 512 * r);
#pragma unroll
        for (int q = 0; q < CT; ++q) b[q][s] = *reinterpret_cast<const u32x4*>(arow + at + s * PLANE + 512 * q);
      }
#pragma unroll
      for (int s = 0; s < kTerms; ++s) {
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
          for (int q = 0; q < CT; ++q) acc[r][q] = multiply(a[r][kTermW[s]], b[q][kTermA[s]], acc[r][q]);
        // the next slot's pieces meanwhile
        if (j == 0) {
#pragma unroll
          for (int i = 0; i < P; ++i)
            if (i * (kTerms - 1) / P == s) convert(buf ^ 1, i, slot + 1);
        }
      }
      if (j == 0) fetch(buf ^ 1, slot + 3);
      if (--left == 0) {
        end_chain();
        left = chain;
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  };
  // in the order in which the turns ask, so that a turn waits for its own slot alone (the operands are not __restrict__: the
  // compiler would move these loads behind one another)
  fetch(0, 0);
  asm volatile("" ::: "memory");
  fetch(1, 1);
  asm volatile("" ::: "memory");
#pragma unroll
  for (int i = 0; i < P; ++i) convert(0, i, 0);
  fetch(0, 2);
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  int slot = 0;
  for (; slot + 2 <= slots; slot += 2) {  // (no way round turn 1: the compiler's waits are those of the worst way)
    turn(0, slot);
    turn(1, slot + 1);
  }
  if (slot < slots) turn(0, slot);
  end_chain();  // a last, shorter chain (or nothing)
  const bool rows_of_16 = (ldo & 3) == 0 && (reinterpret_cast<uintptr_t>(out) & 15) == 0;
  const int m = m0 + 32 * wm * CT + c, n = n0 + 32 * wn * RT + 4 * half;
  bool bad = false;
#pragma unroll
  for (int q = 0; q < CT; ++q) {
    if (m + 32 * q >= M) continue;
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        bad |= store4(f32x4{total[r][q][4 * i], total[r][q][4 * i + 1], total[r][q][4 * i + 2], total[r][q][4 * i + 3]}, !WHOLE,
                      out + static_cast<size_t>(m + 32 * q) * ldo, rows_of_16, n + 32 * r + 8 * i, N);
  }
  finish<WHOLE>(bad, A + kbeg, lda, W + kbeg, ldw, bias, s.bias_dt, out, ldo, m, CT, M, n, RT, N, len, chain);
}

template <int BM, int BN, int SL, int OCC, bool TAIL, bool WHOLE>
__global__ __launch_bounds__(256, OCC) void gemm_f32_tile_kernel(const TileArgs s, int mt) {
  __shared__ __attribute__((aligned(64))) unsigned char lds[tile_bytes<BM, BN, SL>()];
  gemm_f32_tile<BM, BN, 2, 2, SL, TAIL, WHOLE>(lds, s, 0, mt, blockIdx.x, gridDim.x);
}

// Tiles of 128 x 128 for the first 128 mt rows, the first `big` blocks, and of 64 x 128 for up to 64 rows behind them: where those would
// be half of a tile's rows or less, and so that the last round of blocks has smaller ones to fill it with.
template <bool TAIL, bool WHOLE>
__global__ __launch_bounds__(256, 2) void gemm_f32_mixed_kernel(const TileArgs s, int mt, int big) {
  __shared__ __attribute__((aligned(64))) unsigned char lds[tile_bytes<64, 128, 2>()];
  static_assert(tile_bytes<128, 128, 1>() <= tile_bytes<64, 128, 2>(), "room for either");
  const int block = blockIdx.x;
  if (block < big) gemm_f32_tile<128, 128, 2, 2, 1, TAIL, WHOLE>(lds, s, 0, mt, block, big);
  else gemm_f32_tile<64, 128, 2, 2, 2, TAIL, WHOLE>(lds, s, 128 * mt, 1, block - big, gridDim.x - big);
}

constexpr int kStreamMaxRows = 32;
constexpr int kSlotK = 32;  // k of a slot of the ring: rows of 128 bytes

// 16 bytes per lane straight into LDS: lane x's piece lands at lds_addr + 16 x. The s_nop is the wait state that the instruction
// needs behind a scalar write of m0; the compiler puts none into inline assembly.

__device__ inline void load_to_lds(const void* src, unsigned lds_addr) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" : : "v"(src), "s"(lds_addr) : "memory", "m0");
}
// (past the caches: weights that this launch reads once)
__device__ inline void load_to_lds_nt(const void* src, unsigned lds_addr) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off nt" : : "v"(src), "s"(lds_addr) : "memory", "m0");
}
template <int N>
__device__ inline void wait_loads() {
  asm volatile("s_waitcnt vmcnt(%0)" : : "n"(N) : "memory");
}
__device__ __attribute__((aligned(16))) const unsigned kZeroPiece[4] = {0u, 0u, 0u, 0u};

// Up to 32 rows (k a multiple of four, rows on 16 bytes): the weights as a stream. A block has C times 32 output columns and a
// ring of R slots in LDS; a slot is 32 k (two steps) of the block's rows of W and of 32 rows of A, filled by loads
// that go from memory straight into LDS (whole 128-byte lines: 8 rows x 32 k an instruction; the 16-byte pieces of a row are
// exchanged among themselves by the row's number so that the reads spread over the banks). Waves have one task each: C of them
// multiply, 32 columns each, and split the weights that they multiply, a step's while the one before it is multiplied; C bring
// the weights; four bring eight rows of A each and split them, once for the block, into one of two buffers. Behind the one barrier
// of slot j the weights and pieces of slot j + 1 are read into registers and slot j is multiplied; R - 2 slots are on their way. The
// loops are kept short: between other kernels' launches the instructions come from memory, and 2.7 KB of them less are 0.9 us less.
//
// What bounds it: a compute unit has about 32 KB of loads under way (27 GB/s from memory, 84 from L2), so that a stream
// reaches the memory's rate only if all units pull, and equally much; C is chosen for that. Against the float32 instruction with
// a wave a block up to 16 rows and four above (us, alone in a graph): the 1.5B shape's gate/up 38 -> 30 at 20 rows, its way down 18.4 -> 14.7,
// q/k/v 8.2 -> 6.7, the 7B shape's gate/up 138 -> 97 and 109 -> 95 at 8 rows; at 1 to 16 rows the 1.5B shape's products, which are start
// and end, take 5 to 10 % more (gate/up 27 -> 29, way down 13.1 -> 13.9). Whole steps: 1,299 -> 1,307 us at one request of the 1.5B shape
// (14 layers), 1,334 -> 1,347 at 8, 2,132 -> 1,919 at one of the 7B shape (8 layers), 2,153 -> 1,976 at 8; with the weights kept in the
// caches on their way 6 % more.
// (Weights straight into the registers that they are multiplied from, a lane's eight k at a time, take twice as long: a line is
// asked for eight times there, and the lines that a block's waves have under way do not fit the vector cache.)
constexpr int kRowWaves = 4;
constexpr int kStreamPiece = 512 + 32, kStreamPlane = 4 * kStreamPiece;       // [8 k][row] of a plane of pieces, off each other's banks
constexpr int ring_slots(int C) { return C == 3 || C == 4 ? 6 : 5; }
constexpr int slot_bytes(int C) { return 4096 * (C + 1); }
constexpr int stream_bytes(int C) { return ring_slots(C) * slot_bytes(C) + 2 * 3 * kStreamPlane; }
extern __shared__ __attribute__((aligned(1024))) unsigned char stream_lds[];

template <int C>
__global__ __launch_bounds__(64 * (2 * C + kRowWaves)) void gemm_f32_stream_kernel(
    const float* __restrict__ A, size_t lda, const float* __restrict__ W, size_t ldw,
    const void* __restrict__ bias, int bias_dt, float* __restrict__ out, size_t ldo, size_t part_stride, int M,
    int N, int K, int kper, int chain) {
  constexpr int R = ring_slots(C), SLOT = slot_bytes(C);
  unsigned char* const ring = stream_lds;
  unsigned char* const planes = stream_lds + R * SLOT;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, half = lane >> 5, c = lane & 31;
  const int kbeg = blockIdx.z * kper;
  K = min(K, kbeg + kper);  // this part's end
  out += blockIdx.z * part_stride;
  if (blockIdx.z) bias = nullptr;  // the bias belongs to one part only
  const int slots = (K - kbeg + kSlotK - 1) / kSlotK;
  const unsigned mine = __builtin_amdgcn_readfirstlane(static_cast<unsigned>(reinterpret_cast<uintptr_t>(ring)));
  const float* zero = reinterpret_cast<const float*>(kZeroPiece);
  // A load instruction brings 8 rows: lane x's piece lands at row x / 8, place x % 8, and is piece (place ^ swizzle of the row)
  // of the row's 32 k. Columns past the end are the last one once more and are not stored; rows of A past M are zeros.
  const int lr = lane >> 3, lp = lane & 7;
  int fill = 0;  // ring position of the next slot to load
  auto barrier = [] { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
  if (wave >= 2 * C) {
    const int xr = 8 * (wave - 2 * C) + lr, xk = 4 * (lp ^ ((xr >> 1) & 7));
    const float* const xsrc = A + static_cast<size_t>(xr < M ? xr : 0) * lda + kbeg + xk;
    auto issue = [&](int j) {
      const unsigned dst = mine + fill * SLOT + 4096 * C + 1024 * (wave - 2 * C);
      fill = fill + 1 == R ? 0 : fill + 1;
      const int k0 = kSlotK * j, left = j < slots ? K - kbeg - k0 : 0;  // k of this part from the slot's start on
      load_to_lds(xr < M && xk < left ? xsrc + k0 : zero, dst);
    };
    // Four k of a row a lane, of the rows that this wave has brought: the lane's own piece, and its place among the pieces of eight.
    const unsigned char* const raw = ring + 4096 * C + 1024 * (wave - 2 * C) + 16 * lane;
    unsigned char* const dst = planes + (xk >> 3) * kStreamPiece + 16 * xr + 2 * (xk & 4);
    int at = 0;  // ring position of the next slot whose rows are split
    auto split_rows = [&](int buf) {
      const f32x4 v = *reinterpret_cast<const f32x4*>(raw + at * SLOT);
      at = at + 1 == R ? 0 : at + 1;
      const Pieces p = split8(v, v);
#pragma unroll
      for (int s = 0; s < 3; ++s)
        *reinterpret_cast<uint2*>(dst + (3 * buf + s) * kStreamPlane) = make_uint2(p.p[s][0], p.p[s][1]);
    };
#pragma unroll 1
    for (int j = 0; j < R - 1; ++j) issue(j);
    wait_loads<R - 2>();
    split_rows(0);
    barrier();
    for (int j = 0; j < slots; ++j) {
      issue(j + R - 1);         // into the position of slot j - 1
      wait_loads<R - 2>();      // slot j + 1 is there (loads finish in the order of issue)
      split_rows((j + 1) & 1);  // where the multiplying waves have read those of slot j - 1
      barrier();
    }
    wait_loads<0>();  // the loads past the end
    return;
  }
  if (wave >= C) {
    const int load = wave - C;
    const float* wsrc[4];
    int wk[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = 8 * i + lr;
      wk[i] = 4 * (lp ^ ((r >> 1) & 7));
      wsrc[i] = W + static_cast<size_t>(min((static_cast<int>(blockIdx.x) * C + load) * 32 + r, N - 1)) * ldw + kbeg + wk[i];
    }
    auto issue = [&](int j) {
      const unsigned dst = mine + fill * SLOT + 4096 * load;
      fill = fill + 1 == R ? 0 : fill + 1;
      const int k0 = kSlotK * j, left = j < slots ? K - kbeg - k0 : 0;
#pragma unroll
      for (int i = 0; i < 4; ++i) load_to_lds_nt(wk[i] < left ? wsrc[i] + k0 : zero, dst + 1024 * i);
    };
#pragma unroll 1
    for (int j = 0; j < R - 1; ++j) issue(j);
    wait_loads<4 * (R - 2)>();
    barrier();
    for (int j = 0; j < slots; ++j) {
      issue(j + R - 1);           // into the position of slot j - 1
      wait_loads<4 * (R - 2)>();  // slot j + 1 is there
      barrier();
    }
    wait_loads<0>();  // the loads past the end
    return;
  }
  const int n0 = (blockIdx.x * C + wave) * 32;
  const unsigned char* const wpiece = ring + 4096 * wave + c * 128;
  const unsigned char* const xpiece = planes + half * kStreamPiece + 16 * c;
  const int swz = (c >> 1) & 7;
  int at = 0;  // ring position of the next slot whose weights are read
  f32x4 w[2][2];
  u32x4 x[2][3];
  auto read_w = [&](int t) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
      w[t][h] = *reinterpret_cast<const f32x4*>(wpiece + at * SLOT + 16 * ((4 * t + 2 * half + h) ^ swz));
  };
  auto read_x = [&](int t, int buf) {
#pragma unroll
    for (int s = 0; s < 3; ++s)
      x[t][s] = *reinterpret_cast<const u32x4*>(xpiece + (3 * buf + s) * kStreamPlane + 2 * t * kStreamPiece);
  };
  f32x16 acc, total;
#pragma unroll
  for (int i = 0; i < 16; ++i) acc[i] = total[i] = 0.f;
  auto end_chain = [&]() {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      total[i] += acc[i];
      acc[i] = 0.f;
    }
  };
  auto interleave = [] {
#pragma unroll
    for (int s = 0; s < kTerms; ++s) {
      __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);  // a matrix instruction,
      __builtin_amdgcn_sched_group_barrier(0x2, 11, 0);  // eleven vector instructions (nine: a product of up to 32 rows 1 to 3 % slower)
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  barrier();
  read_w(0);
  read_w(1);
  read_x(0, 0);
  read_x(1, 0);
  Pieces p[2];  // of the two steps' weights
  p[0] = split8(w[0][0], w[0][1]);
#pragma unroll 1
  for (int j = 0; j < slots; ++j) {
    barrier();  // the weights and pieces of the next slot are there
    at = at + 1 == R ? 0 : at + 1;
    p[1] = split8(w[1][0], w[1][1]);
#pragma unroll
    for (int s = 0; s < kTerms; ++s) acc = multiply(p[0].p[kTermW[s]], x[0][kTermA[s]], acc);
    interleave();
    read_w(0);
    read_x(0, (j + 1) & 1);
    read_w(1);
    p[0] = split8(w[0][0], w[0][1]);
#pragma unroll
    for (int s = 0; s < kTerms; ++s) acc = multiply(p[1].p[kTermW[s]], x[1][kTermA[s]], acc);
    interleave();
    read_x(1, (j + 1) & 1);
    if (chain == kChain && j % (kChain / 2) == kChain / 2 - 1) end_chain();
  }
  end_chain();

  // total[4 i + j]: output column n = tile row 8 i + 4 half + j, output row m = tile column c.
  const bool rows_of_16 = (ldo & 3) == 0 && (reinterpret_cast<uintptr_t>(out) & 15) == 0;
  bool bad = false;
  if (c < M) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      bad |= store4(f32x4{total[4 * i], total[4 * i + 1], total[4 * i + 2], total[4 * i + 3]}, true, out + static_cast<size_t>(c) * ldo,
                    rows_of_16, n0 + 4 * half + 8 * i, N);
  }
  finish(bad, A + kbeg, lda, W + kbeg, ldw, bias, bias_dt, out, ldo, c, 1, M, n0 + 4 * half, 1, N, K - kbeg, chain);
}

template <int C>
bool launch_stream(const float* A, long lda, const float* W, long ldw, const void* bias, int bias_dt, float* out, long ldo, long part_stride,
                   int M, int N, int K, int kper, int parts, int chain, hipStream_t stream) {
  static LdsLimit limit;
  if (!allow_lds(limit, reinterpret_cast<const void*>(&gemm_f32_stream_kernel<C>), stream_bytes(C))) return false;
  hipLaunchKernelGGL(gemm_f32_stream_kernel<C>, dim3((N + 32 * C - 1) / (32 * C), 1, parts), dim3(64 * (2 * C + kRowWaves)), stream_bytes(C),
                     stream, A, static_cast<size_t>(lda), W, static_cast<size_t>(ldw), bias, bias_dt, out, static_cast<size_t>(ldo),
                     static_cast<size_t>(part_stride), M, N, K, kper, chain);
  return true;
}

// How many times 32 columns a block has: the least time of the busiest unit, where a block costs half as much as 32 columns for its
// start and its rows of A. (The 1.5B shape's head: 239 us with 32 columns a block, which leave the units least unequal.)
int stream_columns(int N, int parts) {
  int best = 1;
  long least = 0;
  for (int c = 1; c <= 5; ++c) {
    const long blocks = static_cast<long>((N + 32 * c - 1) / (32 * c)) * parts, most = (blocks + compute_units() - 1) / compute_units() * (2 * c + 1);
    if (c == 1 || most <= least) least = most, best = c;
  }
  return best;
}

// The tile with the least work on the busiest unit (a block of two or three shares its matrix cores' time, so that is its
// tiles), smaller ones costing more for the same: their operands come from LDS more often. The three sizes in turn (us): the 1.5B
// shape's gate/up 68, 74, 66 at 99 rows, 187, 158, 176 at 400, 197, 207, 230 at 566; the 7B shape's way down 111, 116, 135, then 344,
// 375, 414 and 440, 484, 545 (without the operands' scale, which adds three per cent to all).
struct TileRows {
  int bm, bn;
  double cost;
};
constexpr int kSizes = 3;
constexpr TileRows kTiles[kSizes] = {{128, 128, 1.0}, {64, 128, 1.2}, {64, 64, 1.4}};
constexpr double kMacsPerUs = 3.9e5;    // of a compute unit
constexpr double kBytesPerUs = 5e6;     // of memory, both ways
constexpr double kFillUs = 0.004;       // a k of a block's chain before the unit's other blocks hide it

// 128 x 128 and, for the last rows, 64 x 128, in one launch (us, one size of tiles and the two: the 1.5B shape's gate/up 250 and 225 at 650
// rows, its way down 107 and 100 at 566, 87 and 82 at 400, q/k/v 25 and 21 at 270, the head 1,551 and 1,501 at 566; the 7B shape's
// gate/up 899 and 851, its way down 439 and 418, at 150 rows 175 and 146). Against tiles of 64 x 128 alone only where that says a
// tenth less: at 8 % less it was slower (the 7B shape's gate/up at 150 rows 369 and 398, the 1.5B shape's at 400 162 and 177).
constexpr int kMixed = kSizes;
constexpr double kMixedLeast = 0.9;

// How many tiles of 128 x 128 the busiest unit's tiles are worth where `big` of them and then `small` ones, each worth 0.6, go to
// whichever unit is free.
double mixed_rounds(long big, long small) {
  const double cost = kTiles[1].cost * kTiles[1].bm / kTiles[0].bm;
  const long units = compute_units();
  long n[2] = {units - big % units, big % units};
  double level[2] = {static_cast<double>(big / units), static_cast<double>(big / units + 1)};
  double most = n[1] ? level[1] : level[0];
  while (small > 0) {
    const int i = n[1] && level[1] < level[0] ? 1 : 0;
    level[i] += cost;
    if (level[i] > most) most = level[i];
    small -= n[i];
  }
  return most;
}

// The tile size for so many rows and `parts` parts of kper, and what it takes in microseconds.
int best_tile(int M, int N, int kper, int parts, double* us) {
  int best = 0;
  double least = 1e300;
  for (int i = 0; i < kSizes; ++i) {
    const long tiles = static_cast<long>((M + kTiles[i].bm - 1) / kTiles[i].bm) * ((N + kTiles[i].bn - 1) / kTiles[i].bn) * parts;
    const double work = kTiles[i].cost * kTiles[i].bm * kTiles[i].bn * kper * ((tiles + compute_units() - 1) / compute_units());
    if (work < least) least = work, best = i;
  }
  if (M > 128 && M % 128 > 0 && M % 128 <= 64) {
    const long columns = static_cast<long>((N + 127) / 128) * parts;
    const double work = 128.0 * 128.0 * kper * mixed_rounds(M / 128 * columns, columns);
    if (work < (best == 1 ? kMixedLeast : 1.0) * least) least = work, best = kMixed;
  }
  if (us) *us = least / kMacsPerUs + 8.0 * parts * M * static_cast<double>(N) / kBytesPerUs + kFillUs * kper;
  return best;
}

// (The last loads of a row lie up to eight k before its end.)
bool takes_tiles(int M, int N, int K) { return K >= kShort && static_cast<long>((M + 63) / 64) * ((N + 63) / 64) < (1L << 24); }
// What is offered as sums of all parts: rows on 16 bytes, whole steps.
bool takes_whole(int M, int N, int K, long lda, long ldw) {
  return M > 16 && lda % 4 == 0 && ldw % 4 == 0 && K % BK == 0 && 4 * lda * M < (1L << 32) && 4 * ldw * N < (1L << 32) && takes_tiles(M, N, K);
}

// Chains of `chain` steps. `whole`: in one part, whose chains are the parts of a product in several.
void launch_tiles(const float* A, long lda, const float* W, long ldw, const void* bias, int bias_dt, float* out, long ldo, long part_stride,
                  int M, int N, int K, int kper, int parts, int chain, bool whole, hipStream_t stream) {
  const int nt = (N + 127) / 128, best = best_tile(M, N, kper, parts, nullptr);
  const bool tail = K % BK != 0;
  TileArgs s{A, lda, W, ldw, bias, bias_dt, out, static_cast<size_t>(ldo), static_cast<size_t>(part_stride), M, N, K, kper, chain, nt};
  if (best == kMixed) {
    const int mt = M / 128, big = mt * nt * parts;
    const auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3(big + nt * parts), dim3(256), 0, stream, s, mt, big); };
    if (whole) go(gemm_f32_mixed_kernel<false, true>);
    else if (tail) go(gemm_f32_mixed_kernel<true, false>);
    else go(gemm_f32_mixed_kernel<false, false>);
    return;
  }
  const auto tile = [&](auto kernel, int bm, int bn) {
    const int mt = (M + bm - 1) / bm;
    s.nt = (N + bn - 1) / bn;
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(mt) * s.nt * parts), dim3(256), 0, stream, s, mt);
  };
#define PYRE_F32_TILE(BM, BN, SL, OCC)                                              \
  tile(whole  ? gemm_f32_tile_kernel<BM, BN, SL, OCC, false, true>                  \
       : tail ? gemm_f32_tile_kernel<BM, BN, SL, OCC, true, false>                  \
              : gemm_f32_tile_kernel<BM, BN, SL, OCC, false, false>, BM, BN)
  if (best == 0) PYRE_F32_TILE(128, 128, 1, 2);
  else if (best == 1) PYRE_F32_TILE(64, 128, 2, 2);
  else PYRE_F32_TILE(64, 64, 2, 3);
#undef PYRE_F32_TILE
}

int part_of(int K, int ksplit) { return ((K + ksplit - 1) / ksplit + BK - 1) / BK * BK; }
// Steps of a chain: a part, or less where there is one part only.
int chain_of(int K, int ksplit) { return ksplit > 1 ? part_of(K, ksplit) / BK : kChain; }

}  // namespace

// Whether the sums of all parts of k are better made by the blocks themselves: where that takes less than the same work in
// parts with their way through memory, there and back (the 1.5B shape's q/k/v in 8 parts, us with the consumer's reading: 28 apart
// and 38 whole at 300 rows, 45 and 61 at 566, 96 and 83 at 1,200, 148 and 111 at 2,000; the 7B shape's o in 9: 120 and 138 at
// 400, 148 and 140 at 566, 926 and 799 at 4,000).
extern "C" int pyre_gemm_f32_adds(int M, int N, int K, long lda, long ldw, int ksplit) {
  if (ksplit <= 1 || M <= 64 || !takes_whole(M, N, K, lda, ldw)) return 0;
  double apart, whole;
  best_tile(M, N, part_of(K, ksplit), ksplit, &apart);
  best_tile(M, N, K, 1, &whole);
  return whole < apart;
}

// Which of the tiles' sizes a product of more than 32 rows takes (`ksplit` parts, or 1: also for the sums of all parts).
extern "C" int pyre_gemm_f32_tile_choice(int M, int N, int K, int ksplit) {
  PYRE_REQUIRE(M > 0 && N > 0 && K > 0 && ksplit > 0, "gemm_f32_tile_choice: bad sizes");
  const int i = best_tile(M, N, part_of(K, ksplit), ksplit, nullptr);
  return i == kMixed ? 1000 * (128 + 64) + 128 : 1000 * kTiles[i].bm + kTiles[i].bn;
}

// Whether up to 64 rows behind those that fill tiles of 128 go to tiles of 64 x 128.
extern "C" int pyre_gemm_f32_tile_mixed(int M, int N, int K, int ksplit) {
  PYRE_REQUIRE(M > 0 && N > 0 && K > 0 && ksplit > 0, "gemm_f32_tile_mixed: bad sizes");
  return best_tile(M, N, part_of(K, ksplit), ksplit, nullptr) == kMixed;
}

extern "C" int pyre_gemm_f32_whole(const float* A, long lda, const float* W, long ldw, float* out, long ldo, int M, int N, int K,
                                   int ksplit, hipStream_t stream) {
  PYRE_REQUIRE(takes_whole(M, N, K, lda, ldw) && lda >= K && ldw >= K && ldo >= N && reinterpret_cast<uintptr_t>(A) % 16 == 0 &&
                   reinterpret_cast<uintptr_t>(W) % 16 == 0,
               "gemm_f32_whole: M=%d (more than 16) N=%d K=%d (a multiple of 16) lda=%ld ldw=%ld (of 4) are not supported", M, N, K, lda, ldw);
  PYRE_REQUIRE(ksplit >= 1 && ksplit <= 64 && static_cast<long>(ksplit - 1) * part_of(K, ksplit) < K, "gemm_f32_whole: ksplit=%d", ksplit);
  launch_tiles(A, lda, W, ldw, nullptr, 0, out, ldo, 0, M, N, K, K, 1, chain_of(K, ksplit), ksplit > 1, stream);
  return check_launch("gemm_f32_whole");
}

extern "C" int pyre_gemm_f32(const float* A, long lda, const float* W, long ldw, const void* bias, int bias_dt,
                             float* out, long ldo, long part_stride, int M, int N, int K, int ksplit,
                             hipStream_t stream) {
  PYRE_REQUIRE(!bias || known_dtype(bias_dt), "gemm_f32: unknown bias dtype");
  PYRE_REQUIRE(M >= 0 && N > 0 && K > 0, "gemm_f32: bad sizes M=%d N=%d K=%d", M, N, K);
  PYRE_REQUIRE(lda >= K && ldw >= K && ldo >= N, "gemm_f32: a leading dimension is too small");
  PYRE_REQUIRE(ksplit >= 1 && ksplit <= 64 && (ksplit == 1 || part_stride >= static_cast<long>(M) * ldo),
               "gemm_f32: ksplit=%d, partial sums %ld apart", ksplit, part_stride);
  if (M == 0) return 0;
  const int kper = part_of(K, ksplit);
  PYRE_REQUIRE(static_cast<long>(ksplit - 1) * kper < K, "gemm_f32: a part of k would be empty (K=%d, ksplit=%d)", K, ksplit);
  // loads that go straight into LDS, 16 bytes a lane, need rows that start on 16 bytes
  const bool vec_ok = lda % 4 == 0 && ldw % 4 == 0 && reinterpret_cast<uintptr_t>(A) % 16 == 0 &&
                     reinterpret_cast<uintptr_t>(W) % 16 == 0;
  const int chain = chain_of(K, ksplit);
  if (K < kShort) {  // (one part: a part has 16 k)
    const long mt = (M + 31) / 32, blocks = mt * ((N + 127) / 128);
    PYRE_REQUIRE(blocks < (1L << 24), "gemm_f32: M=%d N=%d are more than a launch holds", M, N);
    hipLaunchKernelGGL(gemm_f32_short_kernel, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, stream, A, static_cast<size_t>(lda), W,
                       static_cast<size_t>(ldw), bias, bias_dt, out, static_cast<size_t>(ldo), M, N, K, static_cast<int>(mt));
  } else if (M <= kStreamMaxRows && vec_ok && K % 4 == 0) {  // a decode step's rows
    const auto launch = [&](auto f) { return f(A, lda, W, ldw, bias, bias_dt, out, ldo, part_stride, M, N, K, kper, ksplit, chain, stream); };
    const int c = stream_columns(N, ksplit);
    PYRE_REQUIRE(c == 1   ? launch(launch_stream<1>)
                 : c == 2 ? launch(launch_stream<2>)
                 : c == 3 ? launch(launch_stream<3>)
                 : c == 4 ? launch(launch_stream<4>)
                          : launch(launch_stream<5>),
                 "gemm_f32: no device, or too little LDS");
  } else {
    PYRE_REQUIRE(takes_tiles(M, N, K), "gemm_f32: M=%d N=%d are more than a launch holds", M, N);
    launch_tiles(A, lda, W, ldw, bias, bias_dt, out, ldo, part_stride, M, N, K, kper, ksplit, chain, false, stream);
  }
  return check_launch("gemm_f32");
}
