// out[m, n] = sum_k X[m, k] W[n, k] for up to 256 rows of X in bfloat16: the matrix products of
// a decode step (pyre/model.py:315-319,338-342 at the batch sizes of pyre/scheduler.py), above all
// of many requests, where every weight is still read once but the arithmetic is no longer
// free. For products with few output columns (q/k/v, the attention output, the feed-forward's
// way down) the BLAS library's kernels take 19 us or more whatever the size; this kernel keeps
// all rows of X of a step against 64 rows of W and splits k over blocks instead.
//
// The product is computed transposed, out^T = W X^T, on MFMA 32x32x16: A = 32 rows of W, B = 32
// rows of X, both read along k as they are stored. A block owns 32 RTW RW rows of W and BM = 32 to 256
// rows of X: RW groups of XW = 1 to 4 or 6 multiplying waves (a group on RTW tiles of 32 rows of W, its wave q
// on the rows 32 CW q .. of X, CW = 1 or 2 tiles, against all tiles of the group) and some waves that only
// load. k is walked in stages of 64 through a ring in LDS that is filled by loads from memory
// straight into LDS, S - 1 stages ahead; a stage holds its rows as 128-byte rows whose eight
// 16-byte pieces are exchanged among themselves by the row's number, so that the operand reads
// of 32 lanes (32 rows, the same k) spread over all banks. One barrier per stage: it publishes
// the stage that has landed and frees the one before it.
//
// kPartials: `ksplit` blocks share rows of W (grid.y); each writes a partial sum, float32
// [ksplit][M][N], that the consumer adds in the order 0..ksplit-1. kSiluMul (W = gate rows, then
// up rows; ksplit = 1): bfloat16 silu(gate) * up, [M][N / 2]; a tile of W is 16 gate rows and the up rows of the same features. The order of an element's sums
// is a function of k alone: a row's result does not depend on the other rows of the step or on
// their number. The time is set by the bytes a compute unit can take from L2 (the rows of X
// come again for every block): it pays where the blocks fill the chip in one round, which the
// caller checks.
#include "pyre_api.h"
#include "pyre_common.h"

using namespace pyre;

namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) float f32x4;

constexpr int BN = 64;   // rows of W per block (kPartials; or twice as many)
constexpr int BK = 64;   // k per stage: rows of 128 bytes

// 16 bytes per lane from global memory straight into LDS: lane x's piece lands at
// lds_addr + 16 x. The compiler does not know of these loads; whoever reads the bytes
// waits for them with wait_loads (they finish in the order of issue) and a barrier. The s_nop is the wait state that the instruction
// needs behind a scalar write of m0; the compiler puts none into inline assembly.
__device__ inline void load_to_lds(const void* src, unsigned lds_addr) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" : : "v"(src), "s"(lds_addr) : "memory", "m0");
}
// The same for bytes that are read once (the weights): past the caches.
__device__ inline void load_to_lds_once(const void* src, unsigned lds_addr) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off nt" : : "v"(src), "s"(lds_addr) : "memory", "m0");
}
template <int N>
__device__ inline void wait_loads() {
  asm volatile("s_waitcnt vmcnt(%0)" : : "n"(N) : "memory");
}
__device__ __attribute__((aligned(16))) const unsigned kZeroPiece[4] = {0u, 0u, 0u, 0u};

enum Epilogue { kPartials = 0, kSiluMul = 1 };

// RW groups of XW multiplying waves, each group on RTW tiles of W, and NL waves that only load; S
// stages in the ring. What a wave can have loaded per microsecond is limited (about 9 GB/s from
// L2, whatever the pattern and however many loads it has on their way; a compute unit takes
// about 84 GB/s), so the loads of a stage are dealt to all waves, and there are more waves than
// multiply; a stage is the rows of W, then the BM rows of X. kSiluMul: a tile's 32 rows
// are 16 gate rows and the up rows of the same features, so that a lane holds both for its
// elements; a block has 8 NG features: where NG is odd, the last tile has eight gate rows and eight up rows, and no others are
// loaded; out is bfloat16 [M][N / 2]. Of the rows of X the first 8 XG are loaded, the others are zeros once
// and for all. The number of waves divides the loads of a stage where it can: a spare turn costs as much as a load.
template <int CW, int XW, int RTW, int RW, int NG, int XG, int EPI, int NL, int S>
__global__ __launch_bounds__(64 * (XW * RW + NL)) void gemm_mid_kernel(const bf16* __restrict__ X, size_t ldx,
                                                                      const bf16* __restrict__ W, size_t ldw,
                                                                      void* __restrict__ out, int M, int N, int K,
                                                                      int kper, GateShape act) {
  constexpr int BM = 32 * CW * XW, BW = EPI == kSiluMul ? 16 * NG : 32 * RTW * RW, ROWS = BW + BM, STAGE = ROWS * 128;
  constexpr int NWAVES = XW * RW + NL, LOADED = BW + 8 * XG, LOADS = LOADED / 8;
  constexpr int HALF = EPI == kSiluMul && NG % 2 ? NG / 2 : -1;  // the tile of sixteen rows
  static_assert(EPI != kSiluMul || (NG + 1) / 2 == RTW * RW, "the tiles hold the features");
  constexpr int PER = (LOADS + NWAVES - 1) / NWAVES;  // loads of 8 rows per wave and stage
  // Where the loads of a stage do not divide evenly over the waves, the spare turns load zeros
  // into a kilobyte behind the ring, so that every wave counts the same number of loads.
  constexpr bool SPARE = LOADS % NWAVES != 0;
  __shared__ __attribute__((aligned(1024))) unsigned char lds[S * STAGE + (SPARE ? 1024 : 0)];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int c = lane & 31, half = lane >> 5;
  const int ks = blockIdx.y, kbeg = ks * kper, kend = min(K, kbeg + kper);
  const int stages = (kend - kbeg + BK - 1) / BK;
  const int inter = N / 2;

  // Every wave loads: of load j = wave + NWAVES i (rows 8 j .. 8 j + 7 of the stage) this lane
  // brings the piece that lands at row 8 j + lane / 8, place lane % 8, which is piece
  // (place ^ swizzle of the row) of the row's 64 k. Rows past the end are zeros.
  const unsigned lds_base = __builtin_amdgcn_readfirstlane(static_cast<unsigned>(reinterpret_cast<uintptr_t>(lds)));
  const bf16* zero = reinterpret_cast<const bf16*>(kZeroPiece);
  const bf16* src[PER];
  int kofs[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int row = 8 * (wave + NWAVES * i) + (lane >> 3);
    kofs[i] = 8 * ((lane & 7) ^ ((row >> 1) & 7));
    const bf16* base = nullptr;
    if (row >= LOADED) {
      // a spare turn
    } else if (row < BW) {
      int n;  // the row of W behind row `row` of the block's tile, or past the end
      if (EPI == kSiluMul) {
        const int half_rows = (row >> 5) == HALF ? 8 : 16, in_tile = row & 31;
        const int f = blockIdx.x * (8 * NG) + 16 * (row >> 5) + (in_tile & (half_rows - 1));
        n = f < inter ? (in_tile / half_rows) * inter + f : N;
      } else {
        n = blockIdx.x * BW + row;
      }
      if (n < N) base = W + static_cast<size_t>(n) * ldw;
    } else if (row - BW < M) {
      base = X + static_cast<size_t>(row - BW) * ldx;
    }
    src[i] = base ? base + kbeg + kofs[i] : nullptr;
  }
  auto issue = [&](int st, int slot) {
    const int left = st < stages ? kend - kbeg - BK * st : 0;  // k of this part from the stage's start on
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int j = wave + NWAVES * i;  // rows 8 j .. of the stage: of W up to BW / 8
      const bf16* from = src[i] && kofs[i] < left ? src[i] + BK * st : zero;
      const unsigned to = j < LOADS ? lds_base + slot * STAGE + j * 1024 : lds_base + S * STAGE;
      if (j < BW / 8) load_to_lds_once(from, to);
      else load_to_lds(from, to);
    }
  };
#pragma unroll
  for (int st = 0; st < S - 1; ++st) issue(st, st);
  if constexpr (LOADED < ROWS) {  // before the first barrier, so before anybody reads them
    constexpr int UNITS = (ROWS - LOADED) * 8;  // of sixteen bytes, a stage
    for (int i = threadIdx.x; i < S * UNITS; i += 64 * NWAVES)
      *reinterpret_cast<uint4*>(lds + i / UNITS * STAGE + LOADED * 128 + i % UNITS * 16) = uint4{0u, 0u, 0u, 0u};
  }

  if (wave >= XW * RW) {
    // ---- a wave that only loads
    int slot = 0;
    for (int st = 0; st < stages; ++st) {
      wait_loads<PER * (S - 2)>();  // loads finish in the order of issue: this wave's share of stage st is there
      __syncthreads();              // everyone knows, and stage st - 1 has been multiplied
      issue(st + S - 1, slot == 0 ? S - 1 : slot - 1);
      slot = slot + 1 == S ? 0 : slot + 1;
    }
    wait_loads<0>();  // the loads past the end
    return;
  }

  // ---- a multiplying wave: its own 32 CW rows of X against its group's tiles of W.
  const int group = wave / XW, quarter = wave % XW;
  f32x16 acc[RTW][CW];
#pragma unroll
  for (int rt = 0; rt < RTW; ++rt)
#pragma unroll
    for (int ct = 0; ct < CW; ++ct)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[rt][ct][i] = 0.f;

  const int swz = (c >> 1) & 7;
  // This lane's rows of W in the stage and how their pieces are exchanged; in the tile of sixteen rows eight lanes read rows of others.
  int wrow[RTW], wswz[RTW];
#pragma unroll
  for (int rt = 0; rt < RTW; ++rt) {
    const int t = RTW * group + rt, in_tile = t == HALF ? (c & 7) + 8 * (c >> 4) : c;
    wrow[rt] = (32 * t + in_tile) * 128;
    wswz[rt] = HALF < 0 ? swz : (in_tile >> 1) & 7;
  }
  const int xrow0 = BW + 32 * CW * quarter + c;    // and of X
  int slot = 0;
  for (int st = 0; st < stages; ++st) {
    wait_loads<PER * (S - 2)>();  // this wave's share of stage st is there
    __syncthreads();              // and everyone's; and everyone has multiplied stage st - 1
    issue(st + S - 1, slot == 0 ? S - 1 : slot - 1);
    const unsigned char* sb = lds + slot * STAGE;
    // The operands of step kk + 1 are read from LDS while step kk is multiplied.
    bf16x8 a[RTW], b[CW], an[RTW], bn[CW];
    auto read = [&](int kk, bf16x8 (&ra)[RTW], bf16x8 (&rb)[CW]) {
      const int piece = 16 * ((2 * kk + half) ^ swz);
#pragma unroll
      for (int rt = 0; rt < RTW; ++rt) ra[rt] = *reinterpret_cast<const bf16x8*>(sb + wrow[rt] + 16 * ((2 * kk + half) ^ wswz[rt]));
#pragma unroll
      for (int ct = 0; ct < CW; ++ct) rb[ct] = *reinterpret_cast<const bf16x8*>(sb + (xrow0 + 32 * ct) * 128 + piece);
    };
    if constexpr (RTW + CW <= 3 && XW <= 2) {  // few operands: a stage's are all asked for together
      bf16x8 wa[BK / 16][RTW], xb[BK / 16][CW];
#pragma unroll
      for (int kk = 0; kk < BK / 16; ++kk) read(kk, wa[kk], xb[kk]);
#pragma unroll
      for (int kk = 0; kk < BK / 16; ++kk)
#pragma unroll
        for (int rt = 0; rt < RTW; ++rt)
#pragma unroll
          for (int ct = 0; ct < CW; ++ct)
            acc[rt][ct] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wa[kk][rt], xb[kk][ct], acc[rt][ct], 0, 0, 0);
      slot = slot + 1 == S ? 0 : slot + 1;
      continue;
    }
    read(0, a, b);
#pragma unroll
    for (int kk = 0; kk < BK / 16; ++kk) {
      if (kk + 1 < BK / 16) read(kk + 1, an, bn);
#pragma unroll
      for (int rt = 0; rt < RTW; ++rt)
#pragma unroll
        for (int ct = 0; ct < CW; ++ct)
          acc[rt][ct] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[rt], b[ct], acc[rt][ct], 0, 0, 0);
#pragma unroll
      for (int rt = 0; rt < RTW; ++rt) a[rt] = an[rt];
#pragma unroll
      for (int ct = 0; ct < CW; ++ct) b[ct] = bn[ct];
    }
    slot = slot + 1 == S ? 0 : slot + 1;
  }
  wait_loads<0>();  // the loads past the end

  // acc[rt][ct][4 q + j]: row 32 rt + 8 q + 4 half + j of the group's tiles of W, row
  // 32 (CW quarter + ct) + c of X.
  if (EPI == kPartials) {
    float* o = static_cast<float*>(out) + static_cast<size_t>(ks) * M * N;
    const bool vec = (N & 3) == 0 && (reinterpret_cast<uintptr_t>(out) & 15) == 0;
#pragma unroll
    for (int ct = 0; ct < CW; ++ct) {
      const int m = 32 * (CW * quarter + ct) + c;
      if (m >= M) continue;
#pragma unroll
      for (int rt = 0; rt < RTW; ++rt)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int n = blockIdx.x * BW + 32 * RTW * group + 32 * rt + 8 * q + 4 * half;
          if (n >= N) continue;
          float* dst = o + static_cast<size_t>(m) * N + n;
          if (vec && n + 3 < N) {
            *reinterpret_cast<f32x4*>(dst) =
                f32x4{acc[rt][ct][4 * q], acc[rt][ct][4 * q + 1], acc[rt][ct][4 * q + 2], acc[rt][ct][4 * q + 3]};
          } else {
            for (int j = 0; j < 4 && n + j < N; ++j) dst[j] = acc[rt][ct][4 * q + j];
          }
        }
    }
  } else {
    bf16* o = static_cast<bf16*>(out);
    const bool vec = (inter & 3) == 0 && (reinterpret_cast<uintptr_t>(out) & 7) == 0;
#pragma unroll
    for (int ct = 0; ct < CW; ++ct) {
      const int m = 32 * (CW * quarter + ct) + c;
      if (m >= M) continue;
#pragma unroll
      for (int rt = 0; rt < RTW; ++rt)
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          const int in_block = 16 * (RTW * group + rt) + 8 * q + 4 * half, f = blockIdx.x * (8 * NG) + in_block;
          if (in_block >= 8 * NG || f >= inter) continue;
          float y[4];
#pragma unroll
          for (int j = 0; j < 4; ++j) y[j] = gated_unit(acc[rt][ct][4 * q + j], acc[rt][ct][4 * (q + 2) + j], act);
          bf16* dst = o + static_cast<size_t>(m) * inter + f;
          if (vec && f + 3 < inter) {
            *reinterpret_cast<uint2*>(dst) = uint2{pack_bf16x2(y[0], y[1]), pack_bf16x2(y[2], y[3])};
          } else {
            for (int j = 0; j < 4 && f + j < inter; ++j) dst[j] = from_float<bf16>(y[j]);
          }
        }
    }
  }
}

int check_mid(const char* name, const void* X, const void* W, int M, int N, int K, long ldx, long ldw) {
  PYRE_REQUIRE(pyre_gemm_mid_supports(M, N, K, ldx, ldw),
               "%s: M=%d (1..256) N=%d K=%d (multiples of 8) ldx=%ld ldw=%ld (multiples of 8, >= K) are not supported",
               name, M, N, K, ldx, ldw);
  PYRE_REQUIRE(reinterpret_cast<uintptr_t>(X) % 16 == 0 && reinterpret_cast<uintptr_t>(W) % 16 == 0,
               "%s: operands must lie on 16 bytes", name);
  return 0;
}

}  // namespace

extern "C" int pyre_gemm_mid_supports(int M, int N, int K, long ldx, long ldw) {
  return M >= 1 && M <= 256 && N >= 1 && K >= 8 && K % 8 == 0 && ldx >= K && ldx % 8 == 0 && ldw >= K && ldw % 8 == 0;
}

// out: float32 [ksplit][M][N].
extern "C" int pyre_gemm_mid_bf16(const void* X, long ldx, const void* W, long ldw, float* out, int M, int N,
                                  int K, int ksplit, int wide, hipStream_t stream) {
  const GateShape act{};  // partial sums: no unit to finish
  if (int rc = check_mid("gemm_mid_bf16", X, W, M, N, K, ldx, ldw)) return rc;
  PYRE_REQUIRE(ksplit >= 1 && ksplit <= 64, "gemm_mid_bf16: ksplit=%d", ksplit);
  const int kper = ((K + ksplit - 1) / ksplit + BK - 1) / BK * BK;
  PYRE_REQUIRE(static_cast<long>(ksplit - 1) * kper < K, "gemm_mid_bf16: a part of k would be empty (K=%d, ksplit=%d)", K, ksplit);
  const auto go = [&](auto kernel, int rows, int waves) {
    hipLaunchKernelGGL(kernel, dim3((N + rows - 1) / rows, ksplit), dim3(64 * waves), 0, stream, static_cast<const bf16*>(X),
                       static_cast<size_t>(ldx), static_cast<const bf16*>(W), static_cast<size_t>(ldw), static_cast<void*>(out), M, N, K, kper, act);
  };
  if (wide) {
    // Twice the rows of W a block, over half as much of k where the caller splits k further: a
    // block's bytes (its rows of W and all rows of X, over its part of k) are fewest where the two
    // are equally many, and at few rows of X a stage (and the barrier that goes with it) carries
    // twice the bytes. Measured on the 7B shape's way down, weights from memory: 25.6 us at 64
    // rows of X where 64 rows of W a block take 29.8 and the weight-streaming kernel 31.9.
    if (M <= 32) go(gemm_mid_kernel<1, 1, 1, 4, 0, 4, kPartials, 6, 6>, 2 * BN, 10);
    else if (M <= 64) go(gemm_mid_kernel<1, 2, 1, 4, 0, 8, kPartials, 4, 5>, 2 * BN, 12);
    else if (M <= 128) go(gemm_mid_kernel<1, 4, 2, 2, 0, 16, kPartials, 8, 4>, 2 * BN, 16);
    else if (M <= 192) go(gemm_mid_kernel<2, 3, 2, 2, 0, 24, kPartials, 8, 3>, 2 * BN, 14);
    else go(gemm_mid_kernel<2, 4, 2, 2, 0, 32, kPartials, 8, 3>, 2 * BN, 16);
  } else if (M > 192) {
    go(gemm_mid_kernel<2, 4, 2, 1, 0, 32, kPartials, 6, 3>, BN, 10);
  } else if (M > 128) {
    go(gemm_mid_kernel<1, 6, 1, 2, 0, 24, kPartials, 4, 4>, BN, 16);
  } else if (M > 64) {
    go(gemm_mid_kernel<1, 4, 1, 2, 0, 16, kPartials, 4, 4>, BN, 12);
  } else if (M > 32) {
    go(gemm_mid_kernel<1, 2, 1, 2, 0, 8, kPartials, 12, 5>, BN, 16);
  } else if (M > 16) {
    go(gemm_mid_kernel<1, 1, 1, 2, 0, 4, kPartials, 10, 8>, BN, 12);
  } else if (M > 8) {
    go(gemm_mid_kernel<1, 1, 1, 2, 0, 2, kPartials, 8, 8>, BN, 10);
  } else {
    go(gemm_mid_kernel<1, 1, 1, 2, 0, 1, kPartials, 7, 8>, BN, 9);
  }
  return check_launch("gemm_mid_bf16");
}

// W = [gate rows; up rows] (two_i x K); out: bfloat16 [M][two_i / 2] = silu(X gate^T) * (X up^T).
// The most features that a block takes: 64, or 96 for up to 128 rows of X (128 for 25 to 64 rows) where one round of blocks would
// not hold them otherwise.
namespace {
int most_features(int M, int two_i) {
  const int inter = two_i / 2, units = compute_units();
  if ((inter + 63) / 64 <= units || M > 128) return 64;
  // 128 features: the 32B shape's 27,648 in 216 blocks, for 25 to 64 rows of X (measured in its
  // decode steps against the weight-streaming kernel: 34.2 against 35.0 ms at 64 requests, 22.7
  // against 22.9 at 32, the same at 8, 13.0 against 12.7 at one)
  return M >= 25 && M <= 64 && (inter + 95) / 96 > units ? 128 : 96;
}

// Features of a block where one round of blocks holds them all, in eights: as few as let the blocks fill the chip, since what a compute
// unit has on its way from memory is limited. With that, with waves that divide a stage's loads, with rows of X that are not there
// left out of them and a tile of W a wave (more waves wait for LDS at a time), us from -> to, weights from memory: the 1.5B shape's
// gate/up in 224 blocks of 40 instead of 140 of 64, 15.2 -> 12.4 at one row, 17.6 -> 14.5 at 64, 20.3 -> 17.3 at 99, 26.5 -> 22.8 at 190,
// 28.7 -> 25.1 at 256; the 7B shape's in 237 of 80 instead of 198 of 96, 47.0 -> 45.6 at 8, 52.7 -> 48.4 at 64, 62.1 -> 57.6 at 128. The
// 1.5B shape's q/k/v 5.1 -> 4.5 at one row, 5.9 -> 5.3 at 64, 9.1 -> 8.5 at 190, its way down 8.1 -> 7.2, 9.4 -> 8.9, 15.5 -> 14.9.
// Of the other sizes, the kernel alone, at 1, 64, 128 and 256 rows: 32 features (8,192 of k = 2,048) 20.2 -> 16.7, 21.0 -> 16.6,
// 25.4 -> 20.2, 35.2 -> 28.5; 48 (11,008 of 2,048) 21.6 -> 19.7, 22.5 -> 20.9, 25.9 -> 24.0, 35.8 -> 35.2; 64 (13,824 of 5,120) 46.9 -> 46.1,
// 52.8 -> 52.4, 63.5 -> 63.2, 91.3 -> 91.2; 96 (22,016 of 4,096) 68.3 -> 65.8, 66.6 -> 65.6, 73.4 -> 72.3.
int feature_groups(int M, int two_i) {
  const int inter = two_i / 2, units = compute_units(), most = most_features(M, two_i);
  if ((inter + most - 1) / most > units) return most / 8;
  const int even = (inter + 8 * units - 1) / (8 * units);
  for (const int groups : {4, 5, 6, 8, 10, 12})
    if (even <= groups && groups <= most / 8) return groups;
  return most / 8;
}
}  // namespace

extern "C" int pyre_gemm_mid_silu_blocks(int M, int two_i) {
  const int f = most_features(M, two_i);
  return (two_i / 2 + f - 1) / f;
}

static int mid_gated(const void* X, long ldx, const void* W, long ldw, void* out, int M, int two_i, int K, GateShape act,
                     hipStream_t stream) {
  if (int rc = check_mid("gemm_mid_silu_bf16", X, W, M, two_i, K, ldx, ldw)) return rc;
  PYRE_REQUIRE(two_i % 2 == 0, "gemm_mid_silu_bf16: gate and up rows must be equally many");
  const int kper = (K + BK - 1) / BK * BK, groups = feature_groups(M, two_i);
  const auto go = [&](auto kernel, int waves) {
    hipLaunchKernelGGL(kernel, dim3((two_i / 2 + 8 * groups - 1) / (8 * groups)), dim3(64 * waves), 0, stream, static_cast<const bf16*>(X),
                       static_cast<size_t>(ldx), static_cast<const bf16*>(W), static_cast<size_t>(ldw), out, M, two_i, K, kper, act);
  };
  // By rows of X and groups of features: fewer of either are fewer multiplying waves, fewer loads and a deeper ring.
  if (M > 192) {
    if (groups == 4) go(gemm_mid_kernel<2, 4, 1, 2, 4, 32, kSiluMul, 6, 3>, 14);
    else if (groups == 5) go(gemm_mid_kernel<2, 4, 1, 3, 5, 32, kSiluMul, 2, 3>, 14);
    else if (groups == 6) go(gemm_mid_kernel<2, 4, 1, 3, 6, 32, kSiluMul, 3, 3>, 15);
    else go(gemm_mid_kernel<2, 4, 2, 2, 8, 32, kSiluMul, 8, 3>, 16);
  } else if (M > 128) {
    if (groups == 4) go(gemm_mid_kernel<1, 6, 1, 2, 4, 24, kSiluMul, 4, 4>, 16);
    else if (groups == 5) go(gemm_mid_kernel<1, 6, 3, 1, 5, 24, kSiluMul, 6, 3>, 12);
    else if (groups == 6) go(gemm_mid_kernel<1, 6, 3, 1, 6, 24, kSiluMul, 6, 3>, 12);
    else go(gemm_mid_kernel<2, 3, 2, 2, 8, 24, kSiluMul, 8, 3>, 14);
  } else if (M > 64) {
    if (groups == 4) go(gemm_mid_kernel<1, 4, 1, 2, 4, 16, kSiluMul, 4, 5>, 12);
    else if (groups == 5) go(gemm_mid_kernel<1, 4, 1, 3, 5, 16, kSiluMul, 1, 4>, 13);
    else if (groups == 6) go(gemm_mid_kernel<1, 4, 1, 3, 6, 16, kSiluMul, 2, 4>, 14);
    else if (groups == 8) go(gemm_mid_kernel<1, 4, 2, 2, 8, 16, kSiluMul, 8, 4>, 16);
    // (96 rows of X: 46.0 us at 65 and 49.0 at 96 on the 7B shape, where the 128 rows of the form below take 50.8 and 53.5)
    else if (groups == 10 && M <= 96) go(gemm_mid_kernel<1, 3, 1, 5, 10, 12, kSiluMul, 1, 4>, 16);
    else if (groups == 10) go(gemm_mid_kernel<2, 2, 1, 5, 10, 16, kSiluMul, 2, 4>, 12);
    else if (M <= 96) go(gemm_mid_kernel<1, 3, 2, 3, 12, 12, kSiluMul, 3, 4>, 12);
    else go(gemm_mid_kernel<1, 4, 2, 3, 12, 16, kSiluMul, 2, 3>, 14);
  } else if (M > 32) {
    if (groups == 4) go(gemm_mid_kernel<1, 2, 1, 2, 4, 8, kSiluMul, 4, 6>, 8);
    else if (groups == 5) go(gemm_mid_kernel<1, 2, 1, 3, 5, 8, kSiluMul, 3, 6>, 9);
    else if (groups == 6) go(gemm_mid_kernel<1, 2, 1, 3, 6, 8, kSiluMul, 4, 6>, 10);
    else if (groups == 8) go(gemm_mid_kernel<1, 2, 1, 4, 8, 8, kSiluMul, 4, 5>, 12);
    else if (groups == 10) go(gemm_mid_kernel<1, 2, 1, 5, 10, 8, kSiluMul, 4, 5>, 14);
    else if (groups == 12) go(gemm_mid_kernel<1, 2, 1, 6, 12, 8, kSiluMul, 4, 4>, 16);
    else go(gemm_mid_kernel<1, 2, 2, 4, 16, 8, kSiluMul, 6, 3>, 14);
  } else if (M > 8) {
    if (groups == 4) go(gemm_mid_kernel<1, 1, 1, 2, 4, 4, kSiluMul, 10, 8>, 12);
    else if (groups == 5) go(gemm_mid_kernel<1, 1, 1, 3, 5, 4, kSiluMul, 11, 8>, 14);
    else if (groups == 6) go(gemm_mid_kernel<1, 1, 1, 3, 6, 4, kSiluMul, 13, 8>, 16);
    else if (groups == 8) go(gemm_mid_kernel<1, 1, 1, 4, 8, 4, kSiluMul, 6, 6>, 10);
    else if (groups == 10) go(gemm_mid_kernel<1, 1, 1, 5, 10, 4, kSiluMul, 7, 6>, 12);
    else if (groups == 12) go(gemm_mid_kernel<1, 1, 1, 6, 12, 4, kSiluMul, 8, 5>, 14);
    // (the 32B shape at 25 and 32 rows: 91.4 and 90.7 us, with two tiles a wave 94.0 and 93.5; with one or eight waves that only load
    // beside these eight 93.2 and 92.1, 93.6 and 92.5)
    else go(gemm_mid_kernel<1, 1, 1, 8, 16, 4, kSiluMul, 4, 4>, 12);
  } else {
    if (groups == 4) go(gemm_mid_kernel<1, 1, 1, 2, 4, 1, kSiluMul, 7, 8>, 9);
    else if (groups == 5) go(gemm_mid_kernel<1, 1, 1, 3, 5, 1, kSiluMul, 8, 8>, 11);
    else if (groups == 6) go(gemm_mid_kernel<1, 1, 1, 3, 6, 1, kSiluMul, 10, 8>, 13);
    else if (groups == 8) go(gemm_mid_kernel<1, 1, 1, 4, 8, 1, kSiluMul, 5, 6>, 9);
    else if (groups == 10) go(gemm_mid_kernel<1, 1, 1, 5, 10, 1, kSiluMul, 6, 6>, 11);
    else go(gemm_mid_kernel<1, 1, 1, 6, 12, 1, kSiluMul, 7, 5>, 13);
  }
  return check_launch("gemm_mid_silu_bf16");
}

extern "C" int pyre_gemm_mid_silu_bf16(const void* X, long ldx, const void* W, long ldw, void* out, int M,
                                       int two_i, int K, hipStream_t stream) {
  return mid_gated(X, ldx, W, ldw, out, M, two_i, K, GateShape{}, stream);
}

// The same with another gated unit in the epilogue: g sigmoid(slope (g + cubic g^3)) (u + shift), inputs clipped at `limit`.
extern "C" int pyre_gemm_mid_glu_bf16(const void* X, long ldx, const void* W, long ldw, void* out, int M, int two_i,
                                      int K, float limit, float slope, float shift, float cubic, hipStream_t stream) {
  return mid_gated(X, ldx, W, ldw, out, M, two_i, K, GateShape{limit, slope, shift, cubic}, stream);
}
