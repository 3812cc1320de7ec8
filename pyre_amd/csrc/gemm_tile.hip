// out[m, n] = sum_k X[m, k] W[n, k] in bfloat16 with float32 sums, for the many rows of prompts and mixed steps
// (pyre/model.py:84-87,92-94,133-139 with a whole prompt as their rows).
//
// The product is computed transposed, out^T = W X^T, on MFMA 32x32x16: A = 32 rows of W, B = 32 rows of X, both read
// along k as they are stored. A block owns BM rows of X and BN rows of W, its WM x WN waves a part of that each; k is
// walked in stages of 64 through a ring of S slots in LDS that loads from memory fill directly, rows of 128 bytes whose
// eight 16-byte pieces are exchanged among themselves by the row's number, so that the operand reads of 32 lanes spread
// over all banks. The operands of the next 16 k are read while the present ones are multiplied; the one barrier of a stage
// stands before its last 16 k: by then every wave has read the slot for the last time, so the loads of S stages further on
// go into it, and the next stage's slot, which everybody has waited for, is read from.
//
// A block takes tiles one after the other until none is left: the first loads of the next tile are on their way before
// the results of the present one are stored. The tiles that the 32 compute units of a die work on at a time are neighbours
// (eight tiles along m by four along n): its L2 then serves every row several times.
//
// kF32Out: float32 [ksplit][M][N], part `ks` of k; kGated: W = gate rows, then up rows; bfloat16 [M][N / 2], the gated
// unit of the two; kPaged: X's rows lie in the pages of a cache, 32 consecutive positions of a request at a time; bfloat16 [N / ldo][M][ldo].
// Results pass through four kilobytes of LDS of the wave's own, so that a store writes whole lines: a
// lane's own four elements are 8 or 16 bytes of a row, and 32 rows of such pieces to a store make the L2's rate of
// requests the limit.
#include "pyre_api.h"
#include "pyre_common.h"

#include <type_traits>

using namespace pyre;

namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) float f32x4;

constexpr int BK = 64;             // k of a stage
constexpr int ROW = 2 * BK;        // bytes of a row in a stage
constexpr int GROUP = 8;           // tiles along m that are neighbours in time

// 16 bytes per lane from `base + off` straight into LDS: lane x's piece lands at lds_addr + 16 x. The compiler does not
// know of these loads; whoever reads the bytes waits for them with wait_loads (they finish in the order of issue, stores
// among them) and a barrier. The s_nop is the wait state that the instruction
// needs behind a scalar write of m0; the compiler puts none into inline assembly.
__device__ inline void load_to_lds(const void* base, unsigned off, unsigned lds_addr) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(off), "s"(base), "s"(lds_addr) : "memory", "m0");
}
template <int N>
__device__ inline void wait_loads() {
  asm volatile("s_waitcnt vmcnt(%0)" : : "n"(N < 63 ? N : 63) : "memory");
}
__device__ inline void barrier() {
  asm volatile("s_barrier" : : : "memory");
}

enum Out { kF32Out = 0, kGated = 1, kPaged = 2 };

struct TileShape {
  int M, N, K, kper;  // kper: k of a part, a multiple of 64
  int mt, nt, parts;  // tiles along m and n, parts of k
  int ldo, up;        // length of a row of the results, rows of W from a feature's gate to its up row
  size_t plane;       // results of a part of k
  const int* groups;  // kPaged: of every 32 rows the request's row of the block table, its first and its last position
  const int* table;
  int table_stride, page_size;
};

template <int BM, int BN, int WM, int WN, int S, int OUT, int OCC>
__global__ __launch_bounds__(64 * WM * WN, OCC) void gemm_tile_kernel(const bf16* __restrict__ X, long ldx,
                                                                      const bf16* __restrict__ W, long ldw,
                                                                      void* __restrict__ out, TileShape sh, GateShape act) {
  constexpr int NW = WM * WN, STAGE = (BM + BN) * ROW;
  constexpr int LX = BM / 8 / NW, LW = BN / 8 / NW, L = LX + LW;      // loads (of eight rows) of a wave and stage
  constexpr int CT = BM / WM / 32, RT = BN / WN / 32;                 // tiles of 32 rows of X and of W of a wave
  constexpr int STORES = CT * (OUT == kGated ? (RT + 3) / 4 : OUT == kPaged ? (RT + 1) / 2 : RT) * 4;  // stores of a wave for a whole tile
  constexpr int MF = RT * CT, RD = RT + CT;
  static_assert(BM % (8 * NW) == 0 && BN % (8 * NW) == 0 && (OUT != kGated || RT % 2 == 0), "rows divide over the waves");
  __shared__ __attribute__((aligned(1024))) unsigned char lds[S * STAGE + NW * 4096];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int c = lane & 31, half = lane >> 5, wm = wave % WM, wn = wave / WM;
  const int inter = sh.N / 2;

  // This die's run of the tiles (blocks are dealt to the eight dies in turn), of which this block takes every step'th.
  const int tiles = sh.mt * sh.nt * sh.parts, die = blockIdx.x & 7;
  const int share = tiles >> 3, rest = tiles & 7;
  const int begin = die * share + min(die, rest), end = begin + share + (die < rest ? 1 : 0);
  const int step = (gridDim.x - die + 7) >> 3;
  int t = begin + (blockIdx.x >> 3);
  if (t >= end) return;

  const unsigned lds_base = __builtin_amdgcn_readfirstlane(static_cast<unsigned>(reinterpret_cast<uintptr_t>(lds)));
  const int lrow = lane >> 3, lpiece = lane & 7;
  unsigned offx[LX], offw[LW];
  const char *xb, *wb;
  int im, in, ks, stages;
  auto place = [&](int tile) {
    const int per = sh.mt * sh.nt;
    ks = tile / per;
    tile -= ks * per;
    const int group = tile / (GROUP * sh.nt), first = group * GROUP, gm = min(GROUP, sh.mt - first);
    tile -= GROUP * sh.nt * group;
    im = first + tile % gm;
    in = tile / gm;
    const int kbeg = ks * sh.kper;
    stages = (min(sh.K, kbeg + sh.kper) - kbeg) / BK;
    // Rows past the end are the last row once more; nobody stores what comes of them.
#pragma unroll
    for (int i = 0; i < LX; ++i) {
      const int row = 8 * (NW * i + wave) + lrow;
      int at = min(im * BM + row, sh.M - 1);
      if (OUT == kPaged) {  // (positions behind the request's last one are the last one once more)
        const int* const group = sh.groups + 3 * (at / 32);
        const int pos = min(group[1] + at % 32, group[2]);
        at = max(sh.table[static_cast<size_t>(group[0]) * sh.table_stride + pos / sh.page_size], 0) * sh.page_size + pos % sh.page_size;
      }
      offx[i] = static_cast<unsigned>(at) * static_cast<unsigned>(2 * ldx) + 16 * (lpiece ^ ((row >> 1) & 7));
    }
#pragma unroll
    for (int i = 0; i < LW; ++i) {
      const int row = 8 * (NW * i + wave) + lrow;
      int n;
      if (OUT == kGated) {  // 32 gate rows, then the up rows of the same features
        const int f = in * (BN / 2) + 32 * (row >> 6) + (row & 31);
        n = min(f, inter - 1) + ((row >> 5) & 1) * sh.up;
      } else {
        n = min(in * BN + row, sh.N - 1);
      }
      offw[i] = static_cast<unsigned>(n) * static_cast<unsigned>(2 * ldw) + 16 * (lpiece ^ ((row >> 1) & 7));
    }
    xb = reinterpret_cast<const char*>(X + kbeg);
    wb = reinterpret_cast<const char*>(W + kbeg);
  };
  auto issue = [&](int i, unsigned slot_base) {
    if (i < LX) load_to_lds(xb, offx[i < LX ? i : 0], slot_base + (NW * i + wave) * 1024);
    else load_to_lds(wb, offw[i < LX ? 0 : i - LX], slot_base + BM * ROW + (NW * (i - LX) + wave) * 1024);
  };
  auto begin_tile = [&]() {
#pragma unroll
    for (int s = 0; s < S; ++s) {
      if (s < stages) {
#pragma unroll
        for (int i = 0; i < L; ++i) issue(i, lds_base + s * STAGE);
        xb += ROW;
        wb += ROW;
      }
    }
  };

  const unsigned char* const xrow = lds + (wm * 32 * CT + c) * ROW;
  const unsigned char* const wrow = lds + BM * ROW + (wn * 32 * RT + c) * ROW;
  const int swz = (c >> 1) & 7;
  bf16x8 a[2][RT], b[2][CT];
  auto read = [&](int x, int kk, int buf, int slot) {
    const int at = slot * STAGE + 16 * ((2 * kk + half) ^ swz);
    if (x < RT) a[buf][x < RT ? x : 0] = *reinterpret_cast<const bf16x8*>(wrow + at + x * 32 * ROW);
    else b[buf][x < RT ? 0 : x - RT] = *reinterpret_cast<const bf16x8*>(xrow + at + (x - RT) * 32 * ROW);
  };

  place(t);
  begin_tile();
  bool stored = false;  // STORES stores of every wave came after the first S stages' loads
  while (true) {
    if (stages < S) wait_loads<0>();
    else if (stored) wait_loads<(S - 1) * L + STORES>();
    else wait_loads<(S - 1) * L>();
    barrier();
#pragma unroll
    for (int x = 0; x < RD; ++x) read(x, 0, 0, 0);
    f32x16 acc[RT][CT];
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
      for (int q = 0; q < CT; ++q)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[r][q][i] = 0.f;

    int slot = 0;
    for (int st = 0; st < stages; ++st) {
      const int next = slot + 1 == S ? 0 : slot + 1;
#pragma unroll
      for (int kk = 0; kk < BK / 16; ++kk) {
        const int cur = kk & 1, nxt = cur ^ 1;
        const bool last = kk == BK / 16 - 1;
        bool more = false;
        if (last) {
          asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");
          if (st + S > stages) wait_loads<0>();
          else if (stored && st < S - 1) wait_loads<(S - 2) * L + STORES>();
          else wait_loads<(S - 2) * L>();
          barrier();
          more = st + S < stages;
        }
#pragma unroll
        for (int g = 0; g < MF; ++g) {
#pragma unroll
          for (int x = 0; x < RD; ++x)
            if ((RD > MF ? x * MF / RD : x) == g) read(x, last ? 0 : kk + 1, nxt, last ? next : slot);
          acc[g / CT][g % CT] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[cur][g / CT], b[cur][g % CT], acc[g / CT][g % CT], 0, 0, 0);
          __builtin_amdgcn_sched_barrier(0);
          if (last && more) {
#pragma unroll
            for (int i = 0; i < L; ++i)
              if (i * MF / L == g) issue(i, lds_base + slot * STAGE);
          }
        }
        if (last && more) {
          xb += ROW;
          wb += ROW;
        }
      }
      slot = next;
    }

    // The next tile's first loads, then this one's results. Everybody has read every slot for the last time; what the
    // last step read ahead is not used.
    const int m0 = im * BM, n0 = in * BN, part = ks, fcol = in * (BN / 2);
    t += step;
    const bool again = t < end;
    if (again) {
      place(t);
      begin_tile();
    }
    stored = m0 + BM <= sh.M && (OUT == kGated ? fcol + BN / 2 <= inter : n0 + BN <= sh.N);
    // acc[r][q][4 p + j]: row 32 (RT wn + r) + 8 p + 4 half + j of the tile of W, row 32 (CT wm + q) + c of X. A piece of
    // 32 rows of 128 bytes at a time goes to the wave's LDS, its 16-byte parts exchanged by the row's number, and from
    // there eight lanes to a row to memory.
    unsigned char* const own = lds + S * STAGE + wave * 4096;
#pragma unroll
    for (int q = 0; q < CT; ++q)
#pragma unroll
      for (int r = 0; r < RT; r += OUT == kF32Out ? 1 : 2) {
        if (OUT == kGated && r % 4 == 2) continue;  // written with the pair before it
        asm volatile("" : : : "memory");
        if (OUT == kGated) {
          auto finish = [&](auto silu_) {
            constexpr bool silu = decltype(silu_)::value;
#pragma unroll
            for (int pair = 0; pair < 2; ++pair) {
              const int g = r + 2 * pair;
              if (g >= RT) continue;
#pragma unroll
              for (int p = 0; p < 4; ++p) {
                float y[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                  const float gate = acc[g < RT ? g : 0][q][4 * p + j], up = acc[g + 1 < RT ? g + 1 : 0][q][4 * p + j];
                  y[j] = silu ? silu_unit(gate, up) : gated_unit(gate, up, act);
                }
                *reinterpret_cast<uint2*>(own + c * 128 + 16 * ((4 * pair + p) ^ (c & 7)) + 8 * half) =
                    uint2{pack_bf16x2(y[0], y[1]), pack_bf16x2(y[2], y[3])};
              }
            }
          };
          if (is_silu(act)) finish(std::true_type{});
          else finish(std::false_type{});
        } else if (OUT == kPaged) {
#pragma unroll
          for (int pair = 0; pair < 2; ++pair) {
            if (r + pair >= RT) continue;
            const f32x16& t = acc[r + pair < RT ? r + pair : 0][q];
#pragma unroll
            for (int p = 0; p < 4; ++p)
              *reinterpret_cast<uint2*>(own + c * 128 + 16 * ((4 * pair + p) ^ (c & 7)) + 8 * half) =
                  uint2{pack_bf16x2(t[4 * p], t[4 * p + 1]), pack_bf16x2(t[4 * p + 2], t[4 * p + 3])};
          }
        } else {
#pragma unroll
          for (int p = 0; p < 4; ++p)
            *reinterpret_cast<f32x4*>(own + c * 128 + 16 * ((2 * p + half) ^ (c & 7))) =
                f32x4{acc[r][q][4 * p], acc[r][q][4 * p + 1], acc[r][q][4 * p + 2], acc[r][q][4 * p + 3]};
        }
        asm volatile("" : : : "memory");
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int row = 8 * i + lrow, m = m0 + 32 * (wm * CT + q) + row;
          const uint4 y = *reinterpret_cast<const uint4*>(own + row * 128 + 16 * (lpiece ^ (row & 7)));
          if (OUT == kGated) {
            const int f = fcol + 16 * (wn * RT + r) + 8 * lpiece;
            if (!stored && (m >= sh.M || f >= inter)) continue;
            if (RT - r < 4 && lpiece >= 4) continue;  // a lone pair of tiles: half a row
            *reinterpret_cast<uint4*>(static_cast<bf16*>(out) + static_cast<size_t>(m) * sh.ldo + f) = y;
          } else if (OUT == kPaged) {
            const int n = n0 + 32 * (wn * RT + r) + 8 * lpiece;
            if (!stored && (m >= sh.M || n >= sh.N)) continue;
            if (RT - r < 2 && lpiece >= 4) continue;  // a lone tile: half a row
            *reinterpret_cast<uint4*>(static_cast<bf16*>(out) + n / sh.ldo * sh.plane + static_cast<size_t>(m) * sh.ldo + n % sh.ldo) = y;
          } else {
            const int n = n0 + 32 * (wn * RT + r) + 4 * lpiece;
            if (!stored && (m >= sh.M || n >= sh.N)) continue;
            *reinterpret_cast<uint4*>(static_cast<float*>(out) + part * sh.plane + static_cast<size_t>(m) * sh.ldo + n) = y;
          }
        }
      }
    if (!again) break;
    if (!stored) wait_loads<0>();  // an edge's stores are not counted
  }
}
}  // namespace

// ---- the choice of a tile and of the parts of k

namespace {

// What a tile size takes, in microseconds: a launch, a round of blocks (one a compute unit) and a stage of its tiles, a
// megabyte of results and of weights. Fitted to 24 row counts from 72 to 3,000 on nine weights (the 1.5B and 7B shapes'
// q/k/v, attention output, gate/up and way down, and two of 8,960 x 1,536 and 5,560 x 3,584), each with 1 to 6 parts of k,
// weights from memory: 2 to 5 % off on average. What it chooses takes 1.6 % (gated: 0.7 %) longer on average than the best
// of all sizes and parts measured. Larger tiles need fewer bytes a product; smaller ones fill the last round better.
struct TileCost {
  int bm, bn;
  double launch, round, stage, out_mb, weight_mb;
};
constexpr TileCost kSums[] = {{256, 256, 0.0, 3.7, 1.217, 0.167, 0.089},
                              {256, 192, 0.6, 1.8, 1.041, 0.183, 0.107},
                              {128, 192, 2.0, 2.1, 0.605, 0.180, 0.057},
                              {128, 128, 1.9, 1.3, 0.471, 0.194, 0.057},
                              {64, 128, 2.3, 1.5, 0.360, 0.168, 0.058}};
constexpr TileCost kUnits[] = {{256, 256, 3.1, 0.0, 1.471, 0.291, 0.000},
                               {192, 256, 5.0, 0.0, 1.219, 0.246, 0.033},
                               {192, 192, 3.8, 1.5, 1.015, 0.400, 0.035},
                               {128, 256, 3.9, 0.0, 0.903, 0.430, 0.018},
                               {96, 256, 4.7, 1.1, 0.654, 0.660, 0.050},
                               {96, 192, 4.1, 0.9, 0.586, 0.768, 0.041}};
// Paged rows: the sums' times (their results are half as many bytes); the product is short in k, what counts are its rounds.
constexpr TileCost kPages[] = {kSums[0], kSums[2], kSums[3]};
constexpr int kMaxParts = 6;
constexpr double kReadMb = 0.2;              // the consumer's reading of a further part, a megabyte
// A product cut in two (see TileChoice) pays for a second launch, and full rounds run at lower clocks than a nearly empty one:
// of twenty sizes, what these sums promise came out 4.5 % lower on average, so a cut has to look that much better. One launch
// against two, us: the 7B shape's gate/up 440 -> 417 at 1,777 rows and 278 -> 259 at 1,000, its q/k/v 135 -> 127 at 4,000 and
// 353 -> 339 at 12,001, the 1.5B shape's gate/up 116 -> 108 at 2,048; not cut, the former's gate/up at 800 rows (262 against 281).
constexpr double kSecondLaunchUs = 2.0, kCutCost = 1.045;
constexpr double kMostPartsBytes = 536870912.0;  // parts of k together take no more scratch memory than this

// Which tiles, in how many parts of k; and, where that leaves the last round of blocks nearly empty, a cut: tiles of `cfg`
// make the first `cut` rows of X (by_rows) or of W (gated: features), which fill their rounds, tiles of `rest` the others in a
// launch of its own.
struct TileChoice {
  int cfg, parts, kper;
  double us;
  int cut, by_rows, rest;
};

// `bytes`: of a result of a part.
double tile_us(const TileCost& c, int bytes, int M, int N, int K, int kper, int parts) {
  const double units = compute_units(), rows_mb = static_cast<double>(M) * N * 1e-6;
  const double tiles = static_cast<double>((M + c.bm - 1) / c.bm) * ((N + c.bn - 1) / c.bn) * parts;
  const double rounds = static_cast<double>(static_cast<long>((tiles + units - 1) / units));
  const double out_mb = rows_mb * bytes * parts;
  return c.launch + rounds * (c.round + kper / BK * c.stage) + out_mb * c.out_mb + 2e-6 * N * static_cast<double>(K) * c.weight_mb +
         (parts - 1) * 4.0 * rows_mb * kReadMb;
}

TileChoice choose(const TileCost* costs, int n_costs, bool gated, int M, int N, int K, int only_parts) {
  const int bytes = gated ? 1 : 4;  // (a unit of two bytes is of two rows of W)
  TileChoice best{0, 1, K, 1e30, 0, 0, 0};
  const int units = compute_units();
  for (int parts = 1; parts <= (gated ? 1 : kMaxParts); ++parts) {
    if (only_parts && parts != only_parts) continue;
    const int kper = ((K + parts - 1) / parts + BK - 1) / BK * BK;
    // A part is at least 256 k, none is empty; a caller that names the number of parts has asked here before.
    if (parts > 1 && (K / parts < 256 || static_cast<long>(parts - 1) * kper >= K)) continue;
    if (parts > 1 && 4.0 * M * N * parts > kMostPartsBytes) continue;
    for (int i = 0; i < n_costs; ++i) {
      const TileCost& c = costs[i];
      const double us = tile_us(c, bytes, M, N, K, kper, parts);
      if (us < best.us) best = TileChoice{i, parts, kper, us, 0, 0, 0};
      const long mt = (M + c.bm - 1) / c.bm, nt = (N + c.bn - 1) / c.bn, rounds = (mt * nt * parts + units - 1) / units;
      for (long full = rounds - 1; full >= 1 && full >= rounds - 2; --full) {
        for (int by_rows = 0; by_rows < 2; ++by_rows) {
          const long cut = full * units / parts / (by_rows ? nt : mt);
          if (cut < 1 || cut >= (by_rows ? mt : nt)) continue;
          const int m1 = by_rows ? static_cast<int>(cut) * c.bm : M, n1 = by_rows ? N : static_cast<int>(cut) * c.bn;
          const int m2 = by_rows ? M - m1 : M, n2 = by_rows ? N : N - n1;
          const double first = kCutCost * (tile_us(c, bytes, m1, n1, K, kper, parts) + kSecondLaunchUs);
          if (first >= best.us) continue;
          for (int j = 0; j < n_costs; ++j) {
            const double both = first + kCutCost * tile_us(costs[j], bytes, m2, n2, K, kper, parts);
            if (both < best.us) best = TileChoice{i, parts, kper, both, by_rows ? m1 : gated ? n1 / 2 : n1, by_rows, j};
          }
        }
      }
    }
  }
  return best;
}

// Rows [m0, m0 + M) of X against rows (gated: features) [n0, n0 + N) of W, of a product of all_m x all_n.
struct Region {
  int m0, M, n0, N, all_m, all_n;
};

template <int BM, int BN, int WM, int WN, int S, int OUT, int OCC>
void launch(const bf16* X, long ldx, const bf16* W, long ldw, void* out, const Region& r, int K, int kper, int parts, GateShape act,
            hipStream_t stream) {
  const bool gated = OUT == kGated;
  const int rows = gated ? 2 * r.N : r.N;  // of W
  const TileShape sh{r.M, rows, K, kper, (r.M + BM - 1) / BM, (rows + BN - 1) / BN, parts, r.all_n, r.all_n,
                     static_cast<size_t>(r.all_m) * r.all_n, nullptr, nullptr, 0, 0};
  const int tiles = sh.mt * sh.nt * parts;
  const size_t at = static_cast<size_t>(r.m0) * r.all_n + r.n0;
  void* to = gated ? static_cast<void*>(static_cast<bf16*>(out) + at) : static_cast<void*>(static_cast<float*>(out) + at);
  hipLaunchKernelGGL((gemm_tile_kernel<BM, BN, WM, WN, S, OUT, OCC>), dim3(tiles < compute_units() ? tiles : compute_units()),
                     dim3(64 * WM * WN), 0, stream, X + static_cast<size_t>(r.m0) * ldx, ldx, W + static_cast<size_t>(r.n0) * ldw, ldw, to,
                     sh, act);
}

// The whole product, or its two regions.
template <typename Launch>
void launch_regions(const TileChoice& c, int M, int N, const Launch& go) {
  if (!c.cut) return go(c.cfg, Region{0, M, 0, N, M, N});
  go(c.cfg, Region{0, c.by_rows ? c.cut : M, 0, c.by_rows ? N : c.cut, M, N});
  if (c.by_rows) go(c.rest, Region{c.cut, M - c.cut, 0, N, M, N});
  else go(c.rest, Region{0, M, c.cut, N - c.cut, M, N});
}

int check_tile(const char* name, const void* X, const void* W, const void* out, int M, int N, int K, long ldx, long ldw) {
  PYRE_REQUIRE(pyre_gemm_tile_supports(M, N, K, ldx, ldw),
               "%s: M=%d N=%d (a multiple of 16) K=%d (a multiple of 64) ldx=%ld ldw=%ld (multiples of 8, >= K; a matrix "
               "within 4 GiB) are not supported", name, M, N, K, ldx, ldw);
  PYRE_REQUIRE(reinterpret_cast<uintptr_t>(X) % 16 == 0 && reinterpret_cast<uintptr_t>(W) % 16 == 0 &&
                   reinterpret_cast<uintptr_t>(out) % 16 == 0, "%s: operands must lie on 16 bytes", name);
  return 0;
}

}  // namespace

extern "C" int pyre_gemm_tile_supports(int M, int N, int K, long ldx, long ldw) {
  return M >= 1 && N >= 16 && N % 16 == 0 && K >= BK && K % BK == 0 && ldx >= K && ldx % 8 == 0 && ldw >= K && ldw % 8 == 0 &&
         2 * ldx * M < (1L << 32) && 2 * ldw * N < (1L << 32) &&
         static_cast<long>((M + 63) / 64) * ((N + 127) / 128) * kMaxParts < (1L << 30);
}

extern "C" int pyre_gemm_tile_parts(int M, int N, int K) {
  return choose(kSums, sizeof(kSums) / sizeof(kSums[0]), false, M, N, K, 0).parts;
}

extern "C" int pyre_gemm_tile_choice(int M, int N, int K, int gated, int parts, int* tiles) {
  const TileCost* costs = gated ? kUnits : kSums;
  const int n = gated ? sizeof(kUnits) / sizeof(kUnits[0]) : sizeof(kSums) / sizeof(kSums[0]);
  const TileChoice c = choose(costs, n, gated, M, N, K, parts);
  PYRE_REQUIRE(c.us < 1e30, "gemm_tile_choice: K=%d cannot be taken in %d parts", K, parts);
  const int says[6] = {costs[c.cfg].bm, costs[c.cfg].bn, c.cut, c.by_rows, c.cut ? costs[c.rest].bm : 0, c.cut ? costs[c.rest].bn : 0};
  for (int i = 0; i < 6; ++i) tiles[i] = says[i];
  return 0;
}

// out: float32 [parts][M][N].
extern "C" int pyre_gemm_tile_bf16(const void* X, long ldx, const void* W, long ldw, float* out, int M, int N, int K, int parts,
                                   hipStream_t stream) {
  if (int rc = check_tile("gemm_tile_bf16", X, W, out, M, N, K, ldx, ldw)) return rc;
  const TileChoice c = choose(kSums, sizeof(kSums) / sizeof(kSums[0]), false, M, N, K, parts);
  PYRE_REQUIRE(parts >= 1 && parts <= kMaxParts && c.us < 1e30, "gemm_tile_bf16: K=%d cannot be taken in %d parts", K, parts);
  const bf16* x = static_cast<const bf16*>(X);
  const bf16* w = static_cast<const bf16*>(W);
  const GateShape act{};
  launch_regions(c, M, N, [&](int cfg, const Region& r) {
    if (cfg == 0) launch<256, 256, 4, 2, 2, kF32Out, 2>(x, ldx, w, ldw, out, r, K, c.kper, parts, act, stream);
    else if (cfg == 1) launch<256, 192, 4, 2, 2, kF32Out, 2>(x, ldx, w, ldw, out, r, K, c.kper, parts, act, stream);
    else if (cfg == 2) launch<128, 192, 2, 2, 3, kF32Out, 1>(x, ldx, w, ldw, out, r, K, c.kper, parts, act, stream);
    else if (cfg == 3) launch<128, 128, 2, 4, 4, kF32Out, 2>(x, ldx, w, ldw, out, r, K, c.kper, parts, act, stream);
    else launch<64, 128, 1, 4, 6, kF32Out, 1>(x, ldx, w, ldw, out, r, K, c.kper, parts, act, stream);
  });
  return check_launch("gemm_tile_bf16");
}

// W = [gate rows; up rows] (two_i x K); out: bfloat16 [M][two_i / 2], the gated unit (see GateShape; limit 0, slope 1, shift
// 0, cubic 0: the SiLU-gate).
extern "C" int pyre_gemm_tile_glu_bf16(const void* X, long ldx, const void* W, long ldw, void* out, int M, int two_i, int K,
                                       float limit, float slope, float shift, float cubic, hipStream_t stream) {
  if (int rc = check_tile("gemm_tile_glu_bf16", X, W, out, M, two_i, K, ldx, ldw)) return rc;
  const TileChoice c = choose(kUnits, sizeof(kUnits) / sizeof(kUnits[0]), true, M, two_i, K, 0);
  const bf16* x = static_cast<const bf16*>(X);
  const bf16* w = static_cast<const bf16*>(W);
  const GateShape act{limit, slope, shift, cubic};
  launch_regions(c, M, two_i / 2, [&](int cfg, const Region& r) {
    if (cfg == 0) launch<256, 256, 4, 2, 2, kGated, 2>(x, ldx, w, ldw, out, r, K, c.kper, 1, act, stream);
    else if (cfg == 1) launch<192, 256, 2, 4, 2, kGated, 2>(x, ldx, w, ldw, out, r, K, c.kper, 1, act, stream);
    else if (cfg == 2) launch<192, 192, 2, 3, 2, kGated, 2>(x, ldx, w, ldw, out, r, K, c.kper, 1, act, stream);
    else if (cfg == 3) launch<128, 256, 2, 2, 3, kGated, 1>(x, ldx, w, ldw, out, r, K, c.kper, 1, act, stream);
    else if (cfg == 4) launch<96, 256, 1, 4, 3, kGated, 1>(x, ldx, w, ldw, out, r, K, c.kper, 1, act, stream);
    else launch<96, 192, 1, 3, 3, kGated, 1>(x, ldx, w, ldw, out, r, K, c.kper, 1, act, stream);
  });
  return check_launch("gemm_tile_glu_bf16");
}

// X [pages][1][page][row]: rows of n_groups x 32 positions (see TileShape); out: bfloat16 [N / head][32 n_groups][head].
extern "C" int pyre_gemm_tile_paged_bf16(const void* X, int pages, int page_size, int row, const int* groups, int n_groups,
                                         const int* block_table, int table_stride, const void* W, void* out, int N, int K, int head,
                                         hipStream_t stream) {
  PYRE_REQUIRE(n_groups >= 0 && n_groups < (1 << 24) && pages > 0 && page_size > 0 && table_stride > 0 && head > 0 && head % 8 == 0 && N % head == 0, "gemm_tile_paged_bf16: bad geometry");
  if (n_groups == 0) return 0;
  const int M = 32 * n_groups;
  if (int rc = check_tile("gemm_tile_paged_bf16", X, W, out, M, N, K, row, K)) return rc;
  PYRE_REQUIRE(groups && block_table && 2L * pages * page_size * row < (1L << 32), "gemm_tile_paged_bf16: a cache of %d x %d rows of %d is not within 4 GiB",
               pages, page_size, row);
  int cfg = 0;
  for (int i = 1; i < 3; ++i)
    if (tile_us(kPages[i], 2, M, N, K, K, 1) < tile_us(kPages[cfg], 2, M, N, K, K, 1)) cfg = i;
  const TileCost& c = kPages[cfg];
  const TileShape sh{M, N, K, K, (M + c.bm - 1) / c.bm, (N + c.bn - 1) / c.bn, 1, head, 0, static_cast<size_t>(M) * head, groups, block_table, table_stride, page_size};
  const int tiles = sh.mt * sh.nt, blocks = tiles < compute_units() ? tiles : compute_units();
  const auto go = [&](auto kernel, int threads) {
    hipLaunchKernelGGL(kernel, dim3(blocks), dim3(threads), 0, stream, static_cast<const bf16*>(X), static_cast<long>(row),
                       static_cast<const bf16*>(W), static_cast<long>(K), out, sh, GateShape{});
  };
  if (cfg == 0) go(gemm_tile_kernel<256, 256, 4, 2, 2, kPaged, 2>, 512);
  else if (cfg == 1) go(gemm_tile_kernel<128, 192, 2, 2, 3, kPaged, 1>, 256);
  else go(gemm_tile_kernel<128, 128, 2, 2, 4, kPaged, 1>, 256);
  return check_launch("gemm_tile_paged_bf16");
}
