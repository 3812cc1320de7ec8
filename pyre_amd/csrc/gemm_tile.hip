// out[m, n] = sum_k X[m, k] W[n, k] in bfloat16 with float32 sums, for the many rows of prompts and mixed steps
// (pyre/model.py:84-87,92-94,133-139 with a whole prompt as their rows).
//
// The product is computed transposed, out^T = W X^T, on MFMA 16x16x32: A = 16 rows of W, B = 16 rows of X, both read
// along k as they are stored. A block owns BM rows of X and BN rows of W, its WM x WN waves a part of that each; k is
// walked in stages of 64 through a ring of S slots in LDS that loads from memory fill directly, rows of 128 bytes whose
// eight 16-byte pieces are exchanged among themselves by the row's number, so that the operand reads of 16 lanes spread
// over all banks.
//
// What bounds it is the card's power: with random values the clocks fall to 1.4 to 1.9 GHz. MFMA 16x16x32 needs less of it than
// 32x32x16 (nothing but products, operands in registers: 2.0 against 1.74 PFLOP/s; operands from LDS as here 1.67 against 1.54; the
// sums have the same bits), and less when one operand stays as it is from one instruction to the next: 2 % more. What else counts
// is that the matrix cores never wait, so the loop has no branch and no case: the loads run on from a tile into the block's next one, and behind
// its last one they fetch a single line that nobody reads. 4,096 x 4,096 x 8,192 takes 184 us (205 with 32x32x16, a stage's loads
// asked for at once and waits behind conditions), the 7B shape's gate/up at 2,048 rows 408 (455), its way down 202 (226).
//
// Where LDS has room for two stages only, a wave's rows of W are two parts of RT0 and RT1 tiles of sixteen, and a stage is four
// steps: the first part against k 0..31 and 32..63 of the stage, then the second part. Every operand is in registers once, read when its
// registers are free: a slot's first part and X from the last step of the stage before to the first one of its own, its second
// part in the two steps between. Two barriers a stage, behind the first and the third step, free them one after the other for
// the loads of two stages further on, which have a stage and a half to arrive. With three slots and more (RT0 = all) a stage is
// two steps, the operands of the next one are read during the present one, and the one barrier between them, behind the slot's last
// read, frees it for the loads of S stages further on.
//
// A block takes tiles one after the other until none is left. The tiles that the 32 compute units of a die work on at a time
// are neighbours (eight tiles along m by four along n): its L2 then serves every row several times.
//
// kF32Out: float32 [ksplit][M][N], part `ks` of k; kGated: W = gate rows, then up rows; bfloat16 [M][N / 2], the gated
// unit of the two; kPaged: X's rows lie in the pages of a cache, 32 consecutive positions of a request at a time; bfloat16 [N / ldo][M][ldo].
// Results pass through four kilobytes of LDS of the wave's own, so that a store writes whole lines: a
// lane's own four elements are 8 or 16 bytes of a row, and 32 rows of such pieces to a store make the L2's rate of
// requests the limit.
#include "pyre_api.h"
#include "pyre_common.h"

#include <algorithm>
#include <type_traits>

using namespace pyre;

namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
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

// Waits for the wave's reads from LDS and for all but its last N loads and stores (Many while `behind` counts down), then for the block.
template <int N, int Many>
__device__ inline void sync(int& behind) {
  asm volatile("s_cmp_gt_i32 %0, 0\n\ts_cbranch_scc1 1f\n\ts_waitcnt vmcnt(%1)\n1:\n\ts_waitcnt vmcnt(%2) lgkmcnt(0)\n\ts_barrier"
               : : "s"(behind), "n"(N), "n"(Many) : "memory", "scc");
  behind = __builtin_amdgcn_readfirstlane(max(behind - 1, 0));
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

template <int BM, int BN, int WM, int WN, int S, int OUT, int OCC, int RT0 = BN / WN / 16>
__global__ __launch_bounds__(64 * WM * WN, OCC) void gemm_tile_kernel(const bf16* __restrict__ X, long ldx, const bf16* __restrict__ W, long ldw,
                                                                      void* __restrict__ out, TileShape sh, GateShape act) {
  constexpr int NW = WM * WN, STAGE = (BM + BN) * ROW;
  constexpr int RT = BN / WN / 16, CT = BM / WM / 16, RT1 = RT - RT0;  // tiles of 16 rows of W and of X of a wave
  constexpr int LX = (BM / 8 + NW - 1) / NW, LA = 2 * WN * RT0 / NW, LB = 2 * WN * RT1 / NW;  // loads (of eight rows) of a wave: X, W's parts
  constexpr int EARLY = LX + LA, L = EARLY + LB;
  constexpr bool two = RT1 > 0;
  constexpr int STORES = CT * 2 * (OUT == kF32Out ? RT / 2 : OUT == kGated ? (RT + 7) / 8 : (RT + 3) / 4);
  static_assert(BM % (16 * WM) == 0 && BN % (16 * WN) == 0 && 2 * WN * RT0 % NW == 0 && 2 * WN * RT1 % NW == 0 && RT % 2 == 0 &&
                    (two ? L : (S - 2) * L) + STORES < 64 && (S - 1) * L + LB < 64, "rows divide over the waves, waits can be counted");
  static_assert(RT0 * CT >= RT0 + CT && (!two || (S == 2 && RT1 * CT >= RT0 + CT && RT0 * CT >= RT1)),
                "a step has a product for every operand that is read during it");
  __shared__ __attribute__((aligned(1024))) unsigned char lds[S * STAGE + NW * 4096];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int c = lane & 15, quad = lane >> 4, wm = wave % WM, wn = wave / WM;
  const int inter = sh.N / 2;

  const int tiles = sh.mt * sh.nt * sh.parts, die = blockIdx.x & 7;
  const int share = tiles >> 3, rest = tiles & 7;
  const int begin = die * share + min(die, rest), end = begin + share + (die < rest ? 1 : 0);
  const int step = (gridDim.x - die + 7) >> 3;
  int t = begin + (blockIdx.x >> 3);
  if (t >= end) return;

  const unsigned lds_base = __builtin_amdgcn_readfirstlane(static_cast<unsigned>(reinterpret_cast<uintptr_t>(lds)));
  const int lrow = lane >> 3, lpiece = lane & 7;

  struct At { int im, in, ks, stages; };
  auto locate = [&](int tile) {
    const int per = sh.mt * sh.nt, ks = tile / per;
    tile -= ks * per;
    const int group = tile / (GROUP * sh.nt), first = group * GROUP, gm = min(GROUP, sh.mt - first);
    tile -= GROUP * sh.nt * group;
    return At{first + tile % gm, tile / gm, ks, (min(sh.K, (ks + 1) * sh.kper) - ks * sh.kper) / BK};
  };
  unsigned offx[LX], offw[LA + LB];
  const char *xb, *wb;
  int coming = t, left;  // the tile whose stages are being asked for, and how many of them are left
  auto place = [&](int tile) {
    const At at_tile = locate(tile);
    left = at_tile.stages;
    // Rows past the end are the last row once more; nobody stores what comes of them.
#pragma unroll
    for (int i = 0; i < LX; ++i) {
      const int row = 8 * ((NW * i + wave) % (BM / 8)) + lrow;  // (where they do not divide, some are asked for twice)
      int at = min(at_tile.im * BM + row, sh.M - 1);
      if (OUT == kPaged) {  // (positions behind the request's last one are the last one once more)
        const int* const group = sh.groups + 3 * (at / 32);
        const int pos = min(group[1] + at % 32, group[2]);
        at = max(sh.table[static_cast<size_t>(group[0]) * sh.table_stride + pos / sh.page_size], 0) * sh.page_size + pos % sh.page_size;
      }
      offx[i] = static_cast<unsigned>(at) * static_cast<unsigned>(2 * ldx) + 16 * (lpiece ^ ((row >> 1) & 7));
    }
#pragma unroll
    for (int i = 0; i < LA + LB; ++i) {
      const int lines = i < LA ? 16 * RT0 : 16 * RT1, at = 8 * (NW * (i < LA ? i : i - LA) + wave) + lrow;  // of a wave's part; in the part
      const int row = at / lines * 16 * RT + (i < LA ? 0 : 16 * RT0) + at % lines;
      int n;
      if (OUT == kGated) {  // 16 gate rows, then the up rows of the same features
        const int f = at_tile.in * (BN / 2) + 16 * (row >> 5) + (row & 15);
        n = min(f, inter - 1) + ((row >> 4) & 1) * sh.up;
      } else {
        n = min(at_tile.in * BN + row, sh.N - 1);
      }
      offw[i] = static_cast<unsigned>(n) * static_cast<unsigned>(2 * ldw) + 16 * (lpiece ^ ((at >> 1) & 7));
    }
    xb = reinterpret_cast<const char*>(X + at_tile.ks * sh.kper);
    wb = reinterpret_cast<const char*>(W + at_tile.ks * sh.kper);
  };
  // A slot: W's first parts of all waves, their second parts, X.
  auto issue = [&](int i, unsigned slot_base) {
    if (i < LA) load_to_lds(wb, offw[i < LA ? i : 0], slot_base + (NW * i + wave) * 1024);
    else if (i < EARLY) load_to_lds(xb, offx[i < LA || i >= EARLY ? 0 : i - LA], slot_base + BN * ROW + (NW * (i - LA) + wave) % (BM / 8) * 1024);
    else load_to_lds(wb, offw[i < EARLY ? 0 : i - LX], slot_base + WN * RT0 * 16 * ROW + (NW * (i - EARLY) + wave) * 1024);
  };
  // On to the next stage to be asked for. Behind the last one of all it is that one again: what a slot holds then is not read,
  // and every stage has the same loads before and behind it.
  int advance = ROW;
  auto dry = [&]() {
    if (advance) xb -= ROW, wb -= ROW;
    advance = 0;
    left = 1;
#pragma unroll
    for (int i = 0; i < LX; ++i) offx[i] = 0;
#pragma unroll
    for (int i = 0; i < LA + LB; ++i) offw[i] = 0;
  };
  auto next_stage = [&]() {
    if (left == 0) {
      if (coming + step < end) place(coming += step);
      else dry();
    }
    --left;
  };

  const int piece = 16 * (quad ^ ((c >> 1) & 7));
  const unsigned char* const row0 = lds + (wn * RT0 * 16 + c) * ROW;
  const unsigned char* const row1 = lds + (WN * RT0 + wn * RT1) * 16 * ROW + c * ROW;
  const unsigned char* const rowx = lds + BN * ROW + (wm * CT * 16 + c) * ROW;
  bf16x8 a0[2][RT0], a1[2][two ? RT1 : 1], b[2][CT];
  auto get = [&](const unsigned char* row, int x, int kk, int slot) {
    return *reinterpret_cast<const bf16x8*>(row + (piece ^ (64 * kk)) + slot * STAGE + x * 16 * ROW);
  };
  auto read0 = [&](int x, int kk, int slot) {  // of the first part and X
    if (x < RT0) a0[kk][x < RT0 ? x : 0] = get(row0, x, kk, slot);
    else b[kk][x < RT0 ? 0 : x - RT0] = get(rowx, x - RT0, kk, slot);
  };

  place(t);
#pragma unroll
  for (int x = 0; x < S; ++x) {
    next_stage();
#pragma unroll
    for (int i = 0; i < L; ++i) issue(i, lds_base + x * STAGE);
    xb += advance, wb += advance;
  }
  wait_loads<LB + (S - 1) * L>();
  barrier();
  int behind = 0;  // of the next waits, so many have the stores of the tile before behind their loads
  int slot = 0;
  while (true) {
    const At here = locate(t);
#pragma unroll
    for (int x = 0; x < RT0 + CT; ++x) read0(x, 0, slot);
    f32x4 acc[RT][CT];
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
      for (int q = 0; q < CT; ++q) acc[r][q] = f32x4{0.f, 0.f, 0.f, 0.f};

#pragma nounroll
    for (int st = 0; st < here.stages; ++st) {
      const int next = slot + 1 == S ? 0 : slot + 1;
      // Every other row of W takes X from the other end: an operand less that changes.
      if constexpr (two) {
#pragma unroll
        for (int g = 0; g < RT0 * CT; ++g) {
          const int r = g / CT, q = r & 1 ? CT - 1 - g % CT : g % CT;
          acc[r][q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0[0][r], b[0][q], acc[r][q], 0, 0, 0);
          __builtin_amdgcn_sched_barrier(0);
          if (g < RT0 + CT) read0(g, 1, slot);
        }
        sync<L, L + STORES>(behind);
        next_stage();
#pragma unroll
        for (int g = 0; g < RT0 * CT; ++g) {
          const int r = g / CT, q = r & 1 ? CT - 1 - g % CT : g % CT;
          acc[r][q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0[1][r], b[1][q], acc[r][q], 0, 0, 0);
          __builtin_amdgcn_sched_barrier(0);
          if (g < RT1) a1[0][g < RT1 ? g : 0] = get(row1, g, 0, slot);
#pragma unroll
          for (int i = 0; i < EARLY / 2; ++i)
            if ((i + 1) * RT0 * CT / (EARLY / 2 + 1) == g) issue(i, lds_base + slot * STAGE);
        }
#pragma unroll
        for (int g = 0; g < RT1 * CT; ++g) {
          const int r = g / CT, q = r & 1 ? CT - 1 - g % CT : g % CT;
          acc[RT0 + r][q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1[0][r], b[0][q], acc[RT0 + r][q], 0, 0, 0);
          __builtin_amdgcn_sched_barrier(0);
          if (g < RT1) a1[1][g < RT1 ? g : 0] = get(row1, g, 1, slot);
#pragma unroll
          for (int i = EARLY / 2; i < EARLY; ++i)
            if ((i - EARLY / 2 + 1) * RT1 * CT / (EARLY - EARLY / 2 + 1) == g) issue(i, lds_base + slot * STAGE);
        }
        sync<L, L + STORES>(behind);
#pragma unroll
        for (int g = 0; g < RT1 * CT; ++g) {
          const int r = g / CT, q = r & 1 ? CT - 1 - g % CT : g % CT;
          acc[RT0 + r][q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1[1][r], b[1][q], acc[RT0 + r][q], 0, 0, 0);
          __builtin_amdgcn_sched_barrier(0);
          if (g < RT0 + CT) read0(g, 0, next);
#pragma unroll
          for (int i = EARLY; i < L; ++i)
            if ((i - EARLY + 1) * RT1 * CT / (LB + 1) == g) issue(i, lds_base + slot * STAGE);
        }
      } else {
#pragma unroll
        for (int g = 0; g < RT * CT; ++g) {
          const int r = g / CT, q = r & 1 ? CT - 1 - g % CT : g % CT;
          acc[r][q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0[0][r], b[0][q], acc[r][q], 0, 0, 0);
          __builtin_amdgcn_sched_barrier(0);
          if (g < RT + CT) read0(g, 1, slot);
        }
        sync<(S - 2) * L, (S - 2) * L + STORES>(behind);
        next_stage();
#pragma unroll
        for (int g = 0; g < RT * CT; ++g) {
          const int r = g / CT, q = r & 1 ? CT - 1 - g % CT : g % CT;
          acc[r][q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0[1][r], b[1][q], acc[r][q], 0, 0, 0);
          __builtin_amdgcn_sched_barrier(0);
          if (g < RT + CT) read0(g, 0, next);
#pragma unroll
          for (int i = 0; i < L; ++i)
            if (i * RT * CT / L == g) issue(i, lds_base + slot * STAGE);
        }
      }
      xb += advance, wb += advance;
      slot = next;
    }

    // (What the last step read ahead is read again.)
    const int m0 = here.im * BM, n0 = here.in * BN, part = here.ks, fcol = here.in * (BN / 2);
    t += step;
    const bool again = t < end;
    const bool stored = m0 + BM <= sh.M && (OUT == kGated ? fcol + BN / 2 <= inter : n0 + BN <= sh.N);  // STORES stores a wave
    // acc[r][q][j]: row 16 (RT wn + r) + 4 quad + j of the tile of W, row 16 (CT wm + q) + c of X. A piece of
    // 32 rows of 128 bytes at a time goes to the wave's LDS, its 16-byte parts exchanged by the row's number, and from
    // there eight lanes to a row to memory.
    unsigned char* const own = lds + S * STAGE + wave * 4096;
    constexpr int WIDE = OUT == kF32Out ? 2 : OUT == kGated ? 8 : 4;  // tiles of W that make a piece
#pragma unroll
    for (int q = 0; q < CT; q += 2)
#pragma unroll
      for (int r = 0; r < RT; r += WIDE) {
        asm volatile("" : : : "memory");
#pragma unroll
        for (int x = 0; x < 2; ++x) {
          if (q + x >= CT) continue;
          const int qx = q + x < CT ? q + x : 0;
          unsigned char* const line = own + (16 * x + c) * 128;
          const int swz = (c >> 1) & 7;
          if (OUT == kGated) {
            auto finish = [&](auto silu_) {
              constexpr bool silu = decltype(silu_)::value;
#pragma unroll
              for (int u = 0; u < 4; ++u) {
                const int g = r + 2 * u;
                if (g >= RT) continue;
                float y[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                  const float gate = acc[g < RT ? g : 0][qx][j], up = acc[g + 1 < RT ? g + 1 : 0][qx][j];
                  y[j] = silu ? silu_unit(gate, up) : gated_unit(gate, up, act);
                }
                *reinterpret_cast<uint2*>(line + 16 * ((2 * u + (quad >> 1)) ^ swz) + 8 * (quad & 1)) =
                    uint2{pack_bf16x2(y[0], y[1]), pack_bf16x2(y[2], y[3])};
              }
            };
            if (is_silu(act)) finish(std::true_type{});
            else finish(std::false_type{});
          } else if (OUT == kPaged) {
#pragma unroll
            for (int u = 0; u < 4; ++u) {
              if (r + u >= RT) continue;
              const f32x4& y = acc[r + u < RT ? r + u : 0][qx];
              *reinterpret_cast<uint2*>(line + 16 * ((2 * u + (quad >> 1)) ^ swz) + 8 * (quad & 1)) = uint2{pack_bf16x2(y[0], y[1]), pack_bf16x2(y[2], y[3])};
            }
          } else {
#pragma unroll
            for (int u = 0; u < 2; ++u) *reinterpret_cast<f32x4*>(line + 16 * ((4 * u + quad) ^ swz)) = acc[r + u][qx];
          }
        }
        asm volatile("" : : : "memory");
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if (q + 1 >= CT && i >= 2) continue;  // sixteen rows are left
          const int row = 8 * i + lrow, m = m0 + 16 * (wm * CT + q) + row;
          const uint4 y = *reinterpret_cast<const uint4*>(own + row * 128 + 16 * (lpiece ^ ((row >> 1) & 7)));
          if (OUT == kGated) {
            const int f = fcol + 8 * (wn * RT + r) + 8 * lpiece;
            if (!stored && (m >= sh.M || f >= inter)) continue;
            if (lpiece >= RT - r) continue;  // a part of a row
            *reinterpret_cast<uint4*>(static_cast<bf16*>(out) + static_cast<size_t>(m) * sh.ldo + f) = y;
          } else if (OUT == kPaged) {
            const int n = n0 + 16 * (wn * RT + r) + 8 * lpiece;
            if (!stored && (m >= sh.M || n >= sh.N)) continue;
            if (RT - r < 4 && lpiece >= 4) continue;  // half a row
            *reinterpret_cast<uint4*>(static_cast<bf16*>(out) + n / sh.ldo * sh.plane + static_cast<size_t>(m) * sh.ldo + n % sh.ldo) = y;
          } else {
            const int n = n0 + 16 * (wn * RT + r) + 4 * lpiece;
            if (!stored && (m >= sh.M || n >= sh.N)) continue;
            *reinterpret_cast<uint4*>(static_cast<float*>(out) + part * sh.plane + static_cast<size_t>(m) * sh.ldo + n) = y;
          }
        }
      }
    if (!again) {
      wait_loads<0>();  // (nothing is to arrive in LDS that is another block's by then)
      break;
    }
    behind = __builtin_amdgcn_readfirstlane(stored ? (two ? 3 : S - 1) : 0);
    if (!stored) wait_loads<0>();  // an edge's stores are not counted
  }
}
}  // namespace

// ---- the choice of a tile and of the parts of k

namespace {

// What a tile size takes, in microseconds: a launch, a round of blocks (one a compute unit), a stage of its tiles, the same again
// where every unit has a tile (the card's power then leaves lower clocks), a megabyte of results and of weights. Fitted to 25 row
// counts from 72 to 3,000 on nineteen weights (the 1.5B and 7B shapes' q/k/v, attention output, gate/up and way down, and others of
// 64 to 1,536 k), each with 1 to 6 parts of k, weights from memory and launches one behind the other: 2 to 7 % off
// on average. What it chooses takes 0.9 % (gated: 0.2 %) longer on average than the best of all sizes and parts measured. Larger
// tiles need fewer bytes a product; smaller ones fill the last round better. A product cut in two (see TileChoice) is two of these
// times: over 39 row counts from 257 to 12,001 on nine weights the cuts so chosen save 0.7 % on average, 1.4 % on the 7B shape's.
struct TileCost {
  int bm, bn;
  double launch, round, stage, full, out_mb, weight_mb;
};
constexpr TileCost kSums[] = {{256, 256, 1.4, 5.0, 0.947, 0.360, 0.095, 0.015},
                              {256, 192, 1.9, 3.8, 0.743, 0.301, 0.095, 0.006},
                              {128, 192, 2.5, 2.0, 0.392, 0.251, 0.104, 0.065},
                              {128, 128, 2.8, 1.4, 0.290, 0.209, 0.086, 0.053},
                              {64, 128, 2.9, 1.0, 0.235, 0.111, 0.065, 0.049}};
constexpr TileCost kUnits[] = {{256, 256, 3.4, 2.8, 0.871, 0.499, 0.093, 0.028},
                               {192, 256, 3.2, 2.6, 0.630, 0.446, 0.081, 0.047},
                               {192, 192, 3.1, 2.6, 0.680, 0.256, 0.093, 0.029},
                               {128, 256, 2.8, 2.1, 0.438, 0.339, 0.065, 0.085},
                               {96, 256, 2.9, 1.8, 0.319, 0.377, 0.051, 0.096},
                               {96, 192, 3.0, 1.7, 0.251, 0.306, 0.042, 0.077}};
// Paged rows: the sums' times (their results are half as many bytes); the product is short in k, what counts are its rounds.
constexpr TileCost kPages[] = {kSums[0], kSums[2], kSums[3]};
constexpr int kMaxParts = 6;
constexpr double kReadMb = 0.2;              // the consumer's reading of a further part, a megabyte
// Megabytes a microsecond that weights come with at the most: a head's few last rows are a second pass over
// weights that no cache holds (151,936 x 1,536, 54 rows: 92 us, 70 without this; 566 rows cut behind 512 took 346 us, whole 309).
constexpr double kMbPerUs = 5.0;
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
  return c.launch + rounds * (c.round + kper / BK * c.stage) + tiles / units * (kper / BK) * c.full + out_mb * c.out_mb + 2e-6 * N * static_cast<double>(K) * c.weight_mb +
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
          const double first = tile_us(c, bytes, m1, n1, K, kper, parts);
          if (first >= best.us) continue;
          const double again = by_rows ? 2e-6 * N * static_cast<double>(K) / kMbPerUs : 0.0;
          for (int j = 0; j < n_costs; ++j) {
            const double both = first + std::max(tile_us(costs[j], bytes, m2, n2, K, kper, parts), again);
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

template <int BM, int BN, int WM, int WN, int S, int OUT, int OCC, int RT0 = BN / WN / 16>
void launch(const bf16* X, long ldx, const bf16* W, long ldw, void* out, const Region& r, int K, int kper, int parts, GateShape act,
            hipStream_t stream) {
  const bool gated = OUT == kGated;
  const int rows = gated ? 2 * r.N : r.N;  // of W
  const TileShape sh{r.M, rows, K, kper, (r.M + BM - 1) / BM, (rows + BN - 1) / BN, parts, r.all_n, r.all_n,
                     static_cast<size_t>(r.all_m) * r.all_n, nullptr, nullptr, 0, 0};
  const int tiles = sh.mt * sh.nt * parts;
  const size_t at = static_cast<size_t>(r.m0) * r.all_n + r.n0;
  void* to = gated ? static_cast<void*>(static_cast<bf16*>(out) + at) : static_cast<void*>(static_cast<float*>(out) + at);
  hipLaunchKernelGGL((gemm_tile_kernel<BM, BN, WM, WN, S, OUT, OCC, RT0>), dim3(tiles < compute_units() ? tiles : compute_units()),
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
    if (cfg == 0) launch<256, 256, 4, 2, 2, kF32Out, 2, 4>(x, ldx, w, ldw, out, r, K, c.kper, parts, act, stream);
    else if (cfg == 1) launch<256, 192, 4, 2, 2, kF32Out, 2, 2>(x, ldx, w, ldw, out, r, K, c.kper, parts, act, stream);
    else if (cfg == 2) launch<128, 192, 4, 2, 3, kF32Out, 2>(x, ldx, w, ldw, out, r, K, c.kper, parts, act, stream);
    else if (cfg == 3) launch<128, 128, 4, 2, 4, kF32Out, 2>(x, ldx, w, ldw, out, r, K, c.kper, parts, act, stream);
    else launch<64, 128, 2, 4, 5, kF32Out, 2>(x, ldx, w, ldw, out, r, K, c.kper, parts, act, stream);
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
    if (cfg == 0) launch<256, 256, 4, 2, 2, kGated, 2, 4>(x, ldx, w, ldw, out, r, K, c.kper, 1, act, stream);
    else if (cfg == 1) launch<192, 256, 2, 4, 2, kGated, 2, 2>(x, ldx, w, ldw, out, r, K, c.kper, 1, act, stream);
    else if (cfg == 2) launch<192, 192, 2, 3, 2, kGated, 2, 2>(x, ldx, w, ldw, out, r, K, c.kper, 1, act, stream);
    else if (cfg == 3) launch<128, 256, 2, 4, 2, kGated, 2, 2>(x, ldx, w, ldw, out, r, K, c.kper, 1, act, stream);
    else if (cfg == 4) launch<96, 256, 2, 4, 2, kGated, 2, 2>(x, ldx, w, ldw, out, r, K, c.kper, 1, act, stream);
    else launch<96, 192, 3, 2, 3, kGated, 2>(x, ldx, w, ldw, out, r, K, c.kper, 1, act, stream);
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
  if (cfg == 0) go(gemm_tile_kernel<256, 256, 4, 2, 2, kPaged, 2, 4>, 512);
  else if (cfg == 1) go(gemm_tile_kernel<128, 192, 4, 2, 3, kPaged, 2>, 512);
  else go(gemm_tile_kernel<128, 128, 2, 4, 4, kPaged, 2>, 512);
  return check_launch("gemm_tile_paged_bf16");
}
