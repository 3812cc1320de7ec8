// Causal (optionally windowed) attention of prompt portions over the paged cache in true
// float32 on the matrix cores (v_mfma_f32_16x16x4_f32: float32 operands, products and sums):
// the 32-bit path's attention for requests that bring more than one token. Single tokens stay
// with attention_generic.hip, whose blocks are of one token and cannot fill sixteen columns.
//
//   scores = (q k^T) * scale, masked to lo..pos       (pyre/model.py:109-120)
//   probs  = softmax(scores), out = probs v            (pyre/model.py:122-123)
//
// A tile is up to 32 consecutive tokens of one request (tiles[i] = first token in the flat
// batch, count). A wave has sixteen of them for one query head. The keys are in KS parts: of every
// KS chunks of 32, each goes to one, which has a maximum, a sum and an output of its own; the
// parts are joined at the end in their order. Two forms with the same sums, bit for bit: "wide", a block
// of sixteen tokens and two heads with a wave for every part, and "shared", a block of the whole tile and
// two heads with half as many waves for the parts, two parts a wave (see the kernel for why). What
// a block reads in a round, a chunk for each of its parts' waves, lies in LDS (K as stored, V transposed
// back: [d][key]). The transposed problem is computed on 16 x 16 x 4, so that the scores come out in the
// layout the second product wants them in:
//   S^T[key, token]  = sum_d K[key, d] Q[token, d]      A = K (LDS), B = Q^T (registers)
//   O^T[d, token]   += sum_key V^T[d, key] P^T[key, token]   A = V^T (LDS), B = P^T = the lane's
//                                                           own eight scores, one per step
// A step's four elements of the summed index are 4 g + j of sixteen (g = lane / 16), so that the
// operands of four steps are one 16-byte read; element j of a tile of scores is key 4 g + j.
// Chunks start at multiples of 32 keys and go to parts by their number, so the order of every sum
// of a token depends on its own bounds (lo, pos) alone, not on the tile it is in or on what
// else is in the step.
#include <algorithm>

#include "pyre_api.h"
#include "pyre_common.h"

using namespace pyre;

namespace {

typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef f32x4 f32x4_anywhere __attribute__((aligned(4)));
constexpr int kKeys = 32;    // keys of a chunk
constexpr int kTokens = 16;  // tokens of a wave

// HDP: the head size rounded up to a multiple of 32 (the rest is zeros). VEC (heads and pages of a multiple of four elements and
// tokens): keys and values come in 16-byte pieces, asked for while the chunks before them are multiplied, and the pages
// they lie in a round earlier still. A round is KW chunks, KW waves have the KS parts of a head and sixteen tokens, HALVES times
// sixteen tokens and HEADS heads share what the block reads.
//
// The matrix instruction has a sixteenth of the 16-bit one's rate: a chunk's 128 instructions are 1.7 us of a wave's SIMD. A step of a
// few hundred tokens is a few dozen tiles, so what counts is that they fill the chip: three prompts of 333, 206 and 27 tokens on twelve
// heads of 128 are 228 blocks of eight waves in the wide form (27 us), where 32 tokens and four heads a block made 76 of four, one wave a
// SIMD (90). Then that an instruction does not cost an LDS read of four bytes, and that the loads of a round are asked for without a
// wait between them (a branch around each made them wait for one another: 30.5 us). The root mean square distance from 64 bits is 2.9e-7
// for the three prompts (3.2e-7 with one part) and 8.7e-7 behind 6,000 tokens (15.6e-7): the parts' sums are shorter.
//
// Where tiles fill the chip by themselves, more waves for the parts only mean that every block reads more for fewer tokens, and of a tile
// that sees few keys they have nothing to do. Us a launch in 32 tokens and four heads with one part, the wide and the shared form: 120
// prompts of 16 tokens on the 7B heads 68, 139, 79, behind 120 others 191, 247, 176, in a window of 64 160, 242, 160; on fourteen heads of 64 17, 48,
// 18, 43, 81, 47, 37, 80, 41; 100 prompts of 32 tokens 88, 120, 77 and 23, 43, 22. Of a single chunk the one part is up to a quarter ahead
// still (200 prompts of two tokens 90, 203, 113), from two on the shared form is.
//
// Blocks start in the order of their tiles, all heads of the last tokens first: with the heads as the slow dimension the long
// blocks of the last head started late. Wide before, wide and shared now: 2,048 tokens of 40 heads 893, 748, 661, two prompts of 3,000 on the 7B
// heads 2,190, 2,028, 1,830, 2,048 behind 6,000 3,089, 3,019, 2,775 (47 % of the instruction's rate); two prompts of 1,000 on sixteen heads of 256 852,
// 570, 469, on five heads of 96 118, 81, 82.
//
// Registers: a wave's parts take turns in the same ones, and the barriers in the products keep the scheduler from reading far ahead; 128 for heads
// of 64 (168 and spills without), so that two blocks of eight waves share a unit.
template <int HDP, int KS, bool SHARED>
constexpr int kWavesPerSimd = HDP > 128 ? 1 : HDP > 64 || !SHARED ? 2 : 4;
template <int HDP, int KS, bool SHARED, bool VEC>
__global__ __launch_bounds__(128 * KS, (kWavesPerSimd<HDP, KS, SHARED>)) void attn_prefill_f32_kernel(
    const float* __restrict__ q, const float* __restrict__ k_cache, const float* __restrict__ v_cache,
    float* __restrict__ out, const int* __restrict__ tiles, const int* __restrict__ positions,
    const int* __restrict__ seq_of_token, const int* __restrict__ block_table, int table_stride, int nq, int nkv,
    int hd, int page_size, float scale, int window) {
  constexpr int HEADS = 2, HALVES = SHARED ? 2 : 1, KW = SHARED ? KS / 2 : KS, ACC = KS / KW;  // ACC: parts that a wave keeps
  constexpr int THREADS = 64 * HEADS * HALVES * KW, KEYS = kKeys * KW;
  constexpr int KROW = HDP + 4, VROW = kKeys + 4;  // elements of a row in LDS: sixteen rows start on all banks in turn
  constexpr int GROUPS = HEADS * HALVES, JOINED = GROUPS * KW * kTokens;  // a wave's tokens and head; rows of outputs that are joined at a time
  constexpr int KSIZE = KEYS * KROW, VSIZE = KW * HDP * VROW, JSIZE = JOINED * (KROW + 2 * ACC);
  __shared__ __attribute__((aligned(16))) float lds[KSIZE + VSIZE > JSIZE ? KSIZE + VSIZE : JSIZE];
  float* const Ks = lds;
  float* const Vt = lds + KSIZE;
  __shared__ __attribute__((aligned(16))) int pages[3][KEYS];    // of three rounds' keys; -1: not there
  // Where a key's row and its column of values start, worked out once: a piece's address is an addition.
  __shared__ __attribute__((aligned(16))) longlong2 where[3][KEYS];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, g = lane >> 4, c = lane & 15;
  const int n_rep = nq / nkv, hgroups = (n_rep + HEADS - 1) / HEADS, per_piece = hgroups * nkv;
  const int hgroup = blockIdx.x % per_piece % hgroups, kvh = blockIdx.x % per_piece / hgroups;
  const int part = wave / GROUPS, hin = hgroup * HEADS + wave % HEADS;
  const int wt = HALVES == 1 ? 0 : kTokens * (wave / HEADS % HALVES);  // the wave's first token of the block's
  const int piece = (gridDim.x - 1 - blockIdx.x) / per_piece;  // of a tile; the last tokens, which see the most keys, first
  const int tile = 2 * (HALVES == 1 ? piece >> 1 : piece), skip = HALVES == 1 ? kTokens * (piece & 1) : 0;
  const int t0 = tiles[tile] + skip, ntok = min(kTokens * HALVES, tiles[tile + 1] - skip);
  if (ntok <= 0) return;
  const bool active = hin < n_rep && wt < ntok;  // a wave without a head or tokens still helps loading
  const int head = kvh * n_rep + (hin < n_rep ? hin : 0);
  const int pos0 = positions[t0];
  const int* table = block_table + static_cast<size_t>(seq_of_token[t0]) * table_stride;

  // Column c of this wave: token t0 + c, which sees keys lo..hi. Columns past the tile's end
  // compute on zeros over the first token's keys and are not stored.
  const bool live = active && wt + c < ntok;
  const int hi = wt + c < ntok ? pos0 + wt + c : pos0;
  const int lo = window > 0 ? max(0, hi - window + 1) : 0;
  f32x4 qr[HDP / 16];  // Q[token c][d = 16 s + 4 g ..]
#pragma unroll
  for (int s = 0; s < HDP / 16; ++s) {
    const int d = 16 * s + 4 * g;
    const float* from = q + (static_cast<size_t>(t0 + wt + c) * nq + head) * hd + d;
    qr[s] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (VEC) {
      if (live && d < hd) qr[s] = *reinterpret_cast<const f32x4_anywhere*>(from);
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (live && d + j < hd) qr[s][j] = from[j];
    }
  }
  f32x4 o[ACC][HDP / 16];
  float m[ACC], l[ACC];  // l: this lane's share of the column's sum (its eight keys of every chunk)
#pragma unroll
  for (int a = 0; a < ACC; ++a) {
    m[a] = -INFINITY, l[a] = 0.f;
#pragma unroll
    for (int dt = 0; dt < HDP / 16; ++dt) o[a][dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  }

  const int lo_all = window > 0 ? max(0, pos0 - window + 1) : 0;
  const int hi_all = pos0 + ntok - 1;
  const int first_chunk = lo_all / kKeys, last_chunk = hi_all / kKeys;
  const int first = first_chunk / KW, last = last_chunk / KW;  // rounds
  // the chunks that the wave's own tokens see
  const int wave_first = HALVES == 1 ? first_chunk : (window > 0 ? max(0, pos0 + wt - window + 1) : 0) / kKeys;
  const int wave_last = HALVES == 1 ? last_chunk : min(pos0 + wt + kTokens - 1, hi_all) / kKeys;
  auto look_up = [&](int round) {  // the page of key KEYS round + tid
    const int key = KEYS * round + tid, entry = key / page_size;
    return tid < KEYS && key >= kKeys * first_chunk && key <= hi_all && entry < table_stride ? table[entry] : -1;
  };
  auto note = [&](int round, int to, int page) {
    if (tid >= KEYS) return;
    const int at = (KEYS * round + tid) % page_size;
    const long long row = (static_cast<long long>(page) * nkv + kvh) * page_size;
    pages[to][tid] = page;
    where[to][tid] = longlong2{(row + at) * hd, row * hd + at};
  };
  constexpr int PIECES = HDP / (8 * HEADS * HALVES);  // 16-byte pieces of keys, and of values, of a thread and round
  // Loads without a branch: a piece that is not there is read from the queries and becomes zeros when it is stored in LDS.
  f32x4 kp[VEC ? PIECES : 1], vp[VEC ? PIECES : 1];
  unsigned kgone = 0, vgone = 0;  // a bit a piece
  auto fetch = [&](int from) {
    kgone = vgone = 0;
#pragma unroll
    for (int i = 0; i < PIECES; ++i) {
      const int key = (tid + THREADS * i) / (HDP / 4), d = 4 * ((tid + THREADS * i) % (HDP / 4));
      const long long at = where[from][key].x;
      const bool there = at >= 0 && d < hd;
      kp[i] = *reinterpret_cast<const f32x4_anywhere*>(there ? k_cache + at + d : q);
      kgone |= there ? 0u : 1u << i;
    }
#pragma unroll
    for (int i = 0; i < PIECES; ++i) {
      const int row = (tid + THREADS * i) / 8, key = kKeys * (row / HDP) + 4 * (tid & 7), d = row % HDP;
      const long long at = where[from][key].y;
      const bool there = at >= 0 && d < hd;
      vp[i] = *reinterpret_cast<const f32x4_anywhere*>(there ? v_cache + at + d * page_size : q);
      vgone |= there ? 0u : 1u << i;
    }
  };
  auto put = [&](int round) {
    if (__ballot(kgone | vgone)) {
#pragma unroll
      for (int i = 0; i < PIECES; ++i) {
        if (kgone >> i & 1) kp[i] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (vgone >> i & 1) vp[i] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
    }
    if (KEYS * round + KEYS - 1 > hi_all) {  // behind the step's last key lies what nobody has written
#pragma unroll
      for (int i = 0; i < PIECES; ++i) {
        const int key = KEYS * round + kKeys * ((tid + THREADS * i) / 8 / HDP) + 4 * (tid & 7);
#pragma unroll
        for (int j = 1; j < 4; ++j)
          if (key + j > hi_all) vp[i][j] = 0.f;
      }
    }
#pragma unroll
    for (int i = 0; i < PIECES; ++i) {
      const int key = (tid + THREADS * i) / (HDP / 4), d = 4 * ((tid + THREADS * i) % (HDP / 4));
      *reinterpret_cast<f32x4*>(Ks + key * KROW + d) = kp[i];
    }
#pragma unroll
    for (int i = 0; i < PIECES; ++i) {
      const int row = (tid + THREADS * i) / 8;
      *reinterpret_cast<f32x4*>(Vt + row * VROW + 4 * (tid & 7)) = vp[i];
    }
  };
  const int page0 = look_up(first), page1 = look_up(first + 1);
  int ahead = look_up(first + 2);
  note(first, 0, page0);
  note(first + 1, 1, page1);
  if (VEC) {
    __syncthreads();
    fetch(0);
  }
  // A chunk of the part whose turn it is, a = 0.
  auto attend = [&](int chunk, int here) __attribute__((always_inline)) {
    f32x4 s[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int st = 0; st < HDP / 16; ++st) {
      f32x4 a[2];
#pragma unroll
      for (int kt = 0; kt < 2; ++kt) a[kt] = *reinterpret_cast<const f32x4*>(Ks + (kKeys * part + 16 * kt + c) * KROW + 16 * st + 4 * g);
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int kt = 0; kt < 2; ++kt) s[kt] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[kt][j], qr[st][j], s[kt], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
    float mx = -INFINITY;
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int kk = 16 * kt + 4 * g + j, key = kKeys * chunk + kk;
        s[kt][j] = key < lo || key > hi || pages[here][kKeys * part + kk] < 0 ? -INFINITY : s[kt][j] * scale;
        mx = fmaxf(mx, s[kt][j]);
      }
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    const float m_new = fmaxf(m[0], mx);
    const float m_use = m_new == -INFINITY ? 0.f : m_new;  // a column without a visible key so far
    const float alpha = expf(m[0] - m_use);
    m[0] = m_new;
    float sum = 0.f;
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        s[kt][j] = expf(s[kt][j] - m_use);
        sum += s[kt][j];
      }
    l[0] = l[0] * alpha + sum;
#pragma unroll
    for (int dt = 0; dt < HDP / 16; ++dt) o[0][dt] *= alpha;
    constexpr int GROUP = HDP % 64 == 0 && HDP > 64 ? 4 : 2;  // tiles of d whose chains of products are in flight together
#pragma unroll
    for (int dt = 0; dt < HDP / 16; dt += GROUP)
#pragma unroll
      for (int kt = 0; kt < 2; ++kt) {
        f32x4 a[GROUP];
#pragma unroll
        for (int t = 0; t < GROUP; ++t)
          a[t] = *reinterpret_cast<const f32x4*>(Vt + (HDP * part + 16 * (dt + t) + c) * VROW + 16 * kt + 4 * g);
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int t = 0; t < GROUP; ++t) o[0][dt + t] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[t][j], s[kt][j], o[0][dt + t], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
  };
  // The wave's other part takes the place of this one.
  auto turn = [&]() __attribute__((always_inline)) {
    if constexpr (ACC == 2) {
      const float m0 = m[0], l0 = l[0];
      m[0] = m[1], m[1] = m0, l[0] = l[1], l[1] = l0;
#pragma unroll
      for (int dt = 0; dt < HDP / 16; ++dt) {
        const f32x4 o0 = o[0][dt];
        o[0][dt] = o[1][dt], o[1][dt] = o0;
      }
    }
  };
  int slot = 0;
  for (int round = first; round <= last; ++round) {
    const int next = slot == 2 ? 0 : slot + 1;
    __syncthreads();  // the round before has been read by every wave
    note(round + 2, next == 2 ? 0 : next + 1, ahead);
    if (VEC) {
      put(round);
      __syncthreads();
      if (round < last) fetch(next);
    } else {  // eight loads on their way: 600 tokens twice, nine heads of 250, 391 us, one behind the other 433
#pragma unroll 8
      for (int i = tid; i < KEYS * HDP; i += THREADS) {  // K: d fastest, as it lies in the cache
        const int key = i / HDP, d = i % HDP;
        const long long at = where[slot][key].x;
        float v = 0.f;
        if (at >= 0 && d < hd) v = k_cache[at + d];
        Ks[key * KROW + d] = v;
      }
#pragma unroll 8
      for (int i = tid; i < KEYS * HDP; i += THREADS) {  // V: the key fastest, as the cache stores it transposed
        const int row = i / kKeys, key = i % kKeys, d = row % HDP;
        const long long at = where[slot][kKeys * (row / HDP) + key].y;
        float v = 0.f;
        if (at >= 0 && d < hd) v = v_cache[at + d * page_size];
        Vt[row * VROW + key] = v;
      }
      __syncthreads();
    }
    if (round + 2 < last) ahead = look_up(round + 3);
    const int chunk = KW * round + part, here = slot;
    slot = next;
    if (active && chunk >= wave_first && chunk <= wave_last) attend(chunk, here);
    turn();
  }
  if ((last + 1) % ACC) turn();  // o[a] is that of parts KW a .. again
#pragma unroll
  for (int a = 0; a < ACC; ++a) {
    l[a] += __shfl_xor(l[a], 16, 64);
    l[a] += __shfl_xor(l[a], 32, 64);
  }
  // The parts of a head, joined in their order, in the keys' and values' place: outputs of KW parts at a time, maxima and sums behind them.
  float* const ml = lds + JOINED * KROW;
  constexpr int UNITS = GROUPS * kTokens * (HDP / 4), ITEMS = (UNITS + THREADS - 1) / THREADS;
  f32x4 y[ITEMS];
#pragma unroll
  for (int a = 0; a < ACC; ++a) {
    __syncthreads();
#pragma unroll
    for (int dt = 0; dt < HDP / 16; ++dt)  // element j of o[a][dt]: d = 16 dt + 4 g + j of token c
      *reinterpret_cast<f32x4*>(lds + (kTokens * wave + c) * KROW + 16 * dt + 4 * g) = o[a][dt];
    if (a == 0 && g == 0) {
#pragma unroll
      for (int b = 0; b < ACC; ++b) {
        ml[2 * (JOINED * b + kTokens * wave + c)] = m[b];
        ml[2 * (JOINED * b + kTokens * wave + c) + 1] = l[b];
      }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
      const int unit = tid + THREADS * i, d = 4 * (unit % (HDP / 4)), row = unit / (HDP / 4), token = row % kTokens, group = row / kTokens;
      const int in_block = kTokens * (group / HEADS) + token, h = hgroup * HEADS + group % HEADS;
      if (unit >= UNITS || d >= hd || in_block >= ntok || h >= n_rep) continue;
      const auto place = [&](int p) { return JOINED * (p / KW) + kTokens * (GROUPS * (p % KW) + group) + token; };  // of part p's maximum and sum
      float most = -INFINITY;
#pragma unroll
      for (int p = 0; p < KS; ++p) most = fmaxf(most, ml[2 * place(p)]);
      const auto weight = [&](int p) { return ml[2 * place(p)] == -INFINITY ? 0.f : expf(ml[2 * place(p)] - most); };
      if (a == 0) y[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int w = 0; w < KW; ++w) y[i] += weight(KW * a + w) * *reinterpret_cast<const f32x4*>(lds + (kTokens * (GROUPS * w + group) + token) * KROW + d);
      if (a + 1 < ACC) continue;
      float total = 0.f;
#pragma unroll
      for (int p = 0; p < KS; ++p) total += weight(p) * ml[2 * place(p) + 1];
      y[i] *= total > 0.f ? 1.f / total : 0.f;
      float* dst = out + (static_cast<size_t>(t0 + in_block) * nq + kvh * n_rep + h) * hd + d;
      if (VEC) {
        *reinterpret_cast<f32x4_anywhere*>(dst) = y[i];
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (d + j < hd) dst[j] = y[i][j];
      }
    }
  }
}

}  // namespace

extern "C" int pyre_attn_prefill_f32(const float* q, float* out, const float* k_cache, const float* v_cache,
                                     const int* tiles, int n_tiles, const int* positions, const int* seq_of_token,
                                     const int* block_table, int table_stride, int nq, int nkv, int hd, int page_size,
                                     float scale, int window, hipStream_t stream) {
  PYRE_REQUIRE(nq > 0 && nkv > 0 && nq % nkv == 0, "attn_prefill_f32: %d query heads do not divide over %d kv heads", nq, nkv);
  PYRE_REQUIRE(hd > 0 && hd <= 256, "attn_prefill_f32: head_dim %d is outside 1..256", hd);
  PYRE_REQUIRE(page_size > 0 && table_stride > 0, "attn_prefill_f32: bad page geometry");
  if (n_tiles <= 0) return 0;
  const int hgroups = (nq / nkv + 1) / 2;
  PYRE_REQUIRE(nkv <= 65535 && hgroups <= 65535 && n_tiles < (1 << 22) && static_cast<long>(nkv) * hgroups < (1 << 22), "attn_prefill_f32: grid too large");
  const bool vec = hd % 4 == 0 && page_size % 4 == 0 && reinterpret_cast<uintptr_t>(k_cache) % 16 == 0 &&
                   reinterpret_cast<uintptr_t>(v_cache) % 16 == 0;
  // Both forms have the same bits; whole tiles share what they read where their blocks fill the chip, one and a half times for heads of 65
  // to 128 in pieces of 16 bytes (one block a unit). Us wide and shared, heads of 128: 60 blocks 25 and 38 (300 tokens) or 13 and 19 (ten portions of two
  // behind 120 tokens), 252 36 and 30 (six prompts of 200), 300 36 and 46 (50 portions of ten behind 120) or 41 and 57, 304 66 and 70 (600
  // tokens), 320 696 and 772 (five tokens each behind 4,000), 480 42 to 101 and 31 to 82, 640 84 and 72, 720 76 and 72; heads of 64: 176
  // 28 and 46 (700 tokens), 320 32 and 24, 400 40 and 23, 800 73 and 47; an element at a time, one
  // behind the other, heads of 250 228 429 and 468, 360 113 and 73, pages of three tokens 360 62 and 35.
  const bool shared = 2L * n_tiles * hgroups * nkv > compute_units() * (vec && hd > 64 && hd <= 128 ? 3L : 2L);
  const auto go = [&](auto kernel, int threads, int pieces) {  // pieces of a tile
    const int most = static_cast<int>(std::max(1L, ((1L << 32) - 1) / threads / (static_cast<long>(pieces) * hgroups * nkv)));  // tiles of a launch
    for (int at = 0; at < n_tiles; at += most)
      hipLaunchKernelGGL(kernel, dim3(pieces * std::min(most, n_tiles - at) * hgroups * nkv), dim3(threads), 0, stream, q, k_cache, v_cache, out,
                         tiles + 2 * static_cast<size_t>(at), positions, seq_of_token, block_table, table_stride, nq, nkv, hd, page_size, scale, window);
  };
#define PYRE_F32_ATTN_OF(HDP, KS, VEC)                                                 \
  if (shared) go(attn_prefill_f32_kernel<HDP, KS, true, VEC>, 128 * KS, 1);            \
  else go(attn_prefill_f32_kernel<HDP, KS, false, VEC>, 128 * KS, 2)
#define PYRE_F32_ATTN(HDP, KS)              \
  if (vec) {                                \
    PYRE_F32_ATTN_OF(HDP, KS, true);        \
  } else {                                  \
    PYRE_F32_ATTN_OF(HDP, KS, false);       \
  }
  // Parts by the head size alone, as far as LDS holds their chunks: a token's sums do not depend on the step.
  switch ((hd + 31) / 32) {
    case 1: PYRE_F32_ATTN(32, 4); break;
    case 2: PYRE_F32_ATTN(64, 4); break;
    case 3: PYRE_F32_ATTN(96, 4); break;
    case 4: PYRE_F32_ATTN(128, 4); break;
    case 5: PYRE_F32_ATTN(160, 2); break;
    case 6: PYRE_F32_ATTN(192, 2); break;
    case 7: PYRE_F32_ATTN(224, 2); break;
    default: PYRE_F32_ATTN(256, 2); break;
  }
#undef PYRE_F32_ATTN
#undef PYRE_F32_ATTN_OF
  return check_launch("attn_prefill_f32");
}
