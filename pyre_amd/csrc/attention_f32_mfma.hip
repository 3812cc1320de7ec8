// Causal (optionally windowed) attention of prompt portions over the paged cache in true
// float32 on the matrix cores (v_mfma_f32_16x16x4_f32: float32 operands, products and sums):
// the 32-bit path's attention for requests that bring more than one token. Single tokens stay
// with attention_generic.hip, whose blocks are of one token and cannot fill sixteen columns.
//
//   scores = (q k^T) * scale, masked to lo..pos       (pyre/model.py:109-120)
//   probs  = softmax(scores), out = probs v            (pyre/model.py:122-123)
//
// A tile is up to 32 consecutive tokens of one request (tiles[i] = first token in the flat
// batch, count); a block takes sixteen of them for HEADS query heads of one key/value head. Its
// waves are a head's each, KS waves a head: of every KS chunks of 32 keys, which the block keeps
// in LDS together (K as stored, V transposed back: [d][key]), a wave takes one, with a maximum,
// a sum and an output of its own; they are joined at the end, in the order of the parts. The
// transposed problem is computed on 16 x 16 x 4, so that the scores come out in the layout the
// second product wants them in:
//   S^T[key, token]  = sum_d K[key, d] Q[token, d]      A = K (LDS), B = Q^T (registers)
//   O^T[d, token]   += sum_key V^T[d, key] P^T[key, token]   A = V^T (LDS), B = P^T = the lane's
//                                                           own eight scores, one per step
// A step's four elements of the summed index are 4 g + j of sixteen (g = lane / 16), so that the
// operands of four steps are one 16-byte read; element j of a tile of scores is key 4 g + j.
// Chunks start at multiples of 32 keys and go to waves by their number, so the order of every sum
// of a token depends on its own bounds (lo, pos) alone, not on the tile it is in or on what
// else is in the step.
#include "pyre_api.h"
#include "pyre_common.h"

using namespace pyre;

namespace {

typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef f32x4 f32x4_anywhere __attribute__((aligned(4)));
constexpr int kKeys = 32;    // keys of a chunk
constexpr int kTokens = 16;  // tokens of a block

// HDP: the head size rounded up to a multiple of 32 (the rest is zeros). VEC (heads and pages of a multiple of four elements and
// tokens): keys and values come in 16-byte pieces, asked for while the chunks before them are multiplied, and the pages
// they lie in a round earlier still. A round is KS chunks.
//
// The matrix instruction has a sixteenth of the 16-bit one's rate: a chunk's 128 instructions are 1.7 us of a wave's SIMD. A step of a
// few hundred tokens is a few dozen tiles, so what counts is that they fill the chip (sixteen tokens and two heads a block, the keys
// dealt to four waves: three prompts of 333, 206 and 27 tokens on twelve heads of 128 are 228 blocks of eight waves where 32 tokens and
// four heads made 76 of four, one wave a SIMD), that an instruction does not cost an LDS read of four bytes, and that the
// loads of a round are asked for without a wait between them (a branch around each made them wait for one another: 30.5 us). Us a
// launch before and now: those three prompts 90 and 27, 150 tokens of the 7B heads 48 and 18, 600 156 and 78, 2,048 1,003 and 619, 2,048
// behind 6,000 others 3,797 and 3,119 (42 % of the instruction's rate); heads of 64, 96, 192 and 256, 700 tokens, 97 and 37, 132 and 51,
// 260 and 99, 332 and 96. KS = 2 of heads of 128: 41 for the three prompts, 1,101 for 2,048 tokens (both with the branches; 757 with
// KS = 4). The root mean square distance from 64 bits is 2.9e-7 for the three prompts (3.2e-7 before) and 8.7e-7 behind 6,000 tokens
// (15.6e-7): the parts' sums are shorter.
template <int HDP, int HEADS, int KS, bool VEC>
__global__ __launch_bounds__(64 * HEADS * KS) void attn_prefill_f32_kernel(
    const float* __restrict__ q, const float* __restrict__ k_cache, const float* __restrict__ v_cache,
    float* __restrict__ out, const int* __restrict__ tiles, const int* __restrict__ positions,
    const int* __restrict__ seq_of_token, const int* __restrict__ block_table, int table_stride, int nq, int nkv,
    int hd, int page_size, float scale, int window) {
  constexpr int THREADS = 64 * HEADS * KS, KEYS = kKeys * KS;
  constexpr int KROW = HDP + 4, VROW = kKeys + 4;  // elements of a row in LDS: sixteen rows start on all banks in turn
  constexpr int KSIZE = KEYS * KROW, VSIZE = KS * HDP * VROW;
  static_assert(HEADS * KS * kTokens * KROW <= KSIZE && 2 * HEADS * KS * kTokens <= VSIZE, "what is joined lies where the keys lay");
  __shared__ __attribute__((aligned(16))) float Ks[KSIZE];
  __shared__ __attribute__((aligned(16))) float Vt[VSIZE];
  __shared__ __attribute__((aligned(16))) int pages[3][KEYS];    // of three rounds' keys; -1: not there
  // Where a key's row and its column of values start, worked out once: a piece's address is an addition.
  __shared__ __attribute__((aligned(16))) longlong2 where[3][KEYS];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, g = lane >> 4, c = lane & 15;
  const int n_rep = nq / nkv, kvh = blockIdx.z;
  const int part = wave / HEADS, hin = blockIdx.y * HEADS + wave % HEADS;
  const bool active = hin < n_rep;  // a wave without a head still helps loading
  const int head = kvh * n_rep + (active ? hin : 0);
  const int half_tile = gridDim.x - 1 - blockIdx.x;  // the last tokens, which see the most keys, first
  const int t0 = tiles[half_tile & ~1] + kTokens * (half_tile & 1);
  const int ntok = min(kTokens, tiles[half_tile | 1] - kTokens * (half_tile & 1));
  if (ntok <= 0) return;
  const int pos0 = positions[t0];
  const int* table = block_table + static_cast<size_t>(seq_of_token[t0]) * table_stride;

  // Column c of this wave: token t0 + c, which sees keys lo..hi. Columns past the tile's end
  // compute on zeros over the first token's keys and are not stored.
  const bool live = active && c < ntok;
  const int hi = c < ntok ? pos0 + c : pos0;
  const int lo = window > 0 ? max(0, hi - window + 1) : 0;
  f32x4 qr[HDP / 16];  // Q[token c][d = 16 s + 4 g ..]
#pragma unroll
  for (int s = 0; s < HDP / 16; ++s) {
    const int d = 16 * s + 4 * g;
    const float* from = q + (static_cast<size_t>(t0 + c) * nq + head) * hd + d;
    qr[s] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (VEC) {
      if (live && d < hd) qr[s] = *reinterpret_cast<const f32x4_anywhere*>(from);
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (live && d + j < hd) qr[s][j] = from[j];
    }
  }
  f32x4 o[HDP / 16];
#pragma unroll
  for (int dt = 0; dt < HDP / 16; ++dt) o[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;  // l: this lane's share of the column's sum (its eight keys of every chunk)

  const int lo_all = window > 0 ? max(0, pos0 - window + 1) : 0;
  const int hi_all = pos0 + ntok - 1;
  const int first_chunk = lo_all / kKeys, last_chunk = hi_all / kKeys;
  const int first = first_chunk / KS, last = last_chunk / KS;  // rounds
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
  constexpr int PIECES = HDP / (8 * HEADS);  // 16-byte pieces of keys, and of values, of a thread and round
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
  int slot = 0;
  for (int round = first; round <= last; ++round) {
    const int next = slot == 2 ? 0 : slot + 1;
    __syncthreads();  // the round before has been read by every wave
    note(round + 2, next == 2 ? 0 : next + 1, ahead);
    if (VEC) {
      put(round);
      __syncthreads();
      if (round < last) fetch(next);
    } else {
      for (int i = tid; i < KEYS * HDP; i += THREADS) {  // K: d fastest, as it lies in the cache
        const int key = i / HDP, d = i % HDP;
        const long long at = where[slot][key].x;
        float v = 0.f;
        if (at >= 0 && d < hd) v = k_cache[at + d];
        Ks[key * KROW + d] = v;
      }
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
    const int chunk = KS * round + part, here = slot;
    slot = next;
    if (!active || chunk < first_chunk || chunk > last_chunk) continue;

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
    const float m_new = fmaxf(m, mx);
    const float m_use = m_new == -INFINITY ? 0.f : m_new;  // a column without a visible key so far
    const float alpha = expf(m - m_use);
    m = m_new;
    float sum = 0.f;
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        s[kt][j] = expf(s[kt][j] - m_use);
        sum += s[kt][j];
      }
    l = l * alpha + sum;
#pragma unroll
    for (int dt = 0; dt < HDP / 16; ++dt) o[dt] *= alpha;
    constexpr int GROUP = HDP % 64 == 0 ? 4 : 2;  // tiles of d whose chains of products are in flight together
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
          for (int t = 0; t < GROUP; ++t) o[dt + t] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[t][j], s[kt][j], o[dt + t], 0, 0, 0);
      }
  }

  // The parts of a head, joined in their order: outputs where the keys lay, maxima and sums where the values lay.
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  __syncthreads();
#pragma unroll
  for (int dt = 0; dt < HDP / 16; ++dt)  // element j of o[dt]: d = 16 dt + 4 g + j of token c
    *reinterpret_cast<f32x4*>(Ks + (kTokens * wave + c) * KROW + 16 * dt + 4 * g) = o[dt];
  if (g == 0) {
    Vt[2 * (kTokens * wave + c)] = m;
    Vt[2 * (kTokens * wave + c) + 1] = l;
  }
  __syncthreads();
  for (int i = tid; i < HEADS * kTokens * (HDP / 4); i += THREADS) {
    const int d = 4 * (i % (HDP / 4)), row = i / (HDP / 4), token = row % kTokens, which = row / kTokens;
    if (d >= hd || token >= ntok || static_cast<int>(blockIdx.y) * HEADS + which >= n_rep) continue;
    float most = -INFINITY, total = 0.f;
#pragma unroll
    for (int p = 0; p < KS; ++p) most = fmaxf(most, Vt[2 * (kTokens * (HEADS * p + which) + token)]);
    f32x4 y{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int p = 0; p < KS; ++p) {
      const int at = kTokens * (HEADS * p + which) + token;
      const float weight = Vt[2 * at] == -INFINITY ? 0.f : expf(Vt[2 * at] - most);
      total += weight * Vt[2 * at + 1];
      y += weight * *reinterpret_cast<const f32x4*>(Ks + at * KROW + d);
    }
    y *= total > 0.f ? 1.f / total : 0.f;
    float* dst = out + (static_cast<size_t>(t0 + token) * nq + kvh * n_rep + blockIdx.y * HEADS + which) * hd + d;
    if (VEC) {
      *reinterpret_cast<f32x4_anywhere*>(dst) = y;
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (d + j < hd) dst[j] = y[j];
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
  constexpr int kHeads = 2;
  const int hgroups = (nq / nkv + kHeads - 1) / kHeads;
  PYRE_REQUIRE(nkv <= 65535 && hgroups <= 65535 && n_tiles < (1 << 22), "attn_prefill_f32: grid too large");
  const dim3 grid(2 * n_tiles, hgroups, nkv);
  const bool vec = hd % 4 == 0 && page_size % 4 == 0 && reinterpret_cast<uintptr_t>(k_cache) % 16 == 0 &&
                   reinterpret_cast<uintptr_t>(v_cache) % 16 == 0;
#define PYRE_F32_ATTN_OF(HDP, KS, VEC)                                                                                  \
  hipLaunchKernelGGL((attn_prefill_f32_kernel<HDP, kHeads, KS, VEC>), grid, dim3(64 * kHeads * KS), 0, stream, q, k_cache, \
                     v_cache, out, tiles, positions, seq_of_token, block_table, table_stride, nq, nkv, hd, page_size, scale, window)
#define PYRE_F32_ATTN(HDP, KS)            \
  if (vec) PYRE_F32_ATTN_OF(HDP, KS, true); \
  else PYRE_F32_ATTN_OF(HDP, KS, false)
  // Waves a head by the head size alone, as far as LDS holds their chunks: a token's sums do not depend on the step.
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
