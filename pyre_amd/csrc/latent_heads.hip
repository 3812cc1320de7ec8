// Softmax attention of prompt portions over compressed rows [c | r] (see latent_attention.hip), with every head's keys and
// values made once: k_h = [Wuk_h c | r] and v_h = Wuv_h c. A pair of a query and a key then takes KD + ROT multiply-adds for its score
// and VD for its sum, where the rows themselves take rank + ROT and rank (576 + 512 against 192 + 128 with a row of 512); a
// key pays rank x (KD + VD) for it, which many queries share. Which portions are worth it: parts/latent_attention.py.
//
//   s(i, j) = (q_i . k_j) * scale;  i sees j iff j <= i and (window == 0 or i - j < window)
//   out_i   = gate_i * sum_j softmax_j(s(i, .)) v_j, with exp(sink[head]) in the denominator if there is a sink
//
// A block has 64 queries of one head and four waves: two tiles of 32 queries, for each of which two waves take every chunk of
// 64 keys half and half and join their sums at the end, so that the waves share nothing but the keys. The problem is
// transposed, S^T[key, query] = K Q^T and O^T[d, query] = V^T P, so that a lane's scores are operands of the second product
// as they are; values are read transposed by ds_read_b64_tr_b16. Scores, maxima, weights and sums are float32, the exponentials
// base two on scores times log2(e), and a weight goes into the second product as three bfloat16 pieces that sum to it exactly.
// One buffer of keys and values; the next chunk's are on their way in registers, and another block on the same unit works meanwhile.
//
// What bounds it: a chunk is 36 matrix instructions of 32 cycles a wave, 24 of them for the pieces, and some 330 vector
// instructions for the softmax, the pieces and the rescaling; a block alone takes 1.35 us a chunk. 12 heads, a window of 1,024: 42 us
// for the first 2,048 tokens, 35 for the next 952; 28 heads 76 and 51 (latent_attn_tile: 157, 99, 289 and 190). Blocks of 128 queries with
// chunks from memory straight into a ring of three in LDS: 46 and 43, 81 and 47; the next chunk's score beside the softmax
// besides: 50 and 47, 85 and 50; all tiles of a head on one die: 49 and 35, 82 and 52.
//
// Chunks start at multiples of 64 positions: the order of a query's sums follows from its own position alone.
#include "pyre_api.h"
#include "pyre_common.h"
#include "pyre_vec4.h"

#include <type_traits>

using namespace pyre;

namespace {

typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) short s16x4;
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kTiles = 2, kTokens = 32 * kTiles, kKeys = 64, kWaves = 2 * kTiles, kThreads = 64 * kWaves;
constexpr int kTileInts = 5;
constexpr float kLog2e = 1.44269504088896340736f;

struct HeadsArgs {
  const bf16* q;            // [n][heads][KD]
  const bf16* turned;       // the queries' turned parts: ROT elements each, turned_token and turned_head apart
  const bf16* kv;           // [heads][kv_rows][KD | VD]
  const bf16* rows;         // [pages][1][page][row]; a row's last ROT elements are its turned part
  bf16* out;                // [n][heads][VD]
  const float* gate;        // [n][heads * VD] or null
  const int* tiles;         // first token, count, its position, its request's row of the block table, kv row of position 0
  const int* table;
  const float* sink;        // [heads] or null
  long turned_token, turned_head;
  long kv_head;             // elements of a head's keys and values
  int table_stride, heads, row, page_size, window;
  unsigned page_magic;      // (2^32 - 1) / page_size
  float scale2;             // scale * log2(e)
};

// A barrier that waits for LDS traffic alone: the next chunk stays on its way.
__device__ inline void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

__device__ inline float exp2_hw(float x) { return __builtin_amdgcn_exp2f(x); }

// The larger of a lane's number and that of the lane 32 further on or back.
__device__ inline float both_halves_max(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

// 1 / denominator for sums made against the maximum m (base two), a sink included.
__device__ inline float heads_factor(float m, float l, const float* sink, int head) {
  if (!sink) return l > 0.f ? 1.f / l : 0.f;
  const float sk = sink[head] * kLog2e, M = fmaxf(m, sk);
  const float a = m == -INFINITY ? 0.f : exp2_hw(m - M);
  return a / (l * a + exp2_hw(sk - M));
}

// Four keys of sixteen neighbouring columns, transposed on the way out of LDS: of each group of sixteen lanes, lane j
// gives the address of four columns 4 (j % 4) .. of key j / 4 and receives column j of the four keys.
__device__ inline uint2 read_transposed(const bf16* p) {
  const auto v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(const_cast<bf16*>(p)));
  return __builtin_bit_cast(uint2, v);
}

template <int KD, int ROT, int VD>
__global__ __launch_bounds__(kThreads, 2) void latent_heads_kernel(const HeadsArgs a) {
  constexpr int STEPS = (KD + ROT) / 16, VT = VD / 32;
  constexpr int LDK = KD + ROT + 8, LDV = VD + 32;  // the reads of 16 lanes (of 8 rows of values) spread over all banks
  constexpr int KU = KD / 8, RU = ROT / 8, VU = VD / 8;  // 16-byte units of a key, its turned part, a value
  constexpr int KN = kKeys * KU / kThreads, RN = kKeys * RU / kThreads, VN = kKeys * VU / kThreads;
  static_assert(KN * kThreads == kKeys * KU && RN * kThreads == kKeys * RU && VN * kThreads == kKeys * VU && VT % 2 == 0, "whole rounds");
  constexpr int KV_BYTES = kKeys * (LDK + LDV) * 2, JOIN_BYTES = kWaves * (VT / 2) * 4096;
  __shared__ __attribute__((aligned(16))) unsigned char lds[KV_BYTES > JOIN_BYTES ? KV_BYTES : JOIN_BYTES];
  __shared__ float ml_s[kWaves][2][32];  // the waves' maxima and weights
  bf16* const Ks = reinterpret_cast<bf16*>(lds);
  bf16* const Vs = Ks + kKeys * LDK;

  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, h = lane >> 5, c = lane & 31;
  const int tw = wave % kTiles, kw = wave / kTiles, head = blockIdx.x;
  const int* const tile = a.tiles + kTileInts * blockIdx.y;
  const int t0 = tile[0], count = tile[1], pos0 = tile[2], base = tile[4];
  const int* const table = a.table + static_cast<size_t>(tile[3]) * a.table_stride;
  if (count <= 0) return;
  const auto first_seen = [&](int pos) { return a.window > 0 ? max(0, pos - a.window + 1) : 0; };
  const int lo_all = first_seen(pos0), hi_all = pos0 + count - 1;
  const int chunk0 = lo_all / kKeys, n_chunks = hi_all / kKeys - chunk0 + 1;
  // this wave's queries, and the lane's own
  const int wpos = pos0 + 32 * tw, wlast = min(wpos + 31, hi_all);
  const bool active = 32 * tw < count, live = 32 * tw + c < count;
  const int hi = min(wpos + c, hi_all), lo = first_seen(hi);
  const int lo_last = first_seen(wlast);  // keys from here to wpos are seen by every query of the wave

  const bf16* const kv = a.kv + head * a.kv_head + static_cast<long>(base) * (KD + VD);
  const bf16* const r_src = a.rows + a.row - ROT + 8 * (tid % RU);
  const auto seen = [&](int key) { return min(max(key, lo_all), hi_all); };  // keys outside are others once more: nobody sees them
  u32x4 k_reg[KN], v_reg[VN], r_reg[RN];
  int page[RN], in_page[RN];  // of the turned parts of the chunk that is asked for next
  const auto look_up = [&](int it) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < RN; ++i) {
      const int key = seen((chunk0 + it) * kKeys + tid / RU + kThreads / RU * i);
      int entry = __umulhi(key, a.page_magic);  // the quotient, or one less
      in_page[i] = key - entry * a.page_size;
      if (in_page[i] >= a.page_size) in_page[i] -= a.page_size, ++entry;
      page[i] = table[entry];
    }
  };
  const auto ask = [&](int it) __attribute__((always_inline)) {
    const int key0 = (chunk0 + it) * kKeys;
#pragma unroll
    for (int i = 0; i < KN; ++i)
      k_reg[i] = *reinterpret_cast<const u32x4*>(kv + seen(key0 + tid / KU + kThreads / KU * i) * (KD + VD) + 8 * (tid % KU));
#pragma unroll
    for (int i = 0; i < VN; ++i)
      v_reg[i] = *reinterpret_cast<const u32x4*>(kv + seen(key0 + tid / VU + kThreads / VU * i) * (KD + VD) + KD + 8 * (tid % VU));
#pragma unroll
    for (int i = 0; i < RN; ++i)
      r_reg[i] = *reinterpret_cast<const u32x4*>(r_src + (static_cast<size_t>(max(page[i], 0)) * a.page_size + in_page[i]) * a.row);
    if (it + 1 < n_chunks) look_up(it + 1);
  };
  const auto stash = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < KN; ++i) *reinterpret_cast<u32x4*>(Ks + (tid / KU + kThreads / KU * i) * LDK + 8 * (tid % KU)) = k_reg[i];
#pragma unroll
    for (int i = 0; i < VN; ++i) *reinterpret_cast<u32x4*>(Vs + (tid / VU + kThreads / VU * i) * LDV + 8 * (tid % VU)) = v_reg[i];
#pragma unroll
    for (int i = 0; i < RN; ++i) *reinterpret_cast<u32x4*>(Ks + (tid / RU + kThreads / RU * i) * LDK + KD + 8 * (tid % RU)) = r_reg[i];
  };

  look_up(0);
  uint4 qf[STEPS];
  {
    const size_t token = t0 + min(32 * tw + c, count - 1);
    const bf16* const qrow = a.q + (token * a.heads + head) * KD + 8 * h;
    const bf16* const trow = a.turned + token * a.turned_token + head * a.turned_head + 8 * h;
#pragma unroll
    for (int st = 0; st < STEPS; ++st)
      qf[st] = *reinterpret_cast<const uint4*>(st < KD / 16 ? qrow + 16 * st : trow + 16 * st - KD);
  }
  __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): the queries are there, and no wait for them comes behind the chunks asked for ahead
  ask(0);

  f32x16 o[VT];
#pragma unroll
  for (int dt = 0; dt < VT; ++dt)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[dt][i] = 0.f;
  float m = -INFINITY, l = 0.f;
  const bf16* const krow = Ks + (32 * kw + c) * LDK + 8 * h;
  const bf16* const vrow = Vs + (32 * kw + 4 * h + ((lane & 15) >> 2)) * LDV + 16 * ((lane >> 4) & 1) + 4 * (lane & 3);

  for (int it = 0; it < n_chunks; ++it) {
    if (it) lds_barrier();  // everybody has read the chunk before
    stash();
    if (it + 1 < n_chunks) ask(it + 1);
    lds_barrier();
    const int key0 = (chunk0 + it) * kKeys + 32 * kw;
    if (!active || key0 > wlast || key0 + 31 < first_seen(wpos)) continue;
    // element i of the scores is of key 8 (i / 4) + 4 h + i % 4, query c
    bf16x8 k8[STEPS], v8[2][VT];
    f32x16 s;
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] = 0.f;
#pragma unroll
    for (int st = 0; st < 8; ++st) k8[st] = *reinterpret_cast<const bf16x8*>(krow + 16 * st);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int st = 0; st < STEPS; ++st) {
      s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(k8[st], __builtin_bit_cast(bf16x8, qf[st]), s, 0, 0, 0);
      if (st + 8 < STEPS) k8[st + 8] = *reinterpret_cast<const bf16x8*>(krow + 16 * (st + 8));
      __builtin_amdgcn_sched_barrier(0);
    }
    const auto values = [&](int b) {
#pragma unroll
      for (int dt = 0; dt < VT; ++dt) {
        const uint2 v0 = read_transposed(vrow + 16 * b * LDV + 32 * dt), v1 = read_transposed(vrow + (16 * b + 8) * LDV + 32 * dt);
        v8[b][dt] = __builtin_bit_cast(bf16x8, uint4{v0.x, v0.y, v1.x, v1.y});
      }
    };
    values(0);  // beside the softmax
    __builtin_amdgcn_sched_barrier(0);
    float w[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) w[i] = s[i] * a.scale2;
    if (key0 < lo_last || key0 + 31 > wpos) {
      const unsigned last = static_cast<unsigned>(hi - lo), first = static_cast<unsigned>(key0 + 4 * h - lo);
#pragma unroll
      for (int i = 0; i < 16; ++i) w[i] = first + 8 * (i >> 2) + (i & 3) <= last ? w[i] : -INFINITY;
    }
    float mx = w[0];
#pragma unroll
    for (int i = 1; i < 15; i += 2) mx = fmaxf(fmaxf(mx, w[i]), w[i + 1]);
    mx = both_halves_max(fmaxf(mx, w[15]));
    const float m_new = fmaxf(m, mx), m_use = m_new == -INFINITY ? 0.f : m_new;
    const float alpha = exp2_hw(m - m_use);
    m = m_new;
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) w[i] = exp2_hw(w[i] - m_use), sum += w[i];
    l = l * alpha + sum;
    if (__ballot(alpha != 1.f))
#pragma unroll
      for (int dt = 0; dt < VT; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[dt][i] *= alpha;
    // keys 16 b .. 16 b + 15: the lane's eight are 16 b + 4 h + u and 16 b + 8 + 4 h + u, elements 8 b .. 8 b + 7 of its weights
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      if (b == 0) values(1);
      uint32_t p[3][4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const float p0 = w[8 * b + 2 * u], p1 = w[8 * b + 2 * u + 1];
        p[0][u] = pack_bf16x2(p0, p1);
        const float r0 = p0 - __uint_as_float(p[0][u] << 16), r1 = p1 - __uint_as_float(p[0][u] & 0xffff0000u);
        p[1][u] = pack_bf16x2(r0, r1);
        p[2][u] = pack_bf16x2(r0 - __uint_as_float(p[1][u] << 16), r1 - __uint_as_float(p[1][u] & 0xffff0000u));
      }
#pragma unroll
      for (int pc = 2; pc >= 0; --pc) {
        const bf16x8 p8 = __builtin_bit_cast(bf16x8, uint4{p[pc][0], p[pc][1], p[pc][2], p[pc][3]});
#pragma unroll
        for (int dt = 0; dt < VT; ++dt) o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(v8[b][dt], p8, o[dt], 0, 0, 0);
      }
    }
  }

  // The two waves of a query tile join: each takes half of the columns.
  l += __shfl_xor(l, 32, 64);
  if (h == 0) ml_s[wave][0][c] = m, ml_s[wave][1][c] = l;
  lds_barrier();
  const float m0 = ml_s[tw][0][c], m1 = ml_s[tw + kTiles][0][c], M = fmaxf(m0, m1);
  const float a0 = m0 == -INFINITY ? 0.f : exp2_hw(m0 - M), a1 = m1 == -INFINITY ? 0.f : exp2_hw(m1 - M);
  const float total = ml_s[tw][1][c] * a0 + ml_s[tw + kTiles][1][c] * a1, mine = kw ? a1 : a0;
  float* const join = reinterpret_cast<float*>(lds);  // [wave][column tile][4][64 lanes][4]
  auto give = [&](auto other_) {
    constexpr int other = decltype(other_)::value;  // the other wave's half
#pragma unroll
    for (int d = 0; d < VT / 2; ++d)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const f32x16& t = o[other * (VT / 2) + d];
        *reinterpret_cast<f32x4*>(join + ((wave * (VT / 2) + d) * 4 + j) * 256 + 4 * lane) =
            f32x4{t[4 * j] * mine, t[4 * j + 1] * mine, t[4 * j + 2] * mine, t[4 * j + 3] * mine};
      }
  };
  if (kw) give(std::integral_constant<int, 0>{});
  else give(std::integral_constant<int, 1>{});
  lds_barrier();
  if (!live) return;
  const float f = heads_factor(M, total, a.sink, head);
  const size_t at = (static_cast<size_t>(t0 + 32 * tw + c) * a.heads + head) * VD;
  auto finish = [&](auto half_) {
    constexpr int half = decltype(half_)::value;
#pragma unroll
    for (int d = 0; d < VT / 2; ++d)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const f32x16& t = o[half * (VT / 2) + d];
        const f32x4 theirs = *reinterpret_cast<const f32x4*>(join + (((wave ^ kTiles) * (VT / 2) + d) * 4 + j) * 256 + 4 * lane);
        const size_t e = at + 32 * (half * (VT / 2) + d) + 8 * j + 4 * h;
        float4 y = {(t[4 * j] * mine + theirs[0]) * f, (t[4 * j + 1] * mine + theirs[1]) * f, (t[4 * j + 2] * mine + theirs[2]) * f,
                    (t[4 * j + 3] * mine + theirs[3]) * f};
        if (a.gate) {
          const float4 g = *reinterpret_cast<const float4*>(a.gate + e);
          y.x *= g.x, y.y *= g.y, y.z *= g.z, y.w *= g.w;
        }
        Vec4<bf16>::store(a.out + e, y);
      }
  };
  if (kw) finish(std::integral_constant<int, 1>{});
  else finish(std::integral_constant<int, 0>{});
}

}  // namespace

extern "C" int pyre_latent_heads_supports(int key_dim, int rot, int value_dim) { return key_dim == 128 && rot == 64 && value_dim == 128; }

extern "C" int pyre_latent_heads(const void* q, const void* turned, long turned_token, long turned_head, const void* kv, int kv_rows, const void* rows,
                                 int row, int page_size, void* out, const float* gate, const int* tiles, int n_tiles,
                                 const int* block_table, int table_stride, int heads, int key_dim, int rot, int value_dim, float scale,
                                 int window, const float* sink, hipStream_t stream) {
  PYRE_REQUIRE(pyre_latent_heads_supports(key_dim, rot, value_dim), "latent_heads: head sizes %d + %d / %d are not supported", key_dim, rot, value_dim);
  PYRE_REQUIRE(n_tiles >= 0 && n_tiles <= 65535, "latent_heads: %d tiles are not a launch", n_tiles);
  if (n_tiles == 0) return 0;
  PYRE_REQUIRE(q && turned && kv && rows && out && tiles && block_table, "latent_heads: bad arguments");
  PYRE_REQUIRE(heads > 0 && heads <= 65535 && kv_rows > 0 && kv_rows < (1 << 22) && page_size > 0 && table_stride > 0 && window >= 0 && row > rot && row % 8 == 0 && turned_token % 8 == 0 &&
                   turned_head % 8 == 0, "latent_heads: bad geometry");
  for (const void* p : {q, turned, kv, rows, static_cast<const void*>(out), static_cast<const void*>(gate)})
    PYRE_REQUIRE(reinterpret_cast<uintptr_t>(p) % 16 == 0, "latent_heads: operands must lie on 16 bytes");
  HeadsArgs a{};
  a.q = static_cast<const bf16*>(q), a.turned = static_cast<const bf16*>(turned), a.kv = static_cast<const bf16*>(kv);
  a.rows = static_cast<const bf16*>(rows), a.out = static_cast<bf16*>(out), a.gate = gate, a.tiles = tiles, a.table = block_table;
  a.kv_head = static_cast<long>(kv_rows) * (key_dim + value_dim), a.sink = sink, a.turned_token = turned_token, a.turned_head = turned_head, a.table_stride = table_stride, a.heads = heads, a.row = row;
  a.page_size = page_size, a.window = window, a.page_magic = 0xffffffffu / page_size, a.scale2 = scale * kLog2e;
  hipLaunchKernelGGL((latent_heads_kernel<128, 64, 128>), dim3(heads, n_tiles), dim3(kThreads), 0, stream, a);
  return check_launch("latent_heads");
}
