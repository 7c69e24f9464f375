// Causal attention of prefill chunks on packed spikes (head_dim <= 128).
//
// Reference semantics: spikeinfer/attention.py:161-178, :320-330 -- query i of a
// chunk (position ctx + i of its sequence) attends to positions 0..ctx + i with
// softmax(popc(q & k) / sqrt(head_dim)) @ bits(v); there by unpacking K and V to
// dense spikes and SDPA with an additive mask.
//
// MI355X design: no dense spikes, no score matrix, no mask tensor; the packed
// words are the only operands.
//   * A workgroup owns 32 * QT rows of one (t, kv head): row r = token r / n_rep,
//     query head r % n_rep, so all the heads of a kv head share its K/V tiles and
//     a tile spans few tokens (little causal waste).  Its four waves take the
//     32-key tiles round-robin and add their sums at the end in wave order, so a
//     row's sums depend on its own sequence only, never on the batch or on QT.
//   * Scores: S^T[key, row] = K Q^T as one v_mfma_scale_f32_32x32x64_f8f6f4 per
//     64 channels, bits as fp4 0.5 (bit i of nibble group i in place), block scales
//     2^-72 and 2^-73: an accumulator is the subnormal 4 * popc(q & k) * 2^-149, so
//     its bits are the integer 4 * popc(q & k) and need no conversion (the matrix
//     cores keep subnormals; 16 conversions a tile: 145 -> 138 us on the prompt
//     below).
//   * A score is an integer in 0..head_dim, so its weight exp(score * scale) is a
//     table entry at byte 4 * score: (hi, lo) halves of an f16 pair with hi + lo
//     the weight to 2^-23 (the table spans e^sqrt(head_dim) <= 2^17 below 2^15, so
//     both halves are normal or lose nothing that counts).  Equal entries broadcast
//     and different ones lie in different banks, save scores 64 apart (0 and 64
//     at head_dim 64; at 128, s and s + 64, far apart for words of one density).
//     No running maximum, no rescaling: any fixed offset cancels in a / l.
//   * Values: O^T[channel, row] += V^T P^T with v_mfma_f32_32x32x16_f16 over
//     (key, hi/lo) pairs.  The score layout (lane l: row l % 32, keys 4 * (l / 32) +
//     0..3 of each 8) is this instruction's B operand layout, so a looked-up pair
//     is an operand register as it is.  V^T comes from a 32 x 32 bit transpose of
//     the wave's V words (five lane-exchange steps), each bit as the pair 1.0, 1.0;
//     it is built once per key tile and shared by the QT row tiles.
//   * Denominators: v_dot2_f32_f16 of the pair with (1, 1), 16 weights to a
//     partial sum and the partial sums in fp32 (one long dot2 chain per row lost
//     1e-6 at 4,000 keys).
//   * fp32 outputs take the hi and the lo products to accumulators of their own, two
//     keys a register (v_perm), the same number of instructions of the matrix cores.
//     Sums of 11-bit halves are exact in fp32 until they pass 2^24 of the smallest
//     one's units, so the sums lose next to nothing; they are added, and divided, in
//     fp64 and rounded once.  Error against float64 in the 2-norm, head_dim 32 to
//     128, 2 to 12,000 keys, a fifth or half of the bits set: 1.6e-8 to 4.1e-8;
//     one accumulator with rounded sums 3.1e-8 to 7e-8 up to 64 keys and up to
//     1.6e-6 beyond; fp32 SDPA 2.7e-8 to 1.1e-7 and up to 1e-5.  The prompt below
//     172 us against 143 with one accumulator, whose bits 16-bit outputs do not show.
// What bounds it: issue.  A 32 x 32 tile at head_dim 64 takes 288 cycles of matrix
// core (two f16 products a weight keep it at 32-bit precision) and about 330 of
// VALU, and the two overlap little: 720 measured (a 4,096-token prompt, 14 / 2
// heads, T = 4: 135 us; row tiles one after the other, without the next one's
// lookups under this one's products: 175).  Against unpack + SDPA (one layer, LIF
// included, bf16): that prompt 8,693 -> 142 us; 32 decodes with chunks of 509 and
// 472 behind 1,024 and 923 cached tokens 1,035 -> 59 us.
#include <cmath>
#include <cstring>
#include <type_traits>

#include "common.hpp"

namespace spk {
namespace prefill {

typedef int v8i __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef _Float16 v2h __attribute__((ext_vector_type(2)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef unsigned v4u __attribute__((ext_vector_type(4)));

#define SPK_LDS __attribute__((address_space(3)))

constexpr int kWaves = 4;
constexpr int kKeys = 32;       // keys per tile
constexpr int kMaxChunks = 32;  // chunks per launch (kernel arguments)
constexpr int kTab = 129;       // weights of scores 0..head_dim (<= 128)

struct Chunk {
  int64_t start;         // first batch row
  const int32_t *table;  // block-table row (any readable word when direct)
  int64_t tstride;
  int n_table, q_len, ctx;
  int direct;            // key j is slot start + j, no table
  int tile0;             // first row tile of the chunk in the launch
};

struct Params {
  const uint32_t *q;           // words of (t, batch row, query head)
  int64_t qs0, qs1, qs2;
  const uint32_t *k, *v;       // words of (t, kv head, slot), the same strides
  int64_t ks0, ks1, ks2;
  int64_t num_slots;
  void *out;                   // (t, batch row, query head, channel)
  int64_t os0, os1, os2;
  int out_dtype, out_vec;      // out_vec: rows take aligned 4-channel stores
  uint32_t rep_mul;            // floor(r / nrep) = r * rep_mul >> 32 for every row
  int units, Hkv, nrep, D, W, bs_log2, nchunks;
  uint32_t tab[kTab];
  Chunk c[kMaxChunks];
};

// The value of x in the lane whose number differs by J (1, 2, 4, 8 or 16).
template <int J>
__device__ __forceinline__ uint32_t lane_xor(uint32_t x) {
  const int v = static_cast<int>(x);
  if constexpr (J == 1) return static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, v, 0xB1, 0xF, 0xF, false));
  else if constexpr (J == 2) return static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, v, 0x4E, 0xF, 0xF, false));
  else if constexpr (J == 8)  // rotation by 8 within a row of 16
    return static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, v, 0x128, 0xF, 0xF, false));
  else return static_cast<uint32_t>(__builtin_amdgcn_ds_swizzle(v, (J << 10) | 0x1f));
}

// One step of the 32 x 32 bit transpose within each 32-lane half (lane = row,
// bit = column): lanes without bit J trade their J-columns for the partner's
// others.
template <int J>
__device__ __forceinline__ uint32_t transpose_step(uint32_t x, int lane) {
  constexpr uint32_t m = J == 16 ? 0x0000ffffu : J == 8 ? 0x00ff00ffu : J == 4 ? 0x0f0f0f0fu
                         : J == 2 ? 0x33333333u : 0x55555555u;
  const uint32_t y = lane_xor<J>(x);
  const bool up = lane & J;
  const uint32_t keep = up ? ~m : m;
  const uint32_t r = __builtin_amdgcn_alignbit(y, y, up ? J : 32 - J);  // rotate right
  return (x & keep) | (r & ~keep);
}

__device__ __forceinline__ uint32_t transpose32(uint32_t x, int lane) {
  x = transpose_step<16>(x, lane);
  x = transpose_step<8>(x, lane);
  x = transpose_step<4>(x, lane);
  x = transpose_step<2>(x, lane);
  return transpose_step<1>(x, lane);
}

// 32 bits as 32 fp4 values of 0.5: nibble n of word i is bit 4n + i.
__device__ __forceinline__ v8i fp4_bits(uint32_t w) {
  v8i r = {};
#pragma unroll
  for (int i = 0; i < 4; ++i) r[i] = static_cast<int>((w >> i) & 0x11111111u);
  return r;
}

// QT row tiles of 32 rows a workgroup; NC = channel tiles of 32 (ceil(D / 32)).
// F32: the outputs are fp32.
template <int QT, int NC, bool F32>
__global__ __launch_bounds__(kWaves * 64) __attribute__((amdgpu_waves_per_eu(2))) void prefill_attn_kernel(
    Params p) {
  constexpr int NK = (NC + 1) / 2;         // 64-channel score steps
  constexpr int kUnits = QT * NC;          // 32 x 32 output tiles a workgroup
  constexpr int kParts = F32 ? 2 : 1;      // accumulators of a tile: the hi and the lo products apart
  constexpr int kTiles = kWaves / kParts;  // output tiles a round of the final sums
  constexpr int kRounds = (kUnits + kTiles - 1) / kTiles;
  struct Smem {
    uint32_t tab[kTab + 3];  // first: a score's accumulator is its entry's LDS address
    float lsum[QT][kParts][kWaves][64];
    float red[kUnits * kParts < kWaves ? kUnits * kParts : kWaves][kWaves][16][64];
  };
  __shared__ Smem sm;
  auto &tab = sm.tab;
  auto &lsum = sm.lsum;
  auto &red = sm.red;
  const uint32_t tab0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((SPK_LDS char *)(void *)tab));

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int half = lane >> 5, col = lane & 31;
  const int tile = blockIdx.x / p.units, unit = blockIdx.x - tile * p.units;
  const int kvh = unit % p.Hkv, t = unit / p.Hkv;
  int ci = 0;
  for (int k = 1; k < p.nchunks; ++k) ci += tile >= p.c[k].tile0 ? 1 : 0;
  const int64_t start = p.c[ci].start;
  const int q_len = p.c[ci].q_len, ctx = p.c[ci].ctx;
  const int rows = q_len * p.nrep;
  const int ntile = (rows + 32 * QT - 1) / (32 * QT);
  const int r0 = (ntile - 1 - (tile - p.c[ci].tile0)) * 32 * QT;  // longest tiles first
  const int nq = min(QT, (rows - r0 + 31) >> 5);
  auto token_of = [&](int r) {
    return p.nrep == 1 ? r : static_cast<int>(__umulhi(static_cast<uint32_t>(r), p.rep_mul));
  };

  if (tid <= p.D) tab[tid] = p.tab[tid];

  // Row tiles: each lane's row (clamped to the last), its last visible key and
  // its query words as score operands.
  v8i qop[QT][NK];
  int lim[QT];
  int lo[QT], hi[QT];  // last visible key of the tile's first and last row (uniform)
#pragma unroll
  for (int i = 0; i < QT; ++i) {
    const int r = min(r0 + 32 * i + col, rows - 1);
    const int tok = token_of(r), h = r - tok * p.nrep;
    lim[i] = ctx + tok;
    lo[i] = ctx + token_of(min(r0 + 32 * i, rows - 1));
    hi[i] = ctx + token_of(min(r0 + 32 * i + 31, rows - 1));
    const uint32_t *qp = p.q + t * p.qs0 + (start + tok) * p.qs1 + (kvh * p.nrep + h) * p.qs2;
#pragma unroll
    for (int s = 0; s < NK; ++s) {
      const int w = 2 * s + half;
      qop[i][s] = fp4_bits(w < p.W ? qp[w] : 0u);
    }
  }

  const int32_t *table = p.c[ci].table;
  const int64_t tstride = p.c[ci].tstride;
  const int n_table = p.c[ci].n_table;
  const bool direct = p.c[ci].direct;
  const int kv_len = ctx + q_len;
  const int bs_mask = (1 << p.bs_log2) - 1;
  const uint32_t nblocks = static_cast<uint32_t>(min<int64_t>(p.num_slots >> p.bs_log2, 0xffffffffll));
  const uint32_t *kbase = p.k + t * p.ks0 + kvh * p.ks1;
  const uint32_t *vbase = p.v + t * p.ks0 + kvh * p.ks1;
  // Loads are unconditional (indices clamped into range, the value dropped where
  // the sequence, its table or the cache ends: zero spikes), so that the wave
  // waits for none of them before it is used an iteration later.
  auto block_of = [&](int kt) -> uint32_t {
    const int blk = (kt * kKeys + col) >> p.bs_log2;
    return static_cast<uint32_t>(table[min(blk, n_table - 1) * tstride]);
  };
  auto load = [&](int kt, uint32_t phys, uint32_t (&kw)[NK], uint32_t (&vw)[NK], bool &ok) {
    const int j = kt * kKeys + col;
    ok = j < kv_len && (direct || ((j >> p.bs_log2) < n_table && phys < nblocks));
    const int64_t slot = direct ? start + j : (static_cast<int64_t>(phys) << p.bs_log2) | (j & bs_mask);
    const int64_t at = ok ? slot * p.ks2 : (direct ? start * p.ks2 : 0);
#pragma unroll
    for (int s = 0; s < NK; ++s) {
      const int w = min(2 * s + half, p.W - 1);
      kw[s] = kbase[at + w];
      vw[s] = vbase[at + w];
    }
  };
  auto keep = [&](uint32_t x, int s, bool ok) { return ok && 2 * s + half < p.W ? x : 0u; };

  v16f acc[QT][NC * kParts];
  float l[QT][kParts];
#pragma unroll
  for (int i = 0; i < QT; ++i) {
#pragma unroll
    for (int p2 = 0; p2 < kParts; ++p2) l[i][p2] = 0.f;
#pragma unroll
    for (int c = 0; c < NC * kParts; ++c) acc[i][c] = v16f{};
  }
  __syncthreads();

  const int nkt = (ctx + token_of(min(r0 + 32 * nq - 1, rows - 1))) / kKeys + 1;
  uint32_t kw[NK], vw[NK];
  bool ok;
  load(wave, block_of(wave), kw, vw, ok);
  uint32_t pnext = block_of(wave + kWaves);
  for (int kt = wave; kt < nkt; kt += kWaves) {
    // Operands of this tile; the next tile's words and the block of the one
    // after are requested before they are used.
    v8i kop[NK];
    uint32_t vt[2 * NK];
#pragma unroll
    for (int s = 0; s < NK; ++s) {
      kop[s] = fp4_bits(keep(kw[s], s, ok));
      const uint32_t x = transpose32(keep(vw[s], s, ok), lane);
      // Both halves of the wave need every channel tile: lanes l and l + 32 take
      // keys 4 * (l / 32) + 0..3 of each eight.
      const auto sw = __builtin_amdgcn_permlane32_swap(x, x, false, false);
      vt[2 * s] = sw[0] >> (4 * half);
      vt[2 * s + 1] = sw[1] >> (4 * half);
    }
    load(kt + kWaves, pnext, kw, vw, ok);
    pnext = block_of(kt + 2 * kWaves);
    v8h vop[NC][4 / kParts];
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int g = 0; g < 4 / kParts; ++g) {
        v4u x;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if constexpr (F32) {  // two keys a register
            const uint32_t b = vt[c] >> (16 * g + 8 * (i >> 1) + 2 * (i & 1));
            x[i] = ((b & 1u) | ((b & 2u) << 15)) * 0x3c00u;
          } else {
            x[i] = static_cast<uint32_t>(static_cast<int>(vt[c] << (31 - 8 * g - i)) >> 31) & 0x3c003c00u;
          }
        }
        vop[c][g] = __builtin_bit_cast(v8h, x);
      }
    auto scores = [&](int i) {
      v16f s = {};
#pragma unroll
      for (int k = 0; k < NK; ++k)
        s = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(kop[k], qop[i][k], s, 4, 4, 0, 55, 0, 54);
      return s;
    };
    auto lookup = [&](const v16f &s, uint32_t (&w)[16]) {
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const uint32_t at = tab0 + __float_as_uint(s[e]);
        w[e] = *reinterpret_cast<const SPK_LDS uint32_t *>(static_cast<uintptr_t>(at));
      }
    };
    auto products = [&](int i, const uint32_t (&w)[16], auto masked) {
      auto weight = [&](int n) {  // the n-th of the lane's sixteen
        if constexpr (decltype(masked)::value)
          return kt * kKeys + 8 * (n >> 2) + 4 * half + (n & 3) <= lim[i] ? w[n] : 0u;
        else return w[n];
      };
      float d[4] = {0.f, 0.f, 0.f, 0.f};  // (a chain of dot2 on one register waits for itself)
      if constexpr (F32) {
#pragma unroll
        for (int g = 0; g < 2; ++g) {
          v4u x[2];  // hi and lo halves, two keys a register
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const uint32_t y0 = weight(8 * g + 2 * e), y1 = weight(8 * g + 2 * e + 1);
#pragma unroll
            for (int q = 0; q < 2; ++q) {
              const uint32_t y = __builtin_amdgcn_perm(y1, y0, q ? 0x07060302u : 0x05040100u);
              float &dq = d[2 * (e & 1) + q];
              dq = __builtin_amdgcn_fdot2(__builtin_bit_cast(v2h, y), v2h{1, 1}, dq, false);
              x[q][e] = y;
            }
          }
#pragma unroll
          for (int c = 0; c < NC; ++c)
#pragma unroll
            for (int q = 0; q < 2; ++q) {
              v16f &a = acc[i][2 * c + q];
              a = __builtin_amdgcn_mfma_f32_32x32x16_f16(vop[c][g], __builtin_bit_cast(v8h, x[q]), a, 0, 0, 0);
            }
        }
        l[i][0] += d[0] + d[2];
        l[i][kParts - 1] += d[1] + d[3];
      } else {
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          v4u x;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const uint32_t y = weight(4 * g + e);
            d[e] = __builtin_amdgcn_fdot2(__builtin_bit_cast(v2h, y), v2h{1, 1}, d[e], false);
            x[e] = y;
          }
          const v8h pw = __builtin_bit_cast(v8h, x);
#pragma unroll
          for (int c = 0; c < NC; ++c)
            acc[i][c] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vop[c][g], pw, acc[i][c], 0, 0, 0);
        }
        l[i][0] += (d[0] + d[1]) + (d[2] + d[3]);
      }
    };
    if (nq == QT && kt * kKeys + kKeys - 1 <= lo[0]) {
      // The next row tile's scores are computed and looked up under this one's
      // products.
      uint32_t w[2][16];
      lookup(scores(0), w[0]);
#pragma unroll
      for (int i = 0; i < QT; ++i) {
        if (i + 1 < QT) lookup(scores(i + 1), w[(i + 1) & 1]);
        products(i, w[i & 1], std::false_type{});
        // Row tile by row tile: left free, the scheduler hoists lookups of several
        // and spills (head_dim 128: 198 us instead of 77).
        __builtin_amdgcn_sched_barrier(0);
      }
    } else {
#pragma unroll
      for (int i = 0; i < QT; ++i) {
        if (i >= nq || kt * kKeys > hi[i]) continue;
        uint32_t w[16];
        lookup(scores(i), w);
        products(i, w, std::true_type{});
      }
    }
  }

  // Sums of the four waves, in wave order: each round the waves put kTiles of the
  // output tiles (row tile i, channel tile c) into LDS and each finishes one of them,
  // or, of an fp32 tile in two parts, one half.
#pragma unroll
  for (int i = 0; i < QT; ++i)
#pragma unroll
    for (int q = 0; q < kParts; ++q) lsum[i][q][wave][lane] = l[i][q];
#pragma unroll
  for (int rd = 0; rd < kRounds; ++rd) {
    if (rd) __syncthreads();
#pragma unroll
    for (int u = 0; u < kWaves; ++u) {
      constexpr int kU = kUnits;
      const int x = rd * kTiles + u / kParts;
      if (x < kU) {
#pragma unroll
        for (int j = 0; j < 16; ++j) red[u][wave][j][lane] = acc[x / NC][x % NC * kParts + u % kParts][j];
      }
    }
    __syncthreads();
    const int x = rd * kTiles + wave / kParts;
    const int i = x / NC, c = x - i * NC;
    const int r = r0 + 32 * i + col;
    if (x >= kUnits || r >= rows) continue;
    const int slot = wave / kParts * kParts;        // the tile's place in red
    const int g0 = F32 ? wave % kParts * 2 : 0;      // first of the wave's 4-channel groups
    constexpr int kGroups = F32 ? 2 : 4;
    // fp32 outputs: the parts' sums and the quotient in fp64, rounded once.
    typedef std::conditional_t<F32, double, float> Sum;
    Sum den = 0;
#pragma unroll
    for (int q = 0; q < kParts; ++q)
#pragma unroll
      for (int w = 0; w < kWaves; ++w)
        den += static_cast<Sum>(lsum[i][q][w][col]) + static_cast<Sum>(lsum[i][q][w][col + 32]);
    const Sum inv = Sum(1) / den;
    const int tok = token_of(r), h = r - tok * p.nrep;
    const int64_t row = t * p.os0 + (start + tok) * p.os1 + (kvh * p.nrep + h) * p.os2;
    auto value = [&](int j) {
      Sum a = 0;
#pragma unroll
      for (int q = 0; q < kParts; ++q)
#pragma unroll
        for (int w = 0; w < kWaves; ++w) a += red[slot + q][w][j][lane];
      return static_cast<float>(a * inv);
    };
    if (p.out_vec) {  // D % 4 == 0: four channels lie in or out together
#pragma unroll
      for (int k = 0; k < kGroups; ++k) {
        const int g = g0 + k, ch = 32 * c + 8 * g + 4 * half;
        const float o[4] = {value(4 * g), value(4 * g + 1), value(4 * g + 2), value(4 * g + 3)};
        if (ch >= p.D) continue;
        if constexpr (F32) {
          *reinterpret_cast<v4f *>(static_cast<float *>(p.out) + row + ch) = v4f{o[0], o[1], o[2], o[3]};
          continue;
        }
        uint32_t w2[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          uint16_t x0, x1;
          if (p.out_dtype == SPK_BF16) {
            x0 = f32_to_bf16_bits(o[2 * e]);
            x1 = f32_to_bf16_bits(o[2 * e + 1]);
          } else {
            x0 = __builtin_bit_cast(uint16_t, static_cast<_Float16>(o[2 * e]));
            x1 = __builtin_bit_cast(uint16_t, static_cast<_Float16>(o[2 * e + 1]));
          }
          w2[e] = x0 | (static_cast<uint32_t>(x1) << 16);
        }
        *reinterpret_cast<uint2 *>(static_cast<uint16_t *>(p.out) + row + ch) = make_uint2(w2[0], w2[1]);
      }
    } else {
#pragma unroll 1
      for (int j = 4 * g0; j < 4 * (g0 + kGroups); ++j) {
        const int ch = 32 * c + 8 * (j >> 2) + 4 * half + (j & 3);
        if (ch < p.D) store_f32_as(p.out, row + ch, p.out_dtype, value(j));
      }
    }
  }
}

// (hi, lo) f16 pairs of exp(s * scale) * 2^15 / exp(D * scale), s = 0..D.
static void build_table(float scale, int D, uint32_t *tab) {
  static thread_local float last_scale = -1.f;
  static thread_local int last_d = 0;
  static thread_local uint32_t last[kTab];
  if (scale != last_scale || D != last_d) {
    for (int s = 0; s <= D; ++s) {
      const double w = std::ldexp(std::exp((s - D) * static_cast<double>(scale)), 15);
      const _Float16 hi = static_cast<_Float16>(w);
      const _Float16 lo = static_cast<_Float16>(w - static_cast<double>(hi));
      uint16_t a, b;
      std::memcpy(&a, &hi, 2);
      std::memcpy(&b, &lo, 2);
      last[s] = a | (static_cast<uint32_t>(b) << 16);
    }
    last_scale = scale;
    last_d = D;
  }
  std::memcpy(tab, last, sizeof(uint32_t) * (D + 1));
}

// Row tiles a workgroup takes of the `qt` asked for: as many as its sums leave
// registers for (fp32 outputs have two accumulators a tile).
constexpr int row_tiles(int qt, int NC, bool f32) {
  const int most = NC > 3 ? 1 : (NC > 2 ? (f32 ? 1 : 2) : (f32 ? 2 : 4));
  return qt < most ? qt : most;
}

template <int QT, bool F32>
static void launch(const Params &p, unsigned grid, hipStream_t s) {
  switch ((p.D + 31) / 32) {
    case 1: prefill_attn_kernel<row_tiles(QT, 1, F32), 1, F32><<<grid, kWaves * 64, 0, s>>>(p); break;
    case 2: prefill_attn_kernel<row_tiles(QT, 2, F32), 2, F32><<<grid, kWaves * 64, 0, s>>>(p); break;
    case 3: prefill_attn_kernel<row_tiles(QT, 3, F32), 3, F32><<<grid, kWaves * 64, 0, s>>>(p); break;
    default: prefill_attn_kernel<row_tiles(QT, 4, F32), 4, F32><<<grid, kWaves * 64, 0, s>>>(p); break;
  }
}

}  // namespace prefill
}  // namespace spk

using namespace spk;

extern "C" int spk_prefill_attn(const int32_t *q, const int64_t q_strides[3], const int32_t *k,
                                const int32_t *v, const int64_t kv_strides[3], int64_t num_slots,
                                const SpkPrefillChunk *chunks, int nchunks, void *out, int out_dtype,
                                const int64_t out_strides[3], int T, int Hq, int Hkv, int head_dim,
                                int block_size, float scale, void *stream) {
  if (T <= 0 || Hq <= 0 || Hkv <= 0 || Hq % Hkv || head_dim <= 0 || nchunks < 0)
    return fail(SPK_EINVAL, "prefill_attn: bad sizes T=%d Hq=%d Hkv=%d D=%d chunks=%d", T, Hq, Hkv, head_dim, nchunks);
  if (head_dim > 128) return fail(SPK_EUNSUPPORTED, "prefill_attn: head_dim=%d (at most 128)", head_dim);
  if (!valid_float_dtype(out_dtype)) return fail(SPK_EINVAL, "prefill_attn: out dtype %d not a float type", out_dtype);
  if (!is_pow2(block_size)) return fail(SPK_EINVAL, "prefill_attn: block_size=%d is not a power of two", block_size);
  if (!(scale > 0.f) || scale * head_dim > 12.f)  // the table's span within f16
    return fail(SPK_EINVAL, "prefill_attn: scale=%g outside (0, 12/head_dim]", (double)scale);
  if (nchunks == 0) return SPK_OK;
  if (!q || !out || !chunks || (num_slots > 0 && (!k || !v))) return fail(SPK_EINVAL, "prefill_attn: null pointer");
  const int nrep = Hq / Hkv;
  int64_t total = 0;  // rows of all chunks
  for (int i = 0; i < nchunks; ++i) {
    const SpkPrefillChunk &c = chunks[i];
    if (c.start < 0 || c.q_len < 0 || c.ctx < 0 || c.n_table < 0 || (!c.table && c.ctx != 0))
      return fail(SPK_EINVAL, "prefill_attn: chunk %d: start=%lld q_len=%d ctx=%d", i, (long long)c.start, c.q_len, c.ctx);
    const int64_t rows = static_cast<int64_t>(c.q_len) * nrep;
    if (rows > (1 << 28) || rows * nrep > 0xffffffffll || static_cast<int64_t>(c.q_len) + c.ctx > (1 << 30))
      return fail(SPK_EUNSUPPORTED, "prefill_attn: chunk %d of %d + %d tokens is too long", i, c.ctx, c.q_len);
    if (!c.table && c.start > num_slots - c.q_len)
      return fail(SPK_EINVAL, "prefill_attn: chunk %d reaches past %lld slots", i, (long long)num_slots);
    total += static_cast<int64_t>(c.q_len) * nrep;
  }
  prefill::Params p{};
  p.q = reinterpret_cast<const uint32_t *>(q);
  p.qs0 = q_strides[0]; p.qs1 = q_strides[1]; p.qs2 = q_strides[2];
  p.k = reinterpret_cast<const uint32_t *>(k);
  p.v = reinterpret_cast<const uint32_t *>(v);
  p.ks0 = kv_strides[0]; p.ks1 = kv_strides[1]; p.ks2 = kv_strides[2];
  p.num_slots = num_slots;
  if (num_slots <= 0) {  // an empty cache: every key is dropped, the loads read q's first words
    p.k = p.v = p.q;
    p.ks0 = p.ks1 = p.ks2 = 0;
  }
  p.out = out; p.out_dtype = out_dtype;
  p.os0 = out_strides[0]; p.os1 = out_strides[1]; p.os2 = out_strides[2];
  p.out_vec = head_dim % 4 == 0 && p.os0 % 4 == 0 && p.os1 % 4 == 0 && p.os2 % 4 == 0 &&
              (reinterpret_cast<uintptr_t>(out) & 15) == 0;
  p.units = T * Hkv; p.Hkv = Hkv; p.nrep = nrep; p.D = head_dim; p.W = (head_dim + 31) / 32;
  p.bs_log2 = ilog2(block_size);
  // ceil(2^32 / nrep): its product with r is off by less than r * nrep <= 2^32
  p.rep_mul = static_cast<uint32_t>(((int64_t(1) << 32) + nrep - 1) / nrep);
  prefill::build_table(scale, head_dim, p.tab);
  // Row tiles per workgroup: four share a key tile's V operands; fewer while
  // that leaves under two workgroups a CU, and where their sums would not fit
  // the registers (head_dim 128, 2,000 tokens: one 60 us, two 77).  The sums do
  // not depend on it.
  const int64_t tiles = (total + 31) / 32 * p.units;
  const int qt = tiles >= 4 * 512 ? 4 : (tiles >= 2 * 512 ? 2 : 1);
  const bool f32 = out_dtype == SPK_F32;
  const int qt_used = prefill::row_tiles(qt, p.W, f32);
  hipStream_t s = static_cast<hipStream_t>(stream);
  for (int i = 0; i < nchunks;) {
    int64_t grid = 0;
    p.nchunks = 0;
    for (; i < nchunks && p.nchunks < prefill::kMaxChunks; ++i) {
      const SpkPrefillChunk &c = chunks[i];
      if (c.q_len == 0) continue;
      const int64_t nt = (static_cast<int64_t>(c.q_len) * nrep + 32 * qt_used - 1) / (32 * qt_used);
      if ((grid + nt) * p.units > 0x7fffffffll) {
        if (p.nchunks) break;
        return fail(SPK_EUNSUPPORTED, "prefill_attn: chunk %d is too large for one launch", i);
      }
      // The kernel loads a table entry whether it uses it or not: a direct chunk
      // or an empty table gets a readable word.
      const bool none = !c.table || c.n_table == 0;
      p.c[p.nchunks++] = prefill::Chunk{c.start, none ? q : c.table, none ? 0 : c.table_stride,
                                        c.table ? c.n_table : 0, c.q_len, c.ctx, c.table ? 0 : 1,
                                        static_cast<int>(grid)};
      grid += nt;
    }
    if (!p.nchunks) break;
    const unsigned g = static_cast<unsigned>(grid * p.units);
    if (f32) {
      if (qt >= 2) prefill::launch<2, true>(p, g, s);
      else prefill::launch<1, true>(p, g, s);
    } else if (qt == 4) {
      prefill::launch<4, false>(p, g, s);
    } else if (qt == 2) {
      prefill::launch<2, false>(p, g, s);
    } else {
      prefill::launch<1, false>(p, g, s);
    }
    const int rc = check_launch("prefill_attn");
    if (rc) return rc;
  }
  return SPK_OK;
}
