// Paged GQA attention for any head_dim up to 512 and any block size: the
// shapes libsde_paged's tile kernels (head_dim 64 / 128, block sizes that
// are multiples of 8) do not take.  Head sizes that are multiples of 8 up to
// 256 run a matrix-core form here (gen_tile_kernel); the rest -- odd sizes,
// whose rows no 16-byte load fits, and larger ones, whose tiles and sums
// outgrow a workgroup's LDS -- run the plain fp32 work unit of
// sde/attention_generic_device.hpp (gen_unit), shared with the device API's
// fallback, one workgroup of 256 threads per (partition, KV head, row
// group), with the partition combine as a kernel of its own.
#include <hip/hip_runtime.h>

#include <cmath>

#include "attention_generic.hpp"
#include "sde/attention_device.hpp"
#include "sde/wave_uniform.hpp"
#include "sde_internal.hpp"

namespace sde {
namespace gen {
namespace {

constexpr int kThreads = 256;

// kv_cache_append of the window with k rotated (model_layer_kv_phase,
// model.cu:346-384): thread per (window row m, feature e), fp16 RNE.
__global__ __launch_bounds__(kThreads) void gen_rope_append_kernel(GenArgs a, GenRope rp) {
  const int m = blockIdx.y;
  const int e = blockIdx.x * kThreads + threadIdx.x;
  if (e >= a.kv_dim) return;
  const int pos = a.pos_base + m;
  const int h = e / a.dph, d = e - h * a.dph;
  const float* krow = rp.k_new + (size_t)m * a.kv_dim + (size_t)h * a.dph;
  const size_t ko = k_row(a, pos);
  a.pool[ko + e] = f2h(rope_elem(krow, d, a.dph, pos, rp));
  a.pool[ko + (size_t)a.bs * a.kv_dim + e] = f2h(rp.v_new[(size_t)m * a.kv_dim + e]);
}

// ---- matrix-core form: head sizes that are multiples of 8, up to 256 ------
//
// The fp32 work unit (gen_unit) computes a token's logits on one thread,
// which reads its K row two bytes at a time; at head size 96 a decode step
// took 188 us over 37 MB of K and V.  Here a workgroup takes up to 16 rows
// and its four waves take the partition's 32-token tiles in turn, each wave
// on its own:
//  * K and V tiles go from memory straight into the wave's LDS, 16 bytes per
//    lane in row order whatever the head size and block size (the lane's
//    token and unit are computed, its block looked up per token), the next K
//    tile while this tile's weights are formed, the next V tile after its
//    product, so a wave keeps at least a tile of loads in flight and needs no
//    barrier;
//  * logits K . Q^T and output V^T . P^T are 16x16x32 fp16 MFMA over the
//    head size padded to 32, q and the weights as fp16 hi + lo pairs, sums
//    in fp32 (the layouts of attention_device.hpp's tile path).  A row of q
//    is scaled by a power of two into fp16's range first and its logits back
//    (any finite q works, and a lo part never loses bits to fp16's least
//    exponent), the weights by kWeightScale;
//  * the waves' sums meet in LDS, the partitions' in a combine kernel.
// Bound by the latency of a few tiles in turn and, as they grow, by memory.
// Measured on MI355X, us per layer, fp32 form / this: decode over 3000 keys,
// 32 KV heads of 96, 188 + 13 (combine) / 14.4 + 3.8; a 5-query window over
// 4000 keys, 16/8 heads of 256, RoPE and the append included, 212 / 26.5.
// Errors against float64 fell too (4.7e-7 -> 2.4e-7, 6.4e-7 -> 3.4e-7 of the
// output's norm): shorter sums.
// DPHP: the head size rounded up to a multiple of 32.
constexpr int kTileWaves = 4;
constexpr int kTileRows = 16;
// The softmax weights, at most 1, enter the matrix cores times this (and
// leave the sums exactly): fp16 then resolves 2^-40 of a row's largest weight
// and not 2^-25, below which a key beside a dominant one was lost or rounded
// to few bits (an attention sink 14 nats above the other keys, its V 0.02 of
// theirs, 16/16 heads of 96, 1200 keys: error 1.2e-5, this 2.4e-7, the fp32
// form 9e-7).
constexpr float kWeightScale = 32768.f;

using attn::f4_t;
using attn::h8_t;
using attn::lds_s4_t;
using attn::s4_t;

template <int DPHP>
struct TileShape {
  static constexpr int KS = DPHP / 32;                     // k-steps of the logits product
  static constexpr int DB = DPHP / 16;                     // 16-feature output blocks
  static constexpr int NI = DPHP / 16;                     // wave loads of a tile (at most)
  static constexpr int TILEB = attn::kTile * 2 * DPHP;     // a staged tile (at most)
  static constexpr int WAVEB = 2 * TILEB;                  // a wave's K and V tile
  // the next smaller form's head size: features below it always exist
  static constexpr int kLeast = DPHP == 256 ? 192 : DPHP - 32;
  // fp16 parts of q: two carry 22-23 of its 24 bits, which is less than the
  // rounding of a long sum of products and more than that of a short one
  // (q x 16 at head size 32, largest error over the output's: fp32 form
  // 1.7e-6, two parts 2.7e-6, three 0.8e-6; at 48 5.3e-6, 1.2e-6, 1.2e-6).
  static constexpr int QP = DPHP <= 32 ? 3 : 2;
};

template <int DPHP>
struct TileLds {
  using Sh = TileShape<DPHP>;
  // (+ 1 KiB: a feature block past the head size is read, and dropped, from
  // behind the tile's last row)
  union {
    char st[kTileWaves * Sh::WAVEB + 1024] __attribute__((aligned(16)));
    GenLds unit;
  };
  h8_t qop[Sh::QP * Sh::KS * 64];
  int qexp[kTileRows];  // rows of q: the exponent of the power of two on it
  float2 ml[kTileWaves][kTileRows];
  int nonfinite[kTileWaves];
  static_assert(kTileRows * DPHP * 4 <= Sh::WAVEB, "a wave's sums fit its tiles");
};

// 16 bytes per lane from p into LDS at lds_off + 16 * lane (lds_off
// wave-uniform); asynchronous (vmcnt).  m0 is a reserved register, which a
// clobber list may not name: nothing else in the kernel may need it (nothing
// does in the assembly of these kernels; LDS operations take no m0 here).
__device__ __forceinline__ void tile_load_to_lds(const char* p, uint32_t lds_off) {
  asm volatile(
      "s_mov_b32 m0, %0\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %1, off"
      :
      : "s"(lds_off), "v"(p)
      : "memory");
}

// Byte offset of unit u of token t in a staged tile of U units per token:
// the unit index is xor-ed within an aligned power-of-two group so that
// tokens whose rows start at the same bank (a period of 16 / 2^swz_v tokens,
// 2^swz_v the largest power of two dividing U, at most 16) differ.
struct TileRow {
  int U, shift, mask;
  __device__ __forceinline__ int at(int t, int u) const {
    return (t * U + (u ^ ((t >> shift) & mask))) * 16;
  }
};

// Weight of sums (max, sum) against the row's max: 0 where no key was seen;
// a sum of NaN logits alone (max -inf, sum NaN) is kept.
__device__ __forceinline__ float part_weight(float2 ml, float mx) {
  if (ml.x == -__builtin_inff()) return ml.y == 0.f ? 0.f : 1.f;
  return __builtin_amdgcn_exp2f(ml.x - mx);
}

// Max over the 16 lanes of a wave's row, returned to all of them.
__device__ __forceinline__ float max16(float x) {
#define SDE_ROR(n)                                                                          \
  x = fmaxf(x, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(                       \
                                             0, __builtin_bit_cast(int, x), 0x120 + n, 0xf, \
                                             0xf, false)))
  SDE_ROR(8);
  SDE_ROR(4);
  SDE_ROR(2);
  SDE_ROR(1);
#undef SDE_ROR
  return x;
}

template <int DPHP>
__global__ __launch_bounds__(64 * kTileWaves) void gen_tile_kernel(GenArgs a, GenRope rp,
                                                                   int use_rope) {
  using Sh = TileShape<DPHP>;
  __shared__ TileLds<DPHP> lds;
  constexpr float kNegInf = -__builtin_inff();
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int l16 = lane & 15, grp = lane >> 4;
  const int part = blockIdx.x, kvh = blockIdx.y, rg = blockIdx.z;
  const int dph = a.dph, U = dph / 8;
  TileRow tr;
  {
    const int v = min(4, __builtin_ctz((unsigned)U));
    tr.U = U;
    tr.shift = 4 - v;
    tr.mask = (1 << v) - 1;
  }
  const int r0 = rg * kTileRows;
  const int nr = min(kTileRows, a.R - r0);
  const int row_max = wave_uniform(a.pos_base + (r0 + nr - 1) / a.G);  // last position seen
  const int wmin = wave_uniform(a.pos_base + r0 / a.G);  // seen by every row
  const int t0 = part * a.part_len;
  const int t1 = min(min(a.L_max, t0 + a.part_len), row_max + 1);

  // ---- tile loads ------------------------------------------------------
  char* const kst = lds.st + wave * Sh::WAVEB;
  char* const vst = kst + Sh::TILEB;
  const uint32_t k_off = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)kst;
  const int ni = (U + 1) / 2;  // 32 U units, 64 per load
  const size_t row_bytes = 2 * (size_t)a.kv_dim;
  const char* head = reinterpret_cast<const char*>(a.pool) + (size_t)kvh * dph * 2;
  // lane l's token of load j (low 5 bits) and the byte offset of its unit in
  // the row (a multiple of 16)
  int at[Sh::NI];
#pragma unroll
  for (int j = 0; j < Sh::NI; j++) {
    const int f = 64 * j + lane;
    const int t = min(f / U, attn::kTile - 1);
    const int u = f - (f / U) * U;
    at[j] = t | (16 * (u ^ ((t >> tr.shift) & tr.mask)) << 4);
  }
  // K row (in rows of the pool; the V row is block_size further) of token
  // ts + lane % 32, tokens past the partition's last taking that one.
  auto row_of = [&](int ts) {
    const int pos = min(ts + (lane & 31), t1 - 1);
    const int lb = pos / a.bs;
    return (uint32_t)a.table[lb] * 2u * (uint32_t)a.bs + (uint32_t)(pos - lb * a.bs);
  };
  auto load = [&](uint32_t row, uint32_t dst) {
    uint32_t r[Sh::NI];
#pragma unroll
    for (int j = 0; j < Sh::NI; j++) r[j] = (uint32_t)__shfl((int)row, at[j] & 31);
#pragma unroll
    for (int j = 0; j < Sh::NI; j++)
      if (j < ni)
        tile_load_to_lds(head + (uint64_t)r[j] * row_bytes + ((uint32_t)at[j] >> 4 & ~15u),
                         dst + 1024u * j);
  };

  // ---- q: thread -> row tid / 16, units (tid % 16) + 16 n; with RoPE
  // instead the wave -> a run of rows, the lane -> pairs, features j and j +
  // dph / 2.  These loads go out before the block table's, whose wait covers
  // them; behind the tile loads they would come back after the tiles.
  auto q_row = [&](int r) {
    const int m = (r0 + r) / a.G, h = kvh * a.G + (r0 + r - m * a.G);
    return a.q + (size_t)m * a.nh * dph + (size_t)h * dph;
  };
  constexpr int kUnits = (DPHP / 8 + 15) / 16;
  const int qr = tid >> 4, qs = tid & 15;
  float x[kUnits][8];
#pragma unroll
  for (int n = 0; n < kUnits; n++)
#pragma unroll
    for (int e = 0; e < 8; e++) x[n][e] = 0.f;
  constexpr int kWaveRows = kTileRows / kTileWaves, kPairs = (DPHP / 2 + 63) / 64;
  const int half = dph / 2;
  const int wave_rows = (nr + kTileWaves - 1) / kTileWaves, wr0 = wave * wave_rows;
  float qa[kWaveRows][kPairs], qb[kWaveRows][kPairs], qf[kPairs];
  if (use_rope) {
#pragma unroll
    for (int k = 0; k < kPairs; k++) qf[k] = rp.inv_freq[min(lane + 64 * k, half - 1)];
#pragma unroll
    for (int i = 0; i < kWaveRows; i++) {
      if (i >= wave_rows || wr0 + i >= nr) break;
      const float* qrow = wave_uniform(q_row(wr0 + i));
#pragma unroll
      for (int k = 0; k < kPairs; k++) {
        const int j = min(lane + 64 * k, half - 1);
        qa[i][k] = qrow[j];
        qb[i][k] = qrow[j + half];
      }
    }
  } else if (qr < nr) {
    const float* qrow = q_row(qr);
#pragma unroll
    for (int n = 0; n < kUnits; n++)
      if (qs + 16 * n < U) {
#pragma unroll
        for (int e = 0; e < 8; e++) x[n][e] = qrow[8 * (qs + 16 * n) + e];
      }
  }

  const int ts0 = t0 + attn::kTile * wave;
  constexpr int kStride = attn::kTile * kTileWaves;
  uint32_t row_n = 0;  // the rows of the next tile to load
  if (ts0 < t1) {
    const uint32_t row = row_of(ts0);
    load(row, k_off);
    if (ts0 + kStride < t1) row_n = row_of(ts0 + kStride);
    load(row + (uint32_t)a.bs, k_off + Sh::TILEB);
  }

  // ---- q operand, while the tiles are on their way ----------------------
  // (part p of k-step ks at qop[(p KS + ks) 64 + lane]; lane = row +
  // 16 (unit % 4)).  A row's largest element is brought to [2^14, 2^15) by a
  // power of two (2^exponent and its inverse are normal numbers; zero, Inf
  // and NaN take 2^15), a rotated one thus below 2^15.5.
  auto exponent = [](float mx) { return min(15 - __builtin_amdgcn_frexp_expf(mx), 126); };
  {
    float mx = 0.f;
#pragma unroll
    for (int n = 0; n < kUnits; n++)
#pragma unroll
      for (int e = 0; e < 8; e++) {
        x[n][e] *= a.qscale;
        mx = fmaxf(mx, fabsf(x[n][e]));
      }
    const int qe = exponent(max16(mx));
    if (qs == 0 && !(use_rope && qr < nr)) lds.qexp[qr] = qe;
#pragma unroll
    for (int n = 0; n < kUnits; n++) {
      const int u = qs + 16 * n;
      if (u >= DPHP / 8 || (use_rope && qr < nr && u < U)) continue;
      const int at = (u >> 2) * 64 + (u & 3) * 16 + qr;
#pragma unroll
      for (int e = 0; e < 8; e++) x[n][e] = ldexpf(x[n][e], qe);
#pragma unroll
      for (int p = 0; p < Sh::QP; p++) {
        h8_t part;
#pragma unroll
        for (int e = 0; e < 8; e++) {
          asm("" : "+v"(x[n][e]));  // (rounded once, as in split_h8)
          part[e] = (_Float16)x[n][e];
          x[n][e] -= (float)part[e];
        }
        lds.qop[p * Sh::KS * 64 + at] = part;
      }
    }
  }
  // With RoPE one angle per pair and query: the rows of a query (its heads)
  // follow each other in the wave's run (an angle per element: 5-query window
  // over 4000 keys, 16/8 heads of 256, the whole layer 29.8 us; this 26.4).
  if (use_rope) {
    float sn[kPairs], cs[kPairs];
    int m_last = -1;
#pragma unroll
    for (int i = 0; i < kWaveRows; i++) {
      const int r = wr0 + i;
      if (i >= wave_rows || r >= nr) break;
      const int m = wave_uniform((r0 + r) / a.G);
      if (m != m_last) {
#pragma unroll
        for (int k = 0; k < kPairs; k++)
          sincosf(((float)(a.pos_base + m) / rp.pos_div) * qf[k], &sn[k], &cs[k]);
        m_last = m;
      }
      float mx = 0.f;
#pragma unroll
      for (int k = 0; k < kPairs; k++) {
        const float x0 = qa[i][k], x1 = qb[i][k];
        mx = fmaxf(mx, fmaxf(fabsf(x0), fabsf(x1)));
        qa[i][k] = (x0 * cs[k] - x1 * sn[k]) * a.qscale;
        qb[i][k] = (x0 * sn[k] + x1 * cs[k]) * a.qscale;
      }
      const int qe = exponent(attn::groups_max(max16(mx)) * a.qscale);
      if (lane == 0) lds.qexp[r] = qe;
#pragma unroll
      for (int k = 0; k < kPairs; k++) {
        const int j = lane + 64 * k;
        if (j >= half) break;
#pragma unroll
        for (int b = 0; b < 2; b++) {
          const int d = j + b * half, u = d >> 3;
          const int at = (u >> 2) * 64 + (u & 3) * 16 + r;
          float v = ldexpf(b ? qb[i][k] : qa[i][k], qe);
#pragma unroll
          for (int p = 0; p < Sh::QP; p++) {
            asm("" : "+v"(v));
            const _Float16 h = (_Float16)v;
            reinterpret_cast<_Float16*>(&lds.qop[p * Sh::KS * 64 + at])[d & 7] = h;
            v -= (float)h;
          }
        }
      }
    }
  }
  __syncthreads();
  const int unscale = -lds.qexp[l16];  // of this lane's row's logits

  // ---- the wave's tiles --------------------------------------------------
  const int lim = l16 < nr ? a.pos_base + (r0 + l16) / a.G : -1;
  float m_run = kNegInf, l_run = 0.f;
  f4_t o[Sh::DB];
#pragma unroll
  for (int db = 0; db < Sh::DB; db++) o[db] = f4_t{0.f, 0.f, 0.f, 0.f};
  for (int ts = ts0; ts < t1; ts += kStride) {
    asm volatile("s_waitcnt vmcnt(0)" : : : "memory");
    const uint32_t row = row_n;  // of the next tile
    const bool more = ts + kStride < t1;
    // Operand reads run a batch ahead of the products (the scheduling
    // barriers): left alone, the compiler reads each operand right before its
    // product and waits out the LDS latency every time.
    f4_t s[2] = {f4_t{0.f, 0.f, 0.f, 0.f}, f4_t{0.f, 0.f, 0.f, 0.f}};
    {
      struct Batch {
        h8_t q[2][Sh::QP];
        uint4 k[2][2];
      } cur, nxt;
      auto read = [&](int k0, Batch& f) {
#pragma unroll
        for (int i = 0; i < 2; i++) {
          const int ks = k0 + i;
          if (ks >= Sh::KS) break;
#pragma unroll
          for (int p = 0; p < Sh::QP; p++) f.q[i][p] = lds.qop[(p * Sh::KS + ks) * 64 + lane];
#pragma unroll
          for (int tb = 0; tb < 2; tb++)
            f.k[i][tb] = *reinterpret_cast<const uint4*>(kst + tr.at(16 * tb + l16, 4 * ks + grp));
        }
      };
      read(0, cur);
#pragma unroll
      for (int k0 = 0; k0 < Sh::KS; k0 += 2) {
        if (k0 + 2 < Sh::KS) read(k0 + 2, nxt);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 2; i++) {
          const int ks = k0 + i;
          if (ks >= Sh::KS) break;
#pragma unroll
          for (int tb = 0; tb < 2; tb++) {
            // (past the head size: another token's features, whatever they hold)
            uint4 kx = cur.k[i][tb];
            if (32 * ks + 32 > Sh::kLeast && 8 * (4 * ks + grp) >= dph)
              kx = make_uint4(0u, 0u, 0u, 0u);
            const h8_t k8 = __builtin_bit_cast(h8_t, kx);
            // the smallest part first: fewer sums are rounded at the logit's
            // magnitude (error at q x 16, head size 96: 2.0e-6 -> 1.2e-6)
#pragma unroll
            for (int p = Sh::QP - 1; p >= 0; p--)
              s[tb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(k8, cur.q[i][p], s[tb], 0, 0, 0);
          }
        }
        cur = nxt;
      }
    }
    // Every operand read has returned (the products took them): the K tile
    // is free.
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");
    // a tile that reaches a position some row may not see: non-finite V at
    // such a position must not meet its zero weight in the matrix product
    // (such a tile is the wave's last: the rows' last positions differ by
    // less than kTileRows, and the wave's next tile lies kStride further)
    static_assert(kStride >= kTileRows + attn::kTile, "no tile after an exact one");
    bool exact = false;
    if (ts + attn::kTile - 1 > wmin) {
      uint32_t bad = 0;
#pragma unroll
      for (int j = 0; j < Sh::NI; j++)
        if (j < ni && ts + (at[j] & 31) > wmin) {
          const uint4 v = *reinterpret_cast<const uint4*>(vst + 1024 * j + 16 * lane);
          bad |= attn::nonfinite_h2(v.x) | attn::nonfinite_h2(v.y) | attn::nonfinite_h2(v.z) |
                 attn::nonfinite_h2(v.w);
        }
      exact = __builtin_amdgcn_ballot_w64(bad != 0) != 0;
    }
    if (more) load(row, k_off);
    float mx = kNegInf;
#pragma unroll
    for (int tb = 0; tb < 2; tb++)
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const int pos = ts + 16 * tb + 4 * grp + i;
        s[tb][i] = pos <= lim && pos < t1 ? ldexpf(s[tb][i], unscale) : kNegInf;
        mx = fmaxf(mx, s[tb][i]);
      }
    const float m_new = fmaxf(m_run, attn::groups_max(mx));
    const float m_use = m_new == kNegInf ? 0.f : m_new;
    const float al = __builtin_amdgcn_exp2f(m_run - m_use);
    m_run = m_new;
    float p[8], ps = 0.f;
#pragma unroll
    for (int tb = 0; tb < 2; tb++)
#pragma unroll
      for (int i = 0; i < 4; i++) {
        p[4 * tb + i] = __builtin_amdgcn_exp2f(s[tb][i] - m_use);
        ps += p[4 * tb + i];
      }
    l_run = l_run * al + ps;
    if (__builtin_amdgcn_ballot_w64(al != 1.f) != 0) {  // (a new max in some row)
#pragma unroll
      for (int db = 0; db < Sh::DB; db++) o[db] *= al;
    }
    if (!exact) {
      const int vt = 4 * grp + (l16 >> 2);
      const int vu = (l16 & 3) >> 1, vsub = 8 * (l16 & 1);
      constexpr int kBatch = 4;
      struct Batch {
        s4_t v[kBatch][2];
      } cur, nxt;
      auto read = [&](int d0, Batch& f) {
#pragma unroll
        for (int i = 0; i < kBatch; i++)
#pragma unroll
          for (int g = 0; g < 2; g++)
            if (d0 + i < Sh::DB)
              f.v[i][g] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                  (lds_s4_t*)(vst + tr.at(vt + 16 * g, 2 * (d0 + i) + vu) + vsub));
      };
      read(0, cur);
      __builtin_amdgcn_sched_barrier(0);
      h8_t ph, pl;
#pragma unroll
      for (int i = 0; i < 8; i++) p[i] *= kWeightScale;
      attn::split_h8(p, ph, pl);
#pragma unroll
      for (int d0 = 0; d0 < Sh::DB; d0 += kBatch) {
        if (d0 + kBatch < Sh::DB) read(d0 + kBatch, nxt);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < kBatch; i++)
          if (d0 + i < Sh::DB)
            o[d0 + i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                __builtin_bit_cast(h8_t, cur.v[i]), ph, o[d0 + i], 0, 0, 0);
#pragma unroll
        for (int i = 0; i < kBatch; i++)
          if (d0 + i < Sh::DB)
            o[d0 + i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                __builtin_bit_cast(h8_t, cur.v[i]), pl, o[d0 + i], 0, 0, 0);
        cur = nxt;
      }
    } else {
      // over the tokens each row sees; the weights go over the K tile
      float* pt = reinterpret_cast<float*>(kst);
#pragma unroll
      for (int tb = 0; tb < 2; tb++)
#pragma unroll
        for (int i = 0; i < 4; i++)
          pt[l16 * attn::kTile + 16 * tb + 4 * grp + i] = p[4 * tb + i] * kWeightScale;
#pragma unroll 1
      for (int t = 0; t < attn::kTile; t++) {
        const float w = pt[l16 * attn::kTile + t];
        const bool vis = ts + t <= lim && ts + t < t1;
#pragma unroll
        for (int db = 0; db < Sh::DB; db++) {
          // features 16db + 4grp .. +3: unit 2db + grp/2, byte 8(grp%2)
          const uint2 v = *reinterpret_cast<const uint2*>(
              vst + tr.at(t, 2 * db + (grp >> 1)) + 8 * (grp & 1));
          const float x[4] = {h2f((uint16_t)(v.x & 0xffffu)), h2f((uint16_t)(v.x >> 16)),
                              h2f((uint16_t)(v.y & 0xffffu)), h2f((uint16_t)(v.y >> 16))};
#pragma unroll
          for (int i = 0; i < 4; i++) o[db][i] = vis ? fmaf(w, x[i], o[db][i]) : o[db][i];
        }
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");  // the V tile is free
    if (more) {
      if (ts + 2 * kStride < t1) row_n = row_of(ts + 2 * kStride);
      load(row + (uint32_t)a.bs, k_off + Sh::TILEB);
    }
  }
  const float l_row = attn::groups_sum(l_run);
  // The wave's sums go over its tiles, whose reads are done: [row][feature].
  float* acc = reinterpret_cast<float*>(kst);
#pragma unroll
  for (int db = 0; db < Sh::DB; db++)
    *reinterpret_cast<f4_t*>(acc + l16 * DPHP + 16 * db + 4 * grp) = o[db];
  if (grp == 0) lds.ml[wave][l16] = make_float2(m_run, l_row);
  __syncthreads();

  // ---- the waves' sums meet: thread -> (row, 2 features) ---------------
  const size_t n_acc = (size_t)a.nkv * a.R * a.n_parts * dph;  // then (max, sum) pairs
  const int hp = dph / 2;
  float finite = 0.f;  // NaN where a sum is not finite
  for (int i = tid; i < nr * hp; i += 64 * kTileWaves) {
    const int r = i / hp, d = 2 * (i - r * hp);
    float2 ml[kTileWaves];
    float mx = kNegInf;
#pragma unroll
    for (int w = 0; w < kTileWaves; w++) {
      ml[w] = lds.ml[w][r];
      mx = fmaxf(mx, ml[w].x);
    }
    float l = 0.f, x0 = 0.f, x1 = 0.f;
#pragma unroll
    for (int w = 0; w < kTileWaves; w++) {
      const float wt = part_weight(ml[w], mx);
      const float2 x = *reinterpret_cast<const float2*>(
          reinterpret_cast<const float*>(lds.st + w * Sh::WAVEB) + r * DPHP + d);
      l += ml[w].y * wt;
      x0 += x.x * (wt * (1.f / kWeightScale));
      x1 += x.y * (wt * (1.f / kWeightScale));
    }
    finite = fmaf(l, 0.f, fmaf(x0, 0.f, fmaf(x1, 0.f, finite)));
    const int gr = r0 + r;
    if (a.n_parts == 1) {
      const int m = gr / a.G, h = kvh * a.G + (gr - m * a.G);
      const float inv = 1.f / l;
      *reinterpret_cast<float2*>(a.out + (size_t)m * a.nh * dph + (size_t)h * dph + d) =
          make_float2(x0 * inv, x1 * inv);
    } else {
      const size_t pr = ((size_t)kvh * a.R + gr) * a.n_parts + part;
      *reinterpret_cast<float2*>(a.partials + pr * dph + d) = make_float2(x0, x1);
      if (d == 0) *reinterpret_cast<float2*>(a.partials + n_acc + pr * 2) = make_float2(mx, l);
    }
  }

  // A part of a pair can make NaN (Inf x 0, Inf - Inf) of a product with Inf
  // that is Inf, or weighs nothing, in fp32: where a row's sums are not finite
  // the fp32 work unit does the partition's rows over, after these stores.
  // (The test costs 0.1 us of a layer's 20 at 32 heads of 96.)
  const bool nonfinite = __builtin_amdgcn_ballot_w64(finite != finite) != 0;
  if (lane == 0) lds.nonfinite[wave] = nonfinite;
  __syncthreads();
  if ((lds.nonfinite[0] | lds.nonfinite[1] | lds.nonfinite[2] | lds.nonfinite[3]) == 0) return;
  __builtin_amdgcn_s_waitcnt(0);
  for (int g = rg * (kTileRows / kGenRows); g * kGenRows < r0 + nr; g++) {
    if (use_rope)
      gen_unit<true, 64 * kTileWaves, true>(a, &rp, part, kvh, g, lds.unit);
    else
      gen_unit<false, 64 * kTileWaves, true>(a, &rp, part, kvh, g, lds.unit);
  }
}

template <bool ROPE>
__global__ __launch_bounds__(kThreads) void gen_attn_kernel(GenArgs a, GenRope rp) {
  __shared__ GenLds lds;
  gen_unit<ROPE, kThreads>(a, &rp, blockIdx.x, blockIdx.y, blockIdx.z, lds);
}

// Log-sum-exp merge of the matrix-core form's partitions: four adjacent lanes
// per (KV head, row, 4 features), lane s taking partitions s, s + 4, ...,
// eight of them in flight; the lanes meet in a fixed order.  A kernel of its
// own on all CUs: run by the last workgroup of a (KV head, row group), which
// one CU's ~35 GB/s of partials bounds, calls measured slower from a few KB
// on (5 queries of 16/8 heads of 256 over 3000 keys 24.8 us against 19.2;
// one query of 32 heads of 96, the least partials, 16.9 against 17.3).
__global__ __launch_bounds__(kThreads) void gen_tile_combine_kernel(GenArgs a) {
  const int sub = threadIdx.x & 3;
  const int cols = a.dph / 4;
  const int64_t n = (int64_t)a.nkv * a.R * cols;
  const int64_t item = ((int64_t)blockIdx.x * kThreads + threadIdx.x) >> 2;
  const int64_t it = item < n ? item : n - 1;  // (whole waves for the exchanges)
  const int64_t row = it / cols;               // kvh * R + rho
  const int c = (int)(it - row * cols);
  const int P = a.n_parts;
  const float* acc = a.partials + row * P * a.dph + 4 * c;
  const float2* mls =
      reinterpret_cast<const float2*>(a.partials + (int64_t)a.nkv * a.R * P * a.dph) + row * P;
  float mx = -__builtin_inff(), l = 0.f;
  float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
  for (int p0 = sub; p0 < P; p0 += 32) {
    float2 ml[8];
    float4 x[8];
#pragma unroll
    for (int k = 0; k < 8; k++) {
      const int p = min(p0 + 4 * k, P - 1);
      ml[k] = mls[p];
      x[k] = *reinterpret_cast<const float4*>(acc + (int64_t)p * a.dph);
    }
    float top = mx;
#pragma unroll
    for (int k = 0; k < 8; k++) top = fmaxf(top, ml[k].x);
    const float old = part_weight(make_float2(mx, l), top);
    mx = top;
    l *= old;
    o.x *= old;
    o.y *= old;
    o.z *= old;
    o.w *= old;
#pragma unroll
    for (int k = 0; k < 8; k++) {
      if (p0 + 4 * k >= P) break;  // (a weight of 0 would make NaN of Inf)
      const float w = part_weight(ml[k], mx);
      l += ml[k].y * w;
      o.x += x[k].x * w;
      o.y += x[k].y * w;
      o.z += x[k].z * w;
      o.w += x[k].w * w;
    }
  }
  float top = fmaxf(mx, __shfl_xor(mx, 1));
  top = fmaxf(top, __shfl_xor(top, 2));
  const float w = part_weight(make_float2(mx, l), top);
  float v[5] = {l * w, o.x * w, o.y * w, o.z * w, o.w * w};
#pragma unroll
  for (int i = 0; i < 5; i++) {
    v[i] += __shfl_xor(v[i], 1);
    v[i] += __shfl_xor(v[i], 2);
  }
  if (sub != 0 || item >= n) return;
  const int h = (int)(row / a.R), rho = (int)(row - (int64_t)h * a.R);
  const int m = rho / a.G, head = h * a.G + (rho - m * a.G);
  const float inv = 1.f / v[0];
  float2* d =
      reinterpret_cast<float2*>(a.out + (size_t)m * a.nh * a.dph + (size_t)head * a.dph + 4 * c);
  d[0] = make_float2(v[1] * inv, v[2] * inv);
  d[1] = make_float2(v[3] * inv, v[4] * inv);
}

// Log-sum-exp merge of a row's partitions: workgroup (row rho, KV head).
__global__ __launch_bounds__(kThreads) void gen_combine_kernel(GenArgs a) {
  gen_combine_row(a, blockIdx.y, blockIdx.x, threadIdx.x, kThreads);
}

}  // namespace

GenPlan generic_plan(int L_max, int nkv, int R, int dph, int n_cus, int max_parts) {
  GenPlan p;
  p.row_groups = (R + kGenRows - 1) / kGenRows;
  const int64_t units = (int64_t)nkv * p.row_groups;
  int64_t parts = (2 * (int64_t)n_cus) / units;
  if (parts > max_parts) parts = max_parts;
  const int64_t by_len = ((int64_t)L_max + 63) / 64;
  if (parts > by_len) parts = by_len;
  // Every plan's partials fit the static array of the allocation-free entry
  // point, so both entry points run the same plan (same results, same errors).
  const int64_t by_bytes =
      (int64_t)(SDE_NOALLOC_SCRATCH_BYTES / ((size_t)nkv * R * (size_t)(dph + 2) * sizeof(float)));
  if (parts > by_bytes) parts = by_bytes;
  if (parts < 1) parts = 1;
  const int64_t len = ((L_max + parts - 1) / parts + 63) / 64 * 64;
  p.part_len = (int)len;
  p.n_parts = (int)((L_max + len - 1) / len);
  return p;
}

bool tile_serves(int dph, int block_size, int64_t pool_blocks) {
  return dph % 8 == 0 && dph <= 256 &&
         pool_blocks * 2 * block_size <= (int64_t)UINT32_MAX;  // (rows are 32-bit)
}

GenPlan tile_plan(int L_max, int nkv, int R, int dph, int n_cus, int max_parts,
                  size_t max_bytes) {
  GenPlan p;
  p.row_groups = (R + kTileRows - 1) / kTileRows;
  const int64_t units = (int64_t)nkv * p.row_groups;
  // (two workgroups' tiles fit a CU's LDS up to head size 128)
  int64_t parts = (dph <= 128 ? 2 : 1) * (int64_t)n_cus / units;
  if (parts > max_parts) parts = max_parts;
  const int64_t by_bytes =
      (int64_t)(max_bytes / ((size_t)nkv * R * (size_t)(dph + 2) * sizeof(float)));
  if (parts > by_bytes) parts = by_bytes;
  if (parts < 1) parts = 1;
  constexpr int kStep = attn::kTile * kTileWaves;
  const int64_t len = ((L_max + parts - 1) / parts + kStep - 1) / kStep * kStep;
  p.part_len = (int)len;
  p.n_parts = (int)((L_max + len - 1) / len);
  return p;
}

size_t generic_partial_bytes(const GenPlan& p, int nkv, int R, int dph) {
  return p.n_parts > 1 ? (size_t)nkv * R * p.n_parts * (size_t)(dph + 2) * sizeof(float) : 0;
}

int generic_attention(uint16_t* pool, const int32_t* table, int kv_dim, int block_size,
                      const float* q, float* out, float* partials, int nh, int nkv, int dph,
                      int pos_base, int n_queries, const GenPlan& plan, const GenRope* rope,
                      bool tiles, hipStream_t stream) {
  if (dph > kMaxDph) return SDE_ERR_UNSUPPORTED;
  GenArgs a;
  a.pool = pool;
  a.table = table;
  a.q = q;
  a.out = out;
  a.partials = partials;
  a.kv_dim = kv_dim;
  a.bs = block_size;
  a.nh = nh;
  a.nkv = nkv;
  a.dph = dph;
  a.G = nh / nkv;
  a.R = n_queries * a.G;
  a.pos_base = pos_base;
  a.L_max = pos_base + n_queries;
  a.n_parts = plan.n_parts;
  a.part_len = plan.part_len;
  a.qscale = (float)(1.4426950408889634 / std::sqrt((double)dph));
  GenRope rp{};
  rp.pos_div = 1.f;
  if (rope) {
    rp = *rope;
    const dim3 grid((kv_dim + kThreads - 1) / kThreads, n_queries);
    gen_rope_append_kernel<<<grid, kThreads, 0, stream>>>(a, rp);
    const int st = launch_status();
    if (st != SDE_OK) return st;
  }
  const dim3 grid(plan.n_parts, nkv, plan.row_groups);
  if (tiles) {
    const dim3 block(64 * kTileWaves);
    const int r = rope ? 1 : 0;
    if (dph <= 32)
      gen_tile_kernel<32><<<grid, block, 0, stream>>>(a, rp, r);
    else if (dph <= 64)
      gen_tile_kernel<64><<<grid, block, 0, stream>>>(a, rp, r);
    else if (dph <= 96)
      gen_tile_kernel<96><<<grid, block, 0, stream>>>(a, rp, r);
    else if (dph <= 128)
      gen_tile_kernel<128><<<grid, block, 0, stream>>>(a, rp, r);
    else if (dph <= 160)
      gen_tile_kernel<160><<<grid, block, 0, stream>>>(a, rp, r);
    else if (dph <= 192)
      gen_tile_kernel<192><<<grid, block, 0, stream>>>(a, rp, r);
    else
      gen_tile_kernel<256><<<grid, block, 0, stream>>>(a, rp, r);
    const int st = launch_status();
    if (st != SDE_OK || plan.n_parts == 1) return st;
    const int64_t threads = (int64_t)nkv * a.R * dph;  // four per 4 features
    gen_tile_combine_kernel<<<(unsigned)((threads + kThreads - 1) / kThreads), kThreads, 0,
                              stream>>>(a);
    return launch_status();
  }
  if (rope)
    gen_attn_kernel<true><<<grid, kThreads, 0, stream>>>(a, rp);
  else
    gen_attn_kernel<false><<<grid, kThreads, 0, stream>>>(a, rp);
  int st = launch_status();
  if (st != SDE_OK || plan.n_parts == 1) return st;
  gen_combine_kernel<<<dim3(a.R, nkv), kThreads, 0, stream>>>(a);
  return launch_status();
}

}  // namespace gen
}  // namespace sde
