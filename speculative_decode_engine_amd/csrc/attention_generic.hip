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
//    in fp32 (the layouts of attention_device.hpp's tile path);
//  * the waves' sums meet in LDS, the partitions' in a combine run by the
//    last workgroup of a (KV head, row group) to finish (a kernel of its own,
//    a thread per feature walking the partitions one load after another, took
//    13-15 us).
// Bound by the latency of a few tiles in turn and, as they grow, by memory.
// Measured on MI355X, us per layer, fp32 form / this: decode over 3000 keys,
// 32 KV heads of 96, 188 + 13 (combine) / 17.4; a 5-query window over 4000
// keys, 16/8 heads of 256, RoPE of q included, 193 + 15 / 32.4.  Errors
// against float64 fell too (4.7e-7 -> 3.0e-7, 6.5e-7 -> 4.2e-7 of the
// output's norm): shorter sums.
// DPHP: the head size rounded up to a multiple of 32.
constexpr int kTileWaves = 4;
constexpr int kTileRows = 16;

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
};

template <int DPHP>
struct TileLds {
  using Sh = TileShape<DPHP>;
  // (+ 1 KiB: a feature block past the head size is read, and dropped, from
  // behind the tile's last row)
  char st[kTileWaves * Sh::WAVEB + 1024] __attribute__((aligned(16)));
  h8_t qop[2 * Sh::KS * 64];
  float2 ml[kTileWaves][kTileRows];
  float wgt[kTileRows][attn::kStreamMaxParts + 1];  // a row's partition weights, then 1 / sum
  int last;
  static_assert(kTileRows * DPHP * 4 <= Sh::WAVEB, "a wave's sums fit its tiles");
};

// 16 bytes per lane from p into LDS at lds_off + 16 * lane (lds_off
// wave-uniform); asynchronous (vmcnt).
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

template <int DPHP>
__global__ __launch_bounds__(64 * kTileWaves) void gen_tile_kernel(GenArgs a, GenRope rp,
                                                                   int use_rope,
                                                                   uint32_t* counters) {
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
  // lane l's token of load j and the byte offset of its unit in the row
  int tok[Sh::NI], uoff[Sh::NI];
#pragma unroll
  for (int j = 0; j < Sh::NI; j++) {
    const int f = 64 * j + lane;
    tok[j] = min(f / U, attn::kTile - 1);
    const int u = f - (f / U) * U;
    uoff[j] = 16 * (u ^ ((tok[j] >> tr.shift) & tr.mask));
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
    for (int j = 0; j < Sh::NI; j++) r[j] = (uint32_t)__shfl((int)row, tok[j]);
#pragma unroll
    for (int j = 0; j < Sh::NI; j++)
      if (j < ni)
        tile_load_to_lds(head + (uint64_t)r[j] * row_bytes + uoff[j], dst + 1024u * j);
  };

  const int ts0 = t0 + attn::kTile * wave;
  constexpr int kStride = attn::kTile * kTileWaves;
  uint32_t row_n = 0;  // the rows of the next tile to load
  if (ts0 < t1) {
    const uint32_t row = row_of(ts0);
    load(row, k_off);
    if (ts0 + kStride < t1) row_n = row_of(ts0 + kStride);
    load(row + (uint32_t)a.bs, k_off + Sh::TILEB);
  }

  // ---- q operand: thread -> units of 8 features of a row ----------------
  // (hi part of k-step ks at qop[64 ks + lane], lo behind all of them; lane =
  // row + 16 (unit % 4))
  for (int i = tid; i < kTileRows * (DPHP / 8); i += 64 * kTileWaves) {
    const int r = i / (DPHP / 8), u = i - r * (DPHP / 8);
    float x[8];
#pragma unroll
    for (int e = 0; e < 8; e++) x[e] = 0.f;
    if (r < nr && u < U) {
      const int gr = r0 + r;
      const int m = gr / a.G, h = kvh * a.G + (gr - m * a.G);
      const float* qrow = a.q + (size_t)m * a.nh * dph + (size_t)h * dph;
#pragma unroll
      for (int e = 0; e < 8; e++) {
        const int d = 8 * u + e;
        x[e] = (use_rope ? rope_elem(qrow, d, dph, a.pos_base + m, rp) : qrow[d]) * a.qscale;
      }
    }
    h8_t hi, lo;
    attn::split_h8(x, hi, lo);
    const int at = (u >> 2) * 64 + (u & 3) * 16 + r;
    lds.qop[at] = hi;
    lds.qop[Sh::KS * 64 + at] = lo;
  }
  __syncthreads();

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
    f4_t s[2] = {f4_t{0.f, 0.f, 0.f, 0.f}, f4_t{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int ks = 0; ks < Sh::KS; ks++) {
      const h8_t qh = lds.qop[ks * 64 + lane];
      const h8_t ql = lds.qop[(Sh::KS + ks) * 64 + lane];
#pragma unroll
      for (int tb = 0; tb < 2; tb++) {
        uint4 kx = *reinterpret_cast<const uint4*>(kst + tr.at(16 * tb + l16, 4 * ks + grp));
        // (past the head size: another token's features, whatever they hold)
        if (8 * (4 * ks + grp) >= dph) kx = make_uint4(0u, 0u, 0u, 0u);
        const h8_t k8 = __builtin_bit_cast(h8_t, kx);
        s[tb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(k8, qh, s[tb], 0, 0, 0);
        s[tb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(k8, ql, s[tb], 0, 0, 0);
      }
    }
    // Every operand read has returned (the products took them): the K tile
    // is free.
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");
    // a tile that reaches a position some row may not see: non-finite V at
    // such a position must not meet its zero weight in the matrix product
    bool exact = false;
    if (ts + attn::kTile - 1 > wmin) {
      uint32_t bad = 0;
#pragma unroll
      for (int j = 0; j < Sh::NI; j++)
        if (j < ni && ts + tok[j] > wmin) {
          const uint4 v = *reinterpret_cast<const uint4*>(vst + 1024 * j + 16 * lane);
          bad |= attn::nonfinite_h2(v.x) | attn::nonfinite_h2(v.y) | attn::nonfinite_h2(v.z) |
                 attn::nonfinite_h2(v.w);
        }
      exact = __builtin_amdgcn_ballot_w64(bad != 0) != 0;
    }
    if (more && !exact) load(row, k_off);
    float mx = kNegInf;
#pragma unroll
    for (int tb = 0; tb < 2; tb++)
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const int pos = ts + 16 * tb + 4 * grp + i;
        s[tb][i] = pos <= lim && pos < t1 ? s[tb][i] : kNegInf;
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
#pragma unroll
    for (int db = 0; db < Sh::DB; db++) o[db] *= al;
    if (!exact) {
      h8_t ph, pl;
      attn::split_h8(p, ph, pl);
      const int vt = 4 * grp + (l16 >> 2);
      const int vu = (l16 & 3) >> 1, vsub = 8 * (l16 & 1);
#pragma unroll
      for (int db = 0; db < Sh::DB; db++) {
        const s4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (lds_s4_t*)(vst + tr.at(vt, 2 * db + vu) + vsub));
        const s4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (lds_s4_t*)(vst + tr.at(vt + 16, 2 * db + vu) + vsub));
        const s4_t both[2] = {lo, hi};
        const h8_t v8 = __builtin_bit_cast(h8_t, both);
        o[db] = __builtin_amdgcn_mfma_f32_16x16x32_f16(v8, ph, o[db], 0, 0, 0);
        o[db] = __builtin_amdgcn_mfma_f32_16x16x32_f16(v8, pl, o[db], 0, 0, 0);
      }
    } else {
      // over the tokens each row sees; the weights go over the K tile
      float* pt = reinterpret_cast<float*>(kst);
#pragma unroll
      for (int tb = 0; tb < 2; tb++)
#pragma unroll
        for (int i = 0; i < 4; i++)
          pt[l16 * attn::kTile + 16 * tb + 4 * grp + i] = p[4 * tb + i];
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
      if (exact) load(row, k_off);
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
      x0 += x.x * wt;
      x1 += x.y * wt;
    }
    const int gr = r0 + r;
    if (a.n_parts == 1) {
      const int m = gr / a.G, h = kvh * a.G + (gr - m * a.G);
      const float inv = 1.f / l;
      *reinterpret_cast<float2*>(a.out + (size_t)m * a.nh * dph + (size_t)h * dph + d) =
          make_float2(x0 * inv, x1 * inv);
    } else {
      const size_t pr = ((size_t)kvh * a.R + gr) * a.n_parts + part;
      attn::store_dev2(a.partials + pr * dph + d, x0, x1);
      if (d == 0) attn::store_dev2(a.partials + n_acc + pr * 2, mx, l);
    }
  }
  if (a.n_parts == 1) return;

  // ---- the last workgroup of the (KV head, row group) combines ----------
  // (device-scope stores, waited for before the arrival: store_dev2)
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  if (tid == 0) {
    uint32_t* ctr = counters + (size_t)kvh * gridDim.z + rg;
    const uint32_t prev =
        __hip_atomic_fetch_add(ctr, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    lds.last = prev == (uint32_t)(a.n_parts - 1);
    if (lds.last) __hip_atomic_store(ctr, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
  if (!lds.last) return;
  const int P = a.n_parts;
  const uint32_t acc_bytes = (uint32_t)(n_acc * 4);
  const uint32_t all_bytes = (uint32_t)((n_acc + (size_t)a.nkv * a.R * P * 2) * 4);
  // a wave per row: lane p holds partition p's (max, sum)
  for (int r = wave; r < nr; r += kTileWaves) {
    const size_t row = (size_t)kvh * a.R + r0 + r;
    const float2 ml = attn::load_dev8(
        a.partials, all_bytes,
        lane < P ? (uint32_t)((n_acc + (row * P + lane) * 2) * 4) : attn::kOutOfRange);
    const float mx = attn::wave_max(lane < P ? ml.x : kNegInf);
    const float w = lane < P ? part_weight(ml, mx) : 0.f;
    const float l = attn::wave_sum(lane < P ? ml.y * w : 0.f);
    if (lane < P) lds.wgt[r][lane] = w;
    if (lane == 0) lds.wgt[r][attn::kStreamMaxParts] = 1.f / l;
  }
  __syncthreads();
  // Thread -> (row, 4 features, slice of the partitions): few rows leave
  // threads free, so up to 8 of them share a column's partitions (p = slice,
  // slice + n_slices, ...) and meet in LDS, in slice order.
  const int cols = dph / 4, items = nr * cols;
  int n_slices = 1;
  while (n_slices < 8 && 2 * n_slices * items <= 64 * kTileWaves && 2 * n_slices <= P) n_slices *= 2;
  float4* meet = reinterpret_cast<float4*>(lds.st);
  for (int i = tid; i < items * n_slices; i += 64 * kTileWaves) {
    const int sl = i / items, it = i - sl * items;
    const int r = it / cols, c = it - r * cols;
    const size_t row = (size_t)kvh * a.R + r0 + r;
    float4 sum = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int p0 = sl; p0 < P; p0 += 8 * n_slices) {
      float4 v[8];
#pragma unroll
      for (int k = 0; k < 8; k++) {
        const int p = p0 + k * n_slices;
        v[k] = attn::load_dev16(a.partials, acc_bytes,
                                p < P ? (uint32_t)(((row * P + p) * dph + 4 * c) * 4)
                                      : attn::kOutOfRange);
      }
#pragma unroll
      for (int k = 0; k < 8; k++) {
        const int p = p0 + k * n_slices;
        const float w = p < P ? lds.wgt[r][p] : 0.f;
        sum.x += w * v[k].x;
        sum.y += w * v[k].y;
        sum.z += w * v[k].z;
        sum.w += w * v[k].w;
      }
    }
    if (n_slices > 1) {
      meet[i] = sum;
    } else {
      const int gr = r0 + r;
      const int m = gr / a.G, h = kvh * a.G + (gr - m * a.G);
      const float inv = lds.wgt[r][attn::kStreamMaxParts];
      float2* dst = reinterpret_cast<float2*>(a.out + (size_t)m * a.nh * dph + (size_t)h * dph +
                                              4 * c);
      dst[0] = make_float2(sum.x * inv, sum.y * inv);
      dst[1] = make_float2(sum.z * inv, sum.w * inv);
    }
  }
  if (n_slices == 1) return;
  __syncthreads();
  if (tid < items) {
    const int r = tid / cols, c = tid - r * cols;
    float4 sum = meet[tid];
    for (int sl = 1; sl < n_slices; sl++) {
      const float4 y = meet[sl * items + tid];
      sum.x += y.x;
      sum.y += y.y;
      sum.z += y.z;
      sum.w += y.w;
    }
    const int gr = r0 + r;
    const int m = gr / a.G, h = kvh * a.G + (gr - m * a.G);
    const float inv = lds.wgt[r][attn::kStreamMaxParts];
    float2* dst =
        reinterpret_cast<float2*>(a.out + (size_t)m * a.nh * dph + (size_t)h * dph + 4 * c);
    dst[0] = make_float2(sum.x * inv, sum.y * inv);
    dst[1] = make_float2(sum.z * inv, sum.w * inv);
  }
}

template <bool ROPE>
__global__ __launch_bounds__(kThreads) void gen_attn_kernel(GenArgs a, GenRope rp) {
  __shared__ GenLds lds;
  gen_unit<ROPE, kThreads>(a, &rp, blockIdx.x, blockIdx.y, blockIdx.z, lds);
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
                      uint32_t* counters, hipStream_t stream) {
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
  if (counters) {
    const dim3 block(64 * kTileWaves);
    const int r = rope ? 1 : 0;
    if (dph <= 32)
      gen_tile_kernel<32><<<grid, block, 0, stream>>>(a, rp, r, counters);
    else if (dph <= 64)
      gen_tile_kernel<64><<<grid, block, 0, stream>>>(a, rp, r, counters);
    else if (dph <= 96)
      gen_tile_kernel<96><<<grid, block, 0, stream>>>(a, rp, r, counters);
    else if (dph <= 128)
      gen_tile_kernel<128><<<grid, block, 0, stream>>>(a, rp, r, counters);
    else if (dph <= 160)
      gen_tile_kernel<160><<<grid, block, 0, stream>>>(a, rp, r, counters);
    else if (dph <= 192)
      gen_tile_kernel<192><<<grid, block, 0, stream>>>(a, rp, r, counters);
    else
      gen_tile_kernel<256><<<grid, block, 0, stream>>>(a, rp, r, counters);
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
