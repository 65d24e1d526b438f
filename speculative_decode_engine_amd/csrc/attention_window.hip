// Causal paged GQA attention for wide windows: a prompt, or a chunk of one,
// whose rows -- (query, head in group) pairs of a KV head -- number many
// more than a verify window's.  Same semantics as the tile kernels of
// paged_attention.hip (query m of the window sees positions
// [0, pos_base + m]; positions a row does not see never enter its sums).
//
// What it costs is arithmetic: every K/V byte serves all rows of the window
// and stays in the caches.  So, against the decode kernels' 16 rows per
// workgroup with the waves splitting the context:
//  * a workgroup holds 128 rows of one KV head, 32 per wave, and its waves
//    share every K/V tile (64 tokens) staged in LDS -- a tile is loaded once
//    for 128 rows, not once for 16;
//  * two waves share 32 rows and take a tile's token halves (merged at the
//    end), so a SIMD has two waves to run however few row groups are left;
//  * the products are 32x32x16 fp16 MFMA (twice the arithmetic per LDS
//    operand byte of the 16x16x32 form), q and the softmax weights as fp16
//    hi + lo pairs, sums in fp32;
//  * tiles past a row group's last visible position are never loaded, tiles
//    past a wave's are not multiplied;
//  * the weights' reference (the running max) enters the logits product as
//    its initial accumulator and is raised only when a row's max is more
//    than 2^8 above it, which skips most rescales of the output registers;
//    the weights enter the products times 2^7 (kWeightScale), below 2^15.
// Tiles go from memory straight into LDS, one ahead of the one multiplied
// (two buffers, one barrier per tile): carried in registers instead, the
// next tile's 16-32 registers made the kernel spill, and its loads, 2 us
// away on a fragmented pool, were waited for.
//
// Measured on MI355X: 2003 queries of 32/8 heads of 128, no context, 417 us
// on the 16-row kernel (L2-bound: 4.1 GB read at ~10 TB/s), 97 here (33
// GFLOP of products, twice that with the hi/lo split); 256 queries of 32/4
// heads of 64 after 1500 keys 32.7 us, 20.7 + 4.6 for the combine here, of
// which ~5 us pass before the first tile arrives.  Neither unit is full: of
// the SIMD cycles of the long prompt the matrix cores are busy for 28 % and
// the vector unit for 31 %, of the chunk's 13 % and 29 %; the waves wait a
// third of their cycles for tiles and barriers and a third to issue.
#include <hip/hip_runtime.h>

#include "attention_window.hpp"
#include "sde_internal.hpp"

namespace sde {
namespace win {

using attn::AttnArgs;
using attn::f4_t;
using attn::h8_t;
using attn::lds_s4_t;
using attn::s4_t;

typedef float f16_t __attribute__((ext_vector_type(16)));

constexpr int kWinThreads = 64 * kWinWaves;
constexpr int kHalf = 32;       // tokens of a tile that one wave takes
constexpr int kWinBuffers = 2;  // tiles in LDS: one multiplied, one on its way
constexpr int kWinTable = 2048; // block table entries in LDS
constexpr float kLazyMax = 8.f;  // log2 growth of a row's max that triggers a rescale
// On the weights (up to 2^kLazyMax) where they enter the matrix cores, taken
// back from the sums exactly: fp16's quantum is then 2^-32 of the reference
// and not 2^-25, which a key beside a dominant one is rounded to.  One
// reference spans a row's partition here, where the 16-row kernels have one
// per wave (a sink 14 nats above the other keys, its V 0.02 of theirs, 2003
// keys, 32/8 heads of 128: error 2.0e-5, this 3.7e-7, 16-row kernel 1.0e-5).
constexpr float kWeightScale = 128.f;

template <int DPH>
struct WinShape {
  static constexpr int KS = DPH / 16;     // k-steps of the logits product
  static constexpr int DB = DPH / 32;     // 32-feature blocks of the output
  static constexpr int UNITS = DPH / 8;   // 16-byte units per token row
  static constexpr int ROWB = 2 * DPH;    // bytes per staged row
  static constexpr int TILEB = kWinTok * ROWB;
  static constexpr int NU = kWinTok * UNITS / kWinThreads;  // units per thread, K or V
};

// 16 bytes per lane from base + off straight into LDS: lane l's go to
// lds_off + 16l (lds_off wave-uniform).  Asynchronous (vmcnt); the memory
// clobber and the waits below order it.  m0 is a reserved register, which a
// clobber list may not name: nothing else in the kernel may need it (nothing
// does in its assembly; LDS operations take no m0 here).
__device__ __forceinline__ void load_to_lds(const char* base, uint32_t off, uint32_t lds_off) {
  asm volatile(
      "s_mov_b32 m0, %0\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %1, %2"
      :
      : "s"(lds_off), "v"(off), "s"(base)
      : "memory");
}

// Waits for the wave's loads in flight.
__device__ __forceinline__ void wait_loads() { asm volatile("s_waitcnt vmcnt(0)" : : : "memory"); }

// Byte offset of 16-byte unit u of token row t in a staged tile.  The unit
// index is xor-ed with a value that differs over any 16 consecutive tokens
// (K operand reads: 16 tokens, one unit) and puts 4 consecutive tokens into
// different 64-byte groups (transposed V reads: 4 tokens, 64 bytes each), so
// both read all 64 banks.
template <int DPH>
__device__ __forceinline__ int win_staged(int t, int u) {
  const int f = DPH == 128 ? ((t & 3) << 2) | ((t >> 2) & 3)
                           : (((t >> 1) & 1) << 2) | ((t >> 2) & 3);
  return t * WinShape<DPH>::ROWB + 16 * (u ^ f);
}

// x = hi + lo (attn::split_h8) for softmax weights, in pairs.
__device__ __forceinline__ void split_weights(const float (&x)[8], h8_t& hi, h8_t& lo) {
  typedef _Float16 h2_t __attribute__((ext_vector_type(2)));
  typedef float f2_t __attribute__((ext_vector_type(2)));
#pragma unroll
  for (int e = 0; e < 8; e += 2) {
    const h2_t h = __builtin_convertvector((f2_t{x[e], x[e + 1]}), h2_t);
    const h2_t l =
        __builtin_convertvector((f2_t{x[e] - (float)h[0], x[e + 1] - (float)h[1]}), h2_t);
    hi[e] = h[0];
    hi[e + 1] = h[1];
    lo[e] = l[0];
    lo[e + 1] = l[1];
  }
}

// Weight of sums (max m, sum l) against the max `top`: 0 where no key was
// seen; a sum of NaN logits alone (max -inf, sum NaN) is kept.
__device__ __forceinline__ float sums_weight(float m, float l, float top) {
  if (m == -INFINITY) return l == 0.f ? 0.f : 1.f;
  return __builtin_amdgcn_exp2f(m - top);
}

__device__ __forceinline__ float half_max(float x) {
  const int v = __builtin_bit_cast(int, x);
  const auto h = __builtin_amdgcn_permlane32_swap(v, v, false, false);
  return fmaxf(__builtin_bit_cast(float, (int)h[0]), __builtin_bit_cast(float, (int)h[1]));
}

// o += P . V over 32 tokens (from position ts on) that each row sees,
// skipping the rest, for a tile in which a position
// hidden from some row of the workgroup holds a non-finite V element (0 x
// Inf would reach that row through the matrix product): every wave takes
// it, its weights going through its own 1 KiB share of those tokens' staged
// K rows, which are dead (the caller's barrier).
template <int DPH>
__device__ __forceinline__ void win_exact_pv(int ts, int lane, int lim, const f16_t& s,
                                             char* pt_bytes, const char* vst,
                                             f16_t (&o)[WinShape<DPH>::DB]) {
  using Sh = WinShape<DPH>;
  constexpr int CT = 8;  // tokens per pass: 32 rows x 8 x 4 bytes = 1 KiB per wave
  static_assert(kWinWaves / 2 * 32 * CT * 4 <= kHalf * Sh::ROWB, "weights fit 32 staged K rows");
  float* pt = reinterpret_cast<float*>(pt_bytes);
  const int l32 = lane & 31, hf = lane >> 5;
  // Rolled loops over an output copy in scratch memory: this rare path must
  // not cost the caller's loop registers.
  float acc[16 * Sh::DB];
#pragma unroll
  for (int i = 0; i < 16 * Sh::DB; i++) acc[i] = o[i / 16][i % 16];
#pragma unroll
  for (int c = 0; c < 32 / CT; c++) {
    // tokens 8c .. 8c+7: registers 4c .. 4c+3 of both halves
#pragma unroll
    for (int i = 0; i < 4; i++) pt[l32 * CT + 4 * hf + i] = s[4 * c + i] * kWeightScale;
#pragma unroll 1
    for (int t = 0; t < CT; t++) {
      const float w = pt[l32 * CT + t];
      const int tok = CT * c + t;
      if (ts + tok > lim) continue;
#pragma unroll 1
      for (int q = 0; q < 16 * Sh::DB; q += 4) {
        // registers q .. q+3: features 32(q / 16) + 8(q % 16 / 4) + 4hf .. +3,
        // unit q / 4, byte 8hf of it
        const char* vp = vst + win_staged<DPH>(tok, q / 4) + 8 * hf;
#pragma unroll 1
        for (int i = 0; i < 4; i++)
          acc[q + i] = fmaf(w, (float)reinterpret_cast<const _Float16*>(vp)[i], acc[q + i]);
      }
    }
  }
#pragma unroll
  for (int i = 0; i < 16 * Sh::DB; i++) o[i / 16][i % 16] = acc[i];
}

template <int DPH>
__global__ __launch_bounds__(kWinThreads) void attn_window_kernel(AttnArgs a) {
  using Sh = WinShape<DPH>;
  __shared__ __attribute__((aligned(16))) char lds[kWinBuffers * 2 * Sh::TILEB];  // [K, V]
  __shared__ int32_t tab[kWinTable];
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int l32 = lane & 31, hf = lane >> 5;

  // Grid position -> (KV head fastest, partition, row group from the heaviest
  // down: a row group's work grows with its place in the window, and the
  // groups that start last should be the short ones).
  const int n = blockIdx.x;
  const int u = wave_uniform(n / a.nkv);
  const int kvh = n - u * a.nkv;
  int rg = wave_uniform(u / a.n_parts);
  const int part = u - rg * a.n_parts;
  rg = a.row_groups - 1 - rg;

  const int r0 = rg * kWinRows;
  const int w0 = r0 + 32 * (wave & 3);  // the wave's first row
  const int half = wave >> 2;           // and its half of every tile's tokens
  const int row = w0 + l32;
  const bool real = row < a.R;
  const int lim = real ? a.pos_base + row / a.G : -1;
  // (divisions run on the vector unit; the loop's bounds and branches below
  // need scalars)
  const int wg_max = wave_uniform(a.pos_base + (min(a.R, r0 + kWinRows) - 1) / a.G);
  const int wg_min = wave_uniform(a.pos_base + r0 / a.G);
  const int wave_max =
      wave_uniform(w0 < a.R ? a.pos_base + (min(a.R, w0 + 32) - 1) / a.G : -1);
  const int wave_min = wave_uniform(a.pos_base + w0 / a.G);
  const int t_begin = part * a.tiles_per_part;
  const int t_end = min(t_begin + a.tiles_per_part, wg_max / kWinTok + 1);
  if (t_begin >= t_end) return;  // nothing here is visible to the row group

  // ---- tile loads, straight into LDS.  A wave's load brings SL consecutive
  // tokens at a multiple of SL (4 or 8; block sizes are multiples of 8), so
  // they share a block, and the address is a scalar base plus a lane offset
  // that never changes.  Lane l's 16 bytes
  // land at unit l % UNITS of token l / UNITS, so it fetches the unit that
  // belongs there (win_staged; its xor depends on the token mod 16 alone).
  constexpr int SL = 64 / Sh::UNITS;             // tokens per wave load
  constexpr int TSTEP = SL * kWinWaves;          // tokens per workgroup load
  static_assert(TSTEP % 16 == 0, "a lane's swizzle is the same in every load");
  const int lt = tid / Sh::UNITS;                // this lane's token of a tile (+ j * TSTEP)
  const int bs = a.src.bs;
  const uint32_t row_bytes = 2u * (uint32_t)a.src.kv_dim;
  const uint32_t v_bytes = (uint32_t)bs * row_bytes;
  const char* head = reinterpret_cast<const char*>(a.src.pool) + (size_t)kvh * Sh::ROWB;
  const uint32_t unit_off =
      (uint32_t)(win_staged<DPH>(lt, lane % Sh::UNITS) - lt * Sh::ROWB);
  const uint32_t lane_off = (uint32_t)(lane / Sh::UNITS) * row_bytes + unit_off;
  const uint32_t lds0 =
      (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lds + 1024u * wave;
  const int step_q = wave_uniform(kWinTok / bs), step_r = kWinTok - step_q * bs;
  const int last_lb = wave_uniform((a.src.L_max - 1) / bs);
  // The block table goes through LDS, kWinTable entries from block tab0 on at
  // a time (a scalar load per tile would be waited for with the LDS operand
  // reads, which share its counter: 1000 cycles of a 2800-cycle step).
  const attn::const_table_t table = attn::const_table(a.src);
  int tab0 = 0;
  auto fill_table = [&](int first) {
    tab0 = first;
#pragma unroll 1
    for (int i = tid; i < kWinTable && first + i <= last_lb; i += kWinThreads)
      tab[i] = a.src.table[first + i];
    __syncthreads();
  };
  int blk[Sh::NU], lb[Sh::NU], slot[Sh::NU], lslot[Sh::NU];
  // logical block and slot of this wave's groups of tile t_begin
#pragma unroll
  for (int j = 0; j < Sh::NU; j++) {
    const int g = t_begin * kWinTok + wave * SL + j * TSTEP;
    lb[j] = wave_uniform(g / bs);
    slot[j] = g - lb[j] * bs;
  }
  // Looks up the blocks of tile t (called for t_begin, t_begin + 1, ...).
  // Groups past L_max take the last written token's block and slot.
  int lb_hi = wave_uniform((t_begin * kWinTok + kWinTok - 1) / bs), slot_hi =
      t_begin * kWinTok + kWinTok - 1 - lb_hi * bs;  // the tile's last token
  // `first`: read from memory (scalar loads), before the table is in LDS.
  auto load_blk = [&](int t, bool first) {
    if (!first && min(lb_hi, last_lb) - tab0 >= kWinTable) {
      __syncthreads();
      fill_table(min(lb_hi - step_q - 1, last_lb));  // (from the tile's first block or before)
    }
    lb_hi += step_q;
    slot_hi += step_r;
    if (slot_hi >= bs) {
      slot_hi -= bs;
      ++lb_hi;
    }
#pragma unroll
    for (int j = 0; j < Sh::NU; j++) {
      const bool in = t * kWinTok + wave * SL + j * TSTEP < a.src.L_max;
      const int at = in ? lb[j] : last_lb;
      if (first)
        blk[j] = table[at];
      else
        blk[j] = tab[at - tab0];
      lslot[j] = in ? slot[j] : a.src.L_max - 1 - last_lb * bs;
      lb[j] += step_q;
      slot[j] += step_r;
      if (slot[j] >= bs) {
        slot[j] -= bs;
        ++lb[j];
      }
    }
  };
  // Lanes whose token is at or past L_max read their group's first token
  // (its logits are masked).
  auto load_tile = [&](int t) {
    const uint32_t dst = lds0 + (uint32_t)((t - t_begin) % kWinBuffers) * (2 * Sh::TILEB);
    const bool full = (t + 1) * kWinTok <= a.src.L_max;
#pragma unroll
    for (int j = 0; j < Sh::NU; j++) {
      const char* p = head + (uint64_t)(uint32_t)wave_uniform(blk[j]) * (2ull * v_bytes) +
                      (uint64_t)((uint32_t)lslot[j] * row_bytes);
      const uint32_t off =
          full || t * kWinTok + lt + j * TSTEP < a.src.L_max ? lane_off : unit_off;
      load_to_lds(p, off, dst + j * (1024 * kWinWaves));
      load_to_lds(p + v_bytes, off, dst + Sh::TILEB + j * (1024 * kWinWaves));
    }
  };
  // Tile t is in LDS for every wave afterwards; whether a position hidden
  // from some row of the workgroup holds a non-finite V element in it.
  auto arrive = [&](int t, const char* vst) {
    wait_loads();
    if ((t + 1) * kWinTok - 1 <= wg_min) {
      __syncthreads();
      return 0;
    }
    int bad = 0;
#pragma unroll
    for (int j = 0; j < Sh::NU; j++) {  // (what this lane's own loads brought)
      const uint4 v =
          *reinterpret_cast<const uint4*>(vst + j * (1024 * kWinWaves) + 1024 * wave + 16 * lane);
      if (t * kWinTok + lt + j * TSTEP > wg_min &&
          (attn::nonfinite_h2(v.x) | attn::nonfinite_h2(v.y) | attn::nonfinite_h2(v.z) |
           attn::nonfinite_h2(v.w)) != 0)
        bad = 1;
    }
    return wave_uniform(__syncthreads_or(bad));
  };

  load_blk(t_begin, true);
  load_tile(t_begin);

  // ---- q operand: row l % 32, features 16ks + 8(l / 32) .. +7
  h8_t qh[Sh::KS], ql[Sh::KS];
  {
    const int gr = min(row, a.R - 1);
    const int m = gr / a.G;
    const int h = kvh * a.G + (gr - m * a.G);
    const float* qp = a.q + (size_t)m * a.nh * DPH + (size_t)h * DPH + 8 * hf;
    const float sc = real ? a.qscale : 0.f;
#pragma unroll
    for (int ks = 0; ks < Sh::KS; ks++) {
      float x[8];
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const float2 v = *reinterpret_cast<const float2*>(qp + 16 * ks + 2 * i);
        x[2 * i] = v.x * sc;
        x[2 * i + 1] = v.y * sc;
      }
      attn::split_h8(x, qh[ks], ql[ks]);
    }
  }

  // (the first tile is on its way)
  fill_table(wave_uniform((t_begin + 1) * kWinTok / bs));
  if (t_begin + 1 < t_end) load_blk(t_begin + 1, false);

  // The weights' reference (a running max, raised lazily) enters the logits
  // product as its initial accumulator.
  float m_neg = 0.f, seen = 0.f, l_run = 0.f;
  f16_t o[Sh::DB];
#pragma unroll
  for (int db = 0; db < Sh::DB; db++)
#pragma unroll
    for (int i = 0; i < 16; i++) o[db][i] = 0.f;

  // transposed V reads: lane -> token 4(l/32) + (l%16)/4 of an 8-token
  // group's half, features 32db + 16((l/16)%2) + 4(l%4) .. +3
  const int vt = 4 * hf + ((lane & 15) >> 2);
  const int vu = 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1);
  const int vsub = 8 * (lane & 1);
  // Logits of 32 tokens from position ts on, relative to the reference: lane
  // holds row l % 32, tokens 8(i / 4) + 4(l / 32) + i % 4.  Operand reads are
  // issued in batches ahead of their products (the scheduling barriers): read
  // one by one, each product would wait out the LDS latency.  k8: the first
  // batch, already read.  The hi and lo products go to accumulators of their
  // own: one chain of dependent products would run at their latency, twice
  // their issue time.
  constexpr int kBatch = 4;
  auto read_k = [&](const char* kst, int k0, h8_t (&k8)[kBatch]) {
#pragma unroll
    for (int ks = 0; ks < kBatch; ks++)
      k8[ks] = __builtin_bit_cast(
          h8_t, *reinterpret_cast<const uint4*>(kst + win_staged<DPH>(l32, 2 * (k0 + ks) + hf)));
  };
  auto logits = [&](int ts, const char* kst, h8_t (&k8)[kBatch]) {
    f16_t s, s2;
#pragma unroll
    for (int i = 0; i < 16; i++) {
      s[i] = m_neg;
      s2[i] = 0.f;
    }
#pragma unroll
    for (int k0 = 0; k0 < Sh::KS; k0 += kBatch) {
      h8_t kn[kBatch];
      if (k0 + kBatch < Sh::KS) read_k(kst, k0 + kBatch, kn);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int ks = 0; ks < kBatch; ks++) {
        s = __builtin_amdgcn_mfma_f32_32x32x16_f16(k8[ks], qh[k0 + ks], s, 0, 0, 0);
        s2 = __builtin_amdgcn_mfma_f32_32x32x16_f16(k8[ks], ql[k0 + ks], s2, 0, 0, 0);
      }
      if (k0 + kBatch < Sh::KS) {
#pragma unroll
        for (int ks = 0; ks < kBatch; ks++) k8[ks] = kn[ks];
      }
    }
#pragma unroll
    for (int i = 0; i < 16; i++) s[i] += s2[i];
    if (ts + 31 > wave_min) {
      const int left = lim - ts - 4 * hf;
#pragma unroll
      for (int i = 0; i < 16; i++) s[i] = 8 * (i / 4) + (i & 3) <= left ? s[i] : -INFINITY;
    }
    float mx = s[0];
#pragma unroll
    for (int i = 1; i < 16; i++) mx = fmaxf(mx, s[i]);
    mx = half_max(mx);
    // Raise the reference when a row's max is more than 2^kLazyMax above it,
    // or is the row's first.
    if (__builtin_amdgcn_ballot_w64(mx > kLazyMax || (seen == 0.f && mx > -INFINITY)) != 0) {
      const float up = seen == 0.f ? mx : fmaxf(mx, 0.f);
      const float d = up == -INFINITY ? 0.f : up;
      const float al = seen == 0.f ? 0.f : __builtin_amdgcn_exp2f(-d);
      m_neg -= d;
      seen = seen != 0.f || mx > -INFINITY ? 1.f : 0.f;
      l_run *= al;
#pragma unroll
      for (int db = 0; db < Sh::DB; db++) o[db] *= al;
#pragma unroll
      for (int i = 0; i < 16; i++) s[i] -= d;
    }
    return s;
  };
  auto weights = [&](f16_t& s) {
    float ps[2] = {0.f, 0.f};
#pragma unroll
    for (int i = 0; i < 16; i++) {
      s[i] = __builtin_amdgcn_exp2f(s[i]);
      ps[i & 1] += s[i];
    }
    l_run += ps[0] + ps[1];
  };

  // Step t: tile t arrives; the loads of tile t + 1 start into the buffer of
  // tile t - 1, which every wave left before that barrier.
  int t = t_begin, exact = 0;
  const char* kst = nullptr;
  auto next = [&]() {
    kst = lds + ((t - t_begin) % kWinBuffers) * 2 * Sh::TILEB;
    exact = arrive(t, kst + Sh::TILEB);
    if (t + 1 < t_end) {
      load_tile(t + 1);
      load_blk(t + 2, false);
    }
  };
  for (next(); !exact;) {
    const int ts = t * kWinTok + kHalf * half;
    const char* kh = kst + half * kHalf * Sh::ROWB;
    const char* vh = kh + Sh::TILEB;
    if (ts <= wave_max) {  // wave-uniform
      h8_t k8[kBatch];
      read_k(kh, 0, k8);
      f16_t s = logits(ts, kh, k8);
      // The V operand reads of the first 16 tokens are in flight while the
      // weights are formed, those of the last 16 during the products.
      s4_t vr[2][Sh::DB][2];
      auto read_v = [&](int k2) {
#pragma unroll
        for (int db = 0; db < Sh::DB; db++)
#pragma unroll
          for (int g = 0; g < 2; g++)
            vr[k2][db][g] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4_t*)(
                vh + win_staged<DPH>(16 * k2 + 8 * g + vt, 4 * db + vu) + vsub));
      };
      read_v(0);
      __builtin_amdgcn_sched_barrier(0);
      weights(s);
      h8_t ph[2], pl[2];
#pragma unroll
      for (int k2 = 0; k2 < 2; k2++) {
        float x[8];
#pragma unroll
        for (int i = 0; i < 8; i++) x[i] = s[8 * k2 + i] * kWeightScale;
        split_weights(x, ph[k2], pl[k2]);
      }
      read_v(1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int k2 = 0; k2 < 2; k2++) {
#pragma unroll
        for (int db = 0; db < Sh::DB; db++)
          o[db] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(h8_t, vr[k2][db]),
                                                         ph[k2], o[db], 0, 0, 0);
#pragma unroll
        for (int db = 0; db < Sh::DB; db++)
          o[db] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(h8_t, vr[k2][db]),
                                                         pl[k2], o[db], 0, 0, 0);
      }
    }
    if (++t == t_end) break;
    next();
  }
  // From a tile that needs it on, every product takes the exact form.
  while (t < t_end) {
    const int ts = t * kWinTok + kHalf * half;
    char* kh = const_cast<char*>(kst) + half * kHalf * Sh::ROWB;
    f16_t s;
    if (ts <= wave_max) {
      h8_t k8[kBatch];
      read_k(kh, 0, k8);
      s = logits(ts, kh, k8);
      weights(s);
    }
    __syncthreads();  // every wave is past its logits: the K tile is dead
    if (ts <= wave_max)
      win_exact_pv<DPH>(ts, lane, lim, s, kh + (wave & 3) * 1024, kh + Sh::TILEB, o);
    if (++t < t_end) next();
  }

  // ---- the token halves meet: the upper half's waves leave their sums in
  // LDS (the tiles are dead), the lower half's merge them
  static_assert(4 * 32 * DPH * 4 <= sizeof(lds), "sums fit the tiles' LDS");
  float l_row = attn::half_pair_total(l_run, l_run);
  float m_row = seen != 0.f ? -m_neg : -INFINITY;
  f4_t* xo = reinterpret_cast<f4_t*>(lds) + (wave & 3) * (8 * DPH) + lane;  // [i][lane]
  float2* xml = reinterpret_cast<float2*>(tab) + (wave & 3) * 32 + l32;
  __syncthreads();
  if (half == 1) {
#pragma unroll
    for (int i = 0; i < 4 * Sh::DB; i++)
      xo[64 * i] = f4_t{o[i / 4][4 * (i & 3)], o[i / 4][4 * (i & 3) + 1],
                        o[i / 4][4 * (i & 3) + 2], o[i / 4][4 * (i & 3) + 3]};
    *xml = make_float2(m_row, l_row);
  }
  __syncthreads();
  if (half == 1 || !real) return;
  {
    const float2 y = *xml;
    const float m = fmaxf(m_row, y.x);
    const float wa0 = sums_weight(m_row, l_row, m);
    const float wa1 = sums_weight(y.x, y.y, m);
    m_row = m;
    l_row = l_row * wa0 + y.y * wa1;
    const float wo0 = wa0 * (1.f / kWeightScale), wo1 = wa1 * (1.f / kWeightScale);
#pragma unroll
    for (int i = 0; i < 4 * Sh::DB; i++) {
      const f4_t x = xo[64 * i];
#pragma unroll
      for (int e = 0; e < 4; e++)
        o[i / 4][4 * (i & 3) + e] = o[i / 4][4 * (i & 3) + e] * wo0 + x[e] * wo1;
    }
  }
  const int m = row / a.G;
  const int h = kvh * a.G + (row - m * a.G);
  if (a.n_parts == 1) {
    const float inv = attn::finish_scale(l_row);
    // (out is 8-byte aligned)
    float* dst = a.out + (size_t)m * a.nh * DPH + (size_t)h * DPH + 4 * hf;
#pragma unroll
    for (int db = 0; db < Sh::DB; db++)
#pragma unroll
      for (int j = 0; j < 4; j++) {
        float2* d = reinterpret_cast<float2*>(dst + 32 * db + 8 * j);
        d[0] = make_float2(o[db][4 * j] * inv, o[db][4 * j + 1] * inv);
        d[1] = make_float2(o[db][4 * j + 2] * inv, o[db][4 * j + 3] * inv);
      }
  } else {
    const size_t pr = ((size_t)kvh * a.R + row) * a.n_parts + part;
    float* dst = a.partials + pr * DPH + 4 * hf;
#pragma unroll
    for (int db = 0; db < Sh::DB; db++)
#pragma unroll
      for (int j = 0; j < 4; j++)
        *reinterpret_cast<float4*>(dst + 32 * db + 8 * j) =
            make_float4(o[db][4 * j], o[db][4 * j + 1], o[db][4 * j + 2], o[db][4 * j + 3]);
    if (hf == 0)
      reinterpret_cast<float2*>(a.partials + (size_t)a.nkv * a.R * a.n_parts * DPH)[pr] =
          make_float2(m_row, l_row);
  }
}

// Log-sum-exp merge of the partitions a row sees, in partition order: one
// thread per (KV head, row, 4 features).  A kernel of its own: the rows'
// partials are read by all CUs, where one workgroup per row group would
// wait for them alone.
template <int DPH>
__global__ __launch_bounds__(256) void window_combine_kernel(AttnArgs a) {
  constexpr int C = DPH / 4;
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  const size_t kr = i / C;
  if (kr >= (size_t)a.nkv * a.R) return;
  const int c = (int)(i - kr * C);
  const int kvh = (int)(kr / a.R), row = (int)(kr - (size_t)kvh * a.R);
  const int m = row / a.G;
  const int h = kvh * a.G + (row - m * a.G);
  const int P = (a.pos_base + m) / (a.tiles_per_part * kWinTok) + 1;
  const float* acc = a.partials + kr * a.n_parts * DPH + 4 * c;
  const float2* ml = reinterpret_cast<const float2*>(
                         a.partials + (size_t)a.nkv * a.R * a.n_parts * DPH) + kr * a.n_parts;
  float mx = -INFINITY, l = 0.f;
  float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
  // Batches of four partitions, every load of a batch in flight together
  // (partitions past the last re-read it and are left out: a weight of 0 would
  // make NaN of Inf).
  for (int p0 = 0; p0 < P; p0 += 4) {
    float2 v[4];
    float4 x[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int p = min(p0 + i, P - 1);
      v[i] = ml[p];
      x[i] = *reinterpret_cast<const float4*>(acc + (size_t)p * DPH);
    }
    float top = mx;
#pragma unroll
    for (int i = 0; i < 4; i++) top = fmaxf(top, v[i].x);
    const float old = mx == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mx - top);
    mx = top;
    l *= old;
    o.x *= old;
    o.y *= old;
    o.z *= old;
    o.w *= old;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const bool in = p0 + i < P;
      const float w = sums_weight(v[i].x, v[i].y, mx);
      l += in ? v[i].y * w : 0.f;
      o.x += in ? x[i].x * w : 0.f;
      o.y += in ? x[i].y * w : 0.f;
      o.z += in ? x[i].z * w : 0.f;
      o.w += in ? x[i].w * w : 0.f;
    }
  }
  const float inv = attn::finish_scale(l);
  float2* d = reinterpret_cast<float2*>(a.out + (size_t)m * a.nh * DPH + (size_t)h * DPH + 4 * c);
  d[0] = make_float2(o.x * inv, o.y * inv);
  d[1] = make_float2(o.z * inv, o.w * inv);
}

// The 16-row kernels spread a window over the chip in one round as long as
// its rows and keys are few, and start faster (this kernel's first tile is
// some 4 us away); their cost then grows by rounds, and with every 16 rows
// re-reading the keys.  Measured on MI355X, us per call, 16-row kernels /
// this one, by rows x keys over all KV heads:
//   32/8 heads of 128: 48 queries after 4000 keys (6M) 27.3 / 28.6, 64 (8M)
//     28.0 / 29.2, 96 (12M) 41.2 / 33.9, 128 (16M) 43.6 / 36.6; 24 after 16000
//     (12M) 44.5 / 33.3;
//   32/4 heads of 64: 64 after 4000 (8M) 17.6 / 21.3, 96 (12M) 24.7 / 23.5,
//     128 (16M) 26.1 / 25.7; 24 after 16000 (12M) 27.0 / 26.4;
//   28/4 heads of 128: 64 after 4000 (7M) 28.2 / 29.6, 128 (14M) 43.1 / 34.6.
// So from 11M rows x keys on it serves wherever it was measured faster, and
// from 16384 rows on, where the grid is half full without a split, from 8M.
// Below either line both kernels occur as the faster one: the 16-row kernels
// lose where their groups have just begun another round, without context
// from some 9000 rows on (32/8 heads of 128: 256 queries alone 18.3 / 18.7,
// 320 32.4 / 23.9, 511 42.0 / 29.6, 512 41.9 / 29.4; of 64: 9.9 / 12.2, 18.8 /
// 16.0, 24.8 / 18.6, 24.5 / 18.5; 28/4: 17.5 / 18.2, 31.9 / 22.8, 41.7 / 28.2,
// 41.6 / 28.1), with fewer KV heads later (16/2: 511 22.0 / 24.3, 640 37.8 /
// 26.3) and with context between (256 after 512 keys, 6M, 32/8 heads of 128
// 25.7 / 27.6, after 1000, 10M, 48.5 / 31.9): these lines give that up.
bool window_serves(int L_max, int nkv, int R) {
  const int64_t rows = (int64_t)nkv * R;
  return R >= 96 && rows * L_max >= (rows >= 16384 ? (int64_t)8 << 20 : (int64_t)11 << 20);
}

size_t window_partial_bytes(const WindowPlan& p, int nkv, int R, int dph) {
  return p.n_parts > 1 ? (size_t)nkv * R * p.n_parts * (size_t)(dph + 2) * sizeof(float) : 0;
}

WindowPlan window_plan(int L_max, int nkv, int R, int dph, int n_cus, int max_parts,
                       size_t max_bytes) {
  WindowPlan p;
  p.row_groups = (R + kWinRows - 1) / kWinRows;
  const int n_tiles = (L_max + kWinTok - 1) / kWinTok;
  const int64_t units = (int64_t)nkv * p.row_groups;
  int64_t parts = (int64_t)n_cus / units;  // one workgroup per CU
  if (parts > max_parts) parts = max_parts;
  if (parts > n_tiles / 2) parts = n_tiles / 2;
  const int64_t by_bytes =
      (int64_t)(max_bytes / ((size_t)nkv * R * (size_t)(dph + 2) * sizeof(float)));
  if (parts > by_bytes) parts = by_bytes;
  if (parts < 1) parts = 1;
  p.tiles_per_part = (int)((n_tiles + parts - 1) / parts);
  p.n_parts = (n_tiles + p.tiles_per_part - 1) / p.tiles_per_part;
  return p;
}

template <int DPH>
static int launch_window(const AttnArgs& a, hipStream_t stream) {
  const int64_t total = (int64_t)a.nkv * a.n_parts * a.row_groups;
  attn_window_kernel<DPH><<<dim3((unsigned)total), dim3(kWinThreads), 0, stream>>>(a);
  int st = launch_status();
  if (st != SDE_OK || a.n_parts == 1) return st;
  const int64_t threads = (int64_t)a.nkv * a.R * (DPH / 4);
  window_combine_kernel<DPH><<<dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, stream>>>(a);
  return launch_status();
}

int window_attention(const attn::AttnArgs& args, const WindowPlan& p, int dph,
                     hipStream_t stream) {
  AttnArgs a = args;
  a.row_groups = p.row_groups;
  a.n_parts = p.n_parts;
  a.tiles_per_part = p.tiles_per_part;
  return dph == 128 ? launch_window<128>(a, stream) : launch_window<64>(a, stream);
}

}  // namespace win
}  // namespace sde
