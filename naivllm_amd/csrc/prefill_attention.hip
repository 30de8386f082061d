// Causal prefill attention for gfx950 (bf16): every new row of a prompt
// attends keys 0 .. its position, from the paged cache (a prompt behind a
// cached prefix) or from the step's own contiguous K/V.
//
// Behaviour follows the reference's prefill attention
// (src/myvllm/layers/attention.py:123-363: the varlen path over contiguous
// K/V and the paged path behind a cached prefix); the kernel is this
// library's own.
//
// What bounds it: two matrix products of 4 D flops per (row, key) pair,
// against one exponential per pair (a quarter-rate VALU operation, about as
// long as the pair's products).  The host cuts the rows of all sequences
// into tiles (heaviest first); a workgroup takes one tile of rows for HW
// query heads of one kv head, so its K/V tiles, staged once in LDS, serve
// HW heads.  A wave holds 32 rows: S^T = K Q^T on v_mfma_f32_32x32x16_bf16
// puts a row's scores into two lanes' registers (the row maximum is a
// register tree and one permlane swap), and its result layout is the B
// operand of O^T = V^T P^T, V^T coming from the transposing LDS reads.  The
// workgroup ids of one kv head agree mod 8 at 8 kv heads, so a head's K/V
// stays in one XCD's L2.
//
// Measured on MI355X (the verify kernel on causal blocks of 64 / G rows,
// which every prefill ran on before -> this kernel): 8 prompts of ~1000
// tokens, 16/8 heads, 538 -> 69 us (475 TFLOP/s); prompts of 2900 and 4050
// tokens behind 4096 cached keys, 32/8 heads, 5283 -> 790-815 us (820-850);
// 8192 tokens, 32/8 heads, 600 us (916); one prompt of 1206 tokens, 16/8
// heads, 85 -> 32 us.  What the parts of it gave was measured with an exponent
// reference moved lazily, which is less precise (see there): these four 59,
// 725, 535 and 31 us; with K/V staged through registers instead of straight to
// LDS and both waves of a SIMD in step 59-64, 781-793, 590 and 31.

#include "common.h"

#include <algorithm>
#include <array>
#include <new>
#include <vector>

namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef short i16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) i16x4 lds_i16x4;

constexpr int kKeys = 64;          // keys per tile
constexpr int kWaveRows = 32;      // query rows per wave
constexpr int kMaxPages = 2048;    // block-table entries in LDS at a time
constexpr int kTileWords = 8;      // int32 words of a tile record
constexpr float kNegInf = -__builtin_inff();
// keys of a workgroup's range up to which every 32 keys have an exponent
// reference of their own, every 64 beyond
constexpr int kFineKeys = 256;
// how far (log2 domain) a maximum may lie below the row's running one for the
// reference to move down to it (sums stay within 2^16 of their count)
constexpr float kRefDrop = 16.f;

struct PrefillArgs {
  const bf16_t* q;
  const bf16_t* k;
  const bf16_t* v;
  bf16_t* out;
  const int32_t* block_tables;  // null: contiguous K/V
  const int32_t* tiles;         // [ntiles][kTileWords]: sequence, first row, rows, first position, first K/V row,
                                // first key, end key, partial slot (-1: the tile's only part)
  float* part;                  // [slots][H][tile_rows][DH + 2]: unnormalised rows, then (max, sum) pairs
  int tile_rows;
  float scale_log2;
  int H, Hkv, bs_log2, max_blocks;
  int hw;                       // query heads of a kv head one workgroup serves
  int hgroups;                  // workgroups per (tile, kv head): (H / Hkv) / hw
};

__device__ __forceinline__ bf16x8 as_bf16x8(u32x4 v) { return __builtin_bit_cast(bf16x8, v); }

__device__ __forceinline__ uint2 lds_read_tr(const unsigned char* p) {
  const i16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(p));
  return __builtin_bit_cast(uint2, v);
}

// the other half-wave's value of the same row (lane ^ 32) combined
__device__ __forceinline__ float half_max(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float half_sum(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

template <int DH, int NW>
__global__ __launch_bounds__(NW * 64, 2) void prefill_attn_kernel(PrefillArgs a) {
  constexpr int NT = NW * 64;
  constexpr int CPR = DH / 8;              // 16-byte chunks per row
  constexpr int ROWB = DH * 2;             // bytes per staged row
  constexpr int KS = DH / 16;              // k-steps of S^T
  constexpr int DT = DH / 32;              // 32-dim tiles of O^T
  constexpr int RPI = 64 / CPR;            // rows one load instruction of a wave fills
  constexpr int J = kKeys / RPI / NW;      // K (and V) loads per wave and tile
  constexpr int TILEB = kKeys * ROWB;
  constexpr bool SKEW = NW == 8;           // see the loop
  // tiles loading ahead, and the K and V tiles staged for it: two ahead with
  // one workgroup per CU; one ahead for two 4-wave workgroups to fit a CU
  constexpr int DIST = SKEW ? 2 : 1;
  constexpr int KB = DIST + 1, VB = DIST + 1 + SKEW;
  static_assert(J >= 1 && kKeys % (RPI * NW) == 0, "whole tiles per pass");
  struct __attribute__((aligned(16))) Lds {
    int pages[kMaxPages];
    int holes, first;  // some page unmapped; first mapped page
    __attribute__((aligned(16))) unsigned char kt[KB][TILEB];
    __attribute__((aligned(16))) unsigned char vt[VB][TILEB];
  };
  __shared__ Lds lds;

  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 31, h = lane >> 5;
  // workgroup -> (tile, head group, kv head), the kv head fastest
  const int hk = blockIdx.x % a.Hkv;
  const int rest = blockIdx.x / a.Hkv;
  const int hg = rest % a.hgroups;
  const int32_t* rec = a.tiles + (int64_t)(rest / a.hgroups) * kTileWords;
  const int seq = rec[0], row0 = rec[1], nrows = rec[2], pos0 = rec[3], kv0 = rec[4];
  const int key_begin = rec[5], slot = rec[7];
  const int wph = NW / a.hw;               // waves per head
  const int head = hk * (a.H / a.Hkv) + hg * a.hw + w / wph;
  const int r0 = (w % wph) * kWaveRows;    // this wave's first row in the tile
  const bool paged = a.block_tables != nullptr;
  const int bs_mask = (1 << a.bs_log2) - 1;
  int key_end = min(rec[6], pos0 + nrows);  // (keys past the tile's last row are never attended)
  if (paged) key_end = min(key_end, a.max_blocks << a.bs_log2);  // the table's width
  const int64_t tok = (int64_t)a.Hkv * DH; // elements between consecutive keys

  // query rows as the B operand of S^T: lane (h, col) holds row col, dims 16 ks + 8 h .. + 7
  bf16x8 qB[KS];
  {
    const int r = min(r0 + col, nrows - 1);  // rows past the tile's last load it and are not stored
    const bf16_t* src = a.q + ((int64_t)(row0 + r) * a.H + head) * DH + h * 8;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) qB[ks] = as_bf16x8(*reinterpret_cast<const u32x4*>(src + ks * 16));
  }
  const int pos = pos0 + r0 + col;           // position of this lane's row
  const int pos_first = pos0 + r0;           // of the wave's first row
  const int pos_last = min(pos_first + kWaveRows - 1, pos0 + nrows - 1);

  // Block-table entries in LDS: entry i from the first page on at slot i mod
  // kMaxPages, the first kMaxPages here, the rest half a ring at a time once
  // the loop has left the half they replace.
  const int pg0 = key_begin >> a.bs_log2;
  const int npg = ((key_end + bs_mask) >> a.bs_log2) - pg0;
  const int32_t* bt = paged ? a.block_tables + (int64_t)seq * a.max_blocks + pg0 : nullptr;
  int staged = kMaxPages;
  if (paged) {
    if (tid == 0) {
      lds.holes = 0;
      lds.first = 0x7fffffff;
    }
    __syncthreads();
    for (int i = tid; i < npg; i += NT) {
      const int p = bt[i];
      if (i < kMaxPages) lds.pages[i] = p;
      if (p < 0) lds.holes = 1;
    }
    __syncthreads();
  }
  auto page = [&](int key) { return lds.pages[((key >> a.bs_log2) - pg0) & (kMaxPages - 1)]; };
  // the ring's next half, at the start of key tile n0's step (by every wave;
  // the waves a step behind still read tile n0 - kKeys, the loads ahead reach
  // 4 tiles, 256 pages at most, past that one: its first use is behind the
  // step's barrier)
  auto turn_pages = [&](int n0) {
    if (!paged || staged >= npg) return;  // uniform
    const int low = (max(n0 - kKeys, key_begin) >> a.bs_log2) - pg0;
    if (low < staged - kMaxPages / 2) return;  // uniform
    const int end = min(staged + kMaxPages / 2, npg);
    for (int i = staged + tid; i < end; i += NT) lds.pages[i & (kMaxPages - 1)] = bt[i];
    staged += kMaxPages / 2;
  };
  const bool holes = paged && __builtin_amdgcn_readfirstlane(lds.holes) != 0;
  int64_t spare = 0;  // the row an unmapped key reads instead (of a key that exists; its weight is zero)
  if (holes) {        // uniform
    for (int i = tid; i < npg; i += NT)
      if (bt[i] >= 0) atomicMin(&lds.first, i);
    __syncthreads();
    const int first = __builtin_amdgcn_readfirstlane(lds.first);
    if (first >= npg) key_end = key_begin;  // no key at all
    else spare = (int64_t)bt[first] << a.bs_log2;
  }

  // K/V rows of a tile go from memory straight to LDS (no registers, no LDS
  // stores): instruction j of wave w fills rows (w J + j) RPI .. with 16-byte
  // chunk X of row r at slot X ^ (r % CPR) (K), X ^ 4 (r % 4) (V), so that the
  // operand reads of a half-wave touch every bank once; the lane picks the
  // chunk its slot holds.  Rows past the last key read it again (masked).
  auto vswz = [](int r) { return ((r & 3) << 2) & (CPR - 1); };
  // (Issued from asm: the compiler would wait for every such load before the
  // next LDS read of any buffer.  The loads have no register result; the
  // waits below and the barriers order them.)
  auto load_lds = [&](const bf16_t* src, unsigned char* dst) {
    const uint32_t at = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)dst);
    __asm__ volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(at), "v"(src) : "memory", "m0");
  };
  auto issue = [&](int kb, int vb, int n0) {
#pragma unroll
    for (int j = 0; j < J; ++j) {
      const int r0j = (w * J + j) * RPI;
      const int r = r0j + lane / CPR, sl = lane % CPR;
      const int kc = min(n0 + r, key_end - 1);
      int64_t row = kv0 + kc;
      if (paged) {
        const int p = page(kc);
        row = p >= 0 ? ((int64_t)p << a.bs_log2) + (kc & bs_mask) : spare;
      }
      const int64_t off = row * tok + hk * DH;
      load_lds(a.k + off + ((sl ^ (r & (CPR - 1))) << 3), &lds.kt[kb][r0j * ROWB]);
      load_lds(a.v + off + ((sl ^ vswz(r)) << 3), &lds.vt[vb][r0j * ROWB]);
    }
  };
  // tile n0's loads landed, `ahead` tiles after it still in flight (the
  // wave's own; the barrier that follows makes the tile whole)
  auto landed = [&](bool ahead) {
    if (DIST == 2 && ahead) __asm__ volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * J) : "memory");
    else __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");
  };

  f32x16 acc[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[dt][i] = 0.f;
  float m_ref = kNegInf, m_run = kNegInf, l_run = 0.f;  // exponent reference, running maximum, running sum
  const float sc = a.scale_log2;

  f32x16 s[2];
  // scores of a tile (every key of a skipped tile lies past this wave's rows)
  auto scores = [&](int kb, int n0) {
    if (n0 > pos_last) return;  // uniform
    const unsigned char* kt = lds.kt[kb];
    // K operands KH steps at a time, both 32-key halves, the next group's
    // reads in flight while one is multiplied (left to itself the compiler
    // waits for each read before its product); the halves alternate, so no
    // product waits for the one before it
    constexpr int KH = KS / 2;
    u32x4 ka[2][2][KH];
    auto read = [&](int g) {
#pragma unroll
      for (int ks = 0; ks < KH; ++ks)
#pragma unroll
        for (int t = 0; t < 2; ++t)
          ka[g][t][ks] = *reinterpret_cast<const u32x4*>(
              kt + (t * 32 + col) * ROWB + ((((g * KH + ks) * 2 + h) ^ (col & (CPR - 1))) << 4));
    };
    read(0);
    read(1);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int g = 0; g < 2; ++g)
#pragma unroll
      for (int ks = 0; ks < KH; ++ks)
#pragma unroll
        for (int t = 0; t < 2; ++t)
          s[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
              as_bf16x8(ka[g][t][ks]), qB[g * KH + ks],
              g == 0 && ks == 0 ? f32x16{0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f} : s[t],
              0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
  };
  auto values = [&](int vb, int n0) {  // softmax of the tile's scores, O^T += V^T P^T
    if (n0 > pos_last) return;  // uniform
    const unsigned char* vt = lds.vt[vb];
    // lane (h, col), element i of tile t: key n0 + 32 t + 8 (i / 4) + 4 h + i % 4, row col
    if (n0 + kKeys - 1 > pos_first) {  // uniform: some key lies past the wave's first row
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int key = t * 32 + (i >> 2) * 8 + h * 4 + (i & 3);
          s[t][i] = key <= pos - n0 ? s[t][i] : kNegInf;
        }
    }
    if (holes) {  // uniform
      const int key = min(n0 + lane, key_end - 1);
      const uint64_t mapped = __ballot(page(key) >= 0) >> (4 * h);
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i)
          s[t][i] = (mapped >> (t * 32 + (i >> 2) * 8 + (i & 3))) & 1 ? s[t][i] : kNegInf;
    }
    // A weight at its exponent reference is exactly 1 in bf16, every other is
    // rounded: the error falls with the number of references a row has, so
    // the reference is the maximum of each group of 32 keys at first and of
    // each tile later, moved down as well as up (a weight stays <= 1, and the
    // sums within 2^kRefDrop of their count).  Error against 64 bits at N(0, 1)
    // scores, in 1e-5 (the verify kernel on causal blocks; one reference,
    // moved lazily -> these): one prompt of 1,206 tokens 193; 204 -> 192, 40
    // rows behind 256 keys 203; 229 -> 203, 900 behind 2,048 216; 231 -> 205.
    // The rescaling costs up to 8% of the time (lazily moved -> these, 2,900
    // and 4,050 rows of 32/8 heads behind 4,096 keys 730 -> 790 us, 8,192
    // tokens 552 -> 595, one prompt of 1,206 32 -> 33.5), and 4% more where the
    // second reference is moved between the products instead of before them.
    // Not precise enough: a reference every 64 keys from the first key on
    // (1,206 tokens 196, 40 rows behind 256 keys 209), every 128 keys past the
    // first 256 (4,050 rows behind 4,096 keys 221; the verify kernel 220).
    const bool fine = n0 < key_begin + kFineKeys;  // uniform
    float mx[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      mx[t] = s[t][0];
#pragma unroll
      for (int i = 1; i < 16; ++i) mx[t] = fmaxf(mx[t], s[t][i]);
    }
    mx[0] = half_max(fine ? mx[0] : fmaxf(mx[0], mx[1]));
    // the reference moved to a group's maximum; returns the factor of what was summed before
    auto move = [&](float m) {
      m_run = fmaxf(m_run, m);
      const bool on = m > kNegInf && !((m_run - m) * sc > kRefDrop);
      const float alpha = on ? __builtin_amdgcn_exp2f((m_ref - m) * sc) : 1.f;  // (from -inf: 0)
      m_ref = on ? m : m_ref;
      return alpha;
    };
    auto rescale = [&](float alpha) {
      if (!__ballot(alpha != 1.f)) return;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[dt][i] *= alpha;
    };
    const float alpha0 = move(mx[0]);
    const float nb0 = m_ref == kNegInf ? 0.f : -m_ref * sc;
    float alpha1 = 1.f, nb1 = nb0;  // of the tile's second 32 keys
    if (fine) {  // uniform
      alpha1 = move(half_max(mx[1]));
      nb1 = m_ref == kNegInf ? 0.f : -m_ref * sc;
    }
    rescale(alpha0);
    l_run *= alpha0;
    // O^T += V^T P^T, 16 keys per step: element j of lane half h is key
    // 8 (j / 4) + 4 h + j % 4 of the step in both operands.  A step's weights
    // are computed, and its V operands read, during the step before's products.
    constexpr int ST = kKeys / 16;
    uint2 va[2][DT][2];
    auto read = [&](int st) {
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        // 16-lane group (h, g): rows 4 h + 0..3 of the step (then + 8), dims 32 dt + 16 g .. + 15
        const int i = lane & 15, g = (lane >> 4) & 1;
        const int r = h * 4 + (i >> 2);
        const int X = dt * 4 + g * 2 + ((i & 3) >> 1);
        const unsigned char* src = vt + r * ROWB + ((X ^ vswz(r)) << 4) + (i & 1) * 8 + st * 16 * ROWB;
        va[st & 1][dt][0] = lds_read_tr(src);  // (vswz(r + 8) == vswz(r))
        va[st & 1][dt][1] = lds_read_tr(src + 8 * ROWB);
      }
    };
    bf16x8 pB[2];
    auto weights = [&](int st) {
      u32x4 pw;
      float sum = 0.f;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float p0 = __builtin_amdgcn_exp2f(fmaf(s[st >> 1][(st & 1) * 8 + 2 * e], sc, st < ST / 2 ? nb0 : nb1));
        const float p1 = __builtin_amdgcn_exp2f(fmaf(s[st >> 1][(st & 1) * 8 + 2 * e + 1], sc, st < ST / 2 ? nb0 : nb1));
        sum += p0 + p1;
        pw[e] = pack_bf16x2(p0, p1);
      }
      l_run = st == ST / 2 ? fmaf(l_run, alpha1, sum) : l_run + sum;
      pB[st & 1] = as_bf16x8(pw);
    };
    read(0);
    weights(0);
#pragma unroll
    for (int st = 0; st < ST; ++st) {
      if (st + 1 < ST) {
        read(st + 1);
        weights(st + 1);
      }
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        const uint2 lo = va[st & 1][dt][0], hi = va[st & 1][dt][1];
        acc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf16x8(u32x4{lo.x, lo.y, hi.x, hi.y}), pB[st & 1], acc[dt], 0, 0, 0);
      }
      if (st + 1 == ST / 2 && fine) rescale(alpha1);
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  if (key_end > key_begin) {  // (uniform; a paged part past the table's last key has none)
    const int last = key_begin + (key_end - 1 - key_begin) / kKeys * kKeys;  // the last tile's first key
    issue(0, 0, key_begin);
    if (DIST == 2 && key_begin < last) issue(1, 1, key_begin + kKeys);
    // (the query operands are waited for here: a wait for them inside the loop
    // would wait for the tiles loading ahead)
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) __asm__ volatile("" ::"v"(__builtin_bit_cast(u32x4, qB[ks])));
    landed(key_begin < last);
    lds_barrier();
    // The upper waves of the 8 (one of each SIMD's two) run half a tile
    // behind: the softmax of their tile falls into the lower waves' matrix
    // products and back.  Their V tile stays staged one step longer.
    auto next = [](int x, int n) { return x + 1 == n ? 0 : x + 1; };
    int kb = 0, vb = 0, kf = DIST % KB, vf = DIST % VB;  // this tile's buffers, and those of the tile issued beside it
    auto advance = [&]() {
      kb = next(kb, KB);
      vb = next(vb, VB);
      kf = next(kf, KB);
      vf = next(vf, VB);
    };
    if (!SKEW || w < NW / 2) {
      for (int n0 = key_begin; n0 <= last; n0 += kKeys) {
        const int nf = n0 + DIST * kKeys;
        turn_pages(n0);
        if (nf <= last) issue(kf, vf, nf);
        scores(kb, n0);
        values(vb, n0);
        landed(nf <= last);
        lds_barrier();
        advance();
      }
    } else {
      int vp = 0;
      for (int n0 = key_begin; n0 <= last; n0 += kKeys) {
        const int nf = n0 + DIST * kKeys;
        turn_pages(n0);
        if (nf <= last) issue(kf, vf, nf);
        if (n0 > key_begin) values(vp, n0 - kKeys);
        scores(kb, n0);
        vp = vb;
        landed(nf <= last);
        lds_barrier();
        advance();
      }
      values(vp, last);
    }
  }

  // lane (h, col), element i of tile dt: O[row col][32 dt + 8 (i / 4) + 4 h + i % 4]
  const float L = half_sum(l_run);
  const float inv = L > 0.f ? 1.f / L : 0.f;
  const int r = r0 + col;
  if (slot >= 0) {  // one of several key ranges of the tile: an unnormalised partial for the merge
    if (r >= nrows) return;
    float* base = a.part + ((int64_t)slot * a.H + head) * a.tile_rows * (DH + 2);
    float* dst = base + r * DH + h * 4;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        *reinterpret_cast<f32x4*>(dst + dt * 32 + q * 8) =
            f32x4{acc[dt][4 * q], acc[dt][4 * q + 1], acc[dt][4 * q + 2], acc[dt][4 * q + 3]};
    if (h == 0) *reinterpret_cast<float2*>(base + a.tile_rows * DH + 2 * r) = make_float2(m_ref * sc, L);
    return;
  }
  if (r < nrows) {
    bf16_t* dst = a.out + ((int64_t)(row0 + r) * a.H + head) * DH + h * 4;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const uint32_t lo = pack_bf16x2(acc[dt][4 * q] * inv, acc[dt][4 * q + 1] * inv);
        const uint32_t hi = pack_bf16x2(acc[dt][4 * q + 2] * inv, acc[dt][4 * q + 3] * inv);
        *reinterpret_cast<uint2*>(dst + dt * 32 + q * 8) = make_uint2(lo, hi);
      }
  }
}

// Merge of the tiles cut over keys: one workgroup per (tile, head, 256 /
// (DH / 4) rows), one thread per (row, 4 dims):
//   out = sum_s 2^(m_s - M) o_s / sum_s 2^(m_s - M) l_s, in part order.
struct PrefillMergeArgs {
  bf16_t* out;
  const float* part;
  const int32_t* merges;  // [nmerge][4]: first slot, parts, first row, rows
  int H, tile_rows;
};

template <int DH>
__global__ __launch_bounds__(256) void prefill_merge_kernel(PrefillMergeArgs a) {
  constexpr int C4 = DH / 4;
  const int32_t* rec = a.merges + (int64_t)blockIdx.x * 4;
  const int slot = rec[0], parts = rec[1], row0 = rec[2], nrows = rec[3];
  const int head = blockIdx.y;
  const int r = blockIdx.z * (256 / C4) + threadIdx.x / C4, c4 = threadIdx.x % C4;
  if (r >= nrows) return;
  const int64_t stride = (int64_t)a.H * a.tile_rows * (DH + 2);
  const float* base = a.part + (int64_t)slot * stride + (int64_t)head * a.tile_rows * (DH + 2);
  constexpr int CH = 4;  // parts per round trip
  float M = kNegInf, den = 0.f;
  f32x4 num = {0.f, 0.f, 0.f, 0.f};
  for (int s0 = 0; s0 < parts; s0 += CH) {
    float2 ml[CH];
    f32x4 o[CH];
#pragma unroll
    for (int k = 0; k < CH; ++k) {
      const float* p = base + min(s0 + k, parts - 1) * stride;
      ml[k] = *reinterpret_cast<const float2*>(p + a.tile_rows * DH + 2 * r);
      o[k] = *reinterpret_cast<const f32x4*>(p + r * DH + c4 * 4);
    }
    float Mn = M;
#pragma unroll
    for (int k = 0; k < CH; ++k) Mn = fmaxf(Mn, ml[k].x);  // (a part read twice changes nothing here)
    if (Mn == kNegInf) continue;  // no key of this row so far
    const float w0 = __builtin_amdgcn_exp2f(M - Mn);  // from -inf: 0
    den *= w0;
    num *= w0;
#pragma unroll
    for (int k = 0; k < CH; ++k) {
      const float wk = s0 + k < parts ? __builtin_amdgcn_exp2f(ml[k].x - Mn) : 0.f;
      den = fmaf(ml[k].y, wk, den);
      num += o[k] * wk;
    }
    M = Mn;
  }
  const float inv = den > 0.f ? 1.f / den : 0.f;
  bf16_t* dst = a.out + ((int64_t)(row0 + r) * a.H + head) * DH + c4 * 4;
  *reinterpret_cast<uint2*>(dst) =
      make_uint2(pack_bf16x2(num[0] * inv, num[1] * inv), pack_bf16x2(num[2] * inv, num[3] * inv));
}

// ---------------------------------------------------------------------------
// The work list (host).  Rows per tile: a workgroup of 8 waves of 32 rows
// (two query heads of a kv head where the group is even) reads a K/V tile for
// twice the rows of a 4-wave one, but fewer, larger workgroups fill the chip
// worse and idle longer at the causal edge.  Measured on MI355X, 4 against 8
// waves: 8 prompts of 1000 tokens (16/8 heads) 69 against 66 us, one of 1206
// 32 against 34; 32/8 heads: 1206 42 against 47, 2048 70 against 74, 3000 111
// against 112, 4096 194 against 172, two of 2900-4050 behind 4096 cached keys
// 833 against 814: 8 waves from 24 key tiles per tile on average.
//
// Cut over keys: where the tiles alone are fewer than the compute units, a
// tile's chain of key tiles (~2 us each with one wave per SIMD) is the
// call's time, so tiles longer than 1.5 targets are cut into parts of about
// `target` key tiles and merged by a second kernel: 40 rows behind 4096 keys
// 130 -> 22 us, 270 rows of 32/8 heads 141 -> 60, one prompt of 1206 40 -> 32
// (other targets, with a lazily moved reference: 20 us at 3 and 4, 21 at 6, 24
// at 8; 50-62 at 16 and 12; 31 at 4, 35 at 3, 34 at 8).  With more
// tiles than compute units the partials cost what the shorter chain saves
// (1206 of 32/8 heads, 304 workgroups: 41.7 -> 39-43; 8 prompts 59 ->
// 64-172), so those stay whole.
// ---------------------------------------------------------------------------
struct Tiling {
  std::vector<std::array<int32_t, kTileWords>> tiles;
  std::vector<std::array<int32_t, 4>> merges;
  int rows, slots;
};

Tiling make_tiles(const int64_t* ql, const int64_t* kl, int n, int H, int Hkv, int block_size, int cus) {
  const int hw = (H / Hkv) % 2 == 0 ? 2 : 1;
  auto key_tiles = [](int64_t end) { return (end + kKeys - 1) / kKeys; };
  auto count = [&](int rows, int64_t& tiles, int64_t& keys) {
    tiles = keys = 0;
    for (int b = 0; b < n; ++b)
      for (int64_t r = 0; r < ql[b]; r += rows) {
        ++tiles;
        keys += key_tiles(kl[b] - ql[b] + std::min(r + rows, ql[b]));
      }
  };
  Tiling t{{}, {}, 8 * kWaveRows / hw, 0};
  int64_t tiles, keys;
  count(t.rows, tiles, keys);
  if (keys < 24 * tiles) {
    t.rows /= 2;
    count(t.rows, tiles, keys);
  }
  const int64_t units = H / hw;  // workgroups per tile
  const int64_t target = std::max<int64_t>(4, (keys * units * 2 + 3 * cus - 1) / (3 * cus));
  t.tiles.reserve(tiles);
  int64_t q0 = 0, k0 = 0;
  for (int b = 0; b < n; ++b) {
    for (int64_t r = 0; r < ql[b]; r += t.rows) {
      const int64_t nr = std::min<int64_t>(t.rows, ql[b] - r), pos = kl[b] - ql[b] + r, end = pos + nr, nt = key_tiles(end);
      int64_t parts = tiles * units <= cus && 2 * nt > 3 * target ? (nt + target - 1) / target : 1;
      const int64_t per = (nt + parts - 1) / parts;
      parts = (nt + per - 1) / per;
      if (parts > 1) t.merges.push_back({t.slots, (int32_t)parts, (int32_t)(q0 + r), (int32_t)nr});
      for (int64_t i = 0; i < parts; ++i)
        t.tiles.push_back({b, (int32_t)(q0 + r), (int32_t)nr, (int32_t)pos, (int32_t)(block_size > 0 ? 0 : k0),
                           (int32_t)(i * per * kKeys), (int32_t)std::min(end, (i + 1) * per * kKeys),
                           parts > 1 ? t.slots++ : -1});
    }
    q0 += ql[b];
    k0 += kl[b];
  }
  std::stable_sort(t.tiles.begin(), t.tiles.end(),
                   [](const auto& x, const auto& y) { return x[6] - x[5] > y[6] - y[5]; });  // heaviest first
  return t;
}

}  // namespace

extern "C" {

int nsv_prefill_tiles(const int64_t* seqlens_q, const int64_t* seqlens_k, int n, int H, int Hkv, int block_size,
                      int cus, int32_t* out, int64_t capacity, int32_t* counts) {
  if (n < 0 || H <= 0 || Hkv <= 0 || H % Hkv || block_size < 0 || cus <= 0 || capacity < 0 || !counts) return NSV_ERR_ARG;
  if (n > 0 && (!seqlens_q || !seqlens_k || !out)) return NSV_ERR_ARG;
  int64_t rows = 0, keys = 0;
  for (int b = 0; b < n; ++b) {
    if (seqlens_q[b] <= 0 || seqlens_q[b] > seqlens_k[b] || seqlens_k[b] > ((int64_t)1 << 30)) return NSV_ERR_ARG;
    rows += seqlens_q[b];
    keys += seqlens_k[b];
  }
  if (rows > 0x7fffffff || keys > 0x7fffffff) return NSV_ERR_UNSUPPORTED;
  try {
    const Tiling t = make_tiles(seqlens_q, seqlens_k, n, H, Hkv, block_size, cus);
    counts[0] = (int32_t)t.tiles.size();
    counts[1] = (int32_t)t.merges.size();
    counts[2] = t.rows;
    counts[3] = t.slots;
    if ((int64_t)t.tiles.size() * kTileWords + (int64_t)t.merges.size() * 4 > capacity) return NSV_ERR_WORKSPACE;
    for (const auto& x : t.tiles) out = std::copy(x.begin(), x.end(), out);
    for (const auto& x : t.merges) out = std::copy(x.begin(), x.end(), out);
  } catch (const std::bad_alloc&) {
    return NSV_ERR_WORKSPACE;
  }
  return NSV_OK;
}

int nsv_prefill_attention(void* out, const void* q, const void* k, const void* v, const int32_t* block_tables,
                          const int32_t* tiles, int ntiles, int tile_rows, const int32_t* merges, int nmerges,
                          float scale, int H, int Hkv, int D, int block_size, int max_blocks, void* partials,
                          void* stream) {
  if (ntiles < 0 || nmerges < 0 || H <= 0 || Hkv <= 0) return NSV_ERR_ARG;
  if (H % Hkv || (D != 64 && D != 128)) return NSV_ERR_UNSUPPORTED;
  const int G = H / Hkv, hw = G % 2 == 0 ? 2 : 1;
  const int nw = tile_rows * hw / kWaveRows;
  if ((nw != 8 && nw != 4) || nw * kWaveRows != tile_rows * hw) return NSV_ERR_UNSUPPORTED;
  int bs_log2 = 0;
  if (block_tables) {
    if (max_blocks <= 0 || block_size <= 0 || (block_size & (block_size - 1))) return NSV_ERR_UNSUPPORTED;
    while ((1 << bs_log2) < block_size) ++bs_log2;
    if ((int64_t)max_blocks * block_size > ((int64_t)1 << 30)) return NSV_ERR_UNSUPPORTED;
  }
  if (ntiles == 0) return NSV_OK;
  if (!out || !q || !k || !v || !tiles || (nmerges > 0 && !merges)) return NSV_ERR_ARG;
  if (nmerges > 0 && !partials) return NSV_ERR_WORKSPACE;
  const int64_t grid = (int64_t)ntiles * H / hw;
  if (grid > 0x7fffffff) return NSV_ERR_UNSUPPORTED;
  PrefillArgs a;
  a.q = (const bf16_t*)q;
  a.k = (const bf16_t*)k;
  a.v = (const bf16_t*)v;
  a.out = (bf16_t*)out;
  a.block_tables = block_tables;
  a.tiles = tiles;
  a.scale_log2 = scale * 1.44269504088896340736f;
  a.H = H;
  a.Hkv = Hkv;
  a.bs_log2 = bs_log2;
  a.max_blocks = max_blocks;
  a.hw = hw;
  a.hgroups = G / hw;
  a.part = (float*)partials;
  a.tile_rows = tile_rows;
  hipStream_t s = (hipStream_t)stream;
  const dim3 g((unsigned)grid), b(nw * 64);
  if (D == 128) {
    if (nw == 8) hipLaunchKernelGGL((prefill_attn_kernel<128, 8>), g, b, 0, s, a);
    else hipLaunchKernelGGL((prefill_attn_kernel<128, 4>), g, b, 0, s, a);
  } else {
    if (nw == 8) hipLaunchKernelGGL((prefill_attn_kernel<64, 8>), g, b, 0, s, a);
    else hipLaunchKernelGGL((prefill_attn_kernel<64, 4>), g, b, 0, s, a);
  }
  const int rc = nsv_launch_status();
  if (rc || nmerges == 0) return rc;
  PrefillMergeArgs m;
  m.out = (bf16_t*)out;
  m.part = (const float*)partials;
  m.merges = merges;
  m.H = H;
  m.tile_rows = tile_rows;
  if (D == 128) hipLaunchKernelGGL(prefill_merge_kernel<128>, dim3(nmerges, H, tile_rows / 8), dim3(256), 0, s, m);
  else hipLaunchKernelGGL(prefill_merge_kernel<64>, dim3(nmerges, H, tile_rows / 16), dim3(256), 0, s, m);
  return nsv_launch_status();
}

}  // extern "C"
