// Projections of 13 to 128 rows for gfx950 (bf16 in, fp32 accumulation): the
// verify rows of a few sequences at hidden 4096, and the LM head past the
// rows whose activations one CU's LDS holds.
//
// y = x W^T with W [N, K] row-major (or the LM head's packed copy).
// Reference: the F.linear projections of layers/linear.py and the LM head of
// layers/embedding_head.py:71-95; the SwiGLU epilogue is
// layers/activation.py:17-19.
//
// What bounds it: the weights stream from HBM once (the only unavoidable
// traffic), while every CU also takes in the activations its columns need,
// M x (its share of K) x 2 bytes through its L1, at the ~50 GB/s one CU
// sustains.  So a workgroup covers many columns (its waves share one staged
// copy of each activation chunk) and, where the columns alone would leave
// CUs idle or make each read all of x, the reduction is split over
// workgroups: their fp32 partials are summed by the kernel that consumes
// the projection (the residual RMSNorm, the pre-attention epilogue), so the
// split costs no launch and no in-kernel hand-off.
//
// A wave owns 16 weight rows (SwiGLU: 16 gate and the 16 matching up rows).
// Weight loads are whole 128-byte lines: one instruction reads 8 rows x 128
// bytes, and two of them become two MFMA operands by swapping 8-lane halves
// with one DPP rotation per register, because a contraction may take its
// terms in any order as long as both operands agree (operand e holds
// elements 16 g4 + 8 e .. + 7 of each 64).  The 16-rows x 64-bytes loads of
// the plain operand order touch every line twice.

#include "common.h"

#include <type_traits>

namespace {

constexpr int kWlKC = 256;        // reduction elements per chunk
constexpr int kWlMaxRows = 128;
typedef uint32_t u32x2v __attribute__((ext_vector_type(2)));

struct WideArgs {
  const uint16_t* x;  // [M, K]
  const uint16_t* w;  // [N, K], or the packed LM-head layout
  uint16_t* y;        // [M, N] (plain, one split) or [M, N / 2] (SwiGLU)
  float* part;        // [splits, M, N] (plain, several splits)
  int M, N, K;
  int splits;
};

__device__ __forceinline__ bf16x8 wl_bf16x8(u32x4 v) { return __builtin_bit_cast(bf16x8, v); }

// lanes of the 8-lane halves MASK selects take src's other half, the rest old
template <int BANKS>
__device__ __forceinline__ u32x4 swap8(u32x4 old, u32x4 src) {
  u32x4 r;
#pragma unroll
  for (int i = 0; i < 4; ++i)
    r[i] = (uint32_t)__builtin_amdgcn_update_dpp((int)old[i], (int)src[i], 0x128 /* row_ror:8 */, 0xf, BANKS, false);
  return r;
}

constexpr int wl_max(int a, int b) { return a > b ? a : b; }

// EPI 0: plain; 1: SwiGLU.  NW waves: NW / WK column slots, WK waves sharing
// each slot's reduction.
template <int MT, int EPI, int NW, int WK, int NTW, bool PACKED>
__global__ __launch_bounds__(NW * 64, 2) void wide_linear_kernel(WideArgs a) {
  constexpr int NT = NW * 64, WN = NW / WK;
  constexpr int MP = MT * 16;
  constexpr int Q = 4 / WK;                       // 64-element groups per wave and chunk
  constexpr int CPR = kWlKC / 8;                  // 16-byte pieces per staged row
  constexpr int XL = (MP * CPR + NT - 1) / NT;    // activation loads per thread and chunk
  constexpr int XBUF = MP * kWlKC * 2;
  constexpr int RED = WK > 1 ? (WK - 1) * WN * NTW * MT * 1024 : 0;
  static_assert(WK == 1 || WK == 2 || WK == 4, "whole groups per wave");
  __shared__ __attribute__((aligned(16))) unsigned char lds[wl_max(2 * XBUF, RED)];
  __asm__ volatile("" ::"s"(a.x), "s"(a.w), "s"(a.y), "s"(a.part), "s"(a.M), "s"(a.N), "s"(a.K), "s"(a.splits));

  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g4 = lane >> 4, c = lane & 15;
  const int slot = w % WN, kz = w / WN;
  const int M = a.M, K = a.K;
  const int ntiles = a.N / 16 / NTW;              // column slots (SwiGLU: gate tiles)
  // this workgroup's column slots, WN at a time (slots past the last are
  // computed from zeros and not stored)
  const int t0 = (int)((int64_t)blockIdx.x * ntiles / gridDim.x), t1 = (int)((int64_t)(blockIdx.x + 1) * ntiles / gridDim.x);
  const int split = blockIdx.y;
  const int nchunk = K / kWlKC;
  const int c0 = (int)((int64_t)split * nchunk / a.splits), c1 = (int)((int64_t)(split + 1) * nchunk / a.splits);

  // Activations and weights through buffer resources of exactly their sizes:
  // padding rows, tiles past the last and chunks past the range return zeros
  // without a memory access, so every load is unconditional and the
  // compiler's wait counts stay exact.
  const __amdgpu_buffer_rsrc_t xr =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(a.x), (short)0, M * K * 2, 0x00020000);
  const int w_end = (int)((int64_t)a.N * K * 2);
  const __amdgpu_buffer_rsrc_t wr =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(a.w), (short)0, w_end, 0x00020000);

  u32x4 xv[XL];
  auto issue_x = [&](int ch) {
#pragma unroll
    for (int j = 0; j < XL; ++j) {
      const int i = tid + j * NT;
      const int m = i / CPR, p = i % CPR;
      const int off = (i < MP * CPR && ch < c1) ? (m * K + ch * kWlKC + p * 8) * 2 : M * K * 2;
      xv[j] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(xr, off, 0, 0));
    }
  };
  auto stage_x = [&](int buf) {  // piece p of row m at slot p ^ (m % 16)
#pragma unroll
    for (int j = 0; j < XL; ++j) {
      const int i = tid + j * NT;
      const int m = i / CPR, p = i % CPR;
      if (MP * CPR % NT == 0 || i < MP * CPR)
        *reinterpret_cast<u32x4*>(lds + buf * XBUF + m * (kWlKC * 2) + ((p ^ (m & 15)) << 4)) = xv[j];
    }
  };
  // weight loads of one chunk: [tile of the pair][group][half]
  struct W {
    u32x4 v[NTW][Q][2];
  };
  const int lane_off = PACKED ? lane * 16 : ((lane & 7) * K + (lane >> 3) * 8) * 2;
  // chunk ch of the column slots from tbase on
  auto issue_w = [&](W& b, int tbase, int ch) {
    const int tile = tbase + slot;
#pragma unroll
    for (int t = 0; t < NTW; ++t)
#pragma unroll
      for (int q = 0; q < Q; ++q)
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          const int g = kz * Q + q;  // group of the chunk
          const int rel = PACKED ? ch * 8192 + (2 * g + e) * 1024 : (ch * kWlKC + g * 64 + 8 * e * K) * 2;
          const int tt = EPI == 1 ? tile + t * ntiles : tile * NTW + t;
          const int off = tile < t1 && ch < c1 ? tt * 16 * K * 2 + lane_off + rel : w_end;
          b.v[t][q][e] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(wr, off, 0, kCpolNt));
        }
  };
  f32x4 acc[NTW][MT];
#pragma unroll
  for (int t = 0; t < NTW; ++t)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[t][mt] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto compute = [&](const W& b, int buf) {
    const unsigned char* xs = lds + buf * XBUF;
#pragma unroll
    for (int q = 0; q < Q; ++q)
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const int g = kz * Q + q;
        const int p = PACKED ? 8 * g + 4 * e + g4 : 8 * g + 2 * g4 + e;  // this lane's piece of the chunk
        u32x4 op[NTW];
#pragma unroll
        for (int t = 0; t < NTW; ++t) {
          if constexpr (PACKED) op[t] = b.v[t][q][e];
          else op[t] = e == 0 ? swap8<0xc>(b.v[t][q][0], b.v[t][q][1]) : swap8<0x3>(b.v[t][q][1], b.v[t][q][0]);
        }
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          const u32x4 xb = *reinterpret_cast<const u32x4*>(xs + (mt * 16 + c) * (kWlKC * 2) + ((p ^ c) << 4));
#pragma unroll
          for (int t = 0; t < NTW; ++t)
            acc[t][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wl_bf16x8(op[t]), wl_bf16x8(xb), acc[t][mt], 0, 0, 0);
        }
      }
  };

  // lane (g4, c): columns 4 g4 .. + 3 of a 16-column tile, row 16 mt + c
  auto emit = [&](int tile) {
    if (tile >= t1) return;
#pragma unroll
  for (int t = 0; t < (EPI == 1 ? 1 : NTW); ++t)
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int m = mt * 16 + c;
    const int n0 = (EPI == 1 ? tile : tile * NTW + t) * 16 + 4 * g4;
    if (m >= M) continue;
    if constexpr (EPI == 1) {
      float r[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float g = bf16_bits_to_f32(f32_to_bf16_bits(acc[0][mt][i]));
        const float u = bf16_bits_to_f32(f32_to_bf16_bits(acc[NTW - 1][mt][i]));
        r[i] = g / (1.f + __expf(-g)) * u;
      }
      *reinterpret_cast<uint2*>(a.y + (int64_t)m * (a.N / 2) + n0) = make_uint2(pack_bf16x2(r[0], r[1]), pack_bf16x2(r[2], r[3]));
    } else if (a.splits == 1) {
      *reinterpret_cast<uint2*>(a.y + (int64_t)m * a.N + n0) =
          make_uint2(pack_bf16x2(acc[t][mt][0], acc[t][mt][1]), pack_bf16x2(acc[t][mt][2], acc[t][mt][3]));
    } else {
      *reinterpret_cast<f32x4*>(a.part + ((int64_t)split * M + m) * a.N + n0) = acc[t][mt];
    }
  }
  };

  // ---- two weight chunks in flight, the activations one chunk ahead, across
  // the workgroup's column groups (a later group's first chunks load while
  // the one before is multiplied; several groups take an even chunk count)
  const int nck = c1 - c0;
  const int groups = (t1 - t0 + WN - 1) / WN;
  int wt = t0, wc = c0, xc = c0;                  // the next weight and activation chunks to issue
  int left = groups * nck;                        // chunks not yet issued
  auto next_w = [&](W& b) {
    issue_w(b, wt, left > 0 ? wc : c1);
    --left;
    if (++wc == c1 && groups > 1) {               // uniform
      wc = c0;
      wt += WN;
    }
  };
  auto next_x = [&]() {
    issue_x(xc);
    if (++xc == c1 && groups > 1) xc = c0;
  };
  W A, B;
  next_x();
  next_w(A);
  __builtin_amdgcn_sched_barrier(0);
  next_w(B);
  __builtin_amdgcn_sched_barrier(0);
  stage_x(0);
  lds_barrier();
  int done = 0, tile = t0 + slot;
  for (int i = 0; i < groups * nck; i += 2) {
    __builtin_amdgcn_sched_barrier(0);
    next_x();
    __builtin_amdgcn_sched_barrier(0);
    compute(A, 0);
    __builtin_amdgcn_sched_barrier(0);
    next_w(A);
    __builtin_amdgcn_sched_barrier(0);
    stage_x(1);
    lds_barrier();
    __builtin_amdgcn_sched_barrier(0);
    next_x();
    __builtin_amdgcn_sched_barrier(0);
    compute(B, 1);  // (past the range: zeros)
    __builtin_amdgcn_sched_barrier(0);
    next_w(B);
    __builtin_amdgcn_sched_barrier(0);
    stage_x(0);
    lds_barrier();
    if (WK == 1 && (done += 2) == nck && i + 2 < groups * nck) {  // a group is complete
      emit(tile);
      done = 0;
      tile += WN;
#pragma unroll
      for (int t = 0; t < NTW; ++t)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[t][mt] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
  }

  // ---- the WK waves of a slot summed in wave order
  if constexpr (WK > 1) {
    f32x4* red = reinterpret_cast<f32x4*>(lds);
    if (kz > 0) {
#pragma unroll
      for (int t = 0; t < NTW; ++t)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
          red[((((kz - 1) * WN + slot) * NTW + t) * MT + mt) * 64 + lane] = acc[t][mt];
    }
    lds_barrier();
    if (kz > 0) return;
#pragma unroll
    for (int z = 0; z < WK - 1; ++z)
#pragma unroll
      for (int t = 0; t < NTW; ++t)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[t][mt] += red[(((z * WN + slot) * NTW + t) * MT + mt) * 64 + lane];
  }
  emit(tile);
}

template <int EPI, int NW, int WK, int NTW, bool PACKED, int MIN_MT, int MAX_MT>
void launch_wide(const WideArgs& a, int cus, hipStream_t s) {
  const int slots = NW / WK, ntiles = a.N / 16 / NTW;
  int gx = (ntiles + slots - 1) / slots;
  if (WK == 1 && a.splits == 1 && a.K / kWlKC % 2 == 0) gx = gx < cus ? gx : cus;  // several column groups per workgroup
  const dim3 grid(gx, a.splits), block(NW * 64);
  const int mt = (a.M + 15) / 16;
  auto go = [&](auto v) {
    constexpr int MT = decltype(v)::value;
    if constexpr (MT >= MIN_MT && MT <= MAX_MT)
      hipLaunchKernelGGL((wide_linear_kernel<MT, EPI, NW, WK, NTW, PACKED>), grid, block, 0, s, a);
  };
  switch (mt < MIN_MT ? MIN_MT : mt) {
    case 2: go(std::integral_constant<int, 2>{}); break;
    case 3: go(std::integral_constant<int, 3>{}); break;
    case 4: go(std::integral_constant<int, 4>{}); break;
    case 5: go(std::integral_constant<int, 5>{}); break;
    case 6: go(std::integral_constant<int, 6>{}); break;
    case 7: go(std::integral_constant<int, 7>{}); break;
    default: go(std::integral_constant<int, 8>{}); break;
  }
}

// The dispatch of a call: columns per workgroup, and the workgroups its
// reduction is split over.
struct WidePlan {
  int cols;    // plain: 128 (a wave per 16 columns) or 64 (two waves per 16 columns);
               // SwiGLU: gate columns, 16 (four waves share them), 48 or 64 (two waves each)
  int splits;  // 0: shape not taken
};

// Plain: the largest even split of the reduction's 256-element chunks that
// keeps one workgroup per CU and at least two chunks each, or, where the even
// ones leave more than a third of those workgroups unused, an uneven one (an
// odd range costs a chunk of zeros; a whole layer at 72 rows, even only -> so,
// us: 4096 x 11008, 43 chunks, 1 -> 8 splits 224 -> 146, library 171; 3584 x
// 18944, 74 chunks, 2 -> 9 splits 223 -> 169, library 235; 2560 x 9728, 38
// chunks, 2 -> 12 splits 148 -> 122, library 133): 64-column
// workgroups while that leaves at most four chunks (the columns alone are
// few, so each CU reads little of x), 128-column ones beyond (half the
// workgroups read x, twice the splits).  MI355X, 72 rows, graph-replayed over
// rotating weights, us (library GEMM -> this; other splits): 6144 x 4096 23.1
// -> 17.0 (128 columns, 4 splits; 2: 25.4, 8: 21.4; 64 columns, 2 splits
// 18.1); 4096 x 4096 16.2 -> 11.5 (64 columns, 4; 128 columns, 8: 12.5); 4096
// x 12288 42.9 -> 25.5 (128 columns, 8; 4: 38; 64 columns, 4: 27.6).  108
// rows: 4096 x 1024 11.4 -> 8.5 (64 columns, 2), 1024 x 2048 10.8 -> 8.1 (4),
// 1024 x 3072 9.7 -> 8.4 (6).
// SwiGLU: one slot of 16 gate columns per workgroup while that fills the
// chip once (6144 x 1024, 108 rows: 11.1 us with four waves, 20.8 with 48
// columns), else three per workgroup (24576 x 4096, 72 rows: 46 us for 256
// workgroups, 52 with four slots, 58 with one; the library GEMM alone 53.5,
// its SiLU kernel 4 more), or four past 80 rows, whose registers three slots
// of two waves do not hold (108 rows: 54.7 against 74.4), and wherever three
// would leave a second turn of a few workgroups and four do not (intermediate
// size 14336, 299 or 224 workgroups, a whole layer with three -> four: 16 rows
// 137 -> 127 us, 54 167 -> 148, 72 184 -> 163, the library 143, 163 and 189).
WidePlan wide_plan(int M, int N, int K, int epi, bool packed, int cus) {
  if (M <= 0 || M > kWlMaxRows || N <= 0 || K <= 0 || N % 16 || K % kWlKC) return {0, 0};
  // byte offsets into the weight and into the activations' padded row tiles fit an int
  const int64_t rows = (M + 15) / 16 * 16 < 32 ? 32 : (M + 15) / 16 * 16;
  if ((N > rows ? N : rows) * (int64_t)K * 2 > ((int64_t)1 << 31) - (1 << 20)) return {0, 0};
  if (epi == 1) {
    if (N % 32 || packed) return {0, 0};
    if (N / 32 <= cus) return {16, 1};
    const int tiles = N / 32;
    const bool one_turn = (tiles + 2) / 3 <= cus || (tiles + 3) / 4 > cus;  // of 48 columns, or none of 64
    return {M <= 80 && one_turn ? 48 : 64, 1};
  }
  if (packed) return {128, K == 1024 || K == 2048 || K == 4096 ? 1 : 0};  // the packed layout's reductions
  const int nck = K / kWlKC;
  auto cut = [&](int cols) {
    const int groups = (N + cols - 1) / cols;
    int s = cus / groups;
    s = s > nck / 2 ? nck / 2 : s;
    const int most = s < 1 ? 1 : s;
    for (s = most; nck % s; --s) {
    }
    return 3 * s < 2 * most ? most : s;
  };
  const int s64 = cut(64);
  if (nck / s64 <= 4) return {64, s64};
  return {128, cut(128)};
}

int wide_cus() {
  int dev = 0, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
      cus <= 0) {
    (void)hipGetLastError();
    return 256;
  }
  return cus;
}

}  // namespace

extern "C" {

int nsv_wide_linear_splits(int M, int N, int K, int epilogue, int packed) {
  if (epilogue < 0 || epilogue > 1) return 0;
  return wide_plan(M, N, K, epilogue, packed != 0, wide_cus()).splits;
}

int nsv_wide_linear(const void* x, const void* weight, void* y, float* partials, int M, int N, int K, int epilogue,
                    int packed, void* stream) {
  if (M < 0 || N <= 0 || K <= 0 || epilogue < 0 || epilogue > 1) return NSV_ERR_ARG;
  if (M == 0) return NSV_OK;
  const int cus = wide_cus();
  const WidePlan p = wide_plan(M, N, K, epilogue, packed != 0, cus);
  if (p.splits == 0) return NSV_ERR_UNSUPPORTED;
  if (!x || !weight || (p.splits > 1 ? !partials : !y)) return NSV_ERR_ARG;
  const WideArgs a{(const uint16_t*)x, (const uint16_t*)weight, (uint16_t*)y, partials, M, N, K, p.splits};
  hipStream_t s = (hipStream_t)stream;
  if (epilogue == 1) {
    if (p.cols == 16) launch_wide<1, 4, 4, 2, false, 2, 8>(a, cus, s);
    else if (p.cols == 48) launch_wide<1, 6, 2, 2, false, 2, 5>(a, cus, s);
    else launch_wide<1, 8, 2, 2, false, 6, 8>(a, cus, s);
  } else if (packed) {
    launch_wide<0, 8, 1, 1, true, 2, 8>(a, cus, s);
  } else if (p.cols == 64) {
    launch_wide<0, 8, 2, 1, false, 2, 8>(a, cus, s);
  } else {
    launch_wide<0, 8, 1, 1, false, 2, 8>(a, cus, s);
  }
  return nsv_launch_status();
}

}  // extern "C"
