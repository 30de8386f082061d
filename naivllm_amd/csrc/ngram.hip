// GPU n-gram (prompt-lookup) drafter for gfx950.
//
// Behaviour follows NgramDrafter._lookup (src/myvllm/spec_engine/
// drafters.py:63-83), which searches the big-endian uint32 byte encoding of
// the token history with bytes.rfind.  The kernel reproduces that byte-level
// search exactly, including hits at byte offsets inside a token (which move
// the search end left of them and make the reference skip aligned matches
// that overlap them), without building the byte string: the 32-bit word at
// byte offset 4i + r is (h[i] << 8r) | (h[i+1] >> (32 - 8r)).
//
// One workgroup per sequence, one pass over its history for every n-gram
// length at once: the needle of length n is the history's last n words, so
// for each byte offset the words before it are compared backwards with the
// history's end, and the length m of that match makes the offset a hit of
// every n <= m.  The highest hit per length is kept (an LDS maximum each);
// the longest length with a hit decides.  Only a hit inside a token, which
// moves the search's end, needs a search of its own (scan_below).
//
// What bounds it: one CU's intake (~50 GB/s: 2.6 us for 32k tokens) and its
// VALU (four byte offsets of two words per token).  Measured (graph-replayed,
// 8 histories without a long match, text-like token frequencies; a scan per
// length with two barriers per 256 offsets before -> now): 1,200 tokens 53 ->
// 4.7 us, 4,000 168 -> 8.7, 16,000 724 -> 10.9, 32,768 1,512 -> 16.8; a match
// of the longest length at the very end 3.7-4.1 -> 4.7-5.1 (1,024 threads
// start instead of 256, which each of the others needs).

#include "common.h"

#include <type_traits>

namespace {

constexpr int kThreads = 1024;
constexpr int kHistLds = 36864;  // tokens of history staged in LDS (144 KB); longer ones are read in place
constexpr int kMaxN = 64;        // longest n-gram
constexpr int kMaxK = 64;        // longest continuation

struct NgramArgs {
  const int32_t* history;  // [B, stride]
  const int32_t* hist_len; // [B]
  int64_t stride;
  int B, min_n, max_n, K;
  int32_t* out_drafts;     // [B, K]
  int32_t* out_len;        // [B]
};

__global__ __launch_bounds__(kThreads) void ngram_draft_kernel(NgramArgs a) {
  __shared__ uint32_t hs[kHistLds];
  __shared__ uint32_t tail[kMaxN];     // tail[k]: the history's word k from its end
  __shared__ int best[kMaxN + 1];      // highest end of a match of exactly this many words
  __shared__ int red[kThreads / 64];
  const int b = blockIdx.x, tid = threadIdx.x;
  const uint32_t* hg = (const uint32_t*)a.history + (int64_t)b * a.stride;
  const int L = max(0, (int)min((int64_t)a.hist_len[b], a.stride));
  const int nmax = min(min(a.max_n, L - 1), kMaxN);
  if (nmax < a.min_n) {  // uniform
    if (tid == 0) a.out_len[b] = 0;
    return;
  }
  const int off = max(0, L - kHistLds);  // first token that LDS holds, once staged
  // ---- windows of the history from its top down; the longest needle's
  // match ends the search, so the first window is small and nothing is read
  // ahead of it (loads queued before the result's store delay it), the
  // others are read ahead while one is searched
  constexpr int U0 = 2, U = 8;  // tokens per thread of the first window, and of the others
  uint32_t v[U], ahead[U];
  int lo = max(0, L - U0 * kThreads), next = L;  // window [lo, next)
#pragma unroll
  for (int u = 0; u < U0; ++u) v[u] = hg[min(lo + u * kThreads + tid, L - 1)];
  uint32_t under = hg[max(lo - 1, 0)], under_ahead = 0u;  // the token below the window
  if (tid <= kMaxN) best[tid] = -1;
  if (tid < nmax) tail[tid] = hg[L - 1 - tid];
  int staged = L;  // tokens [max(staged, off), L) are in LDS
  auto tok = [&](int i) -> uint32_t {
    if (i >= staged && i >= off) return hs[i - off];
    return hg[i];
  };
  // big-endian 32-bit word at byte offset 4 i + r (hi, lo: the words i and i + 1)
  auto word_of = [](uint32_t hi, uint32_t lo, int r) -> uint32_t {
    return r == 0 ? hi : __builtin_amdgcn_alignbyte(hi, lo, 4 - r);
  };
  auto word = [&](int o) -> uint32_t {
    const int i = o >> 2, r = o & 3;
    return word_of(tok(i), r ? tok(i + 1) : 0u, r);
  };
  auto load = [&](uint32_t (&x)[U], int from, int to) {  // window [from, to)
#pragma unroll
    for (int u = 0; u < U; ++u) x[u] = hg[min(from + u * kThreads + tid, to - 1)];
  };
  // stage window [lo, next) (N tokens per thread, in v; under: the token
  // below it) and search it
  auto search = [&](auto width) {
    constexpr int N = decltype(width)::value;
#pragma unroll
    for (int u = 0; u < N; ++u) {
      const int i = lo + u * kThreads + tid;
      if (i < next && i >= off) hs[i - off] = v[u];
    }
    if (tid == 0 && lo - 1 >= off) hs[lo - 1 - off] = under;
    staged = lo;
    lds_barrier();  // (loads read ahead stay in flight)
    // Every offset 4 i + r whose word is the history's last one, and, where
    // no shorter match is asked for, whose word before it is the last but one
    // (the last token may be a frequent one): z[u] is zero where one of token
    // i's four offsets is such a hit.  Its match ends at byte e = 4 i + r + 4
    // <= 4 (L - 1).
    const bool pair = a.min_n >= 2;  // uniform
    const uint32_t last = tail[0], prior = pair ? tail[1] : 0u, keep = pair ? ~0u : 0u;
    uint32_t z[N], after[N], before[N];
#pragma unroll
    for (int u = 0; u < N; ++u) {
      const int i = lo + u * kThreads + tid;
      const int ia = min(i + 1, L - 1), ib = max(min(i, next) - 1, 0);
      after[u] = hs[max(ia - off, 0)];
      before[u] = hs[max(ib - off, 0)];
      if (off > 0) {  // uniform: a history longer than LDS
        if (ia < off) after[u] = hg[ia];
        if (ib < off) before[u] = hg[ib];
      }
    }
    auto differs = [&](int u, int r) {
      return (word_of(v[u], after[u], r) ^ last) | ((word_of(before[u], v[u], r) ^ prior) & keep);
    };
#pragma unroll
    for (int u = 0; u < N; ++u) {
      const int i = lo + u * kThreads + tid;
      const uint32_t d = min(min(differs(u, 0), differs(u, 1)), min(differs(u, 2), differs(u, 3)));
      z[u] = i < next ? d : 1u;
    }
    // from the top down; of the whole matches of a wave's 64 offsets only the
    // highest is recorded (a repeated token matches everywhere)
#pragma unroll
    for (int u = N - 1; u >= 0; --u) {
      if (!__ballot(z[u] == 0)) continue;
      const int i = lo + u * kThreads + tid;
      for (int r = 3; r >= 0; --r) {
        const int e = 4 * i + r + 4;
        bool ok = z[u] == 0 && differs(u, r) == 0 && e <= 4 * (L - 1) && (!pair || i > 0);
        // (a match of nmax words further up decides every length below it)
        ok = ok && e > *(volatile int*)&best[nmax];
        if (!__ballot(ok)) continue;
        int m = ok ? (pair ? 2 : 1) : 0;
        while (ok && m < nmax && e - 4 * (m + 1) >= 0 && word(e - 4 * (m + 1)) == tail[m]) ++m;
        const uint64_t whole = __ballot(m == nmax);
        if (whole && (tid & 63) == 63 - __builtin_clzll(whole)) atomicMax(&best[m], e);
        if (m >= a.min_n && m < nmax) atomicMax(&best[m], e);
      }
    }
    lds_barrier();
    const int bw = best[nmax];
    return lo == 0 || (bw >= 0 && (bw & 3) == 0);  // uniform
  };
  if (!search(std::integral_constant<int, U0>{})) {
    next = lo;
    lo = max(0, lo - U * kThreads);
    load(v, lo, next);
    under = hg[max(lo - 1, 0)];
    while (true) {
      const int nlo = max(0, lo - U * kThreads);
      if (lo > 0) {  // uniform
        load(ahead, nlo, lo);
        under_ahead = hg[max(nlo - 1, 0)];
      }
      if (search(std::integral_constant<int, U>{})) break;
      next = lo;
      lo = nlo;
#pragma unroll
      for (int u = 0; u < U; ++u) v[u] = ahead[u];
      under = under_ahead;
    }
  }

  // the highest offset o <= end - 4 n whose 4 n bytes are the needle, or -1
  auto scan_below = [&](int n, int end) -> int {
    for (int top = end - 4 * n; top >= 0; top -= kThreads) {
      const int o = top - tid;
      bool ok = o >= 0;
      for (int m = 0; ok && m < n; ++m) ok = word(o + 4 * m) == tail[n - 1 - m];
      const uint64_t bal = __ballot(ok);
      const int w = tid >> 6, lane = tid & 63;
      if (lane == 0) red[w] = bal ? (int)(__builtin_ctzll(bal)) + w * 64 : 0x7fffffff;
      __syncthreads();
      int first = 0x7fffffff;  // the highest matching offset of this step = the lowest matching thread
      for (int q = 0; q < kThreads / 64; ++q) first = min(first, red[q]);
      __syncthreads();
      if (first != 0x7fffffff) return top - first;
    }
    return -1;
  };

  int e = -1;
  for (int n = nmax; n >= a.min_n && n >= 1; --n) {
    e = max(e, best[n]);  // the highest match of at least n words
    int found = e < 0 ? -1 : e - 4 * n;
    while (found >= 0 && (found & 3)) found = scan_below(n, found);  // inside a token: search again left of it
    if (found >= 0) {
      const int start = found / 4 + n;
      const int cnt = min(a.K, L - start);  // >= 1: the match ends before the last token
      for (int j = tid; j < cnt; j += kThreads) a.out_drafts[(int64_t)b * a.K + j] = (int32_t)tok(start + j);
      if (tid == 0) a.out_len[b] = cnt;
      return;
    }
  }
  if (tid == 0) a.out_len[b] = 0;
}

}  // namespace

extern "C" {

int nsv_ngram_draft(const int32_t* history, const int32_t* hist_len, int64_t hist_stride, int B, int min_n,
                    int max_n, int K, int32_t* out_drafts, int32_t* out_len, void* stream) {
  if (B < 0 || hist_stride < 0 || min_n < 1 || max_n < min_n || max_n > kMaxN || K < 1 || K > kMaxK)
    return NSV_ERR_ARG;
  if (B == 0) return NSV_OK;
  if (!history || !hist_len || !out_drafts || !out_len) return NSV_ERR_ARG;
  if (hist_stride > ((int64_t)1 << 29)) return NSV_ERR_UNSUPPORTED;  // byte offsets stay in int range
  NgramArgs a;
  a.history = history;
  a.hist_len = hist_len;
  a.stride = hist_stride;
  a.B = B;
  a.min_n = min_n;
  a.max_n = max_n;
  a.K = K;
  a.out_drafts = out_drafts;
  a.out_len = out_len;
  hipLaunchKernelGGL(ngram_draft_kernel, dim3(B), dim3(kThreads), 0, (hipStream_t)stream, a);
  return nsv_launch_status();
}

}  // extern "C"
