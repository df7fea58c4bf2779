// Exact top-2048 + page-table transform over (sparse-mask) indexer logits, gfx950.
//
// Contract (hcu_ops/csrc/sparse_mask_topk.cu:1-22,141-349): per row, the 2048 tokens t < len
// with the largest keys, ties at the threshold to the lower t; masked-out tokens are +0;
// rows with len <= 2048 copy page_table[0:len] and pad with -1.  Output order: the reference
// single kernel's (sparse_mask_topk.cu:301-345), every token with key > thr in ascending token
// order, then the ties taken in ascending token order -- a function of the scores alone, so
// the layout is the same on every run and every graph replay.
//
// Algorithm (this file's own).  Rows of up to 8192 tokens are held in registers and their threshold
// found by counting (held_row).  Longer rows, one read of the row: a fixed sample of the row
// (256 chunks of 16 tokens) gives a key K* that leaves, with
// overwhelming probability, between 2048 and a few thousand of the row's keys >= K*; one
// unordered pass collects them (positions from wave-aggregated LDS atomics, no barriers in the
// streaming loop); they are resolved exactly by a 12-bit histogram of a digit relative to K*
// (sized from the sample so that the threshold digit holds a handful of keys) and an exact
// (key desc, token asc) rank of that digit's members; the selected tokens are then put in order
// by a bitmap of the row's tokens and a prefix count of its words (emit_held).  A count past the
// list's capacity raises K* from the stored keys (to at most the row's 2048th key) and collects
// once more; a count below 2048, or still past capacity, takes the exact path, so the result
// never depends on the sample.
// Exact path (radix digits 12/12/8 of the 32-bit key):
//   pass 1   histogram of key[31:20] over the nonzero tokens plus positive / zero counts (or
//            taken from the logits kernel).  positives <= 2048 <= positives + zeros means the
//            threshold is +0 (sparse fast path).  Otherwise the threshold digit t1 follows.
//   collect  one unordered pass over the row: tokens in bin t1 become candidates (key, token).
//   select   the candidates (in LDS) go through the remaining digit passes to the exact
//            threshold key and the number of threshold ties to take; candidates that do not fit
//            in LDS are resolved by re-reading the row.
//   emit     an ordered pass over the row writes the tokens above the threshold and the first
//            ties (emit_row).
// Few rows: S CTAs per row collect one slice each and publish their candidates through per-row
// global counters; the last CTA of the row to finish (device-scope atomic) resolves them.
// Many rows: one CTA per row does everything.  No host synchronisation; launch shapes depend
// only on (rows, width, splits), so the whole path can be captured in a hipGraph.
#include <mutex>
#include <type_traits>

#include "dsa_common.h"

namespace dsa {
namespace {

constexpr int kTk = 1024;   // threads of the one-CTA-per-row kernel
constexpr int kTs = 512;    // threads of the split collect / resolve CTAs
constexpr int kCapC = 8192; // candidates the one-CTA-per-row kernel resolves in LDS
constexpr int kCapS = 4096; // candidates of a row the split kernel resolves in LDS
constexpr int kCapW = 5120; // the same for the one-CTA-per-row kernel on scores wider than kWideRow
constexpr int kWideRow = 81920;
constexpr int kMaxSplit = 64;
constexpr int64_t kMaxWidth = int64_t{1} << 29;  // tokens a row may hold: byte offsets stay below 2^31
constexpr int kUnroll = 4;  // float4 groups per lane in one batch (two batches in flight)

struct RowSrc {
  const float* vals;
  const int16_t* mask;  // never null: without a mask it points at the scores and mask_or = 0xFFFF
  uint32_t mask_or;
  int len;
};

// Raw scores of tokens [i0, i0 + 4) (i0 % 4 == 0) and the mask word holding their bits, loaded
// but not yet used, so that a batch of them stays in flight.  A quad that starts at or past the
// row's end reads the row's first quad instead (its tokens are flagged invalid by quad_keys),
// so no load leaves the row and no branch splits the batch.
struct Quad {
  float v[4];
  uint16_t mw;
};

// Token index a quad's loads use: its own start inside the row, 0 past the end.
__device__ __forceinline__ int quad_origin(const RowSrc& r, int i0) { return i0 >= r.len ? 0 : i0; }

template <bool kVec>
__device__ __forceinline__ void load_quad(const RowSrc& r, int i0, Quad& q) {
  const int at = quad_origin(r, i0);
  if constexpr (kVec) {
    // nontemporal: a row's scores are streamed once by its collection (measured: logits + top-k
    // on the 64-request MTP batch 79.7 -> 76.9 us; the 32 x 16K batch unchanged)
    using f32x4v = __attribute__((ext_vector_type(4))) float;
    const f32x4v f = __builtin_nontemporal_load(reinterpret_cast<const f32x4v*>(r.vals + at));
#pragma unroll
    for (int j = 0; j < 4; ++j) q.v[j] = f[j];
  } else {
    // raw buffer loads against a descriptor of the row (base and size wave-uniform): one 32-bit
    // byte offset per token, and tokens past r.len read 0 (the descriptor's range check), not
    // memory
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(r.vals), 0, static_cast<int>(static_cast<uint32_t>(r.len) * 4u), kBufferDword3);
    const int byte0 = at * 4;
#pragma unroll
    for (int j = 0; j < 4; ++j) q.v[j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, byte0 + 4 * j, 0, 0));
  }
  // no mask (mask_or all ones, wave-uniform): no load at all
  const int word = at >> 4;
  if (r.mask_or == 0xFFFFu) {
    q.mw = 0;
  } else if constexpr (kVec) {
    q.mw = static_cast<uint16_t>(r.mask[word]);
  } else {
    const __amdgpu_buffer_rsrc_t ms = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<int16_t*>(r.mask), 0, static_cast<int>((static_cast<uint32_t>(r.len) + 15u) >> 4) * 2, kBufferDword3);
    q.mw = __builtin_amdgcn_raw_buffer_load_b16(ms, word * 2, 0, 0);
  }
}

// Bit j set for each token i0 + j (j < 4) that lies below the row's length: the low n bits for
// the n = clamp(len - i0, 0, 4) tokens of the quad inside the row.
__device__ __forceinline__ uint32_t quad_live(const RowSrc& r, int i0) {
  const int inside = min(max(r.len - i0, 0), 4);
  return (1u << inside) - 1u;
}

// Keys of a loaded quad (masked-out tokens are +0); returns quad_live.
__device__ __forceinline__ uint32_t quad_keys(const RowSrc& r, int i0, const Quad& q, uint32_t (&k)[4]) {
  // the quad's four bits of its 16-bit mask word (i0 % 4 == 0, so the nibble never straddles)
  const int at = i0 < r.len ? i0 : 0;
  const uint32_t bits = ((q.mw | r.mask_or) >> (at & 15)) & 0xFu;
#pragma unroll
  for (int j = 0; j < 4; ++j) k[j] = ((bits >> j) & 1u) ? float_key(q.v[j]) : kZeroKey;
  return quad_live(r, i0);
}

template <bool kVec>
__device__ __forceinline__ uint32_t load_keys4(const RowSrc& r, int i0, uint32_t (&k)[4]) {
  Quad q;
  load_quad<kVec>(r, i0, q);
  return quad_keys(r, i0, q, k);
}

// atomicAdd(&hist[bin], 1) from every active lane, as one add when all of them hold the same bin:
// a constant or near-constant row puts every key of a pass on one counter, and a wave's 64 atomics
// on one LDS word are served one after another (the exact path's passes over a 64K-token row of
// equal keys took ~30 us each that way).  The test costs two ballots per call.
__device__ __forceinline__ void hist_add(int* hist, uint32_t bin) {
  const uint64_t act = __ballot(1);
  const uint32_t b0 = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(bin)));
  if (__ballot(bin == b0) == act) {  // wave-uniform
    if (lane_id() == __builtin_ctzll(act)) atomicAdd(&hist[b0], __popcll(act));
  } else {
    atomicAdd(&hist[bin], 1);
  }
}

template <int NT>
__device__ __forceinline__ int block_sum(int x, int* s_red) {
  constexpr int W = NT / kWave;
  x = wave_sum(x);
  if (lane_id() == 0) s_red[threadIdx.x >> 6] = x;
  __syncthreads();
  int s = 0;
#pragma unroll
  for (int v = 0; v < W; ++v) s += s_red[v];
  __syncthreads();
  return s;
}

// Block-exclusive prefix (thread order) of a per-thread count in [0, 7] (kWide: [0, 31]); one
// barrier, with the wave totals double-buffered by `parity` so back-to-back calls do not race.
template <int NT, bool kWide = false>
__device__ __forceinline__ int block_prefix(int c, int& total, int* s_scan, int parity) {
  constexpr int W = NT / kWave;
  int wt;
  const int x = kWide ? wave_prefix_5(c, wt) : wave_prefix_small(c, wt);
  const int w = threadIdx.x >> 6;
  int* buf = s_scan + parity * W;
  if (lane_id() == 0) buf[w] = wt;
  __syncthreads();
  int before = 0, tot = 0;
#pragma unroll
  for (int v = 0; v < W; ++v) {
    before += v < w ? buf[v] : 0;
    tot += buf[v];
  }
  total = tot;
  return before + x;
}

// Finds, for each need[i], bin t with suffix(t) >= need[i] > suffix(t + 1) of a histogram held
// in registers (thread tid owns bins tid * BPT .. tid * BPT + BPT - 1); s_res[3i..3i+2] = {t,
// suffix(t + 1), count of t} ({0, 0, 0} if the histogram holds fewer than need[i], which
// consistent inputs never do).  Ends with a barrier.
template <int NT, int BPT, int NN>
__device__ __forceinline__ void find_thresholds_regs(const int (&h)[BPT], const int (&need)[NN], int* s_wtot, int* s_res) {
  constexpr int W = NT / kWave;
  const int tid = threadIdx.x;
  const int w = tid >> 6;
  if (tid < 3 * NN) s_res[tid] = 0;
  int mine = 0;  // keys in this thread's bins
#pragma unroll
  for (int j = 0; j < BPT; ++j) mine += h[j];
  // keys in the bins of the higher threads: the wave's inclusive suffix minus this thread's own,
  // plus the totals of the higher waves
  const int from_here = wave_suffix_sum(mine);
  if ((tid & 63) == 0) s_wtot[w] = from_here;
  __syncthreads();
  int higher = from_here - mine;
#pragma unroll
  for (int v = 0; v < W; ++v) higher += v > w ? s_wtot[v] : 0;
  // The thread whose bins hold the need[i]-th key walks its bins upwards from its lowest: the
  // count at or above bin j shrinks as j grows, and the answer is the last bin where it still
  // reaches need[i].
#pragma unroll
  for (int i = 0; i < NN; ++i) {
    if (higher < need[i] && higher + mine >= need[i]) {
      int at_or_above = higher + mine;
#pragma unroll
      for (int j = 0; j < BPT; ++j) {
        const int above_j = at_or_above - h[j];
        if (above_j < need[i]) {
          s_res[3 * i] = tid * BPT + j;
          s_res[3 * i + 1] = above_j;
          s_res[3 * i + 2] = h[j];
          break;
        }
        at_or_above = above_j;
      }
    }
  }
  __syncthreads();
}

template <int NT, int BPT>
__device__ __forceinline__ void find_threshold_regs(const int (&h)[BPT], int need, int* s_wtot, int* s_res) {
  const int n[1] = {need};
  find_thresholds_regs<NT, BPT, 1>(h, n, s_wtot, s_res);
}

// The same over an LDS histogram of NB bins (16-B aligned: every histogram here is the first
// member of an alignas(16) LDS struct).  With at least 4 bins a thread, 16-B reads and no guard
// (measured: the 64-request MTP top-k 23.0 -> 21.9 us, a 4096-row prefill slab 332 -> 327 us).
template <int NB, int NT, int NN>
__device__ __forceinline__ void find_thresholds(const int* hist, const int (&need)[NN], int* s_wtot, int* s_res) {
  constexpr int BPT = NB >= NT ? NB / NT : 1;
  constexpr int ACTIVE = NB / BPT;
  int h[BPT];
  if constexpr (ACTIVE == NT && BPT % 4 == 0) {
    const int4* p = reinterpret_cast<const int4*>(__builtin_assume_aligned(hist, 16)) + threadIdx.x * (BPT / 4);
#pragma unroll
    for (int j = 0; j < BPT / 4; ++j) {
      const int4 v = p[j];
      h[4 * j] = v.x;
      h[4 * j + 1] = v.y;
      h[4 * j + 2] = v.z;
      h[4 * j + 3] = v.w;
    }
  } else {
#pragma unroll
    for (int j = 0; j < BPT; ++j) h[j] = static_cast<int>(threadIdx.x) < ACTIVE ? hist[threadIdx.x * BPT + j] : 0;
  }
  find_thresholds_regs<NT, BPT, NN>(h, need, s_wtot, s_res);
}

template <int NB, int NT>
__device__ __forceinline__ void find_threshold(const int* hist, int need, int* s_wtot, int* s_res) {
  const int n[1] = {need};
  find_thresholds<NB, NT, 1>(hist, n, s_wtot, s_res);
}

// (16-B stores here measured slower than these 4-B ones: 0.1-2 us more per top-k launch.)
template <int NT>
__device__ __forceinline__ void zero_lds(int* p, int n) {
  for (int i = threadIdx.x; i < n; i += NT) p[i] = 0;
}

// Output write guarded to the row's 2048 entries (inputs that break the contract -- e.g. a
// pass-1 histogram built for other lengths -- give wrong rows, never stray writes).
__device__ __forceinline__ void put(int32_t* dst, int i, int32_t v) {
  if (static_cast<unsigned>(i) < static_cast<unsigned>(kTopK)) dst[i] = v;
}

// What a PtRow reads for a row without entries (cols == 0), so that a gather never needs a
// branch around its load.
__device__ int32_t g_pt_none = -1;

// Page-table entry of token t (-1 outside the row's entries).
// shift 0: one entry per token (page_table_size_1); 6: one entry per 64-token page of a block
// table, token t at slot entry * 64 + t % 64 (the expansion page_table_size_1 holds), so the
// transform reads 4 B per 64 tokens instead of 4 B per token.  shift is wave-uniform.
struct PtRow {
  const int32_t* p;  // the row's entries, or &g_pt_none when it has none
  int cols;          // tokens the row covers; tokens past it map to -1
  int shift;
  // The entry of token t, or -1 when !valid or t lies past the row.  The load goes out for every
  // lane (such a lane reads entry 0) and its result is dropped afterwards: with the load inside a
  // branch that also used its result, each gather of a batch waited for the one before (eight
  // round trips for the eight candidates a thread holds; measured: the 32 x 16K decode step
  // 32.9 -> 31.5 us, one 4096-token row 15.8 -> 15.0 us, 4096-row prefill slabs 298 / 340 ->
  // 268 / 301 us).
  __device__ __forceinline__ int32_t at(int t, bool valid) const {
    const bool in = valid && static_cast<unsigned>(t) < static_cast<unsigned>(cols);
    const uint32_t tc = in ? static_cast<uint32_t>(t) : 0u;
    // a 32-bit byte offset from the row's base (cols <= width < 2^29, checked by the host)
    const int32_t v = *reinterpret_cast<const int32_t*>(reinterpret_cast<const char*>(p) + (tc >> shift) * 4u);
    const int32_t e = shift ? v * 64 + (t & 63) : v;
    return in ? e : -1;
  }
  __device__ __forceinline__ int32_t operator[](int t) const { return at(t, true); }
};

// Page-table row of score row `row`: the row itself (decode layout) or its request.
__device__ __forceinline__ int pt_row_of(int row, const int32_t* cu, int n_req) {
  if (cu == nullptr) return row;
  int lo = 0, hi = n_req - 1;  // last b with cu[b] <= row
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (cu[mid] <= row) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

// Threshold facts of a row from its pass-1 histogram: fast path, digit t1, tokens above t1.
struct Meta {
  bool fast;
  uint32_t t1;
  int above1;
  int n_t1;  // keys in bin t1
  int pos;
};

template <int NT>
__device__ __forceinline__ Meta row_meta(const int* hist_lds, int pos, int zeros, int* s_wtot, int* s_res) {
  Meta m;
  m.pos = pos;
  m.fast = pos <= kTopK && pos + zeros >= kTopK;
  m.t1 = 0;
  m.above1 = pos;
  m.n_t1 = 0;
  if (!m.fast) {
    find_threshold<kBins, NT>(hist_lds, kTopK, s_wtot, s_res);
    m.t1 = static_cast<uint32_t>(s_res[0]);
    m.above1 = s_res[1];
    m.n_t1 = s_res[2];
  }
  return m;
}

// One batch: kUnroll quads per lane, NT * 4 tokens apart.
struct Batch {
  Quad q[kUnroll];
};

template <bool kVec, int NT>
__device__ __forceinline__ void load_batch(const RowSrc& rr, int b, Batch& x) {
#pragma unroll
  for (int u = 0; u < kUnroll; ++u) load_quad<kVec>(rr, b + u * NT * 4, x.q[u]);
}

// Streams n_batches batches from lane offset b with two in flight: x0 / x1 hold the first two on
// entry (issued by the caller, possibly before other work), and each is reloaded right after
// fn(b, batch) used it -- no register copies, so the in-order load counter only ever waits for
// the batch being used.
template <bool kVec, int NT, typename Fn>
__device__ __forceinline__ void stream_batches(const RowSrc& rr, int b, int n_batches, Batch& x0, Batch& x1, Fn fn) {
  constexpr int kStep = NT * 4 * kUnroll;
  for (int i = 0; i < n_batches; i += 2) {
    fn(b, x0);
    if (i + 2 < n_batches) load_batch<kVec, NT>(rr, b + 2 * kStep, x0);
    if (i + 1 >= n_batches) break;
    fn(b + kStep, x1);
    if (i + 3 < n_batches) load_batch<kVec, NT>(rr, b + 3 * kStep, x1);
    b += 2 * kStep;
  }
}

// Pass 1 over [begin, end) (end > begin) of the row into the LDS histogram `hist` (zeroed here;
// zeros counted, not binned); returns the range's positive / zero counts (block-uniform).
template <bool kVec, int NT>
__device__ __forceinline__ void pass_hist(const RowSrc& r, int begin, int end, int* hist, int* s_red, int& pos, int& zeros) {
  constexpr int kStep = NT * 4 * kUnroll;
  RowSrc rr = r;
  rr.len = end;
  const int b0 = begin + static_cast<int>(threadIdx.x) * 4;
  Batch x0, x1;
  load_batch<kVec, NT>(rr, b0, x0);
  load_batch<kVec, NT>(rr, b0 + kStep, x1);
  zero_lds<NT>(hist, kBins);  // while the first batches are in flight
  __syncthreads();
  int zc = 0, pc = 0;
  stream_batches<kVec, NT>(rr, b0, (end - begin + kStep - 1) / kStep, x0, x1, [&](int b, const Batch& x) {
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) {
      uint32_t k[4];
      const uint32_t v = quad_keys(rr, b + u * NT * 4, x.q[u], k);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if ((v >> j) & 1u) {
          if (k[j] == kZeroKey) {
            ++zc;
          } else {
            pc += k[j] > kZeroKey;
            hist_add(hist, k[j] >> 20);
          }
        }
      }
    }
  });
  pos = block_sum<NT>(pc, s_red);
  zeros = block_sum<NT>(zc, s_red);
}

// Candidates of the threshold bin: the keys of a batch whose 12-bit digit key[31:20] is t1 go to
// the LDS list (ck, ci) at slots from one wave-aggregated atomic per batch; the count keeps
// growing past cap (the caller sees the overflow), the stores stop at cap.
template <int NT>
__device__ __forceinline__ void process_bin(const RowSrc& rr, int b, const Batch& x, uint32_t t1, uint32_t* ck,
                                            int* ci, int* n, int cap) {
  static_assert(kUnroll * 4 <= 16, "hit masks hold 16 keys");
  uint32_t k[kUnroll][4];
  uint32_t f = 0;
#pragma unroll
  for (int u = 0; u < kUnroll; ++u) {
    const uint32_t v = quad_keys(rr, b + u * NT * 4, x.q[u], k[u]);
#pragma unroll
    for (int j = 0; j < 4; ++j) f |= static_cast<uint32_t>(((v >> j) & 1u) && (k[u][j] >> 20) == t1) << (u * 4 + j);
  }
  int t;
  int p = wave_prefix_5(__popc(f), t);
  if (t == 0) return;  // wave-uniform
  int base = 0;
  if (lane_id() == 0) base = atomicAdd(n, t);
  p += uniform(base);
#pragma unroll
  for (int u = 0; u < kUnroll; ++u) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if ((f >> (u * 4 + j)) & 1u) {
        if (p < cap) {
          ck[p] = k[u][j];
          ci[p] = b + u * NT * 4 + j;
        }
        ++p;
      }
    }
  }
}

// Unordered collection of the bin-t1 keys of n_batches batches from lane offset b (x0 / x1: the
// first two, already issued).  Loads past rr.len are redirected inside the row and masked off.
template <bool kVec, int NT>
__device__ __forceinline__ void collect_bin(const RowSrc& rr, int b, int n_batches, uint32_t t1, uint32_t* ck, int* ci, int* n,
                            int cap, Batch& x0, Batch& x1) {
  stream_batches<kVec, NT>(rr, b, n_batches, x0, x1,
                           [&](int bb, const Batch& x) { process_bin<NT>(rr, bb, x, t1, ck, ci, n, cap); });
}

// ---------------------------------------------------------------------------------------------
// Sampled threshold.  A row of len > 2048 tokens is read once: every key >= K* is collected,
// where K* is a key of a fixed sample of the row chosen so that, with overwhelming probability
// for any ordering of the values, at least 2048 and at most a few thousand keys of the row are
// >= K*.  The top-2048 then lies among the collected keys (every other key is < K*) and is
// resolved exactly among them; when the count misses that window the row takes the exact
// two-pass path instead, so the result never depends on the sample.
//
// Sample: 256 chunks of 16 aligned tokens spread evenly over a row of more than 4096 tokens (one 64-B
// sector of scores and one mask word each).  K* is the lower
// edge of the 4096-key digit (key[31:12]) holding the sample key of rank k (descending), k =
// mu + 4 sqrt(mu) + 2, mu = 2048 * 4096 / len the expected number of sample keys above the row's
// 2048th key: the row has fewer than 2048 keys >= K* only if the sample holds >= k keys above
// the 2048th, a 4-sigma binomial event, and about len * k / 4096 ~ 2048 + 4.5 sqrt(2048 len /
// 4096) keys are collected (plus the few of that digit below the rank-k key).
constexpr int kSampleChunks = 256;
constexpr int kSample = kSampleChunks * 16;

__device__ __forceinline__ int sample_rank(int len) {
  const float mu = static_cast<float>(kTopK) * static_cast<float>(kSample) / static_cast<float>(len);
  const int k = static_cast<int>(ceilf(mu + 4.0f * sqrtf(mu) + 2.0f));
  return k < kSample ? k : kSample;
}

// Rank of the sample key that estimates the row's 2048th key (mu, rounded).
__device__ __forceinline__ int sample_mid_rank(int len) {
  const int m = static_cast<int>(static_cast<float>(kTopK) * static_cast<float>(kSample) / static_cast<float>(len) + 0.5f);
  return m < 1 ? 1 : m;
}

// First token of sample quad s (4 tokens) of a row.
__device__ __forceinline__ int sample_quad(int len, int s) {
  const int c = s >> 2;
  int start = static_cast<int>((static_cast<int64_t>(2 * c + 1) * len) / (2 * kSampleChunks)) & ~15;
  const int last = (len - 16) & ~15;
  start = start < last ? start : last;
  return start + (s & 3) * 4;
}

// The collection threshold of a row and the digit its candidates are resolved on:
// min(4095, (key - thr) >> shift), monotone in the key above thr.  shift is set from the
// sample so that the span from K* to the estimated 2048th key covers ~1000-2000 digits: the
// threshold digit then holds a handful of candidates.
struct SampleCut {
  uint32_t thr;
  int shift;
};

__device__ __forceinline__ uint32_t cand_digit(uint32_t key, const SampleCut& c) {
  const uint32_t d = (key - c.thr) >> c.shift;
  return d < 4095u ? d : 4095u;
}

// A K* of +0, the key of a masked-out token, means that zeros fill the row, and collecting
// them would overflow any list.  It moves up to the positive keys: 2048 of them or more are resolved
// as ever, fewer leave zeros to fill up with (sparse_row).  Before, the overflowing lists sent such rows
// to the exact path (us a launch, 1500 positives a row: 64 x 65,536 71.0 -> 23.7, 1024 x 65,536 231 -> 87,
// 32 x 16,384 32.0 -> 17.8; all zeros, 8 x 65,536 41.2 -> 20.5).  The long list's kernels and the one-CTA
// kernel for unaligned rows, at 128 VGPRs, have no room for it: their rows still take the exact path.
constexpr uint32_t kPositive = kZeroKey + 1u;  // the smallest positive key; no other K* has it (a digit's edge)

__device__ __forceinline__ void positives_only(SampleCut& c) {
  if (c.thr == kZeroKey) c.thr = kPositive;
}

// Scratch of the threshold search (LDS).
struct SampleLds {
  int* hist;      // kBins
  int* wtot;      // NT / kWave
  int* res;       // 6
};

// This thread's share of a row's sample, loaded (sample_issue) but not yet used, so that the
// caller's own loads can follow it into the memory pipeline before the sample is waited for.
template <int NT>
struct SampleLoads {
  static constexpr int QPT = kSample / 4 / NT;  // sample quads per thread
  static_assert(QPT >= 1 && QPT * 4 * NT == kSample, "sample split over the block");
  Quad q[QPT];
  int i0[QPT];
};

template <bool kVec, int NT>
__device__ __forceinline__ void sample_issue(const RowSrc& r, SampleLoads<NT>& x) {
#pragma unroll
  for (int j = 0; j < SampleLoads<NT>::QPT; ++j) {
    x.i0[j] = sample_quad(r.len, static_cast<int>(threadIdx.x) + j * NT);
    load_quad<kVec>(r, x.i0[j], x.q[j]);
  }
}

// K* of row r and the candidate digit from its issued sample (block-uniform; every CTA of the
// row computes the same).  after_sample() runs once every wave holds its share of the sample
// (right after the barrier that follows its first use): the caller issues its first streaming
// batch there, so that the sample does not wait behind it in the memory queues.
template <int NT, typename After>
__device__ __forceinline__ SampleCut sample_threshold(const RowSrc& r, const SampleLoads<NT>& x, const SampleLds& S,
                                                      After after_sample) {
  constexpr int QPT = SampleLoads<NT>::QPT;
  const int tid = threadIdx.x;
  const Quad* q = x.q;
  const int* i0 = x.i0;
  zero_lds<NT>(S.hist, kBins);
  __syncthreads();
  uint32_t k[QPT][4], v[QPT];
#pragma unroll
  for (int j = 0; j < QPT; ++j) {
    v[j] = quad_keys(r, i0[j], q[j], k[j]);
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if ((v[j] >> e) & 1u) atomicAdd(&S.hist[k[j][e] >> 20], 1);
  }
  __syncthreads();
  after_sample();
  const int rank = sample_rank(r.len);
  const int needs[2] = {rank, sample_mid_rank(r.len)};
  find_thresholds<kBins, NT, 2>(S.hist, needs, S.wtot, S.res);
  const uint32_t b = static_cast<uint32_t>(S.res[0]);
  const int need = rank - S.res[1];  // rank of the sample's K* within bin b, 1 .. count(b)
  const uint32_t bm = static_cast<uint32_t>(S.res[3]);  // bin of the 2048th-key estimate (>= b)
  const uint32_t span = bm > b ? bm - b + 1u : 1u;         // <= 4096
  SampleCut cut;
  cut.shift = 9 + (32 - __builtin_clz(span));              // 10 .. 22
  // second digit, key[19:12], over the members of bin b: K* is the lower edge of the digit that
  // holds the rank-`need` member (at most one 4096-key digit below it is collected in excess)
  if (tid < 256) S.hist[tid] = 0;
  __syncthreads();
#pragma unroll
  for (int j = 0; j < QPT; ++j) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (((v[j] >> e) & 1u) && (k[j][e] >> 20) == b) atomicAdd(&S.hist[(k[j][e] >> 12) & 0xFFu], 1);
  }
  __syncthreads();
  find_threshold<256, NT>(S.hist, need, S.wtot, S.res);
  cut.thr = (b << 20) | (static_cast<uint32_t>(S.res[0]) << 12);
  return cut;
}

// Keys >= thr of a batch into the LDS list at slots from one wave-aggregated atomic: ck gets the
// token's raw float bits, ci its index with bit 31 set for a masked-out token (whose key is the
// key of +0); readers take both through collected().  key(x) >= thr is decided on the raw bits,
// the key transform folded into the threshold: keys of floats with the sign clear order like
// their bits as signed integers, keys of negative floats the other way round.  kPos (thr >= key
// of +0): pass iff (int)bits >= (int)(thr ^ 2^31); otherwise every float with the sign clear
// passes and a negative one iff bits <= ~thr.  A masked-out token passes iff +0 >= thr, i.e. iff
// !kPos or thr == key of +0.  kMask: the row has a nonzero mask (else every token is kept).
// The slots are written without branches: every lane writes all 16 of its tokens, the ones that
// do not pass into a word of its own past the list (ck and ci hold cap + kWave entries), so the
// loop costs the same whatever the hits (per-slot branches, taken on nearly every batch since
// about 4% of a row's keys pass, made the collection VALU-bound: a 4096-row prefill slab
// 317 -> 281 us, the 32 x 16K decode step 32.4 -> 31.4 us).  A batch whose slots would cross cap
// takes a guarded path; the count keeps growing past cap (the caller sees the overflow).
template <int NT, bool kPos, bool kMask>
__device__ __forceinline__ void process_ge(const RowSrc& rr, int b, const Batch& x, uint32_t thr, uint32_t* ck,
                                           int* ci, int* n, int cap) {
  const int lo = static_cast<int>(thr ^ kZeroKey);
  const uint32_t hi = ~thr;
  const bool zero_in = kZeroKey >= thr;
  // the block's batch starts at b - 4 tid: a batch inside the row needs no per-token length test
  const bool full = uniform(b - static_cast<int>(threadIdx.x) * 4) + NT * 4 * kUnroll <= rr.len;
  uint32_t f = 0;   // bit 4u + j: token b + u NT 4 + j passes
  uint32_t nm = 0;  // bit 4u + j: that token is masked out
#pragma unroll
  for (int u = 0; u < kUnroll; ++u) {
    const int i0 = b + u * NT * 4;
    uint32_t pass = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t bits = __float_as_uint(x.q[u].v[j]);
      bool ge;
      if constexpr (kPos) ge = static_cast<int>(bits) >= lo;
      else ge = static_cast<int>(bits) >= 0 || bits <= hi;
      pass |= static_cast<uint32_t>(ge) << j;
    }
    if constexpr (kMask) {
      const uint32_t mq = ((x.q[u].mw | rr.mask_or) >> (quad_origin(rr, i0) & 12)) & 0xFu;
      pass = (pass & mq) | (zero_in ? (~mq & 0xFu) : 0u);
      nm |= (~mq & 0xFu) << (u * 4);
    }
    f |= pass << (u * 4);
  }
  if (!full) {  // block-uniform: the row's last batch
    uint32_t live = 0;
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) live |= quad_live(rr, b + u * NT * 4) << (u * 4);
    f &= live;
  }
  int t;
  int p = wave_prefix_5(__popc(f), t);
  if (t == 0) return;  // wave-uniform
  int base = 0;
  if (lane_id() == 0) base = atomicAdd(n, t);
  base = uniform(base);
  p += base;
  if (base + t <= cap) {  // wave-uniform
    // the lane's range [p, p + popc(f)) is filled from its top (the list is unordered): m is all
    // ones for a passing token, which takes slot c and moves c down; the others write the discard
    // word.  One v_bfi selects the slot (the compiler's own select took three operations and its
    // cursor update a quarter-rate multiply); c and trash are byte offsets, into ck and at the
    // same offsets into ci.
    const uint32_t trash = (cap + lane_id()) * 4u;
    uint32_t c = (p + __popc(f) - 1) * 4u;
    char* const kb = reinterpret_cast<char*>(ck);
    char* const ib = reinterpret_cast<char*>(ci);
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int s = u * 4 + j;
        const uint32_t m = static_cast<uint32_t>(__builtin_amdgcn_sbfe(static_cast<int>(f), s, 1));
        uint32_t at;
        asm("v_bfi_b32 %0, %1, %2, %3" : "=v"(at) : "v"(m), "v"(c), "v"(trash));
        int tok = b + u * NT * 4 + j;
        if constexpr (kMask) tok |= static_cast<int>((nm << (31 - s)) & 0x80000000u);
        *reinterpret_cast<uint32_t*>(kb + at) = __float_as_uint(x.q[u].v[j]);
        *reinterpret_cast<int*>(ib + at) = tok;
        asm("v_lshl_add_u32 %0, %1, 2, %0" : "+v"(c) : "v"(m));
      }
    }
  } else {
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int s = u * 4 + j;
        if ((f >> s) & 1u) {
          if (p < cap) {
            int tok = b + u * NT * 4 + j;
            if constexpr (kMask) tok |= static_cast<int>(((nm >> s) & 1u) << 31);
            ck[p] = __float_as_uint(x.q[u].v[j]);
            ci[p] = tok;
          }
          ++p;
        }
      }
    }
  }
}

// Key and token of a collected entry (process_ge's raw bits, bit 31 of the token: masked out).
__device__ __forceinline__ void collected(uint32_t bits, int tok, uint32_t& k, int& t) {
  k = tok < 0 ? kZeroKey : float_key(__uint_as_float(bits));
  t = tok & 0x7FFFFFFF;
}

template <bool kVec, int NT, bool kPos, bool kMask>
__device__ __forceinline__ void collect_ge_as(const RowSrc& rr, int b, int n_batches, uint32_t thr, uint32_t* ck,
                                              int* ci, int* n, int cap, Batch& x0, Batch& x1) {
  stream_batches<kVec, NT>(rr, b, n_batches, x0, x1, [&](int bb, const Batch& x) {
    process_ge<NT, kPos, kMask>(rr, bb, x, thr, ck, ci, n, cap);
  });
}

// collect_ge with one batch in flight and no batches issued by the caller: the second pass of a
// row whose first overflowed the list (rare; registers matter more than depth there).
template <bool kVec, int NT, bool kPos, bool kMask>
__device__ __forceinline__ void collect_ge1_as(const RowSrc& rr, int b, int n_batches, uint32_t thr, uint32_t* ck,
                                               int* ci, int* n, int cap) {
  constexpr int kStep = NT * 4 * kUnroll;
  for (int i = 0; i < n_batches; ++i, b += kStep) {
    Batch x;
    load_batch<kVec, NT>(rr, b, x);
    process_ge<NT, kPos, kMask>(rr, b, x, thr, ck, ci, n, cap);
  }
}

template <bool kVec, int NT>
__device__ __forceinline__ void collect_ge1(const RowSrc& rr, int b, int n_batches, uint32_t thr, uint32_t* ck, int* ci,
                                            int* n, int cap) {
  const bool pos = thr >= kZeroKey;       // block-uniform
  const bool msk = rr.mask_or != 0xFFFFu;  // block-uniform
  if (pos && msk) collect_ge1_as<kVec, NT, true, true>(rr, b, n_batches, thr, ck, ci, n, cap);
  else if (pos) collect_ge1_as<kVec, NT, true, false>(rr, b, n_batches, thr, ck, ci, n, cap);
  else if (msk) collect_ge1_as<kVec, NT, false, true>(rr, b, n_batches, thr, ck, ci, n, cap);
  else collect_ge1_as<kVec, NT, false, false>(rr, b, n_batches, thr, ck, ci, n, cap);
}

// ck / ci: cap + kWave entries each (the last kWave are the lanes' discard words).
template <bool kVec, int NT>
__device__ __forceinline__ void collect_ge(const RowSrc& rr, int b, int n_batches, uint32_t thr, uint32_t* ck, int* ci, int* n,
                           int cap, Batch& x0, Batch& x1) {
  const bool pos = thr >= kZeroKey;       // block-uniform
  const bool msk = rr.mask_or != 0xFFFFu;  // block-uniform
  if (pos && msk) collect_ge_as<kVec, NT, true, true>(rr, b, n_batches, thr, ck, ci, n, cap, x0, x1);
  else if (pos) collect_ge_as<kVec, NT, true, false>(rr, b, n_batches, thr, ck, ci, n, cap, x0, x1);
  else if (msk) collect_ge_as<kVec, NT, false, true>(rr, b, n_batches, thr, ck, ci, n, cap, x0, x1);
  else collect_ge_as<kVec, NT, false, false>(rr, b, n_batches, thr, ck, ci, n, cap, x0, x1);
}

// Radix select over LDS members: the key `thr` such that `need` members have key >= thr and the
// number of members with key > thr (returned in above).  key_of(e) / member(e) index 0..n-1.
// d1_known >= 0: every member's key[31:20] is d1_known (the first digit pass is skipped).
template <int NT, typename KeyOf, typename Member>
__device__ __forceinline__ uint32_t radix_select(int n, int need, KeyOf key_of, Member member, int* hist, int* s_wtot, int* s_res,
                                 int& above, int d1_known = -1) {
  uint32_t d1;
  int ab = 0;
  int need2 = need;
  if (d1_known >= 0) {
    d1 = static_cast<uint32_t>(d1_known);
  } else {
    zero_lds<NT>(hist, kBins);
    __syncthreads();
    for (int e = threadIdx.x; e < n; e += NT)
      if (member(e)) hist_add(hist, key_of(e) >> 20);
    __syncthreads();
    find_threshold<kBins, NT>(hist, need, s_wtot, s_res);
    d1 = static_cast<uint32_t>(s_res[0]);
    ab = s_res[1];
    need2 = need - s_res[1];
  }
  zero_lds<NT>(hist, kBins);
  __syncthreads();
  for (int e = threadIdx.x; e < n; e += NT) {
    if (!member(e)) continue;
    const uint32_t k = key_of(e);
    if ((k >> 20) == d1) hist_add(hist, (k >> 8) & 0xFFFu);
  }
  __syncthreads();
  find_threshold<kBins, NT>(hist, need2, s_wtot, s_res);
  const uint32_t p24 = (d1 << 12) | static_cast<uint32_t>(s_res[0]);
  ab += s_res[1];
  const int need3 = need2 - s_res[1];
  zero_lds<NT>(hist, 256);
  __syncthreads();
  for (int e = threadIdx.x; e < n; e += NT) {
    if (!member(e)) continue;
    const uint32_t k = key_of(e);
    if ((k >> 8) == p24) hist_add(hist, k & 0xFFu);
  }
  __syncthreads();
  find_threshold<256, NT>(hist, need3, s_wtot, s_res);
  above = ab + s_res[1];
  return (p24 << 8) | static_cast<uint32_t>(s_res[0]);
}

template <int NT, int CAP>
struct alignas(16) ResolveLds {  // 16-B LDS accesses into hist, ck and ci
  int hist[kBins];
  uint32_t ck[CAP + kWave];  // + one discard word per lane (collect_ge)
  int ci[CAP + kWave];
  int scan[2 * (NT / kWave)];
  int wtot[NT / kWave];
  int red[NT / kWave];
  int res[6];
  int misc[8];
};

// The threshold of a row from its candidates in LDS (L.ck, n of them, all of 12-bit digit d1,
// or d1 < 0: unknown) of which `need` are to be taken: the key thr of the need-th largest and
// the number of ties at thr among them (taken from the lowest tokens).
template <int NT, int CAP>
__device__ __forceinline__ uint32_t select_lds(ResolveLds<NT, CAP>& L, int n, int d1, int need, int& remaining) {
  int gt;
  const uint32_t thr = radix_select<NT>(
      n, need, [&](int e) { return L.ck[e]; }, [](int) { return true; }, L.hist, L.wtot, L.res, gt, d1);
  remaining = need - gt;
  return thr;
}

// The same by re-reading the row (its bin-t1 candidates did not fit in LDS): digit passes over
// key[19:8], then key[7:0], of the row's tokens in bin t1.
template <bool kVec, int NT, int CAP>
__device__ __forceinline__ uint32_t select_rescan(ResolveLds<NT, CAP>& L, const RowSrc& r, uint32_t t1, int need1, int& remaining) {
  zero_lds<NT>(L.hist, kBins);
  __syncthreads();
  for (int b = static_cast<int>(threadIdx.x) * 4; b < r.len; b += NT * 4) {
    uint32_t k[4];
    const uint32_t v = load_keys4<kVec>(r, b, k);
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (((v >> j) & 1u) && (k[j] >> 20) == t1) hist_add(L.hist, (k[j] >> 8) & 0xFFFu);
  }
  __syncthreads();
  find_threshold<kBins, NT>(L.hist, need1, L.wtot, L.res);
  const uint32_t prefix24 = (t1 << 12) | static_cast<uint32_t>(L.res[0]);
  const int need2 = need1 - L.res[1];
  zero_lds<NT>(L.hist, 256);
  __syncthreads();
  for (int b = static_cast<int>(threadIdx.x) * 4; b < r.len; b += NT * 4) {
    uint32_t k[4];
    const uint32_t v = load_keys4<kVec>(r, b, k);
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (((v >> j) & 1u) && (k[j] >> 8) == prefix24) hist_add(L.hist, k[j] & 0xFFu);
  }
  __syncthreads();
  find_threshold<256, NT>(L.hist, need2, L.wtot, L.res);
  remaining = need2 - L.res[1];
  return (prefix24 << 8) | static_cast<uint32_t>(L.res[0]);
}

// Ordered emission by one CTA streaming the row once more (the exact and heavy-tie paths): every
// token with key > thr to dst[0, kTopK - remaining), the first `remaining` tokens with key ==
// thr to dst[kTopK - remaining, kTopK), each part in ascending token order.  A thread owns 16
// consecutive tokens of each 16 NT-token step (one block prefix per part and step); the next
// step's scores are loaded before this step's prefixes.  Stops once both parts are complete.
template <bool kVec, int NT>
__device__ __forceinline__ void emit_row(const RowSrc& r, uint32_t thr, int remaining, const PtRow& pt, int32_t* dst, int* s_scan) {
  constexpr int kStep = NT * 16;
  const int tie_base = kTopK - remaining;
  const int t0 = static_cast<int>(threadIdx.x) * 16;
  int na = 0, nt = 0, parity = 0;
  Quad cur[4], nxt[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) load_quad<kVec>(r, t0 + 4 * u, cur[u]);
  for (int b = 0; b < r.len && (na < tie_base || nt < remaining); b += kStep) {  // block-uniform
    const int i0 = b + t0;
#pragma unroll
    for (int u = 0; u < 4; ++u) load_quad<kVec>(r, i0 + kStep + 4 * u, nxt[u]);
    uint32_t fa = 0, ft = 0;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      uint32_t k[4];
      const uint32_t v = quad_keys(r, i0 + 4 * u, cur[u], k);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const bool valid = (v >> j) & 1u;
        fa |= static_cast<uint32_t>(valid && k[j] > thr) << (4 * u + j);
        ft |= static_cast<uint32_t>(valid && k[j] == thr) << (4 * u + j);
      }
    }
    int ta, tt;
    int pa = block_prefix<NT, true>(__popc(fa), ta, s_scan, parity);
    parity ^= 1;
    int pq = block_prefix<NT, true>(__popc(ft), tt, s_scan, parity);
    parity ^= 1;
    pa += na;
    pq += nt;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      if ((fa >> e) & 1u) put(dst, pa++, i0 + e);
      if ((ft >> e) & 1u) {
        if (pq < remaining) put(dst, tie_base + pq, i0 + e);
        ++pq;
      }
    }
    na += ta;
    nt += tt;
#pragma unroll
    for (int u = 0; u < 4; ++u) cur[u] = nxt[u];
  }
  // The row's 2048 slots hold token indices now (every slot is written: kTopK - remaining taken
  // above the threshold, remaining ties); the barrier's workgroup fence makes each lane's stores
  // visible to the others.  Then one pass turns them into page-table entries, a thread's gathers
  // going out together (taken one at a time inside the loop's branches, each waited for the one
  // before).
  __syncthreads();
  constexpr int kPer = kTopK / NT;
  int32_t tk[kPer];
#pragma unroll
  for (int j = 0; j < kPer; ++j) tk[j] = dst[threadIdx.x + j * NT];
#pragma unroll
  for (int j = 0; j < kPer; ++j) tk[j] = pt.at(tk[j], true);
#pragma unroll
  for (int j = 0; j < kPer; ++j) dst[threadIdx.x + j * NT] = tk[j];
}

// Ordered emission of a resolved selection whose tokens the block's threads hold in registers:
// each(fn) calls fn(token, tie, value) for every taken token this thread holds (tie: key == the
// threshold, else key above it; value: its page-table entry).  Per window of kEmitWin tokens, a
// bitmap of each part's tokens (`bits`, 4096 words: [0, 2048) above the threshold, [2048, 4096)
// the ties) and the prefix counts of its words (`pre`) give every token its rank within its
// part: slot rank for the first part, n_above + rank for the ties (the reference's order).
// Window 0's bitmap must be zero on entry; *n_ties is read after the first barrier.  Three
// barriers a window; one window covers a row of up to 64K tokens.
constexpr int kEmitWords = kBins / 2;
constexpr int kEmitWin = kEmitWords * 32;

// kLaneId: the lane index computed anew instead of kept since the row's start, a register less there.
template <int NT, bool kLaneId = false, typename Each>
__device__ __forceinline__ void emit_held(Each each, const int* n_ties, uint32_t* bits, uint16_t* pre, int* s_w,
                                          int len, int32_t* dst) {
  constexpr int WPT = kBins / NT;  // words a thread zeroes and counts; all of one part
  static_assert(WPT * NT == kBins && WPT % 4 == 0 && kEmitWords % WPT == 0, "bitmap split over the block");
  const int tid = threadIdx.x;
  uint4* b4 = reinterpret_cast<uint4*>(bits + tid * WPT);
  int base_a = 0, base_t = 0;
  for (int w0 = 0; w0 < len; w0 += kEmitWin) {  // block-uniform
    if (w0 > 0) {
#pragma unroll
      for (int j = 0; j < WPT / 4; ++j) b4[j] = make_uint4(0u, 0u, 0u, 0u);
      __syncthreads();
    }
    each([&](int tok, bool tie, int32_t) {
      const int x = tok - w0;
      if (static_cast<unsigned>(x) < static_cast<unsigned>(kEmitWin))
        atomicOr(&bits[(tie ? kEmitWords : 0) + (x >> 5)], 1u << (x & 31));
    });
    __syncthreads();
    if (w0 == 0) base_t = kTopK - *n_ties;
    int pc[WPT];
    int c = 0;
#pragma unroll
    for (int j = 0; j < WPT / 4; ++j) {
      const uint4 q = b4[j];
      pc[4 * j] = c;
      c += __popc(q.x);
      pc[4 * j + 1] = c;
      c += __popc(q.y);
      pc[4 * j + 2] = c;
      c += __popc(q.z);
      pc[4 * j + 3] = c;
      c += __popc(q.w);
    }
    int total;
    int ex = block_excl_sum<NT, kLaneId>(c, total, s_w);
    int tot_a = 0;  // the first part's count in this window: the words of threads [0, NT / 2)
#pragma unroll
    for (int v = 0; v < NT / kWave / 2; ++v) tot_a += s_w[v];
    if (tid >= NT / 2) ex -= tot_a;
#pragma unroll
    for (int j = 0; j < WPT; ++j) pre[tid * WPT + j] = static_cast<uint16_t>(ex + pc[j]);
    __syncthreads();
    each([&](int tok, bool tie, int32_t v) {
      const int x = tok - w0;
      if (static_cast<unsigned>(x) < static_cast<unsigned>(kEmitWin)) {
        const int wd = (tie ? kEmitWords : 0) + (x >> 5);
        const int rank = pre[wd] + __popc(bits[wd] & ((1u << (x & 31)) - 1u));
        put(dst, (tie ? base_t : base_a) + rank, v);
      }
    });
    base_a += tot_a;
    base_t += total - tot_a;
    if (w0 + kEmitWin < len) __syncthreads();  // the next window reuses bits, pre and s_w
  }
}

// The exact selection of one row by one CTA (the sampled kernels' fallback): pass-1 histogram;
// sparse fast path (threshold +0); or collection of the threshold bin's candidates (up to CAP in
// L.ck / L.ci), their threshold in LDS or by re-reading the row; then the ordered emission.
template <bool kVec, int NT, int CAP>
__device__ __forceinline__ void exact_row(ResolveLds<NT, CAP>& L, const RowSrc& r, const PtRow& pt, int32_t* dst) {
  constexpr int kStep = NT * 4 * kUnroll;
  int pos, zeros;
  pass_hist<kVec, NT>(r, 0, r.len, L.hist, L.red, pos, zeros);
  if (threadIdx.x == 0 && zeros) L.hist[kZeroBin] += zeros;
  __syncthreads();
  const Meta m = row_meta<NT>(L.hist, pos, zeros, L.wtot, L.res);
  if (m.fast) {  // block-uniform
    emit_row<kVec, NT>(r, kZeroKey, kTopK - m.pos, pt, dst, L.scan);
    return;
  }
  const int need1 = kTopK - m.above1;
  int remaining;
  uint32_t thr;
  if (m.n_t1 > CAP) {  // block-uniform: pass 1 counted more keys in bin t1 than the list holds
    thr = select_rescan<kVec>(L, r, m.t1, need1, remaining);
  } else {
    const int b0 = static_cast<int>(threadIdx.x) * 4;
    Batch x0, x1;
    load_batch<kVec, NT>(r, b0, x0);
    load_batch<kVec, NT>(r, b0 + kStep, x1);
    if (threadIdx.x == 0) L.misc[1] = 0;
    __syncthreads();
    collect_bin<kVec, NT>(r, b0, (r.len + kStep - 1) / kStep, m.t1, L.ck, L.ci, &L.misc[1], CAP, x0, x1);
    __syncthreads();
    const int n_c = L.misc[1];
    thr = n_c <= CAP ? select_lds(L, n_c, static_cast<int>(m.t1), need1, remaining)
                     : select_rescan<kVec>(L, r, m.t1, need1, remaining);
  }
  emit_row<kVec, NT>(r, thr, remaining, pt, dst, L.scan);
}

// The reference takes the threshold +0, with no ties, whenever positives <= 2048 <= positives +
// zeros (its sparse fast path, sparse_mask_topk.cu:199-234); that differs from the 2048th largest
// key only when the row holds exactly 2048 positive keys -- then all of them come out in one
// ascending run.  The candidates hold every key >= cut.thr, so exactly 2048 positive candidates
// are the whole selection; the row then has no other positive key if cut.thr <= the smallest
// positive key.  From the n_pos positive candidates: 1 for that case, 0 when the 2048th largest
// key is the reference's threshold, -1 when positives below cut.thr may exist and the count has
// to come from the exact path.
__device__ __forceinline__ int sparse_fast_case(int n_pos, const SampleCut& cut) {
  if (n_pos != kTopK) return 0;
  return cut.thr <= kZeroKey + 1u ? 1 : -1;
}

// The first `need` tokens of key +0 in token order, as page-table entries from dst[kTopK - need] on;
// false, with nothing usable written, when the row holds fewer.  A thread owns 16 consecutive tokens of
// each 16 NT-token step; rows that come here are mostly zeros, so one step is the rule.
template <bool kVec, int NT>
__device__ __forceinline__ bool emit_zeros(const RowSrc& r, int need, const PtRow& pt, int32_t* dst, int* s_scan) {
  constexpr int kStep = NT * 16;
  const int base = kTopK - need;
  int n = 0, parity = 0;
  for (int b = 0; b < r.len && n < need; b += kStep) {  // block-uniform
    const int i0 = b + static_cast<int>(threadIdx.x) * 16;
    uint32_t f = 0;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      uint32_t k[4];
      const uint32_t v = load_keys4<kVec>(r, i0 + 4 * u, k);
#pragma unroll
      for (int j = 0; j < 4; ++j) f |= static_cast<uint32_t>(((v >> j) & 1u) && k[j] == kZeroKey) << (4 * u + j);
    }
    int total;
    int p = n + block_prefix<NT, true>(__popc(f), total, s_scan, parity);
    parity ^= 1;
    for (; f && p < need; f &= f - 1, ++p) put(dst, base + p, i0 + static_cast<int>(__builtin_ctz(f)));
    n += total;
  }
  if (n < need) return false;
  __syncthreads();  // the token indices are there for every lane: turned into entries in one pass
  constexpr int kPer = kTopK / NT;
  int32_t tk[kPer];
#pragma unroll
  for (int j = 0; j < kPer; ++j) {
    const int i = static_cast<int>(threadIdx.x) + j * NT;
    tk[j] = i >= base ? dst[i] : 0;
  }
#pragma unroll
  for (int j = 0; j < kPer; ++j) {
    const int i = static_cast<int>(threadIdx.x) + j * NT;
    const int32_t e = pt.at(tk[j], true);
    if (i >= base) dst[i] = e;
  }
  return true;
}

// A row whose n < 2048 positive keys are all collected (load as resolve_cands): the reference's sparse
// fast path, threshold +0 -- the positives in token order, then the first zeros.  False when the row has
// too few zeros for that (the 2048th key is negative): the caller runs exact_row.
template <bool kVec, int NT, int CAP, typename Load>
__device__ __forceinline__ bool sparse_row(ResolveLds<NT, CAP>& L, int n, const RowSrc& r, const PtRow& pt, int32_t* dst,
                                           Load load) {
  constexpr int EPT = kTopK / NT;
  const int tid = threadIdx.x;
  int tt[EPT];
  int32_t pv[EPT];
#pragma unroll
  for (int j = 0; j < EPT; ++j) {
    const int e = tid + j * NT;
    tt[j] = e < n ? load(e) : 0;
  }
#pragma unroll
  for (int j = 0; j < EPT; ++j) pv[j] = pt.at(tt[j], tid + j * NT < n);
  uint32_t* bits = reinterpret_cast<uint32_t*>(L.hist);
  constexpr int WPT = kBins / NT;
  uint4* b4 = reinterpret_cast<uint4*>(bits + tid * WPT);
#pragma unroll
  for (int j = 0; j < WPT / 4; ++j) b4[j] = make_uint4(0u, 0u, 0u, 0u);
  if (tid == 0) L.misc[3] = 0;
  // (its barriers order the zeroed bitmap and the list's reads before the emission)
  if (!emit_zeros<kVec, NT>(r, kTopK - n, pt, dst, L.scan)) return false;  // block-uniform
  __syncthreads();
  emit_held<NT>(
      [&](auto&& fn) {
#pragma unroll
        for (int j = 0; j < EPT; ++j)
          if (tid + j * NT < n) fn(tt[j], false, pv[j]);
      },
      &L.misc[3], bits, reinterpret_cast<uint16_t*>(L.ci + CAP - kBins / 2), L.wtot, r.len, dst);
  return true;
}

// Resolves n (kTopK <= n <= CAP) collected candidates (keys >= cut.thr) that hold the row's top
// 2048; load(e, k, t) fetches candidate e (from LDS, or from the row's published list).  A
// histogram of their digit cand_digit gives the threshold digit t1: candidates above it are
// taken, its members are ranked exactly by (key desc, token asc) -- a handful by the choice of
// the digit -- which also gives the threshold key; the taken tokens then go out in order
// (emit_held).  More members than threads (heavy ties) select the threshold by radix passes
// and emit by re-reading the row r.
// Returns false, having written nothing, when the row's positive keys must be counted exactly
// first (sparse_fast_case): the caller runs exact_row.
// kGivenPv: load(e, key, token, entry) also hands over each candidate's page-table entry
// (gathered by the CTA that collected it); otherwise load(e, key, token) and the entries are
// gathered here.
template <bool kVec, bool kGivenPv = false, int NT, int CAP, typename Load>
__device__ __forceinline__ bool resolve_cands(ResolveLds<NT, CAP>& L, int n, const SampleCut& cut, const RowSrc& r, const PtRow& pt,
                              int32_t* dst, Load load) {
  constexpr int EPT = CAP / NT;
  static_assert(EPT * NT == CAP, "candidates split over the block");
  static_assert(CAP >= 2 * kTopK && 3 * NT + kBins / 2 <= CAP, "LDS layout of the ordered emission");
  const int tid = threadIdx.x;
  uint32_t kk[EPT];
  int tt[EPT];
  int32_t pv[EPT];
#pragma unroll
  for (int j = 0; j < EPT; ++j) {  // every load in flight before the first use
    const int e = tid + j * NT;
    kk[j] = 0u;
    tt[j] = 0;
    pv[j] = -1;
    if (e < n) {
      if constexpr (kGivenPv) load(e, kk[j], tt[j], pv[j]);
      else load(e, kk[j], tt[j]);
    }
  }
  // page-table entries, fetched while the threshold is searched; with more than 8 candidates a
  // thread (the wide list) only the taken ones, once known, which keeps the registers in hand
  constexpr bool kLatePv = EPT > 8 && !kGivenPv;
  if constexpr (!kLatePv && !kGivenPv) {
#pragma unroll
    for (int j = 0; j < EPT; ++j) pv[j] = pt.at(tt[j], tid + j * NT < n);
  }
  zero_lds<NT>(L.hist, kBins);
  if (tid < 8) L.misc[tid] = 0;
  __syncthreads();
  int n_pos = 0;  // candidates with a positive key
#pragma unroll
  for (int j = 0; j < EPT; ++j) {
    if (tid + j * NT < n) {
      atomicAdd(&L.hist[cand_digit(kk[j], cut)], 1);
      n_pos += kk[j] > kZeroKey;
    }
  }
  n_pos = wave_sum(n_pos);
  if (lane_id() == 0 && n_pos) atomicAdd(&L.misc[4], n_pos);
  __syncthreads();
  find_threshold<kBins, NT>(L.hist, kTopK, L.wtot, L.res);
  const uint32_t t1 = static_cast<uint32_t>(L.res[0]);
  const int above1 = L.res[1];
  const int n_t1 = L.res[2];
  const int need1 = kTopK - above1;
  const int plus0 = sparse_fast_case(L.misc[4], cut);
  if (plus0 < 0) return false;  // block-uniform
  static_assert(EPT <= 16, "masks hold 16 candidates");
  uint32_t fa = 0, fm = 0;
#pragma unroll
  for (int j = 0; j < EPT; ++j) {
    const bool in = tid + j * NT < n;
    const uint32_t d = cand_digit(kk[j], cut);
    fa |= static_cast<uint32_t>(in && d > t1) << j;
    fm |= static_cast<uint32_t>(in && d == t1) << j;
  }
  if constexpr (kLatePv) {
#pragma unroll
    for (int j = 0; j < EPT; ++j) pv[j] = pt.at(tt[j], ((fa | fm) >> j) & 1u);
  }
  if (n_t1 > NT) {  // block-uniform: heavy ties at the threshold digit
    int pm = wave_slot_n(__popc(fm), &L.misc[1]);
#pragma unroll
    for (int j = 0; j < EPT; ++j) {
      if ((fm >> j) & 1u) {
        L.ck[pm] = kk[j];
        L.ci[pm] = tt[j];
        ++pm;
      }
    }
    __syncthreads();
    int remaining;
    const uint32_t thr = select_lds(L, n_t1, -1, need1, remaining);
    emit_row<kVec, NT>(r, plus0 ? kZeroKey : thr, plus0 ? 0 : remaining, pt, dst, L.scan);
    return true;
  }
  // The members of digit t1 go to L.ci, the bitmap of the ordered emission (zeroed here) is
  // L.hist and its word prefixes the end of L.ci; the other taken tokens stay in registers.
  uint32_t* mk = reinterpret_cast<uint32_t*>(L.ci);
  int* mt = L.ci + NT;
  int* mv = L.ci + 2 * NT;
  uint16_t* pre = reinterpret_cast<uint16_t*>(L.ci + CAP - kBins / 2);
  uint32_t* bits = reinterpret_cast<uint32_t*>(L.hist);
  {
    int pm = wave_slot_n(__popc(fm), &L.misc[1]);
#pragma unroll
    for (int j = 0; j < EPT; ++j) {
      if ((fm >> j) & 1u) {
        mk[pm] = kk[j];
        mt[pm] = tt[j];
        mv[pm] = pv[j];
        ++pm;
      }
    }
    constexpr int WPT = kBins / NT;
    uint4* b4 = reinterpret_cast<uint4*>(bits + tid * WPT);
#pragma unroll
    for (int j = 0; j < WPT / 4; ++j) b4[j] = make_uint4(0u, 0u, 0u, 0u);
  }
  __syncthreads();
  bool take = false, tie = false;
  int tok = 0, val = 0;
  {
    // A member is taken when its (key desc, token asc) rank is below need1; it is a tie when the
    // members with a key >= its own reach need1, i.e. its key is the threshold (the need1-th).
    // With exactly 2048 positive keys the reference's threshold is +0 and nothing is a tie.
    const int m1 = __builtin_amdgcn_readfirstlane(n_t1);
    if (m1 <= kWave) {  // block-uniform: wave 0 ranks up to 64 members from registers, each lane
                        // against every other by readlane (9.5 -> 8.5 us for one 4096-token row)
      if (tid < kWave) {
        const uint32_t k = tid < m1 ? mk[tid] : 0u;
        const int tk = tid < m1 ? mt[tid] : 0;
        int rank = 0, ge = 0;
        for (int j = 0; j < m1; ++j) {
          const uint32_t kj = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(k), j));
          const int tj = __builtin_amdgcn_readlane(tk, j);
          rank += kj > k || (kj == k && tj < tk);
          ge += kj >= k;
        }
        if (tid < m1) {
          tok = tk;
          val = mv[tid];
          take = rank < need1;
          tie = take && !plus0 && ge >= need1;
        }
      }
    } else if (tid < n_t1) {
      const uint32_t k = mk[tid];
      tok = mt[tid];
      val = mv[tid];
      int rank = 0, ge = 0;
      int j = 0;
#pragma unroll 4
      for (; j + 4 <= n_t1; j += 4) {  // 16-B LDS reads (mk and mt are 16-B aligned)
        const uint4 kj = *reinterpret_cast<const uint4*>(mk + j);
        const int4 tj = *reinterpret_cast<const int4*>(mt + j);
        rank += (kj.x > k || (kj.x == k && tj.x < tok)) + (kj.y > k || (kj.y == k && tj.y < tok)) +
                (kj.z > k || (kj.z == k && tj.z < tok)) + (kj.w > k || (kj.w == k && tj.w < tok));
        ge += (kj.x >= k) + (kj.y >= k) + (kj.z >= k) + (kj.w >= k);
      }
      for (; j < n_t1; ++j) {
        rank += mk[j] > k || (mk[j] == k && mt[j] < tok);
        ge += mk[j] >= k;
      }
      take = rank < need1;
      tie = take && !plus0 && ge >= need1;
    }
    wave_slot(tie, &L.misc[3]);  // the tie count, read by emit_held after its first barrier
  }
  emit_held<NT, !kVec && CAP == kCapS>(
      [&](auto&& fn) {
#pragma unroll
        for (int j = 0; j < EPT; ++j)
          if ((fa >> j) & 1u) fn(tt[j], false, pv[j]);
        if (take) fn(tok, tie, val);
      },
      &L.misc[3], bits, pre, L.wtot, r.len, dst);
  return true;
}

// ---------------------------------------------------------------------------------------------
// Rows of up to NT * 4 * Q tokens held in registers, one CTA a row, exact whatever the scores: no
// sample, no candidate list, no fallback and no LDS histogram.  The 2048th largest key is found by
// counting: a round counts the keys >= a probe (one compare and one ballot's popcount a key, one barrier
// for the waves' counts), and the probes close in on it until at most 64 keys are left between, which
// every wave ranks for itself.  Probes: the smallest positive key (it settles the rows of the sparse fast
// path in one or two rounds), the row's quantile if its scores were normal (mean and deviation come
// with the first count), a step from there by the normal density, then interpolation of the counts
// between the bracket's float values with the Illinois weights; four or five rounds on the indexer's
// logits.  A round is about 0.65 us, so rows whose scores are far from normal, which take eight to twelve, gain
// nothing from being held where few rows are in flight (64 rows of 2049-4096 tokens, ratios of normals 14.4 ->
// 16.6 us; 1024 x 4096 34 -> 23), nor do 4096 normal scores, whose 2048th lies beside zero, the first count's own
// probe (250 rows 9.4 -> 10.8).  Every third round from the sixth pulls the bracket's ends in to keys of the row, which ends
// the search on heavy ties, and past kHeldGuess rounds the probes halve the key range, so that no input
// takes more than 32 further ones.
constexpr int kHeldGuess = 18;
constexpr int kHeldQ = 4;                      // quads a thread of the kTs-thread kernels
constexpr int kHeldRow = kTs * 4 * kHeldQ;     // rows of up to this many tokens are held

__device__ __forceinline__ float key_value(uint32_t k) {
  return __uint_as_float((k & 0x80000000u) ? (k ^ 0x80000000u) : ~k);
}

// max / min over the wave, in every lane (16-lane rows by DPP, then the rows' first lanes)
template <bool kMax>
__device__ __forceinline__ uint32_t wave_extreme(uint32_t x) {
  auto pick = [](uint32_t p, uint32_t q) { return kMax ? max(p, q) : min(p, q); };
  x = pick(x, static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(static_cast<int>(x), 0xB1, 0xF, 0xF, false)));
  x = pick(x, static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(static_cast<int>(x), 0x4E, 0xF, 0xF, false)));
  x = pick(x, static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(static_cast<int>(x), 0x141, 0xF, 0xF, false)));
  x = pick(x, static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(static_cast<int>(x), 0x140, 0xF, 0xF, false)));
  auto at = [&](int l) { return static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(x), l)); };
  return pick(pick(at(0), at(16)), pick(at(32), at(48)));
}

__device__ __forceinline__ float wave_total(float x) {
  auto dpp = [](float y, auto c) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(y), decltype(c)::value, 0xF, 0xF, false));
  };
  x += dpp(x, std::integral_constant<int, 0xB1>{});
  x += dpp(x, std::integral_constant<int, 0x4E>{});
  x += dpp(x, std::integral_constant<int, 0x141>{});
  x += dpp(x, std::integral_constant<int, 0x140>{});
  auto at = [&](int l) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), l)); };
  return (at(0) + at(16)) + (at(32) + at(48));
}

// z with P(normal > z) = q (Abramowitz and Stegun 26.2.23, |error| < 4.5e-4).
__device__ __forceinline__ float normal_quantile(float q) {
  const float t = sqrtf(-2.0f * __logf(fminf(q, 1.0f - q)));
  const float z = t - (2.515517f + t * (0.802853f + t * 0.010328f)) /
                          (1.0f + t * (1.432788f + t * (0.189269f + t * 0.001308f)));
  return q <= 0.5f ? z : -z;
}

template <int NT, int Q>
struct alignas(16) HeldLds {
  int cnt[2][NT / kWave];
  uint32_t top[NT / kWave];
  uint32_t low[NT / kWave];
  float sum[NT / kWave];
  float sq[NT / kWave];
  uint32_t tot[Q * (NT / kWave)];
  uint32_t mem[kWave];
  int n_mem;
  uint16_t out[kTopK + kWave];  // the selected tokens in output order; then a discard word a lane
};

template <bool kVec, int NT, int Q>
__device__ __forceinline__ void held_row(HeldLds<NT, Q>& L, const RowSrc& r, const PtRow& pt, int32_t* dst) {
  constexpr int W = NT / kWave;
  constexpr int QW = Q * W;
  static_assert(W % 4 == 0 && QW <= 2 * kWave, "counts read 16 B at a time; two totals a lane at most");
  static_assert(NT * 4 * Q <= 65536 && kTopK % NT == 0, "16-bit tokens; the output split over the block");
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int len = r.len;
  // Quad u of thread tid: tokens 4 (u NT + tid) ..; tokens past the row get key 0, which only ties
  // with real tokens before them, and a row has more than 2048 of those.
  uint32_t k[Q][4];
  float sum = 0.0f, sq = 0.0f;
  {
    Quad q[Q];
#pragma unroll
    for (int u = 0; u < Q; ++u) load_quad<kVec>(r, (u * NT + tid) * 4, q[u]);
#pragma unroll
    for (int u = 0; u < Q; ++u) {
      const uint32_t live = quad_keys(r, (u * NT + tid) * 4, q[u], k[u]);
      if ((u + 1) * NT * 4 > len) {  // block-uniform: the quads the row ends in
#pragma unroll
        for (int j = 0; j < 4; ++j) k[u][j] = (live >> j) & 1u ? k[u][j] : 0u;
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float x = k[u][j] ? key_value(k[u][j]) : 0.0f;
        sum += x;
        sq = fmaf(x, x, sq);
      }
    }
  }
  // The row's keys >= key; every thread gets the sum.  parity alternates over the calls: a wave may
  // write its next count while another still reads this one, not the one after.
  int parity = 0;
  auto count_ge = [&](uint32_t key) {
    int c = 0;
#pragma unroll
    for (int u = 0; u < Q; ++u) {
#pragma unroll
      for (int j = 0; j < 4; ++j) c += __popcll(__ballot(k[u][j] >= key));
    }
    if (lane == 0) L.cnt[parity][w] = c;
    __syncthreads();
    int n = 0;
#pragma unroll
    for (int v = 0; v < W / 4; ++v) {
      const int4 x = reinterpret_cast<const int4*>(L.cnt[parity])[v];
      n += x.x + x.y + x.z + x.w;
    }
    parity ^= 1;
    return uniform(n);
  };
  // Pulls lo > 0 up and hi down to the nearest keys of the row (a count follows before the next call).
  auto ends = [&](uint32_t& lo, uint32_t& hi) {
    uint32_t m = 0xFFFFFFFFu, t = 0u;
#pragma unroll
    for (int u = 0; u < Q; ++u) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        m = min(m, k[u][j] >= lo ? k[u][j] : 0xFFFFFFFFu);
        t = max(t, k[u][j] <= hi ? k[u][j] : 0u);
      }
    }
    m = wave_extreme<false>(m);
    t = wave_extreme<true>(t);
    if (lane == 0) {
      L.low[w] = m;
      L.top[w] = t;
    }
    __syncthreads();
#pragma unroll
    for (int v = 0; v < W / 4; ++v) {
      const uint4 x = reinterpret_cast<const uint4*>(L.top)[v];
      const uint4 y = reinterpret_cast<const uint4*>(L.low)[v];
      t = max(max(max(t, x.x), max(x.y, x.z)), x.w);
      m = min(min(min(m, y.x), min(y.y, y.z)), y.w);
    }
    lo = static_cast<uint32_t>(uniform(static_cast<int>(m)));
    hi = static_cast<uint32_t>(uniform(static_cast<int>(t)));
  };
  sum = wave_total(sum);
  sq = wave_total(sq);
  if (lane == 0) {
    L.sum[w] = sum;
    L.sq[w] = sq;
    if (w == 0) L.n_mem = 0;
  }
  const int n_pos = count_ge(kZeroKey + 1u);

  // thr: the 2048th largest key (+0 with no ties when the row holds exactly 2048 positive keys, the
  // reference's sparse fast path, sparse_mask_topk.cu:199-234).  It lies in [lo, hi]; c_lo keys are
  // >= lo, c_hi are > hi.
  uint32_t thr = kZeroKey;
  if (n_pos != kTopK) {  // block-uniform, like everything below
    sum = sq = 0.0f;
#pragma unroll
    for (int v = 0; v < W / 4; ++v) {
      const float4 f = reinterpret_cast<const float4*>(L.sum)[v];
      const float4 g = reinterpret_cast<const float4*>(L.sq)[v];
      sum += (f.x + f.y) + (f.z + f.w);
      sq += (g.x + g.y) + (g.z + g.w);
    }
    uint32_t lo = 0u, hi = 0xFFFFFFFFu;
    int c_lo = len, c_hi = 0;
    if (n_pos > kTopK) {
      lo = kZeroKey + 1u;
      c_lo = n_pos;
    } else {
      hi = kZeroKey;
      c_hi = n_pos;
    }
    float w_lo = static_cast<float>(c_lo - kTopK), w_hi = static_cast<float>(kTopK - c_hi);
    const float inv_n = __builtin_amdgcn_rcpf(static_cast<float>(len));
    const float mean = sum * inv_n;
    const float dev = __builtin_amdgcn_sqrtf(fmaxf(sq * inv_n - mean * mean, 0.0f));
    const float z = normal_quantile(static_cast<float>(kTopK) * inv_n);
    float next = mean + z * dev;  // the next probe's value, for the first two rounds
    int side = 0;
    bool at_zero = n_pos < kTopK;  // first +0 itself: with its ties it may hold the 2048th
    int round = 0;
    while (lo < hi && c_lo - c_hi > kWave) {
      uint32_t p;  // a probe in (lo, hi]
      if (at_zero) {
        p = hi;
      } else {
        p = float_key(next);
        if (round >= 2 || !(p > lo && p <= hi)) {
          if (lo == 0u || hi == 0xFFFFFFFFu || (round >= 6 && round % 3 == 0)) {
            if (lo == 0u) {  // off key 0, which the tokens past the row hold
              const int c = count_ge(1u);
              if (c < kTopK) break;  // the 2048th is a key 0 of the row's own
              lo = 1u;
              c_lo = c;
            }
            ends(lo, hi);
            if (lo == hi) break;
          }
          const float fl = key_value(lo), fh = key_value(hi);
          // aimed a few keys to the near side of the 2048th, to bring the farther end close
          const float aim = c_lo - c_hi <= 48 ? 0.0f : (c_lo - kTopK > kTopK - c_hi ? 12.0f : -12.0f);
          const float f = (w_lo - aim) * __builtin_amdgcn_rcpf(w_lo + w_hi);
          p = float_key(fl + (fh - fl) * fminf(fmaxf(f, 0.02f), 0.98f));
          p = p > lo ? p : lo + 1u;
          p = p < hi ? p : hi;
          if (round >= kHeldGuess) p = lo + (hi - lo + 1u) / 2u;
        }
        ++round;
      }
      p = static_cast<uint32_t>(uniform(static_cast<int>(p)));
      const int c = count_ge(p);
      // a step past the quantile by the normal density there, so that the two probes bracket it
      if (!at_zero && round == 1) {
        const float off = static_cast<float>(c - kTopK) * 1.2f + (c >= kTopK ? 20.0f : -20.0f);
        next = key_value(p) + off * 2.5066283f * dev * inv_n * __expf(0.5f * z * z);
      }
      at_zero = false;
      if (c >= kTopK) {
        lo = p;
        c_lo = c;
        w_lo = static_cast<float>(c - kTopK) + 0.5f;
        if (side > 0) w_hi *= 0.5f;
        side = 1;
      } else {
        hi = p - 1u;
        c_hi = c;
        w_hi = static_cast<float>(kTopK - c);
        if (side < 0) w_lo *= 0.5f;
        side = -1;
      }
    }
    thr = lo;
    if (lo < hi && c_lo - c_hi <= kWave) {  // the 2048th is among the at most 64 keys in [lo, hi]
      // those above 0 (tokens past the row hold key 0); fewer of them than needed: it is a key 0
      const uint32_t from = lo > 0u ? lo : 1u;
      const uint32_t span = hi - from;
#pragma unroll
      for (int u = 0; u < Q; ++u) {
        if (min(min(k[u][0] - from, k[u][1] - from), min(k[u][2] - from, k[u][3] - from)) <= span) {
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            if (k[u][j] - from <= span) {
              const int at = atomicAdd(&L.n_mem, 1);
              if (at < kWave) L.mem[at] = k[u][j];
            }
          }
        }
      }
      __syncthreads();
      const int m = uniform(min(L.n_mem, kWave));
      const int need = kTopK - c_hi;
      const uint32_t km = L.mem[lane];
      int gt = 0, ge = 0;
      for (int j = 0; j < m; ++j) {
        const uint32_t kj = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(km), j));
        gt += kj > km;
        ge += kj >= km;
      }
      const uint64_t hit = __ballot(lane < m && gt < need && need <= ge);
      if (hit) thr = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(km), __builtin_ctzll(hit)));
    }
  }

  // Ordered emission: above the threshold in token order, then the ties.  A (quad, wave)'s counts travel
  // in one word (ties in the upper half); their prefix in token order, which every wave forms for
  // itself, places the selected tokens in LDS, and the block writes the row from there: one coalesced
  // store and one page-table gather per output entry.
  int before[Q];  // tokens above the threshold in the lower lanes' part of the quad row
#pragma unroll
  for (int u = 0; u < Q; ++u) {
    int b4 = 0, n_gt = 0, n_eq = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint64_t m = __ballot(k[u][j] > thr);
      b4 = static_cast<int>(__builtin_amdgcn_mbcnt_hi(
          static_cast<uint32_t>(m >> 32), __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(m), static_cast<uint32_t>(b4))));
      n_gt += __popcll(m);
      n_eq += __popcll(__ballot(k[u][j] == thr));
    }
    before[u] = b4;
    if (lane == 0) L.tot[u * W + w] = static_cast<uint32_t>(n_gt) | (static_cast<uint32_t>(n_eq) << 16);
  }
  __syncthreads();
  const uint32_t t0 = lane < QW ? L.tot[lane] : 0u;
  const uint32_t i0 = static_cast<uint32_t>(wave_prefix_sum(static_cast<int>(t0)));
  uint32_t total = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(i0), 63));
  uint32_t t1 = 0u, i1 = 0u;
  if constexpr (QW > kWave) {
    t1 = kWave + lane < QW ? L.tot[kWave + lane] : 0u;
    i1 = total + static_cast<uint32_t>(wave_prefix_sum(static_cast<int>(t1)));
    total = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(i1), 63));
  }
  const int base_t = static_cast<int>(total & 0xFFFFu);
  const int trash = kTopK + lane;
#pragma unroll
  for (int u = 0; u < Q; ++u) {
    const int at = u * W + w;  // wave-uniform
    const bool second = QW > kWave && at >= kWave;
    const uint32_t cw = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(second ? t1 : t0), at & 63));
    if (cw == 0u) continue;  // wave-uniform: nothing selected here
    const uint32_t b = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(second ? i1 : i0), at & 63)) - cw;
    int pa = static_cast<int>(b & 0xFFFFu) + before[u];
    const int tok = (u * NT + tid) * 4;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const bool above = k[u][j] > thr;
      L.out[above ? pa : trash] = static_cast<uint16_t>(tok + j);
      pa += above;
    }
    if (cw >> 16) {  // wave-uniform: ties among them, in (lane, j) order
      int pq = base_t + static_cast<int>(b >> 16);
      int e = 0;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint64_t m = __ballot(k[u][j] == thr);
        e = static_cast<int>(__builtin_amdgcn_mbcnt_hi(
            static_cast<uint32_t>(m >> 32), __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(m), static_cast<uint32_t>(e))));
      }
      pq += e;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const bool tie = k[u][j] == thr;
        L.out[tie ? min(pq, trash) : trash] = static_cast<uint16_t>(tok + j);
        pq += tie;
      }
    }
  }
  __syncthreads();
  constexpr int kPer = kTopK / NT;
  int32_t e[kPer];
#pragma unroll
  for (int j = 0; j < kPer; ++j) e[j] = pt.at(L.out[tid + j * NT], true);
#pragma unroll
  for (int j = 0; j < kPer; ++j) dst[tid + j * NT] = e[j];
}

struct TopkArgs {
  const float* score;
  int64_t score_stride;
  int width;
  const int16_t* mask;
  int64_t mask_stride;
  const int32_t* lengths;
  int rows;
  const int32_t* pt;
  int64_t pt_stride;
  int pt_cols;   // tokens a page-table row covers; tokens past it map to -1
  int pt_shift;  // 0: an entry per token; 6: an entry per 64-token page (PtRow)
  const int32_t* cu;
  int n_req;
  int32_t* out;
  int S;             // CTAs per row of the sampled split kernel
  int T;             // CTAs the balanced split kernel spreads the rows' tokens over
  int32_t* ghist;    // [rows][kBins]  pass-1 histogram
  int32_t* gcnt;     // [rows][2] = (positives, zeros)
  int32_t* ctr;      // per row (stride ctr_stride, 8-B aligned), zero before the split kernels:
                     // exact split [0] output slots taken, [1] candidates published, [2] slice
                     // CTAs finished; sampled split [0] candidates published, [1] CTAs finished
  int64_t ctr_stride;
  uint32_t* c_keys;  // [rows][cap] candidate keys published by the slice CTAs (cap: cap_for)
  int32_t* c_tok;    // [rows][cap] their tokens
  int32_t* c_pv;     // [rows][cap] their page-table entries (the sampled split kernel)
};

__device__ __forceinline__ RowSrc row_src(const TopkArgs& a, int row, int len) {
  RowSrc r;
  r.vals = a.score + static_cast<int64_t>(row) * a.score_stride;
  // without a mask, a dummy in-row address (word t/16 lies inside the row's first t floats)
  r.mask = a.mask ? a.mask + static_cast<int64_t>(row) * a.mask_stride : reinterpret_cast<const int16_t*>(r.vals);
  r.mask_or = a.mask ? 0u : 0xFFFFu;
  r.len = len;
  return r;
}

__device__ __forceinline__ int row_len(const TopkArgs& a, int row) {
  const int l = a.lengths[row];
  return l < 0 ? 0 : (l < a.width ? l : a.width);
}

__device__ __forceinline__ PtRow pt_row(const TopkArgs& a, int row) {
  PtRow p;
  p.p = a.pt_cols > 0 ? a.pt + static_cast<int64_t>(pt_row_of(row, a.cu, a.n_req)) * a.pt_stride : &g_pt_none;
  p.cols = a.pt_cols;
  p.shift = a.pt_shift;
  return p;
}

template <int NT>
__device__ __forceinline__ void copy_short_row(const PtRow& pt, int32_t* dst, int len) {
  for (int i = threadIdx.x; i < kTopK; i += NT) dst[i] = pt.at(i, i < len);
}

// ---------------------------------------------------------------------------------------------
// One CTA a row for scores of at most NT * 4 * Q tokens: all that held_row needs, so that eight waves
// a SIMD hide each other's rounds.
template <bool kVec, int NT, int Q>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(8))) void topk_held_kernel(const TopkArgs a) {
  __shared__ HeldLds<NT, Q> L;
  const int row = blockIdx.x;
  const int len = row_len(a, row);
  const PtRow pt = pt_row(a, row);
  int32_t* dst = a.out + static_cast<int64_t>(row) * kTopK;
  if (len <= kTopK) copy_short_row<NT>(pt, dst, len);
  else held_row<kVec, NT, Q>(L, row_src(a, row, len), pt, dst);
}

// ---------------------------------------------------------------------------------------------
// One CTA per row with pass 1 (histogram + counts) from a.ghist / a.gcnt (the logits kernel's
// fused pass 1): the row's threshold from its exact threshold bin, then the ordered emission.
template <bool kVec>
__global__ __launch_bounds__(kTk) void topk_single_kernel(const TopkArgs a) {
  __shared__ ResolveLds<kTk, kCapC> L;
  constexpr int kStep = kTk * 4 * kUnroll;
  const int row = blockIdx.x;
  const int len = row_len(a, row);
  const PtRow pt = pt_row(a, row);
  int32_t* dst = a.out + static_cast<int64_t>(row) * kTopK;
  if (len <= kTopK) {
    copy_short_row<kTk>(pt, dst, len);
    return;
  }
  const RowSrc r = row_src(a, row, len);
  const int b0 = static_cast<int>(threadIdx.x) * 4;
  // pass-1 slots (4 bins per thread) first, then the first two batches, so that waiting for
  // the histogram does not wait for the batches
  const int4 h4 = reinterpret_cast<const int4*>(a.ghist + static_cast<int64_t>(row) * kBins)[threadIdx.x];
  const int pos = a.gcnt[2 * row];
  const int zeros = a.gcnt[2 * row + 1];
  if (pos <= kTopK && pos + zeros >= kTopK) {  // block-uniform: the threshold is +0
    emit_row<kVec, kTk>(r, kZeroKey, kTopK - pos, pt, dst, L.scan);
    return;
  }
  Batch x0, x1;
  load_batch<kVec, kTk>(r, b0, x0);
  load_batch<kVec, kTk>(r, b0 + kStep, x1);
  if (threadIdx.x == 0) L.misc[1] = 0;
  const int h[4] = {h4.x, h4.y, h4.z, h4.w};
  find_threshold_regs<kTk, 4>(h, kTopK, L.wtot, L.res);
  const uint32_t t1 = static_cast<uint32_t>(L.res[0]);
  const int need1 = kTopK - L.res[1];
  collect_bin<kVec, kTk>(r, b0, (len + kStep - 1) / kStep, t1, L.ck, L.ci, &L.misc[1], kCapC, x0, x1);
  __syncthreads();
  const int n_c = L.misc[1];
  int remaining;
  const uint32_t thr = n_c <= kCapC ? select_lds(L, n_c, static_cast<int>(t1), need1, remaining)
                                    : select_rescan<kVec>(L, r, t1, need1, remaining);
  emit_row<kVec, kTk>(r, thr, remaining, pt, dst, L.scan);
}

// One 512-thread CTA per row against the sampled threshold K* (one read of the row); a count
// past CAP is collected once more above a raised threshold, and the exact path takes a count
// that still misses [2048, CAP].  Two CTAs share a CU, so one's
// latency-bound phases (sample, resolution) overlap the other's collection.  CAP: kCapS, or
// kCapW for wide scores (the expected count grows with the row: 2048 + (4 sqrt(mu) + 2) len /
// 4096 with mu = 2048 * 4096 / len, ~2800 at 64K tokens and ~3150 at 131K, whose sample-to-row
// spread reached 4553 on Student-t keys: rows past kCapS took the exact path at ~300 us each,
// the slab's tail).  kCapW's resolution gathers its page-table entries only once the taken
// candidates are known (prefetched, 10 a thread would not fit in 128 VGPRs), so narrower scores
// keep kCapS and its prefetch.
template <bool kVec, int CAP>
__global__ __launch_bounds__(kTs) __attribute__((amdgpu_waves_per_eu(4))) void topk_row_sampled_kernel(
    const TopkArgs a) {
  __shared__ union Lds {
    ResolveLds<kTs, CAP> res;
    HeldLds<kTs, kHeldQ> held;
    __device__ Lds() {}
  } lds;
  ResolveLds<kTs, CAP>& L = lds.res;
  constexpr int kStep = kTs * 4 * kUnroll;
  constexpr bool kFillZeros = kVec && CAP == kCapS;  // (the others have no registers left for it)
  const int row = blockIdx.x;
  const int len = row_len(a, row);
  const PtRow pt = pt_row(a, row);
  int32_t* dst = a.out + static_cast<int64_t>(row) * kTopK;
  if (len <= kTopK) {
    copy_short_row<kTs>(pt, dst, len);
    return;
  }
  const RowSrc r = row_src(a, row, len);
  if (len <= kHeldRow) {  // block-uniform
    held_row<kVec, kTs, kHeldQ>(lds.held, r, pt, dst);
    return;
  }
  bool done = false;
  {
    const int b0 = static_cast<int>(threadIdx.x) * 4;
    SampleLoads<kTs> smp;
    sample_issue<kVec, kTs>(r, smp);  // the sample first: it is needed first
    Batch x0, x1;
    const SampleLds S{L.hist, L.wtot, L.res};
    // One batch goes out behind the sample, the second once K* is known: with both (64 KB a CTA)
    // queued at once, the waves stall issuing them and the threshold search's barriers wait for
    // the last (a 4096-row prefill slab 327 -> 323 us; the decode split kernel unchanged).
    SampleCut cut = sample_threshold<kTs>(r, smp, S, [&]() { load_batch<kVec, kTs>(r, b0, x0); });
    load_batch<kVec, kTs>(r, b0 + kStep, x1);
    if constexpr (kFillZeros) positives_only(cut);
    if (threadIdx.x == 0) L.misc[2] = 0;
    __syncthreads();
    collect_ge<kVec, kTs>(r, b0, (len + kStep - 1) / kStep, cut.thr, L.ck, L.ci, &L.misc[2], CAP, x0, x1);
    __syncthreads();
    int n = L.misc[2];
    if (n > CAP) {  // block-uniform: more keys >= K* than the list holds (a sample far from the row)
      // The list holds CAP of them, a subset of the row's keys.  The lower edge of the candidate
      // digit (relative to K*) at which the stored keys' suffix count reaches 2048 leaves at least
      // 2048 stored keys at or above it, so it is at most the row's 2048th key: the row's top 2048
      // and their ties are all >= it.  One more pass collects the keys >= it (~2048 * n / CAP when
      // the stored ones are representative) instead of the exact path's three passes over the
      // row (512 rows of 131,072 tokens with ~7000 keys past K*: 382 -> 102 us).
      zero_lds<kTs>(L.hist, kBins);
      __syncthreads();
      for (int e = threadIdx.x; e < CAP; e += kTs) {
        uint32_t k;
        int t;
        collected(L.ck[e], L.ci[e], k, t);
        atomicAdd(&L.hist[cand_digit(k, cut)], 1);
      }
      __syncthreads();
      find_threshold<kBins, kTs>(L.hist, kTopK, L.wtot, L.res);
      // keys of digit >= d are >= thr + (d << shift), which a stored key of digit d bounds
      cut.thr += static_cast<uint32_t>(L.res[0]) << cut.shift;
      // the stored keys at or above it, scaled to the row, past the list: the pass would overflow
      // again (one heavy digit: constant or narrow rows), so the exact path goes first
      if (static_cast<int64_t>(L.res[1] + L.res[2]) * n <= static_cast<int64_t>(CAP) * CAP) {  // block-uniform
        if (threadIdx.x == 0) L.misc[2] = 0;
        __syncthreads();
        collect_ge1<kVec, kTs>(r, b0, (len + kStep - 1) / kStep, cut.thr, L.ck, L.ci, &L.misc[2], CAP);
      }
      __syncthreads();
      n = L.misc[2];
    }
    if (kFillZeros && cut.thr == kPositive && n < kTopK) {  // block-uniform
      if constexpr (kFillZeros) done = sparse_row<kVec>(L, n, r, pt, dst, [&](int e) { return L.ci[e] & 0x7FFFFFFF; });
    } else if (n >= kTopK && n <= CAP) {  // block-uniform
      done = resolve_cands<kVec>(L, n, cut, r, pt, dst, [&](int e, uint32_t& k, int& t) {
        collected(L.ck[e], L.ci[e], k, t);
      });
    }
  }
  if (!done) exact_row<kVec, kTs>(L, r, pt, dst);  // block-uniform
}

// ---------------------------------------------------------------------------------------------
// Cross-CTA hand-over of a row's published candidates (split kernels).  The candidates are stored
// with relaxed agent-scope atomic stores and read back with relaxed agent-scope atomic loads, which
// gfx950 code carries out as `global_store ... sc1` / `global_load ... sc1`: stores written
// through past the XCD's L2 to the device's coherence point, loads that miss the L1 / L2 and read
// from it.  A slice CTA's waves wait for their stores' completion (s_waitcnt vmcnt(0)) before the
// barrier that precedes thread 0's done mark, a device-scope atomic add; the CTA that sees the
// row's last mark issues its loads only after that mark has returned (a barrier and a branch on
// it).  So every candidate is at the coherence point before the last mark exists, and every read
// of it goes there.  An agent-scope acq_rel mark adds an L2 write-back (buffer_wbl2 sc1) per CTA
// and an invalidate (buffer_inv sc1): on the 64-request MTP decode step 81.6 -> 94.9 us with these
// stores, 96.9 us with plain stores and loads under the acq_rel mark (same registers, no scratch,
// same outputs).
__device__ __forceinline__ void candidates_complete() {
  __builtin_amdgcn_s_waitcnt(0);  // this wave's candidate stores have completed
}

// ---------------------------------------------------------------------------------------------
// Split variant.  CTAs cover balanced slices of the rows (split_assign).
// Zeroes the per-row counters of the split path (4 words a row).
__global__ __launch_bounds__(256) void topk_zero_kernel(int32_t* __restrict__ ctr, int rows) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < 4 * rows) ctr[i] = 0;
}

struct SplitLds {
  union {
    struct {
      uint32_t ck[kCapS];
      int ci[kCapS];
    } col;                          // this CTA's candidates of the threshold bin
    ResolveLds<kTs, kCapS> res;     // the row's resolution (last CTA only)
  } u;
  int wtot[kTs / kWave];
  int res[6];
  int n[6];
  long long lsum[kTs / kWave];
  int slot[3];
};

template <int CAP>
struct SampledLds {
  union {
    struct {
      uint32_t ck[CAP + kWave];
      int ci[CAP + kWave];
    } col;                          // this CTA's keys >= K* (raw bits; discard words past CAP)
    ResolveLds<kTs, CAP> res;       // the threshold search; the row's resolution (last CTA)
    HeldLds<kTs, kHeldQ> held;      // a short row
  } u;
  int wtot[kTs / kWave];
  int res[6];
  int misc[2];
  int n[4];
};

// Balanced split: row r gets c_r = ceil(len_r * T / L) CTAs (L = the summed lengths of the rows
// longer than 2048; a row of <= 2048 tokens gets one CTA, which copies it), in row order, so
// that every CTA streams about L / T tokens whatever the length mix; the sum is <= T + rows, the
// grid.  Needs rows <= kTs.  s_slot = {row (-1: none), index among the row's CTAs, c_r}.
template <typename Lds>
__device__ __forceinline__ void split_assign(const TopkArgs& a, int T, Lds& L) {
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int w = tid >> 6;
  const int len = tid < a.rows ? row_len(a, tid) : 0;
  long long big = len > kTopK ? len : 0;
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) big += __shfl_xor(big, o);
  if (lane == 0) L.lsum[w] = big;
  if (tid == 0) L.slot[0] = -1;
  __syncthreads();
  long long total = 0;
#pragma unroll
  for (int v = 0; v < kTs / kWave; ++v) total += L.lsum[v];
  int c = 0;
  if (tid < a.rows) c = len > kTopK ? static_cast<int>((static_cast<long long>(len) * T + total - 1) / total) : 1;
  int inc = c;
#pragma unroll
  for (int o = 1; o < kWave; o <<= 1) {
    const int y = __shfl_up(inc, o);
    if (lane >= o) inc += y;
  }
  if (lane == 63) L.wtot[w] = inc;
  __syncthreads();
  int before = 0;
#pragma unroll
  for (int v = 0; v < kTs / kWave; ++v) before += v < w ? L.wtot[v] : 0;
  const int first = before + inc - c;
  const int cta = blockIdx.x;
  if (cta >= first && cta < first + c) {
    L.slot[0] = tid;
    L.slot[1] = cta - first;
    L.slot[2] = c;
  }
  __syncthreads();
}

// Slice of a row (by split_assign) this CTA covers: [begin, end) of len tokens, n_sl slices in
// the row; false when the CTA has none.  Slices are whole 256-token blocks.
__device__ __forceinline__ bool split_slice(int len, int c, int j, int& begin, int& end, int& n_sl) {
  const int sl = ((len + c - 1) / c + 255) / 256 * 256;
  begin = j * sl;
  end = min(begin + sl, len);
  n_sl = (len + sl - 1) / sl;
  return begin < len;
}

// Pass 1 of one balanced slice (the split kernel's slices) into the row's global histogram and
// positive / zero counts, which start at zero.
// Split with the sampled threshold: CTA c takes slice c % S of row c / S (S CTAs a row, the
// whole grid resident), so it starts loading without a length-dependent assignment.  Every
// CTA of a row computes the same K* from the row's sample, collects its slice's keys >= K* and
// publishes them (device-coherent stores at slots from the row's counter); the last CTA of the
// row resolves them; past CAP (the list then full) it raises K* from the published keys and
// collects the whole row once more itself, and it runs the exact path over the row when the
// count missed [2048, CAP] after that.
// CAP: the row's candidate list, kCapS or kCapW for wide scores (as in the row kernel: one row
// past it made a 128-row top-k of 131K-token rows take 211 us instead of 32).
// Counters (zero on entry): words 0..1 as one 64-bit word (keys published, CTAs done).
template <bool kVec, int CAP>
__global__ __launch_bounds__(kTs) __attribute__((amdgpu_waves_per_eu(4))) void topk_split_sampled_kernel(const TopkArgs a) {
  __shared__ SampledLds<CAP> L;
  constexpr int kStep = kTs * 4 * kUnroll;
  const int tid = threadIdx.x;
  // The S CTAs of a row on one XCD when the rows fill whole octets (CTAs are spread over the 8
  // XCDs by blockIdx % 8): the row's sample is then fetched from HBM once, the other CTAs hit
  // that XCD's L2.
  int row, slice;
  if ((a.rows & 7) == 0) {
    const int l = static_cast<int>(blockIdx.x) >> 3;
    row = ((l / a.S) << 3) | (static_cast<int>(blockIdx.x) & 7);
    slice = l % a.S;
  } else {
    row = blockIdx.x / a.S;
    slice = blockIdx.x - row * a.S;
  }
  const int len = row_len(a, row);
  if (len <= kTopK) {
    if (slice == 0) copy_short_row<kTs>(pt_row(a, row), a.out + static_cast<int64_t>(row) * kTopK, len);
    return;
  }
  const RowSrc r = row_src(a, row, len);
  // the output row and page-table row are formed where they are used, so that nothing beyond
  // the row's scores stays live across the collection loop
  auto dst = [&]() { return a.out + static_cast<int64_t>(row) * kTopK; };
  bool done = false;
  if (len <= kHeldRow) {  // the whole row in one CTA, no split
    if (slice == 0) held_row<kVec, kTs, kHeldQ>(L.u.held, r, pt_row(a, row), dst());
    return;
  }
  {
    int begin, end, n_sl;
    if (!split_slice(len, a.S, slice, begin, end, n_sl)) return;
    const RowSrc rr = row_src(a, row, end);
    const int b0 = begin + tid * 4;
    SampleLoads<kTs> smp;
    sample_issue<kVec, kTs>(r, smp);  // the sample first: it is needed first
    Batch x0, x1;
    if (tid == 0) L.n[0] = 0;
    const SampleLds S{L.u.res.hist, L.wtot, L.res};
    SampleCut cut = sample_threshold<kTs>(r, smp, S, [&]() { load_batch<kVec, kTs>(rr, b0, x0); });
    if constexpr (CAP == kCapS) positives_only(cut);
    load_batch<kVec, kTs>(rr, b0 + kStep, x1);  // the second batch once K* is known (see the row kernel)
    collect_ge<kVec, kTs>(rr, b0, (end - begin + kStep - 1) / kStep, cut.thr, L.u.col.ck, L.u.col.ci, &L.n[0], CAP,
                          x0, x1);
    __syncthreads();

    const int n_loc = L.n[0];
    const int n_put = min(n_loc, CAP);
    // The page-table entries of this CTA's candidates, gathered here and published with them,
    // their loads in flight across the slot reservation below: the CTA that resolves the row
    // then reads them back with the keys instead of gathering ~3000 scattered entries of a
    // 4-B-per-token table itself (that gather, on the step's critical path, cost the 64-request
    // MTP decode step ~7 us).
    constexpr int kPer = CAP / kTs;
    int32_t pvs[kPer];
    {
      const PtRow ptr = pt_row(a, row);
#pragma unroll
      for (int j = 0; j < kPer; ++j) {
        const int i = tid + j * kTs;
        pvs[j] = ptr.at(L.u.col.ci[i] & 0x7FFFFFFF, i < n_put);
      }
    }
    int32_t* ctr = a.ctr + static_cast<int64_t>(row) * a.ctr_stride;
    // words 0..1 of the row's counters as one 64-bit word: low = keys published, high = CTAs done
    unsigned long long* const pub = reinterpret_cast<unsigned long long*>(ctr);
    if (tid == 0) L.n[1] = n_loc ? static_cast<int>(atomicAdd(pub, static_cast<unsigned long long>(n_loc))) : 0;
    __syncthreads();
    uint32_t* lk = a.c_keys + static_cast<int64_t>(row) * CAP;
    int32_t* lt = a.c_tok + static_cast<int64_t>(row) * CAP;
    int32_t* lp = a.c_pv + static_cast<int64_t>(row) * CAP;
    const int base = L.n[1];
#pragma unroll
    for (int jj = 0; jj < kPer; ++jj) {
      const int i = tid + jj * kTs;
      const int j = base + i;
      if (i < n_put && j < CAP) {
        uint32_t k;
        int t;
        collected(L.u.col.ck[i], L.u.col.ci[i], k, t);
        __hip_atomic_store(&lk[j], k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(&lt[j], t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(&lp[j], pvs[jj], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
    // every wave's stores complete before the barrier, so the row's done mark below comes after
    // them (see candidates_complete); the CTA that completes the row reads them back with
    // agent-scope loads
    candidates_complete();
    __syncthreads();
    if (tid == 0) {
      // every CTA adds its count before its done mark, so the last mark returns the final count
      const unsigned long long old = atomicAdd(pub, 1ull << 32);
      const bool last = static_cast<int>(old >> 32) == n_sl - 1;
      L.n[2] = last;
      L.n[3] = last ? static_cast<int>(old & 0xFFFFFFFFull) : 0;
    }
    __syncthreads();
    if (!L.n[2]) return;

    const int n_tot = L.n[3];
    if (CAP == kCapS && cut.thr == kPositive && n_tot < kTopK) {  // block-uniform
      if constexpr (CAP == kCapS) done = sparse_row<kVec>(L.u.res, n_tot, r, pt_row(a, row), dst(), [&](int e) {
        return __hip_atomic_load(&lt[e], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      });
    } else if (n_tot >= kTopK && n_tot <= CAP) {  // block-uniform
      done = resolve_cands<kVec, true>(L.u.res, n_tot, cut, r, pt_row(a, row), dst(),
                                              [&](int e, uint32_t& k, int& t, int32_t& v) {
        k = __hip_atomic_load(&lk[e], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        t = __hip_atomic_load(&lt[e], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        v = __hip_atomic_load(&lp[e], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      });
    } else if (n_tot > CAP) {  // block-uniform: the row's keys >= K* overflowed its list
      // As in the row kernel: a threshold raised from the published keys (CAP of them, a subset of
      // the row's keys >= K*, so their 2048-th digit edge is at most the row's 2048th key), then
      // this CTA collects the whole row once more above it and resolves from LDS.
      SampleCut c2 = cut;
      ResolveLds<kTs, CAP>& R = L.u.res;
      zero_lds<kTs>(R.hist, kBins);
      __syncthreads();
      for (int e = tid; e < CAP; e += kTs)
        atomicAdd(&R.hist[cand_digit(__hip_atomic_load(&lk[e], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT), c2)], 1);
      __syncthreads();
      find_threshold<kBins, kTs>(R.hist, kTopK, R.wtot, R.res);
      c2.thr += static_cast<uint32_t>(R.res[0]) << c2.shift;
      // as in the row kernel: a pass that the stored keys say would overflow again is skipped
      const bool again = static_cast<int64_t>(R.res[1] + R.res[2]) * n_tot <= static_cast<int64_t>(CAP) * CAP;
      if (tid == 0) R.misc[2] = again ? 0 : CAP + 1;
      __syncthreads();
      if (again) collect_ge1<kVec, kTs>(r, tid * 4, (len + kStep - 1) / kStep, c2.thr, R.ck, R.ci, &R.misc[2], CAP);
      __syncthreads();
      const int n2 = R.misc[2];
      if (n2 >= kTopK && n2 <= CAP) {  // block-uniform
        done = resolve_cands<kVec>(R, n2, c2, r, pt_row(a, row), dst(), [&](int e, uint32_t& k, int& t) {
          collected(R.ck[e], R.ci[e], k, t);
        });
      }
    }
  }
  // the estimate missed, or the positives must be counted: the exact path over the row
  if (!done) exact_row<kVec, kTs>(L.u.res, r, pt_row(a, row), dst());  // block-uniform
}

template <bool kVec>
__global__ __launch_bounds__(kTs) void topk_split_kernel(const TopkArgs a) {
  __shared__ SplitLds L;
  constexpr int kStep = kTs * 4 * kUnroll;
  const int tid = threadIdx.x;
  split_assign(a, a.T, L);
  const int row = L.slot[0];
  if (row < 0) return;  // block-uniform
  const int len = row_len(a, row);
  if (len <= kTopK) {
    copy_short_row<kTs>(pt_row(a, row), a.out + static_cast<int64_t>(row) * kTopK, len);
    return;
  }
  int begin, end, n_sl;
  if (!split_slice(len, L.slot[2], L.slot[1], begin, end, n_sl)) return;

  // pass-1 slots (8 bins per thread) and counts first, then the first two batches
  const int4* gh4 = reinterpret_cast<const int4*>(a.ghist + static_cast<int64_t>(row) * kBins);
  const int4 g0 = gh4[2 * tid];
  const int4 g1 = gh4[2 * tid + 1];
  const int pos = a.gcnt[2 * row];
  const int zeros = a.gcnt[2 * row + 1];
  RowSrc rr = row_src(a, row, end);
  const int b0 = begin + tid * 4;
  Batch x0, x1;
  load_batch<kVec, kTs>(rr, b0, x0);
  load_batch<kVec, kTs>(rr, b0 + kStep, x1);

  const bool fast = pos <= kTopK && pos + zeros >= kTopK;
  uint32_t t1 = 0;
  int need1 = kTopK - pos, cnt_t1 = 0;
  if (tid == 0) L.n[1] = 0;
  if (!fast) {
    const int h[8] = {g0.x, g0.y, g0.z, g0.w, g1.x, g1.y, g1.z, g1.w};
    find_threshold_regs<kTs, 8>(h, kTopK, L.wtot, L.res);
    t1 = static_cast<uint32_t>(L.res[0]);
    need1 = kTopK - L.res[1];
    cnt_t1 = L.res[2];
  } else {
    __syncthreads();
  }
  // every CTA of the row takes the same decision: the threshold bin's candidates are collected
  // and published only if the whole bin t1 of the row fits the resolver's LDS
  const bool publish = !fast && cnt_t1 <= kCapS;
  int32_t* ctr = a.ctr + static_cast<int64_t>(row) * a.ctr_stride;
  uint32_t* lk = a.c_keys + static_cast<int64_t>(row) * kCapS;
  int32_t* lt = a.c_tok + static_cast<int64_t>(row) * kCapS;
  if (publish) {  // block-uniform
    collect_bin<kVec, kTs>(rr, b0, (end - begin + kStep - 1) / kStep, t1, L.u.col.ck, L.u.col.ci, &L.n[1], kCapS, x0,
                           x1);
    __syncthreads();
    const int n_c = min(L.n[1], kCapS);
    if (tid == 0) L.n[3] = n_c ? atomicAdd(&ctr[1], n_c) : 0;
    __syncthreads();
    const int base_c = L.n[3];
    for (int i = tid; i < n_c; i += kTs) {
      const int j = base_c + i;
      if (j < kCapS) {
        __hip_atomic_store(&lk[j], L.u.col.ck[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(&lt[j], L.u.col.ci[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
  }
  // Candidates travel between CTAs (and XCDs) through agent-scope stores and loads: every wave's
  // stores complete before the barrier, so the row's done count below comes after all of this
  // CTA's candidates; the CTA that makes the last increment reads them back with agent-scope
  // loads (see candidates_complete).
  candidates_complete();
  __syncthreads();
  if (tid == 0) L.n[4] = atomicAdd(&ctr[2], 1) == n_sl - 1;
  __syncthreads();
  if (!L.n[4]) return;

  // the last CTA of the row: the threshold, then the ordered emission over the whole row
  const RowSrc r = row_src(a, row, len);
  const PtRow pt = pt_row(a, row);
  int32_t* dst = a.out + static_cast<int64_t>(row) * kTopK;
  uint32_t thr = kZeroKey;
  int remaining = need1;
  if (publish) {
    const int n_tot = cnt_t1;  // every CTA published its share of bin t1 (cnt_t1 <= kCapS)
    for (int i = tid; i < n_tot; i += kTs) {
      L.u.res.ck[i] = __hip_atomic_load(&lk[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      L.u.res.ci[i] = __hip_atomic_load(&lt[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    thr = select_lds(L.u.res, n_tot, static_cast<int>(t1), need1, remaining);
  } else if (!fast) {
    thr = select_rescan<kVec>(L.u.res, r, t1, need1, remaining);
  }
  emit_row<kVec, kTs>(r, thr, remaining, pt, dst, L.u.res.scan);
}

// Slices per row of the split path (1: one CTA per row).  At most ~3 split CTAs fit a CU.
int split_count(int64_t rows, int64_t width, int max_splits, int n_cu) {
  if (rows <= 0 || rows > kTs) return 1;  // the balanced split assigns one row per thread
  // one CTA streams a row of up to ~32K tokens faster than a split pays for its publication
  // round trip (measured on 32 x 16K and 64 x U[2K, 64K] decode batches)
  int64_t s = width > 32768 ? (width + 16383) / 16384 : 1;
  s = s < 1 ? 1 : s;
  const int64_t by_cu = (3 * static_cast<int64_t>(n_cu)) / rows;
  s = s < by_cu ? s : by_cu;
  const int64_t cap = max_splits < kMaxSplit ? max_splits : kMaxSplit;
  s = s < cap ? s : cap;
  return static_cast<int>(s < 1 ? 1 : s);
}

// CTAs the balanced split kernel spreads the rows' tokens over (its grid adds one per row):
// rows * S, capped so that the whole grid is resident at once (per_cu CTAs per CU).
int split_target(int64_t rows, int S, int n_cu, int per_cu) {
  const int64_t fit = per_cu * static_cast<int64_t>(n_cu) - rows;
  int64_t t = rows * S;
  t = t < fit ? t : fit;
  return static_cast<int>(t < rows ? rows : t);
}

// CTAs of a kTs-thread kernel resident per CU (the runtime's occupancy calculator).
template <typename Kernel>
int resident_per_cu(Kernel kernel) {
  int n = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kernel, kTs, 0) != hipSuccess || n < 1) n = 1;
  return n;
}

template <int NT, int Q>
void launch_held(const TopkArgs& a, bool vec, hipStream_t stream) {
  const dim3 grid(static_cast<uint32_t>(a.rows));
  if (vec) hipLaunchKernelGGL((topk_held_kernel<true, NT, Q>), grid, dim3(NT), 0, stream, a);
  else hipLaunchKernelGGL((topk_held_kernel<false, NT, Q>), grid, dim3(NT), 0, stream, a);
}

struct WsLayout {
  size_t ctr, c_keys, c_tok, c_pv, total;
};

int cap_for(int64_t width) { return width > kWideRow ? kCapW : kCapS; }

// cap: the candidate list per row (cap_for: kCapS, or kCapW for wide scores)
WsLayout ws_layout(int64_t rows, int cap) {
  WsLayout l;
  size_t off = 0;
  auto take = [&off](size_t bytes) {
    const size_t o = off;
    off += (bytes + 255) / 256 * 256;
    return o;
  };
  l.ctr = take(sizeof(int32_t) * rows * 4);
  l.c_keys = take(sizeof(uint32_t) * rows * cap);
  l.c_tok = take(sizeof(int32_t) * rows * cap);
  l.c_pv = take(sizeof(int32_t) * rows * cap);
  l.total = off;
  return l;
}

// cols: floats of a score row that may be read (>= width); pt_cols: entries per page-table row;
// pt_shift 6: the entries are 64-token pages (PtRow).
int topk_common(const float* score, int64_t score_stride, int64_t width, int64_t cols, const int16_t* mask, int64_t mask_stride,
                const int32_t* lengths, int64_t rows, const int32_t* page_table, int64_t pt_stride, int64_t pt_cols,
                int pt_shift, const int32_t* cu_seqlens_q, int64_t n_req, int max_splits, int n_cu,
                int32_t* pre_hist, bool pass1_done, void* workspace, size_t workspace_bytes, int32_t* out,
                hipStream_t stream, const char* who) {
  DSA_REQUIRE(rows >= 0 && rows <= 0x7FFFFFFF, "%s: rows out of range", who);
  // token offsets (scores, mask words, page-table entries) are formed as 32-bit byte offsets
  DSA_REQUIRE(width >= 0 && width < kMaxWidth, "%s: width %lld out of range (0 .. 2^29 - 1 tokens)", who,
              static_cast<long long>(width));
  if (rows == 0) return ok();
  DSA_REQUIRE(score && lengths && page_table && out, "%s: null pointer", who);
  DSA_REQUIRE(score_stride >= width, "%s: score_stride < width", who);
  DSA_REQUIRE(mask == nullptr || mask_stride >= (width + 15) / 16, "%s: mask_stride < ceil(width / 16)", who);
  DSA_REQUIRE(cu_seqlens_q == nullptr || n_req >= 1, "%s: cu_seqlens_q needs n_req >= 1", who);
  DSA_REQUIRE(max_splits >= 1, "%s: max_splits must be >= 1", who);
  DSA_REQUIRE(pt_cols >= 0 && pt_cols <= 0x7FFFFFFF && (pt_stride >= pt_cols || pt_stride == 0),
              "%s: page-table row stride < its entries per row (and not 0)", who);
  DSA_REQUIRE(pt_shift == 0 || pt_shift == 6, "%s: page-table entries cover 1 or 64 tokens", who);
  // 16-B loads: a row's last quad, the one its length may end in, lies inside the row's cols floats
  const bool vec = cols % 4 == 0 && score_stride % 4 == 0 && (reinterpret_cast<uintptr_t>(score) & 15u) == 0;

  TopkArgs a;
  a.score = score;
  a.score_stride = score_stride;
  a.width = static_cast<int>(width);
  a.mask = mask;
  a.mask_stride = mask_stride;
  a.lengths = lengths;
  a.rows = static_cast<int>(rows);
  a.pt = page_table;
  a.pt_stride = pt_stride;
  const int64_t pt_tokens = pt_cols << pt_shift;  // pt_cols < 2^31 entries, checked above
  a.pt_cols = static_cast<int>(pt_tokens < width ? pt_tokens : width);
  a.pt_shift = pt_shift;
  a.cu = cu_seqlens_q;
  a.n_req = static_cast<int>(n_req);
  a.out = out;
  const int S = split_count(rows, width, max_splits, n_cu);
  a.S = S;
  a.T = 0;
  a.ghist = a.gcnt = a.ctr = a.c_tok = nullptr;
  a.c_keys = nullptr;
  a.c_pv = nullptr;
  a.ctr_stride = 1;
  const dim3 grid_rows(static_cast<uint32_t>(rows));

  if (pre_hist != nullptr) {
    // [ghist1 rows*4096 | ghist2 rows*4096 | cnt rows*2]; words 0..2 of each ghist2 row are the
    // row's split counters (zeroed by the logits call); ghist1 / cnt hold pass 1 if pass1_done.
    a.ghist = pre_hist;
    a.ctr = pre_hist + rows * kBins;
    a.ctr_stride = kBins;
    a.gcnt = pre_hist + 2 * rows * kBins;
  }
  if (S <= 1) {
    if (pre_hist && pass1_done) {
      if (vec) hipLaunchKernelGGL((topk_single_kernel<true>), grid_rows, dim3(kTk), 0, stream, a);
      else hipLaunchKernelGGL((topk_single_kernel<false>), grid_rows, dim3(kTk), 0, stream, a);
    } else {
      const bool wide = cap_for(width) == kCapW;
      if (width <= kHeldRow) {
        // Every row fits a CTA's registers (us a launch, sampled -> held: 4096 x 2049-4096 tokens 90.0 ->
        // 38.0, 64 x 4096 13.7 -> 9.2, 1 x 4096 10.0 -> 6.7, 3904 x 4096-8000 123 -> 63, 32 x 8192 11.5 ->
        // 10.6).  Up to 4096 tokens 512-thread CTAs while a CU has at most one, the shorter chain (1 x
        // 4096: 6.7 against 8.0 with 256 threads; 250 rows 9.7 / 10.8), else 256 threads (1000 rows
        // 16.7 -> 14.7, 4096 rows 48.3 -> 38.0).
        if (width > 4096) launch_held<512, 4>(a, vec, stream);
        else if (rows <= n_cu) launch_held<512, 2>(a, vec, stream);
        else launch_held<256, 4>(a, vec, stream);
      } else if (vec && wide) hipLaunchKernelGGL((topk_row_sampled_kernel<true, kCapW>), grid_rows, dim3(kTs), 0, stream, a);
      else if (vec) hipLaunchKernelGGL((topk_row_sampled_kernel<true, kCapS>), grid_rows, dim3(kTs), 0, stream, a);
      else if (wide) hipLaunchKernelGGL((topk_row_sampled_kernel<false, kCapW>), grid_rows, dim3(kTs), 0, stream, a);
      else hipLaunchKernelGGL((topk_row_sampled_kernel<false, kCapS>), grid_rows, dim3(kTs), 0, stream, a);
    }
    return check_launch(who);
  }
  const int cap = cap_for(width);
  const WsLayout l = ws_layout(rows, cap);
  DSA_REQUIRE(workspace != nullptr && workspace_bytes >= l.total,
              "%s: workspace of %zu bytes is smaller than the %zu required", who, workspace_bytes, l.total);
  DSA_REQUIRE((reinterpret_cast<uintptr_t>(workspace) & 15u) == 0, "%s: workspace must be 16-B aligned", who);
  char* ws = static_cast<char*>(workspace);
  if (!pre_hist) {
    a.ctr = reinterpret_cast<int32_t*>(ws + l.ctr);
    a.ctr_stride = 4;
    hipLaunchKernelGGL(topk_zero_kernel, dim3(static_cast<uint32_t>((4 * rows + 255) / 256)), dim3(256), 0, stream,
                       a.ctr, static_cast<int>(rows));
  }
  a.c_keys = reinterpret_cast<uint32_t*>(ws + l.c_keys);
  a.c_tok = reinterpret_cast<int32_t*>(ws + l.c_tok);
  a.c_pv = reinterpret_cast<int32_t*>(ws + l.c_pv);
  if (pre_hist && pass1_done) {  // the exact threshold bin from the logits kernel's pass 1
    static const int per_cu_v = resident_per_cu(topk_split_kernel<true>);
    static const int per_cu_s = resident_per_cu(topk_split_kernel<false>);
    a.T = split_target(rows, S, n_cu, vec ? per_cu_v : per_cu_s);
    const dim3 grid(static_cast<uint32_t>(a.T + rows));
    if (vec) hipLaunchKernelGGL((topk_split_kernel<true>), grid, dim3(kTs), 0, stream, a);
    else hipLaunchKernelGGL((topk_split_kernel<false>), grid, dim3(kTs), 0, stream, a);
  } else {
    // CTAs per CU the occupancy calculator allows, per instantiation (the wide list's LDS is larger)
    static const int per_cu[4] = {resident_per_cu(topk_split_sampled_kernel<false, kCapS>),
                                  resident_per_cu(topk_split_sampled_kernel<true, kCapS>),
                                  resident_per_cu(topk_split_sampled_kernel<false, kCapW>),
                                  resident_per_cu(topk_split_sampled_kernel<true, kCapW>)};
    const int pc = per_cu[(cap == kCapW ? 2 : 0) + (vec ? 1 : 0)];
    const int64_t fit = pc * static_cast<int64_t>(n_cu) / rows;
    a.S = static_cast<int>(S < fit ? S : (fit > 1 ? fit : 1));
    const dim3 grid(static_cast<uint32_t>(rows * a.S));
    if (cap == kCapW) {
      if (vec) hipLaunchKernelGGL((topk_split_sampled_kernel<true, kCapW>), grid, dim3(kTs), 0, stream, a);
      else hipLaunchKernelGGL((topk_split_sampled_kernel<false, kCapW>), grid, dim3(kTs), 0, stream, a);
    } else {
      if (vec) hipLaunchKernelGGL((topk_split_sampled_kernel<true, kCapS>), grid, dim3(kTs), 0, stream, a);
      else hipLaunchKernelGGL((topk_split_sampled_kernel<false, kCapS>), grid, dim3(kTs), 0, stream, a);
    }
  }
  return check_launch(who);
}

}  // namespace

int topk_padded(const float* score, int64_t score_stride, int64_t width, int64_t cols, const int32_t* lengths,
                int64_t rows, const int32_t* page_table, int64_t pt_stride, int64_t pt_cols, int pt_shift,
                int max_splits, int n_cu, void* workspace, size_t workspace_bytes, int32_t* out, hipStream_t stream,
                const char* who) {
  return topk_common(score, score_stride, width, cols, nullptr, 0, lengths, rows, page_table, pt_stride, pt_cols,
                     pt_shift, nullptr, rows, max_splits, n_cu, nullptr, false, workspace, workspace_bytes, out, stream, who);
}

}  // namespace dsa

using namespace dsa;

extern "C" int dsa_topk_split_count(int64_t rows, int64_t width, int max_splits, int n_cu) {
  return split_count(rows, width, max_splits < 1 ? 1 : max_splits, n_cu);
}

extern "C" size_t dsa_topk_workspace_bytes(int64_t rows, int64_t width, int max_splits, int n_cu) {
  const int S = split_count(rows, width, max_splits < 1 ? 1 : max_splits, n_cu);
  if (S <= 1 || rows <= 0) return 0;
  return ws_layout(rows, cap_for(width)).total;
}

extern "C" int dsa_topk_transform(const float* score, int64_t score_stride, int64_t width, const int16_t* mask,
                                  int64_t mask_stride, const int32_t* lengths, int64_t rows,
                                  const int32_t* page_table, int64_t pt_stride, int64_t pt_cols,
                                  const int32_t* cu_seqlens_q, int64_t n_req, int max_splits, int n_cu,
                                  void* workspace, size_t workspace_bytes, int32_t* out, hipStream_t stream) {
  return topk_common(score, score_stride, width, width, mask, mask_stride, lengths, rows, page_table, pt_stride, pt_cols, 0,
                     cu_seqlens_q, n_req, max_splits, n_cu, nullptr, false, workspace, workspace_bytes, out, stream,
                     "dsa_topk_transform");
}

extern "C" int dsa_topk_transform_pre(const float* score, int64_t score_stride, int64_t width, const int16_t* mask,
                                      int64_t mask_stride, const int32_t* lengths, int64_t rows,
                                      const int32_t* page_table, int64_t pt_stride, int64_t pt_cols,
                                      const int32_t* cu_seqlens_q, int64_t n_req, int max_splits, int n_cu,
                                      int32_t* hist_ws, int pass1_done, void* workspace, size_t workspace_bytes,
                                      int32_t* out, hipStream_t stream) {
  DSA_REQUIRE(hist_ws != nullptr, "dsa_topk_transform_pre: hist_ws is null");
  return topk_common(score, score_stride, width, width, mask, mask_stride, lengths, rows, page_table, pt_stride, pt_cols, 0,
                     cu_seqlens_q, n_req, max_splits, n_cu, hist_ws, pass1_done != 0, workspace, workspace_bytes, out,
                     stream, "dsa_topk_transform_pre");
}

extern "C" int dsa_topk_transform_blocks(const float* score, int64_t score_stride, int64_t width, const int16_t* mask,
                                         int64_t mask_stride, const int32_t* lengths, int64_t rows,
                                         const int32_t* block_table, int64_t bt_stride, int64_t bt_pages,
                                         const int32_t* cu_seqlens_q, int64_t n_req, int max_splits, int n_cu,
                                         int32_t* hist_ws, int pass1_done, void* workspace, size_t workspace_bytes,
                                         int32_t* out, hipStream_t stream) {
  return topk_common(score, score_stride, width, width, mask, mask_stride, lengths, rows, block_table, bt_stride, bt_pages,
                     6, cu_seqlens_q, n_req, max_splits, n_cu, hist_ws, hist_ws != nullptr && pass1_done != 0,
                     workspace, workspace_bytes, out, stream, "dsa_topk_transform_blocks");
}

// ---------------------------------------------------------------------------------------------
// Allocation-free variant of dsa_topk_transform: the split path's workspace is a file-scope
// device array instead of a caller buffer.  Each device holds its own copy of the array until
// the process ends; its device address is looked up once per device (hipGetSymbolAddress, with
// that device current) and kept.  The host-side name `scratch` is only a stand-in for the
// symbol: host code passes the looked-up address, never the array itself.  Every call on one
// device shares that device's array (the split counters in it are cleared by a fill kernel at
// the start of each call), so calls that overlap on one device race.
namespace dsa {
namespace {

// the split workspace (ws_layout) of up to 256 rows: counters, then candidate keys, tokens and
// page-table entries
constexpr size_t kScratchRows = 256;
constexpr size_t kScratchBytes = (kScratchRows * 16 + 255) / 256 * 256 + 3 * kScratchRows * kCapS * 4;
static __device__ __align__(256) uint8_t scratch[kScratchBytes];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices] = {};

int scratch_address(void** ptr, const char* who) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return fail(DSA_ERR_LAUNCH, "%s: hipGetDevice: %s", who, hipGetErrorString(e));
  if (dev < 0 || dev >= kMaxDevices) return fail(DSA_ERR_INVALID, "%s: device ordinal %d out of range", who, dev);
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (g_scratch_ptr[dev] == nullptr) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || p == nullptr)
      return fail(DSA_ERR_LAUNCH, "%s: hipGetSymbolAddress(scratch): %s", who, hipGetErrorString(e));
    g_scratch_ptr[dev] = p;
  }
  *ptr = g_scratch_ptr[dev];
  return DSA_OK;
}

}  // namespace
}  // namespace dsa

extern "C" size_t dsa_topk_noalloc_max_bytes(void) { return kScratchBytes; }

extern "C" int dsa_topk_transform_noalloc(const float* score, int64_t score_stride, int64_t width,
                                          const int16_t* mask, int64_t mask_stride, const int32_t* lengths,
                                          int64_t rows, const int32_t* page_table, int64_t pt_stride, int64_t pt_cols,
                                          const int32_t* cu_seqlens_q, int64_t n_req, int max_splits, int n_cu,
                                          int32_t* out, hipStream_t stream) {
  const char* who = "dsa_topk_transform_noalloc";
  DSA_REQUIRE(rows >= 0 && rows <= 0x7FFFFFFF && width >= 0 && width < kMaxWidth, "%s: rows / width out of range",
              who);
  const size_t need = dsa_topk_workspace_bytes(rows, width, max_splits, n_cu);
  if (need > kScratchBytes)
    return fail(DSA_ERR_WORKSPACE, "%s: %lld rows of width %lld need a %zu-byte split workspace, above the %zu bytes "
                "of the built-in one (use dsa_topk_transform with a caller workspace, or max_splits = 1)",
                who, static_cast<long long>(rows), static_cast<long long>(width), need, kScratchBytes);
  void* ws = nullptr;
  if (need > 0) {
    const int st = scratch_address(&ws, who);
    if (st != DSA_OK) return st;
  }
  return topk_common(score, score_stride, width, width, mask, mask_stride, lengths, rows, page_table, pt_stride, pt_cols, 0,
                     cu_seqlens_q, n_req, max_splits, n_cu, nullptr, false, ws, need, out, stream, who);
}
