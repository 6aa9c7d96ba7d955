// Running top-k over the label chunks of the inference logits (evaluate.py:158-159,235-236 take topk(100) / topk(5) of
// the dense [B, L] logits that xfc_forward returns, chunked_fp8xmc_clf.py:45-60).  The logits of one chunk at a time are
// written to a chunk-sized buffer and reduced to the k best per batch row, so the [B, L] matrix (172 MB at B = 128,
// L = 670 K) is never allocated.
//
// One workgroup per batch row and list (a row has two lists: a large group of chunks is split between two workgroups,
// and topk_finish_kernel merges the lists at the end).  Candidates = the k entries kept so far (from the chunks before, hence smaller label
// ids) followed by the chunk's logits in label order.  Radix select on a 16-bit key that orders bf16 values (two passes
// of 256 bins find the key T of the k-th largest), then everything above T is taken, entries equal to T are taken in
// candidate order until k are full (ties go to the smaller label id: a second radix select, on the label, among the
// chunk's entries equal to T), and the k entries are sorted by (value descending, label ascending).  NaN orders above every number, as in torch.topk.
// Once k entries are kept, their smallest value is a lower bound of the final k-th value: one pass over the chunk
// keeps only the logits at or above it, in LDS, and the selection passes run over that short list (the chunk is read
// again by every pass only when more than TOPK_CAP logits reach the bound).  The first chunk is therefore fed in two
// parts, a short prefix that fits the list and produces a bound, and the rest.
#include "xmc_common.h"

namespace xmc {

constexpr int TOPK_MAX = 128;   // largest k
constexpr int TOPK_NT = 1024;  // sixteen wavefronts keep enough loads in flight on the workgroup's compute unit
template <int N> struct TopkBins { static constexpr int value = N; };
typedef TopkBins<256> B256;
typedef TopkBins<1024> B1024;
constexpr int TOPK_CAP = 6144;  // chunk logits at or above the bound that one workgroup keeps in LDS
constexpr int TOPK_SMALL = 512; // candidates (kept entries included) that are ranked directly

// z: a row's logits of the chunk at z + row*stride, n_all of them valid (n_all <= 2^17; stride % 4 == 0; z 8-byte aligned)
// run_val/run_idx: [batch][2][TOPK_MAX] entries kept so far: every batch row has two lists, which topk_finish_kernel
// merges.  parts = 1: one workgroup per row adds all n_all logits to list 0 (have0 entries valid).  parts = 2: two
// workgroups per row, so that 128 rows fill 256 compute units; workgroup 2 row + p takes the first topk_split(n_all)
// logits (p = 0) or the rest (p = 1) and updates list p (have0 / have1 entries valid).  Lists are updated in place and
// stay sorted; within a list the entries kept from earlier launches have the smaller label ids.
__host__ __device__ __forceinline__ int topk_split(int n_all) { return ((n_all >> 1) + 3) & ~3; }
__global__ __launch_bounds__(TOPK_NT) void topk_chunk_kernel(const unsigned short* z, long long stride, int n_all, int label_base0, int k,
                                                             int parts, int have0, int have1, unsigned short* run_val, int* run_idx) {
  __shared__ unsigned hist[1024];
  __shared__ __attribute__((aligned(16))) unsigned sel_key[TOPK_MAX];
  __shared__ __attribute__((aligned(16))) int sel_idx[TOPK_MAX];
  __shared__ __attribute__((aligned(16))) unsigned cand_key[TOPK_CAP];
  __shared__ __attribute__((aligned(16))) int cand_idx[TOPK_CAP];   // index in the chunk (negative: an entry kept from earlier chunks)
  __shared__ unsigned s_bin, s_above, s_count, s_ncand, wtot[TOPK_NT / 64];
  const int tid = threadIdx.x;
  const int brow = parts == 2 ? (int)(blockIdx.x >> 1) : (int)blockIdx.x, part = parts == 2 ? (int)(blockIdx.x & 1) : 0;
  const int first = part == 0 ? 0 : topk_split(n_all);                      // this workgroup's range of the chunk
  const int n = parts == 2 ? (part == 0 ? topk_split(n_all) : n_all - first) : n_all;
  const int label_base = label_base0 + first;
  const int have = part == 0 ? have0 : have1;
  const unsigned short* row = z + (size_t)brow * stride + first;
  unsigned short* rv = run_val + ((size_t)brow * 2 + part) * TOPK_MAX;
  int* ri = run_idx + ((size_t)brow * 2 + part) * TOPK_MAX;
  const int total = n + have;
  const int kk = k < total ? k : total;
  const unsigned mykey = tid < have ? topk_key(rv[tid]) : 0u;   // this thread's entry of the running list
  const int myidx = tid < have ? ri[tid] : -1;
  const unsigned floor_key = have >= k ? topk_key(rv[k - 1]) : 0u;   // the list is sorted: entry k-1 is its smallest

  // visits every chunk element once, the workgroup reading 8 KiB of consecutive logits at a time, sixteen such loads in
  // flight (a compute unit runs one workgroup: nothing else hides the latency): f(key, index in chunk)
  auto for_each_global = [&](auto f) {
    constexpr int U = 16;
    for (int base = 0; base < n; base += U * 4 * TOPK_NT) {
      uint2 v[U];
#pragma unroll
      for (int u = 0; u < U; u++) {
        const int i = base + u * 4 * TOPK_NT + 4 * tid;
        v[u] = i + 4 <= n ? *(const uint2*)(row + i) : uint2{0u, 0u};
      }
#pragma unroll
      for (int u = 0; u < U; u++) {
        const int i = base + u * 4 * TOPK_NT + 4 * tid;
        if (i + 4 <= n) {
          f(topk_key((unsigned short)(v[u].x & 0xFFFFu)), i);
          f(topk_key((unsigned short)(v[u].x >> 16)), i + 1);
          f(topk_key((unsigned short)(v[u].y & 0xFFFFu)), i + 2);
          f(topk_key((unsigned short)(v[u].y >> 16)), i + 3);
        } else {
          for (int j = i; j < n; j++) f(topk_key(row[j]), j);
        }
      }
    }
  };
  // one pass over the chunk keeps the logits at or above the bound (key, index) in LDS; the selection then runs over
  // that list.  More than TOPK_CAP of them: every later pass reads the chunk again.
  if (tid == 0) s_ncand = 0;
  __syncthreads();
  for_each_global([&](unsigned key, int i) {
    const bool take = key >= floor_key;
    const unsigned long long m = __ballot(take);   // lanes of this wavefront that are here and take
    if (m != 0) {
      const int lane = tid & 63, leader = __ffsll((long long)m) - 1;
      unsigned base = 0;
      if (lane == leader) base = atomicAdd(&s_ncand, (unsigned)__popcll(m));
      base = __shfl(base, leader, 64);
      const unsigned slot = base + (unsigned)__popcll(m & ((1ull << lane) - 1ull));
      if (take && slot < (unsigned)TOPK_CAP) {
        cand_key[slot] = key;
        cand_idx[slot] = i;
      }
    }
  });
  __syncthreads();
  const bool listed = s_ncand <= (unsigned)TOPK_CAP;
  const int ncand = listed ? (int)s_ncand : 0;
  // rank of (key, idx) among m entries of (keys, idxs) in the order value descending, index ascending; m % 4 == 0
  auto rank_among = [&](const unsigned* keys, const int* idxs, int m, unsigned key, int idx) {
    int rank = 0;
    for (int j = 0; j < m; j += 4) {
      const uint4 kj = *(const uint4*)(keys + j);
      const int4 ij = *(const int4*)(idxs + j);
      rank += (kj.x > key || (kj.x == key && ij.x < idx)) ? 1 : 0;
      rank += (kj.y > key || (kj.y == key && ij.y < idx)) ? 1 : 0;
      rank += (kj.z > key || (kj.z == key && ij.z < idx)) ? 1 : 0;
      rank += (kj.w > key || (kj.w == key && ij.w < idx)) ? 1 : 0;
    }
    return rank;
  };
  if (listed && ncand + have <= TOPK_SMALL) {
    // few candidates (the usual case once a bound exists): the kept entries join the list, every entry finds its rank
    // among all of them and the first kk are written in place.  Kept entries have the smaller label ids.
    const int m = ncand + have, m4 = (m + 3) & ~3;
    if (tid < have) {
      cand_key[ncand + tid] = mykey;
      cand_idx[ncand + tid] = myidx - label_base;
    }
    if (tid < m4 - m) {   // padding that ranks after everything
      cand_key[m + tid] = 0u;
      cand_idx[m + tid] = 0x7FFFFFFF;
    }
    __syncthreads();
    for (int c = tid; c < m; c += TOPK_NT) {
      const unsigned key = cand_key[c];
      const int idx = cand_idx[c];
      const int rank = rank_among(cand_key, cand_idx, m4, key, idx);
      if (rank < kk) {
        rv[rank] = topk_bits(key);
        ri[rank] = label_base + idx;
      }
    }
    if (tid >= kk && tid < TOPK_MAX) {
      rv[tid] = 0xFF80;   // -inf
      ri[tid] = -1;
    }
    return;
  }
  auto for_each = [&](auto f) {
    if (listed) {
      for (int j = tid; j < ncand; j += TOPK_NT) f(cand_key[j], cand_idx[j]);
    } else {
      for_each_global([&](unsigned key, int i) { if (key >= floor_key) f(key, i); });
    }
  };
  auto clear_hist = [&]() {
    __syncthreads();
    for (int q = tid; q < 1024; q += TOPK_NT) hist[q] = 0;
    __syncthreads();
  };
  // exclusive prefix sum of one value per thread over the workgroup (thread order), and the total
  auto block_scan = [&](unsigned val, unsigned& total) {
    const int lane = tid & 63, wave = tid >> 6;
    unsigned x = val;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const unsigned y = __shfl_up(x, off, 64);
      if (lane >= off) x += y;
    }
    __syncthreads();
    if (lane == 63) wtot[wave] = x;
    __syncthreads();
    unsigned before = 0;
    total = 0;
#pragma unroll
    for (int q = 0; q < TOPK_NT / 64; q++) {
      if (q < wave) before += wtot[q];
      total += wtot[q];
    }
    return before + x - val;
  };
  // the bin in which the `want`-th candidate lies, counting from the top (down) or from the bottom: s_bin; s_above =
  // candidates in the bins before it.  Thread t looks at one bin (or bins / threads consecutive bins) in counting order.
  auto pick_bin = [&](unsigned want, auto bins_c, bool from_top) {
    __syncthreads();
    constexpr int bins = decltype(bins_c)::value;
    constexpr int per = bins > TOPK_NT ? bins / TOPK_NT : 1;
    unsigned local[per], sum = 0;
#pragma unroll
    for (int q = 0; q < per; q++) {
      const int pos = tid * per + q;
      local[q] = pos < bins ? hist[from_top ? bins - 1 - pos : pos] : 0u;
      sum += local[q];
    }
    unsigned total;
    unsigned before = block_scan(sum, total);
    if (tid == 0 && (want == 0 || total < want)) {   // nothing asked for, or fewer candidates than asked: the last bin in order
      s_bin = (unsigned)(want == 0 ? (from_top ? bins - 1 : 0) : (from_top ? 0 : bins - 1));
      s_above = want == 0 ? 0u : total - hist[from_top ? 0 : bins - 1];
    }
    if (want > 0 && total >= want) {
#pragma unroll
      for (int q = 0; q < per; q++) {
        if (before < want && want <= before + local[q]) {
          const int pos = tid * per + q;
          s_bin = (unsigned)(from_top ? bins - 1 - pos : pos);
          s_above = before;
        }
        before += local[q];
      }
    }
    __syncthreads();
  };

  clear_hist();
  for_each([&](unsigned key, int) { atomicAdd(&hist[key >> 8], 1u); });
  if (tid < have) atomicAdd(&hist[mykey >> 8], 1u);
  pick_bin((unsigned)kk, B256{}, true);
  const unsigned hi_bin = s_bin, above_hi = s_above;
  clear_hist();
  for_each([&](unsigned key, int) { if ((key >> 8) == hi_bin) atomicAdd(&hist[key & 255u], 1u); });
  if (tid < have && (mykey >> 8) == hi_bin) atomicAdd(&hist[mykey & 255u], 1u);
  pick_bin((unsigned)kk - above_hi, B256{}, true);
  const unsigned T = (hi_bin << 8) | s_bin;
  const unsigned n_gt = above_hi + s_above;          // candidates above T: all taken
  const unsigned need_eq = (unsigned)kk - n_gt;      // candidates equal to T still to take, in candidate order

  // equal candidates of the running list come first
  __syncthreads();
  if (tid == 0) s_count = 0;
  unsigned eq_run;
  const unsigned my_eq_rank = block_scan((tid < have && mykey == T) ? 1u : 0u, eq_run);   // the list is in candidate order
  const unsigned eq_from_run = eq_run < need_eq ? eq_run : need_eq;
  if (tid < have) {
    if (mykey > T || (mykey == T && my_eq_rank < need_eq)) {
      const unsigned slot = atomicAdd(&s_count, 1u);
      sel_key[slot] = mykey;
      sel_idx[slot] = myidx;
    }
  }
  // the chunk's candidates equal to T are taken up to the index limit that admits eq_chunk of them: a second radix
  // select, on the index (high bits i >> 10, then the low 10 bits), over those candidates only
  const unsigned eq_chunk = need_eq - eq_from_run;
  int idx_limit = -1;   // equal candidates with index <= idx_limit are taken
  if (eq_chunk > 0) {
    clear_hist();
    for_each([&](unsigned key, int i) { if (key == T) atomicAdd(&hist[i >> 10], 1u); });
    pick_bin(eq_chunk, B256{}, false);
    const unsigned hi_idx = s_bin, below_hi = s_above;
    clear_hist();
    for_each([&](unsigned key, int i) { if (key == T && (unsigned)(i >> 10) == hi_idx) atomicAdd(&hist[i & 1023], 1u); });
    pick_bin(eq_chunk - below_hi, B1024{}, false);
    idx_limit = (int)((hi_idx << 10) | s_bin);
  }
  __syncthreads();
  for_each([&](unsigned key, int i) {
    if (key > T || (key == T && i <= idx_limit)) {
      const unsigned slot = atomicAdd(&s_count, 1u);
      if (slot < (unsigned)TOPK_MAX) {
        sel_key[slot] = key;
        sel_idx[slot] = label_base + i;
      }
    }
  });
  __syncthreads();
  if (tid >= kk && tid < TOPK_MAX) {   // padding that ranks after everything
    sel_key[tid] = 0u;
    sel_idx[tid] = 0x7FFFFFFF;
  }
  __syncthreads();
  // exactly kk entries: sort by (value descending, label ascending) through ranks
  if (tid < kk) {
    const unsigned key = sel_key[tid];
    const int idx = sel_idx[tid];
    const int rank = rank_among(sel_key, sel_idx, (kk + 3) & ~3, key, idx);
    rv[rank] = topk_bits(key);
    ri[rank] = idx;
  }
  if (tid >= kk && tid < TOPK_MAX) {
    rv[tid] = 0xFF80;   // -inf
    ri[tid] = -1;
  }
}

// merges the two sorted lists of every batch row (have0 and have1 entries valid, have0 + have1 >= k, all label ids
// distinct) and writes the first k entries to the outputs [batch][k]: an entry's position is its index in its own list
// plus the number of entries of the other list that come before it (value descending, label ascending).
// One workgroup of 2 * TOPK_MAX threads per row.
__global__ __launch_bounds__(2 * TOPK_MAX) void topk_finish_kernel(const unsigned short* run_val, const int* run_idx, int k, int have0,
                                                                  int have1, unsigned short* out_val, int* out_idx) {
  __shared__ __attribute__((aligned(16))) unsigned fkey[2][TOPK_MAX];
  __shared__ __attribute__((aligned(16))) int fidx[2][TOPK_MAX];
  const int b = blockIdx.x, list = threadIdx.x / TOPK_MAX, j = threadIdx.x - list * TOPK_MAX;
  const int mine = list == 0 ? have0 : have1;
  const bool valid = j < mine;
  const unsigned short bits = valid ? run_val[((size_t)b * 2 + list) * TOPK_MAX + j] : (unsigned short)0;
  const int idx = valid ? run_idx[((size_t)b * 2 + list) * TOPK_MAX + j] : 0x7FFFFFFF;
  const unsigned key = valid ? topk_key(bits) : 0u;   // an entry that is not there comes before nothing
  fkey[list][j] = key;
  fidx[list][j] = idx;
  __syncthreads();
  if (!valid) return;
  int pos = j;
#pragma unroll 8
  for (int o = 0; o < TOPK_MAX; o += 4) {
    const uint4 ko = *(const uint4*)&fkey[list ^ 1][o];
    const int4 io = *(const int4*)&fidx[list ^ 1][o];
    pos += (ko.x > key || (ko.x == key && io.x < idx)) ? 1 : 0;
    pos += (ko.y > key || (ko.y == key && io.y < idx)) ? 1 : 0;
    pos += (ko.z > key || (ko.z == key && io.z < idx)) ? 1 : 0;
    pos += (ko.w > key || (ko.w == key && io.w < idx)) ? 1 : 0;
  }
  if (pos < k) {
    out_val[(size_t)b * k + pos] = bits;
    out_idx[(size_t)b * k + pos] = idx;
  }
}


// ---- the two small kernels of the two-pass top-k (fp8_forward_select_kernel produces gmax and the candidate lists)

// The k-th largest of the 16-bit keys that the threads of a workgroup hold (U per thread, of which the first `used`, the same for all
// threads, are looked at; 0 = no key), or 0 if there are fewer than k: the largest T with at least k keys >= T, found from the top, two
// bits a round (a round is a barrier and an LDS read's latency; one bit a round, the pick and the bound kernels took 8.4 and 4.9 us).
// Every thread of the workgroup calls this; wcnt = 2 x WAVES double words of LDS.
template <int WAVES, int U>
__device__ __forceinline__ unsigned block_kth_key(const unsigned (&key)[U], int used, int k, unsigned long long* wcnt) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  static_assert(WAVES * 64 * U < 65536, "sixteen bits a count");
  unsigned T = 0u;
#pragma unroll 1
  for (int bit = 14; bit >= 0; bit -= 2) {
    unsigned long long n = 0;   // keys at or above T + 1, 2, 3 steps, 16 bits each
#pragma unroll
    for (int u = 0; u < U; u++)
      if (u < used) {
#pragma unroll
        for (int c = 1; c < 4; c++) n += (unsigned long long)__popcll(__ballot(key[u] >= (T | ((unsigned)c << bit)))) << (16 * (c - 1));
      }
    unsigned long long* mine = wcnt + ((bit & 2) ? WAVES : 0);   // alternating halves: a slow reader is never overtaken by a writer
    if (lane == 0) mine[wave] = n;
    __syncthreads();
    unsigned long long total = 0;
#pragma unroll
    for (int q = 0; q < WAVES; q++) total += mine[q];
    unsigned c = 0u;
#pragma unroll
    for (int q = 0; q < 3; q++) c += (unsigned)(total >> (16 * q)) % 65536u >= (unsigned)k ? 1u : 0u;   // (the counts fall with the step)
    T |= c << bit;
  }
  return T;
}

// bound[b] = k-th largest of the `groups` maxima gmax[g][b] of batch row b (groups >= k); rows at or past `batch` get
// a bound nothing reaches.  Also clears the candidate counts and the status word.  One workgroup of TOPK_GROUPS threads
// per row of the padded batch.
constexpr int TOPK_GROUPS = 512;
__global__ __launch_bounds__(TOPK_GROUPS) void topk_bound_kernel(const unsigned short* gmax, int groups, int k, int batch,
                                                                 unsigned short* bound, unsigned* count, int* status) {
  __shared__ unsigned long long wcnt[2 * (TOPK_GROUPS / 64)];
  const int b = blockIdx.x, g = threadIdx.x;
  if (g == 0) {
    count[b * SEL_COUNT_STRIDE] = 0u;
    count[b * SEL_COUNT_STRIDE + 1] = 0u;                                   // (entries of the row's lists in topk_repair)
    if (b < SEL_ROWS / 32) count[(SEL_ROWS + b) * SEL_COUNT_STRIDE] = 0u;   // (workgroups of topk_repair that are done)
    if (b == 0) *status = 0;
    if (b >= batch) bound[b] = 0xFFFFu;
  }
  if (b >= batch) return;
  const unsigned key[1] = {g < groups ? (unsigned)gmax[(size_t)g * SEL_ROWS + b] : 0u};
  const unsigned T = block_kth_key<TOPK_GROUPS / 64>(key, 1, k, wcnt);
  if (g == 0) bound[b] = (unsigned short)T;
}

// ---- Rows whose list is of no use - more logits at or above the bound than it holds (massive ties, say), or fewer than k - are done
// over by topk_repair, in the launch that ranks the other rows' lists: up to 256 workgroups, which look at the rows' counts and are
// usually done with that.  (Before, the host waited for a status word after every call, to launch the general path if need be: 27 - 32 us
// of a call of 158 in which the GPU had nothing to do.)  The workgroups share the groups of 32 batch rows that have such a row, and
// those of a group the labels.  A workgroup computes its logits anew, 256 labels a round, and keeps the best k of every row in LDS; the
// last one of a group merges their lists.  Nobody waits for anybody.
// Bound by memory: every group reads all weights, each wavefront its sixteen labels of the next round into the registers that this
// round's products have just read.  The row's bound, which k logits at least reach, keeps nearly everything else off the lists.
// us a call, k = 100, 6,000 equal labels the best of one row / of all rows: with the host's wait and the general path / with 64
// workgroups for every group, which loaded nothing ahead and ranked lists against one another / now:
//   128 rows  131 K labels 349/285/179  339/547/328   670 K 667/772/328  627/1121/579   2 M 1370/1944/737  1340/2399/1255
//   256 rows  131 K 692/360/256  668/961/421          670 K 810/864/412  1239/2103/904   2 M 1753/2178/933  2664/4503/2087
// With no such row 131 K 74/48/48, 670 K 160/131/122; with every logit of one row alike, where pass 2 takes nearly all, 670 K 8744/8214/7840.
constexpr int REP_NT = 1024;              // threads: as many as topk_pick's, which shares the launch
constexpr int REP_BLOCKS = 64;            // workgroups for every 32 rows of a batch of up to 128, all of a larger one's: 256
constexpr int REP_SLICES = 128;           // most workgroups of a group: the last one reads as many lists
constexpr int REP_CAP = 256;              // entries of a row's list in LDS; cut to the best k <= TOPK_MAX before it overflows
constexpr int REP_STEP = 256;             // labels a round, sixteen a wavefront
constexpr int REP_KS = REP_STEP + 8;      // stride of a row of keys
constexpr int REP_X = 32 * REP_CAP * 8;                // LDS: lists | operand image of the group's X | keys of two rounds | a word
constexpr int REP_KEYS = REP_X + 12 * 2048;
constexpr int REP_WORD = REP_KEYS + 2 * 32 * REP_KS * 2;
constexpr int REP_LDS = REP_WORD + 64;
constexpr int rep_blocks(int batch) { return (batch < BP ? (batch + 31) / 32 : BP / 32) * REP_BLOCKS; }
constexpr size_t REP_BYTES = (size_t)rep_blocks(SEL_ROWS) * 32 * TOPK_MAX * 8;   // lists of the workgroups
static_assert(REP_CAP >= TOPK_MAX + 64, "a wavefront's worth of new entries behind a cut list");
static_assert(REP_STEP == REP_NT / 64 * 16 && REP_BLOCKS % 8 == 0 && SEL_ROWS == 256, "shares of the wavefronts and the workgroups");

// An entry: order key << 32 | ~label, larger = better value, then smaller label; 0 = none.
struct RepList { unsigned long long* ent; int n; unsigned long long above; };   // entries above `above` are still wanted
// Cuts the list of a wavefront's row to its best k, in no order: the k-th entry bit by bit, as all entries are different (ranked against
// one another instead, 128 rows of 6,000 equal labels: 131 K labels 402 us a call, now 328, 670 K 711, now 579).  label_bits: bits that
// labels differ in.
__device__ __forceinline__ void rep_cut(RepList& l, int k, int label_bits) {
  if (l.n <= k) return;
  const int lane = threadIdx.x & 63;
  unsigned long long e[REP_CAP / 64];
#pragma unroll
  for (int u = 0; u < REP_CAP / 64; u++) e[u] = lane + 64 * u < l.n ? l.ent[lane + 64 * u] : 0ull;
  auto at_least = [&](unsigned long long t) {
    int c = 0;
#pragma unroll
    for (int u = 0; u < REP_CAP / 64; u++) c += __popcll(__ballot(e[u] >= t));
    return c;
  };
  unsigned long long T = 0ull;   // at least k entries at or above it
  int have = l.n;
  for (int bit = 47; bit >= 0 && have > k; bit--) {
    if (bit == 31) {   // (the upper bits of an inverted label are ones)
      T |= 0xFFFFFFFFull >> label_bits << label_bits;
      bit = label_bits - 1;
    }
    const int c = at_least(T | 1ull << bit);
    if (c >= k) { T |= 1ull << bit; have = c; }
  }
  int n = 0;
#pragma unroll
  for (int u = 0; u < REP_CAP / 64; u++) {
    const unsigned long long who = __ballot(e[u] >= T);
    if (e[u] >= T) l.ent[n + (int)__builtin_amdgcn_mbcnt_hi((unsigned)(who >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)who, 0u))] = e[u];
    n += __popcll(who);
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  l.n = n;
  l.above = T - 1ull;
}
// a wavefront's worth of entries, one per lane
__device__ __forceinline__ void rep_add(RepList& l, unsigned long long e, int k, int label_bits) {
  unsigned long long who = __ballot(e > l.above);
  if (who == 0) return;
  if (l.n + __popcll(who) > REP_CAP) {
    rep_cut(l, k, label_bits);
    who = __ballot(e > l.above);
  }
  if (e > l.above) l.ent[l.n + (int)__builtin_amdgcn_mbcnt_hi((unsigned)(who >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)who, 0u))] = e;
  l.n += __popcll(who);
}

__device__ __forceinline__ void topk_write(unsigned short* out_val, void* out_idx, int idx64, size_t at, unsigned long long e) {
  const int lab = (int)(0xFFFFFFFFu - (unsigned)e);
  out_val[at] = topk_bits((unsigned)(e >> 32));
  if (idx64) ((long long*)out_idx)[at] = lab;
  else ((int*)out_idx)[at] = lab;
}

// blk of nblk workgroups
__device__ __forceinline__ void topk_repair(const SelectParams& p, int blk, int nblk, int k, unsigned long long* lists, unsigned short* out_val,
                                            void* out_idx, int idx64, unsigned char* lds) {
  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, l16 = lane & 15, kg = lane >> 4;
  // rows to be done over, a bit each.  (Four wavefronts look at 64 counts each, which are a cache line apart.)
  unsigned* word = (unsigned*)(lds + REP_WORD);
  if (w < SEL_ROWS / 64) {
    const int row = 64 * w + lane;
    const unsigned have = row < p.batch ? p.count[row * SEL_COUNT_STRIDE] : (unsigned)k;
    const unsigned long long m = __ballot(have > (unsigned)SEL_CAP || have < (unsigned)k);
    if (lane < 2) word[2 * w + lane] = (unsigned)(m >> (32 * lane));
  }
  __syncthreads();
  unsigned need[SEL_ROWS / 32];
  int ngroups = 0;
#pragma unroll
  for (int g = 0; g < SEL_ROWS / 32; g++) {
    need[g] = __builtin_amdgcn_readfirstlane(word[g]);
    ngroups += need[g] != 0u ? 1 : 0;
  }
  if (ngroups == 0) return;
  // eight workgroups side by side take neighbouring slices of one group's labels, the eight behind them those of the next group
  const int q8 = (blk >> 3) / ngroups, which = (blk >> 3) - q8 * ngroups, slice = q8 * 8 + (blk & 7);
  const int most = (nblk >> 3) / ngroups * 8, slices = most < REP_SLICES ? most : REP_SLICES;
  if (slice >= slices) return;
  int group = 0;
  unsigned rows = 0u;
  {
    int at = 0;
#pragma unroll
    for (int g = 0; g < SEL_ROWS / 32; g++) {
      if (need[g] == 0u) continue;
      if (at == which) { group = g; rows = need[g]; }
      at++;
    }
  }
  RepList l[2];                                                       // rows 2w, 2w + 1 of the group
  unsigned long long floor[2];   // what their bounds leave out (a row with fewer than k logits at its bound has none)
#pragma unroll
  for (int q = 0; q < 2; q++) {
    const int row = 32 * group + 2 * w + q;
    floor[q] = 0ull;
    if (rows >> (2 * w + q) & 1u) {
      const unsigned bound = p.bound[row];
      if (p.count[row * SEL_COUNT_STRIDE] >= (unsigned)k && bound != 0u) floor[q] = ((unsigned long long)bound << 32) - 1ull;
    }
    l[q] = RepList{(unsigned long long*)lds + (2 * w + q) * REP_CAP, 0, floor[q]};
  }
  // the operand image of X, the two halves of a lane's 32 bytes apart
  for (int i = tid; i < 12 * 128; i += REP_NT)
    *(intx4*)(lds + REP_X + (i >> 7) * 2048 + (i & 1) * 1024 + ((i & 127) >> 1) * 16) = *(const intx4*)(p.xq + (size_t)group * 12 * 2048 + (size_t)i * 16);
  __syncthreads();
  // logits: wavefront w takes sixteen labels of a round, which are rows of one chunk, and all 32 batch rows
  const long long n16 = (p.num_labels + 15) / 16;
  const int label_bits = 32 - __builtin_clz((unsigned)(n16 * 16));   // (fewer than 2^31 labels)
  const int s_begin = (int)(n16 * slice / slices), s_end = (int)(n16 * (slice + 1) / slices);
  if (s_begin < s_end) {
    intx8 a[6];
    auto place = [&](int s) {   // behind the last one: the last one again
      const unsigned label = 16u * (unsigned)(s < s_end ? s : s_end - 1), c = label / (unsigned)p.rows_per_chunk, r0 = label - c * (unsigned)p.rows_per_chunk;
      return p.chunk[__builtin_amdgcn_readfirstlane(c)] + (size_t)(r0 + l16) * D + kg * 32;
    };
    auto load = [&](const unsigned char* src, int ks) {
      const intx4 lo = *(const intx4*)(src + ks * 128), hi = *(const intx4*)(src + ks * 128 + 16);
      a[ks] = intx8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    };
    {
      const unsigned char* src = place(s_begin + w);
#pragma unroll
      for (int ks = 0; ks < 6; ks++) load(src, ks);
    }
    int par = 0;
    for (int s0 = s_begin; s0 < s_end; s0 += REP_STEP / 16, par ^= 1) {
      const int s = s0 + w;
      const unsigned char* next = place(s + REP_STEP / 16);
      unsigned char* keys = lds + REP_KEYS + par * (32 * REP_KS * 2);   // [32 rows][REP_KS]
      floatx4 z[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
      for (int ks = 0; ks < 6; ks++) {
#pragma unroll
        for (int rb = 0; rb < 2; rb++) {
          const unsigned char* x = lds + REP_X + (rb * 6 + ks) * 2048 + lane * 16;
          const intx4 lo = *(const intx4*)x, hi = *(const intx4*)(x + 1024);
          z[rb] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a[ks], intx8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]}, z[rb], 0, 0, 0, 0, 0, 0);
        }
        load(next, ks);
      }
      const long long left = s < s_end ? p.num_labels - 16ll * s - 4 * kg : 0;   // labels from this lane's first on
#pragma unroll
      for (int rb = 0; rb < 2; rb++) {
        unsigned short key4[4];
#pragma unroll
        for (int e = 0; e < 4; e++) key4[e] = e < left ? (unsigned short)topk_key(bf16_bits(z[rb][e] * p.zscale)) : (unsigned short)0;
        *(uint2*)(keys + (16 * rb + l16) * (REP_KS * 2) + (16 * w + 4 * kg) * 2) =
            uint2{(unsigned)key4[0] | ((unsigned)key4[1] << 16), (unsigned)key4[2] | ((unsigned)key4[3] << 16)};
      }
      __syncthreads();   // (the keys of the round before are read by all: its barrier lies behind this round's)
#pragma unroll
      for (int q = 0; q < 2; q++)
        if (rows >> (2 * w + q) & 1u)
          for (int h = 0; h < REP_STEP; h += 64) {
            const unsigned key = *(const unsigned short*)(keys + (2 * w + q) * (REP_KS * 2) + (h + lane) * 2);
            rep_add(l[q], key ? ((unsigned long long)key << 32) | (0xFFFFFFFFu - (16u * (unsigned)s0 + (unsigned)(h + lane))) : 0ull, k, label_bits);
          }
    }
  }
  // the lists of a row, one behind the other in the order of their arrival (the second word of the row's counter line counts)
  lists += (size_t)which * slices * 32 * TOPK_MAX;   // the group's, [row][slices * TOPK_MAX]
#pragma unroll
  for (int q = 0; q < 2; q++)
    if (rows >> (2 * w + q) & 1u) {
      rep_cut(l[q], k, label_bits);
      unsigned at = 0;
      if (lane == 0) at = atomicAdd(p.count + (32 * group + 2 * w + q) * SEL_COUNT_STRIDE + 1, (unsigned)l[q].n);
      at = __builtin_amdgcn_readfirstlane(at);
      for (int h = lane; h < l[q].n; h += 64) lists[(size_t)(2 * w + q) * slices * TOPK_MAX + at + h] = l[q].ent[h];
    }
  __threadfence();
  __syncthreads();
  unsigned* arrived = word + SEL_ROWS / 32;
  if (tid == 0) *arrived = atomicAdd(p.count + (SEL_ROWS + group) * SEL_COUNT_STRIDE, 1u);
  __syncthreads();
  if (*arrived != (unsigned)slices - 1u) return;
  __threadfence();   // the last one: everybody's lists are in memory
#pragma unroll
  for (int q = 0; q < 2; q++) {
    if (!(rows >> (2 * w + q) & 1u)) continue;
    l[q].n = 0;
    l[q].above = floor[q];
    const unsigned long long* src = lists + (size_t)(2 * w + q) * slices * TOPK_MAX;
    const int total = (int)__hip_atomic_load(p.count + (32 * group + 2 * w + q) * SEL_COUNT_STRIDE + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    for (int h = lane; h - lane < total; h += 512) {   // (512 at once, or every 64 would be a memory latency)
      unsigned long long e[8];
#pragma unroll
      for (int u = 0; u < 8; u++) e[u] = h + 64 * u < total ? src[h + 64 * u] : 0ull;
#pragma unroll
      for (int u = 0; u < 8; u++) rep_add(l[q], e[u], k, label_bits);
    }
    rep_cut(l[q], k, label_bits);
    // best first
    const unsigned long long e0 = lane < l[q].n ? l[q].ent[lane] : 0ull, e1 = lane + 64 < l[q].n ? l[q].ent[lane + 64] : 0ull;
    int r0 = 0, r1 = 0;
    for (int j = 0; j < l[q].n; j++) {
      const unsigned long long o = l[q].ent[j];
      r0 += o > e0 ? 1 : 0;
      r1 += o > e1 ? 1 : 0;
    }
    const size_t at = (size_t)(32 * group + 2 * w + q) * k;
    if (e0 != 0ull) topk_write(out_val, out_idx, idx64, at + r0, e0);
    if (e1 != 0ull) topk_write(out_val, out_idx, idx64, at + r1, e1);
  }
}

// Picks the k best of the candidate list of batch row b (label and key per entry, all labels different) and writes
// them to the outputs [batch][k]: value descending, label ascending among equal values; labels as int32 or, with
// idx64, as int64.  The k-th largest key T is found first; the entries at or above it (k plus the ties at T) are then
// ranked against each other, several threads sharing the comparisons of one entry.  status |= 1 if a row collected
// more candidates than its list holds, |= 2 if a row has fewer than k: the outputs of such a row are not to be used, unless the launch
// has workgroups behind the batch's, which then write them (topk_repair).
constexpr int PICK_U = SEL_CAP / REP_NT;   // list entries of a thread
constexpr int PICK_LDS = SEL_CAP * 12 + 2 * (REP_NT / 64) * 8 + 16;
__global__ __launch_bounds__(REP_NT) void topk_pick_kernel(const SelectParams p, int k, unsigned short* out_val, void* out_idx, int idx64, int* status,
                                                           unsigned long long* lists) {
  extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
  const int b = blockIdx.x, tid = threadIdx.x;
  if (b >= p.batch) {
    topk_repair(p, b - p.batch, (int)gridDim.x - p.batch, k, lists, out_val, out_idx, idx64, lds_raw);
    return;
  }
  unsigned long long* ent = (unsigned long long*)lds_raw;
  unsigned* rank = (unsigned*)(ent + SEL_CAP);
  unsigned long long* wcnt = (unsigned long long*)(rank + SEL_CAP);
  unsigned* s_m = (unsigned*)(wcnt + 2 * (REP_NT / 64));
  // (requested together: behind the count, the entries cost another trip to memory; those past the count are not looked at)
  unsigned key[PICK_U], label[PICK_U];
#pragma unroll
  for (int u = 0; u < PICK_U; u++) {
    key[u] = (unsigned)p.cand_key[(size_t)b * SEL_CAP + u * REP_NT + tid];
    label[u] = p.cand_label[(size_t)b * SEL_CAP + u * REP_NT + tid];
  }
  const unsigned have = p.count[b * SEL_COUNT_STRIDE];
  const int n = have < (unsigned)SEL_CAP ? (int)have : SEL_CAP;
  const int used = __builtin_amdgcn_readfirstlane((n + REP_NT - 1) / REP_NT);
#pragma unroll
  for (int u = 0; u < PICK_U; u++)
    if (u * REP_NT + tid >= n) key[u] = 0u;   // (no entry has key 0)
  const bool useless = have > (unsigned)SEL_CAP || n < k;
  if (tid == 0) {
    if (useless) atomicOr(status, have > (unsigned)SEL_CAP ? 1 : 2);
    *s_m = 0u;
  }
  if (useless && lists) return;
#pragma unroll
  for (int u = 0; u < PICK_U; u++)
    if (u < used) rank[u * REP_NT + tid] = 0u;
  const unsigned T = block_kth_key<REP_NT / 64, PICK_U>(key, used, k, wcnt);   // its barriers also publish s_m and rank
#pragma unroll
  for (int u = 0; u < PICK_U; u++)
    if (u * REP_NT + tid < n && key[u] >= T) ent[atomicAdd(s_m, 1u)] = ((unsigned long long)key[u] << 32) | (unsigned long long)(0xFFFFFFFFu - label[u]);
  __syncthreads();
  const int m = (int)*s_m;                      // >= min(k, n) entries, all different
  int mp = 64;
  while (mp < m && mp < REP_NT) mp <<= 1;       // threads per slice; REP_NT / mp slices share an entry's comparisons
  const int slices = REP_NT / mp, sl = tid / mp;
  const int per = (m + slices - 1) / slices, j0 = sl * per, j1 = j0 + per < m ? j0 + per : m;
  for (int i = tid & (mp - 1); i < m; i += mp) {
    const unsigned long long mine = ent[i];
    unsigned r = 0;
    for (int j = j0; j < j1; j++) r += ent[j] > mine ? 1u : 0u;
    if (r != 0u) atomicAdd(&rank[i], r);
  }
  __syncthreads();
  for (int i = tid; i < m; i += REP_NT) {
    const unsigned r = rank[i];
    if (r < (unsigned)k) topk_write(out_val, out_idx, idx64, (size_t)b * k + r, ent[i]);
  }
  if (tid >= m && tid < k) {   // fewer than k candidates (reported above): -inf, label -1
    out_val[(size_t)b * k + tid] = 0xFF80;
    if (idx64) ((long long*)out_idx)[(size_t)b * k + tid] = -1;
    else ((int*)out_idx)[(size_t)b * k + tid] = -1;
  }
}

}  // namespace xmc
