// The small kernels around the one-pass cluster step (xmc_cluster.hip): operand images of X with the clearing of the
// counters in front of it, the fixed-order sum of the grad_X partials behind it; and the layout of its workspace.
#include "xmc_cluster.hip"

namespace xmc {

// members of a cluster for a batch, and 16-row batch blocks of a member.  64 rows per member fill the registers; a batch
// of up to 32 rows takes half of them.
inline int cluster_size(int batch) { return batch <= 64 ? 1 : batch <= 128 ? 2 : batch <= 256 ? 4 : 8; }
inline int cluster_blocks(int batch) { return batch <= 32 ? 2 : 4; }

// Where the launches of a step keep what they pass on to one another.
struct ClusterPlace {
  unsigned char* xq; unsigned short* xt;   // operand images of X
  unsigned* keys; int* flags; int* xcc;    // sorted positives (MAX_POS per 256 batch rows); CLU_FLAG_INTS counters; XCC ids
  float* gx;                               // grad_X of the segments before (label spaces of several segments)
  int* tile_ptr; size_t tp_stride;
  unsigned char* exch; floatx4* partial;
  int* err; int* sticky;
};

// workspace of the cluster path (byte offsets, 256-byte aligned); the first 256 bytes hold the error words
constexpr size_t TW_ERR = 0;        // int: error word of the last step; next int: the error words of all steps, OR-ed
constexpr size_t TW_HEAD = 256;
struct ClusterLayout { size_t xq, xt, keys, flags, xcc, gx, tile_ptr, tp_stride, exch, partial, bytes; int slots; };
inline ClusterLayout cluster_layout(int num_chunks, int rows_per_chunk, int batch) {
  ClusterLayout l;
  const int c = batch <= 64 ? 2 : cluster_size(batch);   // (what a cluster of one needs fits as well)
  const size_t bp = (size_t)c * 64, pairs = (bp + 255) / 256;
  auto up = [](size_t b) { return (b + 255) / 256 * 256; };
  l.xq = TW_HEAD;
  l.xt = l.xq + bp * D * 2;
  l.keys = l.xt + bp * D * 2;
  l.flags = l.keys + pairs * MAX_POS * 4 + 256;   // (the kernels read up to seven keys past the end of a list)
  l.xcc = l.flags + CLU_FLAG_INTS * 4;
  l.gx = l.xcc + CLU_MAXWG * 4;
  l.tile_ptr = l.gx + bp * D * 4;
  const size_t t64 = (size_t)num_chunks * ((rows_per_chunk + TL - 1) / TL), t32 = (size_t)num_chunks * ((rows_per_chunk + 31) / 32);
  l.tp_stride = (t64 + 1 + 63) / 64 * 64;
  l.exch = up(l.tile_ptr + pairs * l.tp_stride * 4);
  l.partial = l.exch + (size_t)CLU_MAXWG * CLU_SLOTS * 8192;
  const size_t clusters = CLU_MAXWG / c;
  l.slots = (int)((t32 < clusters ? t32 : clusters) + num_chunks);
  l.bytes = l.partial + (size_t)l.slots * c * 4 * 6 * 8 * 64 * 16;
  return l;
}

// X -> operand images (zero rows up to the padded batch), one thread per four features of a row:
//   logits, kind 0 (bf16 products with bf16 weights): block (16 rows, 32 features) of 64 lanes x 8: lane = row % 16 + 16 (k / 8 % 4)
//           kind 1 (bf16 products with e4m3 weights, whose rows are read 16 bytes at a time): features 64 j + 16 q + 8 u + i are
//                  element i of lane group q in step 2 j + u
//           kind 2 (FP8 products): e4m3 codes, step of 128 features: lane group q holds bytes 16 q.. and 64 + 16 q..
//   grad_W: X^T: block (16 features, 32 batch rows) of 64 lanes x 8: lane = feature % 16 + 16 (row / 8 % 4)
// Also clears the counters and, unless it is null, the error word.
__device__ __forceinline__ void cluster_prep_thread(int i, const unsigned short* x, int batch, int bp, int kind, unsigned char* xq,
                                                    unsigned short* xt, int* flags, int* err, const DropoutParams& dp) {
  if (i < CLU_FLAG_INTS) flags[i] = 0;
  if (i == 0 && err) *err = 0;
  if (i >= bp * (D / 4)) return;
  const int b = i / (D / 4), k = (i - b * (D / 4)) * 4;
  unsigned short raw[4] = {0, 0, 0, 0};
  if (b < batch) {
    const uint2 r = *(const uint2*)(x + (size_t)b * D + k);
    raw[0] = (unsigned short)r.x; raw[1] = (unsigned short)(r.x >> 16); raw[2] = (unsigned short)r.y; raw[3] = (unsigned short)(r.y >> 16);
#pragma unroll
    for (int q = 0; q < 4; q++) raw[q] = dropout_bf16(raw[q], (unsigned)(b * D + k + q), dp);
  }
  const uint2 packed = uint2{(unsigned)raw[0] | ((unsigned)raw[1] << 16), (unsigned)raw[2] | ((unsigned)raw[3] << 16)};
  const int nb = b >> 4, l16 = b & 15;
  if (kind == 0) {
    *(uint2*)(xq + ((size_t)(nb * 24 + (k >> 5)) * 64 + l16 + 16 * ((k >> 3) & 3)) * 16 + (k & 7) * 2) = packed;
  } else if (kind == 1) {
    *(uint2*)(xq + ((size_t)(nb * 24 + 2 * (k >> 6) + ((k >> 3) & 1)) * 64 + l16 + 16 * ((k >> 4) & 3)) * 16 + (k & 7) * 2) = packed;
  } else {
    int codes = 0;
    codes = __builtin_amdgcn_cvt_pk_fp8_f32(clamp448(bf16_from_bits(raw[0])), clamp448(bf16_from_bits(raw[1])), codes, false);
    codes = __builtin_amdgcn_cvt_pk_fp8_f32(clamp448(bf16_from_bits(raw[2])), clamp448(bf16_from_bits(raw[3])), codes, true);
    const int pk = k & 127;
    *(int*)(xq + ((size_t)(nb * 6 + (k >> 7)) * 64 + l16 + 16 * ((pk >> 4) & 3)) * 32 + (((pk >> 6) << 4) | (pk & 15))) = codes;
  }
#pragma unroll
  for (int q = 0; q < 4; q++) {
    const int f = k + q;
    xt[((size_t)((f >> 4) * (bp / 32) + (b >> 5)) * 64 + (f & 15) + 16 * ((b >> 3) & 3)) * 8 + (b & 7)] = raw[q];
  }
}

// The launch in front of the step kernel, 256 threads a block: sort_blocks blocks per 256 batch rows sort the positives,
// ptr_blocks write the first key of every 64-row tile (first_keys_block), the others prepare X.
struct ClusterPrep {
  const int* coo; int nnz, n_pad, batch, label_base, label_count, pairs, rows_per_chunk, tiles_per_chunk, num_tiles, sort_blocks, ptr_blocks;
  unsigned* keys; int* tile_ptr; size_t tp_stride;
  const unsigned short* x; int bp, kind;
  unsigned char* xq; unsigned short* xt; int* flags; int* err;
};
__global__ __launch_bounds__(256) void cluster_prep_kernel(const ClusterPrep p, const DropoutParams dp) {
  int blk = blockIdx.x;
  if (blk < p.sort_blocks * p.pairs) {
    const int pr = blk / p.sort_blocks;
    quad_sort_block(blk - pr * p.sort_blocks, p.coo, p.nnz, p.n_pad, p.batch, 256 * pr, p.label_base, p.label_count, p.keys + (size_t)pr * MAX_POS);
    return;
  }
  blk -= p.sort_blocks * p.pairs;
  if (blk < p.ptr_blocks * p.pairs) {
    const int pr = blk / p.ptr_blocks, t0 = (blk - pr * p.ptr_blocks) * 256, t = t0 + (int)threadIdx.x;
    int p0, p1;
    first_keys_block(t0, p.coo, p.nnz, p.batch, 256 * pr, p.label_base, p.label_count, p.rows_per_chunk, 1.0f / (float)p.rows_per_chunk,
                     p.tiles_per_chunk, &p0, &p1);
    if (t <= p.num_tiles) p.tile_ptr[pr * p.tp_stride + t] = p0;
    return;
  }
  cluster_prep_thread((blk - p.ptr_blocks * p.pairs) * 256 + (int)threadIdx.x, p.x, p.batch, p.bp, p.kind, p.xq, p.xt, p.flags, p.err, dp);
}

// grad_X = sum of the members' partials in a fixed order.  A block handles 64 positions (floatx4 values) of the partial
// layout; its wavefronts take a share of the slots each: equal shares, or with `flush` the chunks ck = wavefront, wavefront +
// CLU_RW, ... (fewer chunks than wavefronts: several wavefronts share a chunk's slots), each chunk's sum rounded to bf16 by itself (chunked.py:116).  The first block checks that the members
// of every cluster ran on one XCD and passes the error word on to the sticky one.
//   add: continue from gx_total;  final: write grad_X (with the dropout's backward) instead of gx_total
struct ClusterReduce {
  const floatx4* partial; int c, nbk, nclusters, ntiles, tpc, nchunks, flush;
  const int* xcc; int* err; int* sticky; int* failure_word;
  float* gx_total; int add, final_out, batch;
  unsigned short* gx_bf16; float* gx_f32;
};
constexpr int CLU_RW = 8;   // wavefronts of a block
__global__ __launch_bounds__(CLU_RW * 64) void cluster_reduce_kernel(const ClusterReduce r, const DropoutParams dp) {
  const int tid = threadIdx.x, wv = tid >> 6, lane = tid & 63;
  if (blockIdx.x == 0) {
    if (r.c > 1 && tid < r.nclusters)
      for (int m = 1; m < r.c; m++)
        if (r.xcc[((tid >> 3) * r.c + m) * 8 + (tid & 7)] != r.xcc[(tid >> 3) * r.c * 8 + (tid & 7)])
          __hip_atomic_fetch_or(r.err, 2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    if (tid == 0) report_step_error(r.err, r.sticky, r.failure_word);
  }
  __shared__ floatx4 sh[CLU_RW][64];
  const int pslot = r.nbk * 6 * 8 * 64;
  const int pos = blockIdx.x * 64 + lane, m = pos / pslot, q = pos - m * pslot;
  auto sum_slots = [&](int s0, int s1) {
    floatx4 s = {0.f, 0.f, 0.f, 0.f};
    int k = s0;
    for (; k + 8 <= s1; k += 8) {
      floatx4 t[8];
#pragma unroll
      for (int u = 0; u < 8; u++) t[u] = r.partial[(size_t)((k + u) * r.c + m) * pslot + q];
#pragma unroll
      for (int u = 0; u < 8; u++) s += t[u];
    }
    for (; k < s1; k++) s += r.partial[(size_t)(k * r.c + m) * pslot + q];
    return s;
  };
  const int per = r.flush && r.nchunks < CLU_RW ? CLU_RW / r.nchunks : 1;   // wavefronts of a chunk
  floatx4 tot = {0.f, 0.f, 0.f, 0.f};
  if (r.flush) {
    // cluster that walks tile t (see the partition in cluster_step_kernel): the last one whose range starts at or before t
    auto owner = [&](int t) { return (int)((((long long)t + 1) * r.nclusters - 1) / r.ntiles); };
    for (int ck = wv / per; ck < r.nchunks; ck += CLU_RW) {
      const int t1 = ck == r.nchunks - 1 ? r.ntiles : (ck + 1) * r.tpc;
      const int s0 = owner(ck * r.tpc) + ck, ns = owner(t1 - 1) + ck + 1 - s0, q = wv % per;
      const floatx4 s = sum_slots(s0 + ns * q / per, s0 + ns * (q + 1) / per);
#pragma unroll
      for (int e = 0; e < 4; e++) tot[e] += per > 1 ? s[e] : bf16_rt(s[e]);
    }
  } else {
    tot = sum_slots(r.nclusters * wv / CLU_RW, r.nclusters * (wv + 1) / CLU_RW);
  }
  sh[wv][lane] = tot;
  __syncthreads();
  if (wv != 0) return;
  if (per > 1) {
    tot = floatx4{0.f, 0.f, 0.f, 0.f};
    for (int ck = 0; ck < r.nchunks; ck++) {
      floatx4 s = sh[ck * per][lane];
      for (int q = 1; q < per; q++) s += sh[ck * per + q][lane];
#pragma unroll
      for (int e = 0; e < 4; e++) tot[e] += bf16_rt(s[e]);
    }
  } else {
#pragma unroll
    for (int q = 1; q < CLU_RW; q++) tot += sh[q][lane];
  }
  // position -> ((16-row block * 6 + feature block) * 8 + wavefront) * 64 + lane of cluster_step_kernel
  const int fv = (q >> 6) & 7, bk = q >> 9, mb = bk / 6, nn = bk - mb * 6;
  const int col = 96 * fv + 16 * nn + (lane & 15);
#pragma unroll
  for (int e = 0; e < 4; e++) {
    const int b = m * 16 * r.nbk + 16 * mb + 4 * (lane >> 4) + e;
    const size_t at = (size_t)b * D + col;
    float val = tot[e];
    if (r.add) val += r.gx_total[at];
    if (!r.final_out) {
      r.gx_total[at] = val;
    } else if (b < r.batch) {
      val = dropout_backward(val, (unsigned)at, dp);
      if (r.gx_f32) r.gx_f32[at] = val;
      r.gx_bf16[at] = bf16_bits(val);
    }
  }
}

}  // namespace xmc
