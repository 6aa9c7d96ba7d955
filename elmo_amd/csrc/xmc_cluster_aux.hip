// The small kernels around the one-pass cluster step (xmc_cluster.hip): operand images of X with the clearing of the
// counters in front of it, the fixed-order sum of the grad_X partials behind it; and the layout of its workspace.
#include "xmc_cluster.hip"

namespace xmc {

// Members of a cluster for a batch, and 16-row batch blocks of a member.  64 rows per member fill the registers; a batch
// of up to 32 rows takes half of them.  cluster_size is the size that a workspace is laid out for: clusters of three and six, whose
// tile streams are 5/4 as many, fit into the places of four and eight (240 + 3 chunks sums of a member against 256 + 4 chunks).
inline int cluster_size(int batch) { return batch <= 64 ? 1 : batch <= 128 ? 2 : batch <= 256 ? 4 : 8; }
// 129 to 192 and 257 to 384 batch rows would leave every fourth member without rows, a quarter of all matrix work for nothing, and their
// features divide evenly by three and six (16 and 8 blocks for eight wavefronts); 240 of 256 compute units work then.  us a step, clusters of
// four / three (192 rows), eight / six (384):
//   131 K labels   FP8 nearest 151/126 326/260, sr_fast 160/133 327/270, Philox 244/230 404/347;  e4m3 with bf16 products, nearest 200/165 378/302,
//                  Philox 297/269 464/402;  bf16, nearest 214/183 393/312, Philox 305/276 471/408
//   500 K          FP8 500/412 1143/908, 530/439 1149/933, 852/787 1447/1226;  686/547 1344/1064, 1050/930 1666/1439;  765/649 1447/1186, 1070/957 1687/1458
//   8 K            FP8 nearest 40.2/37.5 52.7/48.0;  bf16, Philox 48.2/49.1 62.2/58.7;  3 K labels, bf16, nearest 36.6/38.9 43.8/38.7
// With a few tiles a cluster, three members are 5 % faster to 7 % slower than four, by no rule of tiles or rounds: four below
// 7,680 label rows (FP8 logits) and 10,240 (12 K: FP8 41.7/38.5, e4m3 with bf16 products 46.4/42.8, bf16 47.6/44.7).
inline int cluster_members(int batch, long long rows, bool fp8_logits) {
  return batch > 128 && batch <= 192 && rows >= (fp8_logits ? 7680 : 10240) ? 3 : batch > 256 && batch <= 384 ? 6 : cluster_size(batch);
}
inline int cluster_blocks(int batch) { return batch <= 32 ? 2 : 4; }

// Where the launches of a step keep what they pass on to one another.
struct ClusterPlace {
  unsigned char* xq; unsigned short* xt;   // operand images of X
  unsigned* keys; int* flags; int* xcc;    // positives by tile (MAX_POS per 256 batch rows); CLU_FLAG_INTS counters; XCC ids
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

// The launch in front of the step kernel, PREP_NT threads a block: ptr_blocks per 256 batch rows group the positives by 64-row tile and
// write the first key of each, the others prepare X.
struct ClusterPrep {
  const int* coo; int nnz, batch, label_base, label_count, pairs, rows_per_chunk, tiles_per_chunk, num_tiles, ptr_blocks;
  unsigned* keys; int* tile_ptr; size_t tp_stride;
  const unsigned short* x; int bp, kind;
  unsigned char* xq; unsigned short* xt; int* flags; int* err;
};
__global__ __launch_bounds__(PREP_NT) void cluster_prep_kernel(const ClusterPrep p, const DropoutParams dp) {
  const int blk = blockIdx.x;
  if (blk < p.ptr_blocks * p.pairs) {
    const int pr = blk / p.ptr_blocks, t0 = (blk - pr * p.ptr_blocks) * PREP_NT, t = t0 + (int)threadIdx.x;
    int p0, p1;
    group_positives_block(t0, p.coo, p.nnz, p.batch, 256 * pr, p.label_base, p.label_count, p.rows_per_chunk, 1.0f / (float)p.rows_per_chunk,
                          p.tiles_per_chunk, p.keys + (size_t)pr * MAX_POS, &p0, &p1);
    if (t <= p.num_tiles) p.tile_ptr[pr * p.tp_stride + t] = p0;
    return;
  }
  cluster_prep_thread((blk - p.ptr_blocks * p.pairs) * PREP_NT + (int)threadIdx.x, p.x, p.batch, p.bp, p.kind, p.xq, p.xt, p.flags, p.err, dp);
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
  const int tid = threadIdx.x, wv = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
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
  if (16 * (m * r.nbk + (q >> 9) / 6) >= r.batch) return;   // (the same for the block's 64 positions: rows that are not there)
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
    // the rest at once too: one behind the other, each took a memory latency.  us a step: e4m3, bf16 products, 2 K labels, batch 192
    // 41.5, now 38.4; bf16, nearest, 12 K, batch 272 58.5 with the last one loaded again in place of those that are not there, now 56.7;
    // 131 K, batch 512 397 / 395 / 392
    if (k < s1) {
      floatx4 t[7];
#pragma unroll
      for (int u = 0; u < 7; u++) {
        t[u] = floatx4{0.f, 0.f, 0.f, 0.f};
        if (k + u < s1) t[u] = r.partial[(size_t)((k + u) * r.c + m) * pslot + q];
      }
#pragma unroll
      for (int u = 0; u < 7; u++) s += t[u];   // (a sum is never -0 here, so what is added to it behind its last is nothing)
    }
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
