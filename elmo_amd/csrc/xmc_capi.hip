// extern "C" surface of libelmo_xmc.so: argument validation, workspace carving and kernel launches.
// Declarations and the reference interfaces they replace: include/elmo_xmc.h.
#include "../../include/elmo_xmc.h"
#include "xmc_fp8_forward.hip"
#include "xmc_fp8_quad.hip"
#include "xmc_fp8_role.hip"
#include "xmc_fp8_small.hip"
#include "xmc_tiled.hip"
#include "xmc_cluster_aux.hip"
#include "xmc_topk.hip"
#include "xmc_dropout.hip"
#include <stdlib.h>
#include <atomic>
#include <mutex>

using namespace xmc;

// Operand image of X for xmc_fp8_forward_static, the entry point that takes no workspace: e4m3 X in MFMA operand order
// (BP*D bytes).  Every GPU the library runs on holds its own copy of this array until the process ends.  In host code the name
// stands for the symbol only, never for device memory: the address kernels get is the one hipGetSymbolAddress returned for the
// current device.
static __device__ __align__(256) unsigned char scratch[(size_t)BP * D];

namespace {

struct DeviceInfo { int ok; int cus; unsigned char* scratch_ptr; int* failure_word; };

// Filled once per device, by the first call on it; std::call_once makes concurrent first calls of several host threads
// wait for the one that fills the slot, and publishes the finished slot to all of them.
DeviceInfo g_device_info[64];
std::once_flag g_device_once[64];

void fill_device_info(int dev) {
  DeviceInfo di = {-1, 0, nullptr, nullptr};
  hipDeviceProp_t prop;
  if (hipGetDeviceProperties(&prop, dev) != hipSuccess) { g_device_info[dev] = di; return; }
  di.cus = prop.multiProcessorCount;
  di.ok = (__builtin_strncmp(prop.gcnArchName, "gfx950", 6) == 0) ? 1 : -1;
  // this device's copy of the static scratch array (device `dev` is current here); stays null if the lookup fails
  void* sp = nullptr;
  di.scratch_ptr = (di.ok == 1 && hipGetSymbolAddress(&sp, HIP_SYMBOL(scratch)) == hipSuccess) ? (unsigned char*)sp : nullptr;
  // the two words of host memory in which the kernels of this device announce failed steps; live until the process ends.  A
  // caller may be capturing a graph: the allocation is none of that graph's business
  if (di.ok == 1) {
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    const bool swapped = hipThreadExchangeStreamCaptureMode(&mode) == hipSuccess;
    void* fw = nullptr;
    if (hipHostMalloc(&fw, 64, hipHostMallocMapped) == hipSuccess) {
      ((int*)fw)[0] = ((int*)fw)[1] = 0;
      di.failure_word = (int*)fw;
    }
    if (swapped) (void)hipThreadExchangeStreamCaptureMode(&mode);
  }
  // opt in to the full 160 KiB of LDS once per device
  role_plain_set_lds();
  role_heavy_set_lds();
  small_set_lds();
  cluster_set_lds_bf16();
  cluster_set_lds_sim();
  cluster_set_lds_fp8();
  (void)hipFuncSetAttribute((const void*)cluster_prep_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, MAX_POS * 4);
  (void)hipFuncSetAttribute((const void*)fp8_forward_kernel<1, 1, false>, hipFuncAttributeMaxDynamicSharedMemorySize, FwdGeom<1>::LDS);
  (void)hipFuncSetAttribute((const void*)fp8_forward_kernel<1, 4, false>, hipFuncAttributeMaxDynamicSharedMemorySize, FwdGeom<1>::LDS);
  (void)hipFuncSetAttribute((const void*)fp8_forward_kernel<2, 1, false>, hipFuncAttributeMaxDynamicSharedMemorySize, FwdGeom<2>::LDS);
  (void)hipFuncSetAttribute((const void*)fp8_forward_kernel<1, 1, true>, hipFuncAttributeMaxDynamicSharedMemorySize, FwdGeom<1, true>::LDS);
  (void)hipFuncSetAttribute((const void*)fp8_forward_kernel<1, 4, true>, hipFuncAttributeMaxDynamicSharedMemorySize, FwdGeom<1, true>::LDS);
  (void)hipFuncSetAttribute((const void*)fp8_forward_select_kernel<0, 4>, hipFuncAttributeMaxDynamicSharedMemorySize, SelGeom<4>::LDS);
  (void)hipFuncSetAttribute((const void*)fp8_forward_select_kernel<1, 4>, hipFuncAttributeMaxDynamicSharedMemorySize, SelGeom<4>::LDS);
  (void)hipFuncSetAttribute((const void*)fp8_forward_select_kernel<0, 8>, hipFuncAttributeMaxDynamicSharedMemorySize, SelGeom<8>::LDS);
  (void)hipFuncSetAttribute((const void*)fp8_forward_select_kernel<1, 8>, hipFuncAttributeMaxDynamicSharedMemorySize, SelGeom<8>::LDS);
  (void)hipFuncSetAttribute((const void*)topk_pick_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, REP_LDS > PICK_LDS ? REP_LDS : PICK_LDS);
  (void)hipFuncSetAttribute((const void*)quad_prep_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, MAX_POS * 4);
#define XMC_TILED_ATTR(DD)                                                                                                                        \
  (void)hipFuncSetAttribute((const void*)tiled_prep_kernel<DD>, hipFuncAttributeMaxDynamicSharedMemorySize, MAX_POS * 4);                          \
  (void)hipFuncSetAttribute((const void*)tiled_gradx_kernel<W_BF16, 1, DD>, hipFuncAttributeMaxDynamicSharedMemorySize, TgxGeom<W_BF16, 1, DD>::LDS); \
  (void)hipFuncSetAttribute((const void*)tiled_gradx_kernel<W_E4M3, 1, DD>, hipFuncAttributeMaxDynamicSharedMemorySize, TgxGeom<W_E4M3, 1, DD>::LDS); \
  (void)hipFuncSetAttribute((const void*)tiled_gradx_kernel<W_BF16, 2, DD>, hipFuncAttributeMaxDynamicSharedMemorySize, TgxGeom<W_BF16, 2, DD>::LDS); \
  (void)hipFuncSetAttribute((const void*)tiled_gradx_kernel<W_E4M3, 2, DD>, hipFuncAttributeMaxDynamicSharedMemorySize, TgxGeom<W_E4M3, 2, DD>::LDS); \
  (void)hipFuncSetAttribute((const void*)tiled_logits_kernel<W_BF16, true, DD>, hipFuncAttributeMaxDynamicSharedMemorySize, TlgGeom<W_BF16, DD>::LDS); \
  (void)hipFuncSetAttribute((const void*)tiled_logits_kernel<W_BF16, false, DD>, hipFuncAttributeMaxDynamicSharedMemorySize, TlgGeom<W_BF16, DD>::LDS); \
  (void)hipFuncSetAttribute((const void*)tiled_logits_kernel<W_E4M3, true, DD>, hipFuncAttributeMaxDynamicSharedMemorySize, TlgGeom<W_E4M3, DD>::LDS); \
  (void)hipFuncSetAttribute((const void*)tiled_logits_kernel<W_E4M3, false, DD>, hipFuncAttributeMaxDynamicSharedMemorySize, TlgGeom<W_E4M3, DD>::LDS); \
  (void)hipFuncSetAttribute((const void*)tiled_logits_fp8_kernel<DD>, hipFuncAttributeMaxDynamicSharedMemorySize, TlgGeom<W_E4M3, DD>::LDS)
  XMC_TILED_ATTR(D);
  XMC_TILED_ATTR(1024);
#undef XMC_TILED_ATTR
  (void)hipFuncSetAttribute((const void*)tiled_update2_kernel<ROUND_RTN>, hipFuncAttributeMaxDynamicSharedMemorySize, 2 * TU2_GBUF);
  (void)hipFuncSetAttribute((const void*)tiled_update2_kernel<ROUND_SR_PHILOX>, hipFuncAttributeMaxDynamicSharedMemorySize, 2 * TU2_GBUF);
  (void)hipFuncSetAttribute((const void*)tiled_update2_kernel<ROUND_SR_FAST>, hipFuncAttributeMaxDynamicSharedMemorySize, 2 * TU2_GBUF);
  // the update kernels with two batch halves keep 96 KiB of operands in LDS, more than the default limit
#define XMC_UPD_ATTR_D(WTYPE, RMODE, KH, DD) (void)hipFuncSetAttribute((const void*)tiled_update_kernel<WTYPE, RMODE, 2, KH, DD, BP / 32>, hipFuncAttributeMaxDynamicSharedMemorySize, tup_lds_bytes(2, DD))
#define XMC_UPD_ATTR(WTYPE, RMODE, KH) XMC_UPD_ATTR_D(WTYPE, RMODE, KH, D); XMC_UPD_ATTR_D(WTYPE, RMODE, KH, 1024)
  XMC_UPD_ATTR(W_BF16, ROUND_RTN, false); XMC_UPD_ATTR(W_BF16, ROUND_SR_PHILOX, false); XMC_UPD_ATTR(W_BF16, ROUND_SR_FAST, false);
  XMC_UPD_ATTR(W_E4M3, ROUND_RTN, false); XMC_UPD_ATTR(W_E4M3, ROUND_SR_PHILOX, false); XMC_UPD_ATTR(W_E4M3, ROUND_SR_FAST, false);
  XMC_UPD_ATTR(W_E4M3, ROUND_RTN, true); XMC_UPD_ATTR(W_E4M3, ROUND_SR_PHILOX, true); XMC_UPD_ATTR(W_E4M3, ROUND_SR_FAST, true);
#undef XMC_UPD_ATTR_D
#undef XMC_UPD_ATTR
  g_device_info[dev] = di;
}

DeviceInfo device_info() {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return DeviceInfo{-1, 0, nullptr};
  std::call_once(g_device_once[dev], fill_device_info, dev);
  return g_device_info[dev];
}

// polls of a partner's counter before a workgroup of the fused step gives up (xmc_debug_spin_limit)
std::atomic<int> g_spin_limit{QSPIN_LIMIT};

// optional event pair recorded around the next launch of the fused step kernel by the calling thread (benchmarking aid)
thread_local hipEvent_t g_prof_start = nullptr, g_prof_stop = nullptr;

inline bool aligned16(const void* q) { return ((uintptr_t)q & 15) == 0; }

int check_common(void* const* chunk_ptrs, int num_chunks, int rows_per_chunk, const void* x, int batch, int features,
                 const void* workspace, size_t workspace_bytes, int batch_unit = 16, int most_rows = BP) {
  if (!chunk_ptrs || !x || !workspace) return XMC_ERR_NULL;
  if (features != D || batch <= 0 || batch > most_rows || batch % batch_unit != 0) return XMC_ERR_SHAPE;
  if (rows_per_chunk <= 0 || rows_per_chunk % 16 != 0) return XMC_ERR_SHAPE;
  if (num_chunks <= 0 || num_chunks > MAX_CHUNKS) return XMC_ERR_RANGE;
  if ((long long)num_chunks * rows_per_chunk > 0x7FFFFFFFLL) return XMC_ERR_RANGE;   // the fused step has a lower limit of its own
  for (int c = 0; c < num_chunks; c++) {
    if (!chunk_ptrs[c]) return XMC_ERR_NULL;
    if (!aligned16(chunk_ptrs[c])) return XMC_ERR_ALIGN;
  }
  if (!aligned16(x) || ((uintptr_t)workspace & 255) != 0) return XMC_ERR_ALIGN;
  if (workspace_bytes < xmc_workspace_bytes(num_chunks, rows_per_chunk)) return XMC_ERR_WORKSPACE;
  return XMC_OK;
}

// The error word of a step that ran in a workspace which goes away with the call, passed on behind the step by one thread:
// into the two words of a workspace that stays, or, without one, into the second failure word in host memory (a clock
// reading, so that it changes with every failed step, and the error bits).
__global__ void pass_on_error_kernel(const int* err, int* into_error, int* into_sticky, int* failure_word) {
  const int e = __hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (into_sticky) {
    *into_error = e;
    report_step_error(err, into_sticky, failure_word);
  } else if (e != 0) {
    __hip_atomic_store(failure_word + 1, (int)((unsigned)__builtin_amdgcn_s_memrealtime() << 2 | (unsigned)(e & 3)), __ATOMIC_RELEASE,
                       __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

// plain 16-byte-per-lane copy: the known-size reference against which memory counters are calibrated
__global__ __launch_bounds__(256) void copy_probe_kernel(const uint4* __restrict__ src, uint4* __restrict__ dst, size_t n16) {
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n16; i += (size_t)gridDim.x * 256) dst[i] = src[i];
}

// stride of the order in which a chunk's n tiles are visited: about 0.618 n, coprime to n
int tile_stride(int n) {
  if (n < 3) return 1;
  for (int s = (int)(0.618 * n);; s++) {
    int a = s, b = n;
    while (b) { const int t = a % b; a = b; b = t; }
    if (a == 1) return s;   // (n - 1 at the latest)
  }
}

int launch_status() { return hipGetLastError() == hipSuccess ? XMC_OK : XMC_ERR_LAUNCH; }

// xmc_fp8_forward_topk takes the labels in segments of at most 2^17: as many whole chunks as fit (fewer, larger
// launches), or, for a chunk that is larger than that by itself, pieces of it of 2^17 rows
constexpr int TOPK_SEG = 1 << 17;
int topk_group(int rows_per_chunk) { const int g = TOPK_SEG / rows_per_chunk; return g < 1 ? 1 : g; }
long long topk_segment_rows(int rows_per_chunk) {
  return rows_per_chunk > TOPK_SEG ? (long long)TOPK_SEG : (long long)topk_group(rows_per_chunk) * rows_per_chunk;
}
size_t topk_zbuf_bytes(int rows_per_chunk) {
  return ((size_t)BP * (size_t)topk_segment_rows(rows_per_chunk) * 2 + 255) / 256 * 256;
}

// the operand image of X for the batch blocks of 32 rows in use
void prep_x(const void* x_bf16, int batch, float scale_x, unsigned char* xq, hipStream_t stream) {
  const int n = (batch + 31) / 32 * 32 * (D / 4);
  prep_x_kernel<<<n / 256, 256, 0, stream>>>((const unsigned short*)x_bf16, batch, n, 1.0f / scale_x, xq);
}

// the inverse of s modulo n, for s coprime to n
int tile_stride_inverse(int s, int n) {
  long long r0 = n, r1 = s % n, t0 = 0, t1 = 1;
  while (r1 != 0) {
    const long long q = r0 / r1, r = r0 - q * r1, t = t0 - q * t1;
    r0 = r1; r1 = r; t0 = t1; t1 = t;
  }
  return (int)(((t0 % n) + n) % n);
}

// Whether the workgroups of the logits kernel convert X themselves instead of reading an image that a launch in front has written.
// The launch is 3 us of the GPU, and what bounds small label spaces is the host's 4 us for it; the conversion takes a workgroup longer
// the more rows it has, without loads of tiles on their way from 49 rows on.  us a call, image / conversion, by rows:
//   1   131 K labels 20.0/17.9    40  30 K 12.6/9.9, 131 K 22.1/21.2, 300 K 40.9/40.0, 670 K 118.0/116.6    48  48 K 12.6/11.8
//   64  2 K 12.0/9.4, 32 K 12.1/10.3, 48 K 13.0/13.7, 131 K 23.3/24.4
//   100, 128  2 K 12.0/9.5 11.9/10.0 among others, but 24.5/25.0 24.6/26.0 alone
// Where no host is in the way (replays of a graph) the launch is cheaper, and 57 to 64 rows a little slower without it: 2 K labels, 48 rows
// 6.5/6.2, 56 6.5/6.4, 64 6.5/6.8, 30 K, 64 10.0/10.5; waited for alone, 2 K, 64 23.4/22.2, 30 K 26.1/25.5.
bool forward_converts(int batch, long long tiles, int cus) {
  return batch <= 48 || (batch <= FWD_CONV && tiles <= 4 * (long long)cus);
}
// The launches of the inference logits, shared by xmc_fp8_forward (operand images in the caller's workspace) and
// xmc_fp8_forward_static (operand images in this device's copy of the static array); shapes are checked by the callers.
int forward_launch(void* const* chunk_ptrs, int num_chunks, int rows_per_chunk, const void* x_bf16, int batch, float scale_w,
                   float scale_x, void* out_bf16, long long out_stride, long long num_labels, unsigned char* xq, hipStream_t stream) {
  if (!out_bf16) return XMC_ERR_NULL;
  if (num_labels <= 0 || out_stride < num_labels || num_labels > (long long)num_chunks * rows_per_chunk) return XMC_ERR_SHAPE;
  if (!(scale_w > 0.f) || !(scale_x > 0.f)) return XMC_ERR_SHAPE;
  DeviceInfo di = device_info();
  if (di.ok != 1) return XMC_ERR_DEVICE;
  const bool conv = forward_converts(batch, (num_labels + FT - 1) / FT, di.cus);
  if (!conv) prep_x(x_bf16, batch, scale_x, xq, stream);
  ForwardParams fp;
  for (int c = 0; c < MAX_CHUNKS; c++) fp.chunk[c] = c < num_chunks ? (const unsigned char*)chunk_ptrs[c] : nullptr;
  fp.rows_per_chunk = rows_per_chunk;
  fp.tiles_per_chunk = (rows_per_chunk + FT - 1) / FT;
  fp.x = (const unsigned short*)x_bf16;
  fp.inv_scale_x = 1.0f / scale_x;
  const int last_chunk = (int)((num_labels - 1) / rows_per_chunk);
  fp.tile_begin = 0;
  fp.tile_end = last_chunk * fp.tiles_per_chunk + (int)((num_labels - (long long)last_chunk * rows_per_chunk + FT - 1) / FT);
  fp.xq = xq;
  fp.zscale = scale_w * scale_x;
  fp.out = (unsigned short*)out_bf16;
  fp.out_stride = out_stride;
  fp.col0 = 0;
  fp.num_labels = num_labels;
  fp.batch = batch;
  // A tile is 64 bytes of every row of the output, half a cache line.  With tile after tile on another compute unit the halves are
  // written from different XCDs; runs of four tiles on one are written as whole lines.  us a call, runs of one / four,
  // 40 and 128 rows: 300 K labels 43.9/41.2 68.7/63.4, 400 K 71.4/70.3 95.9/90.1, 670 K 126/121 170/151, 1 M 192/182 285/254;  but 250 K
  // 37.8/35.4 51.0/52.0, 131 K 22.4/22.4 27.5/27.7, 128 rows, 50 K 16.8/17.2: from 32 tiles for each compute unit on.  With more rows by no rule: 256 rows, 400 K 116/126, 500 K 200/193, 800 K 222/244, 1 M 413/386.
  const bool runs = batch <= BP && fp.tile_end >= 32 * di.cus;
  const int grid = fp.tile_end < di.cus ? fp.tile_end : di.cus;   // one workgroup fills the LDS of a compute unit
  if (conv && runs) fp8_forward_kernel<1, 4, true><<<grid, FNT, FwdGeom<1, true>::LDS, stream>>>(fp);
  else if (conv) fp8_forward_kernel<1, 1, true><<<grid, FNT, FwdGeom<1, true>::LDS, stream>>>(fp);
  else if (batch > BP) fp8_forward_kernel<2, 1, false><<<grid, FNT, FwdGeom<2>::LDS, stream>>>(fp);
  else if (runs) fp8_forward_kernel<1, 4, false><<<grid, FNT, FwdGeom<1>::LDS, stream>>>(fp);
  else fp8_forward_kernel<1, 1, false><<<grid, FNT, FwdGeom<1>::LDS, stream>>>(fp);
  return launch_status();
}

// Whether a true-FP8 step of at most 64 batch rows takes the one-pass form in clusters of one (xmc_cluster.hip) rather than the
// fused kernel (xmc_fp8_role.hip).  The four workgroups of a quad share a tile and wait for one another; a cluster of one waits for
// nobody, but walks whole tiles of 64 labels, one per compute unit at a time, with a chain of its own latencies, and stores a grad_X
// sum per workgroup.  With round to nearest the tile's chain is short and the stream of weights bounds a long walk: one pass.  With
// sr_fast the update's vector work counts for more, and with Philox it is all that counts: the fused kernel's A and B wavefronts share
// it better.  us a step, fused / one pass, at 65 K, 131 K, 200 K, 300 K, 500 K, 1 M, 2 M labels:
//   32 rows, nearest  36/36  54/52  75/70  117/97   192/171  365/324  713/628    Philox  79/83  142/160  208/227  306/324  498/524  974/1021  1934/2014
//            sr_fast  35/39  52/59  72/81  107/109  189/189  362/353  714/689
//   64 rows, nearest  38/-   57/66  78/87  128/128  204/197  389/361  765/695    Philox  84/-   151/173  221/243  324/349  528/557  1034/1080 2041/2112
//            sr_fast  41/-   63/72  88/98  128/142  212/221  420/420  824/816
// (The weights are the same to the bit; grad_X's fp32 sum is grouped by 256 workgroups instead of 64 quads.)  The lines, in tiles of 64
// labels per compute unit: nearest 6 and 20 for 32 and 64 rows, sr_fast 32 and 64.
bool small_batch_one_pass(int batch, long long tiles, int round_mode, int cus) {
  if (batch > 64 || round_mode == XMC_ROUND_SR_PHILOX) return false;
  return tiles >= (round_mode == XMC_ROUND_RTN ? (batch <= 32 ? 6 : 20) : (batch <= 32 ? 32 : 64)) * (long long)cus;
}
// Clusters of the one-pass step for a step's tiles, of `most` that the device has.  Every workgroup leaves a sum of grad_X of 192 KiB (96 up to
// 32 rows), written and read again behind the kernel: with fewer tiles than clusters, but not by much, half as many clusters with two tiles
// each are faster, unless a second tile takes longer than the sums (Philox, FP8 logits in clusters of one).  us a step, a cluster for every
// tile / for two, at 2 K, 3 K, 4 K, 5 K, 6.5 K, 8 K labels:
//   (up to 64 rows with a launch in front that prepares X and the positives; without it both are 2 to 3 us less)
//   32 rows   bf16, nearest 18.5/20.2 20.2/20.6 21.4/21.7 23.7/22.8 26.8/23.7 28.3/24.2   sr_fast 22.4/23.1 (4 K) 24.6/24.2 27.6/25.4 28.8/25.8
//             e4m3 with bf16 products, nearest 17.4/18.5 19.5/19.4 21.0/20.1 22.4/21.0 24.3/22.1 27.2/23.1   Philox, either: 3 to 8 us slower
//   64 rows   bf16, nearest 22.4/23.4 26.4/25.1 29.3/26.1 31.6/28.0 32.8/30.6 32.7/31.2   sr_fast 22.9/25.0 27.2/26.8 30.4/27.5 31.7/29.4 32.8/32.4 33.1/33.2
//             e4m3 with bf16 products, nearest 22.2/22.8 25.4/24.4 28.0/25.4 31.7/27.3 33.3/29.0 34.6/31.0
//   128 rows  bf16, nearest 29.8/27.6 33.2/29.8 35.7/32.2   sr_fast 29.4/28.7 33.3/30.4 35.6/32.9   Philox 32.2/34.4 37.3/36.5 38.8/37.7
//             e4m3 with bf16 products, nearest 29.6/27.0 33.3/29.4 35.5/31.6   FP8 logits, sr_fast 25.6/26.7 and 33.1/31.0 (5 K)
//   256 rows  bf16, 1 K, 1.6 K, 2 K nearest 30.9/29.0 33.4/31.5 35.3/33.3   Philox 31.8/32.1 34.7/33.9 36.8/35.6
//             FP8 logits, 2 K, 4 K  nearest 31.2/29.6 36.1/34.5   sr_fast 31.2/30.4 36.4/35.0   Philox 33.8/35.6 39.2/40.0
// (Two tiles each of fewer clusters were measured for no more tiles than clusters, and in clusters of one, two and four: elsewhere as many
// clusters as there are, or as tiles.)
int one_pass_clusters(int tiles, int most, int c, int nbk, bool fp8, int round_mode) {
  if (tiles > most) return most;
  const bool philox = round_mode == XMC_ROUND_SR_PHILOX;
  bool two = false;   // tiles for a cluster
  if (c == 1) two = !philox && !fp8 && 16 * tiles > (nbk == 2 ? 9 : 5) * most;
  else if (c == 2 || c == 4) two = philox ? !fp8 && 4 * tiles >= 3 * most : 8 * tiles >= (c == 2 ? 3 : 4) * most;
  return two ? (tiles + 1) / 2 : tiles;
}
// Whether a true-FP8 step without weight decay, dropout or a compensated head takes the two launches of xmc_fp8_small.hip, a workgroup for
// every 32 labels and one to a compute unit at most.  What they gain is a launch and the latencies of the quads' exchange; what they lose
// grows with the labels, 48 KiB of grad_X sums per 16 batch rows and workgroup, and with Philox, whose words take a workgroup longer than
// the four of a quad.  us a step in replays of a graph, five positives a row, fused kernel / this one, at 1 K, 2 K, 4 K, 6 K, 8 K labels:
//   16 rows  sr_fast 12.7/8.9 13.2/9.9 14.4/12.1 15.6/14.1 16.1/16.0   nearest 12.4/8.7 13.1/9.6 14.2/11.7 15.2/13.8 15.7/15.7
//            Philox 15.5/14.4 16.2/15.4 17.3/17.6 21.4/19.9 21.9/21.4
//   32 rows  sr_fast 12.9/10.6 14.1/12.3 15.8/15.7 17.1/18.4 17.9/21.2   nearest 12.9/10.2 13.9/11.9 15.6/15.3 16.5/17.9 17.4/21.0
//            Philox 15.9/15.8 16.8/17.6 19.1/20.9 22.6/23.7 23.7/24.9
// Launched from the host it gains 1.1 to 1.4 more, a launch less: waited for alone, 32 rows, 5 K 32.1/31.5 (16.5/17.3 in a graph), Philox, 2 K 32.3/31.8,
// 6 K 38.0/37.5.  With more positives the launch that the fused kernel has in front takes longer: 5, 36, 128 a row, sr_fast, 16 rows, 4 K 14.4/12.1
// 14.9/12.2 15.6/12.7, 8 K 16.2/16.1 17.0/16.1 17.8/16.6, 32 rows, 1 K 12.9/10.6 13.5/10.9 17.1/11.8, 5 K 16.5/17.3 17.4/17.4 19.7/18.4, Philox, 2 K 16.8/17.6 17.6/17.9
// 20.4/18.8: at SM_POS, all that SM_BATCH rows have at 128 each, this form has gained.  (Eight pairs of a thread requested together instead of one
// behind the other: 32 rows, 128 a row 0.2 to 0.5 faster, 36 a row and 64 a row of 16 rows 0.1 to 0.5 slower.)
// (Workgroups that take several tiles one after the other, and sum: 8 K, 16 rows 15.9, 16 K 20.3/19.9 with the fused kernel, and half a
// microsecond more with one tile each.)
bool small_step(int batch, int nnz, long long tiles, int round_mode, int grid) {
  const long long most = batch <= 16 ? 256 : round_mode == XMC_ROUND_SR_PHILOX ? 64 : 160;
  return batch <= SM_BATCH && nnz <= SM_POS && tiles <= (most < grid ? most : grid);
}
// Quads of the fused kernel for a step's tiles, of `most` that the device has.  A quad leaves the sum of grad_X of all its tiles, 384 KiB at
// 128 rows, and one without tiles leaves as much: written, and read again behind the kernel.  With few tiles those sums cost more than a
// second tile for every quad, but where sums are short or tiles long: a quad for every tile with up to 48 rows or Philox up to half as many tiles
// as quads, with up to 16 rows (32 with decay, 96 with Philox) up to as many.  Whole numbers of quads on each XCD.  us a step, all quads / now, at 300, 1 K, 2 K, 4 K, 5 K labels:
//   sr_fast  48 rows 16.9/13.7 18.3/14.3 18.5/15.9 18.7/17.8 20.1/18.8     128 rows 26.0/16.4 27.9/19.5 28.3/21.6 28.6/25.5 29.1/27.4
//   Philox   64 rows 21.0/16.6 23.3/17.7 23.1/19.8 23.3/23.3 27.6/25.9     128 rows 26.8/19.2 30.1/21.6 31.5/25.7 32.1/30.9 34.4/32.6
// (Two tiles a quad instead of one: 2 K labels, 48 rows 16.0/16.4, Philox 128 rows 25.0/26.3, but 96 rows 19.4/18.7, 128 rows 22.3/20.9; 4 K, Philox,
// 64 rows 23.3/24.8; 16 rows, 2.6 K labels, dropout, sr_fast 15.6/16.0, more than SM_POS pairs 16.6/17.1, decay 17.2/18.4, 32 rows, 4 K, decay 19.0/19.5.  Three on 48 quads instead of 64, 9 K: 48 rows 22.2/21.2, but 128 rows 30.3/30.6: above two as many quads as there are.)
int fused_quads(int tiles, int batch, int round_mode, bool decay, int most) {
  if (tiles > 2 * most) return most;
  const bool philox = round_mode == XMC_ROUND_SR_PHILOX;
  const bool single = tiles <= most / 2 ? batch <= 48 || philox : tiles <= most && batch <= (philox ? 96 : decay ? 32 : 16);
  const int q = ((single ? tiles : (tiles + 1) / 2) + 7) / 8 * 8;
  return q < most ? q : most;
}
// The same for the launch of a compensated head, whose tiles take twice as long and whose sums are read and written once more, by the launch
// of the other tiles: a quad for a tile, from 65 tiles on as few as two each need.  us a step with a fifth of the labels compensated, bf16 terms,
// sr_fast, all quads in both launches / now, at 8 K, 11 K, 16 K labels: 128 rows 45.9/40.7 47.9/44.3 50.2/49.3, 32 rows 28.5/27.4 29.8/29.2 31.0/31.0;
// e5m2, nearest, 128 rows 45.0/39.8 47.1/43.4 49.4/48.2, 22 K 52.3/51.3, 30 K 55.8/54.8.
int head_quads(int tiles, int most) {
  if (tiles > 2 * most) return most;
  const int q = ((tiles <= most ? tiles : (tiles + 1) / 2) + 7) / 8 * 8;
  return q < most ? q : most;
}
// Its places in the fused step's workspace: the grad_X sums from WS_PARTIAL on (32 rows: as many bytes as the fused kernel's; 64 rows:
// twice that, over the exchange ring and the descriptors, which this form does not use, and up to 14 MiB beyond: only workspaces of
// xmc_workspace_bytes_ex hold them), then the first key of every tile.
constexpr size_t one_pass_partial(int batch) { return (size_t)CLU_MAXWG * CluGeom<CLU_E4M3, 1, 1, 2>::PSLOT * 16 * (batch <= 32 ? 1 : 2); }
size_t one_pass_end(int batch, size_t tiles) { return (WS_PARTIAL + one_pass_partial(batch) + (tiles + 1) * 4 + 255) / 256 * 256; }
static_assert(QF_WORDS - QF_CNT2 >= CLU_FLAG_INTS && WS_PARTIAL + one_pass_partial(32) <= WS_EXCH, "one-pass step in the fused step's workspace");

}  // namespace

extern "C" {

int xmc_version(void) { return 1; }

#ifndef XMC_SOURCE_HASH
#define XMC_SOURCE_HASH "unknown"
#endif
const char* xmc_source_hash(void) { return XMC_SOURCE_HASH; }

const char* xmc_error_string(int status) {
  switch (status) {
    case XMC_OK: return "ok";
    case XMC_ERR_NULL: return "null pointer";
    case XMC_ERR_SHAPE: return "unsupported shape: features (768, the tiled step also 1024), batch (up to 128, wide inference 256, the tiled step 512; a multiple of 16 "
                                "where the function says so), rows per chunk, labels or k";
    case XMC_ERR_ALIGN: return "device pointer not sufficiently aligned";
    case XMC_ERR_RANGE: return "too many chunks, labels or positives";
    case XMC_ERR_WORKSPACE: return "workspace too small";
    case XMC_ERR_MODE: return "unknown rounding mode";
    case XMC_ERR_LAUNCH: return "kernel launch failed";
    case XMC_ERR_DEVICE: return "current device is not a gfx950 GPU with at least 16 compute units";
    default: return "unknown status";
  }
}

size_t xmc_workspace_bytes(int num_chunks, int rows_per_chunk) {
  if (num_chunks <= 0 || num_chunks > MAX_CHUNKS || rows_per_chunk <= 0) return 0;
  size_t tiles = (size_t)num_chunks * ((rows_per_chunk + TL - 1) / TL);
  // 32-byte tile descriptors, one run per quad (up to MAX_WG / 4 runs, each rounded up to whole entries; two tables with a
  // compensated head)
  return WS_DESC + (tiles + MAX_WG / 2) * 32;
}

size_t xmc_workspace_bytes_ex(int num_chunks, int rows_per_chunk, int batch) {
  const size_t base = xmc_workspace_bytes(num_chunks, rows_per_chunk);
  if (base == 0) return 0;
  const size_t tiles = (size_t)num_chunks * ((rows_per_chunk + TL - 1) / TL);
  const size_t one = one_pass_end(batch, tiles);
  // (sizes that callers keep do not follow the lines of small_batch_one_pass, which lie above this one)
  return batch <= 64 && tiles >= 4 * (size_t)MAX_WG && one > base ? one : base;
}

int xmc_fp8_step(void* const* chunk_ptrs, int num_chunks, int rows_per_chunk, const void* x_bf16, int batch,
                 int features, const int32_t* labels_coo, int nnz, float lr, const uint32_t* seeds, int round_mode,
                 float scale_w, float scale_x, void* grad_x_bf16, float* grad_x_f32, void* workspace,
                 size_t workspace_bytes, void* stream_) {
  return xmc_fp8_step_ex(chunk_ptrs, num_chunks, rows_per_chunk, x_bf16, batch, features, labels_coo, nnz, lr, seeds, round_mode,
                         scale_w, scale_x, 0.0f, 0.0f, 0ull, grad_x_bf16, grad_x_f32, workspace, workspace_bytes, stream_);
}

}  // extern "C"

// The one-pass form of the step (xmc_cluster.hip): 768 features, no compensated head, no loss, no weight decay (options
// that would have to stay in its main loop, whose registers are full).  Within these it was faster than the three kernels at every size
// tried, from 2 K to 8.6 M labels and 1 to 512 batch rows; true FP8 of up to 128 rows has the fused kernel besides, and
// small_batch_one_pass decides.  The arguments have been checked by the caller.
static int cluster_step(void* const* chunk_ptrs, int num_chunks, int rows_per_chunk, int rows_last_chunk, int weight_type,
                        const void* x_bf16, int batch, const int32_t* labels_coo, int nnz, float lr, const uint32_t* seeds,
                        int round_mode, int quantize_x, int saturate, const DropoutParams& dp, void* grad_x_bf16, float* grad_x_f32,
                        const ClusterPlace& at, bool profiled, int cus, int* failure_word, hipStream_t stream) {
  const bool bf16 = weight_type == W_BF16, fp8 = !bf16 && quantize_x;
  const int c = cluster_members(batch, (long long)(num_chunks - 1) * rows_per_chunk + rows_last_chunk, fp8), nbk = cluster_blocks(batch), bp = c * 16 * nbk, pairs = (bp + 255) / 256;
  const int tile_rows = fp8 && c <= 4 ? 64 : 32;
  const int tpc64 = (rows_per_chunk + TL - 1) / TL;
  // a key keeps 24 bits for the label: larger label spaces are taken in segments of whole chunks
  int seg_chunks = ((1 << 24) - 2) / rows_per_chunk;
  if (seg_chunks > num_chunks) seg_chunks = num_chunks;
  if (seg_chunks < 1) return XMC_ERR_RANGE;
  const ClusterVariant var = bf16 ? cluster_variant_bf16(c, nbk, round_mode) : fp8 ? cluster_variant_fp8(c, nbk, round_mode) : cluster_variant_sim(c, nbk, round_mode);
  for (int c0 = 0; c0 < num_chunks; c0 += seg_chunks) {
    const int nch = c0 + seg_chunks <= num_chunks ? seg_chunks : num_chunks - c0;
    const bool last = c0 + nch == num_chunks;
    const int ptr_blocks = (nch * tpc64 + PREP_NT) / PREP_NT, prep_blocks = (bp * (D / 4) + PREP_NT - 1) / PREP_NT;
    const ClusterPrep pp = {labels_coo, nnz, batch, c0 * rows_per_chunk, nch * rows_per_chunk, pairs, rows_per_chunk, tpc64, nch * tpc64,
                            ptr_blocks, at.keys, at.tile_ptr, at.tp_stride, (const unsigned short*)x_bf16, bp, bf16 ? 0 : fp8 ? 2 : 1,
                            at.xq, at.xt, at.flags, c0 == 0 ? at.err : nullptr};   // (a failure in one segment stays visible behind the others)
    ClusterParams p;
    for (int k = 0; k < MAX_CHUNKS; k++) {
      p.chunk[k] = k < nch ? (unsigned char*)chunk_ptrs[c0 + k] : nullptr;
      p.seed[k] = k < nch && seeds ? (round_mode == XMC_ROUND_SR_FAST ? fast_seed(seeds[c0 + k]) : seeds[c0 + k]) : 0u;
    }
    p.nchunks = nch;
    p.rows_per_chunk = rows_per_chunk;
    p.rows_last = last ? rows_last_chunk : rows_per_chunk;
    p.tpc = (rows_per_chunk + tile_rows - 1) / tile_rows;
    p.tpc_last = (p.rows_last + tile_rows - 1) / tile_rows;
    p.perm = tile_stride(p.tpc);
    p.perm_last = tile_stride(p.tpc_last);
    p.tpc64 = tpc64;
    p.ntiles = (nch - 1) * p.tpc + p.tpc_last;
    const int most = (cus < CLU_MAXWG ? cus : CLU_MAXWG) / 8 / c * 8;   // whole clusters on every XCD
    p.nclusters = one_pass_clusters(p.ntiles, most, c, nbk, fp8, round_mode);
    p.label0_seg = 0u;
    p.label0 = (unsigned)c0 * (unsigned)rows_per_chunk;
    p.xq = at.xq;
    p.xt = (const bf16x8*)at.xt;
    for (int q = 0; q < 2; q++) {
      const int pr = q < pairs ? q : 0;
      p.keys[q] = at.keys + (size_t)pr * MAX_POS;
      p.tile_ptr[q] = at.tile_ptr + pr * at.tp_stride;
    }
    p.partial = at.partial;
    p.exch = at.exch;
    p.flags = at.flags;
    p.xcc = at.xcc;
    p.err = at.err;
    p.lr = lr;
    p.flush = bf16 ? 1 : 0;   // the reference rounds each chunk's sum where the weights are bf16
    p.saturate = saturate;
    p.spin_limit = g_spin_limit.load(std::memory_order_relaxed);
    p.loads_behind = clu_loads_behind((long long)p.ntiles * tile_rows * (D * 2));
    // Clusters of one with few positives prepare themselves (the products of a tile's number and an inverse are taken in 32 bits).  us a
    // step, prepared by a launch in front / by themselves: 32 rows, bf16, nearest 2 K labels 18.4/15.7, 8 K 24.4/21.8, 131 K 73.0/70.2, 500 K 332/330,
    // Philox, 2 K 24.2/21.4, 131 K 160.2/157.1; e4m3 with bf16 products, nearest, 2 K 17.8/15.2, 131 K 56.9/54.4; 64 rows, bf16, nearest, 2 K 22.2/20.6,
    // 131 K 84.9/83.1, e4m3, Philox, 8 K 37.1/36.0, 500 K 580/580.
    p.self = c == 1 && !fp8 && dp.p == 0.f && seg_chunks == num_chunks && nnz <= CLU_SELF_POS && p.tpc < 65536 &&
             p.ntiles / p.nclusters < CLU_SELF_TILES;
    p.nnz = nnz;
    p.batch = batch;
    p.perm_inv = tile_stride_inverse(p.perm, p.tpc);
    p.perm_inv_last = tile_stride_inverse(p.perm_last, p.tpc_last);
    p.coo = (const int2*)labels_coo;
    p.x = (const unsigned char*)x_bf16;
    if (!p.self) cluster_prep_kernel<<<ptr_blocks * pairs + prep_blocks, PREP_NT, (size_t)nnz * 4, stream>>>(pp, dp);
    if (profiled && g_prof_start) (void)hipEventRecord(g_prof_start, stream);
    var.fn<<<(p.nclusters + 7) / 8 * 8 * c, CLU_NT, var.lds, stream>>>(p);
    if (profiled) {
      if (g_prof_stop) (void)hipEventRecord(g_prof_stop, stream);
      g_prof_start = g_prof_stop = nullptr;
    }
    const ClusterReduce rd = {p.partial, c, nbk, p.nclusters, p.ntiles, p.tpc, nch, p.flush, at.xcc, at.err, at.sticky, failure_word, at.gx, c0 > 0 ? 1 : 0, last ? 1 : 0, batch,
                              (unsigned short*)grad_x_bf16, grad_x_f32};
    cluster_reduce_kernel<<<c * nbk * 6 * 8, CLU_RW * 64, 0, stream>>>(rd, dp);
  }
  return launch_status();
}

// The fused step behind xmc_fp8_step, xmc_fp8_step_ex and xmc_fp8_kahan_step.  kahan_type 0: no compensated head.
static int fused_step(void* const* chunk_ptrs, int num_chunks, int rows_per_chunk, const void* x_bf16, int batch,
                      int features, const int32_t* labels_coo, int nnz, float lr, const uint32_t* seeds, int round_mode,
                      float scale_w, float scale_x, float weight_decay, float dropout_p, unsigned long long dropout_seed,
                      void* kahan, int kahan_type, int num_head,
                      void* grad_x_bf16, float* grad_x_f32, void* workspace, size_t workspace_bytes, void* stream_) {
  int st = check_common(chunk_ptrs, num_chunks, rows_per_chunk, x_bf16, batch, features, workspace, workspace_bytes);
  if (st != XMC_OK) return st;
  // a key keeps 24 bits for the label (xmc_tiled_step takes larger label spaces in segments)
  if ((long long)num_chunks * rows_per_chunk >= (1LL << 24) - 1) return XMC_ERR_RANGE;
  if (!grad_x_bf16 || (nnz > 0 && !labels_coo)) return XMC_ERR_NULL;
  if (((uintptr_t)labels_coo & 7) != 0) return XMC_ERR_ALIGN;   // read as (row, label) pairs
  if (nnz < 0 || nnz > MAX_POS) return XMC_ERR_RANGE;
  if (round_mode < XMC_ROUND_RTN || round_mode > XMC_ROUND_SR_FAST) return XMC_ERR_MODE;
  if (round_mode != XMC_ROUND_RTN && !seeds) return XMC_ERR_NULL;
  if (!(scale_w > 0.f) || !(scale_x > 0.f)) return XMC_ERR_SHAPE;
  if (!(weight_decay >= 0.f) || !(dropout_p >= 0.f) || !(dropout_p < 1.f)) return XMC_ERR_SHAPE;
  if (kahan_type < 0 || kahan_type > 2) return XMC_ERR_MODE;
  if (kahan_type != 0) {
    if (!kahan) return XMC_ERR_NULL;
    if (!aligned16(kahan)) return XMC_ERR_ALIGN;
    if (num_head <= 0 || num_head > rows_per_chunk) return XMC_ERR_SHAPE;
  } else {
    num_head = 0;
  }
  DeviceInfo di = device_info();
  if (di.ok != 1 || di.cus < 16) return XMC_ERR_DEVICE;
  hipStream_t stream = (hipStream_t)stream_;
  unsigned char* ws = (unsigned char*)workspace;
  const DropoutParams dp = {dropout_p, 1.0f - dropout_p, (unsigned)(dropout_seed & 0xFFFFFFFFull), (unsigned)(dropout_seed >> 32)};

  const int grid = di.cus < MAX_WG ? di.cus : MAX_WG;   // one workgroup per compute unit
  const int tiles_per_chunk = (rows_per_chunk + TL - 1) / TL;
  const int num_tiles = num_chunks * tiles_per_chunk;

  // (the one-pass form has neither scales nor decay; a workspace that does not hold its sums keeps the fused kernel)
  if (kahan_type == 0 && weight_decay == 0.f && scale_w == 1.f && scale_x == 1.f && small_batch_one_pass(batch, num_tiles, round_mode, di.cus) &&
      workspace_bytes >= one_pass_end(batch, (size_t)num_tiles)) {
    int* flags = (int*)(ws + WS_FLAGS);
    const ClusterPlace at = {ws + WS_XQ, (unsigned short*)(ws + WS_XT), (unsigned*)(ws + WS_KEYS), flags + QF_CNT2, flags + QF_XCC, nullptr,
                             (int*)(ws + WS_PARTIAL + one_pass_partial(batch)), 0, nullptr, (floatx4*)(ws + WS_PARTIAL), flags + QF_ERR, flags + QF_STICKY};
    return cluster_step(chunk_ptrs, num_chunks, rows_per_chunk, rows_per_chunk, W_E4M3, x_bf16, batch, labels_coo, nnz, lr, seeds, round_mode, 1, 1,
                        dp, grad_x_bf16, grad_x_f32, at, true, di.cus, di.failure_word, stream);
  }
  const int qgrid = grid / 32 * 32;   // whole quads on every XCD
  if (qgrid < 32) return XMC_ERR_DEVICE;
  const int small_per_chunk = (rows_per_chunk + SM_ROWS - 1) / SM_ROWS;
  if (kahan_type == 0 && weight_decay == 0.f && dropout_p == 0.f &&
      small_step(batch, nnz, (long long)num_chunks * small_per_chunk, round_mode, qgrid)) {
    SmallParams p;
    for (int c = 0; c < MAX_CHUNKS; c++) {
      p.chunk[c] = c < num_chunks ? (unsigned char*)chunk_ptrs[c] : nullptr;
      p.seed[c] = (c < num_chunks && seeds) ? (round_mode == XMC_ROUND_SR_FAST ? fast_seed(seeds[c]) : seeds[c]) : 0u;
    }
    p.rows_per_chunk = rows_per_chunk;
    p.tiles_per_chunk = small_per_chunk;
    p.num_tiles = num_chunks * small_per_chunk;
    p.x = (const unsigned short*)x_bf16;
    p.coo = (const int2*)labels_coo;
    p.nnz = nnz;
    p.batch = batch;
    p.inv_scale_x = 1.0f / scale_x;
    p.zscale = scale_w * scale_x;
    p.lr_eff = lr / scale_w;
    p.partial = (floatx4*)(ws + WS_PARTIAL);
    p.flags = (int*)(ws + WS_FLAGS);
    static_assert((size_t)MAX_WG * SM_BATCH * D * 4 <= WS_EXCH - WS_PARTIAL, "grad_X sums of a workgroup for every compute unit");
    if (g_prof_start) (void)hipEventRecord(g_prof_start, stream);
    // (as many workgroups as the fused kernel has: all of them record their XCD)
    small_variant(round_mode, batch)<<<qgrid, SM_NT, SM_LDS, stream>>>(p);
    if (g_prof_stop) (void)hipEventRecord(g_prof_stop, stream);
    g_prof_start = g_prof_stop = nullptr;
    const int blocks = batch / 16 * 48;
    fp8_small_reduce_kernel<<<blocks, SM_RW * 64, 0, stream>>>(p.partial, p.num_tiles, blocks, scale_w, grad_x_f32, (unsigned short*)grad_x_bf16,
                                                               p.flags, di.failure_word);
    return launch_status();
  }
  {
    QuadParams p;
    for (int c = 0; c < MAX_CHUNKS; c++) {
      p.chunk[c] = c < num_chunks ? (unsigned char*)chunk_ptrs[c] : nullptr;
      p.seed[c] = (c < num_chunks && seeds) ? (round_mode == XMC_ROUND_SR_FAST ? fast_seed(seeds[c]) : seeds[c]) : 0u;
    }
    p.num_chunks = num_chunks;
    p.rows_per_chunk = rows_per_chunk;
    p.tiles_per_chunk = tiles_per_chunk;
    p.num_tiles = num_tiles;
    p.run_tiles = num_tiles;
    p.xq = ws + WS_XQ;
    p.xt = (const bf16x8*)(ws + WS_XT);
    p.keys = (const unsigned*)(ws + WS_KEYS);
    p.partial = (floatx4*)(ws + WS_PARTIAL);
    p.exch = ws + WS_EXCH;
    uint4* desc = (uint4*)(ws + WS_DESC);
    p.desc = desc;
    p.flags = (int*)(ws + WS_FLAGS);
    p.zscale = scale_w * scale_x;
    p.lr_eff = lr / scale_w;
    p.wd_eff = weight_decay * scale_w;   // T = c - (lr / s) (A + wd s c) for codes c = W / s
    p.batch = batch;
    // with a compensated head the tiles that hold its rows run first, as a launch of their own
    const int head_tiles = (num_head + TL - 1) / TL, rest_tiles = num_tiles - head_tiles;
    // (their quads' sums are continued by the quads of the other launch: at least as many)
    p.nquads_head = head_quads(head_tiles, qgrid >> 2);
    const int rest_quads = fused_quads(rest_tiles, batch, round_mode, weight_decay != 0.f, qgrid >> 2);
    p.nquads = rest_quads > p.nquads_head ? rest_quads : p.nquads_head;
    p.kahan = (unsigned char*)kahan;
    p.num_head = num_head;
    p.head_tiles = head_tiles;
    p.kmax_head = head_tiles > 0 ? (head_tiles + p.nquads_head - 1) / p.nquads_head : 0;
    p.kmax = (rest_tiles + p.nquads - 1) / p.nquads;
    p.cnt_base = 0;
    p.acc_quads = 0;
    p.spin_limit = g_spin_limit.load(std::memory_order_relaxed);
    const int desc_blocks = (num_tiles + PREP_NT - 1) / PREP_NT;
    quad_prep_kernel<<<desc_blocks + (BP * (D / 4) + PREP_NT - 1) / PREP_NT, PREP_NT, (size_t)nnz * 4, stream>>>(
        p, labels_coo, nnz, (unsigned*)(ws + WS_KEYS), desc, desc_blocks, (const unsigned short*)x_bf16, 1.0f / scale_x,
        ws + WS_XQ, (unsigned short*)(ws + WS_XT), dp);
    if (g_prof_start) (void)hipEventRecord(g_prof_start, stream);
    QuadParams ph = p;   // the head's launch
    ph.run_tiles = head_tiles;
    ph.kmax = p.kmax_head;
    p.run_tiles = rest_tiles;
    p.desc = desc + 2 * (size_t)p.nquads_head * p.kmax_head;
    if (head_tiles > 0) { p.cnt_base = QF_CNT2; p.acc_quads = p.nquads_head; }
    // the variants with the Philox recipe or a compensated head live in the library's second translation unit
    if (kahan_type != 0) role_heavy_launch(round_mode, false, kahan_type, role_blocks(batch, false, kahan_type), 4 * p.nquads_head, stream, ph);
    if (rest_tiles > 0) {
      const bool wd = weight_decay != 0.f;
      const int blocks = role_blocks(batch, wd, 0);
      if (round_mode == XMC_ROUND_SR_PHILOX) role_heavy_launch(round_mode, wd, 0, blocks, 4 * p.nquads, stream, p);
      else role_plain_launch(round_mode, wd, blocks, 4 * p.nquads, stream, p);
    }
    if (g_prof_stop) (void)hipEventRecord(g_prof_stop, stream);
    g_prof_start = g_prof_stop = nullptr;
    reduce_gx_role_kernel<<<(batch + 15) / 16 * 48, 256, 0, stream>>>((const floatx4*)(ws + WS_PARTIAL), 4 * p.nquads, scale_w, grad_x_f32,
                                                 (unsigned short*)grad_x_bf16, batch, (int*)(ws + WS_FLAGS), di.failure_word, dp);
  }
  return launch_status();
}

extern "C" {

int xmc_fp8_step_ex(void* const* chunk_ptrs, int num_chunks, int rows_per_chunk, const void* x_bf16, int batch,
                    int features, const int32_t* labels_coo, int nnz, float lr, const uint32_t* seeds, int round_mode,
                    float scale_w, float scale_x, float weight_decay, float dropout_p, unsigned long long dropout_seed,
                    void* grad_x_bf16, float* grad_x_f32, void* workspace, size_t workspace_bytes, void* stream_) {
  return fused_step(chunk_ptrs, num_chunks, rows_per_chunk, x_bf16, batch, features, labels_coo, nnz, lr, seeds, round_mode,
                    scale_w, scale_x, weight_decay, dropout_p, dropout_seed, nullptr, 0, 0, grad_x_bf16, grad_x_f32, workspace,
                    workspace_bytes, stream_);
}

int xmc_fp8_kahan_step(void* const* chunk_ptrs, int num_chunks, int rows_per_chunk, const void* x_bf16, int batch,
                       int features, const int32_t* labels_coo, int nnz, float lr, const uint32_t* seeds, int round_mode,
                       void* kahan, int kahan_type, int num_head, void* grad_x_bf16, float* grad_x_f32, void* workspace,
                       size_t workspace_bytes, void* stream_) {
  if (kahan_type != 1 && kahan_type != 2) return XMC_ERR_MODE;
  return fused_step(chunk_ptrs, num_chunks, rows_per_chunk, x_bf16, batch, features, labels_coo, nnz, lr, seeds, round_mode,
                    1.0f, 1.0f, 0.0f, 0.0f, 0ull, kahan, kahan_type, num_head, grad_x_bf16, grad_x_f32, workspace,
                    workspace_bytes, stream_);
}

static int forward_checked(void* const* chunk_ptrs, int num_chunks, int rows_per_chunk, const void* x_bf16, int batch, int features,
                           float scale_w, float scale_x, void* out_bf16, long long out_stride, long long num_labels, void* workspace,
                           size_t workspace_bytes, void* stream_, int batch_unit, int most_rows = BP) {
  int st = check_common(chunk_ptrs, num_chunks, rows_per_chunk, x_bf16, batch, features, workspace, workspace_bytes, batch_unit, most_rows);
  if (st != XMC_OK) return st;
  // (the operand image of more than 128 rows goes on where a step keeps X^T)
  static_assert((size_t)FWD_ROWS * D <= WS_KEYS - WS_XQ, "operand image of X in the workspace");
  return forward_launch(chunk_ptrs, num_chunks, rows_per_chunk, x_bf16, batch, scale_w, scale_x, out_bf16, out_stride,
                        num_labels, (unsigned char*)workspace + WS_XQ, (hipStream_t)stream_);
}

int xmc_fp8_forward(void* const* chunk_ptrs, int num_chunks, int rows_per_chunk, const void* x_bf16, int batch,
                    int features, float scale_w, float scale_x, void* out_bf16, long long out_stride,
                    long long num_labels, void* workspace, size_t workspace_bytes, void* stream_) {
  return forward_checked(chunk_ptrs, num_chunks, rows_per_chunk, x_bf16, batch, features, scale_w, scale_x, out_bf16, out_stride,
                         num_labels, workspace, workspace_bytes, stream_, 16);
}

int xmc_fp8_forward_rows(void* const* chunk_ptrs, int num_chunks, int rows_per_chunk, const void* x_bf16, int batch,
                         int features, float scale_w, float scale_x, void* out_bf16, long long out_stride,
                         long long num_labels, void* workspace, size_t workspace_bytes, void* stream_) {
  return forward_checked(chunk_ptrs, num_chunks, rows_per_chunk, x_bf16, batch, features, scale_w, scale_x, out_bf16, out_stride,
                         num_labels, workspace, workspace_bytes, stream_, 1);
}

int xmc_fp8_forward_wide(void* const* chunk_ptrs, int num_chunks, int rows_per_chunk, const void* x_bf16, int batch,
                         int features, float scale_w, float scale_x, void* out_bf16, long long out_stride,
                         long long num_labels, void* workspace, size_t workspace_bytes, void* stream_) {
  return forward_checked(chunk_ptrs, num_chunks, rows_per_chunk, x_bf16, batch, features, scale_w, scale_x, out_bf16, out_stride,
                         num_labels, workspace, workspace_bytes, stream_, 1, FWD_ROWS);
}

int xmc_fp8_forward_static(void* const* chunk_ptrs, int num_chunks, int rows_per_chunk, const void* x_bf16, int batch,
                           int features, float scale_w, float scale_x, void* out_bf16, long long out_stride,
                           long long num_labels, void* stream_) {
  // the same checks as xmc_fp8_forward, without a workspace; the static array holds the operand image of at most
  // BP = 128 batch rows of D = 768 features, which is also the limit of xmc_fp8_forward
  if (!chunk_ptrs || !x_bf16) return XMC_ERR_NULL;
  if (features != D || batch <= 0 || batch > BP || batch % 16 != 0) return XMC_ERR_SHAPE;
  if (rows_per_chunk <= 0 || rows_per_chunk % 16 != 0) return XMC_ERR_SHAPE;
  if (num_chunks <= 0 || num_chunks > MAX_CHUNKS) return XMC_ERR_RANGE;
  if ((long long)num_chunks * rows_per_chunk > 0x7FFFFFFFLL) return XMC_ERR_RANGE;
  for (int c = 0; c < num_chunks; c++) {
    if (!chunk_ptrs[c]) return XMC_ERR_NULL;
    if (!aligned16(chunk_ptrs[c])) return XMC_ERR_ALIGN;
  }
  if (!aligned16(x_bf16)) return XMC_ERR_ALIGN;
  const DeviceInfo di = device_info();
  if (di.ok != 1 || !di.scratch_ptr) return XMC_ERR_DEVICE;
  return forward_launch(chunk_ptrs, num_chunks, rows_per_chunk, x_bf16, batch, scale_w, scale_x, out_bf16, out_stride,
                        num_labels, di.scratch_ptr, (hipStream_t)stream_);
}

size_t xmc_topk_scratch_bytes(int rows_per_chunk) {
  if (rows_per_chunk <= 0 || rows_per_chunk % 16 != 0) return 0;
  // logits of one group of chunks [128][group * rows] bf16, then the running lists, two per batch row: values
  // [128][2][128] bf16, label ids [128][2][128] int32
  return topk_zbuf_bytes(rows_per_chunk) + 2 * ((size_t)BP * TOPK_MAX * 2 + (size_t)BP * TOPK_MAX * 4);
}

int xmc_fp8_forward_topk(void* const* chunk_ptrs, int num_chunks, int rows_per_chunk, const void* x_bf16, int batch,
                         int features, float scale_w, float scale_x, long long num_labels, int k, void* out_val_bf16,
                         int32_t* out_idx, void* workspace, size_t workspace_bytes, void* scratch, size_t scratch_bytes,
                         void* stream_) {
  int st = check_common(chunk_ptrs, num_chunks, rows_per_chunk, x_bf16, batch, features, workspace, workspace_bytes);
  if (st != XMC_OK) return st;
  if (!out_val_bf16 || !out_idx || !scratch) return XMC_ERR_NULL;
  if (((uintptr_t)scratch & 255) != 0) return XMC_ERR_ALIGN;
  if (scratch_bytes < xmc_topk_scratch_bytes(rows_per_chunk)) return XMC_ERR_WORKSPACE;
  if (num_labels <= 0 || num_labels > (long long)num_chunks * rows_per_chunk) return XMC_ERR_SHAPE;
  if (k <= 0 || k > TOPK_MAX || k > num_labels) return XMC_ERR_SHAPE;
  if (!(scale_w > 0.f) || !(scale_x > 0.f)) return XMC_ERR_SHAPE;
  DeviceInfo di = device_info();
  if (di.ok != 1) return XMC_ERR_DEVICE;
  hipStream_t stream = (hipStream_t)stream_;
  unsigned char* xq = (unsigned char*)workspace + WS_XQ;
  unsigned short* zbuf = (unsigned short*)scratch;
  unsigned short* run_val = (unsigned short*)((unsigned char*)scratch + topk_zbuf_bytes(rows_per_chunk));
  int* run_idx = (int*)(run_val + (size_t)BP * 2 * TOPK_MAX);
  prep_x(x_bf16, batch, scale_x, xq, stream);
  ForwardParams fp;
  for (int c = 0; c < MAX_CHUNKS; c++) fp.chunk[c] = c < num_chunks ? (const unsigned char*)chunk_ptrs[c] : nullptr;
  fp.rows_per_chunk = rows_per_chunk;
  fp.tiles_per_chunk = (rows_per_chunk + FT - 1) / FT;
  fp.xq = xq;
  fp.zscale = scale_w * scale_x;
  const int group = topk_group(rows_per_chunk);
  const long long seg_rows = topk_segment_rows(rows_per_chunk);
  fp.out = zbuf;
  fp.out_stride = seg_rows;
  fp.num_labels = num_labels;
  fp.batch = batch;
  // Every batch row keeps two lists.  Large segments are split between two workgroups per row (one list each), so that
  // 128 rows occupy all compute units; small ones go to list 0.  A list without k entries yet is first given a short
  // piece (4,096 logits, which fit the workgroup's candidate store): that leaves k entries whose smallest value bounds
  // the rest.
  int have[2] = {0, 0};
  auto select = [&](const unsigned short* zp, int n, int base, int parts) {
    topk_chunk_kernel<<<batch * parts, TOPK_NT, 0, stream>>>(zp, seg_rows, n, base, k, parts, have[0], have[1], run_val, run_idx);
    const int n0 = parts == 2 ? topk_split(n) : n;
    have[0] = have[0] + n0 < k ? have[0] + n0 : k;
    have[1] = have[1] + (n - n0) < k ? have[1] + (n - n0) : k;
  };
  // one segment: the logits of tiles [tile_begin, tile_end) into the scratch buffer, then their n labels from `base` on
  auto segment = [&](int tile_begin, int tile_end, long long base, int n) {
    fp.tile_begin = tile_begin;
    fp.tile_end = tile_end;
    fp.col0 = base;
    const int tiles = tile_end - tile_begin;
    fp8_forward_kernel<1, 1, false><<<tiles < di.cus ? tiles : di.cus, FNT, FwdGeom<1>::LDS, stream>>>(fp);
    int done = 0;
    if (n > 32768) {          // two workgroups per row
      if (have[0] < k || have[1] < k) {
        done = 8192;
        select(zbuf, done, (int)base, 2);
      }
      select(zbuf + done, n - done, (int)base + done, 2);
    } else {
      if (have[0] < k && n > 8192) {
        done = 4096;
        select(zbuf, done, (int)base, 1);
      }
      select(zbuf + done, n - done, (int)base + done, 1);
    }
  };
  if (rows_per_chunk <= TOPK_SEG) {
    for (int c = 0; c < num_chunks; c += group) {
      const long long base = (long long)c * rows_per_chunk;
      if (base >= num_labels) break;
      const int n = (int)(num_labels - base < seg_rows ? num_labels - base : seg_rows);     // padding rows are dropped
      const int full = n / rows_per_chunk, rest = n - full * rows_per_chunk;                // whole chunks, rows of the last one
      segment(c * fp.tiles_per_chunk, c * fp.tiles_per_chunk + full * fp.tiles_per_chunk + (rest + FT - 1) / FT, base, n);
    }
  } else {
    for (int c = 0; c < num_chunks; c++)
      for (int r0 = 0; r0 < rows_per_chunk; r0 += TOPK_SEG) {       // TOPK_SEG is a multiple of the tile height
        const long long base = (long long)c * rows_per_chunk + r0;
        if (base >= num_labels) break;
        long long n = rows_per_chunk - r0 < TOPK_SEG ? rows_per_chunk - r0 : TOPK_SEG;
        if (n > num_labels - base) n = num_labels - base;
        segment(c * fp.tiles_per_chunk + r0 / FT, c * fp.tiles_per_chunk + r0 / FT + (int)((n + FT - 1) / FT), base, (int)n);
      }
  }
  topk_finish_kernel<<<batch, 2 * TOPK_MAX, 0, stream>>>(run_val, run_idx, k, have[0], have[1], (unsigned short*)out_val_bf16, out_idx);
  return launch_status();
}

// scratch of xmc_fp8_forward_topk_fused: group maxima and bounds (the size callers keep is that of the time when the candidates, 1,024 a
// row, were in it too); and the candidates and the lists of topk_repair, in a part of the workspace that inference has no other use for
constexpr size_t SELS_GMAX = 0;
constexpr size_t SELS_BOUND = SELS_GMAX + (size_t)SEL_GROUPS * SEL_ROWS * 2;
constexpr size_t SELS_BYTES = (size_t)SEL_GROUPS * BP * 2 + 256 + (size_t)BP * 4 + (size_t)BP * 1024 * 6;
constexpr size_t SELW_LABEL = WS_PARTIAL;
constexpr size_t SELW_KEY = SELW_LABEL + (size_t)SEL_ROWS * SEL_CAP * 4;
constexpr size_t SELW_LISTS = SELW_KEY + (size_t)SEL_ROWS * SEL_CAP * 2;
constexpr size_t SELW_COUNT = WS_XQ + (size_t)SEL_ROWS * D;   // (behind the operand image of X)
static_assert(SELW_LISTS + REP_BYTES <= WS_DESC && SELS_BOUND + (size_t)SEL_ROWS * 2 <= SELS_BYTES, "top-k lists in the workspace");
static_assert(SELW_COUNT + (size_t)(SEL_ROWS + SEL_ROWS / 32) * SEL_COUNT_STRIDE * 4 <= WS_KEYS && SEL_GROUPS == TOPK_GROUPS, "the top-k kernels share these sizes");

size_t xmc_topk_fused_scratch_bytes(void) { return SELS_BYTES; }

// Pass 1 visits one tile in `step`: the k-th largest of the group maxima of such a sample leaves about k * step candidates per row, which
// have to stay well below the list size; at least four groups per wanted entry.  What a shorter pass 1 gains, pass 2 loses on candidates:
// more than 512 of them pay from about 3/2 k step^2 tiles on (the time is as c tiles / step + d k step), or in the form for more than
// 128 rows, whose pass 2 has twice the rows behind every tile.  us a call, at most 512 / at most 1,024 candidates:
//   128 rows  k = 40 (step 8 / 16)  90 K labels 38.5/43.8  131 K 42.6/47.9  262 K 58.5/59.8  400 K 77.0/79.1  670 K 119/116  1 M 173/163
//             k = 64 (step 8 / 16)            -            131 K 45.6/56.3  262 K 60.5/68.6  400 K 78.9/84.4  670 K 118/121  1 M 172/169
//             k = 100 (step 4 / 8)            -            131 K 45.8/52.9  262 K 64.2/67.1  400 K 83.7/86.4  670 K 126/122  1 M 189/173
//   8 rows    k = 100                                      131 K 40.7/44.0  262 K 58.7/60.8  400 K 78.7/75.3  670 K 123/117  1 M 182/168
//   256 rows  k = 40                 90 K 55.4/54.5        131 K 65.2/64.2  262 K 94.7/92.1  400 K 129/128    670 K 191/191  1 M 263/266
//             k = 100                                      131 K 71.1/73.0  262 K 104/102    400 K 141/138    670 K 211/204  1 M 295/282
// (2,048 candidates, lists of 4,096: 670 K labels, 128 rows, k = 100 135 us, 131 with 1,024.)
static int topk_fused_step(int tiles, int k, bool wide) {
  auto fits = [&](int step) {
    return tiles / step >= 4 * k && (k * step <= SEL_CAP / 4 || (k * step <= SEL_CAP / 2 && (wide || 2 * tiles >= 3 * k * step * step)));
  };
  int step = 16;
  while (step > 1 && !fits(step)) step >>= 1;
  return fits(step) ? step : 0;
}

static int topk_fused(void* const* chunk_ptrs, int num_chunks, int rows_per_chunk, const void* x_bf16, int batch, int features,
                      float scale_w, float scale_x, long long num_labels, int k, void* out_val_bf16, void* out_idx, int idx_int64,
                      void* workspace, size_t workspace_bytes, void* scratch, size_t scratch_bytes, int32_t* status, void* stream_,
                      int batch_unit, bool repair, int most_rows = BP) {
  int st = check_common(chunk_ptrs, num_chunks, rows_per_chunk, x_bf16, batch, features, workspace, workspace_bytes, batch_unit, most_rows);
  if (st != XMC_OK) return st;
  if (!out_val_bf16 || !out_idx || !scratch || !status) return XMC_ERR_NULL;
  if (((uintptr_t)scratch & 255) != 0 || ((uintptr_t)status & 3) != 0 || ((uintptr_t)out_idx & (idx_int64 ? 7 : 3)) != 0) return XMC_ERR_ALIGN;
  if (scratch_bytes < SELS_BYTES) return XMC_ERR_WORKSPACE;
  if (num_labels <= 0 || num_labels > (long long)num_chunks * rows_per_chunk) return XMC_ERR_SHAPE;
  if (k <= 0 || k > TOPK_MAX || k > num_labels) return XMC_ERR_SHAPE;
  if (!(scale_w > 0.f) || !(scale_x > 0.f)) return XMC_ERR_SHAPE;
  SelectParams sp;
  sp.rows_per_chunk = rows_per_chunk;
  sp.tiles_per_chunk = (rows_per_chunk + FT - 1) / FT;
  const int last_chunk = (int)((num_labels - 1) / rows_per_chunk);
  const int tiles = last_chunk * sp.tiles_per_chunk + (int)((num_labels - (long long)last_chunk * rows_per_chunk + FT - 1) / FT);
  const bool wide = batch > BP;
  const int step = topk_fused_step(tiles, k, wide);
  if (step == 0) return XMC_ERR_RANGE;   // too few labels for a useful bound: xmc_fp8_forward_topk takes these
  DeviceInfo di = device_info();
  if (di.ok != 1) return XMC_ERR_DEVICE;
  hipStream_t stream = (hipStream_t)stream_;
  unsigned char* xq = (unsigned char*)workspace + WS_XQ;
  unsigned char* sc = (unsigned char*)scratch;
  prep_x(x_bf16, batch, scale_x, xq, stream);
  for (int c = 0; c < MAX_CHUNKS; c++) sp.chunk[c] = c < num_chunks ? (const unsigned char*)chunk_ptrs[c] : nullptr;
  sp.xq = xq;
  sp.zscale = scale_w * scale_x;
  sp.num_labels = num_labels;
  sp.batch = batch;
  sp.gmax = (unsigned short*)(sc + SELS_GMAX);
  sp.bound = (const unsigned short*)(sc + SELS_BOUND);
  // (the counters lie a cache line apart, in a part of the workspace that inference has no other use for)
  sp.count = (unsigned*)((unsigned char*)workspace + SELW_COUNT);
  sp.cand_label = (unsigned*)((unsigned char*)workspace + SELW_LABEL);
  sp.cand_key = (unsigned short*)((unsigned char*)workspace + SELW_KEY);
  // pass 1: the sampled tiles, one group of them per workgroup
  sp.tile_step = step;
  sp.n_visit = (tiles + step - 1) / step;
  // (a workgroup to a compute unit, or two: with more, the last ones would start when the first ones are done)
  const int most = wide && di.cus < SEL_GROUPS && di.cus >= 2 * k ? di.cus : SEL_GROUPS;
  const int groups = sp.n_visit < most ? sp.n_visit : most;
  if (wide) fp8_forward_select_kernel<0, 8><<<groups, 512, SelGeom<8>::LDS, stream>>>(sp);
  else fp8_forward_select_kernel<0, 4><<<groups, 256, SelGeom<4>::LDS, stream>>>(sp);
  topk_bound_kernel<<<wide ? SEL_ROWS : BP, TOPK_GROUPS, 0, stream>>>(sp.gmax, groups, k, batch, (unsigned short*)(sc + SELS_BOUND), sp.count, status);
  // pass 2: every tile
  sp.tile_step = 1;
  sp.n_visit = tiles;
  if (wide) fp8_forward_select_kernel<1, 8><<<tiles < di.cus ? tiles : di.cus, 512, SelGeom<8>::LDS, stream>>>(sp);
  else fp8_forward_select_kernel<1, 4><<<tiles < 2 * di.cus ? tiles : 2 * di.cus, 256, SelGeom<4>::LDS, stream>>>(sp);
  const int repairers = repair ? rep_blocks(batch) : 0;
  topk_pick_kernel<<<batch + repairers, REP_NT, repair ? REP_LDS : PICK_LDS, stream>>>(
      sp, k, (unsigned short*)out_val_bf16, out_idx, idx_int64 ? 1 : 0, status,
      repair ? (unsigned long long*)((unsigned char*)workspace + SELW_LISTS) : nullptr);
  return launch_status();
}

int xmc_fp8_forward_topk_fused(void* const* chunk_ptrs, int num_chunks, int rows_per_chunk, const void* x_bf16, int batch,
                               int features, float scale_w, float scale_x, long long num_labels, int k, void* out_val_bf16,
                               void* out_idx, int idx_int64, void* workspace, size_t workspace_bytes, void* scratch,
                               size_t scratch_bytes, int32_t* status, void* stream_) {
  return topk_fused(chunk_ptrs, num_chunks, rows_per_chunk, x_bf16, batch, features, scale_w, scale_x, num_labels, k, out_val_bf16,
                    out_idx, idx_int64, workspace, workspace_bytes, scratch, scratch_bytes, status, stream_, 16, false);
}

int xmc_fp8_forward_topk_fused_rows(void* const* chunk_ptrs, int num_chunks, int rows_per_chunk, const void* x_bf16, int batch,
                               int features, float scale_w, float scale_x, long long num_labels, int k, void* out_val_bf16,
                               void* out_idx, int idx_int64, void* workspace, size_t workspace_bytes, void* scratch,
                               size_t scratch_bytes, int32_t* status, void* stream_) {
  return topk_fused(chunk_ptrs, num_chunks, rows_per_chunk, x_bf16, batch, features, scale_w, scale_x, num_labels, k, out_val_bf16,
                    out_idx, idx_int64, workspace, workspace_bytes, scratch, scratch_bytes, status, stream_, 1, false);
}

int xmc_fp8_forward_topk_wide(void* const* chunk_ptrs, int num_chunks, int rows_per_chunk, const void* x_bf16, int batch,
                              int features, float scale_w, float scale_x, long long num_labels, int k, void* out_val_bf16,
                              void* out_idx, int idx_int64, void* workspace, size_t workspace_bytes, void* scratch,
                              size_t scratch_bytes, int32_t* status, void* stream_) {
  return topk_fused(chunk_ptrs, num_chunks, rows_per_chunk, x_bf16, batch, features, scale_w, scale_x, num_labels, k, out_val_bf16,
                    out_idx, idx_int64, workspace, workspace_bytes, scratch, scratch_bytes, status, stream_, 1, true, SEL_ROWS);
}

int xmc_dropout_quantize(const void* x, int x_type, int rows, int cols, float p, unsigned long long seed, void* out_e4m3,
                         void* stream_) {
  if (!x || !out_e4m3) return XMC_ERR_NULL;
  if (x_type != 0 && x_type != 1) return XMC_ERR_MODE;
  if (rows <= 0 || cols <= 0 || cols % 4 != 0 || !(p >= 0.f) || !(p < 1.f)) return XMC_ERR_SHAPE;
  if ((long long)rows * cols > 0x7FFFFFFFll) return XMC_ERR_RANGE;   // the random offsets are 32-bit element indices
  if (((uintptr_t)x & (x_type == 0 ? 7 : 3)) != 0 || ((uintptr_t)out_e4m3 & 3) != 0) return XMC_ERR_ALIGN;
  DeviceInfo di = device_info();
  if (di.ok != 1) return XMC_ERR_DEVICE;
  const long long n4 = (long long)rows * cols / 4;
  dropout_quantize_kernel<<<(unsigned)((n4 + 255) / 256), 256, 0, (hipStream_t)stream_>>>(x, x_type, n4, cols, p, (unsigned)(seed & 0xFFFFFFFFull),
                                                                                        (unsigned)(seed >> 32), (unsigned*)out_e4m3);
  return launch_status();
}

int xmc_debug_spin_limit(int limit) {
  return g_spin_limit.exchange(limit < 0 ? QSPIN_LIMIT : limit, std::memory_order_relaxed);
}

int xmc_profile_events(void* start_event, void* stop_event) {
  g_prof_start = (hipEvent_t)start_event;
  g_prof_stop = (hipEvent_t)stop_event;
  return XMC_OK;
}

size_t xmc_tiled_workspace_bytes(int num_chunks, int rows_per_chunk, int max_batch) {
  return xmc_tiled_workspace_bytes_ex(num_chunks, rows_per_chunk, max_batch, D);
}

size_t xmc_tiled_workspace_bytes_ex(int num_chunks, int rows_per_chunk, int max_batch, int features) {
  if (features != D && features != 1024) return 0;
  if (num_chunks <= 0 || num_chunks > MAX_CHUNKS || rows_per_chunk <= 0 || max_batch <= 0 || max_batch > T_HALVES * BP) return 0;
  const size_t rows_pad = ((size_t)rows_per_chunk + TL - 1) / TL * TL;
  const size_t tiles = (size_t)num_chunks * (rows_pad / TL);
  const size_t halves = (size_t)tiled_halves(max_batch), pairs = (halves + 1) / 2;
  const size_t rows_buf = (size_t)tiled_group(num_chunks, rows_per_chunk) * rows_pad;   // rows of one launch
  // per batch half G in both orientations; tile_ptr per pair of halves (padded to 64 entries); two loss shares per tile
  const size_t three = TW_HEAD + tiled_layout((int)halves, features).g + halves * 2 * rows_buf * BP * 2 + pairs * ((tiles + 1 + 63) / 64 * 64 * 4) + (tiles * 8 + 255) / 256 * 256;
  const size_t one = features == D ? cluster_layout(num_chunks, rows_per_chunk, max_batch).bytes : 0;
  return three > one ? three : one;
}

int* xmc_failure_word(void) { return device_info().failure_word; }

int xmc_pass_on_error(const int32_t* error_word, int32_t* into_error, int32_t* into_sticky, void* stream_) {
  if (!error_word || !into_error != !into_sticky) return XMC_ERR_NULL;
  if ((((uintptr_t)error_word | (uintptr_t)into_error | (uintptr_t)into_sticky) & 3) != 0) return XMC_ERR_ALIGN;
  const DeviceInfo di = device_info();
  if (di.ok != 1 || !di.failure_word) return XMC_ERR_DEVICE;
  pass_on_error_kernel<<<1, 1, 0, (hipStream_t)stream_>>>(error_word, into_error, into_sticky, di.failure_word);
  return launch_status();
}

size_t xmc_tiled_error_offset(void) { return TW_ERR; }
size_t xmc_tiled_sticky_error_offset(void) { return TW_ERR + 4; }

int xmc_tiled_update_streams(int cus, int features, int batch, int tiles) {
  if ((features != D && features != 1024) || batch <= 0 || batch > T_HALVES * BP || cus <= 0 || tiles <= 0) return XMC_ERR_SHAPE;
  return tup_streams(cus, tiled_halves(batch), features, tiles);
}

int xmc_tiled_step(void* const* chunk_ptrs, int num_chunks, int rows_per_chunk, int rows_last_chunk, int weight_type,
                   const void* x_bf16, int batch, int features, const int32_t* labels_coo, int nnz, float lr,
                   const uint32_t* seeds, int round_mode, int quantize_x, int saturate, void* kahan, int kahan_type,
                   int num_head, void* grad_x_bf16, float* grad_x_f32, float* loss_out, void* workspace,
                   size_t workspace_bytes, void* stream_) {
  return xmc_tiled_step_ex(chunk_ptrs, num_chunks, rows_per_chunk, rows_last_chunk, weight_type, x_bf16, batch, features, labels_coo,
                           nnz, lr, seeds, round_mode, quantize_x, saturate, kahan, kahan_type, num_head, 0.0f, 0.0f, 0ull,
                           grad_x_bf16, grad_x_f32, loss_out, workspace, workspace_bytes, stream_);
}

}  // extern "C"

// xmc_tiled_step_ex for DD features (768 or 1024)
template <int DD>
static int tiled_step_t(void* const* chunk_ptrs, int num_chunks, int rows_per_chunk, int rows_last_chunk, int weight_type,
                        const void* x_bf16, int batch, const int32_t* labels_coo, int nnz, float lr,
                        const uint32_t* seeds, int round_mode, int quantize_x, int saturate, void* kahan, int kahan_type,
                        int num_head, float weight_decay, float dropout_p, unsigned long long dropout_seed, void* grad_x_bf16,
                        float* grad_x_f32, float* loss_out, void* workspace, size_t workspace_bytes, void* stream_) {
  if (!chunk_ptrs || !x_bf16 || !workspace || !grad_x_bf16 || (nnz > 0 && !labels_coo)) return XMC_ERR_NULL;
  if (kahan_type < 0 || kahan_type > 2 || (kahan_type != 0 && (weight_type != W_E4M3 || !kahan))) return XMC_ERR_MODE;
  if (kahan_type != 0 && (num_head < 0 || num_head > rows_per_chunk || !aligned16(kahan))) return XMC_ERR_SHAPE;
  if (kahan_type == 0) num_head = 0;
  if (batch <= 0 || batch > T_HALVES * BP) return XMC_ERR_SHAPE;
  if (rows_per_chunk <= 0 || rows_last_chunk <= 0 || rows_last_chunk > rows_per_chunk) return XMC_ERR_SHAPE;
  if (num_chunks <= 0 || num_chunks > MAX_CHUNKS) return XMC_ERR_RANGE;
  // a key keeps 24 bits for the label: larger label spaces are taken in segments of whole chunks, each with its own
  // list of the positives that fall into it and labels counted from the segment's first
  if (rows_per_chunk >= (1 << 24) - 1 || (long long)num_chunks * rows_per_chunk > 0x7FFFFFFFLL) return XMC_ERR_RANGE;
  if (nnz < 0 || nnz > MAX_POS) return XMC_ERR_RANGE;
  if (weight_type != W_E4M3 && weight_type != W_BF16) return XMC_ERR_MODE;
  if (round_mode != XMC_ROUND_RTN && round_mode != XMC_ROUND_SR_PHILOX && round_mode != XMC_ROUND_SR_FAST) return XMC_ERR_MODE;
  if (round_mode != XMC_ROUND_RTN && !seeds) return XMC_ERR_NULL;
  if (!(weight_decay >= 0.f) || !(dropout_p >= 0.f) || !(dropout_p < 1.f)) return XMC_ERR_SHAPE;
  if (kahan_type != 0 && (weight_decay != 0.f || dropout_p != 0.f)) return XMC_ERR_MODE;   // the head-Kahan layer has neither
  const DropoutParams dp = {dropout_p, 1.0f - dropout_p, (unsigned)(dropout_seed & 0xFFFFFFFFull), (unsigned)(dropout_seed >> 32)};
  const float wd = weight_decay;
  for (int c = 0; c < num_chunks; c++) {
    if (!chunk_ptrs[c]) return XMC_ERR_NULL;
    if (!aligned16(chunk_ptrs[c])) return XMC_ERR_ALIGN;
  }
  if (!aligned16(x_bf16) || ((uintptr_t)workspace & 255) != 0 || ((uintptr_t)labels_coo & 7) != 0) return XMC_ERR_ALIGN;
  if (workspace_bytes < xmc_tiled_workspace_bytes_ex(num_chunks, rows_per_chunk, batch, DD)) return XMC_ERR_WORKSPACE;
  DeviceInfo di = device_info();
  if (di.ok != 1) return XMC_ERR_DEVICE;
  hipStream_t stream = (hipStream_t)stream_;
  // (a cluster needs its members on one XCD at the same time: a partition of the GPU too small for one keeps the three kernels)
  const int cluster = cluster_size(batch);
  if (DD == D && kahan_type == 0 && !loss_out && weight_decay == 0.f && di.cus / 8 / cluster >= 1)
  {
    unsigned char* w0 = (unsigned char*)workspace;
    const ClusterLayout lay = cluster_layout(num_chunks, rows_per_chunk, batch);
    const ClusterPlace at = {w0 + lay.xq, (unsigned short*)(w0 + lay.xt), (unsigned*)(w0 + lay.keys), (int*)(w0 + lay.flags), (int*)(w0 + lay.xcc),
                             (float*)(w0 + lay.gx), (int*)(w0 + lay.tile_ptr), lay.tp_stride, w0 + lay.exch, (floatx4*)(w0 + lay.partial),
                             (int*)(w0 + TW_ERR), (int*)(w0 + TW_ERR) + 1};
    return cluster_step(chunk_ptrs, num_chunks, rows_per_chunk, rows_last_chunk, weight_type, x_bf16, batch, labels_coo, nnz, lr, seeds,
                        round_mode, quantize_x, saturate, dp, grad_x_bf16, grad_x_f32, at, false, di.cus, di.failure_word, stream);
  }
  unsigned char* ws = (unsigned char*)workspace + TW_HEAD;

  const int rows_pad = (rows_per_chunk + TL - 1) / TL * TL;
  const int tiles_per_chunk = rows_pad / TL;
  const int num_tiles = num_chunks * tiles_per_chunk;
  const int halves = tiled_halves(batch), pairs = (halves + 1) / 2;   // halves beyond the batch are zero rows of X
  // Several chunks per launch where they lie one behind the other in memory (the bf16 layer's views of one tensor) and
  // the compensated head is not in play; the buffers are sized for that many rows either way.
  const int group_max = tiled_group(num_chunks, rows_per_chunk);
  int group = kahan_type != 0 ? 1 : group_max;
  for (int c = 0; c + 1 < num_chunks && group > 1; c++)
    if ((const unsigned char*)chunk_ptrs[c + 1] != (const unsigned char*)chunk_ptrs[c] + (size_t)rows_per_chunk * DD * (weight_type == W_BF16 ? 2 : 1))
      group = 1;
  const size_t rows_buf = (size_t)group_max * rows_pad;               // rows the G buffers hold
  const TiledLayout lay = tiled_layout(halves, DD);
  unsigned short* xb = (unsigned short*)(ws + lay.xb);
  unsigned short* xT = (unsigned short*)(ws + lay.xt);
  unsigned* keys = (unsigned*)(ws + lay.keys);
  float* gx_total = (float*)(ws + lay.gx);
  floatx4* partial = (floatx4*)(ws + lay.part);
  const size_t g_half = 2 * rows_buf * BP;    // elements of one half's G and G^T
  unsigned short* glb = (unsigned short*)(ws + lay.g);
  unsigned short* gbl = glb + rows_buf * BP;
  int* tile_ptr = (int*)(glb + halves * g_half);
  const size_t tp_stride = (size_t)(num_tiles + 1 + 63) / 64 * 64;   // entries of one pair's tile_ptr
  float* loss_part = (float*)(tile_ptr + pairs * tp_stride);         // one share per sub-tile of 32 rows

  // chunks per segment of the label space: a multiple of the launch group, fewer than 2^24 - 1 labels
  int seg_chunks = ((1 << 24) - 2) / rows_per_chunk / group * group;
  if (seg_chunks < group) return XMC_ERR_RANGE;
  // true-FP8 arithmetic with two or four batch halves: FP8 matrix products, the logits of a pair of halves in one pass
  const bool fp8_logits = weight_type == W_E4M3 && quantize_x && halves >= 2 && !loss_out;
  // e4m3 weights, two batch halves, no compensated head: the feature-split update kernel (X^T in registers)
  const bool split_update = weight_type == W_E4M3 && halves == 2 && kahan_type == 0 && DD == D;
  // batch rows whose G is written and read; the feature-split update reads the G of both halves whole
  const int live = split_update ? halves * BP : batch;
  for (int c = 0; c < num_chunks; c += group) {
    const int seg0 = c / seg_chunks * seg_chunks;   // first chunk of the segment
    if (c == seg0) {
      // the segment's positives of every 256 batch rows as a list of their own (the key keeps eight bits for the row), grouped by
      // tile, and the first key of each of its tiles; in front of the first segment the images of X besides
      const int seg_n = seg0 + seg_chunks <= num_chunks ? seg_chunks : num_chunks - seg0, seg_tiles = seg_n * tiles_per_chunk;
      const int ptr_blocks = (seg_tiles + PREP_NT) / PREP_NT, x_blocks = c == 0 ? (halves * BP * DD + PREP_NT - 1) / PREP_NT : 0;
      const TiledPrep pp = {labels_coo, nnz, batch, seg0 * rows_per_chunk, seg_n * rows_per_chunk, rows_per_chunk, tiles_per_chunk, seg_tiles, ptr_blocks, pairs,
                            keys, tile_ptr + seg0 * tiles_per_chunk, tp_stride, (const unsigned short*)x_bf16, halves, quantize_x, fp8_logits ? 1 : 0,
                            split_update ? 1 : 0, xb, xT, gx_total, loss_part, loss_out ? 2 * num_tiles : 0, (int*)((unsigned char*)workspace + TW_ERR)};
      tiled_prep_kernel<DD><<<ptr_blocks * pairs + x_blocks, PREP_NT, (size_t)nnz * 4, stream>>>(pp, dp);
    }
    void* w = chunk_ptrs[c];
    const int nch = c + group <= num_chunks ? group : num_chunks - c;                       // chunks of this launch
    const int rows = (nch - 1) * rows_per_chunk + (c + nch == num_chunks ? rows_last_chunk : rows_per_chunk);
    const int rp = (rows + TL - 1) / TL * TL;           // padded rows of this launch (the G buffers use the stride rows_buf)
    const int tiles = rp / TL;
    const unsigned label0 = (unsigned)c * (unsigned)rows_per_chunk;                  // global: the fast rounding's random words
    const unsigned label0_seg = (unsigned)(c - seg0) * (unsigned)rows_per_chunk;     // within the segment: the keys
    TiledSeeds sd;
    for (int k = 0; k < T_GROUP; k++)
      sd.s[k] = seeds && k < nch ? (round_mode == XMC_ROUND_SR_FAST ? fast_seed(seeds[c + k]) : seeds[c + k]) : 0u;
    const int nh = c == 0 ? num_head : 0;   // the compensated head lives in chunk 0 (chunked_head_kahan_fp8xmc_clf.py:127)
    // label ranges of the grad_X kernel: slots shared by the launch's chunks, none across a chunk boundary
    const int cs = nch > 1 ? rows_per_chunk : rp;       // rows of a chunk as the kernels see them
    const int spc_max = tiled_splits(rp) / nch > 0 ? tiled_splits(rp) / nch : 1;   // (a launch has at most eight chunks)
    int range = (cs + spc_max - 1) / spc_max;
    range = (range + TL - 1) / TL * TL;
    const int spc = (cs + range - 1) / range;            // slots (and at most ranges) per chunk
    const int splits = nch * spc;
    float* lp = loss_part + 2 * c * tiles_per_chunk;
    for (int hh = 0; fp8_logits && hh < halves; hh += 2) {
      const int nsub = 2 * tiles, lgrid = nsub < di.cus ? nsub : di.cus;
      tiled_logits_fp8_kernel<DD><<<lgrid, 512, TlgGeom<W_E4M3, DD>::LDS, stream>>>(
          w, rows, nsub, (const unsigned char*)xb + (size_t)hh * BP * DD, keys + (size_t)(hh >> 1) * MAX_POS,
          tile_ptr + (hh >> 1) * tp_stride + c * tiles_per_chunk, label0_seg, glb + hh * g_half, gbl + hh * g_half, g_half, live - hh * BP);
    }
    for (int hh = 0; !fp8_logits && hh < halves; hh++) {
      if (hh * BP >= live) break;   // no batch rows: no G, nothing to add to the loss
      unsigned short* gl = glb + hh * g_half;
      unsigned short* gb = gbl + hh * g_half;
      const unsigned short* xh = xb + (size_t)hh * BP * DD;
      const unsigned* kh = keys + (size_t)(hh >> 1) * MAX_POS;                       // this half's pair: its keys,
      const int* tp = tile_ptr + (hh >> 1) * tp_stride + c * tiles_per_chunk;       // its tile_ptr,
      const unsigned brow0 = (unsigned)((hh & 1) * BP);                             // the half's first row within the pair
      const int pbatch = batch - 256 * (hh >> 1);                                   // and the batch rows the pair has
      const int nsub = 2 * tiles;                                   // sub-tiles of 32 label rows
      const int lgrid = nsub < di.cus ? nsub : di.cus;              // persistent: one workgroup per compute unit
      if (weight_type == W_BF16) {
        if (loss_out) tiled_logits_kernel<W_BF16, true, DD><<<lgrid, 512, TlgGeom<W_BF16, DD>::LDS, stream>>>(w, rows, nsub, xh, kh, tp, label0_seg, gl, gb, pbatch, brow0, live - hh * BP, lp);
        else tiled_logits_kernel<W_BF16, false, DD><<<lgrid, 512, TlgGeom<W_BF16, DD>::LDS, stream>>>(w, rows, nsub, xh, kh, tp, label0_seg, gl, gb, pbatch, brow0, live - hh * BP, lp);
      } else {
        if (loss_out) tiled_logits_kernel<W_E4M3, true, DD><<<lgrid, 512, TlgGeom<W_E4M3, DD>::LDS, stream>>>(w, rows, nsub, xh, kh, tp, label0_seg, gl, gb, pbatch, brow0, live - hh * BP, lp);
        else tiled_logits_kernel<W_E4M3, false, DD><<<lgrid, 512, TlgGeom<W_E4M3, DD>::LDS, stream>>>(w, rows, nsub, xh, kh, tp, label0_seg, gl, gb, pbatch, brow0, live - hh * BP, lp);
      }
    }
    // grad_X of the launch's chunks: one pass over W per pair of batch halves, then the fixed-order sums per half
    const size_t part_half = (size_t)T_SPLITS * 4 * (8 * (DD / 256)) * 256;   // floatx4 elements of one half's partials
    const int ggrid = 4 * ((splits + 7) / 8 * 8);
    for (int h0 = 0; h0 < halves; h0 += 2) {
      const unsigned short* gsrc = gbl + h0 * g_half;
      floatx4* pdst = partial + h0 * part_half;
      if (weight_type == W_BF16) {
        if (halves == 1) tiled_gradx_kernel<W_BF16, 1, DD><<<ggrid, 512, TgxGeom<W_BF16, 1, DD>::LDS, stream>>>(w, rows, (int)rows_buf, rp, range, cs, spc, gsrc, g_half, live - h0 * BP, pdst, part_half);
        else tiled_gradx_kernel<W_BF16, 2, DD><<<ggrid, 512, TgxGeom<W_BF16, 2, DD>::LDS, stream>>>(w, rows, (int)rows_buf, rp, range, cs, spc, gsrc, g_half, live - h0 * BP, pdst, part_half);
      } else {
        if (halves == 1) tiled_gradx_kernel<W_E4M3, 1, DD><<<ggrid, 512, TgxGeom<W_E4M3, 1, DD>::LDS, stream>>>(w, rows, (int)rows_buf, rp, range, cs, spc, gsrc, g_half, live - h0 * BP, pdst, part_half);
        else tiled_gradx_kernel<W_E4M3, 2, DD><<<ggrid, 512, TgxGeom<W_E4M3, 2, DD>::LDS, stream>>>(w, rows, (int)rows_buf, rp, range, cs, spc, gsrc, g_half, live - h0 * BP, pdst, part_half);
      }
    }
    const int ugrid = tred_waves(DD) * halves / (tup_threads(halves) / 64) + (DD / 64) / tup_csteps(halves, DD) * tup_streams(di.cus, halves, DD, tiles);
    const bool final_sum = c + nch == num_chunks;
    const TiledSum sum = {partial, part_half, nch, spc, range, rp, weight_type == W_BF16 ? 1 : 0, gx_total, batch,
                          final_sum ? (unsigned short*)grad_x_bf16 : nullptr, final_sum ? grad_x_f32 : nullptr};
#define XMC_LAUNCH_UPDATE_K(WTYPE, RMODE, HV, KH, NKS)                                                                          \
  tiled_update_kernel<WTYPE, RMODE, HV, KH, DD, NKS><<<ugrid, tup_threads(HV), (size_t)tup_lds_bytes(HV, DD, NKS), stream>>>(   \
      w, rows, tiles, glb, g_half, xT, lr, wd, sd, cs, saturate, kahan, kahan_type, nh, label0, live, sum, dp)
#define XMC_LAUNCH_UPDATE_H(WTYPE, RMODE, KH)                                                                                  \
  do {                                                                                                                         \
    if (halves == 1 && batch <= 32 && !KH) XMC_LAUNCH_UPDATE_K(WTYPE, RMODE, 1, false, 1);                                     \
    else if (halves == 1 && batch <= 64 && !KH) XMC_LAUNCH_UPDATE_K(WTYPE, RMODE, 1, false, 2);                                \
    else if (halves == 1) XMC_LAUNCH_UPDATE_K(WTYPE, RMODE, 1, KH, 4);                                                         \
    else if (halves == 2) XMC_LAUNCH_UPDATE_K(WTYPE, RMODE, 2, KH, 4);                                                         \
    else XMC_LAUNCH_UPDATE_K(WTYPE, RMODE, 4, KH, 4);                                                                          \
  } while (0)
    const bool with_head = kahan_type != 0 && nh > 0;   // only chunk 0 of the head-Kahan layer
    if (split_update) {
      int streams = (tiles + 7) / 8 * 8;
      streams = streams < 128 ? streams : 128;           // two workgroups per compute unit, four per stream
      const int grid2 = tred_waves(D) * 2 / 4 + 4 * streams;
#define XMC_LAUNCH_UPDATE2(RMODE)                                                                                              \
  tiled_update2_kernel<RMODE><<<grid2, 256, 2 * TU2_GBUF, stream>>>(w, rows, tiles, glb, g_half, (const bf16x8*)xT, lr, wd, sd, cs, saturate, \
                                                                    label0, sum, dp)
      if (round_mode == XMC_ROUND_RTN) XMC_LAUNCH_UPDATE2(ROUND_RTN);
      else if (round_mode == XMC_ROUND_SR_FAST) XMC_LAUNCH_UPDATE2(ROUND_SR_FAST);
      else XMC_LAUNCH_UPDATE2(ROUND_SR_PHILOX);
#undef XMC_LAUNCH_UPDATE2
    } else if (weight_type == W_BF16) {
      if (round_mode == XMC_ROUND_RTN) XMC_LAUNCH_UPDATE_H(W_BF16, ROUND_RTN, false);
      else if (round_mode == XMC_ROUND_SR_FAST) XMC_LAUNCH_UPDATE_H(W_BF16, ROUND_SR_FAST, false);
      else XMC_LAUNCH_UPDATE_H(W_BF16, ROUND_SR_PHILOX, false);
    } else if (with_head) {
      if (round_mode == XMC_ROUND_RTN) XMC_LAUNCH_UPDATE_H(W_E4M3, ROUND_RTN, true);
      else if (round_mode == XMC_ROUND_SR_FAST) XMC_LAUNCH_UPDATE_H(W_E4M3, ROUND_SR_FAST, true);
      else XMC_LAUNCH_UPDATE_H(W_E4M3, ROUND_SR_PHILOX, true);
    } else {
      if (round_mode == XMC_ROUND_RTN) XMC_LAUNCH_UPDATE_H(W_E4M3, ROUND_RTN, false);
      else if (round_mode == XMC_ROUND_SR_FAST) XMC_LAUNCH_UPDATE_H(W_E4M3, ROUND_SR_FAST, false);
      else XMC_LAUNCH_UPDATE_H(W_E4M3, ROUND_SR_PHILOX, false);
    }
#undef XMC_LAUNCH_UPDATE_H
#undef XMC_LAUNCH_UPDATE_K
  }
  if (loss_out) tiled_loss_kernel<<<1, 256, 0, stream>>>(loss_part, 2 * num_tiles, loss_out);
  return launch_status();
}

extern "C" {

int xmc_tiled_step_ex(void* const* chunk_ptrs, int num_chunks, int rows_per_chunk, int rows_last_chunk, int weight_type,
                      const void* x_bf16, int batch, int features, const int32_t* labels_coo, int nnz, float lr,
                      const uint32_t* seeds, int round_mode, int quantize_x, int saturate, void* kahan, int kahan_type,
                      int num_head, float weight_decay, float dropout_p, unsigned long long dropout_seed, void* grad_x_bf16,
                      float* grad_x_f32, float* loss_out, void* workspace, size_t workspace_bytes, void* stream_) {
  if (features == D)
    return tiled_step_t<D>(chunk_ptrs, num_chunks, rows_per_chunk, rows_last_chunk, weight_type, x_bf16, batch, labels_coo, nnz, lr, seeds,
                           round_mode, quantize_x, saturate, kahan, kahan_type, num_head, weight_decay, dropout_p, dropout_seed,
                           grad_x_bf16, grad_x_f32, loss_out, workspace, workspace_bytes, stream_);
  if (features == 1024)
    return tiled_step_t<1024>(chunk_ptrs, num_chunks, rows_per_chunk, rows_last_chunk, weight_type, x_bf16, batch, labels_coo, nnz, lr,
                              seeds, round_mode, quantize_x, saturate, kahan, kahan_type, num_head, weight_decay, dropout_p,
                              dropout_seed, grad_x_bf16, grad_x_f32, loss_out, workspace, workspace_bytes, stream_);
  return XMC_ERR_SHAPE;
}

int xmc_copy_probe(void* dst, const void* src, size_t bytes, void* stream_) {
  if (!dst || !src) return XMC_ERR_NULL;
  if (!aligned16(dst) || !aligned16(src) || bytes % 16 != 0) return XMC_ERR_ALIGN;
  if (bytes == 0) return XMC_OK;
  copy_probe_kernel<<<2048, 256, 0, (hipStream_t)stream_>>>((const uint4*)src, (uint4*)dst, bytes / 16);
  return launch_status();
}

int xmc_step_error_word(const void* workspace, int num_chunks, int rows_per_chunk, void* stream_) {
  (void)num_chunks; (void)rows_per_chunk;
  if (!workspace) return XMC_ERR_NULL;
  int word = 0;
  if (hipMemcpyAsync(&word, (const unsigned char*)workspace + xmc_step_error_offset(), 4, hipMemcpyDeviceToHost,
                     (hipStream_t)stream_) != hipSuccess) return XMC_ERR_LAUNCH;
  if (hipStreamSynchronize((hipStream_t)stream_) != hipSuccess) return XMC_ERR_LAUNCH;
  return word;
}

size_t xmc_step_error_offset(void) { return WS_FLAGS + (size_t)QF_ERR * 4; }

size_t xmc_step_sticky_error_offset(void) { return WS_FLAGS + (size_t)QF_STICKY * 4; }

int xmc_step_workgroups(void) {
  DeviceInfo di = device_info();
  if (di.ok != 1) return XMC_ERR_DEVICE;
  return (di.cus < MAX_WG ? di.cus : MAX_WG) / 32 * 32;
}

int xmc_step_xcc_ids(const void* workspace, int32_t* ids_host, int count, void* stream_) {
  if (!workspace || !ids_host) return XMC_ERR_NULL;
  if (count <= 0 || count > MAX_WG) return XMC_ERR_RANGE;
  if (hipMemcpyAsync(ids_host, (const unsigned char*)workspace + WS_FLAGS + (size_t)QF_XCC * 4, (size_t)count * 4,
                     hipMemcpyDeviceToHost, (hipStream_t)stream_) != hipSuccess) return XMC_ERR_LAUNCH;
  if (hipStreamSynchronize((hipStream_t)stream_) != hipSuccess) return XMC_ERR_LAUNCH;
  return XMC_OK;
}

int xmc_quad_placement_check(const int32_t* xcc_ids_host, int num_workgroups) {
  if (!xcc_ids_host) return XMC_ERR_NULL;
  if (num_workgroups < 32 || num_workgroups > MAX_WG || num_workgroups % 32 != 0) return XMC_ERR_RANGE;
  int bad = 0;
  for (int q = 0; q < num_workgroups / 4; q++) bad += quad_xcc_mismatch(xcc_ids_host, q) ? 1 : 0;
  return bad;
}

}  // extern "C"
