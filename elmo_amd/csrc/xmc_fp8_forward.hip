// Inference logits of the FP8 extreme-classifier layer for gfx950 (MI355X), and top-k of them without storing them.
//
// Reference semantics: src/xmc_classifiers/chunked_fp8xmc_clf.py:45-60 (xfc_forward).
#include "xmc_common.h"

namespace xmc {

typedef __attribute__((address_space(3))) unsigned char lds_u8;

// 32 bytes from a 16-byte aligned LDS address
__device__ __forceinline__ intx8 lds_read32(const unsigned char* q) {
  intx4 lo = *(const intx4*)q, hi = *(const intx4*)(q + 16);
  return intx8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
}

// Operand image of X for the inference kernels (but for small batches, whose workgroups convert X themselves): e4m3(X / scale_x) in v_mfma 16x16x128 B-operand order,
// [(w*2+nb)*6+ks][lane][32 bytes]; one thread per four features, rows at or past `batch` are zero.
__global__ void prep_x_kernel(const unsigned short* x, int batch, int n, float inv_scale_x, unsigned char* xq) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int b = i / (D / 4), k = (i - b * (D / 4)) * 4;
  uint2 raw = {0u, 0u};
  if (b < batch) raw = *(const uint2*)(x + (size_t)b * D + k);
  auto val = [&](unsigned bits) { return clamp448(__uint_as_float(bits) * inv_scale_x); };
  int packed = __builtin_amdgcn_cvt_pk_fp8_f32(val(raw.x << 16), val(raw.x & 0xFFFF0000u), 0, false);
  packed = __builtin_amdgcn_cvt_pk_fp8_f32(val(raw.y << 16), val(raw.y & 0xFFFF0000u), packed, true);
  const int w = b >> 5, nb = (b >> 4) & 1, ks = k >> 7, kgq = (k >> 5) & 3, jq = k & 31;
  *(int*)(xq + ((size_t)((w * 2 + nb) * 6 + ks) * 64 + ((b & 15) + 16 * kgq)) * 32 + jq) = packed;
}

// Inference logits: out[b, label - col0] = bf16(zscale * sum_k Xq[b,k] W[label,k]) for the 32-label tiles
// [tile_begin, tile_end) of the chunk list (tile t = chunk t / tiles_per_chunk, rows 32 (t % tiles_per_chunk) ...).
struct ForwardParams {
  const unsigned char* chunk[MAX_CHUNKS];
  int rows_per_chunk, tiles_per_chunk;
  int tile_begin, tile_end;
  const unsigned char* xq;     // operand image of X, or
  const unsigned short* x;     // X itself (FWD_CONV), bf16 [batch][768]
  float inv_scale_x;
  float zscale;
  unsigned short* out;         // bf16 [batch][out_stride]
  long long out_stride;
  long long col0;              // label that column 0 of `out` stands for
  long long num_labels;        // labels at or past this one are not written
  int batch;
};

constexpr int FT = 32;                    // labels per tile of the inference kernels
constexpr int FB = FT * WS;               // one tile in LDS (rows of 48 + 1 pieces of 16 bytes)
constexpr int FNT = 512;                  // eight wavefronts of 32 batch rows: four per half of a tile's labels (128 rows), or eight (256)
constexpr int ZS = FT * 2 + 16;           // LDS row stride of the staged logits [b][32 labels] bf16, bytes
constexpr int FWD_CONV = 64;              // most batch rows whose X the workgroups of fp8_forward_kernel convert themselves
// Geometry for up to HB x 128 batch rows
template <int HB, bool CONV = false> struct FwdGeom {
  static constexpr int BUF = HB == 1 ? 5 : 4;          // tile buffers in LDS, one workgroup to a compute unit
  static constexpr int ZB = HB * BP * ZS;              // a stage of logits
  static constexpr int LDS = CONV ? 160 * 1024 : BUF * FB + 2 * ZB;
  static constexpr int X = LDS - FWD_CONV * WS;        // (CONV) e4m3 X before the first tile; X as it comes lies in front of it
  static_assert(!CONV || (BUF * FB + 2 * ZB <= LDS && X >= FWD_CONV * D * 2 && X % 16 == 0), "LDS budget");
};
constexpr int FWD_ROWS = 2 * BP;          // most batch rows of a launch

// Each of WAVES wavefronts fetches its rows of the tile with exactly one instruction a row (fwd_wait relies on it), 48 lanes
// wide, from a scalar row address: no lane computes one.
template <int WAVES>
__device__ __forceinline__ void fwd_issue_tile(const unsigned char* gtile, int rows_valid, unsigned lds_off, int v, int lane) {
  if (lane < D / 16) {
#pragma unroll
    for (int j = 0; j < FT / WAVES; j++) {
      const int row = FT / WAVES * v + j, src = min(row, rows_valid - 1);   // rows past the end re-read the last valid one
      const unsigned ldsoff = __builtin_amdgcn_readfirstlane(lds_off + (unsigned)(row * WS));
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 3\n\tglobal_load_lds_dwordx4 %1, %2" : : "s"(ldsoff), "v"(lane * 16), "s"(gtile + src * D) : "memory", "m0");
    }
  }
}

// the logits operands of a wavefront: batch rows 32w .. 32w + 31
__device__ __forceinline__ void fwd_load_x(const unsigned char* xq_image, int w, int lane, intx8 (&xq)[2][6]) {
#pragma unroll
  for (int nb = 0; nb < 2; nb++)
#pragma unroll
    for (int ks = 0; ks < 6; ks++)
      xq[nb][ks] = *(const intx8*)(xq_image + ((size_t)((w * 2 + nb) * 6 + ks) * 64 + lane) * 32);
}

// X itself instead of its image, for up to FWD_CONV batch rows: straight to LDS as it comes, converted there, and read as the rows of
// a tile are; it saves the launch in front.  Loops of a few instructions with all loads in flight: the first pass over code costs 1.5
// to 2 clocks a byte (24 pieces of a thread unrolled were 10 KiB of it: 131 K labels, 40 rows 26.8 us a call), and a loop that loaded 16
// rows while it converted 16 others had a miss of the L2 in every round (25.1; an image 22.1, as it is 21.2).  What X holds in LDS behind
// the batch are logits of nobody.
__device__ __forceinline__ void fwd_request_x(const unsigned short* x, int rows, unsigned raw, int v, int lane) {
  const int pieces = rows * (D * 2 / 16);
#pragma unroll 1
  for (int c0 = v * 64; c0 < pieces; c0 += FNT) {
    const unsigned ldsoff = __builtin_amdgcn_readfirstlane(raw + (unsigned)(c0 * 16));
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 3\n\tglobal_load_lds_dwordx4 %1, %2" : : "s"(ldsoff), "v"(min(c0 + lane, pieces - 1) * 16), "s"(x) : "memory", "m0");
  }
}
__device__ __forceinline__ void fwd_convert_x(int rows, float inv_scale_x, const unsigned char* raw, unsigned char* img, int tid) {
  constexpr int PR = D * 2 / 16;
#pragma unroll 1
  for (int ch = tid; ch < rows * PR; ch += FNT) {
    const uint4 r = *(const uint4*)(raw + ch * 16);
    auto val = [&](unsigned bits) { return clamp448(__uint_as_float(bits) * inv_scale_x); };
    auto pack = [&](unsigned a, unsigned b) {
      const int lo = __builtin_amdgcn_cvt_pk_fp8_f32(val(a << 16), val(a & 0xFFFF0000u), 0, false);
      return (unsigned)__builtin_amdgcn_cvt_pk_fp8_f32(val(b << 16), val(b & 0xFFFF0000u), lo, true);
    };
    *(uint2*)(img + ch / PR * WS + ch % PR * 8) = uint2{pack(r.x, r.y), pack(r.z, r.w)};
  }
}

// z[nb]: logits of 16 labels (tile rows from `rows` on) and batch rows 32w + 16nb ..  All operands are requested before the
// first product: two wavefronts per SIMD do not hide an LDS read's latency in front of each of the six steps.  `between` runs
// while they are on their way.
template <class F>
__device__ __forceinline__ void fwd_products(const unsigned char* rows, int l16, int kg, const intx8 (&xq)[2][6], floatx4 (&z)[2], F&& between) {
  intx8 a[6];
#pragma unroll
  for (int ks = 0; ks < 6; ks++) a[ks] = lds_read32(rows + l16 * WS + ks * 128 + kg * 32);
  __builtin_amdgcn_sched_barrier(0);
  between();
  z[0] = z[1] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int ks = 0; ks < 6; ks++) {
    z[0] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a[ks], xq[0][ks], z[0], 0, 0, 0, 0, 0, 0);
    z[1] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a[ks], xq[1][ks], z[1], 0, 0, 0, 0, 0, 0);
  }
}

// Place of a tile in the chunk list: chunk c, tile r within it.
struct FwdPlace {
  int c, r;
  __device__ __forceinline__ FwdPlace(int t, int tiles_per_chunk) : c(t / tiles_per_chunk), r(t - c * tiles_per_chunk) {}
  // n tiles on (no division in the loop)
  __device__ __forceinline__ void advance(int n, int tiles_per_chunk) {
    r += n;
    while (r >= tiles_per_chunk) { r -= tiles_per_chunk; c++; }
  }
};

// The next tile has landed: all loads but those of the AHEAD tiles behind it are complete.  Loads complete in order; stores
// in between only make the wait stricter.  `full`: AHEAD tiles have been requested behind it.
template <int WAVES, int AHEAD>
__device__ __forceinline__ void fwd_wait(bool full) {
  if (full) asm volatile("s_waitcnt vmcnt(%0)" : : "n"(AHEAD * FT / WAVES) : "memory");
  else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

// One workgroup streams its tiles through FBUF LDS buffers, the loads four tiles ahead of the matrix products, with one
// barrier per tile: behind it a tile has landed for everyone, the buffer of the tile before is free for the load, and the
// staged logits of the tile before (two stages in turn) leave as 16 consecutive bytes of a batch row per lane.
// HBM bound: 131 K labels, batch 40 (101 MB in, 10 MB out) 20.9 us = 5.3 TB/s; the same loads without anything else take 17.2.
// Two workgroups of four wavefronts with three buffers and three barriers per tile took 23.2; a batch that is no multiple of
// 16 also cost a padded copy of X and a copy of the logits (42 us the call, 25 without).
// CONV: the workgroups convert X themselves (up to FWD_CONV rows; forward_converts has the line): the call 25.3 / 24.1 us.
// HB = 2: 129 to 256 batch rows from one pass over the weights, every wavefront with 32 rows and both halves of a tile.
// us a call, two slices of 128 rows / now: 256 rows, 8 K labels 22.3 / 13.6, 131 K 54.6 / 39.6, 400 K 190 / 117, 1 M 569 / 414 (1.3 GB in
// and out: 3.1 TB/s);  129 rows, 131 K 48.0 / 32.9, 400 K 160 / 88, 1 M 438 / 288.
// RUN: consecutive tiles that a workgroup takes in a round (a power of two); what is left of the tiles is taken singly.
template <int HB, int RUN, bool CONV>
__global__ __launch_bounds__(FNT, 2) void fp8_forward_kernel(const ForwardParams p) {
  typedef FwdGeom<HB, CONV> Geo;
  constexpr int FBUF = Geo::BUF, ZB = Geo::ZB;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
  const int tid = threadIdx.x, v = __builtin_amdgcn_readfirstlane(tid >> 6), w = HB == 1 ? v & 3 : v, half0 = HB == 1 ? v >> 2 : 0;
  const int lane = tid & 63, l16 = lane & 15, kg = lane >> 4, nblocks = (int)gridDim.x;
  const unsigned lds0 = (unsigned)(size_t)(lds_u8*)lds_raw;
  const bool active = 32 * w < p.batch;   // (wave-uniform) a wavefront without batch rows only helps to load and store
  intx8 xq[2][6];
  if constexpr (!CONV) {
    if (active) fwd_load_x(p.xq, w, lane, xq);
    __builtin_amdgcn_s_waitcnt(0);
  }
  const int mine = (int)blockIdx.x, first = p.tile_begin + mine;
  const int rounds = RUN > 1 ? (p.tile_end - p.tile_begin) / (nblocks * RUN) : 0, in_runs = rounds * RUN;
  int ahead = first;                      // next tile to be requested
  FwdPlace at_ahead(p.tile_begin + mine * (rounds > 0 ? RUN : 1), p.tiles_per_chunk), at_store = at_ahead;   // its place, that of the next one to be stored
  // (`ahead` and t below count as a walk of single tiles does, which has as many)
  int k_ahead = 0, k_store = 0;
  auto step = [&](int& k) {               // from the workgroup's k-th tile to the next
    if constexpr (RUN == 1) return nblocks;
    k++;
    return k > in_runs ? nblocks : k == in_runs ? nblocks * RUN - (mine + 1) * RUN + mine + 1 : (k & (RUN - 1)) == 0 ? 1 + (nblocks - 1) * RUN : 1;
  };
  auto issue = [&](int buf) {
    if (ahead < p.tile_end) {
      const int row0 = at_ahead.r * FT;
      fwd_issue_tile<FNT / 64>(p.chunk[at_ahead.c] + (size_t)row0 * D, min(FT, p.rows_per_chunk - row0), lds0 + (unsigned)buf * FB, v, lane);
    }
    at_ahead.advance(step(k_ahead), p.tiles_per_chunk);
    ahead += nblocks;
  };
  auto store = [&](const unsigned char* stage) {
    const int row0 = at_store.r * FT;
    const int rows_valid = min(FT, p.rows_per_chunk - row0);
    const long long label0 = (long long)at_store.c * p.rows_per_chunk + row0, left = p.num_labels - label0;
    const int nvalid = (int)(left < rows_valid ? (left < 0 ? 0 : left) : rows_valid);
    at_store.advance(step(k_store), p.tiles_per_chunk);
    const int seg = tid & 3;
#pragma unroll
    for (int hb = 0; hb < HB; hb++) {
      const int b = (tid >> 2) + BP * hb;
      if (b >= p.batch) return;
      unsigned short* orow = p.out + (size_t)b * p.out_stride + (label0 - p.col0);
      const unsigned short* zrow = (const unsigned short*)(stage + b * ZS);
      const int s = (int)((8u - (unsigned)(((uintptr_t)orow >> 1) & 7u)) & 7u);   // elements before a 16-byte boundary
      const int a = s + 8 * seg;
      if (a + 8 <= nvalid) {
        uint4 o;
        if (s == 0) {
          o = *(const uint4*)(zrow + a);
        } else {
          o.x = zrow[a] | ((unsigned)zrow[a + 1] << 16);
          o.y = zrow[a + 2] | ((unsigned)zrow[a + 3] << 16);
          o.z = zrow[a + 4] | ((unsigned)zrow[a + 5] << 16);
          o.w = zrow[a + 6] | ((unsigned)zrow[a + 7] << 16);
        }
        *(uint4*)(orow + a) = o;
      } else {
        for (int e = a; e < nvalid && e < a + 8; e++) orow[e] = zrow[e];
      }
      if (seg == 0)
        for (int e = 0; e < s && e < nvalid; e++) orow[e] = zrow[e];
    }
  };
  int k0 = 0;
  if constexpr (CONV) {
    const int raw = Geo::X - ((p.batch + 15) & ~15) * (D * 2);
    fwd_request_x(p.x, p.batch, lds0 + (unsigned)raw, v, lane);
    int n = 0;   // tiles on their way into the buffers in front of X
#pragma unroll 1
    for (; k0 < FBUF - 1 && (k0 + 1) * FB <= raw; k0++) {
      n += ahead < p.tile_end ? 1 : 0;
      issue(k0);
    }
    static_assert(FT * 64 / FNT == 4, "loads of a tile");
    if (n == 3) asm volatile("s_waitcnt vmcnt(12)" ::: "memory");
    else if (n == 2) asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
    else if (n == 1) asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    fwd_convert_x(p.batch, p.inv_scale_x, lds_raw + raw, lds_raw + Geo::X, tid);
    __syncthreads();
    if (active) {
#pragma unroll
      for (int nb = 0; nb < 2; nb++)
#pragma unroll
        for (int ks = 0; ks < 6; ks++) xq[nb][ks] = lds_read32(lds_raw + Geo::X + (32 * w + 16 * nb + l16) * WS + ks * 128 + kg * 32);
    }
    __syncthreads();   // X's places are free
  }
#pragma unroll 1
  for (; k0 < FBUF - 1; k0++) issue(k0);
  int buf = 0, par = 0, t = first;
  for (; t < p.tile_end; t += nblocks) {
    unsigned char* stage = lds_raw + FBUF * FB;
    fwd_wait<FNT / 64, FBUF - 2>(t + (FBUF - 2) * nblocks < p.tile_end);
    __syncthreads();
    auto other = [&] {
      issue(buf == 0 ? FBUF - 1 : buf - 1);
      if (t != first) store(stage + (par ^ 1) * ZB);
    };
    if (!active) {
      other();
    } else {
#pragma unroll
      for (int hb = 0; hb < HB; hb++) {
        const int half = half0 + hb;
        floatx4 z[2];
        if (hb == 0) fwd_products(lds_raw + buf * FB + 16 * half * WS, l16, kg, xq, z, other);
        else fwd_products(lds_raw + buf * FB + 16 * half * WS, l16, kg, xq, z, [] {});
#pragma unroll
        for (int nb = 0; nb < 2; nb++) {
          uint2 o;
          o.x = bf16_pack2(z[nb][0] * p.zscale, z[nb][1] * p.zscale);
          o.y = bf16_pack2(z[nb][2] * p.zscale, z[nb][3] * p.zscale);
          *(uint2*)(stage + par * ZB + (32 * w + 16 * nb + l16) * ZS + (16 * half + 4 * kg) * 2) = o;
        }
      }
    }
    buf = buf == FBUF - 1 ? 0 : buf + 1;
    par ^= 1;
  }
  __syncthreads();
  if (t != first) store(lds_raw + FBUF * FB + (par ^ 1) * ZB);
}


// ---- Top-k of the inference logits without the logits in memory: two passes over the weights.
// Pass 1 (MODE 0) visits every tile_step-th tile; workgroup g keeps, per batch row, the largest logit of the tiles it
// visited (its tiles are spread over the whole label range) and writes these maxima as order keys to gmax[g][b].  The
// k-th largest of a row's maxima is at or below the row's k-th largest logit (k different groups each hold a logit at
// or above it): topk_bound_kernel stores it as the row's bound.  Pass 2 (MODE 1) visits every tile and appends the
// logits at or above the bound to the row's candidate list (label and key), in no particular order;
// topk_pick_kernel ranks the list.  A list holds SEL_CAP entries; the count keeps running past that, and the pick
// kernel reports a row whose count exceeded it.
constexpr int SEL_CAP = 2048;
constexpr int SEL_GROUPS = 512;          // most workgroups of pass 1
// Here two workgroups of four wavefronts share a compute unit, with three tile buffers each: a wavefront that collects
// candidates holds up the barrier of its own workgroup only.  Pass 2 over 670 K labels, batch 128, k = 100: 90 us = 5.7 TB/s
// (the loads alone: 85), one workgroup of eight wavefronts and five buffers 110, one queue per workgroup with LDS atomics 113.
// 129 to 256 batch rows take one workgroup of eight wavefronts with six buffers: one pass over the weights where slices of 128 rows
// take two.  us a call, two slices / now, 256 rows: 131 K labels, k = 5 80.7 / 57.0, 670 K, k = 1 234 / 161, k = 5 235 / 169, k = 100
// 241 / 204, 2 M, k = 5 614 / 435;  129 rows: 30 K, k = 5 47.9 / 28.7, 670 K, k = 5 225 / 144, k = 100 233 / 174.
constexpr int SEL_ROWS = FWD_ROWS;       // most batch rows of a launch
constexpr int SEL_QUEUE = 128;           // candidates a wavefront of pass 2 collects in LDS
template <int WAVES> struct SelGeom {
  static constexpr int BUF = WAVES == 4 ? 3 : 6;
  static constexpr int LDS = BUF * FB + WAVES * SEL_QUEUE * 8;
};
// The rows' counters lie a cache line apart: next to each other 57 K atomics (670 K labels, batch 128, k = 100) on four lines
// took 16 us where they came together.
constexpr int SEL_COUNT_STRIDE = 32;
static_assert(2 * SelGeom<4>::LDS <= 160 * 1024 && SelGeom<8>::LDS <= 160 * 1024, "LDS budget");

struct SelectParams {
  const unsigned char* chunk[MAX_CHUNKS];
  int rows_per_chunk, tiles_per_chunk;
  int n_visit, tile_step;        // the launch visits tiles j * tile_step, j in [0, n_visit)
  const unsigned char* xq;       // operand image of X
  float zscale;
  long long num_labels;          // labels at or past this one do not take part
  int batch;
  unsigned short* gmax;          // MODE 0: [gridDim.x][SEL_ROWS] keys
  const unsigned short* bound;   // MODE 1: [SEL_ROWS] keys
  unsigned* count;               // MODE 1: [SEL_ROWS], SEL_COUNT_STRIDE apart
  unsigned* cand_label;          // MODE 1: [SEL_ROWS][SEL_CAP]
  unsigned short* cand_key;      // MODE 1: [SEL_ROWS][SEL_CAP]
};

typedef unsigned short ushortx2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ unsigned pk_max_u16(unsigned a, unsigned b) {
  return __builtin_bit_cast(unsigned, __builtin_elementwise_max(__builtin_bit_cast(ushortx2, a), __builtin_bit_cast(ushortx2, b)));
}
// order keys of two packed bf16 values (topk_key per half, without its NaN rule: a NaN with the sign bit set gets a small key)
typedef short shortx2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ unsigned key_pair(unsigned w) {
  const unsigned neg = __builtin_bit_cast(unsigned, __builtin_bit_cast(shortx2, w) >> 15);   // 0xFFFF in the negative halves
  return w ^ (neg | 0x80008000u);
}

// WAVES wavefronts of 32 batch rows
template <int MODE, int WAVES>
__global__ __launch_bounds__(64 * WAVES, 2) void fp8_forward_select_kernel(const SelectParams p) {
  constexpr int SEL_BUF = SelGeom<WAVES>::BUF;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, l16 = lane & 15, kg = lane >> 4, block = blockIdx.x, nblocks = gridDim.x;
  const unsigned lds0 = (unsigned)(size_t)(lds_u8*)lds_raw;
  const bool active = 32 * w < p.batch;   // (wave-uniform) a wavefront without batch rows only helps to load
  intx8 xq[2][6];
  if (active) fwd_load_x(p.xq, w, lane, xq);
  unsigned bkey[2] = {0xFFFFu, 0xFFFFu}, bm1[2] = {0xFFFEFFFEu, 0xFFFEFFFEu};
  unsigned rows_in_use = 0u;              // bits 8half + 4nb + e of the batch blocks that this lane has a row of
  if (MODE == 1) {
#pragma unroll
    for (int nb = 0; nb < 2; nb++) {
      const int b = 32 * w + 16 * nb + l16;
      if (b < p.batch) {
        rows_in_use |= 0x0F0Fu << (4 * nb);
        unsigned t = p.bound[b];
        t = t < 1u ? 1u : t;
        bkey[nb] = t;
        bm1[nb] = (t - 1u) * 0x00010001u;
      }
    }
  }
  __builtin_amdgcn_s_waitcnt(0);
  int ahead = block;                      // next visit to be requested
  FwdPlace at_ahead(block * p.tile_step, p.tiles_per_chunk), place = at_ahead;   // its place, that of the visit at hand
  const int stride = nblocks * p.tile_step;
  auto issue = [&](int buf) {
    if (ahead < p.n_visit) {
      const int row0 = at_ahead.r * FT;
      fwd_issue_tile<WAVES>(p.chunk[at_ahead.c] + (size_t)row0 * D, min(FT, p.rows_per_chunk - row0), lds0 + (unsigned)buf * FB, w, lane);
    }
    ahead += nblocks;
    at_ahead.advance(stride, p.tiles_per_chunk);
  };
  unsigned mx[2] = {0u, 0u};
  unsigned long long* q_ent = (unsigned long long*)(lds_raw + SEL_BUF * FB) + w * SEL_QUEUE;
  auto emit = [&](unsigned long long ent) {
    const unsigned b = (unsigned)(ent >> 48);
    const unsigned slot = atomicAdd(p.count + b * SEL_COUNT_STRIDE, 1u);
    if (slot < (unsigned)SEL_CAP) {
      p.cand_label[(size_t)b * SEL_CAP + slot] = 0xFFFFFFFFu - (unsigned)ent;
      p.cand_key[(size_t)b * SEL_CAP + slot] = (unsigned short)(ent >> 32);
    }
  };
  // The queue moves to the rows' lists when it is half full and at the end: the list slots come from atomics whose results a
  // wavefront has to wait for, together with its outstanding tile loads.
  int queued = 0;                         // (wave-uniform) entries, those that went to the list because the queue was full included
  auto flush = [&] {
    const int n = queued < SEL_QUEUE ? queued : SEL_QUEUE;
    for (int i = lane; i < n; i += 64) emit(q_ent[i]);
    queued = 0;
  };
  for (int k = 0; k < SEL_BUF - 1; k++) issue(k);
  int buf = 0;
  for (int j = block; j < p.n_visit; j += nblocks) {
    const int row0 = place.r * FT;
    const int rows_valid = min(FT, p.rows_per_chunk - row0);
    const long long label0 = (long long)place.c * p.rows_per_chunk + row0;
    const long long left = p.num_labels - label0;
    const int nvalid = (int)(left < rows_valid ? (left < 0 ? 0 : left) : rows_valid);
    fwd_wait<WAVES, SEL_BUF - 2>(j + (SEL_BUF - 2) * nblocks < p.n_visit);
    __syncthreads();   // the tile has landed for every wavefront, and the one before has been read by all
    if (MODE == 1 && queued > SEL_QUEUE / 2) flush();
    auto other = [&] { issue(buf == 0 ? SEL_BUF - 1 : buf - 1); };
    if (!active) {
      other();
    } else {
      // a lane holds, for batch rows 32w + 16nb + l16, the logits of tile rows 16half + 4kg + e (e = 0..3): the bf16
      // values the dense kernel would store, two to a word, word 4half + 2nb + e / 2
      unsigned wp[8];
#pragma unroll
      for (int half = 0; half < 2; half++) {
        floatx4 z[2];
        const unsigned char* rows = lds_raw + buf * FB + 16 * half * WS;
        if (half == 0) fwd_products(rows, l16, kg, xq, z, other);
        else fwd_products(rows, l16, kg, xq, z, [] {});
#pragma unroll
        for (int nb = 0; nb < 2; nb++) {
          if (p.zscale != 1.0f) z[nb] *= p.zscale;   // the same product as the dense kernel's
          wp[4 * half + 2 * nb] = bf16_pack2(z[nb][0], z[nb][1]);
          wp[4 * half + 2 * nb + 1] = bf16_pack2(z[nb][2], z[nb][3]);
        }
      }
      if (MODE == 0) {
#pragma unroll
        for (int q = 0; q < 8; q++) {
          unsigned kw = key_pair(wp[q]);
          if (nvalid < FT) {   // rows past the end of the chunk or of the labels do not count
            const int r = 16 * (q >> 2) + 4 * kg + 2 * (q & 1);
            kw &= (r < nvalid ? 0x0000FFFFu : 0u) | (r + 1 < nvalid ? 0xFFFF0000u : 0u);
          }
          mx[(q >> 1) & 1] = pk_max_u16(mx[(q >> 1) & 1], kw);
        }
      } else {
        unsigned hit[8], any = 0u, top = 0u;
#pragma unroll
        for (int q = 0; q < 8; q++) {
          const unsigned below = bm1[(q >> 1) & 1];
          hit[q] = pk_max_u16(key_pair(wp[q]), below) ^ below;   // non-zero: a key above bound - 1
          any |= hit[q];
          top = pk_max_u16(top, wp[q]);                          // a half above 0xFF80: a NaN with the sign bit
        }
        const bool nan = pk_max_u16(top, 0xFF80FF80u) != 0xFF80FF80u;   // (a NaN without it has a key above every bound)
        if (__builtin_amdgcn_ballot_w64(any != 0u || nan) != 0) {
          // Candidates go to the wavefront's queue in LDS, one of every lane that has any at a time; their places come from
          // the lanes' ballot.  (One queue per workgroup, its places from an LDS atomic for each value, a move to the lists
          // every eight tiles: all wavefronts waited at the next barrier for the one that was appending.)
          unsigned mask = 0u;   // bit 2q + e of word q
#pragma unroll
          for (int q = 0; q < 8; q++) {
            mask |= (hit[q] & 0xFFFFu) != 0u ? 1u << (2 * q) : 0u;
            mask |= hit[q] >> 16 != 0u ? 2u << (2 * q) : 0u;
          }
          if (__builtin_amdgcn_ballot_w64(nan) != 0) {   // the exact keys decide
            mask = 0u;
#pragma unroll
            for (int q = 0; q < 16; q++)
              mask |= topk_key((unsigned short)(wp[q >> 1] >> (16 * (q & 1)))) >= bkey[(q >> 2) & 1] ? 1u << q : 0u;
          }
          mask &= rows_in_use;
          if (nvalid < FT) {   // rows past the end of the chunk or of the labels do not count
#pragma unroll
            for (int half = 0; half < 2; half++) {
              const int n = nvalid - 16 * half - 4 * kg;
              mask &= ~((n <= 0 ? 0xFFu : n >= 4 ? 0u : ((0xFu << n) & 0xFu) * 0x11u) << (8 * half));
            }
          }
          for (;;) {
            const unsigned long long who = __builtin_amdgcn_ballot_w64(mask != 0u);
            if (who == 0) break;
            if (mask != 0u) {
              const int q = __builtin_ctz(mask);
              mask &= mask - 1u;
              unsigned word = wp[0];
#pragma unroll
              for (int i = 1; i < 8; i++) word = q >> 1 == i ? wp[i] : word;
              const unsigned key = topk_key((unsigned short)(q & 1 ? word >> 16 : word));
              const unsigned b = (unsigned)(32 * w + 4 * (q & 4) + l16);
              const unsigned label = (unsigned)label0 + (unsigned)(2 * (q & 8) + 4 * kg + (q & 3));
              const unsigned long long ent = ((unsigned long long)((b << 16) | key) << 32) | (unsigned long long)(0xFFFFFFFFu - label);
              const int at = queued + (int)__builtin_amdgcn_mbcnt_hi((unsigned)(who >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)who, 0u));
              if (at < SEL_QUEUE) q_ent[at] = ent;
              else emit(ent);   // queue full (many logits at the bound): straight to the list
            }
            queued += __builtin_popcountll(who);
          }
        }
      }
    }
    buf = buf == SEL_BUF - 1 ? 0 : buf + 1;
    place.advance(stride, p.tiles_per_chunk);
  }
  if (MODE == 1) flush();
  if (MODE == 0) {
#pragma unroll
    for (int nb = 0; nb < 2; nb++) {
      unsigned m = mx[nb] & 0xFFFFu, h = mx[nb] >> 16;
      m = m > h ? m : h;
      const unsigned o1 = __shfl_xor(m, 16, 64);
      m = m > o1 ? m : o1;
      const unsigned o2 = __shfl_xor(m, 32, 64);
      m = m > o2 ? m : o2;
      if (kg == 0) p.gmax[(size_t)block * SEL_ROWS + 32 * w + 16 * nb + l16] = (unsigned short)m;
    }
  }
}

}  // namespace xmc
