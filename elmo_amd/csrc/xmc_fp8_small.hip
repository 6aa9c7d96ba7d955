// Fused FP8 extreme-classifier training step for small label spaces and batches on gfx950 (MI355X): two launches that wait for
// nothing but memory.
//
// Work unit = 32 consecutive label rows of one chunk with all their 768 features, one per workgroup: logits, G, grad_X, grad_W and
// the update of a workgroup need no other's data, so there is no exchange, no counter to clear, no table of tiles, and the operand
// images of X and the positives are taken from X and the pairs themselves, by every workgroup, in LDS.  What bounds it is latency:
// one of memory (X, weights and positives are requested together), those of four short stages with a barrier behind each, and the
// first pass over the kernel's code.  The step of xmc_fp8_role.hip, whose quads share a tile, is a launch more and a chain of an
// exchange longer; its tiles leave a 64th of the sums of grad_X, this one's a sum of 48 KiB per 16 batch rows and 32 labels, which
// is why it is not for large label spaces or batches (small_step).  4 K labels, 16 rows, sr_fast: 12.0 us a step in replays of a graph, 14.1 in three
// launches of all quads; launched from the host, 15.7 a pass among others, where the host is what bounds it (18.4), 33 waited for alone (35);
// traced 8.5 and 4.1 (4.1, 7.2 and 3.2 of the three).  64 labels to a workgroup would halve the sums and double the update's vector work.
//
// Reference semantics: as xmc_fp8_role.hip; the weights are the same to the bit (same operands in the same order into the same
// instructions), grad_X up to the order of its fp32 sum.
#include "xmc_common.h"

namespace xmc {

constexpr int SM_ROWS = 32;                  // label rows of a workgroup
constexpr int SM_BATCH = 32;                 // most batch rows
constexpr int SM_POS = 4096;                 // most positives: every workgroup reads all of them (small_step has what they cost)
constexpr int SM_NT = 512;
constexpr int SM_XBS = D * 2 + 16;           // LDS row stride of X in bf16
constexpr int SM_GS = 80;                    // LDS row stride of G, 32 bf16 values
constexpr int SM_W = 0;                                  // weights, rows of QRS bytes; the updated ones take their places
constexpr int SM_XQ = SM_W + SM_ROWS * QRS;              // e4m3 X, rows of QRS bytes
constexpr int SM_XB = SM_XQ + SM_BATCH * QRS;            // bf16 X, 32 rows
constexpr int SM_GL = SM_XB + 32 * SM_XBS;               // G [label][batch row]
constexpr int SM_GB = SM_GL + SM_ROWS * SM_GS;           // G [batch row][label]
constexpr int SM_POSM = SM_GB + SM_BATCH * SM_GS;        // positives: a word for every label, a bit for every batch row
constexpr int SM_LDS = SM_POSM + SM_ROWS * 4;
static_assert(SM_LDS <= 160 * 1024 && SM_XB % 16 == 0 && SM_GL % 16 == 0, "LDS budget");

struct SmallParams {
  unsigned char* chunk[MAX_CHUNKS];
  unsigned seed[MAX_CHUNKS];
  int rows_per_chunk, tiles_per_chunk, num_tiles;   // tiles of SM_ROWS labels
  const unsigned short* x;
  const int2* coo;
  int nnz, batch;
  float inv_scale_x, zscale, lr_eff;
  floatx4* partial;      // [tile][NB][48 feature blocks][64 lanes]
  int* flags;
};

// NB: blocks of 16 batch rows, 1 or 2
template <int MODE, int NB>
__global__ __launch_bounds__(SM_NT, 1) void fp8_small_step_kernel(const SmallParams p) {
  extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
  qlds_u8* lds = (qlds_u8*)lds_raw;
  typedef __attribute__((address_space(3))) unsigned lds_u32;
  typedef __attribute__((address_space(3))) rux2 lds_u2;
  typedef __attribute__((address_space(3))) intx4 lds_i4;
  typedef __attribute__((address_space(3))) unsigned short lds_u16;
  // fp8 conversions saturate at +-448 instead of returning NaN (MODE.FP16_OVFL), as r_update_piece expects
  asm volatile("s_setreg_imm32_b32 hwreg(HW_REG_MODE, 23, 1), 1");
  const int tid = threadIdx.x, g = blockIdx.x;
  const int v = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, l16 = lane & 15, kg = lane >> 4;
  if (tid == 0) {
    p.flags[QF_XCC + g] = (int)(__builtin_amdgcn_s_getreg((3 << 11) | 20) & 15);   // (xmc_step_xcc_ids)
    if (g == 0) p.flags[QF_ERR] = 0;
  }
  if (g >= p.num_tiles) return;
  const int c = g / p.tiles_per_chunk, row0 = (g - c * p.tiles_per_chunk) * SM_ROWS;
  const int valid = min(SM_ROWS, p.rows_per_chunk - row0);
  const unsigned label0 = (unsigned)(c * p.rows_per_chunk + row0);
  unsigned char* wbase = p.chunk[c] + (size_t)row0 * D;

  // ---- X, the weights and the first positives, all requested at once
  constexpr int XP = D * 2 / 16, XN = 16 * XP / SM_NT, WP = D / 16, WN = SM_ROWS * WP / SM_NT;   // pieces of a row; of a thread
  static_assert(XN * SM_NT == 16 * XP && WN * SM_NT == SM_ROWS * WP, "whole pieces");
  uint4 xr[NB * XN];
  intx4 wr[WN];
#pragma unroll
  for (int s = 0; s < NB * XN; s++) xr[s] = ((const uint4*)p.x)[tid + SM_NT * s];   // (the batch is a multiple of 16)
#pragma unroll
  for (int s = 0; s < WN; s++) {
    const int ch = tid + SM_NT * s, row = min(ch / WP, valid - 1);   // (rows past the end re-read the last: their G is zero)
    wr[s] = *(const intx4*)(wbase + row * D + ch % WP * 16);
  }
  int2 e0 = {-1, -1};
  if (tid < p.nnz) e0 = p.coo[tid];
  if (tid < SM_ROWS) *(lds_u32*)(lds + SM_POSM + tid * 4) = 0u;
  if constexpr (NB == 1) {   // the upper half of a K step of 32 batch rows
    if (tid < SM_ROWS * 2) *(lds_i4*)(lds + SM_GL + (tid >> 1) * SM_GS + 32 + (tid & 1) * 16) = intx4{0, 0, 0, 0};
#pragma unroll
    for (int s = 0; s < XN; s++) {
      const int ch = tid + SM_NT * s;
      *(lds_i4*)(lds + SM_XB + (16 + ch / XP) * SM_XBS + ch % XP * 16) = intx4{0, 0, 0, 0};
    }
  }
  __syncthreads();
#pragma unroll
  for (int s = 0; s < NB * XN; s++) {
    const int ch = tid + SM_NT * s, row = ch / XP, at = ch % XP;
    auto val = [&](unsigned bits) { return clamp448(__uint_as_float(bits) * p.inv_scale_x); };
    auto pack = [&](unsigned a, unsigned b) {
      const int lo = __builtin_amdgcn_cvt_pk_fp8_f32(val(a << 16), val(a & 0xFFFF0000u), 0, false);
      return (unsigned)__builtin_amdgcn_cvt_pk_fp8_f32(val(b << 16), val(b & 0xFFFF0000u), lo, true);
    };
    *(lds_i4*)(lds + SM_XB + row * SM_XBS + at * 16) = __builtin_bit_cast(intx4, xr[s]);
    *(lds_u32*)(lds + SM_XQ + row * QRS + at * 8) = pack(xr[s].x, xr[s].y);
    *(lds_u32*)(lds + SM_XQ + row * QRS + at * 8 + 4) = pack(xr[s].z, xr[s].w);
  }
#pragma unroll
  for (int s = 0; s < WN; s++) {
    const int ch = tid + SM_NT * s;
    *(lds_i4*)(lds + SM_W + ch / WP * QRS + ch % WP * 16) = wr[s];
  }
  for (int i = tid; i < p.nnz;) {
    const unsigned rel = (unsigned)e0.y - label0;
    if (rel < (unsigned)valid && (unsigned)e0.x < (unsigned)p.batch)
      __hip_atomic_fetch_or((lds_u32*)(lds + SM_POSM + rel * 4), 1u << e0.x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    i += SM_NT;
    if (i < p.nnz) e0 = p.coo[i];
  }
  __syncthreads();

  // ---- logits of 16 labels and 16 batch rows, a wavefront each; G to both places
  if (v < 2 * NB) {
    const int rb = v & 1, nb = v >> 1;
    const unsigned wa = (unsigned)(SM_W + (16 * rb + l16) * QRS + kg * 16), xa = (unsigned)(SM_XQ + (16 * nb + l16) * QRS + kg * 16);
    // (the K order of stage A of the role kernel)
    intx4 wl[6], wh[6], xl[6], xh[6];
#pragma unroll
    for (int ks = 0; ks < 6; ks++) {
      wl[ks] = *(const lds_i4*)(lds + wa + ks * 128); wh[ks] = *(const lds_i4*)(lds + wa + ks * 128 + 64);
      xl[ks] = *(const lds_i4*)(lds + xa + ks * 128); xh[ks] = *(const lds_i4*)(lds + xa + ks * 128 + 64);
    }
    floatx4 z = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < 6; ks++) {
      const intx8 a = {wl[ks].x, wl[ks].y, wl[ks].z, wl[ks].w, wh[ks].x, wh[ks].y, wh[ks].z, wh[ks].w};
      const intx8 b = {xl[ks].x, xl[ks].y, xl[ks].z, xl[ks].w, xh[ks].x, xh[ks].y, xh[ks].z, xh[ks].w};
      z = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b, z, 0, 0, 0, 0, 0, 0);
    }
    const float nlog2e = -1.44269504088896340736f;
    const int r0 = 16 * rb + 4 * kg;   // this lane's labels r0 .. r0 + 3 of batch row 16 nb + l16
    unsigned hit = 0u, gp[2];
#pragma unroll
    for (int e = 0; e < 4; e++) hit |= (*(const lds_u32*)(lds + SM_POSM + (r0 + e) * 4) >> (16 * nb + l16) & 1u) << e;
#pragma unroll
    for (int e2 = 0; e2 < 2; e2++) {
      const unsigned zb = bf16_pack2(z[2 * e2] * p.zscale, z[2 * e2 + 1] * p.zscale);
      const float z0 = __uint_as_float(zb << 16), z1 = __uint_as_float(zb & 0xFFFF0000u);
      gp[e2] = bf16_pack2(__builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(z0 * nlog2e)), __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(z1 * nlog2e)));
      gp[e2] = minus_hits(gp[e2], hit, 2 * e2);
      if (r0 + 2 * e2 >= valid) gp[e2] &= 0xFFFF0000u;   // rows past the end of the chunk contribute nothing
      if (r0 + 2 * e2 + 1 >= valid) gp[e2] &= 0x0000FFFFu;
    }
    *(lds_u2*)(lds + SM_GB + (16 * nb + l16) * SM_GS + r0 * 2) = rux2{gp[0], gp[1]};
#pragma unroll
    for (int e = 0; e < 4; e++) *(lds_u16*)(lds + SM_GL + (r0 + e) * SM_GS + (16 * nb + l16) * 2) = (unsigned short)(gp[e >> 1] >> (16 * (e & 1)));
  }
  __syncthreads();

  // ---- grad_X and the update of 96 features, a wavefront each: it alone touches these columns of the weights from here on
  {
    const int f0 = 96 * v;
    bf16x8 gb[NB];
#pragma unroll
    for (int nb = 0; nb < NB; nb++) gb[nb] = *(const __attribute__((address_space(3))) bf16x8*)(lds + SM_GB + (16 * nb + l16) * SM_GS + kg * 16);
    floatx4* dst = p.partial + (size_t)g * (NB * 48 * 64) + lane;
#pragma unroll
    for (int fb = 0; fb < 6; fb++) {
      // labels 8 kg .. 8 kg + 7 of feature f0 + 16 fb + l16
      const intx2 raw = __builtin_amdgcn_ds_read_tr8_b64_v2i32((__attribute__((address_space(3))) intx2*)(lds + SM_W + (8 * kg + (l16 >> 1)) * QRS + f0 + 16 * fb + (l16 & 1) * 8));
      const bf16x8 wb = q_fp8x8_to_bf16x8(raw);
#pragma unroll
      for (int nb = 0; nb < NB; nb++)
        dst[(nb * 48 + 6 * v + fb) * 64] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(gb[nb], wb, floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    }
    QTile qt = {};
    qt.seed = p.seed[c];
    qt.row0 = row0;
    const unsigned hash_tile = label0 * (unsigned)(D / 4) * 0x9E3779B1u + qt.seed;
    const RKahanBlock nok = {};
    // (rolled: the first pass over code costs 1.5 to 2 clocks a byte)
#pragma unroll 1
    for (int f = 0; f < 2; f++) {
      const int fc = f0 + 48 * f;   // features fc + 12 kg .. + 11 of a label row to a lane (layout of xt in xmc_fp8_quad.hip)
      RBlockLane bl = {};
      bl.gcol = (unsigned)(fc + 12 * kg);
      bl.hash_lane = ((unsigned)l16 * (unsigned)(D / 4) + (bl.gcol >> 2)) * 0x9E3779B1u;
      bl.orow_lane = (unsigned)(l16 * QRS) + bl.gcol;
      bf16x8 xt[3];
#pragma unroll
      for (int cg = 0; cg < 3; cg++) {
        const unsigned at = (unsigned)(SM_XB + (8 * kg + (l16 >> 2)) * SM_XBS + 2 * (fc + 12 * (l16 & 3) + 4 * cg));
        const shortx4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) shortx4*)(lds + at));
        const shortx4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) shortx4*)(lds + at + 4 * SM_XBS));
        xt[cg] = __builtin_bit_cast(bf16x8, shortx8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]});
      }
#pragma unroll 1
      for (int rb = 0; rb < 2; rb++) {
        const bf16x8 gl = *(const __attribute__((address_space(3))) bf16x8*)(lds + SM_GL + (16 * rb + l16) * SM_GS + kg * 16);
        floatx4 ab[3];
        unsigned wq[3], hs[3], outw[3], knew[6];
        float t[3][4];
#pragma unroll
        for (int cg = 0; cg < 3; cg++) {
          ab[cg] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xt[cg], gl, floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
          wq[cg] = *(const lds_u32*)(lds + SM_W + 16 * rb * QRS + bl.orow_lane + 4 * cg);
        }
        // (its place in the image counts rows of QCOLS bytes)
#pragma unroll
        for (int pc = 0; pc < 8; pc++)
          r_update_piece<MODE, false, 0>(pc, rb, ab, wq, t, hs, outw, knew, bl, qt, hash_tile, p.lr_eff, 0.f, l16, lds, (unsigned)(SM_W + 16 * rb * (QRS - QCOLS)), nok, 0u, 0);
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int s = 0; s < WN; s++) {
    const int ch = tid + SM_NT * s, row = ch / WP;
    if (row < valid) *(intx4*)(wbase + row * D + ch % WP * 16) = *(const lds_i4*)(lds + SM_W + row * QRS + ch % WP * 16);
  }
}

// grad_X = scale * sum over the tiles' sums, in a fixed order; fp32 and bf16 [batch, 768].  Workgroup (16-row batch block, 16 features),
// its eight wavefronts an eighth of the tiles each, eight loads in flight.
constexpr int SM_RW = 8;
__global__ __launch_bounds__(SM_RW * 64) void fp8_small_reduce_kernel(const floatx4* partial, int tiles, int blocks, float scale, float* gx_f32,
                                                               unsigned short* gx_bf16, int* flags, int* failure_word) {
  if (blockIdx.x == 0 && threadIdx.x == 0) report_step_error(flags + QF_ERR, flags + QF_STICKY, failure_word);
  const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63, l16 = lane & 15, kg = lane >> 4;
  const floatx4* src = partial + (size_t)blockIdx.x * 64 + lane;
  floatx4 sum = {0.f, 0.f, 0.f, 0.f};
  for (int t = wv; t < tiles; t += 8 * SM_RW) {
    floatx4 pv[8];
#pragma unroll
    for (int u = 0; u < 8; u++) pv[u] = t + SM_RW * u < tiles ? src[(size_t)(t + SM_RW * u) * blocks * 64] : floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < 8; u++) sum += pv[u];
  }
  __shared__ floatx4 part[SM_RW - 1][64];
  if (wv > 0) part[wv - 1][lane] = sum;
  __syncthreads();
  if (wv > 0) return;
#pragma unroll
  for (int q = 0; q < SM_RW - 1; q++) sum += part[q][lane];
  const int nb = blockIdx.x / 48, col = (blockIdx.x - nb * 48) * 16 + l16;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int b = 16 * nb + 4 * kg + i;
    const float val = sum[i] * scale;
    if (gx_f32) gx_f32[(size_t)b * D + col] = val;
    if (gx_bf16) gx_bf16[(size_t)b * D + col] = bf16_bits(val);
  }
}

typedef void (*small_kernel_t)(const SmallParams);
inline small_kernel_t small_variant(int round_mode, int batch) {
  const bool one = batch <= 16;
  return round_mode == ROUND_RTN ? (one ? fp8_small_step_kernel<ROUND_RTN, 1> : fp8_small_step_kernel<ROUND_RTN, 2>)
       : round_mode == ROUND_SR_FAST ? (one ? fp8_small_step_kernel<ROUND_SR_FAST, 1> : fp8_small_step_kernel<ROUND_SR_FAST, 2>)
       : (one ? fp8_small_step_kernel<ROUND_SR_PHILOX, 1> : fp8_small_step_kernel<ROUND_SR_PHILOX, 2>);
}
inline void small_set_lds() {
  for (int mode = ROUND_RTN; mode <= ROUND_SR_FAST; mode++)
    for (int batch = 16; batch <= SM_BATCH; batch += 16)
      (void)hipFuncSetAttribute((const void*)small_variant(mode, batch), hipFuncAttributeMaxDynamicSharedMemorySize, SM_LDS);
}

}  // namespace xmc
