// Fused FP8 extreme-classifier training step for gfx950 (MI355X), second generation: the four compute units of a quad
// share a tile stream as in xmc_fp8_quad.hip, but the two wavefronts of every SIMD have different jobs.
//
// Work unit = a tile of 64 consecutive label rows of one chunk (64 x 768 e4m3 bytes, contiguous in HBM).  Member m of
// a quad (four workgroups of 512 threads on one XCD, one per compute unit) owns label rows 16m..16m+15 of every tile
// for the logits ("stage A") and input features 192m..192m+191 for grad_X, grad_W and the update ("stage B").
//
//   wavefronts 0-3 ("A", one per SIMD): every vector-memory instruction of the tile loop (loads of weight rows, weight
//     columns, the G tiles of the partners and counters; stores of G and of the updated weights), and stage A for 32
//     batch rows each:
//       Z[16 labels x 32 rows] = W_t[16m.., :] Xq[32a.., :]^T  v_mfma_scale_f32_16x16x128_f8f6f4, Xq resident (96 registers)
//       G = bf16(sigmoid(bf16(Z))) - [positive], stored to the quad's exchange slot in global memory
//   wavefronts 4-7 ("B", one per SIMD): stage B for 48 features each, all batch rows:
//       grad_X[128 x 48] += G^T W_t   v_mfma_f32_16x16x32_bf16, accumulators resident (96 registers)
//       A^T[48 x 64]      = X^T G^T    same instruction, X^T resident (48 registers)
//       W_t = round(W_t - lr A), 12 bytes per lane and row to an image of the tile's updated weights in LDS; the A
//       wavefronts store the image one iteration later, as whole 192-byte row segments
// A B wavefront issues no memory operation inside the tile loop and never waits for memory: its operands are in LDS
// when the per-tile barrier releases it.  The A wavefronts have slack (their matrix work is a fifth of a B
// wavefront's) and absorb the issue cost and latency of the loads and stores.
//
// The exchange: stage A runs RQ tiles ahead of stage B.  An A wavefront stores its part of G(t), waits for the stores at
// the end of the same iteration and then advances its own "tiles published" counter (sixteen counters per quad: member x
// A wavefront).  A wavefront a gathers block a of the next tile's G (the 4 KiB member a produced) after it has seen the
// four counters of member a's wavefronts, normally in a snapshot that arrived in LDS with the other loads of the
// iteration before; a bounded polling loop with an error word is the fallback.  The G tile is laid out member-major
// with a swizzle ([member][row'][quarter'] of 8 bytes) so that an A wavefront stores 512 contiguous bytes, the gather
// is a linear copy of 16 KiB, and both operand reads of stage B are free of LDS bank conflicts.
//
// Reference semantics: src/xmc_classifiers/chunked_fp8xmc_clf.py:81-123 with
// src/triton_kernels/matmul_kernel.py:204-239 (grad_X) and src/triton_kernels/fuse_kernel.py:63-113 (update).
#include "xmc_common.h"

namespace xmc {

#ifndef XMC_NB_B
#define XMC_NB_B 3
#endif
#ifndef XMC_PD
#define XMC_PD 3
#endif
constexpr int NB_B = XMC_NB_B;              // A^T blocks (16 label rows) of a tile the B wavefronts take; the A wavefronts take the rest
// with a compensated head (KT != 0) the B wavefronts take all four: they alone then touch the compensation buffer, with
// ordinary loads and stores whose completion the compiler tracks (the A wavefronts count their loads by hand)
// With the reference's Philox recipe the update is a hundred vector instructions per weight and bounds the kernel: the
// two wavefronts of a SIMD then share it evenly.
constexpr int r_nbb(int kt, int mode, int nk) { return kt != 0 ? 4 : mode == ROUND_SR_PHILOX ? 2 : nk < 4 ? 4 : NB_B; }
constexpr int RR_RING = 3;                  // own-rows images: in use, landed, landing
constexpr int RG_BUF = 2;                   // gathered G tiles: in use, landing
constexpr int RG_BYTES = 16384;             // one G tile: 4 members x 128 rows x 32 bytes
constexpr int RO_RING = 2;                  // images of updated weights: being written, being stored to memory
constexpr int RO_BYTES = TL * QCOLS;         // image of updated weights: 64 rows x 192 bytes, no padding
constexpr int RROW_BYTES = 16 * QRS;        // own-rows image: 16 rows x 800 bytes (the 13th wave-wide piece is half a piece)
// LDS of the variant for compensation terms of type KT (0: none, 1: bf16, 2: e5m2)
template <int KT> struct RGeom {
  // Stage A runs this many tiles ahead of stage B.  (A member may start tile i when its partners have published tile i + 1, which they do
  // at the end of iteration i + 2 - RQ: with 4 that is an iteration ago, with 3 just now, which the longer tiles of a compensated head
  // do not notice.  2 would be too late.)
  static constexpr int RQ = KT != 0 ? 3 : 4;
  static constexpr int RC_RING = RQ + 1;             // own-column images: in use, RQ - 1 landed, one landing
  static constexpr int C = 0;
  static constexpr int O = C + RC_RING * QWC_BYTES;
  static constexpr int G = O + RO_RING * RO_BYTES;
  static constexpr int R = G + RG_BUF * RG_BYTES;
  static constexpr int M = R + RR_RING * RROW_BYTES;   // per A wavefront two snapshots of four counters (32 bytes); at +128 two abort words
  static constexpr int T = M + 160;                    // what the B wavefronts need to know of a tile: two entries of 16 bytes
  static constexpr int P = M + 256;                    // masks of positives of the A wavefronts, 64 bytes each (positive_hits)
  // compensation terms: per B wavefront KSLOTS blocks of 16 rows x 48 features, as they lie in memory
  static constexpr int K = P + 256;
  static constexpr int KROW = KT == 1 ? 96 : 48;       // bytes of a row of a block
  static constexpr int KSLOT = 16 * KROW;
  static constexpr int KSLOTS = 2;                     // requested this many blocks ahead
  static constexpr int KLOADS = KT == 1 ? 2 : 1;       // loads, and stores, of a block (64 + 32 or 48 pieces of 16 bytes)
  static constexpr int BYTES = K + (KT != 0 ? 4 * KSLOTS * KSLOT : 0);
  static_assert(BYTES <= 160 * 1024, "LDS budget");
};
// tiles-published counters: flags[p.cnt_base + quad*16 + member*4 + A wavefront]

// row permutation within sixteen rows of the G image: rows 8..11 and 12..15 trade places, so that the four row groups
// a transposing read touches (rows 8kg..8kg+3) fall into different halves of the LDS banks
__device__ __forceinline__ int g_row16(int r) { return r ^ ((r >> 1) & 4); }

// Everything a wavefront needs for the A^T blocks it takes (features 192m + 48f .. +47 of label rows 16nb..16nb+15):
// per-lane address parts, the resident X^T operand and the state of the update under way.
struct RBlockLane {
  unsigned bg_lane;      // G tile, transposing read: rows 8kg + l16/4, quarter l16%4
  unsigned wrow_lane;    // own-column image: old weights of row l16, 12 bytes
  unsigned orow_lane;    // image of updated weights: the same 12 bytes
  unsigned gcol;         // first of the lane's 12 features
  unsigned hash_lane;    // lane part of the random-word hash
};

// The compensation terms of one A^T block (head-Kahan layer): 12 per lane, raw (bf16: six dwords, e5m2: three), and
// whether the lane's row carries one at all.
struct RKahanBlock { unsigned raw[6]; bool head; int row; };
typedef unsigned rux2 __attribute__((ext_vector_type(2)));

// piece c (0..7) of the update of A^T block nb (12 weights per lane): pieces 0-2 decode the old weights and form
// T = W - lr A, 3-5 make the random words' hashes, 6-7 round, 7 stores.  Split so that the vector instructions can be
// issued between matrix instructions.  With MODE.FP16_OVFL set the fp8 converters saturate, so nothing is clamped here.
//
// KT != 0 (compensation buffer of bf16 (1) or e5m2 (2) values, chunked_head_kahan_fp8xmc_clf.py:127-131 with
// fuse_kernel.py:237-262): on rows that carry a term k the update is
//   T = (W + k) - lr A,  W' = round(T),  k' = cast(((k + W) - W') - lr A)
// and on the other rows of the tile (behind the head's end) the plain update, whose random offsets count from that end.
template <int MODE, bool WD, int KT>
__device__ __forceinline__ void r_update_piece(int c, int nb, const floatx4 (&ab)[3], const unsigned (&wq)[3], float (&t)[3][4],
                                               unsigned (&hs)[3], unsigned (&outw)[3], unsigned (&knew)[6], const RBlockLane& bl, const QTile& q,
                                               unsigned hash_tile, float lr_eff, float wd_eff, int l16, qlds_u8* lds, unsigned oimg,
                                               const RKahanBlock& kb, unsigned kterm, int num_head) {
  // W + k of column group cg (exact decode of both; k = 0 on rows without a term)
  auto kahan_sum = [&](int cg, float (&s)[4]) {
    const unsigned wv = wq[cg];
    floatx2 w01 = __builtin_amdgcn_cvt_pk_f32_fp8((int)wv, false), w23 = __builtin_amdgcn_cvt_pk_f32_fp8((int)wv, true);
    float k[4];
    if (KT == 1) {
      k[0] = __uint_as_float(kb.raw[2 * cg] << 16); k[1] = __uint_as_float(kb.raw[2 * cg] & 0xFFFF0000u);
      k[2] = __uint_as_float(kb.raw[2 * cg + 1] << 16); k[3] = __uint_as_float(kb.raw[2 * cg + 1] & 0xFFFF0000u);
    } else {
      floatx2 k01 = __builtin_amdgcn_cvt_pk_f32_bf8((int)kb.raw[cg], false), k23 = __builtin_amdgcn_cvt_pk_f32_bf8((int)kb.raw[cg], true);
      k[0] = k01.x; k[1] = k01.y; k[2] = k23.x; k[3] = k23.y;
    }
    s[0] = w01.x + k[0]; s[1] = w01.y + k[1]; s[2] = w23.x + k[2]; s[3] = w23.y + k[3];
  };
  if (c < 3) {
    const int cg = c;
    const unsigned wv = wq[cg];
    floatx2 w01 = __builtin_amdgcn_cvt_pk_f32_fp8((int)wv, false), w23 = __builtin_amdgcn_cvt_pk_f32_fp8((int)wv, true);
    if (KT != 0) {
      float s[4];
      kahan_sum(cg, s);
#pragma unroll
      for (int e = 0; e < 4; e++) t[cg][e] = __builtin_fmaf(-lr_eff, ab[cg][e], s[e]);
    } else if (WD) {   // T = W - lr (A + wd W): the decayed gradient first, in fp32
      t[cg][0] = __builtin_fmaf(-lr_eff, __builtin_fmaf(wd_eff, w01.x, ab[cg][0]), w01.x);
      t[cg][1] = __builtin_fmaf(-lr_eff, __builtin_fmaf(wd_eff, w01.y, ab[cg][1]), w01.y);
      t[cg][2] = __builtin_fmaf(-lr_eff, __builtin_fmaf(wd_eff, w23.x, ab[cg][2]), w23.x);
      t[cg][3] = __builtin_fmaf(-lr_eff, __builtin_fmaf(wd_eff, w23.y, ab[cg][3]), w23.y);
    } else {
      t[cg][0] = __builtin_fmaf(-lr_eff, ab[cg][0], w01.x); t[cg][1] = __builtin_fmaf(-lr_eff, ab[cg][1], w01.y);
      t[cg][2] = __builtin_fmaf(-lr_eff, ab[cg][2], w23.x); t[cg][3] = __builtin_fmaf(-lr_eff, ab[cg][3], w23.y);
    }
  } else if (c < 6) {
    const int cg = c - 3;
    if (MODE == ROUND_SR_FAST) {
      // fast_mix(idx, seed) with idx = (label0 + 16nb + l16) * 192 + (gcol + 4cg) / 4: the product idx * 0x9E3779B1 is
      // the sum of a per-tile scalar, a per-lane constant and a literal
      unsigned h = bl.hash_lane + (hash_tile + (unsigned)(16 * nb * (D / 4) + cg) * 0x9E3779B1u);
      h ^= h >> 16; h *= 0x85EBCA77u; h ^= h >> 15;
      hs[cg] = h;
    }
    if (MODE == ROUND_SR_PHILOX) {
      // the reference's recipe on this column group's four targets, one Philox word after the other: the counter of
      // the next word passes through an opaque statement together with this word's result, so that the four chains of
      // ten rounds are not interleaved (forty live registers that this kernel does not have)
      const int row = 16 * nb + l16;
      const int rrow = KT != 0 ? (kb.head ? kb.row : kb.row - num_head) : q.row0 + row;
      unsigned off = (unsigned)rrow * (unsigned)D + bl.gcol + 4 * cg;
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const unsigned r = philox_word0(off + e, q.seed, 0u) & 0xFFFFFu;
        unsigned tb = (__float_as_uint(t[cg][e]) + r) & 0xFFF00000u;
        asm volatile("" : "+v"(off), "+v"(tb));
        t[cg][e] = __uint_as_float(tb);
      }
    }
  } else {
#pragma unroll
    for (int cg = (c == 6 ? 0 : 2); cg < (c == 6 ? 2 : 3); cg++) {
      if (MODE == ROUND_SR_FAST) {
        int packed;
        asm volatile("" : "=v"(packed));   // every byte is written below
        packed = __builtin_amdgcn_cvt_sr_fp8_f32(t[cg][0], fast_word(hs[cg], 0), packed, 0);
        packed = __builtin_amdgcn_cvt_sr_fp8_f32(t[cg][1], fast_word(hs[cg], 1), packed, 1);
        packed = __builtin_amdgcn_cvt_sr_fp8_f32(t[cg][2], fast_word(hs[cg], 2), packed, 2);
        packed = __builtin_amdgcn_cvt_sr_fp8_f32(t[cg][3], fast_word(hs[cg], 3), packed, 3);
        outw[cg] = (unsigned)packed;
      } else {
        // round to nearest (the Philox recipe has been applied to T by now); the converter saturates
        int packed;
        asm volatile("" : "=v"(packed));   // every byte is written below
        packed = __builtin_amdgcn_cvt_pk_fp8_f32(t[cg][0], t[cg][1], packed, false);
        packed = __builtin_amdgcn_cvt_pk_fp8_f32(t[cg][2], t[cg][3], packed, true);
        outw[cg] = (unsigned)packed;
      }
      if (KT != 0) {
        float s[4], kn[4];
        kahan_sum(cg, s);
        floatx2 n01 = __builtin_amdgcn_cvt_pk_f32_fp8((int)outw[cg], false), n23 = __builtin_amdgcn_cvt_pk_f32_fp8((int)outw[cg], true);
        kn[0] = __builtin_fmaf(-lr_eff, ab[cg][0], s[0] - n01.x); kn[1] = __builtin_fmaf(-lr_eff, ab[cg][1], s[1] - n01.y);
        kn[2] = __builtin_fmaf(-lr_eff, ab[cg][2], s[2] - n23.x); kn[3] = __builtin_fmaf(-lr_eff, ab[cg][3], s[3] - n23.y);
        if (KT == 1) {
          knew[2 * cg] = bf16_pack2(kn[0], kn[1]); knew[2 * cg + 1] = bf16_pack2(kn[2], kn[3]);
        } else {
#pragma unroll
          for (int e = 0; e < 4; e++) kn[e] = __builtin_fminf(__builtin_fmaxf(kn[e], -57344.0f), 57344.0f);
          int pk = 0;
          pk = __builtin_amdgcn_cvt_pk_bf8_f32(kn[0], kn[1], pk, false);
          pk = __builtin_amdgcn_cvt_pk_bf8_f32(kn[2], kn[3], pk, true);
          knew[cg] = (unsigned)pk;
        }
      }
    }
    if (KT != 0 && c == 7) {   // the new terms to the place of the old ones in LDS
#pragma unroll
      for (int cg = 0; cg < 3; cg++) {
        if (KT == 1) *(__attribute__((address_space(3))) rux2*)(lds + kterm + 8 * cg) = rux2{knew[2 * cg], knew[2 * cg + 1]};
        else *(__attribute__((address_space(3))) unsigned*)(lds + kterm + 4 * cg) = knew[cg];
      }
    }
    if (c == 7) {
      // the block's 12 bytes per lane go to the image of updated weights in LDS (rows of 192 bytes);
      // the image is stored to memory as whole 192-byte row segments in the next iteration
      typedef unsigned uintx3 __attribute__((ext_vector_type(3)));
      *(__attribute__((address_space(3))) uintx3*)(lds + oimg + bl.orow_lane + 16 * nb * QCOLS) = uintx3{outw[0], outw[1], outw[2]};
    }
  }
}

template <int MODE, bool WD, int KT, int NK>
__global__ __launch_bounds__(QNT, 1) void fp8_step_role_kernel(const QuadParams p) {
  constexpr int NBB = r_nbb(KT, MODE, NK);      // A^T blocks of a tile the B wavefronts take
  constexpr int NBA = 4 - NBB > 0 ? 4 - NBB : 1;
  typedef RGeom<KT> Geo;
  constexpr int RQ = Geo::RQ, RC_RING = Geo::RC_RING, RLDS_C = Geo::C, RLDS_O = Geo::O, RLDS_G = Geo::G, RLDS_R = Geo::R, RLDS_M = Geo::M, RLDS_T = Geo::T, RLDS_P = Geo::P;
  constexpr int AB = NK > 2 ? 2 : 1;            // 16-row batch blocks of an A wavefront's logits: 4 NK / 2 of the 4 wavefronts' have any
  extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
  qlds_u8* lds = (qlds_u8*)lds_raw;
  // fp8 conversions saturate at +-448 instead of returning NaN (MODE.FP16_OVFL; infinities and NaN still give NaN)
  asm volatile("s_setreg_imm32_b32 hwreg(HW_REG_MODE, 23, 1), 1");

  const int tid = threadIdx.x;
  const int v = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, l16 = lane & 15, kg = lane >> 4;
  const int g = blockIdx.x;
  const int xcd = g & 7, j = g >> 3, m = j & 3;
  const int nquads = gridDim.x >> 2;
  const int quad = (j >> 2) * 8 + xcd;
  int n_it = quad < p.run_tiles ? (p.run_tiles - quad + nquads - 1) / nquads : 0;
  // (test aid: with a polling limit of 0 the second member leaves after three tiles, as if it had stopped, and its partners' waits expire)
  if (m == 1 && p.spin_limit == 0) n_it = min(n_it, 3);

  q_cdesc* cdesc = (q_cdesc*)p.desc;
  // descriptor entry of position k in this quad's sequence; positions past the end fall back to entry 0 (tile 0), whose
  // data is loaded and never used
  auto tile_at = [&](int k) { return k < n_it ? quad * p.kmax + k : 0; };
  unsigned char* exq = p.exch + (size_t)quad * QSLOTS * QG_BYTES;   // this quad's ring of exchange slots
  int* errw = p.flags + QF_ERR;
  typedef __attribute__((address_space(3))) int lds_int;
  // the XCD this workgroup really runs on: the reduction kernel compares the four members of every quad
  if (tid == 0) {
    p.flags[QF_XCC + g] = (int)(__builtin_amdgcn_s_getreg((3 << 11) | 20) & 15);   // XCC_ID
    *(lds_int*)(lds + RLDS_M + 128) = 0;
    *(lds_int*)(lds + RLDS_M + 132) = 0;
  }
  // abort word written during iteration i (a bounded wait expired): slot i & 1; everybody reads it behind the next barrier
  const unsigned abort_base = (unsigned)(RLDS_M + 128);

  // the wavefront's share of stage B: features 192m + 48f .. +47 (f = its SIMD)
  const int f = v & 3;
  RBlockLane bl;
  bl.bg_lane = (unsigned)((kg >> 1) * 512 + g_row16(8 * (kg & 1) + (l16 >> 2)) * 32 + (((((l16 >> 1) & 1) ^ (kg & 1)) << 1) | (l16 & 1)) * 8);
  bl.wrow_lane = (unsigned)(l16 * QWS + 48 * f + 12 * kg);
  bl.orow_lane = (unsigned)(l16 * QCOLS + 48 * f + 12 * kg);
  bl.gcol = (unsigned)(QCOLS * m + 48 * f + 12 * kg);
  bl.hash_lane = ((unsigned)l16 * (unsigned)(D / 4) + (bl.gcol >> 2)) * 0x9E3779B1u;
  bf16x8 xt[3][NK];      // grad_W: feature blocks of this wavefront's 48 features, K steps of 32 batch rows
#pragma unroll
  for (int cg = 0; cg < 3; cg++)
#pragma unroll
    for (int ks = 0; ks < NK; ks++) xt[cg][ks] = p.xt[(size_t)(((4 * m + f) * 3 + cg) * 4 + ks) * 64 + lane];
  // operand of A^T block nb, K step ks (32 batch rows): two transposing reads
  auto read_bg = [&](unsigned gwl, unsigned gwh, int nb, int ks) {
    shortx4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) shortx4*)(lds + gwl + nb * 4096 + ks * 1024));
    shortx4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) shortx4*)(lds + gwh + nb * 4096 + ks * 1024));
    return __builtin_bit_cast(bf16x8, shortx8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]});
  };

  // hash part, seed and first row of the tile of an iteration, for the B wavefronts (slot: iteration & 1)
  typedef __attribute__((address_space(3))) intx4 lds_intx4;
  auto pass_on = [&](int slot, const QTile& q) {
    if (lane == 0) *(lds_intx4*)(lds + RLDS_T + slot * 16) = intx4{(int)(q.label0 * (unsigned)(D / 4) * 0x9E3779B1u + q.seed), (int)q.seed, q.row0, 0};
  };

  if (v < 4) {
    // =========================================================================================== A wavefronts
    const int a = v;
    int* myflag = p.flags + p.cnt_base + quad * 16 + m * 4 + a;
    const int* srcflags = p.flags + p.cnt_base + quad * 16 + a * 4;

    const bool la = 4 * AB == 2 * NK || a * AB < 2 * NK;   // whether this wavefront has logits to compute
    intx8 xq[AB][6];   // logits operands: batch blocks AB a.., K steps of 128
    if (la) {
#pragma unroll
      for (int blk = 0; blk < AB; blk++)
#pragma unroll
        for (int ks = 0; ks < 6; ks++) xq[blk][ks] = *(const intx8*)(p.xq + ((size_t)(((AB * a + blk) * 6 + ks) * 64 + lane)) * 32);
    }

    // Per-lane byte offsets of the wave-wide 1 KiB pieces this wavefront loads.  own-column image: 64 rows x 13 chunks of
    // 16 bytes (12 data + 1 pad) = 13 pieces; own-rows image: rows 16m..16m+15, 16 x 50 chunks (48 data + 2 pad) = 13
    // pieces.  Wavefront a takes column pieces a, a+4, a+8 (and 12 if a == 0) and row pieces ra, ra+4, ra+8 (and 12 if
    // ra == 0) with ra = (a + 3) % 4, so that no wavefront has both extra pieces.
    const int ra = (a + 3) & 3;
    auto wcol_offset = [&](int s, int last_row) {
      const int ch = (a + 4 * s) * 64 + lane, wr = ch / 13;
      return __umul24(min(wr, last_row), D) + (unsigned)(QCOLS * m + min(ch - wr * 13, 11) * 16);
    };
    auto rows_offset = [&](int s, int last_row) {
      const int ch = (ra + 4 * s) * 64 + lane, rr = ch / (QRS / 16);
      return __umul24(min(16 * m + min(rr, 15), last_row), D) + (unsigned)(min(ch - rr * (QRS / 16), 47) * 16);
    };
    unsigned woff[4], roff[4];
#pragma unroll
    for (int s = 0; s < 4; s++) {
      woff[s] = wcol_offset(s, TL - 1);
      roff[s] = rows_offset(s, TL - 1);
    }
    // The offsets belong to tiles of w_valid and r_valid rows; a change (the end of a chunk) computes them anew.  (A choice between
    // a full tile's and the others in front of every load: 670 K labels, batch 128, Philox 774 us a step instead of 764, nearest
    // 344 / 336, with a compensated head 477 / 471; sr_fast the same.)
    // (24-bit products: as plain ones they became 64-bit multiply-adds with register pairs for their lane parts, which are kept over
    // the loop; the sr_fast variant spilled two registers and the Philox one nine, one of them read back in front of every tile's
    // logits.  Now none and four, which are read back where the height changes only; the times are the same.  Without any - offsets
    // two to a register, or their lane parts computed anew - Philox took 781 - 787 us instead of 779, at 131 K labels, batch 96,
    // 170 - 171 instead of 168.)
    int w_valid = TL, r_valid = TL;
    auto w_rows = [&](const QTile& q) {
      if (q.rows_valid == w_valid) return;
      w_valid = q.rows_valid;
#pragma unroll
      for (int s = 0; s < 4; s++) woff[s] = wcol_offset(s, w_valid - 1);
    };
    auto r_rows = [&](const QTile& q) {
      if (q.rows_valid == r_valid) return;
      r_valid = q.rows_valid;
#pragma unroll
      for (int s = 0; s < 4; s++) roff[s] = rows_offset(s, r_valid - 1);
    };
    auto wcol_piece = [&](int slot, const QTile& q, int s) {
      if (a + 4 * s >= 13) return;
      const unsigned off = woff[s];
      q_lds_load16_sbase(q.base, off, (unsigned)(RLDS_C + slot * QWC_BYTES + (a + 4 * s) * 1024));
    };
    auto rows_piece = [&](int slot, const QTile& q, int s) {
      if (ra + 4 * s >= 13) return;
      const unsigned off = roff[s];
      if (ra + 4 * s == 12) {   // the last piece is half a piece: 32 chunks
        if (lane < 32) q_lds_load16_sbase(q.base, off, (unsigned)(RLDS_R + slot * RROW_BYTES + 12 * 1024));
      } else {
        q_lds_load16_sbase(q.base, off, (unsigned)(RLDS_R + slot * RROW_BYTES + (ra + 4 * s) * 1024));
      }
    };
    auto rows_pieces = [&](int slot, const QTile& q) {
      r_rows(q);
#pragma unroll
      for (int s = 0; s < 4; s++) rows_piece(slot, q, s);
    };
    // block a (the part member a produced) of the G tile of position t, NK pieces of 1 KiB (32 batch rows), a linear copy
    const unsigned gsrc_lane = (unsigned)(a * 4096 + lane * 16);
    auto gather = [&](int t, int buf) {
#pragma unroll
      for (int s = 0; s < NK; s++)
        q_lds_load16_l2_sbase(exq + (t & (QSLOTS - 1)) * QG_BYTES + s * 1024, gsrc_lane,
                              (unsigned)(RLDS_G + buf * RG_BYTES + a * 4096 + s * 1024));
    };
    // the four counters of member a's wavefronts, as they are now, into LDS (read in the next iteration)
    auto issue_snapshot = [&](int i) {
      if (lane < 4) q_lds_load4_l2(srcflags + lane, (unsigned)(RLDS_M + a * 32 + (i & 1) * 16));
    };
    // wait until the four producers of block a have published at least `need` tiles
    auto wait_published = [&](int need, int fmin, int i) {
      if (fmin >= need) return;
      for (int spin = 0;; spin++) {
        int fl = __hip_atomic_load(srcflags + (lane & 3), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (__builtin_amdgcn_read_exec() == __builtin_amdgcn_ballot_w64(fl >= need)) break;
        if (spin >= p.spin_limit || ((spin & 1023) == 1023 && __hip_atomic_load(errw, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))) {
          // give up: raise the error word (partners that wait for this workgroup see it and give up too) and the
          // workgroup's abort word; every wavefront leaves the loop behind the next barrier
          if (lane == 0) {
            __hip_atomic_fetch_or(errw, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            *(lds_int*)(lds + abort_base + (i & 1) * 4) = 1;
          }
          break;
        }
        __builtin_amdgcn_s_sleep(2);
      }
    };

    // Stage A of the tile at position t: logits of label rows 16m.. against batch rows 32a..32a+31, sigmoid minus target,
    // this wavefront's part of G to the exchange slot.  Lane (l16, kg) ends up with labels 16m + 4kg..+3 of batch rows
    // 32a + l16 and 32a + 16 + l16: eight bytes each, quarter kg of the row's 32 bytes in block m of the slot.
    // The matrix part takes a callback that runs once per K step: the caller spreads its loads over it.
    unsigned char* gdst_lane = exq + m * 4096 + (16 * AB * a + g_row16(l16)) * 32 + ((((kg >> 1) ^ (l16 >> 3)) << 1) | (kg & 1)) * 8;
    auto stage_a_logits = [&](int slot, floatx4 (&z)[AB], auto&& between) {
      // lane (row l16, k group kg) holds bytes 16kg..16kg+15 and 64+16kg..64+16kg+15 of every 128-byte K step (the X
      // image is built in the same order): two 16-byte reads whose lanes tile the LDS banks
      const unsigned asrc = (unsigned)(RLDS_R + slot * RROW_BYTES) + l16 * QRS + kg * 16;
      intx4 alo[6], ahi[6];
      auto rd = [&](int ks) {
        alo[ks] = *(const __attribute__((address_space(3))) intx4*)(lds + asrc + ks * 128);
        ahi[ks] = *(const __attribute__((address_space(3))) intx4*)(lds + asrc + ks * 128 + 64);
      };
      rd(0); rd(1); rd(2);
      QFENCE();
#pragma unroll
      for (int blk = 0; blk < AB; blk++) z[blk] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < 6; ks++) {
        if (ks + 3 < 6) rd(ks + 3);
        between(ks);
        intx8 av = intx8{alo[ks].x, alo[ks].y, alo[ks].z, alo[ks].w, ahi[ks].x, ahi[ks].y, ahi[ks].z, ahi[ks].w};
#pragma unroll
        for (int blk = 0; blk < AB; blk++) z[blk] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(av, xq[blk][ks], z[blk], 0, 0, 0, 0, 0, 0);
        QFENCE();
      }
    };
    auto stage_a_finish = [&](int t, const QTile& q, const floatx4 (&z)[AB]) {
      const float nlog2e = -1.44269504088896340736f;
      const int r0 = 16 * m + 4 * kg;   // this lane's label rows r0..r0+3
      unsigned sb[AB][2];
#pragma unroll
      for (int blk = 0; blk < AB; blk++)
#pragma unroll
        for (int e2 = 0; e2 < 2; e2++) {
          const unsigned zb = bf16_pack2(z[blk][2 * e2] * p.zscale, z[blk][2 * e2 + 1] * p.zscale);
          const float z0 = __uint_as_float(zb << 16), z1 = __uint_as_float(zb & 0xFFFF0000u);
          sb[blk][e2] = bf16_pack2(__builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(z0 * nlog2e)),
                                   __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(z1 * nlog2e)));
        }
      if (q.p1 > q.p0) {
        // (loads that the compiler waits for itself: the waits counted by hand below are for younger operations only.  The lane number
        // anew: kept over the loop it made the Philox variants spill more)
        const unsigned ln = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
        const unsigned hit = positive_hits<16, 16 * AB>(p.keys, q.p0, q.p1, q.label0 + 16u * (unsigned)m, 16u * AB * (unsigned)a, ln, lds + RLDS_P + a * 64);
#pragma unroll
        for (int blk = 0; blk < AB; blk++)
#pragma unroll
          for (int e2 = 0; e2 < 2; e2++) sb[blk][e2] = minus_hits(sb[blk][e2], hit, 4 * blk + 2 * e2);
      }
      if (q.rows_valid < TL) {   // rows past the end of the chunk contribute nothing
#pragma unroll
        for (int blk = 0; blk < AB; blk++)
#pragma unroll
          for (int e2 = 0; e2 < 2; e2++) {
            if (r0 + 2 * e2 >= q.rows_valid) sb[blk][e2] &= 0xFFFF0000u;
            if (r0 + 2 * e2 + 1 >= q.rows_valid) sb[blk][e2] &= 0x0000FFFFu;
          }
      }
      unsigned char* dst = gdst_lane + (t & (QSLOTS - 1)) * QG_BYTES;
      *(uint2*)dst = uint2{sb[0][0], sb[0][1]};
      if constexpr (AB == 2) *(uint2*)(dst + 512) = uint2{sb[AB - 1][0], sb[AB - 1][1]};
    };

    // ---- prologue: rows and columns of the first RQ positions, their stage A, rows of the next two, G of position 0; all that
    //      only as far as the sequence goes.  A launch spends 6 - 10 us here, most of them waiting for memory, so that nothing
    //      waits for more than it needs: stage A for the rows (the columns, which come from the L2 behind them, land under it),
    //      stage A of position 3 for its rows, and the gather of G(0) for no load at all.
#pragma unroll
    for (int k = 0; k < RR_RING; k++)
      if (k < n_it) rows_pieces(k, q_desc_head(cdesc, tile_at(k)));
    // a wait the compiler knows of: without it, it takes the loads of xq above for outstanding wherever the loop below
    // uses them (it cannot see the waits written as inline assembly) and waits for all memory operations there
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();   // P1
#pragma unroll
    for (int k = 0; k < RQ; k++)
      if (k < n_it) {
        const QTile t = q_desc_head(cdesc, tile_at(k));
        w_rows(t);
#pragma unroll
        for (int s = 0; s < 4; s++) wcol_piece(k, t, s);
      }
    // (stays in the XCD's L2, where the quad's members look for it, as the G tiles do.  At agent scope it is written
    // through to memory, and the loop's waits, which count in order, wait for that: 670 K labels, batch 128, nearest 398 us a step
    // instead of 353; with a compensated head, nearest 527 instead of 478, sr_fast 525 instead of 496; 131 K, batch 96, 86.3 / 85.3)
    auto publish = [&](int tiles) {
      if (lane == 0) __hip_atomic_store(myflag, tiles, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    };
    // stage A of positions 0..RQ-1; the rows image of position k + RR_RING replaces that of position k behind a barrier
    static_assert((RQ == 4 || RQ == 3) && RR_RING == 3, "the waits below");
#pragma unroll
    for (int k = 0; k < RQ; k++) {
      if (k >= n_it) continue;
      if (k == RR_RING) {   // this stage A reads an image that was requested behind position 0
        // (younger than its loads: the stores of G, if any, and the loads of a tile, twice)
        if (n_it <= RR_RING + 2) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        else if (!la && ra == 0) asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
        else if (!la) asm volatile("s_waitcnt vmcnt(6)" ::: "memory");
        else if (ra == 0) asm volatile("s_waitcnt vmcnt(%0)" : : "n"(8 + 2 * AB) : "memory");
        else asm volatile("s_waitcnt vmcnt(%0)" : : "n"(6 + 2 * AB) : "memory");
        publish(1);
        __syncthreads();   // P3
      }
      if (la) {
        floatx4 z[AB];
        stage_a_logits(k % RR_RING, z, [](int) {});
        stage_a_finish(k, q_desc_full(cdesc, tile_at(k)), z);
      }
      if (k < RQ - 1 && k + RR_RING < n_it) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __syncthreads();   // P2.k: every A wavefront has read the rows image
        rows_pieces(k, q_desc_head(cdesc, tile_at(k + RR_RING)));
      }
    }
    if (n_it > 0) {
      if (RQ == RR_RING || n_it <= RR_RING) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the stores of G included
        publish(min(RQ, n_it));
      }
      wait_published(1, 0, 1);   // an expiry here is seen behind the first barrier of the loop (slot 1 = "iteration -1")
      gather(0, 0);
    }
    issue_snapshot(1);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (RQ > RR_RING && n_it > RR_RING) publish(min(RQ, n_it));

    // descriptors of the next iteration: the tile of its stage A (whose columns it also fetches), the tile whose rows it
    // fetches and the tile of its share of stage B; loaded one iteration ahead through the scalar path
    if (a == 0) pass_on(0, q_desc_full(cdesc, tile_at(0)));
    QTile qa_n = q_desc_full(cdesc, tile_at(RQ)), qr_n = q_desc_head(cdesc, tile_at(RQ + RR_RING - 1)), qb_n = q_desc_full(cdesc, tile_at(0));
    unsigned char* qp_base = nullptr;   // the tile of the iteration before: base pointer and valid rows
    int qp_base_valid = 0;
    int sa = RQ % RR_RING;    // (i + RQ) % RR_RING, the rows image stage A reads
    int w0 = 0;               // i % RC_RING
    for (int i = 0; i < n_it; i++) {
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __syncthreads();
      const QTile qa = qa_n, qr = qr_n, qb = qb_n;
      int abort_word = *(const lds_int*)(lds + abort_base + ((i + 1) & 1) * 4);
      // the counters as they were in the middle of the iteration before
      intx4 fl = *(const __attribute__((address_space(3))) intx4*)(lds + RLDS_M + a * 32 + ((i + 1) & 1) * 16);
      asm volatile("" : "+v"(abort_word), "+v"(fl));   // (one wait for both)
      if (__builtin_amdgcn_readfirstlane(abort_word) != 0) break;
      if (i + 1 < n_it) {
        const int fmin = min(min((int)__builtin_amdgcn_readfirstlane(fl.x), (int)__builtin_amdgcn_readfirstlane(fl.y)),
                             min((int)__builtin_amdgcn_readfirstlane(fl.z), (int)__builtin_amdgcn_readfirstlane(fl.w)));
        wait_published(i + 2, fmin, i);
        gather(i + 1, (i + 1) & 1);
      }
      // ---- stage A of position i + RQ, the columns of the same tile requested between its matrix instructions
      const bool do_a = i + RQ < n_it, do_r = i + RQ + RR_RING - 1 < n_it;   // (the sequence's end)
      const int wslot = w0 == 0 ? RC_RING - 1 : w0 - 1;   // (i + RQ) % RC_RING
      floatx4 z[AB];
      if (do_a) {
        w_rows(qa);
        if (la) {
          stage_a_logits(sa, z, [&](int ks) { if (ks < 4) wcol_piece(wslot, qa, ks); });
        } else {
#pragma unroll
          for (int ks = 0; ks < 4; ks++) wcol_piece(wslot, qa, ks);
        }
      }
      // the counters as they are now, for the next iteration; everything behind this point may stay in flight over the
      // barrier
      issue_snapshot(i);
      // ---- this wavefront's A^T blocks of position i: operands, matrix instructions
      const unsigned wc = (unsigned)(RLDS_C + w0 * QWC_BYTES);
      const unsigned gb = (unsigned)(RLDS_G + (i & 1) * RG_BYTES);
      const unsigned gwl = gb + bl.bg_lane, gwh = gb + (bl.bg_lane ^ 128u), wrow = wc + bl.wrow_lane;
      const unsigned oimg = (unsigned)(RLDS_O + (i & 1) * RO_BYTES);
      floatx4 aa[NBA][3];
      unsigned wq[NBA][3];
#pragma unroll
      for (int nb = NBB; nb < 4; nb++) {
        bf16x8 bg[NK];
#pragma unroll
        for (int ks = 0; ks < NK; ks++) bg[ks] = read_bg(gwl, gwh, nb, ks);
#pragma unroll
        for (int cg = 0; cg < 3; cg++) wq[nb - NBB][cg] = *(const unsigned*)(lds + wrow + 16 * nb * QWS + 4 * cg);
#pragma unroll
        for (int ks = 0; ks < NK; ks++)
#pragma unroll
          for (int cg = 0; cg < 3; cg++)
            aa[nb - NBB][cg] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xt[cg][ks], bg[ks], ks == 0 ? floatx4{0.f, 0.f, 0.f, 0.f} : aa[nb - NBB][cg], 0, 0, 0);
        QFENCE();
      }
      // descriptors of the next iteration: requested here, in front of a long stretch of vector work, because every wait
      // for an LDS read also waits for outstanding scalar loads
      qa_n = q_desc_full(cdesc, tile_at(i + 1 + RQ));
      qr_n = q_desc_head(cdesc, tile_at(i + 1 + RQ + RR_RING - 1));
      qb_n = q_desc_full(cdesc, tile_at(i + 1));
      if (do_a && la) stage_a_finish(i + RQ, qa, z);
      // the previous tile's updated weights, from their LDS image to memory: 12 wave-wide pieces of 16 bytes per lane,
      // three per A wavefront (chunk ch = (3a + jj) * 64 + lane is bytes 16 (ch % 12).. of row ch / 12)
      if (i > 0) {
#pragma unroll
        for (int jj = 0; jj < 3; jj++) {
          const int ch = (3 * a + jj) * 64 + lane, row = ch / 12;
          const unsigned off = (unsigned)(row * D + QCOLS * m + (ch - row * 12) * 16);
          const intx4 ov = *(const __attribute__((address_space(3))) intx4*)(lds + RLDS_O + ((i + 1) & 1) * RO_BYTES + ch * 16);
          if (qp_base_valid == TL) {
            // written through (system scope): the updated weights are not read again by this launch, and as ordinary
            // stores they push the exchanged G tiles and the weight tiles between their two fetches out of the XCD's
            // L2 (reads from memory 1.34 instead of 1.12 times the weights); same speed either way
            // (the registers of a store of more than 8 bytes may not be written by a vector instruction within the next two wait
            // states: it is the address of the next read here, and with the other wavefront at a higher priority a few
            // addresses in a hundred thousand were stored for weights.  The compiler keeps that distance only from stores it
            // knows, and waiting instructions in between do not count.)
            asm volatile("s_nop 4\n\tglobal_store_dwordx4 %0, %1, %2 sc0 sc1\n\ts_nop 1" : : "v"(off), "v"(ov), "s"(q_uniform(qp_base)) : "memory");
          } else {
            // rows past the end of the chunk go to a place nobody reads (the padding behind an exchange slot), so that
            // the wavefront issues the same number of memory operations for every tile
            unsigned char* dst = row < qp_base_valid ? qp_base + off : exq + (size_t)(m * 2) * QG_BYTES + RG_BYTES + a * 1024 + lane * 16;
            asm volatile("global_store_dwordx4 %0, %1, off\n\ts_nop 1" : : "v"(dst), "v"(ov) : "memory");
          }
        }
      }
      qp_base = qb.base; qp_base_valid = qb.rows_valid;
      if (a == 0) pass_on((i + 1) & 1, qb_n);
      // ---- the update of those blocks, with the rows of position i + RQ + 2 (the only loads that miss the L2) requested
      //      between its pieces
      {
        float t[3][4];
        unsigned hs[3], outw[3], knew[6];
        const RKahanBlock nok = {};
        const unsigned hash_tile = qb.label0 * (unsigned)(D / 4) * 0x9E3779B1u + qb.seed;
        if (do_r) r_rows(qr);
        const int rslot = sa == 0 ? RR_RING - 1 : sa - 1;   // (i + RQ + RR_RING - 1) % RR_RING
#pragma unroll
        for (int nb = NBB; nb < 4; nb++)
#pragma unroll
          for (int c = 0; c < 8; c++) {
            constexpr int every = 2 * NBA;
            const int pc = (nb - NBB) * 8 + c;
            if (pc % every == 0 && do_r) rows_piece(rslot, qr, pc / every);
            r_update_piece<MODE, WD, 0>(c, nb, aa[nb - NBB], wq[nb - NBB], t, hs, outw, knew, bl, qb, hash_tile, p.lr_eff, p.wd_eff, l16, lds, oimg, nok, 0u, 0);
          }
        if (NBB == 4 && do_r) rows_pieces(rslot, qr);
      }
      // Loads and stores complete in order.  Waiting for all but the stores of G and the rows covers the gather, the
      // columns and the snapshot, all issued long before, and everything of the iteration before, whose stores of G can
      // now be published.
      {
        const int cnt = (do_a && la ? AB : 0) + (i > 0 ? 3 : 0) + (do_r ? (ra == 0 ? 4 : 3) : 0);
        switch (cnt) {
          case 9: asm volatile("s_waitcnt vmcnt(9)" ::: "memory"); break;
          case 8: asm volatile("s_waitcnt vmcnt(8)" ::: "memory"); break;
          case 7: asm volatile("s_waitcnt vmcnt(7)" ::: "memory"); break;
          case 6: asm volatile("s_waitcnt vmcnt(6)" ::: "memory"); break;
          case 5: asm volatile("s_waitcnt vmcnt(5)" ::: "memory"); break;
          case 4: asm volatile("s_waitcnt vmcnt(4)" ::: "memory"); break;
          case 3: asm volatile("s_waitcnt vmcnt(3)" ::: "memory"); break;
          case 2: asm volatile("s_waitcnt vmcnt(2)" ::: "memory"); break;
          default: asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); break;
        }
      }
      publish(min(i + RQ, n_it));
      sa = sa == RR_RING - 1 ? 0 : sa + 1;
      w0 = w0 == RC_RING - 1 ? 0 : w0 + 1;
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __syncthreads();   // the last tile's updated weights are in LDS: the B wavefronts store them
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the last loads still target LDS
    return;
  }

  // ============================================================================================= B wavefronts
  const int s = f;       // features 192m + 48s .. +47
  floatx4 acc2[2 * NK][3];    // grad_X[32 NK batch rows x 48 features]
  {
    // a second launch of a step continues the sums of the first
    const floatx4* prev = p.partial + (size_t)g * 24 * 256;
#pragma unroll
    for (int mb = 0; mb < 2 * NK; mb++)
#pragma unroll
      for (int nn = 0; nn < 3; nn++)
        acc2[mb][nn] = quad < p.acc_quads ? prev[(mb * 3 + nn) * 256 + s * 64 + lane] : floatx4{0.f, 0.f, 0.f, 0.f};
  }

  // per-lane parts of the LDS addresses
  const unsigned ga_lane = (unsigned)((kg >> 1) * 4096 + g_row16(l16) * 32 + ((kg & 1) ^ (l16 >> 3)) * 16);           // grad_X operand
  const unsigned wtr_lane = (unsigned)((8 * kg + (l16 >> 1)) * QWS + 48 * s + (l16 & 1) * 8);                        // W columns, transposed read

  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();   // P1
#pragma unroll
  for (int k = 0; k < RQ - 1; k++)
    if (k + RR_RING < n_it) __syncthreads();   // P2.k
  if (RQ > RR_RING && RR_RING < n_it) __syncthreads();         // P3

  // ---- Compensation terms (KT): a block's are 16 row segments of 96 or 48 consecutive bytes.  They come straight to LDS in 16-byte pieces,
  // are taken from there in the update's layout (24 or 12 bytes a lane), and the new ones go the same way back.  As accesses of 8 bytes a
  // lane, 24 apart, each waited for behind another's, they took longer, and the registers of two blocks' terms made every variant spill:
  // 670 K labels, a fifth of them compensated, batch 128, us a step: bf16 terms, sr_fast 479 / 458, nearest 455 / 432, e5m2 447 / 436.
  // What bounds the head's launch now: 3 times a plain tile's bytes (bf16), half as much vector work again, and both by turns - without
  // any access to the terms the step takes 406 us, without the stores 434, without the loads 453.  Stores: written through (as the weights
  // are) 462, to stay in the L2 459, non-temporal 458; terms brought to the L2 by the A wavefronts two tiles ahead 470 / 462.
  // The loads and stores of a wavefront complete in order: block o's loads, requested KSLOTS blocks before, are complete when all but the
  // (KSLOTS - 1) (stores + loads) behind them are.  That number is the same for every block: the last tile's blocks request something,
  // too, and rows behind the head's end are masked, not jumped over (EXEC is written in the statements; all lanes are active in front
  // of them).
  constexpr int KPR = Geo::KROW / 16, KB = KT == 1 ? 2 : 1;   // pieces of a row, bytes of a term
  const unsigned kslot0 = (unsigned)(Geo::K + f * Geo::KSLOTS * Geo::KSLOT), kterm_lane = (unsigned)(l16 * Geo::KROW + kg * (Geo::KROW / 4));
  auto kplace = [&](int ch) { return (unsigned)(ch / KPR * D * KB + (ch - ch / KPR * KPR) * 16); };   // of a piece, behind the block's first row
  auto lane_now = [] { unsigned l = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)); asm volatile("" : "+v"(l)); return (int)l; };
  auto kahan_request = [&](int it, int o) {   // block o of position it; of rows behind the head's end anything
    int first = TL * (quad + it * nquads) + 16 * o, left = p.num_head - first;
    if (left <= 0) { first = 0; left = p.num_head; }
    const unsigned char* base = q_uniform(p.kahan + ((size_t)first * D + QCOLS * m + 48 * f) * KB);
    const unsigned last = (unsigned)((min(left, 16) - 1) * D * KB + Geo::KROW - 16), slot = kslot0 + (unsigned)((o & (Geo::KSLOTS - 1)) * Geo::KSLOT);
    const int ln = lane_now();
    const unsigned kplace0 = kplace(ln), kplace1 = kplace(ln + 64), at0 = min(kplace0, last);
    if constexpr (KT == 1) {
      const unsigned at1 = min(kplace1, last);
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 3\n\tglobal_load_lds_dwordx4 %1, %3\n\ts_add_u32 m0, %0, 1024\n\ts_bfm_b64 exec, 32, 0\n\ts_nop 3\n\t"
                   "global_load_lds_dwordx4 %2, %3\n\ts_mov_b64 exec, -1" : : "s"(slot), "v"(at0), "v"(at1), "s"(base) : "memory", "m0", "scc");
    } else {
      asm volatile("s_mov_b32 m0, %0\n\ts_bfm_b64 exec, 48, 0\n\ts_nop 3\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b64 exec, -1"
                   : : "s"(slot), "v"(at0), "s"(base) : "memory", "m0");
    }
  };
  auto kahan_store = [&](int it, int o) {     // the new terms of block o of position it, from its slot
    const int ln = lane_now();
    const int first = TL * (quad + it * nquads) + 16 * o, left = max(min(p.num_head - first, 16), 0);
    unsigned char* base = q_uniform(p.kahan + ((size_t)first * D + QCOLS * m + 48 * f) * KB);
    const unsigned slot = kslot0 + (unsigned)((o & (Geo::KSLOTS - 1)) * Geo::KSLOT) + (unsigned)ln * 16u, end = (unsigned)(left * D * KB);
    const unsigned kplace0 = kplace(ln), kplace1 = kplace(ln + 64);
    const intx4 k0 = *(const __attribute__((address_space(3))) intx4*)(lds + slot);
    if constexpr (KT == 1) {
      const intx4 k1 = *(const __attribute__((address_space(3))) intx4*)(lds + slot + ((ln & 32) ? 0u : 1024u));   // (lanes 32.. store none)
      const unsigned long long m0 = __builtin_amdgcn_ballot_w64(kplace0 < end), m1 = __builtin_amdgcn_ballot_w64(kplace1 < end) & 0xFFFFFFFFull;
      asm volatile("s_mov_b64 exec, %5\n\ts_nop 4\n\tglobal_store_dwordx4 %0, %2, %4 nt\n\ts_nop 1\n\ts_mov_b64 exec, %6\n\ts_nop 4\n\t"
                   "global_store_dwordx4 %1, %3, %4 nt\n\ts_nop 1\n\ts_mov_b64 exec, -1"
                   : : "v"(kplace0), "v"(kplace1), "v"(k0), "v"(k1), "s"(base), "s"(m0), "s"(m1) : "memory");
    } else {
      const unsigned long long m0 = __builtin_amdgcn_ballot_w64(kplace0 < end) & 0xFFFFFFFFFFFFull;
      asm volatile("s_mov_b64 exec, %3\n\ts_nop 4\n\tglobal_store_dwordx4 %0, %1, %2 nt\n\ts_nop 1\n\ts_mov_b64 exec, -1"
                   : : "v"(kplace0), "v"(k0), "s"(base), "s"(m0) : "memory");
    }
  };
  if constexpr (KT != 0) {
    if (n_it > 0) {
#pragma unroll
      for (int o = 0; o < Geo::KSLOTS; o++) kahan_request(0, o);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
  }
  int w0 = 0;   // i % RC_RING
  int n_done = 0;
  for (int i = 0; i < n_it; i++) {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __syncthreads();
    const unsigned oimg = (unsigned)(RLDS_O + (i & 1) * RO_BYTES);
    const unsigned wc = (unsigned)(RLDS_C + w0 * QWC_BYTES);
    const unsigned gb = (unsigned)(RLDS_G + (i & 1) * RG_BYTES);
    const unsigned gxa = gb + ga_lane, gwl = gb + bl.bg_lane, gwh = gb + (bl.bg_lane ^ 128u);
    const unsigned wtr = wc + wtr_lane, wrow = wc + bl.wrow_lane;

    // The tile is a sequence of (4 + NBB) NK steps of one LDS operand and three matrix instructions each.  The first
    // 2 NK NBB alternate:
    //   even step 2 NK o + 2ks:      A^T block o (label rows 16o..), K step ks:  aa[cg] += X^T[cg][ks] * G^T   (operand: two transposing reads)
    //   odd  step 2 NK o + 2j + 1:   grad_X step NK o + j
    // and the rest are the remaining grad_X steps; grad_X step x = K step x / 2NK (32 labels), batch block x % 2NK:
    //   acc2[mb][nn] += G^T * W[nn]  (operand: one 16-byte read).
    // The operand of step k + 3 is requested in step k.  The vector work of the update of block o (12 weights per lane,
    // eight pieces) is spread over the steps behind the block's last, so that it issues between the matrix instructions.
    constexpr int NS = (4 + NBB) * NK, SB = 2 * NK, NALT = SB * NBB;   // steps of a tile, of a block, alternating ones
    constexpr int PD = KT != 0 ? (MODE == ROUND_SR_PHILOX ? 1 : 2) : XMC_PD;   // operands are requested this many steps ahead (the head-Kahan variants
                                               // have no registers for a third operand in flight)
    bf16x8 op[NS + PD];
    auto grad_step = [](int k) { return k < NALT ? NK * (k / SB) + (k % SB) / 2 : NALT / 2 + (k - NALT); };
    auto request = [&](int k) {
      if (k >= NS) return;
      if (k < NALT && (k & 1) == 0) {
        op[k] = read_bg(gwl, gwh, k / SB, (k % SB) / 2);
      } else {
        const int x = grad_step(k);
        op[k] = *(const bf16x8*)(lds + gxa + (x / SB) * 8192 + (x % SB) * 512);
      }
    };
    const int abort_word = *(const lds_int*)(lds + abort_base + ((i + 1) & 1) * 4);
    // (the tile's descriptor comes through LDS: a scalar load in this wavefront, whose every wait is for LDS reads, stood in front of
    // the barrier with its whole latency; 131 K labels, batch 96, 88.1 us a step with it, 86.4 without)
    const intx4 qd = *(const lds_intx4*)(lds + RLDS_T + (i & 1) * 16);
#pragma unroll
    for (int k = 0; k < PD; k++) request(k);
    intx2 wraw[2][3];
#pragma unroll
    for (int ks2 = 0; ks2 < 2; ks2++)
#pragma unroll
      for (int nn = 0; nn < 3; nn++)
        wraw[ks2][nn] = __builtin_amdgcn_ds_read_tr8_b64_v2i32((__attribute__((address_space(3))) intx2*)(lds + wtr + ks2 * 32 * QWS + nn * 16));
    if (__builtin_amdgcn_readfirstlane(abort_word) != 0) break;
    QTile q = {};
    const unsigned hash_tile = MODE == ROUND_SR_FAST ? (unsigned)__builtin_amdgcn_readfirstlane(qd.x) : 0u;
    if (MODE == ROUND_SR_PHILOX) q.seed = (unsigned)__builtin_amdgcn_readfirstlane(qd.y);
    if (MODE == ROUND_SR_PHILOX || KT != 0) q.row0 = __builtin_amdgcn_readfirstlane(qd.z);
    n_done = i + 1;
    bf16x8 wb[2][3];

    floatx4 aa[2][3];       // A^T of the block in progress and of the one being rounded
    unsigned wq[2][3];      // their old weights
    float t[3][4];
    unsigned hs[3], outw[3], knew[6];
    RKahanBlock kb = {};      // compensation terms of the block being rounded
    auto kahan_begin = [&](int o) {   // block o's terms have landed: to registers
      asm volatile("s_waitcnt vmcnt(%0)" : : "n"((Geo::KSLOTS - 1) * 2 * Geo::KLOADS) : "memory");
      const unsigned at = kslot0 + kterm_lane + (unsigned)((o & (Geo::KSLOTS - 1)) * Geo::KSLOT);
      kb.row = q.row0 + 16 * o + l16;
      kb.head = kb.row < p.num_head;
#pragma unroll
      for (int cg = 0; cg < 3; cg++) {
        if (KT == 1) {
          const rux2 kv = *(const __attribute__((address_space(3))) rux2*)(lds + at + 8 * cg);
          kb.raw[2 * cg] = kb.head ? kv.x : 0u; kb.raw[2 * cg + 1] = kb.head ? kv.y : 0u;
        } else {
          const unsigned kv = *(const __attribute__((address_space(3))) unsigned*)(lds + at + 4 * cg);
          kb.raw[cg] = kb.head ? kv : 0u;
        }
      }
    };
    auto kahan_end = [&](int o) {     // ... and the new ones are in their place
      kahan_store(i, o);
      if (o + Geo::KSLOTS < 4) kahan_request(i, o + Geo::KSLOTS);
      else kahan_request(min(i + 1, n_it - 1), o + Geo::KSLOTS - 4);
    };
    auto kterm = [&](int o) { return KT != 0 ? kslot0 + kterm_lane + (unsigned)((o & (Geo::KSLOTS - 1)) * Geo::KSLOT) : 0u; };
    // (this loop must be unrolled completely: its register arrays are indexed by k.  The variants with the Philox
    // recipe or a compensated head exceed the compiler's default size limit for "#pragma unroll" and are compiled in a
    // translation unit of their own, xmc_fp8_role_heavy.hip, with a higher limit.)
#pragma unroll
    for (int k = 0; k < NS; k++) {
      request(k + PD);
      // vector pieces of this step
      if (k == 0) {
#pragma unroll
        for (int nn = 0; nn < 3; nn++) wb[0][nn] = q_fp8x8_to_bf16x8(wraw[0][nn]);
      }
      if (k == 2) {
#pragma unroll
        for (int nn = 0; nn < 3; nn++) wb[1][nn] = q_fp8x8_to_bf16x8(wraw[1][nn]);
      }
      if (k < NALT && k % SB == NK) {   // old weights of the block in progress, read before its update starts
        const int o = k / SB;
#pragma unroll
        for (int cg = 0; cg < 3; cg++) wq[o & 1][cg] = *(const unsigned*)(lds + wrow + 16 * o * QWS + 4 * cg);
      }
      if (k >= SB) {
        // behind the alternating steps: the last block's, in the trailing ones (none of them: behind the loop)
        constexpr int TR = NS - NALT > 0 ? NS - NALT : 1;
        const int o = k < NALT ? k / SB - 1 : NBB - 1, kk = k < NALT ? k % SB : k - NALT, n = k < NALT ? SB : TR;
        if (KT != 0 && kk == 0) kahan_begin(o);
#pragma unroll
        for (int c = kk * 8 / n; c < (kk + 1) * 8 / n; c++)
          r_update_piece<MODE, WD, KT>(c, o, aa[o & 1], wq[o & 1], t, hs, outw, knew, bl, q, hash_tile, p.lr_eff, p.wd_eff, l16, lds, oimg, kb, kterm(o), p.num_head);
        if (KT != 0 && kk == n - 1) kahan_end(o);
      }
      if (k < NALT && (k & 1) == 0) {
        const int o = k / SB, ks = (k % SB) / 2;
#pragma unroll
        for (int cg = 0; cg < 3; cg++)
          aa[o & 1][cg] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xt[cg][ks], op[k], ks == 0 ? floatx4{0.f, 0.f, 0.f, 0.f} : aa[o & 1][cg], 0, 0, 0);
      } else {
        const int x = grad_step(k), ks2 = x / SB, mb = x % SB;
#pragma unroll
        for (int nn = 0; nn < 3; nn++) acc2[mb][nn] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(op[k], wb[ks2][nn], acc2[mb][nn], 0, 0, 0);
      }
      QFENCE();
    }
    if (NBB == 4) {
      if constexpr (KT != 0) kahan_begin(3);
#pragma unroll
      for (int c = 0; c < 8; c++) r_update_piece<MODE, WD, KT>(c, 3, aa[1], wq[1], t, hs, outw, knew, bl, q, hash_tile, p.lr_eff, p.wd_eff, l16, lds, oimg, kb, kterm(3), p.num_head);
      if constexpr (KT != 0) kahan_end(3);
    }
    w0 = w0 == RC_RING - 1 ? 0 : w0 + 1;
  }
  if (KT != 0) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the last requests still target LDS
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __syncthreads();   // every wavefront has written its part of the last tile's image
  // The image of the last tile's updated weights (64 rows x 192 bytes) goes to memory as 12 wave-wide stores of 16 bytes
  // per lane, three per B wavefront (the A wavefronts, which store the other tiles' images one iteration later, have
  // left): chunk ch = (3s + jj) * 64 + lane is bytes 16 (ch % 12).. of row ch / 12.
  if (n_done > 0) {
    const QTile q_p = q_desc_head(cdesc, tile_at(n_done - 1));
#pragma unroll
    for (int jj = 0; jj < 3; jj++) {
      const int ch = (3 * s + jj) * 64 + lane, row = ch / 12;
      const intx4 ov = *(const __attribute__((address_space(3))) intx4*)(lds + RLDS_O + ((n_done + 1) & 1) * RO_BYTES + ch * 16);
      if (row < q_p.rows_valid) *(intx4*)(q_p.base + (size_t)(row * D + QCOLS * m + (ch - row * 12) * 16)) = ov;
    }
  }

  // ---- per-workgroup grad_X partial, summed in a fixed order by reduce_gx_role_kernel: [24 blocks][4 B wavefronts][64 lanes]
  floatx4* dst = p.partial + (size_t)g * 24 * 256;
#pragma unroll
  for (int mb = 0; mb < 2 * NK; mb++)
    if (16 * mb < p.batch) {   // (blocks of zero rows are not read)
#pragma unroll
      for (int nn = 0; nn < 3; nn++) dst[(mb * 3 + nn) * 256 + s * 64 + lane] = acc2[mb][nn];
    }
}

#ifndef XMC_HEAVY_TU   // compiled once, in the library's main translation unit
// grad_X = scale * sum over quads of the member partials; writes fp32 and bf16 [batch, 768].  Workgroup (16-row batch block,
// feature block, member, B wavefront of the step) sums the 64 values of that wavefront; its four wavefronts take a quarter
// of the quads each, all loads of a wavefront in flight at once: the kernel is bound by the latency of a few rounds of loads
// (7.0 us with two wavefronts' worth of loads one behind the other and all blocks of 128 batch rows, whatever the batch).
__global__ __launch_bounds__(256) void reduce_gx_role_kernel(const floatx4* partial, int nwg, float scale, float* gx_f32,
                                                             unsigned short* gx_bf16, int batch, int* flags, int* failure_word,
                                                             const DropoutParams dp) {
  // placement check: the members of a quad exchanged G through the L2 of one XCD, which holds only if all four ran there
  if (blockIdx.x == 0) {
    if ((int)threadIdx.x < (nwg >> 2) && quad_xcc_mismatch(flags + QF_XCC, (int)threadIdx.x))
      __hip_atomic_fetch_or(flags + QF_ERR, 2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    if (threadIdx.x == 0) report_step_error(flags + QF_ERR, flags + QF_STICKY, failure_word);
  }
  const int blk = blockIdx.x >> 4, m = (blockIdx.x >> 2) & 3, s = blockIdx.x & 3;   // blk = mb*3+nn
  const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63, l16 = lane & 15, kg = lane >> 4;
  // the workgroups of member m of quads nq wv / 4 .. nq (wv + 1) / 4 - 1 (quad 8 j + x), in a fixed order
  floatx4 sum = {0.f, 0.f, 0.f, 0.f};
  const int nq = nwg >> 5;   // quads per XCD
  for (int jq = nq * wv >> 2; jq < nq * (wv + 1) >> 2; jq++) {
    floatx4 pv[8];
#pragma unroll
    for (int x = 0; x < 8; x++) pv[x] = partial[((size_t)(((jq * 4 + m) << 3) + x) * 24 + blk) * 256 + s * 64 + lane];
#pragma unroll
    for (int x = 0; x < 8; x++) sum += pv[x];
  }
  __shared__ floatx4 part[3][64];
  if (wv > 0) part[wv - 1][lane] = sum;
  __syncthreads();
  if (wv > 0) return;
#pragma unroll
  for (int q = 0; q < 3; q++) sum += part[q][lane];
  const int mb = blk / 3, nn = blk - mb * 3;
  const int col = QCOLS * m + 48 * s + 16 * nn + l16;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int b = 16 * mb + 4 * kg + i;
    if (b < batch) {
      const float val = dropout_backward(sum[i] * scale, (unsigned)(b * D + col), dp);
      if (gx_f32) gx_f32[(size_t)b * D + col] = val;
      if (gx_bf16) gx_bf16[(size_t)b * D + col] = bf16_bits(val);
    }
  }
}

#endif  // XMC_HEAVY_TU

// The variants of fp8_step_role_kernel with the reference's Philox recipe (XMC_ROUND_SR_PHILOX) or a compensated head
// (kahan_type 1, 2), defined in xmc_fp8_role_heavy.hip: opt in to the LDS size (once per device); launch.
// blocks: 32-row batch blocks the kernel computes (role_blocks).
void role_heavy_set_lds();
void role_heavy_launch(int round_mode, bool weight_decay, int kahan_type, int blocks, int grid, hipStream_t stream, const QuadParams& p);
// The other variants (round to nearest, fast stochastic rounding), defined in xmc_fp8_role_plain.hip.
void role_plain_set_lds();
void role_plain_launch(int round_mode, bool weight_decay, int blocks, int grid, hipStream_t stream, const QuadParams& p);
// The kernel is built for 1 to 4 blocks of 32 batch rows (NK), with weight decay for 4 and with a
// compensated head for 2 and 4 only: logits, G and its
// exchange, both gradients for the rows there are instead of always 128.  With fewer than four the A wavefronts, then the longer ones,
// hand their A^T block to the B wavefronts (r_nbb; with four blocks that is 2 % slower).  us a step, 128 rows computed / now:
// 131 K labels, batch 96, sr_fast 83.3 / 75.6, nearest 74.6 / 68.5, Philox 171 / 163; 670 K, batch 96, sr_fast 373 / 337; 16 K, batch 48
// 28.4 / 25.5; 131 K, batch 32 84 / 52, batch 64 87 / 63.
inline int role_blocks(int batch, bool weight_decay, int kahan_type) {
  return weight_decay ? 4 : kahan_type != 0 ? (batch <= 64 ? 2 : 4) : (batch + 31) / 32;
}

}  // namespace xmc
