// Shared device helpers and compile-time geometry for the gfx950 XMC classifier kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace xmc {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef int intx8 __attribute__((ext_vector_type(8)));
typedef int intx4 __attribute__((ext_vector_type(4)));
typedef int intx2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

// ---- geometry of the FP8 kernels
constexpr int D = 768;            // input features (row length of W, bytes per FP8 row)
constexpr int BP = 128;           // padded batch rows
constexpr int TL = 64;            // labels per tile of the training kernels
constexpr int NT = 256;           // threads per workgroup of the inference kernel (4 wavefronts of 64)
constexpr int WS = D + 16;        // LDS row stride of a W tile in the inference kernel, bytes (49 x 16)
constexpr int MAX_CHUNKS = 64;
constexpr int MAX_POS = 32768;    // positives per step (per 256 batch rows on the tiled path): the launches that group them keep them all in LDS

// workspace of the fused step (byte offsets), all 256-byte aligned
constexpr int MAX_WG = 256;                                   // workgroups of the persistent step kernel
constexpr size_t WS_XQ = 0;                                   // FP8 logits operands   BP*D
constexpr size_t WS_XT = WS_XQ + (size_t)BP * D;              // bf16 grad_W operands  BP*D*2
constexpr size_t WS_KEYS = WS_XT + (size_t)BP * D * 2;        // positive keys         MAX_POS*4
constexpr size_t WS_FLAGS = WS_KEYS + (size_t)MAX_POS * 4;    // 4096 ints: counters, XCC ids, error words (below)
constexpr size_t WS_PARTIAL = WS_FLAGS + 16384;               // MAX_WG * 12 * 512 * 16 bytes of grad_X partials
constexpr size_t WS_EXCH = WS_PARTIAL + (size_t)MAX_WG * 12 * 512 * 16;     // G exchange ring: 64 quads x 8 slots x 20 KiB
constexpr size_t WS_DESC = WS_EXCH + (size_t)(MAX_WG / 4) * 8 * 20480;      // the tile descriptors

// Layout of the 4096 ints at WS_FLAGS (all but the sticky word cleared at the start of every step):
//   [0, 1024)             tiles-published counters of the persistent step kernel: sixteen per quad
//   [QF_CNT2, +1024)      the same for the step's second launch (the head-Kahan layer runs the compensated tiles first)
//   [QF_XCC, QF_XCC+256)  XCC id every workgroup of the step kernel found itself on
//   [QF_ERR]              error word: bit 0 = a bounded wait expired, bit 1 = the workgroups of a quad were not placed on
//                         one XCD (their exchange of G through that XCD's L2 is then not coherent, and
//                         their counters do not reach one another: bit 0 comes with it)
//   [QF_STICKY]           the error words of all steps since the caller last cleared it, OR-ed together by the step's
//                         last kernel; no kernel ever clears it
constexpr int QF_WORDS = 4096;
constexpr int QF_CNT2 = 2048;
constexpr int QF_XCC = 1024;
constexpr int QF_ERR = 2044;
constexpr int QF_STICKY = 2047;

// The step kernel assumes that workgroup g runs on XCD g % 8, and builds quads of four workgroups with equal g % 8:
// member m of quad q is workgroup ((q / 8) * 4 + m) * 8 + q % 8.
__host__ __device__ inline int quad_member_workgroup(int quad, int m) { return (((quad >> 3) << 2) + m) * 8 + (quad & 7); }
// true if the four members of `quad` did not all record the same XCC id
__host__ __device__ inline bool quad_xcc_mismatch(const int* xcc_ids, int quad) {
  const int id0 = xcc_ids[quad_member_workgroup(quad, 0)];
  return xcc_ids[quad_member_workgroup(quad, 1)] != id0 || xcc_ids[quad_member_workgroup(quad, 2)] != id0 ||
         xcc_ids[quad_member_workgroup(quad, 3)] != id0;
}

// The end of a step, one thread of its last kernel: the step's error word joins the sticky word, which no kernel clears (a
// caller that looks at it only now and then still learns of every failed step), and as long as the sticky word is not zero
// every step changes the failure word in host memory (to an odd clock reading), which the host can watch without a copy,
// an event or a wait: a step that went well costs two loads here and nothing on the host.
__device__ __forceinline__ void report_step_error(const int* err, int* sticky, int* failure_word) {
  const int e = __hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const int before = __hip_atomic_load(sticky, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (e != 0) __hip_atomic_fetch_or(sticky, e, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if ((e | before) != 0 && failure_word)
    __hip_atomic_store(failure_word, (int)__builtin_amdgcn_s_memrealtime() | 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

__device__ __forceinline__ float bf16_rt(float f) { return (float)(__bf16)f; }

// bf16(a) in the low half, bf16(b) in the high half (round to nearest even), one conversion instruction
__device__ __forceinline__ unsigned bf16_pack2(float a, float b) {
  const bf16x2 r = __builtin_convertvector(floatx2{a, b}, bf16x2);
  return __builtin_bit_cast(unsigned, r);
}

__device__ __forceinline__ unsigned short bf16_bits(float f) {
  __bf16 b = (__bf16)f;
  unsigned short u;
  __builtin_memcpy(&u, &b, 2);
  return u;
}
__device__ __forceinline__ float bf16_from_bits(unsigned short u) { return __uint_as_float((unsigned)u << 16); }

__device__ __forceinline__ float clamp448(float t) { return __builtin_fminf(__builtin_fmaxf(t, -448.0f), 448.0f); }

// a ^ b ^ c in one instruction (0x96: the truth table of the three-input exclusive or).  The compiler does not look into it: operands
// that are zero at compile time are left out here.
__device__ __forceinline__ unsigned xor3(unsigned a, unsigned b, unsigned c) {
  if (__builtin_constant_p(b) && b == 0u) return a ^ c;
  return __builtin_amdgcn_bitop3_b32(a, b, c, 0x96);
}

// Philox-4x32-10, counter (off,0,0,0), key (seed_lo, seed_hi); returns word 0.  Bound by vector issue: 17 products (the
// others fold away, because three counter words start at zero and only word 0 is wanted) and 16 exclusive ors.  A round's
// key enters through the three-input xor: v_xor_b32 with a scalar operand issues at half the rate of the one with two
// vector registers (4.2 against 2.4 clocks), so two of them cost 1.5 x one v_bitop3_b32 (4.2).  Measured, clocks per
// evaluation and wavefront with 2 wavefronts per SIMD: 145 (189 with pairs of v_xor_b32, which is what the compiler makes of
// a ^ b ^ c; 283 with separate high and low products).  All keys in vector registers: 5 % less, for fourteen registers nobody has.
struct PhiloxState { unsigned c0, c1, c2, c3; };
template <int R0, int R1> __device__ __forceinline__ void philox_rounds(PhiloxState& s, unsigned k0, unsigned k1) {   // rounds R0 .. R1-1
#pragma unroll
  for (int r = R0; r < R1; r++) {
    // one 32 x 32 -> 64 bit multiply per product (both halves are needed)
    const unsigned long long p0 = (unsigned long long)0xD2511F53u * (unsigned long long)s.c0;
    const unsigned long long p1 = (unsigned long long)0xCD9E8D57u * (unsigned long long)s.c2;
    const unsigned hi0 = (unsigned)(p0 >> 32), lo0 = (unsigned)p0, hi1 = (unsigned)(p1 >> 32), lo1 = (unsigned)p1;
    s.c0 = xor3(hi1, s.c1, k0 + (unsigned)r * 0x9E3779B9u); s.c1 = lo1;
    s.c2 = xor3(hi0, s.c3, k1 + (unsigned)r * 0xBB67AE85u); s.c3 = lo0;
  }
}
__device__ __forceinline__ unsigned philox_word0(unsigned off, unsigned k0, unsigned k1) {
  PhiloxState s = {off, 0u, 0u, 0u};
  philox_rounds<0, 10>(s, k0, k1);
  return s.c0;
}

// Counter hash of the fast stochastic-rounding mode: one 32-bit mix per 4 consecutive weights of a row; the first
// weight takes the mix itself, the other three its products with odd constants.  idx = global_row * (D/4) + col/4.
// The caller's seed goes through a full 32-bit mixer once, on the host, before it reaches fast_mix: seeds that differ
// in a few bits (s and s + 1, say) must not give related words.
__host__ __device__ inline unsigned fast_seed(unsigned s) {
  s ^= s >> 16; s *= 0x7FEB352Du; s ^= s >> 15; s *= 0x846CA68Bu; s ^= s >> 16;
  return s;
}
constexpr unsigned FAST_MUL = 0x9E3779B1u;
__device__ __forceinline__ unsigned fast_mix_tail(unsigned h) {   // h = idx * FAST_MUL + seed
  h ^= h >> 16; h *= 0x85EBCA77u; h ^= h >> 15;
  return h;
}
__device__ __forceinline__ unsigned fast_mix(unsigned idx, unsigned seed) { return fast_mix_tail(idx * FAST_MUL + seed); }
__device__ __forceinline__ unsigned fast_word(unsigned h, int i) {
  const unsigned k[4] = {1u, 0x27D4EB2Fu, 0x165667B1u, 0x9E3779B1u};
  return h * k[i];
}

// Dropout of the embedding inside the step (training.xmc dropout fused into the preparation of X; the reference keeps a
// prototype of this in src/triton_kernels/tma_gemm.py:7-13): element (b, k) is kept when rand(seed, b * D + k) > p, rand
// being Triton's tl.rand (first Philox-4x32-10 word of counter (offset, 0, 0, 0), key = seed, as a uniform fp32).
struct DropoutParams { float p; float keep_scale; unsigned seed_lo, seed_hi; };   // p == 0: no dropout

__device__ __forceinline__ bool dropout_keep(unsigned off, const DropoutParams& dp) {
  int r = (int)philox_word0(off, dp.seed_lo, dp.seed_hi);
  r = r < 0 ? -r - 1 : r;
  return (float)r * 4.6566127342e-10f > dp.p;
}
// the dropped-out embedding in the layer's type: bf16(keep ? x / (1 - p) : 0)
__device__ __forceinline__ unsigned short dropout_bf16(unsigned short raw, unsigned off, const DropoutParams& dp) {
  if (dp.p == 0.f) return raw;
  return dropout_keep(off, dp) ? bf16_bits(bf16_from_bits(raw) / dp.keep_scale) : (unsigned short)0;
}
// gradient with respect to the embedding in front of the dropout
__device__ __forceinline__ float dropout_backward(float g, unsigned off, const DropoutParams& dp) {
  if (dp.p == 0.f) return g;
  return dropout_keep(off, dp) ? g / dp.keep_scale : 0.f;
}

// The key of a positive: label*256 + (batch row - row0) for the batch rows row0..row0+255 that lie below `batch`;
// 0xFFFFFFFF for every other entry and for labels outside the label space.  Labels are taken relative to label_base, and
// those outside [label_base, label_base + label_count) are dropped: a label space of 2^24 labels and more is taken in
// segments of whole chunks (a key keeps 24 bits for the label).
__device__ __forceinline__ unsigned positive_key(int2 e, int batch, int row0, int label_base, int label_count) {
  const int r = e.x - row0;
  const long long lab = (long long)e.y - label_base;
  return (r >= 0 && r < 256 && r + row0 < batch && e.y >= 0 && lab >= 0 && lab < label_count && lab < (1 << 24) - 1) ? (((unsigned)lab << 8) | (unsigned)r) : 0xFFFFFFFFu;
}

// Which of a wavefront's logits are positives.  The wavefront holds the logits of NLAB labels from label0 on and NROW batch rows from
// row0 on (row0 as the keys count it), one of the two 16, as matrix results: lane l has labels 4 (l / 16).. + 3 of every sixteen and batch
// row l % 16 of every sixteen; with ROWS4 label l % 16 and rows 4 (l / 16).. + 3.  Bit 4 n + e of a lane's result: its e-th label (row)
// of block n (sixteen labels or rows) is a positive.
// keys[p0 .. p1-1] are the positives of the enclosing tile, label * 256 + row, in any order; a repeated one sets its bit again.
//
// Up to eight keys come through the scalar path and are tested one after the other (some 40 clocks each).  More are taken a
// wavefront's worth at a time: a lane tests its own and sets the bit in the wavefront's 64 bytes of LDS, a byte for every lane.  Labels
// sorted by frequency make such tiles: a third of all positives lies in the first, whose cluster everybody waits for at the end.
// us a step, all keys through the scalar path / now, with 5 and with 36 positives a row: fused step, 131 K labels, batch 96, sr_fast
// 90.0 / 81.6 and 149 / 93; one-pass step, FP8, 670 K, batch 256, sr_fast 755 / 728 and 1021 / 780, bf16, 131 K, batch 512, Philox
// 503 / 499 and 769 / 633.  (A line at 16, 32 or 64 keys: the same within 1 %.)
constexpr int POS_SCALAR = 8, POS_LOADS = 4;
template <int NLAB, int NROW, bool ROWS4 = false>
__device__ __forceinline__ unsigned positive_hits(const unsigned* keys, int p0, int p1, unsigned label0, unsigned row0,
                                                  unsigned lane, __attribute__((address_space(3))) unsigned char* mask) {
  static_assert(NLAB == 16 || NROW == 16, "four bits a block");
  unsigned hit = 0;
  auto bit_of = [](unsigned lrel, unsigned br) { return ((lrel >> 4) + (br >> 4)) * 4 + ((ROWS4 ? br : lrel) & 3u); };
  auto lane_of = [](unsigned lrel, unsigned br) { return ROWS4 ? ((br >> 2) & 3u) * 16u + (lrel & 15u) : ((lrel >> 2) & 3u) * 16u + (br & 15u); };
  if (p1 - p0 <= POS_SCALAR) {
    typedef unsigned keysx8 __attribute__((ext_vector_type(POS_SCALAR), aligned(4)));
    // (up to seven keys behind the tile's last are read and ignored: the workspace goes on there)
    const keysx8 kk = *(const __attribute__((address_space(4))) keysx8*)((const __attribute__((address_space(4))) unsigned*)keys + p0);
#pragma unroll
    for (int j = 0; j < POS_SCALAR; j++) {
      const unsigned lrel = (kk[j] >> 8) - label0, br = (kk[j] & 255u) - row0;   // wave-uniform
      if (p0 + j < p1 && lrel < (unsigned)NLAB && br < (unsigned)NROW)
        hit |= lane == lane_of(lrel, br) ? 1u << bit_of(lrel, br) : 0u;
    }
  } else {
    typedef __attribute__((address_space(3))) unsigned lds_u32;
    if (lane < 16u) ((lds_u32*)mask)[lane] = 0u;
    for (int e0 = p0; e0 < p1; e0 += 64 * POS_LOADS) {
      unsigned kk[POS_LOADS];
#pragma unroll
      for (int u = 0; u < POS_LOADS; u++) kk[u] = keys[min(e0 + 64 * u + (int)lane, p1 - 1)];   // (the last one again: it sets the same bit)
#pragma unroll
      for (int u = 0; u < POS_LOADS; u++) {
        const unsigned lrel = (kk[u] >> 8) - label0, br = (kk[u] & 255u) - row0;
        if (lrel < (unsigned)NLAB && br < (unsigned)NROW) {
          const unsigned target = lane_of(lrel, br);
          __hip_atomic_fetch_or((lds_u32*)mask + (target >> 2), 1u << (bit_of(lrel, br) + 8u * (target & 3u)), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
        }
      }
    }
    hit = (((lds_u32*)mask)[lane >> 2] >> (8u * (lane & 3u))) & 255u;
  }
  return hit;
}
// bf16 values a and b (a in the low half) minus one where the bit of `hit` is set
__device__ __forceinline__ unsigned minus_hits(unsigned ab, unsigned hit, int bit_a) {
  const float a = __uint_as_float(ab << 16) - (float)((hit >> bit_a) & 1u), b = __uint_as_float(ab & 0xFFFF0000u) - (float)((hit >> (bit_a + 1)) & 1u);
  return bf16_pack2(a, b);
}

enum RoundMode { ROUND_RTN = 0, ROUND_SR_PHILOX = 1, ROUND_SR_FAST = 2 };

// Round four updated weights (fp32) of one row, columns col..col+3, to e4m3 codes packed in a dword.
//   RTN        round to nearest even, saturating at +-448
//   SR_PHILOX  bits(t) + (philox(seed, row*D+col) & 0xFFFFF), clear low 20 bits, then the RTN cast
//   SR_FAST    true stochastic rounding on the e4m3 grid (subnormals included) by the hardware
//              converter, random word from fast_mix/fast_word
template <int MODE>
__device__ __forceinline__ unsigned round4(float t0, float t1, float t2, float t3, unsigned row_in_chunk,
                                           unsigned grow, unsigned col, unsigned seed) {
  float t[4] = {t0, t1, t2, t3};
  if (MODE == ROUND_SR_PHILOX) {
#pragma unroll
    for (int i = 0; i < 4; i++) {
      unsigned r = philox_word0(row_in_chunk * (unsigned)D + col + i, seed, 0u) & 0xFFFFFu;
      t[i] = __uint_as_float((__float_as_uint(t[i]) + r) & 0xFFF00000u);
    }
  }
  int packed = 0;
  if (MODE == ROUND_SR_FAST) {
    unsigned h = fast_mix(grow * (unsigned)(D / 4) + (col >> 2), seed);
    packed = __builtin_amdgcn_cvt_sr_fp8_f32(clamp448(t[0]), fast_word(h, 0), packed, 0);
    packed = __builtin_amdgcn_cvt_sr_fp8_f32(clamp448(t[1]), fast_word(h, 1), packed, 1);
    packed = __builtin_amdgcn_cvt_sr_fp8_f32(clamp448(t[2]), fast_word(h, 2), packed, 2);
    packed = __builtin_amdgcn_cvt_sr_fp8_f32(clamp448(t[3]), fast_word(h, 3), packed, 3);
  } else {
    packed = __builtin_amdgcn_cvt_pk_fp8_f32(clamp448(t[0]), clamp448(t[1]), packed, false);
    packed = __builtin_amdgcn_cvt_pk_fp8_f32(clamp448(t[2]), clamp448(t[3]), packed, true);
  }
  return (unsigned)packed;
}

// 16-bit key of a bf16 value for the top-k selection: ascending key order == ascending value order, -0 below +0, and
// NaN of either sign above everything (torch.topk treats NaN as the largest value), all NaNs alike.
__device__ __forceinline__ unsigned topk_key(unsigned short bits) {
  if ((bits & 0x7FFFu) > 0x7F80u) return 0xFFFFu;
  return (bits & 0x8000u) ? (unsigned)(~bits & 0xFFFFu) : (unsigned)(bits | 0x8000u);
}
__device__ __forceinline__ unsigned short topk_bits(unsigned key) {   // key 0xFFFF gives back a NaN (0x7FFF)
  return (key & 0x8000u) ? (unsigned short)(key & 0x7FFFu) : (unsigned short)(~key & 0xFFFFu);
}

}  // namespace xmc
