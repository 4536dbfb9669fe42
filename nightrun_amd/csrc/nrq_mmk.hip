// Q4_K x Q8_K prefill matmul in the scalar f32 order (dot_q4k_scalar,
// crates/nr-tensor/src/kquant.rs:192-218) for launches of many tokens: y equals the
// per-token matvec bit for bit (kquant_matmul!, kquant.rs:566-639).
//
// What bounds it: the f32 steps per (row, token) and block, on the VALU, and what a
// wave waits for between blocks. On gfx950 a SIMD with two waves or more issues an f32
// add, multiply or fma every 2.7 clocks, a conversion, a 24-bit integer multiply-add or
// a three-operand integer add every 4.5, so the steps run on f32 alone:
//   - an MFMA result is read as an f32: it accumulates onto 2^16, and the integer's
//     bits are then a denormal, (2^16 + sub) * 2^-149. With scales of 2^120 * sc the
//     sums stand for units of 2^-29, exact as in units of one;
//   - the first four partial sums are below 2^24 in any case, so they start at -2^16 *
//     (sc_0 + .. + sc_3) and take the biased values, one fma each; the last four round
//     as the reference's and take the bias off first;
//   - sum_m comes from f16 MFMA steps, whose result is an f32.
// A wave holds 32 rows x 32 TT tokens, so that weights are unpacked once for TT tiles;
// a workgroup is four waves over 128 rows that share the tokens' blocks, staged through
// LDS in two buffers a block at a time (bsums as f16). Weights go straight to registers
// once the block before has been unpacked (staged through LDS too: 93 us against 86).
// 19456 x 2560 at 512 tokens: 100-106 -> 81 us (these steps without loads and stores 60).
#include "nrq_device.h"
#include "nrq_launch.h"

namespace nrq {

namespace {

typedef int i32x16 __attribute__((ext_vector_type(16)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef int i32x4v __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4d __attribute__((ext_vector_type(4), aligned(4)));

constexpr int kRowsWg = 128;

// A staged block: 16 planes of 16 quants per token, four of bsums as f16 (low bytes,
// high bytes; 16 spare bytes per plane: consecutive ones on different banks), then d
template <int TT>
struct Stage {
  static constexpr int TOK = 32 * TT, PL = 16 * TOK + 16, BS = 16 * PL, D = 20 * PL, BYTES = D + 4 * TOK;
};

struct MkArgs {
  const uint8_t *w0, *w1, *w2;
  float *y0, *y1, *y2;
  const uint8_t* x;
  int rows0, rows1, rows2;
  int tile1, tile2;  // first row tile of matrices 1 and 2
  int bpr, batch, ntt, nrt;
  int whole;  // workgroups per XCD that take whole row tiles
};

__device__ __forceinline__ i32x16 mfma32(const u32x4& a, const u32x4& b, const i32x16& c) {
  const i32x4v av = {(int)a.x, (int)a.y, (int)a.z, (int)a.w};
  const i32x4v bv = {(int)b.x, (int)b.y, (int)b.z, (int)b.w};
  return __builtin_amdgcn_mfma_i32_32x32x32_i8(av, bv, c, 0, 0, 0);
}
__device__ __forceinline__ f32x16 mfma_f16(const u32x4& a, const u32x4& b, const f32x16& c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}
// (1024 + byte) as f16 for two bytes of v, less `off`
__device__ __forceinline__ uint32_t f16_of_bytes(uint32_t v, uint32_t sel, _Float16 off) {
  const f16x2 h = __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(0x64646464u, v, sel));
  return __builtin_bit_cast(uint32_t, h - (f16x2){off, off});
}

__device__ __forceinline__ float f4(const float4& v, int i) { return i == 0 ? v.x : i == 1 ? v.y : i == 2 ? v.z : v.w; }

// ---- Q4_K: a lane's row (lane % 32) and its 16 bytes (half lane / 32) of each sub-block pair
struct Q4 {
  u32x4 h;     // d | dmin, scales[12]
  u32x4 q[4];  // qs bytes 32c + 16kg .. +16
};
__device__ __forceinline__ void load_w(Q4& L, const uint8_t* wb, int kg) {
  L.h = *(const u32x4*)wb;
#pragma unroll
  for (int c = 0; c < 4; c++) L.q[c] = *(const u32x4*)(wb + 16 + 32 * c + 16 * kg);
}
__device__ __forceinline__ u32x4 q4_op(const Q4& L, int j) {
  const u32x4 q = L.q[j >> 1];
  return ((j & 1) ? q >> 4 : q) & 0x0f0f0f0fu;
}

// An empty statement that the sums pass through: left alone, the compiler forms them
// after a block's last step and holds every step's result until then
__device__ __forceinline__ void keep16(float S[16]) {
  asm volatile("" : "+v"(S[0]), "+v"(S[1]), "+v"(S[2]), "+v"(S[3]), "+v"(S[4]), "+v"(S[5]), "+v"(S[6]), "+v"(S[7]),
               "+v"(S[8]), "+v"(S[9]), "+v"(S[10]), "+v"(S[11]), "+v"(S[12]), "+v"(S[13]), "+v"(S[14]), "+v"(S[15]));
}

constexpr int kBias = 1 << 16;        // at least any |sub| (15 * 32 * 128)
constexpr float kUnit = 0x1p-29f;     // what 1 stands for in the sums
constexpr float kUp = 0x1p120f;       // kUnit / 2^-149
constexpr float kBiasF = 0x1p-133f;   // kBias as the bits of an f32

// One block for a wave's TT tiles. st: the stage.
// next() runs once L is no longer read.
template <int TT, typename NX>
__device__ __forceinline__ void block_q4(const Q4& L, const uint8_t* st, int lane, const i32x16& bias,
                                         float acc[16 * TT], NX next) {
  using St = Stage<TT>;
  const int r = lane & 31, kg = lane >> 5;
  const uint8_t* at = st + kg * St::PL + r * 16;
  const u32x4 h = L.h;
  // kquant.rs:83-92, four scales or mins per word
  const uint32_t scA = h.y & 0x3f3f3f3fu, mnA = h.z & 0x3f3f3f3fu;
  const uint32_t scB = (h.w & 0x0f0f0f0fu) | ((h.y >> 2) & 0x30303030u);
  const uint32_t mnB = ((h.w >> 4) & 0x0f0f0f0fu) | ((h.z >> 2) & 0x30303030u);
  const float dw = f16_bits_to_f32(h.x & 0xffffu), dmw = f16_bits_to_f32(h.x >> 16);
  u32x4 a[3][TT];  // operands are read two sub-blocks ahead
  auto ld_a = [&](int j) {
#pragma unroll
    for (int t = 0; t < TT; t++) a[j % 3][t] = *(const u32x4*)(at + 2 * j * St::PL + 512 * t);
  };
  ld_a(0);
  ld_a(1);
  u32x4 w = q4_op(L, 0);
  i32x16 res[2];
  res[0] = mfma32(a[0][0], w, bias);
  // the first four partial sums start at -kBias * (sc_0 + .. + sc_3): every one of
  // them is a multiple of the unit below 2^24, so exact with the bias as without
  float sc0 = 0.0f;
#pragma unroll
  for (int j = 0; j < 4; j++) sc0 = sc0 - (float)((scA >> (8 * j)) & 0xffu);
  sc0 = sc0 * ((float)kBias * kUnit);
  // sum_m = sum_k m_{k/2} * bsums[k] (kquant.rs:209-213), bsum = 256 hi + lo, in f16
  // with f32 sums: all integers below 2^24 for the bsums of int8 quants (|bsum| <= 16 *
  // 128; the quantizer writes no others). Lane half kg holds bsums 8kg .. 8kg+7
  const uint32_t mn = kg ? mnB : mnA;
  auto sum_m = [&](int t) {
    u32x4 m, m256;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const uint32_t v = f16_of_bytes(mn, 0x04000400u + 0x00010001u * i, 1024);
      const f16x2 h2 = __builtin_bit_cast(f16x2, v) * (f16x2){256, 256};
      m[i] = v;
      m256[i] = __builtin_bit_cast(uint32_t, h2);
    }
    const uint8_t* pb = st + St::BS + kg * St::PL + r * 16 + 512 * t;
    const f32x16 z = {};
    return mfma_f16(*(const u32x4*)(pb + 2 * St::PL), m256, mfma_f16(*(const u32x4*)pb, m, z));
  };
  float4 d4[4];
  auto ld_d = [&](int t) {
#pragma unroll
    for (int q = 0; q < 4; q++) d4[q] = *(const float4*)((const float*)(st + St::D) + 32 * t + 4 * kg + 8 * q);
  };
  float sq[TT][16];
  f32x16 sm;
#pragma unroll
  for (int j = 0; j < 8; j++) {
    const float sc = (float)(((j < 4 ? scA : scB) >> (8 * (j & 3))) & 0xffu) * kUp;
#pragma unroll
    for (int t = 0; t < TT; t++) {
      const int s = j * TT + t;
      if (t == 0 && j < 6) ld_a(j + 2);
      if (t == TT - 1 && j < 7) w = q4_op(L, j + 1);
      if (s + 1 < 8 * TT) res[(s + 1) & 1] = mfma32(a[((s + 1) / TT) % 3][(s + 1) % TT], w, bias);
      if (s + 1 == 8 * TT) {
        next();
        sm = sum_m(0);
        ld_d(0);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int e = 0; e < 16; e++) {
        const float m = __int_as_float(res[s & 1][e]);
        sq[t][e] = j < 4 ? fmaf(sc, m, j == 0 ? sc0 : sq[t][e]) : fmaf(sc, m - kBiasF, sq[t][e]);
      }
      keep16(sq[t]);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
#pragma unroll
  for (int t = 0; t < TT; t++) {
#pragma unroll
    for (int e = 0; e < 16; e++) {
      const float x = f4(d4[e >> 2], e & 3);
      const float av = (dw * x) * (sq[t][e] * (1.0f / kUnit)), mv = (dmw * x) * sm[e];
      acc[16 * t + e] = acc[16 * t + e] + (av - mv);  // kquant.rs:215
    }
    if (t + 1 < TT) {
      __builtin_amdgcn_sched_barrier(0);
      sm = sum_m(t + 1);
      ld_d(t + 1);
    }
  }
}

template <int TT>
__global__ __launch_bounds__(256, 2) void mmk_kernel(MkArgs a) {
  __shared__ __align__(16) uint8_t lds[2 * Stage<TT>::BYTES];
  // XCD-aware numbering: the token tiles of one row tile share an XCD and its L2, eight
  // neighbouring row tiles at a time; past the first a.whole tiles of each XCD the rest go
  // round the XCDs one by one
  const int xcd = (int)blockIdx.x & 7, slot = (int)blockIdx.x >> 3, k = (slot - a.whole) * 8 + xcd;
  const int rt = slot < a.whole ? slot / a.ntt * 8 + xcd : (a.nrt & ~7) + k / a.ntt;
  const int tt = slot < a.whole ? slot % a.ntt : k % a.ntt;
  if (rt >= a.nrt) return;  // padding workgroup
  const int m = rt >= a.tile2 ? 2 : rt >= a.tile1 ? 1 : 0;
  const uint8_t* W = m == 2 ? a.w2 : m == 1 ? a.w1 : a.w0;
  float* Y = m == 2 ? a.y2 : m == 1 ? a.y1 : a.y0;
  const int rows = m == 2 ? a.rows2 : m == 1 ? a.rows1 : a.rows0;
  // the last tile of rows and of tokens starts early where it would end past the
  // last one: the values that two tiles then write are the same bits
  const int r0 = min((rt - (m == 2 ? a.tile2 : m == 1 ? a.tile1 : 0)) * kRowsWg, rows - kRowsWg);
  const int t0 = min(tt * Stage<TT>::TOK, a.batch - Stage<TT>::TOK);
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  constexpr int BS = kQ4KBytes;
  const uint8_t* wrow = W + (size_t)(r0 + 32 * wv + (lane & 31)) * a.bpr * BS;
  const uint32_t ld = (uint32_t)a.bpr * kQ8KBytes;  // bytes of a token's row
  const uint8_t* xb = a.x + (size_t)t0 * ld;

  // staging: quants of tokens tid / 16 + 16 k, plane tid % 16; and one piece more:
  // a bsums piece (threads 0 .. 2 Stage<TT>::TOK - 1), or the block's first bytes with d
  const int pl = tid & 15, pt = tid >> 4;
  const uint32_t off = (uint32_t)pt * ld + 4 + 16 * pl;
  const bool isb = tid < 2 * Stage<TT>::TOK;
  const int et = isb ? tid >> 1 : tid & (Stage<TT>::TOK - 1);
  const uint32_t offe = (uint32_t)et * ld + (isb ? 260 + 16 * (tid & 1) : 0);
  u32x4 gx[Stage<TT>::TOK / 16], ge;
  auto load_x = [&](int b) {
    const uint8_t* p = xb + (size_t)b * kQ8KBytes;
#pragma unroll
    for (int k = 0; k < Stage<TT>::TOK / 16; k++) {
      const uint8_t* pk = p + (size_t)k * 16 * ld;
      asm volatile("" : "+s"(pk));
      gx[k] = *(const u32x4d*)(pk + off);
    }
    asm volatile("" : "+s"(p));
    ge = *(const u32x4d*)(p + offe);
  };
  auto store_x = [&](uint8_t* st) {
#pragma unroll
    for (int k = 0; k < Stage<TT>::TOK / 16; k++) *(u32x4*)(st + pl * Stage<TT>::PL + (pt + 16 * k) * 16) = gx[k];
    if (isb) {
      u32x4 lo, hi;
#pragma unroll
      for (int i = 0; i < 4; i++) {
        lo[i] = f16_of_bytes(ge[i], 0x04020400u, 1024);
        hi[i] = f16_of_bytes(ge[i] ^ 0x80008000u, 0x04030401u, 1024 + 128);
      }
      uint8_t* pb = st + Stage<TT>::BS + (tid & 1) * Stage<TT>::PL + et * 16;
      *(u32x4*)pb = lo;
      *(u32x4*)(pb + 2 * Stage<TT>::PL) = hi;
    } else *(uint32_t*)(st + Stage<TT>::D + 4 * et) = ge.x;
  };

  float acc[16 * TT];
#pragma unroll
  for (int e = 0; e < 16 * TT; e++) acc[e] = 0.0f;
  i32x16 bias;
#pragma unroll
  for (int e = 0; e < 16; e++) bias[e] = kBias;
  asm volatile("" : "+v"(bias));  // sixteen registers, not sixteen moves per step
  Q4 L;
  load_x(0);
  load_w(L, wrow, lane >> 5);
  store_x(lds);
  __syncthreads();
  for (int b = 0; b < a.bpr; b++) {
    const int bn = min(b + 1, a.bpr - 1);  // past the last block: the last one again, unused
    load_x(bn);
    __builtin_amdgcn_sched_barrier(0);
    block_q4<TT>(L, lds + (b & 1) * Stage<TT>::BYTES, lane, bias, acc,
                 [&]() { load_w(L, wrow + (size_t)bn * BS, lane >> 5); });
    store_x(lds + ((b + 1) & 1) * Stage<TT>::BYTES);
    __syncthreads();
  }
  const int row = r0 + 32 * wv + (lane & 31);
#pragma unroll
  for (int t = 0; t < TT; t++) {
#pragma unroll
    for (int e = 0; e < 16; e++) {
      const int tok = t0 + 32 * t + 8 * (e >> 2) + 4 * (lane >> 5) + (e & 3);
      Y[(size_t)tok * rows + row] = acc[16 * t + e];
    }
  }
}

template <int TT>
int launch_t(const MatmulGroupLaunch& G) {
  MkArgs a{};
  int n[3] = {0, 0, 0};
  for (int i = 0; i < G.nmat; i++) n[i] = (G.rows[i] + kRowsWg - 1) / kRowsWg;
  a.w0 = a.w1 = a.w2 = (const uint8_t*)G.w[0];
  a.y0 = a.y1 = a.y2 = G.y[0];
  a.rows0 = a.rows1 = a.rows2 = G.rows[0];
  a.tile1 = a.tile2 = 0x7fffffff;
  if (G.nmat > 1) {
    a.w1 = (const uint8_t*)G.w[1];
    a.y1 = G.y[1];
    a.rows1 = G.rows[1];
    a.tile1 = n[0];
  }
  if (G.nmat > 2) {
    a.w2 = (const uint8_t*)G.w[2];
    a.y2 = G.y[2];
    a.rows2 = G.rows[2];
    a.tile2 = n[0] + n[1];
  }
  a.x = (const uint8_t*)G.xs;
  a.bpr = G.bpr;
  a.batch = G.batch;
  a.ntt = (G.batch + Stage<TT>::TOK - 1) / Stage<TT>::TOK;
  a.nrt = n[0] + n[1] + n[2];
  // Whole row tiles per XCD, unless the XCDs that take one more than the others then need
  // a round of workgroups more than the tiles do (4480 x 4864 at 405 tokens, 455 tiles, 35
  // row tiles x 13: 65 workgroups on three XCDs of 32 CUs: 48.9 us, shared out 41.3). Shared out in every
  // launch the last nrt % 8 row tiles lose the L2 (5761 x 3840 at 266: 31.5, 33.4).
  const long all = (long)((a.nrt + 7) / 8) * a.ntt, even = ((long)a.nrt * a.ntt + 7) / 8;
  const bool share = (all + 31) / 32 > (even + 31) / 32;
  const long nwg = 8 * (share ? even : all);
  if (8 * all > 0x7fffffffL) return NRQ_LAUNCH_BAD_ARG;
  a.whole = (int)(share ? (long)(a.nrt / 8) * a.ntt : all);
  hipLaunchKernelGGL((mmk_kernel<TT>), dim3((unsigned)nwg), dim3(256), 0, (hipStream_t)G.stream, a);
  return hipGetLastError() == hipSuccess ? NRQ_LAUNCH_OK : NRQ_LAUNCH_FAILED;
}

long mmk_tiles(const MatmulGroupLaunch& G, int tok) {
  long n = 0;
  for (int i = 0; i < G.nmat; i++) n += (G.rows[i] + kRowsWg - 1) / kRowsWg;
  return n * ((G.batch + tok - 1) / tok);
}

}  // namespace

// Whole tiles (a short one starts early), and enough of them. The splits of
// nrq_mmt.hip are as fast or faster (us here, there)
//  - below 300 workgroups of 128 x 32 (2560 x 4096 at 256 tokens, 160: 29.7, 22.1; from
//    there 5120 x 2560 at 256, 320: 21.1, 22.8; 2560 x 4096 at 512, 320: 32.7, 33.4;
//    5000 x 3328 at 300, 400: 28.2, 31.0), and from 24 blocks a row below 400 (4463 +
//    6013 x 7936 at 110, 328: 61.1, 59.8; 1798 + 587 + 9648 x 6656 at 97, 384: 52.6, 51.8;
//    from there 3759 x 7680 at 424, 420: 58.4, 60.8);
//  - with rows of 32 blocks and more (2560 x 9728 at 512, 320: 71.6, 71.4);
//  - where 128-row tiles make one round of 256 workgroups more than the rows fill, up
//    to the fourth (2472 + 268 + 7968 x 2048 at 258, 774 for 3024 tiles of 32 x 32:
//    37.6, 32.3; 3616 + 168 + 4323 x 5632 at 233, 520 for 2040: 58.1, 49.7).
bool mmk_fits(const MatmulGroupLaunch& G, bool any_size) {
  long n32 = 0;
  for (int i = 0; i < G.nmat; i++) {
    if (G.rows[i] < kRowsWg) return false;
    n32 += (G.rows[i] + 31) / 32;
  }
  if (G.batch < 64 || G.bpr > (1 << 17)) return false;
  if (any_size) return true;
  const long tiles = mmk_tiles(G, 32);
  n32 *= (G.batch + 31) / 32;
  return G.bpr < 32 && tiles >= (G.bpr < 24 ? 300 : 400) && (tiles > 1024 || (tiles + 255) / 256 <= (n32 + 1023) / 1024);
}

int launch_mmk(const MatmulGroupLaunch& G) {
  // two tiles per wave from four workgroups per CU (19456 x 2560 at 512 tokens, 1216:
  // 86 us, one tile 96; at 256, 608: 52.6, one tile 47.0)
  return mmk_tiles(G, 64) >= 1024 ? launch_t<2>(G) : launch_t<1>(G);
}

}  // namespace nrq
