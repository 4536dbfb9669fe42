// Q8_0 x Q8_0 prefill matmul in the scalar f32 order (dot_q8_scalar,
// crates/nr-tensor/src/kernels.rs:72-82: per block, sum += (f32(acc) * dw) * dx)
// for launches of many tokens: y equals the per-token matvec bit for bit
// (matmul_q8, kernels.rs:91-143).
//
// What bounds it. Per (row, token) and 32-value block the order leaves three
// roundings that cannot be merged: a multiply by dw, one by dx and the add. At
// the 2.65 clocks in which a SIMD of two waves or more issues an f32 instruction
// (5.2 with one wave) they cost 127 clocks per 32 x 32 tile and block, four times
// its MFMA step, so everything else is kept off the VALU:
//   - f32(acc) costs nothing: the MFMA accumulates onto the bits of 1.5 * 2^23,
//     so that its result, read as f32, is M = 1.5 * 2^23 + acc (|acc| <= 32 *
//     128 * 128 < 2^22), and fmaf(M, dw, -(1.5 * 2^23 * dw)) rounds acc * dw once
//     (1.5 * 2^23 * dw is exact: dw is an f16). Only acc = 0 against a negative
//     dw may differ, in the sign of a zero, which no sum shows (a sum that starts
//     at +0 is never -0). A weight d that is not finite takes the steps as
//     written instead;
//   - d is converted to f32 once per workgroup and block, when it is staged;
//   - blocks are staged as 16-byte pieces, so an operand is one LDS read at a
//     constant offset. Two 34-byte blocks are 17 dwords: d0|q0q1, seven dwords of
//     block 0, q30q31|d1 and eight dwords of block 1. The dot takes a block's
//     bytes in any order, as long as rows and tokens take the same: dwords 1-4,
//     5-8 with d1 replaced by q0q1, 9-12 and 13-16 need one shuffle in all. Loads
//     are then dword aligned (2-byte aligned 16-byte loads, which would hold the
//     quants in order, cost 31 us of 80 on 2048 x 8192 at 512 tokens);
//   - a wave holds RT 32 x 32 tiles of the same 32 tokens, so a token's operands
//     and d are read once for all of them, and a workgroup of 2 x 2 waves reads
//     each row and token from memory once.
// 16384 x 2048 at 512 tokens: 146 -> 68 us (the arithmetic alone takes 27, this
// kernel's steps without their loads 50); 2048 x 8192: 114 -> 64; 3072 x 2048: 37
// -> 24; 2048 x 2048: 33 -> 19.
#include "nrq_device.h"
#include "nrq_launch.h"

namespace nrq {

namespace {

typedef int i32x16 __attribute__((ext_vector_type(16)));
typedef int i32x4v __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4h __attribute__((ext_vector_type(4), aligned(2)));
typedef uint32_t u32x4d __attribute__((ext_vector_type(4), aligned(4)));

constexpr int kS = 8;     // blocks per stage; the last stage of a row starts early to hold as many
constexpr int kTok = 64;  // tokens of a workgroup
constexpr float kMagic = 12582912.0f;  // 1.5 * 2^23

struct M8Args {
  const uint8_t *w0, *w1, *w2;
  float *y0, *y1, *y2;
  const uint8_t* x;
  int rows0, rows1, rows2;
  int tile1, tile2;  // first row tile of matrices 1 and 2
  int bpr, batch, ntt, nrt;
};

// A stage: planes of 16 quant bytes per row (plane 2b + h: half h of block b;
// 16 spare bytes per plane keep the staging writes of consecutive planes on
// different banks), then d as f32, [block][row].
template <int RT>
struct Stage {
  static constexpr int R = 64 * RT, PW = 16 * R + 16, PX = 16 * kTok + 16;
  static constexpr int W = 0, X = W + 2 * kS * PW, DW = X + 2 * kS * PX, LDW = R + 8, LDX = kTok + 8,
                       DX = DW + 4 * kS * LDW, BYTES = DX + 4 * kS * LDX;
  // one tile per wave: its launches leave one workgroup per CU, whose stores then
  // go to a second buffer; two tiles: two workgroups per CU (57 KB each), one
  // storing while the other computes (two buffers, one workgroup: 100 us against 73)
  static constexpr int NBUF = RT == 1 ? 2 : 1;
};

__device__ __forceinline__ i32x16 mfma_tile(const u32x4& a, const u32x4& b, i32x16 c) {
  const i32x4v av = {(int)a.x, (int)a.y, (int)a.z, (int)a.w};
  const i32x4v bv = {(int)b.x, (int)b.y, (int)b.z, (int)b.w};
  return __builtin_amdgcn_mfma_i32_32x32x32_i8(av, bv, c, 0, 0, 0);
}

// One stage's blocks of a wave's RT tiles: acc[16 rt + e] of row 32 rt + lane % 32
// and token 8(e/4) + 4(lane/32) + e%4. The MFMA step of the next (block, tile)
// issues ahead of this one's f32 steps.
template <int RT, typename PF>
__device__ __forceinline__ void stage_blocks(const uint8_t* st, int wr, int wt, int lane, const i32x16& magic,
                                             float acc[16 * RT], PF prefetch) {
  using St = Stage<RT>;
  const int r = lane & 31, kg = lane >> 5;
  const uint8_t* pw = st + St::W + kg * St::PW + (wr * RT * 32 + r) * 16;
  const uint8_t* px = st + St::X + kg * St::PX + (wt * 32 + r) * 16;
  const float* pdw = (const float*)(st + St::DW) + wr * RT * 32 + r;
  const float* pdx = (const float*)(st + St::DX) + wt * 32 + 4 * kg;
  constexpr int NS = RT == 1 ? 3 : 2;  // operand slots: read a step or two before their MFMA
  u32x4 w[NS][RT], x[NS];
  float4 xd[2][4];
  float dw[2][RT];
  auto ld_op = [&](int b) {
#pragma unroll
    for (int t = 0; t < RT; t++) w[b % NS][t] = *(const u32x4*)(pw + 2 * b * St::PW + 512 * t);
    x[b % NS] = *(const u32x4*)(px + 2 * b * St::PX);
  };
  auto ld_d = [&](int b) {
#pragma unroll
    for (int q = 0; q < 4; q++) xd[b & 1][q] = *(const float4*)(pdx + b * St::LDX + 8 * q);
#pragma unroll
    for (int t = 0; t < RT; t++) dw[b & 1][t] = pdw[b * St::LDW + 32 * t];
  };
  ld_op(0);
  ld_d(0);
  if (NS == 3) ld_op(1);
  i32x16 res[2];
  res[0] = mfma_tile(x[0], w[0][0], magic);
#pragma unroll
  for (int b = 0; b < kS; b++) {
#pragma unroll
    for (int t = 0; t < RT; t++) {
      const int s = b * RT + t, sb = (s + 1) / RT;
      if (t == 0) {
        if (b + 1 < kS) ld_d(b + 1);
        if (b + NS - 1 < kS) ld_op(b + NS - 1);
        prefetch(b);
      }
      if (s + 1 < kS * RT) res[(s + 1) & 1] = mfma_tile(x[sb % NS], w[sb % NS][(s + 1) % RT], magic);
      __builtin_amdgcn_sched_barrier(0);
      const float d = dw[b & 1][t], nk = -(kMagic * d);
      // eight outputs a step at a time: an operation waits for its operand for
      // two issue slots, so that a chain alone would issue every other slot
#pragma unroll
      for (int e0 = 0; e0 < 16; e0 += 8) {
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; e++) v[e] = fmaf(__int_as_float(res[s & 1][e0 + e]), d, nk);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int e = 0; e < 8; e++) {
          const float4 x4 = xd[b & 1][(e0 + e) >> 2];
          v[e] = v[e] * ((e & 3) == 0 ? x4.x : (e & 3) == 1 ? x4.y : (e & 3) == 2 ? x4.z : x4.w);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int e = 0; e < 8; e++) acc[16 * t + e0 + e] = acc[16 * t + e0 + e] + v[e];
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
}

// The same with the reference's steps as written, for any d.
template <int RT>
__device__ __forceinline__ void stage_blocks_any(const uint8_t* st, int wr, int wt, int lane, const i32x16& magic,
                                                 float acc[16 * RT]) {
  using St = Stage<RT>;
  const int r = lane & 31, kg = lane >> 5;
#pragma unroll 1
  for (int b = 0; b < kS; b++) {
    const u32x4 x = *(const u32x4*)(st + St::X + (2 * b + kg) * St::PX + (wt * 32 + r) * 16);
    const float* xd = (const float*)(st + St::DX) + b * St::LDX + wt * 32 + 4 * kg;
#pragma unroll
    for (int t = 0; t < RT; t++) {
      const int row = (wr * RT + t) * 32 + r;
      const i32x16 c = mfma_tile(x, *(const u32x4*)(st + St::W + (2 * b + kg) * St::PW + row * 16), magic);
      const float d = ((const float*)(st + St::DW))[b * St::LDW + row];
#pragma unroll
      for (int e = 0; e < 16; e++)
        acc[16 * t + e] = acc[16 * t + e] + (__int_as_float(c[e]) - kMagic) * d * xd[8 * (e >> 2) + (e & 3)];
    }
  }
}

// EVEN: rows start dword aligned (else two-byte aligned loads, each half block a piece)
template <int RT, bool EVEN>
__global__ __launch_bounds__(256, 2) void mm8_kernel(M8Args a) {
  using St = Stage<RT>;
  constexpr int NBUF = St::NBUF;
  extern __shared__ __align__(16) uint8_t lds[];
  __shared__ int s_bad;  // a weight d that is not finite has been staged
  // XCD-aware numbering: the token tiles of one row tile share an XCD and its L2
  const int wg = (int)blockIdx.x, slot = wg >> 3;
  const int tt = slot % a.ntt, rt = (slot / a.ntt) * 8 + (wg & 7);
  if (rt >= a.nrt) return;  // padding workgroup
  const int m = rt >= a.tile2 ? 2 : rt >= a.tile1 ? 1 : 0;
  const uint8_t* W = m == 2 ? a.w2 : m == 1 ? a.w1 : a.w0;
  float* Y = m == 2 ? a.y2 : m == 1 ? a.y1 : a.y0;
  const int rows = m == 2 ? a.rows2 : m == 1 ? a.rows1 : a.rows0;
  // the last tile of rows and of tokens starts early where it would end past the
  // last one: the values that two tiles then write are the same bits
  const int r0 = min((rt - (m == 2 ? a.tile2 : m == 1 ? a.tile1 : 0)) * St::R, rows - St::R);
  const int t0 = min(tt * kTok, a.batch - kTok);
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wr = wv >> 1, wt = wv & 1;
  const uint32_t ld = (uint32_t)a.bpr * kQ8_0Bytes;  // bytes of a row
  const uint8_t* wb = W + (size_t)r0 * ld;
  const uint8_t* xb = a.x + (size_t)t0 * ld;

  // staging: this thread's 16-byte pieces, row tid / 16 + 16 j, plane tid % 16
  constexpr int NW = St::R / 16, NX = kTok / 16;
  static_assert(2 * kS == 16, "sixteen planes");
  const int pl = tid & 15, pr = tid >> 4, b0 = EVEN ? (pl >> 2) * 2 : pl >> 1;
  const bool tail = EVEN ? (pl & 3) == 1 : (pl & 1) == 0;  // the piece that also takes the pair's first dword, or a block's d
  const uint32_t off = (uint32_t)pr * ld + 34 * b0 + (EVEN ? 4 + 16 * (pl & 3) : 2 + 16 * (pl & 1));
  const uint32_t offh = (uint32_t)pr * ld + 34 * b0;  // the pair's first dword, or the block's d
  u32x4 gw[NW], gx[NX];
  uint32_t hw[NW], hx[NX];
  // part b (of kS) of a stage's loads: six parts hold them all
  auto load = [&](int sp, int b) {
    const uint32_t o = (uint32_t)min(sp * kS, a.bpr - kS) * kQ8_0Bytes;
    constexpr int PER = (NW + NX + 5) / 6;
#pragma unroll
    for (int i = 0; i < NW + NX; i++) {
      if (i / PER != b) continue;
      // a uniform base and one 32-bit offset: no 64-bit address per piece
      const uint8_t* p = i < NW ? wb + o + (size_t)i * 16 * ld : xb + o + (size_t)(i - NW) * 16 * ld;
      asm volatile("" : "+s"(p));
      u32x4 g;
      uint32_t h;
      if constexpr (EVEN) {
        g = *(const u32x4d*)(p + off);
        h = *(const uint32_t*)(p + offh);
      } else {
        g = *(const u32x4h*)(p + off);
        h = *(const uint16_t*)(p + offh);
      }
      if (i < NW) {
        gw[i] = g;
        hw[i] = h;
      } else {
        gx[i - NW] = g;
        hx[i - NW] = h;
      }
    }
  };
  auto store = [&](int sp, uint8_t* st) {
    uint8_t* pw = st + St::W + pl * St::PW + pr * 16;
    uint8_t* px = st + St::X + pl * St::PX + pr * 16;
    if (tail) {
      // blocks that the stage before held contribute zeros: their d are cleared
      const bool seen = min(sp * kS, a.bpr - kS) + b0 < sp * kS;  // of a pair both or neither
      float* pdw = (float*)(st + St::DW) + b0 * St::LDW + pr;
      float* pdx = (float*)(st + St::DX) + b0 * St::LDX + pr;
      bool bad = false;
#pragma unroll
      for (int j = 0; j < NW; j++) {
        const float d0 = f16_bits_to_f32(hw[j] & 0xffffu), d1 = f16_bits_to_f32(gw[j].w >> 16);
        bad |= !(fabsf(d0) <= 65504.0f);
        pdw[16 * j] = seen ? 0.0f : d0;
        if constexpr (EVEN) {
          gw[j].w = __builtin_amdgcn_alignbyte(gw[j].w, hw[j], 2);
          bad |= !(fabsf(d1) <= 65504.0f);
          pdw[16 * j + St::LDW] = seen ? 0.0f : d1;
        }
      }
#pragma unroll
      for (int j = 0; j < NX; j++) {
        const float d0 = f16_bits_to_f32(hx[j] & 0xffffu), d1 = f16_bits_to_f32(gx[j].w >> 16);
        pdx[16 * j] = seen ? 0.0f : d0;
        if constexpr (EVEN) {
          gx[j].w = __builtin_amdgcn_alignbyte(gx[j].w, hx[j], 2);
          pdx[16 * j + St::LDX] = seen ? 0.0f : d1;
        }
      }
      if (bad) s_bad = 1;
    }
#pragma unroll
    for (int j = 0; j < NW; j++) *(u32x4*)(pw + 256 * j) = gw[j];
#pragma unroll
    for (int j = 0; j < NX; j++) *(u32x4*)(px + 256 * j) = gx[j];
  };

  float acc[16 * RT];
#pragma unroll
  for (int e = 0; e < 16 * RT; e++) acc[e] = 0.0f;
  i32x16 magic;
#pragma unroll
  for (int e = 0; e < 16; e++) magic[e] = __float_as_int(kMagic);
  asm volatile("" : "+v"(magic));  // sixteen registers, not sixteen moves per step

  const int nsp = (a.bpr + kS - 1) / kS;
#pragma unroll
  for (int b = 0; b < kS; b++) load(0, b);
  if (tid == 0) s_bad = 0;
  __syncthreads();
  store(0, lds);
  __syncthreads();
  for (int sp = 0; sp < nsp; sp++) {
    const bool more = sp + 1 < nsp;
    auto prefetch = [&](int b) { load(sp + 1, b); };  // past the last stage: the last one again, unused
    const uint8_t* st = lds + (NBUF == 2 ? (sp & 1) * St::BYTES : 0);
    if (__builtin_amdgcn_readfirstlane(s_bad) == 0) {
      stage_blocks<RT>(st, wr, wt, lane, magic, acc, prefetch);
    } else {
      stage_blocks_any<RT>(st, wr, wt, lane, magic, acc);
#pragma unroll
      for (int b = 0; b < kS; b++) prefetch(b);
    }
    if (!more) break;
    if (NBUF == 1) __syncthreads();
    store(sp + 1, lds + (NBUF == 2 ? ((sp + 1) & 1) * St::BYTES : 0));
    __syncthreads();
  }
#pragma unroll
  for (int t = 0; t < RT; t++) {
    const int row = r0 + (wr * RT + t) * 32 + (lane & 31);
#pragma unroll
    for (int e = 0; e < 16; e++) {
      const int tok = t0 + wt * 32 + 8 * (e >> 2) + 4 * (lane >> 5) + (e & 3);
      Y[(size_t)tok * rows + row] = acc[16 * t + e];
    }
  }
}

template <int RT, bool EVEN>
int launch_t(const MatmulGroupLaunch& G) {
  using St = Stage<RT>;
  M8Args a{};
  int n[3] = {0, 0, 0};
  for (int i = 0; i < G.nmat; i++) n[i] = (G.rows[i] + St::R - 1) / St::R;
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
  a.ntt = (G.batch + kTok - 1) / kTok;
  a.nrt = n[0] + n[1] + n[2];
  const long nwg = (long)((a.nrt + 7) / 8) * 8 * a.ntt;
  if (nwg > 0x7fffffffL) return NRQ_LAUNCH_BAD_ARG;
  hipLaunchKernelGGL((mm8_kernel<RT, EVEN>), dim3((unsigned)nwg), dim3(256), St::NBUF * St::BYTES, (hipStream_t)G.stream, a);
  return hipGetLastError() == hipSuccess ? NRQ_LAUNCH_OK : NRQ_LAUNCH_FAILED;
}

}  // namespace

static long mm8_tiles(const MatmulGroupLaunch& G, int tile) {
  long n = 0;
  for (int i = 0; i < G.nmat; i++) n += (G.rows[i] + tile - 1) / tile;
  return n * ((G.batch + kTok - 1) / kTok);
}

static uintptr_t mm8_bases(const MatmulGroupLaunch& G) {
  uintptr_t b = (uintptr_t)G.xs;
  for (int i = 0; i < G.nmat; i++) b |= (uintptr_t)G.w[i];
  return b;
}

// rows start dword aligned
static bool mm8_even(const MatmulGroupLaunch& G) { return G.bpr % 2 == 0 && (mm8_bases(G) & 3u) == 0; }

// Whole stages, and whole tiles (a short one starts early), and enough of them (times:
// us here, on the kernel that takes the launch otherwise).
//  - From 96 workgroups of 64 x 64: with fewer, the splits of nrq_mmt.hip keep more of
//    the chip busy (2048 x 2048 at 128 tokens, 64: 18.0, 14.4; 3072 x 2048 at 128, 96:
//    17.9, 25.6; 2048 x 8192 at 256, 128: 63, 89). Odd rows, whose two-byte loads cost
//    more, from where an XCD has more than two of those kernels' tiles per CU (4266 x
//    1120 at 85, 51 tiles per XCD: 14.1, 13.5; 4643 x 4640 at 84, 57: 41.9, 41.8; 4102 x
//    736 at 118, 68: 10.1, 11.7; 1191 x 4512 at 395, 65: 39.8, 53.6), and not where the
//    whole stages are 1.6 times the row (9908 x 288 at 262: 18.8, 15.1).
//  - Below 1024 rows the other kernel is that of nrq_mmq.hip. Up to two rounds here a
//    launch takes 0.25 us per block of whole stages and 2.5 or (odd rows) 4 us more;
//    there 0.19 to 0.46 us per block as its workgroups per XCD fill two, three, four and
//    more rounds of the CUs, and a fifth more where rows are multiples of 128 bytes (225 x
//    10240 at 371 tokens, 48 per XCD: 82, 63; 370 x 9856 at 455, 87: 76.7, 69.7; 604 x 6144
//    at 277, 90: 48.3, 54.8; 674 x 2432 at 305, 120: 22.1, 23.2; 967 x 1600 at 244, 128:
//    16.5, 15.6; 732 x 1760 at 354, 138: 17.9, 20.5; 517 x 1056 at 456, 145: 13.9, 12.5;
//    742 x 9824 at 344, 154: 80.8, 106.8).
bool mm8_fits(const MatmulGroupLaunch& G, bool any_size) {
  long total = 0, rt32 = 0, rt16 = 0;
  for (int i = 0; i < G.nmat; i++) {
    if (G.rows[i] < Stage<1>::R) return false;
    total += G.rows[i];
    rt32 += (G.rows[i] + 31) / 32;
    rt16 += (G.rows[i] + 15) / 16;
  }
  if (G.batch < kTok || G.bpr < kS || G.bpr > (1 << 22) || (mm8_bases(G) & 1u)) return false;
  if (any_size) return true;
  const bool even = mm8_even(G);
  const double blocks = (G.bpr + kS - 1) / kS * kS;
  if (total >= 1024)
    return mm8_tiles(G, Stage<1>::R) >= 96 &&
           (even || ((rt32 + 7) / 8 * ((G.batch + 31) / 32) > 64 && blocks < 1.6 * G.bpr));
  const long per_xcd = (rt16 + 7) / 8 * ((G.batch + 15) / 16);
  if (per_xcd > 192) return true;
  const double there =
      (per_xcd <= 64 ? 0.19 : per_xcd <= 96 ? 0.24 : per_xcd <= 128 ? 0.31 : per_xcd <= 160 ? 0.38 : 0.46) * G.bpr;
  return 0.25 * blocks + (even ? 2.5 : 4.0) < (G.bpr % 64 ? there : 1.2 * there);
}

// Two launches cost what the others take here (as above, by rounds of two workgroups
// per CU) and about 2 us and 0.12 us per block for each short one; one launch of
// nrq_mmt.hip 3.4 us and 4.2 ns per block and 32 x 32 tile of an XCD. Split where that is
// 10% more (us split, in one: 6 + 5198 x 1472 at 314 tokens 24.9, 42.0; 9769 + 12 x 8608 at
// 135: 132, 216; 62 + 4121 + 2383 x 1536 at 135: 25.2, 34.6; 4870 + 41 x 2400 at 188: 33.3, 42.4;
// 3000 + 40 + 3200 x 1088 at 67: 30.0 in three launches, 16.1).
bool mm8_fits_but_short(const MatmulGroupLaunch& G, MatmulGroupLaunch* tall) {
  *tall = G;
  tall->nmat = 0;
  long rt32 = 0;
  for (int i = 0; i < G.nmat; i++) {
    rt32 += (G.rows[i] + 31) / 32;
    if (G.rows[i] < Stage<1>::R) continue;
    tall->w[tall->nmat] = G.w[i];
    tall->y[tall->nmat] = G.y[i];
    tall->rows[tall->nmat++] = G.rows[i];
  }
  if (tall->nmat == 0 || tall->nmat == G.nmat || !mm8_fits(*tall, false)) return false;
  const double blocks = (G.bpr + kS - 1) / kS * kS, rounds = (mm8_tiles(*tall, Stage<1>::R) + 511) / 512;
  const double split = 0.25 * blocks * rounds + (mm8_even(G) ? 2.5 : 4.0) + (2.0 + 0.12 * G.bpr) * (G.nmat - tall->nmat);
  return 1.1 * split < 3.4 + 0.0042 * G.bpr * ((rt32 + 7) / 8 * ((G.batch + 31) / 32));
}

int launch_mm8(const MatmulGroupLaunch& G) {
  // two tiles per wave where that leaves two workgroups per CU (16384 x 2048 at
  // 512 / 256 / 128 tokens: 73 / 37 / 29 us, one tile 92 / 45 / 25 us)
  bool wide = mm8_tiles(G, Stage<2>::R) >= 512;
  for (int i = 0; i < G.nmat; i++) wide = wide && G.rows[i] >= Stage<2>::R;
  // rows of an odd block count alternate their alignment within a dword
  if (!mm8_even(G)) return wide ? launch_t<2, false>(G) : launch_t<1, false>(G);
  return wide ? launch_t<2, true>(G) : launch_t<1, true>(G);
}

}  // namespace nrq
