// Causal prefill attention (infer.rs:601-759) for many tokens at once, as three
// launches over tiles of four (token, head) rows of one KV head:
//   scores   s[r][t] = dot_f16(k_t, q_r) * scale (kernels.rs:146-160): a lane is
//            a position and holds its key row in f32 registers, q comes
//            through scalar registers, and every sum runs in dimension order;
//   softmax  (vec.rs:30-42) max, expf, the exp-sum in position order (one lane
//            per row), p = e * inv, in place;
//   values   out[r][d] += p[r][t] * v_t[d] in position order (kernels.rs:163-173):
//            a lane is a dimension and holds four rows' sums, p comes through
//            scalar registers and v from a chunk the workgroup's waves share in LDS.
// The two products are what the arithmetic costs: a multiply and an add per
// (row, position, dimension), which the reference rounds separately, so no
// matrix instruction applies, and the VALU rate bounds both. The scalar
// operands keep everything else out of the inner loops: no LDS read and no
// conversion per product (a key or value is converted once per 32 rows or once
// per workgroup).
// The weights pass through memory between the launches (the scalar cache does
// not see vector stores of its own launch).
// Llama-3.2-1B widths, a 512-token chunk at 1000 positions on average: 51 us
// scores + 48 us softmax + 64 us values, against 650 us for one workgroup per
// (KV head, token). Each product's multiplies and adds alone take 35 us at the
// 2.65 clocks in which a SIMD of two waves or more issues an f32 instruction; the
// rest of a product's time (waits for scalar loads, conversions, launch tails) has
// not been taken apart. The softmax's LDS (16 bytes per position) leaves fewer workgroups
// per CU as rows grow, one at 8192 positions: whole prompts of 8000 tokens, two
// layers, still take a third of the other kernels' time (Llama-3.2-1B widths 33 ms
// against 88, Qwen3-4B widths 49 against 152).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "nrq_device.h"
#include "nrq_launch.h"

namespace nrq {

namespace {

constexpr int kRows = kPfRows;  // rows of a tile
constexpr int kChunk = 256;     // positions per softmax step
constexpr int kVT = 32;         // positions per value chunk
constexpr int kBatch = 64 / kRows;  // dimensions or positions whose scalars (64 registers) are loaded together

struct PfArgs {
  const uint16_t* kc;
  const uint16_t* vc;
  float* s;  // [n_kv][nrbc][n64][kRows]
  float* out;
  uint8_t* out_q8;
  uint8_t* out_q8k;
  int gqa, nkv, ctx, layer, base, tokens, nrb, rb0, nrbc, n64, group;
  float scale;
};

// positions row r of tile rb attends to; rows past the last repeat it
__device__ __forceinline__ int row_n(const PfArgs& a, int rb, int r) {
  return a.base + min((rb * kRows + r) / a.gqa, a.tokens - 1) + 1;
}

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef const __attribute__((address_space(4))) f32x16* scalar_ptr;

// acc[r] += x[i] * s[i][r] for i = 0..kBatch-1 in order, the 64 scalars loaded
// together: a scalar load's latency is paid once per 128 VALU instructions. With
// MASK row r stops before i = n[r] (a later value may be anything, NaN included)
template <bool MASK>
__device__ __forceinline__ void scalar_batch(const float* s, const float* x, float acc[kRows], int4 n) {
  const scalar_ptr sp = (scalar_ptr)(uintptr_t)s;
  f32x16 v[4];
#pragma unroll
  for (int j = 0; j < 4; j++) v[j] = sp[j];
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = 0; i < kBatch; i++) {
#pragma unroll
    for (int r = 0; r < kRows; r++) {
      const float y = acc[r] + x[i] * v[(i * kRows + r) / 16][(i * kRows + r) % 16];
      acc[r] = !MASK || i < (r == 0 ? n.x : r == 1 ? n.y : r == 2 ? n.z : n.w) ? y : acc[r];
    }
  }
}

template <int HD>
__global__ __launch_bounds__(256) void pf_scores_kernel(PfArgs a, const float* __restrict__ qt,
                                                        float* __restrict__ s) {
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int g = (int)blockIdx.x % a.nkv, rg = (int)blockIdx.x / a.nkv;
  const int t0 = ((int)blockIdx.y * 4 + w) * 64;
  const int rb_first = rg * a.group, rb_end = min(rb_first + a.group, a.nrbc);
  if (t0 >= row_n(a, a.rb0 + rb_end - 1, kRows - 1)) return;
  const int t = t0 + lane;
  const uint4* src =
      (const uint4*)(a.kc + ((size_t)a.layer * a.nkv + g) * HD * a.ctx) + (size_t)min(t, a.ctx - 1);
  float k[HD];
#pragma unroll
  for (int p = 0; p < HD / 8; p++) {
    const uint4 kr = src[(size_t)p * a.ctx];
    const uint32_t kw[4] = {kr.x, kr.y, kr.z, kr.w};
#pragma unroll
    for (int e = 0; e < 4; e++) {
      k[8 * p + 2 * e] = f16_bits_to_f32(kw[e] & 0xffffu);
      k[8 * p + 2 * e + 1] = f16_bits_to_f32(kw[e] >> 16);
    }
  }
  for (int rb = rb_first; rb < rb_end; rb++) {
    if (t0 >= row_n(a, a.rb0 + rb, kRows - 1)) continue;
    const float* q = qt + (((size_t)g * a.nrb + a.rb0 + rb) * HD) * kRows;
    float acc[kRows];
#pragma unroll
    for (int r = 0; r < kRows; r++) acc[r] = 0.0f;
#pragma unroll
    for (int d = 0; d < HD; d += kBatch) scalar_batch<false>(q + d * kRows, k + d, acc, int4{});
    *(float4*)(s + (((size_t)g * a.nrbc + rb) * a.n64 + t) * kRows) =
        make_float4(acc[0] * a.scale, acc[1] * a.scale, acc[2] * a.scale, acc[3] * a.scale);
  }
}

// One workgroup per tile, whose rows stay in LDS from the maximum to the
// division (one read and one write of the weights in memory): four waves take
// the elements (thread = position of a chunk), the fifth the exp-sum chains, a
// chunk behind.
constexpr int softmax_row(int n) { return ((n + kChunk - 1) & ~(kChunk - 1)) + 4; }  // floats

__global__ __launch_bounds__(320) void pf_softmax_kernel(PfArgs a) {
  static_assert(kRows == 4, "a float4 per position");
  extern __shared__ __align__(16) float rows[];  // [kRows][ld]
  __shared__ __align__(16) float red[4][kRows];
  __shared__ float invs[kRows];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int g = (int)blockIdx.x % a.nkv, rbl = a.nrbc - 1 - (int)blockIdx.x / a.nkv, rb = a.rb0 + rbl;
  float4* s4 = (float4*)(a.s + ((size_t)g * a.nrbc + rbl) * a.n64 * kRows);
  const int n0 = row_n(a, rb, 0), n1 = row_n(a, rb, 1), n2 = row_n(a, rb, 2), n3 = row_n(a, rb, 3);
  const int nc = (n3 + kChunk - 1) / kChunk, ld = softmax_row(n3);
  float4 mx = make_float4(-INFINITY, -INFINITY, -INFINITY, -INFINITY);
  if (w < 4) {
#pragma unroll 4
    for (int t = tid; t < n3; t += kChunk) {
      const float4 v = s4[t];
      rows[t] = v.x;
      rows[ld + t] = v.y;
      rows[2 * ld + t] = v.z;
      rows[3 * ld + t] = v.w;
      if (t < n0) mx.x = fmaxf(mx.x, v.x);
      if (t < n1) mx.y = fmaxf(mx.y, v.y);
      if (t < n2) mx.z = fmaxf(mx.z, v.z);
      mx.w = fmaxf(mx.w, v.w);
    }
    mx = make_float4(wave_max(mx.x), wave_max(mx.y), wave_max(mx.z), wave_max(mx.w));
    if (lane == 0) *(float4*)red[w] = mx;
  }
  __syncthreads();
  mx = *(const float4*)red[0];
#pragma unroll
  for (int i = 1; i < 4; i++) {
    const float4 o = *(const float4*)red[i];
    mx = make_float4(fmaxf(mx.x, o.x), fmaxf(mx.y, o.y), fmaxf(mx.z, o.z), fmaxf(mx.w, o.w));
  }
  float sum = 0.0f;
  for (int c = 0; c <= nc; c++) {
    if (w == 4) {
      // chunk c - 1; zeros past a row's positions leave its non-negative sum as it is
      if (c > 0 && lane < kRows)
        sum = chain_from(rows + lane * ld + (c - 1) * kChunk, min(kChunk, (n3 - (c - 1) * kChunk + 3) & ~3), sum);
    } else if (c < nc) {
      const int t = c * kChunk + tid;  // each thread's own elements: read, and written in place
      rows[t] = t < n0 ? dev_expf(rows[t] - mx.x) : 0.0f;
      rows[ld + t] = t < n1 ? dev_expf(rows[ld + t] - mx.y) : 0.0f;
      rows[2 * ld + t] = t < n2 ? dev_expf(rows[2 * ld + t] - mx.z) : 0.0f;
      rows[3 * ld + t] = t < n3 ? dev_expf(rows[3 * ld + t] - mx.w) : 0.0f;
    }
    __syncthreads();
  }
  if (w == 4 && lane < kRows) invs[lane] = 1.0f / sum;
  __syncthreads();
  if (w < 4) {
    const float4 iv = make_float4(invs[0], invs[1], invs[2], invs[3]);
#pragma unroll 4
    for (int t = tid; t < n3; t += kChunk)
      s4[t] = make_float4(rows[t] * iv.x, rows[ld + t] * iv.y, rows[2 * ld + t] * iv.z, rows[3 * ld + t] * iv.w);
  }
}

// Four waves: four tiles of 64-wide heads, or two of 128-wide ones in halves.
template <int HD>
__global__ __launch_bounds__(256) void pf_values_kernel(PfArgs a) {
  constexpr int DG = HD / 64, TW = 4 / DG, LD = HD + 4;
  constexpr int NP = kVT * (HD / 8) / 256;  // 16-byte value pieces per thread and chunk
  __shared__ __align__(16) float vs[2][kVT * LD];
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ng = (a.nrbc + TW - 1) / TW;
  const int g = (int)blockIdx.x % a.nkv, wt = ng - 1 - (int)blockIdx.x / a.nkv;  // the longest rows first
  const int rbl = wt * TW + w / DG, rbc = min(rbl, a.nrbc - 1), rb = a.rb0 + rbc;
  const int d = (w % DG) * 64 + lane;
  const int nwg = row_n(a, a.rb0 + min(wt * TW + TW - 1, a.nrbc - 1), kRows - 1);
  const int nmin = row_n(a, rb, 0), nmax = row_n(a, rb, kRows - 1);
  const int4 nr = make_int4(nmin, row_n(a, rb, 1), row_n(a, rb, 2), nmax);
  const float* __restrict__ p = a.s + ((size_t)g * a.nrbc + rbc) * a.n64 * kRows;
  const uint16_t* vb = a.vc + ((size_t)a.layer * a.nkv + g) * HD * a.ctx;
  uint4 pr[NP];
  auto load = [&](int c) {
#pragma unroll
    for (int j = 0; j < NP; j++) {
      const int i = tid + 256 * j, t = min(c * kVT + i % kVT, a.ctx - 1);
      pr[j] = *(const uint4*)(vb + ((size_t)(i / kVT) * a.ctx + t) * 8);
    }
  };
  auto store = [&](int b) {
#pragma unroll
    for (int j = 0; j < NP; j++) {
      const int i = tid + 256 * j;
      float4* dst = (float4*)(vs[b] + (i % kVT) * LD + (i / kVT) * 8);
      dst[0] = make_float4(f16_bits_to_f32(pr[j].x & 0xffffu), f16_bits_to_f32(pr[j].x >> 16),
                           f16_bits_to_f32(pr[j].y & 0xffffu), f16_bits_to_f32(pr[j].y >> 16));
      dst[1] = make_float4(f16_bits_to_f32(pr[j].z & 0xffffu), f16_bits_to_f32(pr[j].z >> 16),
                           f16_bits_to_f32(pr[j].w & 0xffffu), f16_bits_to_f32(pr[j].w >> 16));
    }
  };
  float acc[kRows];
#pragma unroll
  for (int r = 0; r < kRows; r++) acc[r] = 0.0f;
  const int nc = (nwg + kVT - 1) / kVT;
  load(0);
  store(0);
  __syncthreads();
  for (int c = 0; c < nc; c++) {
    if (c + 1 < nc) load(c + 1);
    // the weights two chunks ahead, towards this XCD's L2: the scalar loads
    // below cannot be issued that early
    const float2 ahead = ((const float2*)p)[min((c + 2) * (kVT * kRows / 2), a.n64 * kRows / 2 - 64) + lane];
    const float* v = vs[c & 1] + d;
#pragma unroll
    for (int t = 0; t < kVT; t += kBatch) {
      const int tg = c * kVT + t;
      if (tg >= nmax) break;
      float x[kBatch];
#pragma unroll
      for (int i = 0; i < kBatch; i++) x[i] = v[(t + i) * LD];
      if (tg + kBatch <= nmin) scalar_batch<false>(p + tg * kRows, x, acc, nr);
      else scalar_batch<true>(p + tg * kRows, x, acc, make_int4(nr.x - tg, nr.y - tg, nr.z - tg, nr.w - tg));
    }
    asm volatile("" : : "v"(ahead.x), "v"(ahead.y));
    if (c + 1 < nc) store((c + 1) & 1);
    __syncthreads();
  }
  const int nrow = a.tokens * a.gqa, nh = a.gqa * a.nkv;
#pragma unroll
  for (int r = 0; r < kRows; r++) {
    const int i = rb * kRows + r;
    if (rbl >= a.nrbc || i >= nrow) continue;
    const size_t o = ((size_t)(i / a.gqa) * nh + g * a.gqa + i % a.gqa) * HD + d;
    a.out[o] = acc[r];
    if (a.out_q8) {
      uint32_t d_bits;
      const int qv = q8_0_lane(acc[r], &d_bits);
      uint8_t* blk = a.out_q8 + (o >> 5) * kQ8_0Bytes;
      blk[2 + (lane & 31)] = (uint8_t)(int8_t)qv;
      if ((lane & 31) == 0) {
        blk[0] = (uint8_t)(d_bits & 0xff);
        blk[1] = (uint8_t)(d_bits >> 8);
      }
    }
  }
  if (!a.out_q8k) return;
  // Q8_K blocks (kquant.rs:157-187) of 256 / HD neighbouring heads, one per
  // half-wave (the launch checks that a block stays inside a token's KV group)
  constexpr int RB = 256 / HD;
  float* ob = vs[0];  // [TW * kRows][HD]; the last chunk was consumed before the barrier
#pragma unroll
  for (int r = 0; r < kRows; r++) ob[((w / DG) * kRows + r) * HD + d] = acc[r];
  __syncthreads();
  const int hw = tid >> 5, l = tid & 31;
  if (hw >= TW * kRows / RB) return;
  const int lr = hw * RB, i = a.rb0 * kRows + wt * TW * kRows + lr;
  const float4* o4 = (const float4*)(ob + lr * HD);
  const float4 v0 = o4[2 * l], v1 = o4[2 * l + 1];
  const float v8[8] = {v0.x, v0.y, v0.z, v0.w, v1.x, v1.y, v1.z, v1.w};
  uint32_t lo, hi, d_bits;
  int ps;
  q8k_half_lanes(v8, l, &lo, &hi, &ps, &d_bits);
  if (i < nrow && i < (a.rb0 + a.nrbc) * kRows)
    q8k_half_store(a.out_q8k + (((size_t)(i / a.gqa) * nh + g * a.gqa + i % a.gqa) * HD / 256) * kQ8KBytes, l, lo, hi,
                   ps, d_bits);
}

template <int HD>
int launch_hd(const PfAttnLaunch& L, PfArgs a) {
  constexpr int DG = HD / 64, TW = 4 / DG;
  hipStream_t st = (hipStream_t)L.stream;
  // tiles per pass: as many as the weights' scratch holds
  const size_t tile = (size_t)L.n_kv * a.n64 * kRows * 4;
  const int per = (int)std::min<size_t>(L.scratch_bytes / tile, (size_t)a.nrb);
  if (per < 1) return NRQ_LAUNCH_TOO_WIDE;
  for (int rb0 = 0; rb0 < a.nrb; rb0 += per) {
    a.rb0 = rb0;
    a.nrbc = std::min(per, a.nrb - rb0);
    const int nmax = a.base + std::min(((rb0 + a.nrbc) * kRows - 1) / a.gqa, a.tokens - 1) + 1;
    // tiles per wave: the key conversion is spread over more rows, the chip needs the waves
    a.group = 8;
    while (a.group > 1 && (long long)L.n_kv * a.nrbc * ((nmax + 63) / 64) < 8192LL * a.group) a.group /= 2;
    hipLaunchKernelGGL(pf_scores_kernel<HD>,
                       dim3(L.n_kv * ((a.nrbc + a.group - 1) / a.group), (nmax + 255) / 256), dim3(256), 0, st, a, L.qt,
                       L.scratch);
    hipLaunchKernelGGL(pf_softmax_kernel, dim3(L.n_kv * a.nrbc), dim3(320), kRows * softmax_row(nmax) * 4, st, a);
    hipLaunchKernelGGL(pf_values_kernel<HD>, dim3(L.n_kv * ((a.nrbc + TW - 1) / TW)), dim3(256), 0, st, a);
  }
  return hipGetLastError() == hipSuccess ? NRQ_LAUNCH_OK : NRQ_LAUNCH_FAILED;
}

}  // namespace

int launch_pf_attention(const PfAttnLaunch& L) {
  const int gqa = L.n_heads / L.n_kv;
  if (L.head_dim != 64 && L.head_dim != 128) return NRQ_LAUNCH_BAD_ARG;
  if (L.out_q8k && (gqa * L.head_dim) % 256) return NRQ_LAUNCH_BAD_ARG;
  PfArgs a{};
  a.kc = L.kc;
  a.vc = L.vc;
  a.s = L.scratch;
  a.out = L.out;
  a.out_q8 = L.out_q8;
  a.out_q8k = L.out_q8k;
  a.gqa = gqa;
  a.nkv = L.n_kv;
  a.ctx = L.ctx;
  a.layer = L.layer;
  a.base = L.base;
  a.tokens = L.tokens;
  a.nrb = pf_tiles(L.tokens, gqa);
  a.n64 = (L.base + L.tokens + 63) & ~63;
  a.scale = L.scale;
  return L.head_dim == 64 ? launch_hd<64>(L, a) : launch_hd<128>(L, a);
}

}  // namespace nrq
