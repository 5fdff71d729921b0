// AWQ W4A16 linear for the M = 1 (or few-token) modulation layers: bf16
// activations times group-64 asymmetric uint4 weights.
//
// Weight layout (the reference's packed-resident buffers,
// models/svdq_awq_packed.py:181-196 and :240-243): weight uint8 [N, K/2],
// code of column 2j in the LOW nibble of byte j, codes 0..15; wscales and
// wzeros bf16 [N, K/64] (zeros pre-scaled and pre-negated on disk, so the
// dequantized weight is an ADD: w = code * s + z).
//
// Arithmetic = the reference's (models/svdq_awq_packed.py:70-93, and the
// decode path models/svdq_awq.py:74-82): w = RN_bf16(code * s + z) with the
// product exact in fp32 (4-bit code times 8-bit significand) and the sum
// rounded once in fp32, so one fma gives the same value as the reference's
// multiply-then-add; y[m, n] = sum_k w[n, k] * x[m, k] in fp32, + bias in
// fp32, rounded to bf16.
//
// The layer is bound by the weight read (N * K / 2 bytes + the two scale
// grids) and by dequantizing it. The GEMV (up to 4 activation rows) reads every
// weight byte once per MT activation rows; the MFMA kernel (more) once per 16.
// GEMV:
//  * a workgroup stages MT activation rows in LDS (bf16) and owns 16 output
//    rows, one per 16-lane team; lane t of a team takes the 32 codes
//    [512 s + 32 t, +32) of span s (16 weight bytes, one coalesced 256-byte
//    segment per team and span: half a group) and that group's scale and zero;
//  * each 8 codes become four bf16 pairs (nibble split, byte-to-float
//    conversion, one fma each, one v_cvt_pk_bf16_f32 per pair) and each pair
//    meets the matching activation pair in one v_dot2c_f32_bf16 per
//    activation row (fp32 accumulation), the activations read as 16 bytes
//    per lane from LDS, swizzled so the 16 lanes of a team hit distinct banks;
//  * the activations are requested before the weights, so that staging them
//    waits for them alone, and every span of a row of up to 6144 inputs is
//    requested at once (longer rows: batches of 4 spans, two in flight); the
//    team's 16 partial sums are reduced by lane exchanges, and lane 0 adds the
//    bias and stores the bf16 result.
// A second kernel dequantizes the whole weight to bf16 [N, K] (the same
// values) for callers with many activation rows, which then run a library
// GEMM.
#include "gwa_common.h"

namespace {

constexpr int AWQ_THREADS = 256, AWQ_TEAMS = AWQ_THREADS / 16;  // 16 output rows per workgroup
constexpr int AWQ_SPAN = 512;                                    // codes of a row per team step (16 lanes x 32)
constexpr int AWQ_BATCH = 4;                                     // spans per load batch of a long row
constexpr int AWQ_ALL = 12;                                      // rows of up to this many spans load at once
constexpr int AWQ_MFMA_SPAN = 128;                                // codes of a row per wave step of the MFMA kernel
constexpr int AWQ_LDS_MAX = 64 * 1024;                           // activation rows staged in LDS

typedef __bf16 v2bf __attribute__((ext_vector_type(2)));

// eight codes (one dword: code 2b in the low nibble of byte b) of one group -> four bf16 pairs (w_2b, w_2b+1)
__device__ __forceinline__ void dequant8(uint32_t d, float s, float z, uint32_t (&w)[4]) {
  uint32_t lo = d & 0x0F0F0F0Fu, hi = (d >> 4) & 0x0F0F0F0Fu;
  // (float)(byte b) compiles to one v_cvt_f32_ubyte<b> (the empty asm hides the nibble masks, which would
  // otherwise turn each byte into a 4-bit field extract plus a conversion)
  asm("" : "+v"(lo), "+v"(hi));
  const float l0 = (float)(lo & 0xFFu), h0 = (float)(hi & 0xFFu);
  const float l1 = (float)((lo >> 8) & 0xFFu), h1 = (float)((hi >> 8) & 0xFFu);
  const float l2 = (float)((lo >> 16) & 0xFFu), h2 = (float)((hi >> 16) & 0xFFu);
  const float l3 = (float)(lo >> 24), h3 = (float)(hi >> 24);
  w[0] = pack_bf16x2_rn(fmaf(l0, s, z), fmaf(h0, s, z));
  w[1] = pack_bf16x2_rn(fmaf(l1, s, z), fmaf(h1, s, z));
  w[2] = pack_bf16x2_rn(fmaf(l2, s, z), fmaf(h2, s, z));
  w[3] = pack_bf16x2_rn(fmaf(l3, s, z), fmaf(h3, s, z));
}

__device__ __forceinline__ float dot2_bf16(uint32_t a, uint32_t b, float c) {
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(v2bf, a), __builtin_bit_cast(v2bf, b), c, false);
}

// 16-byte unit u of a staged activation row lives at unit u ^ ((u >> 4) & 3): the four 16-byte reads
// of a lane's 64 bytes (units 4t + i of a span, lanes t = 0..15) then hit 16 distinct bank groups
__device__ __forceinline__ int x_unit(int u) { return u ^ ((u >> 4) & 3); }

// a barrier for the LDS writes alone: loads stay in flight
__device__ __forceinline__ void barrier_staged() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(15 | (3 << 14) | (7 << 4));  // lgkmcnt(0)
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// B spans per load batch; PIPED: rows of more than B spans, two batches in flight. Loads return in order: with the
// weights requested first (as this kernel did) no dot product began before the last of them had arrived, and one
// token at 3072 -> 18432 took the launch and staging (3.9 us), the loads (3.5) and the arithmetic (4.5) one after
// the other. us, before -> now: 3072 -> 18432, 1 row 11.8 -> 9.7, 2 13.7 -> 11.8, 4 17.8 -> 15.8; 12288 -> 3072, 1 row
// 14.1 -> 10.4; 15360 -> 18432, 4 rows 117 -> 94. What is left at one row: 3.9 us of launch and staging, 3.5 of loads
// and 4.5 of arithmetic, now partly over one another.
template <int MT, int B, bool PIPED, int XU>
__global__ __launch_bounds__(AWQ_THREADS) void awq_w4a16_gemv_kernel(
    const uint16_t* __restrict__ x, int64_t ldx, const uint8_t* __restrict__ weight,
    const uint16_t* __restrict__ wscales, const uint16_t* __restrict__ wzeros, const uint16_t* __restrict__ bias,
    uint16_t* __restrict__ out, int M, int N, int K) {
  extern __shared__ __attribute__((aligned(16))) uint8_t awq_lds[];
  const int tid = threadIdx.x;
  const int m0 = blockIdx.y * MT;
  const int ku = K >> 3;  // 16-byte units of one activation row

  // team (16 lanes) -> output row n; lane t -> codes [512 s + 32 t, +32) of every span s (half a group)
  const int team = tid >> 4, t = tid & 15;
  const int n = blockIdx.x * AWQ_TEAMS + team;
  const bool row_ok = n < N;
  const int spans = (K + AWQ_SPAN - 1) / AWQ_SPAN, ng = K >> 6;
  const rsrc_t xbuf = make_rsrc(x, (uint32_t)(((int64_t)(M - 1) * ldx + K) * 2));
  const rsrc_t wbuf = make_rsrc(weight, (uint32_t)((int64_t)N * (K >> 1)));
  const rsrc_t sbuf = make_rsrc(wscales, (uint32_t)((int64_t)N * ng * 2));
  const rsrc_t zbuf = make_rsrc(wzeros, (uint32_t)((int64_t)N * ng * 2));
  const uint32_t wrow = (uint32_t)((int64_t)n * (K >> 1)) + 16u * (uint32_t)t;
  const uint32_t grow = (uint32_t)((int64_t)n * ng + (t >> 1)) * 2u;

  // 1. the MT activation rows (rows past M: zeros): the first XU units of each thread into registers, ahead of the
  //    weights (launch_gemv: all of them, as far as registers go)
  auto x_load = [&](int u) __attribute__((always_inline)) {
    const int r = u / ku, c = u - r * ku;
    return buf_load16(xbuf, u < MT * ku && m0 + r < M ? (uint32_t)(((int64_t)(m0 + r) * ldx + 8 * c) * 2) : kOOB);
  };
  auto x_store = [&](int u, v4i v) __attribute__((always_inline)) {
    const int r = u / ku, c = u - r * ku;
    if (u < MT * ku) *(v4i*)(awq_lds + 16 * (r * ku + x_unit(c))) = v;
  };
  v4i xr[XU];
#pragma unroll
  for (int i = 0; i < XU; ++i) xr[i] = x_load(tid + i * AWQ_THREADS);

  // 2. the first batch of weights, scales and zeros
  struct Batch {
    v4i wd[B];
    uint16_t sc[B], ze[B];
  };
  auto load_batch = [&](Batch& bt, int s0) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < B; ++j) {
      const bool ok = row_ok && (s0 + j) * AWQ_SPAN + 32 * t < K;
      bt.sc[j] = buf_load2(sbuf, ok ? grow + 16u * (uint32_t)(s0 + j) : kOOB);
      bt.ze[j] = buf_load2(zbuf, ok ? grow + 16u * (uint32_t)(s0 + j) : kOOB);
      bt.wd[j] = buf_load16(wbuf, ok ? wrow + (uint32_t)(AWQ_SPAN / 2) * (uint32_t)(s0 + j) : kOOB);
    }
  };
  Batch cur;
  load_batch(cur, 0);

  // 3. the activations into LDS, units swizzled by x_unit
#pragma unroll
  for (int i = 0; i < XU; ++i) x_store(tid + i * AWQ_THREADS, xr[i]);
  for (int u = tid + XU * AWQ_THREADS; u < MT * ku; u += AWQ_THREADS) x_store(u, x_load(u));
  barrier_staged();

  // 4. batches of spans: dequantize 32 codes, dot them with every activation row
  float acc[MT];
#pragma unroll
  for (int r = 0; r < MT; ++r) acc[r] = 0.0f;
  auto use_batch = [&](const Batch& bt, int s0) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < B; ++j) {
      if ((s0 + j) * AWQ_SPAN + 32 * t >= K) continue;  // past the row (K % 512 != 0, or fewer spans)
      const float sv = bf16_to_f32(bt.sc[j]), zv = bf16_to_f32(bt.ze[j]);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        uint32_t w[4];
        dequant8((uint32_t)bt.wd[j][q], sv, zv, w);
        const int unit = x_unit(64 * (s0 + j) + 4 * t + q);  // activation columns 512 s + 32 t + 8 q .. +8
#pragma unroll
        for (int r = 0; r < MT; ++r) {
          const v4i xv = *(const v4i*)(awq_lds + 16 * (r * ku + unit));
#pragma unroll
          for (int b = 0; b < 4; ++b) acc[r] = dot2_bf16(w[b], (uint32_t)xv[b], acc[r]);
        }
      }
    }
  };
  if (PIPED) {
    Batch nxt;
    for (int s0 = 0; s0 < spans; s0 += 2 * B) {
      load_batch(nxt, s0 + B);  // past the row: no lane loads
      use_batch(cur, s0);
      load_batch(cur, s0 + 2 * B);
      use_batch(nxt, s0 + B);
    }
  } else {
    use_batch(cur, 0);
  }
  // 5. team sum (lanes t ^ 8, 4, 2, 1), bias, bf16
  const float bv = (bias && row_ok) ? bf16_to_f32(bias[n]) : 0.0f;
#pragma unroll
  for (int r = 0; r < MT; ++r) {
    float v = acc[r];
    v += __shfl_xor(v, 8, 16);
    v += __shfl_xor(v, 4, 16);
    v += __shfl_xor(v, 2, 16);
    v += __shfl_xor(v, 1, 16);
    if (t == 0 && row_ok && m0 + r < M) out[(int64_t)(m0 + r) * N + n] = f32_to_bf16(v + bv);
  }
}

// More than 4 activation rows: one read of the weight for up to 16 of them, on 16x16x32 MFMA (weights the first operand,
// activation rows the second: a lane holds 8 consecutive inputs of one row). The GEMV above reads and dequantizes the
// weight once per 4 rows and spends 4 dot products per 8 codes on each row; here dequantizing (the arithmetic that
// bounds it at few rows) is done once and the products are one instruction per 8 codes of a lane. A workgroup owns 16
// output rows, its W waves take every W-th span of 128 inputs, and their sums meet in LDS; activations come straight
// from memory (staged in LDS they would cost a barrier before the first product and the occupancy that hides the
// loads: 8 waves per SIMD, no load batches, is the fastest; batches of 2, 3 and 6 spans in flight took 16-18 us at 3072 ->
// 9216 and 5 rows, 32 and 64 output rows per workgroup 12.9 and 14.1, this 11.5).
// us, GEMV -> this: 3072 -> 18432 5 rows 25.4 -> 17.9, 16 rows 45 -> 25; 3072 -> 3072 16 rows 11.6 -> 6.4; 12288 ->
// 3072 16 rows 47.6 -> 20.6.
template <int W>
__global__ __launch_bounds__(64 * W) void awq_w4a16_mfma_kernel(
    const uint16_t* __restrict__ x, int64_t ldx, const uint8_t* __restrict__ weight,
    const uint16_t* __restrict__ wscales, const uint16_t* __restrict__ wzeros, const uint16_t* __restrict__ bias,
    uint16_t* __restrict__ out, int M, int N, int K) {
  __shared__ __attribute__((aligned(16))) float part[W][256];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int l16 = lane & 15, g = lane >> 4;
  const int n0 = blockIdx.x * 16, m0 = blockIdx.y * 16, ng = K >> 6;
  const rsrc_t xbuf = make_rsrc(x, (uint32_t)(((int64_t)(M - 1) * ldx + K) * 2));
  const rsrc_t wbuf = make_rsrc(weight, (uint32_t)((int64_t)N * (K >> 1)));
  const rsrc_t sbuf = make_rsrc(wscales, (uint32_t)((int64_t)N * ng * 2));
  const rsrc_t zbuf = make_rsrc(wzeros, (uint32_t)((int64_t)N * ng * 2));
  const uint32_t xoff = (uint32_t)(((int64_t)(m0 + l16) * ldx + 32 * g) * 2);
  const uint32_t woff = (uint32_t)((int64_t)(n0 + l16) * (K >> 1) + 16 * g);
  const uint32_t soff = (uint32_t)(((int64_t)(n0 + l16) * ng + (g >> 1)) * 2);

  v4f acc = {0.0f, 0.0f, 0.0f, 0.0f};
  for (int s = wave; s < K / AWQ_MFMA_SPAN; s += W) {
    const float sv = bf16_to_f32(buf_load2(sbuf, soff + 4u * (uint32_t)s));
    const float zv = bf16_to_f32(buf_load2(zbuf, soff + 4u * (uint32_t)s));
    const v4i wd = buf_load16(wbuf, woff + (uint32_t)(AWQ_MFMA_SPAN / 2) * (uint32_t)s);
    v4i xv[4];
#pragma unroll
    for (int q = 0; q < 4; ++q)
      xv[q] = buf_load16(xbuf, m0 + l16 < M ? xoff + (uint32_t)(2 * AWQ_MFMA_SPAN) * (uint32_t)s + 16u * q : kOOB);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      uint32_t w[4];
      dequant8((uint32_t)wd[q], sv, zv, w);
      const v4i wv = {(int)w[0], (int)w[1], (int)w[2], (int)w[3]};
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, wv), __builtin_bit_cast(v8bf, xv[q]), acc,
                                                    0, 0, 0);
    }
  }
  // the block (row 4 g + i, activation row l16) of this wave at [16 l16 + row]; the waves' sums, bias, bf16
  *(v4f*)&part[wave][16 * l16 + 4 * g] = acc;
  __syncthreads();
  const int m = m0 + (tid >> 4), n = n0 + (tid & 15);
  if (tid >= 256 || m >= M) return;
  float v = part[0][tid];
#pragma unroll
  for (int w = 1; w < W; ++w) v += part[w][tid];
  out[(int64_t)m * N + n] = f32_to_bf16(v + (bias ? bf16_to_f32(bias[n]) : 0.0f));
}

// weight [N, K/2] + scales / zeros [N, K/64] -> bf16 [N, K]: one dword of codes (8 columns) per thread
__global__ __launch_bounds__(256) void awq_w4a16_dequant_kernel(const uint32_t* __restrict__ weight,
                                                                 const uint16_t* __restrict__ wscales,
                                                                 const uint16_t* __restrict__ wzeros,
                                                                 uint16_t* __restrict__ out, int64_t N, int K) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;  // dword index
  const int per_row = K >> 3;
  if (i >= N * per_row) return;
  const int64_t n = i / per_row;
  const int c = (int)(i - n * per_row);
  const int64_t g = n * (K >> 6) + (c >> 3);
  uint32_t w[4];
  dequant8(weight[i], bf16_to_f32(wscales[g]), bf16_to_f32(wzeros[g]), w);
  *(v4i*)(out + 8 * i) = (v4i){(int)w[0], (int)w[1], (int)w[2], (int)w[3]};
}

// Rows of up to AWQ_ALL spans load whole (several batch sizes, so that a row does not issue loads for many spans it does
// not have: two rows 4224 -> 3072 pipelined 8.3 us, 12 spans at once 7.5, 10 7.4; 6144 -> 3072 9.6 and 8.9; 16 at once
// for 8192 11.4, pipelined 10.8). Units of activations ahead of the weights: all of a thread's, which is a whole row
// of up to 16384 in 8 (with 2 ahead 12288 -> 3072 took 11.4 us for 10.4; chunks of two rows with 4, 15360 -> 512 18.8
// for 17.6, with 8 18.1), but no more than there are (two rows 8192 -> 3072 with 16 11.1, with their 8 10.8).
template <int MT>
int launch_gemv(const void* x, int64_t ldx, const void* weight, const void* ws, const void* wz, const void* bias,
                void* out, int64_t M, int64_t N, int64_t K, hipStream_t st) {
  const size_t lds = (size_t)MT * (size_t)K * 2;
  const int64_t spans = (K + AWQ_SPAN - 1) / AWQ_SPAN;
  const dim3 grid((unsigned)((N + AWQ_TEAMS - 1) / AWQ_TEAMS), (unsigned)((M + MT - 1) / MT));
  auto go = [&](auto kern) {
    hipLaunchKernelGGL(kern, grid, dim3(AWQ_THREADS), lds, st, (const uint16_t*)x, ldx, (const uint8_t*)weight,
                       (const uint16_t*)ws, (const uint16_t*)wz, (const uint16_t*)bias, (uint16_t*)out, (int)M, (int)N,
                       (int)K);
  };
#define GWA_AWQ_WHOLE(B) go(awq_w4a16_gemv_kernel<MT, B, false, (MT * B + 3) / 4>)
  if (spans > AWQ_ALL) {
    if constexpr (MT == 1) go(awq_w4a16_gemv_kernel<1, AWQ_BATCH, true, 8>);
    else if (MT == 2 && K <= 8192) go(awq_w4a16_gemv_kernel<2, AWQ_BATCH, true, 8>);
    else go(awq_w4a16_gemv_kernel<MT, AWQ_BATCH, true, 16>);
  } else if (spans > 10) GWA_AWQ_WHOLE(AWQ_ALL);
  else if (spans > 8) GWA_AWQ_WHOLE(10);
  else if (spans > 6) GWA_AWQ_WHOLE(8);
  else if (spans > 4) GWA_AWQ_WHOLE(6);
  else if (spans > 2) GWA_AWQ_WHOLE(4);
  else GWA_AWQ_WHOLE(2);
#undef GWA_AWQ_WHOLE
  return gwa_check_launch("awq_w4a16_mm");
}

template <int W>
int launch_mfma(const void* x, int64_t ldx, const void* weight, const void* ws, const void* wz, const void* bias,
                void* out, int64_t M, int64_t N, int64_t K, hipStream_t st) {
  const dim3 grid((unsigned)(N / 16), (unsigned)((M + 15) / 16));
  hipLaunchKernelGGL((awq_w4a16_mfma_kernel<W>), grid, dim3(64 * W), 0, st, (const uint16_t*)x, ldx,
                     (const uint8_t*)weight, (const uint16_t*)ws, (const uint16_t*)wz, (const uint16_t*)bias,
                     (uint16_t*)out, (int)M, (int)N, (int)K);
  return gwa_check_launch("awq_w4a16_mm");
}

}  // namespace

extern "C" int gwa_awq_w4a16_mm(const void* x, int64_t ldx, const void* weight, const void* wscales,
                                const void* wzeros, const void* bias, void* out, int64_t M, int64_t N, int64_t K,
                                void* stream) {
  const char* what = "awq_w4a16_mm";
  GWA_REQUIRE(M >= 0 && N > 0 && K > 0 && N % 16 == 0 && K % 128 == 0,
              "%s: [N=%lld, K=%lld] breaks the packed contract (N %% 16, K %% 128)", what, (long long)N,
              (long long)K);
  GWA_REQUIRE(ldx >= K && ldx % 8 == 0, "%s: row stride %lld must be >= K and a multiple of 8", what,
              (long long)ldx);
  GWA_REQUIRE(K * 2 <= AWQ_LDS_MAX, "%s: K=%lld exceeds %d (one activation row staged in LDS)", what,
              (long long)K, AWQ_LDS_MAX / 2);
  GWA_REQUIRE(M < (1ll << 31) && N * K / 2 < (1ll << 31) && M * ldx * 2 < (1ll << 31) && M * N < (1ll << 31),
              "%s: operands must stay below 2 GiB (buffer addressing)", what);
  if (M == 0) return GWA_OK;
  GWA_REQUIRE(x && weight && wscales && wzeros && out, "%s: null pointer", what);
  GWA_REQUIRE(GWA_ALIGNED(x, 16) && GWA_ALIGNED(weight, 4) && GWA_ALIGNED(wscales, 2) && GWA_ALIGNED(wzeros, 2) &&
                  GWA_ALIGNED(bias, 2) && GWA_ALIGNED(out, 2),
              "%s: x must be 16-byte and weight 4-byte aligned", what);
  hipStream_t st = (hipStream_t)stream;
  // MFMA from 5 rows on (up to 4 the GEMV reads the weight once too, in whole 256-byte row segments: 5 rows at 3072 ->
  // 18432 25.4 -> 17.9 us, 4 rows 15.8 -> 17.9), except long rows on few output rows: there the GEMV's chunks of rows
  // are the parallelism (15360 -> 512, 16 rows: GEMV 17.7, MFMA 24.6; 15360 -> 1024 26 and 24.9; 8192 -> 512 16.3
  // and 13.9). 8 waves per workgroup for rows past 4096 inputs (15360 -> 2048, 16 rows: 4 waves 32.4, 8 25.0),
  // 4 otherwise (3072 -> 18432, 5 rows: 17.9 and 19.5).
  if (M > 4 && (N >= 1024 || K <= 8192)) {
    if (K > 4096) return launch_mfma<8>(x, ldx, weight, wscales, wzeros, bias, out, M, N, K, st);
    return launch_mfma<4>(x, ldx, weight, wscales, wzeros, bias, out, M, N, K, st);
  }
  // GEMV, activation rows per workgroup: up to 4, as many as fit the LDS budget
  int mt = M == 1 ? 1 : (M == 2 ? 2 : 4);
  while (mt > 1 && (int64_t)mt * K * 2 > AWQ_LDS_MAX) mt /= 2;
  if (mt == 1) return launch_gemv<1>(x, ldx, weight, wscales, wzeros, bias, out, M, N, K, st);
  if (mt == 2) return launch_gemv<2>(x, ldx, weight, wscales, wzeros, bias, out, M, N, K, st);
  return launch_gemv<4>(x, ldx, weight, wscales, wzeros, bias, out, M, N, K, st);
}

extern "C" int gwa_awq_w4a16_dequant(const void* weight, const void* wscales, const void* wzeros, void* out,
                                     int64_t N, int64_t K, void* stream) {
  const char* what = "awq_w4a16_dequant";
  GWA_REQUIRE(N > 0 && K > 0 && K % 64 == 0 && N * K < (1ll << 40), "%s: bad shape [N=%lld, K=%lld]", what,
              (long long)N, (long long)K);
  GWA_REQUIRE(weight && wscales && wzeros && out, "%s: null pointer", what);
  GWA_REQUIRE(GWA_ALIGNED(weight, 4) && GWA_ALIGNED(wscales, 2) && GWA_ALIGNED(wzeros, 2) && GWA_ALIGNED(out, 16),
              "%s: weight must be 4-byte and out 16-byte aligned", what);
  const int64_t dwords = N * (K / 8);
  hipLaunchKernelGGL(awq_w4a16_dequant_kernel, dim3((unsigned)((dwords + 255) / 256)), dim3(256), 0,
                     (hipStream_t)stream, (const uint32_t*)weight, (const uint16_t*)wscales,
                     (const uint16_t*)wzeros, (uint16_t*)out, N, (int)K);
  return gwa_check_launch(what);
}
