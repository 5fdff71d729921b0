// W8A8 GEMM: int8 MFMA with int32 accumulation over the whole K and
// the fp32 epilogue acc * sa * sw[n] + bias[n] of torch._scaled_mm: per-token
// activation scales in the rowwise mode (models/w8a8.py:374-378), one scalar in
// the pertensor mode (:366-372, whose weight scale and bias the reference
// applies as two further bf16 ops; here they are fused in fp32).
//
// Same orientation as the W4A4 kernel: A operand = weight rows (n), B operand
// = activation rows (m); lane l of a 16 x 16 accumulator block D[n][m] holds
// m = l % 16 and n = 4*(l/16) + v.
#include <atomic>

#include "fp6_gemm_common.h"

namespace {

// s_waitcnt lgkmcnt(0), vmcnt and expcnt left at their maxima
__device__ __forceinline__ void wait_lgkm0() { __builtin_amdgcn_s_waitcnt(15 | (3 << 14) | (7 << 4)); }

template <int BIAS_DT>
__device__ __forceinline__ float bias_at(const void* bias, int n) {
  if (BIAS_DT == GWA_DT_F32) return ((const float*)bias)[n];
  if (BIAS_DT == GWA_DT_BF16) return bf16_to_f32(((const uint16_t*)bias)[n]);
  if (BIAS_DT == GWA_DT_F16) return f16_bits_to_f32(((const uint16_t*)bias)[n]);
  return 0.0f;
}

// LDS slot of 16-byte chunk c of operand row r: c ^ l_swz(r), so the 16 rows a quarter of a read instruction
// touches fill all banks
__device__ __forceinline__ int l_swz(int r) { return (r >> 1) & 7; }

// Direct-to-LDS copy of 16 bytes per lane at 64-bit lane addresses: LDS [lds_addr + 16 lane, +16) <- src. Every
// lane's source must be readable; waits are the kernel's (as for dma16).
__device__ __forceinline__ void dma16_at(uint32_t lds_addr, const uint8_t* src) {
  asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, off" : : "s"(lds_addr), "v"(src) : "memory", "m0");
}

// wait until at most min(newer, most) stages of `copies` copies each are still in flight (and no LDS read)
template <int copies, int most>
__device__ __forceinline__ void wait_newer(int newer) {
  if constexpr (most > 0) {
    if (newer < most) {
      wait_newer<copies, most - 1>(newer);
      return;
    }
  }
  wait_vm_lgkm0<copies * most>();
}

// ---------------------------------------------------------------------------
// TM x TN tiles (64 or 128) for grids that leave CUs idle on 256 x 256 ones, 4 waves as a 2 x 2 grid. What
// bounds them is the serial chain of a stage (wait, barrier, operand reads, MFMAs), not bytes: 64 x 64 tiles
// at K = 12288 take 0.27 us a stage with one workgroup on a CU, and a deeper ring changes nothing (3, 4 and 8
// buffers: 8.5, 9.0 and 9.4 us at 256 x 3072 x 3072). So the stages are copied straight to LDS (the
// register-staged form took 22.3 us there on 128 x 128 tiles), each stage's operands are read one stage ahead under
// the MFMAs (11.4 us without), and the ring is as short as lets several workgroups share a CU and fill each
// other's gaps.
// ---------------------------------------------------------------------------
constexpr int S_KS = 128;  // K bytes per row and stage; K % 128 == 64 ends in half a stage (one k-step)

template <int TM, int TN, int NBUF, int BIAS_DT, bool OUT_F16>
__global__ __launch_bounds__(256) void w8a8_gemm_small_kernel(const int8_t* __restrict__ qa,
                                                              const int8_t* __restrict__ qw,
                                                              const float* __restrict__ sa,
                                                              const float* __restrict__ sw,
                                                              const void* __restrict__ bias,
                                                              uint16_t* __restrict__ out, int M, int N, int K,
                                                              int sa_row) {
  constexpr int STAGE = (TM + TN) * S_KS, COPIES = STAGE / 1024 / 4;  // per wave and stage
  constexpr int BM = TM / 32, BN = TN / 32;                           // 16 x 16 blocks of a wave's half tiles
  constexpr int OSTR = TN * 2 + 16;
  static_assert(TM * OSTR <= NBUF * STAGE, "output staging");
  __shared__ __attribute__((aligned(16))) uint8_t g_lds[NBUF * STAGE];
  __shared__ __attribute__((aligned(16))) float g_epi[2 * TN];
  const int tid = threadIdx.x;
  const int tiles_n = (N + TN - 1) / TN, tiles_m = (M + TM - 1) / TM;
  int tm, tn;
  if (!xcd_tile_of(blockIdx.x, tiles_m, tiles_n, tm, tn)) return;  // whole workgroup, before any barrier
  const int m0 = tm * TM, n0 = tn * TN;
  const int nst = (K + S_KS - 1) / S_KS;
  const bool half = K % S_KS != 0;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int wn = wave & 1, wm = wave >> 1, r16 = lane & 15, q4 = lane >> 4;

  float cs = 0.0f, cb = 0.0f;
  if (tid < TN && n0 + tid < N) {
    cs = sw[n0 + tid];
    cb = bias_at<BIAS_DT>(bias, n0 + tid);
  }
  // copy j of this wave is run q = wave + 4 j of a stage: eight rows, lane -> row 8 q + lane / 8, LDS slot
  // lane % 8; the activation rows first. Rows past M or N re-read the last one (their results are not stored).
  const uint8_t* src[COPIES];
  const int chunk = (lane & 7) ^ l_swz((8 * wave + (lane >> 3)) & 15);
#pragma unroll
  for (int j = 0; j < COPIES; ++j) {
    const int row = 8 * (wave + 4 * j) + (lane >> 3);
    src[j] = 4 * j < TM / 8 ? (const uint8_t*)qa + (int64_t)min(m0 + row, M - 1) * K
                            : (const uint8_t*)qw + (int64_t)min(n0 + row - TM, N - 1) * K;
    src[j] += 16 * chunk;
  }
  const uint32_t ldst = (uint32_t)(uintptr_t)(g_lds + wave * 1024);
  auto issue = [&](int u, int st) __attribute__((always_inline)) {
    // half a stage: the upper chunks (which no k-step reads) come from the lower ones
    const int back = half && st == nst - 1 && chunk >= 4 ? 64 : 0;
    int64_t off = (int64_t)st * S_KS - back;
    if (!GWA_DCHECK(off + 16 * chunk + 16 <= K, kDbgW8Copy, off)) off = 0;
#pragma unroll
    for (int j = 0; j < COPIES; ++j) dma16_at(ldst + (uint32_t)(u * STAGE + j * 4096), src[j] + off);
  };

  v4i acc[BN][BM];
#pragma unroll
  for (int bn = 0; bn < BN; ++bn)
#pragma unroll
    for (int bm = 0; bm < BM; ++bm) acc[bn][bm] = (v4i){};
  uint32_t xoff[2], woff[2];
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) {
    const uint32_t c = 16u * (uint32_t)((4 * ks + q4) ^ l_swz(r16));
    xoff[ks] = (uint32_t)((TM / 2 * wm + r16) * S_KS) + c;
    woff[ks] = (uint32_t)((TM + TN / 2 * wn + r16) * S_KS) + c;
  }

  // the operands of a stage are read one stage ahead into the other register set, under this stage's MFMAs
  v4i a[2][2][BN], b[2][2][BM];
  auto read_ops = [&](int set, int u) __attribute__((always_inline)) {
    const uint8_t* buf = g_lds + u * STAGE;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
#pragma unroll
      for (int bm = 0; bm < BM; ++bm) b[set][ks][bm] = *(const v4i*)(buf + xoff[ks] + bm * 16 * S_KS);
#pragma unroll
      for (int bn = 0; bn < BN; ++bn) a[set][ks][bn] = *(const v4i*)(buf + woff[ks] + bn * 16 * S_KS);
    }
  };
  auto mma = [&](int set, int ks) __attribute__((always_inline)) {
#pragma unroll
    for (int bn = 0; bn < BN; ++bn)
#pragma unroll
      for (int bm = 0; bm < BM; ++bm)
        acc[bn][bm] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[set][ks][bn], b[set][ks][bm], acc[bn][bm], 0, 0, 0);
  };
#pragma unroll
  for (int st = 0; st < NBUF; ++st)
    if (st < nst) issue(st, st);
  wait_newer<COPIES, NBUF - 1>(min(NBUF - 1, nst - 1));
  barrier_lds();
  read_ops(0, 0);
  int u = 0;  // buffer of stage st
  auto stage = [&](int set, int st) __attribute__((always_inline)) {
    const int v = u == NBUF - 1 ? 0 : u + 1;
    if (st + 1 < nst) {
      wait_newer<COPIES, NBUF - 2>(min(NBUF - 2, nst - 2 - st));
      barrier_lds();  // everyone's copies of stage st + 1 are in, and everyone's reads of stage st have ended
      read_ops(set ^ 1, v);
      if (st + NBUF < nst) issue(u, st + NBUF);
      __builtin_amdgcn_sched_barrier(0);
    }
    mma(set, 0);
    if (!(half && st == nst - 1)) mma(set, 1);
    __builtin_amdgcn_sched_barrier(0);
    u = v;
  };
  for (int st = 0; st < nst; st += 2) {
    stage(0, st);
    if (st + 1 < nst) stage(1, st + 1);
  }

  // epilogue: y = acc * sa[m] * sw[n] + bias[n], staged as [m][n] rows and stored as whole row segments
  if (tid < TN) {
    g_epi[tid] = cs;
    g_epi[TN + tid] = cb;
  }
  __syncthreads();
#pragma unroll
  for (int bm = 0; bm < BM; ++bm) {
    const int ml = TM / 2 * wm + 16 * bm + r16;
    const float am = sa[sa_row ? min(m0 + ml, M - 1) : 0];  // rows past M are computed but never stored
#pragma unroll
    for (int bn = 0; bn < BN; ++bn) {
      const int nl = TN / 2 * wn + 16 * bn + 4 * q4;
      const v4f cw = *(const v4f*)(g_epi + nl);
      const v4f cv = *(const v4f*)(g_epi + TN + nl);
      float o[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float y = (float)acc[bn][bm][e] * am * cw[e];
        if (BIAS_DT >= 0) y += cv[e];
        o[e] = y;
      }
      uint2 pk;
      if (OUT_F16) {
        pk.x = pack_f16x2(o[0], o[1]);
        pk.y = pack_f16x2(o[2], o[3]);
      } else {
        pk.x = pack_bf16x2_rn(o[0], o[1]);
        pk.y = pack_bf16x2_rn(o[2], o[3]);
      }
      *(uint2*)(g_lds + ml * OSTR + nl * 2) = pk;
    }
  }
  __syncthreads();
  // a descriptor over this tile's output span (127 N + 128 elements < 2^28: N < 2^21 is checked on the host)
  const int rows = min(M - m0, TM), cols = min(N - n0, TN);
  const uint32_t span = (uint32_t)(((rows - 1) * N + cols) * 2);
  const rsrc_t obuf = make_rsrc(out + (int64_t)m0 * N + n0, span);
  constexpr int CPR = TN / 8;  // 16-byte chunks per row
#pragma unroll
  for (int i = tid; i < TM * CPR; i += 256) {
    const int row = i / CPR, c = i % CPR;
    const v4i v = *(const v4i*)(g_lds + row * OSTR + c * 16);
    uint32_t off = row < rows && 8 * c < cols ? (uint32_t)((row * N + 8 * c) * 2) : kOOB;
    if (!GWA_DCHECK(off == kOOB || (int64_t)off + 16 <= (int64_t)span, kDbgW8Out, off)) off = kOOB;
    buf_store16(v, obuf, off);
  }
}

// ---------------------------------------------------------------------------
// 256 x 256 tiles for grids that fill the GPU. Operand delivery is the W4A4 kernels': direct-to-LDS 1 KB
// copies (no staging registers, no ds_write), here into two stage buffers of 128 K-bytes of 256 activation
// rows and 256 weight rows (64 KB each), the next stage's copies in flight while a stage is consumed. A copy
// reads whole 128-byte lines: lane l of a copy takes 16 bytes of row 8 q + l / 8 (eight rows per copy), so
// rows past M or N read zeros through the range-checked per-lane offset and the stage advance rides in the
// scalar offset. In LDS the 16-byte chunk c of row r sits at slot c ^ ((r / 2) % 8) of the row, so the 16
// rows a quarter of a read instruction touches fill all banks. 8 waves form a 2 (n) x 4 (m) grid of
// 128 x 64 wave tiles: per k-step of 64 bytes, 12 operand reads feed 32 int8 MFMAs.
//
// What bounds it: with operands of full range, power (4096^3 takes 44.1 us on zeros and 52.5 on normal data; the
// clock falls as more of the chip is busy), so the form that moves the fewest register bytes wins; with the
// small codes that outlier channels leave, the matrix pipe (85 % busy in the loop), the epilogue and the last
// round's idle CUs. The 16 x 16 x 64 MFMA reads and writes a quarter of the sums per instruction that
// 32 x 32 x 32 does, for half the multiply-adds: the same loop on it ran 62 -> 56 us at 4096^3, and visiting
// the blocks in a snake, so that neighbouring MFMAs always share an operand, took another 1 %.
//
// The two waves of a SIMD alternate: waves 0..3 run one phase ahead of waves 4..7, and in every phase one
// group issues a k-step's 32 MFMAs (512 matrix-pipe cycles, raised priority) while the other reads its next
// k-step's operands into registers and issues its copies; a barrier ends each phase. Against both waves
// running the same read-under-MFMA pipeline this took 118.6 -> 114.1 us at 4608 x 9216 x 3072. Persistent
// workgroups that prefetch the next tile under the epilogue measured 118 us there (the epilogue's phase runs
// beside one MFMA phase only). In all, against the 32 x 32 x 32 pipeline before it, normal data: 4096^3
// 60.1 -> 52.5 us (2620 TOPS), 4608 x 9216 x 3072 122.1 -> 108.9, 4608 x 3072 x 3072 41.4 -> 38.
// ---------------------------------------------------------------------------
constexpr int L_TM = 256, L_TN = 256, L_KS = 128;  // tile rows (m, n); K bytes per stage
constexpr int kCus = 256;                          // MI355X compute units
constexpr int L_REG = 256 * L_KS;                  // one operand region of a stage buffer: 32 KB
constexpr int L_STAGE = 2 * L_REG;                 // activation region, then weight region
constexpr int L_RUNS = L_REG / 1024;               // 1 KB copies per operand and stage: 32
constexpr int L_SLOTS = L_STAGE / 1024 / NWAVES;   // copies per wave and stage: 8 (4 activation, 4 weight)
constexpr int L_LDS = 2 * L_STAGE;
static_assert(L_LDS <= kLdsBytes && L_SLOTS * NWAVES * 1024 == L_STAGE, "stage layout");
static_assert(NWAVES * 64 * 256 <= L_LDS, "output staging");

template <int BIAS_DT, bool OUT_F16>
__global__ __launch_bounds__(NTHREADS, 1) void w8a8_gemm_lds_kernel(const int8_t* __restrict__ qa,
                                                                    const int8_t* __restrict__ qw,
                                                                    const float* __restrict__ sa,
                                                                    const float* __restrict__ sw,
                                                                    const void* __restrict__ bias,
                                                                    uint16_t* __restrict__ out, int M, int N, int K,
                                                                    int sa_row) {
  __shared__ __attribute__((aligned(16))) uint8_t g_lds[L_LDS];
  __shared__ __attribute__((aligned(16))) float g_epi[2 * L_TN];  // the tile's sw, then its bias as fp32
  const int tid = threadIdx.x;
  const int tiles_n = (N + L_TN - 1) / L_TN, tiles_m = (M + L_TM - 1) / L_TM;
  int tm, tn;
  if (!xcd_tile_of(blockIdx.x, tiles_m, tiles_n, tm, tn)) return;  // whole workgroup, before any barrier
  const int m0 = tm * L_TM, n0 = tn * L_TN;
  const int nst = K / L_KS;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int wn = wave & 1, wm = wave >> 1;
  const int r16 = lane & 15, q4 = lane >> 4;

  // descriptors over this tile's rows only (256 K < 2^31 bytes, checked on the host, so kOOB lies past them)
  const v4i xbuf = raw_rsrc(qa + (int64_t)m0 * K, (uint32_t)(min(M - m0, L_TM) * K));
  const v4i wbuf = raw_rsrc(qw + (int64_t)n0 * K, (uint32_t)(min(N - n0, L_TN) * K));
  // copy j of this wave is run q = wave + 8 j of a stage: runs 0..31 carry activation rows, 32..63 weight
  // rows (j < 4: activations); lane -> row 8 (q % 32) + lane / 8 of the region, LDS slot lane % 8
  uint32_t voff[L_SLOTS];
  uint32_t ldst[L_SLOTS];
#pragma unroll
  for (int j = 0; j < L_SLOTS; ++j) {
    const int q = wave + NWAVES * j;
    const bool isx = j < L_SLOTS / 2;
    const int row = 8 * (q % L_RUNS) + (lane >> 3);
    const int chunk = (lane & 7) ^ l_swz(row);
    const bool live = (isx ? m0 : n0) + row < (isx ? M : N);
    voff[j] = live ? (uint32_t)(row * K + 16 * chunk) : kOOB;
    ldst[j] = (uint32_t)(uintptr_t)(g_lds + (isx ? 0 : L_REG) + (q % L_RUNS) * 1024);
  }
  auto issue = [&](int u, int st) __attribute__((always_inline)) {
    // the stage's K bytes lie inside every operand row (the lane offsets are range-checked by the hardware,
    // the stage's scalar offset is not)
    const uint32_t soff = GWA_DCHECK((st + 1) * L_KS <= K, kDbgW8Copy, st * L_KS) ? (uint32_t)(st * L_KS) : 0u;
#pragma unroll
    for (int j = 0; j < L_SLOTS; ++j)
      dma16(j < L_SLOTS / 2 ? xbuf : wbuf, ldst[j] + (uint32_t)(u * L_STAGE), voff[j], soff);
  };

  v4i acc[8][4], a[8], b[4];
#pragma unroll
  for (int bn = 0; bn < 8; ++bn)
#pragma unroll
    for (int bm = 0; bm < 4; ++bm) acc[bn][bm] = (v4i){};
  // this lane's chunk of an operand row at k-step ks (64 bytes): the rows of a wave differ by multiples of 16, so
  // the chunk swizzle is the lane's own
  uint32_t xoff[2], woff[2];
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) {
    const uint32_t c = 16u * (uint32_t)((4 * ks + q4) ^ l_swz(r16));
    xoff[ks] = (uint32_t)((64 * wm + r16) * L_KS) + c;
    woff[ks] = (uint32_t)(L_REG + (128 * wn + r16) * L_KS) + c;
  }
  auto read_ops = [&](const uint8_t* buf, int ks) __attribute__((always_inline)) {
#pragma unroll
    for (int bm = 0; bm < 4; ++bm) b[bm] = *(const v4i*)(buf + xoff[ks] + bm * 16 * L_KS);
#pragma unroll
    for (int bn = 0; bn < 8; ++bn) a[bn] = *(const v4i*)(buf + woff[ks] + bn * 16 * L_KS);
  };
  // one k-step; empty asm on its operands and sums keeps the (pure) MFMAs between the phase's two barriers
  auto mma = [&]() __attribute__((always_inline)) {
    asm volatile("" : "+v"(a[0]), "+v"(a[1]), "+v"(a[2]), "+v"(a[3]), "+v"(b[0]), "+v"(b[1]));
    asm volatile("" : "+v"(a[4]), "+v"(a[5]), "+v"(a[6]), "+v"(a[7]), "+v"(b[2]), "+v"(b[3]));
    __builtin_amdgcn_s_setprio(1);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int bn = 0; bn < 8; ++bn)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int bm = bn & 1 ? 3 - i : i;
        acc[bn][bm] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[bn], b[bm], acc[bn][bm], 0, 0, 0);
      }
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_setprio(0);
#pragma unroll
    for (int bn = 0; bn < 8; ++bn)
      asm volatile("" : "+v"(acc[bn][0]), "+v"(acc[bn][1]), "+v"(acc[bn][2]), "+v"(acc[bn][3]));
  };

  issue(0, 0);
  // the epilogue's per-column constants, once per tile (the first barrier publishes them)
  if (tid < L_TN) {
    const int n = n0 + tid;
    float wv = 0.0f, bv = 0.0f;
    if (n < N) {
      wv = sw[n];
      if (BIAS_DT == GWA_DT_F32) bv = ((const float*)bias)[n];
      if (BIAS_DT == GWA_DT_BF16) bv = bf16_to_f32(((const uint16_t*)bias)[n]);
      if (BIAS_DT == GWA_DT_F16) bv = f16_bits_to_f32(((const uint16_t*)bias)[n]);
    }
    g_epi[tid] = wv;
    g_epi[L_TN + tid] = bv;
  }
  wait_vm_lgkm0<0>();
  barrier_lds();
  if (1 < nst) issue(1, 1);
  // Every group's phases are read, MFMA, read, MFMA for each stage, waves 4..7 one phase late. The copies of
  // stage st + 1 are issued in the first read phase of stage st, when every wave has drained that buffer (the late
  // group's reads of stage st - 1 ended before the last barrier), and each wave waits for its own before the
  // barrier that precedes the early group's first read of stage st + 1.
  const bool early = wave < NWAVES / 2;
  if (!early) barrier_lds();
  for (int st = 0; st < nst; ++st) {
    const uint8_t* buf = g_lds + (st & 1) * L_STAGE;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      read_ops(buf, ks);
      if (ks == 0 && st >= 1 && st + 1 < nst) issue((st + 1) & 1, st + 1);
      if (ks == 1 && !early) wait_vm_lgkm0<0>();
      else wait_lgkm0();
      __builtin_amdgcn_sched_barrier(0);
      barrier_lds();
      mma();
      if (ks == 1 && early) wait_vm_lgkm0<0>();
      barrier_lds();
    }
  }
  if (early) barrier_lds();

  // epilogue: y = acc * sa[m] * sw[n] + bias[n], packed to 16 bits. Every wave stages its own 64 x 128 tile in its
  // own 16 KB of the stage buffers (free once every wave has passed the barrier), so no barrier stands between
  // the arithmetic and the stores, which take 256-byte row segments (four rows a store instruction; as the
  // accumulators lie, a store would touch 16 rows' 32-byte pieces). The 16-byte chunk c of row r lies at slot
  // c ^ (r % 16). The per-column constants are read once per column block. Against one staged tile for the
  // workgroup, with the constants read again for every row block: 53.9 -> 52.5 us at 4096^3 (one round of tiles),
  // 113.2 -> 108.9 at 4608 x 9216 x 3072 (three).
  uint8_t* const stag = g_lds + wave * (64 * 256);
  barrier_lds();
  float am[4];
#pragma unroll
  for (int bm = 0; bm < 4; ++bm)  // rows past M are computed but never stored
    am[bm] = sa[sa_row ? min(m0 + 64 * wm + 16 * bm + r16, M - 1) : 0];
#pragma unroll
  for (int bn = 0; bn < 8; ++bn) {
    const v4f cw = *(const v4f*)(g_epi + 128 * wn + 16 * bn + 4 * q4);
    const v4f cb = *(const v4f*)(g_epi + L_TN + 128 * wn + 16 * bn + 4 * q4);
#pragma unroll
    for (int bm = 0; bm < 4; ++bm) {
      float o[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float y = (float)acc[bn][bm][e] * am[bm] * cw[e];
        if (BIAS_DT >= 0) y += cb[e];
        o[e] = y;
      }
      uint2 pk;
      if (OUT_F16) {
        pk.x = pack_f16x2(o[0], o[1]);
        pk.y = pack_f16x2(o[2], o[3]);
      } else {
        pk.x = pack_bf16x2_rn(o[0], o[1]);
        pk.y = pack_bf16x2_rn(o[2], o[3]);
      }
      *(uint2*)(stag + (16 * bm + r16) * 256 + 16 * ((2 * bn + (q4 >> 1)) ^ r16) + 8 * (q4 & 1)) = pk;
    }
  }
  asm volatile("" ::: "memory");
  // a descriptor over the wave's output span (63 N + 128 elements < 2^28: N < 2^21 is checked on the host)
  const int rows = min(M - m0 - 64 * wm, 64), cols = min(N - n0 - 128 * wn, 128);
  const uint32_t span = rows > 0 && cols > 0 ? (uint32_t)(((rows - 1) * N + cols) * 2) : 0u;
  const rsrc_t obuf = make_rsrc(out + (int64_t)(m0 + 64 * wm) * N + n0 + 128 * wn, span);
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int row = 4 * i + q4;
    const v4i v = *(const v4i*)(stag + row * 256 + 16 * (r16 ^ (row & 15)));
    uint32_t off = row < rows && 8 * r16 < cols ? (uint32_t)((row * N + 8 * r16) * 2) : kOOB;
    if (!GWA_DCHECK(off == kOOB || (int64_t)off + 16 <= (int64_t)span, kDbgW8Out, off)) off = kOOB;
    buf_store16(v, obuf, off);
  }
}

std::atomic<int> g_w8a8_force_tile{-1};  // test / tuning hook (gwa_w8a8_gemm_force_tile)

using W8Kernel = void (*)(const int8_t*, const int8_t*, const float*, const float*, const void*, uint16_t*, int, int,
                          int, int);

// A tile's geometry, the workgroups of it a CU holds at once (LDS), and the time of one to that many of them on a
// CU at K = 3072, in 0.1 us (measured; 256 x 3072 and 9216, 1024 and 2048 x 3072, 512 and 1024 x 9216).
struct W8Tile {
  int tm, tn, held;
  int us10[3];
};
constexpr W8Tile kTiles[] = {{128, 128, 2, {180, 232}}, {256, 256, 1, {335}}, {64, 64, 3, {85, 125, 165}},
                             {64, 128, 2, {114, 158}}};

template <int BD, bool F16>
W8Kernel pick_kernel(int tile) {
  switch (tile) {
    case GWA_W8A8_TILE_256x256: return w8a8_gemm_lds_kernel<BD, F16>;
    case GWA_W8A8_TILE_64x64: return w8a8_gemm_small_kernel<64, 64, 3, BD, F16>;
    case GWA_W8A8_TILE_64x128: return w8a8_gemm_small_kernel<64, 128, 3, BD, F16>;
    default: return w8a8_gemm_small_kernel<128, 128, 2, BD, F16>;
  }
}

int64_t w8a8_tiles(int tile, int64_t M, int64_t N) {
  const W8Tile& t = kTiles[tile];
  return ((M + t.tm - 1) / t.tm) * ((N + t.tn - 1) / t.tn);
}

// The tile that finishes first: the most workgroups a CU gets, in batches of as many as it holds, at the batch
// times above. They are those of K = 3072, and a launch's and an epilogue's share does not grow with K, but their
// order held: of 572 shapes (M 1 to 16384, N 512 to 18432, K 64 to 15360) the pick took more than 5 % over the
// fastest tile at 55 and 12 % at most (one row 18432 x 15360: 57.4 us, 64 x 64 51.1; 118.6 the kernel before), spread
// over all K. Measured at the picks against 128 x 128
// for everything below 256 x 256's grids, register-staged (the form before): 256 x 3072 x 3072 64 x 64 8.5 us
// (22.3), 256 x 9216 64 x 128 16.1 (24.4), 1024 x 3072 64 x 128 15.5 (24.5), 512 x 9216 128 x 128 22.6 (29.1),
// 2048 x 3072 128 x 128 23.7 (31.6), K = 12288 at 256 x 3072 64 x 64 26.7 (83.6). 256 x 256's stages need
// K % 128 == 0 and its descriptors 256 K < 2^31.
int w8a8_tile(int64_t M, int64_t N, int64_t K) {
  const bool big_ok = K % L_KS == 0 && K < (1ll << 23);
  const int forced = g_w8a8_force_tile.load(std::memory_order_relaxed);
  if (forced >= 0) return forced == GWA_W8A8_TILE_256x256 && !big_ok ? GWA_W8A8_TILE_128x128 : forced;
  int best = -1;
  int64_t best_us = 0;
  for (int t = 0; t < (int)(sizeof(kTiles) / sizeof(kTiles[0])); ++t) {
    if (t == GWA_W8A8_TILE_256x256 && !big_ok) continue;
    const int64_t per_cu = (w8a8_tiles(t, M, N) + kCus - 1) / kCus, held = kTiles[t].held;
    int64_t us = per_cu / held * kTiles[t].us10[held - 1];
    if (per_cu % held) us += kTiles[t].us10[per_cu % held - 1];
    if (best < 0 || us < best_us) {
      best = t;
      best_us = us;
    }
  }
  return best;
}

}  // namespace

extern "C" int gwa_w8a8_gemm_tile(int64_t M, int64_t N, int64_t K) {
  return M <= 0 || N <= 0 || K <= 0 ? -1 : w8a8_tile(M, N, K);
}

extern "C" int gwa_w8a8_gemm_force_tile(int tile) {
  return g_w8a8_force_tile.exchange(tile >= 0 && tile <= GWA_W8A8_TILE_64x128 ? tile : -1);
}

extern "C" int gwa_w8a8_gemm(const int8_t* qa, const int8_t* qw, const float* sa, int64_t sa_numel,
                             const float* sw, const void* bias, int bias_dtype, void* out, int out_dtype, int64_t M,
                             int64_t N, int64_t K, void* stream) {
  GWA_REQUIRE(M >= 0 && N > 0 && K > 0, "w8a8_gemm: bad shape M=%lld N=%lld K=%lld", (long long)M, (long long)N,
              (long long)K);
  GWA_REQUIRE(K % 64 == 0, "w8a8_gemm: K=%lld is not a multiple of 64", (long long)K);
  GWA_REQUIRE(N % 16 == 0, "w8a8_gemm: N=%lld is not a multiple of 16", (long long)N);
  GWA_REQUIRE(out_dtype == GWA_DT_BF16 || out_dtype == GWA_DT_F16, "w8a8_gemm: out_dtype %d not bf16/f16",
              out_dtype);
  GWA_REQUIRE(bias == nullptr || bias_dtype == GWA_DT_BF16 || bias_dtype == GWA_DT_F16 || bias_dtype == GWA_DT_F32,
              "w8a8_gemm: bias_dtype %d", bias_dtype);
  GWA_REQUIRE(M < (1ll << 31) && N < (1ll << 21) && K < (1ll << 30), "w8a8_gemm: shape too large");
  if (M == 0) return GWA_OK;
  GWA_REQUIRE(sa_numel == 1 || sa_numel == M, "w8a8_gemm: sa has %lld values for M=%lld (1 or M)",
              (long long)sa_numel, (long long)M);
  GWA_REQUIRE(qa && qw && sa && sw && out, "w8a8_gemm: null pointer");
  GWA_REQUIRE(GWA_ALIGNED(qa, 16) && GWA_ALIGNED(qw, 16) && GWA_ALIGNED(out, 8) && GWA_ALIGNED(sa, 4) &&
                  GWA_ALIGNED(sw, 4) && GWA_ALIGNED(bias, 2),
              "w8a8_gemm: qa/qw must be 16-byte and out 8-byte aligned");
  const int tile = w8a8_tile(M, N, K);
  const int64_t tiles = w8a8_tiles(tile, M, N);
  GWA_REQUIRE(tiles < (1ll << 31) - kXcds && w8a8_tiles(GWA_W8A8_TILE_128x128, M, N) < (1ll << 31),
              "w8a8_gemm: too many tiles");
  hipStream_t s = (hipStream_t)stream;
  const bool f16 = out_dtype == GWA_DT_F16;
  uint16_t* op = (uint16_t*)out;
  const int m = (int)M, n = (int)N, k = (int)K, sr = sa_numel == M && M > 1 ? 1 : 0;
  const dim3 grid((unsigned)((tiles + kXcds - 1) / kXcds * kXcds));
  const dim3 block(tile == GWA_W8A8_TILE_256x256 ? NTHREADS : 256);
  const int bd = bias ? bias_dtype : -1;
  W8Kernel kern = nullptr;
  if (bd == -1) kern = f16 ? pick_kernel<-1, true>(tile) : pick_kernel<-1, false>(tile);
  else if (bd == GWA_DT_F32) kern = f16 ? pick_kernel<GWA_DT_F32, true>(tile) : pick_kernel<GWA_DT_F32, false>(tile);
  else if (bd == GWA_DT_BF16) kern = f16 ? pick_kernel<GWA_DT_BF16, true>(tile) : pick_kernel<GWA_DT_BF16, false>(tile);
  else kern = f16 ? pick_kernel<GWA_DT_F16, true>(tile) : pick_kernel<GWA_DT_F16, false>(tile);
  hipLaunchKernelGGL(kern, grid, block, 0, s, qa, qw, sa, sw, bias, op, m, n, k, sr);
  return gwa_check_launch("w8a8_gemm");
}
