// 1-bit decode projections on either side of attention (M = 1 GEMVs over sign-bit weights).
//
// Replaces matmul_split_sg.wgsl (fusedMM: the qkv and gate/up projections, outputs routed to up
// to three buffers by row range) and matmul_resid_mr_sg.wgsl (residMM: o_proj / down_proj with
// the residual added), src/engine.ts:1344-1380, and fuses the decode attention prologue into
// the qkv projection (src/engine.ts:1526-1540: matmul_split_sg, appendKV(V), rmsnorm_rope_sg(Q),
// ROPE_K / rmsnorm_rope_sg_kv8(K)).
//
// Weights: row n, weight k is bit k % 32 of sign word [n][k / 32] (set = +1, clear = -1) times the
// f32 scale [n][k / 128] (shaders/matmul_split_sg.wgsl:24-35).
//
//   contraction  the signed sums of a row's 128-weight blocks run on the int8 matrix cores
//           (v_mfma_i32_16x16x64_i8), exactly: x becomes a 28-bit fixed-point number over its
//           block's largest power of two, in four signed int8 digits, and the integer sums are
//           scaled back per block. One sign word is the weight operand of two MFMAs after one
//           AND a dword: a byte masked to bit j is 0 or 2^j (-128 for j = 7), and x is prepared
//           with the factor 2^(7-j) for those weights, so no bit is shifted to its place (bits
//           0-3 after one shift by 4). sum (2b - 1) x = sum 2b x - sum x: the second sum is the
//           integers' start, got from the same MFMAs over all-ones weights.
//           Against the table of signed 4-term sums it replaces (8 LDS reads and 24 VALU a word,
//           16 K bytes of table built by every workgroup; rows past 4096 weights 32 sign flips and
//           adds) a word costs 9 ANDs and shifts and a quarter of two MFMAs. us a launch, graph
//           replays over 36 weights (read floor of the same bytes): gate | up 24576 x 4096 10.5 ->
//           6.8 (4.7), down 4096 x 12288 10.3 -> 5.45 (3.6), o_proj 4096 x 4096 3.48 -> 3.3 (2.9),
//           qkv + prologue 4.8 as before (3.05; K = 2560: 4.72 -> 4.46). Bound by the latency of
//           x, its conversion (about 100 VALU a wave), then the weights' arrival.
//   precision  x is rounded to within 2^-28 to 2^-31 (by its bit of the sign byte) of the power of
//           two above its block's largest magnitude, so values far below that one lose low bits that
//           f32 had, at most 4.5e-7 of it in all over the block's 128 weights, less than the bound
//           of an f32 sum of them. The block sums are exact, f32 from there on. Relative error against 64 bits
//           (2048 / 4096 / 12288 weights): normal x 6.4 / 7.6 / 9.0e-8, the f32 sums it replaces 9.4 /
//           9.5 / 10.7e-8; an outlier of 3,000 beside normal x 6.9 / 8.6 / 10.6e-8, 8.1 / 8.2 / 13.0e-8;
//           log-normal (sigma 3) 6.5 / 7.9 / 10.4e-8, 8.2 / 9.8 / 11.1e-8. A block with an infinity or
//           a NaN is summed directly in f32.
//   lanes   a 16-row tile x 4 blocks (512 weights) a step: lane 16 g + n holds the four words of
//           row n, block g (one 16-byte load), so the MFMA's four k groups are the four blocks.
//           The x operand is block diagonal: its row 4 g + p holds digit p of block g in k group
//           g and zeros elsewhere, so lane 16 g + n gets back row n's sum over block g (a digit a
//           register), which its own scale multiplies: 7 VALU for 64 block sums.
//   split   the waves of a workgroup split K (steps of 512; each prepares only its own x, in
//           registers), every wave runs the workgroup's T tiles over its part; the parts meet in
//           LDS. All loads of a wave's step are in flight before x is converted. How K is split
//           depends on K alone, so a row's sum has the same bits in every kernel and grid.
//   fused   the qkv kernel's workgroups own 32 rows of one head; all but the head's last one
//           store their raw rows into the cache's gather buffer (the XCD's L2 when the head's
//           workgroups share an XCD) and are done; the last one polls them in (no arrival
//           ticket, no store acknowledgement), writes the empty markers back at once, normalizes
//           and ropes the head (Q -> q_out; K -> the cache row, unroped in sink mode) or stores it
//           (V), with the fused prologue's row arithmetic (bg_qkrow.h; the rope partner by a lane
//           exchange).
#include "bg_kernels.h"
#include "bg_qkrow.h"

namespace bg {

typedef float floatx4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef int i32x4_t __attribute__((ext_vector_type(4)));

constexpr int kTileRows = 16;    // rows of an MFMA tile
constexpr int kStepK = 512;      // weights a tile and step: 4 blocks of 128
constexpr int kGemvMaxWaves = 16;

// How K is split over a workgroup's waves: wave w takes steps [w per, (w + 1) per). One step a wave
// up to 16 waves; longer rows 2 and more (12288 weights on 12 waves of 2 steps 5.4 us, on 8 waves
// of 3 5.8 us, 4096 rows).
struct GemvSplit {
  int steps, per, waves;
};
__host__ __device__ inline GemvSplit gemv_split(int K) {
  GemvSplit s;
  s.steps = (K + kStepK - 1) / kStepK;
  s.per = (s.steps + kGemvMaxWaves - 1) / kGemvMaxWaves;
  s.waves = (s.steps + s.per - 1) / s.per;
  return s;
}

// A wave's x digits in LDS: 16 rows (block g, digit p) of 128 bytes (digit byte i of weight order
// below), 16 bytes of pad a row so that the 16 lanes reading one column of them fall on distinct
// banks, then 128 bytes of zeros for the lanes off the operand's block diagonal.
constexpr int kDigitRow = 144;
constexpr int kDigitZero = 16 * kDigitRow;
constexpr int kDigitBytes = kDigitZero + 128;

// A step's weights of T tiles and its x values, as loaded
template <int T>
struct GemvStep {
  u32x4_t word[T];
  float sc[T];
  float2 x[4];
};

// x first: it is needed first, and vector-memory waits retire in issue order. Every load is
// unconditional (clamped to the last block; past the end x is scaled to 0 and the sum left out at
// its use, since a change here would wait for the loads).
template <int T>
__device__ __forceinline__ void gemv_load(GemvStep<T>& S, const float* __restrict__ x, int K,
                                          const uint32_t* __restrict__ sign, const float* __restrict__ scales, int n0,
                                          int n_rows, int step, int lane) {
  const int W = K >> 5, NB = K >> 7;
  const int g = lane >> 4, l = lane & 15;
  const int b = 4 * step + g, bc = b < NB ? b : NB - 1;
  // lane l of group g prepares weights 32 (l >> 2) + 8 t + 4 ((l >> 1) & 1) + 2 (l & 1) + {0, 1}
  // of block b, t = 0..3
  const float* xb = x + 128 * bc + 32 * (l >> 2) + 2 * (l & 3);
#pragma unroll
  for (int t = 0; t < 4; t++) S.x[t] = *(const float2*)(xb + 8 * t);
  __builtin_amdgcn_sched_barrier(0);  // the loads keep this order (tile t's wait covers tiles 0..t)
#pragma unroll
  for (int t = 0; t < T; t++) {
    const int n = n0 + kTileRows * t + l, nc = n < n_rows ? n : n_rows - 1;
    S.word[t] = *(const u32x4_t*)(sign + (size_t)nc * W + 4 * bc);
    S.sc[t] = scales[(size_t)nc * NB + bc];
    __builtin_amdgcn_sched_barrier(0);
  }
}

// dword j of the weight operand's half h: bit 4 + j of each byte of the word shifted by 4 h
__device__ __forceinline__ i32x4_t weight_operand(uint32_t w) {
  return i32x4_t{(int)(w & 0x10101010u), (int)(w & 0x20202020u), (int)(w & 0x40404040u), (int)(w & 0x80808080u)};
}

// The x operand of a step: digits a[2 w + h] for sign word w and half h (weights 32 w + 8 t + 4 (1
// - h) + j, byte t of dword j), what the sums start from, and each lane's block exponent.
struct GemvX {
  i32x4_t a[8];
  i32x4_t c;  // minus the half sums over all-ones weights, what the sums start from
  int exp;    // block sum = integer sum x 2^exp
  bool in;    // the lane's block lies in the row
  bool bad;   // the lane's block holds an infinity or a NaN
};

// floor(v + 0.5) in one instruction
__device__ __forceinline__ int round_i32(float v) {
  int r;
  asm("v_cvt_rpi_i32_f32 %0, %1" : "=v"(r) : "v"(v));
  return r;
}

template <int T>
__device__ __forceinline__ void gemv_prepare(GemvX& X, const GemvStep<T>& S, int K, int step, char* dig, int lane) {
  const int g = lane >> 4, l = lane & 15;
  X.in = 4 * step + g < (K >> 7);
  // largest magnitude of the lane's block (over its 16 lanes), as bits: infinities and NaN largest
  uint32_t mb = 0;
#pragma unroll
  for (int t = 0; t < 4; t++)
    mb = max(max(mb, __float_as_uint(S.x[t].x) & 0x7fffffffu), __float_as_uint(S.x[t].y) & 0x7fffffffu);
  auto dppmax = [&](auto ctrl) {
    mb = max(mb, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)mb, decltype(ctrl)::value, 0xf, 0xf, false));
  };
  dppmax(std::integral_constant<int, kDppXor1>{});
  dppmax(std::integral_constant<int, kDppXor2>{});
  dppmax(std::integral_constant<int, kDppHalfMirror>{});
  dppmax(std::integral_constant<int, kDppMirror>{});
  X.bad = X.in && mb >= 0x7f800000u;
  const int e = (int)(mb >> 23) - 126;  // |x| < 2^e
  X.exp = e - 33;
  // weights whose sign bit is masked at bit 4 + j carry 2^(4 + j): x x 2^(27 - e) x 2^(3 - j),
  // at most 2^30; bit 7 reads as -128. An infinity or NaN leaves some integer, which only its own
  // block's sum sees: inside the row that block is summed again in f32; a lane past the row's end
  // (it holds the last block again) scales finite values to 0, and its sum is never used.
  const int jp = 2 * (l & 1);
  const int h = 1 - ((l >> 1) & 1);
  uint32_t y[2][4];
#pragma unroll
  for (int u = 0; u < 2; u++) {
    const int sh = X.in ? 30 - e - (jp + u) : -1024;
    const uint32_t flip = jp + u == 3 ? 0x80000000u : 0u;
#pragma unroll
    for (int t = 0; t < 4; t++) {
      const uint32_t v = __float_as_uint(u == 0 ? S.x[t].x : S.x[t].y);
      const int q = round_i32(ldexpf(__uint_as_float(u == 0 ? v : v ^ flip), sh));
      y[u][t] = ((uint32_t)q + 0x80808080u) ^ 0x80808080u;  // signed base-256 digits
    }
  }
  // 4 x 4 byte transposes: dword of digit p = byte p of y[.][0..3]
  char* row = dig + (4 * g) * kDigitRow + (2 * (l >> 2) + h) * 16 + 4 * jp;
  uint32_t d[2][4];
#pragma unroll
  for (int u = 0; u < 2; u++) {
    const uint32_t p01 = __builtin_amdgcn_perm(y[u][1], y[u][0], 0x05010400u);  // y0.b0 y1.b0 y0.b1 y1.b1
    const uint32_t p23 = __builtin_amdgcn_perm(y[u][3], y[u][2], 0x05010400u);
    const uint32_t q01 = __builtin_amdgcn_perm(y[u][1], y[u][0], 0x07030602u);  // bytes 2, 3
    const uint32_t q23 = __builtin_amdgcn_perm(y[u][3], y[u][2], 0x07030602u);
    d[u][0] = __builtin_amdgcn_perm(p23, p01, 0x05040100u);
    d[u][1] = __builtin_amdgcn_perm(p23, p01, 0x07060302u);
    d[u][2] = __builtin_amdgcn_perm(q23, q01, 0x05040100u);
    d[u][3] = __builtin_amdgcn_perm(q23, q01, 0x07060302u);
  }
  // the reads of the step before are done (their MFMAs have used them); the wave's own LDS
  // accesses complete in order
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
#pragma unroll
  for (int p = 0; p < 4; p++) *(uint2*)(row + p * kDigitRow) = make_uint2(d[0][p], d[1][p]);
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  // row m = l of the operand: digit l & 3 of block l >> 2, nonzero in that block's k group only
  const char* src = dig + ((l >> 2) == g ? l * kDigitRow : kDigitZero);
#pragma unroll
  for (int i = 0; i < 8; i++) X.a[i] = *(const i32x4_t*)(src + 16 * i);
  // minus half of the sums over all-ones weights (those are even: every weight byte is)
  i32x4_t f[2] = {{0, 0, 0, 0}, {0, 0, 0, 0}};
#pragma unroll
  for (int i = 0; i < 8; i++) f[i & 1] = __builtin_amdgcn_mfma_i32_16x16x64_i8(X.a[i], weight_operand(~0u), f[i & 1], 0, 0, 0);
#pragma unroll
  for (int i = 0; i < 4; i++) X.c[i] = -((f[0][i] + f[1][i]) >> 1);
}

// the lane's block sum directly in f32, for a block that holds an infinity or a NaN
__device__ __noinline__ float gemv_block_f32(const float* __restrict__ xb, u32x4_t word) {
  float s = 0.0f;
#pragma unroll
  for (int w = 0; w < 4; w++) {
    const uint32_t nw = ~word[w];
#pragma unroll 1
    for (int i = 0; i < 32; i++) s += __uint_as_float(__float_as_uint(xb[32 * w + i]) ^ ((nw << (31 - i)) & 0x80000000u));
  }
  return s;
}

template <int T>
__device__ __forceinline__ void gemv_accumulate(float (&acc)[T], const GemvStep<T>& S, const GemvX& X,
                                                const float* __restrict__ x, int K, int step, int lane) {
  float s[T];
  // two tiles at a time, or the two halves of one: independent MFMA chains (exact integer sums, so
  // their order does not matter). A single tile does not wait for the start values either.
#pragma unroll
  for (int t0 = 0; t0 < T; t0 += 2) {
    const bool pair = t0 + 1 < T;
    const i32x4_t zero = {0, 0, 0, 0};
    i32x4_t d[2] = {T == 1 ? zero : X.c, pair ? X.c : zero};
#pragma unroll
    for (int i = 0; i < 8; i++)
#pragma unroll
      for (int u = 0; u < (pair ? 2 : 1); u++) {
        const uint32_t w = S.word[t0 + u][i >> 1];
        i32x4_t& dd = d[pair ? u : i & 1];
        dd = __builtin_amdgcn_mfma_i32_16x16x64_i8(X.a[i], weight_operand(i & 1 ? w << 4 : w), dd, 0, 0, 0);
      }
    if (!pair) d[0] += T == 1 ? d[1] + X.c : d[1];
#pragma unroll
    for (int u = 0; u < (pair ? 2 : 1); u++) {
      // digits 0, 1 and 2, 3 join as integers (|d| <= 2^21, so below 2^30), then in f32
      const float lo = (float)(d[u][0] + (d[u][1] << 8)), hi = (float)(d[u][2] + (d[u][3] << 8));
      s[t0 + u] = ldexpf(fmaf(hi, 65536.0f, lo), X.exp);
    }
  }
  if (__any(X.bad)) {
    const int b = min(4 * step + (lane >> 4), (K >> 7) - 1);
#pragma unroll
    for (int t = 0; t < T; t++)
      if (X.bad) s[t] = gemv_block_f32(x + 128 * b, S.word[t]);
  }
#pragma unroll
  for (int t = 0; t < T; t++) acc[t] = X.in ? fmaf(s[t], S.sc[t], acc[t]) : acc[t];
}

// One wave's part of the workgroup's rows n0 .. n0 + 16 T - 1: the sums over its steps into
// red[wave][row]. PER: the steps a wave takes when that is at most 2 (K <= 16384): all their
// loads are issued before the first x is converted; 0: any number, the next step's loads issued
// before this one's x is converted. dig: the wave's kDigitBytes of LDS.
template <int T, int PER>
__device__ __forceinline__ void gemv_part(const float* __restrict__ x, int K, const uint32_t* __restrict__ sign,
                                          const float* __restrict__ scales, int n0, int n_rows, int wave, int lane,
                                          char* dig, float* red) {
  const GemvSplit sp = gemv_split(K);
  const int s0 = wave * sp.per, s1 = min(s0 + sp.per, sp.steps);
  constexpr int NB = PER ? PER : 2;
  GemvStep<T> S[NB];
#pragma unroll
  for (int i = 0; i < (PER ? PER : 1); i++) gemv_load<T>(S[i], x, K, sign, scales, n0, n_rows, min(s0 + i, s1 - 1), lane);
  if (lane < 8) *(uint4*)(dig + kDigitZero + 16 * lane) = make_uint4(0, 0, 0, 0);
  float acc[T];
#pragma unroll
  for (int t = 0; t < T; t++) acc[t] = 0.0f;
  GemvX X;
  auto step = [&](const GemvStep<T>& A, int s) {
    gemv_prepare<T>(X, A, K, s, dig, lane);
    gemv_accumulate<T>(acc, A, X, x, K, s, lane);
  };
  if constexpr (PER > 0) {
#pragma unroll
    for (int i = 0; i < PER; i++)
      if (i == 0 || s0 + i < s1) step(S[i], s0 + i);
  } else {
    for (int s = s0; s < s1; s += 2) {
      gemv_load<T>(S[1], x, K, sign, scales, n0, n_rows, min(s + 1, s1 - 1), lane);
      step(S[0], s);
      if (s + 1 >= s1) break;
      gemv_load<T>(S[0], x, K, sign, scales, n0, n_rows, min(s + 2, s1 - 1), lane);
      step(S[1], s + 1);
    }
  }
#pragma unroll
  for (int t = 0; t < T; t++) {
    float2 r = pair16(acc[t]);
    r = pair32(r.x + r.y);
    if (lane < kTileRows) red[wave * (kTileRows * T) + kTileRows * t + lane] = r.x + r.y;
  }
}

// row r of the workgroup: its parts in wave order (after the barrier)
template <int T, int NW>
__device__ __forceinline__ float gemv_row(const float* red, int r, int waves) {
  float p[NW];
#pragma unroll
  for (int w = 0; w < NW; w++) p[w] = red[min(w, waves - 1) * (kTileRows * T) + r];
  float y = p[0];
#pragma unroll
  for (int w = 1; w < NW; w++) y += w < waves ? p[w] : 0.0f;
  return y;
}

// NW: the most waves of the launch (8 up to K = 4096: a quarter more registers and LDS a wave)
template <int T, int PER, int NW>
__global__ __launch_bounds__(64 * NW) void gemv_kernel(GemvArgs a) {
  __shared__ __align__(16) char dig[NW * kDigitBytes];
  __shared__ float red[NW * kTileRows * T];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int N = a.N0 + a.N1 + a.N2;
  const int n0 = blockIdx.x * kTileRows * T;
  // each thread's first row's residual, loaded before anything waits
  const int nr = n0 + threadIdx.x;
  const float res = a.resid && threadIdx.x < kTileRows * T && nr < N ? a.resid[nr] : 0.0f;
  gemv_part<T, PER>(a.x, a.K, a.sign, a.scales, n0, N, wave, lane, dig + wave * kDigitBytes, red);
  __syncthreads();
  for (int r = threadIdx.x; r < kTileRows * T; r += blockDim.x) {
    const int n = n0 + r;
    if (n >= N) return;
    const float tot = gemv_row<T, NW>(red, r, blockDim.x >> 6);
    const float y = a.resid ? tot + (r == (int)threadIdx.x ? res : a.resid[n]) : tot;
    if (n < a.N0) a.out0[n] = y;
    else if (n < a.N0 + a.N1) a.out1[n - a.N0] = y;
    else a.out2[n - a.N0 - a.N1] = y;
  }
}

template <int T>
static void launch_gemv_t(const GemvArgs& a, int N, hipStream_t st) {
  const dim3 g((N + kTileRows * T - 1) / (kTileRows * T)), b(64 * gemv_split(a.K).waves);
  const GemvSplit sp = gemv_split(a.K);
  if (sp.per == 1 && sp.waves <= 8) hipLaunchKernelGGL((gemv_kernel<T, 1, 8>), g, b, 0, st, a);
  else if (sp.per == 1) hipLaunchKernelGGL((gemv_kernel<T, 1, 16>), g, b, 0, st, a);
  else if (sp.per == 2) hipLaunchKernelGGL((gemv_kernel<T, 2, 16>), g, b, 0, st, a);
  else hipLaunchKernelGGL((gemv_kernel<T, 0, 16>), g, b, 0, st, a);
}

hipError_t launch_gemv(const GemvArgs& a, hipStream_t st) {
  const int N = a.N0 + a.N1 + a.N2;
  if (N <= 0) return hipSuccess;
  // One tile a workgroup spreads few rows over the most CUs (4096 rows: 3.3 us against 3.7 with
  // two). From 512 tiles, two: x is converted half as often (24576 x 4096: 6.8 us against 8.2 with
  // one, 7.2 to 8.0 with three to six; 768 tiles of 2048 weights, 3.7 and 3.8, do not care).
  const int tiles = (N + kTileRows - 1) / kTileRows;
  if (tiles <= 512) launch_gemv_t<1>(a, N, st);
  else launch_gemv_t<2>(a, N, st);
  return hipGetLastError();
}

// ---- fused decode qkv projection + prologue ---------------------------------------------------
// s_waitcnt vmcnt(0) with expcnt and lgkmcnt left alone (gfx9 encoding: vmcnt bits 3:0 and 15:14,
// expcnt 6:4, lgkmcnt 11:8)
constexpr int kWaitVm0 = 0x0F70;

size_t qkv_proj_raw_floats(int heads, int D) { return (size_t)heads * D; }

// Workgroup v owns rows [v RPW, v RPW + RPW) of the [Q heads | K heads | V heads] x D output (RPW
// divides D, so they are one head's). The workgroup holding a head's last rows finishes that head:
// its rows stay in LDS, every other workgroup's go into the gather buffer. The finisher's first
// wave polls the head's earlier rows until none holds the empty marker (the data is the completion
// signal: no ticket, no store acknowledgement to wait for); it then writes the marker back
// (written through: the next launch's workgroups may run on another XCD), normalizes, ropes and
// stores the row with the prologue's arithmetic (bg_qkrow.h: bit-identical to bg_gemv_split
// followed by bg_qkv_prologue). The rows a finisher waits on belong to lower workgroup indices,
// dispatched before it, which finish on their own; the wait is still bounded (a finisher that
// gives up stores NaN and raises the cache's error word). When the grid is a multiple of 8 and
// every eighth of the rows is whole heads, blockIdx 8m + x is workgroup v = x (grid / 8) + m, so
// with round-robin placement each XCD holds a run of whole heads and the raw rows stay in its L2.
template <int D, int DT, int T, int PER, int NW>
__global__ __launch_bounds__(64 * NW) void qkv_proj_kernel(LayerView L, QkvProjArgs a) {
  constexpr int RPW = kTileRows * T;
  constexpr int LPR = D / 4;  // lanes per row in the epilogue
  constexpr int kSC1 = 16;    // cache policy sc1: agent scope
  static_assert(RPW <= 64 && D % RPW == 0, "rows of a workgroup");
  __shared__ __align__(16) char dig[NW * kDigitBytes];
  __shared__ float red[NW * RPW];
  __shared__ __align__(16) float rrow[D];
  __shared__ __align__(16) float own[RPW];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int KV = L.kv_heads;
  const int nq = a.H * D;
  const int N = nq + 2 * KV * D;  // gridDim.x * RPW
  const int nwg = gridDim.x;
  const bool grouped = (nwg & 7) == 0 && ((nwg >> 3) * RPW) % D == 0;
  const int v = grouped ? (blockIdx.x & 7) * (nwg >> 3) + (blockIdx.x >> 3) : blockIdx.x;
  const int r0 = v * RPW;
  const int head = r0 / D;  // 0 .. H-1: Q heads, then K heads, then V heads
  const bool finisher = r0 + RPW == (head + 1) * D;  // holds the head's last rows
  const int own0 = r0 - head * D;                    // the workgroup's first dim of the head
  // raw rows stay in the XCD's L2 when every workgroup of the head shares it
  const bool local = grouped && a.n_xcd == 8;
  gemv_part<T, PER>(a.x, a.K, a.sign, a.scales, r0, N, wave, lane, dig + wave * kDigitBytes, red);
  __syncthreads();
  if (wave != 0) return;
  // the first wave: one row a lane
  if (lane < RPW) {
    const float tot = gemv_row<T, NW>(red, lane, blockDim.x >> 6);
    if (finisher) own[lane] = tot;
    else if (local) a.raw[r0 + lane] = tot;  // into the XCD's L2
    else st_coherent(a.raw + r0 + lane, tot);
  }
  if (!finisher) return;

  // ---- the finishing part of the head: one wave, 4 dims a lane (D=128: both halves of the
  // wave hold the row; the lower one stores) ----
  const int c = lane % LPR;
  const bool writer = lane < LPR;
  const bool isq = head < a.H, isk = !isq && head < a.H + KV;
  const bool mine = 4 * c >= own0;  // own0 is a multiple of 16
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(a.raw + (size_t)head * D, (short)0,
                                                                      D * 4, 0x00020000);
  // the row's gamma and rope tables are loaded before the wait, so the epilogue starts on arrival
  const bool rope = isq || (isk && !L.ring.roll);  // sink mode caches K unroped (src/engine.ts:1530-1533)
  float g[4] = {1.0f, 1.0f, 1.0f, 1.0f}, cs[4], sn[4];
  if (isq || isk) load4((isq ? a.q_gamma : a.k_gamma) + 4 * c, g);
  if (rope) row_tables(a.cos_tab, a.sin_tab, a.pos, a.rot_dim, c, cs, sn);
  // the other workgroups' rows
  float x[4];
  bool gave_up = false;
  if (!mine) {
    const int spins = a.spin_limit > 0 ? a.spin_limit : (1 << 20);
    bool missing = true;
    for (int it = 0; it < spins && missing; it++) {
      // a compiler memory barrier: the load is issued again every round (other workgroups
      // write the rows; without it the compiler may reuse the last round's value)
      __asm__ volatile("" ::: "memory");
      const floatx4_t v = __builtin_bit_cast(floatx4_t, __builtin_amdgcn_raw_buffer_load_b128(rs, 16 * c, 0, kSC1));
#pragma unroll
      for (int e = 0; e < 4; e++) x[e] = v[e];
      missing = false;
#pragma unroll
      for (int e = 0; e < 4; e++) missing = missing || __float_as_uint(x[e]) == kWorkspaceEmpty;
      if (missing) __builtin_amdgcn_s_sleep(1);
    }
    gave_up = missing;
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");  // own[], written by this wave
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  if (mine) {
#pragma unroll
    for (int e = 0; e < 4; e++) x[e] = own[4 * c + e - own0];
  }
  gave_up = __any(gave_up);
  // the empty marker back into the slots read, as soon as they are in registers (before the
  // row's stores: a marker store issued after them would wait for their acknowledgement, since
  // it reuses their data registers). Every load has arrived here (the poll waited for its own,
  // issued after gamma and the tables); the explicit vmcnt(0) says so to the compiler, which
  // would otherwise wait for the marker store's acknowledgement before using gamma.
  __builtin_amdgcn_s_waitcnt(kWaitVm0);
  if (writer && !mine) {
    const u32x4_t empty4 = {kWorkspaceEmpty, kWorkspaceEmpty, kWorkspaceEmpty, kWorkspaceEmpty};
    __builtin_amdgcn_raw_buffer_store_b128(empty4, rs, 16 * c, 0, kSC1);
  }
  if (gave_up) {
#pragma unroll
    for (int e = 0; e < 4; e++) x[e] = __builtin_nanf("");
  }
  if (isq || isk) {
    row_scale(x, row_inv_rms<D, LPR>(x, a.eps), g);
    if (rope) {
      // the rotate_half partners by a lane exchange where the width allows it, else through LDS
      float pr[4];
      if (rope_partner_lanes(x, a.rot_dim, pr)) {
        row_rope_lanes(x, pr, c, a.rot_dim, cs, sn);
      } else {
        if (writer) *(float4*)(rrow + 4 * c) = make_float4(x[0], x[1], x[2], x[3]);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        row_rope(x, rrow, c, a.rot_dim, cs, sn);
      }
    }
    if (isq) {
      if (writer) *(float4*)(a.q_out + head * D + 4 * c) = make_float4(x[0], x[1], x[2], x[3]);
    } else {
      // every lane joins the q8 block maxima; the lower half stores
      if (D == 256 || writer) store_k4<D, DT>(L, L.ring.phys(a.slot), head - a.H, x, c);
    }
  } else {
    if (D == 256 || writer) store_v4<D, DT>(L, L.ring.phys(a.slot), head - a.H - KV, x, c);
  }
  if (gave_up && lane == 0) __hip_atomic_store(a.err, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

template <int D, int T, int PER, int NW>
static hipError_t launch_qkv_proj_t(const LayerView& L, const QkvProjArgs& a, hipStream_t st) {
  const dim3 g((a.H + 2 * L.kv_heads) * D / (kTileRows * T)), b(64 * gemv_split(a.K).waves);
  switch (L.dtype) {
    case KV_F32: hipLaunchKernelGGL((qkv_proj_kernel<D, KV_F32, T, PER, NW>), g, b, 0, st, L, a); break;
    case KV_F16: hipLaunchKernelGGL((qkv_proj_kernel<D, KV_F16, T, PER, NW>), g, b, 0, st, L, a); break;
    default: hipLaunchKernelGGL((qkv_proj_kernel<D, KV_Q8, T, PER, NW>), g, b, 0, st, L, a);
  }
  return hipGetLastError();
}

// 32 rows a workgroup: 192 workgroups for the 8B shape, 4.82 us; 16 rows (384) 5.0, 64 (96) 5.7
template <int D>
static hipError_t launch_qkv_proj_d(const LayerView& L, const QkvProjArgs& a, hipStream_t st) {
  const GemvSplit sp = gemv_split(a.K);
  if (sp.per == 1 && sp.waves <= 8) return launch_qkv_proj_t<D, 2, 1, 8>(L, a, st);
  return sp.per == 1 ? launch_qkv_proj_t<D, 2, 1, 16>(L, a, st) : launch_qkv_proj_t<D, 2, 0, 16>(L, a, st);
}

hipError_t launch_qkv_proj(const LayerView& L, const QkvProjArgs& a, hipStream_t st) {
  return L.D == 128 ? launch_qkv_proj_d<128>(L, a, st) : launch_qkv_proj_d<256>(L, a, st);
}

}  // namespace bg
