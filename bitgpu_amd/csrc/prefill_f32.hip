// Causal GQA prefill over an f32 KV cache (kvCache 'f32', the reference default) on the f32
// matrix cores of gfx950: prefill_f32_kernel at head_dim 256, prefill_f32_split_kernel (below) at
// 128 past the shortest prompts, the same arithmetic.
//
// Replaces attention_sg.wgsl / attention_wg.wgsl (and their _roll and f32
// attention_online_cache forms) for more than 16 rows per kv head: those run one subgroup per
// (query, head) scanning every position serially (attention_sg.wgsl:21-44), each GQA head
// re-reading its group's K/V. Here:
//
//   items  = (query block, kv head): QB = 128 / G queries x the G heads of one kv head, 128 rows,
//            4 waves of 32 rows; every K/V byte a block attends is read once for all its rows.
//            Heaviest (latest queries) first; when a CU holds two workgroups and the grid fits at
//            once, each heavy item is paired with its mirror light item on one CU (workgroups b
//            and b + n/2 share a CU when the grid is dispatched in one wave).
//   tiles  = 32 keys a step, K rows and the cache's transposed 32-slot V tile staged into LDS
//            (double-buffered, one barrier a step); sink mode rotates K at staging by the slot's
//            logical (or absolute) position, in f32 with the reference's operand order
//            (attention_sg_roll.wgsl:40-51).
//   QK     = S^T = K . Q^T on v_mfma_f32_32x32x2_f32 (f32 products, f32 accumulation): K as A
//            (lane = key, one b128 LDS read feeds 4 MFMAs), the row's query (times scale * log2 e)
//            in registers as B; two independent accumulator chains.
//   softmax= online, base 2, per 32-key step; each row's 32 scores sit in lanes l and l ^ 32.
//   PV     = O^T += V^T . P^T on the same instruction: the 32x32 result layout puts key
//            8 (r / 4) + 4 (l / 32) + r % 4 of the row in register r of lane l, and the cache's V
//            tile stores exactly those keys of a dim in panel l / 32 (r < 8) and 2 + l / 32 -- so
//            register r of S^T is the B operand of PV MFMA r and the V operand is two contiguous
//            b128 reads a panel: no transpose of P or V.
// All arithmetic is f32, so the output meets the reference's max-abs 1e-4 bar for f32 storage.
#include <algorithm>
#include <mutex>

#include "bg_kernels.h"

namespace bg {

typedef float floatx16 __attribute__((ext_vector_type(16)));

constexpr int kF32KT = 32;   // keys per step
constexpr int kF32Rows = 128;  // rows per workgroup (4 waves x 32)

template <int D>
struct F32Smem {
  static constexpr int KS = D + 4;                         // padded K row (floats)
  static constexpr size_t k_floats = (size_t)kF32KT * KS;  // one K buffer
  static constexpr size_t v_floats = (size_t)kF32KT * D;   // one V tile (4 panels x D x 8)
  static constexpr size_t bytes = 2 * (k_floats + v_floats) * 4;
};

struct F32PrefillParams {
  LayerView L;
  const float* q;
  int S, H, G, QB;
  int pos_base;
  float qscale;  // scale * log2(e)
  const float* gate;
  int gate_stride;
  float* out;
  int n_scan_fixed;  // >0: physical slots scanned by every block (sink mode after a wrap); 0: causal bound
  int phys_limit;
  int n_qblocks;
  int mirror;
};

template <int D, bool ROLL>
__global__ __launch_bounds__(256) void prefill_f32_kernel(F32PrefillParams p) {
  using SM = F32Smem<D>;
  constexpr int KS = SM::KS;
  constexpr int NQ = D / 8;   // 8-dim blocks: one float4 of Q per lane each
  constexpr int NO = D / 32;  // 32-dim output blocks
  extern __shared__ __align__(16) float smf[];
  // double buffers: K [2][32][KS], then V [2][32 * D]
  auto kb = [&](int buf) { return smf + buf * SM::k_floats; };
  auto vb = [&](int buf) { return smf + 2 * SM::k_floats + buf * SM::v_floats; };

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int n = lane & 31, hk = lane >> 5;
  const LayerView& L = p.L;
  const int KV = L.kv_heads;

  const int bid = blockIdx.x;
  const int n_items = p.n_qblocks * KV;
  const int half = (n_items + 1) / 2;
  const int item = !p.mirror || bid < half ? bid : n_items - 1 - (bid - half);
  const int kvh = item % KV;
  const int qb = p.n_qblocks - 1 - item / KV;
  const int s0 = qb * p.QB;
  const int G = p.G;

  // this lane's row (column n of the wave's 32 x 32 blocks)
  const int r = wave * 32 + n;
  const int qi = s0 + r / G;
  const int h = kvh * G + r % G;
  const bool row_ok = r < p.QB * G && qi < p.S;
  const int limit = row_ok ? p.pos_base + qi : -1;
  const int last_q = min(s0 + p.QB, p.S) - 1;
  // the last query row of this wave (wave-uniform): steps past it are masked for every row
  const int wave_last_q = min(s0 + min((wave * 32 + 31) / G, p.QB - 1), p.S - 1);
  const int wave_limit = (wave * 32 < p.QB * G) ? p.pos_base + wave_last_q : -1;
  const int n_keys = p.n_scan_fixed > 0 ? p.n_scan_fixed : p.pos_base + last_q + 1;
  const int kmax = min(n_keys, p.phys_limit);
  const int steps = (n_keys + kF32KT - 1) / kF32KT;

  // Q as the B operand: lane (n, hk) holds dims 8 t + 4 hk .. + 3 of its row, times qscale
  float4 qv[NQ];
  {
    const float* qr = p.q + ((size_t)(row_ok ? qi : 0) * p.H + (row_ok ? h : 0)) * D + 4 * hk;
#pragma unroll
    for (int t = 0; t < NQ; t++) {
      float4 x = *(const float4*)(qr + 8 * t);
      const float f = row_ok ? p.qscale : 0.0f;
      qv[t] = make_float4(x.x * f, x.y * f, x.z * f, x.w * f);
    }
  }

  const float* Kg = (const float*)L.k + (size_t)kvh * L.cap * D;
  const float* Vg = (const float*)L.v + (size_t)kvh * L.cap * D;
  // staging: thread tid copies K pair items (key, dims c..c+3 and c+D/2..) and V float4s
  constexpr int KPI = kF32KT * (D / 8) / 256;  // K pair items a thread
  constexpr int VPI = kF32KT * D / 4 / 256;    // V float4 a thread
  float4 kr[KPI][2], vr[VPI];
  auto fetch = [&](int step) {
    const int j0 = step * kF32KT;
#pragma unroll
    for (int i = 0; i < KPI; i++) {
      const int it = tid + 256 * i;
      const int key = it / (D / 8), c = 4 * (it % (D / 8));
      const float* row = Kg + (size_t)(j0 + key) * D;
      kr[i][0] = *(const float4*)(row + c);
      kr[i][1] = *(const float4*)(row + c + D / 2);
    }
#pragma unroll
    for (int i = 0; i < VPI; i++) vr[i] = *(const float4*)(Vg + (size_t)j0 * D + 4 * (tid + 256 * i));
  };
  auto stage = [&](int step, int buf) {
    const int j0 = step * kF32KT;
#pragma unroll
    for (int i = 0; i < KPI; i++) {
      const int it = tid + 256 * i;
      const int key = it / (D / 8), c = 4 * (it % (D / 8));
      float4 lo = kr[i][0], hi = kr[i][1];
      if constexpr (ROLL) {
        // k_d cos + rot_d sin, rot = -k_{d+D/2} (d < D/2) or k_{d-D/2}, at the slot's position
        const int P = j0 + key;
        int Lg = L.ring.logical(P);
        Lg = P < p.phys_limit ? Lg : 0;
        long ri = (L.rope_abs && Lg >= L.ring.sinks) ? (long)Lg + L.evicted : (long)Lg;
        ri = ri < L.rope_positions ? ri : 0;
        const float4 cs = *(const float4*)(L.cos_tab + (size_t)ri * (D / 2) + c);
        const float4 sn = *(const float4*)(L.sin_tab + (size_t)ri * (D / 2) + c);
        // two rounded products and a rounded sum, not fused
        auto rot = [](float a, float b, float co, float si) { return add_rn(mul_rn(a, co), mul_rn(-b, si)); };
        auto rot2 = [](float b, float a, float co, float si) { return add_rn(mul_rn(b, co), mul_rn(a, si)); };
        lo = make_float4(rot(kr[i][0].x, kr[i][1].x, cs.x, sn.x), rot(kr[i][0].y, kr[i][1].y, cs.y, sn.y),
                         rot(kr[i][0].z, kr[i][1].z, cs.z, sn.z), rot(kr[i][0].w, kr[i][1].w, cs.w, sn.w));
        hi = make_float4(rot2(kr[i][1].x, kr[i][0].x, cs.x, sn.x), rot2(kr[i][1].y, kr[i][0].y, cs.y, sn.y),
                         rot2(kr[i][1].z, kr[i][0].z, cs.z, sn.z), rot2(kr[i][1].w, kr[i][0].w, cs.w, sn.w));
      }
      *(float4*)(kb(buf) + key * KS + c) = lo;
      *(float4*)(kb(buf) + key * KS + c + D / 2) = hi;
    }
#pragma unroll
    for (int i = 0; i < VPI; i++) {
      // slots past the last valid one read as 0 (their probabilities are 0; 0 * garbage could
      // be NaN)
      const int f = 4 * (tid + 256 * i);  // float offset in the tile: panel (D*8), dim 8, index
      float4 x = vr[i];
      if (j0 + kF32KT > kmax) {
        const int panel = f / (D * 8), idx = f % 8;
        float* e = &x.x;
#pragma unroll
        for (int u = 0; u < 4; u++)
          if (j0 + tile_slot(panel, idx + u) >= kmax) e[u] = 0.0f;
      }
      *(float4*)(vb(buf) + f) = x;
    }
  };

  floatx16 o[NO];
#pragma unroll
  for (int b = 0; b < NO; b++)
#pragma unroll
    for (int i = 0; i < 16; i++) o[b][i] = 0.0f;
  float m = -1e30f, lsum = 0.0f;

  if (steps > 0) {
    fetch(0);
    stage(0, 0);
  }
  __syncthreads();
  for (int step = 0; step < steps; step++) {
    const int buf = step & 1;
    if (step + 1 < steps) fetch(step + 1);
    const int j0 = step * kF32KT;
    // a step past every row of this wave (plain cache) is all masked: nothing to add
    const bool active = p.n_scan_fixed > 0 || j0 <= wave_limit;
    if (active) {
      const float* kt = kb(buf);
      floatx16 s0v, s1v;
#pragma unroll
      for (int i = 0; i < 16; i++) {
        s0v[i] = 0.0f;
        s1v[i] = 0.0f;
      }
#pragma unroll
      for (int t = 0; t < NQ; t++) {
        const float4 kk = *(const float4*)(kt + n * KS + 8 * t + 4 * hk);
        floatx16& acc = (t & 1) ? s1v : s0v;
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(kk.x, qv[t].x, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(kk.y, qv[t].y, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(kk.z, qv[t].z, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(kk.w, qv[t].w, acc, 0, 0, 0);
      }
      // register e holds key 8 (e / 4) + 4 hk + e % 4 of this lane's row
      float sv[16];
      float mt = -INFINITY;
#pragma unroll
      for (int e = 0; e < 16; e++) {
        const int P = j0 + 8 * (e >> 2) + 4 * hk + (e & 3);
        const int Lg = ROLL ? L.ring.logical(P) : P;
        const bool ok = P < kmax && Lg <= limit;
        sv[e] = ok ? s0v[e] + s1v[e] : -INFINITY;
        mt = fmaxf(mt, sv[e]);
      }
      {
        const float2 pr = pair32(mt);
        mt = fmaxf(pr.x, pr.y);
      }
      // the reference maximum is raised only when a step's maximum exceeds it by more than 8
      // (log2 units: probabilities stay below 2^8), so most steps leave O and l unscaled
      if (__any(mt > m + 8.0f)) {
        const float mn = fmaxf(m, mt);
        const float corr = __builtin_amdgcn_exp2f(m - mn);
        m = mn;
        lsum *= corr;
#pragma unroll
        for (int b = 0; b < NO; b++)
#pragma unroll
          for (int i = 0; i < 16; i++) o[b][i] *= corr;
      }
      float ps = 0.0f;
      floatx16 pv;
#pragma unroll
      for (int e = 0; e < 16; e++) {
        pv[e] = __builtin_amdgcn_exp2f(sv[e] - m);
        ps += pv[e];
      }
      {
        const float2 pr = pair32(ps);
        ps = pr.x + pr.y;
      }
      lsum += ps;
      // PV: dim block b, MFMA e takes key slot e of this lane's panel pair
      const float* vt = vb(buf);
#pragma unroll
      for (int b = 0; b < NO; b++) {
        const int d = 32 * b + n;
        const float4 v0 = *(const float4*)(vt + (size_t)hk * (D * 8) + d * 8);
        const float4 v1 = *(const float4*)(vt + (size_t)hk * (D * 8) + d * 8 + 4);
        const float4 v2 = *(const float4*)(vt + (size_t)(2 + hk) * (D * 8) + d * 8);
        const float4 v3 = *(const float4*)(vt + (size_t)(2 + hk) * (D * 8) + d * 8 + 4);
        const float va[16] = {v0.x, v0.y, v0.z, v0.w, v1.x, v1.y, v1.z, v1.w,
                              v2.x, v2.y, v2.z, v2.w, v3.x, v3.y, v3.z, v3.w};
#pragma unroll
        for (int e = 0; e < 16; e++) o[b] = __builtin_amdgcn_mfma_f32_32x32x2f32(va[e], pv[e], o[b], 0, 0, 0);
      }
    }
    if (step + 1 < steps) stage(step + 1, buf ^ 1);
    __syncthreads();
  }

  // O^T block b: register e of lane (n, hk) holds dim 32 b + 8 (e / 4) + 4 hk + e % 4 of row n
  if (row_ok) {
    const float inv_l = 1.0f / lsum;
    float* orow = p.out + ((size_t)qi * p.H + h) * D;
    const float* grow = p.gate ? p.gate + ((size_t)qi * p.H + h) * p.gate_stride : nullptr;
#pragma unroll
    for (int b = 0; b < NO; b++)
#pragma unroll
      for (int e4 = 0; e4 < 4; e4++) {
        const int d = 32 * b + 8 * e4 + 4 * hk;
        float x[4];
#pragma unroll
        for (int u = 0; u < 4; u++) x[u] = o[b][4 * e4 + u] * inv_l;
        if (grow) {
#pragma unroll
          for (int u = 0; u < 4; u++) x[u] = x[u] / (1.0f + expf(-grow[d + u]));
        }
        *(float4*)(orow + d) = make_float4(x[0], x[1], x[2], x[3]);
      }
  }
}

// ---- head_dim 128: a wave's keys in registers, an item's waves sharing rows or keys --------------
// The f32 MFMAs take 8192 cycles a 32-key step of 32 rows (about 3.8 us with the softmax), so
// nothing else has to be fast but every wave has to be busy. KS of an item's four waves share 32
// rows, each taking every KS-th step (KS = 4: an item is 32 rows and a quarter of the chain that
// 128 rows are; 1: 128 rows, a wave its own 32) and merge in LDS at the end. A wave owns its step's keys, so K and V go straight from the
// cache into registers in the MFMAs' operand layout (K: one 16-byte load feeds 4 MFMAs, V: the
// transposed tile's 32 contiguous bytes a dim): no LDS, no barrier in the loop. The K registers
// are loaded again right after the step's QK and V's after its PV, each half a step (about 4000
// cycles) before they are used. Grids that still leave CUs idle split every item's keys over
// workgroups (f32 partials, merged by the f16 prefill's merge kernels, whose layout this has).
// Against the 128-row items of the kernel above, us (floor at 153 TFLOP/s, a large f32 matrix
// product's): 777 tokens, 16 heads 117 -> 44 (16); 2048, 32 heads 320 -> 294 (225); 300 after
// 8,000 1170 -> 344 (268); a verify of 9 after 16,000 2230 -> 48; 300 in a wrapped window 757 ->
// 227. Which KS: f32_plan (777 tokens with KS 4, 2, 1: 44, 69, 88; 2048: 337, 301, 294).
struct F32SplitParams {
  F32PrefillParams b;
  int n_parts, part_steps;  // parts of part_steps 64-key steps; 1: one part
  int skip_t0, skip_n;      // 64-key steps that hold only masked ring room (sink mode): left out
  float4* pws;              // [item][part][4 D / 32][64]: o slots
  float2* pml;              // [item][part][64]: (m, l) of each lane's row
};

template <bool ROLL, int KS>
__global__ __launch_bounds__(256, 1) void prefill_f32_split_kernel(F32SplitParams sp) {
  constexpr int D = 128, NQ = D / 8, NO = D / 32;
  constexpr int RG = 4 / KS;  // 32-row groups of the item
  __shared__ __align__(16) float4 lo[KS > 1 ? 4 : 1][4 * NO][64];
  __shared__ float2 lml[4][64];
  const F32PrefillParams& p = sp.b;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int n = lane & 31, hk = lane >> 5;
  const int rg = wave / KS, ks = wave % KS;  // the wave's rows, its share of the keys
  const LayerView& L = p.L;
  const int KV = L.kv_heads, G = p.G;
  // kv head fastest (an XCD's L2 serves few of them), then the part, heaviest query blocks first
  const int kvh = blockIdx.x % KV;
  const int part = blockIdx.x / KV % sp.n_parts;
  const int rank = blockIdx.x / (KV * sp.n_parts);
  const int qb = p.n_qblocks - 1 - rank;
  const int s0 = qb * p.QB;
  const int r0 = 32 * rg + n;
  const int qi = s0 + r0 / G, h = kvh * G + r0 % G;
  const bool row_ok = r0 < p.QB * G && qi < p.S;
  const int limit = row_ok ? p.pos_base + qi : -1;
  // the rows of this wave end at their last query (the whole item's part range is the last one's)
  const int item_q = min(s0 + p.QB, p.S) - 1;
  const int last_q = min(s0 + min((32 * rg + 31) / G, p.QB - 1), p.S - 1);
  const int first_q = s0 + 32 * rg / G;
  const int item_keys = p.n_scan_fixed > 0 ? p.n_scan_fixed : p.pos_base + item_q + 1;
  const int n_keys = p.n_scan_fixed > 0 ? p.n_scan_fixed : p.pos_base + last_q + 1;
  const int kmax = min(n_keys, p.phys_limit);
  const int steps_all = (n_keys + kF32KT - 1) / kF32KT - (ROLL ? 2 * sp.skip_n : 0);
  // first slot of a step
  auto slot0 = [&](int s) { return kF32KT * (ROLL && s >= 2 * sp.skip_t0 ? s + 2 * sp.skip_n : s); };
  const int first = 2 * part * sp.part_steps;
  const int end = sp.n_parts > 1 ? min(first + 2 * sp.part_steps, steps_all) : steps_all;
  if (first >= (item_keys + kF32KT - 1) / kF32KT - (ROLL ? 2 * sp.skip_n : 0)) return;  // a part past the item's range (the whole workgroup)

  float4 qv[NQ];
  {
    const float* qr = p.q + ((size_t)(row_ok ? qi : 0) * p.H + (row_ok ? h : 0)) * D + 4 * hk;
#pragma unroll
    for (int t = 0; t < NQ; t++) {
      const float4 x = *(const float4*)(qr + 8 * t);
      const float f = row_ok ? p.qscale : 0.0f;
      qv[t] = make_float4(x.x * f, x.y * f, x.z * f, x.w * f);
    }
  }
  const float* Kg = (const float*)L.k + (size_t)kvh * L.cap * D;
  const float* Vg = (const float*)L.v + (size_t)kvh * L.cap * D;
  float4 k[NQ], v[NO][4], cs[ROLL ? NQ / 2 : 1], sn[ROLL ? NQ / 2 : 1];
  auto load_k = [&](int step) {
    const int key = slot0(step) + n;
    const float* row = Kg + (size_t)key * D + 4 * hk;
#pragma unroll
    for (int t = 0; t < NQ; t++) k[t] = *(const float4*)(row + 8 * t);
    if constexpr (ROLL) {
      int Lg = L.ring.logical(key);
      Lg = key < p.phys_limit ? Lg : 0;
      long ri = (L.rope_abs && Lg >= L.ring.sinks) ? (long)Lg + L.evicted : (long)Lg;
      ri = ri < L.rope_positions ? ri : 0;
#pragma unroll
      for (int t = 0; t < NQ / 2; t++) {
        cs[t] = *(const float4*)(L.cos_tab + (size_t)ri * (D / 2) + 8 * t + 4 * hk);
        sn[t] = *(const float4*)(L.sin_tab + (size_t)ri * (D / 2) + 8 * t + 4 * hk);
      }
    }
  };
  auto load_v = [&](int step) {
    const float* vt = Vg + (size_t)slot0(step) * D + hk * (D * 8) + n * 8;
#pragma unroll
    for (int b = 0; b < NO; b++) {
      v[b][0] = *(const float4*)(vt + 256 * b);
      v[b][1] = *(const float4*)(vt + 256 * b + 4);
      v[b][2] = *(const float4*)(vt + 2 * (D * 8) + 256 * b);
      v[b][3] = *(const float4*)(vt + 2 * (D * 8) + 256 * b + 4);
    }
  };

  floatx16 o[NO];
#pragma unroll
  for (int b = 0; b < NO; b++)
#pragma unroll
    for (int i = 0; i < 16; i++) o[b][i] = 0.0f;
  float m = -1e30f, lsum = 0.0f;
  int step = first + ks;
  if (step < end) {
    load_k(step);
    load_v(step);
  }
  for (; step < end; step += KS) {
    const int next = step + KS < end ? step + KS : step;
    const int j0 = slot0(step);
    if constexpr (ROLL) {
      // k_d cos + rot_d sin, rot = -k_{d+D/2} (d < D/2) or k_{d-D/2}: two rounded products and a
      // rounded sum, not fused (attention_sg_roll.wgsl:40-51)
#pragma unroll
      for (int t = 0; t < NQ / 2; t++) {
        float* a = &k[t].x;
        float* b = &k[t + NQ / 2].x;
        const float* c = &cs[t].x;
        const float* z = &sn[t].x;
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const float x = a[e], y = b[e];
          a[e] = add_rn(mul_rn(x, c[e]), mul_rn(-y, z[e]));
          b[e] = add_rn(mul_rn(y, c[e]), mul_rn(x, z[e]));
        }
      }
    }
    floatx16 s0v, s1v;
#pragma unroll
    for (int i = 0; i < 16; i++) s0v[i] = s1v[i] = 0.0f;
#pragma unroll
    for (int t = 0; t < NQ; t++) {
      floatx16& acc = (t & 1) ? s1v : s0v;
      acc = __builtin_amdgcn_mfma_f32_32x32x2f32(k[t].x, qv[t].x, acc, 0, 0, 0);
      acc = __builtin_amdgcn_mfma_f32_32x32x2f32(k[t].y, qv[t].y, acc, 0, 0, 0);
      acc = __builtin_amdgcn_mfma_f32_32x32x2f32(k[t].z, qv[t].z, acc, 0, 0, 0);
      acc = __builtin_amdgcn_mfma_f32_32x32x2f32(k[t].w, qv[t].w, acc, 0, 0, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
    load_k(next);
    __builtin_amdgcn_sched_barrier(0);
    // register e holds key 8 (e / 4) + 4 hk + e % 4 of this lane's row
    float sv[16];
    float mt = -INFINITY;
    bool masked;
    if (!ROLL || L.ring.head == 0) {
      masked = j0 + kF32KT > min(kmax, p.pos_base + first_q + 1);
    } else {  // the newest logical slot sits just before the oldest; elsewhere slots ascend
      const int last = j0 + kF32KT - 1, newest = L.ring.sinks + L.ring.head - 1;
      const int top = j0 <= newest && newest <= last ? L.ring.sinks + L.ring.W - 1 : L.ring.logical(last);
      masked = last >= kmax || top > p.pos_base + first_q;
    }
#pragma unroll
    for (int e = 0; e < 16; e++) sv[e] = s0v[e] + s1v[e];
    if (masked) {
#pragma unroll
      for (int e = 0; e < 16; e++) {
        const int P = j0 + 8 * (e >> 2) + 4 * hk + (e & 3);
        const int Lg = ROLL ? L.ring.logical(P) : P;
        sv[e] = P < kmax && Lg <= limit ? sv[e] : -INFINITY;
      }
    }
#pragma unroll
    for (int e = 0; e < 16; e++) mt = fmaxf(mt, sv[e]);
    {
      const float2 pr = pair32(mt);
      mt = fmaxf(pr.x, pr.y);
    }
    // the reference maximum is raised only when a step's maximum exceeds it by more than 8 (log2
    // units: probabilities stay below 2^8), so most steps leave O and l unscaled
    if (__any(mt > m + 8.0f)) {
      const float mn = fmaxf(m, mt);
      const float corr = __builtin_amdgcn_exp2f(m - mn);
      m = mn;
      lsum *= corr;
#pragma unroll
      for (int b = 0; b < NO; b++)
#pragma unroll
        for (int i = 0; i < 16; i++) o[b][i] *= corr;
    }
    float ps = 0.0f;
    floatx16 pv;
#pragma unroll
    for (int e = 0; e < 16; e++) {
      pv[e] = __builtin_amdgcn_exp2f(sv[e] - m);
      ps += pv[e];
    }
    {
      const float2 pr = pair32(ps);
      ps = pr.x + pr.y;
    }
    lsum += ps;
    if (j0 + kF32KT > kmax) {
      // slots past the last valid one count as 0 (their probabilities are 0; 0 * garbage could be NaN)
#pragma unroll
      for (int e = 0; e < 16; e++)
        if (j0 + 8 * (e >> 2) + 4 * hk + (e & 3) >= kmax) {
#pragma unroll
          for (int b = 0; b < NO; b++) (&v[b][e >> 2].x)[e & 3] = 0.0f;
        }
    }
    // PV: dim block b, MFMA e takes key slot e of this lane's panel pair
#pragma unroll
    for (int e = 0; e < 16; e++)
#pragma unroll
      for (int b = 0; b < NO; b++)
        o[b] = __builtin_amdgcn_mfma_f32_32x32x2f32((&v[b][e >> 2].x)[e & 3], pv[e], o[b], 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
    load_v(next);
    __builtin_amdgcn_sched_barrier(0);
  }

  // the row group's waves meet in LDS; each then owns every KS-th dim block
  float M = m, lt = lsum, w[KS];
  if constexpr (KS > 1) {
    lml[wave][lane] = make_float2(m, lsum);
#pragma unroll
    for (int b = 0; b < NO; b++)
#pragma unroll
      for (int e4 = 0; e4 < 4; e4++)
        lo[wave][4 * b + e4][lane] = make_float4(o[b][4 * e4], o[b][4 * e4 + 1], o[b][4 * e4 + 2], o[b][4 * e4 + 3]);
    __syncthreads();
    M = -INFINITY;
    lt = 0.0f;
#pragma unroll
    for (int q = 0; q < KS; q++) M = fmaxf(M, lml[rg * KS + q][lane].x);
#pragma unroll
    for (int q = 0; q < KS; q++) {
      const float2 x = lml[rg * KS + q][lane];
      w[q] = __builtin_amdgcn_exp2f(x.x - M);
      lt += x.y * w[q];
    }
  }
  const size_t pi = ((size_t)(rank * KV + kvh) * sp.n_parts + part) * RG + rg;
#pragma unroll
  for (int i = 0; i < NO / KS; i++) {
    const int b = KS > 1 ? KS * i + ks : i;
    float4 r[4];
#pragma unroll
    for (int e4 = 0; e4 < 4; e4++) {
      if constexpr (KS > 1) {
        r[e4] = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
        for (int q = 0; q < KS; q++) {
          const float4 x = lo[rg * KS + q][4 * b + e4][lane];
          r[e4].x += x.x * w[q];
          r[e4].y += x.y * w[q];
          r[e4].z += x.z * w[q];
          r[e4].w += x.w * w[q];
        }
      } else {
        r[e4] = make_float4(o[i][4 * e4], o[i][4 * e4 + 1], o[i][4 * e4 + 2], o[i][4 * e4 + 3]);
      }
    }
    if (sp.n_parts > 1) {
#pragma unroll
      for (int e4 = 0; e4 < 4; e4++) sp.pws[(pi * 4 * NO + 4 * b + e4) * 64 + lane] = r[e4];
    } else if (row_ok) {
      float* orow = p.out + ((size_t)qi * p.H + h) * D + 32 * b + 4 * hk;
      const float* grow = p.gate ? p.gate + ((size_t)qi * p.H + h) * p.gate_stride + 32 * b + 4 * hk : nullptr;
#pragma unroll
      for (int e4 = 0; e4 < 4; e4++) {
        float x[4] = {r[e4].x / lt, r[e4].y / lt, r[e4].z / lt, r[e4].w / lt};
        if (grow) {
#pragma unroll
          for (int u = 0; u < 4; u++) x[u] = x[u] / (1.0f + expf(-grow[8 * e4 + u]));
        }
        *(float4*)(orow + 8 * e4) = make_float4(x[0], x[1], x[2], x[3]);
      }
    }
  }
  if (sp.n_parts > 1 && ks == 0) sp.pml[pi * 64 + lane] = make_float2(M, lt);
}

// One 32-key step and at most 96 rows a kv head (a first prompt of a few words): the kernel above, whose
// waves share the one step's K and V through LDS: 20 tokens, 16 heads on 8 9.2 us against 11.0, 32
// on 8 10.0 / 10.9; 128 rows 11.0 / 11.0, 136 11.2 / 10.9; two steps 14.3 / 11.2.
static bool f32_one_step(const LayerView& L, int S, int G, int pos_base) {
  return !(L.ring.roll && L.ring.head != 0) && pos_base + S <= kF32KT && S * G <= 96;
}

// The cheapest by a cost model in us. A step takes 3.8 us of a wave (a CU runs one workgroup); an
// item 2.5 to 4 before and after its steps. Where items are alike (a long context before the rows)
// the grid runs in whole rounds of the CUs, else its longest item or its share of a CU counts,
// whichever is more. Keys and values of a kv head past an XCD's L2 are read at about 5 TB/s for
// every item; a partial (16 KB and (m, l) a row group) is written and read at about 4.5 TB/s and
// the merge adds 5 us. Without room for a plan's partials (`floats` of them) the cheapest of one part:
// what is cheapest in many parts is not (200 rows of 16 heads on 4 after 9,000 keys: nine parts of 128
// rows, but in one part items of 32; captured without a buffer 1,155 -> 303 us).
F32Plan f32_plan(const LayerView& L, int S, int H, int pos_base, int cus, size_t floats) {
  F32Plan best{0, 0, 1, 0};
  const int G = H / L.kv_heads;
  if (L.D != 128 || G > 128 || f32_one_step(L, S, G, pos_base)) return best;
  const bool fixed = L.ring.roll && L.ring.head != 0;
  int skip_t0, skip_n;
  prefill_skip(L, S, pos_base, 64, &skip_t0, &skip_n);
  const int steps = ((fixed ? L.max_seq : pos_base + S) + 63) / 64 - skip_n;  // 64 keys each
  const float avg = fixed ? steps : (pos_base + 0.5f * S) / 64 + 0.25f;
  const bool alike = avg > 0.75f * steps;
  float bt = 0;
  for (int ks = 4; ks >= 1; ks /= 2) {
    const int rg = 4 / ks, QB = 32 * rg / G;
    if (QB < 1) continue;
    const int items = (S + QB - 1) / QB * L.kv_heads;
    auto item = [&](float s) { return 3.8f * (ks == 1 ? 2 * s : 2 * s / ks + 0.4f) + (ks == 1 ? 2.5f : 4.0f); };
    // (beyond four rounds of the CUs nothing is left to fill)
    const int most = std::min(std::min(std::max(1, steps / 2), 4 * cus / items), (int)(floats / ((size_t)items * rg * 4096)));
    for (int np = 1; np <= std::max(1, most) && (np == 1 || (size_t)items * rg * np * 512 <= kPfSplitMlBytes); np++) {
      const int ps = (steps + np - 1) / np;
      if ((steps + ps - 1) / ps != np) continue;
      float t = alike ? (items * np + cus - 1) / cus * item((float)ps)
                      : std::max(item((float)ps), items * np * item(avg / np) / cus);
      if (steps > 64) t = std::max(t, items * avg * 65536 / 5e6f);
      if (np > 1) t += items * rg * np * 0.0073f + 5.0f;
      if (best.QB == 0 || t < bt) {
        bt = t;
        best = F32Plan{ks, QB, np, ps};
      }
    }
  }
  return best;
}

size_t f32_prefill_floats(const LayerView& L, int S, int H, int pos_base, int cus) {
  const F32Plan f = f32_plan(L, S, H, pos_base, cus, kPfSplitBytes / sizeof(float));
  return f.QB && f.n_parts > 1 ? (size_t)((S + f.QB - 1) / f.QB) * L.kv_heads * f.n_parts * (4 / f.ks) * 4096 : 0;
}

template <int KS>
static hipError_t launch_pf32_split(const F32SplitParams& sp, hipStream_t st) {
  const dim3 g(sp.b.n_qblocks * sp.b.L.kv_heads * sp.n_parts);
  if (sp.b.L.ring.roll) hipLaunchKernelGGL((prefill_f32_split_kernel<true, KS>), g, dim3(256), 0, st, sp);
  else hipLaunchKernelGGL((prefill_f32_split_kernel<false, KS>), g, dim3(256), 0, st, sp);
  return hipGetLastError();
}

// workgroups of an instantiation a CU holds at once (its LDS allowance set first), per kernel
template <int D, bool ROLL>
static hipError_t pf32_resident(int* out) {
  static std::mutex mu;
  static int resident = 0;
  std::lock_guard<std::mutex> lock(mu);
  if (resident == 0) {
    const void* fn = (const void*)prefill_f32_kernel<D, ROLL>;
    hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)F32Smem<D>::bytes);
    if (e != hipSuccess) return e;
    int nb = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, fn, 256, F32Smem<D>::bytes) != hipSuccess || nb < 1) {
      (void)hipGetLastError();
      nb = 1;
    }
    resident = nb;
  }
  *out = resident;
  return hipSuccess;
}

template <int D, bool ROLL>
static hipError_t launch_pf32(F32PrefillParams p, int grid, int cus, hipStream_t st) {
  int resident = 1;
  const hipError_t e = pf32_resident<D, ROLL>(&resident);
  if (e != hipSuccess) return e;
  // two or more workgroups a CU and a grid held at once: pair heavy and light items on a CU;
  // otherwise heaviest first (the dispatcher hands each freed CU the next, lighter item)
  p.mirror = (resident >= 2 && grid <= resident * cus) ? 1 : 0;
  hipLaunchKernelGGL((prefill_f32_kernel<D, ROLL>), dim3(grid), dim3(256), F32Smem<D>::bytes, st, p);
  return hipGetLastError();
}

hipError_t launch_attention_f32(const LayerView& L, const AttnArgs& a, hipStream_t st) {
  F32PrefillParams p;
  p.L = L;
  p.q = a.q;
  p.S = a.S;
  p.H = a.H;
  p.G = a.H / L.kv_heads;
  p.QB = kF32Rows / p.G;
  if (p.QB < 1) return hipErrorInvalidValue;  // more than 128 heads per kv head
  p.pos_base = a.pos_base;
  p.qscale = a.scale * 1.4426950408889634f;
  p.gate = a.gate;
  p.gate_stride = a.gate_stride;
  p.out = a.out;
  p.n_scan_fixed = (L.ring.roll && L.ring.head != 0) ? L.max_seq : 0;
  p.phys_limit = L.ring.roll ? L.max_seq : L.cap;
  p.n_qblocks = (a.S + p.QB - 1) / p.QB;
  const size_t room = a.pf_o && a.pf_ml ? std::min(a.pf_floats, kPfSplitBytes / sizeof(float)) : 0;
  const F32Plan f = f32_plan(L, a.S, a.H, a.pos_base, a.num_cus > 0 ? a.num_cus : 256, room);
  if (f.QB) {
    F32SplitParams sp;
    p.QB = f.QB;
    p.n_qblocks = (a.S + f.QB - 1) / f.QB;
    p.mirror = 0;
    sp.n_parts = f.n_parts;
    sp.part_steps = f.part_steps;
    prefill_skip(L, a.S, a.pos_base, 64, &sp.skip_t0, &sp.skip_n);
    sp.pws = (float4*)a.pf_o;
    sp.pml = (float2*)a.pf_ml;
    sp.b = p;
    const hipError_t e = f.ks == 4 ? launch_pf32_split<4>(sp, st) : f.ks == 2 ? launch_pf32_split<2>(sp, st) : launch_pf32_split<1>(sp, st);
    if (e != hipSuccess || sp.n_parts == 1) return e;
    return launch_prefill_merge(L, a, f.QB, sp.n_parts, sp.part_steps, 4 / f.ks, p.n_scan_fixed, sp.skip_n, st);
  }
  const int grid = p.n_qblocks * L.kv_heads;
  const int cus = a.num_cus > 0 ? a.num_cus : 256;
  p.mirror = 0;
  const bool roll = L.ring.roll != 0;
  if (L.D == 128 && f.ks == 0) return roll ? launch_pf32<128, true>(p, grid, cus, st) : launch_pf32<128, false>(p, grid, cus, st);
  if (L.D == 256) return roll ? launch_pf32<256, true>(p, grid, cus, st) : launch_pf32<256, false>(p, grid, cus, st);
  return hipErrorInvalidValue;
}

}  // namespace bg
