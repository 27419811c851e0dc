// KV-cache append (the copy / copy_kv16 / copy_kv8 equivalents) and the snapshot-layout
// export/import gathers.
//
// kv_write: one wave per cache row of D values. Lane l owns D/64 consecutive values, so a q8
// block of 32 values is held by 32/(D/64) adjacent lanes and its absolute maximum is a
// shuffle reduction inside that lane group (shaders/copy_kv8.wgsl:25-36 does the same with a
// shared-memory pass). Rows follow the reference's cache-row numbering (src/engine.ts:1385-1393):
// reference row R = position * KV + kv_head.
#include "bg_kernels.h"
#include "bg_store.h"

namespace bg {

template <int D, int DT>
__global__ __launch_bounds__(64) void kv_write_kernel(LayerView L, int which, const float* __restrict__ src,
                                                      int rows, int dst_row0) {
  constexpr int EPL = D / 64;               // values per lane
  const int r = blockIdx.x;
  if (r >= rows) return;
  const int lane = threadIdx.x;
  const int R = dst_row0 + r;
  const int pos = R / L.kv_heads, kvh = R % L.kv_heads;
  const float* x = src + (size_t)r * D + lane * EPL;
  float v[EPL];
#pragma unroll
  for (int e = 0; e < EPL; e++) v[e] = x[e];
  store_row<D, DT>(L, which, L.ring.phys(pos), kvh, v, lane);
}

template <int D>
static hipError_t kv_write_d(const LayerView& L, int which, const float* src, int rows, int dst_row0, hipStream_t st) {
  dim3 g(rows), b(64);
  switch (L.dtype) {
    case KV_F32: hipLaunchKernelGGL((kv_write_kernel<D, KV_F32>), g, b, 0, st, L, which, src, rows, dst_row0); break;
    case KV_F16: hipLaunchKernelGGL((kv_write_kernel<D, KV_F16>), g, b, 0, st, L, which, src, rows, dst_row0); break;
    default: hipLaunchKernelGGL((kv_write_kernel<D, KV_Q8>), g, b, 0, st, L, which, src, rows, dst_row0); break;
  }
  return hipGetLastError();
}

hipError_t launch_kv_write(const LayerView& L, int which, const float* src, int rows, int dst_row0, hipStream_t st) {
  if (rows <= 0) return hipSuccess;
  // head_dim is 128 or 256 (bg_kv_create rejects the rest)
  switch (L.D) {
    case 128: return kv_write_d<128>(L, which, src, rows, dst_row0, st);
    default: return kv_write_d<256>(L, which, src, rows, dst_row0, st);
  }
}

// ---- snapshot layout gathers: region element e of [count, KV, n] in reference order ----------
// region 0/1: K/V elements (f32 / f16 bits / int8 codes); 2/3: K/V block scales.
__global__ void kv_export_kernel(LayerView L, int region, int base, int count, void* __restrict__ dst, int import_) {
  const int D = L.D;
  const int n = region < 2 ? D : D / kBlock;
  const size_t total = (size_t)count * L.kv_heads * n;
  for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < total; e += (size_t)gridDim.x * blockDim.x) {
    const int i = (int)(e % n);
    const size_t rowi = e / n;
    const int kvh = (int)(rowi % L.kv_heads);
    const int pos = base + (int)(rowi / L.kv_heads);
    const int slot = L.ring.phys(pos);
    if (region >= 2) {
      float* sc = region == 2 ? L.ks : L.vs;
      size_t off = scale_offset(kvh, slot, i, L.cap, D);
      if (import_) sc[off] = ((const float*)dst)[e];
      else ((float*)dst)[e] = sc[off];
      continue;
    }
    size_t off = region == 0 ? k_offset(kvh, slot, i, L.cap, D) : v_offset(kvh, slot, i, L.cap, D);
    void* buf = region == 0 ? L.k : L.v;
    if (L.dtype == KV_F32) {
      if (import_) ((float*)buf)[off] = ((const float*)dst)[e];
      else ((float*)dst)[e] = ((const float*)buf)[off];
    } else if (L.dtype == KV_F16) {
      if (import_) ((uint16_t*)buf)[off] = ((const uint16_t*)dst)[e];
      else ((uint16_t*)dst)[e] = ((const uint16_t*)buf)[off];
    } else {
      if (import_) ((int8_t*)buf)[off] = ((const int8_t*)dst)[e];
      else ((int8_t*)dst)[e] = ((const int8_t*)buf)[off];
    }
  }
}

hipError_t launch_kv_export(const LayerView& L, int region, int base, int count, void* dst, hipStream_t st) {
  if (count <= 0) return hipSuccess;
  hipLaunchKernelGGL(kv_export_kernel, dim3(1024), dim3(256), 0, st, L, region, base, count, dst, 0);
  return hipGetLastError();
}
hipError_t launch_kv_import(const LayerView& L, int region, int base, int count, const void* src, hipStream_t st) {
  if (count <= 0) return hipSuccess;
  hipLaunchKernelGGL(kv_export_kernel, dim3(1024), dim3(256), 0, st, L, region, base, count, const_cast<void*>(src), 1);
  return hipGetLastError();
}

// ---- a layer's positions [p0, p1) between the cache and a staging slot in host memory ----------
// buf (pinned host memory, mapped): the positions' K rows, V rows, then (q8) K and V scales, each
// in reference order. One launch a slot; 16 bytes a thread and access on the host side, so a wave
// moves 1 KB pieces over the bus, which bounds it (the V gather reads its transposed tiles from
// cache). A 1,003-position q8 snapshot of 36 layers, 83 MB:
// saved in 3.1 ms and restored in 2.7 (27 and 31 GB/s), by a call and a staged copy a region 20 ms each.
template <int EB, bool IMPORT>
__global__ __launch_bounds__(256) void kv_stage_kernel(LayerView L, int p0, int p1, char* __restrict__ buf) {
  typedef uint32_t u4 __attribute__((ext_vector_type(4)));
  const int D = L.D, KV = L.kv_heads;
  const size_t rows = (size_t)(p1 - p0) * KV;
  const int cd = D * EB / 16, cs = L.dtype == KV_Q8 ? D / kBlock / 4 : 0;  // 16-byte pieces of a row
  const size_t total = rows * 2 * (cd + cs);
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (size_t)gridDim.x * blockDim.x) {
    u4* host = (u4*)buf + i;
    size_t j = i;
    int region = 0;
    if (j >= rows * 2 * cd) {
      j -= rows * 2 * cd;
      region = 2 + (j >= rows * cs);
      j -= region == 3 ? rows * cs : 0;
    } else if (j >= rows * cd) {
      j -= rows * cd;
      region = 1;
    }
    const int per = region < 2 ? cd : cs;
    const int c = (int)(j % per), kvh = (int)(j / per % KV);
    const int slot = L.ring.phys(p0 + (int)(j / per / KV));
    if (region == 1) {
      constexpr int N = 16 / EB;
      union { u4 u; uint8_t b[16]; uint16_t h[8]; uint32_t w[4]; } x;
      if constexpr (IMPORT) x.u = __builtin_nontemporal_load(host);
      const size_t off = v_offset(kvh, slot, N * c, L.cap, D);  // the next dim is 8 elements on
#pragma unroll
      for (int e = 0; e < N; e++) {
        if constexpr (EB == 1) {
          if constexpr (IMPORT) ((uint8_t*)L.v)[off + 8 * e] = x.b[e];
          else x.b[e] = ((const uint8_t*)L.v)[off + 8 * e];
        } else if constexpr (EB == 2) {
          if constexpr (IMPORT) ((uint16_t*)L.v)[off + 8 * e] = x.h[e];
          else x.h[e] = ((const uint16_t*)L.v)[off + 8 * e];
        } else {
          if constexpr (IMPORT) ((uint32_t*)L.v)[off + 8 * e] = x.w[e];
          else x.w[e] = ((const uint32_t*)L.v)[off + 8 * e];
        }
      }
      if constexpr (!IMPORT) __builtin_nontemporal_store(x.u, host);
      continue;
    }
    u4* dev = region == 0 ? (u4*)((char*)L.k + k_offset(kvh, slot, 0, L.cap, D) * EB) + c
                          : (u4*)((region == 2 ? L.ks : L.vs) + scale_offset(kvh, slot, 0, L.cap, D)) + c;
    if constexpr (IMPORT) *dev = __builtin_nontemporal_load(host);
    else __builtin_nontemporal_store(*dev, host);
  }
}

size_t kv_position_bytes(const LayerView& L) {
  const size_t eb = kv_elem_bytes(L.dtype);
  return 2 * (size_t)L.kv_heads * (L.D * eb + (L.dtype == KV_Q8 ? L.D / kBlock * sizeof(float) : 0));
}

hipError_t launch_kv_stage(const LayerView& L, int p0, int p1, void* buf, bool import_, hipStream_t st) {
  const size_t pieces = (size_t)(p1 - p0) * kv_position_bytes(L) / 16;
  const dim3 g((unsigned)((pieces + 255) / 256 < 2048 ? (pieces + 255) / 256 : 2048)), b(256);
  char* h = (char*)buf;
  switch (L.dtype) {
    case KV_Q8:
      if (import_) hipLaunchKernelGGL((kv_stage_kernel<1, true>), g, b, 0, st, L, p0, p1, h);
      else hipLaunchKernelGGL((kv_stage_kernel<1, false>), g, b, 0, st, L, p0, p1, h);
      break;
    case KV_F16:
      if (import_) hipLaunchKernelGGL((kv_stage_kernel<2, true>), g, b, 0, st, L, p0, p1, h);
      else hipLaunchKernelGGL((kv_stage_kernel<2, false>), g, b, 0, st, L, p0, p1, h);
      break;
    default:
      if (import_) hipLaunchKernelGGL((kv_stage_kernel<4, true>), g, b, 0, st, L, p0, p1, h);
      else hipLaunchKernelGGL((kv_stage_kernel<4, false>), g, b, 0, st, L, p0, p1, h);
  }
  return hipGetLastError();
}

// ---- f16 copy of the attended slots, for a long prefill ----------------------------------------
// A prefill stages every K/V tile once per query block that attends it. Where staging computes
// (q8: dequantize, sink mode: rotate the keys) and there are blocks enough, the attended slots are
// converted once here into a copy laid out like an f16 cache (K row-major, V in 32-slot
// transposed tiles), and the prefill copies its tiles from that straight into LDS. The values
// are exactly the staging's: q8 the code, biased to u = code + 128, times s = scale * (1/127) in
// one f32 fma (u * s - 128 * s); sink mode the pair (x, y) of dims (i, i + D/2) rotated at the
// slot's position in f32, every product and sum rounded; then RNE to f16. Bound by memory: each
// value read once and written once (4100 slots of 8 heads, f16 keys: 17 MB; 12,334 slots q8, K and
// V: 78 MB in 15 us).

template <int D, int DT, bool ROLL>
__global__ __launch_bounds__(256) void kv_prefill_copy_kernel(LayerView L, int n_slots, __half* __restrict__ kdst,
                                                              __half* __restrict__ vdst) {
  constexpr int NB = D / kBlock;
  const size_t per_head = (size_t)n_slots * D / 16;  // 16-value chunks of K (and of V) per kv head
  const size_t total = per_head * L.kv_heads;
  const size_t end = DT == KV_Q8 ? 2 * total : total;
  for (size_t c = (size_t)blockIdx.x * blockDim.x + threadIdx.x; c < end; c += (size_t)gridDim.x * blockDim.x) {
    const bool isv = DT == KV_Q8 && c >= total;
    const size_t cc = isv ? c - total : c;
    const int kvh = (int)(cc / per_head);
    const size_t e0 = (cc % per_head) * 16;  // element offset inside the kv head's region
    const size_t base = (size_t)kvh * L.cap * D;
    _Float16 o[16];
    if (!isv) {
      // 16 dims of one key: consecutive ones, or 8 and their rotation partners
      const int slot = (int)(e0 / D);
      const int d0 = ROLL ? (int)(e0 % D) / 2 : (int)(e0 % D), d1 = ROLL ? d0 + D / 2 : d0 + 8;
      float a[8], b[8];
      if constexpr (DT == KV_Q8) {
        const int8_t* row = (const int8_t*)L.k + base + (size_t)slot * D;
        const uint2 wa = *(const uint2*)(row + d0), wb = *(const uint2*)(row + d1);
        const float* ks = L.ks + ((size_t)kvh * L.cap + slot) * NB;
        const float sa = ks[d0 / kBlock] * (1.0f / 127.0f), sb = ks[d1 / kBlock] * (1.0f / 127.0f);
        const uint32_t ua[2] = {wa.x ^ 0x80808080u, wa.y ^ 0x80808080u}, ub[2] = {wb.x ^ 0x80808080u, wb.y ^ 0x80808080u};
#pragma unroll
        for (int i = 0; i < 8; i++) {
          a[i] = q8_stage_f32((ua[i >> 2] >> (8 * (i & 3))) & 0xffu, sa);
          b[i] = q8_stage_f32((ub[i >> 2] >> (8 * (i & 3))) & 0xffu, sb);
        }
      } else {
        const _Float16* row = (const _Float16*)L.k + base + (size_t)slot * D;
        const uint4 ha = *(const uint4*)(row + d0), hb = *(const uint4*)(row + d1);
#pragma unroll
        for (int i = 0; i < 8; i++) {
          a[i] = (float)((const _Float16*)&ha)[i];
          b[i] = (float)((const _Float16*)&hb)[i];
        }
      }
      if constexpr (ROLL) {
        const int Lg = slot < L.max_seq ? L.ring.logical(slot) : 0;
        long ri = (L.rope_abs && Lg >= L.ring.sinks) ? (long)Lg + L.evicted : (long)Lg;
        ri = ri < L.rope_positions ? ri : 0;  // a masked slot
        const float* ct = L.cos_tab + (size_t)ri * (D / 2) + d0;
        const float* st = L.sin_tab + (size_t)ri * (D / 2) + d0;
#pragma unroll
        for (int i = 0; i < 8; i++) {
          const float x = a[i], y = b[i], cv = ct[i], sv = st[i];
          a[i] = add_rn(mul_rn(x, cv), mul_rn(-y, sv));
          b[i] = add_rn(mul_rn(y, cv), mul_rn(x, sv));
        }
      }
#pragma unroll
      for (int i = 0; i < 8; i++) {
        o[i] = (_Float16)a[i];
        o[8 + i] = (_Float16)b[i];
      }
      __half* dst = kdst + base + (size_t)slot * D;
      *(uint4*)(dst + d0) = *(const uint4*)&o[0];
      *(uint4*)(dst + d1) = *(const uint4*)&o[8];
    } else {
      const uint4 w = *(const uint4*)((const int8_t*)L.v + base + e0);
      const uint32_t ww[4] = {w.x ^ 0x80808080u, w.y ^ 0x80808080u, w.z ^ 0x80808080u, w.w ^ 0x80808080u};
      // 16 bytes of a V tile = 2 dims x the 8 slots of one panel
      const int t = (int)(e0 / ((size_t)kTile * D));
      const int wi = (int)(e0 % ((size_t)kTile * D));
      const int panel = wi / (8 * D), d0 = (wi % (8 * D)) / 8;
#pragma unroll
      for (int h = 0; h < 2; h++) {
        const int d = d0 + h;
#pragma unroll
        for (int e = 0; e < 8; e++) {
          const int slot = t * kTile + tile_slot(panel, e);
          const float s = L.vs[((size_t)kvh * L.cap + slot) * NB + d / kBlock] * (1.0f / 127.0f);
          const int i = 8 * h + e;
          o[i] = q8_stage_f16((ww[i >> 2] >> (8 * (i & 3))) & 0xffu, s);
        }
      }
      uint4* dst = (uint4*)(vdst + base + e0);
      dst[0] = *(const uint4*)&o[0];
      dst[1] = *(const uint4*)&o[8];
    }
  }
}

hipError_t launch_kv_prefill_copy(const LayerView& L, int n_slots, void* kdst, void* vdst, hipStream_t st) {
  const bool q8 = L.dtype == KV_Q8, roll = L.ring.roll != 0;
  if (n_slots <= 0 || n_slots % kTile || n_slots > L.cap || (!q8 && !(L.dtype == KV_F16 && roll))) return hipErrorInvalidValue;
  const size_t chunks = (q8 ? 2 : 1) * (size_t)n_slots * L.D / 16 * L.kv_heads;
  const dim3 grid((unsigned)((chunks + 255) / 256 < 4096 ? (chunks + 255) / 256 : 4096)), block(256);
  __half *k = (__half*)kdst, *v = (__half*)vdst;
  if (L.D == 128) {
    if (!q8) hipLaunchKernelGGL((kv_prefill_copy_kernel<128, KV_F16, true>), grid, block, 0, st, L, n_slots, k, v);
    else if (roll) hipLaunchKernelGGL((kv_prefill_copy_kernel<128, KV_Q8, true>), grid, block, 0, st, L, n_slots, k, v);
    else hipLaunchKernelGGL((kv_prefill_copy_kernel<128, KV_Q8, false>), grid, block, 0, st, L, n_slots, k, v);
  } else {
    if (!q8) hipLaunchKernelGGL((kv_prefill_copy_kernel<256, KV_F16, true>), grid, block, 0, st, L, n_slots, k, v);
    else if (roll) hipLaunchKernelGGL((kv_prefill_copy_kernel<256, KV_Q8, true>), grid, block, 0, st, L, n_slots, k, v);
    else hipLaunchKernelGGL((kv_prefill_copy_kernel<256, KV_Q8, false>), grid, block, 0, st, L, n_slots, k, v);
  }
  return hipGetLastError();
}

}  // namespace bg
