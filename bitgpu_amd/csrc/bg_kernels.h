// Host-side launchers of the gfx950 kernels (defined in the .hip files, called by bg_api.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "bg_common.h"

namespace bg {

// One layer's device buffers plus the geometry the kernels need.
struct LayerView {
  void* k;            // K data
  void* v;            // V data (transposed 32-slot tiles)
  float* ks;          // q8 K scales (nullptr otherwise)
  float* vs;          // q8 V scales
  int cap;            // physical slots (multiple of 32)
  int kv_heads;
  int D;
  int dtype;          // KvType
  Ring ring;
  int max_seq;
  // read-time rotation (sink mode)
  const float* cos_tab;
  const float* sin_tab;
  int rope_positions;
  int rope_abs;       // 1: rotate by absolute position (slot + evicted for slots >= sinks)
  int64_t evicted;    // rows dropped by eviction so far
  int q8_row;         // q8 writes: 1 = one scale per row (its maximum, stored in every 32-value
                      // scale slot), 0 = one scale per 32 values
};

// kv_pack.hip
hipError_t launch_kv_write(const LayerView& L, int which, const float* src, int rows, int dst_row0,
                           hipStream_t st);
hipError_t launch_kv_export(const LayerView& L, int region, int base, int count, void* dst, hipStream_t st);
hipError_t launch_kv_import(const LayerView& L, int region, int base, int count, const void* src, hipStream_t st);
// logical positions [p0, p1) of a layer to or from buf (pinned host memory): K rows, V rows, q8 K
// and V scales, each region in reference order, kv_position_bytes a position in all
size_t kv_position_bytes(const LayerView& L);
hipError_t launch_kv_stage(const LayerView& L, int p0, int p1, void* buf, bool import_, hipStream_t st);
// f16 copy of slots [0, n_slots) (n_slots a multiple of 32) of a q8 or sink-mode layer, laid out
// like an f16 cache of the same capacity, with the prefill staging's exact values: q8 dequantized,
// sink-mode keys rotated at their slot's position. An f16 layer's V is not copied (vdst unused).
hipError_t launch_kv_prefill_copy(const LayerView& L, int n_slots, void* kdst, void* vdst, hipStream_t st);

// norm_rope.hip
struct PrologueArgs {
  const float* q; int q_stride;
  const float* k; const float* v;
  int S, H;
  const float* q_gamma; const float* k_gamma; float eps;
  const float* cos_tab; const float* sin_tab; int rot_dim;
  int pos0, slot0;
  float* q_out;
};
hipError_t launch_qkv_prologue(const LayerView& L, const PrologueArgs& a, hipStream_t st);

// gemv.hip: 1-bit decode projections. Row n, weight k = bit k % 32 of sign[n][k / 32] (set =
// +1) times scales[n][k / 128]; K a multiple of 128.
struct GemvArgs {
  const float* x; int K;
  const uint32_t* sign; const float* scales;
  int N0, N1, N2;                  // rows [0, N0) -> out0, [N0, N0+N1) -> out1, the rest -> out2
  float* out0; float* out1; float* out2;
  const float* resid;              // nullable: added to every output (the residual form)
};
hipError_t launch_gemv(const GemvArgs& a, hipStream_t st);
// fused decode qkv projection + prologue over the rows of H query heads, then KV key and KV
// value heads of the cache's head_dim
struct QkvProjArgs {
  const float* x; int K;
  const uint32_t* sign; const float* scales;
  int H;
  const float* q_gamma; const float* k_gamma; float eps;
  const float* cos_tab; const float* sin_tab; int rot_dim;
  int pos, slot;
  float* q_out;                    // [H, D] normed, roped rows
  float* raw;                      // [H + 2 KV][D] raw rows a head's finishing workgroup gathers;
                                   // every value the empty marker (kWorkspaceEmpty) between launches
  unsigned* err;                   // host-visible error word: a finisher's bounded wait gave up
  int spin_limit;                  // poll rounds before a finisher gives up (0: 2^20)
  int n_xcd;                       // > 0: workgroups go to XCDs round robin (see AttnArgs)
};
// raw-row floats the fused projection's gather buffer holds (heads of every kind x head_dim)
size_t qkv_proj_raw_floats(int heads, int D);
// Arrival counters (the f32 decode's, per kv head) sit 256 bytes apart: many workgroups' atomics on
// counters packed into two lines serialize.
constexpr int kCounterStride = 64;
hipError_t launch_qkv_proj(const LayerView& L, const QkvProjArgs& a, hipStream_t st);

// attention (decode.hip, attn_f32.hip, prefill.hip)
struct AttnArgs {
  const float* q;
  int S, H;
  int pos_base;
  float scale;
  const float* gate; int gate_stride;
  float* out;
  // split-K workspace
  float* ws_o; float* ws_ml; unsigned* ws_count; size_t ws_floats;
  // split-K prefill: the partials (pf_floats long) and their (m, l), kPfSplitMlBytes long; a launch
  // whose plan needs more than is there scans whole key ranges
  float* pf_o; float* pf_ml; size_t pf_floats;
  int k_rotated;   // prefill, sink mode: the layer's keys are already rotated (the f16 copy)
  int num_cus;
  // decode merge: host-visible error word, poll bound (0: default) and a test hook that makes
  // one split store no partial (-1: none)
  unsigned* err; int spin_limit; int withhold_split;
  // XCDs the GPU dispatches workgroups to round robin (workgroup b on XCD (b + r) mod n_xcd, r
  // the same for the whole grid; checked on the device once): the decode kernel then exchanges
  // split partials through one XCD's L2. 0: partials are written through to memory.
  int n_xcd;
};
// workgroup placement check of the current device: n_xcd > 0 when a probe grid's workgroups all
// ran on XCD (blockIdx + r) mod n_xcd for one r (decode.hip)
hipError_t probe_xcd_round_robin(int* n_xcd);
hipError_t launch_attention_f32(const LayerView& L, const AttnArgs& a, hipStream_t st);
// split-K f32 decode / verify (G*S <= 16 rows per kv head), workspace as for the decode kernel
hipError_t launch_attention_f32_split(const LayerView& L, const AttnArgs& a, hipStream_t st);
bool f32_split_supported(const LayerView& L, int S, int H);
size_t f32_workspace_floats(const LayerView& L, int S, int H);
hipError_t launch_attention_decode(const LayerView& L, const AttnArgs& a, hipStream_t st);
hipError_t launch_attention_prefill(const LayerView& L, const AttnArgs& a, hipStream_t st);
// workspace floats needed by the decode kernel for S rows of H heads; a new workspace is filled
// with the 32-bit pattern decode_workspace_empty() before its first use
size_t decode_workspace_floats(const LayerView& L, int S, int H, int num_cus, size_t* counters);
uint32_t decode_workspace_empty();
// floats of the split partials one decode launch with n_splits splits per kv head writes
size_t decode_partial_floats(const LayerView& L, int S, int H, int n_splits);
bool decode_supported(const LayerView& L, int S, int H);
// the dispatch: decode kernel (true) or prefill kernel for S rows of H heads. Decode takes every
// shape whose rows per kv head fit one 16-row set, and every sink-mode shape it supports; more
// rows go to the (split-K) prefill, except q8 at head_dim 128 up to 24 rows (measured faster).
bool decode_preferred(const LayerView& L, int S, int H);
// the split-K plan of a decode launch (host-only arithmetic; false when the kernel does not take
// the shape). resident_per_cu: workgroups of the launch's instantiation a CU holds at once.
struct DecodePlan {
  int waves, nset, passes;
  int n_scan, phys_limit, n_tiles;
  int tiles_per_split, n_splits, n_mergers, grid;
  int xcd_group;  // > 0: splits numbered in groups of this many per kv head (sink mode), grid padded
  int skip_t0, skip_n;  // a run of whole tiles every row masks (sink mode), not scanned
};
bool decode_plan(const LayerView& L, int S, int H, int pos_base, int num_cus, int resident_per_cu, DecodePlan* out);
// streaming-read floor (diag.hip): `workgroups` contiguous slices of `bytes` read with 16-byte
// loads, one XOR word per workgroup into sink
hipError_t launch_stream_read(const void* buf, size_t bytes, int workgroups, bool nontemporal, unsigned* sink,
                              hipStream_t st);
bool prefill_supported(const LayerView& L, int S, int H);
// a q8 or sink-mode prefill of S rows that stages each K/V tile for enough query blocks to run faster
// on an f16 copy of the attended slots
bool prefill_wants_f16_copy(const LayerView& L, int S, int H);
// "not written yet" marker of a split partial slot: a quiet NaN with a payload arithmetic on
// finite inputs never produces. The decode kernel leaves every slot it uses holding it.
constexpr uint32_t kWorkspaceEmpty = 0x7FF1DE5Au;
// A split-K prefill plan's largest partials: 512 workgroups of 64 KB at head_dim 128, 256 of 128 KB
// at 256 (one round of a 256-CU GPU), and 512 x 4 waves x 64 lanes of (m, l).
constexpr size_t kPfSplitBytes = (size_t)32 << 20;
constexpr size_t kPfSplitMlBytes = (size_t)1 << 20;
constexpr int kPfMaxParts = 512;
// floats of the partials a prefill launch uses at pos_base (0: the launch does not split); whether
// S rows of H heads can split at any pos_base (the partials are then at most kPfSplitBytes)
size_t prefill_workspace_floats(const LayerView& L, int S, int H, int pos_base, int num_cus);
// merges the partials of `waves` 32-row waves an item, parts of part_steps 64-key (head_dim 128) or
// 32-key (256) steps
hipError_t launch_prefill_merge(const LayerView& L, const AttnArgs& a, int QB, int n_parts, int part_steps, int waves,
                                int n_scan_fixed, int skip_n, hipStream_t st);
// the KT-slot steps *t0 .. + *n - 1 of a wrapped ring that hold only slots past S rows at pos_base
void prefill_skip(const LayerView& L, int S, int pos_base, int KT, int* t0, int* n);
// The plan of an f32 prefill launch (host-only arithmetic): ks of a workgroup's four waves share 32
// rows and take every ks-th 32-key step (4 / ks row groups an item), QB queries an item, n_parts
// parts of part_steps 64-key steps, at most `floats` floats of partials. ks = QB = 0: the kernel of
// 128-row items staged through LDS (a single step of few rows; head_dim 256, whose K, V, Q and O a step
// would not fit a wave's registers).
struct F32Plan {
  int ks, QB, n_parts, part_steps;
};
F32Plan f32_plan(const LayerView& L, int S, int H, int pos_base, int cus, size_t floats);
// floats of the partials an f32 prefill uses at pos_base (0: none)
size_t f32_prefill_floats(const LayerView& L, int S, int H, int pos_base, int num_cus);
bool prefill_can_split(const LayerView& L, int S, int H, int num_cus);

}  // namespace bg
