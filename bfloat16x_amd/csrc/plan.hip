// Device builder of the overflow plan: what bf16x_plan_host (check = 1) does
// with a dict whose streams and table are already in device memory.
//
// Replaces the overflow preparation of Bf16xFused.__init__
// (bf16x_fused.py:165-182).  plan_count checks every table entry against the
// streams and counts the entries to keep (true delta > 7) per workgroup, a
// one-workgroup scan turns the counts into offsets and a total, and plan_write
// encodes the kept entries and the tile offsets.
//
// Bound: the gathers.  An entry reads its code, sign, mantissa and emax from
// four streams, and at one entry per ~38 elements nearly every cache line of
// them is touched (84 MB at 14336x4096).  Measured there (1.55 M entries):
// 13 + 4 + 16 us (15 + 4 + 18.5 with one entry of a thread in flight at a
// time), 48 us for the call with its one wait for the count; the host builder,
// which copies the streams back first, takes 30-40 ms.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/bf16x_hip.h"
#include "bf16x_device.h"
#include "launch_common.h"

namespace {
using namespace bf16x;

// A wave takes 64 * iters consecutive entries, a workgroup 4 such runs;
// iters keeps the workgroups at or below kMaxBlocks, 4 counts per thread of
// the scan.
constexpr int kMaxBlocks = 4096;
constexpr int kAhead = 2;
constexpr uint32_t kBad = 0x80000000u;     // of a workgroup's count: an entry failed its checks

struct PlanGrid {
  int64_t blocks;
  int iters;
};
PlanGrid plan_grid(int64_t n) {
  PlanGrid g;
  g.iters = (int)std::max<int64_t>(1, (n + 256 * (int64_t)kMaxBlocks - 1) / (256 * (int64_t)kMaxBlocks));
  g.blocks = (n + 256 * (int64_t)g.iters - 1) / (256 * (int64_t)g.iters);
  return g;
}

// nb bits at stream bit `bit` (the second word only when the field crosses)
__device__ __forceinline__ uint32_t field(const uint32_t* __restrict__ w, int64_t bit, int nb) {
  const int64_t wi = bit >> 5;
  const uint32_t sh = (uint32_t)(bit & 31);
  const uint32_t hi = (sh + nb > 32) ? w[wi + 1] : 0u;
  return alignbit(hi, w[wi], sh) & ((1u << nb) - 1u);
}

// entries strictly ascending inside [0, N), true delta in 7 .. emax, code 7
__global__ __launch_bounds__(256) void plan_count_kernel(const int32_t* __restrict__ idx,
                                                         const uint8_t* __restrict__ val, int64_t n, int iters,
                                                         const uint32_t* __restrict__ delta,
                                                         const uint8_t* __restrict__ emax, int64_t N,
                                                         uint32_t* __restrict__ blk_cnt) {
  __shared__ uint32_t red[4];
  const int64_t j0 = (int64_t)blockIdx.x * 256 * iters + threadIdx.x;
  uint32_t kept = 0;
  bool bad = false;
  // kAhead entries of a thread at a time: their table words, then their
  // gathers (the last code word's second word is only read when the field
  // crosses into it, so all reads stay inside the stream)
  for (int it = 0; it < iters; it += kAhead) {
    int64_t p[kAhead], prev[kAhead];
    int v[kAhead];
    bool in[kAhead], ok[kAhead];
#pragma unroll
    for (int k = 0; k < kAhead; ++k) {
      const int64_t j = j0 + 256 * (int64_t)(it + k);
      in[k] = it + k < iters && j < n;
      const int64_t jc = in[k] ? j : n - 1;
      p[k] = idx[jc];
      prev[k] = jc ? (int64_t)idx[jc - 1] : -1;
      v[k] = val[jc];
    }
    uint32_t code[kAhead], em[kAhead];
#pragma unroll
    for (int k = 0; k < kAhead; ++k) {
      ok[k] = p[k] > prev[k] && p[k] >= 0 && p[k] < N && v[k] >= 7;
      const int64_t pc = ok[k] ? p[k] : 0;
      code[k] = field(delta, pc * 3, 3);
      em[k] = emax[pc >> 4];
    }
#pragma unroll
    for (int k = 0; k < kAhead; ++k) {
      bad |= in[k] && !(ok[k] && code[k] == 7u && v[k] <= (int)em[k]);
      kept += in[k] && v[k] > 7 ? 1u : 0u;
    }
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) kept += __shfl_xor(kept, o, 64);
  const bool any = __ballot(bad) != 0;
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = kept | (any ? kBad : 0u);
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t s = 0, b = 0;
    for (int k = 0; k < 4; ++k) { s += red[k] & ~kBad; b |= red[k] & kBad; }
    blk_cnt[blockIdx.x] = s | b;
  }
}

// exclusive scan of the workgroup counts in place; n_fix[0] = the total, or -1
// when any workgroup found a bad entry
__global__ __launch_bounds__(1024) void plan_scan_kernel(uint32_t* __restrict__ cnt, int n_blk,
                                                         int64_t* __restrict__ n_fix) {
  __shared__ uint32_t part[16];
  __shared__ uint32_t badw[16];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  constexpr int kPer = kMaxBlocks / 1024;
  uint32_t c[kPer], own = 0, bad = 0;
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const int i = tid * kPer + k;
    const uint32_t v = i < n_blk ? cnt[i] : 0u;
    bad |= v & kBad;
    c[k] = v & ~kBad;
    own += c[k];
  }
  uint32_t total;
  uint32_t at = wave_prefix(own, lane, total);
  const bool any = __ballot(bad != 0) != 0;
  if (lane == 0) {
    part[wv] = total;
    badw[wv] = any ? 1u : 0u;
  }
  __syncthreads();
  uint32_t allbad = 0;
  for (int k = 0; k < 16; ++k) allbad |= badw[k];
  for (int k = 0; k < wv; ++k) at += part[k];
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const int i = tid * kPer + k;
    if (i < n_blk) cnt[i] = at;
    at += c[k];
  }
  if (tid == 1023) n_fix[0] = allbad ? -1 : (int64_t)at;
}

// Kept entries in table order, and the offset of every tile whose first entry
// (kept or not) is this one: tiles after the previous entry's up to its own.
// A checked table only (strictly ascending, in range).
__global__ __launch_bounds__(256) void plan_write_kernel(
    const int32_t* __restrict__ idx, const uint8_t* __restrict__ val, int64_t n, int iters,
    const uint32_t* __restrict__ blk_off, const uint32_t* __restrict__ sign, const uint32_t* __restrict__ mant,
    const uint8_t* __restrict__ emax, uint32_t in_f, uint32_t tpr, int64_t n_tiles, int64_t n_fix,
    uint32_t* __restrict__ tile_off, uint32_t* __restrict__ ent, uint8_t* __restrict__ sat) {
  __shared__ uint32_t part[2][4];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  auto tile_of = [&](uint32_t p, uint32_t& col) {
    const uint32_t row = p / in_f, c = p - row * in_f;
    col = c & (kPlanTileCols - 1);
    return (int64_t)row * tpr + (c >> 16);
  };
  uint32_t base = blk_off[blockIdx.x];
  // entry j's table words; the next iteration's are requested ahead, and an
  // entry's gathers before the barrier that ranks it
  const int64_t j0 = (int64_t)blockIdx.x * iters * 256 + threadIdx.x;
  uint32_t p = 0, prev = 0;
  int v = 0;
  auto load = [&](int64_t j, uint32_t& pj, uint32_t& pv, int& vj) {
    const int64_t jc = min(j, n - 1);
    pj = (uint32_t)idx[jc];
    pv = (uint32_t)idx[jc ? jc - 1 : 0];
    vj = j < n ? val[jc] : 0;
  };
  load(j0, p, prev, v);
  for (int it = 0; it < iters; ++it) {
    const int64_t j = j0 + 256 * (int64_t)it;
    const bool in = j < n;
    const bool keep = v > 7;
    const uint32_t s = field(sign, p, 1), m = field(mant, (int64_t)p * 7, 7);
    const int em = emax[p >> 4];
    uint32_t pn, prevn;
    int vn;
    load(it + 1 < iters ? j + 256 : n, pn, prevn, vn);
    const uint64_t b = __ballot(keep);
    const uint32_t before = (uint32_t)__builtin_popcountll(b & ((1ull << lane) - 1ull));
    if (lane == 0) part[it & 1][wave] = (uint32_t)__builtin_popcountll(b);
    __syncthreads();                       // (two buffers: one barrier per iteration)
    uint32_t o = base + before, all = 0;
    for (int k = 0; k < 4; ++k) {
      const uint32_t c = part[it & 1][k];
      if (k < wave) o += c;
      all += c;
    }
    base += all;
    uint32_t col = 0, pcol;
    const int64_t t = in ? tile_of(p, col) : -1;
    const int64_t t0 = in ? (j ? tile_of(prev, pcol) + 1 : 0) : 0;
    // a long run of empty tiles is written by the whole wave
    const int64_t gap = in ? t - t0 + 1 : 0;
    for (uint64_t m = __ballot(gap > 16); m; m &= m - 1) {
      const int src = __builtin_ctzll(m);
      const int64_t g0 = __shfl(t0, src, 64), g1 = __shfl(t, src, 64);
      const uint32_t gv = __shfl(o, src, 64);
      for (int64_t k = g0 + lane; k <= g1; k += 64) tile_off[k] = gv;
    }
    if (gap <= 16)
      for (int64_t k = t0; k < t0 + gap; ++k) tile_off[k] = o;
    if (const uint64_t m = __ballot(j == n - 1)) {             // and the tiles after the table's last entry
      const int64_t tl = __shfl(t, __builtin_ctzll(m), 64);
      for (int64_t k = tl + 1 + lane; k <= n_tiles; k += 64) tile_off[k] = (uint32_t)n_fix;
    }
    if (keep && (int64_t)o < n_fix) {
      sat[o] = (uint8_t)max(em - 7, 0);
      ent[o] = (col << 16) | (s << 15) | (((uint32_t)(em - v) & 0xFFu) << 7) | m;   // opqk_linear.py:375
    }
    p = pn;
    prev = prevn;
    v = vn;
  }
}

int plan_checks(int64_t n_ovf, const int32_t* ovf_idx, const uint8_t* ovf_val, int64_t out_f, int64_t in_f) {
  if (n_ovf <= 0 || !ovf_idx || !ovf_val || !aligned4(ovf_idx)) return BF16X_EARG;
  if (out_f <= 0 || in_f <= 0 || out_f * in_f > (int64_t)INT32_MAX) return BF16X_ESHAPE;
  return BF16X_OK;
}

}  // namespace

extern "C" int64_t bf16x_plan_device_workspace(int64_t n_ovf) {
  return n_ovf < 0 ? -1 : std::max<int64_t>(plan_grid(n_ovf).blocks, 1) * 4;
}

extern "C" int bf16x_plan_device_count(const int32_t* ovf_idx, const uint8_t* ovf_val, int64_t n_ovf,
                                       const int32_t* delta, int64_t n_delta, const uint8_t* emax, int64_t n_emax,
                                       int64_t out_f, int64_t in_f, int64_t* n_fix, void* workspace,
                                       int64_t workspace_bytes, bf16x_stream_t stream) {
  const int rc = plan_checks(n_ovf, ovf_idx, ovf_val, out_f, in_f);
  if (rc) return rc;
  if (!delta || !emax || !n_fix || !workspace) return BF16X_EARG;
  if (!aligned4(delta) || !aligned8(n_fix) || !aligned4(workspace)) return BF16X_EARG;
  const int64_t N = out_f * in_f;
  if (n_delta < bf16x_stream_words(N, 3) || n_emax < (N + 15) / 16) return BF16X_ESTREAM_LEN;
  if (workspace_bytes < bf16x_plan_device_workspace(n_ovf)) return BF16X_ECAPACITY;
  const PlanGrid g = plan_grid(n_ovf);
  hipStream_t st = (hipStream_t)stream;
  hipLaunchKernelGGL(plan_count_kernel, dim3((unsigned)g.blocks), dim3(256), 0, st, ovf_idx, ovf_val, n_ovf, g.iters,
                     (const uint32_t*)delta, emax, N, (uint32_t*)workspace);
  const int st1 = launch_status();
  if (st1) return st1;
  hipLaunchKernelGGL(plan_scan_kernel, dim3(1), dim3(1024), 0, st, (uint32_t*)workspace, (int)g.blocks, n_fix);
  return launch_status();
}

extern "C" int bf16x_plan_device_write(const int32_t* ovf_idx, const uint8_t* ovf_val, int64_t n_ovf,
                                       const int32_t* sign, int64_t n_sign, const int32_t* mant, int64_t n_mant,
                                       const uint8_t* emax, int64_t n_emax, int64_t out_f, int64_t in_f,
                                       int64_t n_fix, uint32_t* tile_off, uint32_t* tile_ent, uint8_t* tile_sat,
                                       const void* workspace, int64_t workspace_bytes, bf16x_stream_t stream) {
  const int rc = plan_checks(n_ovf, ovf_idx, ovf_val, out_f, in_f);
  if (rc) return rc;
  if (!sign || !mant || !emax || !tile_off || !workspace) return BF16X_EARG;
  if (n_fix < 0 || n_fix > n_ovf || (n_fix > 0 && (!tile_ent || !tile_sat))) return BF16X_EARG;
  if (!aligned4(sign) || !aligned4(mant) || !aligned4(tile_off) || !aligned4(tile_ent) || !aligned4(workspace))
    return BF16X_EARG;
  const int64_t N = out_f * in_f;
  if (n_sign < bf16x_stream_words(N, 1) || n_mant < bf16x_stream_words(N, 7) || n_emax < (N + 15) / 16)
    return BF16X_ESTREAM_LEN;
  if (workspace_bytes < bf16x_plan_device_workspace(n_ovf)) return BF16X_ECAPACITY;
  const PlanGrid g = plan_grid(n_ovf);
  const int tpr = tiles_per_row(in_f);
  hipLaunchKernelGGL(plan_write_kernel, dim3((unsigned)g.blocks), dim3(256), 0, (hipStream_t)stream, ovf_idx, ovf_val,
                     n_ovf, g.iters, (const uint32_t*)workspace, (const uint32_t*)sign, (const uint32_t*)mant, emax,
                     (uint32_t)in_f, (uint32_t)tpr, out_f * tpr, n_fix, tile_off, tile_ent, tile_sat);
  return launch_status();
}
