// Device encoder: bf16 weight -> packed dict, byte-identical to
// bf16x_quantize (opqk_linear.py:291-324) and to bf16x_encode_host.
//
// An atom (the 32 elements 32a .. 32a+31) becomes sign word a, mant words
// 7a .. 7a+6, delta words 3a .. 3a+2 (3-bit codes min(delta, 7), :314) and emax
// bytes 2a, 2a+1 (sub = 16, opqk_linear.py:305-308; elements past N count as
// exponent 0), each clipped to the reference packer's stream length; the
// words the element padding of pack_bits_stream (:53-64) adds past the last
// atom (a few, for small N) are written as zero.  The overflow table (delta
// >= 7, positions ascending, :311-313) takes three launches: the streams with
// a list of the entries of every segment, a scan of the counts, and a copy of
// the lists to their places.
//
// Bound: HBM (2 bytes read, 1.44 written per element).  What the kernels do
// about it, at 4096x14336 (200 MB; kernel times):
//  * a wave reads its 64 atoms as 4 KB contiguous and hands them to the
//    lanes through LDS, and the mant and delta words go back through LDS so
//    that every store instruction writes 1 KB contiguous.  With one atom per
//    thread stored in place (7 + 3 dword stores, 28 and 12 bytes apart) the
//    same pass was bound by its store instructions;
//  * an atom is encoded as 16 pairs (element j, element j + 16), the
//    decoder's order: exponent maximum, delta and code of two elements per
//    packed 16-bit instruction, both mantissas and both codes placed by one
//    shift-or each.  Together 92-94 -> 43.6 us (4.6 TB/s), 8 workgroups per CU;
//  * the pass leaves (position, delta) of a segment's entries in a list, so
//    the table launch copies 5 bytes per entry instead of reading the weight
//    again: 44-46 -> 8.6 us;
//  * at most 4096 workgroups, so the scan is one step of one workgroup:
//    12 -> 5.9 us.  (8192 workgroups, one iteration each: 39.6 us for the
//    streams, 8.7 for the scan, 11 for the table; 2048: 46.4 / 5.9 / 7.7.)
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/bf16x_hip.h"
#include "bf16x_device.h"
#include "launch_common.h"

namespace {
using namespace bf16x;

// A wave encodes a segment of 64 * iters consecutive atoms, a workgroup 4
// segments.  iters keeps the workgroups at or below kMaxBlocks, so the scan
// is one workgroup with 4 counts per thread.
constexpr int kMaxBlocks = 4096;

struct EncGrid {
  int64_t n_atoms, blocks;
  int iters;
};
EncGrid enc_grid(int64_t N) {
  EncGrid g;
  g.n_atoms = (N + 31) / 32;
  g.iters = (int)std::max<int64_t>(1, (g.n_atoms + 256 * (int64_t)kMaxBlocks - 1) / (256 * (int64_t)kMaxBlocks));
  g.blocks = (g.n_atoms + 256 * (int64_t)g.iters - 1) / (256 * (int64_t)g.iters);
  return g;
}
// entries a segment's list holds (an eighth of its elements); a denser
// segment's entries are recomputed from the weight
__host__ __device__ constexpr int seg_cap(int iters) { return 256 * iters; }

// 16-byte chunk q of atom a of a wave's 4 KB: conflict free for the
// contiguous writes and for the per-atom reads
__device__ __forceinline__ int chunk_slot(int a, int q) { return a * 64 + (((q + (a >> 2)) & 3) << 4); }

__device__ __forceinline__ uint32_t pk_max(uint32_t a, uint32_t b) {
  u16x2 x, y;
  __builtin_memcpy(&x, &a, 4);
  __builtin_memcpy(&y, &b, 4);
  u16x2 r = __builtin_elementwise_max(x, y);
  uint32_t o;
  __builtin_memcpy(&o, &r, 4);
  return o;
}
__device__ __forceinline__ uint32_t pk_min(uint32_t a, uint32_t b) {
  u16x2 x, y;
  __builtin_memcpy(&x, &a, 4);
  __builtin_memcpy(&y, &b, 4);
  u16x2 r = __builtin_elementwise_min(x, y);
  uint32_t o;
  __builtin_memcpy(&o, &r, 4);
  return o;
}
// per-16-bit-lane shifts by a constant
__device__ __forceinline__ uint32_t pk_shl(uint32_t a, int n) {
  return (a << n) & (0x00010001u * ((0xFFFFu << n) & 0xFFFFu));
}
__device__ __forceinline__ uint32_t pk_shr(uint32_t a, int n) { return (a >> n) & (0x00010001u * (0xFFFFu >> n)); }

struct Enc {
  uint32_t s, m[7], d[3];
  uint32_t em;          // emax of half 0 | emax of half 1 << 8
  uint32_t ovf;         // bit j: delta of element j >= 7
};

// p[j] = bf16 bits of element j | bits of element j + 16 << 16
__device__ __forceinline__ Enc encode_pairs(const uint32_t (&p)[16]) {
  Enc r;
  uint32_t E = 0;                                  // exponent maxima, at bits 7..14 of the lanes
#pragma unroll
  for (int j = 0; j < 16; ++j) E = pk_max(E, p[j] & 0x7F807F80u);
  uint32_t pm[8] = {0, 0, 0, 0, 0, 0, 0, 0}, pd[4] = {0, 0, 0, 0};
  r.s = 0;
  r.ovf = 0;
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    const uint32_t d7 = pk_sub_wrap(E, p[j] & 0x7F807F80u);        // delta << 7 (never negative)
    // bit 15 of a lane set iff delta >= 7: (delta << 7) + 0x7C80 reaches 0x8000
    u16x2 dv;
    __builtin_memcpy(&dv, &d7, 4);
    dv += (unsigned short)0x7C80;
    uint32_t ge;
    __builtin_memcpy(&ge, &dv, 4);
    r.ovf |= (ge >> (15 - j)) & (0x00010001u << j);
    r.s |= (p[j] >> (15 - j)) & (0x00010001u << j);
    const uint32_t code = pk_min(d7, 0x03800380u);                  // code << 7
    const int dk = (3 * j) >> 4, dof = (3 * j) & 15;
    if (dof <= 13) {
      pd[dk] |= dof <= 7 ? code >> (7 - dof) : code << (dof - 7);
    } else {
      pd[dk] |= pk_shl(code, dof - 7);
      pd[dk + 1] |= pk_shr(code, 7 + 16 - dof);
    }
    const uint32_t mv = p[j] & 0x007F007Fu;
    const int mk = (7 * j) >> 4, mo = (7 * j) & 15;
    if (mo <= 9) {
      pm[mk] |= mv << mo;
    } else {
      pm[mk] |= pk_shl(mv, mo);
      pm[mk + 1] |= pk_shr(mv, 16 - mo);
    }
  }
  // 16-bit chunk k of elements 0..15 is the low lane of pm[k], of elements
  // 16..31 the high lane (chunk 7 + k of the atom)
  r.m[0] = perm(pm[1], pm[0], 0x05040100u);
  r.m[1] = perm(pm[3], pm[2], 0x05040100u);
  r.m[2] = perm(pm[5], pm[4], 0x05040100u);
  r.m[3] = lo_hi(pm[6], pm[0]);
  r.m[4] = perm(pm[2], pm[1], 0x07060302u);
  r.m[5] = perm(pm[4], pm[3], 0x07060302u);
  r.m[6] = perm(pm[6], pm[5], 0x07060302u);
  r.d[0] = perm(pd[1], pd[0], 0x05040100u);
  r.d[1] = lo_hi(pd[2], pd[0]);
  r.d[2] = perm(pd[2], pd[1], 0x07060302u);
  r.em = ((E >> 7) & 0xFFu) | ((E >> 15) & 0xFF00u);
  return r;
}

// Streams and emax; the entries of every segment (element of the segment
// << 8 | delta, ascending) in its list, their number in seg_cnt, the
// workgroup's number in blk_cnt.
__global__ __launch_bounds__(256) void encode_atoms_kernel(
    const uint16_t* __restrict__ wb, int64_t N, int64_t n_atoms, int iters, uint32_t* __restrict__ sign, int64_t ws,
    uint32_t* __restrict__ mant, int64_t wm, uint32_t* __restrict__ delta, int64_t wd, uint8_t* __restrict__ emax,
    int64_t n_emax, uint32_t* __restrict__ list, uint32_t* __restrict__ seg_cnt, uint32_t* __restrict__ blk_cnt) {
  // the wave's 64 atoms, then their mant words and delta words (16 KB per
  // workgroup: 8 workgroups per CU)
  __shared__ __attribute__((aligned(16))) uint8_t wl[4][4096];
  __shared__ uint32_t red[4];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t seg = (int64_t)blockIdx.x * 4 + wave;
  const int64_t a_seg = seg * 64 * iters;
  const int cap = seg_cap(iters);
  uint32_t* sl = list + seg * cap;
  uint8_t* buf = wl[wave];
  uint32_t* mb = (uint32_t*)buf;
  const bool emax_even = ((uintptr_t)emax & 1u) == 0;
  uint32_t cnt = 0;                                 // entries of the segment so far
  // the 4 KB of iteration it: chunk 64 i + l of the wave's atoms (whole atoms only)
  const int64_t full = N >> 5;                      // atoms with all 32 elements
  auto load = [&](int it, u32x4 (&v)[4]) {
    const int64_t a0 = a_seg + 64 * (int64_t)it;
    if (it < iters && a0 + 64 <= full) {
      const u32x4* src = (const u32x4*)(wb + a0 * 32);
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = src[64 * i + lane];
    }
  };
  u32x4 v[4] = {};
  load(0, v);
  for (int it = 0; it < iters; ++it) {
    const int64_t a0 = a_seg + 64 * (int64_t)it, a = a0 + lane;
    if (a0 >= n_atoms) break;
    const bool whole = a0 + 64 <= full;
    uint32_t p[16];
    if (whole) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int c = 64 * i + lane;
        *(u32x4*)(buf + chunk_slot(c >> 2, c & 3)) = v[i];
      }
      load(it + 1, v);
    } else {                                        // the weight's last atoms, element by element
      for (int j = 0; j < 32; ++j) {
        const int64_t e = a * 32 + j;
        *(uint16_t*)(buf + chunk_slot(lane, j >> 3) + (j & 7) * 2) = e < N ? wb[e] : (uint16_t)0;
      }
    }
    __builtin_amdgcn_wave_barrier();                // lanes read what others wrote: kept in this order
    u32x4 q[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) q[c] = *(const u32x4*)(buf + chunk_slot(lane, c));
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const uint32_t l0 = q[c].x, l1 = q[c].y, l2 = q[c].z, l3 = q[c].w;                        // elements 8c ..
      const uint32_t h0 = q[c + 2].x, h1 = q[c + 2].y, h2 = q[c + 2].z, h3 = q[c + 2].w;        // 16 + 8c ..
      p[8 * c + 0] = perm(h0, l0, 0x05040100u); p[8 * c + 1] = perm(h0, l0, 0x07060302u);
      p[8 * c + 2] = perm(h1, l1, 0x05040100u); p[8 * c + 3] = perm(h1, l1, 0x07060302u);
      p[8 * c + 4] = perm(h2, l2, 0x05040100u); p[8 * c + 5] = perm(h2, l2, 0x07060302u);
      p[8 * c + 6] = perm(h3, l3, 0x05040100u); p[8 * c + 7] = perm(h3, l3, 0x07060302u);
    }
    Enc t = encode_pairs(p);
    if (!whole) {
      const int64_t left = N - a * 32;              // elements of this atom
      if (left < 32) {                              // padding elements: code 0, never in the table
        const int n = (int)max(left, (int64_t)0);
        t.ovf &= n ? (1u << n) - 1u : 0u;
        const int fw = (3 * n) >> 5;                // whole code words kept
        for (int k = 0; k < 3; ++k) t.d[k] &= k < fw ? 0xFFFFFFFFu : (k == fw ? (1u << ((3 * n) & 31)) - 1u : 0u);
      }
    }
    uint32_t total;
    uint32_t pos = cnt + wave_prefix(__builtin_popcount(t.ovf), lane, total);
    for (uint32_t mk = t.ovf; mk; mk &= mk - 1) {
      const int j = __builtin_ctz(mk);
      const uint32_t b = *(const uint16_t*)(buf + chunk_slot(lane, j >> 3) + (j & 7) * 2);
      const uint32_t d = ((t.em >> ((j >> 4) * 8)) & 0xFFu) - ((b >> 7) & 0xFFu);
      if (pos < (uint32_t)cap) sl[pos] = ((uint32_t)(it * 2048 + lane * 32 + j) << 8) | d;
      ++pos;
    }
    cnt += total;
    if (whole) {
      sign[a] = t.s;
      if (emax_even) {
        *(uint16_t*)(emax + 2 * a) = (uint16_t)t.em;
      } else {
        emax[2 * a] = (uint8_t)t.em;
        emax[2 * a + 1] = (uint8_t)(t.em >> 8);
      }
      __builtin_amdgcn_wave_barrier();              // the atoms are read; their place takes the words
#pragma unroll
      for (int k = 0; k < 7; ++k) mb[lane * 7 + k] = t.m[k];
#pragma unroll
      for (int k = 0; k < 3; ++k) mb[448 + lane * 3 + k] = t.d[k];
      __builtin_amdgcn_wave_barrier();
      const u32x4* sc = (const u32x4*)mb;
      u32x4a* md = (u32x4a*)(mant + 7 * a0);
      md[lane] = sc[lane];
      if (lane < 48) {
        md[64 + lane] = sc[64 + lane];
        ((u32x4a*)(delta + 3 * a0))[lane] = sc[112 + lane];
      }
      __builtin_amdgcn_wave_barrier();              // before the next atoms overwrite them
    } else if (a < n_atoms) {
      if (a < ws) sign[a] = t.s;
      for (int k = 0; k < 7; ++k)
        if (7 * a + k < wm) mant[7 * a + k] = t.m[k];
      for (int k = 0; k < 3; ++k)
        if (3 * a + k < wd) delta[3 * a + k] = t.d[k];
      if (2 * a < n_emax) emax[2 * a] = (uint8_t)t.em;
      if (2 * a + 1 < n_emax) emax[2 * a + 1] = (uint8_t)(t.em >> 8);
    }
    if (a == n_atoms - 1) {
      // the packer's element padding can reach past the last atom (N = 5:
      // 34 padded elements, 8 mant words): those words are zero
      for (int64_t k = 7 * n_atoms; k < wm; ++k) mant[k] = 0u;
      for (int64_t k = 3 * n_atoms; k < wd; ++k) delta[k] = 0u;
      for (int64_t k = n_atoms; k < ws; ++k) sign[k] = 0u;
    }
  }
  if (lane == 0) {
    seg_cnt[seg] = cnt;
    red[wave] = cnt;
  }
  __syncthreads();
  if (threadIdx.x == 0) blk_cnt[blockIdx.x] = red[0] + red[1] + red[2] + red[3];
}

// exclusive scan of the workgroup counts (at most kMaxBlocks), one workgroup
__global__ __launch_bounds__(1024) void encode_scan_kernel(const uint32_t* __restrict__ blk_cnt, int n_blk,
                                                           uint32_t* __restrict__ blk_off,
                                                           int64_t* __restrict__ n_ovf) {
  __shared__ uint32_t part[16];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  constexpr int kPer = kMaxBlocks / 1024;
  uint32_t c[kPer], own = 0;
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const int i = tid * kPer + k;
    c[k] = i < n_blk ? blk_cnt[i] : 0u;
    own += c[k];
  }
  uint32_t total;
  uint32_t at = wave_prefix(own, lane, total);
  if (lane == 0) part[wv] = total;
  __syncthreads();
  for (int k = 0; k < wv; ++k) at += part[k];
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const int i = tid * kPer + k;
    if (i < n_blk) blk_off[i] = at;
    at += c[k];
  }
  if (tid == 1023) n_ovf[0] = (int64_t)at;
}

// the lists to the table; a segment with more entries than its list holds
// takes them from the weight again
__global__ __launch_bounds__(256) void encode_table_kernel(const uint16_t* __restrict__ wb, int64_t N, int iters,
                                                           const uint32_t* __restrict__ list,
                                                           const uint32_t* __restrict__ seg_cnt,
                                                           const uint32_t* __restrict__ blk_off,
                                                           int32_t* __restrict__ ovf_idx,
                                                           uint8_t* __restrict__ ovf_val, int64_t cap) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t s0 = (int64_t)blockIdx.x * 4, seg = s0 + wave;
  int64_t pos = blk_off[blockIdx.x];
  for (int k = 0; k < wave; ++k) pos += seg_cnt[s0 + k];
  const uint32_t cnt = seg_cnt[seg];
  const int64_t e_seg = seg * 2048 * iters;
  if (cnt <= (uint32_t)seg_cap(iters)) {
    const uint32_t* sl = list + seg * seg_cap(iters);
    for (uint32_t k = lane; k < cnt; k += 64) {
      const uint32_t v = sl[k];
      if (pos + k < cap) {
        ovf_idx[pos + k] = (int32_t)(e_seg + (v >> 8));
        ovf_val[pos + k] = (uint8_t)v;
      }
    }
    return;
  }
  // 64 elements at a time; a 16-element block's exponent maximum is the
  // maximum over its 16 lanes
  for (int64_t e0 = e_seg; e0 < e_seg + 2048 * (int64_t)iters && e0 < N; e0 += 64) {
    const int64_t e = e0 + lane;
    const uint32_t x = e < N ? ((uint32_t)wb[e] >> 7) & 0xFFu : 0u;
    uint32_t em = x;
#pragma unroll
    for (int o = 8; o >= 1; o >>= 1) em = max(em, (uint32_t)__shfl_xor(em, o, 64));
    const bool in = e < N && em - x >= 7u;
    const uint64_t b = __ballot(in);
    const int64_t at = pos + __builtin_popcountll(b & ((1ull << lane) - 1ull));
    if (in && at < cap) {
      ovf_idx[at] = (int32_t)e;
      ovf_val[at] = (uint8_t)(em - x);
    }
    pos += __builtin_popcountll(b);
  }
}

// workspace: lists, segment counts, workgroup counts, workgroup offsets
struct EncWs {
  int64_t list, seg, cnt, off, bytes;
};
EncWs enc_ws(const EncGrid& g) {
  auto up = [](int64_t b) { return (b + 255) / 256 * 256; };
  EncWs w;
  w.list = 0;
  w.seg = up(g.blocks * 4 * seg_cap(g.iters) * 4);
  w.cnt = w.seg + up(g.blocks * 4 * 4);
  w.off = w.cnt + up(g.blocks * 4);
  w.bytes = w.off + up(g.blocks * 4);
  return w;
}

}  // namespace

extern "C" int64_t bf16x_encode_workspace(int64_t out_f, int64_t in_f) {
  if (out_f <= 0 || in_f <= 0) return -1;
  return enc_ws(enc_grid(out_f * in_f)).bytes;
}

extern "C" int bf16x_encode_streams(const uint16_t* w_bits, int64_t out_f, int64_t in_f, int32_t sub, int32_t* sign,
                                    int64_t n_sign, int32_t* mant, int64_t n_mant, int32_t* delta, int64_t n_delta,
                                    uint8_t* emax, int64_t n_emax, int64_t* n_ovf, void* workspace,
                                    int64_t workspace_bytes, bf16x_stream_t stream) {
  if (!w_bits || !sign || !mant || !delta || !emax || !n_ovf || !workspace) return BF16X_EARG;
  if (out_f <= 0 || in_f <= 0) return BF16X_ESHAPE;
  if (sub != 16) return BF16X_ESUB;
  const int64_t N = out_f * in_f;
  if (N > (int64_t)INT32_MAX) return BF16X_ESHAPE;           // the table stores int32 positions
  const int64_t ws = bf16x_stream_words(N, 1), wm = bf16x_stream_words(N, 7), wd = bf16x_stream_words(N, 3);
  const int64_t ne = (N + 15) / 16;
  if (n_sign < ws || n_mant < wm || n_delta < wd || n_emax < ne) return BF16X_ESTREAM_LEN;
  if (workspace_bytes < bf16x_encode_workspace(out_f, in_f)) return BF16X_ECAPACITY;
  if (!aligned16(w_bits) || !aligned16(workspace) || !aligned4(sign) || !aligned4(mant) || !aligned4(delta) ||
      !aligned8(n_ovf))
    return BF16X_EARG;
  const EncGrid g = enc_grid(N);
  const EncWs o = enc_ws(g);
  uint8_t* w = (uint8_t*)workspace;
  hipStream_t st = (hipStream_t)stream;
  hipLaunchKernelGGL(encode_atoms_kernel, dim3((unsigned)g.blocks), dim3(256), 0, st, w_bits, N, g.n_atoms, g.iters,
                     (uint32_t*)sign, ws, (uint32_t*)mant, wm, (uint32_t*)delta, wd, emax, ne,
                     (uint32_t*)(w + o.list), (uint32_t*)(w + o.seg), (uint32_t*)(w + o.cnt));
  const int rc = launch_status();
  if (rc) return rc;
  hipLaunchKernelGGL(encode_scan_kernel, dim3(1), dim3(1024), 0, st, (const uint32_t*)(w + o.cnt), (int)g.blocks,
                     (uint32_t*)(w + o.off), n_ovf);
  return launch_status();
}

extern "C" int bf16x_encode_table(const uint16_t* w_bits, int64_t out_f, int64_t in_f, int32_t* ovf_idx,
                                  uint8_t* ovf_val, int64_t ovf_cap, const void* workspace, int64_t workspace_bytes,
                                  bf16x_stream_t stream) {
  if (!w_bits || !workspace) return BF16X_EARG;
  if (ovf_cap < 0 || (ovf_cap > 0 && (!ovf_idx || !ovf_val))) return BF16X_EARG;
  if (out_f <= 0 || in_f <= 0 || out_f * in_f > (int64_t)INT32_MAX) return BF16X_ESHAPE;
  if (workspace_bytes < bf16x_encode_workspace(out_f, in_f)) return BF16X_ECAPACITY;
  if (!aligned16(w_bits) || !aligned16(workspace) || !aligned4(ovf_idx)) return BF16X_EARG;
  if (ovf_cap == 0) return BF16X_OK;
  const int64_t N = out_f * in_f;
  const EncGrid g = enc_grid(N);
  const EncWs o = enc_ws(g);
  const uint8_t* w = (const uint8_t*)workspace;
  hipLaunchKernelGGL(encode_table_kernel, dim3((unsigned)g.blocks), dim3(256), 0, (hipStream_t)stream, w_bits, N,
                     g.iters, (const uint32_t*)(w + o.list), (const uint32_t*)(w + o.seg),
                     (const uint32_t*)(w + o.off), ovf_idx, ovf_val, ovf_cap);
  return launch_status();
}

extern "C" int bf16x_encode(const uint16_t* w_bits, int64_t out_f, int64_t in_f, int32_t sub, int32_t* sign,
                            int64_t n_sign, int32_t* mant, int64_t n_mant, int32_t* delta, int64_t n_delta,
                            uint8_t* emax, int64_t n_emax, int32_t* ovf_idx, uint8_t* ovf_val, int64_t ovf_cap,
                            int64_t* n_ovf, void* workspace, int64_t workspace_bytes, bf16x_stream_t stream) {
  if (ovf_cap < 0 || (ovf_cap > 0 && (!ovf_idx || !ovf_val)) || !aligned4(ovf_idx)) return BF16X_EARG;
  const int rc = bf16x_encode_streams(w_bits, out_f, in_f, sub, sign, n_sign, mant, n_mant, delta, n_delta, emax,
                                      n_emax, n_ovf, workspace, workspace_bytes, stream);
  if (rc) return rc;
  return bf16x_encode_table(w_bits, out_f, in_f, ovf_idx, ovf_val, ovf_cap, workspace, workspace_bytes, stream);
}
