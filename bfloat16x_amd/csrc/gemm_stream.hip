// Fused decode + GEMM for up to 16 activation rows, streaming: no barrier and
// no shared x tile in the main loop, no second launch.
//
// y[M, N] = x[M, K] . W[N, K]^T, fp32 accumulation (bf16x_gemm_fused.py:31-114
// contract; EXACT applies the step-major overflow plan).  W is the packed dict
// or GGUF half-blocks (GG).
//
// A workgroup of 16 waves, one per CU, takes 16 W rows at a time; wave w takes
// the 128-column steps w, w + 16, .. of them, so the 16 waves read 2048
// consecutive columns of a row at once and a wave meets the others only when
// the rows are done (their 16 partial tiles are added through LDS in wave
// order, by waves 0-3, while the others go on).  x of a step belongs to one
// wave, so its MFMA operands are loaded from memory straight into registers.
//
//  * Loads: lane l reads and decodes atom 4s + l % 4 of row l / 4 (a quad
//    reads one row's 4 consecutive atoms); x operand i is 64 contiguous bytes
//    of each token.  The sequence of (rows, step) runs on across row groups:
//    W is requested two steps ahead, x, the plan's entries one, their bounds
//    two, in the order plan, x, W, so that waiting for x leaves W in flight.
//  * The decoded words go through a wave-private LDS scratch in natural column
//    order (load order in, MFMA order out); the step's two plan runs of the 16
//    rows, taken as one list, are written over it in between.
//  * v_mfma_f32_16x16x32_bf16, step operand i = atom i: lane l holds columns
//    8 (l / 16) .. + 7 of it, of row l % 16 (A) and of token l % 16 (B);
//    result register v of lane l is D[4 (l / 16) + v][l % 16].
//
// For small weights (bf16x_use_stream): what it saves is the second launch, the
// x tile's prologue and the barriers.  For large ones it is slower than the
// 16x16x32 kernel's shared x tile: 16 rows per group make a wave load 4 KB of
// x per 2.9 KB of weight.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "../../include/bf16x_hip.h"
#include "bf16x_device.h"
#include "launch_common.h"

namespace bf16x {
namespace stream {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kStep = 128;                 // columns per step (4 atoms per row)
constexpr int kRows = 16;                  // W rows per group
constexpr int kWaves = 16;
constexpr int kScratch = 64 * 64 + 64 * 4; // a wave's decoded step + one trash word per lane
constexpr int kMaxRows = 16;               // activation rows served

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const void* p, uint64_t bytes) {
  const uint32_t n = bytes > 0xFFFFFFFFull ? 0xFFFFFFFFu : (uint32_t)bytes;
  return __builtin_amdgcn_make_buffer_rsrc((void*)p, (short)0, (int)n, 0x00020000);
}

struct WAtom {
  uint32_t s, m[7], d[3];
  uint32_t ew;     // dword holding this atom's emax pair (and its neighbour's)
};
struct WBlock {    // a GGUF block: the 48 bytes from the dword at or below it
  u32x4 q0, q1, q2;
};

template <bool GG, bool EXACT, bool YF32>
__global__ __launch_bounds__(64 * kWaves) void gemm_stream_kernel(
    const uint16_t* __restrict__ x, int M, const uint32_t* __restrict__ sign, const uint32_t* __restrict__ mant,
    const uint32_t* __restrict__ delta, const uint16_t* __restrict__ emax2, const uint8_t* __restrict__ blocks,
    const uint32_t* __restrict__ kp_off, const uint32_t* __restrict__ kp_ent, int out_f, int in_f,
    void* __restrict__ y) {
  __shared__ __attribute__((aligned(16))) uint8_t lds[kWaves * kScratch];
  __shared__ float red[2][kWaves][256];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int P = in_f >> 5, S = in_f / kStep;
  const int groups = (out_f + kRows - 1) / kRows;
  const int nw = (S + kWaves - 1) / kWaves;        // steps of a wave per group (the last may lie past S)
  const int r = lane & 15, q = lane >> 4;          // MFMA role
  const int rl = lane >> 2, ql = lane & 3;         // load role: row rl, atom ql of the step

  // position in the wave's sequence: row group and step; past the last group
  // it stays there (re-reads, never used)
  struct Pos { int g, k; };
  auto next = [&](Pos p) {
    if (++p.k == nw) {
      if (p.g + (int)gridDim.x < groups) { p.k = 0; p.g += (int)gridDim.x; }
      else p.k = nw - 1;
    }
    return p;
  };
  auto step_of = [&](Pos p) { return min(p.k * kWaves + wave, S - 1); };

  // ---- W: lane -> (row 16 g + rl, atom 4 s + ql).  16 P and 4 s atoms are
  // whole multiples of 4 bytes in every stream and in the blocks, and keep the
  // parity of ql; rows past out_f re-read the last one
  using WT = typename std::conditional<GG, WBlock, WAtom>::type;
  __amdgpu_buffer_rsrc_t rs_, rm_, rd_, re_, rb_;
  if constexpr (GG) {
    rb_ = rsrc(blocks, ((uint64_t)out_f * P * 46 + 3) & ~3ull);
  } else {
    rs_ = rsrc(sign, (uint64_t)out_f * P * 4);
    rm_ = rsrc(mant, (uint64_t)out_f * P * 28);
    rd_ = rsrc(delta, (uint64_t)out_f * P * 12);
    re_ = rsrc(emax2, (uint64_t)out_f * P * 2);
  }
  const uint32_t esh = 16u * (uint32_t)(ql & 1);
  auto load_w = [&](Pos p, WT& t) {
    const uint32_t av = (uint32_t)(min(rl, out_f - 1 - kRows * p.g) * P + ql);     // from the group's first atom
    const uint32_t sa = (uint32_t)(kRows * p.g) * (uint32_t)P + 4u * (uint32_t)step_of(p);
    if constexpr (GG) {
      const uint32_t vo = (av * 46) & ~3u;
      t.q0 = __builtin_amdgcn_raw_buffer_load_b128(rb_, (int)vo, (int)(sa * 46), 0);
      t.q1 = __builtin_amdgcn_raw_buffer_load_b128(rb_, (int)(vo + 16), (int)(sa * 46), 0);
      t.q2 = __builtin_amdgcn_raw_buffer_load_b128(rb_, (int)(vo + 32), (int)(sa * 46), 0);
    } else {
      const u32x4 m03 = __builtin_amdgcn_raw_buffer_load_b128(rm_, (int)(av * 28), (int)(sa * 28), 0);
      const u32x3 m46 = __builtin_amdgcn_raw_buffer_load_b96(rm_, (int)(av * 28 + 16), (int)(sa * 28), 0);
      const u32x3 d02 = __builtin_amdgcn_raw_buffer_load_b96(rd_, (int)(av * 12), (int)(sa * 12), 0);
      t.s = __builtin_amdgcn_raw_buffer_load_b32(rs_, (int)(av * 4), (int)(sa * 4), 0);
      t.ew = __builtin_amdgcn_raw_buffer_load_b32(re_, (int)((av & ~1u) * 2), (int)(sa * 2), 0);
      const uint32_t c0 = m03.x, c1 = m03.y, c2 = m03.z, c3 = m03.w, c4 = m46.x, c5 = m46.y, c6 = m46.z;
      t.m[0] = c0; t.m[1] = c1; t.m[2] = c2; t.m[3] = c3; t.m[4] = c4; t.m[5] = c5; t.m[6] = c6;
      const uint32_t e0 = d02.x, e1 = d02.y, e2 = d02.z;
      t.d[0] = e0; t.d[1] = e1; t.d[2] = e2;
    }
  };

  // ---- x: operand i of a step, token r (tokens past M re-read the last one)
  const __amdgpu_buffer_rsrc_t rx_ = rsrc(x, (uint64_t)M * in_f * 2);
  const uint32_t vx = (uint32_t)(min(r, M - 1) * in_f * 2 + q * 16);
  auto load_x = [&](Pos p, bf16x8_t (&X)[4]) {
    const uint32_t ks = (uint32_t)step_of(p) * (kStep * 2);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(rx_, (int)(vx + i * 64), (int)ks, 0);
      X[i] = __builtin_bit_cast(bf16x8_t, v);
    }
  };

  // ---- plan: runs (2 s, g) and (2 s + 1, g) as one list.  Bounds: lane
  // 2 b + e loads the start (e = 0) or end of run b
  const int G2 = 2 * ((out_f + 31) / 32);
  uint32_t kp_total = 0;
  if constexpr (EXACT) kp_total = kp_off[(int64_t)2 * S * G2];
  const __amdgpu_buffer_rsrc_t roff = rsrc(kp_off, ((uint64_t)2 * S * G2 + 1) * 4);
  const __amdgpu_buffer_rsrc_t rent = rsrc(kp_ent, (uint64_t)kp_total * 4);
  const uint32_t vo_o = (uint32_t)(((lane >> 1) & 1) * G2 + (lane & 1)) * 4;
  struct Ent { uint32_t b0, b1, c0, c1, e; };     // run starts, list positions where run 0 and the list end
  auto load_bounds = [&](Pos p) {
    return __builtin_amdgcn_raw_buffer_load_b32(roff, (int)vo_o, (int)((2u * (uint32_t)step_of(p) * G2 + p.g) * 4u), 0);
  };
  auto addr_of = [&](const Ent& t, uint32_t k) { return k < t.c0 ? t.b0 + k : t.b1 + k - t.c0; };
  auto load_ents = [&](uint32_t o, Ent& t) {
    t.b0 = __builtin_amdgcn_readlane(o, 0);
    t.c0 = __builtin_amdgcn_readlane(o, 1) - t.b0;
    t.b1 = __builtin_amdgcn_readlane(o, 2);
    t.c1 = t.c0 + __builtin_amdgcn_readlane(o, 3) - t.b1;
    t.e = __builtin_amdgcn_raw_buffer_load_b32(rent, (int)(addr_of(t, lane) * 4), 0, 0);
  };

  // ---- scratch: slot t = row + 16 atom holds the atom's four 16-byte chunks
  // in natural order, chunk k at position k ^ (t / 4 % 4) ^ (t / 16): 16 lanes
  // writing chunk k of slots in load order, or reading chunk q of 16 rows,
  // touch 16 different 16-byte bank groups
  uint8_t* const scr = lds + wave * kScratch;
  uint8_t* const trash = scr + 64 * 64 + lane * 4;
  auto chunk = [&](int t, int k) { return scr + t * 64 + ((k ^ (t >> 2) ^ (t >> 4)) & 3) * 16; };
  auto patch = [&](const Ent& t, uint32_t k, uint32_t e, bool live) {
    const int rg = (int)(e >> 22) & 15;
    const int col = (int)((e >> 16) & 63) + (k >= t.c0 ? 64 : 0);
    __asm__ volatile("" : "+v"(e));            // the compiler waits for the entry here, outside a branch
    uint8_t* dst = live ? chunk(rg + 16 * (col >> 5), (col & 31) >> 3) + 2 * (col & 7) : trash;
    *(uint16_t*)dst = (uint16_t)(e & 0xFFFFu);
  };

  WT A[2];
  bf16x8_t X[2][4];
  Ent E[2] = {};
  uint32_t O = 0;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  int par = 0;

  // step u (registers u & 1) at position p; p1, p2: the next two
  auto step = [&](int u, Pos p, Pos p1, Pos p2) {
    uint32_t w[16];
    if constexpr (GG) {
      decode_pairs<true>(gguf_atom(GgufRaw{A[u].q0, A[u].q1, A[u].q2, esh}), w);
    } else {
      Atom t;
      t.s = A[u].s;
#pragma unroll
      for (int i = 0; i < 7; ++i) t.m[i] = A[u].m[i];
#pragma unroll
      for (int i = 0; i < 3; ++i) t.d[i] = A[u].d[i];
      t.e = (uint16_t)(A[u].ew >> esh);
      decode_pairs(t, w);
    }
    uint32_t n[16];                            // natural order: elements 2i, 2i + 1 in word i
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      n[i] = perm(w[2 * i + 1], w[2 * i], 0x05040100u);
      n[8 + i] = perm(w[2 * i + 1], w[2 * i], 0x07060302u);
    }
    const int tw = rl + 16 * ql;
#pragma unroll
    for (int k = 0; k < 4; ++k) *(u32x4*)chunk(tw, k) = u32x4{n[4 * k], n[4 * k + 1], n[4 * k + 2], n[4 * k + 3]};
    if constexpr (EXACT) {
      patch(E[u], lane, E[u].e, (uint32_t)lane < E[u].c1);
      for (uint32_t k = 64 + lane; k < E[u].c1; k += 64)                   // dense runs (rare)
        patch(E[u], k, kp_ent[min(addr_of(E[u], k), kp_total - 1)], true);
    }
    __builtin_amdgcn_wave_barrier();
    // the requests: their order is the order they are waited for in
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (EXACT) {
      load_ents(O, E[u ^ 1]);
      O = load_bounds(p2);
    }
    load_x(p1, X[u ^ 1]);
    load_w(p2, A[u]);
    __builtin_amdgcn_sched_barrier(0);
    if (p.k * kWaves + wave < S) {             // (a step past the row is not multiplied)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const bf16x8_t a = *(const bf16x8_t*)chunk(r + 16 * i, q);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, X[u][i], acc, 0, 0, 0);
      }
    }
    if (p.k == nw - 1) {                       // the group's partial tiles: added in wave order
#pragma unroll
      for (int v = 0; v < 4; ++v) red[par][wave][v * 64 + lane] = acc[v];
      acc = f32x4{0.f, 0.f, 0.f, 0.f};
      __syncthreads();
      if (wave < 4) {
        float t = red[par][0][tid];
#pragma unroll
        for (int k = 1; k < kWaves; ++k) t += red[par][k][tid];
        const int row = kRows * p.g + 4 * q + wave;
        if (row < out_f && r < M) {
          const int64_t o = (int64_t)r * out_f + row;
          if constexpr (YF32) ((float*)y)[o] = t;
          else ((uint16_t*)y)[o] = (uint16_t)f32_to_bf16_rne(t);
        }
      }
      par ^= 1;                                // (the other buffer's readers passed this barrier's predecessor)
    }
  };

  Pos p{(int)blockIdx.x, 0};
  if (p.g >= groups) return;
  Pos p1 = next(p), p2 = next(p1);
  if constexpr (EXACT) O = load_bounds(p);
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (EXACT) {
    load_ents(O, E[0]);
    O = load_bounds(p1);
  }
  load_x(p, X[0]);
  load_w(p, A[0]);
  load_w(p1, A[1]);
  __builtin_amdgcn_sched_barrier(0);
  const int total = nw * ((groups - (int)blockIdx.x + (int)gridDim.x - 1) / (int)gridDim.x);
  int i = 0;
  for (; i + 1 < total; i += 2) {
    step(0, p, p1, p2);
    p = p1; p1 = p2; p2 = next(p2);
    step(1, p, p1, p2);
    p = p1; p1 = p2; p2 = next(p2);
  }
  if (i < total) step(0, p, p1, p2);
}

}  // namespace stream
}  // namespace bf16x

// Whether the kernel takes the shape (32-bit offsets).
bool bf16x_gemm_stream_fits(int64_t M, int64_t out_f, int64_t in_f, bool gg) {
  using namespace bf16x::stream;
  if (M < 1 || M > kMaxRows || in_f % kStep != 0 || in_f > kPlanTileCols || out_f > INT32_MAX / 2) return false;
  const uint64_t atoms = (uint64_t)out_f * (uint64_t)(in_f >> 5);
  return atoms * (gg ? 46 : 28) < 0xFFFFFFF0ull && (uint64_t)M * (uint64_t)in_f * 2 < 0xFFFFFFFFull;
}

int bf16x_gemm_stream_launch(const uint16_t* x, int64_t M, const uint32_t* s, const uint32_t* m, const uint32_t* d,
                             const uint16_t* e, const uint8_t* blocks, const uint32_t* kp_off, const uint32_t* kp_ent,
                             int64_t out_f, int64_t in_f, bool exact, bool yf32, void* y, hipStream_t st) {
  using namespace bf16x::stream;
  if (!bf16x_gemm_stream_fits(M, out_f, in_f, blocks != nullptr)) return BF16X_ESHAPE;
  const int cus = device_cus() > 0 ? device_cus() : 256;
  const int64_t groups = (out_f + kRows - 1) / kRows;
  const dim3 grid((unsigned)std::min<int64_t>(groups, cus));
#define BF16X_ST(GG_, EX_, YF_)                                                                                 \
  hipLaunchKernelGGL((gemm_stream_kernel<GG_, EX_, YF_>), grid, dim3(64 * kWaves), 0, st, x, (int)M, s, m, d, e, \
                     blocks, kp_off, kp_ent, (int)out_f, (int)in_f, y)
#define BF16X_STX(GG_)                                                                         \
  do {                                                                                         \
    if (exact) { if (yf32) BF16X_ST(GG_, true, true); else BF16X_ST(GG_, true, false); }        \
    else { if (yf32) BF16X_ST(GG_, false, true); else BF16X_ST(GG_, false, false); }            \
  } while (0)
  if (blocks) BF16X_STX(true);
  else BF16X_STX(false);
#undef BF16X_STX
#undef BF16X_ST
  return launch_status();
}

// Whether the dispatch of bf16x_gemm and bf16x_gguf_gemm takes the kernel: a
// wave's steps times the tokens at most 32, and at most 4 steps.  A step costs
// a wave about 4.3 us at 16 tokens and 3.5 at 2 (it loads more x than weight),
// against a fixed ~9 us of the 16x16x32 kernel with its x tile, barriers and
// reduction.  Measured, streaming against that kernel (us), M = 2 / 8 / 16:
// 1024x1024 (1 step) 4.6 / 4.9 / 5.6 against 8.3 / 8.2 / 8.3; 4096x4096 (2)
// 9.9 / 10.9 / 12.4 against 13.4 / 13.5 / 13.9; 300x6144 (3) 9.3 / 10.4 / 11.9
// against 11.6 / 11.7 / 11.9; 2048x8192 (4) 13.1 / 15.0 / 17.7 against 14.5 /
// 14.6 / 15.0; 4096x14336 (7) 28.4 / 31.0 / 34.7 against 28.6 / 29.3 / 29.9.
bool bf16x_use_stream(int64_t M, int64_t out_f, int64_t in_f, bool gg) {
  using namespace bf16x::stream;
  const int64_t t = tuning(BF16X_TUNE_GEMM_STREAM_MAX);
  if (M > (t >= 0 ? t : kMaxRows) || !bf16x_gemm_stream_fits(M, out_f, in_f, gg)) return false;
  if (t >= 0) return true;
  if (tuning(BF16X_TUNE_GEMM_SKINNY2_MAX) >= 0 || tuning(BF16X_TUNE_GEMM_WS_MIN_ROWS) >= 0) return false;
  const int64_t cus = device_cus() > 0 ? device_cus() : 256;
  const int64_t groups = (out_f + kRows - 1) / kRows, S = in_f / kStep;
  const int64_t steps = (groups + cus - 1) / cus * ((S + kWaves - 1) / kWaves);
  return steps <= 4 && steps * M <= 32;
}
