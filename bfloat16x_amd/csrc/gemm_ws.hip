// Fused decode + GEMM for many rows (prefill) on gfx950: wave-specialised
// workgroups.
//
// Replaces _bf16x_gemm_fused_kernel / bf16x_fused_gemm (bf16x_gemm_fused.py:31-114)
// from tens of rows on: y[M, N] = x[M, K] . W[N, K]^T with W decoded on the
// fly, fp32 accumulation (in four-step groups, K % 256 == 0, from 65 rows, or 33
// of a weight of 2^25 elements; one step at a time from 192).  SATURATED reproduces the reference
// kernel's numerics (code 7 -> exponent emax-7, bf16x_gemm_fused.py:84-87);
// EXACT writes the overflow plan's entries over the decoded tile and
// multiplies by the lossless weight.
//
// Measured on MI355X, and the reason for the structure:
//  * VALU instructions in an MFMA wave's own instruction stream do not run
//    under its MFMAs (the step time is close to the sum of both), but an
//    MFMA wave and a VALU wave sharing a SIMD overlap.  Decoding a W element
//    takes ~5 VALU lane-ops, so the decode runs in waves of its own.
//  * LDS sustains ~70 B/clk per CU for writes (ds_write or direct loads) and
//    130-220 B/clk for 16-byte reads.  Register budget (two waves per SIMD,
//    256 registers each) limits an MFMA wave to 128 accumulators.
//
// A workgroup is 8 waves and owns an output tile of 256 x rows (tokens) by 128
// W rows (the grouped kernel below also 128 or 64 by 128, with 12 waves) over a
// range of 64-column K steps (all of K, or one split of it when
// the tile count alone leaves CUs idle; split partials are fp32 and summed in
// split order by a second kernel).
//  * Waves 4-7 decode.  Wave 4+p decodes rows 32p .. 32p+31 of the W tile at
//    each step (lane l: row l%32, atom l/32 of the step), writes them to LDS
//    in natural order and writes the EXACT plan entries of the same rows over
//    them (one wave: its LDS writes land in order).  Atoms and plan entries
//    are requested two steps ahead into registers, the plan offsets one step
//    before their entries.
//  * Waves 0-3 (one per SIMD) issue the MFMAs: wave c owns tokens
//    64c .. 64c+63 and all 128 W rows, 2 x 4 accumulators of
//    v_mfma_f32_32x32x16_bf16.  Each token row belongs to one wave, so x does
//    not pass through LDS: a wave requests its x operands of the next step
//    (8 16-byte loads per lane) straight into registers.  x is first
//    rewritten in MFMA operand order (x_op_kernel, into the workspace), so
//    each of those loads reads 1 KB contiguous: loading the operands from
//    row-major x touches 32 rows per instruction, and the vector memory
//    pipeline's rate in cache lines per clock, not bytes, then set the step
//    time.  W operands come from LDS; each k-quarter first requests the next
//    quarter's 4, then runs its 8 MFMAs.
//  * LDS traffic is the W tile only: 16 KB written and 64 KB read per step.
//    With the x tile staged in LDS as well (144 KB per step), the kernel ran
//    at half this speed: LDS, not the MFMAs, set the step time.
//  * LDS: 2 W slots of 16 KB; one barrier per step.  Tile rows are 128
//    bytes; 16-byte chunk c of row r sits at c ^ ((r >> 1) & 7), so 16 lanes
//    reading one logical chunk of 16 consecutive rows touch 16 different
//    16-byte bank groups (64 banks).
//  * MFMA k-slots: in k-quarter q, lanes 0-31 hold 8 columns of the step's
//    first half and lanes 32-63 the same 8 of its second half, for x (A
//    operand) and W (B operand) alike: columns 4q .. 4q+3 and 16+4q .. 19+4q
//    of the half, interleaved (the order the decode leaves them in, see
//    chunk_of).  Result register v of lane l is D[8(v/4) + 4(l/32) + v%4][l%32]:
//    token row, W row.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "../../include/bf16x_hip.h"
#include "bf16x_device.h"
#include "launch_common.h"

namespace bf16x {
namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

constexpr int kStep = 64;              // K columns per step
constexpr int kRowB = 128;             // bytes of one LDS tile row (64 bf16)
constexpr int kBM = 256;               // tokens per tile
constexpr int kBN = 128;               // W rows per tile
constexpr int kWSlot = kBN * kRowB;    // 16 KB

__device__ __forceinline__ int swz(int row, int chunk) { return chunk ^ ((row >> 1) & 7); }

// K order inside a 64-column step.  decode_pairs leaves element j of an atom
// in the low half of word j and element 16 + j in the high half; W is stored
// as decoded (no permute), so 16-byte chunk c of atom h (words 4c .. 4c+3)
// holds atom columns 4c, 16+4c, 4c+1, 17+4c, 4c+2, 18+4c, 4c+3, 19+4c.  x_op
// writes x's operand chunks in the same column order, so both MFMA operands
// see one permutation of K.  Column c (0..63) of a step sits in chunk
// chunk_of(c) of the step's 8, at bf16 position pos_of(c).
__device__ __forceinline__ int chunk_of(int c) { return ((c >> 5) << 2) | ((c >> 2) & 3); }
__device__ __forceinline__ int pos_of(int c) { return ((c & 3) << 1) | ((c >> 4) & 1); }

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const void* p, uint64_t bytes) {
  const uint32_t n = bytes > 0xFFFFFFFFull ? 0xFFFFFFFFu : (uint32_t)bytes;
  return __builtin_amdgcn_make_buffer_rsrc((void*)p, (short)0, (int)n, 0x00020000);
}

// the words of one atom as loaded (emax as the dword holding both atoms of the step)
struct Raw {
  uint32_t s, m[7], d[3], ew;
};
// a GGUF block as loaded: the 48 bytes from the dword at or below it
struct RawG {
  u32x4 q0, q1, q2;
};

// Block -> work.  Blocks [0, full) each own one output tile over all of K
// (tiles 0 .. full-1); the remaining blocks split K for the last `ltiles`
// tiles in `lunits`-unit ranges (units: steps, or four-step groups) and write
// fp32 partials, summed by ws_tile_reduce_kernel.  full is a multiple of the
// resident block count, so the split blocks fill the last round.  Within
// each range the order is XCD-aware: blocks go round-robin over 8 XCDs, and
// each XCD gets a contiguous run of tiles, M fastest, so the M tiles that
// share a W tile run on one XCD at the same time and share its L2.
struct WsGrid {
  int mtiles, full, ltiles, lunits;
  int bm;         // tokens per tile
};
struct WsWork {
  int64_t m0, n0;
  int u0, nu;     // first unit and unit count of this block
  int lt;         // split tile index (0 .. ltiles-1), or -1 for a full tile
  int kb;         // K range of a split tile
};
__device__ __forceinline__ int xcd_order(int b, int nb) {
  const int per = nb / 8, extra = nb - per * 8;
  return nb >= 8 ? ((b & 7) * per + min(b & 7, extra) + (b >> 3)) : b;
}
__device__ __forceinline__ WsWork ws_work(const WsGrid& g, int units) {
  const int nb = (int)gridDim.x, b = (int)blockIdx.x;
  WsWork w;
  int tile;
  if (b < g.full) {
    tile = xcd_order(b, g.full);
    w.lt = -1; w.kb = 0; w.u0 = 0; w.nu = units;
  } else {
    const int lb = xcd_order(b - g.full, nb - g.full);
    w.lt = lb % g.ltiles; w.kb = lb / g.ltiles;
    tile = g.full + w.lt;
    w.u0 = w.kb * g.lunits;
    w.nu = min(g.lunits, units - w.u0);
  }
  w.m0 = (int64_t)(tile % g.mtiles) * g.bm;
  w.n0 = (int64_t)(tile / g.mtiles) * kBN;
  return w;
}

// The output tile from the MFMA waves' accumulators: register v of lane l ->
// token row 8(v/4) + 4(l/32) + v%4, W row l%32.  A split tile's partial goes
// to its own BM x 128 fp32 tile of `part` (all of it: rows past M and
// columns past out_f hold zeros), in K-range order.  The wave owns NT 32-token
// tiles from token 32 NT (wave % TG) and NJ 32-row W tiles from row
// 32 NJ (wave / TG).
enum { kYBf16 = 0, kYF32 = 1, kYF16 = 2 };     // output types of the kernels below
template <int YT>
__device__ __forceinline__ void store_y(void* __restrict__ y, int64_t i, float v) {
  if constexpr (YT == kYF32) ((float*)y)[i] = v;
  else if constexpr (YT == kYF16) ((_Float16*)y)[i] = (_Float16)v;
  else ((uint16_t*)y)[i] = (uint16_t)f32_to_bf16_rne(v);
}

template <int YT, int NT, int TG, int NJ>
__device__ __forceinline__ void ws_store(const f32x16 (&acc)[NT][NJ], const WsWork& w, int wave, int lane, int64_t M,
                                         int64_t out_f, int ltiles, void* __restrict__ y, float* __restrict__ part) {
  constexpr int BM = 32 * NT * TG;
  const int lr = lane & 31, h = lane >> 5;
  const int t0 = 32 * NT * (wave % TG), r0 = 32 * NJ * (wave / TG);
  if (w.lt >= 0) {
    float* pt = part + ((int64_t)w.kb * ltiles + w.lt) * (BM * kBN);
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
      for (int jj = 0; jj < NJ; ++jj)
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const int r = t0 + i * 32 + 8 * (v >> 2) + 4 * h + (v & 3);
          pt[r * kBN + r0 + jj * 32 + lr] = acc[i][jj][v];
        }
    return;
  }
#pragma unroll
  for (int i = 0; i < NT; ++i) {
#pragma unroll
    for (int jj = 0; jj < NJ; ++jj) {
      const int64_t col = w.n0 + r0 + jj * 32 + lr;
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int64_t row = w.m0 + t0 + i * 32 + 8 * (v >> 2) + 4 * h + (v & 3);
        if (row < M && col < out_f) store_y<YT>(y, row * out_f + col, acc[i][jj][v]);
      }
    }
  }
}

// GG: W is GGUF half-blocks (`blocks`, 46 bytes per 32 elements, row-major;
// the dict stream pointers are unused), decoded with the zero marker
// (bf16x_gguf_block.py:76-87).  Otherwise W is the packed dict.
template <bool GG, bool EXACT, bool YF32>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void gemm_ws_kernel(
    const uint16_t* __restrict__ x, int64_t M, const uint32_t* __restrict__ sign,
    const uint32_t* __restrict__ mant, const uint32_t* __restrict__ delta, const uint16_t* __restrict__ emax2,
    const uint8_t* __restrict__ blocks, const uint32_t* __restrict__ kp_off, const uint32_t* __restrict__ kp_ent,
    int64_t out_f, int64_t in_f, WsGrid grid, void* __restrict__ y, float* __restrict__ part) {
  __shared__ __attribute__((aligned(16))) uint8_t wlds[2 * kWSlot];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  const int S = (int)(in_f >> 6);
  const WsWork wk = ws_work(grid, S);           // units are steps
  const int64_t m0 = wk.m0, n0 = wk.n0;
  const int s0 = wk.u0;
  const int n = wk.nu;                          // steps of this block (>= 1)

  if (wave >= 4) {
    // ===================== staging waves =====================
    const int pw = wave - 4;                    // 0..3
    const int64_t P = in_f >> 5;                // atoms per row
    const int r = 32 * pw + (lane & 31), a = lane >> 5;
    using RawT = typename std::conditional<GG, RawG, Raw>::type;
    const uint64_t wat = (uint64_t)(out_f - n0) * P;   // atoms from the tile's first row
    __amdgpu_buffer_rsrc_t rs_, rm_, rd_, re_, rb_;
    uint32_t vo_s = 0, vo_m = 0, vo_d = 0, vo_e = 0, vo_b = 0, sh = 0;
    // rows past out_f read zeros (buffer range check on the vector offset);
    // their outputs are not stored
    const uint32_t av = (uint32_t)(r * P) + (uint32_t)a;
    if constexpr (GG) {
      // the tile's first block starts at a multiple of 4 bytes (n0 % 128 == 0);
      // the range is the rest of the blocks rounded up to 4 bytes, which the
      // caller guarantees readable.  Block (r, 2s + a) is at av * 46 + s * 92:
      // its offset modulo 4 (0 or 2) does not depend on s.
      rb_ = rsrc(blocks + (uint64_t)n0 * P * 46, (wat * 46 + 3) & ~3ull);
      vo_b = av * 46;
      sh = (vo_b & 2u) * 8u;
      vo_b &= ~3u;
    } else {
      rs_ = rsrc(sign + n0 * P, wat * 4);
      rm_ = rsrc(mant + n0 * P * 7, wat * 28);
      rd_ = rsrc(delta + n0 * P * 3, wat * 12);
      re_ = rsrc(emax2 + n0 * P, wat * 2);
      vo_s = av * 4; vo_m = av * 28; vo_d = av * 12; vo_e = (uint32_t)(r * P) * 2;
    }
    auto load_atoms = [&](int j, RawT& t) {
      const uint32_t s = (uint32_t)(s0 + min(j, n - 1));
      if constexpr (GG) {
        t.q0 = __builtin_amdgcn_raw_buffer_load_b128(rb_, (int)vo_b, (int)(s * 92), 0);
        t.q1 = __builtin_amdgcn_raw_buffer_load_b128(rb_, (int)(vo_b + 16), (int)(s * 92), 0);
        t.q2 = __builtin_amdgcn_raw_buffer_load_b128(rb_, (int)(vo_b + 32), (int)(s * 92), 0);
      } else {
        const u32x4 m03 = __builtin_amdgcn_raw_buffer_load_b128(rm_, (int)vo_m, (int)(s * 56), 0);
        const u32x3 m46 = __builtin_amdgcn_raw_buffer_load_b96(rm_, (int)(vo_m + 16), (int)(s * 56), 0);
        const u32x3 d02 = __builtin_amdgcn_raw_buffer_load_b96(rd_, (int)vo_d, (int)(s * 24), 0);
        t.s = __builtin_amdgcn_raw_buffer_load_b32(rs_, (int)vo_s, (int)(s * 8), 0);
        // the full dword (both atoms' emax pairs) is kept raw until the decode:
        // a value computed from a load at the load site makes the compiler wait
        // for it there
        t.ew = __builtin_amdgcn_raw_buffer_load_b32(re_, (int)vo_e, (int)(s * 4), 0);
        const uint32_t c0 = m03.x, c1 = m03.y, c2 = m03.z, c3 = m03.w, c4 = m46.x, c5 = m46.y, c6 = m46.z;
        t.m[0] = c0; t.m[1] = c1; t.m[2] = c2; t.m[3] = c3; t.m[4] = c4; t.m[5] = c5; t.m[6] = c6;
        const uint32_t e0 = d02.x, e1 = d02.y, e2 = d02.z;
        t.d[0] = e0; t.d[1] = e1; t.d[2] = e2;
      }
    };
    const int wst = r * kRowB;                  // this lane's W row in slot 0
    auto store_w = [&](const RawT& w, int slot) {
      uint32_t p[16];
      if constexpr (GG) {
        decode_pairs<true>(gguf_atom(GgufRaw{w.q0, w.q1, w.q2, sh}), p);
      } else {
        Atom t;
        t.s = w.s;
#pragma unroll
        for (int i = 0; i < 7; ++i) t.m[i] = w.m[i];
#pragma unroll
        for (int i = 0; i < 3; ++i) t.d[i] = w.d[i];
        t.e = (uint16_t)(w.ew >> (16 * a));
        decode_pairs(t, p);
      }
      // chunk c = pairs 4c .. 4c+3 as decoded: K order kchunk(c), as x_op writes x
#pragma unroll
      for (int c = 0; c < 4; ++c)
        *(u32x4*)(wlds + wst + slot * kWSlot + swz(r, 4 * a + c) * 16) =
            u32x4{p[4 * c], p[4 * c + 1], p[4 * c + 2], p[4 * c + 3]};
    };

    // EXACT plan: run of this wave's 32-row group at step s
    const int64_t G = (out_f + 31) / 32, G2 = 2 * G;
    const int64_t g = min(n0 / 32 + pw, G);
    uint32_t kp_total = 0;
    if constexpr (EXACT) kp_total = kp_off[S * G2];
    const __amdgpu_buffer_rsrc_t rent = rsrc(kp_ent, (uint64_t)kp_total * 4);
    const __amdgpu_buffer_rsrc_t roff = rsrc(kp_off, ((uint64_t)S * G2 + 1) * 4);
    const uint32_t ob = (uint32_t)(2 * g) * 4, oe = (uint32_t)min(2 * g + 2, G2) * 4;
    struct Off { uint32_t beg, end; };
    struct Ent { uint32_t beg, end, e0, e1; };
    auto load_off = [&](int j, Off& o) {
      const uint32_t s = (uint32_t)(s0 + min(j, n - 1));
      o.beg = __builtin_amdgcn_raw_buffer_load_b32(roff, (int)ob, (int)(s * G2 * 4), 0);
      o.end = __builtin_amdgcn_raw_buffer_load_b32(roff, (int)oe, (int)(s * G2 * 4), 0);
    };
    auto load_ent = [&](const Off& o, Ent& e) {
      e.beg = __builtin_amdgcn_readfirstlane(o.beg);
      e.end = __builtin_amdgcn_readfirstlane(o.end);
      e.e0 = __builtin_amdgcn_raw_buffer_load_b32(rent, (int)((e.beg + lane) * 4), 0, 0);
      e.e1 = __builtin_amdgcn_raw_buffer_load_b32(rent, (int)((e.beg + lane + 64) * 4), 0, 0);
    };
    // The entry is used outside the branch first (the empty asm), so the
    // compiler waits for its load there with an exact count: a loaded value
    // first used under a divergent branch makes it wait for every
    // outstanding load.
    auto patch_one = [&](uint32_t e, int slot, bool live) {
      const int rr = (int)(e >> 22) & (kBN - 1), c = (int)(e >> 16) & 63;
      const uint32_t dst = (uint32_t)(slot * kWSlot + rr * kRowB + swz(rr, chunk_of(c)) * 16 + pos_of(c) * 2);
      __asm__ volatile("" : "+v"(e));
      if (live) *(uint16_t*)(wlds + dst) = (uint16_t)(e & 0xFFFFu);
    };
    auto patch = [&](const Ent& e, int slot) {
      patch_one(e.e0, slot, e.beg + lane < e.end);
      patch_one(e.e1, slot, e.beg + lane + 64 < e.end);
      for (uint32_t k = e.beg + 128 + lane; k < e.end; k += 64)   // dense runs (rare)
        patch_one(kp_ent[k], slot, true);
    };

    RawT A0, A1;
    Off O0{}, O1{};
    Ent E0{}, E1{};
    // prologue: the requests of steps 0 and 1 (atoms, plan entries), step 0
    // decoded, the requests of step 2.  The loads in flight at the loop entry
    // are then the requests of 1 and 2, the pattern at the top of every
    // iteration, so the waits the compiler derives hold on both paths into
    // the loop
    if constexpr (EXACT) {
      load_off(0, O0);
      load_off(1, O1);
    }
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (EXACT) { load_ent(O0, E0); load_off(2, O0); }
    load_atoms(0, A0);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (EXACT) { load_ent(O1, E1); load_off(3, O1); }
    load_atoms(1, A1);
    __builtin_amdgcn_sched_barrier(0);
    store_w(A0, 0);
    if constexpr (EXACT) patch(E0, 0);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (EXACT) { load_ent(O0, E0); load_off(4, O0); }
    load_atoms(2, A0);
    __builtin_amdgcn_sched_barrier(0);
    __syncthreads();

    // iteration j: step j + 1 decoded (W slot (j + 1) & 1) from its register
    // set, then the atoms of j + 3 requested into that set with the plan
    // entries of j + 3 and the offsets of j + 5
    auto iter = [&](int j, RawT& at, Off& o, Ent& e, int slot) {
      store_w(at, slot);
      if constexpr (EXACT) patch(e, slot);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (EXACT) { load_ent(o, e); load_off(j + 5, o); }
      load_atoms(j + 3, at);
      __builtin_amdgcn_sched_barrier(0);
      __syncthreads();
    };
    int j = 0;
    for (; j + 1 < n; j += 2) {
      iter(j, A1, O1, E1, 1);
      iter(j + 1, A0, O0, E0, 0);
    }
    if (j < n) iter(j, A1, O1, E1, 1);
    return;
  }

  // ===================== MFMA waves =====================
  const int lr = lane & 31, h = lane >> 5;
  // x operand of token tile i, k-quarter q at step s: 1 KB of x in operand
  // order (x_op_kernel), lane l's 16 bytes at l * 16.  The block's tiles
  // start at tile m0 / 32; rows past M hold zeros (outputs not stored).
  const int64_t S64 = S;
  const __amdgpu_buffer_rsrc_t rx_ = rsrc(x + m0 * in_f, (uint64_t)(((M + 31) / 32) * 32 - m0) * (uint64_t)in_f * 2);
  const uint32_t vx0 = (uint32_t)(2 * wave * S64 * 4096 + lane * 16);
  const uint32_t vx1 = vx0 + (uint32_t)(S64 * 4096);
  // the x operands of one step: [token tile][k-quarter]
  auto load_x = [&](int j, bf16x8_t (&X)[2][4]) {
    const uint32_t ks = (uint32_t)(s0 + min(j, n - 1)) * 4096;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(rx_, (int)((i ? vx1 : vx0) + q * 1024), (int)ks, 0);
        X[i][q] = __builtin_bit_cast(bf16x8_t, v);
      }
  };
  // W operand of W tile jj, k-quarter q (the swizzle term depends on lr only)
  uint32_t wo[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) wo[q] = (uint32_t)(lr * kRowB + swz(lr, 4 * h + q) * 16);
  auto load_w = [&](int q, int ws, bf16x8_t (&wb)[4]) {
#pragma unroll
    for (int jj = 0; jj < 4; ++jj) wb[jj] = *(const bf16x8_t*)(wlds + wo[q] + ws * kWSlot + jj * 32 * kRowB);
  };
  f32x16 acc[2][4];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int jj = 0; jj < 4; ++jj)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][jj][v] = 0.f;
  auto mfma = [&](int t, const bf16x8_t (&X)[2][4], int q, const bf16x8_t (&wb)[4]) {
    const int i = t >> 2, jj = t & 3;
    acc[i][jj] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(X[i][q], wb[jj], acc[i][jj], 0, 0, 0);
  };
#define BF16X_SG(mask, cnt) __builtin_amdgcn_sched_group_barrier(mask, cnt, 0)
  bf16x8_t X0[2][4], X1[2][4], W0[4], W1[4];
  // one step from W slot ws with x in X; x of step j + 1 requested into Xn
  // (the set the previous step used) at the start
  auto step = [&](int j, int ws, const bf16x8_t (&X)[2][4], bf16x8_t (&Xn)[2][4]) {
    load_x(j + 1, Xn);
    // quarter 0: the next quarter's W reads, then 8 MFMAs
    load_w(1, ws, W1);
#pragma unroll
    for (int t = 0; t < 8; ++t) mfma(t, X, 0, W0);
    BF16X_SG(0x020, 8);
    BF16X_SG(0x100, 4);
    BF16X_SG(0x008, 8);
    __builtin_amdgcn_sched_barrier(0);
    load_w(2, ws, W0);
#pragma unroll
    for (int t = 0; t < 8; ++t) mfma(t, X, 1, W1);
    BF16X_SG(0x100, 4);
    BF16X_SG(0x008, 8);
    __builtin_amdgcn_sched_barrier(0);
    load_w(3, ws, W1);
#pragma unroll
    for (int t = 0; t < 8; ++t) mfma(t, X, 2, W0);
    BF16X_SG(0x100, 4);
    BF16X_SG(0x008, 8);
    __builtin_amdgcn_sched_barrier(0);
    // last quarter: 4 MFMAs, the barrier, the next step's quarter-0 W reads
    // under the other 4
#pragma unroll
    for (int t = 0; t < 4; ++t) mfma(t, X, 3, W1);
    __builtin_amdgcn_sched_barrier(0);
    __syncthreads();
    load_w(0, ws ^ 1, W0);
#pragma unroll
    for (int t = 4; t < 8; ++t) mfma(t, X, 3, W1);
    BF16X_SG(0x100, 4);
    BF16X_SG(0x008, 4);
    __builtin_amdgcn_sched_barrier(0);
  };
#undef BF16X_SG
  load_x(0, X0);
  __syncthreads();
  load_w(0, 0, W0);
  int j = 0;
  for (; j + 1 < n; j += 2) {
    step(j, 0, X0, X1);
    step(j + 1, 1, X1, X0);
  }
  if (j < n) step(j, 0, X0, X1);
  ws_store<YF32 ? kYF32 : kYBf16, 2, 4, 4>(acc, wk, wave, lane, M, out_f, grid.ltiles, y, part);
}

// ---------------------------------------------------------------------------
// Four-step groups (in_f % 256 == 0): the kernel above with the W tile of one
// barrier interval 256 columns wide (64 KB per slot, two slots), so that the
// decode waves read runs of consecutive atoms of a row.  In round i (0..3)
// lane l of decode wave 4 + p takes tile row 32p + 8i + l/8 and atom l%8 of
// the group: a load instruction reads 8 rows x 8 consecutive atoms (368
// contiguous bytes of a GGUF row, 224 of a mantissa stream) instead of 32
// rows x 2 atoms, about 1.7x fewer cache lines per instruction (a timing copy
// of the one-step kernel with this access pattern ran 11-24 % faster).  Each
// round's registers are refilled with the next group's atoms as soon as they
// are decoded, so one set of 4 rounds is in flight while the other is decoded.
// Tile rows are 512 bytes; 16-byte chunk c of row r sits at
// c ^ (((c >> 4) & 1) << 1) ^ (r & 15): the MFMA waves' reads (16 rows, one
// chunk) and the decode waves' writes (2 rows x 8 atoms, one chunk of each)
// each touch 16 different 16-byte bank groups.  The MFMA waves run the
// one-step kernel's step four times per barrier.
//
// Tiles of 256, 128 or 64 tokens: MFMA wave c owns NT 32-token tiles of token
// group c % TG and 32 TG rows of row group c / TG (256: NT 2, TG 4; 128: NT 1,
// TG 4; 64: NT 1, TG 2).  With fewer MFMAs per tile the decode sets the pace,
// so the 128- and 64-token tiles decode with ND = 8 waves of 16 rows.  What
// bounds them (work-skipping copies, 14336x4096 saturated, 64 tokens, the
// kernel alone): 29 us whole, 25.7 without the MFMAs and their operand loads,
// 23.7 also without the decode arithmetic, 19.8 whole without the atom loads;
// the decode's VALU is 1.0 us of a group's 2.6 us per SIMD (137 instructions
// per atom, two decode waves), and launch, first loads and the partial tiles
// are 9 us.  Two 64-row blocks per CU (16 waves) were no faster (M = 101: 49.8
// against 49.8 us).  Calls against the tiled kernel these tiles replace:
// 14336x4096 M = 101 66.7 -> 44 us, 6144x4096 40.5 -> 28.5, 4096x4096 30.6 ->
// 23.3; 4096x14336 59.6 -> 38.4 (on one weight, partly cached).
// ---------------------------------------------------------------------------
constexpr int kGroup = 4;                    // 64-column steps per group
constexpr int kRowB4 = kGroup * kRowB;       // 512 bytes per tile row
constexpr int kWSlot4 = kBN * kRowB4;        // 64 KB

__device__ __forceinline__ int swz4(int row, int chunk) { return chunk ^ (((chunk >> 4) & 1) << 1) ^ (row & 15); }

template <bool GG, bool EXACT, int YT, int NT, int TG, int ND, int NX>
__global__ __launch_bounds__(64 * (4 + ND)) __attribute__((amdgpu_waves_per_eu((4 + ND) / 4, (4 + ND) / 4)))
void gemm_ws4_kernel(
    const uint16_t* __restrict__ x, int64_t M, const uint32_t* __restrict__ sign,
    const uint32_t* __restrict__ mant, const uint32_t* __restrict__ delta, const uint16_t* __restrict__ emax2,
    const uint8_t* __restrict__ blocks, const uint32_t* __restrict__ kp_off, const uint32_t* __restrict__ kp_ent,
    int64_t out_f, int64_t in_f, WsGrid grid, void* __restrict__ y, float* __restrict__ part) {
  constexpr int NJ = TG;                        // 32-row W tiles per MFMA wave
  constexpr int NR = 16 / ND;                   // rounds of a group per decode wave
  // two W slots, then 256 bytes where the plan patch lanes with no entry write
  __shared__ __attribute__((aligned(16))) uint8_t wlds[2 * kWSlot4 + 256];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  const int S = (int)(in_f >> 6);
  const WsWork wk = ws_work(grid, S / kGroup);  // units are groups
  const int64_t m0 = wk.m0, n0 = wk.n0;
  const int g0 = wk.u0;
  const int ng = wk.nu;                         // groups of this block (>= 1)

  if (wave >= 4) {
    // ===================== decode waves =====================
    const int pw = wave - 4;                    // 0 .. ND - 1
    const int64_t P = in_f >> 5;                // atoms per row (a multiple of 8)
    const int a = lane & 7, rq = lane >> 3;     // atom of the group, row within a round
    using RawT = typename std::conditional<GG, RawG, Raw>::type;
    const uint64_t wat = (uint64_t)(out_f - n0) * P;
    __amdgpu_buffer_rsrc_t rs_, rm_, rd_, re_, rb_;
    uint32_t vo_s = 0, vo_m = 0, vo_d = 0, vo_e = 0, vo_b = 0, sh = 0;
    // round 0's atom from the tile's first atom; rows past out_f read zeros
    // (buffer range check), their outputs are not stored
    const uint32_t av = (uint32_t)((8 * NR * pw + rq) * P) + (uint32_t)a;
    const uint32_t rstep = (uint32_t)(8 * P);   // atoms from one round's row to the next
    if constexpr (GG) {
      // P is even, so block av sits at av * 46, which is 2 (a & 1) modulo 4
      rb_ = rsrc(blocks + (uint64_t)n0 * P * 46, (wat * 46 + 3) & ~3ull);
      vo_b = (av * 46) & ~3u;
      sh = 16u * (uint32_t)(a & 1);
    } else {
      rs_ = rsrc(sign + n0 * P, wat * 4);
      rm_ = rsrc(mant + n0 * P * 7, wat * 28);
      rd_ = rsrc(delta + n0 * P * 3, wat * 12);
      re_ = rsrc(emax2 + n0 * P, wat * 2);
      vo_s = av * 4; vo_m = av * 28; vo_d = av * 12; vo_e = (av & ~1u) * 2;
    }
    // the atoms of round i of group gj (clamped to the block's last group)
    auto load_round = [&](int gj, int i, RawT& t) {
      const uint32_t ra = (uint32_t)(g0 + min(gj, ng - 1)) * 8u + (uint32_t)i * rstep;
      if constexpr (GG) {
        t.q0 = __builtin_amdgcn_raw_buffer_load_b128(rb_, (int)vo_b, (int)(ra * 46), 0);
        t.q1 = __builtin_amdgcn_raw_buffer_load_b128(rb_, (int)(vo_b + 16), (int)(ra * 46), 0);
        t.q2 = __builtin_amdgcn_raw_buffer_load_b128(rb_, (int)(vo_b + 32), (int)(ra * 46), 0);
      } else {
        const u32x4 m03 = __builtin_amdgcn_raw_buffer_load_b128(rm_, (int)vo_m, (int)(ra * 28), 0);
        const u32x3 m46 = __builtin_amdgcn_raw_buffer_load_b96(rm_, (int)(vo_m + 16), (int)(ra * 28), 0);
        const u32x3 d02 = __builtin_amdgcn_raw_buffer_load_b96(rd_, (int)vo_d, (int)(ra * 12), 0);
        t.s = __builtin_amdgcn_raw_buffer_load_b32(rs_, (int)vo_s, (int)(ra * 4), 0);
        t.ew = __builtin_amdgcn_raw_buffer_load_b32(re_, (int)vo_e, (int)(ra * 2), 0);
        const uint32_t c0 = m03.x, c1 = m03.y, c2 = m03.z, c3 = m03.w, c4 = m46.x, c5 = m46.y, c6 = m46.z;
        t.m[0] = c0; t.m[1] = c1; t.m[2] = c2; t.m[3] = c3; t.m[4] = c4; t.m[5] = c5; t.m[6] = c6;
        const uint32_t e0 = d02.x, e1 = d02.y, e2 = d02.z;
        t.d[0] = e0; t.d[1] = e1; t.d[2] = e2;
      }
    };
    auto store_round = [&](const RawT& w, int i, int slot) {
      uint32_t p[16];
      if constexpr (GG) {
        decode_pairs<true>(gguf_atom(GgufRaw{w.q0, w.q1, w.q2, sh}), p);
      } else {
        Atom t;
        t.s = w.s;
#pragma unroll
        for (int k = 0; k < 7; ++k) t.m[k] = w.m[k];
#pragma unroll
        for (int k = 0; k < 3; ++k) t.d[k] = w.d[k];
        t.e = (uint16_t)(w.ew >> (16 * (a & 1)));
        decode_pairs(t, p);
      }
      const int r = 8 * NR * pw + 8 * i + rq;
      uint8_t* row = wlds + slot * kWSlot4 + r * kRowB4;
#pragma unroll
      for (int c = 0; c < 4; ++c)
        *(u32x4*)(row + swz4(r, 4 * a + c) * 16) = u32x4{p[4 * c], p[4 * c + 1], p[4 * c + 2], p[4 * c + 3]};
    };

    // EXACT plan: the runs of this wave's 16-row groups at the 4 steps of a
    // group, taken as one list of their concatenated entries: entry t belongs
    // to step u(t) = (t >= c[0]) + (t >= c[1]) + (t >= c[2]).  Lane l loads
    // entries l, l + 64, .. ahead: NE of them in any case (one entry in 32
    // elements, more than a dict's 1 in 43 to 108), and up to NP where the list
    // goes on, a uniform branch each.  A GGUF table has every element seven
    // steps down in it, 1 in 22 to 54, and most of its lists are longer: with
    // the rest of them loaded where they are written, each such load draining
    // the atoms in flight, 14336x4096 lossless took 83.4 us at M = 300 (74.1
    // here) and 39.0 at M = 64 (36.0).
    constexpr int NE = ND == 4 ? 4 : 2, NP = 2 * NE;
    const int64_t G2 = 2 * ((out_f + 31) / 32);
    const int64_t gr = min(n0 / 16 + (NR / 2) * pw, G2);
    uint32_t kp_total = 0;
    if constexpr (EXACT) kp_total = kp_off[S * G2];
    const __amdgpu_buffer_rsrc_t rent = rsrc(kp_ent, (uint64_t)kp_total * 4);
    const __amdgpu_buffer_rsrc_t roff = rsrc(kp_off, ((uint64_t)S * G2 + 1) * 4);
    // lane 2u + b: the start (b = 0) or end of step u's run
    const uint32_t vo_o =
        (uint32_t)(((lane >> 1) & 3) * G2 + ((lane & 1) ? min(gr + NR / 2, G2) : gr)) * 4;
    struct Ent { uint32_t b[kGroup], c[kGroup], e[NP]; };   // run starts, ends within the list, entries
    auto load_off = [&](int gj) {
      return __builtin_amdgcn_raw_buffer_load_b32(
          roff, (int)vo_o, (int)((uint32_t)(g0 + min(gj, ng - 1)) * kGroup * (uint32_t)G2 * 4u), 0);
    };
    auto addr_of = [&](const Ent& t, uint32_t k) {
      return k + (k < t.c[0] ? t.b[0] : k < t.c[1] ? t.b[1] - t.c[0] : k < t.c[2] ? t.b[2] - t.c[1]
                                                                                 : t.b[3] - t.c[2]);
    };
    auto load_ent = [&](uint32_t o, Ent& t) {
      uint32_t n_ent = 0;
#pragma unroll
      for (int u = 0; u < kGroup; ++u) {
        t.b[u] = __builtin_amdgcn_readlane(o, 2 * u);
        n_ent += __builtin_amdgcn_readlane(o, 2 * u + 1) - t.b[u];
        t.c[u] = n_ent;
      }
      auto load = [&](int k) {
        t.e[k] = __builtin_amdgcn_raw_buffer_load_b32(rent, (int)(addr_of(t, lane + 64 * k) * 4), 0, 0);
      };
#pragma unroll
      for (int k = 0; k < NE; ++k) load(k);
#pragma unroll
      for (int k = NE; k < NP; ++k)
        if (n_ent > 64u * k) load(k);
    };
    // entry -> its bf16 in the group tile; a lane past the list writes its
    // own word of the spare area instead (no exec-mask branch); the empty asm
    // makes the compiler wait for the entry's load there
    auto patch_one = [&](const Ent& t, uint32_t k, uint32_t e, int slot, bool live) {
      const int u = (k >= t.c[0]) + (k >= t.c[1]) + (k >= t.c[2]);
      const int rr = (int)(e >> 22) & (kBN - 1), c = (int)(e >> 16) & 63;
      const uint32_t dst =
          (uint32_t)(slot * kWSlot4 + rr * kRowB4 + swz4(rr, 8 * u + chunk_of(c)) * 16 + pos_of(c) * 2);
      __asm__ volatile("" : "+v"(e));
      *(uint16_t*)(wlds + (live ? dst : (uint32_t)(2 * kWSlot4 + lane * 4))) = (uint16_t)(e & 0xFFFFu);
    };
    auto patch = [&](const Ent& t, int slot) {
#pragma unroll
      for (int k = 0; k < NE; ++k) patch_one(t, lane + 64 * k, t.e[k], slot, lane + 64 * k < t.c[3]);
      if (t.c[3] > 64 * NE) {
#pragma unroll
        for (int k = NE; k < NP; ++k)
          if (t.c[3] > 64u * k) patch_one(t, lane + 64 * k, t.e[k], slot, lane + 64 * k < t.c[3]);
        for (uint32_t k = 64 * NP + lane; k < t.c[3]; k += 64)             // denser still: one load at a time
          patch_one(t, k, kp_ent[min(addr_of(t, k), kp_total - 1)], slot, true);
      }
    };

    RawT R[NR];
    uint32_t O = 0;
    Ent E[2] = {};
    // prologue: group 0's plan offsets and entries and group 1's offsets,
    // group 0's atoms; group 1's entries and group 2's offsets; group 0 decoded
    // round by round, each round's registers refilled with group 1's atoms.
    // The plan is requested ahead of the atoms everywhere (waits are in request
    // order), so waiting for a group's entries leaves the atoms requested
    // after them in flight.  One group of atoms ahead is enough: with two the
    // 8-decode-wave tiles were 1.3 us slower (14336x4096 M = 64: 39.9 against
    // 38.6), the second group only lengthening the prologue's burst.
    if constexpr (EXACT) O = load_off(0);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (EXACT) { load_ent(O, E[0]); O = load_off(1); }
#pragma unroll
    for (int i = 0; i < NR; ++i) load_round(0, i, R[i]);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (EXACT) { load_ent(O, E[1]); O = load_off(2); }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      store_round(R[i], i, 0);
      __builtin_amdgcn_sched_barrier(0);
      load_round(1, i, R[i]);
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (EXACT) patch(E[0], 0);
    __builtin_amdgcn_sched_barrier(0);
    __syncthreads();

    // iteration j: group j + 2's entries and group j + 3's offsets requested;
    // group j + 1 decoded into slot (j + 1) & 1, round by round, each round's
    // registers refilled with group j + 2's atoms; its entries patched
    auto iter = [&](int j, int slot) {
      if constexpr (EXACT) { load_ent(O, E[slot ^ 1]); O = load_off(j + 3); }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < NR; ++i) {
        store_round(R[i], i, slot);
        __builtin_amdgcn_sched_barrier(0);
        load_round(j + 2, i, R[i]);
        __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (EXACT) patch(E[slot], slot);
      __builtin_amdgcn_sched_barrier(0);
      __syncthreads();
    };
    int j = 0;
    for (; j + 1 < ng; j += 2) {
      iter(j, 1);
      iter(j + 1, 0);
    }
    if (j < ng) iter(j, 1);
    return;
  }

  // ===================== MFMA waves =====================
  const int lr = lane & 31, h = lane >> 5;
  const int n = ng * kGroup;                  // steps of this block
  const int s0 = g0 * kGroup;
  const int64_t S64 = S;
  const __amdgpu_buffer_rsrc_t rx_ = rsrc(x + m0 * in_f, (uint64_t)(((M + 31) / 32) * 32 - m0) * (uint64_t)in_f * 2);
  const int tw = wave % TG, jw = wave / TG;   // token group and W row group of this wave
  uint32_t vx[NT];
#pragma unroll
  for (int i = 0; i < NT; ++i) vx[i] = (uint32_t)((NT * tw + i) * S64 * 4096 + lane * 16);
  auto load_x = [&](int jx, bf16x8_t (&X)[NT][4]) {
    const uint32_t ks = (uint32_t)(s0 + min(jx, n - 1)) * 4096;
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(rx_, (int)(vx[i] + q * 1024), (int)ks, 0);
        X[i][q] = __builtin_bit_cast(bf16x8_t, v);
      }
  };
  // W operand of row tile jj, k-quarter q at step u of the group in slot
  // `slot`: chunk 8u + 4h + q of row jj*32 + lr.  The chunk's swizzle splits
  // into a per-lane part (wo[q]) and a constant of u, joined with one XOR;
  // the slot is bit 16 of the address and jj an immediate offset.
  uint32_t wo[4];
#pragma unroll
  for (int q = 0; q < 4; ++q)
    wo[q] = (uint32_t)((jw * NJ * 32 + lr) * kRowB4 + (((4 * h + q) ^ (lr & 15)) * 16));
  auto load_w = [&](int q, int u, int slot, bf16x8_t (&wb)[NJ]) {
    const uint32_t ku = (uint32_t)(((8 * u) ^ ((u >> 1) << 1)) * 16) | ((uint32_t)slot << 16);
    const uint32_t o = wo[q] ^ ku;
#pragma unroll
    for (int jj = 0; jj < NJ; ++jj) wb[jj] = *(const bf16x8_t*)(wlds + o + jj * 32 * kRowB4);
  };
  f32x16 acc[NT][NJ];
#pragma unroll
  for (int i = 0; i < NT; ++i)
#pragma unroll
    for (int jj = 0; jj < NJ; ++jj)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][jj][v] = 0.f;
  constexpr int NM = NT * NJ;                 // MFMAs per k-quarter
  if constexpr (NT == 1) {
    // Few MFMAs per k-quarter: a quarter's operands are requested into the
    // registers of the quarter just multiplied, WQ quarters (W, from LDS) and
    // XD steps (x) ahead, so an LDS read has at least eight MFMAs to arrive.
    // The group's last WQ quarters request the next group's operands: the
    // barrier comes before them, when all of this group's are in registers,
    // which also frees the slot for the decode waves early.  The ring fills
    // the 168 registers: the 128-token kernel spills 1-2 of them and the
    // two-term 64-token kernel 2-3 (8-16 bytes of scratch per lane).
    // NX = 2: x is two terms (hi, lo), both multiplied into the accumulator
    // (4096x4096 fp16 M = 64: 21.5 us for the call, 30.1 with the terms split
    // into 2 M rows and their results added by launches of their own).
    constexpr int WQ = NX == 2 ? (NJ == 4 ? 2 : 4) : (NJ == 4 ? 4 : 8), XD = NJ == 4 || NX == 2 ? 1 : 2;
    constexpr int kQ = 4 * kGroup;             // k-quarters of a group
    bf16x8_t X[XD][4][NX], W[WQ][NJ];
    const int64_t xrows = ((M + 31) / 32) * 32;
    const __amdgpu_buffer_rsrc_t rlo_ =
        rsrc(x + ((NX - 1) * xrows + m0) * in_f, (uint64_t)(xrows - m0) * (uint64_t)in_f * 2);
    auto load_xq = [&](int jx, int q, bf16x8_t (&d)[NX]) {
      const uint32_t ks = (uint32_t)(s0 + min(jx, n - 1)) * 4096;
#pragma unroll
      for (int t = 0; t < NX; ++t) {
        const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(t ? rlo_ : rx_, (int)(vx[0] + q * 1024), (int)ks, 0);
        d[t] = __builtin_bit_cast(bf16x8_t, v);
      }
    };
    auto group = [&](int jg, int slot) {
#pragma unroll
      for (int p = 0; p < kQ; ++p) {
        if (p == kQ - WQ) {
          __builtin_amdgcn_sched_barrier(0);
          __syncthreads();
          __builtin_amdgcn_sched_barrier(0);
        }
        const int u = p >> 2, q = p & 3, np = (p + WQ) % kQ;
#pragma unroll
        for (int t = 0; t < NX; ++t)
#pragma unroll
          for (int jj = 0; jj < NJ; ++jj)
            acc[0][jj] =
                __builtin_amdgcn_mfma_f32_32x32x16_bf16(X[u % XD][q][t], W[p % WQ][jj], acc[0][jj], 0, 0, 0);
        load_xq(4 * jg + u + XD, q, X[u % XD][q]);
        load_w(np & 3, np >> 2, p + WQ >= kQ ? slot ^ 1 : slot, W[p % WQ]);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
#pragma unroll
    for (int u = 0; u < XD; ++u)
#pragma unroll
      for (int q = 0; q < 4; ++q) load_xq(u, q, X[u][q]);
    __syncthreads();
#pragma unroll
    for (int p = 0; p < WQ; ++p) load_w(p & 3, p >> 2, 0, W[p]);
    __builtin_amdgcn_sched_barrier(0);
    int jg = 0;
    for (; jg + 1 < ng; jg += 2) {
      group(jg, 0);
      group(jg + 1, 1);
    }
    if (jg < ng) group(jg, 0);
  } else {
  auto mfma = [&](int t, const bf16x8_t (&X)[NT][4], int q, const bf16x8_t (&wb)[NJ]) {
    const int i = t / NJ, jj = t % NJ;
    acc[i][jj] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(X[i][q], wb[jj], acc[i][jj], 0, 0, 0);
  };
#define BF16X_SG(mask, cnt) __builtin_amdgcn_sched_group_barrier(mask, cnt, 0)
  bf16x8_t X0[NT][4], X1[NT][4], W0[NJ], W1[NJ];
  // step u of the group in `slot` (block step jx) with x in X; x of step
  // jx + 1 requested into Xn first.  The last quarter's second half reads
  // the next step's quarter-0 W operands: after the group's barrier from the
  // other slot at u == 3, from the same slot otherwise.
  auto step = [&](int jx, int u, int slot, const bf16x8_t (&X)[NT][4], bf16x8_t (&Xn)[NT][4]) {
    load_x(jx + 1, Xn);
    load_w(1, u, slot, W1);
#pragma unroll
    for (int t = 0; t < NM; ++t) mfma(t, X, 0, W0);
    BF16X_SG(0x020, 4 * NT);
    BF16X_SG(0x100, NJ);
    BF16X_SG(0x008, NM);
    __builtin_amdgcn_sched_barrier(0);
    load_w(2, u, slot, W0);
#pragma unroll
    for (int t = 0; t < NM; ++t) mfma(t, X, 1, W1);
    BF16X_SG(0x100, NJ);
    BF16X_SG(0x008, NM);
    __builtin_amdgcn_sched_barrier(0);
    load_w(3, u, slot, W1);
#pragma unroll
    for (int t = 0; t < NM; ++t) mfma(t, X, 2, W0);
    BF16X_SG(0x100, NJ);
    BF16X_SG(0x008, NM);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int t = 0; t < NM / 2; ++t) mfma(t, X, 3, W1);
    __builtin_amdgcn_sched_barrier(0);
    if (u == kGroup - 1) {
      __syncthreads();
      load_w(0, 0, slot ^ 1, W0);
    } else {
      load_w(0, u + 1, slot, W0);
    }
#pragma unroll
    for (int t = NM / 2; t < NM; ++t) mfma(t, X, 3, W1);
    BF16X_SG(0x100, NJ);
    BF16X_SG(0x008, NM - NM / 2);
    __builtin_amdgcn_sched_barrier(0);
  };
#undef BF16X_SG
  auto group = [&](int jg, int slot) {
    step(4 * jg + 0, 0, slot, X0, X1);
    step(4 * jg + 1, 1, slot, X1, X0);
    step(4 * jg + 2, 2, slot, X0, X1);
    step(4 * jg + 3, 3, slot, X1, X0);
  };
  load_x(0, X0);
  __syncthreads();
  load_w(0, 0, 0, W0);
  int jg = 0;
  for (; jg + 1 < ng; jg += 2) {
    group(jg, 0);
    group(jg + 1, 1);
  }
  if (jg < ng) group(jg, 0);
  }
  ws_store<YT, NT, TG, NJ>(acc, wk, wave, lane, M, out_f, grid.ltiles, y, part);
}

// x [M, K] -> operand order: 32-row tile T, step s (64 columns), k-quarter q
// is 1 KB at ((T * S + s) * 4 + q) * 1024, lane l = lr + 32 h holding row
// 32 T + lr, columns 64 s + 32 h + {4q, 16+4q, 4q+1, 17+4q, .., 4q+3, 19+4q}
// (the MFMA A operand of the fused kernels, in the K order of the W tile).
// Rows past M (up to the 32-row boundary) are zeros.  XT fp16 or fp32: two
// such matrices, hi = bf16(x) and, behind it, lo = bf16(x - hi).  One thread
// per 16-byte chunk (T, s, q, l): it reads the chunk's two runs of 4 columns
// and writes it (1 KB contiguous per wave; the four waves of a workgroup take
// the quarters of one (T, s), so a row's lines are shared in the L1).  At tens
// of rows the pass is a launch and one memory round trip: with a thread per
// row segment of 32 columns (a quarter of the threads, four chunks each)
// 64x4096 fp16
// took 5.2 us (3.0 here), 101x4096 bf16 4.0 (2.6), 512x4096 5.5 (4.4).
__device__ __forceinline__ u32x4 xo_chunk(u32x2 a, u32x2 b) {
  const uint32_t a0 = a.x, a1 = a.y, b0 = b.x, b1 = b.y;      // columns 4q .. 4q+3 and 16+4q .. 19+4q
  return u32x4{perm(b0, a0, 0x05040100u), perm(b0, a0, 0x07060302u), perm(b1, a1, 0x05040100u),
               perm(b1, a1, 0x07060302u)};
}
template <int XT>
__global__ __launch_bounds__(256) void x_op_kernel(const void* __restrict__ x, int64_t M, int64_t in_f,
                                                   int64_t chunks, u32x4* __restrict__ xo) {
  const uint32_t S = (uint32_t)(in_f / 64);      // (chunks < 2^28: x stays below 4 GiB)
  for (int64_t u = (int64_t)blockIdx.x * 256 + threadIdx.x; u < chunks; u += (int64_t)gridDim.x * 256) {
    const int l = (int)(u & 63), q = (int)(u >> 6) & 3;
    const uint32_t ts = (uint32_t)(u >> 8), T = ts / S, s = ts - T * S;
    const int64_t row = (int64_t)T * 32 + (l & 31);
    const int64_t e0 = row * in_f + s * 64 + (l >> 5) * 32 + 4 * q;
    u32x2 h[2] = {u32x2{0u, 0u}, u32x2{0u, 0u}}, r[2] = {u32x2{0u, 0u}, u32x2{0u, 0u}};
    if (row < M) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int64_t e = e0 + 16 * i;
        if constexpr (XT == BF16X_BF16) {
          const u32x2a v = *(const u32x2a*)((const uint16_t*)x + e);
          const uint32_t v0 = v.x, v1 = v.y;
          h[i] = u32x2{v0, v1};
        } else {
          float f[4];
          if constexpr (XT == BF16X_F16) {
            const u32x2a v = *(const u32x2a*)((const _Float16*)x + e);
            const uint32_t w[2] = {v.x, v.y};
            _Float16 t[4];
            __builtin_memcpy(t, w, 8);
#pragma unroll
            for (int k = 0; k < 4; ++k) f[k] = (float)t[k];
          } else {
            const u32x4a v = *(const u32x4a*)((const float*)x + e);
            const uint32_t w[4] = {v.x, v.y, v.z, v.w};
            __builtin_memcpy(f, w, 16);
          }
          uint32_t hi[4], lo[4];
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            hi[k] = f32_to_bf16_rne(f[k]);
            lo[k] = f32_to_bf16_rne(f[k] - __uint_as_float(hi[k] << 16));
          }
          h[i] = u32x2{hi[0] | (hi[1] << 16), hi[2] | (hi[3] << 16)};
          r[i] = u32x2{lo[0] | (lo[1] << 16), lo[2] | (lo[3] << 16)};
        }
      }
    }
    xo[u] = xo_chunk(h[0], h[1]);
    if constexpr (XT != BF16X_BF16) xo[u + chunks] = xo_chunk(r[0], r[1]);
  }
}

// y over the split tiles: the sum of each element's fp32 partials in K-range
// order (partial tile layout as ws_store writes it), one thread per four
// consecutive elements of the split tiles.
template <int YT>
__global__ __launch_bounds__(256) void ws_tile_reduce_kernel(const float* __restrict__ part, WsGrid g, int nsplit,
                                                             int64_t M, int64_t out_f, void* __restrict__ y,
                                                             bool yal) {
  // four columns of one tile row (kBN % 4 == 0): 16-byte
  // partial loads, an 8-byte (bf16) or 16-byte (fp32) store when the row's
  // four outputs are in range and aligned (yal: y is 16-byte aligned)
  // (at most resident blocks x 256 x 128 elements: 32-bit indexes)
  const uint32_t tsz = (uint32_t)(g.bm * kBN), count = (uint32_t)g.ltiles * tsz, mt = (uint32_t)g.mtiles;
  typedef float f32x4v __attribute__((ext_vector_type(4)));
  for (uint32_t i = (blockIdx.x * 256 + threadIdx.x) * 4; i < count; i += gridDim.x * 256 * 4) {
    const uint32_t lt = i / tsz, e = i - lt * tsz, tile = (uint32_t)g.full + lt;
    const int64_t row = (int64_t)(tile % mt) * g.bm + e / kBN;
    const int64_t col = (int64_t)(tile / mt) * kBN + e % kBN;
    if (row >= M || col >= out_f) continue;
    f32x4v s = *(const f32x4v*)(part + i);
    for (int k = 1; k < nsplit; ++k) s += *(const f32x4v*)(part + (int64_t)k * count + i);
    const float v[4] = {s.x, s.y, s.z, s.w};
    const int64_t o = row * out_f + col;
    if (yal && col + 3 < out_f && (o & 3) == 0) {
      if constexpr (YT == kYF32) {
        *(f32x4v*)((float*)y + o) = s;
      } else if constexpr (YT == kYF16) {
        typedef _Float16 f16x4v __attribute__((ext_vector_type(4)));
        *(f16x4v*)((_Float16*)y + o) = f16x4v{(_Float16)v[0], (_Float16)v[1], (_Float16)v[2], (_Float16)v[3]};
      } else {
        const uint32_t lo = f32_to_bf16_rne(v[0]) | (f32_to_bf16_rne(v[1]) << 16);
        const uint32_t hi = f32_to_bf16_rne(v[2]) | (f32_to_bf16_rne(v[3]) << 16);
        *(u32x2a*)((uint16_t*)y + o) = u32x2a{lo, hi};
      }
    } else {
      for (int c = 0; c < 4 && col + c < out_f; ++c) store_y<YT>(y, o + c, v[c]);
    }
  }
}

struct WsShape {
  WsGrid g;
  int nsplit;       // K ranges of a split tile (1: no split tiles)
  int64_t grid;     // blocks
  bool grouped;     // four-step-group kernel (units are groups, else steps)
};

// Four-step groups when K allows (the grouped kernel reads W in runs of
// consecutive atoms); BF16X_TUNE_GEMM_WS_GROUPED = 0 keeps the one-step kernel.
bool ws_grouped(int64_t in_f) {
  return (in_f / kStep) % kGroup == 0 && tuning(BF16X_TUNE_GEMM_WS_GROUPED) != 0;
}

// Resident blocks of the wave-specialised kernels: one per CU (128 KB of LDS,
// and 8 waves of 256 registers or 12 of 168); 256 CUs when there is no device to ask.
int64_t ws_resident() {
  static int64_t cache[64];
  int dev = 0, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  if (cache[dev] > 0) return cache[dev];
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0) return 256;
  cache[dev] = cus;
  return cus;
}

// Token rows per tile of the grouped kernel.  A tile of 64 tokens decodes its W
// rows in about the time of a 128-token tile (the decode sets the pace), a
// 256-token tile in a third more, so a tile covers all tokens up to 256.  Two
// smaller token tiles decode every W row twice and win only where that is a
// short part of the launch: where they still leave every CU at most one block
// before K is split (C / 4: shorter K ranges and smaller partials), and a
// block's K range is short: at most 12 column groups for a dict; for GGUF
// blocks, whose decode (46-byte blocks, twice the plan entries) takes longer,
// 4 with 64-token and 6 with 128-token tiles.
// Measured, exact, 64 / 128 / 256-token tiles (us): 14336x4096 M = 64 38.6 /
// 42.1 / 48.7, M = 128 52.8 / 45.3 / 51.1, M = 191 74.9 / 60.7 / 54.3;
// 4096x4096 (32 row tiles, two smaller tiles: 4 groups) M = 64 22.6 / 24.1 /
// 28.8, M = 128 23.8 / 24.9 / 29.5, M = 191 30.1 / 27.3 / 30.7.  Time of two
// 64-token tiles over one of 128 at M = 101, and of two of 128 over one of 256
// at M = 160, by groups: dict exact 5 0.97 / 0.89, 8 0.99 / 0.92, 12 1.05 /
// 1.02, 14 1.05 / 1.05 (saturated 0.90 / 0.86, 0.94 / 0.89, 0.94 / 1.00, 1.08
// / 1.01); GGUF lossless 4 0.99 / 0.98, 5 1.06 / 0.97, 6 1.09 / 1.03, 8 1.12 /
// 1.03, 14 1.27 / 1.16 (4096x14336: M = 101 48.4 against 38.3, M = 160 56.5
// against 48.4); without a table 5 1.01 / 0.96, 6 1.03 / 0.98, 8 1.00 / 1.01, 14
// 1.12 / 1.13.
constexpr int64_t kMaxSplit = 16;
int64_t ws_tile_rows(int64_t M, int64_t nt, int64_t units, int64_t C, bool terms, bool gg) {
  const int64_t t = tuning(BF16X_TUNE_GEMM_WS_BM);
  if (t == 64 || t == 128 || (t == 256 && !terms)) return t;
  for (int64_t bm = 64; bm < 256; bm *= 2) {
    const int64_t mt = (M + bm - 1) / bm;
    if (mt == 1) return bm;
    if (mt > 2 || mt * nt > C / 4) continue;
    const int64_t s = std::min<int64_t>(C / (mt * nt), kMaxSplit);      // (as ws_shape splits K)
    if ((units + s - 1) / s <= (!gg ? 12 : bm == 64 ? 4 : 6)) return bm;
  }
  return terms ? 128 : 256;    // two terms: the operands of a 256-token tile do not fit the registers
}

// Tiles run whole-K in full rounds of resident blocks; the f tiles of the
// last, partial round (all tiles when there are fewer than one round) are
// split into s = min(resident / f, 16) K ranges of at least one group (four
// steps for the one-step kernel) so that they fill that round:
// T = 896 tiles on 256 CUs run as 3 rounds of whole tiles and one round of
// 128 tiles x 2 half-K blocks (3.5 rounds instead of 4), with fp32 partials
// only for those 128 tiles.  BF16X_TUNE_GEMM_WS_SPLIT > 0 splits every tile
// into that many K ranges instead; BF16X_TUNE_GEMM_WS_RESIDENT > 0 replaces
// the resident block count (tests reach the mixed plan with few tiles).
WsShape ws_shape(int64_t M, int64_t out_f, int64_t in_f, bool terms, bool gg) {
  WsShape w;
  w.grouped = ws_grouped(in_f);
  const int64_t forced_c = tuning(BF16X_TUNE_GEMM_WS_RESIDENT);
  // (the reduction indexes the split tiles' elements in 32 bits)
  const int64_t C = forced_c > 0 ? std::min<int64_t>(forced_c, 32768) : ws_resident();
  const int64_t nt = (out_f + kBN - 1) / kBN;
  const int64_t S = in_f / kStep, units = w.grouped ? S / kGroup : S;
  const int64_t bm = w.grouped ? ws_tile_rows(M, nt, units, C, terms, gg) : kBM;
  const int64_t mt = (M + bm - 1) / bm, tiles = mt * nt;
  const int64_t max_split = std::max<int64_t>(1, std::min<int64_t>(kMaxSplit, w.grouped ? units : units / 4));
  int64_t f = tiles % C, s = f ? std::min<int64_t>(C / f, max_split) : 1;
  const int64_t forced = tuning(BF16X_TUNE_GEMM_WS_SPLIT);
  if (forced > 0 && tiles <= 32768) {
    f = tiles;
    s = std::min<int64_t>(forced, w.grouped ? units : S);
  }
  const int64_t lunits = (units + s - 1) / s, ks = (units + lunits - 1) / lunits;
  w.g.mtiles = (int)mt;
  w.g.bm = (int)bm;
  if (ks <= 1) {
    w.g.full = (int)tiles; w.g.ltiles = 0; w.g.lunits = (int)units; w.nsplit = 1;
    w.grid = tiles;
  } else {
    w.g.full = (int)(tiles - f); w.g.ltiles = (int)f; w.g.lunits = (int)lunits; w.nsplit = (int)ks;
    w.grid = (tiles - f) + f * ks;
  }
  return w;
}

}  // namespace
}  // namespace bf16x

using namespace bf16x;

namespace {
// workspace: x in operand order (rows rounded up to 32), then the split partials
int64_t ws_xop_bytes(int64_t M, int64_t in_f) { return ((M + 31) / 32) * 32 * in_f * 2; }
}  // namespace

// terms: x is fp16 or fp32, multiplied as two bf16 terms (grouped kernel only)
int64_t bf16x_gemm_ws_workspace(int64_t M, int64_t out_f, int64_t in_f, bool terms, bool gg) {
  const WsShape w = ws_shape(M, out_f, in_f, terms, gg);
  return ws_xop_bytes(M, in_f) * (terms ? 2 : 1) +
         (w.nsplit > 1 ? (int64_t)w.nsplit * w.g.ltiles * ((int64_t)w.g.bm * kBN) * 4 : 0);
}

// Launch of the wave-specialised kernel; arguments checked by the caller
// (bf16x_gemm and bf16x_gemm_terms for the packed dict; bf16x_gguf_gemm for
// GGUF blocks, given as `blocks` with the dict pointers null).  x_dtype fp16
// or fp32: two terms, y in x's type; otherwise yf32 says bf16 or fp32.
int bf16x_gemm_ws_launch(const void* x, int32_t x_dtype, int64_t M, const uint32_t* s, const uint32_t* m,
                         const uint32_t* d, const uint16_t* e, const uint8_t* blocks, const uint32_t* kp_off,
                         const uint32_t* kp_ent, int64_t out_f, int64_t in_f, bool exact, bool yf32, void* y,
                         void* workspace, int64_t workspace_bytes, hipStream_t st) {
  const bool terms = x_dtype != BF16X_BF16;
  const WsShape w = ws_shape(M, out_f, in_f, terms, blocks != nullptr);
  if (terms && (!w.grouped || blocks)) return BF16X_ESHAPE;
  const int64_t xop = ws_xop_bytes(M, in_f);
  if (!workspace || !aligned16(workspace) ||
      workspace_bytes < bf16x_gemm_ws_workspace(M, out_f, in_f, terms, blocks != nullptr))
    return BF16X_ECAPACITY;
  if (xop >= (int64_t)0xFFFFFFFF) return BF16X_ESHAPE;
  if (w.grid > INT32_MAX) return BF16X_ESHAPE;
  const int64_t chunks = xop / 16;
  const dim3 xg((unsigned)std::min<int64_t>((chunks + 255) / 256, 16384));
  if (x_dtype == BF16X_F16)
    hipLaunchKernelGGL(x_op_kernel<BF16X_F16>, xg, dim3(256), 0, st, x, M, in_f, chunks, (u32x4*)workspace);
  else if (x_dtype == BF16X_F32)
    hipLaunchKernelGGL(x_op_kernel<BF16X_F32>, xg, dim3(256), 0, st, x, M, in_f, chunks, (u32x4*)workspace);
  else
    hipLaunchKernelGGL(x_op_kernel<BF16X_BF16>, xg, dim3(256), 0, st, x, M, in_f, chunks, (u32x4*)workspace);
  const uint16_t* xo = (const uint16_t*)workspace;
  float* part = (float*)((uint8_t*)workspace + xop * (terms ? 2 : 1));
  const dim3 grid((unsigned)w.grid);
#define BF16X_WS4(GG_, EX_, YT_, NT_, TG_, ND_, NX_)                                                               \
  hipLaunchKernelGGL((gemm_ws4_kernel<GG_, EX_, YT_, NT_, TG_, ND_, NX_>), grid, dim3(64 * (4 + ND_)), 0, st, xo, M, \
                     s, m, d, e, blocks, kp_off, kp_ent, out_f, in_f, w.g, y, part)
#define BF16X_WS1(GG_, EX_, YF_)                                                                                   \
  do {                                                                                                           \
    if (!w.grouped)                                                                                              \
      hipLaunchKernelGGL((gemm_ws_kernel<GG_, EX_, YF_>), grid, dim3(512), 0, st, xo, M, s, m, d, e, blocks,        \
                         kp_off, kp_ent, out_f, in_f, w.g, y, part);                                              \
    else if (w.g.bm == 64) BF16X_WS4(GG_, EX_, (YF_ ? kYF32 : kYBf16), 1, 2, 8, 1);                                \
    else if (w.g.bm == 128) BF16X_WS4(GG_, EX_, (YF_ ? kYF32 : kYBf16), 1, 4, 8, 1);                               \
    else BF16X_WS4(GG_, EX_, (YF_ ? kYF32 : kYBf16), 2, 4, 4, 1);                                                 \
  } while (0)
#define BF16X_WSX(EX_, YT_)                                 \
  do {                                                      \
    if (w.g.bm == 64) BF16X_WS4(false, EX_, YT_, 1, 2, 8, 2); \
    else BF16X_WS4(false, EX_, YT_, 1, 4, 8, 2);            \
  } while (0)
#define BF16X_WS(GG_)                                        \
  do {                                                       \
    if (exact) {                                             \
      if (yf32) BF16X_WS1(GG_, true, true);                  \
      else BF16X_WS1(GG_, true, false);                      \
    } else {                                                 \
      if (yf32) BF16X_WS1(GG_, false, true);                 \
      else BF16X_WS1(GG_, false, false);                     \
    }                                                        \
  } while (0)
  const int yt = terms ? (x_dtype == BF16X_F16 ? kYF16 : kYF32) : (yf32 ? kYF32 : kYBf16);
  if (terms) {
    if (yt == kYF16) { if (exact) BF16X_WSX(true, kYF16); else BF16X_WSX(false, kYF16); }
    else { if (exact) BF16X_WSX(true, kYF32); else BF16X_WSX(false, kYF32); }
  } else if (blocks) {
    BF16X_WS(true);
  } else {
    BF16X_WS(false);
  }
#undef BF16X_WSX
#undef BF16X_WS
#undef BF16X_WS1
#undef BF16X_WS4
  if (w.nsplit > 1) {
    const int64_t count = (int64_t)w.g.ltiles * ((int64_t)w.g.bm * kBN);
    const int64_t blocks_r = std::min<int64_t>((count / 4 + 255) / 256, 4096);
#define BF16X_RED(YT_)                                                                                            \
  hipLaunchKernelGGL(ws_tile_reduce_kernel<YT_>, dim3((unsigned)blocks_r), dim3(256), 0, st, (const float*)part, w.g, \
                     w.nsplit, M, out_f, y, aligned16(y))
    if (yt == kYF32) BF16X_RED(kYF32);
    else if (yt == kYF16) BF16X_RED(kYF16);
    else BF16X_RED(kYBf16);
#undef BF16X_RED
  }
  return launch_status();
}
