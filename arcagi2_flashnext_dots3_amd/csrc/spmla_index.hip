// Indexer logits and exact top-k selection.
//
// Logits (dotsnote/engine/arcstats_pkg/arcstats/shard_logits_v2.py:49-123, shard_indexer.py:63-91; torch statement
// dotsnote/training/finetune/student.py:219-222):
//   logit[row][j] = min(sum_h w[row][h] * relu(q[row][h] . kcode[j]) * ks[j], 60000) for positions j < ctx[row]
//   (column j holds position j * P + rank of this rank's key store), -inf for j >= ctx (unless noinf); stored as fp32,
//   or rounded to fp16 (the reference's ARC_SHARD_F16OUT buffer, shard_indexer.py:28-29, :124).
//   gfx950: each wave loads the codes of its 32-key tiles straight into the registers of the MFMA B operand (three
//   tiles of loads in flight; the logits of a workgroup staged in LDS and written once its waves are done);
//   S = Q K^T on bf16 MFMA (32x32x16; e4m3 key codes convert exactly to bf16, two per instruction), 64 heads = 2 M
//   blocks, keys as the B operand; the head reduction is in-lane plus one cross-half exchange. (The fp8 MFMA would take the codes directly, but its internal accumulation keeps only
//   ~2^-12 of the largest product on gfx950, too coarse for the selection.)
//
// Top-k (dotsnote/engine/arcstats_pkg/arcstats/fast_topk.py:1-15, csrc/topk_select.cu:1-30 semantics):
//   per row, the K largest values among columns j < n = min(ctx, Lc) by torch's order-preserving key
//   (-0 < +0, NaN largest); equal keys -> lower column first; output positions sorted by (value desc, column asc),
//   -1 where the value is +-inf and in slots >= n. fp32 or fp16 logits: an fp16 key is the same order key of the
//   16-bit pattern placed in the top half of the 32-bit key (low half zero), so one radix code serves both.
//   gfx950: rows of up to 32768 columns, and up to 8 such chunks of a row, are selected and sorted by 4096 bins of the
//   value or the key (topk_row_kernel, topk_chunk_kernel). Longer rows, and the two stages of the rank-sharded selection, go
//   through 11/11/10-bit radix levels with an LDS histogram; keys above the boundary bin are appended at slots from a
//   block scan of per-thread counts (wave scans on DPP); once the boundary bin holds at most the candidate cap the
//   remaining levels run on those candidates alone; ties on the final key take the lowest columns. The K winners are
//   bitonic-sorted in LDS (only the stages whose pairs cross waves take a workgroup barrier); on the several-
//   workgroup path, whose lists arrive in column order, fp16 winners are ordered by a stable radix sort instead.
#include <type_traits>

#include "spmla_common.h"
#include <limits.h>
#include <algorithm>

namespace spmla {
namespace idx {

// torch's order-preserving key of an fp32 value (the top-k's radix key; -0 < +0, NaN largest)
__device__ inline uint32_t okey(float v) {
  const uint32_t x = f2u(v);
  if (v != v) return 0xffffffffu;
  return (x & 0x80000000u) ? ~x : (x | 0x80000000u);
}
// the same key for an fp16 pattern, in the top 16 bits (low 16 bits zero; NaN largest)
__device__ inline uint32_t okey16(uint32_t h) {
  if ((h & 0x7fffu) > 0x7c00u) return 0xffff0000u;
  return ((h & 0x8000u) ? (~h & 0xffffu) : (h | 0x8000u)) << 16;
}

// op over the 16 lanes of a row, in every lane of it: quad permutations and row mirrors
template <class T, class Op>
__device__ inline T row_reduce(T x, Op op) {
  auto dpp = [](T y, auto ctrl) {
    return __builtin_bit_cast(T, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, y), decltype(ctrl)::value, 0xf, 0xf, false));
  };
  x = op(x, dpp(x, std::integral_constant<int, 0xb1>()));      // quad_perm [1, 0, 3, 2]
  x = op(x, dpp(x, std::integral_constant<int, 0x4e>()));      // quad_perm [2, 3, 0, 1]
  x = op(x, dpp(x, std::integral_constant<int, 0x141>()));     // row_half_mirror
  return op(x, dpp(x, std::integral_constant<int, 0x140>()));  // row_mirror
}
template <bool MAX>
__device__ inline uint32_t row_minmax(uint32_t x) {
  return row_reduce(x, [](uint32_t a, uint32_t b) { return MAX ? (a > b ? a : b) : (a < b ? a : b); });
}
__device__ inline uint32_t lane_of(uint32_t x, int l) { return (uint32_t)__builtin_amdgcn_readlane((int)x, l); }
// Minimum / maximum over the wave (uniform): the four rows' results through readlane
template <bool MAX>
__device__ inline uint32_t wave_minmax(uint32_t x) {
  x = row_minmax<MAX>(x);
  const uint32_t a = lane_of(x, 0), b = lane_of(x, 16), c = lane_of(x, 32), d = lane_of(x, 48);
  return MAX ? max(max(a, b), max(c, d)) : min(min(a, b), min(c, d));
}
// ------------------------------------------------------------------------------------------------ logits
constexpr int LG_NWV = 8;                 // waves per logits workgroup (2 per SIMD: 256 registers each)
constexpr int LG_TPW = 16;                // 32-key tiles per wave and workgroup when the rows overfill the device

struct LogitParams {
  const uint16_t* q; long long q_st, q_sh;   // q[row][64][128] bf16
  const float* w; long long w_st;            // w[row][64]
  const uint8_t* store; long long R_local; int rpb; long long blk_stride;
  const int* bt; long long bt_st; int bs;    // block table [req][...], block size (positions per block)
  const int* req; const int* ctx;            // per row
  // per > 0 (req null): rows per request, row r belongs to request r / per; tail: ctx is per request and row r sees
  // per - 1 - r % per keys less
  int per, tail;
  int rows, Lc, P, rank, noinf;
  void* out; long long out_st;              // fp32, or fp16 (F16OUT); stride in elements
  int bs_sh, rpb_sh, p_sh;                   // log2 of bs, rpb, P when a power of two, else -1
  long long lim;                             // R_local * P (< 2^31): valid block-table positions lie below
  int clamp;                                 // 1: logits clamped at 60000 (shard kernels); 0: unclamped (paged)
  const int* lo;                             // optional per-row first valid position (flat layout: cu_seqlen_ks)
  const float* kscale; long long k_st;       // flat layout: key j codes at store + j * k_st, scale kscale[j]
  int tpg;                                   // 32-key tiles per workgroup (the launcher's lg_grid)
  int all;                                   // 1 (P == 1): columns below min(ctx, Lc) are written whatever noinf says
};

typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
__device__ inline uint32_t fp8lo_bf16x2(uint32_t w) {
  return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, 1.0f, false));
}
__device__ inline uint32_t fp8hi_bf16x2(uint32_t w) {
  return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, 1.0f, true));
}

// Logits workgroup: the waves of one CU (one workgroup per CU, so no later-dispatched workgroup waits behind an
// older one's issue priority) share a range of 32-key tiles of one row; each wave computes all 64 heads of one tile
// per step, its first tiles tb + w + k NW (NW = LG_NWV) and later ones claimed from an LDS counter. The key codes go straight from global memory into the
// registers of the MFMA B operand: lane (k, h) of a tile loads 16-byte chunks 2 kp + h (kp = 0..3) of key k, which
// are the key's dims 32 kp + 16 h .. + 15 in the order the operand takes them, and the key's scale. A wave keeps
// LG_D tiles of loads in flight: step t computes tile t, then loads the codes of tile t + LG_D (whose block-table
// entries were loaded at step t - LG_D) and the block-table entries of tile t + 2 LG_D, so the one wait of a step
// (for the loads of step t - LG_D) leaves LG_D - 1 steps of loads outstanding. A workgroup whose range holds at
// most LG_STAGE columns keeps its logits in LDS (with a per-tile mask of the columns to write) and writes them in
// one pass once every wave is done: the logit stores interleaved with the key reads cost 20% of the read rate at
// 131072 columns per row (measured on MI355X with a probe of the same access pattern: 181 us for the reads alone,
// 226 us with a 128-byte store per tile, 201 us with the stores staged to the end).
constexpr int LG_D = 3;                    // steps of loads in flight per wave
constexpr int LG_STAGE = 32768;            // columns a workgroup stages in LDS before writing them (128 KiB fp32)

// Key layouts: LY_ROW 132-byte rows [128 codes | scale] (the rank-sharded store); LY_SHUF vLLM's paged SHUFFLE
// layout (P = 1, rpb = keys per block): key t of a block has its 16-byte chunk c at (t / 16) * 2048 + (t % 16) * 16
// + 256 c and its scale at rpb * 128 + 4 t (dotsnote/engine/arcstats_pkg/arcstats/dsa_sm89.py:63-66); LY_FLAT the
// prefill gather: key j (column j) at store + j * k_st, scale kscale[j], valid for lo[row] <= j < ctx[row], no
// block table (dsa_sm89.py:97-118).
enum { LY_ROW = 0, LY_SHUF = 1, LY_FLAT = 2 };
typedef uint32_t u32x4u __attribute__((ext_vector_type(4), aligned(4)));   // 16 bytes at a 4-byte boundary
template <bool POW2, int LY, bool F16OUT = false>
__global__ void __launch_bounds__(LG_NWV * 64) logits_kernel(LogitParams p) {
  constexpr bool SHUF = LY == LY_SHUF, FLAT = LY == LY_FLAT;
  constexpr int D = LG_D;
  __shared__ float sbuf[LG_STAGE];                          // staged logits of the range's columns
  __shared__ uint32_t smask[LG_STAGE / 32];                 // per tile: the columns to write
  __shared__ int claim;                                     // next unclaimed tile of the range
  const int row = blockIdx.x;
  const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int lane = threadIdx.x & 63;
  const bool stage = 32LL * p.tpg <= LG_STAGE;              // uniform
  const int half = lane >> 5, l32 = lane & 31;
  const int rq = FLAT ? 0 : p.per ? row / p.per : p.req[row];
  const int ctx = p.tail ? p.ctx[rq] - (p.per - 1 - (row - rq * p.per)) : p.ctx[row];
  float* orow = (float*)p.out + (long long)row * p.out_st;            // fp32 output row
  _Float16* hrow = (_Float16*)p.out + (long long)row * p.out_st;      // fp16 output row
  auto put = [&](int j, float v) {
    if constexpr (F16OUT) hrow[j] = (_Float16)v;                       // round to nearest even (+-inf kept)
    else orow[j] = v;
  };
  // tiles [tb, te) of the row; keys j with j P + rank < ctx lie in tiles below tv (computed)
  const int tb = blockIdx.y * p.tpg;
  const int te = min(tb + p.tpg, (p.Lc + 31) >> 5);
  const long long nvalid = ctx > p.rank ? ((long long)ctx - p.rank + p.P - 1) / p.P : 0;   // keys below ctx
  const int tv = p.lim == 0 ? tb : (int)min((long long)te, max((long long)tb, (nvalid + 31) >> 5));
  const int nh = p.all ? min(ctx, p.Lc) : 0;                // columns the caller's top-k reads
  if (!p.noinf || p.all)                                                // keys of the range past ctx
    for (int j = 32 * tv + (int)threadIdx.x; j < 32 * te && j < (p.noinf ? nh : p.Lc); j += LG_NWV * 64)
      put(j, -__builtin_inff());
  if (tv <= tb) return;                                     // uniform over the workgroup: no barrier below
  if (threadIdx.x == 0) claim = tb + 2 * LG_D * LG_NWV;     // steps 0 .. 2 LG_D - 1 take tiles tb + k NW + w
  __syncthreads();
  const int* btr = FLAT ? nullptr : p.bt + (long long)rq * p.bt_st;
  const int lo = p.lo ? p.lo[row] : 0;
  // n / d, n % d: shifts when every divisor is a power of two (POW2), else 32-bit division
  auto dv = [&](uint32_t n, uint32_t d, int sh) -> uint32_t { return POW2 ? n >> sh : n / d; };
  auto md = [&](uint32_t n, uint32_t d, int sh) -> uint32_t { return POW2 ? n & (d - 1u) : n % d; };
  // positions without a block-table entry read the range's first entry (key 32 tb < nvalid: in range)
  const int* bt_dummy = FLAT ? nullptr : btr + dv((uint32_t)(32 * tb * p.P + p.rank), (uint32_t)p.bs, p.bs_sh);
  // key r of tile id: its position, and whether it is a key of the row (id < tv: tiles past tv are no tiles)
  auto key_pos = [&](int id, int r, uint32_t& pos) -> bool {
    const int j = 32 * id + r;
    const long long ps = (long long)j * p.P + p.rank;
    pos = (uint32_t)ps;
    return id < tv && j < p.Lc && ps < ctx && ps >= lo;
  };
  // the block-table entry of this lane's key of tile id (a load from the range's first entry when there is none;
  // the value is first read when the tile's codes are loaded, LG_D steps later)
  auto load_bt = [&](int id) -> int {
    if constexpr (FLAT) return 0;
    uint32_t pos;
    const bool in = key_pos(id, l32, pos);
    return *(in ? btr + dv(pos, (uint32_t)p.bs, p.bs_sh) : bt_dummy);
  };
  // the codes (chunks 2 kp + half) and scale of this lane's key of tile id; keys that are none read row 0
  auto load_codes = [&](int id, int blk, u32x4 (&c)[4], float& sc) -> bool {
    uint32_t pos;
    bool ok = key_pos(id, l32, pos);
    const uint8_t* rp;
    const float* sp;
    uint32_t cs;                                       // bytes from chunk c to chunk c + 1
    if (FLAT) {                                        // key pos itself (pos < Lc = number of keys)
      rp = p.store + (long long)(ok ? pos : 0u) * p.k_st;
      sp = p.kscale + (ok ? pos : 0u);
      cs = 16;
    } else {
      ok = ok && blk >= 0;
      const long long tt = (long long)blk * p.bs + md(pos, (uint32_t)p.bs, p.bs_sh);
      ok = ok && tt < p.lim;
      const uint32_t lrow = ok ? dv((uint32_t)tt, (uint32_t)p.P, p.p_sh) : 0u;   // p.lim > 0: row 0 exists
      const uint8_t* kblk = p.store + (long long)dv(lrow, (uint32_t)p.rpb, p.rpb_sh) * p.blk_stride;
      const uint32_t kt = md(lrow, (uint32_t)p.rpb, p.rpb_sh);
      rp = SHUF ? kblk + (kt >> 4) * 2048u + (kt & 15u) * 16u : kblk + kt * 132u;            // chunk 0
      sp = (const float*)(SHUF ? kblk + (uint32_t)p.rpb * 128u + 4u * kt : rp + 128);      // scale
      cs = SHUF ? 256u : 16u;
    }
#pragma unroll
    for (int kp = 0; kp < 4; ++kp) {
      const u32x4u v = *(const u32x4u*)(rp + cs * (uint32_t)(2 * kp + half));
      c[kp] = u32x4{v[0], v[1], v[2], v[3]};
    }
    sc = *sp;
    return ok;
  };

  // query fragments (bf16 A operand): M block m = heads 32m..32m+31 (lane head 32m + l32); k-pair kp covers dims
  // 32kp + 16half + 0..15, MFMA 2kp taking the first 8 and 2kp+1 the next 8 (same permutation as the key operand)
  const uint16_t* qr = p.q + (long long)row * p.q_st;
  bf16x8 qf[2][8];
  float wl[2][16];
#pragma unroll
  for (int m = 0; m < 2; ++m) {
    const uint16_t* src = qr + (long long)(32 * m + l32) * p.q_sh + 16 * half;
#pragma unroll
    for (int kp = 0; kp < 4; ++kp) {
      qf[m][2 * kp] = __builtin_bit_cast(bf16x8, *(const u32x4*)(src + 32 * kp));
      qf[m][2 * kp + 1] = __builtin_bit_cast(bf16x8, *(const u32x4*)(src + 32 * kp + 8));
    }
    // weights of this lane's C-layout heads (8(i/4) + 4half + i%4 in block m)
    const float myw = p.w[(long long)row * p.w_st + 32 * m + l32];
#pragma unroll
    for (int i = 0; i < 16; ++i) wl[m][i] = __shfl(myw, 8 * (i >> 2) + 4 * half + (i & 3), 64);
  }

  // step t computes tile t
  auto compute = [&](int id, const u32x4 (&c)[4], float sc, bool ok) {
    bf16x8 kb[8];
#pragma unroll
    for (int kp = 0; kp < 4; ++kp) {
      const u32x4 w4 = c[kp];
      i32x4 a0, a1;
      a0[0] = (int)fp8lo_bf16x2(w4[0]); a0[1] = (int)fp8hi_bf16x2(w4[0]);
      a0[2] = (int)fp8lo_bf16x2(w4[1]); a0[3] = (int)fp8hi_bf16x2(w4[1]);
      a1[0] = (int)fp8lo_bf16x2(w4[2]); a1[1] = (int)fp8hi_bf16x2(w4[2]);
      a1[2] = (int)fp8lo_bf16x2(w4[3]); a1[3] = (int)fp8hi_bf16x2(w4[3]);
      kb[2 * kp] = __builtin_bit_cast(bf16x8, a0);
      kb[2 * kp + 1] = __builtin_bit_cast(bf16x8, a1);
    }
    f32x16 acc0 = f32x16{}, acc1 = f32x16{};
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) {
      acc0 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(qf[0][ks], kb[ks], acc0, 0, 0, 0);
      acc1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(qf[1][ks], kb[ks], acc1, 0, 0, 0);
    }
    // relu as an integer max on the bit pattern (one instruction; fmaxf would also canonicalize its operand):
    // non-negative floats keep their value, negative ones (sign bit set: negative as int) become +0
    // (elements are copied out first: __builtin_bit_cast on an ext_vector element subscript reads element 0)
    float pa = 0.f, pb = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const float s0 = acc0[i], s1 = acc1[i];
      pa = __builtin_fmaf(wl[0][i], __builtin_bit_cast(float, max(__builtin_bit_cast(int, s0), 0)), pa);
      pb = __builtin_fmaf(wl[1][i], __builtin_bit_cast(float, max(__builtin_bit_cast(int, s1), 0)), pb);
    }
    float part = pa + pb;
    part += __shfl_xor(part, 32, 64);
    const int j = 32 * id + l32;
    const float lg = p.clamp ? fminf(part * sc, 60000.f) : part * sc;
    const float v = ok ? lg : -__builtin_inff();
    const bool wr = half == 0 && j < p.Lc && (ok || !p.noinf || j < nh);
    if (stage) {
      if (half == 0) sbuf[32 * (id - tb) + l32] = v;
      const uint64_t m = __ballot(wr);
      if (lane == 0) smask[id - tb] = (uint32_t)m;
    } else if (wr) {
      put(j, v);
    }
  };

  // tiles of steps t .. t + 2D - 1 (slot t % 2D, wave-uniform): the first 2D steps take tiles tb + k NW + w, each
  // later one is claimed from the LDS counter 2D steps ahead (when its block-table entries are loaded), so the waves
  // finish together whatever each one's issue priority and memory service (with equal static shares the youngest
  // waves of a workgroup ended up to 31 us after the oldest at 131072 columns). A wave's tiles only grow, so it is
  // done once a whole round of 2D steps holds no tile below tv.
  // loads in flight: codes of steps t .. t + D - 1 (slot t % D), block-table entries of steps t + D .. t + 2D - 1
  // (slot t % 2D). Every step issues the same loads and claim (tiles at or past tv read the row-0 key and the
  // range's first block-table entry, cache hits, and are not computed), so the compiler's wait before a step's first
  // use of its codes counts the loads of the D - 1 steps after it on every path.
  int ids[2 * D];
#pragma unroll
  for (int k = 0; k < 2 * D; ++k) ids[k] = tb + wv + k * LG_NWV;
  u32x4 cd[D][4];
  float scv[D];
  bool okv[D];
  int btv[2 * D];
#pragma unroll
  for (int k = 0; k < 2 * D; ++k) btv[k] = load_bt(ids[k]);
#pragma unroll
  for (int k = 0; k < D; ++k) okv[k] = load_codes(ids[k], btv[k], cd[k], scv[k]);
  bool live = true;
#pragma unroll 1
  while (live) {
    live = false;
#pragma unroll
    for (int s = 0; s < 2 * D; ++s) {
      int nxt = 0;
      if (lane == 0) nxt = atomicAdd(&claim, 1);            // the tile of step t + 2D (an LDS atomic)
      if (ids[s] < tv) {                                    // uniform
        live = true;
        compute(ids[s], cd[s % D], scv[s % D], okv[s % D]);
      }
      okv[s % D] = load_codes(ids[(s + D) % (2 * D)], btv[(s + D) % (2 * D)], cd[s % D], scv[s % D]);
      ids[s] = __builtin_amdgcn_readfirstlane(nxt);
      btv[s] = load_bt(ids[s]);
    }
  }
  if (stage) __syncthreads();                // every wave has computed its tiles
  if (stage) {                               // 4 columns per thread: one 16-byte (fp16: 8-byte) store when all go out
    const int ncol = 32 * (tv - tb);
    const bool vec = ((uintptr_t)p.out & (F16OUT ? 7u : 15u)) == 0 && (p.out_st & 3) == 0;   // j % 4 == 0 below
    for (int i = 4 * (int)threadIdx.x; i < ncol; i += 4 * LG_NWV * 64) {
      const int j = 32 * tb + i;
      const uint32_t m4 = (smask[i >> 5] >> (i & 31)) & 15u;
      const f32x4 v4 = *(const f32x4*)&sbuf[i];
      if (vec && m4 == 15u && j + 3 < p.Lc) {
        if constexpr (F16OUT) {
          typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
          *(f16x4*)(hrow + j) = f16x4{(_Float16)v4[0], (_Float16)v4[1], (_Float16)v4[2], (_Float16)v4[3]};
        } else {
          *(f32x4*)(orow + j) = v4;
        }
      } else {
#pragma unroll
        for (int k = 0; k < 4; ++k)
          if (((m4 >> k) & 1u) && j + k < p.Lc) put(j + k, v4[k]);
      }
    }
  }
}

// ---- prefill logits over gathered keys (many query rows over the same keys) --------------------------------------
// The kernel above reads and converts every key for every query row (2048 rows of 16384 keys: 786 us, a third of them
// matrix-core time). Here a workgroup keeps 512 keys as bf16 MFMA operands in registers, 64 a wave (2
// waves per SIMD), and runs up to 64 query rows past them: a row's 64 heads (16 KiB) and weights go through a 3-deep
// LDS ring by LDS DMA, every wave reads them as the A operand (chunk c of head h at c ^ (h & 7): no bank conflicts) and
// does 32 MFMAs a row, two head blocks by two key blocks; the ReLU and weighting of one product run under the
// MFMAs of the next. Same products and sums in the same order as above. Rows whose range misses the 512 keys are only
// filled; where the ranges of a workgroup's rows (a few requests' keys among many) leave tiles out, the workgroups of those
// take part of the rows of the others (256 rows that each see an eighth of 16384 keys: 48 -> 16 us, row at a time 21).
// Bound by the matrix cores (32 x 32 cycles a row and wave) and, at 60%, the LDS reads; measured: 2048 rows of 16384
// keys (15360 valid on average) 417 us.
constexpr int FL_NWV = 8, FL_KEYS = 64 * FL_NWV;   // waves, keys of a workgroup
constexpr int FL_RING = 3;
constexpr int FL_ROWB = 64 * 256 + 256;            // a query row in LDS: 64 heads x 128 bf16, then 64 fp32 weights

struct FlatParams {
  const uint16_t* q; long long q_st, q_sh;
  const float* w; long long w_st;
  const uint8_t* k; long long k_st; const float* kscale;
  const int* lo; const int* hi;                    // per row: first valid key, end of the valid keys
  int M, N, rw;                                    // rows, keys, rows per workgroup (at most 64)
  float* out; long long out_st;
};

__global__ void __launch_bounds__(FL_NWV * 64, 2) flat_logits_kernel(FlatParams p) {
  __shared__ __attribute__((aligned(16))) uint8_t ring[FL_RING * FL_ROWB];
  SPMLA_LDS uint8_t* lds = (SPMLA_LDS uint8_t*)ring;
  const int ntile = (p.N + FL_KEYS - 1) / FL_KEYS, nchunk = (p.M + p.rw - 1) / p.rw;
  const int f = remap_xcd(blockIdx.x, ntile * nchunk);      // an XCD's workgroups take the same rows past all keys
  if (f < 0) return;
  const int lane = threadIdx.x & 63, half = lane >> 5, l32 = lane & 31;
  const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int m0 = f / ntile * p.rw, own = f % ntile;
  int n0 = own * FL_KEYS, key = n0 + 64 * wv + lane;        // this lane's output column
  // rows of the chunk: lane r holds row m0 + r's range
  const int mr = m0 + lane;
  const bool rok = lane < p.rw && mr < p.M;
  const int lo_l = rok ? p.lo[mr] : 0, hi_l = rok ? p.hi[mr] : 0;
  auto meets = [&]() -> bool { return rok && max(lo_l, n0) < min(hi_l, min(n0 + FL_KEYS, p.N)); };
  uint64_t fill = __ballot(rok && !meets());
  auto put = [&](int r, float v) {                          // column `key` of row m0 + r (beyond N, r < 0: dropped)
    const uint64_t a = (uint64_t)(uintptr_t)(p.out + (long long)(m0 + max(r, 0)) * p.out_st);
    const uint32_t alo = __builtin_amdgcn_readfirstlane((uint32_t)a), ahi = __builtin_amdgcn_readfirstlane((uint32_t)(a >> 32));
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(uintptr_t)(((uint64_t)ahi << 32) | alo), (short)0, r < 0 ? 0 : 4 * p.N, 0x00020000);
    __builtin_amdgcn_raw_buffer_store_b32(f2u(v), rs, 4 * key, 0, 0);
  };
  for (; fill; fill &= fill - 1) put(__builtin_ctzll(fill), -__builtin_inff());
  // The chunk's ranges lie in tiles t0 .. t1: its ntile workgroups share them, n / tiles on one, part of the rows each
  const int lc = max(lo_l, 0), hc = min(hi_l, p.N);
  const bool some = rok && lc < hc;
  const int t0 = (int)wave_minmax<false>(some ? (uint32_t)lc / FL_KEYS : 0x7fffffffu);
  const int nt = (int)wave_minmax<true>(some ? (uint32_t)(hc - 1) / FL_KEYS + 1u : 0u) - t0;
  if (nt <= 0) return;                                      // uniform over the workgroup, as the returns below
  int r0 = 0, r1 = 64;                                      // this workgroup's part of the rows
  if (nt < ntile) {
    const int nsub = ntile / nt, sub = own / nt, per = (p.rw + nsub - 1) / nsub;
    if (sub >= nsub) return;
    n0 = (t0 + own - sub * nt) * FL_KEYS;
    key = n0 + 64 * wv + lane;
    r0 = sub * per;
    r1 = r0 + per;
  }
  uint64_t todo = __ballot(meets() && lane >= r0 && lane < r1);
  if (!todo) return;

  // copies of query row m0 + r into ring slot s: 64 heads, 2 KiB a wave, then 8 weights a wave (3 instructions)
  auto issue = [&](int r, int s) {
    SPMLA_LDS uint8_t* d = lds + s * FL_ROWB;
    const uint16_t* qr = p.q + (long long)(m0 + r) * p.q_st;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int h = 4 * (2 * wv + i) + (lane >> 4);
      dma16(qr + (long long)h * p.q_sh + 8 * ((lane & 15) ^ (h & 7)), d + (2 * wv + i) * 1024);
    }
    if (lane < 8) dma4(p.w + (long long)(m0 + r) * p.w_st + 8 * wv + lane, d + 64 * 256 + 32 * wv);
  };
  // row sequence: the set bits of todo, then the last one again (its copies are repeated, not used)
  uint64_t ahead = todo;
  int last = 0;
  auto next_row = [&]() -> int {
    if (ahead) { last = __builtin_ctzll(ahead); ahead &= ahead - 1; }
    return last;
  };
#pragma unroll
  for (int s = 0; s < FL_RING; ++s) issue(next_row(), s);

  // this wave's keys: block b = keys n0 + 64 wv + 32 b + l32, dims in the order of the A operand's fragments
  bf16x8 kf[2][8];
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    const int kn = min(n0 + 64 * wv + 32 * b + l32, p.N - 1);
    const uint8_t* src = p.k + (long long)kn * p.k_st + 16 * half;
    u32x4 c[4];
#pragma unroll
    for (int kp = 0; kp < 4; ++kp) {
      const u32x4u v = *(const u32x4u*)(src + 32 * kp);
      c[kp] = u32x4{v[0], v[1], v[2], v[3]};
    }
#pragma unroll
    for (int kp = 0; kp < 4; ++kp) {
      i32x4 a0, a1;
      a0[0] = (int)fp8lo_bf16x2(c[kp][0]); a0[1] = (int)fp8hi_bf16x2(c[kp][0]);
      a0[2] = (int)fp8lo_bf16x2(c[kp][1]); a0[3] = (int)fp8hi_bf16x2(c[kp][1]);
      a1[0] = (int)fp8lo_bf16x2(c[kp][2]); a1[1] = (int)fp8hi_bf16x2(c[kp][2]);
      a1[2] = (int)fp8lo_bf16x2(c[kp][3]); a1[3] = (int)fp8hi_bf16x2(c[kp][3]);
      kf[b][2 * kp] = __builtin_bit_cast(bf16x8, a0);
      kf[b][2 * kp + 1] = __builtin_bit_cast(bf16x8, a1);
    }
  }
  const float sc = p.kscale[min(key, p.N - 1)];

  // A fragment ks = 2 kp + e of head block m: chunk 4 kp + 2 half + e of head 32 m + l32
  auto load_a = [&](int s, int m, bf16x8 (&a)[8]) {
    SPMLA_LDS uint8_t* d = lds + s * FL_ROWB + (32 * m + l32) * 256;
#pragma unroll
    for (int ks = 0; ks < 8; ++ks)
      a[ks] = __builtin_bit_cast(bf16x8, *(SPMLA_LDS u32x4*)(d + 16 * ((4 * (ks >> 1) + 2 * half + (ks & 1)) ^ (l32 & 7))));
  };
  auto load_w = [&](int s, int m, f32x4 (&x)[4]) {          // weights of the C layout's rows 8 q + 4 half ..
#pragma unroll
    for (int q = 0; q < 4; ++q) x[q] = *(SPMLA_LDS f32x4*)(lds + s * FL_ROWB + 64 * 256 + (32 * m + 8 * q + 4 * half) * 4);
  };
  auto product = [&](const bf16x8 (&a)[8], const bf16x8 (&k)[8]) -> f32x16 {
    f32x16 acc = f32x16{};
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[ks], k[ks], acc, 0, 0, 0);
    return acc;
  };
  auto weigh = [&](const f32x16& acc, const f32x4 (&x)[4]) -> float {   // sum of w * relu (an integer max: see above)
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const float v = acc[i];
      s = __builtin_fmaf(x[i >> 2][i & 3], __builtin_bit_cast(float, max(__builtin_bit_cast(int, v), 0)), s);
    }
    return s;
  };
  // one MFMA, then a slice of the previous product's 32 VALU instructions, eight times
  auto interleave = [&]() {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);
    }
  };

  wait_vm<0>();
  lds_barrier();
  bf16x8 a0[8], a1[8];
  f32x4 w0[4], w1[4];
  load_a(0, 0, a0);
  load_w(0, 0, w0);
  f32x16 x = f32x16{}, y = f32x16{};
  float pa0 = 0.f, pa1 = 0.f, pb0 = 0.f;
  int prow = -1, slot = 0;
  auto finish = [&](float pb1) {                            // row prow's logits of the lane's key
    const float s0 = pa0 + pb0, s1 = pa1 + pb1;
    const auto t = __builtin_amdgcn_permlane32_swap(f2u(s0), f2u(s1), false, false);
    const float v = (u2f(t[0]) + u2f(t[1])) * sc;           // lanes 0 .. 31: block 0's keys, the others block 1's
    const int lo = __builtin_amdgcn_readlane(lo_l, max(prow, 0)), hi = __builtin_amdgcn_readlane(hi_l, max(prow, 0));
    put(prow, key >= lo && key < hi ? v : -__builtin_inff());
  };
#pragma unroll 1
  for (; todo; todo &= todo - 1) {
    const int r = __builtin_ctzll(todo);
    const int ns = slot == FL_RING - 1 ? 0 : slot + 1;
    load_a(slot, 1, a1);
    x = product(a0, kf[0]);
    float pb1 = weigh(y, w1);                               // the previous row's last product
    interleave();
    asm volatile("" : "+v"(pb1));                           // (keeps the slices here)
    __builtin_amdgcn_sched_barrier(0);
    finish(pb1);                                            // (the first time round: dropped)
    load_w(slot, 1, w1);
    __builtin_amdgcn_sched_barrier(0);
    y = product(a0, kf[1]);
    pa0 = weigh(x, w0);
    interleave();
    asm volatile("" : "+v"(pa0));
    __builtin_amdgcn_sched_barrier(0);
    x = product(a1, kf[0]);
    pa1 = weigh(y, w0);
    interleave();
    asm volatile("" : "+v"(pa1));
    __builtin_amdgcn_sched_barrier(0);
    // the next row's copies have landed (issued two rows ago: after them one row's copies and two stores) and this row
    // is read by every wave: its slot takes the row after the next two
    wait_vm<5>();
    lds_barrier();
    issue(next_row(), slot);
    load_a(ns, 0, a0);
    load_w(ns, 0, w0);
    __builtin_amdgcn_sched_barrier(0);
    y = product(a1, kf[1]);
    pb0 = weigh(x, w1);
    interleave();
    asm volatile("" : "+v"(pb0));
    __builtin_amdgcn_sched_barrier(0);
    prow = r;
    slot = ns;
  }
  finish(weigh(y, w1));
  wait_vm<0>();                                             // no copy in flight when the LDS is given back
}

// ------------------------------------------------------------------------------------------------ top-k
constexpr int TK_NT = 1024;
constexpr int TK_KMAX = 2048;
constexpr int TK_CAP = 8192;              // candidate list capacity (workspace and LDS)
constexpr int TK_CAP1 = 4096;             // the one-workgroup path's candidate threshold

// key of logit j of a row (fp32 or fp16 elements)
template <bool F16>
__device__ inline uint32_t lkey(const void* x, long long j) {
  if constexpr (F16) return okey16(((const uint16_t*)x)[j]);
  else return okey(((const float*)x)[j]);
}
// keys of +inf and -inf
template <bool F16>
__device__ inline bool inf_key(uint32_t k) {
  if constexpr (F16) return k == 0xfc000000u || k == 0x03ff0000u;
  else return k == 0xff800000u || k == 0x007fffffu;
}
// row `row` of a logits matrix with element stride st
template <bool F16>
__device__ inline const void* lrow(const void* lg, int row, long long st) {
  return (const uint8_t*)lg + (long long)row * st * (F16 ? 2 : 4);
}

// Inclusive prefix sum over the 64 lanes of a wave on the VALU: DPP row shifts 1, 2, 4, 8 scan each 16-lane row,
// then row_bcast:15 adds row 0's total to row 1 and row 2's to row 3, and row_bcast:31 adds rows 0-1's total to rows
// 2 and 3 (gfx9 DPP controls). A lane whose DPP source is outside its row adds 0.
__device__ inline uint32_t wave_incl_scan(uint32_t x) {
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x111, 0xf, 0xf, false);   // row_shr:1
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x112, 0xf, 0xf, false);   // row_shr:2
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x114, 0xf, 0xf, false);   // row_shr:4
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x118, 0xf, 0xf, false);   // row_shr:8
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x142, 0xa, 0xf, false);   // row_bcast:15, rows 1, 3
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x143, 0xc, 0xf, false);   // row_bcast:31, rows 2, 3
  return x;
}
// block-wide exclusive scan of a per-thread count (1024 threads = 16 waves): wave scans on the VALU, the 16 wave
// totals through LDS (wsum: 16-byte aligned, 16 words); every thread sums the totals of the waves before its own
__device__ inline uint32_t block_excl_scan(uint32_t v, uint32_t* wsum, uint32_t* total) {
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const uint32_t inc = wave_incl_scan(v);
  if (lane == 63) wsum[wv] = inc;
  __syncthreads();
  uint32_t before = 0u, tot = 0u;
#pragma unroll
  for (int q = 0; q < TK_NT / 256; ++q) {
    const u32x4 s4 = ((const u32x4*)wsum)[q];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      before += 4 * q + e < wv ? s4[e] : 0u;
      tot += s4[e];
    }
  }
  *total = tot;
  __syncthreads();                                   // wsum is free for the next scan
  return before + inc - v;
}

// bitonic sort of n (power of two) uint64 in LDS, descending. Thread t handles pairs t, t + 1024, ...; for a
// stride <= 64 both elements of its pairs lie in the 128-element block of its wave, so such a stage needs no
// workgroup barrier (LDS operations of one wave complete in issue order), only a compiler fence.
__device__ inline void bitonic_desc(unsigned long long* a, int n) {
  for (int size = 2; size <= n; size <<= 1) {
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
      for (int t = threadIdx.x; t < n / 2; t += TK_NT) {
        const int lo = 2 * t - (t & (stride - 1));
        const int hi = lo + stride;
        const bool desc = (lo & size) == 0;
        const unsigned long long x = a[lo], y = a[hi];
        if ((x < y) == desc) { a[lo] = y; a[hi] = x; }
      }
      const int next = stride > 1 ? stride >> 1 : size;   // stride of the next stage (size << 1 >> 1)
      if (stride >= 128 || next >= 128) __syncthreads();
      else __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    }
  }
  __syncthreads();
}

// Lane-xor exchange of a 64-bit value. Masks 1 and 2 are DPP quad permutations and 32 is v_permlane32_swap, all on
// the SIMD's own VALU; 4, 8 and 16 go through the LDS crossbar (ds_swizzle, bit mode). The sort's stages are bound by
// the LDS pipe that the CU's 16 waves share, so every exchange moved to the VALU shortens them.
template <int M>
__device__ inline unsigned long long xchg64(unsigned long long v, int perm32) {
  (void)perm32;
  const int vlo = (int)(uint32_t)v, vhi = (int)(uint32_t)(v >> 32);
  int lo, hi;
  if constexpr (M == 1 || M == 2) {
    constexpr int ctl = M == 1 ? 0xB1 : 0x4E;          // quad_perm [1, 0, 3, 2] / [2, 3, 0, 1]
    lo = __builtin_amdgcn_mov_dpp(vlo, ctl, 0xF, 0xF, false);
    hi = __builtin_amdgcn_mov_dpp(vhi, ctl, 0xF, 0xF, false);
  } else if constexpr (M == 32) {
    const auto a = __builtin_amdgcn_permlane32_swap((uint32_t)vlo, (uint32_t)vlo, false, false);
    const auto b = __builtin_amdgcn_permlane32_swap((uint32_t)vhi, (uint32_t)vhi, false, false);
    const bool up = (__lane_id() & 32) != 0;
    lo = (int)(up ? a[0] : a[1]);
    hi = (int)(up ? b[0] : b[1]);
  } else {
    lo = __builtin_amdgcn_ds_swizzle(vlo, (M << 10) | 0x1f);
    hi = __builtin_amdgcn_ds_swizzle(vhi, (M << 10) | 0x1f);
  }
  return ((unsigned long long)(uint32_t)hi << 32) | (uint32_t)lo;
}

// One compare-exchange stage of the bitonic network held in VGPRs (block size SIZE, lane-xor stride S < 64);
// thread t of wave w holds entries e0 = 128w + l and e0 + 64 (l = lane).
template <int SIZE, int S>
__device__ inline void bstage(unsigned long long& x0, unsigned long long& x1, int e0, int l, int perm32) {
  const bool d0 = (e0 & SIZE) == 0, d1 = ((e0 + 64) & SIZE) == 0;
  const unsigned long long y0 = xchg64<S>(x0, perm32), y1 = xchg64<S>(x1, perm32);
  const bool lower = (l & S) == 0;
  // the lower element of a pair keeps the max when descending, the upper one the min (and the reverse)
  x0 = ((lower == d0) == (x0 > y0)) ? x0 : y0;
  x1 = ((lower == d1) == (x1 > y1)) ? x1 : y1;
}

// The stages of a SIZE block with strides <= 64 (stride 64: the thread's own two entries, same block).
template <int SIZE>
__device__ inline void bmerge(unsigned long long& x0, unsigned long long& x1, int e0, int l, int perm32) {
  if constexpr (SIZE >= 128) {
    if ((x0 < x1) == ((e0 & SIZE) == 0)) { const unsigned long long t = x0; x0 = x1; x1 = t; }
  }
  if constexpr (SIZE >= 64) bstage<SIZE, 32>(x0, x1, e0, l, perm32);
  if constexpr (SIZE >= 32) bstage<SIZE, 16>(x0, x1, e0, l, perm32);
  if constexpr (SIZE >= 16) bstage<SIZE, 8>(x0, x1, e0, l, perm32);
  if constexpr (SIZE >= 8) bstage<SIZE, 4>(x0, x1, e0, l, perm32);
  if constexpr (SIZE >= 4) bstage<SIZE, 2>(x0, x1, e0, l, perm32);
  bstage<SIZE, 1>(x0, x1, e0, l, perm32);
}

// The stages of a SIZE block with strides >= 128, through LDS (one pair per thread, a barrier per stage).
template <int SIZE>
__device__ inline void bmerge_lds(unsigned long long* a, unsigned long long& x0, unsigned long long& x1, int e0) {
  const int t = threadIdx.x;
  a[e0] = x0;
  a[e0 + 64] = x1;
  __syncthreads();
#pragma unroll
  for (int stride = SIZE >> 1; stride >= 128; stride >>= 1) {
    const int lo = 2 * t - (t & (stride - 1)), hi = lo + stride;
    const bool desc = (lo & SIZE) == 0;
    const unsigned long long x = a[lo], y = a[hi];
    if ((x < y) == desc) { a[lo] = y; a[hi] = x; }
    __syncthreads();
  }
  x0 = a[e0];
  x1 = a[e0 + 64];
}

// Bitonic sort of a[0, 2048) descending with the data in VGPRs: 56 of the 66 stages are in-thread or lane-xor
// exchanges (ds_swizzle), the 10 with strides >= 128 go through LDS.
__device__ inline void sort2048_desc(unsigned long long* a) {
  const int t = threadIdx.x, l = t & 63;
  const int e0 = 128 * (t >> 6) + l;
  const int perm32 = (l ^ 32) << 2;
  unsigned long long x0 = a[e0], x1 = a[e0 + 64];
  bmerge<2>(x0, x1, e0, l, perm32);
  bmerge<4>(x0, x1, e0, l, perm32);
  bmerge<8>(x0, x1, e0, l, perm32);
  bmerge<16>(x0, x1, e0, l, perm32);
  bmerge<32>(x0, x1, e0, l, perm32);
  bmerge<64>(x0, x1, e0, l, perm32);
  bmerge<128>(x0, x1, e0, l, perm32);
  bmerge_lds<256>(a, x0, x1, e0);
  bmerge<256>(x0, x1, e0, l, perm32);
  bmerge_lds<512>(a, x0, x1, e0);
  bmerge<512>(x0, x1, e0, l, perm32);
  bmerge_lds<1024>(a, x0, x1, e0);
  bmerge<1024>(x0, x1, e0, l, perm32);
  bmerge_lds<2048>(a, x0, x1, e0);
  bmerge<2048>(x0, x1, e0, l, perm32);
  __syncthreads();                                   // every thread has read a: write the sorted data back
  a[e0] = x0;
  a[e0 + 64] = x1;
  __syncthreads();
}

// Sorts a[0, n) descending (entries nonzero); pads with zeros to the sorting network's size.
__device__ inline void tk_sort_desc(unsigned long long* a, int n) {
  int np2 = 1;
  while (np2 < n) np2 <<= 1;
  if (np2 > 256 && np2 <= 2048) np2 = 2048;
  for (int i = n + (int)threadIdx.x; i < np2; i += TK_NT) a[i] = 0ull;
  __syncthreads();
  if (np2 == 2048) sort2048_desc(a);
  else if (np2 > 1) bitonic_desc(a, np2);
}

template <bool F16>
struct RowSrc {     // a logits row (fp32 or fp16): candidate j = column j
  const void* x; int n;
  __device__ uint32_t key(int j) const { return lkey<F16>(x, j); }
  __device__ float val(int j) const {
    if constexpr (F16) return (float)((const _Float16*)x)[j];
    else return ((const float*)x)[j];
  }
  __device__ int id(int j) const { return j; }
  __device__ static bool inf(uint32_t k) { return inf_key<F16>(k); }
};
struct MergeSrc {   // all-gathered payloads [P][nrows][2 * kl] = [values | positions]: candidate c = (c / kl, c % kl)
  const float* allp; long long nrows; int row, kl, n;
  __device__ const float* seg(int c, int& i) const {
    const int r = c / kl;
    i = c - r * kl;
    return allp + ((long long)r * nrows + row) * 2 * kl;
  }
  __device__ float val(int c) const { int i; const float* b = seg(c, i); return b[i]; }
  __device__ uint32_t key(int c) const { return okey(val(c)); }
  __device__ int id(int c) const { int i; const float* b = seg(c, i); return (int)f2u(b[kl + i]); }
  __device__ static bool inf(uint32_t k) { return inf_key<false>(k); }
};

// Four copies of the 2048-bin histogram (lane & 3 picks one) split same-bin atomics of a wave four ways; a copy
// stride of 2049 words keeps the copies of a bin in different banks.
constexpr int TK_HCOPY = 4;
constexpr int TK_HSTR = 2049;

struct TopkLds {
  uint32_t hist[TK_HCOPY * TK_HSTR];
  unsigned long long sel[TK_KMAX];
  unsigned long long cand[TK_CAP];
  __attribute__((aligned(16))) uint32_t wsum[17];
  uint32_t sh[8];
};

__device__ inline unsigned long long tk_pack(uint32_t key, int j) {
  return ((unsigned long long)key << 32) | (uint32_t)(~(uint32_t)j);
}

__device__ inline void tk_hist_add(TopkLds& L, uint32_t bin) {
  atomicAdd(&L.hist[(threadIdx.x & (TK_HCOPY - 1)) * TK_HSTR + bin], 1u);
}

// Radix level bookkeeping: digit d = (key >> shift) & dm of the keys under (prefix, mask).
__device__ inline int tk_shift(int level) { return level == 0 ? 21 : (level == 1 ? 10 : 0); }
__device__ inline uint32_t tk_dmask(int level) { return level == 2 ? 0x3ffu : 0x7ffu; }

// From the level's histogram: the boundary bin b holding the need-th largest key, the count above it and in it.
__device__ inline void tk_bin(TopkLds& L, uint32_t need, uint32_t& b, uint32_t& above, uint32_t& binc) {
  const int tid = threadIdx.x;
  const int b0 = 2047 - 2 * tid, b1 = b0 - 1;   // thread t owns bins 2047 - 2t, 2046 - 2t (descending)
  uint32_t h0 = 0, h1 = 0;
#pragma unroll
  for (int c = 0; c < TK_HCOPY; ++c) { h0 += L.hist[c * TK_HSTR + b0]; h1 += L.hist[c * TK_HSTR + b1]; }
  uint32_t tot;
  const uint32_t before = block_excl_scan(h0 + h1, L.wsum, &tot);
  if (before < need && before + h0 >= need) { L.sh[1] = (uint32_t)b0; L.sh[2] = before; L.sh[3] = h0; }
  if (before + h0 < need && before + h0 + h1 >= need) { L.sh[1] = (uint32_t)b1; L.sh[2] = before + h0; L.sh[3] = h1; }
  __syncthreads();
  b = L.sh[1]; above = L.sh[2]; binc = L.sh[3];
}

__device__ inline void tk_clear_hist(TopkLds& L) {
  for (int i = threadIdx.x; i < TK_HCOPY * TK_HSTR; i += TK_NT) L.hist[i] = 0;
  __syncthreads();
}

// Block-wide placement of per-thread selections: each thread passes how many entries it appends to sel and to cand;
// returns its first slot in each (after the bases *sb, *cb, which advance by the block totals on every thread).
__device__ inline void tk_slots(uint32_t ns, uint32_t nc, TopkLds& L, uint32_t& sb, uint32_t& cb, uint32_t& so,
                                uint32_t& co) {
  uint32_t tot;
  const uint32_t off = block_excl_scan(ns | (nc << 16), L.wsum, &tot);   // both totals < 65536
  so = sb + (off & 0xffffu);
  co = cb + (off >> 16);
  sb += tot & 0xffffu;
  cb += tot >> 16;
}

constexpr int TK_KPT = 32;                 // keys per thread per chunk (held in VGPRs)
constexpr int TK_CH = TK_KPT * TK_NT;      // 32768 columns per chunk
constexpr int TK_EPT = TK_CAP / TK_NT;     // boundary-bin candidates per thread at the full capacity

template <class Src>
__device__ inline void tk_load(const Src& src, int base, uint32_t (&k)[TK_KPT]) {
#pragma unroll
  for (int i = 0; i < TK_KPT; ++i) {
    const int j = base + i * TK_NT + (int)threadIdx.x;
    k[i] = j < src.n ? src.key(j) : 0u;
  }
}

// Finishes a selection from the boundary-bin candidates L.cand[0, nc) (all under (prefix, mask) of level lvl - 1):
// radix levels lvl..2 on the candidates held in registers; equal final keys go to the lowest columns. sb = entries
// already in L.sel.
template <int EPT = TK_EPT>                       // candidates per thread: nc <= EPT * TK_NT
__device__ __forceinline__ void tk_resolve_cands(TopkLds& L, int nc, int lvl, uint32_t prefix, uint32_t mask,
                                                 uint32_t need, uint32_t sb, int ncols) {
  const int tid = threadIdx.x;
  unsigned long long e[EPT];
  uint32_t vm = 0;                                   // bit i: e[i] is a candidate
  int t = tid;                                       // opaque copy: keeps the slot indices from being hoisted
  asm volatile("" : "+v"(t));
#pragma unroll
  for (int i = 0; i < EPT; ++i) {              // consecutive candidates: the winners appended below keep their
    const int c = EPT * t + i;                  // order in L.cand (column order for the workspace path)
    vm |= (uint32_t)(c < nc) << i;
    e[i] = c < nc ? L.cand[c] : 0ull;
  }
  for (int level = lvl; level < 3; ++level) {
    const int shift = tk_shift(level);
    const uint32_t dm = tk_dmask(level);
    tk_clear_hist(L);
#pragma unroll
    for (int i = 0; i < EPT; ++i) {
      const uint32_t k = (uint32_t)(e[i] >> 32);
      if (((vm >> i) & 1u) && (k & mask) == prefix) tk_hist_add(L, (k >> shift) & dm);
    }
    __syncthreads();
    uint32_t b, above, binc;
    tk_bin(L, need, b, above, binc);
    const bool whole = above + binc == need;
    uint32_t selm = 0;
#pragma unroll
    for (int i = 0; i < EPT; ++i) {
      const uint32_t k = (uint32_t)(e[i] >> 32);
      const uint32_t d = (k >> shift) & dm;
      const bool in = ((vm >> i) & 1u) && (k & mask) == prefix;
      selm |= (uint32_t)(in && (d > b || (whole && d == b))) << i;
    }
    uint32_t cb = 0, so, co;
    tk_slots(__popc(selm), 0u, L, sb, cb, so, co);
#pragma unroll
    for (int i = 0; i < EPT; ++i)
      if ((selm >> i) & 1u) L.sel[so++] = e[i];
    if (whole) { __syncthreads(); return; }
    prefix |= b << shift;
    mask |= dm << shift;
    need -= above;
    if (level == 2) {
      // binc candidates carry the final key; the need lowest columns win
      uint32_t eqm = 0;
#pragma unroll
      for (int i = 0; i < EPT; ++i)
        eqm |= (uint32_t)(((vm >> i) & 1u) && (uint32_t)(e[i] >> 32) == prefix) << i;
      constexpr int BM_WPT = 8;                    // bitmap words per thread: TK_NT * 8 words in the histogram space
      static_assert(TK_NT * BM_WPT <= TK_HCOPY * TK_HSTR, "bitmap fits the histogram space");
      if (ncols <= 32 * TK_NT * BM_WPT) {
        // a bitmap of the tied columns in the histogram space (free after the last level), then each column's rank
        // among them from prefix sums of per-word bit counts: the need lowest are taken, no sort (the final output
        // sort orders every winner anyway)
        const int words = (ncols + 31) >> 5;
        __syncthreads();
        for (int w = tid; w < words; w += TK_NT) L.hist[w] = 0u;
        __syncthreads();
#pragma unroll
        for (int i = 0; i < EPT; ++i)
          if ((eqm >> i) & 1u) {
            const uint32_t j = ~(uint32_t)e[i];
            atomicOr(&L.hist[j >> 5], 1u << (j & 31u));
          }
        __syncthreads();
        const int w0 = tid * BM_WPT;
        uint32_t cnt = 0;
#pragma unroll
        for (int k = 0; k < BM_WPT; ++k)
          if (w0 + k < words) cnt += (uint32_t)__popc(L.hist[w0 + k]);
        uint32_t tot;
        uint32_t r = block_excl_scan(cnt, L.wsum, &tot);   // ranks of this thread's first tied column
#pragma unroll
        for (int k = 0; k < BM_WPT; ++k) {
          uint32_t bits = w0 + k < words ? L.hist[w0 + k] : 0u;
          while (bits && r < need) {
            const uint32_t j = 32u * (uint32_t)(w0 + k) + (uint32_t)(__ffs(bits) - 1);
            bits &= bits - 1u;
            L.sel[sb + r] = (((unsigned long long)prefix) << 32) | (uint32_t)~j;
            ++r;
          }
        }
        __syncthreads();
        return;
      }
      // wider rows: sort the tied candidates by column ascending
      __syncthreads();                             // every thread has read its candidates: L.cand is free
      uint32_t cb2 = 0, sb2 = 0;
      tk_slots(0u, __popc(eqm), L, sb2, cb2, so, co);
#pragma unroll
      for (int i = 0; i < EPT; ++i)
        if ((eqm >> i) & 1u) L.cand[co++] = (unsigned long long)(uint32_t)e[i] << 32;   // ~j high: desc = j asc
      __syncthreads();
      tk_sort_desc(L.cand, (int)binc);
      for (uint32_t i = tid; i < need; i += TK_NT) L.sel[sb + i] = (((unsigned long long)prefix) << 32) | (L.cand[i] >> 32);
      __syncthreads();
      return;
    }
  }
}

// Selects the K largest candidates (key desc, j asc) of src into L.sel (unordered); returns their number min(n, K).
// The row's keys sit in VGPRs (32 per thread; longer rows are re-read per 32768-column chunk with all loads of a
// chunk in flight). Each radix level builds an LDS histogram; the keys above the boundary bin are written to slots
// from one block scan of per-thread counts; a boundary bin of at most TK_CAP1 keys is finished on the candidates alone.
template <class Src>
__device__ __forceinline__ int tk_select(const Src& src, int K, TopkLds& L) {
  const int tid = threadIdx.x, n = src.n;
  if (n <= K) {
    for (int j = tid; j < n; j += TK_NT) L.sel[j] = tk_pack(src.key(j), j);
    __syncthreads();
    return n;
  }
  const int nch = (n + TK_CH - 1) / TK_CH;
  uint32_t key[TK_KPT];
  if (nch == 1) tk_load(src, 0, key);
  uint32_t prefix = 0, mask = 0, need = (uint32_t)K, sb = 0;
  for (int level = 0; level < 3; ++level) {
    const int shift = tk_shift(level);
    const uint32_t dm = tk_dmask(level);
    // the column of key[i] is recomputed per level from an opaque copy of tid: hoisting the 32 columns (and the
    // packed entries built from them) out of the level loop would spill them
    int t = tid;
    asm volatile("" : "+v"(t));
    tk_clear_hist(L);
    for (int c = 0; c < nch; ++c) {
      if (nch > 1) tk_load(src, c * TK_CH, key);
#pragma unroll
      for (int i = 0; i < TK_KPT; ++i) {
        const int j = c * TK_CH + i * TK_NT + t;
        if (j < n && (key[i] & mask) == prefix) tk_hist_add(L, (key[i] >> shift) & dm);
      }
    }
    __syncthreads();
    uint32_t b, above, binc;
    tk_bin(L, need, b, above, binc);
    const bool whole = above + binc == need;
    const bool fits = !whole && level < 2 && binc <= (uint32_t)TK_CAP1;
    uint32_t cb = 0;
    for (int c = 0; c < nch; ++c) {
      if (nch > 1) tk_load(src, c * TK_CH, key);
      uint32_t selm = 0, candm = 0;
#pragma unroll
      for (int i = 0; i < TK_KPT; ++i) {
        const int j = c * TK_CH + i * TK_NT + t;
        const uint32_t d = (key[i] >> shift) & dm;
        const bool in = j < n && (key[i] & mask) == prefix;
        selm |= (uint32_t)(in && (d > b || (whole && d == b))) << i;
        candm |= (uint32_t)(fits && in && d == b) << i;
      }
      uint32_t so, co;
      tk_slots(__popc(selm), __popc(candm), L, sb, cb, so, co);
#pragma unroll
      for (int i = 0; i < TK_KPT; ++i) {
        const int j = c * TK_CH + i * TK_NT + t;
        if ((selm >> i) & 1u) L.sel[so++] = tk_pack(key[i], j);
        if ((candm >> i) & 1u) L.cand[co++] = tk_pack(key[i], j);
      }
    }
    __syncthreads();
    if (whole) return K;
    if (fits) {
      tk_resolve_cands<TK_CAP1 / TK_NT>(L, (int)binc, level + 1, prefix | (b << shift), mask | (dm << shift), need - above, sb, n);
      return K;
    }
    prefix |= b << shift;
    mask |= dm << shift;
    need -= above;
  }
  // the boundary key is fully known (prefix); the need lowest columns holding it win, in column order
  uint32_t got = 0;
  for (int c = 0; c < nch && got < need; ++c) {
    if (nch > 1) tk_load(src, c * TK_CH, key);
#pragma unroll
    for (int i = 0; i < TK_KPT; ++i) {
      if (got < need) {                          // uniform: got is a block-wide total
        const int j = c * TK_CH + i * TK_NT + tid;
        const bool eq = j < n && key[i] == prefix;
        uint32_t tot;
        const uint32_t r = block_excl_scan(eq ? 1u : 0u, L.wsum, &tot);
        if (eq && got + r < need) L.sel[sb + got + r] = tk_pack(prefix, j);
        got += tot;
      }
    }
  }
  __syncthreads();
  return K;
}

// Sorts the nsel selected entries by (key desc, j asc) and writes src.id of the first kout slots to o
// (-1 where the value is +-inf and for slots >= nsel).
template <class Src>
__device__ __forceinline__ void tk_emit_sorted(const Src& src, int nsel, int kout, int* o, TopkLds& L) {
  const int tid = threadIdx.x;
  tk_sort_desc(L.sel, nsel);
  for (int s = tid; s < kout; s += TK_NT) {
    int r = -1;
    if (s < nsel) {
      const unsigned long long e = L.sel[s];
      const uint32_t key = (uint32_t)(e >> 32);
      const int j = (int)(~(uint32_t)e);
      if (!Src::inf(key)) r = src.id(j);                  // +-inf: no position
    }
    o[s] = r;
  }
}

// Stable LSD radix sort of L.sel[0, n) (n <= 2048) by key (the high word) descending, then the emit of
// tk_emit_sorted. Entries with equal keys keep their order in L.sel, so lists appended in column order come out
// (key desc, column asc) with no sort on the columns. Keys are offset by the smallest key, and only the bytes that
// the offsets span are sorted (fp16 keys: their low half is zero). One pass: wave-local stable ranks from 16 ballots
// (entries 2t, 2t + 1 of thread t, waves in order), per-wave digit counts, one scan over (digit, wave), a scatter.
// LDS: L.cand as the scatter buffer, L.hist for the counts and offsets.
template <class Src, bool F16>
__device__ __forceinline__ void tk_emit_radix(const Src& src, int n, int kout, int* o, TopkLds& L) {
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  unsigned long long* tmp = L.cand;
  uint32_t* whist = L.hist;                      // [digit][wave] counts of the pass
  uint32_t* woff = L.hist + 4096;                // [digit][wave] first slot of the wave's entries of the digit
  uint32_t* red = (uint32_t*)(L.cand + TK_KMAX); // 16 waves x (min, max)
  static_assert(2 * 4096 <= TK_HCOPY * TK_HSTR && TK_CAP >= TK_KMAX + 16, "radix sort LDS");
  for (int i = tid; i < 4096; i += TK_NT) whist[i] = 0u;
  const bool v0 = 2 * tid < n, v1 = 2 * tid + 1 < n;   // entries past n: zero, sorted last
  unsigned long long x0 = v0 ? L.sel[2 * tid] : 0ull, x1 = v1 ? L.sel[2 * tid + 1] : 0ull;
  uint32_t kmn = 0xffffffffu, kmx = 0u;
  if (v0) { kmn = (uint32_t)(x0 >> 32); kmx = kmn; }
  if (v1) { kmn = min(kmn, (uint32_t)(x1 >> 32)); kmx = max(kmx, (uint32_t)(x1 >> 32)); }
  kmn = wave_minmax<false>(kmn);
  kmx = wave_minmax<true>(kmx);
  if (lane == 0) { red[2 * wv] = kmn; red[2 * wv + 1] = kmx; }
  __syncthreads();
#pragma unroll
  for (int v = 0; v < TK_NT / 64; ++v) { kmn = min(kmn, red[2 * v]); kmx = max(kmx, red[2 * v + 1]); }
  const uint32_t range = kmx > kmn ? kmx - kmn : 0u;
  const int first = F16 ? 2 : 0;                 // lowest byte that can differ
  const int last = range ? (31 - __builtin_clz(range)) >> 3 : -1;
  const unsigned long long below = (1ull << lane) - 1ull;
  for (int byte = first; byte <= last; ++byte) {   // uniform
    const int sh = 8 * byte;
    // padding entries (key 0: every real key is at least -inf's 0x007fffff) take digit 255 in every pass
    const uint32_t k0 = (uint32_t)(x0 >> 32), k1 = (uint32_t)(x1 >> 32);
    const uint32_t d0 = k0 ? 255u - ((k0 - kmn) >> sh & 255u) : 255u;
    const uint32_t d1 = k1 ? 255u - ((k1 - kmn) >> sh & 255u) : 255u;
    // lanes whose entry 0 / entry 1 has this lane's digit d0 (ma / mb) or d1 (mc / md)
    unsigned long long ma = ~0ull, mb = ~0ull, mc = ~0ull, md = ~0ull;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const unsigned long long b0 = __ballot((d0 >> k) & 1u), b1 = __ballot((d1 >> k) & 1u);
      const unsigned long long s0 = (unsigned long long)(long long)-(int)((d0 >> k) & 1u);
      const unsigned long long s1 = (unsigned long long)(long long)-(int)((d1 >> k) & 1u);
      ma &= ~(b0 ^ s0); mb &= ~(b1 ^ s0); mc &= ~(b0 ^ s1); md &= ~(b1 ^ s1);
    }
    // stable rank among the wave's entries of the same digit (order: lane, then entry)
    const uint32_t r0 = (uint32_t)(__popcll(ma & below) + __popcll(mb & below));
    const uint32_t r1 = (uint32_t)(__popcll(mc & below) + __popcll(md & below)) + (d0 == d1 ? 1u : 0u);
    if (r0 == 0u) whist[d0 * 16 + wv] = (uint32_t)(__popcll(ma) + __popcll(mb));
    if (r1 == 0u) whist[d1 * 16 + wv] = (uint32_t)(__popcll(mc) + __popcll(md));
    __syncthreads();
    uint32_t c[16], tot = 0u, incl = 0u;
    if (tid < 256) {                              // digit tid: offsets over the waves, then over the digits
      u32x4* hp = (u32x4*)(whist + tid * 16);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const u32x4 v = hp[q];
        hp[q] = u32x4{0u, 0u, 0u, 0u};           // cleared for the next pass
#pragma unroll
        for (int e = 0; e < 4; ++e) { c[4 * q + e] = tot; tot += v[e]; }
      }
      incl = wave_incl_scan(tot);
      if (lane == 63) L.wsum[wv] = incl;
    }
    __syncthreads();
    if (tid < 256) {
      uint32_t bse = incl - tot;
      for (int v = 0; v < wv; ++v) bse += L.wsum[v];
      u32x4* op = (u32x4*)(woff + tid * 16);
#pragma unroll
      for (int q = 0; q < 4; ++q) op[q] = u32x4{bse + c[4 * q], bse + c[4 * q + 1], bse + c[4 * q + 2], bse + c[4 * q + 3]};
    }
    __syncthreads();
    tmp[woff[d0 * 16 + wv] + r0] = x0;
    tmp[woff[d1 * 16 + wv] + r1] = x1;
    __syncthreads();
    x0 = tmp[2 * tid];
    x1 = tmp[2 * tid + 1];
  }
  // entries 2t, 2t + 1 of the sorted order are in this thread's registers
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const int slot = 2 * tid + e;
    if (slot < kout) {
      int r = -1;
      const unsigned long long x = e ? x1 : x0;
      if (slot < n) {
        const uint32_t key = (uint32_t)(x >> 32);
        const int j = (int)(~(uint32_t)x);
        if (!Src::inf(key)) r = src.id(j);
      }
      o[slot] = r;
    }
  }
}

struct TopkParams {
  const void* lg; long long lg_st;                // fp32 or fp16 (the kernel's F16), stride in elements
  const int* ctx; int rows, Lc, K;
  int* out; long long out_st;
};

template <bool F16>
__global__ void __launch_bounds__(TK_NT) topk_kernel(TopkParams p) {
  __shared__ TopkLds L;
  const int row = blockIdx.x;
  int n = p.ctx[row];
  n = n < 0 ? 0 : (n > p.Lc ? p.Lc : n);
  const RowSrc<F16> src{lrow<F16>(p.lg, row, p.lg_st), n};
  const int nsel = tk_select(src, p.K, L);
  tk_emit_sorted(src, nsel, p.K, p.out + (long long)row * p.out_st, L);
}

// ---- bucket selection: rows of at most 32768 columns, and chunks of longer rows ------------------------------
// One 1024-thread workgroup holds up to 32768 keys in VGPRs and selects and sorts in one go: the values' range is cut
// into 4096 equal bins (a float subtract and multiply round monotonically, so a larger value never gets a lower bin);
// an LDS histogram and one scan give every bin's first slot in descending order and the bin of the K-th key; the keys
// of that bin and above go to their bin's slots (an LDS atomic each), and an entry's final slot is its bin's first plus
// the number of larger entries (key, then lower column) in its bin. Bins of equal width are nearly evenly filled by
// indexer logits (a few entries each at the K-th key, where the 11-bit radix digits of the key put a fifth of the row
// into one bin), so there is no second level and no sort of the winners. A row is a chain of barriers, LDS atomics and
// one read of the row; in graphs, against a radix level over several workgroups, a second on its bin and a finishing
// sort: 4 rows of 16000 columns 9.8 us (32.7), 64 of 32768 15.3 us (39.0), 2048 of 16384 55.6 us (356).
// Where the high values crowd at the low end of the range (far outliers, skewed distributions) the bins are of the key's
// integer instead, which spaces them by magnitude. A row whose bins from the K-th key's on still hold more than BK_LIM
// entries somewhere (heavy ties, no finite value) has the K-th key's bin cut further (bk_refine). A whole row (K = n) needs
// no cut, only the sort, which is faster from 128 entries a bin on (512 rows of 2048 with 25 distinct values 36 -> 23 us).
constexpr int BK_BINS = 4096;
constexpr int BK_LIM = 256;                  // entries of a bin that are ranked by counting
constexpr int BK_LIST = TK_KMAX + BK_LIM;    // entries from the K-th key's bin on
constexpr int BK_COLS = 32768;               // columns of one workgroup
static_assert(BK_BINS == 4 * TK_NT, "a thread owns 4 bins");

struct BkLds {
  __attribute__((aligned(16))) uint32_t off[BK_BINS];   // counts, then first slots, then ends
  unsigned long long list[BK_LIST];
  __attribute__((aligned(16))) uint32_t wsum[16];
  __attribute__((aligned(16))) uint32_t red[64];        // per wave: smallest, largest finite key, smallest of its threads' largest (twice)
  uint32_t sh[8];
};

__device__ inline float unkey(uint32_t k) { return u2f((k & 0x80000000u) ? k & 0x7fffffffu : ~k); }   // okey's inverse
// vmin, scale: bins of the value; kmin, sh (by_key): of the key. bin of the K-th key (-1: none), entries from it on, in it
struct BkRange { float vmin, scale; uint32_t kmin; int sh; bool by_key; int bin; uint32_t n, c; };
template <bool KEY>
__device__ inline int bk_bin(float v, const BkRange& r) {
  if constexpr (KEY) {
    const uint32_t k = okey(v);
    return k < r.kmin ? 0 : (int)min((k - r.kmin) >> r.sh, (uint32_t)(BK_BINS - 1));
  }
  const float t = fminf(fmaxf((v - r.vmin) * r.scale, 0.f), (float)(BK_BINS - 1));   // -inf: 0; +inf: the last bin
  return v != v ? BK_BINS - 1 : (int)t;                                                // NaN is the largest key
}
__device__ inline int bk_bin(float v, const BkRange& r) { return r.by_key ? bk_bin<true>(v, r) : bk_bin<false>(v, r); }

// Bins of the n keys v (bit i of vm: v[i] is one), K of them wanted (0 < K <= n): L.off = every bin's first slot. False
// (uniform) when bk_refine has to do it. upper: the range starts at the smallest of the threads' largest values instead of
// the smallest value (2 K <= n, columns dealt to the threads: 1024 values at least and of independent ones a fifth to
// four fifths of the row lie above it; where the K-th does not, bk_refine finds it in bin 0), so that values far below
// cost no resolution. The lowest bin is not counted but is what the others leave: a floor of equal values, -inf and
// everything below the range would queue at its counter. us, 64 rows of 32768, K = 2048, radix passes / range from
// the smallest value, all bins counted / this: half the row at a floor 32 / 27 / 15.5, Cauchy 31 / 62 / 17, far outlier above 31
// / 37 / 18, Gaussian 31 / 15.8 / 15.5.
template <int EPT>
__device__ inline bool bk_bins(BkLds& L, const float (&v)[EPT], uint32_t vm, uint32_t n, uint32_t K, bool upper, BkRange& r) {
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  float mn = __builtin_inff(), mx = -__builtin_inff();
#pragma unroll
  for (int i = 0; i < EPT; ++i) {
    const bool fin = ((vm >> i) & 1u) && __builtin_fabsf(v[i]) < __builtin_inff();
    mn = fin ? fminf(mn, v[i]) : mn;
    mx = fin ? fmaxf(mx, v[i]) : mx;
  }
  const uint32_t kn = wave_minmax<false>(okey(mn)), kx = wave_minmax<true>(okey(mx));
  const uint32_t kq = wave_minmax<false>(mx == -__builtin_inff() ? ~0u : okey(mx));        // (~0: no finite key)
  if (lane == 0) { L.red[wv] = kn; L.red[16 + wv] = kx; L.red[32 + wv] = kq; L.red[48 + wv] = kq == ~0u ? 0u : kq; }
  ((u32x4*)L.off)[tid] = u32x4{0u, 0u, 0u, 0u};
  if (tid < 8) L.sh[tid] = 0u;
  __syncthreads();
  const uint32_t x = L.red[lane];                         // a 16-lane row each
  const uint32_t xx = row_minmax<true>(x), xn = row_minmax<false>(x);
  const uint32_t an = lane_of(xn, 0), ax = lane_of(xx, 16), aq = lane_of(xn, 32);
  const float q = unkey(lane_of(xx, 48));                 // (of a wave's 64 threads with EPT values each: a high quantile)
  const bool high = upper && aq < ax;
  r.bin = -1;
  r.kmin = high ? aq : an;
  r.vmin = unkey(r.kmin);
  const float span = unkey(ax) - r.vmin;
  r.scale = ((float)BK_BINS - 0.01f) / span;
  if (!(r.scale > 0.f && r.scale < __builtin_inff())) return false;   // no finite value, one value, or an overflow
  r.sh = max(0, 20 - (int)__builtin_clz((ax - r.kmin) | 1u));         // (ax - kmin) >> sh < 4096
  // by key when the high values lie that low in the range: bins of equal width would hold hundreds of them each
  r.by_key = q >= r.vmin && (q - r.vmin) * (high ? 128.f : 2048.f / (float)EPT) < span;
  auto count = [&](auto key) {
#pragma unroll
    for (int i = 0; i < EPT; ++i)
      if ((vm >> i) & 1u) {
        const int b = bk_bin<decltype(key)::value>(v[i], r);
        if (b) atomicAdd(&L.off[b], 1u);
      }
  };
  if (r.by_key) count(std::true_type()); else count(std::false_type());
  __syncthreads();
  u32x4* own = (u32x4*)L.off + (TK_NT - 1 - tid);      // bins 4095 - 4 t (element 3) down to 4092 - 4 t
  u32x4 h = *own;
  uint32_t tot;
  uint32_t run = block_excl_scan(h[0] + h[1] + h[2] + h[3], L.wsum, &tot);
  uint32_t big = 0;
#pragma unroll
  for (int e = 3; e >= 0; --e) {
    const uint32_t c = e == 0 && tid == TK_NT - 1 ? n - run : h[e];
    if (run < K) big = max(big, c);
    if (run < K && run + c >= K) { L.sh[1] = (uint32_t)(BK_BINS - 4 - 4 * tid + e); L.sh[2] = run + c; L.sh[3] = c; }
    h[e] = run;
    run += c;
  }
  *own = h;
  big = wave_minmax<true>(big);
  if (lane == 0) atomicMax(&L.sh[0], big);
  __syncthreads();
  r.bin = (int)L.sh[1];
  r.n = L.sh[2];
  r.c = L.sh[3];
  return L.sh[0] <= (K == n ? (uint32_t)BK_LIM / 2 : (uint32_t)BK_LIM);
}

// Entries in registers: (key, ~column) of entry i as key(i), low(i), its value val(i). fence: what follows is computed from the registers
// again (the compiler would keep keys and columns of all entries beside them, and spill).
template <int EPT>
struct RowRegs {                                           // columns c + 4096 (i / 4) + i % 4 of a row
  float (&v)[EPT];
  int c;
  __device__ float val(int i) const { return v[i]; }
  __device__ uint32_t key(int i) const { return okey(v[i]); }
  __device__ uint32_t low(int i) const { return ~(uint32_t)(c + 4 * TK_NT * (i >> 2) + (i & 3)); }
  __device__ void fence() {
#pragma unroll
    for (int i = 0; i < EPT; ++i) asm volatile("" : "+v"(v[i]));
    asm volatile("" : "+v"(c));
  }
};
template <int EPT>
struct ListRegs {
  unsigned long long (&e)[EPT];
  __device__ float val(int i) const { return unkey(key(i)); }
  __device__ uint32_t key(int i) const { return (uint32_t)(e[i] >> 32); }
  __device__ uint32_t low(int i) const { return (uint32_t)e[i]; }
  __device__ void fence() {
#pragma unroll
    for (int i = 0; i < EPT; ++i) asm volatile("" : "+v"(e[i]));
  }
};

// The K best of the n entries ent (bit i of vm: entry i is one; all different) into L.list in no order, after bk_bins gave
// up: the bin of the K-th key (r.bin; -1: all) is cut by its keys' range into 4096 bins of a power of two, then that bin
// again, then, between equal keys, by column (lo .. hi: the range of ~column), until the bin is taken whole or its entries
// can be ranked by counting. A chain of barriers and of same-bin atomics of the equal values. us, several workgroups' radix
// passes / a radix select over (key, column) that re-read the row / this: 64 rows of 32768: 25 distinct values 35 / 73 / 34
// (fp16 33 / 75 / 35), 1 % of the values not zero 107 / 196 / 35, one value 107 / 161 / 27; 64 of 131072: 55 / 113 / 52 (fp16
// 46 / 111 / 50), 477 / 254 / 55, 478 / 214 / 45.
template <int EPT, class Ent>
__device__ inline void bk_refine(BkLds& L, Ent ent, uint32_t vm, uint32_t n, const BkRange& r, uint32_t K, uint32_t lo,
                                 uint32_t hi) {
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  uint32_t sm = 0u, cm = vm, above = 0u, c = n;            // selected entries, candidates; their numbers
  auto fence = [&]() { ent.fence(); asm volatile("" : "+v"(sm), "+v"(cm)); };
  auto above_bin = [&](auto key) {
    fence();
#pragma unroll
    for (int i = 0; i < EPT; ++i) {
      const int b = bk_bin<decltype(key)::value>(ent.val(i), r);
      const uint32_t bit = cm & (1u << i);
      sm |= b > r.bin ? bit : 0u;
      cm &= b != r.bin ? ~bit : ~0u;
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  if (r.bin >= 0) {
    above = r.n - r.c;
    c = r.c;
    if (r.by_key) above_bin(std::true_type()); else above_bin(std::false_type());
  }
  bool col = false;
  uint32_t rl = 0u, rw = 0u;                               // the candidates' keys (or ~columns): rl .. rl + rw
  // a cut leaves 12 bits less of the range: at most 3 by key and 2 by column, after which one entry is left
#pragma unroll 1
  for (int cut = 0; cut < 5 && c > (uint32_t)BK_LIM && above + c != K; ++cut) {       // uniform
    __syncthreads();                                       // L.red, L.sh are read
    if (!col) {
      uint32_t mn = 0xffffffffu, mx = 0u;
      fence();
#pragma unroll
      for (int i = 0; i < EPT; ++i) {
        const uint32_t k = ent.key(i);
        mn = min(mn, (cm >> i) & 1u ? k : 0xffffffffu);
        mx = max(mx, (cm >> i) & 1u ? k : 0u);
        __builtin_amdgcn_sched_barrier(0);
      }
      mn = wave_minmax<false>(mn);
      mx = wave_minmax<true>(mx);
      if (lane == 0) { L.red[wv] = mn; L.red[16 + wv] = mx; }
      __syncthreads();
      rl = wave_minmax<false>(L.red[lane & 15]);
      rw = wave_minmax<true>(L.red[16 + (lane & 15)]) - rl;
      if (rw == 0u) { col = true; rl = lo; rw = hi - lo; }
    }
    const int s = max(0, 20 - (int)__builtin_clz(rw | 1u));            // rw >> s < 4096
    auto digit = [&](int i) -> uint32_t { return ((col ? ent.low(i) : ent.key(i)) - rl) >> s; };
    ((u32x4*)L.off)[tid] = u32x4{0u, 0u, 0u, 0u};
    __syncthreads();
    fence();
#pragma unroll
    for (int i = 0; i < EPT; ++i)
      if ((cm >> i) & 1u) atomicAdd(&L.off[digit(i)], 1u);
    __syncthreads();
    const u32x4 h = ((u32x4*)L.off)[TK_NT - 1 - tid];      // bins 4095 - 4 t (element 3) down to 4092 - 4 t
    uint32_t tot;
    uint32_t run = above + block_excl_scan(h[0] + h[1] + h[2] + h[3], L.wsum, &tot);
#pragma unroll
    for (int e = 3; e >= 0; --e) {
      if (run < K && run + h[e] >= K) { L.sh[1] = (uint32_t)(BK_BINS - 4 - 4 * tid + e); L.sh[2] = run; L.sh[3] = h[e]; }
      run += h[e];
    }
    __syncthreads();
    const uint32_t b = L.sh[1];
    above = L.sh[2];
    c = L.sh[3];
    fence();
#pragma unroll
    for (int i = 0; i < EPT; ++i) {
      const uint32_t d = digit(i), bit = cm & (1u << i);
      sm |= d > b ? bit : 0u;
      cm &= d != b ? ~bit : ~0u;
      __builtin_amdgcn_sched_barrier(0);
    }
    rl += b << s;
    rw = min(rw - (b << s), (1u << s) - 1u);
  }
  // the selected, and the candidates (at most BK_LIM, unless they are all taken)
  const bool whole = above + c == K;
  if (whole) { sm |= cm; cm = 0u; }
  unsigned long long* cand = (unsigned long long*)L.off;
  __syncthreads();                                         // L.off is read
  uint32_t tot;
  const uint32_t at = block_excl_scan((uint32_t)__popc(sm) | ((uint32_t)__popc(cm) << 16), L.wsum, &tot);
  uint32_t so = at & 0xffffu, co = at >> 16;
  fence();
#pragma unroll
  for (int i = 0; i < EPT; ++i) {
    const unsigned long long e = ((unsigned long long)ent.key(i) << 32) | ent.low(i);
    if ((sm >> i) & 1u) { if (so < (uint32_t)BK_LIST) L.list[so] = e; ++so; }
    if ((cm >> i) & 1u) { if (co < (uint32_t)BK_LIM) cand[co] = e; ++co; }
    __builtin_amdgcn_sched_barrier(0);
  }
  __syncthreads();
  if (!whole) {                                            // four lanes rank a candidate
    const uint32_t i = (uint32_t)tid >> 2, nc = min(c, (uint32_t)BK_LIM);
    const unsigned long long e = i < nc ? cand[i] : 0ull;
    uint32_t rank = 0u;
#pragma unroll 4
    for (uint32_t j = (uint32_t)tid & 3u; j < nc; j += 4u) rank += (uint32_t)(cand[j] > e);
    rank += (uint32_t)__builtin_amdgcn_mov_dpp((int)rank, 0xb1, 0xf, 0xf, false);
    rank += (uint32_t)__builtin_amdgcn_mov_dpp((int)rank, 0x4e, 0xf, 0xf, false);
    if ((tid & 3) == 0 && i < nc && rank < K - above) L.list[above + rank] = e;
  }
  __syncthreads();
}

// Columns c0 .. c1 - 1 of a logits row (at most EPT * 1024): v[4 g + e] = column c0 + 4 (tid + 1024 g) + e as fp32, and
// the mask of the columns that exist. Through a buffer that ends at c1 (reads past it give 0), so no load is under a
// branch; 4 columns a load on aligned rows (the last, partial four by single loads).
template <bool F16, int EPT>
__device__ inline uint32_t bk_load(const void* row, int c0, int c1, float (&v)[EPT]) {
  constexpr int ES = F16 ? 2 : 4;
  const int tid = threadIdx.x, n = c1 - c0;
  const uint64_t a = (uint64_t)(uintptr_t)row + (uint64_t)c0 * ES;
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)a), hi = __builtin_amdgcn_readfirstlane((uint32_t)(a >> 32));
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(uintptr_t)(((uint64_t)hi << 32) | lo), (short)0, n * ES, 0x00020000);
  auto one = [&](int j) -> float {
    if constexpr (F16) return (float)__builtin_bit_cast(_Float16, (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(rs, 2 * j, 0, 0));
    else return u2f(__builtin_amdgcn_raw_buffer_load_b32(rs, 4 * j, 0, 0));
  };
  uint32_t vm = 0;
  if ((lo & (4 * ES - 1)) == 0u) {
#pragma unroll
    for (int g = 0; g < EPT / 4; ++g) {
      const int j = 4 * (tid + TK_NT * g);
      const int at = j + 4 <= n ? j * ES : n * ES;         // past the end: zeros
      if constexpr (F16) {
        typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
        typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
        const f16x4 x = __builtin_bit_cast(f16x4, (u32x2)__builtin_amdgcn_raw_buffer_load_b64(rs, at, 0, 0));
#pragma unroll
        for (int e = 0; e < 4; ++e) v[4 * g + e] = (float)x[e];
      } else {
        const f32x4 x = __builtin_bit_cast(f32x4, (u32x4)__builtin_amdgcn_raw_buffer_load_b128(rs, at, 0, 0));
#pragma unroll
        for (int e = 0; e < 4; ++e) v[4 * g + e] = x[e];
      }
    }
    const int q = n >> 2;                                  // the partial four, if any, is group q / 1024 of thread q % 1024
    if ((n & 3) && tid == (q & (TK_NT - 1))) {
#pragma unroll
      for (int g = 0; g < EPT / 4; ++g)
        if (g == q >> 10) {
#pragma unroll
          for (int e = 0; e < 3; ++e) v[4 * g + e] = one(4 * q + e);
        }
    }
  } else {
#pragma unroll
    for (int i = 0; i < EPT; ++i) v[i] = one(4 * (tid + TK_NT * (i >> 2)) + (i & 3));
  }
#pragma unroll
  for (int i = 0; i < EPT; ++i) {
    vm |= (uint32_t)(4 * (tid + TK_NT * (i >> 2)) + (i & 3) < n) << i;
    if constexpr (F16) asm volatile("" : "+v"(v[i]));     // (the fp16 values would be kept beside them)
  }
  return vm;
}

// The entries of L.list from the K-th key's bin on, in final order, to o[0, K) (column, -1 for +-inf), and -1 to kout.
__device__ inline void bk_emit(BkLds& L, const BkRange& r, uint32_t K, int kout, int* o) {
  for (uint32_t i = threadIdx.x; i < r.n; i += TK_NT) {
    const unsigned long long e = L.list[i];
    const int b = bk_bin(unkey((uint32_t)(e >> 32)), r);
    const uint32_t end = L.off[b];                        // the appends moved a bin's first slot to its end
    uint32_t at = b + 1 < BK_BINS ? L.off[b + 1] : 0u, first = at;
    for (uint32_t j = first; j < end; ++j) at += (uint32_t)(L.list[j] > e);
    if (at < K) o[at] = inf_key<false>((uint32_t)(e >> 32)) ? -1 : (int)~(uint32_t)e;
  }
  for (int s = (int)K + (int)threadIdx.x; s < kout; s += TK_NT) o[s] = -1;
}
__device__ inline void bk_emit_sorted(BkLds& L, uint32_t K, int kout, int* o) {   // after bk_refine
  tk_sort_desc(L.list, (int)K);
  for (int s = threadIdx.x; s < kout; s += TK_NT) {
    int c = -1;
    if (s < (int)K) {
      const unsigned long long e = L.list[s];
      if (!inf_key<false>((uint32_t)(e >> 32))) c = (int)~(uint32_t)e;
    }
    o[s] = c;
  }
}

// Rows of at most EPT * 1024 columns, one workgroup each. Two workgroups share a compute unit up to 16 keys a thread.
template <bool F16, int EPT>
__global__ void __launch_bounds__(TK_NT, EPT <= 16 ? 8 : 4) topk_row_kernel(TopkParams p) {
  __shared__ BkLds L;
  const int row = blockIdx.x, tid = threadIdx.x;
  int n = p.ctx[row];
  n = n < 0 ? 0 : (n > p.Lc ? p.Lc : n);
  int* o = p.out + (long long)row * p.out_st;
  const uint32_t K = (uint32_t)min(n, p.K);
  if (K == 0) {                                           // uniform
    for (int s = tid; s < p.K; s += TK_NT) o[s] = -1;
    return;
  }
  const void* x = lrow<F16>(p.lg, row, p.lg_st);
  float v[EPT];
  const uint32_t vm = bk_load<F16, EPT>(x, 0, n, v);
  BkRange r;
  if (!bk_bins<EPT>(L, v, vm, (uint32_t)n, K, 2u * K <= (uint32_t)n, r)) {
    bk_refine<EPT>(L, RowRegs<EPT>{v, 4 * tid}, vm, (uint32_t)n, r, K, ~(uint32_t)(n - 1), ~0u);
    bk_emit_sorted(L, K, p.K, o);
    return;
  }
  auto append = [&](auto key) {
#pragma unroll
    for (int i = 0; i < EPT; ++i) {
      const int b = bk_bin<decltype(key)::value>(v[i], r);
      if (((vm >> i) & 1u) && b >= r.bin) L.list[atomicAdd(&L.off[b], 1u)] = tk_pack(okey(v[i]), 4 * (tid + TK_NT * (i >> 2)) + (i & 3));
    }
  };
  if (r.by_key) append(std::true_type()); else append(std::false_type());
  __syncthreads();
  bk_emit(L, r, K, p.K, o);
}

// Longer rows: a workgroup per chunk of at most 32768 columns writes its entries that can be among the row's K (its
// own K best and the rest of their last bin) to a list in the workspace, then one workgroup per row selects and sorts
// over the lists. 64 rows of 131072 columns 26.7 us against 50.6 for the radix passes, 1024 of 65536 132 against 560.
struct BkWs {                                             // workspace of a row: G list lengths, then G lists
  static constexpr int GMAX = 8;
  static constexpr long long LISTS = 64;                  // bytes before the lists
  static constexpr long long row_bytes(int G) { return LISTS + (long long)G * BK_LIST * 8; }
};
static_assert(BkWs::GMAX * 4 <= BkWs::LISTS && BkWs::row_bytes(1) % 64 == 0, "lengths before the lists, rows 64-byte aligned");
struct TopkChunkParams {
  const void* lg; long long lg_st;
  const int* ctx; int rows, Lc, K;
  int* out; long long out_st;
  uint8_t* ws; long long row_bytes; int G, CL;            // chunks per row, columns per chunk
};

template <bool F16>
__global__ void __launch_bounds__(TK_NT) topk_chunk_kernel(TopkChunkParams p) {
  constexpr int EPT = BK_COLS / TK_NT;
  __shared__ BkLds L;
  const int row = blockIdx.x, g = blockIdx.y, tid = threadIdx.x;
  int n = p.ctx[row];
  n = n < 0 ? 0 : (n > p.Lc ? p.Lc : n);
  uint8_t* wr = p.ws + (long long)row * p.row_bytes;
  unsigned long long* list = (unsigned long long*)(wr + BkWs::LISTS) + (long long)g * BK_LIST;
  const int c0 = min(g * p.CL, n), c1 = min(c0 + p.CL, n);
  const uint32_t K = (uint32_t)min(c1 - c0, p.K);
  if (K == 0) {
    if (tid == 0) ((uint32_t*)wr)[g] = 0u;
    return;
  }
  const void* x = lrow<F16>(p.lg, row, p.lg_st);
  float v[EPT];
  const uint32_t vm = bk_load<F16, EPT>(x, c0, c1, v);
  BkRange r;
  if (!bk_bins<EPT>(L, v, vm, (uint32_t)(c1 - c0), K, 2u * K <= (uint32_t)(c1 - c0), r)) {
    bk_refine<EPT>(L, RowRegs<EPT>{v, c0 + 4 * tid}, vm, (uint32_t)(c1 - c0), r, K, ~(uint32_t)(c1 - 1), ~(uint32_t)c0);
    for (uint32_t i = tid; i < K; i += TK_NT) list[i] = L.list[i];
    if (tid == 0) ((uint32_t*)wr)[g] = K;
    return;
  }
  auto append = [&](auto key) {
#pragma unroll
    for (int i = 0; i < EPT; ++i) {
      const int b = bk_bin<decltype(key)::value>(v[i], r);
      if (((vm >> i) & 1u) && b >= r.bin) list[atomicAdd(&L.off[b], 1u)] = tk_pack(okey(v[i]), c0 + 4 * (tid + TK_NT * (i >> 2)) + (i & 3));
    }
  };
  if (r.by_key) append(std::true_type()); else append(std::false_type());
  if (tid == 0) ((uint32_t*)wr)[g] = r.n;
}

template <int G>                                          // lists per row, rounded up
__global__ void __launch_bounds__(TK_NT) topk_lists_kernel(TopkChunkParams p) {
  constexpr int EPT = (G * BK_LIST + TK_NT - 1) / TK_NT;
  __shared__ BkLds L;
  const int row = blockIdx.x, tid = threadIdx.x;
  int n = p.ctx[row];
  n = n < 0 ? 0 : (n > p.Lc ? p.Lc : n);
  int* o = p.out + (long long)row * p.out_st;
  const uint32_t K = (uint32_t)min(n, p.K);
  if (K == 0) {
    for (int s = tid; s < p.K; s += TK_NT) o[s] = -1;
    return;
  }
  const uint8_t* wr = p.ws + (long long)row * p.row_bytes;
  const int m = p.G * BK_LIST;                            // places of the row's lists one after another
  unsigned long long e[EPT];
  float v[EPT];
  uint32_t vm = 0, cnt[EPT];
#pragma unroll
  for (int i = 0; i < EPT; ++i) {                         // every place is read, the unused ones dropped
    const int j = min(tid + TK_NT * i, m - 1);
    e[i] = ((const unsigned long long*)(wr + BkWs::LISTS))[j];
    cnt[i] = ((const uint32_t*)wr)[j / BK_LIST];
  }
#pragma unroll
  for (int i = 0; i < EPT; ++i) {
    const int j = tid + TK_NT * i;
    if (j >= m || (uint32_t)(j % BK_LIST) >= cnt[i]) e[i] = 0ull;
  }
#pragma unroll
  for (int i = 0; i < EPT; ++i) {
    vm |= (uint32_t)(e[i] != 0ull) << i;
    v[i] = unkey((uint32_t)(e[i] >> 32));
  }
  BkRange r;
  uint32_t have = 0u;
  for (int g = 0; g < p.G; ++g) have += ((const uint32_t*)wr)[g];
  if (!bk_bins<EPT>(L, v, vm, have, K, false, r)) {
    bk_refine<EPT>(L, ListRegs<EPT>{e}, vm, have, r, K, ~(uint32_t)(n - 1), ~0u);
    bk_emit_sorted(L, K, p.K, o);
    return;
  }
  auto append = [&](auto key) {
#pragma unroll
    for (int i = 0; i < EPT; ++i) {
      const int b = bk_bin<decltype(key)::value>(v[i], r);
      if (((vm >> i) & 1u) && b >= r.bin) L.list[atomicAdd(&L.off[b], 1u)] = e[i];
    }
  };
  if (r.by_key) append(std::true_type()); else append(std::false_type());
  __syncthreads();
  bk_emit(L, r, K, p.K, o);
}

// ---- top-k over several workgroups per row (workspace variant) -------------------------------------------
// Two radix levels run across G workgroups per row (chunks of at most CL columns):
//   hist:    the histogram of the level-0 11-bit digit over each chunk's keys;
//   collect: every workgroup sums the G histograms of the level and finds the boundary bin b of the row's
//            remaining need; it writes its chunk's keys above b (and in b when that completes the need) to the row's
//            winner list, and the keys in b to the candidate list when the bin holds at most TK_CAP1 keys. A chunk's
//            entries start at the offset the histograms of the chunks before it give; inside the chunk each wave
//            takes its slots from a block scan per pass over 8 consecutive columns per thread, so every list is
//            in column order (the finishing pass's stable radix sort of fp16 keys relies on it). Otherwise the
//            next level narrows the prefix to b, and this pass also builds its chunk's histogram of that level
//            (into the other half of the histogram buffer, which no workgroup of the row is reading).
// A finishing pass (one workgroup per row) resolves the candidates' remaining levels, sorts the K winners and
// writes the positions. Rows with n <= K, and rows whose bin is still too large after two levels (heavy ties), run
// the one-workgroup selection there. Per-row state lives in the workspace, one header per level (the collect pass
// of level L reads header L and its first workgroup writes header L + 1).
enum : int { TKW_SELECT = 0, TKW_WHOLE = 1, TKW_CANDS = 2, TKW_FALLBACK = 3 };
struct __attribute__((aligned(32))) TkwHdr { int state, prefix, mask, need, sb, binc, lvl; };

struct TopkWs {
  int G, CL;                                      // chunks per row, columns per chunk (multiple of 1024)
  long long row_bytes;                            // workspace bytes per row
  __host__ __device__ TkwHdr* hdr(uint8_t* ws, int row) const { return (TkwHdr*)(ws + row * row_bytes); }
  __host__ __device__ unsigned long long* sel(uint8_t* ws, int row) const {
    return (unsigned long long*)(ws + row * row_bytes + 3 * sizeof(TkwHdr));
  }
  __host__ __device__ unsigned long long* cand(uint8_t* ws, int row) const { return sel(ws, row) + TK_KMAX; }
  __host__ __device__ uint32_t* hist(uint8_t* ws, int row) const { return (uint32_t*)(cand(ws, row) + TK_CAP); }
};

__host__ inline TopkWs topk_ws_layout(int Lc) {
  TopkWs w;
  // chunks of 8192 columns, at most 4 per row (every collect workgroup reads all G histograms of its row; with
  // 8 chunks at 131072 columns the passes took 69.6 us against 58.8 with 4, B = 64). The passes run above 262144
  // columns; below, the layout only gives the limits of spmla_topk_scratch and spmla_index_logits_hist.
  int G = (Lc + 8191) / 8192;
  if (G > 4) G = 4;
  if (G < 1) G = 1;
  int CL = (Lc + G - 1) / G;
  CL = (CL + 1023) / 1024 * 1024;
  w.G = G; w.CL = CL;
  w.row_bytes = 3 * (long long)sizeof(TkwHdr) + (long long)(TK_KMAX + TK_CAP) * 8 + 2LL * G * 2048 * 4 + 16;
  w.row_bytes = (w.row_bytes + 15) / 16 * 16;
  return w;
}

struct TopkWsParams {
  const void* lg; long long lg_st;                // fp32 or fp16 (the kernels' F16), stride in elements
  const int* ctx; int rows, Lc, K;
  int* out; long long out_st;
  uint8_t* ws; TopkWs w;
  int level;
};

__device__ inline int tkw_n(const TopkWsParams& p, int row) {
  const int n = p.ctx[row];
  return n < 0 ? 0 : (n > p.Lc ? p.Lc : n);
}

// the row's state entering level p.level (level 0: select everything, need K)
__device__ inline TkwHdr tkw_state(const TopkWsParams& p, int row) {
  if (p.level == 0) return TkwHdr{TKW_SELECT, 0, 0, p.K, 0, 0, 0};
  return p.w.hdr(p.ws, row)[p.level];
}

template <bool F16>
__global__ void __launch_bounds__(TK_NT) topk_hist_kernel(TopkWsParams p) {
  __shared__ uint32_t hist[TK_HCOPY * TK_HSTR];
  const int row = blockIdx.x, g = blockIdx.y, tid = threadIdx.x;
  const int n = tkw_n(p, row);
  if (n <= p.K) return;
  const TkwHdr st = tkw_state(p, row);
  if (st.state != TKW_SELECT) return;
  const int shift = tk_shift(p.level);
  const uint32_t prefix = (uint32_t)st.prefix, mask = (uint32_t)st.mask;
  for (int i = tid; i < TK_HCOPY * TK_HSTR; i += TK_NT) hist[i] = 0;
  __syncthreads();
  const void* x = lrow<F16>(p.lg, row, p.lg_st);
  const int c0 = g * p.w.CL, c1 = min(c0 + p.w.CL, n);
  for (int base = c0; base < c1; base += 8 * TK_NT) {
    uint32_t k[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int j = base + i * TK_NT + tid;
      k[i] = j < c1 ? lkey<F16>(x, j) : 0u;
    }
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (base + i * TK_NT + tid < c1 && (k[i] & mask) == prefix)
        atomicAdd(&hist[(tid & (TK_HCOPY - 1)) * TK_HSTR + ((k[i] >> shift) & 0x7ffu)], 1u);
  }
  __syncthreads();
  uint32_t* out = p.w.hist(p.ws, row) + (long long)g * 2048;
  for (int b = tid; b < 2048; b += TK_NT) {
    uint32_t h = 0;
#pragma unroll
    for (int c = 0; c < TK_HCOPY; ++c) h += hist[c * TK_HSTR + b];
    out[b] = h;
  }
}

template <bool F16>
__global__ void __launch_bounds__(TK_NT) topk_collect_kernel(TopkWsParams p) {
  __shared__ __attribute__((aligned(16))) uint32_t wsum[17];
  __shared__ uint32_t sh[8];
  __shared__ uint32_t nh[TK_HCOPY * TK_HSTR];       // the next level's histogram of this chunk (when narrowing)
  const int row = blockIdx.x, g = blockIdx.y, tid = threadIdx.x;
  const TkwHdr st = tkw_state(p, row);              // read beside the row length: one round trip for both
  const int n = tkw_n(p, row);
  if (n <= p.K) return;
  TkwHdr* next = p.w.hdr(p.ws, row) + p.level + 1;
  if (st.state != TKW_SELECT) {                     // settled at an earlier level: carry the state forward
    if (g == 0 && tid == 0) *next = st;
    return;
  }
  const int shift = tk_shift(p.level);
  const uint32_t prefix = (uint32_t)st.prefix, mask = (uint32_t)st.mask, need = (uint32_t)st.need;
  // thread t owns bins 2047 - 2t, 2046 - 2t: totals over the G chunks and over the chunks before g
  const int b0 = 2047 - 2 * tid, b1 = b0 - 1;
  const uint32_t* hs = p.w.hist(p.ws, row) + (long long)(p.level & 1) * p.w.G * 2048;
  uint32_t t0 = 0, t1 = 0, q0 = 0, q1 = 0;
  for (int c = 0; c < p.w.G; ++c) {
    const uint32_t h0 = hs[(long long)c * 2048 + b0], h1 = hs[(long long)c * 2048 + b1];
    t0 += h0; t1 += h1;
    if (c < g) { q0 += h0; q1 += h1; }
  }
  // defaults: with histograms that do not add up to the row (a workspace that was never filled for these logits) no
  // thread finds the boundary; the lists below are bounds-checked either way, so such a call writes only its own lists
  if (tid == 0) { sh[1] = 0u; sh[2] = 0u; sh[3] = 0u; sh[4] = 0u; }
  uint32_t tot;
  const uint32_t before = block_excl_scan(t0 + t1, wsum, &tot);
  if (before < need && before + t0 >= need) { sh[1] = (uint32_t)b0; sh[2] = before; sh[3] = t0; }
  if (before + t0 < need && before + t0 + t1 >= need) { sh[1] = (uint32_t)b1; sh[2] = before + t0; sh[3] = t1; }
  __syncthreads();
  const uint32_t b = sh[1], above = sh[2], binc = sh[3];
  const bool whole = above + binc == need;
  const bool fits = !whole && binc <= (uint32_t)TK_CAP1;
  // this chunk's offsets: winners of the chunks before g (bins above b, and b itself when whole); candidates in b
  const uint32_t mine = ((uint32_t)b0 > b || (whole && (uint32_t)b0 == b) ? q0 : 0u) +
                        ((uint32_t)b1 > b || (whole && (uint32_t)b1 == b) ? q1 : 0u);
  uint32_t sum;
  (void)block_excl_scan(mine, wsum, &sum);
  if ((uint32_t)b0 == b) sh[4] = q0;
  if ((uint32_t)b1 == b) sh[4] = q1;
  __syncthreads();
  const uint32_t sb = (uint32_t)st.sb + sum, cb = sh[4];   // this chunk's first winner / candidate slot
  const bool narrow = !whole && !fits && p.level + 1 < 2;   // uniform per row: the next level runs on bin b
  const int nshift = tk_shift(p.level + 1);
  if (narrow) {
    for (int i = tid; i < TK_HCOPY * TK_HSTR; i += TK_NT) nh[i] = 0;
    __syncthreads();
  }
  if (g == 0 && tid == 0) {
    TkwHdr h = st;
    h.prefix = (int)(prefix | (b << shift));
    h.mask = (int)(mask | (0x7ffu << shift));
    h.need = (int)(need - above);
    h.sb = st.sb + (int)above;
    h.binc = (int)binc;
    h.lvl = p.level + 1;
    if (whole) { h.state = TKW_WHOLE; h.sb = st.sb + (int)need; }
    else if (fits) h.state = TKW_CANDS;
    else h.state = p.level + 1 < 2 ? TKW_SELECT : TKW_FALLBACK;
    *next = h;
  }
  unsigned long long* sel = p.w.sel(p.ws, row);
  unsigned long long* cand = p.w.cand(p.ws, row);
  const void* x = lrow<F16>(p.lg, row, p.lg_st);
  const int c0 = g * p.w.CL, c1 = min(c0 + p.w.CL, n);      // the columns this workgroup visits
  // thread t visits the 8 consecutive entries 8t .. 8t + 7 of each 8192-entry pass, and the slots of a pass come
  // from one block scan of the per-thread counts: every list the pass appends to stays in column order (the
  // finishing pass's stable sort relies on it to order equal keys by column)
  const bool vec = ((uintptr_t)x & 15u) == 0u;              // 16-byte aligned row: vector loads
  uint32_t sbase = sb, cbase = cb;                  // running slot bases of this chunk's lists
  for (int base = c0; base < c1; base += 8 * TK_NT) {
    uint32_t k[8];
    const int j0 = base + 8 * tid;
    if (vec && j0 + 8 <= c1) {
      if constexpr (F16) {
        const u32x4 v = *(const u32x4*)((const uint16_t*)x + j0);
#pragma unroll
        for (int i = 0; i < 4; ++i) { k[2 * i] = okey16(v[i] & 0xffffu); k[2 * i + 1] = okey16(v[i] >> 16); }
      } else {
        const f32x4 a = *(const f32x4*)((const float*)x + j0), b = *(const f32x4*)((const float*)x + j0 + 4);
#pragma unroll
        for (int i = 0; i < 4; ++i) { k[i] = okey(a[i]); k[4 + i] = okey(b[i]); }
      }
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) k[i] = j0 + i < c1 ? lkey<F16>(x, j0 + i) : 0u;
    }
    uint32_t selm = 0, candm = 0, binm = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const bool in = j0 + i < c1 && (k[i] & mask) == prefix;
      const uint32_t d = (k[i] >> shift) & 0x7ffu;
      selm |= (uint32_t)(in && (d > b || (whole && d == b))) << i;
      candm |= (uint32_t)(in && fits && d == b) << i;
      binm |= (uint32_t)(in && d == b) << i;
    }
    // both counts stay below 2^16: a pass holds 8192 entries
    uint32_t tot;
    const uint32_t off = block_excl_scan((uint32_t)__popc(selm) | ((uint32_t)__popc(candm) << 16), wsum, &tot);
    uint32_t so = sbase + (off & 0xffffu), co = cbase + (off >> 16);
    sbase += tot & 0xffffu;
    cbase += tot >> 16;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      if ((selm >> i) & 1u) { if (so < (uint32_t)TK_KMAX) sel[so] = tk_pack(k[i], j0 + i); ++so; }
      if ((candm >> i) & 1u) { if (co < (uint32_t)TK_CAP) cand[co] = tk_pack(k[i], j0 + i); ++co; }
      if (narrow && ((binm >> i) & 1u))
        atomicAdd(&nh[(tid & (TK_HCOPY - 1)) * TK_HSTR + ((k[i] >> nshift) & 0x7ffu)], 1u);
    }
  }
  if (narrow) {                                     // level L + 1's histograms go to the other half of the buffer
    __syncthreads();
    uint32_t* out = p.w.hist(p.ws, row) + (long long)(((p.level + 1) & 1) * p.w.G + g) * 2048;
    for (int bb = tid; bb < 2048; bb += TK_NT) {
      uint32_t h = 0;
#pragma unroll
      for (int c = 0; c < TK_HCOPY; ++c) h += nh[c * TK_HSTR + bb];
      out[bb] = h;
    }
  }
}

template <bool F16>
__global__ void __launch_bounds__(TK_NT) topk_finish_kernel(TopkWsParams p) {
  __shared__ TopkLds L;
  const int row = blockIdx.x, tid = threadIdx.x;
  const int n = tkw_n(p, row);
  const RowSrc<F16> src{lrow<F16>(p.lg, row, p.lg_st), n};
  int* o = p.out + (long long)row * p.out_st;
  int nsel = 0;
  const TkwHdr st = p.w.hdr(p.ws, row)[p.level];   // read beside the row length (unused when n <= K)
  const bool full = n <= p.K || (st.state != TKW_WHOLE && st.state != TKW_CANDS);
  if (full) {
    nsel = tk_select(src, p.K, L);                  // few columns, or ties too heavy for the lists
  } else {
    // the header's counts, kept inside the lists (they are, whenever the histograms were this row's)
    const int nsb = min(max(st.sb, 0), p.K), nbc = min(max(st.binc, 0), TK_CAP1);
    const uint32_t nneed = (uint32_t)min(max(st.need, 0), p.K - nsb);
    const unsigned long long* sel = p.w.sel(p.ws, row);
    for (int i = tid; i < nsb; i += TK_NT) L.sel[i] = sel[i];
    if (st.state == TKW_CANDS) {
      const unsigned long long* cand = p.w.cand(p.ws, row);
      for (int i = tid; i < nbc; i += TK_NT) L.cand[i] = cand[i];
    }
    __syncthreads();
    if (st.state == TKW_CANDS)
      tk_resolve_cands<TK_CAP1 / TK_NT>(L, nbc, st.lvl, (uint32_t)st.prefix, (uint32_t)st.mask, nneed, (uint32_t)nsb, n);
    if constexpr (F16) {
      // fp16 keys: at most two radix passes (the keys' low half is zero), faster than the bitonic network here;
      // fp32 keys need three or four, slower than it (measured on the bench's indexer logits)
      tk_emit_radix<RowSrc<F16>, F16>(src, p.K, p.K, o, L);   // the lists arrive in column order
      return;
    }
    nsel = p.K;
  }
  tk_emit_sorted(src, nsel, p.K, o, L);
}

// fast_topk.local (dotsnote/engine/arcstats_pkg/arcstats/fast_topk.py:52-66, csrc/topk_select.cu:1-13, :75-201):
// the row's valid columns are j < ceil((ctx - rank) / P) (clipped to Lc); the top kl of them go to the payload
// pk[row] = [values fp32 | positions j * P + rank as int32 bits] in ascending column order; fewer than kl valid
// columns: the rest is padded with -inf values and positions s * P + rank.
struct LocalParams {
  const void* lg; long long lg_st;                // fp32 or fp16 (the kernel's F16), stride in elements
  const int* ctx; int rows, rank, P, Lc, kl;
  float* pk;
};

template <bool F16>
__global__ void __launch_bounds__(TK_NT) topk_local_kernel(LocalParams p) {
  __shared__ TopkLds L;
  const int row = blockIdx.x, tid = threadIdx.x;
  const int c = p.ctx[row];
  int n = c > p.rank ? (int)(((long long)c - p.rank + p.P - 1) / p.P) : 0;
  if (n > p.Lc) n = p.Lc;
  const RowSrc<F16> src{lrow<F16>(p.lg, row, p.lg_st), n};
  const int nsel = tk_select(src, p.kl, L);
  // ascending column order: sort descending on ~j (the low word of a selected entry)
  for (int i = tid; i < nsel; i += TK_NT) L.sel[i] = (unsigned long long)(uint32_t)L.sel[i] << 32;
  tk_sort_desc(L.sel, nsel);
  float* pv = p.pk + (long long)row * 2 * p.kl;
  int* pp = reinterpret_cast<int*>(pv + p.kl);
  for (int s = tid; s < p.kl; s += TK_NT) {
    if (s < nsel) {
      const int j = (int)(~(uint32_t)(L.sel[s] >> 32));
      pv[s] = src.val(j);
      pp[s] = j * p.P + p.rank;
    } else {
      pv[s] = u2f(0xff800000u);
      pp[s] = s * p.P + p.rank;
    }
  }
}

// fast_topk.merge (dotsnote/engine/arcstats_pkg/arcstats/fast_topk.py:69-78, csrc/topk_select.cu:203-244): per row,
// the top kk of the P * kl all-gathered candidates by (value key desc, concatenation index asc) -> their positions,
// -1 where the value is +-inf, slots [kk, topk_tokens) = -1.
struct MergeParams {
  const float* allp; int n, P, kl, kk, topk_tokens;
  int* out; long long out_st;
};

__global__ void __launch_bounds__(TK_NT) topk_merge_kernel(MergeParams p) {
  __shared__ TopkLds L;
  const int row = blockIdx.x;
  const MergeSrc src{p.allp, p.n, row, p.kl, p.P * p.kl};
  const int nsel = tk_select(src, p.kk, L);
  tk_emit_sorted(src, nsel, p.topk_tokens, p.out + (long long)row * p.out_st, L);
}

// ------------------------------------------------------------------------------------------------ rows
// rows[t][k] = block_table[req[t]][p / bs] * stride_rows + p % bs for p = topk[t][k] >= 0 (and a valid block),
// else -1. vLLM triton_convert_req_index_to_global_index semantics (call sites dsa_sm89.py:314-315, :467-469).
__global__ void rows_kernel(const int* topk, long long tk_st, const int* req, const int* bt, long long bt_st,
                            int bt_cols, int bs, long long stride_rows, int T, int K, int* rows, long long r_st,
                            int* counts) {
  const int t = blockIdx.y;
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= T) return;
  int r = -1;
  if (k < K) {
    const int pp = topk[(long long)t * tk_st + k];
    if (pp >= 0 && pp / bs < bt_cols) {
      const int blk = bt[(long long)req[t] * bt_st + pp / bs];
      if (blk >= 0) r = (int)((long long)blk * stride_rows + pp % bs);
    }
    rows[(long long)t * r_st + k] = r;
  }
  if (counts) {
    const unsigned long long b = __ballot(k < K && r >= 0);
    if ((threadIdx.x & 63) == 0 && b) atomicAdd(&counts[t], __popcll(b));
  }
}

__global__ void zero_i32(int* p, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0;
}

// ---- scratch of the no-allocation top-k entry point (spmla_topk_scratch) ---------------------------------------
// File-scope device memory (each GPU holds its own copy from module load until the process ends). Host code never
// passes `scratch` itself to a kernel: its name is a host-side stand-in, not a device address. The device address
// comes from hipGetSymbolAddress, once per device, and is kept in scratch_dev[].
constexpr long long TOPK_SCRATCH_BYTES = 16ll << 20;
static __device__ __align__(256) uint8_t scratch[TOPK_SCRATCH_BYTES];

}  // namespace idx
}  // namespace spmla

#include <mutex>

namespace {
constexpr int SCRATCH_MAX_DEV = 64;
std::mutex scratch_mu;
void* scratch_dev[SCRATCH_MAX_DEV] = {};

// Device address of this device's `scratch` array (looked up on the first call on the device).
int scratch_ptr(void** out) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return (int)e;
  if (dev < 0 || dev >= SCRATCH_MAX_DEV) return spmla::SPMLA_ELIMIT;
  std::lock_guard<std::mutex> lock(scratch_mu);
  if (scratch_dev[dev] == nullptr) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(spmla::idx::scratch));
    if (e != hipSuccess) return (int)e;
    if (p == nullptr) return (int)hipErrorInvalidSymbol;
    scratch_dev[dev] = p;
  }
  *out = scratch_dev[dev];
  return spmla::SPMLA_OK;
}
}  // namespace

namespace spmla {
namespace idx {
// rows of at most BK_COLS columns: one workgroup each, 8 / 16 / 32 keys a thread (fewer registers and loads)
static void topk_rows(const TopkParams& p, int dtype, hipStream_t st) {
  const int v = (p.Lc <= 8 * TK_NT ? 0 : p.Lc <= 16 * TK_NT ? 2 : 4) + (dtype == 1 ? 1 : 0);
  const dim3 g(p.rows), b(TK_NT);
  switch (v) {
    case 0: hipLaunchKernelGGL((topk_row_kernel<false, 8>), g, b, 0, st, p); break;
    case 1: hipLaunchKernelGGL((topk_row_kernel<true, 8>), g, b, 0, st, p); break;
    case 2: hipLaunchKernelGGL((topk_row_kernel<false, 16>), g, b, 0, st, p); break;
    case 3: hipLaunchKernelGGL((topk_row_kernel<true, 16>), g, b, 0, st, p); break;
    case 4: hipLaunchKernelGGL((topk_row_kernel<false, 32>), g, b, 0, st, p); break;
    default: hipLaunchKernelGGL((topk_row_kernel<true, 32>), g, b, 0, st, p); break;
  }
}
static void topk_chunks(const TopkChunkParams& p, int dtype, hipStream_t st) {
  const dim3 g(p.rows, p.G), b(TK_NT);
  if (dtype == 1) hipLaunchKernelGGL(topk_chunk_kernel<true>, g, b, 0, st, p);
  else hipLaunchKernelGGL(topk_chunk_kernel<false>, g, b, 0, st, p);
  if (p.G <= 2) hipLaunchKernelGGL(topk_lists_kernel<2>, dim3(p.rows), b, 0, st, p);
  else if (p.G <= 4) hipLaunchKernelGGL(topk_lists_kernel<4>, dim3(p.rows), b, 0, st, p);
  else hipLaunchKernelGGL(topk_lists_kernel<BkWs::GMAX>, dim3(p.rows), b, 0, st, p);
}

// longer rows: the radix passes on fp32 (F16 false) or fp16 logits
template <bool F16>
static void topk_ws_passes(TopkWsParams p, hipStream_t stream) {
  p.level = 0;
  hipLaunchKernelGGL(topk_hist_kernel<F16>, dim3(p.rows, p.w.G), dim3(TK_NT), 0, stream, p);
  for (int level = 0; level < 2; ++level) {        // the level-1 histograms come from the level-0 collect
    p.level = level;
    hipLaunchKernelGGL(topk_collect_kernel<F16>, dim3(p.rows, p.w.G), dim3(TK_NT), 0, stream, p);
  }
  p.level = 2;                                      // header 2: the state after both levels
  hipLaunchKernelGGL(topk_finish_kernel<F16>, dim3(p.rows), dim3(TK_NT), 0, stream, p);
}

}  // namespace idx
}  // namespace spmla

using namespace spmla;

// Logits grid: one 8-wave workgroup per CU. With at most as many rows as CUs, each row's tiles are split over
// CUs / rows workgroups, one round of the whole grid (a wave pays its two-round-trip prologue, ~6 us under load,
// once); with more rows, workgroups of LG_TPW tiles per wave, rounds fine enough for a short tail.
inline int lg_cus() {
  static std::atomic<int> cached[64];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) dev = 0;
  int n = cached[dev].load(std::memory_order_relaxed);
  if (n <= 0) {
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
    cached[dev].store(n, std::memory_order_relaxed);
  }
  return n;
}
inline dim3 lg_grid(int rows, int cols, int& tpg) {
  const long long tiles = ((long long)cols + 31) / 32;      // per row
  const long long cus = lg_cus();
  const long long g = rows <= cus ? cus / rows : std::max(1LL, tiles / ((long long)idx::LG_NWV * idx::LG_TPW));
  tpg = (int)std::max(1LL, (tiles + g - 1) / g);
  return dim3(rows, (unsigned)((tiles + tpg - 1) / tpg));
}


// Rows per workgroup of flat_logits_kernel (0: the row-at-a-time kernel, which spreads a few rows over all compute
// units). A workgroup takes 4.2 us for its keys and 1.33 us a row, one workgroup per compute unit at a time: the count
// with the shortest rounds. Against the row-at-a-time kernel, including ~12 us of host time a call (us): 2048 x 16384 417
// / 786, 256 x 16384 56 / 72, 64 x 16384 18 / 25, 16 x 65536 18 / 26, 64 x 4096 12 / 15, 2048 x 1024 32 / 76.
inline int flat_rows(int M, int N) {
  if (M < 8 || N > (1 << 28)) return 0;                     // (32-bit byte offsets in a row)
  const long long tiles = (N + idx::FL_KEYS - 1) / idx::FL_KEYS;
  int best = 0;
  double cost = 0;
  for (int rw = 64; rw >= 2; rw /= 2) {
    const long long wgs = tiles * ((M + rw - 1) / rw);
    const double c = (double)((wgs + lg_cus() - 1) / lg_cus()) * (4.2 + 1.33 * rw);
    if (!best || c < cost) { best = rw; cost = c; }
  }
  return best;
}

// Workspace bytes of a row by its route: none up to BK_COLS columns, the chunks' lists up to GMAX chunks, the radix state
static int topk_chunks_of(int Lc) { return (Lc + idx::BK_COLS - 1) / idx::BK_COLS; }
static long long topk_ws_row(int Lc) {
  if (Lc <= idx::BK_COLS) return 0;
  return topk_chunks_of(Lc) <= idx::BkWs::GMAX ? idx::BkWs::row_bytes(topk_chunks_of(Lc)) : idx::topk_ws_layout(Lc).row_bytes;
}

extern "C" {

static int logits_row(const void* q, long long q_st, long long q_sh, const float* w, long long w_st,
                      const void* store, long long R_local, int rows_per_block, long long block_stride,
                      const int* block_table, long long bt_st, int block_size, const int* req, const int* ctx,
                      int rows, int H, int D, int Lc, int P, int rank, int noinf, void* out, long long out_st,
                      int out_dtype, void* stream, int all) {
  if (rows < 0 || Lc < 0 || P <= 0 || rank < 0 || rank >= P || block_size <= 0 || rows_per_block <= 0) return SPMLA_EARG;
  if (out_dtype != 0 && out_dtype != 1) return SPMLA_EARG;
  if (rows == 0 || Lc == 0) return SPMLA_OK;
  if (H != 64 || D != 128) return SPMLA_ELIMIT;
  if (R_local < 0 || R_local > (long long)INT_MAX / P) return SPMLA_ELIMIT;   // 32-bit row arithmetic
  if (!q || !w || !store || !block_table || !req || !ctx || !out) return SPMLA_EARG;
  if (((uintptr_t)q & 15) || (q_st & 7) || (q_sh & 7) || ((uintptr_t)store & 3) || (block_stride & 3))
    return SPMLA_EALIGN;
  idx::LogitParams p{};
  p.q = (const uint16_t*)q; p.q_st = q_st; p.q_sh = q_sh; p.w = w; p.w_st = w_st;
  p.store = (const uint8_t*)store; p.R_local = R_local; p.rpb = rows_per_block; p.blk_stride = block_stride;
  p.bt = block_table; p.bt_st = bt_st; p.bs = block_size; p.req = req; p.ctx = ctx;
  p.rows = rows; p.Lc = Lc; p.P = P; p.rank = rank; p.noinf = noinf; p.out = out; p.out_st = out_st;
  auto log2_or = [](long long v) { return (v & (v - 1)) == 0 ? __builtin_ctzll((unsigned long long)v) : -1; };
  p.bs_sh = log2_or(block_size); p.rpb_sh = log2_or(rows_per_block); p.p_sh = log2_or(P);
  p.lim = R_local * P;
  p.clamp = 1;
  p.lo = nullptr; p.kscale = nullptr; p.k_st = 0;
  const dim3 grid = lg_grid(rows, Lc, p.tpg);
  p.all = all;
  const bool pow2 = p.bs_sh >= 0 && p.rpb_sh >= 0 && p.p_sh >= 0;
  if (out_dtype == 1) {
    if (pow2) hipLaunchKernelGGL((idx::logits_kernel<true, idx::LY_ROW, true>), grid, dim3(idx::LG_NWV * 64), 0, (hipStream_t)stream, p);
    else hipLaunchKernelGGL((idx::logits_kernel<false, idx::LY_ROW, true>), grid, dim3(idx::LG_NWV * 64), 0, (hipStream_t)stream, p);
  } else {
    if (pow2) hipLaunchKernelGGL((idx::logits_kernel<true, idx::LY_ROW>), grid, dim3(idx::LG_NWV * 64), 0, (hipStream_t)stream, p);
    else hipLaunchKernelGGL((idx::logits_kernel<false, idx::LY_ROW>), grid, dim3(idx::LG_NWV * 64), 0, (hipStream_t)stream, p);
  }
  return (int)hipGetLastError();
}

int spmla_index_logits(const void* q, long long q_st, long long q_sh, const float* w, long long w_st,
                       const void* store, long long R_local, int rows_per_block, long long block_stride,
                       const int* block_table, long long bt_st, int block_size, const int* req, const int* ctx,
                       int rows, int H, int D, int Lc, int P, int rank, int noinf, void* out, long long out_st,
                       int out_dtype, void* stream) {
  return logits_row(q, q_st, q_sh, w, w_st, store, R_local, rows_per_block, block_stride, block_table, bt_st,
                    block_size, req, ctx, rows, H, D, Lc, P, rank, noinf, out, out_st, out_dtype, stream, 0);
}

int spmla_index_logits_hist(const void* q, long long q_st, long long q_sh, const float* w, long long w_st,
                            const void* store, long long R_local, int rows_per_block, long long block_stride,
                            const int* block_table, long long bt_st, int block_size, const int* req, const int* ctx,
                            int rows, int H, int D, int Lc, int noinf, void* out, long long out_st, int out_dtype,
                            void* topk_ws, long long ws_bytes, int K, void* stream) {
  if (rows < 0 || Lc < 0 || K <= 0 || (out_dtype != 0 && out_dtype != 1)) return SPMLA_EARG;
  if (K > idx::TK_KMAX) return SPMLA_ELIMIT;
  if (rows == 0 || Lc == 0) return SPMLA_OK;
  const idx::TopkWs tw = idx::topk_ws_layout(Lc);
  if (!topk_ws || ((uintptr_t)topk_ws & 15) || ws_bytes < rows * topk_ws_row(Lc)) return SPMLA_EARG;
  if (tw.CL >= 65536) return SPMLA_ELIMIT;                  // (kept from 16-bit histogram counts, as the workspace check)
  return logits_row(q, q_st, q_sh, w, w_st, store, R_local, rows_per_block, block_stride, block_table, bt_st,
                    block_size, req, ctx, rows, H, D, Lc, 1, 0, noinf, out, out_st, out_dtype, stream, 1);
}

// per, tail: see LogitParams
static int paged_launch(const void* q, long long q_st, long long q_sh, const float* w, long long w_st,
                        const void* cache, long long num_blocks, int block_size, long long block_stride,
                        const int* block_table, long long bt_st, const int* req, const int* ctx, int per, int tail,
                        int rows, int H, int D, int Lc, int noinf, float* out, long long out_st, void* stream) {
  if (rows < 0 || Lc < 0 || block_size <= 0 || (block_size & 15) || num_blocks < 0) return SPMLA_EARG;
  if (rows == 0 || Lc == 0) return SPMLA_OK;
  if (H != 64 || D != 128) return SPMLA_ELIMIT;
  if (num_blocks > (long long)INT_MAX / block_size) return SPMLA_ELIMIT;
  if (!q || !w || !cache || !block_table || !(req || per) || !ctx || !out) return SPMLA_EARG;
  if (((uintptr_t)q & 15) || (q_st & 7) || (q_sh & 7) || ((uintptr_t)cache & 3) || (block_stride & 3) ||
      block_stride < (long long)block_size * 132)
    return SPMLA_EALIGN;
  idx::LogitParams p{};
  p.q = (const uint16_t*)q; p.q_st = q_st; p.q_sh = q_sh; p.w = w; p.w_st = w_st;
  p.store = (const uint8_t*)cache; p.R_local = num_blocks * block_size; p.rpb = block_size;
  p.blk_stride = block_stride; p.bt = block_table; p.bt_st = bt_st; p.bs = block_size; p.req = req; p.ctx = ctx;
  p.per = per; p.tail = tail;
  p.rows = rows; p.Lc = Lc; p.P = 1; p.rank = 0; p.noinf = noinf; p.out = out; p.out_st = out_st;
  auto log2_or = [](long long v) { return (v & (v - 1)) == 0 ? __builtin_ctzll((unsigned long long)v) : -1; };
  p.bs_sh = log2_or(block_size); p.rpb_sh = p.bs_sh; p.p_sh = 0;
  p.lim = p.R_local;
  p.clamp = 0;
  p.lo = nullptr; p.kscale = nullptr; p.k_st = 0;
  const dim3 grid = lg_grid(rows, Lc, p.tpg);
  if (p.bs_sh >= 0)
    hipLaunchKernelGGL((idx::logits_kernel<true, idx::LY_SHUF>), grid, dim3(idx::LG_NWV * 64), 0, (hipStream_t)stream, p);
  else
    hipLaunchKernelGGL((idx::logits_kernel<false, idx::LY_SHUF>), grid, dim3(idx::LG_NWV * 64), 0, (hipStream_t)stream, p);
  return (int)hipGetLastError();
}

int spmla_paged_mqa_logits(const void* q, long long q_st, long long q_sh, const float* w, long long w_st,
                           const void* cache, long long num_blocks, int block_size, long long block_stride,
                           const int* block_table, long long bt_st, const int* req, const int* ctx, int rows, int H,
                           int D, int Lc, int noinf, float* out, long long out_st, void* stream) {
  return paged_launch(q, q_st, q_sh, w, w_st, cache, num_blocks, block_size, block_stride, block_table, bt_st, req, ctx,
                      0, 0, rows, H, D, Lc, noinf, out, out_st, stream);
}

int spmla_paged_mqa_logits_seq(const void* q, long long q_st, long long q_sh, const float* w, long long w_st,
                               const void* cache, long long num_blocks, int block_size, long long block_stride,
                               const int* block_table, long long bt_st, const int* seq_lens, int per_row, int next_n,
                               int rows, int H, int D, int Lc, int noinf, float* out, long long out_st, void* stream) {
  if (next_n <= 0) return SPMLA_EARG;
  return paged_launch(q, q_st, q_sh, w, w_st, cache, num_blocks, block_size, block_stride, block_table, bt_st, nullptr,
                      seq_lens, next_n, per_row == 0, rows, H, D, Lc, noinf, out, out_st, stream);
}

int spmla_mqa_logits(const void* q, long long q_st, long long q_sh, const float* w, long long w_st, const void* k,
                     long long k_st, const float* kscale, int N, const int* ks, const int* ke, int M, int H, int D,
                     float* out, long long out_st, void* stream) {
  if (M < 0 || N < 0) return SPMLA_EARG;
  if (M == 0 || N == 0) return SPMLA_OK;
  if (H != 64 || D != 128) return SPMLA_ELIMIT;
  if (!q || !w || !k || !kscale || !ks || !ke || !out) return SPMLA_EARG;
  if (((uintptr_t)q & 15) || (q_st & 7) || (q_sh & 7) || ((uintptr_t)k & 3) || (k_st & 3) || k_st < 128 ||
      ((uintptr_t)kscale & 3))
    return SPMLA_EALIGN;
  if (const int rw = flat_rows(M, N)) {
    const idx::FlatParams p{(const uint16_t*)q, q_st, q_sh, w, w_st, (const uint8_t*)k, k_st, kscale, ks, ke, M, N, rw,
                            out, out_st};
    const long long n = (long long)((N + idx::FL_KEYS - 1) / idx::FL_KEYS) * ((M + rw - 1) / rw);
    hipLaunchKernelGGL(idx::flat_logits_kernel, dim3((unsigned)((n + 7) / 8 * 8)), dim3(idx::FL_NWV * 64), 0,
                       (hipStream_t)stream, p);
    return (int)hipGetLastError();
  }
  idx::LogitParams p{};
  p.q = (const uint16_t*)q; p.q_st = q_st; p.q_sh = q_sh; p.w = w; p.w_st = w_st;
  p.store = (const uint8_t*)k; p.R_local = N; p.rpb = 1; p.blk_stride = 0;
  p.bt = nullptr; p.bt_st = 0; p.bs = 1; p.req = nullptr; p.ctx = ke;
  p.rows = M; p.Lc = N; p.P = 1; p.rank = 0; p.noinf = 0; p.out = out; p.out_st = out_st;
  p.bs_sh = p.rpb_sh = p.p_sh = 0;
  p.lim = N;
  p.clamp = 0;
  p.lo = ks; p.kscale = kscale; p.k_st = k_st;
  const dim3 grid = lg_grid(M, N, p.tpg);
  hipLaunchKernelGGL((idx::logits_kernel<true, idx::LY_FLAT>), grid, dim3(idx::LG_NWV * 64), 0, (hipStream_t)stream, p);
  return (int)hipGetLastError();
}

int spmla_topk(const void* logits, long long lg_st, const int* ctx, int rows, int Lc, int K, int* out,
               long long out_st, int dtype, void* stream) {
  if (rows < 0 || Lc < 0 || K <= 0 || (dtype != 0 && dtype != 1)) return SPMLA_EARG;
  if (K > idx::TK_KMAX) return SPMLA_ELIMIT;
  if (rows == 0) return SPMLA_OK;
  if (!logits || !ctx || !out) return SPMLA_EARG;
  idx::TopkParams p;
  p.lg = logits; p.lg_st = lg_st; p.ctx = ctx; p.rows = rows; p.Lc = Lc; p.K = K; p.out = out; p.out_st = out_st;
  if (Lc <= idx::BK_COLS) idx::topk_rows(p, dtype, (hipStream_t)stream);
  else if (dtype == 1) hipLaunchKernelGGL(idx::topk_kernel<true>, dim3(rows), dim3(idx::TK_NT), 0, (hipStream_t)stream, p);
  else hipLaunchKernelGGL(idx::topk_kernel<false>, dim3(rows), dim3(idx::TK_NT), 0, (hipStream_t)stream, p);
  return (int)hipGetLastError();
}

// (never 0 for a row, so that a buffer of this size has an address: 64 bytes more a row)
long long spmla_topk_ws_bytes(int rows, int Lc, int K) {
  if (rows < 0 || Lc < 0 || K <= 0) return 0;
  return (long long)rows * (topk_ws_row(Lc) + 64);
}

int spmla_topk_ws(const void* logits, long long lg_st, const int* ctx, int rows, int Lc, int K, int* out,
                  long long out_st, void* ws, long long ws_bytes, int dtype, void* stream) {
  if (rows < 0 || Lc < 0 || K <= 0 || (dtype != 0 && dtype != 1)) return SPMLA_EARG;
  if (K > idx::TK_KMAX) return SPMLA_ELIMIT;
  if (rows == 0) return SPMLA_OK;
  if (!logits || !ctx || !out || !ws) return SPMLA_EARG;
  if (((uintptr_t)ws & 15) || ws_bytes < rows * topk_ws_row(Lc)) return SPMLA_EARG;
  if (Lc <= idx::BK_COLS) {                         // a row fits one workgroup's registers
    idx::topk_rows(idx::TopkParams{logits, lg_st, ctx, rows, Lc, K, out, out_st}, dtype, (hipStream_t)stream);
    return (int)hipGetLastError();
  }
  const int G = topk_chunks_of(Lc);
  if (G <= idx::BkWs::GMAX) {                       // the chunks' lists fit one workgroup's registers
    idx::topk_chunks(idx::TopkChunkParams{logits, lg_st, ctx, rows, Lc, K, out, out_st, (uint8_t*)ws, topk_ws_row(Lc), G,
                                          ((Lc + G - 1) / G + 1023) / 1024 * 1024},
                     dtype, (hipStream_t)stream);
    return (int)hipGetLastError();
  }
  idx::TopkWsParams p;
  p.lg = logits; p.lg_st = lg_st; p.ctx = ctx; p.rows = rows; p.Lc = Lc; p.K = K; p.out = out; p.out_st = out_st;
  p.ws = (uint8_t*)ws; p.w = idx::topk_ws_layout(Lc);
  if (dtype == 1) idx::topk_ws_passes<true>(p, (hipStream_t)stream);
  else idx::topk_ws_passes<false>(p, (hipStream_t)stream);
  return (int)hipGetLastError();
}

int spmla_topk_ws_prehist(const void* logits, long long lg_st, const int* ctx, int rows, int Lc, int K, int* out,
                          long long out_st, void* ws, long long ws_bytes, int dtype, void* stream) {
  return spmla_topk_ws(logits, lg_st, ctx, rows, Lc, K, out, out_st, ws, ws_bytes, dtype, stream);
}

long long spmla_topk_scratch_bytes(void) { return idx::TOPK_SCRATCH_BYTES; }

int spmla_topk_scratch(const void* logits, long long lg_st, const int* ctx, int rows, int Lc, int K, int* out,
                       long long out_st, int dtype, void* stream) {
  if (rows < 0 || Lc < 0 || K <= 0 || (dtype != 0 && dtype != 1)) return SPMLA_EARG;
  if (K > idx::TK_KMAX) return SPMLA_ELIMIT;
  if (rows == 0) return SPMLA_OK;
  if (!logits || !ctx || !out) return SPMLA_EARG;
  const long long radix = (long long)rows * idx::topk_ws_layout(Lc).row_bytes, need = rows * topk_ws_row(Lc);
  if (max(radix, need) > idx::TOPK_SCRATCH_BYTES) return SPMLA_ELIMIT;   // (as long as every row took the radix state)
  void* ws = nullptr;
  const int rc = scratch_ptr(&ws);
  if (rc != SPMLA_OK) return rc;
  return spmla_topk_ws(logits, lg_st, ctx, rows, Lc, K, out, out_st, ws, need, dtype, stream);
}

int spmla_topk_local(const void* logits, long long lg_st, const int* ctx, int rows, int rank, int P, int Lc, int kl,
                     float* pk, int dtype, void* stream) {
  if (rows < 0 || Lc < 0 || kl <= 0 || P <= 0 || rank < 0 || rank >= P || (dtype != 0 && dtype != 1))
    return SPMLA_EARG;
  if (kl > idx::TK_KMAX) return SPMLA_ELIMIT;
  if (rows == 0) return SPMLA_OK;
  if (!logits || !ctx || !pk) return SPMLA_EARG;
  idx::LocalParams p;
  p.lg = logits; p.lg_st = lg_st; p.ctx = ctx; p.rows = rows; p.rank = rank; p.P = P; p.Lc = Lc; p.kl = kl; p.pk = pk;
  if (dtype == 1) hipLaunchKernelGGL(idx::topk_local_kernel<true>, dim3(rows), dim3(idx::TK_NT), 0, (hipStream_t)stream, p);
  else hipLaunchKernelGGL(idx::topk_local_kernel<false>, dim3(rows), dim3(idx::TK_NT), 0, (hipStream_t)stream, p);
  return (int)hipGetLastError();
}

int spmla_topk_merge(const float* allp, int n, int P, int kl, int kk, int topk_tokens, int* out, long long out_st,
                     void* stream) {
  if (n < 0 || P <= 0 || kl <= 0 || kk < 0 || kk > P * kl || topk_tokens < kk) return SPMLA_EARG;
  if (kk > idx::TK_KMAX) return SPMLA_ELIMIT;
  if (n == 0 || topk_tokens == 0) return SPMLA_OK;
  if (!allp || !out) return SPMLA_EARG;
  idx::MergeParams p;
  p.allp = allp; p.n = n; p.P = P; p.kl = kl; p.kk = kk; p.topk_tokens = topk_tokens; p.out = out; p.out_st = out_st;
  hipLaunchKernelGGL(idx::topk_merge_kernel, dim3(n), dim3(idx::TK_NT), 0, (hipStream_t)stream, p);
  return (int)hipGetLastError();
}

int spmla_rows_from_topk(const int* topk, long long tk_st, const int* req, const int* block_table, long long bt_st,
                         int bt_cols, int block_size, long long stride_rows, int T, int K, int* rows, long long r_st,
                         int* counts, void* stream) {
  if (T < 0 || K < 0 || block_size <= 0 || bt_cols < 0) return SPMLA_EARG;
  if (T == 0 || K == 0) return SPMLA_OK;
  if (!topk || !req || !block_table || !rows) return SPMLA_EARG;
  if (T > 65535) return SPMLA_ELIMIT;
  if (counts)   // a fill kernel, not hipMemsetAsync: safe inside captured graphs
    hipLaunchKernelGGL(idx::zero_i32, dim3((T + 255) / 256), dim3(256), 0, (hipStream_t)stream, counts, T);
  dim3 grid((K + 255) / 256, T);
  hipLaunchKernelGGL(idx::rows_kernel, grid, dim3(256), 0, (hipStream_t)stream, topk, tk_st, req, block_table, bt_st,
                     bt_cols, block_size, stride_rows, T, K, rows, r_st, counts);
  return (int)hipGetLastError();
}

}  // extern "C"
