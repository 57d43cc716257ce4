// KV-cache write (quantize + pack) and indexer-key write.
//
// Row656 (per token): per 128 latent values s = max(amax / 448, 1e-12) (fp32, correctly rounded),
//   code = e4m3fn_rne(x / s); layout [512 codes | 4 x fp32 s | 64 x bf16 rope (bit copy)].
//   Closed form of the reference's per-128 FP8 activation quantizer: dotsnote/training/finetune/student.py:80-87;
//   656-byte layout: dotsnote/engine/vllm_patch/vllm/v1/hisparse/runtime.py:35-36.
// Row576 (the reference's deployed offload row, dotsnote/engine/arcstats_pkg/arcstats/sparse_offload.py:252-270):
//   code = e4m3fn_rne(clamp(x * inv_scale, -448, 448)) for the 512 latent and the 64 rope values.
// Row400 (the reference's compact e2m2b32 host row, dotsnote/engine/arcstats_pkg/arcstats/offload_rowfmt.py:81-129,
//   torch statement ref_quant / ref_pack :336-388): x = clamp(v * inv_scale, +-448); per 32 values
//   k = smallest integer with 2^k >= amax / 7 (fp32 amax / 7; zero or subnormal quotients give k = -126), y = |x| 2^-k,
//   mag = floor(4y + 0.5) for y < 1, else ((e2 + 1) << 2) + floor(y / 2^(e2 - 2) + 0.5) - 4 with e2 = [y >= 2] +
//   [y >= 4], capped at 15; the sign bit is set for x < 0 with mag > 0. Rope as in Row576.
// Index key (dotsnote/engine/arcstats_pkg/arcstats/shard_indexer.py:42-60): s = max(amax, 1e-4) / 448 (optionally
//   rounded up to a power of two, UE8M0), code = e4m3fn_rne(k / s); 132-byte row [128 codes | fp32 s].
//
// One wave per token, 4 tokens per 256-thread block; tokens with slot < 0 (padding), slot >= R or another rank's slot are
// skipped and their values are not read (a padded batch may hold fewer rows of values than slots). The encoding bounded
// these kernels (a branchy software encoder and one division per value): finite groups now use the hardware's conversion,
// which equals e4m3_rne on every fp32 value except the sign of NaNs (all 2^32 compared), and one reciprocal per group.
// 8192 tokens: rows 8.2 -> 4.9 us, index keys 5.0 -> 3.8; 8 tokens: 4.1 -> 2.6 and 2.9 -> 2.7.
#include "spmla_common.h"

namespace spmla {
namespace wr {

__device__ inline float wave_max16(float v) {   // max over aligned groups of 16 lanes
  v = fmaxf(v, __shfl_xor(v, 1, 64));
  v = fmaxf(v, __shfl_xor(v, 2, 64));
  v = fmaxf(v, __shfl_xor(v, 4, 64));
  v = fmaxf(v, __shfl_xor(v, 8, 64));
  return v;
}

// e2m2 magnitude index of y = |x| 2^-k >= 0 (offload_rowfmt.py:93-101 with M = 2). The products are exact
// (powers of two), so the one rounding is the fp32 add of 0.5, as in the reference.
__device__ inline uint32_t e2m2_mag(float y) {
  if (y < 1.0f) return (uint32_t)floorf(y * 4.0f + 0.5f);       // 0 .. 4
  const int e2 = (y >= 2.0f) + (y >= 4.0f);
  const float inv_stp = u2f((uint32_t)(127 + 2 - e2) << 23);     // 2^(2 - e2)
  const uint32_t nrm = ((uint32_t)(e2 + 1) << 2) + (uint32_t)floorf(y * inv_stp + 0.5f) - 4u;
  return nrm < 15u ? nrm : 15u;
}

__device__ inline uint32_t e4m3x4(float a, float b, float c, float d) {    // no NaN
  const int w = __builtin_amdgcn_cvt_pk_fp8_f32(a, b, 0, false);
  return (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(c, d, w, true);
}
// x / s correctly rounded, r = 1 / s correctly rounded, x and s finite (Markstein's division step: the remainder is exact
// unless x is below 2^-78, where the quotient by s >= 1e-12 encodes to zero either way); the sign is x's
__device__ inline float quotient(float x, float s, float r) {
  const float q = x * r;
  return copysignf(__builtin_fmaf(__builtin_fmaf(-q, s, x), r, q), x);
}
// (slot / n, slot % n) for 0 <= slot: sh = log2 n for a power of two, else -1
__device__ inline void div_slot(long long slot, int n, int sh, long long& blk, int& off) {
  if (sh >= 0) { blk = slot >> sh; off = (int)(slot & (n - 1)); }
  else if ((slot >> 31) == 0) { blk = (uint32_t)slot / (uint32_t)n; off = (int)((uint32_t)slot % (uint32_t)n); }
  else { blk = slot / n; off = (int)(slot % n); }
}
inline int log2_or(int n) { return n > 0 && (n & (n - 1)) == 0 ? __builtin_ctz((unsigned)n) : -1; }

struct WriteParams {
  const uint16_t* kv; long long kv_st;      // kv_c_normed[n][512] bf16
  const uint16_t* pe; long long pe_st;      // k_pe[n][64] bf16
  const long long* slots; int n;
  uint8_t* cache; long long R; int bs, sh; long long blk_stride;   // row of slot: (slot / bs) * blk_stride + (slot % bs) * row
  int fmt;                                  // 0: Row656, 1: Row576, 2: Row400
  float inv_scale;                          // Row576 / Row400
};

__global__ void __launch_bounds__(256) cache_write_kernel(WriteParams p) {
  const int tok = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * 4 + (threadIdx.x >> 6)));
  const int lane = threadIdx.x & 63;
  if (tok >= p.n) return;
  const long long slot = p.slots[tok];
  if (slot < 0 || slot >= p.R) return;
  const u32x4 raw = *(const u32x4*)(p.kv + (long long)tok * p.kv_st + lane * 8);
  const uint2 rope = *(const uint2*)(p.pe + (long long)tok * p.pe_st + (lane & 15) * 4);
  const int rowb = p.fmt == 0 ? ROW656 : (p.fmt == 1 ? ROW576 : ROW400);
  long long blk;
  int off;
  div_slot(slot, p.bs, p.sh, blk, off);
  uint8_t* row = p.cache + blk * p.blk_stride + (long long)off * rowb;
  float x[8];
#pragma unroll
  for (int e = 0; e < 4; ++e) { x[2 * e] = u2f(raw[e] << 16); x[2 * e + 1] = u2f(raw[e] & 0xffff0000u); }
  uint32_t lo = 0, hi = 0;
  auto clamped = [&](float v) -> float { return fminf(fmaxf(v * p.inv_scale, -448.f), 448.f); };   // (a NaN becomes -448)
  if (p.fmt == 0) {
    float am = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) am = fmaxf(am, fabsf(x[e]));
    am = wave_max16(am);
    const float s = fmaxf(am / 448.0f, 1e-12f);
    uint32_t mag = 0;                  // largest magnitude as an integer: infinities and NaNs lie above the finite ones
#pragma unroll
    for (int e = 0; e < 8; ++e) mag = max(mag, f2u(x[e]) & 0x7fffffffu);
    if (__builtin_expect(__ballot(mag >= 0x7f800000u) == 0ull, 1)) {
      const float r = 1.0f / s;
      float y[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) y[e] = quotient(x[e], s, r);
      lo = e4m3x4(y[0], y[1], y[2], y[3]);
      hi = e4m3x4(y[4], y[5], y[6], y[7]);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        lo |= (uint32_t)e4m3_rne(x[e] / s) << (8 * e);
        hi |= (uint32_t)e4m3_rne(x[4 + e] / s) << (8 * e);
      }
    }
    *(uint2*)(row + lane * 8) = make_uint2(lo, hi);
    if ((lane & 15) == 0) *(float*)(row + SC_OFF + (lane >> 4) * 4) = s;
    if (lane < 16) *(uint2*)(row + ROPE_OFF + lane * 8) = rope;   // 64 bf16 = 16 x 8 bytes
  } else if (p.fmt == 2) {
    // Row400: lane l holds values 8l .. 8l + 7; the 4 lanes 4b .. 4b + 3 form exponent block b
    float am = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      x[e] = fminf(fmaxf(x[e] * p.inv_scale, -448.f), 448.f);
      am = fmaxf(am, fabsf(x[e]));
    }
    am = fmaxf(am, __shfl_xor(am, 1, 64));
    am = fmaxf(am, __shfl_xor(am, 2, 64));
    const uint32_t rb = f2u(am / 7.0f);
    const int ex = (int)((rb >> 23) & 255u) - 127;
    int k = ex + ((rb & 0x7fffffu) != 0u);
    k = ex < -126 ? -126 : (k < 127 ? k : 127);
    const float inv = u2f((uint32_t)(127 - k) << 23);                // 2^-k
    uint32_t nib = 0, sgn = 0;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const uint32_t mag = e2m2_mag(fabsf(x[e]) * inv);
      nib |= mag << (4 * e);
      sgn |= (x[e] < 0.f && mag > 0u ? 1u : 0u) << e;
    }
    *(uint32_t*)(row + 4 * lane) = nib;
    row[R4_SIGN + lane] = (uint8_t)sgn;
    if ((lane & 3) == 0) row[R4_K + (lane >> 2)] = (uint8_t)(int8_t)k;
    if (lane < 16) {   // rope: 64 values -> 64 e4m3 codes, 4 per lane
      const uint32_t c = e4m3x4(clamped(u2f(rope.x << 16)), clamped(u2f(rope.x & 0xffff0000u)), clamped(u2f(rope.y << 16)),
                                clamped(u2f(rope.y & 0xffff0000u)));
      *(uint32_t*)(row + R4_ROPE + lane * 4) = c;
    }
  } else {
    lo = e4m3x4(clamped(x[0]), clamped(x[1]), clamped(x[2]), clamped(x[3]));
    hi = e4m3x4(clamped(x[4]), clamped(x[5]), clamped(x[6]), clamped(x[7]));
    *(uint2*)(row + lane * 8) = make_uint2(lo, hi);
    if (lane < 16) {   // rope: 64 values -> 64 codes, 4 per lane
      const uint32_t c = e4m3x4(clamped(u2f(rope.x << 16)), clamped(u2f(rope.x & 0xffff0000u)), clamped(u2f(rope.y << 16)),
                                clamped(u2f(rope.y & 0xffff0000u)));
      *(uint32_t*)(row + D_LAT + lane * 4) = c;
    }
  }
}

struct KeyParams {
  const uint16_t* k; long long k_st;       // k[n][128] bf16
  const long long* slots; int n;
  uint8_t* store; long long R_local;       // local rows
  int P, rank, rpb, sh; long long blk_stride;  // row r at (r / rpb) * blk_stride + (r % rpb) * 132
  int ue8m0;
  int shuf;                                // vLLM's paged SHUFFLE layout (P = 1): key t of a block of rpb keys has
                                           // its 16-byte chunk c at (t / 16) * 2048 + (t % 16) * 16 + 256 c and its
                                           // scale at rpb * 128 + 4 t
};

__global__ void __launch_bounds__(256) key_write_kernel(KeyParams p) {
  const int tok = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * 4 + (threadIdx.x >> 6)));
  const int lane = threadIdx.x & 63;
  if (tok >= p.n) return;
  const long long slot = p.slots[tok];
  if (slot < 0 || (p.P > 1 && slot % p.P != p.rank)) return;
  const long long r = p.P > 1 ? slot / p.P : slot;
  if (r >= p.R_local) return;
  const uint32_t raw = *(const uint32_t*)(p.k + (long long)tok * p.k_st + lane * 2);
  long long b;
  int t;
  div_slot(r, p.rpb, p.sh, b, t);
  uint8_t* blk = p.store + b * p.blk_stride;
  uint8_t* row = blk + t * 132;                                        // 132-byte rows
  uint8_t* code = p.shuf ? blk + (t >> 4) * 2048 + (t & 15) * 16 + (lane >> 3) * 256 + (lane & 7) * 2
                         : row + lane * 2;
  float* scale = (float*)(p.shuf ? blk + p.rpb * 128 + 4 * t : row + 128);
  const float x0 = u2f(raw << 16), x1 = u2f(raw & 0xffff0000u);
  float am = fmaxf(fabsf(x0), fabsf(x1));
  am = wave_max16(am);
  am = fmaxf(am, __shfl_xor(am, 16, 64));
  am = fmaxf(am, __shfl_xor(am, 32, 64));
  float s = fmaxf(am, 1e-4f) / 448.0f;
  if (p.ue8m0) {   // next power of two >= s (s is positive and normal here)
    uint32_t u = f2u(s);
    if (u & 0x7fffffu) u = (u & 0xff800000u) + 0x800000u;
    s = u2f(u);
  }
  uint32_t c;
  if (__builtin_expect(__ballot(max(f2u(x0) & 0x7fffffffu, f2u(x1) & 0x7fffffffu) >= 0x7f800000u) == 0ull, 1)) {
    const float rs = 1.0f / s;
    c = (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(quotient(x0, s, rs), quotient(x1, s, rs), 0, false);
  } else {
    c = (uint32_t)e4m3_rne(x0 / s) | ((uint32_t)e4m3_rne(x1 / s) << 8);
  }
  *(uint16_t*)code = (uint16_t)c;
  if (lane == 0) *scale = s;
}

}  // namespace wr
}  // namespace spmla

using namespace spmla;

extern "C" {

int spmla_cache_write(const void* kv_c, long long kv_st, const void* k_pe, long long pe_st, const long long* slots,
                      int n, void* cache, long long R, int block_size, long long block_stride, int fmt,
                      float kv_scale, void* stream) {
  if (n < 0 || R < 0 || fmt < 0 || fmt > 2 || block_size <= 0) return SPMLA_EARG;
  if (n == 0) return SPMLA_OK;
  if (!kv_c || !k_pe || !slots || !cache) return SPMLA_EARG;
  if (((uintptr_t)kv_c & 15) || (kv_st & 7) || ((uintptr_t)k_pe & 7) || (pe_st & 3)) return SPMLA_EALIGN;
  const int rowb = fmt == 0 ? ROW656 : (fmt == 1 ? ROW576 : ROW400);
  if (((uintptr_t)cache & 7) || (block_stride & 7) || block_stride < (long long)block_size * rowb) return SPMLA_EALIGN;
  if (fmt != 0 && !(kv_scale > 0.f)) return SPMLA_EARG;
  wr::WriteParams p;
  p.kv = (const uint16_t*)kv_c; p.kv_st = kv_st; p.pe = (const uint16_t*)k_pe; p.pe_st = pe_st;
  p.slots = slots; p.n = n; p.cache = (uint8_t*)cache; p.R = R; p.bs = block_size; p.sh = wr::log2_or(block_size); p.blk_stride = block_stride;
  p.fmt = fmt; p.inv_scale = fmt != 0 ? 1.0f / kv_scale : 1.0f;
  hipLaunchKernelGGL(wr::cache_write_kernel, dim3((n + 3) / 4), dim3(256), 0, (hipStream_t)stream, p);
  return (int)hipGetLastError();
}

int spmla_index_key_write(const void* k, long long k_st, const long long* slots, int n, void* store,
                          long long R_local, int P, int rank, int rows_per_block, long long block_stride, int ue8m0,
                          void* stream) {
  if (n < 0 || P <= 0 || rank < 0 || rank >= P || rows_per_block <= 0 || R_local < 0) return SPMLA_EARG;
  if (n == 0) return SPMLA_OK;
  if (!k || !slots || !store) return SPMLA_EARG;
  if (((uintptr_t)k & 3) || (k_st & 1) || ((uintptr_t)store & 3) || (block_stride & 3) ||
      block_stride < (long long)rows_per_block * 132)
    return SPMLA_EALIGN;
  wr::KeyParams p;
  p.k = (const uint16_t*)k; p.k_st = k_st; p.slots = slots; p.n = n; p.store = (uint8_t*)store;
  p.R_local = R_local; p.P = P; p.rank = rank; p.rpb = rows_per_block; p.sh = wr::log2_or(rows_per_block); p.blk_stride = block_stride; p.ue8m0 = ue8m0;
  p.shuf = 0;
  hipLaunchKernelGGL(wr::key_write_kernel, dim3((n + 3) / 4), dim3(256), 0, (hipStream_t)stream, p);
  return (int)hipGetLastError();
}

int spmla_index_key_write_shuffle(const void* k, long long k_st, const long long* slots, int n, void* cache,
                                  long long num_blocks, int block_size, long long block_stride, int ue8m0,
                                  void* stream) {
  if (n < 0 || num_blocks < 0 || block_size <= 0 || (block_size & 15)) return SPMLA_EARG;
  if (n == 0) return SPMLA_OK;
  if (!k || !slots || !cache) return SPMLA_EARG;
  if (((uintptr_t)k & 3) || (k_st & 1) || ((uintptr_t)cache & 3) || (block_stride & 3) ||
      block_stride < (long long)block_size * 132)
    return SPMLA_EALIGN;
  wr::KeyParams p;
  p.k = (const uint16_t*)k; p.k_st = k_st; p.slots = slots; p.n = n; p.store = (uint8_t*)cache;
  p.R_local = num_blocks * block_size; p.P = 1; p.rank = 0; p.rpb = block_size; p.sh = wr::log2_or(block_size); p.blk_stride = block_stride;
  p.ue8m0 = ue8m0; p.shuf = 1;
  hipLaunchKernelGGL(wr::key_write_kernel, dim3((n + 3) / 4), dim3(256), 0, (hipStream_t)stream, p);
  return (int)hipGetLastError();
}

}  // extern "C"
