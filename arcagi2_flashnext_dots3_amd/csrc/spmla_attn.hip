// Sparse-MLA decode / prefill attention over gathered Row656 KV rows, and the log-sum-exp merge of partials.
//
// Math (reference: dotsnote/kaggle/runtime_dataset/bench_offload_attn2.py:77-93 and
// dotsnote/engine/vllm_patch/vllm/v1/attention/ops/xpu_mla_sparse.py:77-161):
//   row r of token t = idx[t][k] (valid iff 0 <= idx < R); latent_d = e4m3(code_d) * scale[d / 128], rope bf16
//   s[h][k] = sm_scale * kv_scale * (q[h][:512] . latent + q[h][512:] . rope)           (fp32)
//   p = exp2(s * log2e - m), o[h] = kv_scale * sum_k p latent / sum_k p,  lse = ln sum_k exp(s)
//   invalid entries contribute nothing; a token with no valid entry gives o = 0 and lse = -inf.
//
// gfx950 mapping of fwd_kernel (prefill chunks). One workgroup = (token t, group of up to 128 heads, split s of the
// token's rows), 4 waves, one per SIMD. The latent dims are split over the waves: wave w owns scale group w (128 dims) of
// all 128 heads, so that a row's codes are copied, read and converted by one wave only (heads split over the waves, as
// it was before, read and convert every row four times, or hand converted V^T tiles through LDS):
//   * staging: wave w copies the codes of its group, a quarter of the rope and its scale of the tile's 32 rows into LDS
//     rings (3 deep; the rope's 2) with direct global->LDS copies, two tiles ahead; a lane copies from one row only, so
//     a tile costs one row address per lane. Entries that are invalid or past the split's end copy a file-scope zero row;
//   * QK: S^T partials (32 rows x 32 heads, bf16 MFMA 32x32x16, codes converted exactly) of the group for the four head
//     blocks in turn; three go through LDS to the waves that own those heads, in fp32, where they are combined with the
//     rows' fp32 scales (a DPP operand: see fmac8_dpp), so no product of a code and a scale is rounded; each wave adds
//     the rope of its own heads (Row576: a quarter of the rope dims is a ninth MFMA of every partial);
//   * softmax: wave w owns heads 32 w .. 32 w + 31: the C layout puts one head in each lane (16 rows; the other 16 in
//     lane + 32): in-lane plus one cross-half exchange, base 2, lazy rescaling (a head's reference max moves only when a
//     tile exceeds it by more than TAU, so p <= 2^TAU and O is rescaled rarely). P returns through LDS: fp32 (Row656,
//     each wave rounds P' = P * scale(row, group) to f16 itself), f16 (Row576);
//   * PV: f16 MFMA, V^T operands with the 8-bit transposing read straight from the wave's codes; a power-of-two factor
//     2^-eps carried by P' and O keeps P' inside f16's range for any row scale.
// The loop is software-pipelined over the two halves of a step (QK of tile j + 1 with the rounding of P' of tile j; PV of
// tile j with the softmax of tile j + 1), one barrier after each, and written in slices: every MFMA is followed by a
// fence and carries the side work that fits under its 32 cycles. What bounds it is issue: one wave per SIMD (512
// registers) issues about one instruction per 4 cycles (8-byte ones 4.6, scalar ones 8: measured), 620 (Row656) or 480
// per tile, 68 of them MFMAs; matrix cores are busy 39 % (Row656) and 44 % (Row576) of the time, LDS 28 and 26 %. Hence
// addresses that are a register plus immediates, no wait states where none are needed, no scalar work per slice.
// T = 2048, H = 128, K = 2048: Row656 1304 us (896 TFLOP/s), before (heads split over the waves) 1580 us; Row576 1160 us,
// before (head-group kernel) 1440 us; back to back for a second the card lowers its clock: 1400 us against 1545, Row576
// T = 1455 900 us against 1050.
#include <type_traits>

#include "spmla_common.h"
#include "spmla_rules.h"

namespace spmla {
namespace attn {

constexpr int NW = 4;                 // waves per workgroup = head blocks
constexpr int HB = 32;                // heads per wave
constexpr int HGW = NW * HB;          // heads per workgroup
constexpr int TR = 32;                // rows per tile
constexpr int KMAX = 2048;            // rows per (token, split): their ids are staged in LDS
constexpr float TAU = 6.0f;
// LDS map (bytes): a region per wave (so that the own wave's places are one base register plus immediates, and another
// wave's a constant apart), then what the workgroup shares.
constexpr int NRING = 3;                      // depth of the code and scale rings (the rope's is 2)
constexpr int RP_TILE = TR * 128;             // bf16 rope tile [8 chunks][32 rows][16]
template <bool R5>
struct Lds {
  // a ring slot: the codes of the wave's scale group, [16-byte chunk][32 rows][16]; then Row576: 16 bytes of rope per row,
  // Row656: the group's fp32 scales by row (the copy of the upper lanes lands behind them)
  static constexpr int CODE = 8 * TR * 16 + (R5 ? TR * 16 : 64 * 4);
  static constexpr int NQL = R5 ? 9 : 3;                               // query operands in LDS (see q_lds)
  static constexpr int PB = R5 ? 2048 : 4096;                          // P of a head block: f16 operands, or fp32
  static constexpr int S = NRING * CODE;                               // partials [step][4][64 lanes][16]
  static constexpr int P = S + 3 * 4096;
  static constexpr int QR = P + PB;                                    // query rope, [8 chunks][32 heads][16]
  static constexpr int QL = QR + (R5 ? 0 : HB * 128);                  // NQL query operands [64 lanes][16]
  static constexpr int WAVE = QL + NQL * 1024;                         // bytes of a wave's region
  static constexpr int RP = NW * WAVE;
  static constexpr int IDS = RP + (R5 ? 0 : 2 * RP_TILE);              // validated row ids (-1: none), and three tiles of -1
  static constexpr int ST = IDS + (KMAX + 3 * TR) * 4;                 // per head: rescale factors; at the end 1 / l
  static constexpr int FLAG = ST + HGW * 4;                            // per wave: it has factors other than 1
  static constexpr int TOTAL = FLAG + 16;
  static_assert(TOTAL <= 160 * 1024, "LDS budget");
  static_assert(WAVE < 65536, "immediate offsets");
};
constexpr int OROW = 272;                     // output staging: a head's 128 dims in bf16, padded
static_assert(HB * OROW <= Lds<true>::S && HB * OROW <= Lds<false>::S, "a head block of output per wave fits in its rings");

// Source of invalid and padding rows: zero codes, zero scales, zero rope.
__device__ __attribute__((aligned(16))) uint8_t zero_row[ROW656];

// e4m3 pairs -> bf16 / f16 pairs (exact), through the compiler builtins so that the hazard recognizer sees the VALU
// writes. The packed result is bit-cast whole.
__device__ inline uint32_t fp8lo_bf16x2(uint32_t w) {
  return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, 1.0f, false));
}
__device__ inline uint32_t fp8hi_bf16x2(uint32_t w) {
  return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, 1.0f, true));
}
__device__ inline uint32_t fp8lo_f16x2(uint32_t w) {
  return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w, 1.0f, false));
}
__device__ inline uint32_t fp8hi_f16x2(uint32_t w) {
  return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w, 1.0f, true));
}
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
__device__ inline uint32_t pk_bf16(float a, float b) {      // v_cvt_pk_bf16_f32, round to nearest even
  const bf16x2_t v = {(__bf16)a, (__bf16)b};
  return __builtin_bit_cast(uint32_t, v);
}
__device__ inline uint32_t pk_f16(float a, float b) {       // round to nearest even
  const f16x2_t v = {(_Float16)a, (_Float16)b};
  return __builtin_bit_cast(uint32_t, v);
}
// 8 e4m3 codes (two dwords) -> 8 bf16 / f16, exact
__device__ inline bf16x8 codes8_bf16(uint32_t a, uint32_t b) {
  return __builtin_bit_cast(bf16x8, u32x4{fp8lo_bf16x2(a), fp8hi_bf16x2(a), fp8lo_bf16x2(b), fp8hi_bf16x2(b)});
}
__device__ inline f16x8 codes8_f16(uint32_t a, uint32_t b) {
  return __builtin_bit_cast(f16x8, u32x4{fp8lo_f16x2(a), fp8hi_f16x2(a), fp8lo_f16x2(b), fp8hi_f16x2(b)});
}

// The value of lane l ^ 32 (v_permlane32_swap: one VALU op, no LDS round trip).
__device__ inline float half_swap(float x) {
  const uint32_t u = __builtin_bit_cast(uint32_t, x);
  const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return __builtin_bit_cast(float, (__lane_id() & 32) ? r[0] : r[1]);
}

// QK MFMAs with the accumulator in VGPRs. The compiler builtin puts every MFMA result in AGPRs when the function
// uses AGPRs, which here would evict part of the PV accumulator around each QK phase; inline asm pins the QK
// accumulator to VGPRs; the statements are volatile so that they keep their order. Hazards the compiler cannot see inside
// asm are kept off by the order of the slices, not by wait states (each would take an issue slot): an operand comes from
// LDS or was converted a slice or more before (2 wait states after a VALU write), a chain's result is read, and its
// registers written, three or more MFMAs after its last one. Back-to-back MFMAs of one chain have srcC == vdst exactly
// (forwarded). tests/test_attention_hazards.py checks the compiled order.
__device__ inline f32x16 qk_first(bf16x8 a, bf16x8 b) {
  f32x16 d;
  asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, 0" : "=&v"(d) : "v"(a), "v"(b));
  return d;
}
__device__ inline f32x16 qk_next(bf16x8 a, bf16x8 b, f32x16 c) {
  asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(c) : "v"(a), "v"(b));
  return c;
}
// Maxima without the canonicalization that fmaxf puts on operands which come out of asm statements: of three, and of the
// 16 values of an accumulator in two statements (the compiler separates dependent ones by a wait state).
__device__ inline float max3(float a, float b, float c) {
  float d;
  asm("v_max3_f32 %0, %1, %2, %3" : "=v"(d) : "v"(a), "v"(b), "v"(c));
  return d;
}
__device__ inline void max15(float (&m)[4], const f32x16& s) {
  asm volatile("v_max3_f32 %0, %4, %5, %6\n\tv_max3_f32 %1, %7, %8, %9\n\tv_max3_f32 %2, %10, %11, %12\n\tv_max3_f32 %3, %13, %14, %15"
               : "=&v"(m[0]), "=&v"(m[1]), "=&v"(m[2]), "=&v"(m[3])
               : "v"(s[0]), "v"(s[1]), "v"(s[2]), "v"(s[3]), "v"(s[4]), "v"(s[5]), "v"(s[6]), "v"(s[7]), "v"(s[8]), "v"(s[9]),
                 "v"(s[10]), "v"(s[11]));
}
__device__ inline float max_rest(const float (&m)[4], const f32x16& s) {
  float d, e;
  asm volatile("v_max3_f32 %0, %2, %3, %4\n\tv_max3_f32 %1, %5, %6, %7\n\tv_max3_f32 %0, %0, %8, %9\n\tv_max_f32 %0, %0, %1"
               : "=&v"(d), "=&v"(e)
               : "v"(m[0]), "v"(m[1]), "v"(s[12]), "v"(m[2]), "v"(m[3]), "v"(s[13]), "v"(s[14]), "v"(s[15]));
  return d;
}
// the maximum of x over the two lanes l, l ^ 32
__device__ inline float half_max(float x) {
  const uint32_t u = __builtin_bit_cast(uint32_t, x);
  const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  const uint32_t a = r[0], b = r[1];           // (a bit cast of an element would take element 0)
  return max3(__builtin_bit_cast(float, a), __builtin_bit_cast(float, b), __builtin_bit_cast(float, b));
}

// O *= a for the 64 AGPR accumulator values of a head block, one register at a time through one VGPR (a plain C++
// multiply makes the register allocator move the whole accumulator into VGPRs; the rescale is a rare path).
__device__ inline void scale_acc(f32x16 (&O)[4], float a) {
#pragma unroll
  for (int b = 0; b < 4; ++b)
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      float tmp;
      asm volatile("v_accvgpr_read_b32 %1, %0\n\tv_mul_f32 %1, %1, %2\n\tv_accvgpr_write_b32 %0, %1"
                   : "+a"(O[b][e]), "=&v"(tmp)
                   : "v"(a));
    }
}

template <int N>
using ic = std::integral_constant<int, N>;

struct Params {
  const uint16_t* q; long long q_st, q_sh;        // q[t][h][576] bf16 (last dim contiguous)
  const uint8_t* pool; long long R;               // Row656 (or Row576) rows
  const int* idx; long long idx_st; int K;        // idx[t][k]
  const int* kcount;                              // optional per-token count of leading valid entries
  int T, H, S, HG;                                // tokens, heads, splits, head groups of 128
  float c;                                        // sm_scale * kv_scale * log2(e)
  float kv_scale;
  uint16_t* out; long long o_st, o_sh;            // bf16 out[t][h][512] (when opart is null)
  float* lse; long long lse_st;                   // lse[t][h]
  float* opart; float* lsepart;                   // fp32 partials: opart[s][t][h][512], lsepart[s][t][h]
  // optional prior partial merged into the bf16 output (S == 1): normalized fp32 o and natural-log lse
  const float* prior_o; long long po_st, po_sh;
  const float* prior_lse; long long pl_st;
  Pages pg;                                       // idx holds positions (pg.bt) or rows
};

// Row scales as DPP operands. z[a] of lane l = scale g of row 8 a + 4 hh + l % 4; value i = 4 a + b of a C-layout
// accumulator (row 8 a + 4 hh + b) takes its scale from lane 4 (l / 4) + b of the same quad (quad_perm b,b,b,b), so one
// register per a serves the four rows of a quad. A DPP source may not have been written by the VALU within 2 wait
// states, which the compiler cannot see inside asm: the scales come from LDS or were multiplied a tile half earlier.
// s[8 A + b] += z0 (row of value 8 A + b) * x[b], s[8 A + 4 + b] += z1 (...) * y[b], b = 0..3
template <int A>
__device__ inline void fmac8_dpp(f32x16& s, float z0, float z1, f32x4 x, f32x4 y) {
  asm volatile("v_fmac_f32_dpp %0, %8, %10 quad_perm:[0,0,0,0] row_mask:0xf bank_mask:0xf\n\t"
               "v_fmac_f32_dpp %1, %8, %11 quad_perm:[1,1,1,1] row_mask:0xf bank_mask:0xf\n\t"
               "v_fmac_f32_dpp %2, %8, %12 quad_perm:[2,2,2,2] row_mask:0xf bank_mask:0xf\n\t"
               "v_fmac_f32_dpp %3, %8, %13 quad_perm:[3,3,3,3] row_mask:0xf bank_mask:0xf\n\t"
               "v_fmac_f32_dpp %4, %9, %14 quad_perm:[0,0,0,0] row_mask:0xf bank_mask:0xf\n\t"
               "v_fmac_f32_dpp %5, %9, %15 quad_perm:[1,1,1,1] row_mask:0xf bank_mask:0xf\n\t"
               "v_fmac_f32_dpp %6, %9, %16 quad_perm:[2,2,2,2] row_mask:0xf bank_mask:0xf\n\t"
               "v_fmac_f32_dpp %7, %9, %17 quad_perm:[3,3,3,3] row_mask:0xf bank_mask:0xf"
               : "+v"(s[8 * A]), "+v"(s[8 * A + 1]), "+v"(s[8 * A + 2]), "+v"(s[8 * A + 3]), "+v"(s[8 * A + 4]),
                 "+v"(s[8 * A + 5]), "+v"(s[8 * A + 6]), "+v"(s[8 * A + 7])
               : "v"(z0), "v"(z1), "v"(x[0]), "v"(x[1]), "v"(x[2]), "v"(x[3]), "v"(y[0]), "v"(y[1]), "v"(y[2]), "v"(y[3]));
}
template <int A>
__device__ inline f32x4 quarter(const f32x16& x) { return f32x4{x[4 * A], x[4 * A + 1], x[4 * A + 2], x[4 * A + 3]}; }
// (p z) of two groups of four values with the row scales as above, as four packed f16 pairs (round to nearest even).
// The packing is part of the statement: the compiler would move it behind the barrier and keep the fp32 products live.
__device__ inline u32x4 mul8_dpp_f16(float z0, float z1, f32x4 p, f32x4 q) {
  float t0, t1, t2, t3;
  uint32_t o0, o1, o2, o3;
  asm volatile("v_mul_f32_dpp %0, %8, %10 quad_perm:[0,0,0,0] row_mask:0xf bank_mask:0xf\n\t"
               "v_mul_f32_dpp %1, %8, %11 quad_perm:[1,1,1,1] row_mask:0xf bank_mask:0xf\n\t"
               "v_mul_f32_dpp %2, %8, %12 quad_perm:[2,2,2,2] row_mask:0xf bank_mask:0xf\n\t"
               "v_mul_f32_dpp %3, %8, %13 quad_perm:[3,3,3,3] row_mask:0xf bank_mask:0xf\n\t"
               "v_cvt_pk_f16_f32 %4, %0, %1\n\t"
               "v_cvt_pk_f16_f32 %5, %2, %3\n\t"
               "v_mul_f32_dpp %0, %9, %14 quad_perm:[0,0,0,0] row_mask:0xf bank_mask:0xf\n\t"
               "v_mul_f32_dpp %1, %9, %15 quad_perm:[1,1,1,1] row_mask:0xf bank_mask:0xf\n\t"
               "v_mul_f32_dpp %2, %9, %16 quad_perm:[2,2,2,2] row_mask:0xf bank_mask:0xf\n\t"
               "v_mul_f32_dpp %3, %9, %17 quad_perm:[3,3,3,3] row_mask:0xf bank_mask:0xf\n\t"
               "v_cvt_pk_f16_f32 %6, %0, %1\n\t"
               "v_cvt_pk_f16_f32 %7, %2, %3"
               : "=&v"(t0), "=&v"(t1), "=&v"(t2), "=&v"(t3), "=&v"(o0), "=&v"(o1), "=&v"(o2), "=&v"(o3)
               : "v"(z0), "v"(z1), "v"(p[0]), "v"(p[1]), "v"(p[2]), "v"(p[3]), "v"(q[0]), "v"(q[1]), "v"(q[2]), "v"(q[3]));
  return u32x4{o0, o1, o2, o3};
}

// LDS place of query operand n = r NK + ks (-1: in registers): every fourth one, or the last of steps 1 to 3
template <bool R5>
__device__ constexpr int q_lds(int n) {
  return R5 ? ((n & 3) == 3 ? n / 4 : -1) : ((n & 7) == 7 && n > 8 ? n / 8 - 1 : -1);
}

template <bool R5>
__global__ void __launch_bounds__(256, 1) fwd_kernel(Params p) {
  using L = Lds<R5>;
  constexpr int RB = R5 ? ROW576 : ROW656;
  constexpr int NK = R5 ? 9 : 8;                  // QK MFMAs per head block: the group's 128 dims (and 16 of the rope)
  constexpr int VM_TILE = R5 ? 5 : 6;             // copies per wave and tile
  extern __shared__ __attribute__((aligned(16))) uint8_t smem_generic[];
  SPMLA_LDS uint8_t* lds = (SPMLA_LDS uint8_t*)smem_generic;

  const int nwork = p.T * p.S * p.HG;
  const int f = remap_xcd(blockIdx.x, nwork);
  if (f < 0) return;
  const int hg = f % p.HG;
  const int ts = f / p.HG;
  const int s = ts % p.S;
  const int t = ts / p.S;

  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);   // wave-uniform: scalar control flow
  const int hh = lane >> 5, l32 = lane & 31;
  const int h = hg * HGW + w * HB + l32;                    // this lane's head of the wave's own block
  const bool hval = h < p.H;
  auto block_of = [&](int r) -> int { return (w + 1 + r) & 3; };   // head block of step r (r = 3: the wave's own)

  // ---- row range of this split
  const int kc = ((p.K + p.S - 1) / p.S + TR - 1) / TR * TR;
  const int kb = s * kc;
  int ke = kb + kc < p.K ? kb + kc : p.K;
  if (p.kcount) { const int cc = p.kcount[t]; ke = ke < cc ? ke : cc; }
  const int nrow = ke > kb ? ke - kb : 0;
  const int ntile = p.R > 0 ? (nrow + TR - 1) / TR : 0;     // no rows to read: o = 0, lse = -inf

  // ---- prologue: validated row ids -> LDS; this wave's group of the query of all four head blocks -> VGPRs (B operands:
  // lane half hh holds the dims of 16-byte code chunk 2 kp + hh, MFMA 2 kp + e its bytes 8 e .. 8 e + 7); query rope
  const int* idxrow = p.idx + (long long)t * p.idx_st + kb;
  int xs[KMAX / 256];
#pragma unroll
  for (int k = 0; k < KMAX / 256; ++k) {
    const int i = tid + 256 * k;
    int x = -1;
    if (i < nrow) x = idxrow[i];
    xs[k] = x;
  }
  if (p.pg.bt) {
    const int* btrow = p.pg.bt + (long long)p.pg.req[t] * p.pg.bt_st;
    int b[KMAX / 256];
#pragma unroll
    for (int k = 0; k < KMAX / 256; ++k) b[k] = page_entry(p.pg, btrow, xs[k], p.pg.req + t);
#pragma unroll
    for (int k = 0; k < KMAX / 256; ++k) xs[k] = page_row(p.pg, xs[k], b[k]);
  }
#pragma unroll
  for (int k = 0; k < KMAX / 256; ++k) xs[k] = xs[k] >= 0 && (long long)xs[k] < p.R ? xs[k] : -1;
  bf16x8 qf[4 * NK];                                         // operand r NK + ks; NQL of them move to LDS below
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int hr = hg * HGW + block_of(r) * HB + l32;
    const uint32_t qmask = hr < p.H ? 0xffffffffu : 0u;     // heads past H: zero query
    const uint16_t* qrow = p.q + (long long)t * p.q_st + (long long)(hr < p.H ? hr : 0) * p.q_sh;
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) {
      const u32x4 v = *(const u32x4*)(qrow + 128 * w + 16 * (2 * (ks >> 1) + hh) + 8 * (ks & 1)) & qmask;
      qf[r * NK + ks] = __builtin_bit_cast(bf16x8, v);
    }
    if constexpr (R5) {                                      // rope dims 16 w + 8 hh .. + 7
      const u32x4 v = *(const u32x4*)(qrow + D_LAT + 16 * w + 8 * hh) & qmask;
      qf[r * NK + 8] = __builtin_bit_cast(bf16x8, v);
    }
  }
  u32x4 qrv[4];
  if constexpr (!R5) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {                            // rope of the own block: 32 heads x 8 chunks, 4 per lane
      const uint16_t* src = p.q + (long long)t * p.q_st + (long long)(hval ? h : 0) * p.q_sh + D_LAT + 8 * (2 * k + hh);
      qrv[k] = *(const u32x4*)src & (hval ? 0xffffffffu : 0u);
    }
  }
  wait_vm<0>();
  SPMLA_LDS int* ids = (SPMLA_LDS int*)(lds + L::IDS);
#pragma unroll
  for (int k = 0; k < KMAX / 256; ++k) ids[tid + 256 * k] = xs[k];
  if (tid < 3 * TR) ids[KMAX + tid] = -1;
  SPMLA_LDS uint8_t* reg = lds + w * L::WAVE;               // this wave's region
  if constexpr (!R5) {
#pragma unroll
    for (int k = 0; k < 4; ++k) *(SPMLA_LDS u32x4*)(reg + L::QR + k * 1024 + lane * 16) = qrv[k];
  }
#pragma unroll
  for (int n = 0; n < 4 * NK; ++n)
    if (q_lds<R5>(n) >= 0) *(SPMLA_LDS u32x4*)(reg + L::QL + q_lds<R5>(n) * 1024 + lane * 16) = __builtin_bit_cast(u32x4, qf[n]);
  // "tile -1", whose PV the first step runs: zero codes, scales and P
#pragma unroll
  for (int k = 0; k < 4; ++k) *(SPMLA_LDS u32x4*)(reg + 2 * L::CODE + (k * 64 + lane) * 16) = u32x4{0, 0, 0, 0};
#pragma unroll
  for (int k = 0; k < L::PB / 1024; ++k) *(SPMLA_LDS u32x4*)(reg + L::P + (k * 64 + lane) * 16) = u32x4{0, 0, 0, 0};
  SPMLA_LDS int* flags = (SPMLA_LDS int*)(lds + L::FLAG);
  if (lane == 0) flags[w] = 0;
  SPMLA_LDS float* st = (SPMLA_LDS float*)(lds + L::ST);
  lds_barrier();

  // Copies of tile jj into the ring slot at sl for wave w, all of lane l from row l % 32 of the tile: the codes of scale
  // group w (copy i fills chunks 2 i + l / 32); Row656: chunk 2 w + l / 32 of the rope and scale w; Row576: 16 bytes of
  // rope. VM_TILE instructions whatever the tile: rows and tiles that do not exist copy the zero row.
  uint64_t zrow = (uint64_t)(uintptr_t)zero_row;       // source of rows that do not exist
  asm volatile("" : "+s"(zrow));                       // (its address would be formed again in every step)
  auto row_at = [&](int x, int ln) -> uint64_t {       // address of the lane's first code chunk of row x, without a branch
    uint64_t a = (uint64_t)(uintptr_t)p.pool + (uint64_t)(uint32_t)x * RB;
    asm volatile("" : "+v"(a));
    return (x >= 0 ? a : zrow) + (uint32_t)(128 * w + 16 * (ln >> 5));
  };
  auto issue_code = [&](int sl, uint64_t row, auto i) {
    dma16_off<32 * decltype(i)::value, 1024 * decltype(i)::value>(row, reg + sl);
  };
  auto issue_rope = [&](int ln, int jj, int sl, uint64_t row) {
    if constexpr (R5) { if (ln < 32) dma16((const void*)(row + (uint64_t)(D_LAT - 112 * w)), reg + sl + 4096); }
    else dma16((const void*)(row + (uint64_t)(ROPE_OFF - 96 * w)), lds + L::RP + (jj & 1) * RP_TILE + w * 1024);
  };
  auto issue_scale = [&](int sl, uint64_t row) {       // (the upper lanes' 16 bytes more: the next scales or the rope)
    if constexpr (!R5) dma4((const void*)(row + (uint64_t)(SC_OFF - 124 * w)), reg + sl + 4096);
  };
  auto issue = [&](int jj, int sl) {
    const uint64_t r0 = row_at(ids[jj * TR + l32], lane);
    issue_code(sl, r0, ic<0>());
    issue_code(sl, r0, ic<1>());
    issue_code(sl, r0, ic<2>());
    issue_code(sl, r0, ic<3>());
    issue_rope(lane, jj, sl, r0);
    issue_scale(sl, r0);
  };

  const float c = p.c;
  float m_run = -__builtin_inff();     // reference max of this lane's head (log2 units)
  float l_run = 0.f;                   // sum of p over this lane's 16 rows of every tile
  // Row576: the sum of the rounded p, which the output is divided by (an error of a row that dominates a head cancels)
  float l_rnd = 0.f;
  constexpr float PUP = R5 ? 9.f : 0.f;   // Row576: P, O and l carry a factor 2^9 (P < 2^15: few f16 subnormals)
  int eps = 0;                         // P' and O carry a factor 2^-eps (f16 range of P')
  float elim = 0.f, zmul = 1.f;        // 2^(9 + eps) once eps is set; 2^-eps

  f32x16 O[4][4];                      // [step r: head block][32 dims] of group w
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int b = 0; b < 4; ++b) O[r][b] = f32x16{};

  u32x4 kr[4];                         // codes of the next tile's K operands (and its rope codes)
  u32x2 krr = {};
  auto k_read = [&](int own, int sl, int kp) -> u32x4 {       // chunk 2 kp + half of row ln % 32
    return *(SPMLA_LDS u32x4*)(lds + own + sl + kp * 1024);
  };
  auto kr_read = [&](int ln, int sl) -> u32x2 { return *(SPMLA_LDS u32x2*)(reg + sl + 4096 + (ln & 31) * 16 + 8 * (ln >> 5)); };
  // scales as DPP operands (see fmac8_dpp); zb: the own slot's at ring offset 0; d: another wave's region, and the slot
  auto zload = [&](SPMLA_LDS uint8_t* zb, int d) -> f32x4 {
    SPMLA_LDS float* a = (SPMLA_LDS float*)(zb + d);
    return f32x4{a[0], a[8], a[16], a[24]};
  };

  f32x4 zj = {};                       // scales of group w of tile j, times 2^-eps (P')
  if (ntile > 0) {
    issue(0, 0);
    issue(1, L::CODE);
    wait_vm<VM_TILE>();
#pragma unroll
    for (int kp = 0; kp < 4; ++kp) kr[kp] = k_read(w * L::WAVE + lane * 16, 0, kp);
    if constexpr (R5) krr = kr_read(lane, 0);
    lds_barrier();
  }
  int s0 = 2 * L::CODE, s1 = 0, s2 = L::CODE;   // ring slots of tiles j, j + 1, j + 2
  bool dirty = false;                  // the wave's factors were not all 1
  // regions of the waves of steps 0 to 2 from the wave's own
  const int d0 = (block_of(0) - w) * L::WAVE, d1 = (block_of(1) - w) * L::WAVE, d2 = (block_of(2) - w) * L::WAVE;
#pragma unroll 1
  for (int j = -1; j < ntile && ntile > 0; ++j) {
    // ======== first half: S of tile j + 1 for group w, all four head blocks; P' of tile j for group w
    // (tile j + 1 has landed for every wave; P and the factors of tile j are written)
    // the lane id, opaque in every step: the LDS addresses made of it would be hoisted and spilled
    int lo = lane;
    asm volatile("" : "+v"(lo));
    const int own = w * L::WAVE + lo * 16;
    auto oth = [&](int r) -> int { return own + (r == 0 ? d0 : r == 1 ? d1 : r == 2 ? d2 : 0); };
    auto blk = [&](int r) -> int { return (w + 1 + r) & 3; };
    const i32x4 fl = *(SPMLA_LDS i32x4*)flags;
    f32x4 zn;                           // scales of group w of tile j + 1
    bf16x8 kf[NK];
    auto k_conv = [&](int k) {
      kf[k] = k == 8 ? codes8_bf16(krr[0], krr[1]) : (k & 1) ? codes8_bf16(kr[k >> 1][2], kr[k >> 1][3]) : codes8_bf16(kr[k >> 1][0], kr[k >> 1][1]);
    };
    k_conv(0);
    k_conv(1);
    f16x8 pb[4][2];                     // P' of tile j: B operands per head block and k half
    f32x4 pr[2];                        // raw P values in flight
    f32x16 acc[2], S;
    bf16x8 ra[2], rb[2];                // rope operands (Row656)
    bf16x8 qn;                          // query operand from LDS
    auto p_read = [&](int cb) {         // operand cb = 2 r + ks
      const int r = cb >> 1, ks = cb & 1;
      SPMLA_LDS uint8_t* pa = lds + oth(r) + L::P;
      if constexpr (R5) pb[r][ks] = __builtin_bit_cast(f16x8, *(SPMLA_LDS u32x4*)(pa + ks * 1024));
      else {
        pr[0] = *(SPMLA_LDS f32x4*)(pa + 2 * ks * 1024);
        pr[1] = *(SPMLA_LDS f32x4*)(pa + (2 * ks + 1) * 1024);
      }
    };
    auto p_scale = [&](int cb) {        // values 8 ks .. 8 ks + 7: row groups 2 ks, 2 ks + 1
      if constexpr (!R5)
        pb[cb >> 1][cb & 1] = __builtin_bit_cast(f16x8, mul8_dpp_f16(zj[2 * (cb & 1)], zj[2 * (cb & 1) + 1], pr[0], pr[1]));
    };
    auto s_write = [&](int r, int a) {  // rows 8 a + 4 hh .. of step r's partial to its owner
      SPMLA_LDS uint8_t* d = lds + own + L::S + r * 4096 + a * 1024;
      const f32x16& x = acc[r & 1];
      *(SPMLA_LDS f32x4*)d = f32x4{x[4 * a], x[4 * a + 1], x[4 * a + 2], x[4 * a + 3]};
    };
    auto p_slices = [&](int m) {        // slices of P': operand cb is read at MFMA 12 + 3 cb and scaled three later
      if (m >= 12 && m % 3 == 0) {
        if (m >= 15) p_scale((m - 15) / 3);
        p_read((m - 12) / 3);
      }
    };
    auto rope_read = [&](int ks) {
      ra[ks & 1] = __builtin_bit_cast(bf16x8, *(SPMLA_LDS u32x4*)(lds + L::RP + ((j + 1) & 1) * RP_TILE + lo * 16 + ks * 1024));
      rb[ks & 1] = __builtin_bit_cast(bf16x8, *(SPMLA_LDS u32x4*)(lds + own + L::QR + ks * 1024));
    };
    // V^T operand reads (16-lane group G of the transposing read: lane 2 i + c supplies row i, bytes 8 c .. 8 c + 7; the
    // rows follow the C-layout rows of the lane's P values)
    SPMLA_LDS uint8_t *vb = nullptr, *zb = nullptr, *idp = nullptr;   // (addresses: set after the first chain)
    auto addresses = [&]() {
      int ln = lane;
      asm volatile("" : "+v"(ln));
      vb = reg + s0 + (((ln >> 4) & 1) * 32 + 8 * ((ln >> 3) & 1) + 4 * (ln >> 5) + ((ln >> 1) & 3)) * 16 + (ln & 1) * 8;
      zb = reg + 4096 + (4 * (ln >> 5) + (ln & 3)) * 4;
      idp = lds + L::IDS + (j + 1) * (TR * 4) + (ln & 31) * 4;
    };
    auto vread = [&](int v) -> i32x2 {          // operand v = 2 db + ks: dims 32 db .. of the group, rows 16 ks ..
      return __builtin_amdgcn_ds_read_tr8_b64_v2i32((SPMLA_LDS i32x2*)(vb + (v >> 1) * 1024 + (v & 1) * 256));
    };
    constexpr int NV = R5 ? 4 : 2;      // operands converted in the first half (the rest: one operand ahead)
    i32x2 tv[8];
    f16x8 va[8];
    auto v_conv = [&](int v) { va[v] = codes8_f16((uint32_t)tv[v][0], (uint32_t)tv[v][1]); };
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if constexpr (!R5) {
        if (r == 3) {                   // rope of the own block
#pragma unroll
          for (int ks = 0; ks < 4; ++ks) {
            if (ks < 3) rope_read(ks + 1);
            if (ks == 3) s_write(2, 0);
            p_slices(24 + ks);
            S = ks == 0 ? qk_first(ra[0], rb[0]) : qk_next(ra[ks & 1], rb[ks & 1], S);
            __builtin_amdgcn_sched_barrier(0);
          }
        }
      }
#pragma unroll
      for (int ks = 0; ks < NK; ++ks) {
        const int m = r * NK + ks + (!R5 && r == 3 ? 4 : 0);
        // slices of side work
        if (r == 1 && ks == 0) addresses();
        if (r == 0 && ks + 2 < NK) k_conv(ks + 2);   // the K operands, used by all four steps
        if (r >= 1 && ks >= 3 && ks < 7 && (r < 3 || R5)) s_write(r - 1, ks - 3);
        if (r == 3 && !R5 && ks < 3) s_write(2, 1 + ks);
        if (r == 2 && ks == 5 && !R5) rope_read(0);
        if (r == 3 && ks == 4 && !R5) zn = zload(zb, s1);
        p_slices(m);
        if (r == 3 && ks < NV + 1) tv[ks] = vread(ks);
        if (r == 3 && ks >= NK - NV) {
          v_conv(ks - (NK - NV));
          asm volatile("" : "+v"(va[ks - (NK - NV)]));
        }
        const int n = r * NK + ks;      // query operand; one from LDS is read three MFMAs ahead
        if (n + 3 < 4 * NK && q_lds<R5>(n + 3) >= 0)
          qn = __builtin_bit_cast(bf16x8, *(SPMLA_LDS u32x4*)(lds + own + L::QL + q_lds<R5>(n + 3) * 1024));
        const bf16x8 b = q_lds<R5>(n) < 0 ? qf[n] : qn;
        f32x16& x = acc[r & 1];
        if (ks == 0) x = qk_first(kf[0], b);
        else x = qk_next(kf[ks], b, x);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    p_scale(7);
    // the factors of tile j (rare; before tile 0 there is nothing to scale)
    if (__builtin_amdgcn_readfirstlane(fl[0] | fl[1] | fl[2] | fl[3]) && j > 0) {
#pragma unroll
      for (int r = 0; r < 4; ++r) scale_acc(O[r], st[blk(r) * HB + (lo & 31)]);
    }
    lds_barrier();                      // partials exchanged; P and the factors of tile j are read

    // ======== second half: PV of tile j; the softmax of tile j + 1 for the wave's own heads under its MFMAs
    f32x4 x[4];                                 // partials in flight: quarter a of source step r (wave (w - 1 - r) & 3)
    auto x_read = [&](int r, int a) { x[a] = *(SPMLA_LDS f32x4*)(lds + oth(2 - r) + L::S + r * 4096 + a * 1024); };
    f32x4 z[2];
    auto z_read = [&](int r) { if constexpr (!R5) z[r & 1] = zload(zb, s1 + (r == 0 ? d2 : r == 1 ? d1 : d0)); };
#pragma unroll
    for (int a = 0; a < 4; ++a) x_read(0, a);
    z_read(0);
    auto combine = [&](int r, int a) {          // row groups 2 a, 2 a + 1
      if constexpr (R5) {
#pragma unroll
        for (int e = 0; e < 4; ++e) { S[8 * a + e] += x[2 * a][e]; S[8 * a + 4 + e] += x[2 * a + 1][e]; }
      } else {
        if (a == 0) fmac8_dpp<0>(S, z[r & 1][0], z[r & 1][1], x[0], x[1]);
        else fmac8_dpp<1>(S, z[r & 1][2], z[r & 1][3], x[2], x[3]);
      }
    };
    int idv = -1, nx = -1;                      // ids of the lane's row of tiles j + 1, j + 3
    uint64_t nrow_at = 0;
    float P[16];
    float m8[4], mref = 0.f, alpha = 1.f;
    bool resc = false;
    if constexpr (R5) S = acc[1];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int v = 0; v < 8; ++v) {
      const int db = v >> 1, ks = v & 1;
      if (v >= NV - 1 && v + 2 < 8) tv[v + 2] = vread(v + 2);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = 4 * v + r;
        // slices of side work: the partials of the other three groups, the maximum, the exponentials, their sum
        if (m >= 4 && m < 16 && (m & 1) == 0) {
          combine(m / 4 - 1, (m & 2) / 2);
          if (m < 12) { x_read(m / 4, m & 2); x_read(m / 4, (m & 2) + 1); }
        }
        if constexpr (!R5) {            // the own block's group: its chain ended three MFMAs ago
          if (m == 3) fmac8_dpp<0>(S, zn[0], zn[1], quarter<0>(acc[1]), quarter<1>(acc[1]));
          if (m == 5) fmac8_dpp<1>(S, zn[2], zn[3], quarter<2>(acc[1]), quarter<3>(acc[1]));
        }
        if (m == 3) z_read(1);
        if (m == 8) z_read(2);
        if (m == 12) idv = *(SPMLA_LDS int*)idp;
        if (m == 16) {                  // rows that do not exist: -inf (C-layout row of value i: 8 (i / 4) + 4 hh + i % 4)
          const unsigned vmask = (unsigned)__ballot(idv >= 0);
          if (__builtin_expect(vmask != 0xffffffffu, 0)) {     // rare: keep it a branch, not 16 selects per tile
            asm volatile("" ::: "memory");
            const unsigned lm = vmask >> (4 * (lo >> 5));
#pragma unroll
            for (int i = 0; i < 16; ++i)
              if (!((lm >> (8 * (i >> 2) + (i & 3))) & 1u)) S[i] = -__builtin_inff();
          }
          max15(m8, S);
        }
        if (m == 17) m8[0] = max_rest(m8, S);
        if (m == 19) {                  // online softmax of this lane's head
          const float mx = half_max(m8[0]) * c;   // c > 0; -inf stays -inf
          const bool need = mx > m_run + TAU;                    // also true for the first finite tile
          if (__ballot(need)) {
            const float mn = need ? mx : m_run;
            alpha = need ? (m_run > -__builtin_inff() ? __builtin_amdgcn_exp2f(m_run - mn) : 0.f) : 1.f;
            l_run *= alpha;
            if constexpr (R5) l_rnd *= alpha;
            m_run = mn;
            resc = true;
          }
          mref = (m_run > -__builtin_inff() ? m_run : 0.f) - PUP;
        }
        if (m >= 20 && m < 28) {
#pragma unroll
          for (int i = 2 * (m - 20); i < 2 * (m - 20) + 2; ++i)
            P[i] = __builtin_amdgcn_exp2f(__builtin_fmaf(S[i], c, -mref));   // exp2(-inf) = 0
        }
        if (m >= 22 && (m & 1) == 0 && m < 30) {                 // P of value group a to the other waves
          const int a = (m - 22) >> 1;
          if constexpr (!R5)
            *(SPMLA_LDS f32x4*)(lds + own + L::P + a * 1024) = f32x4{P[4 * a], P[4 * a + 1], P[4 * a + 2], P[4 * a + 3]};
          else if (a & 1) {                                      // P' = P in f16, for every group
            const int q = 4 * a - 4;
            const u32x4 ph = u32x4{pk_f16(P[q], P[q + 1]), pk_f16(P[q + 2], P[q + 3]), pk_f16(P[q + 4], P[q + 5]), pk_f16(P[q + 6], P[q + 7])};
            *(SPMLA_LDS u32x4*)(lds + own + L::P + (a / 2) * 1024) = ph;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const uint32_t x2 = ph[e];
              l_rnd = __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2_t, x2), f16x2_t{1, 1}, l_rnd, false);
            }
            asm volatile("" : "+v"(l_rnd));
          }
        }
        if (m >= 28) {
          const int q = 4 * (m - 28);
          l_run += (P[q] + P[q + 1]) + (P[q + 2] + P[q + 3]);
          asm volatile("" : "+v"(l_run));               // (not after the last MFMA)
        }
        // the copies of tile j + 3, into the slot of tile j once its last V operand is in registers
        if (m == 21) nx = *(SPMLA_LDS int*)(idp + 2 * TR * 4);
        if (m == 27) nrow_at = row_at(nx, lo);
        if (m == 20) wait_vm<0>();      // tile j + 2 has landed (its copies were issued a tile ago)
        if (m >= 28) {
          kr[m - 28] = k_read(own, s2, m - 28);
          if (m == 28) issue_code(s0, nrow_at, ic<0>());
          if (m == 29) issue_code(s0, nrow_at, ic<1>());
          if (m == 30) issue_code(s0, nrow_at, ic<2>());
          if (m == 31) issue_code(s0, nrow_at, ic<3>());
        }
        if (m == 31) {
          if constexpr (R5) krr = kr_read(lo, s2);
          issue_rope(lo, j + 3, s0, nrow_at);
          issue_scale(s0, nrow_at);
        }
        if (r == 2 && v + 1 < 8 && v + 1 >= NV) v_conv(v + 1);
        O[r][db] = __builtin_amdgcn_mfma_f32_32x32x16_f16(va[v], pb[r][ks], O[r][db], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    if (resc | dirty) {                                          // (uniform; rare)
      st[w * HB + (lo & 31)] = alpha;
      if (lo == 0) flags[w] = resc;
      dirty = resc;
    }
    if constexpr (!R5) {
      // f16 range of P' = P * scale: it and O carry a factor 2^-eps, so that P' < 2^TAU * 2^9 = 2^15 while every scale of
      // the wave's group is below 2^(9 + eps). eps is set by the first tile with a positive scale and rises (exact
      // power-of-two rescale of O) when a later tile's largest scale passes 2^(9 + eps) -- rare: scales sit near amax
      // / 448 of their rows.
      const float sx = max3(max3(zn[0], zn[1], zn[2]), zn[3], 0.f);
      if (__builtin_expect(__ballot(sx > elim) != 0ull, 0)) {
        // (lanes of one quad and half hold different rows)
        auto q_perm = [](float y, auto ctrl) { return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, y), decltype(ctrl)::value, 0xf, 0xf, true)); };
        float wm = half_max(sx);
        wm = fmaxf(wm, q_perm(wm, ic<0xB1>()));
        wm = fmaxf(wm, q_perm(wm, ic<0x4E>()));
        const int en = __builtin_amdgcn_readfirstlane(__builtin_amdgcn_frexp_expf(wm) - 9);   // wm * 2^-en < 2^9
        if (elim == 0.f || en > eps) {
          if (elim != 0.f) {
            const float fe = __builtin_ldexpf(1.f, eps - en);
#pragma unroll
            for (int r = 0; r < 4; ++r) scale_acc(O[r], fe);
          }
          eps = en;
          elim = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, __builtin_ldexpf(1.f, 9 + eps))));
          zmul = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, __builtin_ldexpf(1.f, -eps))));
        }
      }
      zj = zn * zmul;
    }
    lds_barrier();
    const int sn = s0;
    s0 = s1; s1 = s2; s2 = sn;
  }
  wait_vm<0>();                                                  // no copy in flight: the LDS is reused below

  // ---- epilogue: wave w holds dims 128 w .. 128 w + 127 of all heads, its own heads' sums. C layout of O[r][b]: lane
  // holds head l32 of block_of(r), dims 32 b + 8 a + 4 hh + e of the group in value 4 a + e.
  l_run += half_swap(l_run);
  if constexpr (R5) l_rnd += half_swap(l_rnd);
  SPMLA_LDS float* stp = (SPMLA_LDS float*)ids;                   // per head: weight of the prior (the ids are read)
  {
    const float Ls = l_run;
    float lse_v = Ls > 0.f ? (m_run + (log2f(Ls) - PUP)) * 0.69314718055994531f : -__builtin_inff();
    float inv = Ls > 0.f ? p.kv_scale / (R5 ? l_rnd : Ls) : 0.f;
    float wp = 0.f;                       // weight of the prior partial (merge of two normalized partials)
    if (p.prior_o && hval) {
      const float lp = p.prior_lse[(long long)t * p.pl_st + h];
      const float mf = fmaxf(lse_v, lp);
      if (mf > -__builtin_inff()) {
        const float a = expf(lse_v - mf), b = expf(lp - mf);     // exp(-inf) = 0
        const float zz = a + b;
        inv *= a / zz;
        wp = b / zz;
        lse_v = mf + logf(zz);
      }
    }
    if (hh == 0) {
      st[w * HB + l32] = inv;
      stp[w * HB + l32] = wp;
      if (hval) {
        if (p.opart) p.lsepart[((long long)s * p.T + t) * p.H + h] = lse_v;
        else p.lse[(long long)t * p.lse_st + h] = lse_v;
      }
    }
  }
  lds_barrier();
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int hb = block_of(r), h0 = hg * HGW + hb * HB;
    const float inv = st[hb * HB + l32] * __builtin_ldexpf(1.f, eps);   // (O carries 2^-eps of this wave's group)
    if (!p.opart && !p.prior_o) {          // bf16 through this wave's LDS: a head's 256 bytes in 16-byte stores
#pragma unroll
      for (int b = 0; b < 4; ++b) {
#pragma unroll
        for (int a = 0; a < 4; ++a)
          *(SPMLA_LDS u32x2*)(reg + l32 * OROW + (32 * b + 8 * a + 4 * hh) * 2) =
              u32x2{pk_bf16(O[r][b][4 * a] * inv, O[r][b][4 * a + 1] * inv), pk_bf16(O[r][b][4 * a + 2] * inv, O[r][b][4 * a + 3] * inv)};
        __builtin_amdgcn_sched_barrier(0);
      }
      const bool al16 = !(((uintptr_t)p.out | (uintptr_t)(p.o_st * 2) | (uintptr_t)(p.o_sh * 2)) & 15);
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const int hr = 4 * k + (lane >> 4);
        const u32x4 x = *(SPMLA_LDS u32x4*)(reg + hr * OROW + 16 * (lane & 15));
        uint16_t* dst = p.out + (long long)t * p.o_st + (long long)(h0 + hr) * p.o_sh + 128 * w + 8 * (lane & 15);
        if (h0 + hr < p.H) {
          if (al16) *(u32x4*)dst = x;
          else { *(uint2*)dst = make_uint2(x[0], x[1]); *(uint2*)(dst + 4) = make_uint2(x[2], x[3]); }
        }
      }
      continue;
    }
    // One block at a time (the fences keep the compiler from reading all accumulators into VGPRs at once).
    const float wp = stp[hb * HB + l32];
    const int ho = h0 + l32;
    const bool part = p.opart != nullptr;
    if (ho < p.H) {
      uint16_t* orow = part ? nullptr : p.out + (long long)t * p.o_st + (long long)ho * p.o_sh;
      float* frow = part ? p.opart + (((long long)s * p.T + t) * p.H + ho) * D_LAT : nullptr;
      const float* prow = p.prior_o ? p.prior_o + (long long)t * p.po_st + (long long)ho * p.po_sh : nullptr;
#pragma unroll
      for (int b = 0; b < 4; ++b) {
#pragma unroll
        for (int a = 0; a < 4; ++a) {
          const int col = 128 * w + 32 * b + 8 * a + 4 * hh;
          f32x4 v = f32x4{O[r][b][4 * a] * inv, O[r][b][4 * a + 1] * inv, O[r][b][4 * a + 2] * inv, O[r][b][4 * a + 3] * inv};
          if (prow) {
            const f32x4 x = *(const f32x4*)(prow + col);
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = __builtin_fmaf(x[e], wp, v[e]);
          }
          if (part) *(f32x4*)(frow + col) = v;
          else *(uint2*)(orow + col) = make_uint2(pk_bf16(v[0], v[1]), pk_bf16(v[2], v[3]));
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
}

// ---- LSE merge ------------------------------------------------------------------------------------------
// o = sum_i w_i o_i, w_i = exp(lse_i - L), L = ln sum_i exp(lse_i); all parts -inf -> o = 0, L = -inf.
// Reference: dotsnote/engine/arcstats_pkg/arcstats/sparse_offload.py:519-538 (split partials) and the
// merge_attn_states call of VP/model_executor/layers/attention/sparse_mla_attention.py:1091-1097 (tiers).
// One wave per (t, h); lane covers 8 consecutive output columns. Parts are fp32 or bf16.
struct MergeParams {
  const void* o; int o_bf16; long long o_ps, o_st, o_sh;   // part i of (t, h) at o + i*o_ps + t*o_st + h*o_sh
  const float* lse; long long l_ps, l_st;                   // lse[i*l_ps + t*l_st + h]
  int n, T, H;
  uint16_t* out; long long out_st, out_sh;                  // bf16
  float* out_f32;                                           // optional fp32 output (same strides)
  float* lse_out; long long lo_st;
};

__global__ void __launch_bounds__(256) merge_kernel(MergeParams p) {
  const int wv = blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (wv >= p.T * p.H) return;
  const int t = wv / p.H, h = wv % p.H;
  float M = -__builtin_inff();
  for (int i = 0; i < p.n; ++i) M = fmaxf(M, p.lse[i * p.l_ps + t * p.l_st + h]);
  float acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  float L = 0.f;
  if (M > -__builtin_inff()) {
    for (int i = 0; i < p.n; ++i) {
      const float li = p.lse[i * p.l_ps + t * p.l_st + h];
      if (!(li > -__builtin_inff())) continue;
      const float w = expf(li - M);
      L += w;
      const long long off = i * p.o_ps + t * p.o_st + h * p.o_sh + lane * 8;
      if (p.o_bf16) {
        const u32x4 v = *(const u32x4*)((const uint16_t*)p.o + off);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          acc[2 * e] += w * u2f(v[e] << 16);
          acc[2 * e + 1] += w * u2f(v[e] & 0xffff0000u);
        }
      } else {
        const f32x4 a = *(const f32x4*)((const float*)p.o + off);
        const f32x4 b = *(const f32x4*)((const float*)p.o + off + 4);
#pragma unroll
        for (int e = 0; e < 4; ++e) { acc[e] += w * a[e]; acc[4 + e] += w * b[e]; }
      }
    }
  }
  const float inv = L > 0.f ? 1.f / L : 0.f;
  const long long oo = t * p.out_st + h * p.out_sh + lane * 8;
  if (p.out) {
    u32x4 v;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      v[e] = (uint32_t)f2bf_rne(acc[2 * e] * inv) | ((uint32_t)f2bf_rne(acc[2 * e + 1] * inv) << 16);
    *(u32x4*)(p.out + oo) = v;
  }
  if (p.out_f32) {
    *(f32x4*)(p.out_f32 + oo) = f32x4{acc[0] * inv, acc[1] * inv, acc[2] * inv, acc[3] * inv};
    *(f32x4*)(p.out_f32 + oo + 4) = f32x4{acc[4] * inv, acc[5] * inv, acc[6] * inv, acc[7] * inv};
  }
  if (lane == 0 && p.lse_out) p.lse_out[t * p.lo_st + h] = L > 0.f ? M + logf(L) : -__builtin_inff();
}

}  // namespace attn
}  // namespace spmla

using namespace spmla;

namespace spmla {
namespace pk {
// the head-group kernel's per-token launch (spmla_attn_hg.hip)
int launch_tokens(const void* q, long long q_st, long long q_sh, const void* pool, long long R, const int* idx,
                  long long idx_st, int K, const int* kcount, int T, int H, float sm_scale, float kv_scale, int S,
                  void* out, long long o_st, long long o_sh, float* lse, long long lse_st, float* opart,
                  float* lsepart, const float* prior_o, long long po_st, long long po_sh, const float* prior_lse,
                  long long pl_st, void* ws, void* stream, bool r576, const Pages& pg);
long long ws_bytes(int T, int H, int S);
}  // namespace pk
}  // namespace spmla

extern "C" {

static bool attn_wide(int T, int H, int K, int S) {       // fwd_kernel and not the head-group kernel
  static_assert(attn::KMAX == rules::WIDE_ROWS && attn::HGW == 128 && attn::TR == 32, "what the rule was measured with");
  return rules::attn_wide(T, H, K, S);
}

static attn::Params wide_params(const void* q, long long q_st, long long q_sh, const void* pool, long long R,
                                const int* idx, long long idx_st, int K, const int* kcount, int T, int H,
                                float sm_scale, float kv_scale, int S, void* out, long long o_st, long long o_sh,
                                float* lse, long long lse_st, float* opart, float* lsepart, const float* prior_o,
                                long long po_st, long long po_sh, const float* prior_lse, long long pl_st,
                                const Pages& pg) {
  attn::Params p;
  p.pg = pg;
  p.q = (const uint16_t*)q; p.q_st = q_st; p.q_sh = q_sh;
  p.pool = (const uint8_t*)pool; p.R = R;
  p.idx = idx; p.idx_st = idx_st; p.K = K; p.kcount = kcount;
  p.T = T; p.H = H; p.S = S; p.HG = (H + attn::HGW - 1) / attn::HGW;
  p.c = sm_scale * kv_scale * 1.4426950408889634f;
  p.kv_scale = kv_scale;
  p.out = (uint16_t*)out; p.o_st = o_st; p.o_sh = o_sh; p.lse = lse; p.lse_st = lse_st;
  p.opart = opart; p.lsepart = lsepart;
  p.prior_o = prior_o; p.po_st = po_st; p.po_sh = po_sh; p.prior_lse = prior_lse; p.pl_st = pl_st;
  return p;
}

static int wide_launch(const attn::Params& p, bool r576, void* stream) {
  const long long nwork = (long long)p.T * p.S * p.HG;
  if (nwork > (1ll << 30)) return SPMLA_ELIMIT;
  const dim3 grid((unsigned)((nwork + 7) / 8 * 8));
  static DynLds lds_attr[2];
  const void* fn = r576 ? (const void*)attn::fwd_kernel<true> : (const void*)attn::fwd_kernel<false>;
  const int bytes = r576 ? attn::Lds<true>::TOTAL : attn::Lds<false>::TOTAL;
  if (const int e = lds_attr[r576].ensure(fn, bytes)) return e;
  if (r576) hipLaunchKernelGGL(attn::fwd_kernel<true>, grid, dim3(256), bytes, (hipStream_t)stream, p);
  else hipLaunchKernelGGL(attn::fwd_kernel<false>, grid, dim3(256), bytes, (hipStream_t)stream, p);
  return (int)hipGetLastError();
}

static int attn_launch(const void* q, long long q_st, long long q_sh, const void* pool, long long R, const int* idx,
                       long long idx_st, int K, const int* kcount, int T, int H, float sm_scale, float kv_scale, int S,
                       void* out, long long o_st, long long o_sh, float* lse, long long lse_st, float* opart,
                       float* lsepart, const float* prior_o, long long po_st, long long po_sh, const float* prior_lse,
                       long long pl_st, void* ws, long long ws_bytes, void* stream, const Pages& pg = Pages{}) {
  if (T < 0 || H <= 0 || K < 0 || S <= 0 || R < 0) return SPMLA_EARG;
  if (T == 0) return SPMLA_OK;
  if (!q || !idx || (R > 0 && !pool)) return SPMLA_EARG;
  const bool f32part = opart != nullptr;   // fp32 partials (any S) instead of the bf16 output
  bool fused = !f32part && S > 1;          // bf16 output of S splits merged in the kernel (workspace ws)
  if (f32part ? !lsepart : (!out || !lse)) return SPMLA_EARG;
  if (fused) {
    if (!ws || prior_o) return SPMLA_EARG;
    if (S > 8) return SPMLA_ELIMIT;
    if ((uintptr_t)ws & 255) return SPMLA_EALIGN;
    if (ws_bytes < pk::ws_bytes(T, H, S)) return SPMLA_EARG;
  }
  if (((uintptr_t)q & 15) || (q_st & 7) || (q_sh & 7) || ((uintptr_t)pool & 15)) return SPMLA_EALIGN;
  if (out && (((uintptr_t)out & 7) || (o_st & 3) || (o_sh & 3))) return SPMLA_EALIGN;
  if (f32part && ((uintptr_t)opart & 15)) return SPMLA_EALIGN;
  if (fused && ((K + S - 1) / S + attn::TR - 1) / attn::TR * attn::TR > attn::KMAX) return SPMLA_ELIMIT;   // (a limit kept
  // from the kernel that merged before; the head-group kernel has none)
  if (fused) {
    S = rules::merged_splits(T, H, K, S, false);
    fused = S > 1;
  }
  if (fused || !attn_wide(T, H, K, S))
    return pk::launch_tokens(q, q_st, q_sh, pool, R, idx, idx_st, K, kcount, T, H, sm_scale, kv_scale, S, out, o_st,
                             o_sh, lse, lse_st, opart, lsepart, prior_o, po_st, po_sh, prior_lse, pl_st,
                             fused ? ws : nullptr, stream, false, pg);
  return wide_launch(wide_params(q, q_st, q_sh, pool, R, idx, idx_st, K, kcount, T, H, sm_scale, kv_scale, S, out, o_st,
                                 o_sh, lse, lse_st, opart, lsepart, prior_o, po_st, po_sh, prior_lse, pl_st, pg), false,
                     stream);
}

// See include/spmla.h for the contracts.
int spmla_attn_splitk(const void* q, long long q_st, long long q_sh, const void* pool, long long R,
                      const int* idx, long long idx_st, int K, const int* kcount, int T, int H, float sm_scale,
                      float kv_scale, int S, void* out, long long o_st, long long o_sh, float* lse,
                      long long lse_st, float* opart, float* lsepart, void* stream) {
  return attn_launch(q, q_st, q_sh, pool, R, idx, idx_st, K, kcount, T, H, sm_scale, kv_scale, S, out, o_st, o_sh, lse,
                     lse_st, opart, lsepart, nullptr, 0, 0, nullptr, 0, nullptr, 0, stream);
}

long long spmla_attn_ws_bytes(int T, int H, int S) {
  if (T < 0 || H <= 0 || S <= 0) return -1;
  return S == 1 ? 0 : pk::ws_bytes(T, H, S);
}

int spmla_attn(const void* q, long long q_st, long long q_sh, const void* pool, long long R, const int* idx,
               long long idx_st, int K, const int* kcount, int T, int H, float sm_scale, float kv_scale, int S,
               void* out, long long o_st, long long o_sh, float* lse, long long lse_st, void* ws, long long ws_bytes,
               void* stream) {
  return attn_launch(q, q_st, q_sh, pool, R, idx, idx_st, K, kcount, T, H, sm_scale, kv_scale, S, out, o_st, o_sh, lse,
                     lse_st, nullptr, nullptr, nullptr, 0, 0, nullptr, 0, S > 1 ? ws : nullptr, ws_bytes, stream);
}

static int attn576_launch(const void* q, long long q_st, long long q_sh, const void* pool, long long R, const int* idx,
                  long long idx_st, int K, const int* kcount, int T, int H, float sm_scale, float kv_scale, int S,
                  void* out, long long o_st, long long o_sh, float* lse, long long lse_st, float* opart,
                  float* lsepart, void* ws, long long ws_bytes, void* stream, const Pages& pg = Pages{}) {
  if (T < 0 || H <= 0 || K < 0 || S <= 0 || R < 0) return SPMLA_EARG;
  if (T == 0) return SPMLA_OK;
  if (!q || !idx || (R > 0 && !pool)) return SPMLA_EARG;
  const bool f32part = opart != nullptr;
  bool fused = !f32part && S > 1;
  if (f32part ? !lsepart : (!out || !lse || (fused && !ws))) return SPMLA_EARG;
  if (fused) {
    if (S > 8) return SPMLA_ELIMIT;
    if ((uintptr_t)ws & 255) return SPMLA_EALIGN;
    if (ws_bytes < pk::ws_bytes(T, H, S)) return SPMLA_EARG;
  }
  if (((uintptr_t)q & 15) || (q_st & 7) || (q_sh & 7) || ((uintptr_t)pool & 15)) return SPMLA_EALIGN;
  if (out && (((uintptr_t)out & 7) || (o_st & 3) || (o_sh & 3))) return SPMLA_EALIGN;
  if (f32part && ((uintptr_t)opart & 15)) return SPMLA_EALIGN;
  if (fused) {
    S = rules::merged_splits(T, H, K, S, true);
    fused = S > 1;
  }
  if (!fused && attn_wide(T, H, K, S))
    return wide_launch(wide_params(q, q_st, q_sh, pool, R, idx, idx_st, K, kcount, T, H, sm_scale, kv_scale, S, out,
                                   o_st, o_sh, lse, lse_st, opart, lsepart, nullptr, 0, 0, nullptr, 0, pg), true, stream);
  return pk::launch_tokens(q, q_st, q_sh, pool, R, idx, idx_st, K, kcount, T, H, sm_scale, kv_scale, S, out, o_st,
                           o_sh, lse, lse_st, opart, lsepart, nullptr, 0, 0, nullptr, 0, fused ? ws : nullptr, stream,
                           true, pg);
}

int spmla_attn576(const void* q, long long q_st, long long q_sh, const void* pool, long long R, const int* idx,
                  long long idx_st, int K, const int* kcount, int T, int H, float sm_scale, float kv_scale, int S,
                  void* out, long long o_st, long long o_sh, float* lse, long long lse_st, float* opart,
                  float* lsepart, void* stream) {
  return attn576_launch(q, q_st, q_sh, pool, R, idx, idx_st, K, kcount, T, H, sm_scale, kv_scale, S, out, o_st, o_sh,
                        lse, lse_st, opart, lsepart, nullptr, 0, stream);
}

int spmla_attn576_ws(const void* q, long long q_st, long long q_sh, const void* pool, long long R, const int* idx,
                     long long idx_st, int K, const int* kcount, int T, int H, float sm_scale, float kv_scale, int S,
                     void* out, long long o_st, long long o_sh, float* lse, long long lse_st, void* ws,
                     long long ws_bytes, void* stream) {
  return attn576_launch(q, q_st, q_sh, pool, R, idx, idx_st, K, kcount, T, H, sm_scale, kv_scale, S, out, o_st, o_sh,
                        lse, lse_st, nullptr, nullptr, ws, ws_bytes, stream);
}

int spmla_attn_paged(const void* q, long long q_st, long long q_sh, const void* pool, long long R, const int* topk,
                     long long tk_st, int K, const int* req, const int* block_table, long long bt_st, int bt_cols,
                     int block_size, long long stride_rows, int T, int H, float sm_scale, float kv_scale, int row_bytes,
                     int S, void* out, long long o_st, long long o_sh, float* lse, long long lse_st, void* ws,
                     long long ws_bytes, void* stream) {
  if (row_bytes != ROW656 && row_bytes != ROW576) return SPMLA_EARG;
  if (block_size <= 0 || bt_cols <= 0) return SPMLA_EARG;
  if (block_size & (block_size - 1)) return SPMLA_ELIMIT;
  if (T > 0 && (!req || !block_table)) return SPMLA_EARG;
  const Pages pg{req, block_table, bt_st, bt_cols, __builtin_ctz((unsigned)block_size), stride_rows};
  if (row_bytes == ROW576)
    return attn576_launch(q, q_st, q_sh, pool, R, topk, tk_st, K, nullptr, T, H, sm_scale, kv_scale, S, out, o_st, o_sh,
                          lse, lse_st, nullptr, nullptr, S > 1 ? ws : nullptr, ws_bytes, stream, pg);
  return attn_launch(q, q_st, q_sh, pool, R, topk, tk_st, K, nullptr, T, H, sm_scale, kv_scale, S, out, o_st, o_sh, lse,
                     lse_st, nullptr, nullptr, nullptr, 0, 0, nullptr, 0, S > 1 ? ws : nullptr, ws_bytes, stream, pg);
}

int spmla_attn_merge(const void* q, long long q_st, long long q_sh, const void* pool, long long R, const int* idx,
                     long long idx_st, int K, const int* kcount, int T, int H, float sm_scale, float kv_scale,
                     const float* prior_o, long long po_st, long long po_sh, const float* prior_lse, long long pl_st,
                     void* out, long long o_st, long long o_sh, float* lse, long long lse_st, void* stream) {
  if (T > 0 && (!prior_o || !prior_lse)) return SPMLA_EARG;
  if (((uintptr_t)prior_o & 15) || (po_st & 3) || (po_sh & 3)) return SPMLA_EALIGN;
  return attn_launch(q, q_st, q_sh, pool, R, idx, idx_st, K, kcount, T, H, sm_scale, kv_scale, 1, out, o_st, o_sh, lse,
                     lse_st, nullptr, nullptr, prior_o, po_st, po_sh, prior_lse, pl_st, nullptr, 0, stream);
}

int spmla_lse_merge(const void* parts, int parts_bf16, long long o_ps, long long o_st, long long o_sh,
                    const float* lse, long long l_ps, long long l_st, int n, int T, int H, void* out,
                    long long out_st, long long out_sh, float* out_f32, float* lse_out, long long lo_st,
                    void* stream) {
  if (n <= 0 || T < 0 || H <= 0) return SPMLA_EARG;
  if (T == 0) return SPMLA_OK;
  if (!parts || !lse || (!out && !out_f32)) return SPMLA_EARG;
  const int eb = parts_bf16 ? 2 : 4;
  if (((uintptr_t)parts & 15) || ((o_ps * eb) & 15) || ((o_st * eb) & 15) || ((o_sh * eb) & 15))
    return SPMLA_EALIGN;
  if ((out && (((uintptr_t)out & 15) || (out_st & 7) || (out_sh & 7))) ||
      (out_f32 && (((uintptr_t)out_f32 & 15) || (out_st & 3) || (out_sh & 3))))
    return SPMLA_EALIGN;
  attn::MergeParams p;
  p.o = parts; p.o_bf16 = parts_bf16; p.o_ps = o_ps; p.o_st = o_st; p.o_sh = o_sh;
  p.lse = lse; p.l_ps = l_ps; p.l_st = l_st; p.n = n; p.T = T; p.H = H;
  p.out = (uint16_t*)out; p.out_st = out_st; p.out_sh = out_sh; p.out_f32 = out_f32;
  p.lse_out = lse_out; p.lo_st = lo_st;
  const long long waves = (long long)T * H;
  hipLaunchKernelGGL(attn::merge_kernel, dim3((unsigned)((waves + 3) / 4)), dim3(256), 0, (hipStream_t)stream, p);
  return (int)hipGetLastError();
}

}  // extern "C"
