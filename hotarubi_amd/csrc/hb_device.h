// Device-side VEC lane arithmetic for the fused epilogue and the VEC engine
// kernels.  Each operation uses the hardware FP32 unit (compiled with FP32
// denormals flushed, no contraction) where that gives the NPU's bits, and the
// integer routines of hb_fp32.h otherwise:
//   add  : identical to the NPU's add unless an operand has exponent 255;
//          a zero result is returned as +0.
//   mul  : identical when both operands are normal with exponent < 255 and
//          the product's exponent is 2..255 (no rounding near 2^-126).
// Lane formulas follow tools/iss/lane.cpp:163-179 (FloatResult),
// :305-320 (LaneOutput), :322-335 (PostAdd), :337-355 (Interpolate,
// Activation) and :406-424 (QuantizeBlock).
#pragma once

#include "hb_fp32.h"
#include "hb_internal.h"

namespace hb {

constexpr uint32_t kOne = 0x3F800000u;
constexpr uint32_t kSign = 0x80000000u;

namespace fp8 {
// Four OCP E4M3 codes (one per byte) split into two operand planes by
// exponent field: codes with exponent 8..15 (bit 6 set) go to `hi`, codes
// with exponent 0..7 (subnormals included) to `lo`; the other plane holds
// +0 there.  The block-scaled matrix cores sum an instruction's 64 FP8 x
// FP4 products exactly only while they span few binades: a full E4M3 block
// spans 17, each plane at most 9 (measured on the GPU over config 1's
// shapes: one plane 1.7e-5 of the row maximum and 2^-14.3 of the sum of
// |block values| per element, two planes 3.3e-7 and 2^-21.6).
__device__ __forceinline__ void Split(uint32_t x, uint32_t& lo, uint32_t& hi) {
  const uint32_t big = (x >> 6) & 0x01010101u;
  const uint32_t mask = (big << 8) - big;  // 0xFF in each byte with bit 6 set
  hi = x & mask;
  lo = x & ~mask;
}
}  // namespace fp8

__device__ __forceinline__ uint32_t AsBits(float f) { return __float_as_uint(f); }
__device__ __forceinline__ float AsFloat(uint32_t u) { return __uint_as_float(u); }

__device__ __forceinline__ uint32_t FAdd(uint32_t a, uint32_t b) {
  if (ExpField(a) == 0xFFu || ExpField(b) == 0xFFu) return AddBits(a, b);
  const uint32_t r = AsBits(AsFloat(a) + AsFloat(b));
  return (r << 1) == 0 ? 0u : r;
}

__device__ __forceinline__ uint32_t FMul(uint32_t a, uint32_t b) {
  const uint32_t ea = ExpField(a), eb = ExpField(b);
  if (ea == 0 || eb == 0) return 0u;
  const uint32_t r = AsBits(AsFloat(a) * AsFloat(b));
  const uint32_t er = ExpField(r);
  if (ea == 0xFFu || eb == 0xFFu || er <= 1u) return MulBits(a, b);
  return r;
}

// sign-magnitude prod >= other, both zeros equal (lane.cpp:45-58)
__device__ __forceinline__ bool MaxGreaterEqual(uint32_t prod, uint32_t other) {
  const uint32_t pm = prod & ~kSign, om = other & ~kSign;
  if (pm == 0 && om == 0) return true;
  const bool pn = (prod >> 31) != 0, on = (other >> 31) != 0;
  if (pn != on) return !pn;
  return pn ? pm <= om : pm >= om;
}

// y = v + RNE(s * frac / 2^16), entry = {s[63:32], v[31:0]}
__device__ __forceinline__ uint32_t Interpolate(uint64_t entry, uint32_t fraction) {
  return FAdd((uint32_t)entry, MulFractionBits((uint32_t)(entry >> 32), fraction));
}

// T(|x|) from the activation half of TBUF, t = TBUF + 512 (the 512 entries
// of [512, 1024)): |x| truncated to UQ4.21, 9-bit index, 16-bit fraction;
// 1.0 at |x| >= 16.
__device__ __forceinline__ uint32_t Activation(uint32_t prod, const uint64_t* t) {
  const uint32_t e = ExpField(prod);
  if (e >= 131u) return kOne;
  const uint32_t sig = Significand(prod);
  uint32_t fixed = 0;
  if (e == 130u) fixed = sig << 1;
  else if (e >= 105u) fixed = sig >> (129u - e);
  return Interpolate(t[fixed >> 16], fixed & 0xFFFFu);
}

// One VEC lane with c0 = 0, b = 1, post = ADD: Add(Mul(Add(x, c0), b), c1).
__device__ __forceinline__ uint32_t LaneAddMul(uint32_t x, uint32_t c0, uint32_t b, uint32_t c1) {
  return FAdd(FMul(FAdd(x, c0), b), c1);
}

// Epilogue op kinds (library entry numbers; ADD residual = 0x100).
enum : uint32_t {
  kEpAdd0 = 0, kEpMul = 1, kEpMax = 2, kEpAddP = 3, kEpMulP = 4, kEpScale = 5,
  kEpCopy = 6, kEpRelu = 7, kEpAct = 8, kEpActMul = 9, kEpAdd = 0x100
};

// ACT gate pass: x < 0 ? -(x*T) + x : x*T  (post = SIGNFIX, c1 = raw x);
// t = TBUF + 512.
__device__ __forceinline__ uint32_t ActGate(uint32_t x, const uint64_t* t) {
  const uint32_t pre = FAdd(x, 0u);
  const uint32_t a = Activation(FMul(pre, kOne), t);
  const uint32_t prod = FMul(pre, a);
  return (x >> 31) ? FAdd(prod ^ kSign, x) : FAdd(prod, 0u);
}

// One fused epilogue op on one element y (lane formulas of the VEC library
// entries).  Its operands are passed in already loaded: x2 the element of
// the op's [m][n] tensor (ADD, ACT_MUL), p the column's vector value (ADDP,
// MULP), imm the SCALE factor; t = TBUF + 512.
__device__ __forceinline__ uint32_t EpApply(uint32_t kind, uint32_t imm, uint32_t y, uint32_t x2,
                                            uint32_t p, const uint64_t* t) {
  switch (kind) {
    case kEpAddP: return LaneAddMul(y, p, kOne, 0u);
    case kEpMulP: return LaneAddMul(y, 0u, p, 0u);
    case kEpScale: return LaneAddMul(y, 0u, imm, 0u);
    case kEpCopy: return LaneAddMul(y, 0u, kOne, 0u);
    case kEpRelu: {
      const uint32_t prod = FMul(FAdd(y, 0u), kOne);
      return FAdd(MaxGreaterEqual(prod, 0u) ? prod : 0u, 0u);
    }
    case kEpAdd: return LaneAddMul(y, x2, kOne, 0u);
    case kEpAct: return ActGate(y, t);
    case kEpActMul: return LaneAddMul(ActGate(y, t), 0u, x2, 0u);
    default: return y;
  }
}

// The same ops in plain FP32 hardware arithmetic (flush-to-zero, round to
// nearest even, one rounding per operation), for HB_LINEAR_FAST.  Equal to
// the lane formulas above except for operands or results with exponent
// field 255, where the NPU's add and multiply differ from IEEE; zero
// results are +0 as there.  The table interpolation v + s * (frac / 2^16)
// is one correctly rounded product (frac / 2^16 is exact) and one add, as
// in the exact path.
// (Branch-free: the index is computed for every exponent and always lies in
// the table; exponents from 131 on then take 1.0.)
__device__ __forceinline__ float ActivationFast(float prod, const uint64_t* t) {
  const uint32_t bits = __float_as_uint(prod), e = ExpField(bits);
  const uint32_t sig = Significand(bits);
  const uint32_t sh = e >= 105u && e <= 129u ? 129u - e : 31u;
  const uint32_t fixed = e == 130u ? sig << 1 : e < 105u || e > 130u ? 0u : sig >> sh;
  const uint64_t entry = t[fixed >> 16];
  const float v = __uint_as_float((uint32_t)entry) +
                  __uint_as_float((uint32_t)(entry >> 32)) * ((float)(fixed & 0xFFFFu) * (1.0f / 65536.0f));
  return e >= 131u ? 1.0f : v;
}

__device__ __forceinline__ float ActGateFast(float x, const uint64_t* t) {
  const float pre = x + 0.0f;
  const float prod = pre * ActivationFast(pre, t);
  return (__float_as_uint(x) >> 31) ? (-prod + x) + 0.0f : prod + 0.0f;
}

__device__ __forceinline__ float EpApplyFast(uint32_t kind, uint32_t imm, float y, float x2,
                                             float p, const uint64_t* t) {
  switch (kind) {
    case kEpAddP: return (y + p) + 0.0f;
    case kEpMulP: return (y + 0.0f) * p + 0.0f;
    case kEpScale: return (y + 0.0f) * __uint_as_float(imm) + 0.0f;
    case kEpCopy: return y + 0.0f;
    case kEpRelu: {
      const float prod = y + 0.0f;
      return (prod > 0.0f ? prod : 0.0f) + 0.0f;
    }
    case kEpAdd: return (y + x2) + 0.0f;
    case kEpAct: return ActGateFast(y, t);
    case kEpActMul: return (ActGateFast(y, t) + 0.0f) * x2 + 0.0f;
    default: return y;
  }
}

// EpApplyFast over N (4, 16) values of a lane: the kind is resolved once, each
// case is a straight run.  x2 holds the op's [m][n] operand, p the vector
// value of each element's column (P = float: one column for all 16; P =
// f32x16_t: one per element).  kSerial keeps the 16 table lookups of an
// activation from all being in flight at once (for callers short of
// registers); otherwise their latencies overlap.
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
template <bool kSerial = true, typename V, typename P>
__device__ __forceinline__ void EpApplyFastN(uint32_t kind, uint32_t imm, V& y, const V& x2,
                                             const P& p, const uint64_t* t) {
  constexpr int kN = sizeof(V) / sizeof(float);
  switch (kind) {
    case kEpAddP: y = (y + p) + 0.0f; break;
    case kEpMulP: y = (y + 0.0f) * p + 0.0f; break;
    case kEpScale: y = (y + 0.0f) * __uint_as_float(imm) + 0.0f; break;
    case kEpCopy: y = y + 0.0f; break;
    case kEpAdd: y = (y + x2) + 0.0f; break;
    case kEpRelu:
#pragma unroll
      for (int r = 0; r < kN; ++r) {
        const float prod = y[r] + 0.0f;
        y[r] = (prod > 0.0f ? prod : 0.0f) + 0.0f;
      }
      break;
    case kEpAct:
#pragma unroll
      for (int r = 0; r < kN; ++r) {
        y[r] = ActGateFast(y[r], t);
        if (kSerial) __builtin_amdgcn_sched_barrier(0);
      }
      break;
    case kEpActMul:
#pragma unroll
      for (int r = 0; r < kN; ++r) {
        y[r] = (ActGateFast(y[r], t) + 0.0f) * x2[r] + 0.0f;
        if (kSerial) __builtin_amdgcn_sched_barrier(0);
      }
      break;
    default: break;
  }
}
template <bool kSerial = true, typename P>
__device__ __forceinline__ void EpApplyFast16(uint32_t kind, uint32_t imm, f32x16_t& y,
                                              const f32x16_t& x2, const P& p, const uint64_t* t) {
  EpApplyFastN<kSerial>(kind, imm, y, x2, p, t);
}

// EpApply over 4 values of a lane.  The FP32 unit gives the lane formulas'
// bits except where an operand or a result has exponent field 255 or a
// product of nonzero operands comes out with field 0 or 1 (it may have
// rounded up to, or been flushed below, 2^-126), so the hardware form runs
// first (EpApplyFastN's arithmetic) and a lane that saw such a field takes
// the integer routines for its 4 values.  About 12 instructions a value and
// op against 40 with every operation guarded.
__device__ __forceinline__ bool ProductOdd(uint32_t a, uint32_t b, uint32_t r) {
  return ExpField(a) != 0 && ExpField(b) != 0 && ExpField(r) <= 1u;
}
__device__ __forceinline__ bool TopField(uint32_t x) { return ExpField(x) == 255u; }

// x T(|x|) as ActGateFast, *odd raised where a step may differ from ActGate.
__device__ __forceinline__ float ActGateChecked(float x, const uint64_t* t, bool* odd) {
  const float pre = x + 0.0f;
  const uint32_t bits = __float_as_uint(pre), e = ExpField(bits);
  const uint32_t sig = Significand(bits);
  const uint32_t sh = e >= 105u && e <= 129u ? 129u - e : 31u;
  const uint32_t fixed = e == 130u ? sig << 1 : e < 105u || e > 130u ? 0u : sig >> sh;
  const uint64_t entry = t[fixed >> 16];
  const uint32_t ev = (uint32_t)entry, es = (uint32_t)(entry >> 32);
  const float frac = (float)(fixed & 0xFFFFu) * (1.0f / 65536.0f);
  const float step = __uint_as_float(es) * frac;
  float v = __uint_as_float(ev) + step;
  *odd |= TopField(ev) || TopField(es) || TopField(__float_as_uint(v)) ||
          ProductOdd(es, __float_as_uint(frac), __float_as_uint(step));
  v = e >= 131u ? 1.0f : v;
  const float prod = pre * v;
  const float y = (__float_as_uint(x) >> 31) ? (-prod + x) + 0.0f : prod + 0.0f;
  *odd |= TopField(bits) || TopField(__float_as_uint(prod)) || TopField(__float_as_uint(y)) ||
          ProductOdd(bits, __float_as_uint(v), __float_as_uint(prod));
  return y;
}

__device__ __forceinline__ void EpApply4(uint32_t kind, uint32_t imm, f32x4_t& y,
                                         const f32x4_t& x2, const f32x4_t& p, const uint64_t* t) {
  f32x4_t r;
  bool odd = false;
  switch (kind) {
    case kEpAct:
#pragma unroll
      for (int k = 0; k < 4; ++k) r[k] = ActGateChecked(y[k], t, &odd);
      break;
    case kEpActMul:
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const float gate = ActGateChecked(y[k], t, &odd);
        const float prod = gate * x2[k];
        odd |= TopField(__float_as_uint(x2[k])) || TopField(__float_as_uint(prod)) ||
               ProductOdd(__float_as_uint(gate), __float_as_uint(x2[k]), __float_as_uint(prod));
        r[k] = prod + 0.0f;
      }
      break;
    case kEpMulP:
    case kEpScale:
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const float f = kind == kEpScale ? __uint_as_float(imm) : p[k], prod = y[k] * f;
        odd |= TopField(__float_as_uint(y[k])) || TopField(__float_as_uint(f)) ||
               TopField(__float_as_uint(prod)) ||
               ProductOdd(__float_as_uint(y[k]), __float_as_uint(f), __float_as_uint(prod));
        r[k] = prod + 0.0f;
      }
      break;
    default:  // sums, copies, ReLU
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const float b = kind == kEpAdd ? x2[k] : kind == kEpAddP ? p[k] : 0.0f;
        const float sum = (y[k] + b) + 0.0f;
        odd |= TopField(__float_as_uint(y[k])) || TopField(__float_as_uint(b)) ||
               TopField(__float_as_uint(sum));
        r[k] = kind == kEpRelu ? (sum > 0.0f ? sum : 0.0f) : sum;
      }
      break;
  }
  if (odd) {
#pragma unroll 1
    for (int k = 0; k < 4; ++k)
      r[k] = __uint_as_float(EpApply(kind, imm, __float_as_uint(y[k]), __float_as_uint(x2[k]),
                                     __float_as_uint(p[k]), t));
  }
  y = r;
}

// Reads one dword of every 64-byte line of a kernel argument at once, with
// one wait for all, so the argument reads that follow (scattered over the
// structure, many behind branches) hit the scalar cache instead of each
// waiting for memory in turn.
__device__ __forceinline__ void TouchArgs(const void* args, size_t bytes) {
  const uint32_t* p = static_cast<const uint32_t*>(args);
  uint32_t x = 0;
  for (size_t i = 0; i < bytes / 64; ++i) x ^= p[i * 16];
  asm volatile("; args touched %0" ::"s"(x));
}

// Largest value over the 16 lanes of each DPP row (lanes 16r .. 16r + 15):
// xor 1 and xor 2 (quad permutes), the half-row mirror (lane i and 7 - i of
// each 8), the row mirror (i and 15 - i).  All four are register moves of
// the DPP unit, with no trip through LDS.
__device__ __forceinline__ uint32_t RowMax16(uint32_t x) {
  x = max(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0xB1, 0xF, 0xF, false));
  x = max(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x4E, 0xF, 0xF, false));
  x = max(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x141, 0xF, 0xF, false));
  x = max(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x140, 0xF, 0xF, false));
  return x;
}
// ... over the 32 lanes of each half of the wave: the two rows of a half
// meet through one swizzle (bit mode, lane i reads lane i ^ 16 of its 32).
__device__ __forceinline__ uint32_t HalfMax32(uint32_t x) {
  x = RowMax16(x);
  return max(x, (uint32_t)__builtin_amdgcn_ds_swizzle((int)x, 0x401F));
}

// QuantizeBlock for one token: values[32] -> bytes and scale byte.
// emax = largest exponent field (0 -> scale byte 127).
__device__ __forceinline__ uint32_t ScaleByteOf(uint32_t emax) { return emax == 0 ? 127u : emax; }

// QuantizeElement (tools/iss/lane.cpp:384-404) in FP32 hardware arithmetic,
// bit for bit, for emax at least the value's exponent field e (emax is the
// block's largest field):
//  * e in 1..254: the significand shifted right emax - e + 17 places with
//    round-to-nearest-even is |v| * 2^(133 - emax) rounded to an integer
//    the same way.  The product is exact in FP32 (it is below 2^7), or
//    below 2^-126 where both give 0; saturation to [-128, 127] matches the
//    NPU's (+128 and above -> 127, -128 and below -> -128).
//  * e = 0 (zero, subnormal): 0, as the integer path takes the significand
//    as 0.
//  * e = 255 (inf, NaN): the integer path shifts the significand with its
//    leading 1 by 17 places (emax is 255); the same bits with field 254 and
//    emax 254 give that value.
// About 10 instructions against the integer path's 22.
__device__ __forceinline__ uint8_t QuantizeElementHw(uint32_t value, uint32_t emax) {
  const uint32_t e = ExpField(value);
  const bool top = e == 255u;
  const uint32_t bits = top ? value - 0x00800000u : (e == 0u ? 0u : value);
  const int32_t sh = 133 - (int32_t)(top ? emax - 1u : emax);
  const float q = __builtin_amdgcn_fmed3f(__builtin_rintf(__builtin_amdgcn_ldexpf(__uint_as_float(bits), sh)),
                                          -128.0f, 127.0f);
  return (uint8_t)(int32_t)q;
}

// Block blk of column col, plane l of W8 panels (w: the panels): the dot
// product of the 32 int8 codes at a32 with the plane's nibble values (each
// decoded from its FP6 code v / 2), and the plane's scale byte.
typedef uint32_t W8Codes __attribute__((ext_vector_type(6)));
typedef _Float16 W8Halves __attribute__((ext_vector_type(32)));
__device__ __forceinline__ int32_t W8PanelDot(const GemmArgs& g, const uint8_t* w, uint32_t col,
                                              uint32_t blk, uint32_t l, const uint8_t* a32,
                                              uint32_t* wscale) {
  const uint32_t cc = col % kPanelCols, b = blk % 2, i = (b * 2 + l) * kPanelCols + cc;
  const uint8_t* chunk = w + ((size_t)(col / kPanelCols) * g.w_steps + blk / 2) * kW8Chunk;
  const uint4 d0 = *reinterpret_cast<const uint4*>(chunk + i * 16);
  const uint2 d1 = *reinterpret_cast<const uint2*>(chunk + kW8Part8 + i * 8);
  const W8Codes codes = {d0.x, d0.y, d0.z, d0.w, d1.x, d1.y};
  const W8Halves v = __builtin_amdgcn_cvt_scalef32_pk32_f16_fp6(codes, 1.0f);
  *wscale = (chunk[kW8Scales + (b * 32 + cc % 32) * 4 + 2 * (cc / 32) + l] + (l ? 5u : 1u)) & 0xFFu;
  int32_t sum = 0;
#pragma unroll
  for (int k = 0; k < 32; ++k)
    sum += (int32_t)(int8_t)a32[k] * (int32_t)(float)(v[k] * (_Float16)2.0f);
  return sum;
}

// Exact recomputation of one output of a linear layer over DDR words (the
// NPU's ordered fold, tools/iss/gemm_array.cpp:123-147 as emitted per
// tools/compiler/kernels.cpp:343-395: pieces, then planes, then blocks),
// starting from acc.
// kLayout: 0 reads g.w_panels and g.w_fp6, 1 DDR words, 2 panels, 3 W8
// panels (known to the caller).
template <int kLayout = 0>
__device__ __forceinline__ uint32_t SlowLinear(const GemmArgs& g, const uint8_t* a,
                                               const uint8_t* w0, const uint8_t* w1, uint32_t acc,
                                               uint32_t row, uint32_t col) {
  const bool fp6 = kLayout == 0 ? g.w_fp6 != 0 : kLayout == 3;
  const bool panels = kLayout == 0 ? g.w_panels != 0 : kLayout == 2;
  const uint32_t quad = row >> 2, t = row & 3;
  const WLaneOff wo = WLane(g, col, panels);
  for (uint32_t p = 0; p < g.n_pieces; ++p)
    for (uint32_t l = 0; l < g.n_planes; ++l)
      for (uint32_t b = 0; b < g.piece_kb[p]; ++b) {
        const uint32_t blk = g.piece_off[p] + b, mode = g.modes[l];
        const uint8_t* aw = a + ((size_t)quad * g.a_row + blk) * kDdrWord;
        const uint8_t* wp = l ? w1 : w0;
        if (fp6) {
          uint32_t ws = 0;
          const int32_t dot = W8PanelDot(g, wp, col, blk, l, aw + t * 32, &ws);
          acc = AddBits(acc, BlockValue(dot, aw[128 + t], ws, mode));
          continue;
        }
        const uint8_t* codes;
        uint32_t wscale;
        if (panels) {
          codes = wp + wo.codes + WBlockCodes(g, blk, true);
          wscale = wp[wo.scale + WBlockScale(g, blk, true) + wo.shift / 8];
        } else {  // the column's 16 code bytes and its scale byte in the block's word
          const uint8_t* ww = wp + ((size_t)(col >> 3) * g.kb_total + blk) * kDdrWord;
          codes = ww + (col & 7) * 16;
          wscale = ww[128 + (col & 7)];
        }
        int32_t sum = 0;
        for (uint32_t k = 0; k < 32; ++k) {
          const uint32_t byte = codes[k >> 1];
          sum += (int32_t)(int8_t)aw[t * 32 + k] * WeightValue((k & 1) ? (byte >> 4) : byte, mode);
        }
        acc = AddBits(acc, BlockValue(sum, aw[128 + t], wscale, mode));
      }
  return acc;
}

// SlowLinear for MXFP8 E4M3 activations over one MXFP4 plane (DDR words or
// weight panels): each block's exact sum of Fp8Int(a) x WeightValue(w),
// BlockValueFp8, folded with the reference's add in its order.
__device__ __forceinline__ uint32_t SlowLinearFp8(const GemmArgs& g, const uint8_t* a,
                                                  const uint8_t* w, uint32_t acc, uint32_t row,
                                                  uint32_t col) {
  const bool panels = g.w_panels != 0;
  const uint32_t quad = row >> 2, t = row & 3;
  const WLaneOff wo = WLane(g, col, panels);
  for (uint32_t p = 0; p < g.n_pieces; ++p)
    for (uint32_t b = 0; b < g.piece_kb[p]; ++b) {
      const uint32_t blk = g.piece_off[p] + b;
      const uint8_t* aw = a + ((size_t)quad * g.a_row + blk) * kDdrWord;
      const uint8_t* codes;
      uint32_t wscale;
      if (panels) {
        codes = w + wo.codes + WBlockCodes(g, blk, true);
        wscale = w[wo.scale + WBlockScale(g, blk, true) + wo.shift / 8];
      } else {
        const uint8_t* ww = w + ((size_t)(col >> 3) * g.kb_total + blk) * kDdrWord;
        codes = ww + (col & 7) * 16;
        wscale = ww[128 + (col & 7)];
      }
      int32_t sum = 0;
      for (uint32_t k = 0; k < 32; ++k) {
        const uint32_t byte = codes[k >> 1];
        sum += Fp8Int(aw[t * 32 + k]) * WeightValue((k & 1) ? (byte >> 4) : byte, kModeFp4);
      }
      acc = AddBits(acc, BlockValueFp8(sum, aw[128 + t], wscale));
    }
  return acc;
}

// Starts kT accumulator tiles (16 values per lane each) from C.  A tile's
// 16 loads issue together, before their first wait: with a branch around each load
// the compiler waits for each in turn (measured on a 128 x 256 tile, 64
// values per lane: 19 us against 2).  An element outside the m x n output
// reads C's first word and starts from +0.  at(j, r, row, col) names value
// r of tile j.  Returns whether a start value's exponent field exceeds 252.
template <int kT, typename Acc, typename At>
__device__ __forceinline__ bool AccFromC(Acc (&acc)[kT], const uint32_t* c, uint32_t m,
                                         uint32_t n, At at) {
  bool unsafe = false;
#pragma unroll
  for (int j = 0; j < kT; ++j) {
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      uint32_t row, col;
      at(j, r, row, col);
      acc[j][r] = __uint_as_float(c[row < m && col < n ? (size_t)row * n + col : 0]);
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      uint32_t row, col;
      at(j, r, row, col);
      const uint32_t v = row < m && col < n ? __float_as_uint(acc[j][r]) : 0u;
      acc[j][r] = __uint_as_float(v);
      unsafe |= ExpField(v) > 252u;
    }
    __builtin_amdgcn_sched_barrier(0);  // one tile's loads in flight at a time
  }
  return unsafe;
}

// The lane's index within its wave, read afresh where it is called: the
// asm is opaque to the compiler, so lane-derived addresses computed from it
// are not hoisted out of a loop to stay live (and spill) across its body.
__device__ __forceinline__ uint32_t LaneNow() {
  uint32_t l;
  asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(l));
  return l;
}

}  // namespace hb
