// GEMM kernels for gfx950: the hotarubi GEMM instruction (ISS images) and
// the linear layer it is emitted for (DDR words), both exact.
//
// Arithmetic (tools/iss/gemm_array.cpp:51-69, 99-110): per output and per
// 32-element K block, the block value s * 2^(ea + ew + SBIAS) with s the exact
// integer dot product, folded into an FP32 accumulator in block order.
//
// Matrix-core mapping.  Per K block the tile's operands are staged in LDS as
// f16: A' = q * 2^d with d = ea - 130 held to [-14, 5], and W' = v, the
// unscaled weight value.  q (int8) and v (4-bit value) have at most 8
// significant bits, so A' and W' are exact, normal f16 values.  One
// v_mfma_f32_16x16x32_f16 with a zero accumulator then covers exactly one K
// block, and every product and every partial sum it forms is an integer
// multiple of 2^d below 2^17 of that unit: all exactly representable, so the
// MFMA returns the exact block value up to the scales.  The ordered fold is
// one fma per output and block, acc = fma(value, 2^(ew+ea-d-254+SBIAS), acc)
// with ea - d = 130: a single rounding of an exact sum (FTZ mode), which is
// the NPU's RNE add for normal operands; a -0 result can only appear where
// the NPU has +0 and is fixed once after the fold.  Where a row's ea lies
// outside [116, 135] the rest of its exponent, 2^(ea-130-d), multiplies the
// block value first (exact): such steps are flagged and take a second copy
// of the fold.
//
// The argument needs every scale byte of the tile in [70, 179] (exponents
// -57..52) and |initial C| < 2^126: then operands and products stay normal
// and the fold cannot overflow (steps <= 8192).  A tile that sees anything
// else recomputes itself with the integer routines of hb_fp32.h, so the
// result is bit-exact for every input.
#include <type_traits>

#include "hb_device.h"
#include "hb_internal.h"

namespace hb {
namespace {

typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kThreads = 512;  // 8 waves: 4 stage A, 4 stage W, all fold
constexpr uint32_t kCheck = 8;  // stages between two looks at the rows' scales (even)
constexpr uint32_t kSafeLo = 70, kSafeHi = 179;
// What a kernel knows of the planes' modes: all FP4; W8 hi then lo; anything.
enum : int { kFmtFp4, kFmtW8, kFmtAny };
constexpr int32_t kAUnit = 130, kAMin = -14, kAMax = 5;  // d = ea - kAUnit, held to [kAMin, kAMax]

// Tile geometry.  kBM x kBN outputs per workgroup; the 8 waves tile it as
// kWaveM x kWaveN with a kTM x kTN wave tile of 16x16 MFMA tiles.  kC: K
// blocks staged per barrier.  A staging thread has one unit per stage: half a
// row-block of A (16 of its 32 bytes), or a column-block of W (16 bytes).
template <int kBM_, int kBN_, int kWaveM, int kC_, int kWavesPerSimd_>
struct Tile {
  static constexpr int kWavesPerSimd = kWavesPerSimd_;
  static constexpr int kBM = kBM_, kBN = kBN_, kC = kC_;
  static constexpr int kWaveN = 8 / kWaveM;
  static constexpr int kTM = kBM / kWaveM, kTN = kBN / kWaveN;
  static constexpr int kTI = kTM / 16, kTJ = kTN / 16;
  static constexpr int kAUnits = kBM * 2 * kC, kWUnits = kBN * kC;
  static constexpr int kOutRow = kBN + 4;  // floats per row of the staged outputs
  static_assert(kTM % 16 == 0 && kTN % 16 == 0, "whole MFMA tiles");
  static_assert(kAUnits <= 256 && kWUnits <= 256, "a unit per staging thread");
};

// LDS: two stages of kC blocks.  A block's operands lie as the MFMAs read
// them: 16 rows (columns) of one tile are 64 slots of 16 bytes (8 f16), slot
// Slot(kq, row) for K elements 8 kq .. + 7, so a wave's read covers 64
// consecutive slots, each once.  Rows of kq 2, 3 are swapped by eights: a
// staging lane pair writes kq 0 and 2 (or 1 and 3) of a row at once, and the
// 16 lanes of a write then use 16 different bank groups.
template <class T>
struct Lds {
  static constexpr int kBM = T::kBM, kBN = T::kBN, kC = T::kC;
  union {
    struct {
      uint4 a[2][kC][kBM / 16][64];
      uint4 w[2][kC][kBN / 16][64];
    };
    struct {  // after the K loop
      float out[kBM * T::kOutRow];
      uint64_t act[512];  // activation half of TBUF
    };
  };
  float fw[2][kC][kBN];  // 2^(ew + SBIAS + kAUnit - 254) per column and block
  float fr[2][kC][kBM];  // 2^(ea - kAUnit - d) per row and block
  uint32_t unsafe, wide;
};
__device__ __forceinline__ uint32_t Slot(uint32_t kq, uint32_t row16) {
  return kq * 16 + (row16 ^ ((kq & 2) * 4));
}

// A stage of the fold: up to kC consecutive blocks of one piece and plane,
// `live` of them; a stage past the end has none.  Its dead blocks repeat the
// last live one with A staged as zeros, adding +0.
struct Stage {
  uint32_t l, blk, live;
};
// The stages in fold order (pieces outer, planes inner).
template <bool kMulti, int kC>
struct Cursor {
  uint32_t p = 0, l = 0, b = 0;
  __device__ __forceinline__ Stage Take(const GemmArgs& g) {
    const uint32_t kb = g.piece_kb[kMulti ? p : 0], left = b < kb ? kb - b : 0u;
    const Stage s{l, g.piece_off[kMulti ? p : 0] + min(b, kb - 1), min(left, (uint32_t)kC)};
    b += kC;
    if (b >= kb) {  // the next plane or piece; past the last, b stays at kb or more
      if (l + 1 < g.n_planes) {
        ++l;
        b = 0;
      } else if (kMulti && p + 1 < g.n_pieces) {
        ++p;
        l = b = 0;
      }
    }
    return s;
  }
};
template <int kC>
__device__ __forceinline__ uint32_t StageCount(const GemmArgs& g) {
  uint32_t n = 0;
  for (uint32_t p = 0; p < g.n_pieces; ++p) n += (g.piece_kb[p] + kC - 1) / kC;
  return n * g.n_planes;
}

template <bool kLinear>
__device__ __forceinline__ const uint8_t* AWord(const GemmArgs& g, const uint8_t* a, uint32_t q,
                                                uint32_t blk) {
  if (kLinear) return a + ((size_t)q * g.a_row + blk) * kDdrWord;
  return a + (size_t)((g.a_base + q * g.a_stride + blk) & (kAbufDepth - 1)) * kAbufWord;
}

template <bool kLinear>
__device__ __forceinline__ const uint8_t* WWord(const GemmArgs& g, const uint8_t* w, uint32_t grp,
                                                uint32_t blk) {
  if (kLinear) return w + ((size_t)grp * g.kb_total + blk) * kDdrWord;
  return w + (size_t)((g.w_base + grp * g.w_stride + blk) & (kWbufDepth - 1)) * kWbufWord;
}

// FP32 bits of the C element (row, col) of the tile's global index space.
template <bool kLinear>
__device__ __forceinline__ uint32_t* CElem(const GemmArgs& g, uint32_t* c, uint32_t row,
                                           uint32_t col) {
  if (kLinear) return c + (size_t)row * g.n + col;
  const uint32_t word = (g.c_base + (row >> 2) * g.groups + (col >> 3)) & (kFbufDepth - 1);
  return c + (size_t)word * 32 + (row & 3) * 8 + (col & 7);
}

// Raw operand bytes of one stage, as one thread stages them, and the aligned
// dword that holds their scale byte.  Loads are issued unconditionally: rows
// and columns past the edge of the layer (and units past the stage's) read
// the last valid one instead, which only feeds outputs that are never stored
// (rows of a GEMM depend on their own A row, columns on their own W column).
struct Staged {
  u32x4 v;
  uint32_t scale;
};

// Where a thread's staging unit lies: unit u of A is half u % 2 of row u / 2
// % kBM of the stage's block u / (2 kBM); unit u of W is column u % kBN of
// block u / kBN.  (8 consecutive lanes read the 128 bytes of a quad's, or a
// column group's, block.)  Block blk of the unit's operand lies at
// (blk >> half) * chunk + (blk & half) * codes from the layer's base, its
// scale dwords at scales in place of codes (DDR words, or panels of two
// blocks a chunk: WBlockCodes, WBlockScale without a branch).
template <bool kLinear, class T>
struct Lane {
  bool w;           // stages W (wave-uniform)
  uint32_t u;       // the unit
  uint32_t block;   // its block of the stage
  uint32_t codes, scale, shift;  // its byte offsets in a block's words (linear); scale bit
  uint32_t line;    // its quad or column group (instruction level)
  uint32_t half, chunk, c_step, s_step;
  __device__ __forceinline__ Lane(const GemmArgs& g, uint32_t q0, uint32_t g0) {
    w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8) != 0;
    u = min(threadIdx.x & 255u, (w ? T::kWUnits : T::kAUnits) - 1u);
    half = kLinear && w && g.w_panels ? 1u : 0u;
    chunk = half ? kPanelChunk : kDdrWord;
    c_step = kPanelCols * 16;
    s_step = kPanelCols;
    if (w) {
      const uint32_t col = u % T::kBN, grp = min(g0 + (col >> 3), g.groups - 1), cl = col & 7;
      block = u / T::kBN;
      line = grp;
      if (kLinear) {
        const WLaneOff wo = WLane(g, grp * 8 + cl);
        codes = wo.codes;
        scale = wo.scale;
        shift = wo.shift;
      } else {
        codes = cl * 16;
        scale = 128 + (cl & 4);
        shift = 8 * (cl & 3);
      }
    } else {
      const uint32_t r = u / 2 % T::kBM, quad = min(q0 + (r >> 2), g.quads - 1);
      block = u / (2 * T::kBM);
      line = quad;
      codes = (kLinear ? quad * g.a_row * kDdrWord : 0u) + (r & 3) * 32 + (u % 2) * 16;
      scale = (kLinear ? quad * g.a_row * kDdrWord : 0u) + 128;
      shift = 8 * (r & 3);
    }
  }
};

// Loads the thread's unit of a stage.
template <bool kLinear, class T>
__device__ __forceinline__ void LoadStage(const GemmArgs& g, const uint8_t* a, const uint8_t* w0,
                                          const uint8_t* w1, const Lane<kLinear, T>& ln,
                                          const Stage& s, Staged& st) {
  const uint32_t last = max(s.live, 1u) - 1, blk = s.blk + min(ln.block, last);
  const uint8_t* base = ln.w ? (s.l ? w1 : w0) : a;
  if (kLinear) {
    const uint32_t at = (blk >> ln.half) * ln.chunk, odd = blk & ln.half;
    st.v = *reinterpret_cast<const u32x4*>(base + (size_t)(ln.codes + at + odd * ln.c_step));
    st.scale = *reinterpret_cast<const uint32_t*>(base + (size_t)(ln.scale + at + odd * ln.s_step));
  } else if (ln.w) {
    const uint8_t* word = WWord<false>(g, base, ln.line, blk);
    st.v = *reinterpret_cast<const u32x4*>(word + ln.codes);
    st.scale = *reinterpret_cast<const uint32_t*>(word + ln.scale);
  } else {  // ISS ABUF words are 132 B: only 4-byte aligned
    const uint8_t* word = AWord<false>(g, base, ln.line, blk);
    const uint32_t* src = reinterpret_cast<const uint32_t*>(word + ln.codes);
#pragma unroll
    for (int k = 0; k < 4; ++k) st.v[k] = src[k];
    st.scale = *reinterpret_cast<const uint32_t*>(word + ln.scale);
  }
}

// A byte n under the f16 exponent byte 0x64 is exactly 1024 + n.
// perm(0x64646464, x, Sel(i, j)) is the f16 pair {1024 + byte i, 1024 + byte j}.
constexpr uint32_t Sel(uint32_t i, uint32_t j) { return 0x04000400u | i | (j << 16); }
__device__ __forceinline__ f16x2 Pair(uint32_t x, uint32_t sel) {
  return __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(0x64646464u, x, sel));
}
__device__ __forceinline__ uint32_t Bits(f16x2 v) { return __builtin_bit_cast(uint32_t, v); }

// What a staging thread has seen: a scale byte outside the window the
// matrix-core path is exact for, or a row whose ea lies outside f16's.
struct Seen {
  bool unsafe = false, wide = false;
};

// Converts a stage into LDS buffer `buf`: A scaled to f16, W as unscaled f16
// weight integers (FP4 codes by v_cvt_scalef32_pk_f16_fp4, nibbles by the
// perm above), and the scale factors.  A W8 byte holds two K positions, so a
// W8 block's elements come out in the order 0,2,1,3 of each 4; A is staged in
// the same order for it (a block's sum does not depend on the order).
template <int kFmt, bool kLinear, class T>
__device__ __forceinline__ void StoreStage(const GemmArgs& g, const Lane<kLinear, T>& ln,
                                           const Stage& s, const Staged& st, Lds<T>& lds,
                                           uint32_t buf, Seen& seen) {
  // the plane's mode (a W8 layer's planes are hi, lo)
  const uint32_t mode = kFmt == kFmtFp4  ? (uint32_t)kModeFp4
                        : kFmt == kFmtW8 ? (s.l ? (uint32_t)kModeW8Lo : (uint32_t)kModeW8Hi)
                                         : (s.l ? g.modes[1] : g.modes[0]);
  const bool fp4 = mode == kModeFp4;
  const uint32_t e = __builtin_amdgcn_ubfe(st.scale, ln.shift, 8);
  seen.unsafe |= e - kSafeLo > kSafeHi - kSafeLo;
  if (!ln.w) {
    if (T::kAUnits < 256 && (threadIdx.x & 255u) >= (uint32_t)T::kAUnits) return;
    const uint32_t s01 = fp4 ? Sel(0, 1) : Sel(0, 2), s23 = fp4 ? Sel(2, 3) : Sel(1, 3);
    const uint32_t r = ln.u / 2 % T::kBM, h = ln.u % 2;
    const int32_t d = min(max((int32_t)e - kAUnit, kAMin), kAMax);
    // f16 2^d and -1152 * 2^d: fma(1024 + q + 128, 2^d, -1152 * 2^d) = q * 2^d
    const uint32_t live = ln.block < s.live ? 0xFFFFFFFFu : 0u;
    const uint32_t d2 = __umul24((uint32_t)(d + 15), 0x000400u) * 0x00010001u;
    const f16x2 f = __builtin_bit_cast(f16x2, d2 & live);
    const f16x2 c = __builtin_bit_cast(f16x2, ((d2 + 0x28002800u) | 0x80808080u) & live);
    uint32_t o[8];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const uint32_t x = st.v[k] ^ 0x80808080u;
      o[2 * k] = Bits(__builtin_elementwise_fma(Pair(x, s01), f, c));
      o[2 * k + 1] = Bits(__builtin_elementwise_fma(Pair(x, s23), f, c));
    }
    uint4* tile = lds.a[buf][ln.block][r / 16];
    tile[Slot(2 * h, r % 16)] = uint4{o[0], o[1], o[2], o[3]};
    tile[Slot(2 * h + 1, r % 16)] = uint4{o[4], o[5], o[6], o[7]};
    const int32_t rest = (int32_t)e - kAUnit - d;
    lds.fr[buf][ln.block][r] = __uint_as_float((uint32_t)(rest + 127) << 23);
    seen.wide |= rest != 0;
  } else {
    if (T::kWUnits < 256 && (threadIdx.x & 255u) >= (uint32_t)T::kWUnits) return;
    const uint32_t col = ln.u % T::kBN;
    uint4* tile = lds.w[buf][ln.block][col / 16];
    if (fp4) {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const uint32_t v = st.v[k];
        tile[Slot(k, col % 16)] =
            uint4{Bits(__builtin_amdgcn_cvt_scalef32_pk_f16_fp4(v, 2.0f, 0)),
                  Bits(__builtin_amdgcn_cvt_scalef32_pk_f16_fp4(v, 2.0f, 1)),
                  Bits(__builtin_amdgcn_cvt_scalef32_pk_f16_fp4(v, 2.0f, 2)),
                  Bits(__builtin_amdgcn_cvt_scalef32_pk_f16_fp4(v, 2.0f, 3))};
      }
    } else {
      const uint32_t flip = mode == kModeW8Hi ? 0x88888888u : 0u;
      const _Float16 bias = mode == kModeW8Hi ? (_Float16)1032.0f : (_Float16)1024.0f;
      const f16x2 sub = {bias, bias};
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const uint32_t v = st.v[k] ^ flip;
        const uint32_t ev = v & 0x0F0F0F0Fu, od = (v >> 4) & 0x0F0F0F0Fu;
        tile[Slot(k, col % 16)] =
            uint4{Bits(Pair(ev, Sel(0, 1)) - sub), Bits(Pair(od, Sel(0, 1)) - sub),
                  Bits(Pair(ev, Sel(2, 3)) - sub), Bits(Pair(od, Sel(2, 3)) - sub)};
      }
    }
    lds.fw[buf][ln.block][col] =
        __uint_as_float((uint32_t)((int32_t)e + ScaleBias(mode) + kAUnit - 127) << 23);
  }
}

// Exact integer recomputation of one output (the NPU's arithmetic verbatim).
template <bool kLinear>
__device__ __forceinline__ uint32_t SlowOutput(const GemmArgs& g, const uint8_t* a,
                                               const uint8_t* w0, const uint8_t* w1, uint32_t acc,
                                               uint32_t row, uint32_t col) {
  if (kLinear) return SlowLinear(g, a, w0, w1, acc, row, col);
  const uint32_t quad = row >> 2, t = row & 3, grp = col >> 3, cl = col & 7;
  for (uint32_t p = 0; p < g.n_pieces; ++p) {
    for (uint32_t l = 0; l < g.n_planes; ++l) {
      const uint32_t mode = g.modes[l];
      for (uint32_t b = 0; b < g.piece_kb[p]; ++b) {
        const uint32_t blk = g.piece_off[p] + b;
        const uint8_t* aw = AWord<kLinear>(g, a, quad, blk);
        const uint8_t* ww = WWord<kLinear>(g, l ? w1 : w0, grp, blk);
        int32_t sum = 0;
        for (uint32_t k = 0; k < 32; ++k) {
          const uint32_t byte = ww[cl * 16 + (k >> 1)];
          sum += (int32_t)(int8_t)aw[t * 32 + k] * WeightValue((k & 1) ? (byte >> 4) : byte, mode);
        }
        acc = AddBits(acc, BlockValue(sum, aw[128 + t], ww[128 + cl], mode));
      }
    }
  }
  return acc;
}

// The exact tile kernel.  A stage is kC K blocks; while a stage is folded,
// the raw bytes of the next two are on their way into registers; the next one
// is converted into the other LDS buffer: one barrier per stage.  Per block
// and 16x16 tile one MFMA with a zero accumulator gives s * 2^d exactly, and
// the fold is an fma per output.
//
// Bound: no one unit.  A 16x16x32 MFMA takes 16.5 cycles and the 4 folds of
// its outputs as long; both together 23.3 where 3 waves of a SIMD take turns,
// 24.2 with 2, 37 with one (measured), so tiles leave room for 2 or 3
// workgroups per CU, and a 64 x 96 tile costs a SIMD 140 cycles per block.
// Next to that stands conversion: 5 instructions per 4 activations (an xor,
// two byte permutes, two packed f16 fmas; with bf16 operands, which have no
// packed arithmetic, it was 11) and one per 2 FP4 weights.  The K loop takes
// about 1.6 times the cycles of both; the LDS moves 65 KB per 64 x 96 tile
// and stage, 0.6 of its rate.
//
// Measured, one launch: 4512 x 960, K 2560, MXFP4 with the residual 129 -> 56
// us (14 of them MFMAs and folds); 2048 x 2304, K 768, W8 with MULP and ADDP
// 111 -> 45 us (8.5) (bf16 operands, 128 x 128 tiles of 4 waves, one block a
// barrier, and the ops in integers before).  The 64 x 96 tile's 80 registers
// spill 18 to 30 outside the MFMA loop (68 bytes a lane).
//
// The loop runs with the rows' factors fr left out, which are 1 for every
// ea in [116, 135]; every kCheck stages it looks whether a row had another,
// and then starts again with them.
template <bool kLinear, bool kMulti, int kFmt, class T>
__global__ __launch_bounds__(kThreads, T::kWavesPerSimd) void GemmTileKernel(GemmArgs g) {
  constexpr int kBM = T::kBM, kBN = T::kBN, kC = T::kC;
  __shared__ __attribute__((aligned(16))) Lds<T> lds;

  const uint8_t* a = g.a;
  const uint8_t* w0 = g.w[0];
  const uint8_t* w1 = g.w[1];
  uint32_t* c = g.c;
  uint8_t* q_out = g.q_out;
  const TileId tile = LogicalTile(g.gx, g.gy, g.gz);
  const uint32_t z = kLinear ? tile.z : 0u;  // layer of a batched linear launch
  if (kLinear) {
    a += z * g.a_batch;
    w0 += z * g.w_batch;
    w1 += z * g.w_batch;
    c += z * g.c_batch;
    if (q_out) q_out += z * g.q_batch;
  }

  const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const uint32_t wm = wave / T::kWaveN, wn = wave % T::kWaveN;
  const uint32_t row16 = lane & 15, kq = lane >> 4;
  const uint32_t q0 = tile.y * (kBM / 4), g0 = tile.x * (kBN / 8);
  const uint32_t row0 = q0 * 4, col0 = g0 * 8;

  const Lane<kLinear, T> ln(g, q0, g0);
  if (tid == 0) lds.unsafe = lds.wide = 0;

  // Output (i, j, v) of this lane: tile row wm*kTM + i*16 + kq*4 + v,
  // tile column wn*kTN + j*16 + row16 (16x16 MFMA accumulator layout).
  f32x4 acc[T::kTI][T::kTJ];
  Seen seen;
  auto start = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < T::kTI; ++i)
#pragma unroll
      for (int j = 0; j < T::kTJ; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (!g.acc) return;
#pragma unroll
    for (int i = 0; i < T::kTI; ++i)
#pragma unroll
      for (int j = 0; j < T::kTJ; ++j)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const uint32_t row = row0 + wm * T::kTM + i * 16 + kq * 4 + v;
          const uint32_t col = col0 + wn * T::kTN + j * 16 + row16;
          const bool in = (row >> 2) < g.quads && (col >> 3) < g.groups && (!kLinear || row < g.m);
          const uint32_t init = in ? *CElem<kLinear>(g, c, row, col) : 0u;
          seen.unsafe |= ExpField(init) > 252u;
          acc[i][j][v] = __uint_as_float(init);
        }
  };

  const uint32_t stages = StageCount<kC>(g);
  struct Operands {
    f16x8 a[T::kTI], w[T::kTJ];
    float fw[T::kTJ];
  };
  auto read = [&](uint32_t buf, int b, Operands& o) __attribute__((always_inline)) {
    const uint32_t slot = Slot(kq, row16);
#pragma unroll
    for (int j = 0; j < T::kTJ; ++j) {
      o.w[j] = __builtin_bit_cast(f16x8, lds.w[buf][b][wn * T::kTJ + j][slot]);
      o.fw[j] = lds.fw[buf][b][wn * T::kTN + j * 16 + row16];
    }
#pragma unroll
    for (int i = 0; i < T::kTI; ++i)
      o.a[i] = __builtin_bit_cast(f16x8, lds.a[buf][b][wm * T::kTI + i][slot]);
  };
  // The fold of one stage; kWide: with the rows' own factors.
  auto fold = [&](uint32_t buf, auto wide) __attribute__((always_inline)) {
    constexpr bool kWide = decltype(wide)::value;
#pragma unroll
    for (int b = 0; b < kC; ++b) {
      Operands x;
      read(buf, b, x);
#pragma unroll
      for (int i = 0; i < T::kTI; ++i) {
        f32x4 fr, bv[T::kTJ];
        if (kWide)
          fr = *reinterpret_cast<const f32x4*>(&lds.fr[buf][b][wm * T::kTM + i * 16 + kq * 4]);
#pragma unroll
        for (int j = 0; j < T::kTJ; ++j) {
          const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
          bv[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(x.a[i], x.w[j], zero, 0, 0, 0);
        }
#pragma unroll
        for (int j = 0; j < T::kTJ; ++j) {
          if (kWide) bv[j] = bv[j] * fr;
#pragma unroll
          for (int v = 0; v < 4; ++v)
            acc[i][j][v] = __builtin_fmaf(bv[j][v], x.fw[j], acc[i][j][v]);
        }
      }
      // Anchor the fold here: left free, the compiler sinks every block's
      // (pure) folds to the end of the stage, keeping all the blocks'
      // values live at once.  The empty asm emits no instruction.
#pragma unroll
      for (int i = 0; i < T::kTI; ++i)
#pragma unroll
        for (int j = 0; j < T::kTJ; ++j) asm volatile("" : "+v"(acc[i][j]));
      if (b + 1 < kC) __builtin_amdgcn_sched_barrier(0);
    }
  };
  // The whole fold; false if it met a row that needs its factor (without
  // kWide).  Two stages a round, without a branch between the loads and their
  // use, so that the loads of two stages stay in flight across the barriers.
  auto run = [&](auto wide) __attribute__((always_inline)) {
    constexpr bool kWide = decltype(wide)::value;
    Cursor<kMulti, kC> cursor;
    Stage cur[2];
    Staged raw[2];
    auto load = [&](int i) __attribute__((always_inline)) {
      cur[i] = cursor.Take(g);
      LoadStage<kLinear, T>(g, a, w0, w1, ln, cur[i], raw[i]);
    };
    auto store = [&](int i, uint32_t buf) __attribute__((always_inline)) {
      StoreStage<kFmt, kLinear, T>(g, ln, cur[i], raw[i], lds, buf, seen);
    };
    load(0);
    load(1);
    start();
    store(0, 0);
    load(0);
    __syncthreads();
    for (uint32_t s = 0; s + 1 < stages; s += 2) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        fold(i, wide);
        store(1 - i, 1 - i);
        load(1 - i);
        if (!kWide && i == 1 && seen.wide && s % kCheck == 0) lds.wide = 1;
        __syncthreads();
      }
      // (uniform: the flag was raised before the barrier, and every wave is
      // past the next one before it can be raised again)
      if (!kWide && s % kCheck == 0 && __builtin_amdgcn_readfirstlane(lds.wide) != 0) return false;
    }
    if (stages & 1) fold(0, wide);
    if (!kWide && seen.wide) lds.wide = 1;
    __syncthreads();
    return kWide || __builtin_amdgcn_readfirstlane(lds.wide) == 0;
  };
  if (!run(std::false_type{})) run(std::true_type{});
  if (seen.unsafe) lds.unsafe = 1;
  if (kLinear && g.tbuf != nullptr)
    for (uint32_t i = tid; i < 512; i += kThreads) lds.act[i] = g.tbuf[512 + i];
  // The outputs meet row by row in the staging buffers, -0 as +0.
#pragma unroll
  for (int i = 0; i < T::kTI; ++i)
#pragma unroll
    for (int j = 0; j < T::kTJ; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v)
        lds.out[(wm * T::kTM + i * 16 + kq * 4 + v) * T::kOutRow + wn * T::kTN + j * 16 + row16] =
            acc[i][j][v] + 0.0f;
  __syncthreads();
  const bool slow = lds.unsafe != 0;

  // Epilogue: 4 consecutive columns of a row per thread and round, the ops
  // in order, C as 16-byte stores; a row's 32-column block is 8 consecutive
  // lanes, whose largest exponent field meets in three register moves.
  const uint32_t rows4 = g.quads * 4, n = g.groups * 8;
  const bool c16 = (reinterpret_cast<uintptr_t>(c) & 15u) == 0;  // uniform
  constexpr uint32_t kUnits = kBM * kBN / 4;
#pragma unroll 1
  for (uint32_t u = tid; u < kUnits; u += kThreads) {
    const uint32_t r = u / (kBN / 4), cc = u % (kBN / 4) * 4;
    const uint32_t row = row0 + r, col = col0 + cc;
    const bool in = row < rows4 && col < n;
    f32x4 y = *reinterpret_cast<const f32x4*>(&lds.out[r * T::kOutRow + cc]);
    if (slow && in) {  // the tile exactly
#pragma unroll 1
      for (uint32_t k = 0; k < 4; ++k) {
        uint32_t init = 0;
        if (g.acc && (!kLinear || row < g.m)) init = *CElem<kLinear>(g, c, row, col + k);
        y[k] = __uint_as_float(SlowOutput<kLinear>(g, a, w0, w1, init, row, col + k));
      }
    }
    if (kLinear) {
      for (uint32_t o = 0; o < g.n_ops; ++o) {
        const uint32_t kind = g.op_kind[o];
        f32x4 x2 = {0.f, 0.f, 0.f, 0.f}, p = x2;
        if ((kind == kEpAdd || kind == kEpActMul) && in && row < g.m) {
          const uint32_t* v = g.op_x2[o] + z * g.op_x2_batch[o] + (size_t)row * g.n + col;
          if ((reinterpret_cast<uintptr_t>(g.op_x2[o] + z * g.op_x2_batch[o]) & 15u) == 0 &&
              g.n % 4 == 0) {
            x2 = *reinterpret_cast<const f32x4*>(v);
          } else {
#pragma unroll
            for (int k = 0; k < 4; ++k) x2[k] = __uint_as_float(v[k]);
          }
        }
        if ((kind == kEpAddP || kind == kEpMulP) && in) {
          const uint32_t* v = g.op_vec[o] + z * g.op_vec_batch[o] + col;
#pragma unroll
          for (int k = 0; k < 4; ++k) p[k] = __uint_as_float(v[k]);
        }
        EpApply4(kind, g.op_imm[o], y, x2, p, lds.act);
      }
    }
    if (in && (!kLinear || (row < g.m && g.c != nullptr))) {
      uint32_t* dst = CElem<kLinear>(g, c, row, col);
      if (c16) {
        *reinterpret_cast<f32x4*>(dst) = y;
      } else {
#pragma unroll
        for (int k = 0; k < 4; ++k) dst[k] = __float_as_uint(y[k]);
      }
    }
    if (kLinear && q_out != nullptr) {  // MXINT8 requantize (n % 32 == 0)
      uint32_t e = 0;
#pragma unroll
      for (int k = 0; k < 4; ++k) e = max(e, ExpField(__float_as_uint(y[k])));
      e = max(e, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)e, 0xB1, 0xF, 0xF, false));
      e = max(e, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)e, 0x4E, 0xF, 0xF, false));
      e = max(e, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)e, 0x141, 0xF, 0xF, false));
      if (in) {
        uint8_t* word = q_out + ((size_t)(row >> 2) * (n >> 5) + (col >> 5)) * kDdrWord;
        uint32_t codes = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k)
          codes |= (uint32_t)QuantizeElementHw(__float_as_uint(y[k]), e) << (8 * k);
        const uint32_t part = (col >> 2) & 7;
        *reinterpret_cast<uint32_t*>(word + (row & 3) * 32 + part * 4) = codes;  // (4-aligned)
        if (part == 0) word[128 + (row & 3)] = (uint8_t)ScaleByteOf(e);
        if ((row & 3) == 0 && part >= 1 && part < 4)  // bytes 132..143
          *reinterpret_cast<uint32_t*>(word + 128 + 4 * part) = 0u;
      }
    }
  }
}

// An instruction whose output words wrap around FBUF (m/4 * n8 > 4096) writes
// some words more than once; with acc the later writers read what the earlier
// ones wrote.  This kernel keeps the reference's (g outer, q inner) order per
// FBUF word: one workgroup per word, one thread per element.
__global__ __launch_bounds__(32) void GemmAliasKernel(GemmArgs g) {
  const uint32_t total = g.quads * g.groups;
  const uint32_t i0 = blockIdx.x;
  uint32_t keys[16];
  uint32_t n = 0;
  for (uint32_t i = i0; i < total && n < 16; i += kFbufDepth)
    keys[n++] = (i % g.groups) * g.quads + i / g.groups;
  for (uint32_t x = 1; x < n; ++x) {  // ascending (g, q) order
    const uint32_t k = keys[x];
    uint32_t y = x;
    for (; y > 0 && keys[y - 1] > k; --y) keys[y] = keys[y - 1];
    keys[y] = k;
  }
  const uint32_t e = threadIdx.x, t = e >> 3, cl = e & 7;
  const uint32_t word = (g.c_base + i0) & (kFbufDepth - 1);
  uint32_t* elem = g.c + (size_t)word * 32 + e;
  const uint32_t mode = g.modes[0];
  for (uint32_t x = 0; x < n; ++x) {
    const uint32_t grp = keys[x] / g.quads, quad = keys[x] % g.quads;
    uint32_t acc = g.acc ? *elem : 0u;
    for (uint32_t b = 0; b < g.piece_kb[0]; ++b) {
      const uint8_t* aw = AWord<false>(g, g.a, quad, b);
      const uint8_t* ww = WWord<false>(g, g.w[0], grp, b);
      int32_t sum = 0;
      for (uint32_t k = 0; k < 32; ++k) {
        const uint32_t byte = ww[cl * 16 + (k >> 1)];
        sum += (int32_t)(int8_t)aw[t * 32 + k] * WeightValue((k & 1) ? (byte >> 4) : byte, mode);
      }
      acc = AddBits(acc, BlockValue(sum, aw[128 + t], ww[128 + cl], mode));
    }
    *elem = acc;
  }
}

}  // namespace

namespace {
template <bool kLinear, class T>
void LaunchTile(GemmArgs args, uint32_t batch, hipStream_t stream) {
  args.gz = batch;
  args.gx = (args.groups * 8 + T::kBN - 1) / T::kBN;
  args.gy = (args.quads * 4 + T::kBM - 1) / T::kBM;
  const dim3 grid(args.gx * args.gy * batch), block(kThreads);
  if constexpr (!kLinear) {
    hipLaunchKernelGGL((GemmTileKernel<false, false, kFmtAny, T>), grid, block, 0, stream, args);
  } else {
    const bool fp4 = args.n_planes == 1 && args.modes[0] == kModeFp4;
    const bool w8 = args.n_planes == 2 && args.modes[0] == kModeW8Hi && args.modes[1] == kModeW8Lo;
    if (args.n_pieces == 1 && fp4)
      hipLaunchKernelGGL((GemmTileKernel<true, false, kFmtFp4, T>), grid, block, 0, stream, args);
    else if (args.n_pieces == 1 && w8)
      hipLaunchKernelGGL((GemmTileKernel<true, false, kFmtW8, T>), grid, block, 0, stream, args);
    else
      hipLaunchKernelGGL((GemmTileKernel<true, true, kFmtAny, T>), grid, block, 0, stream, args);
  }
}
}  // namespace

// The tile of a launch: the one with the least estimated time per K block, a
// CU's tiles one after the other at the shape's rate, or one tile's latency.
// Each output's fold is sequential over K, so a launch is parallel only over
// its tiles: large tiles convert less per output, small ones fill the CUs.
// The rates (ns per tile and block, and the least per block) are fitted to
// these times, one launch each (us, 64x96 / 64x128 / 32x64):
//   4512 x 960, K 2560    56 / 75 / 96     141 x 2560, K 960   17 / 20 / 11
//   2048 x 2304, W8 768   45 / 55 / 67     141 x 960, K 2560   29 / 31 / 17
//   2048 x 768, W8 768    27 / 26 / 26     1 x 960, K 960      13 / 13 / 9
//   4512 x 320, K 960     25 / 21 / 22     928 x 512, W8 512   21 / 22 / 11
//   32 layers of 128 x 960, K 2560   60 / 51 / 85
// Up to 32 rows, half of a larger tile would be padding: 54 layers of 16 x
// 3,072, W8 768 91 / 92 / 78; 54 of 16 x 3,072, K 768 53 / 60 / 49.
template <bool kLinear>
hipError_t LaunchTiles(const GemmArgs& args, uint32_t batch, hipStream_t stream) {
  const uint64_t cus = DeviceCus(), cols = args.groups * 8ull, rows = args.quads * 4ull;
  auto time = [&](uint64_t bm, uint64_t bn, uint64_t rate, uint64_t latency) {
    const uint64_t tiles = ((rows + bm - 1) / bm) * ((cols + bn - 1) / bn) * batch;
    const uint64_t t = (tiles + cus - 1) / cus * rate;
    return t > latency ? t : latency;
  };
  const uint64_t t0 = time(32, 64, 130, 200), t1 = time(64, 96, 200, 400),
                 t2 = time(64, 128, 260, 460);
  if (rows <= 32 || (t0 <= t1 && t0 <= t2))
    LaunchTile<kLinear, Tile<32, 64, 2, 4, 4>>(args, batch, stream);
  else if (t1 <= t2) LaunchTile<kLinear, Tile<64, 96, 4, 2, 6>>(args, batch, stream);
  else LaunchTile<kLinear, Tile<64, 128, 2, 2, 4>>(args, batch, stream);
  return hipGetLastError();
}

hipError_t LaunchGemmInstr(const GemmArgs& args, hipStream_t stream) {
  return LaunchTiles<false>(args, 1, stream);
}

hipError_t LaunchGemmInstrAliased(const GemmArgs& args, hipStream_t stream) {
  const uint32_t total = args.quads * args.groups;
  const uint32_t words = total < kFbufDepth ? total : kFbufDepth;
  hipLaunchKernelGGL(GemmAliasKernel, dim3(words), dim3(32), 0, stream, args);
  return hipGetLastError();
}

namespace {
// A single fast layer with fewer tiles than this splits its K range (to
// about kTargetWorkgroups workgroups, at least kMinSplitSteps K-steps each)
// and finishes in the element-parallel deferred epilogue.  Measured on the
// SmolVLA chains (M = 141 and 1,600): 128 workgroups of at least 4 steps beat
// 256 of 2 by 9-13% (the split sums written and read again cost more than the
// parallelism gains); 32 workgroups, or no split, lost 50-70% at M = 141.
constexpr uint32_t kSmallGrid = 128, kTargetWorkgroups = 128, kMinSplitSteps = 4;
constexpr uint32_t kSplitMidRows = 1024, kSplitMidWork = 65536;

// K splits of args' gx x gy tiles: as many as fit in one round of
// kTargetWorkgroups workgroups.
void PlanKSplits(GemmArgs& args) {
  uint32_t nblocks = 0;
  for (uint32_t p = 0; p < args.n_pieces; ++p) nblocks += args.piece_kb[p];
  const uint32_t steps = (nblocks + 1) / 2, tiles = args.gx * args.gy;
  const uint32_t want = kTargetWorkgroups > tiles ? kTargetWorkgroups / tiles : 1u;
  uint32_t per = (steps + want - 1) / want;
  per = per < kMinSplitSteps ? kMinSplitSteps : per;
  args.splits = (steps + per - 1) / per;
  args.split_steps = per;
}
}  // namespace

hipError_t GrowWorkspace(Workspace& ws, size_t bytes, hipStream_t stream) {
  bytes += kSplitCounterBytes;
  if (ws.bytes >= bytes) return hipSuccess;
  // at least double, so a run of growing shapes retires few buffers
  size_t want = ws.bytes * 2 > bytes ? ws.bytes * 2 : bytes;
  want = (want + 0xFFFFF) & ~(size_t)0xFFFFF;
  if (ws.ptr != nullptr && ws.n_retired == sizeof ws.retired / sizeof ws.retired[0])
    return hipErrorOutOfMemory;  // (64 doublings: unreachable in practice)
  float* p = nullptr;
  hipError_t err = hipMalloc(&p, want);
  if (err != hipSuccess) return err;
  err = hipMemsetAsync(p, 0, kSplitCounterBytes, stream);  // the split counters start at zero
  if (err != hipSuccess) {
    (void)hipFree(p);
    return err;
  }
  if (ws.ptr != nullptr) ws.retired[ws.n_retired++] = ws.ptr;
  ws.ptr = p;
  ws.bytes = want;
  return hipSuccess;
}

void FreeWorkspace(Workspace& ws) {
  if (ws.ptr != nullptr) (void)hipFree(ws.ptr);
  for (uint32_t i = 0; i < ws.n_retired; ++i) (void)hipFree(ws.retired[i]);
  ws = Workspace{};
}

// MXFP8 E4M3 activations (one MXFP4 plane): in fast mode a layer of up to
// kSplitMidRows rows runs the single-launch split kernel with A straight
// into the FP8 x FP4 matrix cores; every other layer (exact mode, batches,
// more rows) is folded exactly per output by the epilogue kernel, one
// launch per layer (which meets the fast-mode tolerance too).
hipError_t LaunchFp8Linear(const GemmArgs& in, uint32_t batch, bool fast, hipStream_t stream) {
  GemmArgs args = in;
  args.ws = nullptr;
  args.splits = 1;
  args.split_steps = 0;
  if (fast && batch == 1 && args.quads * 4 <= kSplitMidRows) {
    SplitPlan(args);
    args.fast_ep = 1u;
    return LaunchSplitLinear(args, stream);
  }
  // batches of layers of up to 16 rows: the skinny kernel (the streaming
  // kernel's 128-row tiles would be mostly padding)
  if (fast && args.quads * 4 <= 16) {
    args.fast_ep = 1u;
    return LaunchLinearSkinny(args, batch, stream);
  }
  // batches and larger layers over weight panels (ops and the requantize
  // included): the streaming kernel, not the per-output exact fold below
  if (fast && StreamEligible(args)) {
    args.fast_ep = 1u;
    return LaunchStream(args, batch, stream);
  }
  args.fast_ep = 0u;
  for (uint32_t z = 0; z < batch; ++z) {
    GemmArgs one = args;
    one.a += z * args.a_batch;
    one.w[0] += z * args.w_batch;
    one.w[1] = one.w[0];
    one.c += z * args.c_batch;
    if (one.q_out != nullptr) one.q_out += z * args.q_batch;
    for (uint32_t o = 0; o < args.n_ops; ++o) {
      if (one.op_vec[o] != nullptr) one.op_vec[o] += z * args.op_vec_batch[o];
      if (one.op_x2[o] != nullptr) one.op_x2[o] += z * args.op_x2_batch[o];
    }
    one.a_batch = one.w_batch = one.c_batch = one.q_batch = 0;
    const hipError_t err = LaunchEpilogue(one, stream);
    if (err != hipSuccess) return err;
  }
  return hipSuccess;
}

hipError_t LaunchLinear(const GemmArgs& in, uint32_t batch, bool fast, Workspace& ws,
                        hipStream_t stream, FixedScratch* fixed) {
  // W8 panels: their own kernel, every shape and mode.
  if (in.w_fp6) return LaunchW8Linear(in, batch, fast, stream);
  if (in.a_fp8) return LaunchFp8Linear(in, batch, fast, stream);
  GemmArgs args = in;
  args.ws = nullptr;
  args.splits = 1;
  args.split_steps = 0;
  // Fast mode runs MXFP4 and W8 (hi, lo) on the block-scaled matrix cores;
  // any other plane list runs exactly (which meets the fast-mode tolerance).
  const bool fastk = fast && FastEligible(args);
  // A single small layer: one launch, K split over workgroups (the last
  // split of each tile finishes it).  Workspace: the counters, then the
  // partial sums.
  if (fastk && SplitEligible(args, batch)) {
    const size_t part = SplitPlan(args);
    args.fast_ep = 1u;
    if (part > 0) {
      float* base = nullptr;
      if (fixed != nullptr) {
        fixed->need = kSplitCounterBytes + part;
        if (fixed->need > fixed->bytes || fixed->ptr == nullptr) return hipErrorOutOfMemory;
        base = static_cast<float*>(fixed->ptr);
      } else {
        const hipError_t grown = GrowWorkspace(ws, part, stream);
        if (grown != hipSuccess) return grown;
        base = ws.ptr;
      }
      args.ws = base;
    }
    return LaunchSplitLinear(args, stream);
  }
  // Batched layers of up to 16 rows: split-K over the waves of one
  // workgroup, which holds every row.
  if (fastk && args.quads * 4 <= 16) return LaunchLinearSkinny(args, batch, stream);
  if (!fastk) return LaunchTiles<true>(args, batch, stream);
  // A batch of such layers whose 32 x 32 tiles are at most two to a CU:
  // the split kernel's tiles too, where the tile kernel's 64-row tiles leave
  // most CUs idle.  Measured, a launch (us, tile kernel / split tiles):
  // 32 layers of 50 x 192, W8 K 64 (attention scores; 384 split tiles) 10.0
  // / 5.5; 128 of 50 x 64, K 192 (512) 10.3 / 6.5; 16 of 64 x 320, K 960
  // (320) 15.3 / 9.5; 4 of 128 x 960, K 2560 (480) 26.2 / 14.3; past two to
  // a CU the larger tiles win: 128 of 50 x 192, K 64 (1,536) 10.6 / 13.9; 8
  // of 141 x 960, K 960 (1,200) 16.0 / 22.4.
  if (batch > 1 && args.quads * 4 <= kSplitMaxRows) {
    GemmArgs split = args;
    SplitPlan(split);
    if ((uint64_t)split.gx * split.gy * batch <= 2ull * DeviceCus()) {
      split.fast_ep = 1u;
      return LaunchSplitBatch(split, batch, stream);
    }
  }
  uint32_t gx, gy;
  FastGrid(args, batch, &gx, &gy, &args.tile_rows);
  args.gx = gx;
  args.gy = gy;
  const bool small = batch == 1 && gx * gy < kSmallGrid;
  // A layer of up to kSplitMidRows rows whose 128-row grid is small: the
  // single-launch split kernel's 32 x 32 tiles (enough workgroups, no
  // partial sums through memory, no second launch) instead of K splits of
  // 128-row tiles and the epilogue kernel, while rows x K blocks stays
  // within kSplitMidWork (measured, one layer per launch: 928 x 512 x 512
  // 7.3 against 16.1 us, 512 x 2560 x 960 18.1 against 25.9 us, 768 rows
  // even, 1024 x 2560 x 960 34.3 against 28.9 us).
  uint32_t blocks = 0;
  for (uint32_t p = 0; p < args.n_pieces; ++p) blocks += args.piece_kb[p];
  args.fast_ep = 1u;
  // MXFP4 layers the wave kernel can take keep these tiles up to two a CU:
  // 513 x 960, K 800, 510 tiles, 8.8 against 9.7 us; 300 x 2,560, K 960, 800
  // tiles, 15.2 against 9.2 us.  Up to three where they requantize (493 x
  // 1,408, K 416, 704 tiles, 9.1 against 10.6 us; 863 x 1,024, K 64, 864
  // tiles, 8.7 against 8.8 us) and for folds that the 8 splits shorten most
  // (676 x 768, K 3072, 528 tiles, 21.0 against 23.1 us).
  const uint32_t rows = args.quads * 4;
  if (small && rows <= kSplitMidRows && rows * blocks <= kSplitMidWork) {
    const uint32_t tiles = (args.n + 31) / 32 * ((rows + 31) / 32);
    const uint32_t per_cu = args.q_out != nullptr || blocks > 70 ? 3 : 2;
    if (tiles <= per_cu * (uint32_t)DeviceCus() || WaveColumns(args, batch) == 0) {
      SplitPlan(args);
      return LaunchSplitLinear(args, stream);
    }
  }
  const uint32_t wave_columns = WaveColumns(args, batch);
  if (wave_columns != 0) return LaunchWave(args, batch, wave_columns, stream);
  // What the wave kernel leaves: over panels the streaming kernel takes plain
  // batched layers (and MXFP8), the panel kernel a plain single layer of a
  // long fold (its 8 waves per CU hide more latency where a workgroup has one
  // or two tiles).  Layers with ops or the requantize stay on the tile kernel:
  // its epilogue runs on 16 waves per CU, the streaming kernel's on 4.
  if (!small && StreamEligible(args) && batch > 1)
    return LaunchStream(args, batch, stream);
  if (!small && PanelEligible(args)) return LaunchPanel(args, batch, stream);
  if (small) PlanKSplits(args);
  if (args.splits <= 1) return LaunchLinearFast(args, batch, stream);

  // (the partial sums start after the split counters)
  if (fixed != nullptr) {  // no allocation: the caller's buffer, or an error
    fixed->need = kSplitCounterBytes + WorkspaceBytes(args);
    if (fixed->need > fixed->bytes || fixed->ptr == nullptr) return hipErrorOutOfMemory;
    args.ws = static_cast<float*>(fixed->ptr) + kSplitCounterBytes / sizeof(float);
  } else {
    const hipError_t grown = GrowWorkspace(ws, WorkspaceBytes(args), stream);
    if (grown != hipSuccess) return grown;
    args.ws = ws.ptr + kSplitCounterBytes / sizeof(float);
  }
  const hipError_t err = LaunchLinearFast(args, args.splits, stream);  // z = split
  if (err != hipSuccess) return err;
  return LaunchEpilogue(args, stream);
}

}  // namespace hb
