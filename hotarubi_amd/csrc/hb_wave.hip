// MXFP4 tile kernel of independent waves (HB_LINEAR_FAST, DDR words or weight
// panels, every epilogue): a wave owns 32 rows x 32 kTN columns and takes
// them from the first load to the last store, with no barrier and no operand
// in LDS.
//
// Arithmetic as in the other fast kernels: A as two exact FP6 E2M3 planes
// h = fp6(q / 32) and (q - 32 h) / 2 with scale bytes ea - 1 and ea - 5
// (ring::SplitA), W's E2M1 codes and E8M0 bytes untouched (hb_panel.hip);
// plane h, then plane r of a step into each accumulator.
//
// Why waves on their own.  Lane l of an A operand is row l % 32, block l / 32:
// 32 consecutive bytes of a DDR word, so a lane loads and converts its own
// operand; a B operand is 16 consecutive bytes of a word or a panel.  A
// workgroup that shares converted operands through LDS (FastKernel: 128 x
// 256 tiles, 144 KB of LDS, one workgroup to a CU) runs prologue, K loop and
// epilogue one after the other, in rounds of 256 tiles; here 8 to 12 waves a
// CU are each at a point of their own, so one's stores and operand loads run
// under another's conversions and matrix work.  Each wave converts its rows
// again for every 128 columns (about 500 cycles a step against 256 of matrix
// work), which is what bounds the wide layers; the narrow ones are bound by
// HBM.
#include "hb_device.h"
#include "hb_internal.h"
#include "hb_ring.h"

namespace hb {
namespace {

typedef int i32x8 __attribute__((ext_vector_type(8)));
typedef float f32x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
// 4 floats at any 4-byte address (operands and C of the caller's tensors)
typedef float f32x4_u __attribute__((ext_vector_type(4), aligned(4)));

constexpr uint32_t kSafeLo = 70, kSafeHi = 179;
constexpr int kWaveRows = 32, kWaves = 4;

// Largest value over the 8 lanes 8 p .. 8 p + 7 (xor 1, xor 2, half-row mirror).
__device__ __forceinline__ uint32_t Max8(uint32_t x) {
  x = max(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0xB1, 0xF, 0xF, false));
  x = max(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x4E, 0xF, 0xF, false));
  return max(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x141, 0xF, 0xF, false));
}

// One step's raw operands of a lane: 32 bytes of A and the dword of its
// scale byte; the column-block of each n-tile and the dword of its scale byte
// (panels: one dword holds those of both n-tiles of a panel).
struct RawA {
  u32x4 a0, a1;
  uint32_t sa, mask;
};
template <int kTN, bool kPanels>
struct RawW {
  static constexpr int kScales = kPanels ? kTN / 2 : kTN;
  u32x4 w[kTN];
  uint32_t sw[kScales];
};
// A step's A operand in the matrix cores' form: both planes, and their scale
// bytes (0: h, 1: r).
struct PlanesA {
  i32x8 h, r;
  int sa;
};

template <int kTN, bool kPanels>
__global__ __launch_bounds__(64 * kWaves, 2) void WaveKernel(GemmArgs g) {
  __shared__ __attribute__((aligned(16))) float lds_out[kWaves][kTN][32 * 32];
  __shared__ uint64_t lds_act[512];  // activation half of TBUF
  __shared__ __attribute__((aligned(16))) float lds_vec[kMaxOps][32 * kTN];  // the ops' columns

  TouchArgs(&g, sizeof g);
  const uint32_t lane = threadIdx.x & 63;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const TileId tile = LogicalTile(g.gx, g.gy, g.gz);
  const uint32_t z = tile.z, rows4 = g.quads * 4;
  const uint32_t row0 = (tile.y * kWaves + wave) * kWaveRows, col0 = tile.x * (32 * kTN);
  const uint8_t* a = g.a + z * g.a_batch;
  const uint8_t* w = g.w[0] + z * g.w_batch;
  uint32_t* c = g.c + z * g.c_batch;
  uint8_t* q_out = g.q_out ? g.q_out + z * g.q_batch : nullptr;

  const uint32_t nblocks = g.piece_kb[0], first = g.piece_off[0], steps = (nblocks + 1) / 2;
  // The epilogue's small operands, which every wave shares: fetched first,
  // in LDS by the only barrier, which waits for them alone.
  constexpr int kActLoads = 512 / (64 * kWaves), kVecLoads = kMaxOps * 32 * kTN / (64 * kWaves);
  // (no branch around a load: a value that no op reads comes from the first
  // A word of the fold; `a` itself may lie before the buffer, moved by the
  // piece's place among the W blocks)
  const uint8_t* const any = a + (size_t)first * kDdrWord;
  const uint64_t* act_src = g.tbuf != nullptr ? g.tbuf + 512 : reinterpret_cast<const uint64_t*>(any);
  uint64_t act_v[kActLoads];
  uint32_t vec_v[kVecLoads];
  if (g.n_ops > 0) {  // uniform
#pragma unroll
    for (int k = 0; k < kActLoads; ++k)
      act_v[k] = act_src[g.tbuf != nullptr ? threadIdx.x + 64 * kWaves * k : 0u];
#pragma unroll
    for (int k = 0; k < kVecLoads; ++k) {
      const uint32_t o = (wave + kWaves * k) * 64 / (32 * kTN);  // the wave's op
      const uint32_t col = col0 + (threadIdx.x + 64 * kWaves * k) % (32 * kTN);
      const bool live = o < g.n_ops && (g.op_kind[o] == kEpAddP || g.op_kind[o] == kEpMulP);
      const uint32_t* src = live ? g.op_vec[o] + z * g.op_vec_batch[o]
                                 : reinterpret_cast<const uint32_t*>(any);
      vec_v[k] = src[live && col < g.n ? col : 0u];
    }
  }

  const uint32_t h = lane >> 5, l32 = lane & 31;
  const uint32_t quad = min((row0 + l32) >> 2, g.quads - 1);
  const uint32_t o_a = (quad * g.a_row + first) * kDdrWord, o_codes = (lane & 3) * 32;
  uint32_t o_w[kTN], o_sw[RawW<kTN, kPanels>::kScales];
  if constexpr (kPanels) {  // (columns past n are zero codes inside their panel)
    const uint32_t panels = (g.n + kPanelCols - 1) / kPanelCols;
#pragma unroll
    for (int p = 0; p < kTN / 2; ++p) {
      const uint32_t panel = min(col0 / kPanelCols + p, panels - 1);
      const uint32_t base = (panel * g.w_steps + first / 2) * kPanelChunk;
      o_w[2 * p] = base + (h * kPanelCols + l32) * 16;
      o_w[2 * p + 1] = o_w[2 * p] + 512;
      o_sw[p] = base + kPanelScales + 4 * (lane >> 1);
    }
  } else {
#pragma unroll
    for (int t = 0; t < kTN; ++t) {
      const uint32_t col = col0 + 32 * t + l32, grp = min(col >> 3, g.groups - 1);
      const uint32_t base = (grp * g.kb_total + first) * kDdrWord;
      o_w[t] = base + (lane & 7) * 16;
      o_sw[t] = base + 128 + (lane & 4);
    }
  }
  const uint32_t sw_shift = kPanels ? 16 * (lane & 1) : 8 * (lane & 3);

  // Steps past the last reload it (cache hits); the second block of an odd
  // last step reloads the first with A masked to zero.
  auto load_a = [&](RawA& rw, uint32_t step) __attribute__((always_inline)) {
    __builtin_amdgcn_sched_barrier(0);
    const uint32_t want = 2 * min(step, steps - 1) + h;
    const uint8_t* aw = a + (o_a + min(want, nblocks - 1) * kDdrWord);
    rw.a0 = *reinterpret_cast<const u32x4*>(aw + o_codes);
    rw.a1 = *reinterpret_cast<const u32x4*>(aw + o_codes + 16);
    rw.sa = *reinterpret_cast<const uint32_t*>(aw + 128);
    rw.mask = want < nblocks ? 0xFFFFFFFFu : 0u;
    __builtin_amdgcn_sched_barrier(0);
  };
  auto load_w = [&](RawW<kTN, kPanels>& rw, uint32_t step) __attribute__((always_inline)) {
    __builtin_amdgcn_sched_barrier(0);
    const uint32_t s = min(step, steps - 1);
    const uint32_t ub = kPanels ? s * kPanelChunk : min(2 * s + h, nblocks - 1) * kDdrWord;
#pragma unroll
    for (int t = 0; t < kTN; ++t) rw.w[t] = *reinterpret_cast<const u32x4*>(w + (o_w[t] + ub));
#pragma unroll
    for (int t = 0; t < RawW<kTN, kPanels>::kScales; ++t)
      rw.sw[t] = *reinterpret_cast<const uint32_t*>(w + (o_sw[t] + ub));
    __builtin_amdgcn_sched_barrier(0);
  };

  // MFMA tile j, register r of this lane: row row0 + 4 h + 8 (r / 4) + r % 4,
  // column col0 + 32 j + l32.
  f32x16 acc[kTN];
  bool unsafe = false;
  if (g.acc) {  // uniform: start from C
    unsafe = AccFromC(acc, c, g.m, g.n, [&](uint32_t j, uint32_t r, uint32_t& row, uint32_t& col) {
      row = row0 + 4 * h + 8 * (r / 4) + (r & 3);
      col = col0 + 32 * j + l32;
    });
  } else {
#pragma unroll
    for (int j = 0; j < kTN; ++j) acc[j] = f32x16{};
  }

  uint32_t bad = 0;
  auto convert = [&](const RawA& rw, PlanesA& p) __attribute__((always_inline)) {
    const uint32_t x[8] = {rw.a0[0], rw.a0[1], rw.a0[2], rw.a0[3],
                           rw.a1[0], rw.a1[1], rw.a1[2], rw.a1[3]};
    ring::u32x6 h6, r6;
    ring::SplitA(x, rw.mask, h6, r6);
#pragma unroll
    for (int i = 0; i < 6; ++i) {
      p.h[i] = (int)h6[i];
      p.r[i] = (int)r6[i];
    }
    p.h[6] = p.h[7] = p.r[6] = p.r[7] = 0;
    const uint32_t ea = __builtin_amdgcn_ubfe(rw.sa, 8 * (lane & 3), 8);  // row % 4 == lane % 4
    p.sa = (int)(((ea - 1u) & 0xFFu) | ((ea - 5u) << 8));
    bad |= (uint32_t)(ea - kSafeLo > kSafeHi - kSafeLo);
  };
  auto matrix = [&](const PlanesA& p, const RawW<kTN, kPanels>& rw) __attribute__((always_inline)) {
    int sw[kTN];
#pragma unroll
    for (int t = 0; t < kTN; ++t) {
      sw[t] = (int)(rw.sw[kPanels ? t / 2 : t] >> sw_shift);
      const uint32_t ew = __builtin_amdgcn_ubfe((uint32_t)sw[t], kPanels ? 8 * (t % 2) : 0, 8);
      bad |= (uint32_t)(ew - kSafeLo > kSafeHi - kSafeLo);
    }
    ring::Unroll<2>([&](auto plane) {
      ring::Unroll<kTN>([&](auto jj) {
        constexpr int kJ = decltype(jj)::value, kP = decltype(plane)::value;
        const u32x4 wv = rw.w[kJ];
        const i32x8 b = {(int)wv[0], (int)wv[1], (int)wv[2], (int)wv[3], 0, 0, 0, 0};
        acc[kJ] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(
            kP ? p.r : p.h, b, acc[kJ], 2, 4, kP, p.sa, kPanels ? kJ % 2 : 0, sw[kJ]);
      });
    });
  };
  // the work so far stays ahead of what follows
  auto anchor = [&]() __attribute__((always_inline)) {
    asm volatile("" : "+v"(bad));
#pragma unroll
    for (int j = 0; j < kTN; ++j) asm volatile("" : "+v"(acc[j]));
  };

  // Step s: its matrix work beside the conversion of step s + 1, then the
  // refills, each a whole step ahead of its use: A of step s + 3 (converted
  // in step s + 2) and W of step s + 2.  Two steps a round, with no way out
  // of the middle: a branch there would have the compiler wait for every
  // load at the loop's head.
  RawA ra[2];
  RawW<kTN, kPanels> rw[2];
  PlanesA pl[2];
  load_a(ra[0], 0);
  load_w(rw[0], 0);
  load_a(ra[1], 1);
  load_w(rw[1], 1);
  if (g.n_ops > 0) {  // uniform
#pragma unroll
    for (int k = 0; k < kActLoads; ++k) lds_act[threadIdx.x + 64 * kWaves * k] = act_v[k];
#pragma unroll
    for (int k = 0; k < kVecLoads; ++k) (&lds_vec[0][0])[threadIdx.x + 64 * kWaves * k] = __uint_as_float(vec_v[k]);
    __syncthreads();
  }
  if (row0 >= rows4) return;  // (past the only barrier)
  convert(ra[0], pl[0]);
  load_a(ra[0], 2);
  uint32_t s0 = 0;
  for (; s0 + 2 <= steps; s0 += 2) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      matrix(pl[i], rw[i]);
      convert(ra[1 - i], pl[1 - i]);
#pragma unroll
      for (int k = 0; k < 2 * kTN; ++k) {  // a matrix instruction, then what fits beside it
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, 64 / kTN / 2, 0);
      }
      anchor();
      load_a(ra[1 - i], s0 + i + 3);
      load_w(rw[i], s0 + i + 2);
    }
  }
  if (s0 < steps) matrix(pl[0], rw[0]);
  const bool slow = __builtin_amdgcn_ballot_w64(unsafe || bad != 0) != 0;

  // Epilogue: the MFMA tiles through the wave's own LDS (4 KB each) into rows
  // of 4 columns a lane (slot p holds row p ^ ((p >> 2) & 1), free of bank
  // conflicts both ways); a row's 32-column block is the 8 lanes 8 p .. + 7.
  const uint32_t ln = LaneNow();
  const uint32_t slot = ln >> 3, cc = 4 * (ln & 7);
  const uint32_t row_a = row0 + (slot ^ ((slot >> 2) & 1));  // and + 8, + 16, + 24
  // The first op with an [m][n] operand (a residual, the gate's partner): its
  // loads for every tile go out at once.
  uint32_t pre_op = kMaxOps;
  for (uint32_t o = g.n_ops; o-- > 0;)
    if (g.op_kind[o] == kEpAdd || g.op_kind[o] == kEpActMul) pre_op = o;
  auto load_x2 = [&](uint32_t o, uint32_t col) __attribute__((always_inline)) {
    const uint32_t* src = g.op_x2[o] + z * g.op_x2_batch[o];
    f32x16 v = {};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t row = row_a + 8 * i;
      if (row < g.m && col < g.n) {
        const f32x4_u x = *reinterpret_cast<const f32x4_u*>(src + (size_t)row * g.n + col);
#pragma unroll
        for (int k = 0; k < 4; ++k) v[4 * i + k] = x[k];
      }
    }
    return v;
  };
  f32x16 pre[kTN];
#pragma unroll
  for (int j = 0; j < kTN; ++j)
    pre[j] = pre_op < kMaxOps ? load_x2(pre_op, col0 + 32 * j + cc) : f32x16{};

#pragma unroll
  for (int j = 0; j < kTN; ++j)
#pragma unroll
    for (int r = 0; r < 16; ++r) {  // +0 maps -0 (and a flushed denormal) to +0
      const uint32_t row = 8 * (r / 4) + 4 * (ln >> 5) + (r & 3);
      lds_out[wave][j][(row ^ ((row >> 2) & 1)) * 32 + (ln & 31)] = acc[j][r] + 0.0f;
    }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  if (slow) {  // a scale byte or an initial C left the window: each lane its outputs exactly
    for (uint32_t t = 0; t < 16 * kTN; ++t) {
      const uint32_t j = t >> 4, i = (t >> 2) & 3, row = row_a + 8 * i, col = col0 + 32 * j + cc + (t & 3);
      if (row >= rows4 || col >= g.n) continue;
      const uint32_t init = (g.acc && row < g.m) ? c[(size_t)row * g.n + col] : 0u;
      lds_out[wave][j][(slot + 8 * i) * 32 + cc + (t & 3)] =
          __uint_as_float(SlowLinear<kPanels ? 2 : 1>(g, a, w, w, init, row, col));
    }
  }

  // The operands are waited for here, once: a wait inside the loop would be
  // for the stores of the tiles before as well (one in-order counter).
#pragma unroll
  for (int j = 0; j < kTN; ++j) asm volatile("" : "+v"(pre[j]));
  // (a loop, not unrolled: every tile through the same code, which a short
  // launch fetches once; the prefetched operand is picked by a uniform branch)
#pragma unroll 1
  for (uint32_t j = 0; j < kTN; ++j) {
    const uint32_t colt = col0 + 32 * j, col = colt + cc;
    if (colt >= g.n) break;  // uniform
    const bool col_in = col < g.n;  // (n is a multiple of 8: 4 columns in or out together)
    const float* const src = &lds_out[wave][j][slot * 32 + cc];  // + 256 i: row row_a + 8 i
    f32x16 y;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const f32x4_t v = *reinterpret_cast<const f32x4_t*>(src + 256 * i);
#pragma unroll
      for (int k = 0; k < 4; ++k) y[4 * i + k] = v[k];
    }
    for (uint32_t o = 0; o < g.n_ops; ++o) {
      const uint32_t kind = g.op_kind[o];
      f32x4_t p = {};
      f32x16 x2 = {};
      if (o == pre_op) {
        x2 = j == 0 ? pre[0] : j == 1 || kTN == 2 ? pre[1] : j == 2 ? pre[kTN - 2] : pre[kTN - 1];
      } else if (kind == kEpAdd || kind == kEpActMul) {
        x2 = load_x2(o, col);
        asm volatile("" : "+v"(x2));
      } else if (kind == kEpAddP || kind == kEpMulP) {
        p = *reinterpret_cast<const f32x4_t*>(&lds_vec[o][32 * j + cc]);
      }
      // two rows' worth at a time: 16 table entries in flight would spill
      ring::Unroll<2>([&](auto hh) {
        constexpr int kB = decltype(hh)::value * 8;
        f32x8 v, x, pv;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          v[i] = y[kB + i];
          x[i] = x2[kB + i];
          pv[i] = p[i & 3];
        }
        EpApplyFastN<false>(kind, g.op_imm[o], v, x, pv, lds_act);
#pragma unroll
        for (int i = 0; i < 8; ++i) y[kB + i] = v[i];
      });
    }
    if (c != nullptr) {  // uniform
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint32_t row = row_a + 8 * i;
        if (row < g.m && col_in)
          *reinterpret_cast<f32x4_u*>(c + (size_t)row * g.n + col) =
              f32x4_u{y[4 * i], y[4 * i + 1], y[4 * i + 2], y[4 * i + 3]};
      }
    }
    if (q_out != nullptr) {  // MXINT8 requantize
      const uint32_t nb = g.n >> 5;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint32_t row = row_a + 8 * i;
        uint32_t e = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) e = max(e, ExpField(__float_as_uint(y[4 * i + k])));
        e = Max8(e);
        if (row >= rows4 || !col_in) continue;
        uint8_t* word = q_out + ((size_t)(row >> 2) * nb + (colt >> 5)) * kDdrWord;
        uint32_t codes = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k)
          codes |= (uint32_t)QuantizeElementHw(__float_as_uint(y[4 * i + k]), e) << (8 * k);
        *reinterpret_cast<uint32_t*>(word + (row & 3) * 32 + cc) = codes;
        if ((ln & 7) == 0) word[128 + (row & 3)] = (uint8_t)ScaleByteOf(e);
        if ((ln & 7) == 1 && (row & 3) == 0) {  // bytes 132 .. 143 of the word are zero
          uint32_t* pad = reinterpret_cast<uint32_t*>(word + 132);
          pad[0] = pad[1] = pad[2] = 0u;
        }
      }
    }
  }
}

template <int kTN>
void Launch(const GemmArgs& args, hipStream_t stream) {
  const dim3 grid(args.gx * args.gy * args.gz), block(64 * kWaves);
  if (args.w_panels) hipLaunchKernelGGL((WaveKernel<kTN, true>), grid, block, 0, stream, args);
  else hipLaunchKernelGGL((WaveKernel<kTN, false>), grid, block, 0, stream, args);
}

}  // namespace

// The line between this kernel's two wave tiles and the others.  Measured,
// one launch (us: the other kernel / 128 / 64 columns a wave):
//   67,584 x 64, K 576 with bias, ReLU, requantize   44.1 / 26.6 / 21.9
//   67,584 x 256, K 64 with a residual               41.0 / 31.0 / 25.0
//   4,512 x 2,560, K 960, requantized                52.3 / 39.8 / 43.4
//   4,512 x 960, K 2560 with a residual              36.2 / 38.6 / 41.3
//   1,600 x 2,048, K 736, requantized                20.3 / 20.0 / 18.7
//   1,613 x 960, K 1024, requantized                 20.7 / 20.0 / 14.4
//   29 layers of 514 x 384, K 1504                   50.4 / 29.5 / 38.6
//   64 layers of 48 x 960, K 960, requantized        23.1 / 25.6 / 24.5
//   1,056 x 256, K 2304, requantized                 17.4 / 26.3 / 19.6
//   256 layers of 128 x 960, K 960                   81.2 / 88.7 / -
//   300 x 2,560, K 960 / 513 x 960, K 800            16.4 / 14.2 / 10.4,  8.8 / 13.2 / 9.7
// So: 64 columns a wave (3 waves to a SIMD, each converting A for half the
// columns) while 128 columns would give fewer than one wave to two SIMDs or
// the fold is under 4 steps.  Others: the split kernel's 32 x 32 tiles while
// they are at most two or three to a CU (LaunchLinear; its K splits are
// parallel, a wave's fold is not), K splits of large tiles for a long fold
// over few waves, and tiles that share converted operands where a long fold
// over many waves is all conversion, where 64 rows fill their tile, or where
// the weights of many layers of up to 128 rows are the traffic (their one
// tile reads them once).  Plain batches over DDR words stay on their
// streaming kernel (hb_fast4.hip: 200 layers of 128 x 2,048, K 736, 107.8
// against 134.3 us; 40 of 200 x 256, K 320, 10.1 against 9.5).
//
// The lines past that are for launches whose workgroups (4 waves) just miss
// a round of the CUs, or whose columns just miss a tile; each with the times
// on both sides (us: the other kernel / 128 / 64 columns):
//   64 columns for at most 5 column tiles that 128 would leave a quarter
//   empty: 9,894 x 160, K 992, requantized 18.9 / 20.4 / 15.1 (folds under 24
//   steps: 12,241 x 160, K 2976 32.7 / 31.7 / 37.5)
//   128 columns for a long fold that they fit in one round and 64 do not: 15
//   layers of 144 x 768, K 3072 32.4 / 28.2 / 35.2
//   the others for a long fold past one round, up to one and a half: 11
//   layers of 391 x 736, K 2048 26.7 / 33.7 / 36.8
//   the tile kernel where its 64-row tiles fill the one round that this
//   kernel just misses: 1,589 x 2,560, K 960, requantized 22.0 / 26.4 / 25.9
//   the tile kernel for requantized 64 columns and up to 4 steps over few
//   waves: 1,141 x 64, K 128 8.2 / 9.5 / 8.7
//   K splits from 24 steps on where the layer requantizes: 1,211 x 96, K
//   1760 14.2 / 21.1 / 16.9
//   the panel kernel (plain, whole 256-column tiles) where its rounds are
//   nearly full or its one round is this kernel's second: 7,952 x 3,072, K
//   768 40.9 / 43.6 / 58.9, 10,602 x 512, K 512 12.9 / 14.1 / 14.6 (but
//   15,943 x 768, K 768, rounds 0.73 full, 27.2 / 24.3 / 29.6)
// Over 6,031 calls of 8 us and more, drawn after these lines were set (17 to
// 70,000 rows, K 32 to 3,072, 64 to 3,072 columns, up to 64 layers), 10 take
// over 8% longer than on the other kernels (51 without the lines), the worst
// 1.21 times as long (27 layers of 174 x 736, K 864, requantized 21.9 / 26.1
// / 25.9), and the mean is 0.79 of theirs.
uint32_t WaveColumns(const GemmArgs& args, uint32_t batch) {
  // one MXFP4 plane, one run of blocks (over panels from the start of a step:
  // a chunk's two blocks are one step's)
  if (args.n_planes != 1 || args.modes[0] != kModeFp4 || args.a_fp8 || args.n_pieces != 1 ||
      (args.w_panels && args.piece_off[0] % 2 != 0))
    return 0;
  const uint64_t cus = DeviceCus(), simds = 4 * cus;
  const uint64_t rows = args.quads * 4ull, cols = args.groups * 8ull;
  const uint64_t cols128 = (cols + 127) / 128, cols64 = (cols + 63) / 64;
  // waves, and workgroups, of 128 and 64 columns
  const uint64_t row_waves = (rows + kWaveRows - 1) / kWaveRows * batch;
  const uint64_t wide = row_waves * cols128, narrow = row_waves * cols64;
  const uint64_t row_groups = (rows + kWaves * kWaveRows - 1) / (kWaves * kWaveRows) * batch;
  const uint64_t wide_groups = row_groups * cols128, narrow_groups = row_groups * cols64;
  const uint32_t steps = (args.piece_kb[0] + 1) / 2;
  const bool quantize = args.q_out != nullptr, plain = args.n_ops == 0 && !quantize;
  if (rows <= 64 ? narrow > simds : steps >= 32 && wide >= simds) return 0;
  if (rows <= 128 && wide > 2 * simds) return 0;
  if (batch > 1 && !args.w_panels && plain) return 0;
  if (batch == 1 && steps >= (quantize ? 24u : 32u) && narrow < cus) return 0;
  if (quantize && cols <= 64 && steps <= 4 && narrow <= simds / 2) return 0;
  if (steps >= 24 && wide_groups > cus && 2 * wide_groups <= 3 * cus) return 0;
  const uint64_t tiles64 = (rows + 63) / 64 * ((cols + 255) / 256) * batch;
  if (steps >= 12 && wide_groups > cus && 4 * wide_groups <= 5 * cus &&
      16 * tiles64 >= 15 * cus && tiles64 <= cus)
    return 0;
  if (batch == 1 && steps >= 8 && steps <= 24 && cols % 256 == 0 && PanelEligible(args)) {
    const uint64_t tiles = (rows + 127) / 128 * (cols / 256);
    if (6 * tiles >= 5 * ((tiles + cus - 1) / cus * cus) ||
        (tiles <= cus && wide_groups > cus && 10 * wide_groups <= 13 * cus))
      return 0;
  }
  if (!plain && steps < 24 && 3 * cols64 <= 5 * cols128) return 64;
  if (steps >= 24 && wide_groups <= cus && narrow_groups > cus) return 128;
  return cols <= 64 || wide < simds / 2 || steps < 4 ? 64 : 128;
}

hipError_t LaunchWave(const GemmArgs& in, uint32_t batch, uint32_t columns, hipStream_t stream) {
  GemmArgs args = in;
  const uint32_t row_waves = (args.quads * 4 + kWaveRows - 1) / kWaveRows;
  args.gx = (args.groups * 8 + columns - 1) / columns;
  args.gy = (row_waves + kWaves - 1) / kWaves;
  args.gz = batch;
  if (columns == 64) Launch<2>(args, stream);
  else Launch<4>(args, stream);
  return hipGetLastError();
}

}  // namespace hb
