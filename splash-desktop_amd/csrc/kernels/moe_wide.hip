// The MoE expert passes over 32-row tiles (reference: kernels/shared/moe_gguf.metal:121-206, moe_expert_slab.h:13-99):
// exact bf16 operands 128 + q against bf16 activations with a per-scale-group fp32 close, as the row tile's
// (rowtile.hpp), on the 32x32x16 MFMA.
//
// CDNA4 mapping. A workgroup of eight waves takes up to two consecutive tiles of one expert (64 grouped rows); a wave
// streams 32 columns of one tensor over all of K (a gate/up pass: waves 0..3 gate, 4..7 up of the same columns, which
// meet in LDS at the end), 128 registers, so four waves share a SIMD and cover each other's dependency stalls (a wave
// of both tensors' 32 columns, two a SIMD, took 206 us where this takes 160: Q4_K gate/up of 1999 rows of 8 routes over
// 256 experts of 2048 x 512; the row tile's 16x16x32 walk of 32 rows, 213). Per step of 64 inputs
//  - the workgroup's rows come 128 bytes a row (eight lanes a row, whole cache lines) through registers into LDS, one
//    step ahead (32 rows and fewer: two), in two stages with one barrier each, with each group's input sums (four lanes
//    a group) beside them; every wave reads its MFMA fragments from there;
//  - a lane holds one column's codes of one of the step's groups (lane l: column l % 32, group l / 32), so two
//    v_permlane32_swap turn a block's words into both groups' B operands, the lane derives one (column, group)'s
//    coefficients, one more swap gives every lane its column's scales of both groups, and the offsets already lie in
//    the fp32 MFMA's B layout;
//  - each scale group closes as acc += s * sum x (128 + q) on the VALU, and the offsets of both groups, (z - 128 s) *
//    sum x, in one 32x32x2 fp32 MFMA a row block.
// The passes are bound by instruction issue (VALU issue 59% of the gate/up dispatch above) and, where tiles hold few rows,
// by their steps' waits. Of the instances (128 registers) all but af4g64's spill, 28 to 128 bytes a lane; in the hot loops
// only Q5_K's and Q6_K's over 64 rows (two and seven reloads or stores every four steps). A row's result depends only on
// its own activations.
#include <type_traits>

#include "kernels.hpp"
#include "rowtile.hpp"

namespace sq::kern {
namespace {

typedef __attribute__((__vector_size__(16 * sizeof(float)))) float f32x16;

__device__ __forceinline__ f32x16 mfma32(u32x4 a, u32x4 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0,
                                                 0);
}
__device__ __forceinline__ f32x16 mfma32_f32(float a, float b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}
// The lower halves of a and b, and the upper ones: {a.lo | b.lo}, {a.hi | b.hi}.
__device__ __forceinline__ void swap32(uint32_t &a, uint32_t &b) {
  const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
  a = r[0];
  b = r[1];
}
__device__ __forceinline__ u32x4 half_of(const u32x4 &a, const u32x4 &b, int m) {
  return u32x4{a[2 * m], a[2 * m + 1], b[2 * m], b[2 * m + 1]};
}
// LDS writes done, then the workgroup's barrier; loads in flight stay so (a __syncthreads() would wait for them).
__device__ __forceinline__ void step_barrier() {
  __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0)
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}
// Byte offset of 16-byte chunk c of row r of a stage: rows r and r + 1 of any even r hold a chunk 128 bytes apart, and
// sixteen neighbouring rows' reads of one chunk cover all banks once.
__device__ __forceinline__ uint32_t stage_at(uint32_t r, uint32_t c) { return r * 128 + ((c ^ ((r >> 1) & 7)) << 4); }

// A stage: 64 rows of 128 bytes, then each row's input sums [half][group] (formats without half scales: [group]).
constexpr int kStageRows = 64, kRowBytes = kStageRows * 128, kStageBytes = kRowBytes + kStageRows * 16;
constexpr int kWaves = 8, kTensorWaves = 4;

// The sums of a 16-byte chunk's first and last four bf16 values, in a fixed order.
__device__ __forceinline__ float quad_of(uint32_t a, uint32_t b) {
  const float x0 = __uint_as_float(a << 16), x1 = __uint_as_float(a & 0xFFFF0000u);
  const float x2 = __uint_as_float(b << 16), x3 = __uint_as_float(b & 0xFFFF0000u);
  return (x0 + x1) + (x2 + x3);
}
// v added over the four lanes of a quad (quad_perm [1,0,3,2], then [2,3,0,1]).
__device__ __forceinline__ float quad_total(float v) {
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xF, 0xF, false));
  return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4E, 0xF, 0xF, false));
}

// The row of the workgroup's whose chunk lane % 8 the lane stages.
template <int RB>
__device__ __forceinline__ uint32_t stage_row() {
  return RB == 2 ? threadIdx.x >> 3 : 4 * (threadIdx.x >> 6) + ((threadIdx.x >> 3) & 3);
}
// That row in the input: a pointer to the lane's chunk, or, in the formats whose walk would spill the pointer (each
// reload then waits for every load in flight), the 64-input span it begins at. Measured, block times at 33 / 128 rows
// of eight routes over 256 experts of 2048 x 512, pointer -> span: af4g128 99 / 139 -> 89 / 130 us, Q6_K 143 / 199 ->
// 137 / 194; af4g64 84 / 123 -> 86 / 127 (the span's address takes instructions), so the formats that don't spill keep
// the pointer.
template <uint32_t FMT>
constexpr bool kRowSpans = FMT == SQ_FMT_AF4G128 || FMT == SQ_FMT_Q6K;
template <uint32_t FMT>
using RowSource = std::conditional_t<kRowSpans<FMT>, uint32_t, const uint16_t *>;

// The walk of one wave over RB blocks of 32 rows: acc[b] += its 32 columns' sums, in registers 0..LIVE - 1 (LIVE 8:
// rows 0..15 of a block). plane, high and meta: the plane tile, c0 the wave's first column of it; row: the lane's row,
// of the workgroup's `rows`. One block stages two steps at a time (lanes 0..31 the even step's rows, 32..63 the odd
// one's), in four half stages: one barrier and one wait for rows every two steps. Tiles of few rows run as many steps
// as tall ones and hold little to do in each, so they were bound by that wait: 64 rows of eight routes over 256 af4g64
// experts of 2048 x 512, a step at a time with every wave staging and sixteen registers closed, 143 us the block; so,
// 115 to 119. (Four steps at a time up to 16 rows: 1.01 x that; rings of six or eight steps of codes 1.08 and 1.17.)
template <uint32_t FMT, int RB, int LIVE>
__device__ __forceinline__ void wide_walk(const MoeExpertArgs &a, const uint8_t *plane, const uint8_t *high,
                                          const uint8_t *meta, uint32_t c0, RowSource<FMT> row, uint32_t rows,
                                          uint8_t *lds, f32x16 (&acc)[RB]) {
  using F = Fmt<FMT>;
  constexpr int SG = F::SG, NH = F::HALVES ? 2 : 1;
  const int lane = threadIdx.x & 63, l32 = lane & 31, h = lane >> 5;
  constexpr uint32_t kSteps = RB == 2 ? 1 : 2;   // steps staged at a time
  constexpr int kRows = RB * 32 * 128, kStage = kStageBytes / kSteps;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), G = a.K >> 5, steps = G / 2;
  const CodeConstants cc = make_code_constants();

  const uint32_t col = c0 + l32;
  const auto planes = buffer_rsrc(plane, G * 64 * F::P0), metas = buffer_rsrc(meta, G / F::UNIT * 64 * F::META);
  const auto highs = buffer_rsrc(high, F::P1 ? G * 64 * F::P1 : 0);
  const uint32_t pv = (h * 64 + col) * F::P0, hv = (h * 64 + col) * F::P1;
  const uint32_t mv = ((F::UNIT == 1 ? h * 64 : 0) + col) * F::META;
  // A step's words: codes (8-bit codes: two vectors) and plane1 bits of the lane's (column, group).
  struct Words {
    u32x4 lo, hi;
    u32x2 high;
  };
  const auto load = [&](uint32_t step, Words &w) __attribute__((always_inline)) {
    const uint32_t at = 2 * step * 64 * F::P0;
    w.lo = buffer_b128(planes, pv, at);
    if constexpr (F::P0 == 32) w.hi = buffer_b128(planes, pv, at + 16);
    if constexpr (F::P1 == 4) w.high[0] = buffer_b32(highs, hv, 2 * step * 64 * 4);
    if constexpr (F::P1 == 8) w.high = buffer_b64(highs, hv, 2 * step * 64 * 8);
  };
  const auto load_meta_of = [&](uint32_t step) __attribute__((always_inline)) {
    return buffer_meta<FMT>(metas, mv, 2 * step / F::UNIT * 64 * F::META);
  };
  // Waves whose rows all lie past the workgroup's stage none: what the stages hold there reaches only outputs that are
  // not stored.
  u32x4 x;
  const uint32_t my_row = stage_row<RB>();
  const bool loads = RB == 2 || 4 * wave < rows;
  const auto load_rows = [&](uint32_t step) __attribute__((always_inline)) {
    const uint32_t at = min(RB == 2 ? step : step + h, steps - 1);
    if (!loads) return;
    if constexpr (!kRowSpans<FMT>) x = *(const u32x4 *)(row + at * 64);
    else if constexpr (RB == 2) x = ((const u32x4 *)a.input + 8 * at)[8 * (size_t)row + (lane & 7)];
    else x = ((const u32x4 *)a.input)[8 * (size_t)(row + at) + (lane & 7)];
  };
  const auto store_rows = [&](uint32_t step) __attribute__((always_inline)) {
    uint8_t *const to = lds + (RB == 2 ? step & 1 : (step & 2) + h) * kStage;
    if (loads) {
      *(u32x4 *)(to + stage_at(my_row, lane & 7)) = x;
      float *const sums = (float *)(to + kRows) + my_row * (2 * NH) + ((lane >> 2) & 1);
      const float first = quad_of(x[0], x[1]), second = quad_of(x[2], x[3]);
      if constexpr (F::HALVES) {
        const float s0 = quad_total(first), s1 = quad_total(second);
        if ((lane & 3) == 0) {
          sums[0] = s0;
          sums[2] = s1;
        }
      } else {
        const float s0 = quad_total(first + second);
        if ((lane & 3) == 0) sums[0] = s0;
      }
    }
  };

  f32x16 zero;
#pragma unroll
  for (int r = 0; r < 16; ++r) zero[r] = 0.0f;
  f32x16 C[RB];
  const auto close = [&](f32x16 &to, float scale, const f32x16 &c) __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < LIVE; ++r) to[r] = fmaf(scale, c[r], to[r]);
  };

  const auto compute = [&](uint32_t step, const Words &w, const MetaWords &meta_words) __attribute__((always_inline)) {
    const uint8_t *stage = lds + (step & (2 * kSteps - 1)) * kStage;
    const float *sums = (const float *)(stage + kRows);
    // The lane's coefficients (its column's in group 2 step + h).
    float s[2], zc[2];
    const uint32_t own = 2 * step + h;
    if constexpr (F::HALVES) {
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        s[m] = q6k_scale(meta_words, own, m);
        zc[m] = -160.0f * s[m];
      }
    } else {
      const Coef k = coef<FMT>(meta_words, own);
      s[0] = k.s;
      zc[0] = F::P0 == 32 ? fmaf(-2176.0f, k.s, FMT == SQ_FMT_Q80 ? -128.0f * k.s : k.z) : fmaf(-128.0f, k.s, k.z);
    }
    // Both groups' words: word[g][i] chunk 2 h + i of the lane's column (8-bit codes: and its second word).
    uint32_t word[2][2], second[2][2], bits[2];
    if constexpr (F::P0 == 32) {
      // Chunks 0, 1 are words 0..3, chunks 2, 3 words 4..7.
      uint32_t v[8] = {w.lo[0], w.lo[1], w.lo[2], w.lo[3], w.hi[0], w.hi[1], w.hi[2], w.hi[3]};
#pragma unroll
      for (int i = 0; i < 4; ++i) swap32(v[i], v[4 + i]);
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        word[0][i] = v[2 * i];
        second[0][i] = v[2 * i + 1];
        word[1][i] = v[4 + 2 * i];
        second[1][i] = v[5 + 2 * i];
      }
    } else {
      uint32_t v[4] = {w.lo[0], w.lo[1], w.lo[2], w.lo[3]};
      swap32(v[0], v[2]);
      swap32(v[1], v[3]);
      word[0][0] = v[0];
      word[0][1] = v[1];
      word[1][0] = v[2];
      word[1][1] = v[3];
    }
    if constexpr (F::P1 != 0) {
      bits[0] = w.high[0];
      bits[1] = F::P1 == 4 ? w.high[0] : w.high[1];
      swap32(bits[0], bits[1]);
    }
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      u32x4 lo[2], hi[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        uint32_t hb = 0;
        if constexpr (F::P1 == 4) hb = (bits[g] >> (16 * h + 8 * i)) & 0xFFu;
        if constexpr (F::P1 == 8) hb = (bits[g] >> (16 * i)) & 0xFFFFu;
        chunk_operands<FMT, true>(word[g][i], F::P0 == 32 ? second[g][i] : 0u, hb, cc, lo[i], hi[i]);
      }
      float sg[2];   // every lane its column's scale of group g
#pragma unroll
      for (int m = 0; m < NH; ++m) {
        if constexpr (SG == 1) {
          uint32_t p = __float_as_uint(s[m]), q = p;
          swap32(p, q);
          sg[m] = __uint_as_float(g ? q : p);
        } else {
          sg[m] = s[m];
        }
      }
      const bool first = SG == 1 || (g == 0 && (SG == 2 || step % 2 == 0));
      const bool last = SG == 1 || (g == 1 && (SG == 2 || step % 2 == 1));
      u32x4 xa[RB], xb[RB];
#pragma unroll
      for (int b = 0; b < RB; ++b) {
        xa[b] = *(const u32x4 *)(stage + stage_at(32 * b + l32, 4 * g + 2 * h));
        xb[b] = *(const u32x4 *)(stage + stage_at(32 * b + l32, 4 * g + 2 * h + 1));
      }
      if constexpr (F::HALVES) {
#pragma unroll
        for (int m = 0; m < 2; ++m) {
#pragma unroll
          for (int b = 0; b < RB; ++b) C[b] = mfma32(half_of(xa[b], xb[b], m), half_of(lo[0], lo[1], m), zero);
#pragma unroll
          for (int b = 0; b < RB; ++b) close(acc[b], sg[m], C[b]);
        }
      } else {
#pragma unroll
        for (int b = 0; b < RB; ++b) C[b] = mfma32(xa[b], lo[0], first ? zero : C[b]);
#pragma unroll
        for (int b = 0; b < RB; ++b) C[b] = mfma32(xb[b], lo[1], C[b]);
        if constexpr (F::P0 == 32) {
#pragma unroll
          for (int b = 0; b < RB; ++b) C[b] = mfma32(xa[b], hi[0], C[b]);
#pragma unroll
          for (int b = 0; b < RB; ++b) C[b] = mfma32(xb[b], hi[1], C[b]);
        }
        if (last)
#pragma unroll
          for (int b = 0; b < RB; ++b) close(acc[b], sg[0], C[b]);
      }
    }
    // Both groups' offsets (a scale group over both or over several steps: its offset times each group's sum).
#pragma unroll
    for (int m = 0; m < NH; ++m)
#pragma unroll
      for (int b = 0; b < RB; ++b) acc[b] = mfma32_f32(sums[(32 * b + l32) * (2 * NH) + 2 * m + h], zc[m], acc[b]);
  };

  // Codes come `kAhead` steps ahead into a ring of four (8-bit codes, of twice the registers: two), the meta with them
  // or, where a unit spans the ring's four steps, a unit ahead.
  constexpr int kRing = F::P0 == 32 ? 2 : 4, kAhead = kRing - 1;
  constexpr bool kUnitMeta = F::UNIT == 8;
  Words w[kRing];
  MetaWords m[kUnitMeta ? 2 : kRing];
  load_rows(0);
  store_rows(0);
  load_rows(kSteps);   // before the codes, as in the loop, so that waiting for them does not wait for those
#pragma unroll
  for (int k = 0; k < kAhead; ++k) {
    load(min((uint32_t)k, steps - 1), w[k]);
    if constexpr (!kUnitMeta) m[k] = load_meta_of(min((uint32_t)k, steps - 1));
  }
  if constexpr (kUnitMeta) m[0] = load_meta_of(0);
  const auto run = [&](uint32_t at, int k) __attribute__((always_inline)) {
    if (RB == 2 || k % 2 == 0) {
      step_barrier();   // the stage's rows are in, and the other stage's reads are done
      store_rows(at + kSteps);
      load_rows(at + 2 * kSteps);
    }
    load(min(at + kAhead, steps - 1), w[(k + kAhead) % kRing]);
    if constexpr (!kUnitMeta) m[(k + kAhead) % kRing] = load_meta_of(min(at + kAhead, steps - 1));
    compute(at, w[k], m[kUnitMeta ? 0 : k]);
  };
  uint32_t step = 0;
#pragma unroll 1
  for (; step + kRing <= steps; step += kRing) {
    if constexpr (kUnitMeta) m[1] = load_meta_of(min(step + kRing, steps - 1));
#pragma unroll
    for (int k = 0; k < kRing; ++k) run(step + k, k);
    if constexpr (kUnitMeta) m[0] = m[1];
  }
  // The steps past the last whole ring (a unit's formats have none).
  if constexpr (!kUnitMeta)
#pragma unroll
    for (int k = 0; k < kRing - 1; ++k)
      if (step + k < steps) run(step + k, k);
}

// The wave's sums to their places: acc[b][r] is row 32 b + 8 (r / 4) + 4 h + r % 4, column l32 of the wave's.
template <int RB>
__device__ __forceinline__ void wide_store(const MoeExpertArgs &a, const f32x16 (&acc)[RB], uint32_t first_row,
                                           uint32_t rows, uint32_t column, bool live, uint8_t *lds) {
  const int lane = threadIdx.x & 63, l32 = lane & 31, h = lane >> 5;
  const uint32_t wave = threadIdx.x >> 6;
  // The gathering passes store in the read order (chunk (col / 4) % 4 of a group, half col / 16), the down pass in
  // column order.
  const uint32_t col = column + (a.gather ? 8 * ((l32 >> 2) & 3) + 4 * (l32 >> 4) + (l32 & 3) : l32);
  float *const gates = (float *)lds;   // [wave][b][r][lane]
  if (a.gate_up) {
    __syncthreads();   // every wave's reads of the stages are done
    if (wave < kTensorWaves)
#pragma unroll
      for (int b = 0; b < RB; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) gates[((wave * RB + b) * 16 + r) * 64 + lane] = acc[b][r];
    __syncthreads();
    if (wave < kTensorWaves) return;
  }
  if (!live) return;
#pragma unroll
  for (int b = 0; b < RB; ++b)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const uint32_t row = 32 * b + 8 * (r >> 2) + 4 * h + (r & 3);
      if (row >= rows) continue;
      const size_t at = (size_t)(first_row + row) * a.output_size + col;
      float v = acc[b][r];
      if (a.gate_up || a.gate) {
        const uint32_t place = (((wave - kTensorWaves) * RB + b) * 16 + r) * 64 + lane;
        const float g = bf16_to_f32(a.gate_up ? f32_to_bf16(gates[place]) : a.gate[at]);
        v = bf16_to_f32(f32_to_bf16(v)) * silu(g);
      }
      a.output[at] = f32_to_bf16(v);
    }
}

// The launch's work list in LDS: its tiles taken two of an expert at a time from the expert's first on (`single`: each
// alone), as 2 tile + (1 if it takes the next tile too), those of two tiles first, so that the long ones do not trail.
// Returns its entries. experts: LDS room for the tiles' experts.
constexpr uint32_t kMaxTiles =
    SQ_PREFILL_TOKEN_BUDGET * 64 / 32 + SQ_MOE_WIDE_EXPERT_SLOTS + 2 * SQ_PREFILL_TOKEN_BUDGET / 32;
__device__ uint32_t work_list(const MoeExpertArgs &a, uint32_t n, uint16_t *experts, uint16_t *list) {
  constexpr uint32_t kThreads = 64 * kWaves;
  __shared__ uint32_t wave_start[kWaves], wave_count[kWaves];
  const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  for (uint32_t t = tid; t < n; t += kThreads) experts[t] = (uint16_t)a.tiles[t].expert;
  __syncthreads();
  const uint32_t each = (n + kThreads - 1) / kThreads, begin = min(n, tid * each), end = min(n, begin + each);
  const auto starts = [&](uint32_t t) { return t == 0 || experts[t] != experts[t - 1]; };
  // The first tile (plus one) of the expert that holds tile begin - 1: the last start before the run.
  uint32_t latest = 0;
  for (uint32_t t = begin; t < end; ++t)
    if (starts(t)) latest = t + 1;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const uint32_t up = (uint32_t)__shfl_up((int)latest, d);
    if (lane >= (uint32_t)d) latest = max(latest, up);
  }
  if (lane == 63) wave_start[wave] = latest;
  uint32_t before = (uint32_t)__shfl_up((int)latest, 1);
  if (lane == 0) before = 0;
  __syncthreads();
  for (uint32_t w = 0; w < wave; ++w) before = max(before, wave_start[w]);
  // The entry of tile t: 0 none, 1 alone, 2 with the next tile.
  const auto entry = [&](uint32_t t, uint32_t &first) -> uint32_t {
    if (starts(t)) first = t + 1;
    const uint32_t expert = experts[t];
    if (a.mode != 2 && (expert >= a.experts) != (a.mode == 1)) return 0;
    if (a.single) return 1;
    if ((t + 1 - first) & 1) return 0;
    return t + 1 < n && experts[t + 1] == expert ? 2 : 1;
  };
  uint32_t mine = 0, first = before;   // entries of two tiles << 16 | of one
  for (uint32_t t = begin; t < end; ++t) {
    const uint32_t e = entry(t, first);
    mine += e == 2 ? 1u << 16 : e;
  }
  uint32_t inclusive = mine;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const uint32_t up = (uint32_t)__shfl_up((int)inclusive, d);
    if (lane >= (uint32_t)d) inclusive += up;
  }
  if (lane == 63) wave_count[wave] = inclusive;
  __syncthreads();
  uint32_t at = inclusive - mine, all = 0;
#pragma unroll
  for (uint32_t w = 0; w < kWaves; ++w) {
    at += w < wave ? wave_count[w] : 0u;
    all += wave_count[w];
  }
  uint32_t pair = at >> 16, one = (all >> 16) + (at & 0xFFFFu);
  first = before;
  for (uint32_t t = begin; t < end; ++t) {
    const uint32_t e = entry(t, first);
    if (e == 2) list[pair++] = (uint16_t)(2 * t + 1);
    if (e == 1) list[one++] = (uint16_t)(2 * t);
  }
  __syncthreads();
  return (all >> 16) + (all & 0xFFFFu);
}

// A workgroup runs one column group of a tile and, if it is the expert's next, the tile after it (tiles pair from the
// expert's first on). Over a long K it takes its tiles from the work list, the tall ones first: entries go round the
// XCDs (workgroup b runs on XCD b % 8), an entry's column groups on one XCD, whose L2 they share its rows in. Over a
// short K, or where the routed experts hold at most 24 rows on average (most are then one tile, and the order has
// nothing to put first), the list costs more than the order gains, and the workgroups go by tile, those of a pair's
// second tile returning at once; tiles go round the XCDs two by two, so that those do not idle the XCDs of one parity.
// Measured (35B layer, 1999 rows), list against tiles: gate/up of K 2048 160 against 178 us, down of K 512 136 against
// 121; 512 rows, down of K 768 45 against 50. By rows an expert, af4g64 blocks, list against tiles: 4 (256 experts of
// 2048 x 512) 130 against 125 us, 17 (60 of 2048 x 1280) 103 against 100, 32 (128 of 2048 x 768) 157 against 167, 34
// (60) 139 against 153. Launches that hold shared tiles keep the list: Q8_0 with its shared slice, 64 rows, 198 against
// 219.
constexpr uint32_t kListedRows = 24;
template <uint32_t FMT>
__global__ __launch_bounds__(64 * kWaves) __attribute__((amdgpu_waves_per_eu(4)))
void expert_wide_kernel(MoeExpertArgs a) {
  using F = Fmt<FMT>;
  constexpr int kLds = 2 * kStageBytes > kTensorWaves * 2 * 4096 ? 2 * kStageBytes : kTensorWaves * 2 * 4096;
  static_assert(kMaxTiles * 4 <= kLds, "the list and the experts fit the stages");
  __shared__ __attribute__((aligned(1024))) uint8_t lds[kLds];
  const int lane = threadIdx.x & 63;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t turn = blockIdx.x / 8 / a.column_groups, group = blockIdx.x / 8 % a.column_groups, xcd = blockIdx.x % 8;
  uint32_t tile, rows;
  SqMoeTileDescriptor d;
  if (a.listed) {
    const uint32_t n = min(a.tile_count->tiles, kMaxTiles), which = turn * 8 + xcd;
    if (which >= n) return;
    uint16_t *const list = (uint16_t *)lds;
    if (which >= work_list(a, n, list + kMaxTiles, list)) return;
    const uint32_t entry = __builtin_amdgcn_readfirstlane(list[which]);
    __syncthreads();   // the list's place is the stages'
    tile = entry >> 1;
    d = a.tiles[tile];
    rows = d.rows + (entry & 1 ? a.tiles[tile + 1].rows : 0u);
  } else {
    tile = turn / 2 * 16 + xcd * 2 + turn % 2;
    // The lane's tile before this one, the tile and the next, with the count: one round of loads.
    const uint32_t count = a.tile_count->tiles, back = lane + 1;
    const bool in = tile < a.max_tiles;
    const uint32_t earlier = in && back <= tile ? a.tiles[tile - back].expert : ~0u;
    const SqMoeTileDescriptor none{~0u, 0};
    const SqMoeTileDescriptor next = tile + 1 < a.max_tiles ? a.tiles[tile + 1] : none;
    d = in ? a.tiles[tile] : none;
    if (tile >= count || (a.mode != 2 && (d.expert >= a.experts) != (a.mode == 1))) return;
    rows = d.rows;
    if (!a.single) {
      uint64_t alike = __ballot(earlier == d.expert);
      uint32_t before = 0;
      while (alike == ~0ull) {
        before += 64;
        alike = __ballot(before + back <= tile && a.tiles[tile - before - back].expert == d.expert);
      }
      if ((before + __builtin_ctzll(~alike)) & 1) return;
      if (tile + 1 < count && next.expert == d.expert) rows += next.rows;
    }
  }
  // Wave-uniform, spelled out: the walk's buffer resources are built from them.
  tile = __builtin_amdgcn_readfirstlane(tile);
  rows = __builtin_amdgcn_readfirstlane(rows);
  const uint32_t expert = __builtin_amdgcn_readfirstlane(d.expert);
  const bool shared = expert >= a.experts;
  const uint32_t first_row = tile * a.tile_rows, G = a.K >> 5, column_tiles = a.output_size / 64;
  // The wave's 32 columns: block c of its tensor.
  const int t = a.gate_up && wave >= kTensorWaves ? 1 : 0;
  const uint32_t c = a.gate_up ? group * kTensorWaves + wave % kTensorWaves : group * kWaves + wave;
  const bool live = c < 2 * column_tiles;   // a spare wave walks the last block and stores nothing
  const uint32_t block = live ? c : 2 * column_tiles - 1;
  const size_t pt = (size_t)(shared ? expert - a.experts : a.slots[expert]) * column_tiles + block / 2;
  const uint8_t *const plane = (shared ? a.shared_plane0[t] : a.plane0[t]) + pt * G * 64 * F::P0;
  const uint8_t *const high = F::P1 ? (shared ? a.shared_plane1[t] : a.plane1[t]) + pt * G * 64 * F::P1 : nullptr;
  const uint8_t *const meta = (shared ? a.shared_meta[t] : a.meta[t]) + pt * (G / F::UNIT) * 64 * F::META;
  const bool tall = rows > 32;
  const uint32_t r = tall ? stage_row<2>() : stage_row<1>(), row = r < rows ? r : 0u;
  const uint32_t source = a.gather ? a.routes[first_row + row] / a.routes_per_row : first_row + row;
  RowSource<FMT> from;
  if constexpr (kRowSpans<FMT>) from = source * (a.K / 64);
  else from = a.input + (size_t)source * a.K + 8 * (lane & 7);
  const auto clear16 = [&](f32x16 &v) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 16; ++i) v[i] = 0.0f;
  };
  if (tall) {
    f32x16 acc[2];
    clear16(acc[0]);
    clear16(acc[1]);
    wide_walk<FMT, 2, 16>(a, plane, high, meta, 32 * (block & 1), from, rows, lds, acc);
    wide_store(a, acc, first_row, rows, 32 * c, live, lds);
  } else {
    f32x16 acc[1];
    clear16(acc[0]);
    if (rows > 16) wide_walk<FMT, 1, 16>(a, plane, high, meta, 32 * (block & 1), from, rows, lds, acc);
    else wide_walk<FMT, 1, 8>(a, plane, high, meta, 32 * (block & 1), from, rows, lds, acc);
    wide_store(a, acc, first_row, rows, 32 * c, live, lds);
  }
}

template <uint32_t FMT>
hipError_t launch_format(const MoeExpertArgs &args, hipStream_t stream) {
  MoeExpertArgs a = args;
  const uint32_t blocks = a.output_size / 32, per = a.gate_up ? kTensorWaves : kWaves;
  a.column_groups = (blocks + per - 1) / per;
  a.listed = a.K >= 768 && (a.mode != 0 || a.routed > kListedRows * a.experts);
  const uint32_t grid = a.column_groups * ((a.max_tiles + 15) / 16) * 16;
  hipLaunchKernelGGL(expert_wide_kernel<FMT>, dim3(grid), dim3(64 * kWaves), 0, stream, a);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_moe_expert(const MoeExpertArgs &a, hipStream_t stream) {
  if (a.tile_rows != 32 || !a.max_tiles || a.max_tiles > kMaxTiles) return hipErrorInvalidValue;
  switch (a.fmt) {
    case SQ_FMT_AF4G32: return launch_format<SQ_FMT_AF4G32>(a, stream);
    case SQ_FMT_AF4G64: return launch_format<SQ_FMT_AF4G64>(a, stream);
    case SQ_FMT_AF4G128: return launch_format<SQ_FMT_AF4G128>(a, stream);
    case SQ_FMT_Q4K: return launch_format<SQ_FMT_Q4K>(a, stream);
    case SQ_FMT_Q5K: return launch_format<SQ_FMT_Q5K>(a, stream);
    case SQ_FMT_Q6K: return launch_format<SQ_FMT_Q6K>(a, stream);
    case SQ_FMT_Q80: return launch_format<SQ_FMT_Q80>(a, stream);
    case SQ_FMT_AF8G64: return launch_format<SQ_FMT_AF8G64>(a, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace sq::kern
