// The narrow prefill tile: the prefill projection (prefill.hip: fp16 weights rounded once from fp32, the half rows
// table, fp32 sums) for dispatches whose 256-column tiles would leave most compute units idle.
//
// CDNA4 mapping. A workgroup of eight waves computes 64 or 96 rows x 32 or 64 columns; the waves split K in slices
// of whole 64-input steps and each walks its slice by itself, so the step loop has no barrier; the slices' fp32 sums
// meet in LDS in slice order. It costs more a step than the wide tile for the same outputs (its weights are dequantised
// for fewer rows, its rows read for fewer columns), and pays where the wide one would run a few workgroups through all
// of K: measured, Q4_K, wide -> narrow, N 5120 x K 6144 at 77 / 256 / 512 rows 98 / 100 / 102 -> 22 / 31 / 64 us, N
// 4096 x K 14336 at 48 / 256 / 512 rows 223 / 226 / 227 -> 32 / 54 / 104, N 1024 x K 4096 at 1024 rows 68 -> 20; N
// 14336 x K 4096 at 512 rows would go 87 -> 129 (prefill_narrow draws the line). Bound by instruction issue (the
// dequantisation) where the chip is full, by the waves' step chains where it is not; sixteen waves a workgroup measured
// no faster. Per step a wave
//  - brings the rows' 128 bytes as they lie (eight lanes a row, whole cache lines; fragment loads straight from memory
//    would touch a line a lane) into registers a step ahead, and turns them into the MFMA's layout through its own LDS
//    (the swizzle of chunk_slot, conflict-free both ways);
//  - brings 32 columns' codes of both groups (64 columns: of a group) with one 16-byte load a lane and transposes the
//    words across the wave's 16-lane rows in registers (transpose4), and derives one (column, group)'s coefficients a
//    lane, which the others read from LDS;
//  - dequantises a group's words and runs its 16x16x32 f16 MFMAs, weights x activations, so a lane ends with four
//    consecutive columns of a row.
#include <algorithm>

#include "device.hpp"
#include "half_rows.hpp"
#include "kernels.hpp"
#include "rowtile.hpp"

namespace sq::kern {
namespace {

constexpr int kNarrowWaves = 8;
typedef _Float16 half2 __attribute__((ext_vector_type(2)));
typedef float float2v __attribute__((ext_vector_type(2)));

__device__ __forceinline__ float byte_of(uint32_t v, int b) { return (float)((v >> (8 * b)) & 0xFFu); }
// fp16(fma(q, s, z)) of two codes: rounded to fp32 by the fma, then to fp16 (the empty asm keeps the two apart).
__device__ __forceinline__ uint32_t weight_pair(float q0, float q1, Coef k) {
  float v0 = fmaf(q0, k.s, k.z), v1 = fmaf(q1, k.s, k.z);
  asm volatile("" : "+v"(v0), "+v"(v1));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(float2v{v0, v1}, half2));
}
// Byte offset of 16-byte chunk c of row r of a wave's activations.
__device__ __forceinline__ uint32_t chunk_slot(uint32_t r, uint32_t c) { return r * 128 + ((c ^ (r & 7)) << 4); }

// The eight fp16 weights of a chunk (the MFMA's A operand): plane word w0 (8-bit codes: w0 then w1), its plane1 bits,
// and the group's coefficients (Q6_K: of its two halves).
template <uint32_t FMT>
__device__ __forceinline__ u32x4 chunk_weights(uint32_t w0, uint32_t w1, uint32_t high, uint32_t mask, Coef k,
                                               Coef k2) {
  using F = Fmt<FMT>;
  u32x4 o;
  if constexpr (F::P0 == 32) {
    const uint32_t flip = FMT == SQ_FMT_Q80 ? 0x80808080u : 0u;   // the signed byte v as v + 128
    const uint32_t a = w0 ^ flip, b = w1 ^ flip;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const uint32_t src = r >> 1 ? b : a;
      o[r] = weight_pair(byte_of(src, 2 * (r & 1)), byte_of(src, 2 * (r & 1) + 1), k);
    }
  } else {
    // lo: the word's slots 0, 4, 1, 5, hi: 2, 6, 3, 7, a byte each; plane1 bits go above them.
    uint32_t lo = w0 & mask, hi = (w0 >> 4) & mask;
    if constexpr (F::P1 == 4) {
      lo |= ((high & 0x33u) * 0x880110u) & 0x10101010u;
      hi |= (((high >> 2) & 0x33u) * 0x880110u) & 0x10101010u;
    } else if constexpr (F::P1 == 8) {
      lo |= ((high & 0x0303u) << 4) | ((high & 0x0C0Cu) << 18);
      hi |= (high & 0x3030u) | ((high & 0xC0C0u) << 14);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const uint32_t src = r & 1 ? hi : lo;
      o[r] = weight_pair(byte_of(src, r >> 1), byte_of(src, (r >> 1) + 2), F::HALVES && r >= 2 ? k2 : k);
    }
  }
  return o;
}

// NT column blocks of 16 (2 or 4), MI row blocks of 16 (4 or 6).
template <uint32_t FMT, int MI, int NT>
__global__ __launch_bounds__(64 * kNarrowWaves) __attribute__((amdgpu_waves_per_eu(2)))
void narrow_kernel(PrefillArgs a, uint32_t epilogue) {
  using F = Fmt<FMT>;
  constexpr int W = kNarrowWaves, BM = 16 * MI, NC = 16 * NT, XL = BM / 8;   // XL: 16-byte loads a lane for a step's rows
  constexpr int kRowBytes = BM * 128, kWave = kRowBytes + 2 * NC * 8;
  constexpr int kUnits = MI * NT, kPass = W < kUnits ? W : kUnits;   // f32x4 sums a lane, and those met at a time
  constexpr int kLds = W * (kWave > kPass * 1024 ? kWave : kPass * 1024);
  static_assert(kLds <= 160 * 1024, "the waves' activations and the sums fit the LDS");
  __shared__ __attribute__((aligned(1024))) uint8_t lds[kLds];
  const int lane = threadIdx.x & 63, j = lane & 15, q = lane >> 4;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t G = a.K >> 5, units = G / F::UNIT, steps = a.K / 64;
  const uint32_t first = __builtin_amdgcn_readfirstlane(steps * wave / W);
  const uint32_t end = __builtin_amdgcn_readfirstlane(steps * (wave + 1) / W);
  const uint32_t row0 = blockIdx.y * BM;
  uint32_t ptile = NT == 4 ? blockIdx.x : blockIdx.x >> 1, s = 0;
  const uint32_t c0 = NT == 4 ? 0u : (blockIdx.x & 1) * 32;   // the workgroup's first column of the plane tile
  while (s + 1 < a.segments && ptile >= a.seg[s].tiles) ptile -= a.seg[s++].tiles;
  const Segment seg = a.seg[s];

  f32x4 acc[MI][NT];
#pragma unroll
  for (int mi = 0; mi < MI; ++mi)
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[mi][t] = f32x4{0.f, 0.f, 0.f, 0.f};

  if (first < end) {
    uint8_t *const xs = lds + wave * kWave;
    float *const cs = (float *)(xs + kRowBytes);   // (s, z) or half scales of [group][column]
    // The lane's column and (32 columns) its group of a step.
    const uint32_t col = NT == 4 ? lane : c0 + (lane & 31), half = NT == 4 ? 0u : lane >> 5;
    // Buffer resources over the tile's planes and the workgroup's own rows (32-bit lane offsets, the step's offset
    // scalar; the extent of a whole chunk's rows would wrap from 4 GiB on, 2048 rows of K 2^20, and every load then
    // read zeros).
    const uint32_t live = min((uint32_t)BM, a.rows - row0);
    const auto planes = buffer_rsrc(seg.plane0 + (size_t)ptile * G * 64 * F::P0, G * 64 * F::P0);
    const auto metas = buffer_rsrc(seg.meta + (size_t)ptile * units * 64 * F::META, units * 64 * F::META);
    const auto highs = buffer_rsrc(F::P1 ? seg.plane1 + (size_t)ptile * G * 64 * F::P1 : nullptr, G * 64 * F::P1);
    const auto rows = buffer_rsrc(a.half_input + (size_t)row0 * a.K, live * a.K * 2);
    const uint32_t pv = (half * 64 + col) * F::P0, hv = (c0 + j) * F::P1 + q * (F::P1 / 4);
    const uint32_t mv = (F::UNIT == 1 ? half * 64 + col : col) * F::META;
    uint32_t xv[XL];
#pragma unroll
    for (int i = 0; i < XL; ++i)
      xv[i] = min(8u * i + (lane >> 3), live - 1) * a.K * 2 + (lane & 7) * 16;
    constexpr int CG = NT / 2;                            // code loads a step: groups a lane holds (1 or 2)
    constexpr int MU = NT == 4 && F::UNIT == 1 ? 2 : 1;   // meta units a lane reads a step
    u32x4 x[XL], codes[CG], codes_hi[F::P0 == 32 ? CG : 1];
    uint32_t hb[F::P1 ? 2 : 1][NT];
    MetaWords mw[MU];
    const auto issue = [&](uint32_t step) __attribute__((always_inline)) {
#pragma unroll
      for (int c = 0; c < CG; ++c) {
        const uint32_t at = (2 * step + c) * 64 * F::P0;
        codes[c] = buffer_b128<0>(planes, pv, at);
        if constexpr (F::P0 == 32) codes_hi[c] = buffer_b128<0>(planes, pv, at + 16);
      }
#pragma unroll
      for (int m = 0; m < MU; ++m)
        mw[m] = buffer_meta<FMT>(metas, mv, (2 * step + m) / F::UNIT * 64 * F::META);
      if constexpr (F::P1 != 0) {
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int t = 0; t < NT; ++t) {
            const uint32_t at = ((2 * step + h) * 64 + 16 * t) * F::P1;
            if constexpr (F::P1 == 4) hb[h][t] = __builtin_amdgcn_raw_buffer_load_b8(highs, hv, at, 0);
            else hb[h][t] = __builtin_amdgcn_raw_buffer_load_b16(highs, hv, at, 0);
          }
      }
#pragma unroll
      for (int i = 0; i < XL; ++i) x[i] = buffer_b128<0>(rows, xv[i], step * 128);
    };
    uint32_t mask = 0x0F0F0F0Fu;
    asm volatile("" : "+s"(mask));
    const uint32_t to = chunk_slot(lane >> 3, lane & 7);
    issue(first);
#pragma unroll 1
    for (uint32_t step = first; step < end; ++step) {
      // This step's words, coefficients and rows; the next step's loads go out as soon as theirs are used.
      uint32_t w0[2][NT], w1[2][NT], h1[2][NT];
#pragma unroll
      for (int c = 0; c < CG; ++c) {
        if constexpr (F::P0 == 32) {
          uint32_t e[4] = {codes[c][0], codes[c][2], codes_hi[c][0], codes_hi[c][2]};
          uint32_t o[4] = {codes[c][1], codes[c][3], codes_hi[c][1], codes_hi[c][3]};
          transpose4(e);
          transpose4(o);
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            w0[NT == 4 ? c : r >> 1][NT == 4 ? r : r & 1] = e[r];
            w1[NT == 4 ? c : r >> 1][NT == 4 ? r : r & 1] = o[r];
          }
        } else {
          uint32_t r4[4] = {codes[c][0], codes[c][1], codes[c][2], codes[c][3]};
          transpose4(r4);
#pragma unroll
          for (int r = 0; r < 4; ++r) w0[NT == 4 ? c : r >> 1][NT == 4 ? r : r & 1] = r4[r];
        }
      }
#pragma unroll
      for (int g = 0; g < (NT == 4 ? 2 : 1); ++g) {
        const uint32_t group = 2 * step + half + g;
        const MetaWords &m = mw[MU == 2 ? g : 0];
        f32x4 k;
        if constexpr (F::HALVES) {
          k[0] = q6k_scale(m, group, 0);
          k[1] = q6k_scale(m, group, 1);
        } else {
          const Coef c = coef<FMT>(m, group);
          k[0] = c.s;
          k[1] = FMT == SQ_FMT_Q80 ? -128.0f * c.s : c.z;
        }
        const uint32_t at = ((half + g) * NC + (NT == 4 ? lane : lane & 31)) * 2;
        *(float2v *)(cs + at) = float2v{k[0], k[1]};
      }
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int t = 0; t < NT; ++t) h1[h][t] = F::P1 ? hb[F::P1 ? h : 0][t] : 0u;
#pragma unroll
      for (int i = 0; i < XL; ++i) *(u32x4 *)(xs + i * 1024 + to) = x[i];
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      issue(__builtin_amdgcn_readfirstlane(min(step + 1, end - 1)));
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        u32x4 w[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          const float2v k = *(const float2v *)(cs + (h * NC + 16 * t + j) * 2);
          const Coef k1 = F::HALVES ? Coef{k[0], -32.0f * k[0]} : Coef{k[0], k[1]};
          const Coef k2 = F::HALVES ? Coef{k[1], -32.0f * k[1]} : k1;
          w[t] = chunk_weights<FMT>(w0[h][t], F::P0 == 32 ? w1[h][t] : 0u, h1[h][t], mask, k1, k2);
        }
#pragma unroll
        for (int mi = 0; mi < MI; ++mi) {
          const u32x4 f = *(const u32x4 *)(xs + chunk_slot(16 * mi + j, 4 * h + q));
#pragma unroll
          for (int t = 0; t < NT; ++t) acc[mi][t] = mfma_f16(w[t], f, acc[mi][t]);
        }
      }
      // The wave's reads precede its next step's writes.
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
  }

  // The slices meet in LDS, kPass of the lane's sums at a time: unit u (row block u / NT, column block u % NT) belongs
  // to wave u % 8, which adds it over the slices in slice order and stores its four columns of a row.
  f32x4 *const red = (f32x4 *)lds;   // [slice][unit of the pass][lane]
  const uint32_t col0 = seg.out_offset + ptile * 64 + c0;
#pragma unroll
  for (int p = 0; p < kUnits; p += kPass) {
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kPass && p + u < kUnits; ++u)
      red[(wave * kPass + u) * 64 + lane] = acc[(p + u) / NT][(p + u) % NT];
    __syncthreads();
    const uint32_t u = wave < kPass ? wave : kUnits, r = row0 + (p + u) / NT * 16 + j, c = col0 + (p + u) % NT * 16 + 4 * q;
    if (p + u < kUnits && r < a.rows) {
      f32x4 part[W];
#pragma unroll
      for (int k = 0; k < W; ++k) part[k] = red[(k * kPass + u) * 64 + lane];
      f32x4 sum = part[0];
#pragma unroll
      for (int k = 1; k < W; ++k) sum += part[k];
      const float scale = a.row_scale[r];
      const size_t at = (size_t)r * a.out_stride + c;
      u32x2 x = {0u, 0u}, out;
      if (epilogue != EpNone) x = *(const u32x2 *)(a.aux + at);
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        float v0 = sum[2 * e] * scale, v1 = sum[2 * e + 1] * scale;
        if (epilogue == EpResidual) {
          v0 = epilogue_bits<EpResidual>(v0, x[e] & 0xFFFFu);
          v1 = epilogue_bits<EpResidual>(v1, x[e] >> 16);
        } else if (epilogue == EpUpWithGate) {
          v0 = epilogue_bits<EpUpWithGate>(v0, x[e] & 0xFFFFu);
          v1 = epilogue_bits<EpUpWithGate>(v1, x[e] >> 16);
        }
        out[e] = (uint32_t)f32_to_bf16(v0) | ((uint32_t)f32_to_bf16(v1) << 16);
      }
      *(u32x2 *)(a.output + at) = out;
    }
  }
}

template <uint32_t FMT>
hipError_t launch_format(uint32_t epilogue, const PrefillArgs &a, PrefillNarrow n, hipStream_t stream) {
  uint32_t tiles = 0;
  for (uint32_t s = 0; s < a.segments; ++s) tiles += a.seg[s].tiles;
  const dim3 grid(tiles * 64 / n.columns, (a.rows + n.rows - 1) / n.rows), block(64 * kNarrowWaves);
  const uint32_t shape = n.rows * 100 + n.columns;
  switch (shape) {
#define SQ_NARROW(MI, NT) \
  case 1600 * MI + 16 * NT: \
    hipLaunchKernelGGL((narrow_kernel<FMT, MI, NT>), grid, block, 0, stream, a, epilogue); \
    break;
    SQ_NARROW(4, 2) SQ_NARROW(4, 4) SQ_NARROW(6, 2) SQ_NARROW(6, 4)
#undef SQ_NARROW
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace

hipError_t launch_prefill_narrow(uint32_t fmt, uint32_t epilogue, const PrefillArgs &a, PrefillNarrow n,
                                 hipStream_t stream) {
  switch (fmt) {
    case SQ_FMT_AF4G32: return launch_format<SQ_FMT_AF4G32>(epilogue, a, n, stream);
    case SQ_FMT_AF4G64: return launch_format<SQ_FMT_AF4G64>(epilogue, a, n, stream);
    case SQ_FMT_AF4G128: return launch_format<SQ_FMT_AF4G128>(epilogue, a, n, stream);
    case SQ_FMT_Q4K: return launch_format<SQ_FMT_Q4K>(epilogue, a, n, stream);
    case SQ_FMT_Q5K: return launch_format<SQ_FMT_Q5K>(epilogue, a, n, stream);
    case SQ_FMT_Q6K: return launch_format<SQ_FMT_Q6K>(epilogue, a, n, stream);
    case SQ_FMT_Q80: return launch_format<SQ_FMT_Q80>(epilogue, a, n, stream);
    case SQ_FMT_AF8G64: return launch_format<SQ_FMT_AF8G64>(epilogue, a, n, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace sq::kern
