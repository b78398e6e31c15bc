// MoE block: top-k route select and shared-slice weights, grouping of routes into expert tiles, the expert passes
// (gate and up in one pass, then down) and the combine (reference: kernels/shared/moe.metal:23-162,175-331,480-505
// and kernels/shared/moe_gguf.metal:21-206).
//
// CDNA4 mapping. Each expert pass is the decode row tile's exact-operand arithmetic (rowtile.hpp) per expert tile: the
// 8-row tiles here, the 32-row ones in moe_wide.hip. The passes read their input rows in the tile's read order (one
// 16-byte chunk holds an MFMA operand): the routed work opens by writing the block's input rows in that order, and the
// gate/up pass writes the intermediate rows in it.
#include "kernels.hpp"
#include "rowtile.hpp"

namespace sq::kern {
namespace {

// A 64-lane reduction by DPP row operations (dpp_ctrl quad_perm [1,0,3,2], quad_perm [2,3,0,1], row_half_mirror,
// row_mirror, then row_bcast15 into rows 1 and 3 and row_bcast31 into rows 2 and 3): after the six steps lane 63
// holds op over all 64 lanes, which readlane gives every lane. op must be associative, commutative and idempotent
// (a row the mask leaves out combines a value with itself).
template <int CTRL, int ROWS>
__device__ __forceinline__ uint32_t dpp_row(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, CTRL, ROWS, 0xF, false);
}
template <typename Op>
__device__ __forceinline__ uint32_t wave_reduce(uint32_t v, Op op) {
  v = op(v, dpp_row<0xB1, 0xF>(v));
  v = op(v, dpp_row<0x4E, 0xF>(v));
  v = op(v, dpp_row<0x141, 0xF>(v));
  v = op(v, dpp_row<0x140, 0xF>(v));
  v = op(v, dpp_row<0x142, 0xA>(v));
  v = op(v, dpp_row<0x143, 0xC>(v));
  return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}

// One wave per row (moe.metal:23-112). Rank by rank, the highest remaining score wins, the lowest expert id among
// equal scores; the router then weights the top_k routes in rank order: Softmax weight_r =
// 2^((s_r - s_0) log2 e) / sum_o 2^((s_o - s_0) log2 e), SigmoidNormalized weight_r = sigmoid(s_r) /
// (sum_o sigmoid(s_o) + 1e-20). The row's routes top_k .. top_k + shared - 1 are the shared expert's slices (ids
// experts on), each weighted by sigmoid(x . g) of the block's fp32 scalar gate g (gated) or by 1.
__global__ __launch_bounds__(128) void route_select_kernel(const float *scores, uint32_t stride, uint32_t *selected,
                                                          float *weights, SqMoeRouteParams p, const uint16_t *input,
                                                          const float *shared_gate, uint32_t router, uint32_t shared,
                                                          uint16_t *rows_table) {
  constexpr int kPer = SQ_MOE_WIDE_EXPERT_SLOTS / 64;
  const uint32_t row = blockIdx.x, lane = threadIdx.x & 63, per_row = p.top_k + shared;
  const size_t base = (size_t)row * per_row;
  if (threadIdx.x >= 64) {
    // The second wave (launched with rows_table only): the row in the tiles' read order (input_rows_kernel's 16-byte
    // chunks, lane l the row's chunks l, l + 64, ...), beside the first wave's selection.
    const uint16_t *xr = input + (size_t)row * p.input_size;
    uint16_t *out = rows_table + (size_t)row * p.input_size;
    for (uint32_t i = lane; i < p.input_size / 8; i += 64) {
      const uint32_t *in = (const uint32_t *)(xr + 32 * (i / 4)) + 2 * (i % 4);
      const u32x2 lo = *(const u32x2 *)in, hi = *(const u32x2 *)(in + 8);
      *(u32x4 *)(out + 8 * i) = u32x4{lo[0], lo[1], hi[0], hi[1]};
    }
    return;
  }
  if (shared) {
    float gate = 1.0f;
    if (shared_gate) {
      float dot = 0.0f;
      const uint16_t *xr = input + (size_t)row * p.input_size;
      if (p.input_size % 512 == 0) {
        // Eight inputs a lane a step (one 16-byte load of the row, two of the gate), four steps' loads in flight.
#pragma unroll 4
        for (uint32_t d = 8 * lane; d < p.input_size; d += 512) {
          const u32x4 x = *(const u32x4 *)(xr + d);
          const f32x4 g0 = *(const f32x4 *)(shared_gate + d), g1 = *(const f32x4 *)(shared_gate + d + 4);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float ge = e < 2 ? g0[2 * e] : g1[2 * e - 4], go = e < 2 ? g0[2 * e + 1] : g1[2 * e - 3];
            dot = fmaf(bf16_to_f32(x[e] & 0xFFFFu), ge, dot);
            dot = fmaf(bf16_to_f32(x[e] >> 16), go, dot);
          }
        }
      } else {
        for (uint32_t d = lane; d < p.input_size; d += 64) dot = fmaf(bf16_to_f32(xr[d]), shared_gate[d], dot);
      }
#pragma unroll
      for (int m = 32; m >= 1; m >>= 1) dot += __shfl_xor(dot, m);
      gate = sigmoid(dot);
    }
    if (lane < shared) {
      selected[base + p.top_k + lane] = p.experts + lane;
      weights[base + p.top_k + lane] = gate;
    }
  }
  float v[kPer];
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const uint32_t e = lane + 64u * i;
    v[i] = e < p.experts ? scores[(size_t)row * stride + e] : -INFINITY;
  }
  __shared__ float ordered[64];
  // A lane's best starts at -inf in its first slot and moves only to a strictly greater score, so a NaN score never
  // becomes a lane's best and the wave maximum sees no NaN; a taken expert's score becomes -inf (moe.metal:77-93).
  // Every lane offers at least its first slot, so the winner is always an expert id below `experts`: when no finite
  // score is left, every lane's best is -inf and lane 0's expert 0 wins (the reference's choice too).
  for (uint32_t rank = 0; rank < p.top_k; ++rank) {
    float best = -INFINITY;
    int at = 0;
#pragma unroll
    for (int i = 0; i < kPer; ++i)
      if (v[i] > best) best = v[i], at = i;
    const float top = __uint_as_float(wave_reduce(__float_as_uint(best), [](uint32_t a, uint32_t b) {
      return __float_as_uint(fmaxf(__uint_as_float(a), __uint_as_float(b)));
    }));
    const uint32_t candidate = best == top ? lane + 64u * at : 0xFFFFFFFFu;
    const uint32_t winner = wave_reduce(candidate, [](uint32_t a, uint32_t b) { return min(a, b); });
#pragma unroll
    for (int i = 0; i < kPer; ++i)
      if (candidate == winner && i == at) v[i] = -INFINITY;
    if (lane == 0) {
      selected[base + rank] = winner;
      ordered[rank] = top;
    }
  }
  // One wave selects (a second one, if any, returned above): lane 0's LDS writes reach its other lanes.
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  for (uint32_t rank = lane; rank < p.top_k; rank += 64) {
    float denominator = 0.0f;
    if (router == SQ_MOE_ROUTER_SOFTMAX) {
      for (uint32_t o = 0; o < p.top_k; ++o) denominator += exp2f((ordered[o] - ordered[0]) * 1.44269504089f);
      weights[base + rank] = exp2f((ordered[rank] - ordered[0]) * 1.44269504089f) / denominator;
    } else {
      for (uint32_t o = 0; o < p.top_k; ++o) denominator += sigmoid(ordered[o]);
      weights[base + rank] = sigmoid(ordered[rank]) / (denominator + 1e-20f);
    }
  }
}

// One workgroup groups every route (moe.metal:184-278): count per expert, exclusive prefix of the experts' tiles in
// expert order, tile descriptors, then each routed route's grouped row. Routes of an expert take its rows in route
// order (a bitmap of the rows that route to each expert, 512 rows at a time, gives a route's rank), so the
// grouping, and every expert pass after it, is deterministic. The `shared` slices' tiles follow the routed tiles,
// slice after slice, each slice's holding every row in order (route row * (top_k + shared) + top_k + slice).
// With verify_rows (a verify step: a live-row count per lane of lane_rows rows) the routed routes of a row past its
// lane's count are grouped into no tile and their route_rows are ~0u (moe_group_routes_verified,
// moe.metal:164-173); the shared slices still hold every row.
__global__ __launch_bounds__(512) void group_kernel(const uint32_t *selected, SqMoeTileDescriptor *tiles,
                                                    SqMoeTileCount *tile_count, uint32_t *grouped_routes,
                                                    uint32_t *route_rows, const uint32_t *verify_rows,
                                                    SqMoeGroupParams p, uint32_t shared) {
  // The row bitmaps and their prefixes: an expert's kWords words at a stride of kStride, so that the threads that
  // walk their experts' words together (thread e, word w) take different LDS banks.
  constexpr uint32_t kChunk = 512, kWords = kChunk / 32, kStride = kWords + 1;
  __shared__ uint32_t counts[SQ_MOE_WIDE_EXPERT_SLOTS], offsets[SQ_MOE_WIDE_EXPERT_SLOTS],
      running[SQ_MOE_WIDE_EXPERT_SLOTS];
  __shared__ uint32_t bits[SQ_MOE_WIDE_EXPERT_SLOTS * kStride], prefix[SQ_MOE_WIDE_EXPERT_SLOTS * kStride];
  __shared__ uint32_t total;
  const uint32_t tid = threadIdx.x, per_row = p.top_k + shared, tr = p.tile_rows;
  // Routed route k of row r: selected[r * per_row + k].
  const auto route_of = [&](uint32_t i) { return i / p.top_k * per_row + i % p.top_k; };
  // The route select writes expert ids below `experts` only; the clamp keeps a corrupted selection inside the
  // tables below.
  const auto expert_of = [&](uint32_t i) { return min(selected[route_of(i)], p.experts - 1u); };
  const auto dead = [&](uint32_t i) {
    const uint32_t row = i / p.top_k;
    return verify_rows != nullptr && row % p.lane_rows >= verify_rows[row / p.lane_rows];
  };
  // When one chunk takes every row and a row has at most kHeld routes, each thread loads its routes' expert ids once
  // (route tid + 512 k, k < top_k), counts them and sets their row bits in one pass, and ranks them from registers:
  // one read of the selection instead of three. Up to kStaged routes otherwise go through LDS once (each route's
  // expert id, ~0u for a dead one), which the passes below read instead of the selection.
  constexpr uint32_t kHeld = 8, kStaged = 4 * kChunk * kHeld;
  const uint32_t routes = p.rows * p.top_k;
  const bool one = p.rows <= kChunk && p.top_k <= kHeld, staged = !one && routes <= kStaged;
  __shared__ uint32_t stage[kStaged];
  // Route i's expert, or ~0u for a dead route.
  const auto live_expert = [&](uint32_t i) __attribute__((always_inline)) {
    return staged ? stage[i] : dead(i) ? ~0u : expert_of(i);
  };
  uint32_t held[kHeld];
#pragma unroll
  for (uint32_t k = 0; k < kHeld; ++k) {
    const uint32_t i = tid + 512 * k;
    held[k] = one && i < routes && !dead(i) ? expert_of(i) : ~0u;   // ~0u: no live route
  }
  __shared__ uint32_t duplicated;
  counts[tid] = 0;
  running[tid] = 0;
  if (one) {
    for (uint32_t i = tid; i < p.experts * kStride; i += 512) bits[i] = 0;
    if (tid == 0) duplicated = 0;
  }
  __syncthreads();
  if (one) {
#pragma unroll
    for (uint32_t k = 0; k < kHeld; ++k) {
      const uint32_t i = tid + 512 * k;
      if (i >= routes) continue;
      if (held[k] == ~0u) {
        route_rows[route_of(i)] = ~0u;
        continue;
      }
      const uint32_t local = i / p.top_k, bit = 1u << (local % 32);
      atomicAdd(&counts[held[k]], 1u);
      // A bit already set names another route of the same row to the same expert (see below).
      if (atomicOr(&bits[held[k] * kStride + local / 32], bit) & bit) duplicated = 1;
    }
  } else {
    for (uint32_t i = tid; i < routes; i += 512) {
      const uint32_t e = dead(i) ? ~0u : expert_of(i);
      if (staged) stage[i] = e;
      if (e != ~0u) atomicAdd(&counts[e], 1u);
    }
  }
  __syncthreads();
  {
    // Exclusive prefix of the experts' tile counts: a scan within each wave, then over the eight wave totals.
    __shared__ uint32_t wave_sum[8];
    const uint32_t mine = tid < p.experts ? (counts[tid] + tr - 1) / tr : 0u, lane = tid & 63, wave = tid >> 6;
    uint32_t inclusive = mine;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const uint32_t up = (uint32_t)__shfl_up((int)inclusive, d);
      if (lane >= (uint32_t)d) inclusive += up;
    }
    if (lane == 63) wave_sum[wave] = inclusive;
    __syncthreads();
    uint32_t before = 0;
    for (uint32_t w = 0; w < wave; ++w) before += wave_sum[w];
    offsets[tid] = before + inclusive - mine;
    if (tid == 511) total = before + inclusive;
  }
  __syncthreads();
  if (tid < p.experts) {
    const uint32_t c = counts[tid], n = (c + tr - 1) / tr, first = offsets[tid];
    for (uint32_t t = 0; t < n; ++t) tiles[first + t] = SqMoeTileDescriptor{tid, min(tr, c - t * tr)};
    for (uint32_t row = first * tr + c; row < (first + n) * tr; ++row) grouped_routes[row] = ~0u;
  }
  for (uint32_t chunk = 0; chunk < p.rows; chunk += kChunk) {
    const uint32_t i0 = chunk * p.top_k, i1 = min(p.rows, chunk + kChunk) * p.top_k;
    if (!one) {
      for (uint32_t i = tid; i < p.experts * kStride; i += 512) bits[i] = 0;
      if (tid == 0) duplicated = 0;
      __syncthreads();
    }
    for (uint32_t i = i0 + tid; !one && i < i1; i += 512) {
      const uint32_t e = live_expert(i);
      if (e == ~0u) {
        route_rows[route_of(i)] = ~0u;
        continue;
      }
      const uint32_t local = i / p.top_k - chunk, bit = 1u << (local % 32);
      // A bit already set names another route of the same row to the same expert: a row with fewer scores above
      // -inf than top_k routes (an all-NaN row selects expert 0 at every rank). Such a chunk is ranked serially.
      if (atomicOr(&bits[e * kStride + local / 32], bit) & bit) duplicated = 1;
    }
    __syncthreads();
    if (!duplicated) {
      // Rows of the chunk before word w that route to expert e: one pass per expert, then each route's rank is a
      // table read and one population count.
      if (tid < p.experts) {
        uint32_t before = 0;
        for (uint32_t w = 0; w < kWords; ++w) {
          prefix[tid * kStride + w] = before;
          before += __popc(bits[tid * kStride + w]);
        }
      }
      __syncthreads();
      const auto place = [&](uint32_t i, uint32_t e) __attribute__((always_inline)) {
        const uint32_t r = route_of(i), local = i / p.top_k - chunk;
        uint32_t rank = running[e] + prefix[e * kStride + local / 32];
        rank += __popc(bits[e * kStride + local / 32] & ((1u << (local % 32)) - 1u));
        const uint32_t row = offsets[e] * tr + rank;
        grouped_routes[row] = r;
        route_rows[r] = row;
      };
      if (one) {
#pragma unroll
        for (uint32_t k = 0; k < kHeld; ++k)
          if (tid + 512 * k < routes && held[k] != ~0u) place(tid + 512 * k, held[k]);
      } else {
        for (uint32_t i = i0 + tid; i < i1; i += 512) {
          const uint32_t e = live_expert(i);
          if (e != ~0u) place(i, e);
        }
      }
      __syncthreads();
      if (tid < p.experts) {
        uint32_t ranked = running[tid];
        for (uint32_t w = 0; w < kWords; ++w) ranked += __popc(bits[tid * kStride + w]);
        running[tid] = ranked;
      }
    } else if (tid < p.experts) {
      // Thread e takes its expert's routes of the chunk in route order.
      for (uint32_t i = i0; i < i1; ++i) {
        if (live_expert(i) != tid) continue;
        const uint32_t r = route_of(i), row = offsets[tid] * tr + running[tid]++;
        grouped_routes[row] = r;
        route_rows[r] = row;
      }
    }
    __syncthreads();
  }
  // Shared slices (moe.metal:245-270): slice s's tiles after slice s - 1's, each of every row in order.
  const uint32_t shared_tiles = (p.rows + tr - 1) / tr, shared_base = total * tr;
  for (uint32_t i = tid; i < shared * shared_tiles; i += 512) {
    const uint32_t slice = i / shared_tiles, t = i % shared_tiles;
    tiles[total + i] = SqMoeTileDescriptor{p.experts + slice, min(tr, p.rows - t * tr)};
  }
  for (uint32_t i = tid; i < shared * shared_tiles * tr; i += 512) {
    const uint32_t slice = i / (shared_tiles * tr), row = i % (shared_tiles * tr);
    if (row < p.rows) {
      const uint32_t r = row * per_row + p.top_k + slice;
      grouped_routes[shared_base + i] = r;
      route_rows[r] = shared_base + i;
    } else {
      grouped_routes[shared_base + i] = ~0u;
    }
  }
  if (tid == 0) {
    const uint32_t live = total + shared * shared_tiles;
    *tile_count = SqMoeTileCount{live, {p.gate_up_columns, live, 1}, {p.down_columns, live, 1}, {0, 0, 0}};
  }
}

// Wave `slice`'s groups of tensor slot n of column tile ct against the at most 16 rows of a small tile, into acc.
template <uint32_t FMT>
__device__ __forceinline__ void small_walk(const MoeExpertArgs &a, SqMoeTileDescriptor d, uint32_t first_row, int n,
                                           uint32_t ct, uint32_t slice, float (&acc)[1][4][1][4]) {
  using F = Fmt<FMT>;
  const int lane = threadIdx.x & 63, j = lane & 15, q = lane >> 4;
  const uint32_t G = a.K >> 5, spans = (G + 3) / 4;
  const uint32_t first = spans * slice / a.slices * 4, end = min(G, spans * (slice + 1) / a.slices * 4);
  if (first >= end) return;
  const bool shared = d.expert >= a.experts;
  const size_t pt = (size_t)(shared ? d.expert - a.experts : a.slots[d.expert]) * (a.output_size / 64) + ct;
  const uint8_t *const plane = (shared ? a.shared_plane0[n] : a.plane0[n]) + (pt * G * 64 + lane) * F::P0;
  const uint8_t *const high =
      F::P1 ? (shared ? a.shared_plane1[n] : a.plane1[n]) + (pt * G * 64 + lane) * F::P1 : nullptr;
  const uint8_t *const meta = (shared ? a.shared_meta[n] : a.meta[n]) + (pt * (G / F::UNIT) * 64 + lane) * F::META;
  const uint32_t r = (uint32_t)j < d.rows ? j : 0u;
  const uint32_t source = a.gather ? a.routes[first_row + r] / a.routes_per_row : first_row + r;
  const uint16_t *const xrow = a.input + (size_t)source * a.K + 8 * q;
  row_stream<FMT, F::SG <= 2 ? 2 : 4>(plane, high, meta, xrow, first, end, acc);
}

// The expert passes of 8-row tiles (decode steps and the smallest chunks: an expert's one to eight rows). There are few
// tiles and each wave's walk over K is a chain of loads it waits on, so K is cut into `slices` slices, a wave each, and
// a gate/up pass gives gate and up waves of their own: a workgroup's eight waves are the slices of the tensors of 8 /
// (slices x tensors) column tiles, their sums meet in LDS in slice order. One launch runs the routed and the shared
// tiles, each in its own format, so that the shared slices' long chains overlap the routed ones. 128 registers a wave
// (chunks of two groups, the shortest that hold whole scale groups), so that four waves share a SIMD. A pass of one
// tensor takes workgroups of four waves: a workgroup's registers and LDS are free again only when its last wave is
// done, and a pass of many tiles runs in rounds of them. Measured, 8 rows over 256 experts of 2048 x 512 (Q4_K gate/up,
// Q5_K down, a Q8_0 shared slice): gate/up 40.6 us routed and 62.5 us shared in two launches of whole-K waves -> 25 us;
// down 17.1 and 10.2 -> 17.5; at 170 registers 33 and 24. The block of 16 / 32 rows over 256 af4g64 experts of 2048 x
// 512: whole-K waves 64 / 87 us, eight waves and chunks of four groups 69 / 90, four waves in the down pass 66 / 87,
// and chunks of two 64 / 85; one wave running its column tile's slices in turn took 90 / 129, gate and up (or two
// column tiles) in one wave 75 / 106.
template <uint32_t WAVES>
__global__ __launch_bounds__(64 * WAVES) __attribute__((amdgpu_waves_per_eu(4)))
void expert_small_kernel(MoeExpertArgs a) {
  const uint32_t tile = blockIdx.y;
  if (tile >= a.tile_count->tiles) return;
  const SqMoeTileDescriptor d = a.tiles[tile];
  const int lane = threadIdx.x & 63, j = lane & 15, q = lane >> 4;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), tensors = a.gate_up ? 2 : 1;
  const uint32_t per = WAVES / (a.slices * tensors), ct0 = blockIdx.x * per;
  const uint32_t column = wave / (a.slices * tensors), n = wave / a.slices % tensors, slice = wave % a.slices;
  const uint32_t column_tiles = a.output_size / 64, first_row = tile * a.tile_rows;
  float acc[1][4][1][4];
  clear(acc);
  if (ct0 + column < column_tiles) {
    const uint32_t fmt = d.expert >= a.experts ? a.shared_fmt : a.fmt;
    with_format(fmt, [&](auto f) { small_walk<decltype(f)::value>(a, d, first_row, n, ct0 + column, slice, acc); });
  }
  // red[wave][4 t + i][lane]: column block t, row 4 q + i.
  __shared__ float red[WAVES][16][64];
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) red[wave][4 * t + i][lane] = acc[0][t][0][i];
  __syncthreads();
  const auto total = [&](uint32_t from, uint32_t f) __attribute__((always_inline)) {
    float v = 0.0f;
    for (uint32_t s = 0; s < a.slices; ++s) v += red[from + s][f][lane];
    return v;
  };
  for (uint32_t o = wave; o < per * 16; o += WAVES) {
    const uint32_t c = o / 16, f = o % 16, ct = ct0 + c, r = 4u * q + (f & 3), t = f >> 2;
    if (ct >= column_tiles || r >= d.rows) continue;
    // The gathering passes store at the column's place in the read order (chunk 4 g + j / 4 of its group, position
    // 4 (t % 2) + j % 4), the down pass in column order.
    const uint32_t place = a.gather ? 32 * (t >> 1) + 4 * (t & 1) + 8 * (j >> 2) + (j & 3) : 16 * t + j;
    const size_t at = (size_t)(first_row + r) * a.output_size + ct * 64 + place;
    const uint32_t from = c * a.slices * tensors;
    float v = total(from, f);
    if (a.gate_up) {
      const float u = bf16_to_f32(f32_to_bf16(total(from + a.slices, f)));
      v = u * silu(bf16_to_f32(f32_to_bf16(v)));
    } else if (a.gate) {
      v = bf16_to_f32(f32_to_bf16(v)) * silu(bf16_to_f32(a.gate[at]));
    }
    a.output[at] = f32_to_bf16(v);
  }
}

// Thread: one 16-byte chunk of the table, chunk c of a group of 32 inputs: its 4-input units c and c + 4 (inputs
// 4c..4c+3 and 16+4c..19+4c, the group's dwords 2c, 2c + 1 and 8 + 2c, 9 + 2c), the prefill's half rows order
// (half_rows.hpp). The reference's routed pass opens with its gather of the input rows into the grouped input
// (MoE.cpp:480-517); here the rows keep their order and the gate/up pass gathers through the routes as it reads.
// Four threads a group, so each wave reads and writes 1 KiB contiguous.
__global__ __launch_bounds__(256) void input_rows_kernel(const uint16_t *input, uint64_t chunks, uint16_t *table) {
  const uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;   // chunk i % 4 of group i / 4, rows back to back
  if (i >= chunks) return;
  const uint32_t *in = (const uint32_t *)(input + 32 * (i / 4)) + 2 * (i % 4);
  const u32x2 lo = *(const u32x2 *)in, hi = *(const u32x2 *)(in + 8);
  *(u32x4 *)(table + 8 * i) = u32x4{lo[0], lo[1], hi[0], hi[1]};
}

// out[r][d] = bf16(residual + sum_slot w_slot * expert_out[route_rows[slot]][d]) in slot order (moe.metal:480-505).
__global__ __launch_bounds__(256) void combine_kernel(const uint16_t *expert_output, const uint32_t *route_rows,
                                                      const float *weights, const uint16_t *residual,
                                                      uint16_t *output, SqMoeCombineParams p) {
  // Thread: eight consecutive outputs of row blockIdx.x (the hidden size is a multiple of 64).
  const uint32_t r = blockIdx.x, d = (blockIdx.y * 256 + threadIdx.x) * 8;
  if (d >= p.hidden_size) return;
  const size_t at = (size_t)r * p.hidden_size + d;
  float v[8];
  const u32x4 res = residual ? *(const u32x4 *)(residual + at) : u32x4{0u, 0u, 0u, 0u};
#pragma unroll
  for (int e = 0; e < 4; ++e) v[2 * e] = bf16_to_f32(res[e] & 0xFFFFu), v[2 * e + 1] = bf16_to_f32(res[e] >> 16);
  const size_t route = (size_t)r * p.routes_per_row;
  // Eight slots at a time: their route rows (one scalar load each: the row is the workgroup's), then every live
  // slot's 16 bytes in flight together, then the sums in slot order; the slots past the last eight one at a time. A
  // route row of ~0u (a dead verify row) adds nothing, not even a zero.
  constexpr uint32_t kBatch = 8;
  uint32_t s0 = 0;
  for (; s0 + kBatch <= p.routes_per_row; s0 += kBatch) {
    uint32_t grouped[kBatch];
    u32x4 x[kBatch];
    float w[kBatch];
#pragma unroll
    for (uint32_t k = 0; k < kBatch; ++k) {
      grouped[k] = route_rows[route + s0 + k];
      w[k] = 0.0f;
      x[k] = u32x4{0u, 0u, 0u, 0u};
      if (grouped[k] != ~0u) {
        w[k] = weights[route + s0 + k];
        x[k] = *(const u32x4 *)(expert_output + (size_t)grouped[k] * p.hidden_size + d);
      }
    }
#pragma unroll
    for (uint32_t k = 0; k < kBatch; ++k) {
      if (grouped[k] == ~0u) continue;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        v[2 * e] = fmaf(w[k], bf16_to_f32(x[k][e] & 0xFFFFu), v[2 * e]);
        v[2 * e + 1] = fmaf(w[k], bf16_to_f32(x[k][e] >> 16), v[2 * e + 1]);
      }
    }
  }
  for (; s0 < p.routes_per_row; ++s0) {
    const uint32_t grouped = route_rows[route + s0];
    if (grouped == ~0u) continue;
    const float w = weights[route + s0];
    const u32x4 x = *(const u32x4 *)(expert_output + (size_t)grouped * p.hidden_size + d);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      v[2 * e] = fmaf(w, bf16_to_f32(x[e] & 0xFFFFu), v[2 * e]);
      v[2 * e + 1] = fmaf(w, bf16_to_f32(x[e] >> 16), v[2 * e + 1]);
    }
  }
  u32x4 out;
#pragma unroll
  for (int e = 0; e < 4; ++e) out[e] = (uint32_t)f32_to_bf16(v[2 * e]) | ((uint32_t)f32_to_bf16(v[2 * e + 1]) << 16);
  *(u32x4 *)(output + at) = out;
}

}  // namespace

hipError_t launch_moe_route_select(const float *scores, uint32_t stride, uint32_t *selected, float *weights,
                                   const SqMoeRouteParams &p, const uint16_t *input, const float *shared_gate,
                                   uint32_t router, uint32_t shared, uint16_t *rows_table, hipStream_t stream) {
  if (rows_table && p.input_size % 32) return hipErrorInvalidValue;
  hipLaunchKernelGGL(route_select_kernel, dim3(p.rows), dim3(rows_table ? 128 : 64), 0, stream, scores, stride,
                     selected, weights, p, input, shared_gate, router, shared, rows_table);
  return hipGetLastError();
}

hipError_t launch_moe_group(const uint32_t *selected, SqMoeTileDescriptor *tiles, SqMoeTileCount *tile_count,
                            uint32_t *grouped_routes, uint32_t *route_rows, const uint32_t *verify_rows,
                            const SqMoeGroupParams &p, uint32_t shared, hipStream_t stream) {
  hipLaunchKernelGGL(group_kernel, dim3(1), dim3(512), 0, stream, selected, tiles, tile_count, grouped_routes,
                     route_rows, verify_rows, p, shared);
  return hipGetLastError();
}

hipError_t launch_moe_input_rows(const uint16_t *input, uint32_t rows, uint32_t K, uint16_t *table,
                                 hipStream_t stream) {
  if (K % 32) return hipErrorInvalidValue;
  const uint64_t chunks = (uint64_t)rows * (K / 32) * 4;
  hipLaunchKernelGGL(input_rows_kernel, dim3((uint32_t)((chunks + 255) / 256)), dim3(256), 0, stream, input, chunks,
                     table);
  return hipGetLastError();
}

hipError_t launch_moe_expert_small(const MoeExpertArgs &args, hipStream_t stream) {
  if (args.tile_rows > 16 || !args.max_tiles) return hipErrorInvalidValue;
  MoeExpertArgs a = args;
  // Slices of at least eight groups (the loads a wave keeps in flight) and at most four of them, in a power of two.
  const uint32_t spans = a.K / 32 / 4;
  a.slices = spans >= 8 ? 4 : spans >= 4 ? 2 : 1;
  const uint32_t waves = a.gate_up ? 8 : 4, per = waves / (a.slices * (a.gate_up ? 2 : 1));
  hipLaunchKernelGGL(waves == 4 ? expert_small_kernel<4> : expert_small_kernel<8>,
                     dim3((a.output_size / 64 + per - 1) / per, a.max_tiles), dim3(64 * waves), 0, stream, a);
  return hipGetLastError();
}

hipError_t launch_moe_combine(const uint16_t *expert_output, const uint32_t *route_rows, const float *weights,
                              const uint16_t *residual, uint16_t *output, const SqMoeCombineParams &p,
                              hipStream_t stream) {
  hipLaunchKernelGGL(combine_kernel, dim3(p.rows, (p.hidden_size / 8 + 255) / 256), dim3(256), 0, stream, expert_output,
                     route_rows, weights, residual, output, p);
  return hipGetLastError();
}

}  // namespace sq::kern
