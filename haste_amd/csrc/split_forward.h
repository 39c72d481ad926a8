// The forward recurrence of one XCD per batch tile with the step's product on the bf16 matrix cores, for any
// cell whose step is "sums of h * R per gate, then the pointwise step": the kernel, and what a cell supplies.
#pragma once

#include "split_operands.h"

namespace haste_hip {

template <int N>
__device__ __forceinline__ bool all_parts_written(const uint4_t (&v)[N]) {
  unsigned int m = 0u;
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const unsigned int xy = v[i].x > v[i].y ? v[i].x : v[i].y, zw = v[i].z > v[i].w ? v[i].z : v[i].w;
    const unsigned int q = xy > zw ? xy : zw;
    m = m > q ? m : q;
  }
  return __all(m != kUnwrittenBits) != 0;
}

template <int LANE>
__device__ __forceinline__ unsigned int quad_lane(unsigned int v) {
  return (unsigned int)__builtin_amdgcn_update_dpp(0, (int)v, LANE * 0x55, 0xf, 0xf, false);
}

// The parts of h, hi | mid << 16 in p12, lo in p3.  RAW (states that do not split): bits 31..16, 15..8 and 7..0.
__device__ __forceinline__ void split_state(float h, bool raw, unsigned int& p12, unsigned int& p3) {
  h = h != h ? __uint_as_float(0x7fc00000u) : h;
  if (raw) {
    const unsigned int bits = __float_as_uint(h);
    p12 = (bits >> 16) | ((bits << 8) & 0xff0000u);
    p3 = bits & 0xffu;
    return;
  }
  float rest = h * kSplitScale;
  const unsigned int hi = pack_bf16(rest, 0.f);
  rest -= bf16_low(hi);
  const unsigned int mid = pack_bf16(rest, 0.f);
  rest -= bf16_low(mid);
  p12 = hi | (mid << 16);
  p3 = pack_bf16(rest, 0.f);
}

// What the four lanes of a quad hold of four consecutive units, rearranged: lane 0, 1, 2 gets part 1, 2, 3 of all
// four, as two words to be stored side by side (lane 3: nothing of use).  All four lanes must be active.
__device__ __forceinline__ uint2 quad_parts(unsigned int p12, unsigned int p3) {
  const int part = threadIdx.x & 3;
  // (every lane makes both exchanges: a lane that skipped one would leave its neighbours without its value)
  const unsigned int x0 = quad_lane<0>(p12), x1 = quad_lane<1>(p12), x2 = quad_lane<2>(p12), x3 = quad_lane<3>(p12);
  const unsigned int y0 = quad_lane<0>(p3), y1 = quad_lane<1>(p3), y2 = quad_lane<2>(p3), y3 = quad_lane<3>(p3);
  const unsigned int a0 = part < 2 ? x0 : y0, a1 = part < 2 ? x1 : y1;
  const unsigned int a2 = part < 2 ? x2 : y2, a3 = part < 2 ? x3 : y3;
  const unsigned int sel = part == 1 ? 0x07060302u : 0x05040100u;  // the high halves : the low halves
  return make_uint2(__builtin_amdgcn_perm(a1, a0, sel), __builtin_amdgcn_perm(a3, a2, sel));
}

// A workgroup's LDS: the wavefronts' sums of an element (gates side by side), a step's inputs x * W and zoneout mask, the
// caller's copies; all twice, by step parity.
template <int NB>
struct SplitForwardLds {
  float sums[2][4][NB][16][4];
  float in[2][NB][16][4];
  float mask[2][NB][16];
  float out[2][6][NB][16];
};

// A wavefront's share of a matrix `src` [rows, G*H], split: lane 16*q + c holds unit j0 + c of every gate, k = 8*q ..
// 8*q+7 of the groups wave*KS .. wave*KS+KS-1.  `largest`: raised to the largest magnitude.  DropConnect: `mask`, `scale`.
template <int KS, int G>
__device__ __forceinline__ void load_split_weights(bf16x8_t (&w)[KS][G][3], const float* src, int rows, const float* mask,
                                                   float scale, int j0, int H, int wave, float& largest) {
  const int lane = threadIdx.x & 63;
  const int unit = j0 + (lane & 15);
  // (Rows and units beyond the matrix lie beyond the buffer and read as zero.)
  const int bytes = rows * G * H * 4;
  const __amdgpu_buffer_rsrc_t from = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(src), 0, bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t from_mask = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(mask), 0, bytes, 0x00020000);
  const int base = unit < H ? ((wave * KS * 32 + 8 * (lane >> 4)) * G * H + unit) * 4 : 0x70000000;
  float f[2][G][8];  // the groups are read one ahead of the one being split
  auto read = [&](float (&to)[G][8], __amdgpu_buffer_rsrc_t r, int j) {
#pragma unroll
    for (int e = 0; e < 8; ++e)
#pragma unroll
      for (int g = 0; g < G; ++g)
        to[g][e] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, base + ((j * 32 + e) * G + g) * H * 4, 0, 0));
    __builtin_amdgcn_sched_barrier(0);
  };
  read(f[0], from, 0);
#pragma unroll
  for (int j = 0; j < KS; ++j) {
    if (j + 1 < KS) read(f[(j + 1) & 1], from, j + 1);
    float (&x)[G][8] = f[j & 1];
    if (mask != nullptr) {
      float m[G][8];
      read(m, from_mask, j);
#pragma unroll
      for (int g = 0; g < G; ++g)
#pragma unroll
        for (int e = 0; e < 8; ++e) x[g][e] = x[g][e] * m[g][e] * scale;
    }
#pragma unroll
    for (int g = 0; g < G; ++g) {
      uint4_t parts[3];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        largest = fmaxf(largest, fmaxf(fabsf(x[g][2 * e]), fabsf(x[g][2 * e + 1])));
        unsigned int hi, mid, lo;
        split_pair(x[g][2 * e] * kSplitScale, x[g][2 * e + 1] * kSplitScale, hi, mid, lo);
        parts[0][e] = hi;
        parts[1][e] = mid;
        parts[2][e] = lo;
      }
#pragma unroll
      for (int q = 0; q < 3; ++q) w[j][g][q] = __builtin_bit_cast(bf16x8_t, parts[q]);
    }
  }
}

// acc[g] += rows * weights of a step, the small products of all k first, then the large ones: the sums of the former
// are not rounded to the size of the latter again and again.  One instruction per gate at a time, in the order written:
// left alone, the scheduler strings together those of one gate, each of which waits for the one before it.
template <int NB, int KS, int G, int FR>
__device__ __forceinline__ void split_products(const uint4_t (&a)[FR], const bf16x8_t (&w)[KS][G][3], float4_t (&acc)[G]) {
  const int lane = threadIdx.x & 63;
  auto mfma = [&](const uint4_t& x, int j, int part) {
#pragma unroll
    for (int g = 0; g < G; ++g)
      acc[g] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, x), w[j][g][part], acc[g], 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
  };
  if constexpr (NB == 16) {
#pragma unroll
    for (int j = 0; j < KS; ++j) {
      mfma(a[3 * j + 2], j, 0);
      mfma(a[3 * j + 1], j, 1);
      mfma(a[3 * j], j, 2);
    }
#pragma unroll
    for (int j = 0; j < KS; ++j) {
      mfma(a[3 * j + 1], j, 0);
      mfma(a[3 * j], j, 1);
    }
#pragma unroll
    for (int j = 0; j < KS; ++j) mfma(a[3 * j], j, 0);
  } else {
#pragma unroll
    for (int j = 0; j < KS; ++j) {
      if constexpr (NB == 8) {
        uint4_t part3 = a[KS + j / 2];
        const bool keep = ((lane >> 3) & 1) == (j & 1);
#pragma unroll
        for (int e = 0; e < 4; ++e) part3[e] = keep ? part3[e] : 0u;
        mfma(part3, j, 0);
      }
      mfma(a[j], j, 2);
    }
#pragma unroll
    for (int j = 0; j < KS; ++j) mfma(a[j], j, 1);
    // The last ones of gates 0 and 2 before those of the others: what follows for the former goes beside the latter.
#pragma unroll
    for (int half = 0; half < 2; ++half) {
#pragma unroll
      for (int j = 0; j < KS; ++j)
#pragma unroll
        for (int g = half; g < G; g += 2)
          acc[g] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a[j]), w[j][g][0], acc[g], 0, 0, 0);
      if (half == 0) __builtin_amdgcn_sched_barrier(0);
    }
  }
}

// A group of workgroups on one XCD runs all steps of NB batch rows; a workgroup owns 16 hidden units.  Its 256
// threads are four wavefronts, one per SIMD, that share the contraction: wavefront w keeps rows
// [32*KST*w, 32*KST*(w+1)) of its gates' columns of R, split into parts, in registers for the whole launch (48 * kGates
// of them at H = 512).  A step: poll the operands (h[t], already split by its producers), multiply, add the four
// wavefronts' sums through LDS, the pointwise step, split and publish h[t+1].
// What bounds it: the chain of a step.  LSTM, N = 64, H = 512 (cycles at 2.25 GHz, of about 3 700): the operands' request
// to their arrival 1 100 (24 KiB per CU at 57 bytes a cycle behind 220 of latency, and the time the publications take to
// land), 64 matrix instructions 1 075 and the sums' way to LDS 300, barrier 100, pointwise step and publication 1 000.
// Everything that is not part of it is kept off the wavefronts while they are on it: the inputs of a step and the
// caller's copies come from and go to memory that is cold in this launch, and a memory instruction costs its wavefront
// 50 - 100 cycles to issue, so they are moved 16 bytes per lane through LDS, at 4 and 8 rows by the wavefronts without
// hidden units of their own.
// Measured, C = H = 512, T = 100: LSTM N = 64, 358 us beside x * W on the fp32 matrix instructions -> 203 and 85 for the
// GEMM; N = 128 (GEMM before and now) 360 -> 288.  Training passes: LSTM 850 -> 814, N = 128 1411 -> 1335, GRU with
// masks 775 -> 750.  x * W inside this recurrence, behind the publication, was slower at 8 rows (287 for both) than the GEMM:
// its instructions are not hidden, only moved.
//
// A Cell supplies
//   Params                  the kernel's arguments: T, N, H, R [H, G*H], dc_mask, dc_scale, h [N,H], zoneout_prob,
//                           zoneout_mask, training, xh, ls, and whatever the cell reads and writes
//   kGates                  columns of R per unit, each with an input of its own
//   kOut, kStates           caller's copies per element and step; the first kStates of them also without training
//   load_state(p, row, unit, mine)         `h` is zero where the element is not the thread's
//   aligned(p)              the rows below start on 16 bytes where H is a multiple of 4
//   in_row(p, gate, row)    x * W of a gate at step 0: a row of H floats; in_stride(p): floats between steps
//   out_row(p, i, row), out_stride(p, i)   the same for the copies
//   step(p, in, mask, sums, zoneout)       the pointwise step; `h` holds the new state afterwards
//   out(i)                  copy i of the last step
template <class Cell, int NB, int KST>
__global__ __launch_bounds__(256, 1)
void split_forward_kernel(typename Cell::Params p) {
  using Tile = SplitTile<NB, KST>;
  constexpr int G = Cell::kGates;
  constexpr int HS = 16;
  constexpr int FR = Tile::kFrags;
  constexpr int OWNERS = NB * HS;                         // threads with an element of their own
  constexpr int HELPERS = NB == 16 ? 256 : 256 - OWNERS;  // threads that move inputs and copies: the last ones
  constexpr int ITEMS = NB * 4;                           // groups of four units per plane of inputs or copies
  constexpr int IN_N = ((G + 1) * ITEMS + HELPERS - 1) / HELPERS;  // (planes of inputs: the gates, the mask)
  constexpr int OUT_N = (Cell::kOut * ITEMS + HELPERS - 1) / HELPERS;
  using Lds = SplitForwardLds<NB>;
  extern __shared__ __attribute__((aligned(16))) float lds[];
  Lds& s = *reinterpret_cast<Lds*>(lds);
  const Role role = take_role(p.ls, reinterpret_cast<unsigned int*>(&s.sums));
  if (!role.active) return;

  const int H = p.H, N = p.N, T = p.T;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int j0 = role.cw * HS;
  const int n0 = role.bt * NB;
  const int rows_here = (N - n0) < NB ? (N - n0) : NB;

  char* xh = reinterpret_cast<char*>(p.xh) + (size_t)role.bt * kPolledTiles * Tile::kBytes;
  const TileBuffer xhb = make_tile_buffer(reinterpret_cast<float*>(xh), kPolledTiles * Tile::kBytes / 4);

  GroupSync gs;
  group_sync_init(gs, p.ls, role);

  // States that do not split are published raw, by all workgroups of the group alike.  (fmaxf passes over NaNs.)
  float state[NB * KST / 2];
#pragma unroll
  for (int i = 0; i < NB * KST / 2; ++i) {
    const int at = tid + 256 * i;
    state[i] = p.h[(size_t)n0 * H + (at < rows_here * H ? at : 0)];
  }
  // This workgroup's chunks of the exchange tiles: rows and units beyond the problem stay zero for the launch.
  for (int i = tid; i < Tile::kBytes / 16; i += 256) {
    int owner = Tile::chunk_unit(i) / HS;
    owner = owner < p.ls.gx ? owner : p.ls.gx - 1;
    if (owner == role.cw)
      for (int b = 0; b < kPolledTiles; ++b)
        *reinterpret_cast<uint4_t*>(xh + (size_t)b * Tile::kBytes + i * 16) = uint4_t{0u, 0u, 0u, 0u};
  }
  float largest = 0.f;
#pragma unroll
  for (int i = 0; i < NB * KST / 2; ++i) largest = fmaxf(largest, fabsf(state[i]));
  const bool raw = __syncthreads_or(largest >= kSplitLimit) != 0;

  // The weights.  The matrix instructions take most of them from the upper half of the register file, which nothing
  // else can use directly: left alone, the compiler copies what does not fit the lower half back and forth.
  largest = 0.f;
  bf16x8_t w[KST][G][3];
  load_split_weights<KST, G>(w, p.R, H, p.dc_mask, p.dc_scale, j0, H, wave, largest);
#pragma unroll
  for (int j = 0; j < KST; ++j)
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
      for (int q = 1; q < 3; ++q)
        if (KST > 2) asm volatile("" : "+a"(w[j][g][q]));
  const bool exact = __syncthreads_or(largest >= kSplitLimit) != 0 || raw;

  // Pointwise ownership: thread 16*r + u of the first NB*16 handles batch row n0 + r, hidden unit j0 + u.
  const bool owns = wave < OWNERS / 64;
  const int pr = tid / HS, pu = tid % HS;
  const bool act = owns && pr < rows_here && j0 + pu < H;
  const size_t row = act ? (size_t)(n0 + pr) : 0, unit = act ? (size_t)(j0 + pu) : 0;
  const bool zoneout = p.zoneout_prob != 0.f && p.zoneout_mask != nullptr;
  Cell cell;
  cell.load_state(p, row, unit, act);
  // What this lane publishes: one part of four units of its row (see quad_parts); elsewhere its stores go beyond the
  // buffer, where nothing is written.
  const bool pub = owns && pr < rows_here && j0 + (pu & ~3) < H && (pu & 3) < 3;
  const int pub_at = pub ? Tile::byte(j0 + (pu & ~3), pu & 3, pr < NB ? pr : 0) : 0x7ffffff0;
  auto store_parts = [&](int tile, uint2 v) {
    typedef unsigned int uint2_t __attribute__((ext_vector_type(2)));
    __builtin_amdgcn_raw_buffer_store_b64(uint2_t{v.x, v.y}, xhb.rsrc, pub_at, tile * Tile::kBytes, 0);
  };
  auto publish = [&](int tile, float h) {
    unsigned int p12, p3;
    split_state(h, raw, p12, p3);
    store_parts(tile, quad_parts(p12, p3));
  };
  auto unwrite = [&](int tile) { store_parts(tile, make_uint2(kUnwrittenBits, kUnwrittenBits)); };
  // The zeros above have landed before anything is published over them.
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (owns) {
    publish(0, cell.h);
    for (int b = 1; b < kPolledTiles; ++b) unwrite(b);
  }

  // What this thread moves: group i of four units is plane i / ITEMS, row i / 4 % NB, units 4 * (i % 4) of the
  // workgroup's.  Rows of H floats that do not start on 16 bytes are moved element by element.
  const int helper = tid - (256 - HELPERS);
  const bool helps = wave >= 4 - HELPERS / 64;
  const bool masked = zoneout && p.training;
  const int in_planes = G + (masked ? 1 : 0), out_planes = p.training ? Cell::kOut : Cell::kStates;
  const bool wide = H % 4 == 0 && Cell::aligned(p);
  const float* in_at[IN_N];
  float* out_at[OUT_N];
  float4_t moved[IN_N];
  bool in_ok[IN_N], out_ok[OUT_N];
  auto item_unit = [&](int i) { return j0 + 4 * (i & 3); };
#pragma unroll
  for (int n = 0; n < IN_N; ++n) {
    const int i = helper + HELPERS * n, plane = i / ITEMS, r = (i >> 2) % NB;
    in_ok[n] = helps && plane < in_planes && r < rows_here && item_unit(i) < H;
    const size_t at = in_ok[n] ? (size_t)(n0 + r) : 0;
    in_at[n] = (plane < G ? Cell::in_row(p, in_ok[n] ? plane : 0, at) : p.zoneout_mask + at * H) + (in_ok[n] ? item_unit(i) : 0);
    moved[n] = float4_t{0.f, 0.f, 0.f, 0.f};
  }
#pragma unroll
  for (int n = 0; n < OUT_N; ++n) {
    const int i = helper + HELPERS * n, plane = i / ITEMS, r = (i >> 2) % NB;
    out_ok[n] = helps && plane < out_planes && r < rows_here && item_unit(i) < H;
    out_at[n] = out_ok[n] ? Cell::out_row(p, plane, (size_t)(n0 + r)) + item_unit(i) : nullptr;
  }
  auto request = [&] {
#pragma unroll
    for (int n = 0; n < IN_N; ++n)
      if (in_ok[n]) {
        if (wide) {
          moved[n] = *reinterpret_cast<const float4_t*>(in_at[n]);
        } else {
          const int i = helper + HELPERS * n;
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (item_unit(i) + e < H) moved[n][e] = in_at[n][e];
        }
        in_at[n] += (helper + HELPERS * n) / ITEMS < G ? Cell::in_stride(p) : (size_t)N * H;
      }
  };
  auto park_inputs = [&](int t) {
#pragma unroll
    for (int n = 0; n < IN_N; ++n)
      if (in_ok[n]) {
        const int i = helper + HELPERS * n, plane = i / ITEMS, r = (i >> 2) % NB;
        if (plane < G) {
#pragma unroll
          for (int e = 0; e < 4; ++e) s.in[t & 1][r][4 * (i & 3) + e][plane] = moved[n][e];
        } else {
          *reinterpret_cast<float4_t*>(&s.mask[t & 1][r][4 * (i & 3)]) = moved[n];
        }
      }
  };
  auto leave_copies = [&](int t) {
#pragma unroll
    for (int i = 0; i < Cell::kOut; ++i)
      if (i < out_planes) s.out[t & 1][i][pr][pu] = cell.out(i);
  };
  // The caller's copies of step t, which the owners have left in LDS.
  auto write_copies = [&](int t) {
#pragma unroll
    for (int n = 0; n < OUT_N; ++n)
      if (out_ok[n]) {
        const int i = helper + HELPERS * n, plane = i / ITEMS, r = (i >> 2) % NB;
        const float4_t v = *reinterpret_cast<const float4_t*>(&s.out[t & 1][plane][r][4 * (i & 3)]);
        if (wide) {
          *reinterpret_cast<float4_t*>(out_at[n]) = v;
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (item_unit(i) + e < H) out_at[n][e] = v[e];
        }
        out_at[n] += Cell::out_stride(p, plane);
      }
  };

  // A step's operands.
  uint4_t a[FR];
  const int frag_at = wave * FR * 1024 + lane * 16;
  auto load = [&](int tile) {
    constexpr int kAgentScope = 16;  // the sc1 bit of the cache policy
#pragma unroll
    for (int f = 0; f < FR; ++f)
      a[f] = __builtin_amdgcn_raw_buffer_load_b128(xhb.rsrc, frag_at + f * 1024, tile * Tile::kBytes, kAgentScope);
  };

  // Step t finds its inputs parked in area t % 2; those of step t + 1 are on their way in registers.
  request();
  park_inputs(0);
  if (T > 1) request();
  group_arrive(gs);
  group_wait(gs);
  load(0);

  for (int t = 0; t < T; ++t) {
    poll_until_written(gs, [&] { load(t & 3); }, [&] { return all_parts_written(a); });
    // (In the order issued, everything this wavefront stored before -- the reset of a tile among it -- has landed too.)
    if (NB == 16 && t > 0 && t + 1 < T) request();

    float (&sums)[4][NB][16][4] = s.sums[t & 1];
    if (!exact) {
      float4_t acc[G];
#pragma unroll
      for (int g = 0; g < G; ++g) acc[g] = float4_t{0.f, 0.f, 0.f, 0.f};
      split_products<NB, KST, G>(a, w, acc);
      // Element e of an accumulator in lane 16*q + c: operand row 4*q + e, column c.  The rows that hold parts of
      // the same batch row are added here; a lane stores the gates it has of an element side by side.
      const int q = lane >> 4, c = lane & 15;
      if constexpr (NB == 16) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          *reinterpret_cast<float4_t*>(sums[wave][4 * q + e][c]) = float4_t{acc[0][e], acc[1][e], acc[2][e], acc[G - 1][e]};
      } else if constexpr (NB == 8) {
        // rows 8..15 (lanes 32..63) are part 2 of rows 0..7: the lower lanes take gates 0 and 1, the upper 2 and 3
        const int r = 4 * (q & 1), up = q >> 1;
#pragma unroll
        for (int e = 0; e < 4; ++e)
          *reinterpret_cast<float2_t*>(&sums[wave][r + e][c][2 * up]) =
              float2_t{swap_add32(acc[0][e], acc[2][e]), swap_add32(acc[1][e], acc[G - 1][e])};
      } else {
        // every lane group holds a part of the four rows: lane group 0, 1, 2, 3 ends up with row 0, 2, 1, 3
        auto total = [](const float4_t& v) { return swap_add32(swap_add16(v.x, v.z), swap_add16(v.y, v.w)); };
        *reinterpret_cast<float4_t*>(sums[wave][scatter_row(q)][c]) =
            float4_t{total(acc[0]), total(acc[1]), total(acc[2]), total(acc[G - 1])};
      }
    }
    __syncthreads();

    if (owns) {
      float4_t rh = {0.f, 0.f, 0.f, 0.f};
      const float4_t in = *reinterpret_cast<const float4_t*>(s.in[t & 1][pr][pu]);
      const float mask = masked ? s.mask[t & 1][pr][pu] : 1.f;
      if (!exact) {
        float4_t v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = *reinterpret_cast<const float4_t*>(sums[i][pr][pu]);
        rh = ((v[0] + v[1]) + (v[2] + v[3])) * kProductScale;
      } else if (act) {
        const char* tile = xh + (size_t)(t & 3) * Tile::kBytes;
        for (int k = 0; k < H; ++k) {
          unsigned int part[3];
#pragma unroll
          for (int q = 0; q < 3; ++q)
            part[q] = __hip_atomic_load(reinterpret_cast<const unsigned short*>(tile + Tile::byte(k, q, pr)),
                                        __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          const float hk = raw ? __uint_as_float((part[0] << 16) | (part[1] << 8) | part[2])
                               : ((bf16_low(part[2]) + bf16_low(part[1])) + bf16_low(part[0])) * (1.0f / kSplitScale);
          for (int g = 0; g < G; ++g) {
            const size_t off = ((size_t)k * G + g) * H + unit;
            float x = p.R[off];
            if (p.dc_mask != nullptr) x = x * p.dc_mask[off] * p.dc_scale;
            rh[g] = fmaf(hk, x, rh[g]);
          }
        }
      }
      if (act) cell.step(p, in, mask, rh, zoneout);
      if (t + 1 < T) {
        publish((t + 1) & 3, cell.h);
        if (t + 3 < T) unwrite((t + 3) & 3);  // read at step t-1: nobody needs it any more
      }
    }
    // Between the step's barrier and the next step's the helpers own area (t+1) % 2 of the inputs and read area
    // (t-1) % 2 of the copies, the owners the other areas.
    if (helps) {
      if (t > 0) write_copies(t - 1);
      if (t + 1 < T) park_inputs(t + 1);
      if (NB < 16 && t + 2 < T) request();
    }
    // (8 rows: the wavefronts without hidden units sleep until the others have published.  Polling earlier, they keep the
    // publication waiting for the memory pipeline.)
    if (NB < 16) __syncthreads();
    if (t + 1 < T) load((t + 1) & 3);
    if (owns && t + 1 < T) leave_copies(t);  // while these are on their way
  }
  if (owns) leave_copies(T - 1);
  __syncthreads();
  if (helps) write_copies(T - 1);
}

inline size_t split_forward_tile_bytes(int N, int H, int nb) {
  const int kst = (H + 127) / 128;
  const int frags = nb == 4 ? kst : (nb == 8 ? kst + (kst + 1) / 2 : 3 * kst);
  return (size_t)((N + nb - 1) / nb) * kPolledTiles * 4 * frags * 1024;
}

// The rows of a batch tile where a forward recurrence takes this kernel (0: it does not), behind the GEMM for
// x * W (C inputs, `columns` outputs; `ready`: x * W exists; `beside`: the other kernels compute it beside their waits).
// With few hidden units a step is the chain alone, which the other kernels, with fewer units per workgroup, have
// shorter; with few steps the weights' splitting and the GEMM's launch are not made up for.  Measured, inference, the
// others -> this one with its GEMM, us:
//   T = 100  LSTM N = 128 C = H = 512  469 -> 409   N = 128 C = 128 H = 256  244 -> 223   N = 100 C = 128 H = 192  206 -> 214
//            LSTM N = 64 C = H = 512  308 -> 279   C = 256 H = 272  236 -> 202   C = 75 H = 192  159 -> 170
//            LSTM N = 20 C = 512 H = 336  198 -> 186   N = 4 C = 300 H = 512  222 -> 178   N = 16 C = 128 H = 256  108 -> 146
//            GRU N = 128 C = H = 512  389 -> 357   N = 64  262 -> 247   N = 32 C = 512  204 -> 185
//   C = 256 H = 320 N = 64, T = 25 / 50  LSTM 73 / 128 -> 80 / 126   GRU 64 / 109 -> 76 / 118
//   C = 75 (nothing beside the waits) H = 300 N = 16, T = 25 / 50  LSTM 64 / 101 -> 62 / 96   GRU 62 / 98 -> 57 / 89
inline int split_forward_rule(hipStream_t stream, int T, int N, int C, int H, int columns, bool ready, bool beside,
                              int* rows) {
  *rows = 0;
  int nb = 0;
  for (int rows_of_tile : {16, 8, 4})
    if (xcd_local_fits((H + 15) / 16, (N + rows_of_tile - 1) / rows_of_tile)) nb = rows_of_tile;
  if (nb == 0 || H > 512 || H <= (nb == 16 ? 224 : 256)) return HASTE_HIP_OK;
  if (T < (nb == 16 ? 2 : (beside ? 64 : 24))) return HASTE_HIP_OK;
  size_t bytes = split_forward_tile_bytes(N, H, nb);
  const size_t product = ready ? 0 : gemm_f32_scratch_bytes(T * N, columns, C);
  bytes = bytes > product ? bytes : product;
  bool room = false;
  HASTE_HIP_PROPAGATE(workspace_has_room(stream, bytes, &room));
  if (room) *rows = nb;
  return HASTE_HIP_OK;
}

template <class Cell, int NB, int KST>
int launch_split_forward_tile(const char* name, hipStream_t stream, const Workspace& ws, typename Cell::Params& p) {
  LaunchPlan plan;
  HASTE_HIP_PROPAGATE(plan_launch(stream, ws, (p.H + 15) / 16, (p.N + NB - 1) / NB, NB, sizeof(SplitForwardLds<NB>),
                                  (unsigned)p.T + 1, &plan));
  p.ls = plan.shape;
  plan.kernel = kPlanSplit;
  return launch_persistent(name, split_forward_kernel<Cell, NB, KST>, plan, p, stream);
}
template <class Cell, int NB>
int launch_split_forward_rows(const char* name, hipStream_t stream, const Workspace& ws, typename Cell::Params& p) {
  if constexpr (NB == 16)
    if (p.H <= 256) return launch_split_forward_tile<Cell, NB, 2>(name, stream, ws, p);
  if (p.H <= 384) return launch_split_forward_tile<Cell, NB, 3>(name, stream, ws, p);
  return launch_split_forward_tile<Cell, NB, 4>(name, stream, ws, p);
}

// Launches the kernel for the rows split_forward_rule() gives, on p.xh of split_forward_tile_bytes(N, H, nb).
template <class Cell>
int launch_split_forward(const char* name, hipStream_t stream, const Workspace& ws, int nb, typename Cell::Params& p) {
  if (nb == 4) return launch_split_forward_rows<Cell, 4>(name, stream, ws, p);
  if (nb == 8) return launch_split_forward_rows<Cell, 8>(name, stream, ws, p);
  return launch_split_forward_rows<Cell, 16>(name, stream, ws, p);
}

}  // namespace haste_hip
