// The recurrence of a group of XCDs for hidden sizes whose weights one XCD does not hold: the step's product cut along
// both the contraction and the columns, on the bf16 matrix cores.  For the cells of split_forward.h and
// scatter_backward.h.
#pragma once

#include <algorithm>

#include "split_forward.h"
#include "split_backward.h"

namespace haste_hip {

// How a group works.  A group is `span` XCDs and takes every groups-th tile of 16 batch rows; per XCD `chunks` ranges of
// the contraction (128 * KS each) times `blocks` blocks of 16 * CT columns of the weights, a workgroup each.
//   Forward: a block is 4 * CT hidden units (four columns each); an XCD has blocks of its own and all of the
//   contraction, so that h goes to all XCDs and partial sums stay on one.
//   Backward: an XCD has units of its own, whose gate gradients are its contraction (k = 4 * unit + gate), and all
//   columns, so that the gate gradients stay on the XCD and partial sums of dh go to all.
// Every workgroup also finishes `own` units (a multiple of 4): forward some of its block's, backward some of its XCD's.
struct CutShape {
  int xcds, span, groups;
  int chunks, blocks, own;
  int xcd_units;  // backward: units of an XCD
  int tiles;      // batch tiles of 16 rows
  int areas;      // of inputs and copies in LDS
  float* pieces;
  char* operands;
  float* sums;    // backward: column sums [groups][sums][H]
};

template <class Params>
struct CutParams {
  Params p;
  CutShape s;
};

constexpr int kCutRows = 16;
constexpr int kCutLoads = 4;  // pieces a lane adds up

// Column tiles whose weights' last parts are kept in LDS: what the registers do not hold.
template <int KS, int CT>
constexpr int cut_lds_tiles() {
  return KS * CT <= 18 ? 0 : CT - 1;
}
// Where the wavefronts have two column tiles each to add up, they keep their own sums of those in registers.
template <int CT>
constexpr bool cut_keeps_sums() {
  return CT == 8;
}
template <int CT>
constexpr int cut_sum_tiles() {  // a wavefront leaves in LDS
  return cut_keeps_sums<CT>() ? CT - 2 : CT;
}

// Words of LDS for an element's inputs and for what a step leaves for the caller's copies: whole 16 bytes, read and
// written as such, or else an odd number.
template <class Cell, bool BACK>
constexpr int cut_in_words() {
  if constexpr (BACK) return (Cell::kCutInputs + 3) / 4 * 4;
  else return (Cell::kGates + 1) | 1;
}
template <class Cell, bool BACK>
constexpr int cut_out_words() {
  return BACK ? 4 : Cell::kOut | 1;
}

// The LDS of a workgroup, in bytes.
template <int KS, int CT>
constexpr size_t cut_fixed_lds_bytes() {
  return (size_t)KS * cut_lds_tiles<KS, CT>() * 4 * 1024 + (size_t)cut_sum_tiles<CT>() * 4 * 1024 + 64 * CT;
}
inline size_t cut_lds_bytes(size_t fixed, int areas, int inputs, int copies, int carried, int sums, int own, int row_tiles) {
  const size_t plane = (size_t)own * kCutRows * sizeof(float);
  return fixed + (size_t)(areas * (inputs + copies) + carried * row_tiles + (sums > 0 ? 4 : 0)) * plane +
         (size_t)sums * own * 2 * sizeof(float);
}

// ---- values that do not split -------------------------------------------------------------------
// A float whose scaled first part would be infinite (2^104 and more, infinities) travels as its bits, marked by a NaN in
// the first part; a NaN as a mark of its own.  The product then is not finite, which is what a workgroup looks for: it
// forms such sums again from the floats.  No word of two parts is all ones.
constexpr unsigned int kBitsMark = 0x7fc0u, kNanMark = 0x7fe0u;

__device__ __forceinline__ void mark_large(float v, int shift, unsigned int& hi, unsigned int& mid, unsigned int& lo) {
  if (fabsf(v) < 0x1p103f) return;
  const unsigned int bits = __float_as_uint(v), keep = 0xffff0000u >> shift;
  const bool nan = v != v;
  hi = (hi & keep) | (nan ? kNanMark : kBitsMark | (bits & 1u)) << shift;
  mid = (mid & keep) | (nan ? 0x7fc0u : bits >> 16) << shift;
  lo = (lo & keep) | (nan ? 0u : (bits & 0xffffu) >> 1) << shift;
}
// The parts of two floats side by side.
__device__ __forceinline__ void cut_pair(float a, float b, unsigned int& hi, unsigned int& mid, unsigned int& lo) {
  split_pair(a * kSplitScale, b * kSplitScale, hi, mid, lo);
  if (__any(!(fmaxf(fabsf(a), fabsf(b)) < 0x1p103f) || a != a || b != b)) {
    mark_large(a, 0, hi, mid, lo);
    mark_large(b, 16, hi, mid, lo);
  }
}
__device__ __forceinline__ float cut_value(unsigned int p0, unsigned int p1, unsigned int p2) {
  if ((p0 & 0x7f80u) == 0x7f80u)
    return (p0 & 0xfffeu) == kBitsMark ? __uint_as_float((p1 << 16) | (p2 << 1) | (p0 & 1u)) : __uint_as_float(0x7fc00000u);
  return ((bf16_low(p2) + bf16_low(p1)) + bf16_low(p0)) * (1.0f / kSplitScale);
}

// r[0..3] hold a word each for the four 16-lane groups: afterwards group g holds in r[j] what group j held in r[g].
__device__ __forceinline__ void transpose_groups(unsigned int (&r)[4]) {
  auto swap32 = [](unsigned int& a, unsigned int& b) {
    const auto s = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    a = s[0];
    b = s[1];
  };
  auto swap16 = [](unsigned int& a, unsigned int& b) {
    const auto s = __builtin_amdgcn_permlane16_swap(a, b, false, false);
    a = s[0];
    b = s[1];
  };
  swap32(r[0], r[2]);
  swap32(r[1], r[3]);
  swap16(r[0], r[1]);
  swap16(r[2], r[3]);
}

// The wavefront's weights, split: lane 16*q + m holds column m of tile ct, k = 8*q + e of group j of 32.  The first two
// parts and the last one of tiles 0 .. CT-LDS-1 in registers, the others' last parts in `lds` (the lane's first word, a
// wavefront's operands 1 KiB each).  offset(j, ct, e): where the element is in `src`, in bytes, beyond the buffer
// where there is none.  nans: bit ct is set where a weight of column tile ct is a NaN.
template <int KS, int CT, int LDS, class OffsetFn>
__device__ __forceinline__ void load_cut_weights(bf16x8_t (&w)[KS][CT][2], uint4_t (&lo)[KS][CT - LDS > 0 ? CT - LDS : 1],
                                                 uint4_t* lds, const float* src, int bytes,
                                                 OffsetFn offset, unsigned int& nans) {
  const __amdgpu_buffer_rsrc_t from = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(src), 0, bytes, 0x00020000);
  constexpr int HALF = CT / 2;
  float f[2][HALF][8];  // half the tiles of a group of k are read ahead of those being split
  auto read = [&](float (&to)[HALF][8], __amdgpu_buffer_rsrc_t r, int step) {
#pragma unroll
    for (int e = 0; e < 8; ++e)
#pragma unroll
      for (int i = 0; i < HALF; ++i)
        to[i][e] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, offset(step >> 1, (step & 1) * HALF + i, e), 0, 0));
    __builtin_amdgcn_sched_barrier(0);
  };
  nans = 0u;
  read(f[0], from, 0);
#pragma unroll
  for (int step = 0; step < 2 * KS; ++step) {
    const int j = step >> 1;
    const float (&x)[HALF][8] = f[step & 1];
    if (step + 1 < 2 * KS) read(f[(step + 1) & 1], from, step + 1);
#pragma unroll
    for (int i = 0; i < HALF; ++i) {
      const int ct = (step & 1) * HALF + i;
      uint4_t parts[3];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float a = x[i][2 * e], b = x[i][2 * e + 1];
        nans |= (a != a || b != b ? 1u : 0u) << ct;
        unsigned int hi, mid, last;
        split_pair(a * kSplitScale, b * kSplitScale, hi, mid, last);
        parts[0][e] = hi;
        parts[1][e] = mid;
        parts[2][e] = last;
      }
#pragma unroll
      for (int part = 0; part < 2; ++part) {
        w[j][ct][part] = __builtin_bit_cast(bf16x8_t, parts[part]);
        // (see split_forward_kernel; the accumulators need some of the upper half themselves)
        if (KS * CT * 2 <= 56 || part == 0 || j < KS - 1) asm volatile("" : "+a"(w[j][ct][part]));
      }
      if (ct < CT - LDS) lo[j][ct] = parts[2];
      else lds[(j * LDS + ct - (CT - LDS)) * 64] = parts[2];
      __builtin_amdgcn_sched_barrier(0);
    }
  }
}

// acc[ct] += weights * rows for the three parts `a` of 16 rows: small products first, in two halves, of which the second
// takes the rows' first parts only.  The weights' last parts are read from LDS ahead of the matrix instructions, which go
// through the accumulators in turn.
template <int KS, int CT, int LDS>
__device__ __forceinline__ void cut_small_products(const uint4_t (&a)[KS][3], const bf16x8_t (&w)[KS][CT][2],
                                             const uint4_t (&lo)[KS][CT - LDS > 0 ? CT - LDS : 1], const uint4_t* lds,
                                             float4_t (&acc)[CT]) {
  constexpr int STEP = 2, STEPS = CT / STEP;  // column tiles of a step
  constexpr int AHEAD = 1;                    // steps
  auto mfma = [&](const bf16x8_t& x, const uint4_t& y, int ct) {
    acc[ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, __builtin_bit_cast(bf16x8_t, y), acc[ct], 0, 0, 0);
  };
  uint4_t ahead[AHEAD + 1][STEP];
  auto read = [&](int step) {
#pragma unroll
    for (int i = 0; i < STEP; ++i) {
      const int ct = step % STEPS * STEP + i;
      if (ct >= CT - LDS) ahead[step % (AHEAD + 1)][i] = lds[(step / STEPS * LDS + ct - (CT - LDS)) * 64];
    }
  };
  if (LDS > 0) {
#pragma unroll
    for (int step = 0; step < AHEAD; ++step) read(step);
    __builtin_amdgcn_sched_barrier(0);
  }
#pragma unroll
  for (int step = 0; step < STEPS * KS; ++step) {
    const int j = step / STEPS, first = step % STEPS * STEP;
    if (LDS > 0 && step + AHEAD < STEPS * KS) {
      read(step + AHEAD);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int i = 0; i < STEP; ++i) mfma(w[j][first + i][0], a[j][2], first + i);
#pragma unroll
    for (int i = 0; i < STEP; ++i) mfma(w[j][first + i][1], a[j][1], first + i);
#pragma unroll
    for (int i = 0; i < STEP; ++i) {
      const int ct = first + i;
      const uint4_t last = ct >= CT - LDS ? ahead[step % (AHEAD + 1)][i] : lo[j][ct < CT - LDS ? ct : 0];
      mfma(__builtin_bit_cast(bf16x8_t, last), a[j][0], ct);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
#pragma unroll
  for (int j = 0; j < KS; ++j) {
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) mfma(w[j][ct][0], a[j][1], ct);
    __builtin_amdgcn_sched_barrier(0);
  }
}
template <int KS, int CT>
__device__ __forceinline__ void cut_large_products(const uint4_t (&a)[KS][3], const bf16x8_t (&w)[KS][CT][2], float4_t (&acc)[CT]) {
#pragma unroll
  for (int part = 1; part >= 0; --part)
#pragma unroll
    for (int j = 0; j < KS; ++j) {
#pragma unroll
      for (int ct = 0; ct < CT; ++ct)
        acc[ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[j][ct][part], __builtin_bit_cast(bf16x8_t, a[j][0]), acc[ct], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
}

// (Addresses that pass through a structure would otherwise be accessed as if they could lie in LDS.)
typedef __attribute__((address_space(1))) char GlobalByte;
typedef __attribute__((address_space(1))) float GlobalFloat;
typedef __attribute__((address_space(1))) float4_t GlobalFloat4;

// The sum over the 16 rows of a unit, in all their lanes.
__device__ __forceinline__ float sum_of_rows(float v) {
  auto add = [&](auto control) {
    constexpr int kControl = decltype(control)::value;
    v += __uint_as_float((unsigned int)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(v), kControl, 0xf, 0xf, false));
  };
  add(std::integral_constant<int, 0xb1>{});   // quad_perm 1, 0, 3, 2
  add(std::integral_constant<int, 0x4e>{});   // quad_perm 2, 3, 0, 1
  add(std::integral_constant<int, 0x141>{});  // row_half_mirror
  add(std::integral_constant<int, 0x140>{});  // row_mirror
  return v;
}

// A step of a batch tile and where it is kept: time (or reverse time) and the group's row tile.
struct CutSlot {
  int step, tile;
  __device__ __forceinline__ void next(int tiles) {
    if (++tile == tiles) {
      tile = 0;
      ++step;
    }
  }
};

// The 256 threads of a workgroup are four wavefronts, one per SIMD, which share the workgroup's range of the contraction:
// wavefront w keeps 32 * KS of k times the block's columns, split into parts, in registers (and LDS) for the whole launch.
// The batch tiles of the group go through in turn; for each a slot of work is
//   product     poll the operands (parts of 16 rows, as the matrix instruction takes them), multiply; the weights are
//               the first operand, so that a lane ends up with four columns of one row: the gates of a unit
//   pieces      the four wavefronts' sums meet in LDS, and the workgroup's partial sums go to those who finish the units
//   finish      who finishes units adds up the pieces of all chunks, takes the pointwise step and publishes operands
// With several batch tiles a workgroup finishes its units of the tile before, whose pieces have been on their way during
// the product: only one tile waits for two exchanges a step.  Pieces are tagged as in split_backward.h (two buffers), the
// operands polled as in split_forward.h (four buffers); either is overwritten only by those who, through others, have
// heard from all its readers: a step's operands hang together with the pieces of all chunks of the step before.
// What bounds it.  With a batch tile per group the chain of two exchanges: LSTM, 16 rows, H = 768 (cycles at 2.4 GHz, of
// about 8 600 a step forward, 11 000 backward): operands 1 300 (backward 950), product 1 730, sums 540, pieces out 620
// and in 1 400 (from other XCDs 3 000), pointwise step 550, publication 650, copies and inputs 1 200.  With four tiles,
// N = 64, H = 2 048: 8 400 a tile forward, 8 800 backward, of which 192 matrix instructions take 3 130 with the loads of
// the next tile beside them (48 KiB per CU and tile: 900 cycles of the memory pipeline), the sums through LDS and the
// pieces 1 100, the finish 2 600 (two wavefronts of four; the others move inputs and copies).  A wavefront per SIMD has
// nothing to run beside its own vector instructions; two do not fit, the weights take 400 of the 512 registers.
// Measured, whole passes, C = 64, T = 60: LSTM N = 64, H = 2 048 forward 1 380 -> 879 us (the fp32 instruction, every
// workgroup reading all of h), backward 2 131 -> 1 530 (a GEMM per step); C = 512, T = 50, training 3 693 -> 2 658.
// WIDE: what a thread moves starts on 16 bytes and is four units.  MANY: a group has more than two batch tiles.
template <class Cell, bool BACK, int KS, int CT, bool WIDE, bool MANY>
__global__ __launch_bounds__(256, 1)
void cut_recurrence_kernel(CutParams<typename Cell::Params> cp) {
  constexpr int G = Cell::kGates;
  constexpr int LDS = cut_lds_tiles<KS, CT>();
  constexpr int KR = 128 * KS;      // a workgroup's range of the contraction
  constexpr bool KEEPS = cut_keeps_sums<CT>();
  constexpr int ITEMS = CT * 64;    // groups of four columns of a row that it has sums of
  constexpr int ITEM_N = (ITEMS + 255) / 256;
  constexpr int IN_PLANES = [] {
    if constexpr (BACK) return Cell::kCutInputs;
    else return Cell::kGates + 1;
  }();
  constexpr int IN_N = (IN_PLANES + 3) / 4, OUT_N = (Cell::kOut + 3) / 4;  // (a plane is at most 64 groups of four)
  constexpr int CARRIED = Cell::kCarried;
  constexpr int SUMS = [] {
    if constexpr (BACK) return Cell::kSums;
    else return 1;
  }();
  typename Cell::Params& p = cp.p;
  const CutShape& cs = cp.s;
  extern __shared__ __attribute__((aligned(16))) float lds[];
  uint4_t* lds_lo = reinterpret_cast<uint4_t*>(lds);                            // [4][KS*LDS][64]
  // Sums: [4][ITEMS]; KEEPS: [wavefront they are for][the other three][two tiles][64]
  float4_t* lds_sums = reinterpret_cast<float4_t*>(lds_lo + 4 * KS * LDS * 64);
  unsigned int* lds_nan = reinterpret_cast<unsigned int*>(lds_sums + 4 * 64 * cut_sum_tiles<CT>());  // [16*CT]
  float* lds_in = reinterpret_cast<float*>(lds_nan + 16 * CT);
  const int O = cs.own, plane = O * kCutRows;
  // Inputs and copies, element by element, and what is carried.
  constexpr int IN_P = cut_in_words<Cell, BACK>(), OUT_P = cut_out_words<Cell, BACK>();
  const int in_floats = IN_P * plane, out_floats = OUT_P * plane;
  float* lds_out = lds_in + cs.areas * in_floats;
  float* lds_state = lds_out + cs.areas * out_floats;

  const Role role = take_role(p.ls, lds_nan);
  __syncthreads();
  const int T = p.T, N = p.N, H = p.H;
  const int group = role.bt / cs.span, xi = role.bt % cs.span, wi = role.cw;
  if (!role.active || group >= cs.groups) return;
  const int RT = (cs.tiles - group + cs.groups - 1) / cs.groups;  // (every group has a tile)
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int q = lane >> 4, c = lane & 15;
  const bool cross = cs.span > 1;

  GroupSync gs;
  gs.flags = &p.ls.cb->step_flags[group * cs.span * p.ls.gx];
  gs.abort_flag = &p.ls.cb->abort_flag[0];
  gs.host_status = p.ls.host_status;
  gs.group_size = (unsigned int)(cs.span * p.ls.gx + p.ls.absent);
  gs.my_index = (unsigned int)(xi * p.ls.gx + wi);
  gs.epoch = p.ls.epoch;
  gs.arrivals = 0;
  gs.spin_limit = p.ls.spin_limit;
  gs.same_xcd = !cross;

  // The workgroup's part of the product and the units it finishes.
  const int xcd_base = xi * cs.xcd_units;
  const int xcd_units = BACK ? max(0, min(cs.xcd_units, H - xcd_base)) : 0;
  const int chunk = wi % cs.chunks, block = wi / cs.chunks + (BACK ? 0 : xi * cs.blocks);
  const bool in_grid = wi < cs.chunks * cs.blocks;
  const int k0 = chunk * KR;
  const int block_unit = block * (BACK ? 16 : 4) * CT;  // first unit of the block's columns
  const bool multiplies = in_grid && block_unit < H && k0 < (BACK ? 4 * xcd_units : H);
  const int u0 = BACK ? xcd_base + wi * O : block_unit + chunk * O;
  const int u_end = BACK ? xcd_base + xcd_units : min(H, block_unit + 4 * CT);
  const int units = (BACK || in_grid) ? max(0, min(O, u_end - u0)) : 0;
  const bool finishes = units > 0;

  // Operands: [row tile][4][groups of 32 k][part][lane]; backward, those of an XCD.
  const int k_groups = cs.chunks * 4 * KS;
  const int tile_bytes = k_groups * 3 * 1024;
  const int set_bytes = kPolledTiles * tile_bytes;
  const int max_tiles = (cs.tiles + cs.groups - 1) / cs.groups;
  char* operands = cs.operands + (size_t)(group * (BACK ? cs.span : 1) + (BACK ? xi : 0)) * max_tiles * set_bytes;
  const TileBuffer ob = make_tile_buffer(reinterpret_cast<float*>(operands), max_tiles * (set_bytes / 4));
  // Pieces: [row tile][2][destination][source][groups of four columns of a row].
  const int sources = BACK ? cs.span * cs.chunks : cs.chunks;
  const int finishers = BACK ? cs.xcd_units / O : cs.chunks;  // of an XCD or a block
  const int piece_bytes = (BACK ? O / 4 : O) * kCutRows * 16;
  const int pieces_bytes = (BACK ? cs.span * finishers : cs.span * cs.blocks * cs.chunks) * sources * piece_bytes;
  float* pieces = cs.pieces + (size_t)group * max_tiles * 2 * (pieces_bytes / 4);
  const TileBuffer pb = make_tile_buffer(pieces, max_tiles * 2 * (pieces_bytes / 4));
  constexpr int kAgentScope = 16;  // the sc1 bit of the cache policy
  constexpr int kNowhere = 0x70000000;
  typedef unsigned int uint2_t __attribute__((ext_vector_type(2)));

  // Operands go to all XCDs of the group forward and stay on one backward; pieces the other way round.
  auto store_operand = [&](int at, int tile_at, uint2_t v) {
    if (!BACK && cross) __builtin_amdgcn_raw_buffer_store_b64(v, ob.rsrc, at, tile_at, kAgentScope);
    else __builtin_amdgcn_raw_buffer_store_b64(v, ob.rsrc, at, tile_at, 0);
  };
  auto store_piece = [&](int at, int tile_at, const float4_t& v) {
    const uint4_t bits = __builtin_bit_cast(uint4_t, v);
    if (BACK && cross) __builtin_amdgcn_raw_buffer_store_b128(bits, pb.rsrc, at, tile_at, kAgentScope);
    else __builtin_amdgcn_raw_buffer_store_b128(bits, pb.rsrc, at, tile_at, 0);
  };
  // Byte of (k, part 0, row) within a buffer; parts are 1 KiB apart, k up to a multiple of 8 contiguous.
  auto operand_byte = [](int k, int row) { return (k >> 5) * 3 * 1024 + (((k >> 3) & 3) * 16 + row) * 16 + (k & 7) * 2; };

  // The batch rows of row tile r start at n0(r).
  auto n0 = [&](int r) { return (group + r * cs.groups) * kCutRows; };

  // ---- set-up
  for (int i = tid; i < 16 * CT; i += 256) lds_nan[i] = 0u;
  __syncthreads();
  // The weights: lane 16*q + m has column m of every tile, k = 8*q .. 8*q+7 of every group of 32.  KEEPS: a wavefront
  // starts with the two tiles that it adds up the sums of.
  auto tile_of = [&](int ct) { return KEEPS ? (2 * wave + ct) % CT : ct; };
  bf16x8_t w[KS][CT][2];
  uint4_t lo[KS][CT - LDS > 0 ? CT - LDS : 1];
  {
    const int base_k = k0 + wave * KS * 32 + 8 * q;
    int column_at[CT];  // forward: of k = base_k; backward: of gate 0 of unit base_k / 4
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
      const int u = block_unit + 4 * tile_of(ct) + c / 4, col = block_unit + 16 * tile_of(ct) + c;
      const int at = BACK ? ((xcd_base + base_k / 4) * H + col) * 4 : ((base_k * G + c % 4) * H + u) * 4;
      const bool ok = multiplies && (BACK ? col < H : c % 4 < G && u < H);
      column_at[ct] = ok ? at : kNowhere;
    }
    // (conditions that could become branches: every load would then wait for the one before it)
    auto offset = [&](int j, int ct, int el) {
      const int k = 32 * j + el;
      int at;
      if constexpr (BACK) {
        const int unit = base_k / 4 + k / 4;
        at = (unit < xcd_units && el % 4 < G ? column_at[ct] : kNowhere) + (el % 4 * H + k / 4) * H * 4;
      } else {
        at = column_at[ct] + k * G * H * 4;
      }
      asm volatile("" : "+v"(at));
      return at;
    };
    unsigned int nans = 0u;
    uint4_t* lds_own = lds_lo + wave * KS * LDS * 64 + lane;
    if constexpr (BACK) load_cut_weights<KS, CT, LDS>(w, lo, lds_own, p.R_t, G * H * H * 4, offset, nans);
    else load_cut_weights<KS, CT, LDS>(w, lo, lds_own, p.R, G * H * H * 4, offset, nans);
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
      if (nans >> ct & 1u) lds_nan[16 * tile_of(ct) + c] = 1u;
  }

  // Pointwise ownership: lane 16*q + c of wavefront w handles row c of the tile, unit u0 + 4*w + q.
  const int eu = 4 * wave + q;
  const int e = eu * kCutRows + c;  // (of the elements in LDS)
  const bool owner = wave < O / 4 && finishes;
  const bool mine = owner && eu < units;
  const int unit = mine ? u0 + eu : 0;
  // What the lane publishes: forward part q of units u0+4w .. +3 of row c, backward the gates of its unit, all parts.
  const bool pub = BACK ? mine : owner && 4 * wave < units && q < 3;
  const int pub_at = !pub ? kNowhere
                          : (BACK ? operand_byte(4 * (unit - xcd_base), c) : operand_byte(u0 + 4 * wave, c) + q * 1024);
  auto publish_words = [&](int slot_tile, int buffer, const uint2_t (&v)[BACK ? 3 : 1], bool ok) {
#pragma unroll
    for (int i = 0; i < (BACK ? 3 : 1); ++i)
      store_operand((ok ? pub_at : kNowhere) + i * 1024, (slot_tile * kPolledTiles + buffer) * tile_bytes, v[i]);
  };
  auto publish_unwritten = [&](int slot_tile, int buffer, bool ok) {
    uint2_t v[BACK ? 3 : 1];
#pragma unroll
    for (int i = 0; i < (BACK ? 3 : 1); ++i) v[i] = uint2_t{kUnwrittenBits, kUnwrittenBits};
    publish_words(slot_tile, buffer, v, ok);
  };
  auto publish_state = [&](int slot_tile, int buffer, float h, bool ok) {
    unsigned int r[4] = {0u, 0u, 0u, 0u};
    cut_pair(h, 0.f, r[0], r[1], r[2]);
    transpose_groups(r);
    uint2_t v[BACK ? 3 : 1];
    // (the low halves: the second float's parts, zero but for the sign, are in the high ones)
    v[0] = uint2_t{__builtin_amdgcn_perm(r[1], r[0], 0x05040100u), __builtin_amdgcn_perm(r[3], r[2], 0x05040100u)};
    publish_words(slot_tile, buffer, v, ok);
  };

  // Operands nobody publishes stay zero: k beyond the problem, rows beyond the batch.
  {
    const int k_end = BACK ? 4 * xcd_units : (H + 3) / 4 * 4;
    const int quads = (k_groups * 32 - k_end) / 4;
    const int workers = BACK ? p.ls.gx : cs.span * p.ls.gx;
    const int me = BACK ? wi : (int)gs.my_index;
    for (int i = me * 256 + tid; i < quads * 48 * RT * kPolledTiles; i += workers * 256) {
      const int row = i % 16, part = i / 16 % 3, rest = i / 48;
      store_operand(operand_byte(k_end + 4 * (rest % quads), row) + part * 1024 + rest / quads * tile_bytes, 0, uint2_t{0u, 0u});
    }
  }
  Cell cell;
  for (int r = 0; r < RT; ++r) {
    const bool row_ok = n0(r) + c < N, act = mine && row_ok;
    if constexpr (BACK) cell.load_carried(p, act ? (size_t)(n0(r) + c) * H + unit : 0, act);
    else cell.load_state(p, act ? (size_t)(n0(r) + c) : 0, (size_t)unit, act);
    if (owner)
#pragma unroll
      for (int i = 0; i < CARRIED; ++i) lds_state[(r * plane + e) * CARRIED + i] = cell.carried(i);
    if (row_ok) {
      if constexpr (!BACK) publish_state(r, 0, cell.carried(0), true);
      for (int b = BACK ? 0 : 1; b < kPolledTiles; ++b) publish_unwritten(r, b, true);
    } else {
      uint2_t zero[BACK ? 3 : 1];
#pragma unroll
      for (int i = 0; i < (BACK ? 3 : 1); ++i) zero[i] = uint2_t{0u, 0u};
      for (int b = 0; b < kPolledTiles; ++b) publish_words(r, b, zero, true);
    }
  }

  // The partial sums of a workgroup: item i = 64*ct + 16*q + c is columns 16*ct + 4*q .. +3 of row c.
  auto item = [&](int n) { return KEEPS ? (2 * wave + n) * 64 + lane : tid + 256 * n; };
  auto has_item = [&](int n) { return ITEMS % 256 == 0 || n < ITEM_N - 1 || wave < ITEMS % 256 / 64; };
  int piece_at[ITEM_N];
#pragma unroll
  for (int n = 0; n < ITEM_N; ++n) {
    const int i = item(n), col = (i >> 4) * 4, row = i & 15;
    int to, at;
    bool ok = multiplies && i < ITEMS;
    if constexpr (BACK) {
      const int u = block_unit + col, in_xcd = u % cs.xcd_units;
      ok = ok && u < H;
      to = u / cs.xcd_units * finishers + in_xcd / O;
      at = in_xcd % O / 4 * 16 + row;
    } else {
      const int u = col / 4;
      ok = ok && block_unit + u < H;
      to = block * cs.chunks + u / O;
      at = u % O * 16 + row;
    }
    piece_at[n] = ok ? (to * sources + (BACK ? xi * cs.chunks : 0) + chunk) * piece_bytes + at * 16 : kNowhere;
  }
  {
    const float stale = __uint_as_float(1u ^ scatter_tag(0));
    for (int b = 0; b < 2 * RT; ++b)
#pragma unroll
      for (int n = 0; n < ITEM_N; ++n) store_piece(piece_at[n], b * pieces_bytes, float4_t{stale, stale, stale, stale});
  }
  // The pieces a lane adds up.  Forward: those of its element.  Backward: wavefront w takes every fourth source (or pair of
  // sources, where a piece is half a KiB), lane by lane.
  const int dest = BACK ? xi * finishers + wi : block * cs.chunks + chunk;
  const int per_load = BACK && O <= 8 ? 2 : 1;  // sources a wavefront reads with one load
  int gather_at = kNowhere;
  unsigned int real = 0u;  // bit f: load f of the lane is of a source
#pragma unroll
  for (int f = 0; f < kCutLoads; ++f) {
    int source = f, at = tid;
    bool ok = mine;
    if constexpr (BACK) {
      source = (4 * f + wave) * per_load + (per_load == 2 ? lane >> 5 : 0);
      at = per_load == 2 ? lane & 31 : lane;
      const int from = source / cs.chunks, k = source % cs.chunks * KR;
      ok = finishes && at / 16 * 4 < units && k < 4 * max(0, min(cs.xcd_units, H - from * cs.xcd_units));
    }
    ok = ok && source < sources;
    if (f == 0 && (BACK ? finishes && at / 16 * 4 < units : mine)) gather_at = (dest * sources + source) * piece_bytes + at * 16;
    real |= ok ? 1u << f : 0u;
  }
  const int gather_step = (BACK ? 4 * per_load : 1) * piece_bytes;  // from load to load
  const int loads = BACK ? (sources + 4 * per_load - 1) / (4 * per_load) : sources;

  // What a thread moves between the caller's memory and LDS: four units of a row of a plane.
  const bool zoneout = [&] {
    if constexpr (BACK) return p.zoneout_mask != nullptr;
    else return p.zoneout_prob != 0.f && p.zoneout_mask != nullptr;
  }();
  const int quads = O / 4, per_plane = quads * kCutRows;
  const bool masked = [&] {
    if constexpr (BACK) return zoneout;
    else return zoneout && p.training;
  }();
  const int out_planes = [&] {
    if constexpr (BACK) return (int)Cell::kOut;
    else return p.training ? (int)Cell::kOut : (int)Cell::kStates;
  }();
  auto in_used = [&](int i) {
    if constexpr (BACK) return Cell::in_used(p, Cell::cut_input(i), zoneout);
    else return i < G || masked;
  };
  auto in_row = [&](int i, size_t row) -> const float* {
    if constexpr (BACK) return Cell::in_row(p, Cell::cut_input(i), row);
    else return i < G ? Cell::in_row(p, i, row) : p.zoneout_mask + row * H;
  };
  // (A row that a thread does not move: 255.  The addresses go from slot to slot by what a tile and a step are apart.)
  struct Moved {
    GlobalByte* at;
    int row, lds, pitch;  // pitch: bytes between batch rows
  };
  Moved in[IN_N], out[OUT_N];
  float4_t moved[IN_N];
  const int tile_rows = cs.groups * kCutRows, step_rows = (BACK ? -N : N) - (RT - 1) * tile_rows;
  // Two wavefronts without units of their own to finish move everything while the others finish theirs.
  const bool helpers = O <= 8 && cs.areas == 2;
  const bool helps = !helpers || wave >= 2;
  const int helper = tid - (helpers ? 128 : 0), movers = helpers ? 128 : 256;
  auto set_up_item = [&](Moved& m, int i, bool used, auto row_of) {
    const int first_unit = 4 * (i % quads), row = i / quads % kCutRows;
    const bool ok = helps && used && first_unit < units;
    m.row = ok ? row : 255;
    const size_t first = (size_t)(BACK ? T - 1 : 0) * N + n0(0) + row;
    const char* start = reinterpret_cast<const char*>(row_of(0));
    const int row_bytes = (int)(reinterpret_cast<const char*>(row_of(1)) - start);
    m.at = (GlobalByte*)(const_cast<char*>(start) + (ok ? first * row_bytes + (u0 + first_unit) * 4 : 0));
    m.pitch = ok ? row_bytes : 0;
  };
#pragma unroll
  for (int n = 0; n < IN_N; ++n) {
    const int i = max(0, helper) + movers * n, pl = i / per_plane < IN_PLANES ? i / per_plane : 0;
    set_up_item(in[n], i, i / per_plane < IN_PLANES && in_used(pl), [&](size_t row) { return in_row(pl, row); });
    in[n].lds = (4 * (i % quads) * kCutRows + i / quads % kCutRows) * IN_P + pl;
    moved[n] = float4_t{0.f, 0.f, 0.f, 0.f};
  }
#pragma unroll
  for (int n = 0; n < OUT_N; ++n) {
    const int i = max(0, helper) + movers * n, pl = i / per_plane < Cell::kOut ? i / per_plane : 0;
    set_up_item(out[n], i, i / per_plane < out_planes, [&](size_t row) { return Cell::out_row(p, pl, row); });
    int value = pl;
    if constexpr (BACK) value = Cell::out_value(pl);
    out[n].lds = (4 * (i % quads) * kCutRows + i / quads % kCutRows) * OUT_P + value;
  }
  auto advance = [&](Moved& m, const CutSlot& s) { m.at += __mul24(m.pitch, s.tile == RT - 1 ? step_rows : tile_rows); };
  // (units of the workgroup from item i's first on)
  auto units_left = [&](int n) { return units - 4 * ((max(0, helper) + movers * n) % quads); };
  auto request = [&](const CutSlot& s) {
    if (s.step >= T) return;
    const int rows = min(N - n0(s.tile), 255);
    if constexpr (WIDE) {
#pragma unroll
      for (int n = 0; n < IN_N; ++n)
        if (in[n].row < rows) moved[n] = *(const GlobalFloat4*)in[n].at;
    } else {
#pragma unroll
      for (int n = 0; n < IN_N; ++n)
        if (in[n].row < rows)
#pragma unroll
          for (int k = 0; k < 4; ++k) moved[n][k] = ((const GlobalFloat*)in[n].at)[k < units_left(n) ? k : 0];
    }
#pragma unroll
    for (int n = 0; n < IN_N; ++n) advance(in[n], s);
  };
  auto park = [&](const CutSlot& s, int area) {
    if (s.step >= T) return;
#pragma unroll
    for (int n = 0; n < IN_N; ++n)
      if (in[n].row < 255) {
        float* to = lds_in + area * in_floats + in[n].lds;
#pragma unroll
        for (int k = 0; k < 4; ++k) to[k * kCutRows * IN_P] = moved[n][k];
      }
  };
  auto write_copies = [&](const CutSlot& s, int area) {
    if (s.step >= T) return;
    const int rows = min(N - n0(s.tile), 255);
#pragma unroll
    for (int n = 0; n < OUT_N; ++n) {
      if (out[n].row < rows) {
        const float* from = lds_out + area * out_floats + out[n].lds;
        float4_t v;
#pragma unroll
        for (int k = 0; k < 4; ++k) v[k] = from[k * kCutRows * OUT_P];
        if constexpr (WIDE) {
          *(GlobalFloat4*)out[n].at = v;
        } else {
#pragma unroll
          for (int k = 0; k < 4; ++k)
            if (k < units_left(n)) ((GlobalFloat*)out[n].at)[k] = v[k];
        }
      }
      advance(out[n], s);
    }
  };

  // The operands of a slot.
  uint4_t a[KS][3];
  const int operand_at = multiplies ? (k0 / 32 + wave * KS) * 3 * 1024 + lane * 16 : kNowhere;  // (beyond it: zeros)
  auto load_parts = [&](const CutSlot& s, int first, int end) {
    const int tile_at = (s.tile * kPolledTiles + (s.step & 3)) * tile_bytes;
#pragma unroll
    for (int j = 0; j < KS; ++j)
#pragma unroll
      for (int part = first; part < end; ++part)
        // (what does not fit an instruction's offset goes into the scalar one: no register per address)
        a[j][part] = __builtin_amdgcn_raw_buffer_load_b128(ob.rsrc, operand_at + (3 * j + part) % 4 * 1024,
                                                           tile_at + (3 * j + part) / 4 * 4096, kAgentScope);
  };
  auto load_operands = [&](const CutSlot& s) { load_parts(s, 0, 3); };
  // The pieces of a slot.
  static_assert(kCutLoads == 4, "pieces of a lane");
  float4_t piece[kCutLoads];
  auto load_pieces = [&](const CutSlot& s) {
    const int tile_at = (s.tile * 2 + (s.step & 1)) * pieces_bytes;
    auto load = [&](int f) {
      piece[f] = __builtin_bit_cast(float4_t, __builtin_amdgcn_raw_buffer_load_b128(pb.rsrc, gather_at, tile_at + f * gather_step, kAgentScope));
    };
    load(0);
    load(1);
    if (loads > 2) {
      load(2);
      load(3);
    }
  };
  auto add_pieces = [&](const CutSlot& s) {
    const unsigned int tag = scatter_tag(s.step);
    auto arrived = [&] {
      auto missing = [&](int f) {
        const uint4_t b = __builtin_bit_cast(uint4_t, piece[f]);
        const unsigned int x = tag ? ~b.x | ~b.y | ~b.z | ~b.w : b.x | b.y | b.z | b.w;
        return x & (real >> f);
      };
      unsigned int m = missing(0) | missing(1);
      if (loads > 2) m |= missing(2) | missing(3);
      return __all((m & 1u) == 0u) != 0;
    };
    // (The first look by itself: inside the loop it would wait for everything stored since the loads, too.)
    if (!arrived()) {
      load_pieces(s);
      poll_until_written(gs, [&] { load_pieces(s); }, arrived);
    }
    auto of_source = [&](int f) { return real >> f & 1u ? piece[f] : float4_t{0.f, 0.f, 0.f, 0.f}; };
    auto total = [&] {
      const float4_t two = of_source(0) + of_source(1);
      return loads > 2 ? two + (of_source(2) + of_source(3)) : two;
    };
    float4_t v = total();
    // An infinite partial sum tagged 1 reads as a signalling NaN, which arithmetic does not make.
    const float all = (v.x + v.y) + (v.z + v.w);
    if (__any(all != all)) {
#pragma unroll
      for (int f = 0; f < kCutLoads; ++f)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const unsigned int b = __float_as_uint(piece[f][i]);
          piece[f][i] = (b & 0x7fffffffu) == 0x7f800001u ? __uint_as_float(b & ~1u) : piece[f][i];
        }
      v = total();
    }
    return v;
  };

  float step_sums[SUMS];
#pragma unroll
  for (int i = 0; i < SUMS; ++i) step_sums[i] = 0.f;
  // Backward, odd rows go through the product with their signs changed (see split_backward_kernel).
  const float sign_scale = BACK && (c & 1) ? -kProductScale : kProductScale;
  float* lds_part = lds_state + CARRIED * RT * plane;  // backward: [4][own][16] floats, four units of a row side by side
  float2_t* lds_totals = reinterpret_cast<float2_t*>(lds_part + 4 * plane);  // backward: column sums [own][SUMS]
  if (BACK && owner && c == 0)
#pragma unroll
    for (int i = 0; i < SUMS; ++i) lds_totals[eu * SUMS + i] = float2_t{0.f, 0.f};
  auto leave_parts = [&](const CutSlot& s) {
    const float4_t v = add_pieces(s);
    if (per_load == 2) {
      // both halves of the wavefront hold sums of the same elements; each ends up with two units
      const float2_t two = {swap_add32(v.x, v.z), swap_add32(v.y, v.w)};
      if ((lane & 31) < O * 4)
        *reinterpret_cast<float2_t*>(lds_part + wave * plane + (lane & 31) * 4 + 2 * (lane >> 5)) = two;
    } else if (lane < O * 4) {
      *reinterpret_cast<float4_t*>(lds_part + wave * plane + lane * 4) = v;
    }
  };
  // The end of slot `s`: forward with the sums of its products, backward (sums: whether there are any yet) those that
  // were asked for a step before.
  auto finish = [&](const CutSlot& s, bool gathered, int area) {
    const float* from = lds_in + area * in_floats + e * IN_P;
    float* to = lds_out + area * out_floats + e * OUT_P;
    const bool act = mine && n0(s.tile) + c < N;
    float* state = lds_state + (s.tile * plane + e) * CARRIED;
    if constexpr (BACK) {
      if (!owner) return;
#pragma unroll
      for (int i = 0; i < CARRIED; ++i) cell.carried(i) = state[i];
      float dh = 0.f;
      if (gathered) {
        const float* part = lds_part + (eu >> 2) * 64 + c * 4 + (eu & 3);
        dh = (part[0] + part[plane]) + (part[2 * plane] + part[3 * plane]);
      }
      cell.add_gathered(dh);
      float4_t dv = {0.f, 0.f, 0.f, 0.f};
      if (s.step < T) {
        float in[Cell::kInputs];
        float4_t words[IN_P / 4];
#pragma unroll
        for (int i = 0; i < IN_P / 4; ++i) words[i] = *reinterpret_cast<const float4_t*>(from + 4 * i);
#pragma unroll
        for (int i = 0; i < IN_PLANES; ++i) in[Cell::cut_input(i)] = words[i / 4][i % 4];
        cell.carry_inputs(in);
        cell.prepare(in);
        dv = cell.step(act, zoneout, step_sums);
        const float sign = c & 1 ? -1.f : 1.f;
        const float dg[4] = {sign * dv[0], sign * dv[1], sign * dv[2], G > 3 ? sign * dv[3] : 0.f};
        unsigned int low[3], high[3];
        cut_pair(dg[0], dg[1], low[0], low[1], low[2]);
        cut_pair(dg[2], dg[3], high[0], high[1], high[2]);
        uint2_t v[BACK ? 3 : 1];
#pragma unroll
        for (int i = 0; i < (BACK ? 3 : 1); ++i) v[i] = uint2_t{low[i], high[i]};
        publish_words(s.tile, s.step & 3, v, act);
        if (s.step + 2 < T) publish_unwritten(s.tile, (s.step + 2) & 3, act);
        *reinterpret_cast<float4_t*>(to) = dv;
        if (s.tile == RT - 1) {
#pragma unroll
          for (int i = 0; i < SUMS; ++i) {
            const float rows = sum_of_rows(step_sums[i]);
            if (c == 0) {  // (with what an addition loses, which hundreds of them would add up to)
              float2_t& total = lds_totals[eu * SUMS + i];
              const float next = rows - total.y, sum = total.x + next;
              total = float2_t{sum, (sum - total.x) - next};
            }
            step_sums[i] = 0.f;
          }
        }
#pragma unroll
        for (int i = 0; i < CARRIED; ++i) state[i] = cell.carried(i);
      } else if (act) {
        cell.store_state(p, (size_t)(n0(s.tile) + c) * H + unit);
      }
    } else {
      if (!owner) return;
      const float4_t rh = add_pieces(s);
      float4_t in = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int g = 0; g < G; ++g) in[g] = from[g];
      const float mask = masked ? from[G] : 1.f;
#pragma unroll
      for (int i = 0; i < CARRIED; ++i) cell.carried(i) = state[i];
      if (act) cell.step(p, in, mask, rh, zoneout);
      if (s.step + 1 < T) {
        const bool ok = n0(s.tile) + c < N;
        publish_state(s.tile, (s.step + 1) & 3, act ? cell.carried(0) : 0.f, ok);
        if (s.step + 3 < T) publish_unwritten(s.tile, (s.step + 3) & 3, ok);
      }
#pragma unroll
      for (int i = 0; i < CARRIED; ++i) state[i] = cell.carried(i);
#pragma unroll
      for (int i = 0; i < Cell::kOut; ++i)
        if (i < out_planes) to[i] = cell.out(i);
    }
  };
  // Sums that are not finite, formed again from the floats themselves (something did not split or grew too large) unless
  // a NaN among their operands accounts for them.
  auto sum_again = [&](const CutSlot& s, int i, float4_t v) {
    const int tile_at = (s.tile * kPolledTiles + (s.step & 3)) * tile_bytes;
    const char* tile = operands + tile_at;
    bool row_nan = false;
#pragma nounroll
    for (int g = 0; g < 4 * KS; ++g) {
      const uint4_t x = __builtin_amdgcn_raw_buffer_load_b128(ob.rsrc, (k0 / 32 + g) * 3 * 1024 + lane * 16, tile_at, kAgentScope);
#pragma unroll
      for (int j = 0; j < 4; ++j) row_nan = row_nan || (x[j] & 0xffffu) == kNanMark || x[j] >> 16 == kNanMark;
    }
    const unsigned long long rows = __ballot(row_nan);
    row_nan = ((rows | rows >> 16 | rows >> 32 | rows >> 48) >> c & 1ull) != 0;
    const int col = (i >> 4) * 4;
    bool again[4];
    bool any = false;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      again[j] = !(fabsf(v[j]) <= 0x1.fffffep127f) && !row_nan && lds_nan[col + j] == 0u;
      any = any || again[j];
    }
    if (!__any(any)) return v;
    float4_t sum = {0.f, 0.f, 0.f, 0.f};
    const int k_end = min(KR, (BACK ? 4 * xcd_units : H) - k0);
#pragma unroll 2
    for (int k = 0; k < k_end; ++k) {
      const unsigned short* at = reinterpret_cast<const unsigned short*>(tile + operand_byte(k0 + k, c));
      unsigned int part[3];
#pragma unroll
      for (int j = 0; j < 3; ++j) part[j] = __hip_atomic_load(at + j * 512, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      const float x = cut_value(part[0], part[1], part[2]);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        float weight = 0.f;
        if constexpr (BACK) {
          const int u = xcd_base + (k0 + k) / 4, gate = (k0 + k) % 4, column = block_unit + col + j;
          if (gate < G && column < H) weight = p.R_t[((size_t)gate * H + u) * H + column];
        } else {
          const int u = block_unit + col / 4;
          if (j < G && u < H) weight = p.R[((size_t)(k0 + k) * G + j) * H + u];
        }
        sum[j] = fmaf(x, weight, sum[j]);
      }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (again[j]) v[j] = BACK && (c & 1) ? -sum[j] : sum[j];
    return v;
  };

  // ---- the steps
  const bool single = !MANY && RT == 1;  // (where there are many, a group has at least two)
  CutSlot in_slot{0, 0};  // whose inputs are parked next
  int area = 0;           // of the inputs and copies that the next finish takes
  group_arrive(gs);
  if (!multiplies && !finishes) return;
  group_wait(gs);
  const bool ahead = helpers && !single;  // inputs of a finish are parked during the one before it, else before its product ends
  if (BACK || ahead) {
    request(in_slot);
    park(in_slot, 0);
    in_slot.next(RT);
  }
  if constexpr (BACK) {
    // The gradients of the last step come from outside alone.
    for (CutSlot s{0, 0}; s.step == 0; s.next(RT)) {
      __syncthreads();
      finish(s, false, 0);
      __syncthreads();
      write_copies(s, 0);
      if (ahead || s.tile + 1 < RT) {
        request(in_slot);
        park(in_slot, 0);
        in_slot.next(RT);
      }
    }
  }
  if (ahead) request(in_slot);
  // What a finish leaves is written while the next one is at work (the wavefronts without units have the time), or else
  // where others are waited for.
  CutSlot written{0, 0};
  if (BACK) written.step = 1;
  bool left = false;
  auto write_left = [&](int from_area) {
    if (!left) return;
    write_copies(written, from_area);
    written.next(RT);
    left = false;
  };
  auto finish_slot = [&](CutSlot target) {
    if (BACK) ++target.step;
    if (ahead && helps) {
      write_left(area ^ 1);
      park(in_slot, area ^ 1);
      in_slot.next(RT);
      request(in_slot);
    }
    finish(target, true, area);
    __syncthreads();
    left = target.step < T;
    if (ahead) area ^= 1;
  };
  CutSlot slot{0, 0}, done{0, 0};  // `done`: the slot that is finished beside this one's product
  load_operands(slot);
  for (bool first = true; slot.step < T; first = false) {
    const bool ends = !single && !first;
    CutSlot next = slot;
    next.next(RT);
    auto arrived = [&] {
      unsigned int m = 0u;
#pragma unroll
      for (int j = 0; j < KS; ++j)
#pragma unroll
        for (int part = 0; part < 3; ++part) {
          const uint4_t& v = a[j][part];
          const unsigned int xy = v.x > v.y ? v.x : v.y, zw = v.z > v.w ? v.z : v.w;
          const unsigned int x = xy > zw ? xy : zw;
          m = m > x ? m : x;
        }
      return __all(m != kUnwrittenBits) != 0;
    };
    if (!arrived()) {  // (see add_pieces)
      load_operands(slot);
      poll_until_written(gs, [&] { load_operands(slot); }, arrived);
    }
    if (!ahead && (single || ends)) request(in_slot);
    float4_t acc[CT];
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) acc[ct] = float4_t{0.f, 0.f, 0.f, 0.f};
    cut_small_products<KS, CT, LDS>(a, w, lo, lds_lo + wave * KS * LDS * 64 + lane, acc);
    // What the end of this slot and the next slot need, where it has been published by now, comes beside the rest: a
    // wavefront's loads take the memory pipeline as long as these products take the matrix cores.
    // (Nothing here depends on a condition, or the wait for the pieces would have to be one for everything: what a slot
    // beyond the last one would read lies within the buffers.)
    if (MANY || ends) load_pieces(done);
    if (MANY) load_parts(next, 1, 3);
    __builtin_amdgcn_sched_barrier(0);
    cut_large_products<KS, CT>(a, w, acc);
    if (MANY) load_parts(next, 0, 1);
#pragma unroll
    for (int ct = KEEPS ? 2 : 0; ct < CT; ++ct) {
      // (the wavefronts after this one, in turn, have it as the third, second and first before them)
      if (KEEPS) lds_sums[(((wave + ct / 2) % 4 * 3 + ct / 2 - 1) * 2 + ct % 2) * 64 + lane] = acc[ct];
      else lds_sums[wave * ITEMS + ct * 64 + lane] = acc[ct];
    }
    if (!ahead && (single || ends)) {
      park(in_slot, 0);
      in_slot.next(RT);
    }
    if (BACK && ends && finishes) leave_parts(done);
    __syncthreads();
    if (multiplies) {
      const unsigned int tag = scatter_tag(slot.step);
      const int tile_at = (slot.tile * 2 + (slot.step & 1)) * pieces_bytes;
      static_assert(ITEM_N <= 2, "items of a thread");
      constexpr int OTHERS = KEEPS ? 3 : 4;
      float4_t v[ITEM_N], other[ITEM_N][OTHERS];
#pragma unroll
      for (int n = 0; n < ITEM_N; ++n)
#pragma unroll
        for (int i = 0; i < OTHERS; ++i)  // (the items of wavefronts that have one less: anything)
          other[n][i] = lds_sums[KEEPS ? (wave * 3 + i) * 128 + n * 64 + lane : (has_item(n) ? item(n) : 0) + i * ITEMS];
      __builtin_amdgcn_sched_barrier(0);
      float finite = 0.f;
#pragma unroll
      for (int n = 0; n < ITEM_N; ++n) {
        v[n] = ((KEEPS ? acc[n] : other[n][OTHERS - 1]) + other[n][0]) + (other[n][1] + other[n][2]);
        finite += (v[n].x + v[n].y) + (v[n].z + v[n].w);
        v[n] *= sign_scale;
      }
      if (__any(!(fabsf(finite) <= 0x1.fffffep127f))) {
#pragma nounroll
        for (int n = 0; n < ITEM_N; ++n) {
          if (!has_item(n)) break;
          const float4_t again = sum_again(slot, item(n), n == 0 ? v[0] : v[ITEM_N - 1]);
          if (n == 0) v[0] = again;
          else v[ITEM_N - 1] = again;
        }
      }
#pragma unroll
      for (int n = 0; n < ITEM_N; ++n) store_piece(piece_at[n], tile_at, tagged4(v[n], tag));
    }
    if (single) {
      if (BACK) write_left(0);
      if (finishes) load_pieces(done);
      if (BACK) {
        if (finishes) leave_parts(done);
        __syncthreads();
      }
    }
    if (single || ends) {
      finish_slot(done);
      done.next(RT);
    } else {
      __syncthreads();
    }
    // (The copies first: operands requested too early have to be requested again.)
    if (!ahead && !(BACK && single)) write_left(0);
    if (!MANY && next.step < T) load_operands(next);
    slot = next;
  }
  if (!single) {
    if (!ahead) {
      request(in_slot);
      park(in_slot, 0);
    }
    if (finishes) load_pieces(done);
    if (BACK && finishes) leave_parts(done);
    __syncthreads();
    finish_slot(done);
  }
  write_left(ahead ? area ^ 1 : 0);

  if constexpr (BACK) {
    if (finishes) {
      // Column sums (bias gradients), parked per group; the last group to finish adds them in order.
      __syncthreads();
      const int sum = tid / 16, su = tid % 16;
      if (sum < SUMS && su < units) {
        const float total = lds_totals[su * SUMS + sum].x;
        store_agent(&cs.sums[((size_t)group * SUMS + sum) * H + u0 + su], total);
      }
      if (column_last_arrival(p.ls.cb, (int)gs.my_index, (unsigned)cs.groups, lds_nan)) {
        if (sum < SUMS && su < units) {
          const int col = sum * H + u0 + su;
          Cell::add_sums(p, col, sum_over_tiles(cs.sums + col, (size_t)SUMS * H, cs.groups));
        }
      }
    }
  }
}

// ---- which calls take it -----------------------------------------------------------------------

struct CutPlan {
  bool ok = false;
  int ks = 0, ct = 0, row_tiles = 0;
  CutShape s{};
  size_t lds = 0, sum_floats = 0, weight_floats = 0, piece_floats = 0, operand_bytes = 0;
  size_t bytes() const { return (sum_floats + weight_floats + piece_floats) * sizeof(float) + operand_bytes; }
};

// The geometry for N rows and H units on `cus` compute units in `xcds` XCDs: the fewest XCDs per group that hold the weights
// (more groups, fewer tiles each).
template <class Cell, bool BACK>
CutPlan cut_plan(int N, int H, int cus, int xcds) {
  CutPlan plan;
  if (xcds <= 0 || cus % xcds != 0) return plan;
  const int per_xcd = cus / xcds;
  auto up = [](int a, int b) { return (a + b - 1) / b; };
  for (int span = 1; span <= xcds; span *= 2) {
    if (xcds % span != 0) continue;
    for (int variant = 0; variant < 2; ++variant) {
      const int ks = variant == 0 ? 3 : 4, ct = variant == 0 ? 6 : 8, range = 128 * ks;
      CutShape s{};
      s.xcds = xcds;
      s.span = span;
      s.tiles = up(N, kCutRows);
      s.groups = std::min(xcds / span, s.tiles);
      if (BACK) {
        s.blocks = up(H, 16 * ct);
        // (the workgroups that share an XCD's units take a multiple of four each)
        const int fair = up(H, span);
        s.own = up(up(fair, per_xcd), 4) * 4;
        s.xcd_units = up(fair, s.own) * s.own;
        s.chunks = up(4 * s.xcd_units, range);
        if (s.chunks * s.blocks > per_xcd || s.xcd_units / s.own > per_xcd) continue;
        const int per_load = s.own <= 8 ? 2 : 1;
        if (up(span * s.chunks, 4 * per_load) > kCutLoads) continue;
      } else {
        s.chunks = up(H, range);
        s.blocks = per_xcd / s.chunks;
        if (s.chunks > kCutLoads || s.blocks * span * 4 * ct < H) continue;
        s.own = up(up(4 * ct, s.chunks), 4) * 4;
      }
      if (s.own > 16) continue;
      const int row_tiles = up(s.tiles, s.groups);
      const size_t fixed = variant == 0 ? cut_fixed_lds_bytes<3, 6>() : cut_fixed_lds_bytes<4, 8>();
      constexpr int inputs = cut_in_words<Cell, BACK>(), copies = cut_out_words<Cell, BACK>();
      int sums = 0;
      if constexpr (BACK) sums = Cell::kSums;
      s.areas = s.own <= 8 && row_tiles > 1 ? 2 : 1;
      if (cut_lds_bytes(fixed, s.areas, inputs, copies, Cell::kCarried, sums, s.own, row_tiles) > kWorkgroupLdsBytes) s.areas = 1;
      const size_t lds = cut_lds_bytes(fixed, s.areas, inputs, copies, Cell::kCarried, sums, s.own, row_tiles);
      if (lds > kWorkgroupLdsBytes) continue;
      plan.ok = true;
      plan.ks = ks;
      plan.ct = ct;
      plan.row_tiles = row_tiles;
      plan.s = s;
      plan.lds = lds;
      const int sources = BACK ? span * s.chunks : s.chunks;
      const int dests = BACK ? span * (s.xcd_units / s.own) : span * s.blocks * s.chunks;
      const size_t piece = (size_t)(BACK ? s.own / 4 : s.own) * kCutRows * 4;
      plan.piece_floats = (size_t)s.groups * row_tiles * 2 * dests * sources * piece;
      plan.operand_bytes = (size_t)s.groups * (BACK ? span : 1) * row_tiles * kPolledTiles * s.chunks * 4 * ks * 3 * 1024;
      if constexpr (BACK) plan.sum_floats = ((size_t)s.groups * Cell::kSums * H + 63) / 64 * 64;
      return plan;
    }
  }
  return plan;
}

// Whether it pays.  Here a step takes a turn per batch tile of a group (the plan's row_tiles: 4, 2 or 1 groups share them,
// H <= 1024, 1280 and beyond); the others' step grows with the rows of their tiles, which all go at once.  So it does where
// theirs have many rows for every turn here, and where they stream the weights, always.  Measured, C = 64, T = 60, N rows in
// tiles of theirs / turns here, the others -> this one, us:
//   LSTM forward   H =  544  N = 40 8/1 241 -> 262   N = 64 16/1 282 -> 269 (not taken)  N = 96 16/2 293 -> 437  N = 128 64/2 537 -> 447
//                  H =  640  N = 32 16/1 277 -> 262 (not taken)  N = 52 32/1 345 -> 263  N = 72 32/2 361 -> 436  N = 144 64/3 620 -> 623
//                  H =  736  N = 12 8/1 220 -> 262   N = 20 16/1 305 -> 265  N = 40 32/1 417 -> 266  N = 96 64/2 645 -> 475
//                  H = 1024  N = 28 16/1 297 -> 318  N = 48 32/1 447 -> 326  N = 128 64/2 900 -> 604
//                  H = 1056  N = 16 16/1 305 -> 345  N = 28 32/1 457 -> 343  N = 52 64/2 765 -> 533
//       beyond LDS H = 1280  N = 12 16/1 381 -> 348
//                  H = 1536  N = 1 362 -> 284   N = 64 1092 -> 732   N = 128 2048 -> 1407  N = 160 2573 -> 1728
//                  H = 2048  N = 1 430 -> 337   N = 64 1432 -> 940   N = 128 2458 -> 1790  N = 160 3649 -> 2216
//   LSTM backward  H =  544  N = 28 4/1 320 -> 372   N = 40 8/1 388 -> 387   N = 52 8/1 428 -> 397   N = 96 16/2 528 -> 570
//                  H =  608  N = 32 8/1 405 -> 387   N = 64 16/1 587 -> 421  N = 72 16/2 604 -> 558  N = 160 32/3 970 -> 838
//                  H =  800  N = 72 16/2 691 -> 708  N = 96 32/2 1005 -> 771 N = 160 32/5 1188 -> 1277
//                  H =  848  N = 160 64/5 1789 -> 1294
//       beyond LDS H =  640  N = 1 16/1 400 -> 348   N = 72 16/2 524 -> 563  N = 160 32/3 925 -> 854
//                  H = 1536  N = 1 792 -> 383   N = 64 1840 -> 1167  N = 128 2846 -> 2295  N = 160 3736 -> 2824
//                  H = 2048  N = 1 1049 -> 455  N = 64 2368 -> 1699  N = 128 3986 -> 3350  N = 160 5343 -> 4130
//   GRU forward    H =  544  N = 64 16/1 244 -> 267  N = 128 32/2 396 -> 435 H = 672  N = 64 16/1 310 -> 264  N = 96 16/2 323 -> 452
//                  H =  736  N = 28 8/1 236 -> 266   N = 48 16/1 340 -> 264  N = 72 16/2 351 -> 449  N = 96 64/2 625 -> 455
//                  H =  832  N = 20 16/1 326 -> 302  N = 40 32/1 433 -> 305  H = 1024 N = 28 16/1 290 -> 302
//                  H = 1056  N = 28 32/1 441 -> 334
//       beyond LDS H =  736  N = 144 32/3 566 -> 618
//                  H = 1056  N = 40 16/2 368 -> 503  N = 52 32/2 594 -> 528  N = 96 32/3 626 -> 737  N = 128 64/4 1048 -> 914
//                  H = 2048  N = 1 422 -> 323   N = 64 1369 -> 894   N = 160 2938 -> 2059
//   GRU backward   H =  544  N = 28 4/1 373 -> 375   N = 40 8/1 449 -> 383   N = 96 16/2 619 -> 581  N = 144 32/3 736 -> 775
//                  H =  672  N = 28 8/1 434 -> 385   N = 80 16/2 510 -> 604  N = 160 32/3 881 -> 892
//                  H =  736  N = 72 16/2 616 -> 602  N = 160 32/3 988 -> 932
//       beyond LDS H =  864  N = 8 16/1 527 -> 429   H = 1056 N = 48 16/2 651 -> 710  H = 1152 N = 48 16/2 754 -> 712
//                  H = 1312  N = 40 16/3 899 -> 753  N = 80 32/5 1340 -> 1270
//                  H = 2048  N = 1 891 -> 437   N = 64 2223 -> 1553  N = 160 4572 -> 3622
// Whole passes of three steps are level with the others, of eight 0.65 - 1 of theirs.
inline bool cut_pays(bool backward, int gates, int N, int H, const CutPlan& plan, const CutOther& other) {
  const int turns = plan.row_tiles;
  if (other.rows == 0) return true;
  if (!backward) {
    if (other.rows > 16 * turns) return gates == 3 || turns <= 2 || H > 608;
    // as many rows as a turn has: level with them, by how well either fits the size
    return other.rows == 16 * turns && (other.beyond_lds || (turns == 1 && H > 640 && H <= 960));
  }
  // Their backward steps take longer, these hardly do, least where a group is the whole chip.
  if (other.rows >= 16 * turns) return true;
  if (other.rows < (plan.s.span == plan.s.xcds ? 5 : 8) * turns) return false;
  if (gates == 4) {
    if (turns == 1) return H > 576 || N > 48;
    return other.rows > 16 || (H > 576 && (H <= 632 || H > 656));
  }
  if (turns == 1) return true;
  if (other.rows > 16) return H > 576;
  return H <= 656 || (H > 720 && H <= 1024) || H > 1100;
}

// `masked`: the weights are multiplied with a DropConnect mask first, which takes room for them.
template <class Cell, bool BACK>
int cut_rule(hipStream_t stream, int T, int N, int H, const CutOther& other, bool masked, CutPlan* plan) {
  *plan = CutPlan();
  if (T < kCutMinSteps || H <= 512 || N > kCutMaxRows) return HASTE_HIP_OK;
  CutPlan found = cut_plan<Cell, BACK>(N, H, device_cu_count(), device_xcd_count());
  if (!found.ok || !cut_pays(BACK, Cell::kGates, N, H, found, other)) return HASTE_HIP_OK;
  if (masked) found.weight_floats = ((size_t)Cell::kGates * H * H + 63) / 64 * 64;
  bool room = false;
  HASTE_HIP_PROPAGATE(workspace_has_room(stream, found.bytes(), &room));
  if (room) *plan = found;
  return HASTE_HIP_OK;
}

// Launches the kernel for a plan that cut_rule() made (the workspace is looked up here: a GEMM before it may have replaced
// the stream's scratch buffer with a larger one).
template <class Cell, bool BACK>
int launch_cut(const char* name, hipStream_t stream, const CutPlan& cut, typename Cell::Params& p) {
  Workspace ws;
  HASTE_HIP_PROPAGATE(get_workspace(stream, cut.bytes(), &ws));
  HASTE_HIP_PROPAGATE(check_and_clear_abort(stream, &ws));
  LaunchPlan plan;
  HASTE_HIP_PROPAGATE(plan_launch(stream, ws, device_cu_count() / cut.s.xcds, cut.s.xcds, kCutRows, cut.lds, 4, &plan));
  plan.kernel = kPlanSplit;
  plan.group_workgroups = cut.s.span * plan.shape.gx;
  plan.groups = cut.s.groups;
  plan.tiles_each = cut.row_tiles;
  CutParams<typename Cell::Params> cp{p, cut.s};
  cp.p.ls = plan.shape;
  cp.s.sums = ws.scratch;
  float* weights = ws.scratch + cut.sum_floats;
  if constexpr (!BACK) {
    if (p.dc_mask != nullptr) {
      HASTE_HIP_PROPAGATE(scale_weights(stream, (size_t)Cell::kGates * p.H * p.H, p.R, p.dc_mask, p.dc_scale, weights));
      cp.p.R = weights;
    }
  }
  cp.s.pieces = weights + cut.weight_floats;
  cp.s.operands = reinterpret_cast<char*>(cp.s.pieces + cut.piece_floats);
  auto launch = [&](auto kernel) { return launch_persistent(name, kernel, plan, cp, stream); };
  const bool wide = p.H % 4 == 0 && Cell::aligned(p);
  if (cut.ks == 3) {
    if (!wide) return launch(cut_recurrence_kernel<Cell, BACK, 3, 6, false, false>);
    return cut.row_tiles > 2 ? launch(cut_recurrence_kernel<Cell, BACK, 3, 6, true, true>)
                             : launch(cut_recurrence_kernel<Cell, BACK, 3, 6, true, false>);
  }
  if (!wide) return launch(cut_recurrence_kernel<Cell, BACK, 4, 8, false, false>);
  return cut.row_tiles > 2 ? launch(cut_recurrence_kernel<Cell, BACK, 4, 8, true, true>)
                           : launch(cut_recurrence_kernel<Cell, BACK, 4, 8, true, false>);
}

}  // namespace haste_hip
