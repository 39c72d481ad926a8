// The backward recurrence of 8- and 16-row batch tiles in scattered form with the step's product on the bf16 matrix
// cores, for any cell scatter_backward.h can run.
#pragma once

#include "scatter_backward.h"
#include "split_bf16.h"
#include "split_operands.h"

namespace haste_hip {

// A workgroup's LDS: the operands of the step's product; the gathering wavefronts' sums; a step's inputs and its gate
// gradients by step parity; whether some of those do not split.
template <class Cell, int NB>
struct SplitBackwardLds {
  uint4_t operand[NB == 8 ? 3 : 6][64];
  float part[4][16][NB];  // [wavefront][unit][row]
  float in[2][Cell::kInputs][NB][16];
  float out[2][4][NB][16];
  unsigned int large[2][4];
};

constexpr int kSplitPieceTiles = 2;
inline size_t split_piece_floats(int gx, int ctw, int nb) { return (size_t)gx * 4 * ctw * 16 * nb; }

// See "scattered partial sums" in recurrent.h for the ownership, the pieces and their tags, and scatter_backward.h for
// the cells.  Here a workgroup is four wavefronts, one per SIMD, that work on the same NB batch rows: a step is
//   gather      every wavefront adds up the pieces of its quarter of the producers, requested behind the publication of
//               the step before; the sums meet in LDS
//   pointwise   the owners (one thread per row and unit) finish dh and compute the gate gradients, which go, as three
//               bfloat16 each, to LDS as operands of v_mfma_f32_16x16x32_bf16: row, k = 4 * unit + gate.  8 rows share an
//               operand with another part of theirs (see split_operands.h)
//   product     every wavefront multiplies them with the rows of R_t of the workgroup's units and CTW owners' columns,
//               split, in registers for the whole launch (24 * CTW), and publishes the owners' pieces: 16 * NB floats
//               [unit][row], in [owner][producer] order, producers padded to 4 * CTW
// Inputs and the caller's copies move through LDS, 16 bytes per lane; at 8 rows the wavefronts without elements move
// them while the others are at the pointwise step.
// What bounds it: the chain of a step.  LSTM, N = 64, H = 512 (cycles at 2.3 GHz, of about 4 100): the pieces' request to
// their sums 800, barrier 130, pointwise step and split 740, barrier 130, 64 matrix instructions with the publication
// beside them 1 950 (1 075 the instructions alone), the next step's inputs and the copies, while the pieces are on their
// way, 300.  Measured, C = H = 512, T = 100: LSTM N = 64, two sets of 4 rows on the fp32 matrix instructions 264 us ->
// 211; N = 128, gathering the gate gradients instead 480 -> 357.
// Beyond what scatter_backward.h adds to Cell: kOut copies per element, copy i of element value out_value(i) of step();
// in_row(p, i, row), out_row(p, i, row) with their strides between steps, for row = t*N + n; in_used(p, i, zoneout);
// aligned(p): those rows start on 16 bytes where H is a multiple of 4.
template <class Cell, int NB, int CTW>
__global__ __launch_bounds__(256, 1)
void split_backward_kernel(typename Cell::Params p) {
  constexpr int G = Cell::kGates;
  constexpr int HS = 16;
  constexpr int PIECE = 16 * NB;
  constexpr int PRODUCERS = 4 * CTW;
  constexpr int LOADS = NB == 8 ? CTW / 2 : CTW;  // a wavefront's share of the pieces, 1 KiB each
  constexpr int kInputs = Cell::kInputs, kSums = Cell::kSums;
  constexpr int OWNERS = NB * HS;
  constexpr int HELPERS = NB == 16 ? 256 : 256 - OWNERS;
  constexpr int ITEMS = NB * 4;  // groups of four units per plane of inputs or copies
  constexpr int IN_N = (kInputs * ITEMS + HELPERS - 1) / HELPERS;
  constexpr int OUT_N = (Cell::kOut * ITEMS + HELPERS - 1) / HELPERS;
  static_assert(NB == 8 || NB == 16, "rows of a split tile");
  static_assert(CTW % 2 == 0 && G <= 4 && kSums <= 2 * kInputs, "pairs of owners, operand, room for the column sums");
  extern __shared__ __attribute__((aligned(16))) float lds[];
  using Lds = SplitBackwardLds<Cell, NB>;
  Lds& s = *reinterpret_cast<Lds*>(lds);
  const Role role = take_role(p.ls, &s.large[0][0]);
  if (!role.active) return;

  const int H = p.H, N = p.N, T = p.T, gx = p.ls.gx;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int cw = role.cw, bt = role.bt;
  const int j0 = cw * HS;
  const int n0 = bt * NB;
  const int rows_here = (N - n0) < NB ? (N - n0) : NB;
  const int q = lane >> 4, c = lane & 15;

  GroupSync gs;
  group_sync_init(gs, p.ls, role);

  const int tile_bytes = gx * PRODUCERS * PIECE * 4;
  float* xp = Cell::pieces(p) + (size_t)bt * kSplitPieceTiles * (tile_bytes / 4);
  const TileBuffer xpb = make_tile_buffer(xp, kSplitPieceTiles * (tile_bytes / 4));

  // The wavefront's weights, split: lane 16*q + c holds column c of owner wave*CTW + i, k = 32*j + 8*q + e: unit
  // 8*j + 2*q + e/4 of the workgroup, gate e%4.
  float largest = 0.f;
  bf16x8_t w[2][CTW][3];
  {
    const __amdgpu_buffer_rsrc_t from =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p.R_t), 0, G * H * H * 4, 0x00020000);
    float f[2][CTW / 2][8];
    auto read = [&](float (&to)[CTW / 2][8], int step) {  // step: (k group, half of the owners)
#pragma unroll
      for (int e = 0; e < 8; ++e)
#pragma unroll
        for (int i = 0; i < CTW / 2; ++i) {
          const int owner = wave * CTW + (step & 1) * (CTW / 2) + i;
          const int unit = j0 + 8 * (step >> 1) + 2 * q + e / 4, gate = e % 4;
          // (elements that do not exist lie beyond the buffer and read as zero)
          const bool ok = gate < G && unit < H && owner * 16 + c < H;
          const int off = ok ? ((gate * H + unit) * H + owner * 16 + c) * 4 : 0x7ffffff0;
          to[i][e] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(from, off, 0, 0));
        }
      __builtin_amdgcn_sched_barrier(0);
    };
    read(f[0], 0);
#pragma unroll
    for (int step = 0; step < 4; ++step) {
      if (step < 3) read(f[(step + 1) & 1], step + 1);
#pragma unroll
      for (int i = 0; i < CTW / 2; ++i) {
        const float (&x)[8] = f[step & 1][i];
        uint4_t parts[3];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          largest = fmaxf(largest, fmaxf(fabsf(x[2 * e]), fabsf(x[2 * e + 1])));
          unsigned int hi, mid, lo;
          split_pair(x[2 * e] * kSplitScale, x[2 * e + 1] * kSplitScale, hi, mid, lo);
          parts[0][e] = hi;
          parts[1][e] = mid;
          parts[2][e] = lo;
        }
#pragma unroll
        for (int part = 0; part < 3; ++part) {
          bf16x8_t& to = w[step >> 1][(step & 1) * (CTW / 2) + i][part];
          to = __builtin_bit_cast(bf16x8_t, parts[part]);
          if (CTW > 4 && part > 0) asm volatile("" : "+a"(to));  // see split_forward_kernel
        }
      }
    }
  }
  const bool large_weights = __syncthreads_or(largest >= kSplitLimit) != 0;

  // Where the wavefront publishes.  8 rows: lanes 0..31 take the even owner of a pair, lanes 32..63 the odd one, a lane
  // four rows of a unit; 16 rows: a lane four rows of a unit of every owner.
  constexpr int PUBS = NB == 8 ? CTW / 2 : CTW;
  int pub_at[PUBS];
#pragma unroll
  for (int i = 0; i < PUBS; ++i) {
    const int owner = wave * CTW + (NB == 8 ? 2 * i + (q >> 1) : i);
    const int at = NB == 8 ? c * 8 + 4 * (q & 1) : c * 16 + 4 * q;
    pub_at[i] = owner < gx ? ((owner * PRODUCERS + cw) * PIECE + at) * 4 : 0x7ffffff0;
  }
  auto publish = [&](int parity, int i, const float4_t& v) {
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(uint4_t, v), xpb.rsrc, pub_at[i], parity * tile_bytes, 0);
  };
  // All pieces start out with the tag their first publication does not have; producers that do not exist hold zeros.
  {
    const float stale = __uint_as_float(1u ^ scatter_tag(0));
#pragma unroll
    for (int i = 0; i < PUBS; ++i)
      for (int b = 0; b < kSplitPieceTiles; ++b) publish(b, i, float4_t{stale, stale, stale, stale});
    for (int i = tid; i < (PRODUCERS - gx) * PIECE; i += 256)
      for (int b = 0; b < kSplitPieceTiles; ++b)
        xp[(size_t)b * (tile_bytes / 4) + ((size_t)cw * PRODUCERS + gx) * PIECE + i] = 0.f;
  }

  // Pointwise ownership: thread 16*r + u of the first NB*16 handles batch row n0 + r, hidden unit j0 + u.
  const bool owns = wave < OWNERS / 64;
  const int pr = tid / HS, pu = tid % HS;
  const bool act = owns && pr < rows_here && j0 + pu < H;
  const size_t row = act ? (size_t)(n0 + pr) : 0, unit = act ? (size_t)(j0 + pu) : 0;
  const bool zoneout = p.zoneout_mask != nullptr;
  Cell cell;
  cell.load_state(p, row * H + unit, act);
  float sums[kSums];
#pragma unroll
  for (int i = 0; i < kSums; ++i) sums[i] = 0.f;
  // The matrix instructions round their sums down, not to nearest: a bias of 2^-28 or so of a value that adds up in sums
  // over steps and rows (the bias gradients' error doubled).  Odd rows go in and come out with their signs changed.
  const float sign_scale = pr & 1 ? -kSplitScale : kSplitScale;
  const float4_t unscale = {kProductScale, -kProductScale, kProductScale, -kProductScale};
  // Where the element's operands go: parts of gates 0..3, side by side.
  int operand_at[3];
#pragma unroll
  for (int part = 0; part < 3; ++part) operand_at[part] = SplitTile<NB, 2>::byte_in_wave(4 * pu, part, pr < NB ? pr : 0);

  // What this thread moves (see split_forward_kernel).  Step d works on time step T-1-d.
  const int helper = tid - (256 - HELPERS);
  const bool helps = wave >= 4 - HELPERS / 64;
  const bool wide = H % 4 == 0 && Cell::aligned(p);
  const float* in_at[IN_N];
  float* out_at[OUT_N];
  float4_t moved[IN_N];
  bool in_ok[IN_N], out_ok[OUT_N];
  auto item_unit = [&](int i) { return j0 + 4 * (i & 3); };
#pragma unroll
  for (int n = 0; n < IN_N; ++n) {
    const int i = helper + HELPERS * n, plane = i / ITEMS, r = (i >> 2) % NB;
    in_ok[n] = helps && plane < kInputs && Cell::in_used(p, plane, zoneout) && r < rows_here && item_unit(i) < H;
    in_at[n] = in_ok[n] ? Cell::in_row(p, plane, (size_t)(T - 1) * N + n0 + r) + item_unit(i) : nullptr;
    moved[n] = float4_t{0.f, 0.f, 0.f, 0.f};
  }
#pragma unroll
  for (int n = 0; n < OUT_N; ++n) {
    const int i = helper + HELPERS * n, plane = i / ITEMS, r = (i >> 2) % NB;
    out_ok[n] = helps && plane < Cell::kOut && r < rows_here && item_unit(i) < H;
    out_at[n] = out_ok[n] ? Cell::out_row(p, plane, (size_t)(T - 1) * N + n0 + r) + item_unit(i) : nullptr;
  }
  auto request = [&] {
#pragma unroll
    for (int n = 0; n < IN_N; ++n)
      if (in_ok[n]) {
        const int i = helper + HELPERS * n;
        if (wide) {
          moved[n] = *reinterpret_cast<const float4_t*>(in_at[n]);
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (item_unit(i) + e < H) moved[n][e] = in_at[n][e];
        }
        in_at[n] -= Cell::in_stride(p, i / ITEMS);
      }
  };
  auto park_inputs = [&](int d) {
#pragma unroll
    for (int n = 0; n < IN_N; ++n)
      if (in_ok[n]) {
        const int i = helper + HELPERS * n;
        *reinterpret_cast<float4_t*>(&s.in[d & 1][i / ITEMS][(i >> 2) % NB][4 * (i & 3)]) = moved[n];
      }
  };
  auto write_copies = [&](int d) {
#pragma unroll
    for (int n = 0; n < OUT_N; ++n)
      if (out_ok[n]) {
        const int i = helper + HELPERS * n, plane = i / ITEMS, r = (i >> 2) % NB;
        const float4_t v = *reinterpret_cast<const float4_t*>(&s.out[d & 1][Cell::out_value(plane)][r][4 * (i & 3)]);
        if (wide) {
          *reinterpret_cast<float4_t*>(out_at[n]) = v;
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (item_unit(i) + e < H) out_at[n][e] = v[e];
        }
        out_at[n] -= Cell::out_stride(p, plane);
      }
  };
  auto prepare = [&](int d) {
    float sv[kInputs];
#pragma unroll
    for (int i = 0; i < kInputs; ++i) sv[i] = s.in[d & 1][i][pr][pu];
    cell.prepare(sv);
  };

  // The pieces of this wavefront's producers.
  float4_t piece[LOADS];
  unsigned int real[LOADS];
#pragma unroll
  for (int f = 0; f < LOADS; ++f) real[f] = wave * CTW + (NB == 8 ? 2 * f + (lane >> 5) : f) < gx ? 1u : 0u;
  const int gather_at = (cw * PRODUCERS + wave * CTW) * PIECE * 4 + lane * 16;
  auto request_pieces = [&](int d) {
    constexpr int kAgentScope = 16;  // the sc1 bit of the cache policy
#pragma unroll
    for (int f = 0; f < LOADS; ++f)
      piece[f] = __builtin_bit_cast(float4_t, __builtin_amdgcn_raw_buffer_load_b128(
                                                  xpb.rsrc, gather_at + f * 1024, (d & 1) * tile_bytes, kAgentScope));
  };
  auto gather = [&](int d) {
    const unsigned int tag = scatter_tag(d);
    poll_until_written(gs, [&] { request_pieces(d); }, [&] {
      unsigned int m = 0u;
#pragma unroll
      for (int f = 0; f < LOADS; ++f) {
        const uint4_t b = __builtin_bit_cast(uint4_t, piece[f]);
        m |= ((b.x ^ tag) | (b.y ^ tag) | (b.z ^ tag) | (b.w ^ tag)) & real[f];
      }
      return __all(m == 0u) != 0;
    });
    auto total = [&] {
      float4_t v = piece[0];
#pragma unroll
      for (int f = 1; f < LOADS; ++f) v += piece[f];
      return v;
    };
    float4_t v = total();
    // An infinite partial sum tagged 1 reads as a signalling NaN, which arithmetic does not make.
    const bool nan = v.x != v.x || v.y != v.y || v.z != v.z || v.w != v.w;
    if (__any(nan)) {
#pragma unroll
      for (int f = 0; f < LOADS; ++f)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const unsigned int b = __float_as_uint(piece[f][e]);
          piece[f][e] = (b & 0x7fffffffu) == 0x7f800001u ? __uint_as_float(b & ~1u) : piece[f][e];
        }
      v = total();
    }
    if constexpr (NB == 8) {
      // lanes 0..31 and 32..63 hold different producers' sums of the same elements; each half ends up with two rows
      const float2_t two = {swap_add32(v.x, v.z), swap_add32(v.y, v.w)};
      *reinterpret_cast<float2_t*>(&s.part[wave][(lane & 31) >> 1][4 * (lane & 1) + 2 * (lane >> 5)]) = two;
    } else {
      *reinterpret_cast<float4_t*>(&s.part[wave][lane >> 2][4 * (lane & 3)]) = v;
    }
  };
  auto gathered = [&] {
    return (s.part[0][pu][pr] + s.part[1][pu][pr]) + (s.part[2][pu][pr] + s.part[3][pu][pr]);
  };

  request();
  park_inputs(0);
  if (T > 1) request();
  group_arrive(gs);
  group_wait(gs);
  if (owns) prepare(0);

  for (int d = 0; d < T; ++d) {
    if (d > 0) gather(d - 1);
    // (The loads of cold memory are issued where the wavefront's next polls are far.)
    if (NB == 16 && d > 0 && d + 1 < T) request();
    __syncthreads();
    if (owns) {
      if (d > 0) cell.add_gathered(gathered());
      const float4_t dv = cell.step(act, zoneout, sums);
      float biggest = 0.f;
      unsigned int p01[3], p23[3];
      const float4_t v = dv * sign_scale;
      split_pair(v.x, v.y, p01[0], p01[1], p01[2]);
      split_pair(v.z, G > 3 ? v.w : 0.f, p23[0], p23[1], p23[2]);
#pragma unroll
      for (int part = 0; part < 3; ++part)
        *reinterpret_cast<uint2*>(reinterpret_cast<char*>(s.operand) + operand_at[part]) = make_uint2(p01[part], p23[part]);
#pragma unroll
      for (int g = 0; g < 4; ++g) s.out[d & 1][g][pr][pu] = dv[g];
#pragma unroll
      for (int g = 0; g < G; ++g) biggest = fmaxf(biggest, fabsf(dv[g]));
      const unsigned int any = __any(biggest >= kSplitLimit) ? 1u : 0u;
      if (lane == 0) s.large[d & 1][wave] = any;
    } else if (NB == 8 && helps) {
      if (d + 1 < T) park_inputs(d + 1);
      if (d + 2 < T) request();
    }
    __syncthreads();

    const unsigned int tag = scatter_tag(d);
    constexpr int OPERANDS = NB == 8 ? 3 : 6;
    uint4_t a[OPERANDS];
#pragma unroll
    for (int f = OPERANDS - 1; f >= 0; --f) a[f] = s.operand[f][lane];
    unsigned int any = large_weights ? 1u : 0u;
#pragma unroll
    for (int i = 0; i < OWNERS / 64; ++i) any |= s.large[d & 1][i];
    __builtin_amdgcn_sched_barrier(0);
    if (__builtin_amdgcn_readfirstlane(any) == 0u) {
      if constexpr (NB == 8) {
        uint4_t third[2];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          third[0][e] = (lane & 8) == 0 ? a[2][e] : 0u;
          third[1][e] = (lane & 8) != 0 ? a[2][e] : 0u;
        }
#pragma unroll
        for (int i = 0; i < CTW; i += 2) {
          float4_t acc[2] = {float4_t{0.f, 0.f, 0.f, 0.f}, float4_t{0.f, 0.f, 0.f, 0.f}};
          auto mfma = [&](const uint4_t& x, int j, int part) {
#pragma unroll
            for (int h = 0; h < 2; ++h)
              acc[h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, x), w[j][i + h][part], acc[h], 0, 0, 0);
          };
          mfma(third[0], 0, 0);
          mfma(third[1], 1, 0);
          mfma(a[0], 0, 2);
          mfma(a[1], 1, 2);
          mfma(a[0], 0, 1);
          mfma(a[1], 1, 1);
          mfma(a[0], 0, 0);
          mfma(a[1], 1, 0);
          float4_t v;
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = swap_add32(acc[0][e], acc[1][e]);
          publish(d & 1, i / 2, tagged4(v * unscale, tag));
        }
      } else {
#pragma unroll
        for (int i = 0; i < CTW; i += 2) {
          float4_t acc[2] = {float4_t{0.f, 0.f, 0.f, 0.f}, float4_t{0.f, 0.f, 0.f, 0.f}};
          constexpr int pa[6] = {2, 1, 0, 1, 0, 0}, pb[6] = {0, 1, 2, 0, 1, 0};
#pragma unroll
          for (int m = 0; m < 6; ++m)
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
              for (int h = 0; h < 2; ++h)
                acc[h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a[3 * j + pa[m]]),
                                                                 w[j][i + h][pb[m]], acc[h], 0, 0, 0);
#pragma unroll
          for (int h = 0; h < 2; ++h) publish(d & 1, i + h, tagged4(acc[h] * unscale, tag));
        }
      }
    } else {
      // Something does not split: the same sums in fp32.
      for (int i = 0; i < PUBS; ++i) {
        const int owner = wave * CTW + (NB == 8 ? 2 * i + (q >> 1) : i), col = owner * 16 + c;
        const int r = 4 * (NB == 8 ? q & 1 : q);
        float4_t v = {0.f, 0.f, 0.f, 0.f};
        for (int k = 0; k < 16 * G; ++k) {
          const int u = k % 16, g = k / 16;
          const bool ok = j0 + u < H && col < H;
          const float weight = ok ? p.R_t[((size_t)g * H + j0 + u) * H + col] : 0.f;
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = fmaf(ok ? s.out[d & 1][g][r + e][u] : 0.f, weight, v[e]);
        }
        int at = 0x7ffffff0;
#pragma unroll
        for (int n = 0; n < PUBS; ++n) at = n == i ? pub_at[n] : at;
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(uint4_t, tagged4(v, tag)), xpb.rsrc, at,
                                               (d & 1) * tile_bytes, 0);
      }
    }
    // What does not depend on the pieces, while they are on their way.  (They are requested afterwards: a request that
    // comes too early has to be made again, 700 cycles later at 16 rows.)
    if (d + 1 < T) {
      if (NB == 16) {
        park_inputs(d + 1);
        __syncthreads();
      }
      if (owns) prepare(d + 1);
    }
    if (helps) write_copies(d);
    request_pieces(d);
  }
  gather(T - 1);
  __syncthreads();
  if (owns) {
    cell.add_gathered(gathered());
    if (act) cell.store_state(p, (size_t)(n0 + pr) * H + j0 + pu);
  }

  // Column sums (bias gradients): the tile's rows in order, parked per tile; the last workgroup of the column block to
  // finish adds the tiles in order.
  float (*red)[NB][16] = reinterpret_cast<float (*)[NB][16]>(&s.in[0][0][0][0]);
  if (owns) {
#pragma unroll
    for (int i = 0; i < kSums; ++i) red[i][pr][pu] = act ? sums[i] : 0.f;
  }
  __syncthreads();
  const int sum = tid / HS, su = tid % HS;
  if (sum < kSums && j0 + su < H) {
    float total = 0.f;
    for (int r = 0; r < NB; ++r) total += red[sum][r][su];
    store_agent(&p.db_partial[(size_t)bt * kSums * H + (size_t)sum * H + j0 + su], total);
  }
  if (column_last_arrival(p.ls.cb, cw, (unsigned)p.ls.gy, &s.large[0][0])) {
    if (sum < kSums && j0 + su < H) {
      const int col = sum * H + j0 + su;
      Cell::add_sums(p, col, sum_over_tiles(p.db_partial + col, (size_t)kSums * H, p.ls.gy));
    }
  }
}

// The owners a wavefront's columns cover.
inline int split_backward_columns(int H) { return H <= 256 ? 4 : (H <= 384 ? 6 : 8); }

// The rows of a batch tile where a backward recurrence takes this kernel (0: it does not) and the floats it needs of
// scratch, column sums (`sums` per unit) first.  With few hidden units a step is the chain alone, and the other kernels'
// is shorter.  Measured, C = 64, T = 100, whole training passes, the others -> this one, us:
//   LSTM N = 64  H = 64 325 -> 344  H = 128 360 -> 369  H = 256 424 -> 403  H = 320 520 -> 478  H = 512 633 -> 587
//        N = 128 H = 64 404 -> 423  H = 128 537 -> 465  H = 256 607 -> 562  H = 384 884 -> 690  H = 512 997 -> 860
//   GRU  N = 64  H = 128 342 -> 350  H = 256 399 -> 391  H = 512 566 -> 539
//        N = 128 H = 64 408 -> 406  H = 128 515 -> 441  H = 256 729 -> 525  H = 512 1027 -> 839
inline int split_backward_rule(hipStream_t stream, int N, int H, int sums, int* rows, size_t* sum_floats, size_t* floats) {
  *rows = 0;
  const int gx = (H + 15) / 16;
  int nb = 0;
  for (int rows_of_tile : {16, 8})
    if (xcd_local_fits(gx, (N + rows_of_tile - 1) / rows_of_tile)) nb = rows_of_tile;
  if (nb == 0 || N <= 32 || H > 512 || H <= (nb == 16 ? 64 : 128)) return HASTE_HIP_OK;
  const int gy = (N + nb - 1) / nb;
  *sum_floats = ((size_t)gy * sums * H + 3) / 4 * 4;
  *floats = *sum_floats + (size_t)gy * kSplitPieceTiles * split_piece_floats(gx, split_backward_columns(H), nb);
  bool room = false;
  HASTE_HIP_PROPAGATE(workspace_has_room(stream, *floats * sizeof(float), &room));
  if (room) *rows = nb;
  return HASTE_HIP_OK;
}

// Launches the kernel for the rows split_backward_rule() gives.
template <class Cell, int NB>
int launch_split_backward_rows(const char* name, hipStream_t stream, const Workspace& ws, typename Cell::Params& p) {
  const int gx = (p.H + 15) / 16, ctw = split_backward_columns(p.H);
  LaunchPlan plan;
  HASTE_HIP_PROPAGATE(plan_launch(stream, ws, gx, (p.N + NB - 1) / NB, NB, sizeof(SplitBackwardLds<Cell, NB>),
                                  (unsigned)p.T + 1, &plan));
  p.ls = plan.shape;
  plan.kernel = kPlanSplit;
  if (ctw == 4) return launch_persistent(name, split_backward_kernel<Cell, NB, 4>, plan, p, stream);
  if (ctw == 6) return launch_persistent(name, split_backward_kernel<Cell, NB, 6>, plan, p, stream);
  return launch_persistent(name, split_backward_kernel<Cell, NB, 8>, plan, p, stream);
}
template <class Cell>
int launch_split_backward(const char* name, hipStream_t stream, const Workspace& ws, int nb, typename Cell::Params& p) {
  if (nb == 8) return launch_split_backward_rows<Cell, 8>(name, stream, ws, p);
  return launch_split_backward_rows<Cell, 16>(name, stream, ws, p);
}

}  // namespace haste_hip
