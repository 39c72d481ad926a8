// Operands of the bf16 matrix instructions made of floats' three parts: their layout for batch tiles of 4, 8 and 16 rows.
#pragma once

#include "recurrent.h"
#include "split_bf16.h"

namespace haste_hip {

// ---- exchange tiles of split h -------------------------------------------------------------
// h is published as its three bfloat16 parts, laid out as the A operands of v_mfma_f32_16x16x32_bf16: lane
// 16*q + i of a wavefront holds row i, k = 8*q .. 8*q+7 of a group of 32 hidden units.  The operand has 16 rows
// whatever the batch tile; short tiles put the PARTS of their rows there, so that one instruction multiplies
// several of them with the same part of R:
//   16 rows: one operand per part; R's three parts take 3 + 2 + 1 = 6 instructions per 32 k and 16 columns
//    8 rows: parts 1 and 2 of the 8 rows in one operand (3 instructions, one for each part of R), part 3 of two
//            groups of k in another (1 instruction per group; the other group's rows are masked): 4
//    4 rows: parts 1, 2 and 3 in one operand (the last 4 rows are zero): 3
// Wavefront w contracts over the groups w*KST .. w*KST+KST-1 and reads its operands, kFrags contiguous KiB,
// straight from the tile: its loads are the wait, as with the polled tiles of floats in recurrent.h (four
// tiles rotate, elements not yet published are all ones; two parts share a 32-bit word and neither is ever 0xffff).
template <int NB, int KST>
struct SplitTile {
  static_assert(NB == 4 || NB == 8 || NB == 16, "rows of a split tile");
  static constexpr int kFrags = NB == 4 ? KST : (NB == 8 ? KST + (KST + 1) / 2 : 3 * KST);
  static constexpr int kBytes = 4 * kFrags * 1024;

  // Where part `part` of (unit k, row) lies; four consecutive k from a multiple of 4 on are contiguous.
  __device__ __forceinline__ static int byte(int k, int part, int row) {
    return k / (32 * KST) * kFrags * 1024 + byte_in_wave(k % (32 * KST), part, row);
  }
  // The same within a wavefront's operands (k < 32 * KST).
  __device__ __forceinline__ static int byte_in_wave(int k, int part, int row) {
    const int j = k >> 5;
    int frag = 0, row16;
    if (NB == 16) {
      frag += 3 * j + part;
      row16 = row;
    } else if (NB == 8) {
      frag += part < 2 ? j : KST + (j >> 1);
      row16 = (part < 2 ? part : (j & 1)) * 8 + row;
    } else {
      frag += j;
      row16 = part * 4 + row;
    }
    return frag * 1024 + (((k >> 3) & 3) * 16 + row16) * 16 + (k & 7) * 2;
  }

  // The unit whose owner sets up 16-byte chunk `chunk` of the tile (units beyond H: the last workgroup).
  __device__ __forceinline__ static int chunk_unit(int chunk) {
    const int frag = chunk >> 6, w = frag / kFrags, f = frag % kFrags;
    const int q = (chunk >> 4) & 3, row16 = chunk & 15;
    int j = NB == 16 ? f / 3 : f;
    if (NB == 8 && f >= KST) j = 2 * (f - KST) + (row16 >> 3);
    return j < KST ? (w * KST + j) * 32 + 8 * q : 128 * KST;
  }
};

// Floats beyond this (infinities too) would overflow as scaled parts: a launch that meets one in R or in the
// initial h (nothing later is larger: the cells' states after a step are bounded by 1 or by the state before)
// computes with floats, element by element.  NaNs need no such care, they come out of either as NaN.
constexpr float kSplitLimit = 0x1p35f;

}  // namespace haste_hip
