// fp32 GEMM for gfx950: C[M,N] = op(A)[M,K] * B[K,N] (+ C).
//
// Replaces the cuBLAS sgemm calls of the reference (lib/blas.h:48-61): the
// time-fused input projection x*W (lib/lstm_forward_gpu.cu.cc:340-348) and the
// three batched backward products dW, dR, dx (lib/lstm_backward_gpu.cu.cc:374-402).
//
// The product runs on the bf16 matrix cores, which multiply 16 times as fast as the fp32 ones,
// without giving up precision: every float is the exact sum of three bfloat16 (8 + 8 + 8 bits
// of significand), the products of those are exact in fp32, and of the nine the six that can
// reach a float's 24 bits are accumulated in fp32 (Henry, Tang and Heinecke, "Leveraging the
// bfloat16 artificial intelligence datatype for higher-precision computations", 2019).  The
// three left out are below 2^-24 of the largest.  The five small products have an accumulator
// of their own, so that the large one is rounded once per 16 k where the fp32 instruction
// (32x32x2) rounds eight times.  Measured against float64, normal operands: 0.3 - 0.4 of the
// fp32 instruction's error (2-norm, K = 75 .. 160000).  Operands are scaled by a power of two, so
// that the parts of the smallest floats are bfloat16 too; a tile in which that does not work --
// infinities, NaNs, operands from 2^104 or results from 2^80 on -- is computed again with the fp32
// instruction.
//
// Design: 128x128 output tile per 256-thread workgroup (4 wavefronts, each a 64x64 quadrant =
// 2x2 v_mfma_f32_32x32x16_bf16 tiles), K consumed 32 at a time.  A stage is read as float,
// split in registers and put into LDS as three planes of [k / 8][row][k % 8]: an operand of
// the instruction is then one 16-byte LDS read per lane at consecutive addresses.  Operands
// whose rows run along the output (B, and A stored transposed) are read 8 k deep per thread,
// so that putting 8 k side by side is a choice of registers.  Two workgroups share a CU and one
// splits while the other multiplies; the multiplying one has the higher wave priority (3-8 %).
// What bounds it: the SIMDs' instructions.  At 8192^3 the bf16 matrix cores execute for 66 % of the time and the
// other vector instructions, nearly all of them the splitting's 6.5 per element, take 38 % of a SIMD's cycles; the two
// hardly overlap (counters).  A bare loop of these MFMAs on random data reaches 1700 TFLOP/s = 283 of fp32 product,
// 1430 with the splitting's share of vector instructions beside them.  Measured, fp32 instruction before -> now:
// 8192^3 140 -> 193 TFLOP/s; 6400 x 2048 x 512 110 -> 155; 6400 x 512 x 2048 113 -> 153;
// 512 x 2048 x 6400 119 -> 166 (with the kernel that adds the K pieces).  Before operands were scaled (see kSplitScale)
// 8192^3 ran at 199; against that:
// One accumulator instead of two leaves registers for three workgroups per CU: 213 TFLOP/s at
// 8192^3 and 0-5 % on the other shapes, with 2.5 times the error.  256x128 tiles (8 wavefronts, two LDS
// stages) 195; 16x16x32 instructions 197 with one accumulator.
//
// Work distribution: whole tiles for as long as they fill rounds of two per CU; the tiles of
// the last, partial round (all tiles, when there are few: dW, dR with K = T*N) are cut along K
// into pieces so that the pieces again fill the chip evenly.  Pieces park partial tiles; a
// second, bandwidth-bound kernel adds the pieces of a tile in index order, so results do not
// depend on scheduling.  Whole tiles are numbered so that each XCD (one L2) works on a
// contiguous run of them; the pieces follow, dealt round-robin over the XCDs.
#include "common.h"
#include "split_bf16.h"

namespace haste_hip {
namespace {

typedef float float4_t __attribute__((ext_vector_type(4)));
typedef float float16_t __attribute__((ext_vector_type(16)));

constexpr int BN = 128;
constexpr int BK = 16;
constexpr int LDB = BN + 4;
constexpr int B_STAGE = BK * LDB;
constexpr int kXcds = 8;

// Operand panels are read through buffer resources: a 16-byte load at any 4-byte aligned
// offset, elements beyond the resource's range read as zero and never fault.  That keeps the
// K loops free of branches (the compiler can then overlap the loads of the next step with the
// MFMAs of this one).
typedef unsigned int uint4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_panel(const float* base, long long floats) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(base), 0, (int)(floats * 4), 0x00020000);
}

// The load is issued here; `valid` (how many of the four elements belong to the problem) is
// applied by masked4() when the data is used, so that nothing waits for the load in between.
__device__ __forceinline__ uint4_t load4_raw(__amdgpu_buffer_rsrc_t panel, long long float_offset,
                                             int valid) {
  const unsigned int off = valid > 0 ? (unsigned int)(float_offset * 4) : 0x7ffffff0u;
  return __builtin_amdgcn_raw_buffer_load_b128(panel, off, 0, 0);
}

__device__ __forceinline__ float4_t masked4(uint4_t u, int valid) {
  float4_t v;
  v.x = valid > 0 ? __uint_as_float(u.x) : 0.f;
  v.y = valid > 1 ? __uint_as_float(u.y) : 0.f;
  v.z = valid > 2 ? __uint_as_float(u.z) : 0.f;
  v.w = valid > 3 ? __uint_as_float(u.w) : 0.f;
  return v;
}

// One BM x 128 output tile over the K range [k_begin, k_end) with the fp32 instruction: what
// split_tile() falls back on when its operands do not split.  Arguments as there; `smem`:
// 2 * (BK * (BM + 4) + B_STAGE) floats.
template <bool TRANS_A, int BM>
__device__ __forceinline__ void float_tile(int M, int N, int K,
                                          const float* __restrict__ A, int lda,
                                          const float* __restrict__ B, int ldb,
                                          float* __restrict__ C, int ldc, int accumulate,
                                          int tm, int tn, int k_begin, int k_end,
                                          float* __restrict__ part, float* smem) {
  // A tile k-major in LDS: leading dimension BM+2 when it is written with transposing
  // scalar stores (bank-conflict free), BM+4 when written with 16-byte stores.
  constexpr int LDA = TRANS_A ? BM + 4 : BM + 2;
  constexpr int A_STAGE = BK * (BM + 4);
  constexpr int MI = BM / 64;       // 32x32 MFMA tiles per wavefront along M
  constexpr int A_PASSES = BM / 64; // passes of 256 threads to load the A tile
  float* As = smem;
  float* Bs = smem + 2 * A_STAGE;
  const int m0 = tm * BM, n0 = tn * BN;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int wm = (wave >> 1) * (32 * MI);
  const int wn = (wave & 1) * 64;

  float16_t acc[MI][2];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

  uint4_t a_raw[A_PASSES], b_raw[2];
  int a_valid[A_PASSES], b_valid[2];
  // A tile stored [K][M] in memory: one pass covers (256*4/BM) k-rows of BM columns.
  constexpr int TA_ROWS = 1024 / BM;
  constexpr int TA_COLS = BM / 4;

  // This workgroup's operand panels: its BM rows (TRANS_A: columns) of A and its 128 columns
  // of B, all of K.  Offsets below are in floats from the panel's first element.
  const int rows_here = (M - m0) < BM ? (M - m0) : BM;
  const int cols_here = (N - n0) < BN ? (N - n0) : BN;
  const __amdgpu_buffer_rsrc_t a_panel =
      TRANS_A ? make_panel(A + m0, (long long)(K - 1) * lda + rows_here)
              : make_panel(A + (size_t)m0 * lda, (long long)(rows_here - 1) * lda + K);
  const __amdgpu_buffer_rsrc_t b_panel = make_panel(B + n0, (long long)(K - 1) * ldb + cols_here);

  auto load_global = [&](int kk) {
#pragma unroll
    for (int i = 0; i < A_PASSES; ++i) {
      if (TRANS_A) {
        const int ak = (tid / TA_COLS) + TA_ROWS * i;
        const int am = (tid % TA_COLS) * 4;
        const int k = kk + ak;
        a_valid[i] = (k < k_end) ? (rows_here - am) : 0;
        a_raw[i] = load4_raw(a_panel, (long long)k * lda + am, a_valid[i]);
      } else {
        const int arow = (tid >> 2) + 64 * i;
        const int ak = (tid & 3) * 4;
        const int k = kk + ak;
        a_valid[i] = (arow < rows_here) ? (k_end - k) : 0;
        a_raw[i] = load4_raw(a_panel, (long long)arow * lda + k, a_valid[i]);
      }
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int bk = (tid >> 5) + 8 * i;
      const int bn = (tid & 31) * 4;
      const int k = kk + bk;
      b_valid[i] = (k < k_end) ? (cols_here - bn) : 0;
      b_raw[i] = load4_raw(b_panel, (long long)k * ldb + bn, b_valid[i]);
    }
  };

  auto store_lds = [&](int buf) {
    float* as = As + buf * A_STAGE;
    float* bs = Bs + buf * B_STAGE;
#pragma unroll
    for (int i = 0; i < A_PASSES; ++i) {
      const float4_t a = masked4(a_raw[i], a_valid[i]);
      if (TRANS_A) {
        const int ak = (tid / TA_COLS) + TA_ROWS * i;
        const int am = (tid % TA_COLS) * 4;
        *reinterpret_cast<float4_t*>(as + ak * LDA + am) = a;
      } else {
        const int arow = (tid >> 2) + 64 * i;
        const int ak = (tid & 3) * 4;
        as[(ak + 0) * LDA + arow] = a.x;
        as[(ak + 1) * LDA + arow] = a.y;
        as[(ak + 2) * LDA + arow] = a.z;
        as[(ak + 3) * LDA + arow] = a.w;
      }
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int bk = (tid >> 5) + 8 * i;
      const int bn = (tid & 31) * 4;
      *reinterpret_cast<float4_t*>(bs + bk * LDB + bn) = masked4(b_raw[i], b_valid[i]);
    }
  };

  auto compute = [&](int buf) {
    const float* as = As + buf * A_STAGE + (lane >> 5) * LDA + wm + (lane & 31);
    const float* bs = Bs + buf * B_STAGE + (lane >> 5) * LDB + wn + (lane & 31);
    // The LDS reads of K pair k2+2 are issued before the MFMAs of pair k2.
    float b_nxt[2], a_nxt[MI];
    b_nxt[0] = bs[0];
    b_nxt[1] = bs[32];
#pragma unroll
    for (int i = 0; i < MI; ++i) a_nxt[i] = as[32 * i];
#pragma unroll
    for (int k2 = 0; k2 < BK; k2 += 2) {
      const float b0 = b_nxt[0], b1 = b_nxt[1];
      float av[MI];
#pragma unroll
      for (int i = 0; i < MI; ++i) av[i] = a_nxt[i];
      if (k2 + 2 < BK) {
        b_nxt[0] = bs[(k2 + 2) * LDB];
        b_nxt[1] = bs[(k2 + 2) * LDB + 32];
#pragma unroll
        for (int i = 0; i < MI; ++i) a_nxt[i] = as[(k2 + 2) * LDA + 32 * i];
        // keep the reads here: the scheduler would otherwise sink them to just before their use
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int i = 0; i < MI; ++i) {
        acc[i][0] = __builtin_amdgcn_mfma_f32_32x32x2f32(av[i], b0, acc[i][0], 0, 0, 0);
        acc[i][1] = __builtin_amdgcn_mfma_f32_32x32x2f32(av[i], b1, acc[i][1], 0, 0, 0);
      }
    }
  };

  if (k_begin < k_end) {
    load_global(k_begin);
    store_lds(0);
    __syncthreads();
    int buf = 0;
    for (int kk = k_begin; kk < k_end; kk += BK) {
      const bool more = kk + BK < k_end;
      if (more) load_global(kk + BK);
      compute(buf);
      if (more) store_lds(buf ^ 1);
      __syncthreads();
      buf ^= 1;
    }
  }

  // Output element (row, col) of accumulator register e in a 32x32 tile:
  // col = lane % 32, row = 8*(e/4) + 4*(lane/32) + e%4.
  const int col_in = lane & 31;
  const int row_in = (lane >> 5) * 4;
  if (part == nullptr) {
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int col = n0 + wn + 32 * j + col_in;
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int row = m0 + wm + 32 * i + 8 * (e >> 2) + row_in + (e & 3);
          if (row < M && col < N) {
            float* p = C + (size_t)row * ldc + col;
            *p = accumulate ? (*p + acc[i][j][e]) : acc[i][j][e];
          }
        }
      }
    return;
  }

  // A K piece: park the whole [BM][BN] partial tile (rows and columns beyond the problem
  // hold zeros); a second, bandwidth-bound kernel adds a tile's pieces in order (the kernel
  // boundary makes them visible, so no cache-wide fence is needed here).
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int col = wn + 32 * j + col_in;
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int row = wm + 32 * i + 8 * (e >> 2) + row_in + (e & 3);
        part[row * BN + col] = acc[i][j][e];
      }
    }
}


// ---- the product on the bf16 matrix cores ------------------------------------------------
constexpr int SK = 32;  // k of one LDS stage
// Bytes of one group of 8 k of `rows` rows in one plane (the padding puts the groups that a
// wavefront writes side by side on different banks), and of an operand's three planes.
constexpr int split_group_bytes(int rows) { return rows * 16 + 64; }
constexpr int split_operand_bytes(int rows) { return 3 * (SK / 8) * split_group_bytes(rows); }

// The scaling (split_bf16.h) is one vector instruction more per element: 8192^3 5.42 -> 5.55 ms, 6400 x 512 x 2048
// 85.6 -> 87.5 us.
// Eight consecutive k of one row, scaled, split into three bf16 each and stored into the three planes.
__device__ __forceinline__ void split_store(const float (&f)[8], char* at, int plane_bytes) {
  uint4_t p[3];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    unsigned int hi, mid, lo;
    split_pair(f[2 * j] * kSplitScale, f[2 * j + 1] * kSplitScale, hi, mid, lo);
    p[0][j] = hi;
    p[1][j] = mid;
    p[2][j] = lo;
  }
#pragma unroll
  for (int q = 0; q < 3; ++q) *reinterpret_cast<uint4_t*>(at + q * plane_bytes) = p[q];
}

// One BM x 128 output tile, BM = 64 * MI, over the K range [k_begin, k_end): MI = 2 (each
// wavefront a 64x64 quadrant) or 1 (each a 32x64 quadrant) for outputs of at most 64 rows.
// k_begin is a multiple of SK, k_end too unless it is K.  part == null: the tile goes to C
// (+= when accumulate); otherwise the whole [BM][BN] partial tile is parked at `part` (columns
// and rows beyond the problem hold nothing of use).
// `smem`: split_operand_bytes(BM) + split_operand_bytes(BN) bytes.
template <bool TRANS_A, int MI>
__device__ __forceinline__ void split_tile(int M, int N, int K, const float* __restrict__ A, int lda,
                                           const float* __restrict__ B, int ldb, float* __restrict__ C,
                                           int ldc, int accumulate, int tm, int tn, int k_begin, int k_end,
                                           float* __restrict__ part, char* smem) {
  constexpr int BM = 64 * MI;
  constexpr int WM = 32 * MI;
  constexpr int A_GROUP = split_group_bytes(BM), B_GROUP = split_group_bytes(BN);
  constexpr int A_PLANE = (SK / 8) * A_GROUP, B_PLANE = (SK / 8) * B_GROUP;
  char* As = smem;
  char* Bs = smem + split_operand_bytes(BM);
  const int m0 = tm * BM, n0 = tn * BN;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wr = wave >> 1, wc = wave & 1;

  const int rows_here = (M - m0) < BM ? (M - m0) : BM;
  const int cols_here = (N - n0) < BN ? (N - n0) : BN;
  const __amdgpu_buffer_rsrc_t a_panel =
      TRANS_A ? make_panel(A + m0, (long long)(K - 1) * lda + rows_here)
              : make_panel(A + (size_t)m0 * lda, (long long)(rows_here - 1) * lda + K);
  const __amdgpu_buffer_rsrc_t b_panel = make_panel(B + n0, (long long)(K - 1) * ldb + cols_here);

  float16_t acc[MI][2], low[MI][2];  // the products of the first parts; the five smaller ones
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = low[i][j][e] = 0.f;

  // A thread's share of a stage: 8 consecutive k of MI rows of A and 2 columns of B.  Rows, columns
  // and k beyond the problem read as zero or as what lies there, which reaches only outputs
  // that nobody keeps -- except k beyond the end of a row of A, masked in store_lds().
  // Where the rows run along the output, a wavefront takes 8 k of all of them, a lane MI (2)
  // neighbours, and neighbour i goes to MFMA tile i: writes to LDS stay consecutive, and a lane
  // ends up with two neighbouring columns of C.
  float a_raw[MI][8], b_raw[2][8];
  // Where row k of a panel starts; rows from K on are beyond every panel (with few of them and a long
  // stride their own offset need not be: it wraps at 2^32).  Scalar arithmetic: a wavefront's k are its own.
  const int wave_k = 8 * __builtin_amdgcn_readfirstlane(wave);
  auto row_at = [&](int k, int ld) { return k < K ? (unsigned)k * (unsigned)ld * 4u : 0x80000000u; };
  auto load_global = [&](int kk) {
    if constexpr (TRANS_A) {
#pragma unroll
      for (int r = 0; r < 8; ++r) {
        const unsigned int off = row_at(kk + wave_k + r, lda) + (unsigned)(lane * MI) * 4u;
        if constexpr (MI == 2) {
          const auto u = __builtin_amdgcn_raw_buffer_load_b64(a_panel, off, 0, 0);
          a_raw[0][r] = __uint_as_float(u[0]);
          a_raw[1][r] = __uint_as_float(u[1]);
        } else {
          a_raw[0][r] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(a_panel, off, 0, 0));
        }
      }
    } else {
      const unsigned int base = ((unsigned)(tid >> 2) * (unsigned)lda + (unsigned)(kk + 8 * (tid & 3))) * 4u;
#pragma unroll
      for (int i = 0; i < MI; ++i) {
        const unsigned int off = base + (unsigned)(64 * i * lda) * 4u;
        const uint4_t u = __builtin_amdgcn_raw_buffer_load_b128(a_panel, off, 0, 0);
        const uint4_t w = __builtin_amdgcn_raw_buffer_load_b128(a_panel, off + 16u, 0, 0);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          a_raw[i][e] = __uint_as_float(u[e]);
          a_raw[i][4 + e] = __uint_as_float(w[e]);
        }
      }
    }
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      const auto u = __builtin_amdgcn_raw_buffer_load_b64(b_panel, row_at(kk + wave_k + r, ldb) + (unsigned)(lane * 2) * 4u, 0, 0);
      b_raw[0][r] = __uint_as_float(u[0]);
      b_raw[1][r] = __uint_as_float(u[1]);
    }
  };

  auto store_lds = [&](int kk) {
    if constexpr (TRANS_A) {
#pragma unroll
      for (int i = 0; i < MI; ++i)
        split_store(a_raw[i], As + wave * A_GROUP + ((lane >> 5) * WM + 32 * i + (lane & 31)) * 16, A_PLANE);
    } else {
      if (kk + SK > k_end) {  // the last stage of a ragged K: what follows a row is another row
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
          for (int e = 0; e < 8; ++e) a_raw[i][e] = kk + 8 * (tid & 3) + e < k_end ? a_raw[i][e] : 0.f;
      }
#pragma unroll
      for (int i = 0; i < MI; ++i)
        split_store(a_raw[i], As + (tid & 3) * A_GROUP + ((tid >> 2) + 64 * i) * 16, A_PLANE);
    }
#pragma unroll
    for (int j = 0; j < 2; ++j)
      split_store(b_raw[j], Bs + wave * B_GROUP + ((lane >> 5) * 64 + 32 * j + (lane & 31)) * 16, B_PLANE);
  };

  auto fragment = [&](const char* at) { return *reinterpret_cast<const bf16x8_t*>(at); };
  auto compute = [&]() {
    const char* as = As + (lane >> 5) * A_GROUP + (wr * WM + (lane & 31)) * 16;
    const char* bs = Bs + (lane >> 5) * B_GROUP + (wc * 64 + (lane & 31)) * 16;
#pragma unroll
    for (int s = 0; s < SK / 16; ++s) {
      bf16x8_t b[2][3];
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int q = 0; q < 3; ++q) b[j][q] = fragment(bs + q * B_PLANE + 2 * s * B_GROUP + 32 * 16 * j);
#pragma unroll
      for (int i = 0; i < MI; ++i) {
        bf16x8_t a[3];
#pragma unroll
        for (int q = 0; q < 3; ++q) a[q] = fragment(as + q * A_PLANE + 2 * s * A_GROUP + 32 * 16 * i);
          // the smallest partial products first
        constexpr int pa[6] = {2, 0, 1, 1, 0, 0}, pb[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
        for (int p = 0; p < 6; ++p)
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            float16_t& to = p < 5 ? low[i][j] : acc[i][j];
            to = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[pa[p]], b[j][pb[p]], to, 0, 0, 0);
          }
      }
    }
  };

  load_global(k_begin);
  for (int kk = k_begin; kk < k_end; kk += SK) {
    store_lds(kk);
    __syncthreads();
    if (kk + SK < k_end) load_global(kk + SK);
    __builtin_amdgcn_s_setprio(1);
    compute();
    __builtin_amdgcn_s_setprio(0);
    __syncthreads();
  }

#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = (acc[i][j] + low[i][j]) * kProductScale;
  const int col = wc * 64 + 2 * (lane & 31);
  auto row_of = [&](int i, int e) {
    const int q = 8 * (e >> 2) + 4 * (lane >> 5) + (e & 3);
    return TRANS_A ? wr * WM + MI * q + i : wr * WM + 32 * i + q;
  };
  // An operand that is not finite, or is not once it is scaled, gives infinities or NaNs here, and so do
  // results that scaled are beyond the largest float: such tiles are computed again on the float matrix cores.
  float finite = 0.f;
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        // what lies beside the matrices (between rows of a longer stride) is nobody's to judge by
        const bool inside = row_of(i, e) < rows_here && col + j < cols_here;
        finite = fmaf(inside ? acc[i][j][e] : 0.f, 0.f, finite);
      }
  if (__syncthreads_or(!(finite == 0.f))) {
    float_tile<TRANS_A, BM>(M, N, K, A, lda, B, ldb, C, ldc, accumulate, tm, tn, k_begin, k_end, part,
                           reinterpret_cast<float*>(smem));
    return;
  }

  // Whole tiles with 8-byte aligned rows: a lane's two columns in one store.
  const bool wide = cols_here == BN && (ldc & 1) == 0 && (reinterpret_cast<uintptr_t>(C) & 7) == 0;
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const int row = row_of(i, e);
      if (part != nullptr) {
        const float2_t v = {acc[i][0][e], acc[i][1][e]};
        *reinterpret_cast<float2_t*>(part + row * BN + col) = v;
      } else if (row < rows_here) {
        float* p = C + (size_t)(m0 + row) * ldc + n0 + col;
        if (wide) {
          float2_t v = {acc[i][0][e], acc[i][1][e]};
          if (accumulate) v += *reinterpret_cast<const float2_t*>(p);
          *reinterpret_cast<float2_t*>(p) = v;
          continue;
        }
        if (col < cols_here) p[0] = accumulate ? p[0] + acc[i][0][e] : acc[i][0][e];
        if (col + 1 < cols_here) p[1] = accumulate ? p[1] + acc[i][1][e] : acc[i][1][e];
      }
    }
}

template <bool TRANS_A, int BM>
__global__ __launch_bounds__(256, 2)
void gemm_f32_kernel(int M, int N, int K,
                     const float* __restrict__ A, int lda,
                     const float* __restrict__ B, int ldb,
                     float* __restrict__ C, int ldc, int accumulate,
                     int tiles_n, int whole_tiles, int splits, int k_per_split,
                     float* __restrict__ partial) {
  __shared__ __attribute__((aligned(16))) float smem[(split_operand_bytes(BM) + split_operand_bytes(BN)) / 4];
  // Workgroups [0, whole_tiles) compute one whole tile each.  Ids are handed to the XCDs
  // round-robin; XCD x gets the x-th contiguous chunk of the tile list so that neighbours
  // in the list share an L2.  Workgroups from whole_tiles on compute one K piece of one of
  // the remaining tiles: piece j = id - whole_tiles is split j % splits of tile
  // whole_tiles + j / splits, and parks its result at partial + j * BM * BN.
  const int id = blockIdx.x;
  int tile, k_begin, k_end;
  float* part = nullptr;
  if (id < whole_tiles) {
    const int q = whole_tiles / kXcds, r = whole_tiles % kXcds;
    const int xcd = id % kXcds, local = id / kXcds;
    tile = xcd * q + (xcd < r ? xcd : r) + local;
    k_begin = 0;
    k_end = K;
  } else {
    // Pieces that read the same rows of A -- the same split of the tiles of one row of tiles --
    // form a group, and the groups are dealt to the XCDs (workgroup ids go to them round-robin)
    // so that a group's pieces have consecutive places on one XCD: its rows of A then come
    // from HBM once and from that XCD's L2 afterwards.  (dx of the headline shape, 4 tiles per
    // row: 245 -> 100 MiB fetched.)  Groups beyond the last whole round of 8, and lists that do
    // not consist of whole rows of tiles, keep the plain order.  Where a piece's result is
    // parked does not depend on the order.
    const int j = id - whole_tiles;
    const int rest = (int)gridDim.x - whole_tiles;          // pieces
    int t = j / splits, split = j % splits;                 // plain order
    if ((rest / splits) % tiles_n == 0 && whole_tiles % tiles_n == 0) {
      const int groups = rest / tiles_n;                    // (row of tiles, split) pairs
      const int dealt = groups / kXcds * kXcds * tiles_n;   // pieces in whole rounds of groups
      int group, member;
      if (j < dealt) {
        const int xcd = j % kXcds, place = j / kXcds;
        group = place / tiles_n * kXcds + xcd;
        member = place % tiles_n;
      } else {
        group = (groups / kXcds) * kXcds + (j - dealt) / tiles_n;
        member = (j - dealt) % tiles_n;
      }
      t = (group / splits) * tiles_n + member;
      split = group % splits;
    }
    tile = whole_tiles + t;
    k_begin = split * k_per_split;
    k_end = (k_begin + k_per_split < K) ? (k_begin + k_per_split) : K;
    part = partial + ((size_t)t * splits + split) * BM * BN;
  }
  split_tile<TRANS_A, BM / 64>(M, N, K, A, lda, B, ldb, C, ldc, accumulate, tile / tiles_n, tile % tiles_n,
                             k_begin, k_end, part, reinterpret_cast<char*>(smem));
}

// Two products with the same N and K in one launch (dW = x^T dv and dR = h^T dv of a backward
// pass): A1 row-major [M1,K], A2 stored transposed [K,M2].  Their tiles form one list, every
// tile cut into `splits` K pieces (splits == 1: whole tiles); piece j of the list parks its
// result at partial + j * BM * BN.  One launch of twice the tiles needs half the pieces per
// tile to fill the chip, i.e. half the partial-tile traffic.
struct GemmPair {
  int M1, M2, N, K;
  const float* A1; int lda1; const float* B1; int ldb1; float* C1; int ldc1;
  const float* A2; int lda2; const float* B2; int ldb2; float* C2; int ldc2;
  int accumulate, tiles_n, tiles_m1, splits, k_per_split;
  float* partial;
};

template <int BM>
__global__ __launch_bounds__(256, 2)
void gemm_f32_pair_kernel(GemmPair p) {
  __shared__ __attribute__((aligned(16))) float smem[(split_operand_bytes(BM) + split_operand_bytes(BN)) / 4];
  const int j = blockIdx.x;
  const int tile = j / p.splits;
  const int k_begin = (j % p.splits) * p.k_per_split;
  const int k_end = (k_begin + p.k_per_split < p.K) ? (k_begin + p.k_per_split) : p.K;
  float* part = p.splits > 1 ? p.partial + (size_t)j * BM * BN : nullptr;
  const int tm = tile / p.tiles_n, tn = tile % p.tiles_n;
  if (tm < p.tiles_m1)
    split_tile<false, BM / 64>(p.M1, p.N, p.K, p.A1, p.lda1, p.B1, p.ldb1, p.C1, p.ldc1, p.accumulate,
                             tm, tn, k_begin, k_end, part, reinterpret_cast<char*>(smem));
  else
    split_tile<true, BM / 64>(p.M2, p.N, p.K, p.A2, p.lda2, p.B2, p.ldb2, p.C2, p.ldc2, p.accumulate,
                            tm - p.tiles_m1, tn, k_begin, k_end, part, reinterpret_cast<char*>(smem));
}

// For the split tiles (tile index whole_tiles + blockIdx.x): C tile (+)= sum over its
// `splits` pieces of partial[(blockIdx.x * splits + piece)][BM][BN], pieces added in index
// order.  blockIdx.y selects 8 of the tile's rows; a thread owns 4 consecutive columns.
template <int BM>
__global__ __launch_bounds__(256)
void split_reduce_kernel(int M, int N, int splits, int tiles_n, int whole_tiles,
                         const float* __restrict__ partial, float* __restrict__ C, int ldc,
                         int accumulate, int vec_ok) {
  const int tile = whole_tiles + blockIdx.x;
  const int tm = tile / tiles_n, tn = tile % tiles_n;
  const int r = blockIdx.y * 8 + (threadIdx.x >> 5);
  const int c = (threadIdx.x & 31) * 4;
  const int row = tm * BM + r, col = tn * BN + c;
  if (r >= BM || row >= M || col >= N) return;
  const float* p = partial + ((size_t)blockIdx.x * splits) * BM * BN + r * BN + c;
  float4_t s = *reinterpret_cast<const float4_t*>(p);
  for (int sp = 1; sp < splits; ++sp)
    s += *reinterpret_cast<const float4_t*>(p + (size_t)sp * BM * BN);
  float* out = C + (size_t)row * ldc + col;
  if (vec_ok && col + 3 < N) {
    float4_t* o = reinterpret_cast<float4_t*>(out);
    *o = accumulate ? (*o + s) : s;
  } else {
    const float v[4] = {s.x, s.y, s.z, s.w};
    for (int i = 0; i < 4 && col + i < N; ++i) out[i] = accumulate ? (out[i] + v[i]) : v[i];
  }
}

// The same for the tile list of gemm_f32_pair_kernel: tile rows below tiles_m1 belong to the
// first product.
template <int BM>
__global__ __launch_bounds__(256)
void split_reduce_pair_kernel(int M1, int M2, int N, int splits, int tiles_n, int tiles_m1,
                              const float* __restrict__ partial, float* __restrict__ C1, int ldc1,
                              float* __restrict__ C2, int ldc2, int accumulate, int vec_ok) {
  const int tile = blockIdx.x;
  int tm = tile / tiles_n;
  const int tn = tile % tiles_n;
  const bool second = tm >= tiles_m1;
  if (second) tm -= tiles_m1;
  const int M = second ? M2 : M1;
  float* C = second ? C2 : C1;
  const int ldc = second ? ldc2 : ldc1;
  const int r = blockIdx.y * 8 + (threadIdx.x >> 5);
  const int c = (threadIdx.x & 31) * 4;
  const int row = tm * BM + r, col = tn * BN + c;
  if (r >= BM || row >= M || col >= N) return;
  const float* p = partial + ((size_t)blockIdx.x * splits) * BM * BN + r * BN + c;
  float4_t s = *reinterpret_cast<const float4_t*>(p);
  for (int sp = 1; sp < splits; ++sp)
    s += *reinterpret_cast<const float4_t*>(p + (size_t)sp * BM * BN);
  float* out = C + (size_t)row * ldc + col;
  if (vec_ok && col + 3 < N) {
    float4_t* o = reinterpret_cast<float4_t*>(out);
    *o = accumulate ? (*o + s) : s;
  } else {
    const float v[4] = {s.x, s.y, s.z, s.w};
    for (int i = 0; i < 4 && col + i < N; ++i) out[i] = accumulate ? (out[i] + v[i]) : v[i];
  }
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// How a product is cut into workgroups (depends on the shape only).
struct GemmPlan {
  int bm, tiles_n, whole_tiles, rest, splits, k_per_split, pieces;
  size_t scratch_bytes;
};

// What `tiles` tiles cut into s pieces each cost, in units of what one CU needs for a whole tile
// while two workgroups share it (41 ns * K).  A piece costs as much as 48 k more (its first
// loads, its write-out); workgroups run in rounds of two per CU, and a round of at most one
// per CU takes three quarters of a full one; the partial tiles cost 128 KiB of traffic a piece
// at 4.5 TB/s, the kernel that adds them up 3 us.
double list_cost(long long tiles, int s, int K, int cus) {
  const long long pieces = tiles * s, slots = 2LL * cus, left = pieces % slots;
  const double rounds = (double)(pieces / slots) + (left == 0 ? 0.0 : left <= cus ? 0.75 : 1.0);
  double c = 2.0 * rounds * (1.0 / s + 48.0 / K);
  if (s > 1) c += (0.71 * (double)pieces + 73.0) / K;
  return c;
}

GemmPlan plan_gemm(int M, int N, int K) {
  GemmPlan g;
  g.tiles_n = (N + BN - 1) / BN;
  const int cus = device_cu_count() > 0 ? device_cu_count() : 256;

  // Tile height: 64 rows only when the output has no more than that.
  g.bm = M <= 64 ? 64 : 128;
  const int tiles_m = (M + g.bm - 1) / g.bm;
  const long long tiles = (long long)tiles_m * g.tiles_n;

  // Either all tiles whole, or whole tiles for full rounds of two per CU and the `rest` cut
  // into the cheapest number of K pieces; the choice depends on the shape only, so results are
  // reproducible.  (Measured, us: 6400 x 512 x 2048, 200 tiles, in 1 / 2 / 4 / 5 pieces 122 / 84 /
  // 91 / 87; 512 x 8192 x 3200, 256 tiles, in 1 / 2 / 4: 190 / 143 / 154; 12800 x 2048 x 512, 1600
  // tiles, whole 162, the last 64 in 4 pieces 150; 6400 x 2048 x 512, 800 tiles, whole 82, the
  // last 32 in 4 pieces 85.)
  const long long whole = tiles / (2 * cus) * (2 * cus);
  int splits = 1;
  g.rest = (int)(tiles - whole);
  if (g.rest > 0) {
    int s_max = K / 64;
    if (s_max > 64) s_max = 64;
    double best = list_cost(tiles, 1, K, cus) - list_cost(whole, 1, K, cus);
    // At most four pieces per CU: that bounds the partial tiles of any product (64 KiB a
    // piece) by a size callers who lend the library its scratch memory can plan for.
    for (int s = 2; s <= s_max && (long long)g.rest * s <= 4LL * cus; ++s) {
      const double c = list_cost(g.rest, s, K, cus);
      if (c < best - 1e-9) { best = c; splits = s; }
    }
  }
  g.k_per_split = (K + splits - 1) / splits;
  g.k_per_split = (g.k_per_split + SK - 1) / SK * SK;
  g.splits = (K + g.k_per_split - 1) / g.k_per_split;
  const bool split = g.splits > 1;
  // Unsplit "rest" tiles are ordinary whole tiles.
  g.whole_tiles = split ? (int)whole : (int)tiles;
  g.pieces = split ? g.rest * g.splits : 0;
  g.scratch_bytes = (size_t)g.pieces * g.bm * BN * sizeof(float);
  return g;
}

}  // namespace

size_t gemm_f32_scratch_bytes(int M, int N, int K) {
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  // Which kernel runs also depends on the operands' alignment: room for either.
  const size_t tiled = plan_gemm(M, N, K).scratch_bytes;
  const size_t skinny = gemm_f32_skinny_shape(false, M, N, K) ? gemm_f32_skinny_scratch_bytes(M, N, K) : 0;
  return tiled > skinny ? tiled : skinny;
}

namespace {
int gemm_f32_once(hipStream_t stream, bool trans_a, int M, int N, int K,
                  const float* A, int lda, const float* B, int ldb,
                  float* C, int ldc, bool accumulate, size_t scratch_offset);
}  // namespace

// A workgroup of the tile kernel addresses its operand panels (its rows of A, its columns of
// B, all of K) with 32-bit byte offsets, so a panel must stay under 2 GiB.  A longer
// contraction -- the dW and dR products of a backward pass contract over T*N with rows of 4H
// floats, 2 GiB from T*N*H = 2^27 on -- is cut into runs of K that fit, each accumulating into
// C; where the cuts fall depends on the shape only.
int gemm_f32(hipStream_t stream, bool trans_a, int M, int N, int K,
             const float* A, int lda, const float* B, int ldb,
             float* C, int ldc, bool accumulate, size_t scratch_offset) {
  HASTE_HIP_REQUIRE(M > 0 && N > 0 && K > 0);
  HASTE_HIP_REQUIRE(A != nullptr && B != nullptr && C != nullptr);
  HASTE_HIP_REQUIRE(lda >= (trans_a ? M : K) && ldb >= N && ldc >= N);
  const long long limit = (1ll << 29) - 256;  // floats a panel may span
  long long run = (limit - BN) / ldb;
  if (trans_a) {
    const long long a_run = (limit - 128) / lda;
    run = a_run < run ? a_run : run;
  } else if (128ll * lda + K >= limit) {
    run = 0;  // 128 rows of A alone exceed the limit
  }
  if (run >= K) return gemm_f32_once(stream, trans_a, M, N, K, A, lda, B, ldb, C, ldc, accumulate, scratch_offset);
  run = run / 1024 * 1024;
  if (run <= 0) {
    set_error_text("gemm: a row of an operand is too long for the kernel's 32-bit panel offsets "
                   "(leading dimension of 2^19 floats or more per 1024 rows)");
    return HASTE_HIP_ERROR_UNSUPPORTED_SIZE;
  }
  for (long long k0 = 0; k0 < K; k0 += run) {
    const int kc = (int)(K - k0 < run ? K - k0 : run);
    const float* a = trans_a ? A + (size_t)k0 * lda : A + k0;
    HASTE_HIP_PROPAGATE(gemm_f32_once(stream, trans_a, M, N, kc, a, lda, B + (size_t)k0 * ldb, ldb, C, ldc,
                                      accumulate || k0 > 0, scratch_offset));
  }
  return HASTE_HIP_OK;
}

namespace {
int gemm_f32_once(hipStream_t stream, bool trans_a, int M, int N, int K,
                  const float* A, int lda, const float* B, int ldb,
                  float* C, int ldc, bool accumulate, size_t scratch_offset) {
  HASTE_HIP_REQUIRE(M > 0 && N > 0 && K > 0);
  HASTE_HIP_REQUIRE(A != nullptr && B != nullptr && C != nullptr);
  HASTE_HIP_REQUIRE(lda >= (trans_a ? M : K) && ldb >= N && ldc >= N);
  HASTE_HIP_REQUIRE((long long)((M + 63) / 64) * ((N + BN - 1) / BN) < (1ll << 26));
  if (gemm_f32_skinny_applies(trans_a, M, N, K, A, lda, B, ldb, C, ldc))
    return gemm_f32_skinny(stream, M, N, K, A, lda, B, ldb, C, ldc, accumulate, scratch_offset);
  const GemmPlan g = plan_gemm(M, N, K);
  const int bm = g.bm, tiles_n = g.tiles_n, whole_tiles = g.whole_tiles, rest = g.rest;
  const int splits = g.splits, k_per_split = g.k_per_split, pieces = g.pieces;
  const bool split = splits > 1;

  // The partial tiles live `scratch_offset` bytes (a multiple of 16) into the stream's
  // scratch buffer; callers that keep data of their own in front of them say so.
  Workspace ws;
  float* partial = nullptr;
  if (split) {
    HASTE_HIP_PROPAGATE(get_workspace(stream, scratch_offset + g.scratch_bytes, &ws));
    partial = ws.scratch + scratch_offset / sizeof(float);
  }
  // A workgroup addresses its operand panels (its rows of A, its columns of B, all of K)
  // with 32-bit byte offsets.
  HASTE_HIP_REQUIRE(((long long)(trans_a ? K : bm) * lda + (trans_a ? bm : K)) * 4 < (1ll << 31));
  HASTE_HIP_REQUIRE(((long long)K * ldb + BN) * 4 < (1ll << 31));
  if (planned_pass() != nullptr) return HASTE_HIP_OK;
  dim3 grid((unsigned)(whole_tiles + pieces)), block(256);
  ScopedKernelTimer timer("gemm_f32", stream);
#define HASTE_GEMM_LAUNCH(TA_, BM_)                                                          \
  if (trans_a == TA_ && bm == BM_)                                                           \
    gemm_f32_kernel<TA_, BM_><<<grid, block, 0, stream>>>(                                   \
        M, N, K, A, lda, B, ldb, C, ldc, accumulate ? 1 : 0, tiles_n, whole_tiles, splits,   \
        k_per_split, partial);
  HASTE_GEMM_LAUNCH(false, 128) HASTE_GEMM_LAUNCH(false, 64)
  HASTE_GEMM_LAUNCH(true, 128) HASTE_GEMM_LAUNCH(true, 64)
#undef HASTE_GEMM_LAUNCH
  HASTE_HIP_TRY(hipGetLastError());
  if (split) {
    const int vec = (ldc % 4 == 0) && aligned16(C);
    const dim3 rgrid((unsigned)rest, (unsigned)(bm / 8));
    if (bm == 128)
      split_reduce_kernel<128><<<rgrid, dim3(256), 0, stream>>>(
          M, N, splits, tiles_n, whole_tiles, partial, C, ldc, accumulate ? 1 : 0, vec);
    else
      split_reduce_kernel<64><<<rgrid, dim3(256), 0, stream>>>(
          M, N, splits, tiles_n, whole_tiles, partial, C, ldc, accumulate ? 1 : 0, vec);
    HASTE_HIP_TRY(hipGetLastError());
  }
  return HASTE_HIP_OK;
}
}  // namespace

// C1[M1,N] (+)= A1[M1,K] * B1 and C2[M2,N] (+)= A2^T * B2 (A2 stored [K,M2]) in one launch when
// together they have fewer tiles than the chip has CUs (then each alone would be cut into
// twice the pieces); otherwise two ordinary products.  `products` of the timer: 2.
int gemm_f32_pair(hipStream_t stream, int M1, int M2, int N, int K, const float* A1, int lda1,
                  const float* B1, int ldb1, float* C1, int ldc1, const float* A2, int lda2,
                  const float* B2, int ldb2, float* C2, int ldc2, bool accumulate) {
  HASTE_HIP_REQUIRE(M1 > 0 && M2 > 0 && N > 0 && K > 0 && A1 && B1 && C1 && A2 && B2 && C2);
  HASTE_HIP_REQUIRE(lda1 >= K && lda2 >= M2 && ldb1 >= N && ldb2 >= N && ldc1 >= N && ldc2 >= N);
  const int cus = device_cu_count() > 0 ? device_cu_count() : 256;
  const int tiles_n = (N + BN - 1) / BN;
  const int tiles_m1 = (M1 + 127) / 128, tiles_m2 = (M2 + 127) / 128;
  const long long tiles = (long long)(tiles_m1 + tiles_m2) * tiles_n;
  const bool panels_ok = ((long long)128 * lda1 + K) * 4 < (1ll << 31) && ((long long)K * lda2 + 128) * 4 < (1ll << 31) &&
                         ((long long)K * ldb1 + BN) * 4 < (1ll << 31) && ((long long)K * ldb2 + BN) * 4 < (1ll << 31);
  if (tiles >= cus || M1 <= 64 || M2 <= 64 || !panels_ok) {
    HASTE_HIP_PROPAGATE(gemm_f32(stream, false, M1, N, K, A1, lda1, B1, ldb1, C1, ldc1, accumulate));
    return gemm_f32(stream, true, M2, N, K, A2, lda2, B2, ldb2, C2, ldc2, accumulate);
  }
  int s_max = K / 64;
  if (s_max > 64) s_max = 64;
  int splits = 1;
  double best = list_cost(tiles, 1, K, cus);
  for (int s = 2; s <= s_max && tiles * s <= 4LL * cus; ++s)
    if (list_cost(tiles, s, K, cus) < best - 1e-9) { best = list_cost(tiles, s, K, cus); splits = s; }
  int k_per_split = (K + splits - 1) / splits;
  k_per_split = (k_per_split + SK - 1) / SK * SK;
  splits = (K + k_per_split - 1) / k_per_split;

  GemmPair p;
  p.M1 = M1; p.M2 = M2; p.N = N; p.K = K;
  p.A1 = A1; p.lda1 = lda1; p.B1 = B1; p.ldb1 = ldb1; p.C1 = C1; p.ldc1 = ldc1;
  p.A2 = A2; p.lda2 = lda2; p.B2 = B2; p.ldb2 = ldb2; p.C2 = C2; p.ldc2 = ldc2;
  p.accumulate = accumulate ? 1 : 0;
  p.tiles_n = tiles_n; p.tiles_m1 = tiles_m1; p.splits = splits; p.k_per_split = k_per_split;
  p.partial = nullptr;
  if (splits > 1) {
    Workspace ws;
    HASTE_HIP_PROPAGATE(get_workspace(stream, (size_t)tiles * splits * 128 * BN * sizeof(float), &ws));
    p.partial = ws.scratch;
  }
  if (planned_pass() != nullptr) return HASTE_HIP_OK;
  ScopedKernelTimer timer("gemm_f32", stream, 2);
  gemm_f32_pair_kernel<128><<<dim3((unsigned)(tiles * splits)), dim3(256), 0, stream>>>(p);
  HASTE_HIP_TRY(hipGetLastError());
  if (splits > 1) {
    const int vec = (ldc1 % 4 == 0) && (ldc2 % 4 == 0) && aligned16(C1) && aligned16(C2);
    split_reduce_pair_kernel<128><<<dim3((unsigned)tiles, 16), dim3(256), 0, stream>>>(
        M1, M2, N, splits, tiles_n, tiles_m1, p.partial, C1, ldc1, C2, ldc2, p.accumulate, vec);
    HASTE_HIP_TRY(hipGetLastError());
  }
  return HASTE_HIP_OK;
}

// The product as its K pieces, for a consumer that adds them itself (in piece order): only the
// tile kernel is launched.  Possible when every tile of the product is cut into pieces and
// the output is one tile high; *splits == 0 otherwise (nothing launched).  Element (row, col)
// of piece s lies at partial[((col / 128 * splits + s) * bm + row) * 128 + col % 128]; valid
// until the next product on the stream.
int gemm_f32_pieces(hipStream_t stream, int M, int N, int K, const float* A, int lda,
                    const float* B, int ldb, size_t scratch_offset, const float** partial,
                    int* splits, int* bm) {
  *splits = 0;
  HASTE_HIP_REQUIRE(M > 0 && N > 0 && K > 0 && A != nullptr && B != nullptr);
  HASTE_HIP_REQUIRE(lda >= K && ldb >= N);
  const GemmPlan g = plan_gemm(M, N, K);
  if (g.splits <= 1 || g.whole_tiles != 0 || M > g.bm) return HASTE_HIP_OK;
  if (((long long)g.bm * lda + K) * 4 >= (1ll << 31) || ((long long)K * ldb + BN) * 4 >= (1ll << 31))
    return HASTE_HIP_OK;
  Workspace ws;
  HASTE_HIP_PROPAGATE(get_workspace(stream, scratch_offset + g.scratch_bytes, &ws));
  float* part = ws.scratch + scratch_offset / sizeof(float);
  dim3 grid((unsigned)g.pieces), block(256);
  ScopedKernelTimer timer("gemm_f32", stream);
  if (g.bm == 128)
    gemm_f32_kernel<false, 128><<<grid, block, 0, stream>>>(M, N, K, A, lda, B, ldb, nullptr, 0, 0, g.tiles_n,
                                                            0, g.splits, g.k_per_split, part);
  else
    gemm_f32_kernel<false, 64><<<grid, block, 0, stream>>>(M, N, K, A, lda, B, ldb, nullptr, 0, 0, g.tiles_n,
                                                           0, g.splits, g.k_per_split, part);
  HASTE_HIP_TRY(hipGetLastError());
  *partial = part;
  *splits = g.splits;
  *bm = g.bm;
  return HASTE_HIP_OK;
}

}  // namespace haste_hip

extern "C" int haste_hip_gemm_f32(int trans_a, int M, int N, int K,
                                  const float* A, int lda, const float* B, int ldb,
                                  float* C, int ldc, int accumulate, void* stream) {
  return haste_hip::gemm_f32(haste_hip::as_stream(stream), trans_a != 0, M, N, K, A, lda, B, ldb,
                             C, ldc, accumulate != 0);
}
