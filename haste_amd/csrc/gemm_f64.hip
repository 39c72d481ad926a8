// C[M,N] (+)= op(A)[M,K] * B[K,N] in double precision on the fp64 matrix cores
// (v_mfma_f64_16x16x4_f64): what the `double` instantiations of the reference get from
// cublasDgemm (lib/blas.h:48-61).
//
// Bound: MFMA (fp64 peak 78.6 TFLOP/s), algorithmic flops 2*M*N*K.  A workgroup of four
// wavefronts owns a 64 x 64 tile of C; a wavefront owns 32 x 32 of it as 2 x 2 MFMA tiles.
// Operand panels of 32 k go through LDS k-major ([k][m], [k][n]): the lanes of one MFMA
// operand read 16 consecutive doubles of one k row.  Panels are loaded in runs of 256 - 512
// bytes and requested three ahead.  Two workgroups share a CU (256 registers a lane, accumulators and
// operands alike: given 512, the compiler computed in one half of the file and kept the accumulators in the other,
// 64 moves and a wait for the matrix cores every two panels), and the tiles that would fill a last round of
// workgroups only partly are cut along K, as is a product of few tiles and a long contraction (the product of one step
// over 70 rows: 128 x 512 x 2048 is 16 tiles): each piece a workgroup of its own, which parks partial results in the
// stream's scratch buffer; a second kernel adds a tile's pieces in index order.  Measured, launches back to back, before and
// after those two, the loop and the order of tiles below: 6400 x 2048 x 512 255 -> 230 us, 6400 x 512 x 2048 306 -> 222,
// 512 x 2048 x 6400 299 -> 237, with A transposed 281 -> 222 (60 TFLOP/s), 4096^3 59 -> 64 TFLOP/s (the library: 72);
// a step's product 16 x 256 x 64 5.3 -> 5.2, 16 x 808 x 202 15.1 -> 12.2, 16 x 3072 x 768 13.1 -> 13.0.
// How a product is cut depends on its shape and the device, and where the scratch buffer has no room for the pieces it is
// not: the same call gives the same bits with any workspace that holds them.  Lane layout of the instruction (checked on the hardware): a = A[i = lane%16][k = lane/16], b = B[k = lane/16][j = lane%16],
// d[r] = D[i = 4*r + lane/16][j = lane%16].
#include "common.h"

namespace haste_hip {
namespace {

typedef double double4_t __attribute__((ext_vector_type(4)));
typedef double double2_t __attribute__((ext_vector_type(2)));
typedef unsigned int uint2_t __attribute__((ext_vector_type(2)));
typedef unsigned int uint4_t __attribute__((ext_vector_type(4)));
constexpr unsigned int kNowhere = 0x7ffffff0u;  // an offset beyond any buffer resource's range: the load returns zeros

constexpr int DM = 64, DN = 64, DK = 32;

// Where element i (row of A, column of B) of panel row k lies in LDS.  The operand reads of an
// instruction take 16 elements of four consecutive k, the transposing stores of A one k of every
// second of 32 and four rows: the exclusive or with bits of k spreads both evenly over the banks
// (two words each) and keeps neighbouring elements side by side.
__device__ __forceinline__ int panel_at(int k, int i) {
  return k * 64 + (i ^ (((k >> 1) & 3) << 2) ^ (((k >> 3) ^ k) & 1) << 4);
}

// How a product is cut: the first `whole` tiles (row by row) are not, the others into `pieces` of k_per_piece each.
struct F64Plan {
  int whole, pieces, k_per_piece;
  int in_order = 0;
};
constexpr int kXcds = 8;

// How a workgroup's operands are loaded: pairs in whole panels, pairs with a ragged last panel, or single elements.
enum { kWhole, kPairs, kSingle };

template <bool TRANS_A>
__global__ __launch_bounds__(256, 2)
void gemm_f64_kernel(int M, int N, int K, const double* __restrict__ A, int lda,
                     const double* __restrict__ B, int ldb, double* __restrict__ C, int ldc,
                     int accumulate, F64Plan plan, int tiles_n, double* __restrict__ part, int chunks, int panels_ok) {
  __shared__ double2_t panels[2][2][DK * 64 / 2];  // [buffer][A, B]
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  // Workgroups [0, whole) take a tile each, in_order or with a contiguous run of them for every XCD (ids go to the XCDs
  // round-robin; see tiles_in_order), the others a piece of one of the remaining tiles, an XCD a run of them.
  int tile, piece = 0;
  {
    const int id = blockIdx.x;
    auto mine = [](int at, int count) {
      const int xcd = at % kXcds, q = count / kXcds, r = count % kXcds;
      return xcd * q + (xcd < r ? xcd : r) + at / kXcds;
    };
    if (id < plan.whole) {
      tile = plan.in_order ? id : mine(id, plan.whole);
    } else {
      const int at = mine(id - plan.whole, (int)gridDim.x - plan.whole);
      tile = plan.whole + at / plan.pieces;
      piece = at % plan.pieces;
    }
  }
  const int m0 = tile / tiles_n * DM, n0 = tile % tiles_n * DN;
  const int wm = (wave >> 1) * 32, wn = (wave & 1) * 32;
  // Loads go through buffer resources, 16 bytes at a time and without a branch: pairs beyond the problem take an offset
  // beyond the resource's range and read as zero, as do rows of A beyond M.  A pair must lie inside or outside as a
  // whole: a piece of K (A not transposed), a last tile's columns or transposed rows of odd number load every element
  // under its own bounds check (one branch each).  (Ragged pieces took that path too: 768 x 3072 x 2000, A
  // transposed, 272 -> 164 us, 300 x 1200 x 3071 87 -> 54.)
  const bool cut = tile >= plan.whole;
  const int piece_begin = cut ? piece * plan.k_per_piece : 0;
  const int piece_end = cut && piece_begin + plan.k_per_piece < K ? piece_begin + plan.k_per_piece : K;
  const bool fast = panels_ok != 0 && (n0 + DN <= N || N % 2 == 0) &&
                    (TRANS_A ? m0 + DM <= M || M % 2 == 0 : (piece_end - piece_begin) % 2 == 0);
  const __amdgpu_buffer_rsrc_t pa = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<double*>(A), 0,
      fast ? (int)((TRANS_A ? (long long)(K - 1) * lda + M : (long long)(M - 1) * lda + K) * 8) : 0, 0x00020000);
  const __amdgpu_buffer_rsrc_t pb = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<double*>(B), 0, fast ? (int)(((long long)(K - 1) * ldb + N) * 8) : 0, 0x00020000);
  // Load i of a panel: where rows run along k (A not transposed) 16 lanes take the 32 k of a row and
  // i counts 16 rows, otherwise 32 lanes take the 64 elements of one k and i counts 8 k -- a
  // wavefront's load is runs of 256 or 512 bytes.
  const int rrow = tid >> 4, rk = (tid & 15) * 2;
  const int ck = tid >> 5, ci = (tid & 31) * 2;
  const unsigned int a_voff = TRANS_A ? m0 + ci < M ? (unsigned int)((ck * lda + m0 + ci) * 8) : kNowhere
                                      : (unsigned int)(((m0 + rrow) * lda + rk) * 8);
  const unsigned int a_step = (unsigned int)((TRANS_A ? 8 : 16) * lda) * 8u, b_step = (unsigned int)ldb * 64u;
  const unsigned int b_voff = n0 + ci < N ? (unsigned int)((ck * ldb + n0 + ci) * 8) : kNowhere;
  double4_t acc[2][2];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) acc[a][b] = double4_t{0.0, 0.0, 0.0, 0.0};

  // A thread's 8 elements of each operand panel.  Panels are requested three ahead of the MFMAs
  // (two in registers, one in LDS): a product with one workgroup per CU has nothing else to do
  // while it waits for memory.
  double2_t ra[2][4], rb[2][4];
  auto request = [&](auto fast_c, int set, int k0) {
    if constexpr (decltype(fast_c)::value != kSingle) {
      const int sa = TRANS_A ? k0 * lda * 8 : k0 * 8, sb = k0 * ldb * 8;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const bool whole = decltype(fast_c)::value == kWhole;
        const bool b_in = whole || k0 + ck + 8 * i < K, a_in = TRANS_A ? b_in : whole || k0 + rk < K;
        const unsigned int ao = a_in ? a_voff + i * a_step : kNowhere, bo = b_in ? b_voff + i * b_step : kNowhere;
        ra[set][i] = __builtin_bit_cast(double2_t, __builtin_amdgcn_raw_buffer_load_b128(pa, ao, sa, 0));
        rb[set][i] = __builtin_bit_cast(double2_t, __builtin_amdgcn_raw_buffer_load_b128(pb, bo, sb, 0));
      }
      return;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        if (TRANS_A) {
          const int gk = k0 + ck + 8 * i, gm = m0 + ci + e;
          ra[set][i][e] = (gm < M && gk < K) ? A[(size_t)gk * lda + gm] : 0.0;
        } else {
          const int gk = k0 + rk + e, gm = m0 + rrow + 16 * i;
          ra[set][i][e] = (gm < M && gk < K) ? A[(size_t)gm * lda + gk] : 0.0;
        }
        const int gk = k0 + ck + 8 * i, gn = n0 + ci + e;
        rb[set][i][e] = (gn < N && gk < K) ? B[(size_t)gk * ldb + gn] : 0.0;
      }
  };
  auto park = [&](int set, int buffer) {
    double2_t* as = panels[buffer][0];
    double2_t* bs = panels[buffer][1];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (TRANS_A) {
        as[panel_at(ck + 8 * i, ci) / 2] = ra[set][i];
      } else {
#pragma unroll
        for (int e = 0; e < 2; ++e)
          reinterpret_cast<double*>(as)[panel_at(rk + e, rrow + 16 * i)] = ra[set][i][e];
      }
      bs[panel_at(ck + 8 * i, ci) / 2] = rb[set][i];
    }
  };

  // this workgroup's piece of the contraction; request() and the loop below see its end as K
  const int k_begin = piece_begin;
  K = piece_end;
  int row0 = m0, col0 = n0, rows = M, cols = N;
  if (cut && chunks) {  // piece z parks [M][N] at part + z * M * N
    C = part + (size_t)piece * M * N;
    ldc = N;
    accumulate = 0;
  } else if (cut) {
    // A tile's pieces park [64][64] one behind the other, what there is of them (the zeros of 60 rows that do
    // not exist, 9 MB at 4 x 768 x 3072, took 1.2 us of 15.4).
    C = part + ((size_t)(tile - plan.whole) * plan.pieces + piece) * DM * DN;
    ldc = DN;
    row0 = col0 = accumulate = 0;
    rows = M - m0;
    cols = N - n0;
  }
  // The operands of an instruction group are read one group ahead: a wavefront issues in order, so a read behind the
  // group before it comes back when the matrix cores have run dry.  between(g): what is issued behind group g.
  auto multiply = [&](int buffer, auto&& between) {
    const double* as = reinterpret_cast<const double*>(panels[buffer][0]);
    const double* bs = reinterpret_cast<const double*>(panels[buffer][1]);
    double a[2][2], b[2][2];
    auto read = [&](int g) {
      const int k = 4 * g + (lane >> 4), o = lane & 15;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        a[g & 1][i] = as[panel_at(k, wm + 16 * i + o)];
        b[g & 1][i] = bs[panel_at(k, wn + 16 * i + o)];
      }
    };
    read(0);
#pragma unroll
    for (int g = 0; g < DK / 4; ++g) {
      if (g + 1 < DK / 4) read(g + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[g & 1][i], b[g & 1][j], acc[i][j], 0, 0, 0);
      between(g);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // Panel p lies in buffer p % 2; at its turn the panel behind it is parked in the other buffer,
  // which everybody has finished with, and the one three behind requested.  Without a branch: with one the compiler cannot
  // tell which loads a panel waits for, and waited for all of them, and read the operands of a group when its instructions
  // were due.  (6400 x 2048 x 512 271 -> 262 us, 512 x 2048 x 6400 296 -> 277, with A transposed 278 -> 258.)  The last
  // one or two panels are written out: a turn of the barrier or a wait for nobody shows in the product of a step.
  auto run = [&](auto fast_c) {
    const int last = k_begin + (K - k_begin - 1) / DK * DK;
    auto panel = [&](auto parity, int k0) {
      constexpr int P = decltype(parity)::value;
      multiply(P, [&](int g) {
        if (g == 1) park(P ^ 1, P ^ 1);
        if (g == 3) request(fast_c, P ^ 1, k0 + 3 * DK < last ? k0 + 3 * DK : last);
      });
      __syncthreads();
    };
    auto finish = [&](int k0) {
      const bool two = k0 + DK < K;
      multiply(0, [&](int g) {
        if (g == 1 && two) park(1, 1);
      });
      if (!two) return;
      __syncthreads();
      multiply(1, [](int) {});
    };
    request(fast_c, 0, k_begin);
    if (K - k_begin <= 2 * DK) {
      if (k_begin + DK < K) request(fast_c, 1, k_begin + DK);
      park(0, 0);
      __syncthreads();
      return finish(k_begin);
    }
    request(fast_c, 1, k_begin + DK);
    park(0, 0);
    request(fast_c, 0, k_begin + 2 * DK);
    __syncthreads();
    int k0 = k_begin;
    for (; k0 + 2 * DK < K; k0 += 2 * DK) {
      panel(std::integral_constant<int, 0>{}, k0);
      panel(std::integral_constant<int, 1>{}, k0 + DK);
    }
    finish(k0);
  };
  // Element by element the loads are branches, many instructions each: all of them in front of a panel's product.
  auto run_single = [&] {
    const std::integral_constant<int, kSingle> single{};
    auto panel = [&](int p, int k0) {
      if (k0 + DK < K) park(p ^ 1, p ^ 1);
      if (k0 + 3 * DK < K) request(single, p ^ 1, k0 + 3 * DK);
      multiply(p, [](int) {});
      __syncthreads();
    };
    request(single, 0, k_begin);
    if (k_begin + DK < K) request(single, 1, k_begin + DK);
    park(0, 0);
    if (k_begin + 2 * DK < K) request(single, 0, k_begin + 2 * DK);
    __syncthreads();
    for (int k0 = k_begin; k0 < K; k0 += 2 * DK) {
      panel(0, k0);
      if (k0 + DK < K) panel(1, k0 + DK);
    }
  };
  if (!fast) run_single();
  else if ((K - k_begin) % DK == 0) run(std::integral_constant<int, kWhole>{});
  else run(std::integral_constant<int, kPairs>{});
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int gm = row0 + wm + 16 * a + 4 * r + (lane >> 4);
        const int gn = col0 + wn + 16 * b + (lane & 15);
        if (gm < rows && gn < cols) {
          double* p = C + (size_t)gm * ldc + gn;
          *p = accumulate ? *p + acc[a][b][r] : acc[a][b][r];
        }
      }
}

// C (+)= the pieces of every element of the cut tiles, added in index order.  A workgroup takes kReduceRows rows of a tile, a
// thread two columns.
constexpr int kReduceRows = 8;
__global__ __launch_bounds__(256)
void gemm_f64_reduce_kernel(int M, int N, F64Plan plan, int tiles_n, const double* __restrict__ part,
                            double* __restrict__ C, int ldc, int accumulate) {
  const int tile = plan.whole + blockIdx.x;
  const int r = blockIdx.y * kReduceRows + (threadIdx.x >> 5), c = (threadIdx.x & 31) * 2;
  const int row = tile / tiles_n * DM + r, col = tile % tiles_n * DN + c;
  if (row >= M || col >= N) return;
  const double* p = part + (size_t)blockIdx.x * plan.pieces * DM * DN + r * DN + c;
  double2_t s = *reinterpret_cast<const double2_t*>(p);
#pragma unroll 8  // (eight pieces' loads in flight: 24 pieces of 4 x 768 4.5 -> 4.0 us)
  for (int z = 1; z < plan.pieces; ++z) s += *reinterpret_cast<const double2_t*>(p + (size_t)z * DM * DN);
  double* out = C + (size_t)row * ldc + col;
#pragma unroll
  for (int i = 0; i < 2; ++i)
    if (col + i < N) out[i] = accumulate ? out[i] + s[i] : s[i];
}

// Whether the whole tiles go to the workgroups as they are numbered, so that XCD x (one L2) gets number x and every eighth
// from there, rather than in a contiguous run per XCD: what reads fewer panels of A and B into an L2.  With a multiple of eight
// columns of tiles an XCD's are the same in every row and only the tiles in flight count; with four they alternate; otherwise all
// columns take turns.  (In order / in runs, us: 32 columns, 6400 x 2048 x 512 228 / 235, 768 x 2048 x 256 added to C 23.1 / 27.3;
// 28 columns, 512 x 1792 x 256 15.1 / 18.4; 8 columns, 6400 x 512 x 2048 225 / 222; 13 columns, 6400 x 808 x 512 106 / 103,
// 1500 x 808 x 128 added to C 17.8 / 15.0.)
bool tiles_in_order(long long tiles_m, long long tiles_n, long long whole, long long cus) {
  const int every = tiles_n % 8 == 0 ? 8 : (tiles_n % 4 == 0 ? 4 : 1);
  if (every == 1) return false;
  long long mine = whole / kXcds;
  if (every == 8 && mine > 2 * cus / kXcds) mine = 2 * cus / kXcds;
  const long long run_rows = (mine + tiles_n - 1) / tiles_n, order_rows = (mine * kXcds + tiles_n - 1) / tiles_n;
  return (order_rows < tiles_m ? order_rows : tiles_m) + tiles_n / every < run_rows + (mine < tiles_n ? mine : tiles_n);
}

// Whole tiles for full rounds of one per CU (a CU holds two workgroups, which share its matrix cores); the tiles of the
// last, partial round are cut along K into pieces that make about two per CU, a piece keeping at least 8 panels of the
// contraction (its first panel's load and its 64 KiB of partial results show below that).  A last round of more than
// three quarters of the CUs has too little to give: stays whole (6400 x 512 x 2048, 800 tiles: 295 us whole, 222 with the last
// 32 in 8).  A product of no more tiles than CUs is cut into the number of pieces that is expected to be fastest, of at
// least 4 panels.  Measured, in us: 5.5 and 1.25 a panel for whole tiles; 4.5 and 0.02 a workgroup for the pieces' way through
// memory, 1.25 a panel again, 2 where two workgroups share a CU.  (512 x 2048 x 256 / 1024 / 6400, 256 tiles: 15.3 / 46.5 / 258
// whole, 22.8 / 48.5 / 238 in two; 256 x 2048 x 1024: 45.7 whole, 31.3 in four; 64 x 2048 x 2048: 22.4 in 16, 19.4 in 8; 4 x
// 768 x 3072: 14.2 in 24, 10.4 in 20.)
F64Plan plan_f64(int M, int N, int K) {
  const long long tiles_m = (M + DM - 1) / DM, tiles_n = (N + DN - 1) / DN, tiles = tiles_m * tiles_n;
  const long long cus = device_cu_count() > 0 ? device_cu_count() : 256;
  const F64Plan uncut{(int)tiles, 1, K, tiles_in_order(tiles_m, tiles_n, tiles, cus)};
  const long long whole = tiles > cus ? tiles / cus * cus : 0;
  const long long rest = tiles - whole;
  if (rest == 0) return uncut;
  auto cut = [&](long long pieces) {
    const int per = ((int)((K + pieces - 1) / pieces) + DK - 1) / DK * DK;
    return F64Plan{(int)whole, (K + per - 1) / per, per, tiles_in_order(tiles_m, tiles_n, whole, cus)};
  };
  long long most = K / ((whole > 0 ? 8 : 4) * DK);
  most = most < 64 ? most : 64;
  if (whole > 0) {
    const long long pieces = 2 * cus / rest < most ? 2 * cus / rest : most;
    if (pieces <= 1 || 4 * rest > 3 * cus) return uncut;
    const F64Plan p = cut(pieces);
    return p.pieces > 1 ? p : uncut;
  }
  F64Plan best = uncut;
  long long best_cost = 275 + 62ll * ((K + DK - 1) / DK);  // 1/50 us
  for (long long pieces = 2; pieces <= most && tiles * pieces <= 2 * cus; ++pieces) {
    const F64Plan p = cut(pieces);
    const long long workgroups = tiles * p.pieces;
    const long long cost = 225 + workgroups + (workgroups > cus ? 100 : 62) * (p.k_per_piece / DK);
    if (p.pieces > 1 && cost < best_cost) {
      best = p;
      best_cost = cost;
    }
  }
  return best;
}
// The same for a consumer that adds the pieces itself: all tiles, about one piece per CU.
F64Plan plan_f64_chunks(int M, int N, int K) {
  const long long tiles = (long long)((M + DM - 1) / DM) * ((N + DN - 1) / DN);
  int s = 1;
  if (tiles < 128) {
    s = (int)(256 / tiles);
    const int most = K / (4 * DK);
    s = s < most ? s : most;
    s = s < 64 ? s : 64;
    s = s > 1 ? s : 1;
  }
  int per = (K + s - 1) / s;
  per = (per + DK - 1) / DK * DK;
  return F64Plan{0, (K + per - 1) / per, per};
}
size_t f64_piece_bytes(const F64Plan& plan, int M, int N) {
  const long long tiles = (long long)((M + DM - 1) / DM) * ((N + DN - 1) / DN);
  return plan.pieces > 1 ? (size_t)(tiles - plan.whole) * plan.pieces * DM * DN * sizeof(double) : 0;
}

// ---- The product of one step of the step-wise regime: at most 64 rows (the batch), a few
// hundred to a few thousand columns and as long a contraction.  The tile kernel above gives
// it a handful of tiles whose workgroups walk their K range panel by panel, a load latency
// each; here everything a wavefront needs is requested at once and goes from memory straight
// into the MFMA operand registers -- no LDS, no barrier before the last sum.
//   * A workgroup takes 16 columns, all rows (RB blocks of 16) and k_per_wg of the contraction;
//     its four wavefronts take a quarter of that each and their blocks are added through LDS
//     in wavefront order; the workgroups of a column block leave [chunk][M][N] for the consumer
//     to add in chunk order.
//   * v_mfma_f64_16x16x4_f64 wants A[row = lane % 16][k = lane / 16] and B[k = lane / 16]
//     [col = lane % 16] of a lane.  Which four k one instruction contracts is free as long as
//     both operands agree: a lane loads A[row][k0 + 2 q], A[row][k0 + 2 q + 1] (q = lane / 16)
//     with one 16-byte load and the two B elements of the same k, and a stage of 8 k is two
//     instructions per row block, one on the even and one on the odd k.
//   * Rounds of four stages alternate between two register sets, the next round's loads in
//     flight while this one's MFMAs run.  Stages beyond a wavefront's range are loaded from an
//     offset beyond the buffer resources' range (zeros, no traffic), as are columns beyond N,
//     rows beyond M and B's k beyond K; A's k beyond K (the next row) is masked.
constexpr int kRoundStages = 4;   // stages of 8 k per round and wavefront

template <int RB>
__global__ __launch_bounds__(256)
void skinny_f64_kernel(int M, int N, int K, const double* __restrict__ A, int lda,
                       const double* __restrict__ B, int ldb, double* __restrict__ part, int k_per_wg) {
  __shared__ double red[3][RB][4][64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int c = lane & 15, q = lane >> 4;
  const int n0 = blockIdx.x * 16;
  const int kb = blockIdx.y * k_per_wg;
  const int ke = kb + k_per_wg < K ? kb + k_per_wg : K;
  const int kw = k_per_wg / 4;  // a multiple of 8
  const int kws = kb + wave * kw;
  const int kwe = kws + kw < ke ? kws + kw : ke;  // <= kws: a wavefront without work

  const __amdgpu_buffer_rsrc_t pa = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<double*>(A), 0, (int)(((long long)(M - 1) * lda + K) * 8), 0x00020000);
  const __amdgpu_buffer_rsrc_t pb = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<double*>(B), 0, (int)(((long long)(K - 1) * ldb + N) * 8), 0x00020000);
  unsigned int a_voff[RB];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) a_voff[rb] = (unsigned int)(((16 * rb + c) * lda + 2 * q) * 8);
  const unsigned int b_voff = n0 + c < N ? (unsigned int)((2 * q * ldb + n0 + c) * 8) : kNowhere;
  const unsigned int b_next = (unsigned int)(ldb * 8);

  double2_t a[2][kRoundStages][RB];
  double b[2][kRoundStages][2];
  double4_t acc[RB];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) acc[rb] = double4_t{0.0, 0.0, 0.0, 0.0};

  auto request = [&](auto set_c, int k_first) {
    constexpr int SET = decltype(set_c)::value;
#pragma unroll
    for (int s = 0; s < kRoundStages; ++s) {
      const int k0 = k_first + 8 * s;
      const bool in = k0 < kwe;  // the same for a whole wavefront
      unsigned int ob = in ? b_voff : kNowhere, ob1 = in ? b_voff + b_next : kNowhere;
      asm volatile("" : "+v"(ob), "+v"(ob1));
      b[SET][s][0] = __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(pb, ob, k0 * ldb * 8, 0));
      b[SET][s][1] = __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(pb, ob1, k0 * ldb * 8, 0));
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) {
        unsigned int oa = in ? a_voff[rb] : kNowhere;
        asm volatile("" : "+v"(oa));
        a[SET][s][rb] = __builtin_bit_cast(double2_t, __builtin_amdgcn_raw_buffer_load_b128(pa, oa, k0 * 8, 0));
      }
    }
  };
  auto multiply = [&](auto set_c, int k_first) {
    constexpr int SET = decltype(set_c)::value;
#pragma unroll
    for (int s = 0; s < kRoundStages; ++s) {
      const int left = K - (k_first + 8 * s + 2 * q);  // of this lane's two k, how many exist
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) {
        const double a0 = left > 0 ? a[SET][s][rb][0] : 0.0;
        acc[rb] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b[SET][s][0], acc[rb], 0, 0, 0);
      }
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) {
        const double a1 = left > 1 ? a[SET][s][rb][1] : 0.0;
        acc[rb] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b[SET][s][1], acc[rb], 0, 0, 0);
      }
    }
  };
  using Set0 = std::integral_constant<int, 0>;
  using Set1 = std::integral_constant<int, 1>;
  constexpr int kRound = 8 * kRoundStages;
  request(Set0{}, kws);
  for (int k = kws; k < kwe; k += 2 * kRound) {
    request(Set1{}, k + kRound);
    multiply(Set0{}, k);
    if (k + kRound >= kwe) break;
    request(Set0{}, k + 2 * kRound);
    multiply(Set1{}, k + kRound);
  }

  if (wave > 0) {
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
      for (int e = 0; e < 4; ++e) red[wave - 1][rb][e][lane] = acc[rb][e];
  }
  __syncthreads();
  if (wave > 0 || n0 + c >= N) return;
  double* out = part + (size_t)blockIdx.y * M * N + n0 + c;
#pragma unroll
  for (int rb = 0; rb < RB; ++rb)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int row = 16 * rb + 4 * e + q;
      const double sum = ((acc[rb][e] + red[0][rb][e][lane]) + red[1][rb][e][lane]) + red[2][rb][e][lane];
      if (row < M) out[(size_t)row * N] = sum;
    }
}

// k_per_wg: 256 (a wavefront then has two rounds, everything in flight at once) unless that
// leaves CUs without a workgroup (then 128), and never more than 8 chunks for the consumer.
void plan_skinny_f64(int M, int N, int K, int* chunks, int* k_per_wg) {
  (void)M;
  const int cus = device_cu_count() > 0 ? device_cu_count() : 256;
  const long long col_blocks = (N + 15) / 16;
  int per = 256;
  if (col_blocks * ((K + 255) / 256) < cus) per = 128;
  const int least = ((K + 7) / 8 + 31) / 32 * 32;  // at most 8 chunks
  if (per < least) per = least;
  const int whole = (K + 31) / 32 * 32;
  if (per > whole) per = whole;
  *k_per_wg = per;
  *chunks = (K + per - 1) / per;
}

// The operands fit the 32-bit byte offsets of a buffer resource.
int panels_fit(bool trans_a, int M, int N, int K, int lda, int ldb) {
  const long long a = trans_a ? (long long)K * lda + M : (long long)M * lda + K, b = (long long)K * ldb + N;
  return a * 8 < (1ll << 31) - 64 && b * 8 < (1ll << 31) - 64 ? 1 : 0;
}

bool skinny_f64_applies(int M, int N, int K, int lda, int ldb) {
  return M <= 64 && ((long long)M * lda + K) * 8 < (1ll << 31) - 64 && ((long long)K * ldb + N) * 8 < (1ll << 31) - 64 &&
         (long long)ldb * 8 < (1ll << 28);
}

}  // namespace

// *need: what a product takes at least (its chunks, where a consumer adds them); *wish: with the pieces of a cut one.
void gemm_f64_scratch_bytes(int M, int N, int K, size_t* need, size_t* wish) {
  *need = *wish = 0;
  if (M <= 0 || N <= 0 || K <= 0) return;
  const F64Plan chunked = plan_f64_chunks(M, N, K);
  if (chunked.pieces > 1) *need = (size_t)chunked.pieces * M * N * sizeof(double);
  if (M <= 64) {
    int pieces, per;
    plan_skinny_f64(M, N, K, &pieces, &per);
    const size_t skinny = (size_t)pieces * M * N * sizeof(double);
    *need = *need > skinny ? *need : skinny;
  }
  const size_t cut = f64_piece_bytes(plan_f64(M, N, K), M, N);
  *wish = *need > cut ? *need : cut;
}

// The partial results of a cut product lie `scratch_offset` bytes (a multiple of 16) into the
// stream's scratch buffer.
int gemm_f64(hipStream_t stream, bool trans_a, int M, int N, int K, const double* A, int lda,
             const double* B, int ldb, double* C, int ldc, bool accumulate, size_t scratch_offset) {
  HASTE_HIP_REQUIRE(M > 0 && N > 0 && K > 0 && A && B && C);
  HASTE_HIP_REQUIRE(lda >= (trans_a ? M : K) && ldb >= N && ldc >= N);
  const int tiles_n = (N + DN - 1) / DN;
  const long long tiles = (long long)((M + DM - 1) / DM) * tiles_n;
  HASTE_HIP_REQUIRE(tiles < (1ll << 30));
  F64Plan plan = plan_f64(M, N, K);
  double* part = nullptr;
  if (plan.pieces > 1) {  // not cut without room for the pieces (a caller's own buffer, a capture, a buffer in use)
    const size_t bytes = scratch_offset + f64_piece_bytes(plan, M, N);
    bool room = false;
    if (scratch_offset == 0) HASTE_HIP_PROPAGATE(workspace_has_room(stream, bytes, &room));
    Workspace ws;
    HASTE_HIP_PROPAGATE(get_workspace(stream, room ? bytes : 0, &ws));
    if (ws.scratch_bytes >= bytes) part = reinterpret_cast<double*>(reinterpret_cast<char*>(ws.scratch) + scratch_offset);
    else plan = F64Plan{(int)tiles, 1, K};
  }
  const int rest = (int)(tiles - plan.whole);
  HASTE_HIP_REQUIRE(rest == 0 || part != nullptr);  // a tile that is not whole is parked
  const dim3 grid((unsigned)(plan.whole + (long long)rest * plan.pieces));
  ScopedKernelTimer timer("gemm_f64", stream);
  if (trans_a)
    gemm_f64_kernel<true><<<grid, dim3(256), 0, stream>>>(M, N, K, A, lda, B, ldb, C, ldc, accumulate, plan, tiles_n, part, 0,
                                                          panels_fit(true, M, N, K, lda, ldb));
  else
    gemm_f64_kernel<false><<<grid, dim3(256), 0, stream>>>(M, N, K, A, lda, B, ldb, C, ldc, accumulate, plan, tiles_n, part, 0,
                                                           panels_fit(false, M, N, K, lda, ldb));
  HASTE_HIP_TRY(hipGetLastError());
  if (rest > 0) {
    gemm_f64_reduce_kernel<<<dim3((unsigned)rest, DM / kReduceRows), dim3(256), 0, stream>>>(M, N, plan, tiles_n, part, C, ldc,
                                                                                     accumulate ? 1 : 0);
    HASTE_HIP_TRY(hipGetLastError());
  }
  return HASTE_HIP_OK;
}

// The product left as chunks of its contraction, [chunk][M][N] in the stream's scratch buffer,
// for a consumer that adds them itself in chunk order (one launch less per step than adding
// them here); *chunks == 0, and nothing launched, when the product is not cut.  Valid until the
// next product on the stream.
int gemm_f64_chunks(hipStream_t stream, int M, int N, int K, const double* A, int lda, const double* B,
                    int ldb, size_t scratch_offset, const double** partial, int* chunks) {
  *chunks = 0;
  HASTE_HIP_REQUIRE(M > 0 && N > 0 && K > 0 && A && B);
  HASTE_HIP_REQUIRE(lda >= K && ldb >= N);
  int pieces, per = 0;
  const bool skinny = skinny_f64_applies(M, N, K, lda, ldb);
  const F64Plan plan = plan_f64_chunks(M, N, K);
  if (skinny) plan_skinny_f64(M, N, K, &pieces, &per);
  else pieces = plan.pieces;
  if (!skinny && pieces <= 1) return HASTE_HIP_OK;
  Workspace ws;
  HASTE_HIP_PROPAGATE(get_workspace(stream, scratch_offset + (size_t)pieces * M * N * sizeof(double), &ws));
  double* part = reinterpret_cast<double*>(reinterpret_cast<char*>(ws.scratch) + scratch_offset);
  if (skinny) {
    const dim3 grid((unsigned)((N + 15) / 16), (unsigned)pieces);
    ScopedKernelTimer timer("gemm_f64_skinny", stream);
    if (M <= 16) skinny_f64_kernel<1><<<grid, dim3(256), 0, stream>>>(M, N, K, A, lda, B, ldb, part, per);
    else if (M <= 32) skinny_f64_kernel<2><<<grid, dim3(256), 0, stream>>>(M, N, K, A, lda, B, ldb, part, per);
    else skinny_f64_kernel<4><<<grid, dim3(256), 0, stream>>>(M, N, K, A, lda, B, ldb, part, per);
    HASTE_HIP_TRY(hipGetLastError());
  } else {
    const int tiles_n = (N + DN - 1) / DN;
    const dim3 grid((unsigned)((M + DM - 1) / DM * tiles_n * pieces));
    ScopedKernelTimer timer("gemm_f64", stream);
    gemm_f64_kernel<false><<<grid, dim3(256), 0, stream>>>(M, N, K, A, lda, B, ldb, nullptr, 0, 0, plan, tiles_n, part, 1,
                                                           panels_fit(false, M, N, K, lda, ldb));
    HASTE_HIP_TRY(hipGetLastError());
  }
  *partial = part;
  *chunks = pieces;
  return HASTE_HIP_OK;
}

}  // namespace haste_hip

extern "C" int haste_hip_gemm_f64(int trans_a, int M, int N, int K, const double* A, int lda,
                                  const double* B, int ldb, double* C, int ldc, int accumulate,
                                  void* stream) {
  return haste_hip::gemm_f64(haste_hip::as_stream(stream), trans_a != 0, M, N, K, A, lda, B, ldb,
                             C, ldc, accumulate != 0, 0);
}
