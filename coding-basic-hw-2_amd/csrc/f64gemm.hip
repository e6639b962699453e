// f64gemm.hip -- grouped native FP64 GEMM on gfx950 MFMA: C = alpha A B + beta C, column-major,
// no transpose.  Replaces the reference's cuBLAS calls for its native routes (K_ZERO, ALPHA_ZERO,
// K_TOO_LARGE, SMALL_K, TINY, UNPROFITABLE, PRECISION) and the two native paths
// (src/ggemm.cu:102-184, src/ggemm_graph.cu:88-102).
//
// One launch per group: output tiles of all problems in one table, workgroup b takes tile b.  One tile
// shape per group (f64_build_schedule):
//   128 x 128: 4 waves, 4 x 4 blocks of 16 x 16 each, 64 KB of LDS, two workgroups per compute unit:
//            half the operand traffic per flop of the next and four times the MFMA work per fragment
//            read -- groups that fill their rounds;
//   64 x 64: 2 x 2 blocks per wave, 32 KB of LDS, five workgroups per compute unit -- the others;
//   16 x 128, 32 x 128: groups of problems with at most 16 / 32 rows, which stream B once;
//   32 x 32: one block per wave (f64_chain_kernel) -- few outputs, where one chain per wave is what
//            fills the GPU.
// A wave owns the 16-row and 16-column blocks of its tile in turn with the other waves, so the blocks
// of a tile that hangs over the problem's edge are dealt evenly and the ones outside are skipped.
// Every output entry takes the same k-ordered chain of MFMAs (zero-padded beyond k) at every shape, so
// all give bit-identical results.  Descriptors live in device memory, so a captured graph replays
// with new pointers after one small H2D.
//
// What bounds it: the FP64 matrix cores, 64 cycles per v_mfma_f64_16x16x4 (75 TFLOP/s measured on
// register operands); thin groups, HBM; 32 x 32 tiles, the chain's latency.  Measured before -> after
// B's stages came in as whole 128-byte lines, partial tiles loaded without a test per element and
// skipped their outside blocks, neighbouring tiles shared an XCD's L2 and a workgroup's priority rose
// with its progress (same GPU): 64 x 1024^3, beta 0.5, 2.29 -> 2.18 ms (63 TFLOP/s), 96 x 679x600x515
// 1.11 -> 0.78 ms, 1024 thin panels (5 or 14 rows, 128 columns, k about 880) 0.317 -> 0.217 ms
// (4.5 TB/s); on 32 x 32 tiles 500x500x60000 3.95 -> 0.73 ms, 3 x 209x197x10380 0.69 -> 0.13 ms.
// BLAS semantics: alpha == 0 or k == 0 never reads A or B; beta == 0 never reads C.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <type_traits>

#include "common.hpp"

namespace ggemm {
namespace {

typedef double v4d __attribute__((ext_vector_type(4)));
typedef double v2d __attribute__((ext_vector_type(2)));
// global address space: the descriptor pointers would otherwise compile to flat loads, which also
// count in lgkmcnt, so every LDS fragment wait would wait for the next stage's prefetch as well
#define GLOBAL __attribute__((address_space(1)))
constexpr int kThreads = 256;
constexpr int kBK = 16;

// LDS positions without padding.  A tile, k-major: row c of k row k, 16-row blocks XOR-swizzled by
// k mod 4, so that the four k rows a fragment read touches fall into different banks (a tile of one or
// two blocks needs less).  B tile, in 16-deep k groups, column-major inside a group (the 16 k of a
// column are one 128-byte line, stored by eight lanes two k each): 16-byte pairs XOR-swizzled by the
// column, so that a fragment read (16 columns, the 32 bytes of 4 k each) covers every bank evenly.
template <int W>
__device__ __forceinline__ int swa(int k, int c) {
  return W >= 64 ? c ^ (k & 3) << 4 : W == 32 ? c ^ (k & 1) << 4 : c;
}
template <int W>
__device__ __forceinline__ int swb(int k, int c) {
  return (k >> 4) * (W * 16) + c * 16 + ((((k & 15) >> 1) ^ (c & 7)) << 1 | (k & 1));
}

// Workgroup -> tile: the dispatcher deals consecutive workgroups to the XCDs in turn, so chunks of
// 32 consecutive tiles (which share operand panels) go to one XCD's L2.  The tiles come longest first,
// so the chunks' order turns from one round of chunks to the next.
__device__ __forceinline__ int tile_of(int b, int total) {
  constexpr int kChunk = 32;
  const int super = b / (kXcds * kChunk) * (kXcds * kChunk);
  if (super + kXcds * kChunk > total) return b;
  const int i = b - super;
  return super + ((i + b / (kXcds * kChunk)) % kXcds) * kChunk + i / kXcds;
}

// The problem of a tile and the tile's index in it.
struct TileRef {
  int problem, local;
};
__device__ __forceinline__ TileRef find_tile(const int* __restrict__ sched, int block) {
  const int tile = tile_of(block, sched[0]);
  const int ne = sched[1];
  const int* prefix = sched + kSchedHdr;
  const int* entry = prefix + ne + 1;
  int lo = 0;
  if (const int per = sched[2]) {   // equal tile counts
    lo = tile / per;
  } else {
    int hi = ne - 1;
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (prefix[mid] <= tile) lo = mid; else hi = mid - 1;
    }
  }
  return TileRef{entry[lo] >> 2, tile - prefix[lo]};
}

// Stages of BK k of a BM x BN tile's operands, HBM to LDS through the registers of 256 threads.  Thread
// t: A elements (ar, ak + KSA q); B elements (bk, bk + 1) of column bc + 32 c and 16-deep k group g,
// q = c + CP g, eight lanes to a column's 128 bytes of the group (one request per line: a thread per
// 64-byte run of a column came back to each line four times, and the lines of a compute unit's
// workgroups do not fit its L1).  Rows and columns past the problem read its last one (their outputs
// are not stored), so only a stage that crosses k needs a test per element.
template <int BM, int BN, int BK>
struct Loader {
  static constexpr int KSA = kThreads / BM, NA = BK / KSA, NB = BN * BK / (2 * kThreads), CP = BN / 32;
  struct Regs {
    double a[NA], b[NB][2];
  };
  const GLOBAL double* Ag;
  const GLOBAL double* Bg[CP];
  size_t lda;
  int k, ar, ak, bc, bk;
  __device__ __forceinline__ void init(const F64Problem& P, int row0, int col0, int t) {
    ar = t % BM, ak = t / BM;
    bc = t / 8, bk = (t % 8) * 2;
    k = P.k;
    lda = (size_t)P.lda;
    Ag = (const GLOBAL double*)P.A + min(row0 + ar, P.m - 1);
#pragma unroll
    for (int c = 0; c < CP; ++c)
      Bg[c] = (const GLOBAL double*)P.B + (size_t)min(col0 + bc + 32 * c, P.n - 1) * (size_t)P.ldb;
  }
  __device__ __forceinline__ void load(Regs& r, int kt) const {
    const int k0 = kt * BK;
    if (k - k0 >= BK) {
      const GLOBAL double* pa = Ag + (size_t)(k0 + ak) * lda;
#pragma unroll
      for (int q = 0; q < NA; ++q) r.a[q] = pa[(size_t)(KSA * q) * lda];
#pragma unroll
      for (int q = 0; q < NB; ++q) {
        r.b[q][0] = Bg[q % CP][k0 + 16 * (q / CP) + bk];
        r.b[q][1] = Bg[q % CP][k0 + 16 * (q / CP) + bk + 1];
      }
      return;
    }
#pragma unroll
    for (int q = 0; q < NA; ++q) {
      const int kk = k0 + ak + KSA * q;
      const double v = Ag[(size_t)min(kk, k - 1) * lda];
      r.a[q] = kk < k ? v : 0.0;
    }
#pragma unroll
    for (int q = 0; q < 2 * NB; ++q) {
      const int kk = k0 + 16 * (q / 2 / CP) + bk + (q & 1);
      const double v = Bg[q / 2 % CP][min(kk, k - 1)];
      r.b[q / 2][q & 1] = kk < k ? v : 0.0;
    }
  }
  __device__ __forceinline__ void store(const Regs& r, double (&sA)[BK][BM], double (&sB)[BK * BN]) const {
#pragma unroll
    for (int q = 0; q < NA; ++q) sA[ak + KSA * q][swa<BM>(ak + KSA * q, ar)] = r.a[q];
#pragma unroll
    for (int q = 0; q < NB; ++q)
      *reinterpret_cast<v2d*>(&sB[swb<BN>(16 * (q / CP) + bk, bc + 32 * (q % CP))]) = v2d{r.b[q][0], r.b[q][1]};
  }
};

// BM x BN tile, WM waves along the rows and 4 / WM along the columns, OCC workgroups per compute unit
template <int BM, int BN, int WM, int OCC>
__global__ void __launch_bounds__(kThreads, OCC) f64_grouped_kernel(const F64Problem* __restrict__ probs,
                                                                 const int* __restrict__ sched) {
  constexpr int WN = 4 / WM;
  constexpr int FM = BM / (16 * WM), FN = BN / (16 * WN);   // 16 x 16 blocks per wave
  constexpr int BK = kBK;
  __shared__ double sA[2][BK][BM];
  __shared__ __align__(16) double sB[2][BK * BN];
  const TileRef t = find_tile(sched, blockIdx.x);
  const F64Problem P = probs[t.problem];
  const int local = t.local;
  const int tiles_m = ceil_div(P.m, BM);
  const int row0 = (local % tiles_m) * BM, col0 = (local / tiles_m) * BN;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave % WM, wn = wave / WM;
  // this wave's blocks inside the problem: block i covers rows row0 + 16 (WM i + wm) ..
  const int nbm = min(FM, ceil_div(max(0, P.m - row0 - 16 * wm), 16 * WM));
  const int nbn = min(FN, ceil_div(max(0, P.n - col0 - 16 * wn), 16 * WN));

  v4d acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = v4d{0.0, 0.0, 0.0, 0.0};

  const bool compute = P.alpha != 0.0 && P.k > 0;
  if (compute) {
    Loader<BM, BN, BK> ld;
    ld.init(P, row0, col0, tid);
    const int nk = ceil_div(P.k, BK);
    const int fr = lane & 15, fk = lane >> 4;
    // The product is taken transposed (B's columns as the MFMA rows), so that a lane's four results
    // are four columns of one row and 16 lanes store 16 consecutive rows of a column: 128-byte
    // segments of C.
    auto loop = [&](auto edge) {
      constexpr bool kEdge = decltype(edge)::value;
      // step s of the stage in buffer st: k = 4 s .. 4 s + 3
      auto step = [&](int st, int s) {
        double a[FM], b[FN];
#pragma unroll
        for (int i = 0; i < FM; ++i) a[i] = sA[st][4 * s + fk][swa<BM>(fk, (WM * i + wm) * 16 + fr)];
#pragma unroll
        for (int j = 0; j < FN; ++j) b[j] = sB[st][swb<BN>(4 * s + fk, fr) + (WN * j + wn) * 256];
#pragma unroll
        for (int i = 0; i < FM; ++i) {
          if (kEdge && i >= nbm) break;
#pragma unroll
          for (int j = 0; j < FN; ++j) {
            if (kEdge && j >= nbn) break;
            acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(b[j], a[i], acc[i][j], 0, 0, 0);
          }
        }
      };
      typename Loader<BM, BN, BK>::Regs r;
      ld.load(r, 0);
      ld.store(r, sA[0], sB[0]);
      __syncthreads();
      const int quarter = nk >> 2;
      for (int kt = 0; kt < nk; ++kt) {
        // a workgroup's priority rises with its progress: the ones sharing a compute unit drift apart,
        // and one's epilogue and prologue run under the others' MFMAs
        if (kt == quarter) __builtin_amdgcn_s_setprio(1);
        if (kt == 2 * quarter) __builtin_amdgcn_s_setprio(2);
        if (kt == 3 * quarter) __builtin_amdgcn_s_setprio(3);
        const int st = kt & 1;
        if (kt + 1 < nk) ld.load(r, kt + 1);
#pragma unroll
        for (int s = 0; s < BK / 4; ++s) step(st, s);
        if (kt + 1 < nk) ld.store(r, sA[st ^ 1], sB[st ^ 1]);
        __syncthreads();
      }
    };
    if (nbm == FM && nbn == FN)
      loop(std::false_type{});
    else
      loop(std::true_type{});
  }

  // D block layout of v_mfma_f64_16x16x4f64: lane l, register r -> MFMA row 4 r + l / 16, column
  // l % 16 (four single-row groups; the INT8 / F32 16 x 16 instructions use four consecutive rows
  // instead); transposed, so lane l, register r holds C row l % 16, column 4 r + l / 16 of the block.
  // With beta != 0 the C0 values of a batch of blocks are all loaded before the batch's stores:
  // entry by entry, each C0 load waited for its data before the store (the stores might alias
  // the next loads), one memory round trip per entry.
  // C0 rows and columns past the problem are read from its last one, so the loads need no test.  The
  // product by alpha is rounded, the one by beta fused, at every shape.
  const size_t ldc = (size_t)P.ldc;
  GLOBAL double* const Cg = (GLOBAL double*)P.C;
  const bool rd = P.beta != 0.0;
  constexpr int NBLK = FM * FN, BATCH = NBLK < 8 ? NBLK : 8;
  auto epilogue = [&](auto inside) {
    constexpr bool kInside = decltype(inside)::value;   // the whole tile
#pragma unroll
    for (int b0 = 0; b0 < NBLK; b0 += BATCH) {
      double c0[BATCH][4];
      if (rd) {
#pragma unroll
        for (int q = 0; q < BATCH; ++q) {
          const int i = (b0 + q) / FN, j = (b0 + q) % FN;
          const int row = row0 + (WM * i + wm) * 16 + (lane & 15), rc = kInside ? row : min(row, P.m - 1);
          const int cbase = col0 + (WN * j + wn) * 16 + (lane >> 4);
#pragma unroll
          for (int r = 0; r < 4; ++r)
            c0[q][r] = Cg[(size_t)rc + (size_t)(kInside ? cbase + 4 * r : min(cbase + 4 * r, P.n - 1)) * ldc];
        }
      }
#pragma unroll
      for (int q = 0; q < BATCH; ++q) {
        const int i = (b0 + q) / FN, j = (b0 + q) % FN;
        const int row = row0 + (WM * i + wm) * 16 + (lane & 15);
        const int cbase = col0 + (WN * j + wn) * 16 + (lane >> 4);
        if (!kInside && row >= P.m) continue;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int col = cbase + 4 * r;
          if (!kInside && col >= P.n) continue;
          const double ab = compute ? P.alpha * acc[i][j][r] : 0.0;
          Cg[(size_t)row + (size_t)col * ldc] = !rd ? ab : (compute ? __builtin_fma(P.beta, c0[q][r], ab) : P.beta * c0[q][r]);
        }
      }
    }
  };
  if (P.m - row0 >= BM && P.n - col0 >= BN)
    epilogue(std::true_type{});
  else
    epilogue(std::false_type{});
}

// Few outputs (32 x 32 tiles, 512 threads): waves 0-3 run one
// accumulator chain each -- 16 x 16 outputs, the whole k -- and waves 4-7, one beside each on its SIMD,
// stream the operands in stages of BK k, two stages ahead in registers.  The time is that of the chain's
// k / 4 dependent MFMAs: 64 cycles of the matrix core each, 103 as measured (500x500x60000, 0.73 ms) -- the
// loader wave's address arithmetic and LDS stores issue on the same SIMD, and a stage's first fragments are
// read after its barrier.  Compute waves that load for themselves take 145 (64x64x90000 1.42 against 1.01 ms).
constexpr int kChainTile = 32;
template <int BK>
__global__ void __launch_bounds__(2 * kThreads, 2) f64_chain_kernel(const F64Problem* __restrict__ probs,
                                                                  const int* __restrict__ sched) {
  constexpr int T = kChainTile;
  __shared__ double sA[2][BK][T];
  __shared__ __align__(16) double sB[2][BK * T];
  const TileRef t = find_tile(sched, blockIdx.x);
  const F64Problem P = probs[t.problem];
  const int tiles_m = ceil_div(P.m, T);
  const int row0 = (t.local % tiles_m) * T, col0 = (t.local / tiles_m) * T;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const bool compute = P.alpha != 0.0 && P.k > 0;
  const int nk = compute ? ceil_div(P.k, BK) : 0;
  if (wave >= 4) {
    if (!compute) return;
    Loader<T, T, BK> ld;
    ld.init(P, row0, col0, tid - kThreads);
    typename Loader<T, T, BK>::Regs r0, r1;
    ld.load(r0, 0);
    if (nk > 1) ld.load(r1, 1);
    ld.store(r0, sA[0], sB[0]);
    __syncthreads();
    for (int kt = 0; kt < nk; kt += 2) {   // stage kt + 1 to LDS while stage kt is multiplied
      if (kt + 2 < nk) ld.load(r0, kt + 2);
      if (kt + 1 < nk) ld.store(r1, sA[1], sB[1]);
      __syncthreads();
      if (kt + 1 >= nk) break;
      if (kt + 3 < nk) ld.load(r1, kt + 3);
      if (kt + 2 < nk) ld.store(r0, sA[0], sB[0]);
      __syncthreads();
    }
    return;
  }
  const int wm = wave & 1, wn = wave >> 1;
  const int row = row0 + 16 * wm + (lane & 15), cbase = col0 + 16 * wn + (lane >> 4);
  v4d acc = v4d{0.0, 0.0, 0.0, 0.0};
  if (compute) {
    const int fr = lane & 15, fk = lane >> 4;
    auto step = [&](int st, int s) {
      const double a = sA[st][4 * s + fk][swa<T>(fk, 16 * wm + fr)];
      const double b = sB[st][swb<T>(4 * s + fk, fr) + 256 * wn];
      acc = __builtin_amdgcn_mfma_f64_16x16x4f64(b, a, acc, 0, 0, 0);   // transposed, as above
    };
    __builtin_amdgcn_s_setprio(3);
    __syncthreads();
    for (int kt = 0; kt < nk; ++kt) {
      const int left = P.k - kt * BK;
      if (left > BK - 4) {
#pragma unroll
        for (int s = 0; s < BK / 4; ++s) step(kt & 1, s);
      } else {
#pragma unroll 4
        for (int s = 0; 4 * s < left; ++s) step(kt & 1, s);
      }
      __syncthreads();
    }
    // the other shapes run zeros up to a multiple of 16 k; all they can change is a chain of -0 (negative
    // products that underflow), which the +0 of a padded step turns into +0
    if (P.k % kBK != 0 && P.k % kBK <= kBK - 4) acc = acc + v4d{0.0, 0.0, 0.0, 0.0};
  }
  const size_t ldc = (size_t)P.ldc;
  GLOBAL double* const Cg = (GLOBAL double*)P.C;
  const bool rd = P.beta != 0.0;
  double c0[4];
#pragma unroll
  for (int r = 0; r < 4; ++r)
    c0[r] = (rd && row < P.m && cbase + 4 * r < P.n) ? Cg[(size_t)row + (size_t)(cbase + 4 * r) * ldc] : 0.0;
  if (row >= P.m) return;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    if (cbase + 4 * r >= P.n) continue;
    const double ab = compute ? P.alpha * acc[r] : 0.0;
    Cg[(size_t)row + (size_t)(cbase + 4 * r) * ldc] = !rd ? ab : (compute ? __builtin_fma(P.beta, c0[r], ab) : P.beta * c0[r]);
  }
}

constexpr int kCus = 256;
// log2 of the tile sizes: a group's tiles are counted for every shape, per problem and call, and divisions
// took a sixth of the schedule's time (host, 20000 problems 1.22 ms, 1024 53 us; with shifts 1.05 and 45)
struct F64Shape {
  int bm, bn;
};
constexpr F64Shape kShapes[kF64Shapes] = {{6, 6}, {7, 7}, {4, 7}, {5, 7}, {5, 5}, {5, 5}};

inline long long tiles_of(const F64Problem& p, const F64Shape& t) {   // m, n >= 1
  return (long long)(((p.m - 1) >> t.bm) + 1) * (((p.n - 1) >> t.bn) + 1);
}

}  // namespace

int f64_build_schedule(const F64Problem* h, int num, void* h_ws, size_t ws_bytes, int* launch, size_t* bytes_used,
                       int tile_mode) {
  if (num < 0 || (num > 0 && !h) || !h_ws || !launch) return 1;
  if (ws_bytes < sched_bytes(num)) return 2;
  // problems with outputs, longest k first (ties by index: the order a stable sort keeps), sorted
  // in place in the image's entry array -- no host scratch
  int* img = static_cast<int*>(h_ws);
  size_t ne = 0;
  for (int i = 0; i < num; ++i) ne += h[i].m > 0 && h[i].n > 0;
  int* prefix = img + kSchedHdr;
  int* entry = prefix + ne + 1;
  int mmax = 0, kmax = 0;
  long long tiles[kF64Shapes] = {};
  double work128 = 0, workc = 0, area = 0;
  for (int i = 0, j = 0; i < num; ++i) {
    const F64Problem& p = h[i];
    if (p.m <= 0 || p.n <= 0) continue;
    entry[j++] = i;
    mmax = std::max(mmax, p.m);
    const int k = p.alpha == 0.0 ? 0 : p.k;
    kmax = std::max(kmax, k);
    tiles[kF64Tile64] += tiles_of(p, kShapes[kF64Tile64]);
    tiles[kF64Tile16] += tiles_of(p, kShapes[kF64Tile16]);
    tiles[kF64Tile32] += tiles_of(p, kShapes[kF64Tile32]);
    const long long t128 = tiles_of(p, kShapes[kF64Tile128]), tc = tiles_of(p, kShapes[kF64TileChain]);
    tiles[kF64Tile128] += t128;
    tiles[kF64TileChain] += tc;
    work128 += (double)t128 * k;
    workc += (double)tc * k;
    area += (double)p.m * p.n;
  }
  std::sort(entry, entry + ne, [h](int a, int b) {
    const int ka = std::max(h[a].k, 1), kb = std::max(h[b].k, 1);
    return ka != kb ? ka > kb : a < b;
  });

  // Tile shape.  Microseconds per 16 k, measured on groups of 1 to 3000 tiles: a round of 32 x 32 tiles
  // (one per compute unit) 0.22 with 128-deep stages, 0.20 with 64-deep ones, of 64 x 64 tiles 0.58 but at
  // least 0.85 in all, of the thin ones 1.0 but at least 1.2 (their problems differ in k, and then a round
  // of 32 x 32 ones takes 0.4).  128 x 128 (67 TFLOP/s on long k against 61 of the 64 x 64 tiles) when little
  // of the tiles hangs over the problems' edges and their rounds of two workgroups per compute unit are
  // nearly filled: a short last round leaves compute units idle for as long as a full one, unless it has
  // at most one tile for each.  At most one tile per compute unit in all stays on 64 x 64 tiles, four
  // workgroups of which hide each other's waits: 2048^2 x 2048 323 against 297 us, x 64 23.9 / 21.4,
  // 16 x 512^3 91 / 84.
  int shape = tile_mode == 128 ? kF64Tile128 : kF64Tile64;
  if (tile_mode == 0 && kmax > 0) {
    auto rounds = [&](int s) { return std::ceil((double)tiles[s] / kCus); };
    // 32 x 32 tiles: a grid has fewer than 2^32 threads, and these tiles take twice as many each.  Past the
    // two workgroups per compute unit that run at once, each further round costs about 1 us before its first
    // MFMA, which only a longer k makes up for -- 32 (mean over the tiles) for each round, 384 whatever the
    // rounds.  Below the line, us at 32 x 32 against the shape taken: 2000 x 8x8x16 16.8 / 13.4,
    // 1000 x 30x60x128 33.8 / 24.6, 600 x 96x96x16 43 / 21, 300 x 96x96x300 71 / 68; above: 71 x 96x96x128
    // 16.0 / 19.1, 222 x 96x96x256 40.5 / 46.2, 300 x 96x96x400 70 / 82, 5000 x 32x32x400 210 / 217.
    const double crounds = rounds(kF64TileChain);
    const bool small = tiles[kF64TileChain] < (1LL << 32) / (2 * kThreads) &&
                       (crounds <= 2.0 || workc >= std::min(32.0 * crounds, 384.0) * tiles[kF64TileChain]);
    if (mmax <= 32) {
      const int thin = mmax <= 16 ? kF64Tile16 : kF64Tile32;
      shape = small && 0.4 * crounds < std::max(1.2, 1.0 * rounds(thin)) ? kF64TileChain : thin;
    } else if (small && 0.22 * crounds < std::max(0.85, 0.58 * rounds(kF64Tile64))) {
      shape = kF64TileChain;
    } else if (area >= 0.95 * 16384.0 * tiles[kF64Tile128]) {
      const double share = work128 / kmax / (2.0 * kCus);
      const double full = std::floor(share), left = share - full;
      if (share >= 0.87 * (full + (left <= 0.0 ? 0.0 : left <= 0.5 && full > 0.0 ? 0.5 : 1.0))) shape = kF64Tile128;
    }
  }
  // 32 x 32 tiles: 128-deep stages, one workgroup per compute unit, or 64-deep ones and two of them, when
  // there is more than a tile for each (3 x 300x300x4096: 106 -> 91 us) or k is too short for the long
  // stages' start-up (3 x 300x300x100 19.2 -> 14.8; 500x500x512 18, 500x500x4096 58 against 64 us)
  if (shape == kF64TileChain && (tiles[kF64TileChain] > kCus || kmax <= 512)) shape = kF64TileShort;
  const F64Shape t = kShapes[shape];
  const long long per = ne ? tiles_of(h[entry[0]], t) : 0;
  long long tot = 0;
  bool equal = true;
  for (size_t j = 0; j < ne; ++j) {
    const long long n = tiles_of(h[entry[j]], t);
    prefix[j] = (int)tot;
    tot += n;
    if (tot > kF64MaxTiles) return 5;
    equal = equal && n == per;
  }
  prefix[ne] = (int)tot;
  std::memset(img, 0, sizeof(int) * kSchedHdr);
  img[0] = (int)tot;
  img[1] = (int)ne;
  img[2] = equal ? (int)per : 0;
  for (size_t j = 0; j < ne; ++j) entry[j] <<= 2;
  *launch = tot == 0 ? 0 : (int)tot | shape << kF64ShapeBit;
  if (bytes_used) *bytes_used = sizeof(int) * (kSchedHdr + 2 * ne + 1);
  return 0;
}

int f64_launch(const F64Problem* d_probs, const void* d_sched, int launch, hipStream_t s) {
  if (launch <= 0) return 0;
  const unsigned tiles = (unsigned)(launch & kF64MaxTiles);
  const int shape = launch >> kF64ShapeBit;
  const int* sched = static_cast<const int*>(d_sched);
  if (shape == kF64TileChain || shape == kF64TileShort) {
    const auto kernel = shape == kF64TileChain ? f64_chain_kernel<128> : f64_chain_kernel<64>;
    hipLaunchKernelGGL(kernel, dim3(tiles), dim3(2 * kThreads), 0, s, d_probs, sched);
  } else {
    const auto kernel = shape == kF64Tile128  ? f64_grouped_kernel<128, 128, 2, 2>
                        : shape == kF64Tile16 ? f64_grouped_kernel<16, 128, 1, 4>
                        : shape == kF64Tile32 ? f64_grouped_kernel<32, 128, 2, 4>
                                              : f64_grouped_kernel<64, 64, 2, 5>;
    hipLaunchKernelGGL(kernel, dim3(tiles), dim3(kThreads), 0, s, d_probs, sched);
  }
  return hipGetLastError() == hipSuccess ? 0 : 1;
}

}  // namespace ggemm
