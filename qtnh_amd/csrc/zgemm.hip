// Complex FP64 GEMM on CDNA matrix cores: C[MxN] = A[MxK] * B[KxN], row-major,
// complex128 interleaved.
//
// Each 16x16 complex output tile keeps a real and an imaginary accumulator
// and takes four v_mfma_f64_16x16x4_f64 per 4-deep k step:
//   Cr += Ar*Br, Ci += Ar*Bi, Cr += (-Ai)*Bi, Ci += Ai*Br.
// A workgroup of 2 x 2 waves owns a BM x BN complex tile.  Operands are staged
// through two LDS buffers BK complex deep: the loads of stage s + 1 are issued
// into registers before the MFMAs of stage s and written to the other buffer
// between them, so that a stage costs one barrier and the matrix cores (64
// cycles per f64 MFMA) wait for little else.  Every kFold terms the
// accumulators are added into a second set: sums of partial sums, whose error
// does not grow with the depth as one long sum's does.
#include <algorithm>

#include "internal.hpp"

namespace qtnh_hip {
namespace {

typedef double double4_t __attribute__((ext_vector_type(4)));
typedef double double2_t __attribute__((ext_vector_type(2)));

constexpr int BK = 16;
constexpr int kThreads = 256;

constexpr int kFold = 256;  // terms per accumulator set

constexpr uint64_t kMaxTiles = (1ull << 32) / kThreads - 1;  // a launch takes fewer than 2^32 threads

template <int BM, int BN>
struct ZTile {
  static constexpr int LDA = BK + 1;  // padded LDS rows (complex elements)
  static constexpr int LDB = BN + 1;
  static constexpr int kA = BM * LDA, kBuf = kA + BK * LDB;  // one stage's LDS elements
  static constexpr int A_PER = BM * BK / kThreads;            // complex loads per thread per stage
  static constexpr int B_PER = BK * BN / kThreads;
  static constexpr int TM = BM / 32, TN = BN / 32;  // MFMA tiles per wave
  static_assert(A_PER >= 1 && B_PER >= 1 && TM >= 1 && TN >= 1, "tile too small");
};

// Compile-time flags of a stage.
struct No {
  static constexpr bool value = false;
};
struct Yes {
  static constexpr bool value = true;
};

// The BM x BN output tile at (m0, n0) of C = A * B over k in [kb, ke), written
// to C.  lds: the workgroup's 2 kBuf staging elements.
template <int BM, int BN>
__device__ __forceinline__ void zgemm_tile(const c128 *__restrict__ A, const c128 *__restrict__ B,
                                           c128 *__restrict__ C, uint64_t M, uint64_t N, uint64_t lda, uint64_t ldb,
                                           uint64_t ldc, uint64_t kb, uint64_t ke, uint64_t m0, uint64_t n0,
                                           double2_t *lds) {
  using Z = ZTile<BM, BN>;
  constexpr int TM = Z::TM, TN = Z::TN;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int wm = (wave >> 1) * (BM / 2);  // wave tile origin inside the block tile
  const int wn = (wave & 1) * (BN / 2);

  double4_t accR[TM][TN], accI[TM][TN], sumR[TM][TN], sumI[TM][TN];
  const double4_t zero4 = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) accR[i][j] = accI[i][j] = zero4;

  // Loads of a stage: A rows 16 apart and B rows kThreads / BN apart.  Rows and
  // columns past the result's take the last one's values (their outputs are not
  // stored); terms past the depth take the last one's address and become zeros
  // on their way to LDS.
  constexpr int kBStep = kThreads / BN, kLoads = Z::A_PER + Z::B_PER;
  const int ar = tid / BK, ac = tid % BK, br = tid / BN, bc = tid % BN;
  const double2_t *pa[Z::A_PER];
#pragma unroll
  for (int r = 0; r < Z::A_PER; ++r) {
    const uint64_t m = m0 + ar + r * 16;
    pa[r] = reinterpret_cast<const double2_t *>(A) + (m < M ? m : M - 1) * lda;
  }
  const double2_t *pb = reinterpret_cast<const double2_t *>(B) + (n0 + bc < N ? n0 + bc : N - 1);
  double2_t v[kLoads];
  auto load = [&](int i, uint64_t k0, auto tail) {
    uint64_t k = i < Z::A_PER ? k0 + ac : k0 + br + (i - Z::A_PER) * kBStep;
    if (decltype(tail)::value) k = k < ke ? k : ke - 1;
    v[i] = i < Z::A_PER ? pa[i < Z::A_PER ? i : 0][k] : pb[k * ldb];
  };
  auto put = [&](int i, double2_t *buf, uint64_t k0, auto tail) {
    double2_t x = v[i];
    if (decltype(tail)::value && (i < Z::A_PER ? k0 + ac : k0 + br + (i - Z::A_PER) * kBStep) >= ke)
      x = double2_t{0.0, 0.0};
    if (i < Z::A_PER)
      buf[(ar + i * 16) * Z::LDA + ac] = x;
    else
      buf[Z::kA + (br + (i - Z::A_PER) * kBStep) * Z::LDB + bc] = x;
  };
  struct Frag {
    double2_t x[TM + TN];  // A rows, then B columns
  };
  constexpr int kReads = TM + TN;
  auto read = [&](Frag &f, int i, const double2_t *buf, int kk) {
    const int kl = kk + (lane >> 4);
    f.x[i] = i < TM ? buf[(wm + i * 16 + (lane & 15)) * Z::LDA + kl]
                    : buf[Z::kA + kl * Z::LDB + wn + (i - TM) * 16 + (lane & 15)];
  };
  // The four products of a step; between(n) after the n-th MFMA: the memory
  // work of the stage, a piece at a time, under the MFMAs (64 cycles each,
  // issued in order: anything between two groups of them leaves the matrix
  // core idle).  The last argument negates A.
  constexpr int kMfma = 4 * TM * TN;
  auto mma = [&](const Frag &f, auto between) {
#pragma unroll
    for (int p = 0; p < 4; ++p)
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          const double2_t x = f.x[i], y = f.x[TM + j];
          if (p == 0) accR[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(x.x, y.x, accR[i][j], 0, 0, 0);
          if (p == 1) accI[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(x.x, y.y, accI[i][j], 0, 0, 0);
          if (p == 2) accR[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(x.y, y.y, accR[i][j], 0, 0, 1);
          if (p == 3) accI[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(x.y, y.x, accI[i][j], 0, 0, 0);
          between((p * TM + i) * TN + j);
          __builtin_amdgcn_sched_barrier(0);
        }
  };
  // Pieces [0, count) dealt evenly over a step's MFMAs.
  auto deal = [&](int n, int count, auto piece) {
#pragma unroll
    for (int q = 0; q < count; ++q)
      if (q * kMfma / count == n) piece(q);
  };
  bool folded = false;
  int cur = 0, until = kFold / BK;
  Frag f0, f1;
  // One stage at k0: each fragment step is read a step ahead; the next stage
  // goes from registers to the other buffer (last read before the barrier of
  // the stage before) and the one after it is requested in its place; the
  // barrier comes before the last step, whose MFMAs cover the next stage's
  // first read.  PUT / GET: there is such a stage; *_TAIL: it may be partial.
  auto stage = [&](uint64_t k0, auto put_it, auto put_tail, auto get_it, auto get_tail) {
    const double2_t *buf = lds + cur;
    double2_t *next = lds + (Z::kBuf - cur);
    mma(f0, [&](int n) { deal(n, kReads, [&](int q) { read(f1, q, buf, 4); }); });
    mma(f1, [&](int n) { deal(n, kReads, [&](int q) { read(f0, q, buf, 8); }); });
    mma(f0, [&](int n) {
      deal(n, kReads, [&](int q) { read(f1, q, buf, 12); });
      deal(n, kLoads, [&](int q) {
        if (decltype(put_it)::value) put(q, next, k0 + BK, put_tail);
        if (decltype(get_it)::value) load(q, k0 + 2 * BK, get_tail);
      });
    });
    cur = Z::kBuf - cur;
    if (decltype(put_it)::value) lds_barrier();
    mma(f1, [&](int n) {
      if (decltype(put_it)::value) deal(n, kReads, [&](int q) { read(f0, q, next, 0); });
    });
    if (--until == 0 && decltype(put_it)::value) {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          sumR[i][j] = folded ? sumR[i][j] + accR[i][j] : accR[i][j];
          sumI[i][j] = folded ? sumI[i][j] + accI[i][j] : accI[i][j];
          accR[i][j] = accI[i][j] = zero4;
        }
      folded = true;
      until = kFold / BK;
    }
  };
#pragma unroll
  for (int i = 0; i < kLoads; ++i) load(i, kb, Yes{});
#pragma unroll
  for (int i = 0; i < kLoads; ++i) put(i, lds, kb, Yes{});
  if (kb + BK < ke) {
#pragma unroll
    for (int i = 0; i < kLoads; ++i) load(i, kb + BK, Yes{});
  }
  lds_barrier();
#pragma unroll
  for (int i = 0; i < kReads; ++i) read(f0, i, lds, 0);
  uint64_t k0 = kb;
  for (; k0 + 3 * BK <= ke; k0 += BK) stage(k0, Yes{}, No{}, Yes{}, No{});
  if (k0 + 2 * BK < ke) {
    stage(k0, Yes{}, No{}, Yes{}, Yes{});
    k0 += BK;
  }
  if (k0 + BK < ke) {
    stage(k0, Yes{}, Yes{}, No{}, No{});
    k0 += BK;
  }
  stage(k0, No{}, No{}, No{}, No{});
  lds_barrier();  // the buffers are free for another tile
  // Result layout of the 16x16 f64 MFMA (measured on gfx950): lane l holds
  // column l % 16 of rows l / 16 + 4 v, v = 0..3.
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      if (folded) {
        accR[i][j] = sumR[i][j] + accR[i][j];
        accI[i][j] = sumI[i][j] + accI[i][j];
      }
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const uint64_t gm = m0 + wm + i * 16 + (lane >> 4) + 4 * v;
        const uint64_t gn = n0 + wn + j * 16 + (lane & 15);
        if (gm < M && gn < N) {
          c128 out;
          out.re = accR[i][j][v];
          out.im = accI[i][j][v];
          C[gm * ldc + gn] = out;
        }
      }
    }
}

// Workgroup blk of `total` as a position in the tile order: workgroups are
// dealt to the 8 XCDs in turn, and XCD x takes the x-th stretch of the order,
// so that the tiles that share operand rows and columns meet in one L2.
__device__ __forceinline__ uint32_t xcd_order(uint32_t blk, uint32_t total) {
  const uint32_t q = total >> 3, r = total & 7u, x = blk & 7u;
  return x * q + (x < r ? x : r) + (blk >> 3);
}

// One BM x BN tile of one depth chunk per workgroup (chunk c: k in [c kc,
// (c + 1) kc), written to C + c cstride).  Tiles in groups of 8 tile rows,
// down each column of a group.
template <int BM, int BN>
__global__ void __launch_bounds__(kThreads, 2) zgemm_f64_kernel(const c128 *__restrict__ A, const c128 *__restrict__ B,
                                                             c128 *__restrict__ C, uint64_t M, uint64_t N, uint64_t K,
                                                             uint64_t lda, uint64_t ldb, uint64_t ldc, uint64_t kc,
                                                             uint64_t cstride, uint32_t ntm, uint32_t ntn) {
  __shared__ double2_t lds[2 * ZTile<BM, BN>::kBuf];
  const uint32_t tiles = ntm * ntn, l = xcd_order(blockIdx.x, gridDim.x);
  const uint32_t chunk = l / tiles, tile = l - chunk * tiles;
  const uint32_t group = tile / (8 * ntn), rows = min(8u, ntm - 8 * group), in = tile - group * 8 * ntn;
  const uint32_t tm = 8 * group + in % rows, tn = in / rows;
  const uint64_t kb = chunk * kc, ke = kb + kc < K ? kb + kc : K;
  zgemm_tile<BM, BN>(A, B, C + chunk * cstride, M, N, lda, ldb, ldc, kb, ke, (uint64_t)tm * BM, (uint64_t)tn * BN,
                     lds);
}

// Element of a sum of chunks, in chunk order, several of them requested at a time
// (the grouped sums of 32 networks of 4 x 5 grid circuits: 47 us, 62 one at a time).
template <int U>
__device__ __forceinline__ void add_chunks(double2_t &s, const double2_t *part, uint64_t stride, uint64_t &c,
                                           uint64_t chunks) {
  for (; c + U <= chunks; c += U) {
    double2_t v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = part[(c + u) * stride];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      s.x = s.x + v[u].x;
      s.y = s.y + v[u].y;
    }
  }
}

__device__ __forceinline__ double2_t sum_chunks(const double2_t *part, uint64_t stride, uint64_t chunks) {
  double2_t s = part[0];
  uint64_t c = 1;
  add_chunks<8>(s, part, stride, c, chunks);
  add_chunks<3>(s, part, stride, c, chunks);
  add_chunks<1>(s, part, stride, c, chunks);
  return s;
}

// Many GEMMs in one launch: each block of a grid-stride walk over every
// GEMM's (chunk, tile) blocks computes one tile, exactly as zgemm_f64_kernel.
template <int BM, int BN>
__global__ void __launch_bounds__(kThreads, 2) zgemm_grouped_kernel(const ZGroupDesc *__restrict__ d, int nd,
                                                                 uint64_t total) {
  __shared__ double2_t lds[2 * ZTile<BM, BN>::kBuf];
  for (uint64_t blk = blockIdx.x; blk < total; blk += gridDim.x) {
    const ZGroupDesc &D = d[find_entry(d, nd, blk)];
    const uint64_t local = blk - D.first, chunk = local / D.tiles, tile = local % D.tiles;
    const uint64_t ntn = (D.N + BN - 1) / BN, kb = chunk * D.kc, ke = kb + D.kc < D.K ? kb + D.kc : D.K;
    zgemm_tile<BM, BN>(D.A, D.B, D.C + chunk * D.cstride, D.M, D.N, D.K, D.N, D.N, kb, ke, tile / ntn * BM,
                       tile % ntn * BN, lds);
  }
}

// Sums of depth-chunk partials of many GEMMs: C = sum over chunks of part[c], in chunk order.
__global__ void zgemm_grouped_sum_kernel(const ZSumDesc *__restrict__ d, int nd, uint64_t total) {
  for (uint64_t blk = blockIdx.x; blk < total; blk += gridDim.x) {
    const ZSumDesc &D = d[find_entry(d, nd, blk)];
    const uint64_t i = (blk - D.first) * blockDim.x + threadIdx.x;
    if (i < D.MN) ((double2_t *)D.C)[i] = sum_chunks((const double2_t *)D.part + i, D.MN, D.chunks);
  }
}

constexpr int kSkThreads = 256;

// Partial sum s of output mn = m N + n: ordered per-thread sums over the
// chunk's terms, then a fixed tree in LDS; red: the workgroup's LDS buffer.
__device__ __forceinline__ void splitk_partial(const double2_t *__restrict__ A, const double2_t *__restrict__ Bt,
                                               uint64_t N, uint64_t K, uint64_t kc, uint64_t mn, uint64_t s,
                                               double2_t *__restrict__ out, double2_t *red) {
  const uint64_t m = mn / N, n = mn % N;
  const double2_t *a = A + m * K, *b = Bt + n * K;
  const uint64_t k1 = std::min(K, (s + 1) * kc);
  double re = 0.0, im = 0.0;
  for (uint64_t k = s * kc + threadIdx.x; k < k1; k += kSkThreads) {
    const double2_t x = a[k], y = b[k];
    double pr, pi;
    cmul_parts(x.x, x.y, y.x, y.y, &pr, &pi);
    re = re + pr;
    im = im + pi;
  }
  red[threadIdx.x] = double2_t{re, im};
  __syncthreads();
  for (int w = kSkThreads / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) {
      const double2_t u = red[threadIdx.x], v = red[threadIdx.x + w];
      red[threadIdx.x] = double2_t{u.x + v.x, u.y + v.y};
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) *out = red[0];
  __syncthreads();  // red is reused by the workgroup's next partial
}

// Block (output mn, chunk s).
__global__ void __launch_bounds__(kSkThreads) splitk_partial_kernel(const double2_t *__restrict__ A,
                                                                    const double2_t *__restrict__ Bt, uint64_t N,
                                                                    uint64_t K, uint64_t kc, uint64_t S,
                                                                    double2_t *__restrict__ part) {
  __shared__ double2_t red[kSkThreads];
  splitk_partial(A, Bt, N, K, kc, blockIdx.x / S, blockIdx.x % S, part + blockIdx.x, red);
}

__device__ __forceinline__ double2_t splitk_sum(const double2_t *__restrict__ part, uint64_t mn, uint64_t S) {
  double re = 0.0, im = 0.0;
  for (uint64_t s = 0; s < S; ++s) {
    const double2_t v = part[mn * S + s];
    re = re + v.x;
    im = im + v.y;
  }
  return double2_t{re, im};
}

__global__ void splitk_final_kernel(const double2_t *__restrict__ part, uint64_t MN, uint64_t S,
                                    double2_t *__restrict__ C) {
  for (uint64_t mn = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; mn < MN; mn += (uint64_t)gridDim.x * blockDim.x)
    C[mn] = splitk_sum(part, mn, S);
}

// Split-K partials of many contractions: blocks [first, first + MN S) of a
// descriptor are its (output, chunk) pairs.
__global__ void __launch_bounds__(kSkThreads) splitk_grouped_partial_kernel(const SkDesc *__restrict__ d, int nd,
                                                                            uint64_t total) {
  __shared__ double2_t red[kSkThreads];
  for (uint64_t blk = blockIdx.x; blk < total; blk += gridDim.x) {
    const SkDesc &D = d[find_entry(d, nd, blk)];
    const uint64_t local = blk - D.first;
    splitk_partial((const double2_t *)D.A, (const double2_t *)D.Bt, D.N, D.K, D.kc, local / D.S, local % D.S,
                   (double2_t *)D.part + local, red);
  }
}

// Their final sums: element i of descriptor j in block (i / 256) + D.first2.
__global__ void splitk_grouped_final_kernel(const SkDesc *__restrict__ d, int nd, uint64_t total) {
  for (uint64_t blk = blockIdx.x; blk < total; blk += gridDim.x) {
    int lo = 0, hi = nd - 1;
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (d[mid].first2 <= blk)
        lo = mid;
      else
        hi = mid - 1;
    }
    const SkDesc &D = d[lo];
    const uint64_t mn = (blk - D.first2) * blockDim.x + threadIdx.x;
    if (mn < D.MN) ((double2_t *)D.C)[mn] = splitk_sum((const double2_t *)D.part, mn, D.S);
  }
}
}  // namespace

qtnh_status launch_zgemm_splitk(qtnh_ctx_t ctx, const c128 *A, const c128 *Bt, c128 *C, uint64_t M, uint64_t N,
                                uint64_t K, uint64_t chunks, c128 *partials) {
  const uint64_t MN = M * N;
  const uint64_t kc = splitk_chunk_len(K, chunks);
  if (MN * chunks > 0x7fffffffull) return set_error(ctx, QTNH_EUNSUPPORTED, "splitk: grid too large");
  hipLaunchKernelGGL(splitk_partial_kernel, dim3((unsigned)(MN * chunks)), dim3(kSkThreads), 0, ctx->stream,
                     (const double2_t *)A, (const double2_t *)Bt, N, K, kc, chunks, (double2_t *)partials);
  qtnh_status st = check_hip(ctx, hipGetLastError(), "splitk launch");
  if (st) return st;
  hipLaunchKernelGGL(splitk_final_kernel, dim3(grid_for(MN, 256, 4096)), dim3(256), 0, ctx->stream,
                     (const double2_t *)partials, MN, chunks, (double2_t *)C);
  return check_hip(ctx, hipGetLastError(), "splitk final launch");
}

// Block width asked for: 0 none, 64 or 128.
static int g_zgemm_bn = 0;

extern "C" void qtnh_tune_zgemm(int bn) { g_zgemm_bn = (bn == 64 || bn == 128) ? bn : 0; }

// Most depth chunks of a shape whose operands are large: about 1024 tiles
// times chunks of 64 x 128 tiles, 256 terms each.  (Their partials are
// workspace that callers with a fixed one have to find room for.)
uint64_t zgemm_chunks_large(uint64_t M, uint64_t N, uint64_t K) {
  const uint64_t bn = (N < 128 || ((M + 63) / 64) * ((N + 63) / 64) >= 2048) ? 64 : 128;
  const uint64_t tiles = ((N + bn - 1) / bn) * ((M + 63) / 64);
  if (tiles == 0 || tiles * 2 > 1024 || K < 512) return 1;
  return std::max<uint64_t>(1, std::min<uint64_t>((1024 + tiles - 1) / tiles, K / 256));
}

// Tile and depth chunks of a shape: the least estimated time over the tiles
// and chunk counts, from measured rates: 5 us for a launch, its first loads and
// its stores; a 16-deep stage of a 64 x 64 tile 1.9 us of a compute unit, of a
// 32 x 64 tile 0.96, of a 32 x 32 tile 0.5 (1.0 and 0.6 where a compute unit
// has only one); the second kernel that sums depth chunks 5.5 us and its
// traffic.  A launch takes as long as the fullest of 256 compute units.
// The chunks depend on the shape only, also where the tiles are set: the network
// planner sizes workspaces with them, and every caller of a shape runs the same
// ones.  (64 x 64 tiles or 64 x 128
// ones alone, the rule before: 512^3 92 us, now 25 with 32 x 32 tiles; 256 x
// 512 x 256 85 and 14; 700^3 107 and 57; 4096^3 8.10 and 7.74 ms.)
struct ZShape {
  int bm, bn;
  uint64_t kc, chunks;
};
static ZShape zgemm_shape(uint64_t M, uint64_t N, uint64_t K) {
  struct Tile {
    int bm, bn;
    double stage, alone;  // us per stage of a compute unit, and more where it has one workgroup
  };
  static const Tile kTiles[] = {{64, 64, 1.9, 0.0}, {32, 64, 0.96, 0.04}, {32, 32, 0.5, 0.1}};
  // Up to here operands, result and partials fit the 64 MiB of the contraction without allocation.
  const uint64_t room = (uint64_t)(60 << 20) / sizeof(c128);
  const uint64_t large = zgemm_chunks_large(M, N, K), own = M * K + K * N + M * N;
  ZShape best{64, 64, K, 1};
  double t_best = 0.0;
  for (const Tile &t : kTiles) {
    const uint64_t tiles = ((M + t.bm - 1) / t.bm) * ((N + t.bn - 1) / t.bn);
    uint64_t last = 0;
    for (uint64_t want = 1; want <= 64; want += want < 4 ? 1 : want / 2) {
      uint64_t kc = (K + want - 1) / want;
      if (want > 1) kc = (kc + BK - 1) / BK * BK;
      const uint64_t chunks = (K + kc - 1) / kc;
      if (chunks > 1 && (kc < 64 || chunks == last)) continue;
      if (chunks > large && own + chunks * M * N > room) continue;
      if (tiles > kMaxTiles / chunks) continue;
      last = chunks;
      const double per = (double)((tiles * chunks + 255) / 256), stages = (double)((kc + BK - 1) / BK);
      double us = 5.0 + stages * (per * t.stage + (per > 1 ? 0.0 : t.alone));
      if (chunks > 1) us += 5.5 + (double)(M * N) * 16.0 * (double)(chunks + 1) / 4.5e6;
      if (t_best == 0.0 || us < 0.97 * t_best) {
        t_best = us;
        best = ZShape{t.bm, t.bn, kc, chunks};
      }
    }
  }
  if (g_zgemm_bn) best.bm = best.bn = 64;
  return best;
}

uint64_t zgemm_chunks(uint64_t M, uint64_t N, uint64_t K) { return zgemm_shape(M, N, K).chunks; }

// C = sum over chunks of part[c] (M x N each), in chunk order.
__global__ void zgemm_chunk_sum_kernel(const double2_t *__restrict__ part, double2_t *__restrict__ C, uint64_t M,
                                       uint64_t N, uint64_t ldc, uint64_t chunks) {
  const uint64_t MN = M * N;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < MN; i += (uint64_t)gridDim.x * blockDim.x) {
    C[(i / N) * ldc + i % N] = sum_chunks(part + i, MN, chunks);
  }
}

template <int BM, int BN>
static void launch_tile_gemm(qtnh_ctx_t ctx, const c128 *A, const c128 *B, c128 *out, uint64_t M, uint64_t N,
                             uint64_t K, uint64_t lda, uint64_t ldb, uint64_t ld, uint64_t cstride, const ZShape &z) {
  const uint32_t ntm = (uint32_t)((M + BM - 1) / BM), ntn = (uint32_t)((N + BN - 1) / BN);
  hipLaunchKernelGGL((zgemm_f64_kernel<BM, BN>), dim3((unsigned)(ntm * ntn * z.chunks)), dim3(kThreads), 0, ctx->stream,
                     A, B, out, M, N, K, lda, ldb, ld, z.kc, cstride, ntm, ntn);
}

qtnh_status launch_zgemm_f64(qtnh_ctx_t ctx, const c128 *A, const c128 *B, c128 *C, uint64_t M, uint64_t N, uint64_t K,
                             uint64_t lda, uint64_t ldb, uint64_t ldc, c128 *partials) {
  const ZShape z = zgemm_shape(M, N, K);
  const uint64_t tiles = ((N + z.bn - 1) / z.bn) * ((M + z.bm - 1) / z.bm);
  if (tiles > kMaxTiles / z.chunks) return set_error(ctx, QTNH_EUNSUPPORTED, "zgemm: grid too large");
  if (z.chunks > 1 && !partials) return set_error(ctx, QTNH_EINVAL, "zgemm: depth chunks need a partial buffer");
  c128 *out = z.chunks > 1 ? partials : C;
  const uint64_t ld = z.chunks > 1 ? N : ldc, cstride = z.chunks > 1 ? M * N : 0;
  if (z.bm == 64)
    launch_tile_gemm<64, 64>(ctx, A, B, out, M, N, K, lda, ldb, ld, cstride, z);
  else if (z.bn == 64)
    launch_tile_gemm<32, 64>(ctx, A, B, out, M, N, K, lda, ldb, ld, cstride, z);
  else
    launch_tile_gemm<32, 32>(ctx, A, B, out, M, N, K, lda, ldb, ld, cstride, z);
  qtnh_status st = check_hip(ctx, hipGetLastError(), "zgemm launch");
  if (st || z.chunks <= 1) return st;
  hipLaunchKernelGGL(zgemm_chunk_sum_kernel, dim3(grid_for(M * N, 256, 65536)), dim3(256), 0, ctx->stream,
                     (const double2_t *)partials, (double2_t *)C, M, N, ldc, z.chunks);
  return check_hip(ctx, hipGetLastError(), "zgemm chunk sum launch");
}


uint64_t splitk_chunk_len(uint64_t K, uint64_t chunks) {
  return ((K + chunks - 1) / chunks + kSkThreads - 1) / kSkThreads * kSkThreads;
}

// Depth chunks of launch_zgemm_f64 on BK steps: (chunk length, chunk count).
void zgemm_chunk_shape(uint64_t M, uint64_t N, uint64_t K, uint64_t *kc_out, uint64_t *n_out) {
  const ZShape z = zgemm_shape(M, N, K);
  *kc_out = z.kc;
  *n_out = z.chunks;
}

// Tile edge of a shape's GEMM in grouped launches (other shapes fill the GPU
// beside it): 64 where that wastes little of its tiles, else 32.
int zgemm_group_tile(uint64_t M, uint64_t N) {
  auto padded = [&](uint64_t b) { return ((M + b - 1) / b) * ((N + b - 1) / b) * b * b; };
  return M > 32 && N > 32 && padded(64) * 4 <= padded(32) * 5 ? 64 : 32;
}

qtnh_status launch_zgemm_grouped(qtnh_ctx_t ctx, int tile, const ZGroupDesc *d, int nd, uint64_t total) {
  if (nd <= 0 || total == 0) return QTNH_OK;
  const unsigned grid = (unsigned)std::min<uint64_t>(total, (uint64_t)ctx->num_cus * 8);
  if (tile == 64)
    hipLaunchKernelGGL((zgemm_grouped_kernel<64, 64>), dim3(grid), dim3(kThreads), 0, ctx->stream, d, nd, total);
  else
    hipLaunchKernelGGL((zgemm_grouped_kernel<32, 32>), dim3(grid), dim3(kThreads), 0, ctx->stream, d, nd, total);
  return check_hip(ctx, hipGetLastError(), "grouped zgemm launch");
}

qtnh_status launch_zgemm_grouped_sum(qtnh_ctx_t ctx, const ZSumDesc *d, int nd, uint64_t total) {
  if (nd <= 0 || total == 0) return QTNH_OK;
  const unsigned grid = (unsigned)std::min<uint64_t>(total, (uint64_t)ctx->num_cus * 16);
  hipLaunchKernelGGL(zgemm_grouped_sum_kernel, dim3(grid), dim3(256), 0, ctx->stream, d, nd, total);
  return check_hip(ctx, hipGetLastError(), "grouped chunk sum launch");
}

qtnh_status launch_splitk_grouped(qtnh_ctx_t ctx, const SkDesc *d, int nd, uint64_t total_partial,
                                  uint64_t total_final) {
  if (nd <= 0) return QTNH_OK;
  unsigned grid = (unsigned)std::min<uint64_t>(total_partial, (uint64_t)ctx->num_cus * 16);
  hipLaunchKernelGGL(splitk_grouped_partial_kernel, dim3(grid), dim3(kSkThreads), 0, ctx->stream, d, nd,
                     total_partial);
  qtnh_status st = check_hip(ctx, hipGetLastError(), "grouped splitk launch");
  if (st) return st;
  grid = (unsigned)std::min<uint64_t>(total_final, (uint64_t)ctx->num_cus * 16);
  hipLaunchKernelGGL(splitk_grouped_final_kernel, dim3(grid), dim3(256), 0, ctx->stream, d, nd, total_final);
  return check_hip(ctx, hipGetLastError(), "grouped splitk final launch");
}

}  // namespace qtnh_hip
