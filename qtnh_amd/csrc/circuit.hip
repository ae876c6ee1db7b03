// Gate sequences on resident state vectors: qubit circuits as chains of the
// in-place gate and diagonal contractions of the contraction path.
//
// The reference applies a circuit as one Tensor::contract per gate against
// the state (examples/qft.cpp; src/tensor/contract.cpp:250-289 places each
// gate's outputs on its inputs' axes).  Here a circuit is a list of ops, each
// a dense k-qubit gate G[in][out] or a diagonal d[x], with qubit q = axis q of
// a rank-n state with every dim 2 (axis 0 is the most significant index bit).
//
// Two executors:
//  * per gate: one launch of the streaming gate / diagonal kernels per op;
//  * fused: consecutive ops are grouped into runs touching at most `tb`
//    distinct index bits.  A run is one pass over the state: each workgroup
//    gathers a tile of 2^tb amplitudes (the run's bits vary, every other bit
//    is fixed) into registers (some forms: LDS), applies the run's ops in order,
//    and scatters the tile back.  Every op does the same arithmetic on the same values as the per
//    gate kernel (sum over inputs in row-major order from zero, products
//    without FMA), so both executors agree bit for bit; the fused one reads
//    and writes the state once per run instead of once per op.
// Batches run the k-th run of many circuits (on many states) in one launch.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <map>
#include <memory>
#include <vector>

#include "internal.hpp"

namespace qtnh_hip {

qtnh_status launch_gate(qtnh_ctx_t ctx, c128 *state, int rank, const uint64_t *dims, int k, const uint16_t *axes,
                        const double *G);
qtnh_status launch_diag(qtnh_ctx_t ctx, c128 *state, int rank, const uint64_t *dims, int k, const uint16_t *axes,
                        const double *d);

namespace {

typedef double double2_t __attribute__((ext_vector_type(2)));

constexpr int kMaxTileBits = 13;  // 2^13 amplitudes = 128 KiB of LDS
constexpr int kMaxOpQubits = 3;
constexpr int kMinRegBits = 2, kMaxRegBits = 4;  // register bits of circuit_reg_kernel

struct TileOp {
  int kind;                 // 0: dense gate, 1: diagonal
  int kb;                   // qubits of the op inside the tile
  int pos[kMaxOpQubits];    // tile bit of op-index bit j (j = 0 most significant)
  int zpos[kMaxOpQubits];   // the same tile bits, ascending
  uint32_t coef;            // first coefficient (complex units)
  // Diagonals only: qubits outside the tile.  Byte 0: their count; byte 1 + j:
  // bit of the run's tile number holding the j-th of them (op order).  Their
  // values are fixed within a tile and pick one block of 2^kb coefficients.
  uint32_t outer;
};

// First coefficient of a diagonal's block for tile number t of its run.
__device__ __forceinline__ uint32_t outer_sel(const TileOp &op, uint64_t t) {
  const uint32_t no = op.outer & 0xffu;
  uint32_t s = 0;
  for (uint32_t j = 0; j < no; ++j) s = (s << 1) | (uint32_t)((t >> ((op.outer >> (8 + 8 * j)) & 0xffu)) & 1u);
  return s << op.kb;
}

// Coefficients of an op: 2^(2 kb) for a gate, 2^(kb + outer qubits) for a diagonal.
__device__ __forceinline__ uint32_t coef_count(const TileOp &op) {
  return op.kind == 1 ? (1u << (op.kb + (op.outer & 0xffu))) : (1u << (2 * op.kb));
}

struct RegOp;
struct RegChunk;

struct RunDesc {
  const TileOp *ops;
  const double2_t *coef;
  double2_t *psi;
  uint64_t first;       // first tile of this run in the launch's tile numbering
  uint64_t outer_mask;  // state bits outside the tile
  uint64_t tile_mask;   // state bits of the tile
  uint32_t op_begin, op_end;
  uint32_t coef_begin;  // first coefficient of op_begin (ops' coefficients are contiguous)
  int tb;               // tile bits
  int n_outer;          // popcount(outer_mask)
  // Register form (circuit_reg_kernel): its ops, coefficients, staging chunks
  // [chunk_begin, chunk_end) and first register bits (packed).
  const RegOp *rops;
  const double2_t *rcoef;
  const RegChunk *rchunks;
  uint32_t chunk_begin, chunk_end;
  uint32_t map0;
  uint32_t where_in, where_out;  // state bits of the first and the last register bits (8 bits each)
  int rbits;  // register bits (0: no register form)
  int has3;   // a run of the launch may hold dense 3-qubit gates
};

constexpr int kChunkOps = 32;     // ops staged in LDS at a time
constexpr int kChunkCoef = 512;   // their coefficients (complex)

// Parallel bit deposit: the low bits of v, in order, onto the set bits of mask.
__device__ __forceinline__ uint64_t deposit(uint64_t v, uint64_t mask) {
  uint64_t r = 0;
  while (mask) {
    const uint64_t low = mask & (0 - mask);
    if (v & 1ull) r |= low;
    v >>= 1;
    mask ^= low;
  }
  return r;
}

__device__ __forceinline__ double2_t cmul2(double2_t a, double2_t b) {
  double r, i;
  cmul_parts(a.x, a.y, b.x, b.y, &r, &i);
  return double2_t{r, i};
}

// Group gi of a k-qubit op: tile index with zero bits inserted at the op's bits.
template <int KB>
__device__ __forceinline__ int group_base(int gi, const TileOp &op) {
  int base = gi;
#pragma unroll
  for (int j = 0; j < KB; ++j) {
    const int p = op.zpos[j];
    base = ((base >> p) << (p + 1)) | (base & ((1 << p) - 1));
  }
  return base;
}

// Dense k-qubit op on a tile in LDS.  U groups per iteration: all their loads
// are issued before any store (the groups are disjoint), so LDS latency
// overlaps across groups.
template <int KB, int NT>
__device__ void gate_in_lds(double2_t *buf, int tb, const TileOp &op, const double2_t *g) {
  constexpr int K = 1 << KB;
  constexpr int U = KB == 3 ? 1 : 2;
  int comb[K];
#pragma unroll
  for (int c = 0; c < K; ++c) {
    int off = 0;
#pragma unroll
    for (int j = 0; j < KB; ++j)
      if ((c >> (KB - 1 - j)) & 1) off |= 1 << op.pos[j];
    comb[c] = off;
  }
  const int groups = 1 << (tb - KB);
  for (int g0 = threadIdx.x; g0 < groups; g0 += NT * U) {
    // Large gates (and 2-qubit gates in 1024-thread blocks, which have 128
    // registers): re-read the coefficients from LDS in every iteration rather
    // than holding them in registers (a compiler barrier, no code).
    if (KB == 3 || (KB == 2 && NT == 1024)) asm volatile("" ::: "memory");
    int base[U];
    bool live[U];
    double2_t in[U][K];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int gi = g0 + u * NT;
      live[u] = gi < groups;
      base[u] = group_base<KB>(live[u] ? gi : g0, op);
#pragma unroll
      for (int c = 0; c < K; ++c) in[u][c] = buf[base[u] + comb[c]];
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (!live[u]) continue;
#pragma unroll
      for (int o = 0; o < K; ++o) {
        double2_t acc = {0.0, 0.0};
#pragma unroll
        for (int i = 0; i < K; ++i) {
          const double2_t p = cmul2(in[u][i], g[i * K + o]);
          acc.x = acc.x + p.x;
          acc.y = acc.y + p.y;
        }
        buf[base[u] + comb[o]] = acc;
      }
    }
  }
}

template <int KB, int NT>
__device__ void diag_in_lds(double2_t *buf, int tb, const TileOp &op, const double2_t *d) {
  constexpr int U = 4;
  const int T = 1 << tb;
  for (int l0 = threadIdx.x; l0 < T; l0 += NT * U) {
    double2_t v[U];
    int c[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int l = l0 + u * NT;
      c[u] = 0;
#pragma unroll
      for (int j = 0; j < KB; ++j) c[u] = (c[u] << 1) | ((l >> op.pos[j]) & 1);
      v[u] = l < T ? buf[l] : double2_t{0.0, 0.0};
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int l = l0 + u * NT;
      if (l < T) buf[l] = cmul2(v[u], d[c[u]]);
    }
  }
}

// One workgroup per tile (persistent over tiles); runs[] sorted by `first`.
// Ops and their coefficients are staged into LDS in chunks; each op is
// followed by one barrier.
template <int TBMAX, int NT>
__global__ void __launch_bounds__(NT, (NT == 256 && TBMAX < 13) ? 2 : 1)
    circuit_tile_kernel(const RunDesc *__restrict__ runs, int nruns, uint64_t total_tiles) {
  constexpr int LB = NT == 1024 ? 10 : 8;  // tile bits taken from the thread index
  __shared__ double2_t buf[1 << TBMAX];
  __shared__ double2_t cbuf[kChunkCoef];
  __shared__ TileOp obuf[kChunkOps];
  __shared__ uint64_t hi_off[(1 << TBMAX) / NT + 1];
  for (uint64_t gt = blockIdx.x; gt < total_tiles; gt += gridDim.x) {
    int lo = 0, hi = nruns - 1;
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (runs[mid].first <= gt)
        lo = mid;
      else
        hi = mid - 1;
    }
    const RunDesc &R = runs[lo];
    const uint64_t t = gt - R.first;
    const int T = 1 << R.tb;
    const int nj = (T + NT - 1) / NT;
    // Tile element l = thread + NT j: its low LB tile bits are the thread's,
    // the others come from j (table hi_off).
    uint64_t lo_mask = 0, rest = R.tile_mask;
    for (int b = 0; b < LB && rest; ++b) {
      const uint64_t low = rest & (0 - rest);
      lo_mask |= low;
      rest ^= low;
    }
    if ((int)threadIdx.x < nj) hi_off[threadIdx.x] = deposit(threadIdx.x, rest);
    double2_t *psi = R.psi + deposit(t, R.outer_mask);
    const uint64_t lo_off = deposit(threadIdx.x, lo_mask);
    __syncthreads();
    for (int l = threadIdx.x, j = 0; l < T; l += NT, ++j) buf[l] = psi[lo_off | hi_off[j]];
    uint32_t o = R.op_begin;
    uint32_t cbase = R.coef_begin;
    while (o < R.op_end) {
      // Stage the next ops whose coefficients fit the chunk.
      __syncthreads();  // previous chunk's ops are done with obuf / cbuf
      uint32_t oe = o, ce = cbase;
      while (oe < R.op_end && oe - o < (uint32_t)kChunkOps) {
        const TileOp &x = R.ops[oe];
        const uint32_t nco = coef_count(x);
        if (x.coef + nco - cbase > (uint32_t)kChunkCoef) break;
        ce = x.coef + nco;
        ++oe;
      }
      for (uint32_t i = threadIdx.x; i < oe - o; i += NT) obuf[i] = R.ops[o + i];
      for (uint32_t i = threadIdx.x; i < ce - cbase; i += NT) cbuf[i] = R.coef[cbase + i];
      __syncthreads();
      for (uint32_t i = 0; i < oe - o; ++i) {
        const TileOp &op = obuf[i];
        const double2_t *g = cbuf + (op.coef - cbase);
        if (op.kind == 1) {
          g += outer_sel(op, t);
          if (op.kb == 0)
            diag_in_lds<0, NT>(buf, R.tb, op, g);
          else if (op.kb == 1)
            diag_in_lds<1, NT>(buf, R.tb, op, g);
          else if (op.kb == 2)
            diag_in_lds<2, NT>(buf, R.tb, op, g);
          else
            diag_in_lds<3, NT>(buf, R.tb, op, g);
        } else if (op.kb == 1) {
          gate_in_lds<1, NT>(buf, R.tb, op, g);
        } else if (op.kb == 2) {
          gate_in_lds<2, NT>(buf, R.tb, op, g);
        } else {
          gate_in_lds<3, NT>(buf, R.tb, op, g);
        }
        __syncthreads();
      }
      o = oe;
      cbase = ce;
    }
    if (R.op_begin == R.op_end) __syncthreads();
    for (int l = threadIdx.x, j = 0; l < T; l += NT, ++j) psi[lo_off | hi_off[j]] = buf[l];
    __syncthreads();
  }
}

// Large states: runs whose tiles have exactly kPipeTB bits.  One 512-thread
// workgroup per CU walks its tiles with two LDS tile buffers: while the ops of
// tile k run on one buffer, tile k+1 streams into the other straight from HBM
// (global_load_lds_dwordx4: each wave instruction gathers 64 tile elements,
// 1 KiB, into consecutive LDS slots), and tile k is written back with
// non-temporal stores.  Same ops, same order, same arithmetic as
// circuit_tile_kernel.
constexpr int kPipeTB = 12, kPipeT = 1 << kPipeTB, kPipeNT = 512;
constexpr int kPipeWaves = kPipeNT / 64, kPipeCPW = kPipeT / 64 / kPipeWaves;  // 8 chunks of 64 per wave

__device__ __forceinline__ int find_run(const RunDesc *__restrict__ runs, int nruns, uint64_t gt) {
  int lo = 0, hi = nruns - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (runs[mid].first <= gt)
      lo = mid;
    else
      hi = mid - 1;
  }
  return lo;
}

// This lane's element offsets in tile t of run R: element l = 64 (wave + kPipeWaves k) + lane.
__device__ __forceinline__ double2_t *pipe_offsets(const RunDesc &R, uint64_t t, int wave, int lane,
                                                   uint64_t (&off)[kPipeCPW]) {
  uint64_t lo6 = 0, rest = R.tile_mask;
  for (int b = 0; b < 6; ++b) {
    const uint64_t low = rest & (0 - rest);
    lo6 |= low;
    rest ^= low;
  }
  const uint64_t lo = deposit(lane, lo6);
#pragma unroll
  for (int k = 0; k < kPipeCPW; ++k) off[k] = lo | deposit(wave + kPipeWaves * k, rest);
  return R.psi + deposit(t, R.outer_mask);
}

__device__ __forceinline__ void pipe_issue(double2_t *dstbuf, const double2_t *psi, const uint64_t (&off)[kPipeCPW],
                                           int wave) {
#pragma unroll
  for (int k = 0; k < kPipeCPW; ++k)
    __builtin_amdgcn_global_load_lds((const void *)(psi + off[k]),
                                     (void __attribute__((address_space(3))) *)(dstbuf + 64 * (wave + kPipeWaves * k)),
                                     16, 0, 0);
}

__global__ void __launch_bounds__(kPipeNT, 1)
    circuit_pipe_kernel(const RunDesc *__restrict__ runs, int nruns, uint64_t total_tiles) {
  __shared__ double2_t buf[2][kPipeT];
  __shared__ double2_t cbuf[kChunkCoef];
  __shared__ TileOp obuf[kChunkOps];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  uint64_t gt = blockIdx.x;
  if (gt >= total_tiles) return;  // uniform: the whole workgroup leaves
  int r = find_run(runs, nruns, gt);
  uint64_t off[kPipeCPW];
  double2_t *psi = pipe_offsets(runs[r], gt - runs[r].first, wave, lane, off);
  pipe_issue(buf[0], psi, off, wave);
  int cur = 0;
  while (true) {
    const RunDesc &R = runs[r];
    // This tile's gather is complete (and the previous tile's stores have been
    // accepted: the counter covers both, and nothing here relies on their order).
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    // Stage the first chunk of ops before the next gather is issued (their
    // loads then do not wait behind it).
    uint32_t o = R.op_begin, cbase = R.coef_begin;
    auto stage = [&](uint32_t &oe, uint32_t &ce) {
      oe = o;
      ce = cbase;
      while (oe < R.op_end && oe - o < (uint32_t)kChunkOps) {
        const TileOp &x = R.ops[oe];
        const uint32_t nco = coef_count(x);
        if (x.coef + nco - cbase > (uint32_t)kChunkCoef) break;
        ce = x.coef + nco;
        ++oe;
      }
      for (uint32_t i = threadIdx.x; i < oe - o; i += kPipeNT) obuf[i] = R.ops[o + i];
      for (uint32_t i = threadIdx.x; i < ce - cbase; i += kPipeNT) cbuf[i] = R.coef[cbase + i];
    };
    uint32_t oe, ce;
    stage(oe, ce);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    const uint64_t gn = gt + gridDim.x;
    const bool more = gn < total_tiles;  // uniform
    int rn = r;
    uint64_t offn[kPipeCPW];
    double2_t *psin = psi;
    if (more) {
      rn = find_run(runs, nruns, gn);
      psin = pipe_offsets(runs[rn], gn - runs[rn].first, wave, lane, offn);
      pipe_issue(buf[cur ^ 1], psin, offn, wave);
    }
    double2_t *tb = buf[cur];
    while (true) {
      for (uint32_t i = 0; i < oe - o; ++i) {
        const TileOp &op = obuf[i];
        const double2_t *g = cbuf + (op.coef - cbase);
        if (op.kind == 1) {
          g += outer_sel(op, gt - R.first);
          if (op.kb == 0)
            diag_in_lds<0, kPipeNT>(tb, kPipeTB, op, g);
          else if (op.kb == 1)
            diag_in_lds<1, kPipeNT>(tb, kPipeTB, op, g);
          else if (op.kb == 2)
            diag_in_lds<2, kPipeNT>(tb, kPipeTB, op, g);
          else
            diag_in_lds<3, kPipeNT>(tb, kPipeTB, op, g);
        } else if (op.kb == 1) {
          gate_in_lds<1, kPipeNT>(tb, kPipeTB, op, g);
        } else if (op.kb == 2) {
          gate_in_lds<2, kPipeNT>(tb, kPipeTB, op, g);
        } else {
          gate_in_lds<3, kPipeNT>(tb, kPipeTB, op, g);
        }
        __syncthreads();
      }
      o = oe;
      cbase = ce;
      if (o >= R.op_end) break;
      // More ops than one chunk: stage the next chunk (waits behind the gather).
      stage(oe, ce);
      __syncthreads();
    }
    // Write the tile back.
#pragma unroll
    for (int k = 0; k < kPipeCPW; ++k)
      __builtin_nontemporal_store(tb[64 * (wave + kPipeWaves * k) + lane], psi + off[k]);
    if (!more) break;
    gt = gn;
    r = rn;
    psi = psin;
#pragma unroll
    for (int k = 0; k < kPipeCPW; ++k) off[k] = offn[k];
    cur ^= 1;
  }
}

// Register-resident runs: a thread holds 2^R amplitudes of its tile in
// registers for the whole run.  The tile's index bits split into R register
// bits (the same for every thread) and the thread bits.  Dense gates act on
// register bits with compile-time indexing; a diagonal may use any bit (its
// register bits pick among up to 8 coefficients, its thread bits and the bits
// outside the tile pick which ones, per lane), so only dense gates ask for
// other register bits.  Such a change passes the tile through LDS.  The first
// register bits are those of the first gates, read straight from the state.
//
// What bounds it (28 qubits, 12-bit tiles, R = 4): a run of one gate takes
// 1.66 ms, 5.2 TB/s, what an in-place pass reaches here in workgroups of
// 64 KiB (5.4 TB/s by a plain kernel); each 1-qubit gate adds 106 us of FP64
// issue once that passes the memory's time (14 instructions per amplitude at
// the 33 T a second the card reaches: 114), a diagonal 44, an exchange 100.
// Four workgroups per compute unit (half the LDS: real and imaginary parts
// are exchanged one after the other; at most 128 VGPRs) hide one another's
// loads and exchanges.  The 28-qubit depth-6 random circuit went from 56.2 to
// 37.7 ms with this form (from a tile kept in LDS between phases, 64 KiB and
// two workgroups per compute unit, whose op switch copied the amplitudes).
//
// The op list and its coefficients are staged in LDS by chunks; an op is one
// 16-byte record, read by every lane from one address and made uniform.
//
// Arithmetic: that of gate_in_lds / diag_in_lds, whose sums start from 0.0.
// Here they start from the first product, which is the same but for a sum of
// zeros: -0 where every product is (exactly or by underflow), and +0 there.  A
// gate's results do not depend on the signs of zeros among its inputs, so a
// dense record turns -0 into +0 (two additions per amplitude, kRegSettle) only
// where a diagonal or the end of the circuit follows.
struct RegOp {
  // One bit per op form.  1-qubit gates on register bits 3..0 (kRegG1): one
  // record may hold several, applied from the highest bit down, their
  // coefficients one after another.  0 ends a chunk.
  uint32_t code;
  uint32_t coef;  // first coefficient (of the run's list)
  // Diagonals: tile positions of the thread bits in bytes 0..2, the least
  // significant last (31, a zero bit, where there are fewer than three), and
  // their count in byte 3.  kRegSpecial: 0 for a dense 3-qubit gate, else a
  // change of register bits: kRegRemapFlag and their tile positions, 4 bits each.
  // Dense gates: kRegSettle or 0.
  uint32_t lane;
  uint32_t outer;  // diagonals: bits of the tile number, likewise (63: a zero bit; no count)
};
constexpr int kRegG1 = 0, kRegG2 = 4, kRegSpecial = 16, kRegD0 = 17, kRegD1 = 18, kRegD2 = 22, kRegD3 = 28;
constexpr uint32_t kRegRemapFlag = 1u << 31, kRegSettle = 1u << 30, kRegNoLane = 0x1f1f1f, kRegNoOuter = 0x3f3f3f;
constexpr int kRegOps = 48, kRegCoef = 384;  // per chunk: with a 32 KiB half tile, four workgroups fit 160 KiB
struct RegChunk {
  uint32_t op_begin, op_end, coef_begin, coef_end;
};

// Read-only tables seen through the constant address space: uniform reads
// become scalar loads.
template <typename T>
__device__ __forceinline__ const __attribute__((address_space(4))) T *as_const(const T *p) {
  return (const __attribute__((address_space(4))) T *)(p);
}

// Tile element l's LDS slot: l with its low five bits mixed with bits 5..11,
// so that the lanes of an access fall on different banks for nearly every
// choice of register bits (the vectors were searched for; at most two-way for
// contiguous ones).  Linear over XOR.
constexpr uint32_t kSlotMix[7] = {31, 11, 28, 26, 25, 3, 9};
__device__ __forceinline__ uint32_t reg_slot(uint32_t l) {
  uint32_t s = l;
#pragma unroll
  for (int i = 0; i < 7; ++i) s ^= (0u - ((l >> (5 + i)) & 1u)) & kSlotMix[i];
  return s;
}
// That of tile bit b (uniform) alone, from the vectors packed five bits a tile bit.
__device__ __forceinline__ uint32_t reg_slot_bit(uint32_t b) {
  uint64_t packed = 0;
#pragma unroll
  for (int i = 0; i < 7; ++i) packed |= (uint64_t)kSlotMix[i] << (5 * (5 + i));
  return (1u << b) ^ ((uint32_t)(packed >> (5 * b)) & 31u);
}

// Deposit over runs of set bits: mask is uniform, so its few runs are walked
// by scalar code.
__device__ __forceinline__ uint64_t deposit_runs(uint32_t v, uint64_t mask) {
  uint64_t r = 0;
  while (mask) {
    const int lo = __builtin_ctzll(mask);
    const uint64_t up = ~(mask >> lo);
    const int len = up ? __builtin_ctzll(up) : 64;
    const uint32_t part = len >= 32 ? v : v & ((1u << len) - 1u);
    r |= (uint64_t)part << lo;
    v = len >= 32 ? 0 : v >> len;
    mask = lo + len >= 64 ? 0 : mask >> (lo + len) << (lo + len);
  }
  return r;
}

__device__ __forceinline__ uint64_t deposit_runs64(uint64_t v, uint64_t mask) {
  uint64_t r = 0;
  while (mask) {
    const int lo = __builtin_ctzll(mask);
    const uint64_t up = ~(mask >> lo);
    const int len = up ? __builtin_ctzll(up) : 64;
    const uint64_t field = len >= 64 ? ~0ull : (1ull << len) - 1ull;
    r |= (v & field) << lo;
    v = len >= 64 ? 0 : v >> len;
    mask &= ~(field << lo);
  }
  return r;
}

// x = a + b and x = a - b into the register x already has: the amplitudes keep
// their registers through every op, so the op loop needs no copies where its
// cases meet (32 moves per op with plain assignments).
__device__ __forceinline__ void add_to(double &x, double a, double b) {
  asm("v_add_f64 %0, %1, %2" : "+v"(x) : "v"(a), "v"(b));
}
__device__ __forceinline__ void sub_to(double &x, double a, double b) {
  asm("v_add_f64 %0, %1, -%2" : "+v"(x) : "v"(a), "v"(b));
}

// -0 becomes +0; other values stay.
template <int R>
__device__ __forceinline__ void rg_settle(double (&re)[1 << R], double (&im)[1 << R]) {
#pragma unroll
  for (int r = 0; r < (1 << R); ++r) {
    asm("v_add_f64 %0, %0, 0" : "+v"(re[r]));
    asm("v_add_f64 %0, %0, 0" : "+v"(im[r]));
  }
}

template <int R, int A>
__device__ __forceinline__ void rg_gate1(double (&re)[1 << R], double (&im)[1 << R], const double2_t *g) {
  const double2_t g00 = g[0], g01 = g[1], g10 = g[2], g11 = g[3];
#pragma unroll
  for (int r = 0; r < (1 << R); ++r) {
    if ((r >> A) & 1) continue;
    const int s = r | (1 << A);
    const double2_t a = {re[r], im[r]}, b = {re[s], im[s]};
    const double2_t p0 = cmul2(a, g00), q0 = cmul2(b, g10);
    const double2_t p1 = cmul2(a, g01), q1 = cmul2(b, g11);
    add_to(re[r], p0.x, q0.x);
    add_to(im[r], p0.y, q0.y);
    add_to(re[s], p1.x, q1.x);
    add_to(im[s], p1.y, q1.y);
  }
}

// KB-qubit gate on register bits A, B, C (most significant first).  ROOM: registers
// for the next input's coefficients.
template <int R, int KB, int A, int B, int C, bool ROOM>
__device__ __forceinline__ void rg_gate(double (&re)[1 << R], double (&im)[1 << R], const double2_t *g) {
  constexpr int K = 1 << KB;
  constexpr int M = (1 << A) | (1 << B) | (KB > 2 ? (1 << C) : 0);
  double2_t row[2][K];  // (ROOM) this input's coefficients and the next one's
  if (ROOM) {
#pragma unroll
    for (int o = 0; o < K; ++o) row[0][o] = g[o];
  }
#pragma unroll
  for (int r0 = 0; r0 < (1 << R); ++r0) {
    if (r0 & M) continue;
    int idx[K];
#pragma unroll
    for (int c = 0; c < K; ++c) {
      int x = r0;
      if ((c >> (KB - 1)) & 1) x |= 1 << A;
      if ((c >> (KB - 2)) & 1) x |= 1 << B;
      if (KB > 2 && (c & 1)) x |= 1 << C;
      idx[c] = x;
    }
    // Every output's sum over all terms but the last, term by term; the last
    // term's addition then puts output o in the registers of input o, which no
    // sum needs any more (the last input's own output comes last).
    double ar[K], ai[K];
#pragma unroll
    for (int i = 0; i < K; ++i) {
      const double2_t x = {re[idx[i]], im[idx[i]]};
      if (ROOM) {
#pragma unroll
        for (int o = 0; o < K; ++o) row[(i + 1) & 1][o] = g[(i + 1) % K * K + o];
        __builtin_amdgcn_sched_barrier(0);  // requested before this input's products
      }
#pragma unroll
      for (int o = 0; o < K; ++o) {
        if (!ROOM && o % 4 == 0) asm volatile("" ::: "memory");  // four coefficients live at a time (likewise)
        const double2_t p = cmul2(x, ROOM ? row[i & 1][o] : g[i * K + o]);
        if (i == 0) {
          ar[o] = p.x;
          ai[o] = p.y;
        } else if (i + 1 < K) {
          ar[o] = ar[o] + p.x;
          ai[o] = ai[o] + p.y;
        } else {
          add_to(re[idx[o]], ar[o], p.x);
          add_to(im[idx[o]], ai[o], p.y);
        }
      }
    }
  }
}

// Diagonal whose register bits are those of MASK: d holds 2^popcount(MASK)
// coefficients, indexed by them (highest bit most significant).
template <int R, int MASK>
__device__ __forceinline__ void rg_diag(double (&re)[1 << R], double (&im)[1 << R], const double2_t *d) {
  constexpr int NB = __builtin_popcount(MASK);
  constexpr int H = NB > 2 ? 2 : 1, NC = (1 << NB) / H;  // at most four coefficients live at a time
#pragma unroll
  for (int h = 0; h < H; ++h) {
    if (h) asm volatile("" ::: "memory");  // (a compiler barrier, no code)
    double2_t c[NC];
#pragma unroll
    for (int i = 0; i < NC; ++i) c[i] = d[h * NC + i];
#pragma unroll
    for (int r = 0; r < (1 << R); ++r) {
      int i = 0;
#pragma unroll
      for (int b = R - 1; b >= 0; --b)
        if ((MASK >> b) & 1) i = (i << 1) | ((r >> b) & 1);
      if (i / NC != h) continue;
      i %= NC;
      // All products before the first result takes its register.
      const double xc = re[r] * c[i].x, ys = im[r] * c[i].y, xs = re[r] * c[i].y, yc = im[r] * c[i].x;
      sub_to(re[r], xc, ys);
      add_to(im[r], xs, yc);
    }
  }
}

// Register bit k sits at tile bit (map >> 4 k) & 15.
template <int R>
__device__ __forceinline__ uint32_t reg_mask(uint32_t map) {
  uint32_t m = 0;
#pragma unroll
  for (int k = 0; k < R; ++k) m |= 1u << ((map >> (4 * k)) & 15u);
  return m;
}
// Tile index of this thread's element 0: the thread's bits with zeros at the register bits.
template <int R>
__device__ __forceinline__ uint32_t reg_base(uint32_t tid, uint32_t map) {
  uint32_t m = reg_mask<R>(map), base = tid;
#pragma unroll
  for (int k = 0; k < R; ++k) {
    const uint32_t low = m & (0u - m);
    m ^= low;
    base = ((base & ~(low - 1u)) << 1) | (base & (low - 1u));
  }
  return base;
}

// This thread's 2^R elements of a tile under one set of register bits: element
// r sits at lane | the state bits of r's register bits.
template <int R>
struct RegRefs {
  uint64_t lane = 0;
  uint64_t bit[R] = {};
  // where: state bits of the register bits (8 bits each).
  __device__ __forceinline__ void set(uint32_t tid, uint64_t tile_mask, uint32_t where) {
    uint64_t regs = 0;
#pragma unroll
    for (int k = 0; k < R; ++k) {
      bit[k] = 1ull << ((where >> (8 * k)) & 63u);
      regs |= bit[k];
    }
    lane = deposit_runs(tid, tile_mask & ~regs);
  }
  __device__ __forceinline__ uint64_t off(int r) const {
    uint64_t o = lane;
#pragma unroll
    for (int k = 0; k < R; ++k)
      if ((r >> k) & 1) o |= bit[k];
    return o;
  }
};

// KD: most qubits of a dense gate among the launch's ops.  MINW of 2: for launches
// that leave a compute unit one or two tiles, so one or two waves per SIMD that
// hide little of one another.  Registers and LDS are there to spare: an exchange
// takes both parts at once, and a gate of 2 or 3 qubits requests the next input's
// coefficients before this one's products.  20 qubits, one tile each: a 2-qubit
// gate 1.7 -> 1.4 us, a 3-qubit one 2.95 -> 2.6, an exchange 1.15 -> 0.8; 24 random
// 2-qubit gates 107 -> 93 us (86 with the tile in LDS between phases).  With four tiles
// (22 qubits) the 128-register form is the faster, 80 against 90 us for 24 1-qubit gates.
constexpr bool reg_room(int minw) { return minw <= 2; }
constexpr size_t reg_slot_bytes(int minw) { return reg_room(minw) ? sizeof(double2_t) : sizeof(double); }

template <int R, int KD, int MINW>
__global__ void __launch_bounds__(256, MINW)
    circuit_reg_kernel(const RunDesc *__restrict__ runs, int nruns, uint64_t total_tiles, int lds_tb) {
  constexpr int E = 1 << R;
  constexpr bool ROOM = reg_room(MINW);
  extern __shared__ double smem[];
  char *bytes = reinterpret_cast<char *>(smem);
  double2_t *cbuf = reinterpret_cast<double2_t *>(bytes + (reg_slot_bytes(MINW) << lds_tb));
  uint4 *obuf = reinterpret_cast<uint4 *>(cbuf + kRegCoef);
  const uint32_t thread = threadIdx.x;
  const RegChunk *staged = nullptr;  // the chunk now in LDS
  uint64_t gt = blockIdx.x;
  if (gt >= total_tiles) return;  // uniform: the whole workgroup leaves
  int run = find_run(runs, nruns, gt), run_in = -1, run_out = -1;
  RegRefs<R> in, out;
  double2_t amp[E];
  // Threads past the tile's (tiles of fewer bits than the launch's widest)
  // repeat another's work: the same values to the same slots, nothing to the
  // state.  (Their loads are over before the barriers of an exchange let the
  // others store; without an exchange they write nothing at all.)
  auto load = [&](int ri, uint64_t tile) {
    const RunDesc &D = runs[ri];
    if (run_in != ri) in.set(thread & ((1u << (D.tb - R)) - 1u), D.tile_mask, D.where_in);
    run_in = ri;
    const auto src =
        (const __attribute__((address_space(1))) double2_t *)(D.psi + deposit_runs64(tile - D.first, D.outer_mask));
#pragma unroll
    for (int r = 0; r < E; ++r) amp[r] = src[in.off(r)];
  };
  load(run, gt);
  while (true) {
    const RunDesc &D = runs[run];
    const uint64_t t = gt - D.first;
    const uint32_t nth = 1u << (D.tb - R);
    const bool live = thread < nth;
    const uint32_t tid = thread & (nth - 1u);
    const RegOp *ops = D.rops;
    const double2_t *coef = D.rcoef;
    double2_t *psi = D.psi + deposit_runs64(t, D.outer_mask);
    const auto chunks = as_const(D.rchunks);
    // Stages chunk c; the barrier before it ends the previous chunk's reads.
    auto stage = [&](const RegChunk *c, const RegChunk &h) {
      if (staged == c) return;
      staged = c;
      __syncthreads();
      for (uint32_t i = thread; i < h.op_end - h.op_begin; i += blockDim.x)
        obuf[i] = reinterpret_cast<const uint4 *>(ops)[h.op_begin + i];
      if (thread < 2) obuf[h.op_end - h.op_begin + thread] = uint4{0, 0, 0, 0};
      for (uint32_t i = thread; i < h.coef_end - h.coef_begin; i += blockDim.x) cbuf[i] = coef[h.coef_begin + i];
      __syncthreads();
    };
    uint32_t map = D.map0;
    uint32_t base = reg_base<R>(tid, map);
    // LDS places under these register bits (bytes): of element 0, and what each
    // register bit adds to it.
    uint32_t slot0, slotb[R];
    auto slots = [&]() {
      constexpr uint32_t kBytes = reg_slot_bytes(MINW);
      slot0 = reg_slot(base) * kBytes;
#pragma unroll
      for (int k = 0; k < R; ++k) slotb[k] = reg_slot_bit((map >> (4 * k)) & 15u) * kBytes;
    };
    slots();
    double re[E], im[E];
#pragma unroll
    for (int r = 0; r < E; ++r) {
      re[r] = amp[r].x;
      im[r] = amp[r].y;
    }
    const uint64_t gn = gt + gridDim.x;
    const bool more = gn < total_tiles;  // uniform
    const int run_next = more ? find_run(runs, nruns, gn) : run;
    for (uint32_t ci = D.chunk_begin; ci < D.chunk_end; ++ci) {
      RegChunk h;
      h.op_begin = chunks[ci].op_begin;
      h.op_end = chunks[ci].op_end;
      h.coef_begin = chunks[ci].coef_begin;
      h.coef_end = chunks[ci].coef_end;
      stage(D.rchunks + ci, h);
      const uint32_t c0 = h.coef_begin;
      uint32_t i = 0, code, co, lane, outer;
      uint4 rec = obuf[0];
      // Takes the record read ahead and reads the next one (a chunk ends with code 0).
      auto next = [&]() {
        code = __builtin_amdgcn_readfirstlane(rec.x);
        co = __builtin_amdgcn_readfirstlane(rec.y) - c0;
        lane = __builtin_amdgcn_readfirstlane(rec.z);
        outer = __builtin_amdgcn_readfirstlane(rec.w);
        rec = obuf[++i];
      };
      // A diagonal's coefficients of this lane: outer bits, then thread bits, pick the block.
      auto block = [&](int nr) {
        uint32_t s = 0;
        if (outer != kRegNoOuter) {
          s = (uint32_t)((t >> (outer & 63u)) & 1u) << 2 | (uint32_t)((t >> ((outer >> 8) & 63u)) & 1u) << 1 |
              (uint32_t)((t >> ((outer >> 16) & 63u)) & 1u);
          s <<= lane >> 24;
        }
        const uint32_t l = ((base >> (lane & 31u)) & 1u) << 2 | ((base >> ((lane >> 8) & 31u)) & 1u) << 1 |
                           ((base >> ((lane >> 16) & 31u)) & 1u);
        return cbuf + co + ((s | l) << nr);
      };
      // Every form is an `if` of its own that changes the amplitudes in place
      // (not one of a switch's exclusive branches): the compiler structures
      // those one after another with copies of the amplitudes between them.
      // A diagonal's form repeats while the records stay of that form.
      next();
      while (code) {
        if (code & 0xfu) {
          const double2_t *g = cbuf + co;
#define QTNH_REG_G1(A)                    \
  if constexpr (A < R)                    \
    if (code & (1u << A)) {               \
      rg_gate1<R, A>(re, im, g);          \
      g += 4;                             \
    }
          QTNH_REG_G1(3)
          QTNH_REG_G1(2)
          QTNH_REG_G1(1)
          QTNH_REG_G1(0)
#undef QTNH_REG_G1
          if (lane & kRegSettle) rg_settle<R>(re, im);
          next();
        }
#define QTNH_REG_DIAG(BIT, NEED, MASK)                                   \
  if constexpr (NEED < R)                                                \
    while (code & (1u << BIT)) {                                         \
      rg_diag<R, MASK>(re, im, block(__builtin_popcount(MASK)));         \
      next();                                                            \
    }
        if (code & (0x1fu << kRegD0)) {
          QTNH_REG_DIAG(17, 0, 0)
          QTNH_REG_DIAG(18, 0, 1)
          QTNH_REG_DIAG(19, 1, 2)
          QTNH_REG_DIAG(20, 2, 4)
          QTNH_REG_DIAG(21, 3, 8)
        }
        if (code & (0x3fu << kRegD2)) {
          QTNH_REG_DIAG(22, 1, 3)
          QTNH_REG_DIAG(23, 2, 5)
          QTNH_REG_DIAG(24, 2, 6)
          QTNH_REG_DIAG(25, 3, 9)
          QTNH_REG_DIAG(26, 3, 10)
          QTNH_REG_DIAG(27, 3, 12)
        }
        if (code & (0xfu << kRegD3)) {
          QTNH_REG_DIAG(28, 2, 7)
          QTNH_REG_DIAG(29, 3, 11)
          QTNH_REG_DIAG(30, 3, 13)
          QTNH_REG_DIAG(31, 3, 14)
        }
#undef QTNH_REG_DIAG
        if constexpr (KD > 1) if (code & (0xfffu << kRegG2)) {
#define QTNH_REG_CASE(BIT, NEED, CALL) \
  if constexpr (NEED < R)              \
    if (code & (1u << BIT)) CALL;
          QTNH_REG_CASE(4, 1, (rg_gate<R, 2, 0, 1, 0, ROOM>(re, im, cbuf + co)))
          QTNH_REG_CASE(5, 2, (rg_gate<R, 2, 0, 2, 0, ROOM>(re, im, cbuf + co)))
          QTNH_REG_CASE(6, 3, (rg_gate<R, 2, 0, 3, 0, ROOM>(re, im, cbuf + co)))
          QTNH_REG_CASE(7, 1, (rg_gate<R, 2, 1, 0, 0, ROOM>(re, im, cbuf + co)))
          QTNH_REG_CASE(8, 2, (rg_gate<R, 2, 1, 2, 0, ROOM>(re, im, cbuf + co)))
          QTNH_REG_CASE(9, 3, (rg_gate<R, 2, 1, 3, 0, ROOM>(re, im, cbuf + co)))
          QTNH_REG_CASE(10, 2, (rg_gate<R, 2, 2, 0, 0, ROOM>(re, im, cbuf + co)))
          QTNH_REG_CASE(11, 2, (rg_gate<R, 2, 2, 1, 0, ROOM>(re, im, cbuf + co)))
          QTNH_REG_CASE(12, 3, (rg_gate<R, 2, 2, 3, 0, ROOM>(re, im, cbuf + co)))
          QTNH_REG_CASE(13, 3, (rg_gate<R, 2, 3, 0, 0, ROOM>(re, im, cbuf + co)))
          QTNH_REG_CASE(14, 3, (rg_gate<R, 2, 3, 1, 0, ROOM>(re, im, cbuf + co)))
          QTNH_REG_CASE(15, 3, (rg_gate<R, 2, 3, 2, 0, ROOM>(re, im, cbuf + co)))
#undef QTNH_REG_CASE
          if (lane & kRegSettle) rg_settle<R>(re, im);
          next();
        }
        if (code & (1u << kRegSpecial)) {
          if constexpr (KD > 2 && R > 2) {
            if (!(lane & kRegRemapFlag)) rg_gate<R, 3, 2, 1, 0, ROOM>(re, im, cbuf + co);
            if (lane & kRegSettle) rg_settle<R>(re, im);
          }
          if (lane & kRegRemapFlag) {
            const uint32_t s0 = slot0;
            uint32_t sb[R];
#pragma unroll
            for (int k = 0; k < R; ++k) sb[k] = slotb[k];
            map = lane;
            base = reg_base<R>(tid, map);
            slots();
            // Element r's place in LDS (bytes).
            auto at = [](uint32_t s, const uint32_t (&b)[R], int r) {
              uint32_t x = 0;
#pragma unroll
              for (int k = 0; k < R; ++k)
                if ((r >> k) & 1) x ^= b[k];
              return s ^ x;
            };
            lds_barrier();  // the previous exchange has been read
            if constexpr (ROOM) {
#pragma unroll
              for (int r = 0; r < E; ++r) *reinterpret_cast<double2_t *>(bytes + at(s0, sb, r)) = double2_t{re[r], im[r]};
              lds_barrier();
#pragma unroll
              for (int r = 0; r < E; ++r) {
                const double2_t x = *reinterpret_cast<const double2_t *>(bytes + at(slot0, slotb, r));
                re[r] = x.x;
                im[r] = x.y;
              }
            } else {
#pragma unroll
              for (int r = 0; r < E; ++r) *reinterpret_cast<double *>(bytes + at(s0, sb, r)) = re[r];
              lds_barrier();
#pragma unroll
              for (int r = 0; r < E; ++r) re[r] = *reinterpret_cast<const double *>(bytes + at(slot0, slotb, r));
              lds_barrier();
#pragma unroll
              for (int r = 0; r < E; ++r) *reinterpret_cast<double *>(bytes + at(s0, sb, r)) = im[r];
              lds_barrier();
#pragma unroll
              for (int r = 0; r < E; ++r) im[r] = *reinterpret_cast<const double *>(bytes + at(slot0, slotb, r));
            }
          }
          next();
        }
      }
    }
    // Write back under the last register bits.
    if (run_out != run) out.set(tid, D.tile_mask, D.where_out);
    run_out = run;
    const auto dst = (__attribute__((address_space(1))) double2_t *)(psi);
    if (live) {
#pragma unroll
      for (int r = 0; r < E; ++r) dst[out.off(r)] = double2_t{re[r], im[r]};
    }
    if (!more) break;
    gt = gn;
    run = run_next;
    load(run, gt);
  }
}

// ---- <Z_q> for a list of qubits --------------------------------------------
// Chunks of 2^kChunkBits consecutive amplitudes.  Per chunk: the total
// probability and, for each of the chunk's own index bits, the probability
// with that bit set (slot s of chunk c at part[s nchunks + c]).  Bits above the
// chunk are constant inside it.
constexpr int kChunkBits = 12;
constexpr int kZThreads = 256;
constexpr int kZSlots = 1 + kChunkBits;

// Memory bounds it: a thread's 16 amplitudes are requested together, and of the
// 13 sums over the threads those of the low eight bits are taken from the same
// totals as the chunk's own, a quarter of them by each wave, with one barrier a
// chunk.  2^20 amplitudes: 4.8 us, and 13.7 with a tree of eight barriers for every
// sum; 2^28: 720 us and 890.  FULL: the chunk has 2^kChunkBits amplitudes.  NT:
// non-temporal loads, for states beyond the 256 MB cache (2^26 amplitudes: 203 us a
// call, 219 without; 2^24: 67 us a call, 62.6 without).
template <bool FULL, bool NT>
__global__ void __launch_bounds__(kZThreads) zchunk_kernel(const double2_t *__restrict__ psi, int cb,
                                                           double *__restrict__ part, uint64_t nchunks) {
  constexpr int kEach = (1 << kChunkBits) / kZThreads, kHigh = kChunkBits - 8;
  __shared__ double red[1 + kHigh][kZThreads];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const uint64_t ch = blockIdx.x;
  // Thread t owns chunk elements t + kZThreads j: bits 0..7 of the element are t's bits.
  double2_t v[kEach];
#pragma unroll
  for (int j = 0; j < kEach; ++j) {
    const int l = tid + kZThreads * j;
    const double2_t *p = psi + (ch << cb) + l;
    v[j] = double2_t{0.0, 0.0};
    if (FULL || l < 1 << cb) v[j] = NT ? __builtin_nontemporal_load(p) : *p;
  }
  double tot = 0.0, hib[kHigh] = {};
#pragma unroll
  for (int j = 0; j < kEach; ++j) {
    double p = v[j].x * v[j].x;
    p = p + v[j].y * v[j].y;
    tot = tot + p;
#pragma unroll
    for (int b = 0; b < kHigh; ++b)
      if (j >> b & 1) hib[b] = hib[b] + p;
  }
  red[0][tid] = tot;
#pragma unroll
  for (int b = 0; b < kHigh; ++b) red[1 + b][tid] = hib[b];
  __syncthreads();
  // slot 0: total; slot 1 + b: probability with bit b set.
#pragma unroll
  for (int i = 0; i < (kZSlots + 3) / 4; ++i) {
    const int s = wave + 4 * i, b = s - 1;
    if (s >= kZSlots) break;
    const double *r = red[s > 8 ? s - 8 : 0];
    double x[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const double y = r[64 * k + lane];
      x[k] = s == 0 || s > 8 || (64 * k + lane) >> b & 1 ? y : 0.0;
    }
    double sum = (x[0] + x[2]) + (x[1] + x[3]);
#pragma unroll
    for (int w = 32; w > 0; w >>= 1) sum = sum + __shfl_down(sum, w, 64);
    if (lane == 0) part[(uint64_t)s * nchunks + ch] = sum;
  }
}

struct ZQubits {
  uint8_t bit[kHostScalars];
};

// One workgroup per requested qubit: <Z_b> = sum over chunks of (total - 2 set_b),
// eight of a thread's chunks read at a time (2^16 chunks: 41 us, 138 one at a time
// from a table of 13 slots a chunk).
__global__ void __launch_bounds__(kZThreads) zfinal_kernel(const double *__restrict__ part, uint64_t nchunks, int cb,
                                                           ZQubits qubits, double *__restrict__ out) {
  __shared__ double red[kZThreads];
  const int b = qubits.bit[blockIdx.x];
  const bool inside = b < cb;
  const double *set = part + (inside ? (uint64_t)(1 + b) * nchunks : 0);
  double s = 0.0;
  for (uint64_t c0 = threadIdx.x; c0 < nchunks; c0 += 8 * kZThreads) {
    double tot[8], on[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const uint64_t ch = c0 + j * kZThreads < nchunks ? c0 + j * kZThreads : c0;
      tot[j] = part[ch];
      on[j] = set[ch];
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const uint64_t ch = c0 + j * kZThreads;
      if (ch >= nchunks) break;
      double v;
      if (inside)
        v = tot[j] - 2.0 * on[j];
      else
        v = (((ch << cb) >> b) & 1) ? -tot[j] : tot[j];
      s = s + v;
    }
  }
  red[threadIdx.x] = s;
  __syncthreads();
  for (int w = kZThreads / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] = red[threadIdx.x] + red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[blockIdx.x] = red[0];
}

}  // namespace
}  // namespace qtnh_hip

using qtnh_hip::c128;
using qtnh_hip::RegChunk;
using qtnh_hip::RegOp;
using qtnh_hip::RunDesc;
using qtnh_hip::TileOp;

// ---- host side ---------------------------------------------------------------
struct qtnh_circuit_s {
  struct Op {
    int kind;  // 0 gate, 1 diagonal
    int k;
    uint16_t q[3];
    std::vector<double> coef;  // interleaved complex: gates (2^k)^2, diagonals 2^k
  };
  int n = 0;
  std::vector<Op> ops;
  // Tile shape chosen for this circuit by qtnh_circuit_tune (0: the context's).
  int tuned_tb = 0, tuned_low = 0;
  struct Run {
    uint32_t begin, end;
    std::vector<int> tbits;  // ascending state bits
  };
  // Register form of the runs with some number of register bits (ops null: not built).
  struct RegForm {
    const RegOp *ops = nullptr;
    const RegChunk *chunks = nullptr;
    const qtnh_hip::double2_t *coef = nullptr;
    struct Run {
      uint32_t chunk_begin, chunk_end, map0, where_in, where_out;
    };
    std::vector<Run> runs;
  };
  // The ops compiled for one tile shape on one device.
  struct Compiled {
    int n = 0;  // qubits
    int tb = 0, low = 0, device = -1;
    void *dev = nullptr;  // everything below that is on the device
    const TileOp *ops = nullptr;
    const qtnh_hip::double2_t *coef = nullptr;
    std::vector<Run> runs;
    std::vector<TileOp> tops;  // host copy of the compiled ops
    RegForm forms[qtnh_hip::kMaxRegBits + 1];  // by register bits
    bool has3 = false;  // a dense 3-qubit gate among the ops
    // Uploaded run descriptors of fused runs, per state buffer: a repeated run
    // on the same state launches kernels only (no copy), so it can be captured
    // into a graph.
    struct DescCache {
      RunDesc *d = nullptr;
      std::vector<RunDesc> h;
      std::vector<size_t> starts;
    };
    std::map<const void *, DescCache> desc_cache;
  };
  // One for each tile shape and device the circuit has run with since ops were
  // last appended.  A graph captured from a fused run reads its memory, so all of
  // them are kept until ops are appended or the circuit is destroyed.
  std::vector<std::unique_ptr<Compiled>> compiled;
  size_t compiled_ops = 0;
};

namespace qtnh_hip {
namespace {

int g_tile_bits = 0;  // 0: by the state's size (default_tile)
// 2 (and 3): register kernel for tiles of 4 to 12 bits; 1: pipelined LDS kernel
// for many 12-bit tiles; 0: plain LDS kernel.
int g_circuit_mode = 2;
int g_low_bits = 4;  // lowest state bits in every tile: 2^4 x 16 B = 256 B contiguous rows

// Tile bits and low bits of an n-qubit circuit in launches over about 2^bits
// amplitudes (its own state's and the others' of a batch), where nothing else is
// set.  12-bit tiles make the fewest passes, which large states need; a launch of
// fewer tiles than compute units is bound by one tile's latency and takes smaller
// tiles, more passes over more workgroups (12 / 10-bit tiles: QFT-12 35 / 24 us,
// random circuits of 16 and 18 qubits 168 / 124 and 163 / 126; 11 bits at 19
// qubits 262 / 228; at 20 qubits 372 us with 12 bits, 431 with 11).  So do
// batches: depth-4 random circuits, 10 / 11 / 12 bits, 8 of 15 qubits 79 / 84 / 102
// us, 16 of them 107 / 98 / 113, 16 of 16 qubits 179 / 158 / 135; of 19 qubits 11
// bits are the best for two, too (175, and 194 with 12).  States that one tile
// holds need a single pass, which eight of them make faster than two over smaller
// tiles (32 of 12 qubits 84 / 87 / 60).
void default_tile(int n, int bits, int *tb, int *low) {
  const bool large = bits >= (n == 19 ? 21 : 20) || (n <= 12 && bits >= n + 3);
  *tb = g_tile_bits ? g_tile_bits : large ? 12 : bits >= 19 ? 11 : 10;
  *low = g_tile_bits ? g_low_bits : large ? 4 : 3;
}

// State bits an op needs inside the tile: all of a gate's; none of a
// diagonal's (a qubit outside the tile is fixed per tile and selects the
// diagonal's coefficients there).
uint64_t mask_of(const qtnh_circuit_s &c, const qtnh_circuit_s::Op &op) {
  uint64_t m = 0;
  if (op.kind == 1) return 0;
  for (int j = 0; j < op.k; ++j) m |= 1ull << (c.n - 1 - op.q[j]);
  return m;
}

// Greedy partition of the op sequence into runs of at most tb distinct gate
// bits, each widened with the lowest free bits (coalesced tile rows) up to
// tb.  Runs are contiguous in op order, so every amplitude sees the ops in
// program order; with that constraint the greedy (longest feasible run first)
// gives the fewest runs.
std::vector<qtnh_circuit_s::Run> plan_runs(const qtnh_circuit_s &c, int tb, int low_bits) {
  std::vector<qtnh_circuit_s::Run> runs;
  const int tbe = std::min(tb, c.n);
  const uint64_t low = (1ull << std::min(std::min(low_bits, tbe - 3 > 0 ? tbe - 3 : 0), c.n)) - 1;
  uint64_t cur = low;
  uint32_t begin = 0;
  auto close = [&](uint32_t end) {
    if (end == begin) return;
    uint64_t m = cur;
    for (int b = 0; b < c.n && __builtin_popcountll(m) < tbe; ++b) m |= 1ull << b;
    qtnh_circuit_s::Run r;
    r.begin = begin;
    r.end = end;
    for (int b = 0; b < c.n; ++b)
      if ((m >> b) & 1) r.tbits.push_back(b);
    runs.push_back(r);
  };
  for (uint32_t i = 0; i < c.ops.size(); ++i) {
    const uint64_t m = mask_of(c, c.ops[i]);
    if (__builtin_popcountll(cur | m) > tbe) {
      close(i);
      begin = i;
      cur = low;
    }
    cur |= m;
  }
  close((uint32_t)c.ops.size());
  return runs;
}

using Compiled = qtnh_circuit_s::Compiled;

// Frees every compiled form (the caller has drained the streams that used them).
void free_compiled(qtnh_circuit_s &c) {
  for (const auto &k : c.compiled) {
    if (k->dev) (void)hipFree(k->dev);
    for (auto &d : k->desc_cache)
      if (d.second.d) (void)hipFree(d.second.d);
  }
  c.compiled.clear();
}

// Register bits for a launch of runs of tb-bit tiles: 64 to 256 threads per
// tile.  More amplitudes per thread mean fewer exchanges and less decoding per
// amplitude, fewer mean more waves per tile, which small tiles need (random
// circuit of 16 qubits, 10-bit tiles: 124 us with 2 register bits, 138 with 3,
// 171 with 4; 24 qubits, 12-bit tiles: 3.74 ms with 2, 2.19 with 3, 1.88 with
// 4).  A dense 3-qubit gate needs three.
int reg_bits(int tb, bool has3) { return std::max(has3 ? 3 : kMinRegBits, std::min(tb - 8, kMaxRegBits)); }

// Register forms a circuit with tb-bit tiles needs: the one for its own runs,
// and the widest (launches that mix circuits of several widths).
bool wants_form(int tb, bool has3, int R) {
  if (tb < kMaxRegBits || tb > 12) return false;
  return R == kMaxRegBits || R == reg_bits(tb, has3);
}

// The register form (R register bits) of run r: appends its ops, coefficients
// and staging chunks.  Consecutive ops whose dense gates fit R tile bits share
// their register bits; free ones take the highest tile bits, so that threads
// vary in the lowest (a read or write of the state then covers whole 128-byte
// lines; where the first or last gates need one of the lowest three bits, an
// exchange is put before or after them instead).
void plan_reg_run(const qtnh_circuit_s &c, const qtnh_circuit_s::Run &r, int R, std::vector<RegOp> &ops,
                  std::vector<double> &coef, std::vector<RegChunk> &chunks,
                  qtnh_circuit_s::RegForm::Run *fr) {
  const int tb = (int)r.tbits.size();
  struct Seg {
    uint32_t begin, end;
    int pos[kMaxRegBits];  // tile bit of each register bit
  };
  auto tile_bit = [&](int q) {
    const auto it = std::lower_bound(r.tbits.begin(), r.tbits.end(), c.n - 1 - q);
    return it != r.tbits.end() && *it == c.n - 1 - q ? (int)(it - r.tbits.begin()) : -1;
  };
  std::vector<Seg> segs;
  uint32_t cur = 0, begin = r.begin;
  bool fixed = false;
  int fpos[kMaxRegBits];
  auto close = [&](uint32_t end) {
    if (end == begin) return;
    Seg s;
    s.begin = begin;
    s.end = end;
    if (fixed) {
      memcpy(s.pos, fpos, sizeof(fpos));
    } else {
      uint32_t m = cur;
      for (int b = tb - 1; b >= 0 && __builtin_popcount(m) < R; --b) m |= 1u << b;
      int k = 0;
      for (int b = 0; b < tb; ++b)
        if ((m >> b) & 1) s.pos[k++] = b;
    }
    segs.push_back(s);
    begin = end;
    cur = 0;
    fixed = false;
  };
  for (uint32_t i = r.begin; i < r.end; ++i) {
    const auto &op = c.ops[i];
    if (op.kind == 1) continue;
    uint32_t m = 0;
    for (int j = 0; j < op.k; ++j) m |= 1u << tile_bit(op.q[j]);
    if (op.k == 3) {
      // Its qubits take register bits 2, 1, 0 in this order.
      if (cur) close(i);  // (diagonals alone join this gate's register bits)
      fixed = true;
      for (int j = 0; j < 3; ++j) fpos[2 - j] = tile_bit(op.q[j]);
      cur = m;
      for (int b = tb - 1, k = 3; k < R; --b)
        if (!((cur >> b) & 1)) {
          fpos[k++] = b;
          cur |= 1u << b;
        }
    } else if (__builtin_popcount(cur | m) > R) {
      close(i);
      cur = m;
    } else {
      cur |= m;
    }
  }
  close(r.end);
  auto pack = [&](const int *pos) {
    uint32_t m = 0;
    for (int k = 0; k < R; ++k) m |= (uint32_t)pos[k] << (4 * k);
    return m;
  };
  int top[kMaxRegBits];
  for (int k = 0; k < R; ++k) top[k] = tb - R + k;
  // Whether the state is read and written in whole lines under these register bits.
  auto whole_lines = [&](const int *pos) {
    for (int k = 0; k < R; ++k)
      if (pos[k] < std::min(3, tb - R)) return false;
    return true;
  };
  uint32_t chunk_op = (uint32_t)ops.size(), chunk_coef = (uint32_t)(coef.size() / 2);
  auto end_chunk = [&]() {
    if (ops.size() == chunk_op) return;
    chunks.push_back(RegChunk{chunk_op, (uint32_t)ops.size(), chunk_coef, (uint32_t)(coef.size() / 2)});
    chunk_op = (uint32_t)ops.size();
    chunk_coef = (uint32_t)(coef.size() / 2);
  };
  auto room = [&](size_t ncoef) {
    if (ops.size() - chunk_op + 1 > (size_t)kRegOps || coef.size() / 2 - chunk_coef + ncoef > (size_t)kRegCoef)
      end_chunk();
  };
  uint32_t map = 0;
  auto remap = [&](const int *pos) {
    if (pack(pos) == map) return;
    map = pack(pos);
    room(0);
    ops.push_back(RegOp{1u << kRegSpecial, (uint32_t)(coef.size() / 2), map | kRegRemapFlag, 0});
  };
  map = fr->map0 = pack(!segs.empty() && whole_lines(segs[0].pos) ? segs[0].pos : top);
  for (const Seg &s : segs) {
    remap(s.pos);
    auto reg_bit = [&](int tbit) {
      for (int k = 0; k < R; ++k)
        if (s.pos[k] == tbit) return k;
      return -1;
    };
    for (uint32_t i = s.begin; i < s.end; ++i) {
      const auto &op = c.ops[i];
      const size_t ncoef = op.coef.size() / 2;
      room(ncoef);
      RegOp o{0, (uint32_t)(coef.size() / 2), 0, 0};
      if (op.kind == 0) {
        // A diagonal comes next, or the circuit ends (a run ends before a dense gate).
        if (i + 1 == c.ops.size() || c.ops[i + 1].kind == 1) o.lane = kRegSettle;
        const int a = reg_bit(tile_bit(op.q[0])), b = op.k > 1 ? reg_bit(tile_bit(op.q[1])) : 0;
        // A 1-qubit gate joins the record before it if its register bit is below all of that one's.
        RegOp *prev = ops.size() > chunk_op ? &ops.back() : nullptr;
        const bool join = op.k == 1 && prev && prev->code && prev->code < 16u && (prev->code & ((2u << a) - 1u)) == 0;
        if (join) {
          prev->code |= 1u << a;
          prev->lane |= o.lane;
        } else {
          o.code = 1u << (op.k == 1 ? kRegG1 + a : op.k == 2 ? kRegG2 + 3 * a + (b > a ? b - 1 : b) : kRegSpecial);
        }
        coef.insert(coef.end(), op.coef.begin(), op.coef.end());
        if (!join) ops.push_back(o);
        continue;
      }
      // Table order, most significant first: outer bits, thread bits, register bits from the highest.
      int order[3], no = 0, nl = 0, nr = 0, regs = 0;
      o.lane = kRegNoLane;
      o.outer = kRegNoOuter;
      for (int j = 0; j < op.k; ++j)
        if (tile_bit(op.q[j]) < 0) {
          const int sb = c.n - 1 - op.q[j];
          const int below = (int)(std::lower_bound(r.tbits.begin(), r.tbits.end(), sb) - r.tbits.begin());
          o.outer = (o.outer >> 8) | (uint32_t)(sb - below) << 16;
          order[no++] = j;
        }
      for (int j = 0; j < op.k; ++j)
        if (tile_bit(op.q[j]) >= 0 && reg_bit(tile_bit(op.q[j])) < 0) {
          o.lane = (o.lane >> 8) | (uint32_t)tile_bit(op.q[j]) << 16;
          order[no + nl++] = j;
        }
      for (int k = R - 1; k >= 0; --k)
        for (int j = 0; j < op.k; ++j)
          if (tile_bit(op.q[j]) >= 0 && reg_bit(tile_bit(op.q[j])) == k) {
            order[no + nl + nr++] = j;
            regs |= 1 << k;
          }
      o.lane |= (uint32_t)nl << 24;
      const int hi = 31 - __builtin_clz((unsigned)regs | 1u), lo = __builtin_ctz((unsigned)regs | 16u);
      o.code = 1u << (nr == 0   ? kRegD0
                      : nr == 1 ? kRegD1 + hi
                      : nr == 2 ? kRegD2 + hi * (hi - 1) / 2 + lo
                                : kRegD3 + 3 - __builtin_ctz(~(unsigned)regs));
      for (int x = 0; x < (1 << op.k); ++x) {
        int idx = 0;
        for (int m = 0; m < op.k; ++m)
          if ((x >> (op.k - 1 - m)) & 1) idx |= 1 << (op.k - 1 - order[m]);
        coef.push_back(op.coef[2 * idx]);
        coef.push_back(op.coef[2 * idx + 1]);
      }
      ops.push_back(o);
    }
  }
  if (!segs.empty() && !whole_lines(segs.back().pos)) remap(top);
  end_chunk();
  auto where = [&](uint32_t packed) {
    uint32_t w = 0;
    for (int k = 0; k < R; ++k) w |= (uint32_t)r.tbits[(packed >> (4 * k)) & 15u] << (8 * k);
    return w;
  };
  fr->where_in = where(fr->map0);
  fr->where_out = where(map);
}

// Device tables gathered on the host, for one allocation and one copy.
struct Tables {
  std::vector<char> host;
  template <typename T>
  size_t add(const std::vector<T> &v) {
    const size_t at = (host.size() + 255) & ~(size_t)255, bytes = v.size() * sizeof(T);
    host.resize(at + bytes);
    if (bytes) memcpy(host.data() + at, v.data(), bytes);
    return at;
  }
};

// Tile shape for an n-qubit circuit in launches over about 2^bits amplitudes: the
// autotuned one of this context, else the process default.
void tile_shape(qtnh_ctx_t ctx, int n, int bits, int *tb, int *low) {
  const bool tuned = n < 64 && ctx->circ_tb[n] > 0;
  default_tile(n, bits, tb, low);
  if (!tuned) return;
  *tb = ctx->circ_tb[n];
  *low = ctx->circ_low[n];
}

// ... and for a circuit: its own tuned one first.
void tile_shape(qtnh_ctx_t ctx, const qtnh_circuit_s &c, int bits, int *tb, int *low) {
  tile_shape(ctx, c.n, bits, tb, low);
  if (c.tuned_tb <= 0) return;
  *tb = c.tuned_tb;
  *low = c.tuned_low;
}

// The circuit compiled on the context's device, for its tile shape in launches
// over about 2^bits amplitudes.
qtnh_status compile(qtnh_ctx_t ctx, qtnh_circuit_s &c, int bits, Compiled **out) {
  int tb, low;
  tile_shape(ctx, c, bits, &tb, &low);
  if (c.compiled_ops != c.ops.size() && !c.compiled.empty()) {
    qtnh_status st = check_hip(ctx, hipStreamSynchronize(ctx->stream), "circuit recompile sync");
    if (st) return st;
    free_compiled(c);
  }
  c.compiled_ops = c.ops.size();
  for (const auto &k : c.compiled)
    if (k->tb == tb && k->low == low && k->device == ctx->device) {
      *out = k.get();
      return QTNH_OK;
    }
  std::unique_ptr<Compiled> k(new Compiled);
  k->n = c.n;
  k->tb = tb;
  k->low = low;
  k->device = ctx->device;
  k->runs = plan_runs(c, tb, low);
  for (const auto &op : c.ops) k->has3 = k->has3 || (op.kind == 0 && op.k == 3);
  std::vector<TileOp> tops(std::max<size_t>(c.ops.size(), 1));
  std::vector<double> coef;
  for (const auto &r : k->runs) {
    for (uint32_t i = r.begin; i < r.end; ++i) {
      const auto &op = c.ops[i];
      TileOp t;
      memset(&t, 0, sizeof(t));
      t.kind = op.kind;
      t.coef = (uint32_t)(coef.size() / 2);
      // Op-index bits j inside the tile (tj) and outside it (oj, diagonals only).
      int tj[3], oj[3], nt = 0, no = 0;
      for (int j = 0; j < op.k; ++j) {
        const int sb = c.n - 1 - op.q[j];
        const auto it = std::find(r.tbits.begin(), r.tbits.end(), sb);
        if (it != r.tbits.end()) {
          t.pos[nt] = (int)(it - r.tbits.begin());
          t.zpos[nt] = t.pos[nt];
          tj[nt++] = j;
        } else {
          // Bit of the tile number: the state bit's rank among the bits outside the tile.
          const int below = (int)(std::lower_bound(r.tbits.begin(), r.tbits.end(), sb) - r.tbits.begin());
          t.outer |= (uint32_t)(sb - below) << (8 + 8 * no);
          oj[no++] = j;
        }
      }
      if (op.kind == 0 && no) return set_error(ctx, QTNH_EINVAL, "circuit: gate outside its tile (planner)");
      t.kb = nt;
      t.outer |= (uint32_t)no;
      std::sort(t.zpos, t.zpos + nt);
      if (op.kind == 0 || no == 0) {
        coef.insert(coef.end(), op.coef.begin(), op.coef.end());
      } else {
        // Block o (outer bits, op order) holds the 2^nt coefficients of the tile bits.
        for (int o = 0; o < (1 << no); ++o)
          for (int tt = 0; tt < (1 << nt); ++tt) {
            int idx = 0;
            for (int m = 0; m < nt; ++m)
              if ((tt >> (nt - 1 - m)) & 1) idx |= 1 << (op.k - 1 - tj[m]);
            for (int m = 0; m < no; ++m)
              if ((o >> (no - 1 - m)) & 1) idx |= 1 << (op.k - 1 - oj[m]);
            coef.push_back(op.coef[2 * idx]);
            coef.push_back(op.coef[2 * idx + 1]);
          }
      }
      tops[i] = t;
    }
  }
  if (coef.empty()) coef.assign(2, 0.0);
  Tables tables;
  const size_t ops_at = tables.add(tops), coef_at = tables.add(coef);
  size_t form_at[kMaxRegBits + 1][3] = {};
  for (int R = kMinRegBits; R <= kMaxRegBits; ++R) {
    if (!wants_form(std::min(tb, c.n), k->has3, R)) continue;
    std::vector<RegOp> rops;
    std::vector<RegChunk> chunks;
    std::vector<double> rcoef;
    for (const auto &r : k->runs) {
      qtnh_circuit_s::RegForm::Run fr;
      fr.chunk_begin = (uint32_t)chunks.size();
      plan_reg_run(c, r, R, rops, rcoef, chunks, &fr);
      fr.chunk_end = (uint32_t)chunks.size();
      k->forms[R].runs.push_back(fr);
    }
    form_at[R][0] = tables.add(rops);
    form_at[R][1] = tables.add(chunks);
    form_at[R][2] = tables.add(rcoef);
  }
  tables.host.resize(tables.host.size() + 16);  // (an address for empty tables)
  qtnh_status st = check_hip(ctx, hipMalloc(&k->dev, tables.host.size()), "circuit alloc");
  if (st) return st;
  st = check_hip(ctx, hipMemcpyAsync(k->dev, tables.host.data(), tables.host.size(), hipMemcpyHostToDevice, ctx->stream),
                 "circuit upload");
  if (st) {
    (void)hipStreamSynchronize(ctx->stream);
    (void)hipFree(k->dev);
    return st;
  }
  const char *dev = (const char *)k->dev;
  k->ops = (const TileOp *)(dev + ops_at);
  k->coef = (const double2_t *)(dev + coef_at);
  for (int R = kMinRegBits; R <= kMaxRegBits; ++R) {
    if (!wants_form(std::min(tb, c.n), k->has3, R)) continue;
    k->forms[R].ops = (const RegOp *)(dev + form_at[R][0]);
    k->forms[R].chunks = (const RegChunk *)(dev + form_at[R][1]);
    k->forms[R].coef = (const double2_t *)(dev + form_at[R][2]);
  }
  k->tops = std::move(tops);
  c.compiled.push_back(std::move(k));
  *out = c.compiled.back().get();
  return QTNH_OK;
}

// Descriptor of run ri on psi, with its register form of R bits (0: none).
RunDesc make_desc(const Compiled &c, size_t ri, c128 *psi, uint64_t first, int R) {
  const qtnh_circuit_s::Run &r = c.runs[ri];
  RunDesc d;
  memset(&d, 0, sizeof(d));
  if (R) {
    const auto &f = c.forms[R];
    d.rops = f.ops;
    d.rcoef = f.coef;
    d.rchunks = f.chunks;
    d.chunk_begin = f.runs[ri].chunk_begin;
    d.chunk_end = f.runs[ri].chunk_end;
    d.map0 = f.runs[ri].map0;
    d.where_in = f.runs[ri].where_in;
    d.where_out = f.runs[ri].where_out;
    d.rbits = R;
  }
  d.ops = c.ops;
  d.coef = c.coef;
  d.psi = (double2_t *)psi;
  d.first = first;
  d.op_begin = r.begin;
  d.op_end = r.end;
  d.coef_begin = r.begin < c.tops.size() ? c.tops[r.begin].coef : 0;
  d.tb = (int)r.tbits.size();
  uint64_t tile = 0;
  for (size_t j = 0; j < r.tbits.size(); ++j) tile |= 1ull << r.tbits[j];
  d.tile_mask = tile;
  const uint64_t all = c.n == 64 ? ~0ull : ((1ull << c.n) - 1);
  d.outer_mask = all & ~tile;
  d.n_outer = __builtin_popcountll(d.outer_mask);
  return d;
}

uint64_t desc_tiles(const RunDesc &d) { return 1ull << d.n_outer; }

// Run ri of circuit c on psi, one of a launch's runs.
struct RunRef {
  const Compiled *c;
  size_t ri;
  c128 *psi;
};

// Appends one launch's descriptors.  All runs of a launch take register forms
// of one width: the width these tiles want, where every circuit has built it,
// else the widest.
void add_group(const std::vector<RunRef> &refs, std::vector<RunDesc> &descs, std::vector<size_t> &starts) {
  starts.push_back(descs.size());
  int tb_max = 0;
  bool has3 = false;
  for (const RunRef &r : refs) {
    tb_max = std::max(tb_max, (int)r.c->runs[r.ri].tbits.size());
    has3 = has3 || r.c->has3;
  }
  int R = reg_bits(tb_max, has3);
  for (const RunRef &r : refs)
    if (!r.c->forms[R].ops) {
      R = kMaxRegBits;
      break;
    }
  for (const RunRef &r : refs)
    if (!r.c->forms[R].ops) {
      R = 0;
      break;
    }
  uint64_t first = 0;
  for (const RunRef &r : refs) {
    descs.push_back(make_desc(*r.c, r.ri, r.psi, first, R));
    descs.back().has3 = has3;
    first += desc_tiles(descs.back());
  }
}

// One workgroup per tile (a grid of resident workgroups walking the tiles ran
// 10% longer at 28 qubits: its workgroups stay in step, all loading at a time),
// up to a grid whose threads stay below 2^32; beyond it, which takes states of
// at least 24 qubits more than their tiles have, workgroups walk several.
constexpr uint64_t kRegMaxBlocks = 1u << 23;

template <int R, int KD, int MINW>
void launch_reg(qtnh_ctx_t ctx, const RunDesc *d, int nr, uint64_t total, int tb) {
  const unsigned threads = std::max(64, 1 << (tb - R));
  const unsigned blocks = (unsigned)std::min(total, kRegMaxBlocks);
  const size_t lds = (reg_slot_bytes(MINW) << tb) + kRegCoef * sizeof(double2_t) + (kRegOps + 2) * sizeof(RegOp);
  hipLaunchKernelGGL((circuit_reg_kernel<R, KD, MINW>), dim3(blocks), dim3(threads), lds, ctx->stream, d, nr, total, tb);
}

// Launches groups of runs: group g covers descs [starts[g], starts[g+1]), one
// launch each, in order.  The descriptors go to the device in one copy.
// Launches the run groups [starts[g], starts[g+1]) of descriptors already on
// the device (dd); descs is their host copy.
qtnh_status launch_groups(qtnh_ctx_t ctx, const RunDesc *dd, const std::vector<RunDesc> &descs,
                          const std::vector<size_t> &starts) {
  qtnh_status st = QTNH_OK;
  for (size_t g = 0; g + 1 < starts.size(); ++g) {
    const size_t b = starts[g], e = starts[g + 1];
    if (b == e) continue;
    int tbmax = 0;
    uint64_t total = 0;
    for (size_t i = b; i < e; ++i) {
      tbmax = std::max(tbmax, descs[i].tb);
      total = descs[i].first + desc_tiles(descs[i]);
    }
    const int nr = (int)(e - b);
    bool all12 = true;
    for (size_t i = b; i < e; ++i) all12 = all12 && descs[i].tb == kPipeTB;
    if (descs[b].rbits && g_circuit_mode >= 2) {
      const bool g3 = descs[b].has3 != 0;
      if (descs[b].rbits == 2)
        launch_reg<2, 2, 4>(ctx, dd + b, nr, total, tbmax);
      else if (descs[b].rbits == 3)
        g3 ? launch_reg<3, 3, 4>(ctx, dd + b, nr, total, tbmax) : launch_reg<3, 2, 4>(ctx, dd + b, nr, total, tbmax);
      else if (total <= 2ull * ctx->num_cus)  // one or two tiles a compute unit
        g3 ? launch_reg<4, 3, 2>(ctx, dd + b, nr, total, tbmax) : launch_reg<4, 2, 2>(ctx, dd + b, nr, total, tbmax);
      else
        g3 ? launch_reg<4, 3, 3>(ctx, dd + b, nr, total, tbmax) : launch_reg<4, 2, 4>(ctx, dd + b, nr, total, tbmax);
      st = check_hip(ctx, hipGetLastError(), "circuit register launch");
      if (st) return st;
      continue;
    }
    if (all12 && total >= 4ull * ctx->num_cus && g_circuit_mode == 1) {
      const unsigned pb = (unsigned)std::min<uint64_t>(total, (uint64_t)ctx->num_cus);
      hipLaunchKernelGGL(circuit_pipe_kernel, dim3(pb), dim3(kPipeNT), 0, ctx->stream, dd + b, nr, total);
      st = check_hip(ctx, hipGetLastError(), "circuit pipe launch");
      if (st) return st;
      continue;
    }
    // Few tiles: 1024 threads per tile; many: 256 threads, several tiles per CU.
    const bool wide = total < (uint64_t)ctx->num_cus;
    const unsigned per_cu = wide ? 1 : tbmax <= 10 ? 8 : tbmax == 11 ? 4 : tbmax == 12 ? 2 : 1;
    const unsigned blocks = (unsigned)std::min<uint64_t>(total, (uint64_t)ctx->num_cus * per_cu);
#define QTNH_TILE_LAUNCH(TBM)                                                                                       \
  if (wide)                                                                                                       \
    hipLaunchKernelGGL((circuit_tile_kernel<TBM, 1024>), dim3(blocks), dim3(1024), 0, ctx->stream, dd + b, nr, total); \
  else                                                                                                            \
    hipLaunchKernelGGL((circuit_tile_kernel<TBM, 256>), dim3(blocks), dim3(256), 0, ctx->stream, dd + b, nr, total);
    if (tbmax <= 10) {
      QTNH_TILE_LAUNCH(10)
    } else if (tbmax == 11) {
      QTNH_TILE_LAUNCH(11)
    } else if (tbmax == 12) {
      QTNH_TILE_LAUNCH(12)
    } else {
      QTNH_TILE_LAUNCH(13)
    }
#undef QTNH_TILE_LAUNCH
    st = check_hip(ctx, hipGetLastError(), "circuit tile launch");
    if (st) return st;
  }
  return QTNH_OK;
}

// Uploads the descriptors into the context's descriptor buffer, then launches.
qtnh_status launch_run_groups(qtnh_ctx_t ctx, const std::vector<RunDesc> &descs, const std::vector<size_t> &starts) {
  if (descs.empty()) return QTNH_OK;
  const uint64_t bytes = descs.size() * sizeof(RunDesc);
  qtnh_status st = grow_buffer(ctx, &ctx->desc, &ctx->desc_bytes, bytes);
  if (st) return st;
  st = check_hip(ctx, hipMemcpyAsync(ctx->desc, descs.data(), bytes, hipMemcpyHostToDevice, ctx->stream),
                 "run descriptor upload");
  if (st) return st;
  return launch_groups(ctx, (const RunDesc *)ctx->desc, descs, starts);
}

constexpr size_t kDescCacheMax = 64;  // states per circuit with cached descriptors

qtnh_status run_fused(qtnh_ctx_t ctx, qtnh_circuit_s &c, c128 *psi) {
  Compiled *k = nullptr;
  qtnh_status st = compile(ctx, c, c.n, &k);
  if (st) return st;
  auto hit = k->desc_cache.find(psi);
  if (hit != k->desc_cache.end()) return launch_groups(ctx, hit->second.d, hit->second.h, hit->second.starts);
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(ctx->stream, &cap) != hipSuccess) {
    (void)hipGetLastError();
    cap = hipStreamCaptureStatusNone;
  }
  if (cap != hipStreamCaptureStatusNone)
    return set_error(ctx, QTNH_EUNSUPPORTED,
                     "circuit_run: first fused run of this circuit on this state during graph capture "
                     "(run it once on the state before capturing)");
  Compiled::DescCache dc;
  for (size_t ri = 0; ri < k->runs.size(); ++ri) add_group({RunRef{k, ri, psi}}, dc.h, dc.starts);
  dc.starts.push_back(dc.h.size());
  if (dc.h.empty()) return QTNH_OK;
  if (k->desc_cache.size() >= kDescCacheMax) return launch_run_groups(ctx, dc.h, dc.starts);
  const uint64_t bytes = dc.h.size() * sizeof(RunDesc);
  st = check_hip(ctx, hipMalloc((void **)&dc.d, bytes), "run descriptor alloc");
  if (st) return st;
  auto &e = k->desc_cache[psi];
  e = std::move(dc);
  st = check_hip(ctx, hipMemcpyAsync(e.d, e.h.data(), bytes, hipMemcpyHostToDevice, ctx->stream),
                 "run descriptor upload");
  if (st) {
    (void)hipFree(e.d);
    k->desc_cache.erase(psi);
    return st;
  }
  return launch_groups(ctx, e.d, e.h, e.starts);
}

qtnh_status run_per_gate(qtnh_ctx_t ctx, const qtnh_circuit_s &c, c128 *psi) {
  std::vector<uint64_t> dims(c.n, 2);
  for (const auto &op : c.ops) {
    qtnh_status st = op.kind == 0 ? launch_gate(ctx, psi, c.n, dims.data(), op.k, op.q, op.coef.data())
                                  : launch_diag(ctx, psi, c.n, dims.data(), op.k, op.q, op.coef.data());
    if (st) return st;
  }
  return QTNH_OK;
}

// ---- seeded generators ----------------------------------------------------
uint64_t mix64(uint64_t seed, uint64_t k) {
  uint64_t z = seed + (k + 1) * 0x9E3779B97F4A7C15ull;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}

struct HostRng {
  uint64_t seed, k = 0;
  explicit HostRng(uint64_t s) : seed(s) {}
  uint64_t next() { return mix64(seed, k++); }
  double uniform() { return (double)(next() >> 11) * 0x1.0p-53; }  // [0, 1)
  void normal2(double *a, double *b) {
    const double u1 = (double)((next() >> 11) + 1) * 0x1.0p-53, u2 = uniform();
    const double r = std::sqrt(-2.0 * std::log(u1));
    *a = r * std::cos(2.0 * M_PI * u2);
    *b = r * std::sin(2.0 * M_PI * u2);
  }
};

// Haar-random SU(2) (Mezzadri 2007): QR of a complex Gaussian 2x2 with the
// phases of R's diagonal moved into Q, then divided by sqrt(det).
// Returns G[in][out] = U[out][in].
void random_su2(HostRng &rng, double *G) {
  double z[4][2];
  for (int i = 0; i < 4; ++i) rng.normal2(&z[i][0], &z[i][1]);
  // columns a = (z00, z10), b = (z01, z11) of Z
  const double ar[2] = {z[0][0], z[2][0]}, ai[2] = {z[0][1], z[2][1]};
  const double br[2] = {z[1][0], z[3][0]}, bi[2] = {z[1][1], z[3][1]};
  const double na = std::sqrt(ar[0] * ar[0] + ai[0] * ai[0] + ar[1] * ar[1] + ai[1] * ai[1]);
  double q0r[2], q0i[2];
  for (int i = 0; i < 2; ++i) {
    q0r[i] = ar[i] / na;
    q0i[i] = ai[i] / na;
  }
  // r01 = <q0, b>; b' = b - q0 r01
  double r01r = 0, r01i = 0;
  for (int i = 0; i < 2; ++i) {
    r01r += q0r[i] * br[i] + q0i[i] * bi[i];
    r01i += q0r[i] * bi[i] - q0i[i] * br[i];
  }
  double cr[2], ci[2];
  for (int i = 0; i < 2; ++i) {
    cr[i] = br[i] - (q0r[i] * r01r - q0i[i] * r01i);
    ci[i] = bi[i] - (q0r[i] * r01i + q0i[i] * r01r);
  }
  const double nc = std::sqrt(cr[0] * cr[0] + ci[0] * ci[0] + cr[1] * cr[1] + ci[1] * ci[1]);
  double q1r[2], q1i[2];
  for (int i = 0; i < 2; ++i) {
    q1r[i] = cr[i] / nc;
    q1i[i] = ci[i] / nc;
  }
  // R's diagonal (na, nc) is real positive, so Q is already phase-fixed.
  // U = Q / sqrt(det Q)
  const double dr = (q0r[0] * q1r[1] - q0i[0] * q1i[1]) - (q1r[0] * q0r[1] - q1i[0] * q0i[1]);
  const double di = (q0r[0] * q1i[1] + q0i[0] * q1r[1]) - (q1r[0] * q0i[1] + q1i[0] * q0r[1]);
  const double ph = std::atan2(di, dr) / 2.0;
  const double sr = std::cos(-ph), si = std::sin(-ph);
  double U[2][2][2];  // U[row][col][re/im]
  for (int i = 0; i < 2; ++i) {
    U[i][0][0] = q0r[i] * sr - q0i[i] * si;
    U[i][0][1] = q0r[i] * si + q0i[i] * sr;
    U[i][1][0] = q1r[i] * sr - q1i[i] * si;
    U[i][1][1] = q1r[i] * si + q1i[i] * sr;
  }
  for (int in = 0; in < 2; ++in)
    for (int out = 0; out < 2; ++out) {
      G[2 * (in * 2 + out)] = U[out][in][0];
      G[2 * (in * 2 + out) + 1] = U[out][in][1];
    }
}

bool qubits_valid(int n, int k, const uint16_t *q) {
  if (k < 1 || k > kMaxOpQubits) return false;
  for (int j = 0; j < k; ++j) {
    if (q[j] >= n) return false;
    for (int i = 0; i < j; ++i)
      if (q[i] == q[j]) return false;
  }
  return true;
}

}  // namespace
}  // namespace qtnh_hip

namespace qtnh_hip {

int circuit_run_count(qtnh_ctx_t ctx, qtnh_circuit_t c, int bits) {
  int tb, low;
  tile_shape(ctx, *c, bits, &tb, &low);
  return (int)plan_runs(*c, tb, low).size();
}

qtnh_status circuit_advance(qtnh_ctx_t ctx, int count, const qtnh_circuit_t *cs, void *const *states,
                            const int *first_run, const int *nrun, int bits) {
  int kmax = 0;
  std::vector<Compiled *> ks(count);
  for (int i = 0; i < count; ++i) {
    qtnh_status st = compile(ctx, *cs[i], bits, &ks[i]);
    if (st) return st;
    if (first_run[i] < 0 || nrun[i] < 0 || (size_t)first_run[i] + (size_t)nrun[i] > ks[i]->runs.size())
      return set_error(ctx, QTNH_EINVAL, "circuit advance: runs out of range");
    kmax = std::max(kmax, nrun[i]);
  }
  std::vector<RunDesc> descs;
  std::vector<size_t> starts;
  for (int k = 0; k < kmax; ++k) {
    std::vector<RunRef> refs;
    for (int i = 0; i < count; ++i)
      if (k < nrun[i]) refs.push_back(RunRef{ks[i], (size_t)(first_run[i] + k), (c128 *)states[i]});
    add_group(refs, descs, starts);
  }
  starts.push_back(descs.size());
  return launch_run_groups(ctx, descs, starts);
}

}  // namespace qtnh_hip

using namespace qtnh_hip;

extern "C" {

void qtnh_tune_circuit(int tile_bits, int low_bits) {
  g_tile_bits = tile_bits <= 0 ? 0 : std::max(3, std::min(tile_bits, kMaxTileBits));
  g_low_bits = std::max(0, std::min(low_bits, 8));
}

void qtnh_tune_circuit_pipeline(int mode) { g_circuit_mode = std::max(0, std::min(mode, 3)); }

qtnh_status qtnh_circuit_create(int n_qubits, qtnh_circuit_t *out) {
  if (!out) return QTNH_EINVAL;
  *out = nullptr;
  if (n_qubits < 1 || n_qubits > 62) return QTNH_EINVAL;
  auto *c = new (std::nothrow) qtnh_circuit_s;
  if (!c) return QTNH_ENOMEM;
  c->n = n_qubits;
  *out = c;
  return QTNH_OK;
}

qtnh_status qtnh_circuit_destroy(qtnh_circuit_t c) {
  if (!c) return QTNH_EINVAL;
  for (const auto &k : c->compiled) {
    (void)hipSetDevice(k->device);
    (void)hipDeviceSynchronize();
  }
  free_compiled(*c);
  delete c;
  return QTNH_OK;
}

qtnh_status qtnh_circuit_gate(qtnh_circuit_t c, int k, const uint16_t *qubits, const double *G) {
  if (!c || !qubits || !G || !qubits_valid(c->n, k, qubits)) return QTNH_EINVAL;
  qtnh_circuit_s::Op op;
  op.kind = 0;
  op.k = k;
  for (int j = 0; j < k; ++j) op.q[j] = qubits[j];
  op.coef.assign(G, G + 2 * (1 << k) * (1 << k));
  c->ops.push_back(std::move(op));
  return QTNH_OK;
}

qtnh_status qtnh_circuit_diag(qtnh_circuit_t c, int k, const uint16_t *qubits, const double *d) {
  if (!c || !qubits || !d || !qubits_valid(c->n, k, qubits)) return QTNH_EINVAL;
  qtnh_circuit_s::Op op;
  op.kind = 1;
  op.k = k;
  for (int j = 0; j < k; ++j) op.q[j] = qubits[j];
  op.coef.assign(d, d + 2 * (1 << k));
  c->ops.push_back(std::move(op));
  return QTNH_OK;
}

qtnh_status qtnh_circuit_qft(qtnh_circuit_t c, const double *phases) {
  if (!c) return QTNH_EINVAL;
  const int n = c->n;
  const double h = 0x1.6a09e667f3bcdp-1;
  const double H[8] = {h, 0, h, 0, h, 0, -h, 0};
  for (int i = 0; i < n; ++i) {
    const uint16_t qi = (uint16_t)i;
    qtnh_status st = qtnh_circuit_gate(c, 1, &qi, H);
    if (st) return st;
    for (int j = i + 1; j < n; ++j) {
      const int m = j - i;
      double pr, pi;
      if (phases) {
        pr = phases[2 * m];
        pi = phases[2 * m + 1];
      } else {
        pr = std::cos(M_PI / std::ldexp(1.0, m));
        pi = std::sin(M_PI / std::ldexp(1.0, m));
      }
      const double d[8] = {1, 0, 1, 0, 1, 0, pr, pi};
      const uint16_t q2[2] = {(uint16_t)i, (uint16_t)j};
      st = qtnh_circuit_diag(c, 2, q2, d);
      if (st) return st;
    }
  }
  return QTNH_OK;
}

qtnh_status qtnh_circuit_random(qtnh_circuit_t c, int depth, uint64_t seed) {
  if (!c || depth < 0) return QTNH_EINVAL;
  const int n = c->n;
  HostRng rng(seed);
  std::vector<uint16_t> perm(n);
  for (int layer = 0; layer < depth; ++layer) {
    for (int q = 0; q < n; ++q) {
      double G[8];
      random_su2(rng, G);
      const uint16_t qq = (uint16_t)q;
      qtnh_status st = qtnh_circuit_gate(c, 1, &qq, G);
      if (st) return st;
    }
    for (int q = 0; q < n; ++q) perm[q] = (uint16_t)q;
    for (int q = n - 1; q > 0; --q) std::swap(perm[q], perm[rng.next() % (uint64_t)(q + 1)]);
    const double cz[8] = {1, 0, 1, 0, 1, 0, -1, 0};
    for (int p = 0; p + 1 < n; p += 2) {
      const uint16_t q2[2] = {perm[p], perm[p + 1]};
      qtnh_status st = qtnh_circuit_diag(c, 2, q2, cz);
      if (st) return st;
    }
  }
  return QTNH_OK;
}

qtnh_status qtnh_circuit_grid(qtnh_circuit_t c, int rows, int cols, int depth, uint64_t seed) {
  if (!c || rows < 1 || cols < 1 || depth < 0 || rows * cols != c->n) return QTNH_EINVAL;
  HostRng rng(seed);
  const double cz[8] = {1, 0, 1, 0, 1, 0, -1, 0};
  for (int layer = 0; layer < depth; ++layer) {
    for (int q = 0; q < c->n; ++q) {
      double G[8];
      random_su2(rng, G);
      const uint16_t qq = (uint16_t)q;
      qtnh_status st = qtnh_circuit_gate(c, 1, &qq, G);
      if (st) return st;
    }
    // Couplers cycle through four patterns: horizontal even / odd columns,
    // vertical even / odd rows.
    const int pat = layer % 4;
    for (int r = 0; r < rows; ++r)
      for (int col = 0; col < cols; ++col) {
        int r2 = r, c2 = col;
        if (pat < 2) {
          if ((col & 1) != pat) continue;
          c2 = col + 1;
        } else {
          if ((r & 1) != pat - 2) continue;
          r2 = r + 1;
        }
        if (r2 >= rows || c2 >= cols) continue;
        const uint16_t q2[2] = {(uint16_t)(r * cols + col), (uint16_t)(r2 * cols + c2)};
        qtnh_status st = qtnh_circuit_diag(c, 2, q2, cz);
        if (st) return st;
      }
  }
  return QTNH_OK;
}

qtnh_status qtnh_circuit_info(qtnh_circuit_t c, int *n_qubits, uint64_t *n_ops, uint64_t *n_runs) {
  if (!c) return QTNH_EINVAL;
  if (n_qubits) *n_qubits = c->n;
  if (n_ops) *n_ops = c->ops.size();
  if (n_runs) {
    int tb = c->tuned_tb, low = c->tuned_low;
    if (tb <= 0) default_tile(c->n, c->n, &tb, &low);
    *n_runs = plan_runs(*c, tb, low).size();
  }
  return QTNH_OK;
}

qtnh_status qtnh_circuit_op(qtnh_circuit_t c, uint64_t i, int *kind, int *k, uint16_t *qubits, double *coef) {
  if (!c || i >= c->ops.size()) return QTNH_EINVAL;
  const auto &op = c->ops[i];
  if (kind) *kind = op.kind;
  if (k) *k = op.k;
  if (qubits)
    for (int j = 0; j < op.k; ++j) qubits[j] = op.q[j];
  if (coef) memcpy(coef, op.coef.data(), op.coef.size() * sizeof(double));
  return QTNH_OK;
}

qtnh_status qtnh_circuit_run(qtnh_ctx_t ctx, qtnh_circuit_t c, void *state, int mode) {
  qtnh_status st = enter_ctx(ctx);
  if (st) return st;
  if (!c || !state) return set_error(ctx, QTNH_EINVAL, "circuit_run: null argument");
  if (mode == QTNH_RUN_PER_GATE) return run_per_gate(ctx, *c, (c128 *)state);
  if (mode == QTNH_RUN_FUSED) return run_fused(ctx, *c, (c128 *)state);
  return set_error(ctx, QTNH_EINVAL, "circuit_run: unknown mode %d", mode);
}

qtnh_status qtnh_circuit_run_batch(qtnh_ctx_t ctx, int count, const qtnh_circuit_t *cs, void *const *states) {
  qtnh_status st = enter_ctx(ctx);
  if (st) return st;
  if (count < 0 || (count > 0 && (!cs || !states))) return set_error(ctx, QTNH_EINVAL, "run_batch: bad arguments");
  size_t steps = 0;
  uint64_t amplitudes = 0;
  for (int i = 0; i < count; ++i) {
    if (!cs[i] || !states[i]) return set_error(ctx, QTNH_EINVAL, "run_batch: null circuit or state %d", i);
    for (int j = 0; j < i; ++j)
      if (states[j] == states[i]) return set_error(ctx, QTNH_EINVAL, "run_batch: state %d repeats state %d", i, j);
    amplitudes += 1ull << cs[i]->n;
  }
  std::vector<Compiled *> ks(count);
  for (int i = 0; i < count; ++i) {
    st = compile(ctx, *cs[i], floor_log2(amplitudes), &ks[i]);
    if (st) return st;
    steps = std::max(steps, ks[i]->runs.size());
  }
  // Step s runs the s-th run of every circuit that has one, in one launch.
  std::vector<RunDesc> descs;
  std::vector<size_t> starts;
  for (size_t s = 0; s < steps; ++s) {
    std::vector<RunRef> refs;
    for (int i = 0; i < count; ++i)
      if (s < ks[i]->runs.size()) refs.push_back(RunRef{ks[i], s, (c128 *)states[i]});
    add_group(refs, descs, starts);
  }
  starts.push_back(descs.size());
  return launch_run_groups(ctx, descs, starts);
}


qtnh_status qtnh_circuit_tune(qtnh_ctx_t ctx, qtnh_circuit_t c, void *scratch, int *tile_bits, int *low_bits,
                              double *us_out) {
  qtnh_status st = enter_ctx(ctx);
  if (st) return st;
  if (!c || !scratch) return set_error(ctx, QTNH_EINVAL, "circuit_tune: null argument");
  if (c->ops.empty()) return QTNH_OK;
  // Candidates: the tile the circuit takes without tuning, then from the largest
  // to smaller ones (more workgroups per run; they win for small states whose runs
  // would otherwise occupy a few CUs).
  int cand[][2] = {{0, 0}, {12, 4}, {11, 4}, {10, 2}, {9, 2}, {8, 2}, {7, 2}};
  tile_shape(ctx, c->n, c->n, &cand[0][0], &cand[0][1]);
  const int reps = c->n >= 20 ? 2 : 10;
  hipEvent_t e0 = nullptr, e1 = nullptr;
  st = check_hip(ctx, hipEventCreate(&e0), "circuit_tune event");
  if (!st) st = check_hip(ctx, hipEventCreate(&e1), "circuit_tune event");
  double best = 1e30;
  int btb = 0, blow = 0;
  for (const auto &cd : cand) {
    if (st) break;
    if (&cd != cand && (cd[0] > std::max(c->n, 7) || (cd[0] == cand[0][0] && cd[1] == cand[0][1]))) continue;
    c->tuned_tb = cd[0];
    c->tuned_low = cd[1];
    st = run_fused(ctx, *c, (c128 *)scratch);  // compile + warm up
    float ms = 0;
    if (!st) st = check_hip(ctx, hipEventRecord(e0, ctx->stream), "circuit_tune record");
    for (int r = 0; r < reps && !st; ++r) st = run_fused(ctx, *c, (c128 *)scratch);
    if (!st) st = check_hip(ctx, hipEventRecord(e1, ctx->stream), "circuit_tune record");
    if (!st) st = check_hip(ctx, hipEventSynchronize(e1), "circuit_tune sync");
    if (!st) st = check_hip(ctx, hipEventElapsedTime(&ms, e0, e1), "circuit_tune elapsed");
    if (!st && ms / reps < best) {
      best = ms / reps;
      btb = cd[0];
      blow = cd[1];
    }
  }
  if (e0) (void)hipEventDestroy(e0);
  if (e1) (void)hipEventDestroy(e1);
  c->tuned_tb = st ? 0 : btb;
  c->tuned_low = st ? 0 : blow;
  if (st) return st;
  // Leave the winning shape compiled, so the next run launches without a recompile.
  Compiled *k = nullptr;
  st = compile(ctx, *c, c->n, &k);
  if (st) return st;
  if (tile_bits) *tile_bits = btb;
  if (low_bits) *low_bits = blow;
  if (us_out) *us_out = best * 1e3;
  return QTNH_OK;
}

qtnh_status qtnh_autotune_circuit(qtnh_ctx_t ctx, int n_qubits, int *tile_bits, int *low_bits, double *ms_out) {
  qtnh_status st = enter_ctx(ctx);
  if (st) return st;
  if (n_qubits < 1 || n_qubits > 62) return set_error(ctx, QTNH_EINVAL, "autotune: bad qubit count");
  // Proxy: a depth-6 random circuit on min(n, 26) qubits (the best tile does
  // not depend on the state size once it spans many tiles); best of two runs.
  const int np = std::min(n_qubits, 26);
  const uint64_t N = 1ull << np;
  void *w = nullptr;
  st = workspace(ctx, N * sizeof(c128), &w);
  if (st) return st;
  st = launch_fill(ctx, (c128 *)w, N, 1, QTNH_DIST_NORMAL);
  if (st) return st;
  const int cand[][2] = {{10, 3}, {11, 3}, {11, 4}, {12, 4}, {12, 5}, {13, 4}, {13, 5}};
  hipEvent_t e0 = nullptr, e1 = nullptr;
  st = check_hip(ctx, hipEventCreate(&e0), "autotune event");
  if (!st) st = check_hip(ctx, hipEventCreate(&e1), "autotune event");
  double best = 1e30;
  int btb, blow;
  default_tile(np, np, &btb, &blow);
  for (const auto &cd : cand) {
    if (st) break;
    if (cd[0] > std::max(np, 10)) continue;
    qtnh_circuit_s c;
    c.n = np;
    (void)qtnh_circuit_random(&c, 6, 12345);
    ctx->circ_tb[np] = (int8_t)cd[0];
    ctx->circ_low[np] = (int8_t)cd[1];
    st = run_fused(ctx, c, (c128 *)w);  // compile + warm up
    float ms = 1e30f;
    for (int rep = 0; rep < 2 && !st; ++rep) {
      float one = 0;
      st = check_hip(ctx, hipEventRecord(e0, ctx->stream), "autotune record");
      if (!st) st = run_fused(ctx, c, (c128 *)w);
      if (!st) st = check_hip(ctx, hipEventRecord(e1, ctx->stream), "autotune record");
      if (!st) st = check_hip(ctx, hipEventSynchronize(e1), "autotune sync");
      if (!st) st = check_hip(ctx, hipEventElapsedTime(&one, e0, e1), "autotune elapsed");
      ms = std::min(ms, one);
    }
    if (!st && ms < best) {
      best = ms;
      btb = cd[0];
      blow = cd[1];
    }
    free_compiled(c);
  }
  if (e0) (void)hipEventDestroy(e0);
  if (e1) (void)hipEventDestroy(e1);
  if (st) {
    ctx->circ_tb[np] = 0;
    return st;
  }
  ctx->circ_tb[n_qubits] = (int8_t)btb;
  ctx->circ_low[n_qubits] = (int8_t)blow;
  if (np != n_qubits) {
    ctx->circ_tb[np] = (int8_t)btb;
    ctx->circ_low[np] = (int8_t)blow;
  }
  if (tile_bits) *tile_bits = btb;
  if (low_bits) *low_bits = blow;
  if (ms_out) *ms_out = best;
  return QTNH_OK;
}

qtnh_status qtnh_expect_z_c128(qtnh_ctx_t ctx, const void *state, int n_qubits, int nq, const uint16_t *qubits,
                               double *out) {
  qtnh_status st = enter_ctx(ctx);
  if (st) return st;
  if (!state || !out || n_qubits < 1 || n_qubits > 62 || nq < 1 || nq > kHostScalars || !qubits)
    return set_error(ctx, QTNH_EINVAL, "expect_z: bad arguments");
  for (int j = 0; j < nq; ++j)
    if (qubits[j] >= n_qubits) return set_error(ctx, QTNH_EINVAL, "expect_z: qubit %d out of range", qubits[j]);
  const uint64_t n = 1ull << n_qubits;
  const int cb = std::min(n_qubits, kChunkBits);
  const uint64_t nchunks = n >> cb;
  st = grow_buffer(ctx, &ctx->red, &ctx->red_bytes, nchunks * kZSlots * sizeof(double));
  if (st) return st;
  double *part = (double *)ctx->red;
  ZQubits bits;
  for (int j = 0; j < nq; ++j) bits.bit[j] = (uint8_t)(n_qubits - 1 - qubits[j]);
  const unsigned blocks = (unsigned)nchunks;
  const auto *psi = (const double2_t *)state;
  if (n_qubits > 24)
    hipLaunchKernelGGL((zchunk_kernel<true, true>), dim3(blocks), dim3(kZThreads), 0, ctx->stream, psi, cb, part,
                       nchunks);
  else if (cb == kChunkBits)
    hipLaunchKernelGGL((zchunk_kernel<true, false>), dim3(blocks), dim3(kZThreads), 0, ctx->stream, psi, cb, part,
                       nchunks);
  else
    hipLaunchKernelGGL((zchunk_kernel<false, false>), dim3(blocks), dim3(kZThreads), 0, ctx->stream, psi, cb, part,
                       nchunks);
  st = check_hip(ctx, hipGetLastError(), "expect_z launch");
  if (st) return st;
  // The results go to pinned host memory from the kernel.
  hipLaunchKernelGGL(zfinal_kernel, dim3(nq), dim3(kZThreads), 0, ctx->stream, part, nchunks, cb, bits,
                     ctx->host_scalar);
  st = check_hip(ctx, hipGetLastError(), "expect_z final launch");
  if (st) return st;
  st = check_hip(ctx, hipStreamSynchronize(ctx->stream), "expect_z sync");
  if (st) return st;
  memcpy(out, ctx->host_scalar, nq * sizeof(double));
  return QTNH_OK;
}

}  // extern "C"
