// Batched matmul C[b] = A[b] . B[b] (+ C_old[b]) on strided views.
//
// fp32 runs on the gfx950 matrix cores (v_mfma_f32_32x32x2_f32; large single
// products on v_mfma_f32_32x32x16_bf16 with each operand split into three
// exact parts, see mm_split_kernel).  The
// reference (src/cpp/ops/matmul.cu) has a SIMT 128x128x16 kernel that only
// accepts contiguous operands and sends every transposed operand -- hence
// both backward products of MatmulOp (ops_binary.py:264-267) -- to a naive
// one-thread-per-output kernel.  Here each operand is read in place in
// whichever orientation it has:
//
//   layout K  : the reduction index k is the unit-stride one (A row-major,
//               or B = W^T of a row-major W).  Stored in LDS as [mn][k].
//   layout MN : the m (or n) index is unit-stride (A = X^T of a row-major
//               X, or B row-major).  Stored in LDS as [k][mn].
//   anything else (odd row lengths, `[:, ::2]` views): 4-byte loads along
//               the axis with the smaller stride, stored either way.
//
// Workgroup tiles of 128x128, 64x64, 32x128 and 128x32 with a 32-deep k-tile
// (mm_f32_tile_kernel, 256 threads = 4 waves), and of 256x256 for large
// products whose sizes fit (mm_f32_mfma_wide_kernel, 8 waves).  Operands go
// from global memory straight into LDS (gfx950's direct loads, 16 bytes per
// lane where the layout allows and 4 bytes otherwise); LDS is double
// buffered and the loads of k-tile t+1 are in flight under the MFMAs of tile
// t, with one barrier per k-tile.  The tile shape and a split of K follow
// the product's size (choose_tile).  Workgroups are numbered so that
// consecutive tiles of a group of 8 tile-rows land on the same XCD (gfx950
// dispatches workgroups round-robin over its 8 XCDs, each with its own L2).
//
// MFMA k assignment: in MFMA step kk (0..15) of a k-tile, the lanes of wave
// half h (lane / 32) supply k = h*16 + kk, for A and B alike, so each lane's
// 16 fragments of a k-tile are contiguous in a [mn][k] LDS row.  The sum over
// k is unchanged; only the fp32 accumulation order differs from the
// reference's sequential loop (|diff| <= 1e-4 * (|A|.|B|) is the parity
// bound).  Accumulate mode adds C_old after the full dot product: one
// rounding, like the reference's `x._grad += grad`.
//
// Other dtypes (fp64, int32, int64) use tiled SIMT kernels that accumulate
// in k order exactly like the reference's CPU loop (matmul.cu:33-45).
#include <algorithm>
#include <limits>

#include "ew_engine.h"

namespace nt {

typedef float floatx16 __attribute__((ext_vector_type(16)));

constexpr int MM_BK = 32, MM_THREADS = 256;
constexpr int MM_MAX_BATCH = NT_MAX_DIMS - 2;

// Unit-stride axis of an operand of the wide kernel.
enum { LAY_K = 0, LAY_MN = 1 };

struct MMArgs {
  const float *A;
  const float *B;
  float *C;
  int64_t M, N, K;
  int64_t sAm, sAk, sBk, sBn, sCm, sCn;
  int nb;
  int64_t bshape[MM_MAX_BATCH];
  int64_t bsA[MM_MAX_BATCH], bsB[MM_MAX_BATCH], bsC[MM_MAX_BATCH];
  int64_t tiles_m, tiles_n;
  uint32_t nbatch;
  int accumulate;
  // Split over K: slice s takes k in [s kslice, (s + 1) kslice) and writes
  // its raw sum to part + s nbatch M N (every batch [M][N] contiguous);
  // mm_splitk_sum_kernel adds the slices.  part == nullptr: no split (one
  // slice, kslice >= K), results go to C.
  int64_t kslice;
  float *part;
  // Optional bias added to every output row in the epilogue, C = fl(acc) +
  // bias[n] (one fp32 rounding after the product's own, as a separate add
  // would give); nullptr: none.  Never combined with accumulate.
  const float *bias;
  int64_t sBias;
  // Flag words of a split product (mm_split_pack_kernel): the kernel runs
  // only if they say `run_if`.  nullptr: it runs.
  const uint32_t *flags;
  bool run_if;
};

// Workgroup -> (slice of K, batch, tile).
struct TileCoord {
  int64_t m0, n0;
  uint32_t slice, batch;
  const float *A, *B;
  float *C;
};

// The 1-D grid holds slices x batches x tiles.  Workgroup ids are dealt to
// the 8 XCDs round-robin; renumbered so that each XCD gets one contiguous run
// (of any grid size), tiles of a run walk groups of 8 tile-rows column by
// column.  The grid is below 2^31 workgroups: 32-bit divisions.
template <int BM, int BN>
__device__ __forceinline__ TileCoord mm_tile_coord(const MMArgs &g) {
  const uint32_t tm = uint32_t(g.tiles_m), tn = uint32_t(g.tiles_n);
  const uint32_t per_batch = tm * tn;
  const uint32_t nblk = gridDim.x, q8 = nblk / 8, r8 = nblk % 8;
  const uint32_t xcd = blockIdx.x % 8;
  const uint32_t bid = xcd * q8 + (xcd < r8 ? xcd : r8) + blockIdx.x / 8;
  TileCoord tc;
  const uint32_t all = bid / per_batch; // slice * batches + batch
  const uint32_t tile = bid - all * per_batch;
  tc.slice = all / g.nbatch;
  tc.batch = all - tc.slice * g.nbatch;
  constexpr uint32_t GROUP = 8;
  const uint32_t group = tile / (GROUP * tn);
  const uint32_t first_m = group * GROUP;
  const uint32_t gsize = tm - first_m < GROUP ? tm - first_m : GROUP;
  const uint32_t in_group = tile - group * GROUP * tn;
  const uint32_t col = in_group / gsize;
  tc.m0 = int64_t(first_m + in_group - col * gsize) * BM;
  tc.n0 = int64_t(col) * BN;
  tc.A = g.A;
  tc.B = g.B;
  tc.C = g.C;
  uint32_t rem = tc.batch;
  for (int d = g.nb - 1; d >= 0; --d) {
    const uint32_t sz = uint32_t(g.bshape[d]);
    const uint32_t q = rem / sz;
    const int64_t c = rem - q * sz;
    rem = q;
    tc.A += c * g.bsA[d];
    tc.B += c * g.bsB[d];
    tc.C += c * g.bsC[d];
  }
  return tc;
}

// One finished value of the product: to its slice's partial array, or to C
// (accumulated, or with the bias).
__device__ __forceinline__ void mm_put(const MMArgs &g, const TileCoord &tc,
                                       int64_t row, int64_t col, float v) {
  if (g.part) {
    const int64_t p = int64_t(tc.slice) * g.nbatch + tc.batch;
    g.part[(p * g.M + row) * g.N + col] = v;
  } else {
    float *dst = tc.C + row * g.sCm + col * g.sCn;
    *dst = g.accumulate ? (*dst + v) : (g.bias ? v + g.bias[col * g.sBias] : v);
  }
}

// ------------------------------------------ direct-to-LDS staging (gfx950)

// gfx950 moves 16 or 4 bytes per lane from global memory straight into LDS
// (global_load_lds): lane L of a wave lands at LDS base + 16 L (or 4 L), with
// the base wave-uniform.  No VGPR round trip, no LDS store instructions.
// An operand's stage is a [mn][32 k] or [32 k][mn] tile, where mn is m for A
// and n for B:
//   ST_K16 : k is unit-stride, 16-byte loads; rows of 32 k, no padding,
//            16-byte chunks swizzled within a row (dl_swz) so that fragment
//            reads are bank-conflict free.  One instruction covers 8 rows.
//   ST_MN16: mn is unit-stride, 16-byte loads; k rows of mn.
//   ST_K4  : any strides, 4-byte loads with consecutive lanes along k (for
//            odd row lengths, unaligned views); two rows of 32 k and 4 pad
//            floats per instruction, which keeps the 16-byte fragment reads
//            of 16 rows on distinct banks.
//   ST_MN4 : any strides, 4-byte loads with consecutive lanes along mn.
// Rows (columns) past M (N) re-read the last valid one: their results are
// never stored.
enum { ST_K16 = 0, ST_MN16 = 1, ST_K4 = 2, ST_MN4 = 3 };

// Chunk swizzle of a [mn][k] stage row.  A fragment read is a 16-byte read
// per lane of one chunk from 16 consecutive rows (lanes li of a half-wave);
// gfx950's LDS serves 16 lanes x 16 bytes over its 64 banks at once, so the
// 16 (row parity, chunk) pairs must differ: chunk c of row r is stored at
// c ^ (r % 8) ^ ((r / 8) % 2).  (With c ^ (r % 8) alone, rows r and r + 8
// collide: rocprof counted one LDS bank conflict per read.)
__device__ __forceinline__ int dl_swz(int r) { return (r & 7) ^ ((r >> 3) & 1); }

// FAR: strides past the 32-bit offsets (64 rows of 2^22 elements and more):
// a 64-bit offset per load.
template <int ST, int B, bool FAR = false> struct StageTile {
  static constexpr int FLOATS = ST == ST_K4 ? B / 2 * 68 : B * MM_BK;
  static constexpr bool WIDE = ST == ST_K16 || ST == ST_MN16;
  static constexpr int NI = WIDE ? B / 32 : B / 8; // instructions per wave
  static constexpr int LDS_STEP = WIDE ? 256 : (ST == ST_K4 ? 68 : 64);
  // Where element (mn, k) of the tile lies in the stage.
  __device__ __forceinline__ static int pos(int mn, int k) {
    if constexpr (ST == ST_K16)
      return mn * 32 + (((k >> 2) ^ dl_swz(mn)) << 2) + (k & 3);
    else if constexpr (ST == ST_K4)
      return (mn >> 1) * 68 + (mn & 1) * 32 + k;
    else
      return k * B + mn;
  }
  using Off = std::conditional_t<FAR, int64_t, uint32_t>;
  const char *base;  // element (mn0, k0) of the operand
  Off off[NI];       // byte offset of this lane's source, instruction j
  int64_t kstep;     // bytes between two k-tiles
  __device__ __forceinline__ void init(const float *p, int64_t mn0, int64_t MN,
                                       int64_t s_mn, int64_t s_k, int wave,
                                       int lane) {
    base = reinterpret_cast<const char *>(p + mn0 * s_mn);
    kstep = 4 * MM_BK * s_k;
    // the last row (16-byte group of rows) that may be read
    const int64_t last = MN - mn0 - (ST == ST_MN16 ? 4 : 1);
    const int lastc = int(last < B - 1 ? last : B - 1);
    const Off bm = Off(4 * s_mn), bk = Off(4 * s_k);
#pragma unroll
    for (int j = 0; j < NI; ++j) {
      const int q = wave * NI + j;
      int mn, k;
      if constexpr (ST == ST_K16) {
        mn = q * 8 + lane / 8;
        k = 4 * ((lane % 8) ^ dl_swz(mn));
      } else if constexpr (ST == ST_MN16) {
        const int flat = q * 256 + lane * 4;
        k = flat / B;
        mn = flat % B;
      } else if constexpr (ST == ST_K4) {
        mn = q * 2 + lane / 32;
        k = lane % 32;
      } else {
        const int flat = q * 64 + lane;
        k = flat / B;
        mn = flat % B;
      }
      mn = mn < lastc ? mn : lastc;
      off[j] = Off(mn) * bm + Off(k) * bk;
    }
  }
  __device__ __forceinline__ void issue(float *stage, int64_t kt,
                                        int wave) const {
    if constexpr (FAR) {
#pragma unroll
      for (int j = 0; j < NI; ++j) {
        auto *from =
            (const __attribute__((address_space(1))) void *)(base + kt * kstep + off[j]);
        auto *to = (__attribute__((address_space(3))) void *)(stage +
                                                              (wave * NI + j) * LDS_STEP);
        if constexpr (WIDE)
          __builtin_amdgcn_global_load_lds(from, to, 16, 0, 0);
        else
          __builtin_amdgcn_global_load_lds(from, to, 4, 0, 0);
      }
      return;
    }
    // Buffer loads: a scalar base and each lane's 32-bit offset.  (With
    // global pointers the compiler kept a 64-bit address per load in
    // registers and advanced them all each k-tile, and spilled in the
    // 128x128 tiles.)  Every offset is in bounds by init's clamp; the range
    // check of the resource is left wide open.
    const char *src = base + kt * kstep;
    const uint64_t ub = reinterpret_cast<uint64_t>(src);
    const uint32_t lo = __builtin_amdgcn_readfirstlane(uint32_t(ub));
    const uint32_t hi = __builtin_amdgcn_readfirstlane(uint32_t(ub >> 32));
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
        reinterpret_cast<void *>((uint64_t(hi) << 32) | lo), 0, -1, BUF_WORD3);
#pragma unroll
    for (int j = 0; j < NI; ++j) {
      auto *to = (__attribute__((address_space(3))) void *)(stage +
                                                            (wave * NI + j) * LDS_STEP);
      if constexpr (WIDE)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, to, 16, int(off[j]), 0, 0, 0);
      else
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, to, 4, int(off[j]), 0, 0, 0);
    }
  }
  // The partial k-tile of K % 32 leading elements k0 .. K - 1, the rest
  // zero: through registers.  p: the operand.
  __device__ __forceinline__ static void stage_tail(float *stage, const float *p,
                                                    int64_t mn0, int64_t MN,
                                                    int64_t s_mn, int64_t s_k,
                                                    int64_t k0, int64_t K, int t) {
    constexpr int E = B * MM_BK / MM_THREADS;
    float v[E];
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const int flat = t + MM_THREADS * e;
      constexpr bool KF = ST == ST_K16 || ST == ST_K4;
      const int mn = KF ? flat / MM_BK : flat % B;
      const int k = KF ? flat % MM_BK : flat / B;
      v[e] = 0.f;
      if (mn0 + mn < MN && k0 + k < K)
        v[e] = p[(mn0 + mn) * s_mn + (k0 + k) * s_k];
    }
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const int flat = t + MM_THREADS * e;
      constexpr bool KF = ST == ST_K16 || ST == ST_K4;
      const int mn = KF ? flat / MM_BK : flat % B;
      const int k = KF ? flat % MM_BK : flat / B;
      stage[pos(mn, k)] = v[e];
    }
  }
};

// f[i][kk] = element (mn + 32 i, h * 16 + kk) of a stage.
template <int ST, int B, int NB>
__device__ __forceinline__ void tile_frags(const float *stage, int mn, int li,
                                           int h, float (&f)[NB][16]) {
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    const int row = mn + 32 * i + li;
    if constexpr (ST == ST_K16 || ST == ST_K4) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const float4 w = *reinterpret_cast<const float4 *>(
            stage + StageTile<ST, B>::pos(row, h * 16 + 4 * q));
        f[i][4 * q + 0] = w.x;
        f[i][4 * q + 1] = w.y;
        f[i][4 * q + 2] = w.z;
        f[i][4 * q + 3] = w.w;
      }
    } else {
#pragma unroll
      for (int kk = 0; kk < 16; ++kk)
        f[i][kk] = stage[(h * 16 + kk) * B + row];
    }
  }
}

// Keeps a stage's direct loads where the source issues them, ahead of the
// MFMAs that overlap their latency.  The loads write LDS, not registers, so
// the scheduler sees no consumer and sank one stage's loads to the end of
// the other stage's MFMAs, right before the wait on them (config-5 step
// 1.8% slower that way).
__device__ __forceinline__ void pin_issued_loads() {
  __builtin_amdgcn_sched_barrier(0);
}

__device__ __forceinline__ void dl_wait_and_sync() {
  // the stage's direct loads have landed in LDS, then every wave sees them
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
}

// Range of a split product (mm_split_pack_kernel).  flags[0], flags[1]: the
// largest biased exponent in A and in B, or SP_HIGH if none is above.  Values
// are packed times 2^SP_SHIFT, so that every part of every float32, subnormal
// ones too, is a normal bfloat16, and what a product of parts loses below the
// normal range is under 2^-170, past the last bit of any float32.  What is
// left is the upper end: finite parts (values below 2^103), and K products
// below 2^(ea + eb + 2) times 2^(2 SP_SHIFT) that cannot overflow.
constexpr int SP_SHIFT = 24;
constexpr uint32_t SP_HIGH = 127 + 10;
__device__ __forceinline__ bool split_ok(const uint32_t *flags, int64_t K) {
  const int bits = 64 - __builtin_clzll(uint64_t(K)); // K < 2^bits
  const uint32_t ea = flags[0], eb = flags[1];
  return ea < 127 + 103 && eb < 127 + 103 &&
         int(ea + eb) - 2 * 127 + 2 + 2 * SP_SHIFT + bits <= 127;
}

// A BM x BN tile of a slice of K: 4 waves in a WM x WN grid, each a
// (BM / WM) x (BN / WN) block of 32x32 MFMA blocks.  Operands staged by
// direct loads into two named stage pairs (the k loop is unrolled by two so
// that every LDS access names its stage at compile time).  A K that is not a
// multiple of 32 starts with its partial k-tile, staged through registers.
//
// Bound: the fp32 MFMA pipe for large products (4000^3 at 134 TFLOP/s of the
// 149 that a large library product reaches here), HBM for a few rows against
// a large matrix (8x4096x4096: 67 MB in 18.8 us with its sum pass, 3.6 TB/s),
// and in between the number of workgroups: hence small tiles, which also
// waste less on ragged edges, and the split of K.  The 4-byte stages cost
// four times the load instructions of the 16-byte ones and run at 0.8 of
// their rate; through registers, one strided element at a time, odd row
// lengths had run at a fifth of it.
template <int SA, int SB, int BM, int BN, bool FAR = false>
__global__ __launch_bounds__(MM_THREADS, BM * BN >= 128 * 128 ? 2 : 3)
void mm_f32_tile_kernel(MMArgs g) {
  using TA = StageTile<SA, BM, FAR>;
  using TB = StageTile<SB, BN, FAR>;
  constexpr int WN = BM == BN ? 2 : (BM < BN ? 4 : 1), WM = 4 / WN;
  constexpr int NM = BM / WM / 32, NN = BN / WN / 32;
  __shared__ __align__(16) float sA0[TA::FLOATS], sB0[TB::FLOATS];
  __shared__ __align__(16) float sA1[TA::FLOATS], sB1[TB::FLOATS];
  const int t = threadIdx.x;
  const int lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int wm = wave / WN, wn = wave % WN;
  const int h = lane >> 5, li = lane & 31;
  if (g.flags && split_ok(g.flags, g.K) != g.run_if)
    return;
  const TileCoord tc = mm_tile_coord<BM, BN>(g);

  floatx16 acc[NM][NN];
#pragma unroll
  for (int i = 0; i < NM; ++i)
#pragma unroll
    for (int j = 0; j < NN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        acc[i][j][r] = 0.f;

  const int64_t k0 = int64_t(tc.slice) * g.kslice;
  const int64_t klen = g.K - k0 < g.kslice ? g.K - k0 : g.kslice;
  const int64_t full = klen / MM_BK;
  const int64_t tail = klen % MM_BK ? 1 : 0; // only in the last slice
  TA ta;
  TB tb;
  ta.init(tc.A + k0 * g.sAk, tc.m0, g.M, g.sAm, g.sAk, wave, lane);
  tb.init(tc.B + k0 * g.sBk, tc.n0, g.N, g.sBn, g.sBk, wave, lane);

  auto compute = [&](const float *sa, const float *sb) {
    float fa[NM][16], fb[NN][16];
    tile_frags<SA, BM, NM>(sa, wm * (BM / WM), li, h, fa);
    tile_frags<SB, BN, NN>(sb, wn * (BN / WN), li, h, fb);
#pragma unroll
    for (int kk = 0; kk < 16; ++kk)
#pragma unroll
      for (int i = 0; i < NM; ++i)
#pragma unroll
        for (int j = 0; j < NN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(
              fa[i][kk], fb[j][kk], acc[i][j], 0, 0, 0);
  };

  const int64_t steps = full + tail; // step 0 is the partial tile, if any
  if (tail) {
    const int64_t kt = k0 + full * MM_BK;
    TA::stage_tail(sA0, tc.A, tc.m0, g.M, g.sAm, g.sAk, kt, g.K, t);
    TB::stage_tail(sB0, tc.B, tc.n0, g.N, g.sBn, g.sBk, kt, g.K, t);
  } else {
    ta.issue(sA0, 0, wave);
    tb.issue(sB0, 0, wave);
  }
  dl_wait_and_sync();
  for (int64_t s = 0; s < steps; s += 2) {
    if (s + 1 < steps) {
      ta.issue(sA1, s + 1 - tail, wave);
      tb.issue(sB1, s + 1 - tail, wave);
    }
    pin_issued_loads();
    compute(sA0, sB0);
    dl_wait_and_sync();
    if (s + 1 >= steps)
      break;
    if (s + 2 < steps) {
      ta.issue(sA0, s + 2 - tail, wave);
      tb.issue(sB0, s + 2 - tail, wave);
    }
    pin_issued_loads();
    compute(sA1, sB1);
    dl_wait_and_sync();
  }

  // lane holds column li of each 32x32 block, rows 8*(r/4) + 4*h + (r%4)
#pragma unroll
  for (int i = 0; i < NM; ++i)
#pragma unroll
    for (int j = 0; j < NN; ++j) {
      const int64_t col = tc.n0 + wn * (BN / WN) + j * 32 + li;
      if (col >= g.N)
        continue;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int64_t row =
            tc.m0 + wm * (BM / WM) + i * 32 + (r >> 2) * 8 + h * 4 + (r & 3);
        if (row < g.M)
          mm_put(g, tc, row, col, acc[i][j][r]);
      }
    }
}

// ---------------------------------------- wide tile (direct-to-LDS, gfx950)

// Workgroup tile 256x256, k-tile 32, 8 waves in a 2x4 grid (two per SIMD),
// each wave owns a 128x64 block = 4x2 MFMA 32x32 blocks (128 accumulator
// registers per lane).  Between two barriers a SIMD runs 256 MFMAs against
// 128 in the 128x128 kernel, each A fragment read from LDS feeds two MFMAs
// and each B fragment four, and every operand element crosses from L2 once
// per 256 (not 128) outputs.  Two direct-loaded stages per operand take
// 128 KB of LDS: one workgroup per CU.  Used for M and N multiples of 256
// and K a multiple of 64 when the 256x256 tiles give every CU one.
constexpr int WD_BM = 256, WD_BN = 256, WD_THREADS = 512;
constexpr int WD_STAGE = WD_BM * MM_BK; // floats per operand stage (32 KB)

// As DirectTile, for 256 rows of full tiles (no row is clamped): each of the
// 4 instructions of a wave fills 1 KB of a stage:
//   layout K : [256 mn][32 k], chunks swizzled (dl_swz); 8 rows each.
//              Instruction j covers rows 32 wave + 8 j + lane / 8, whose
//              swizzle is (lane / 8) ^ (j & 1): two per-lane bases, the
//              rest uniform offsets.
//   layout MN: [32 k][256 mn]; one k row each: one per-lane base.
template <int LAY> struct WideDirectTile {
  const float *base[2];
  int64_t jstep; // elements between instruction j and j + 2 (K) / j + 1 (MN)
  int64_t kstep; // elements between two k-tiles
  __device__ __forceinline__ void init(const float *p, int64_t mn0,
                                       int64_t s_mn, int64_t s_k, int wave,
                                       int lane) {
    if constexpr (LAY == LAY_K) {
      const int64_t row = mn0 + wave * 32 + lane / 8;
#pragma unroll
      for (int par = 0; par < 2; ++par)
        base[par] = p + (row + 8 * par) * s_mn +
                    4 * ((lane % 8) ^ (lane / 8) ^ par);
      jstep = 16 * s_mn;
      kstep = 32;
    } else {
      base[0] = base[1] = p + int64_t(wave * 4) * s_k + mn0 + 4 * lane;
      jstep = s_k;
      kstep = 32 * s_k;
    }
  }
  __device__ __forceinline__ void issue(float *stage, int64_t kt,
                                        int wave) const {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float *src =
          LAY == LAY_K ? base[j & 1] + (j / 2) * jstep + kt * kstep
                       : base[0] + j * jstep + kt * kstep;
      __builtin_amdgcn_global_load_lds(
          (const __attribute__((address_space(1))) void *)src,
          (__attribute__((address_space(3))) void *)(stage +
                                                     (wave * 4 + j) * 256),
          16, 0, 0);
    }
  }
};

// f[i][kk] = element (mn + 32 i, h * 16 + 8 * half + kk) of a wide stage.
template <int LAY, int NB>
__device__ __forceinline__ void wd_frags(const float *stage, int mn, int li,
                                         int h, int half, float (&f)[NB][8]) {
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    const int row = mn + 32 * i + li;
    if constexpr (LAY == LAY_K) {
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const int pc = (4 * h + 2 * half + q) ^ dl_swz(row);
        const float4 w =
            *reinterpret_cast<const float4 *>(stage + row * 32 + pc * 4);
        f[i][4 * q + 0] = w.x;
        f[i][4 * q + 1] = w.y;
        f[i][4 * q + 2] = w.z;
        f[i][4 * q + 3] = w.w;
      }
    } else {
#pragma unroll
      for (int kk = 0; kk < 8; ++kk)
        f[i][kk] = stage[(h * 16 + 8 * half + kk) * WD_BM + row];
    }
  }
}

// The k-tile in two halves of 8 MFMA steps: 48 fragment registers live.
template <int LA, int LB>
__device__ __forceinline__ void wd_compute(const float *sa, const float *sb,
                                           int wm, int wn, int li, int h,
                                           floatx16 (&acc)[4][2]) {
#pragma unroll
  for (int half = 0; half < 2; ++half) {
    float fa[4][8], fb[2][8];
    wd_frags<LA, 4>(sa, wm * 128, li, h, half, fa);
    wd_frags<LB, 2>(sb, wn * 64, li, h, half, fb);
#pragma unroll
    for (int kk = 0; kk < 8; ++kk)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(
              fa[i][kk], fb[j][kk], acc[i][j], 0, 0, 0);
  }
}

template <int LA, int LB>
__global__ __launch_bounds__(WD_THREADS, 1) void mm_f32_mfma_wide_kernel(
    MMArgs g) {
  __shared__ __align__(16) float sA0[WD_STAGE], sB0[WD_STAGE];
  __shared__ __align__(16) float sA1[WD_STAGE], sB1[WD_STAGE];
  const int t = threadIdx.x;
  const int lane = t & 63, wave = t >> 6;
  const int wm = wave >> 2, wn = wave & 3;
  const int h = lane >> 5, li = lane & 31;
  if (g.flags && split_ok(g.flags, g.K) != g.run_if)
    return;
  const TileCoord tc = mm_tile_coord<WD_BM, WD_BN>(g);

  floatx16 acc[4][2];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        acc[i][j][r] = 0.f;

  WideDirectTile<LA> ta;
  WideDirectTile<LB> tb;
  const int64_t k0 = int64_t(tc.slice) * g.kslice;
  ta.init(tc.A + k0 * g.sAk, tc.m0, g.sAm, g.sAk, wave, lane);
  tb.init(tc.B + k0 * g.sBk, tc.n0, g.sBn, g.sBk, wave, lane);
  // The slice is a multiple of 64: k-tiles come in pairs, one per stage,
  // and the loop has a single exit (an exit between the two stages made the
  // compiler copy and spill the accumulators).
  const int64_t ktiles = g.kslice / 32;
  ta.issue(sA0, 0, wave);
  tb.issue(sB0, 0, wave);
  dl_wait_and_sync();
  for (int64_t kt = 0; kt < ktiles; kt += 2) {
    ta.issue(sA1, kt + 1, wave);
    tb.issue(sB1, kt + 1, wave);
    pin_issued_loads();
    wd_compute<LA, LB>(sA0, sB0, wm, wn, li, h, acc);
    dl_wait_and_sync();
    if (kt + 2 < ktiles) {
      ta.issue(sA0, kt + 2, wave);
      tb.issue(sB0, kt + 2, wave);
    }
    pin_issued_loads();
    wd_compute<LA, LB>(sA1, sB1, wm, wn, li, h, acc);
    dl_wait_and_sync();
  }

  // lane holds column li of each 32x32 block, rows 8*(r/4) + 4*h + (r%4)
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int64_t col = tc.n0 + wn * 64 + j * 32 + li;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int64_t row =
            tc.m0 + wm * 128 + i * 32 + (r >> 2) * 8 + h * 4 + (r & 3);
        mm_put(g, tc, row, col, acc[i][j][r]);
      }
    }
}

// ------------------------------------- large products on the bf16 matrix cores

// A float32 is the exact sum of three bfloat16 values (8 + 8 + 8 bits of
// significand), and a product of bfloat16 values is exact in float32.  So
// a . b = (a1 + a2 + a3) . (b1 + b2 + b3) can run on the bf16 MFMA, which does
// 16 times the work of the fp32 one per cycle (Henry, Tang and Heinecke,
// "Leveraging the bfloat16 Artificial Intelligence Datatype for Higher-
// Precision Computations", 2019): six of the nine products.  Of the three left
// out a2 b3 and a3 b2 are at most 2^-25 of a b each (2^-29 of it together in
// the median of normal operands, 2^-24 at most), half an ulp of a float32.
//
// Rounding: the bf16 MFMA rounds its sums down (towards -infinity), so no
// running sum of K stays in it.  The leading products a1 b1 of 32 k's are
// summed on the matrix cores (exactly, for a few terms of like size), and the
// vector unit adds that to the running sum, to nearest: one rounding of the
// sum per 32 k's, where the fp32 MFMA has 16.  Every other pair of steps the
// leading products are formed negated and subtracted: what is rounded down is
// then rounded up, and the results have no mean shift.  The five small
// products, 2^-8 of the leading one, have accumulators of their own on the
// matrix cores, which join the sum at the end: their roundings are 2^-8 of a
// float32's.
//
// Error against 64 bits, fp32 MFMA -> this, 2-norm: normal operands 4000^3
// 1.13e-6 -> 2.1e-7, 4096x300x4096 3.1e-7 -> 7.3e-8, 1024x8192x4096 8.1e-7 ->
// 2.1e-7 (51 non-zeros to a row of 8192: 8.0e-8 -> 5.1e-8); positive operands
// 8192x4096x4096 8.8e-7 -> 1.6e-7.  Mean shift of the results within 5e-10 of
// their mean magnitude (1e-9); of one column's mean 2e-7 (1.1e-6).  Sums of a
// single term, in 2^-24 of it: exact for a one-hot operand, largest error
// 1.0 -> 1.8 and rms 0.425 -> 0.436 for a diagonal one (the products left
// out); of two terms, rms 0.436 -> 0.368.
//
// Three kernels: mm_split_pack_kernel writes both operands as packed bf16
// planes, in the order in which the product's LDS stages hold them, zeros
// past every edge; mm_split_kernel multiplies; the slices of a split K are
// added as for the other tiles.  What six exact products cannot do as the
// fp32 kernel does -- infinities and NaN (0 x inf among the parts), values and
// products near the upper end of float32's range -- the pack kernel reports
// in a word per operand (split_ok): then it packs no further, mm_split_kernel
// returns at once and the fp32 kernel queued behind it does the work;
// otherwise that one returns at once.
constexpr int SP_B = 256, SP_K = 16;             // rows of a block, k of a step
constexpr int SP_PLANE = SP_B * SP_K;            // bf16 values
constexpr int SP_STEP = 3 * SP_PLANE * 2;        // bytes of a block's k step
constexpr int SP_BN = 128;                       // columns of a tile
constexpr int SP_STAGE = SP_STEP + SP_STEP / 2;  // LDS of one step of a tile
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

__global__ void mm_split_flags_kernel(uint32_t *flags) {
  if (threadIdx.x < 2)
    flags[threadIdx.x] = SP_HIGH;
}

struct SplitOperand {
  const float *p;
  int64_t rows, s_mn, s_k;
  char *packed;
  uint32_t blocks; // workgroups for this operand
  int vec;         // k unit-stride, 16-byte aligned
};

// A wave packs 32 rows of one k step: lane l the 8 k's of half l / 32 of row
// l % 32, 16 bytes in each plane, so that a wave writes 1 KB runs.  Packed
// order: [256-row block][k step][plane][32-row block][half][row][8].  The 4
// waves of a workgroup take consecutive k steps (64 k's: 256 bytes of a
// k-contiguous row).  HBM bound: 4 bytes read, 6 written per value.
__global__ __launch_bounds__(256) void mm_split_pack_kernel(
    SplitOperand a, SplitOperand b, int64_t K, uint32_t ksteps, uint32_t *flags) {
  const bool second = blockIdx.x >= a.blocks;
  const SplitOperand &o = second ? b : a;
  const uint32_t w = blockIdx.x - (second ? a.blocks : 0);
  const uint32_t kgroups = (ksteps + 3) / 4;
  const uint32_t rb = w / kgroups; // 32-row block
  const int lane = threadIdx.x & 63;
  const uint32_t step = (w - rb * kgroups) * 4 + (threadIdx.x >> 6);
  if (step >= ksteps)
    return;
  const int64_t row = int64_t(rb) * 32 + lane % 32;
  const int64_t k = int64_t(step) * SP_K + lane / 32 * 8;
  auto read = [&](int i) {
    return uint32_t(__builtin_amdgcn_readfirstlane(
        __hip_atomic_load(flags + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)));
  };
  const uint32_t seen[2] = {read(0), read(1)};
  float v[8];
  if (o.vec && row < o.rows && k + 8 <= K) {
    const float4 *q = reinterpret_cast<const float4 *>(o.p + row * o.s_mn + k);
    const float4 x = q[0], y = q[1];
    v[0] = x.x, v[1] = x.y, v[2] = x.z, v[3] = x.w;
    v[4] = y.x, v[5] = y.y, v[6] = y.z, v[7] = y.w;
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      v[e] = 0.f;
      if (row < o.rows && k + e < K)
        v[e] = o.p[row * o.s_mn + (k + e) * o.s_k];
    }
  }
  if (!split_ok(seen, K)) // another wave has settled it: nothing is packed
    return;
  bf16x8 p1, p2, p3;
  uint32_t high = 0;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const uint32_t ex = (__float_as_uint(v[e]) >> 23) & 255; // 127: 1.x
    high = high > ex ? high : ex;
    const float x = v[e] * float(1 << SP_SHIFT);
    p1[e] = __bf16(x);
    const float r = x - float(p1[e]);
    p2[e] = __bf16(r);
    p3[e] = __bf16(r - float(p2[e]));
  }
  char *dst = o.packed + (int64_t(rb / 8) * ksteps + step) * SP_STEP +
              (rb % 8) * (32 * SP_K * 2) + lane * 16;
  *reinterpret_cast<bf16x8 *>(dst) = p1;
  *reinterpret_cast<bf16x8 *>(dst + 2 * SP_PLANE) = p2;
  *reinterpret_cast<bf16x8 *>(dst + 4 * SP_PLANE) = p3;
  if (__any(high > seen[second])) { // no traffic on the word for ordinary data
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const uint32_t other = __shfl_xor(high, off, 64);
      high = high > other ? high : other;
    }
    if (lane == 0)
      atomicMax(flags + second, high);
  }
}

// 256x128 tiles, 8 waves in a 4x2 grid (two per SIMD) of 64x64: 2x2 blocks of
// 32x32 in two sets of accumulators (128 registers) and the leading products
// of two steps (64 more), 24 MFMAs of 32x32x16 per k step against 12 fragment
// reads (half of the LDS rate), so the matrix pipe and the chip's power (the
// clock falls below 2 GHz) are the bound.  Stages are copies of the packed
// operands (every load 1 KB of consecutive memory, conflict-free reads).
// With packing, in us, fp32 MFMA -> this: 8192x4096x4096 1949 -> 1345,
// 4000^3 1074 -> 708, 1024x8192x4096 511 -> 408, 8192x4096x1000 518 -> 387,
// 4093x301x4090 112 -> 84.  (Where this takes 738 for 4000^3: one running sum
// of all six products in 256x256 tiles, every sum rounded down, 682, with five
// times the error; the leading products of each step added apart, 759.)
__global__ __launch_bounds__(512, 1) void mm_split_kernel(
    MMArgs g, const char *pa, const char *pb, uint32_t ksteps, uint32_t kper,
    const uint32_t *flags) {
  if (!split_ok(flags, g.K))
    return;
  __shared__ __align__(16) char st0[SP_STAGE], st1[SP_STAGE], st2[SP_STAGE], st3[SP_STAGE];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const TileCoord tc = mm_tile_coord<SP_B, SP_BN>(g);
  // the sum of the leading products, that of the five small ones, and the
  // leading products of the present pair of steps
  floatx16 acc[2][2], low[2][2], top[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        acc[i][j][r] = low[i][j][r] = 0.f;
  const uint32_t s0 = tc.slice * kper;
  const uint32_t steps = ksteps - s0 < kper ? ksteps - s0 : kper;
  const char *a0 = pa + (tc.m0 / SP_B * ksteps + s0) * SP_STEP;
  const char *b0 = pb + (tc.n0 / SP_B * ksteps + s0) * SP_STEP;
  // A stage is A's step (24 KB) and B's half of one (3 planes of 4 KB): 36
  // pieces of 1 KB, piece 8 j + wave by this wave (the last 4 twice: every
  // wave then has 5 loads in flight per stage).
  const uint32_t bhalf = uint32_t(tc.n0 / SP_BN % 2) * SP_PLANE;
  auto issue = [&](char *stage, uint32_t s) {
    auto rsrc = [](const char *src) {
      const uint64_t ub = reinterpret_cast<uint64_t>(src);
      const uint32_t lo = __builtin_amdgcn_readfirstlane(uint32_t(ub));
      const uint32_t hi = __builtin_amdgcn_readfirstlane(uint32_t(ub >> 32));
      return __builtin_amdgcn_make_buffer_rsrc(
          reinterpret_cast<void *>((uint64_t(hi) << 32) | lo), 0, SP_STEP, BUF_WORD3);
    };
    const __amdgpu_buffer_rsrc_t ra = rsrc(a0 + int64_t(s) * SP_STEP);
    const __amdgpu_buffer_rsrc_t rb = rsrc(b0 + int64_t(s) * SP_STEP);
#pragma unroll
    for (int j = 0; j < 5; ++j) {
      if (j < 3) {
        const int piece = 8 * j + wave;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            ra, (__attribute__((address_space(3))) void *)(stage + piece * 1024), 16,
            piece * 1024 + lane * 16, 0, 0, 0);
      } else {
        const int q = j == 3 ? wave : 8 + wave % 4; // piece of B
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            rb, (__attribute__((address_space(3))) void *)(stage + SP_STEP + q * 1024),
            16, (q / 4) * (2 * SP_PLANE) + bhalf + (q % 4) * 1024 + lane * 16, 0, 0, 0);
      }
    }
  };
  // NEG: the pair's leading products are formed negated; LAST: its second step.
  auto compute = [&]<bool NEG, bool LAST>(const char *st) {
    bf16x8 a[2][3], b[2][3], b1[2];
#pragma unroll
    for (int p = 0; p < 3; ++p) {
#pragma unroll
      for (int i = 0; i < 2; ++i)
        a[i][p] = *reinterpret_cast<const bf16x8 *>(st + p * 2 * SP_PLANE +
                                                    (wm * 2 + i) * 1024 + lane * 16);
#pragma unroll
      for (int j = 0; j < 2; ++j)
        b[j][p] = *reinterpret_cast<const bf16x8 *>(st + SP_STEP + p * SP_PLANE +
                                                    (wn * 2 + j) * 1024 + lane * 16);
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      b1[j] = b[j][0];
      if constexpr (NEG) {
        typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
        b1[j] = __builtin_bit_cast(bf16x8, __builtin_bit_cast(u32x4, b1[j]) ^ 0x80008000u);
      }
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
        top[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
            a[i][0], b1[j], LAST ? top[i][j] : floatx16{}, 0, 0, 0);
    constexpr int PA[5] = {2, 0, 1, 1, 0}, PB[5] = {0, 2, 1, 0, 1};
#pragma unroll
    for (int q = 0; q < 5; ++q)
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          low[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i][PA[q]], b[j][PB[q]],
                                                              low[i][j], 0, 0, 0);
    if constexpr (LAST)
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            acc[i][j][r] = NEG ? acc[i][j][r] - top[i][j][r] : acc[i][j][r] + top[i][j][r];
  };
  // Four stages: a step's loads have three steps of MFMAs to land in, so the
  // wait leaves the 10 loads of the two steps after next in flight.  Past the
  // end the last step is loaded again, to keep the count.  steps is a
  // multiple of 4: one exit, so that the accumulators stay where they are.
  // lgkmcnt(0): this wave's reads of the stage that is loaded next are done
  // (the MFMAs that wait for them may be scheduled past the barrier).
  auto landed = [] {
    asm volatile("s_waitcnt vmcnt(10) lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  auto at = [&](uint32_t s) { return s < steps ? s : steps - 1; };
  issue(st0, 0);
  issue(st1, 1);
  issue(st2, 2);
  landed();
  for (uint32_t s = 0; s < steps; s += 4) {
    issue(st3, s + 3);
    pin_issued_loads();
    compute.template operator()<false, false>(st0);
    landed();
    issue(st0, at(s + 4));
    pin_issued_loads();
    compute.template operator()<false, true>(st1);
    landed();
    issue(st1, at(s + 5));
    pin_issued_loads();
    compute.template operator()<true, false>(st2);
    landed();
    issue(st2, at(s + 6));
    pin_issued_loads();
    compute.template operator()<true, true>(st3);
    landed();
  }
  // no load may still write the LDS of a workgroup that has ended
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  const int h = lane >> 5, li = lane & 31;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int64_t col = tc.n0 + wn * 64 + j * 32 + li;
      if (col >= g.N)
        continue;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int64_t row =
            tc.m0 + wm * 64 + i * 32 + (r >> 2) * 8 + h * 4 + (r & 3);
        if (row < g.M) // + 0: a sum of zeros is +0, as in the fp32 kernels
          mm_put(g, tc, row, col,
                 (acc[i][j][r] + low[i][j][r]) * (1.f / (1ull << 2 * SP_SHIFT)) + 0.f);
      }
    }
}

// C[b][m][n] (+)= part[0][b][m][n] + part[1][b][m][n] + ... in slice order (a
// fixed order: the result does not depend on scheduling).  V adjacent columns
// per work-item; V == 4 needs N a multiple of 4 and 16-byte rows of C.
template <int S, int V>
__global__ __launch_bounds__(256) void mm_splitk_sum_kernel(
    MMArgs g, FastDivU32 fdn, FastDivU32 fdm, uint32_t total) {
  // one work-item per V columns of one row, in a one-shot grid; the S slice
  // loads are independent (S is a template argument) and go out together
  const uint32_t q = blockIdx.x * 256u + threadIdx.x;
  if (q >= total || (g.flags && split_ok(g.flags, g.K) != g.run_if))
    return;
  const uint32_t rm = fdn.div(q); // batch * M + m
  const int64_t n = int64_t(q - rm * fdn.d) * V;
  uint32_t batch = fdm.div(rm);
  const int64_t m = rm - batch * uint32_t(g.M);
  const int64_t slice = int64_t(g.nbatch) * g.M * g.N;
  const float *p = g.part + int64_t(rm) * g.N + n;
  typedef float fv __attribute__((ext_vector_type(V)));
  fv w[S];
#pragma unroll
  for (int s = 0; s < S; ++s)
    w[s] = __builtin_nontemporal_load(
        reinterpret_cast<const fv *>(p + int64_t(s) * slice));
  fv v = w[0];
#pragma unroll
  for (int s = 1; s < S; ++s)
    v = v + w[s];
  if (g.bias) // the product's value, then the bias add (its own rounding)
#pragma unroll
    for (int e = 0; e < V; ++e)
      v[e] = v[e] + g.bias[(n + e) * g.sBias];
  float *C = g.C;
  for (int d = g.nb - 1; d >= 0; --d) {
    const uint32_t sz = uint32_t(g.bshape[d]);
    const uint32_t r = batch / sz;
    C += int64_t(batch - r * sz) * g.bsC[d];
    batch = r;
  }
  if constexpr (V > 1) {
    fv *dst = reinterpret_cast<fv *>(C + m * g.sCm + n);
    *dst = g.accumulate ? *dst + v : v;
  } else {
    float *dst = C + m * g.sCm + n * g.sCn;
    *dst = g.accumulate ? *dst + v[0] : v[0];
  }
}

// ------------------------------------------------ SIMT (non-fp32) kernel

template <class T> struct MMArgsT {
  const T *A;
  const T *B;
  T *C;
  int64_t M, N, K;
  int64_t sAm, sAk, sBk, sBn, sCm, sCn;
  int nb;
  int64_t bshape[MM_MAX_BATCH];
  int64_t bsA[MM_MAX_BATCH], bsB[MM_MAX_BATCH], bsC[MM_MAX_BATCH];
  int accumulate;
};

// A (16 TM) x (16 TM) tile by 256 work-items of TM x TM outputs each, every
// output summed in k order with the product and the sum rounded apart, as
// the reference's loop does (no split of K, no FMA, no MFMA: their results
// differ in the last bits).  Operands go through registers into [k][mn] LDS
// stages, the next k-tile's loads in flight under this one's arithmetic.
// Bound by the float64 instructions of the one wave that a tile gives each
// SIMD (5.8 cycles each from a single wave, 4 from several; a multiply and an
// add apart reach at most 39 TFLOP/s) and by LDS, where 2 TM values are read
// for TM^2 products; so a work-item holds as many outputs as leave every CU
// a tile (simt_tile).  float64 1000x784x1000: 225 us with one output per
// work-item, 105 with 4 x 4 (15 TFLOP/s; 113 with a k-tile of 16 and no XCD
// order, 125 with LDS reads at their use).
template <class T, int TM>
__global__ __launch_bounds__(256) void mm_simt_kernel(MMArgsT<T> g) {
  constexpr int TS = 16 * TM, BK = 32;
  constexpr int P = TS + 2; // LDS row of a k: 16-byte aligned pairs
  constexpr int E = TS * BK / 256; // values per work-item, operand and k-tile
  __shared__ __align__(16) T As[2][BK][P], Bs[2][BK][P];
  const int t = threadIdx.x;
  const int tx = t & 15, ty = t >> 4;
  // Each XCD (workgroups go to the 8 of them round-robin) takes one run of
  // tiles, in groups of 4 tile-rows walked column by column: its L2 then
  // holds few rows of A and few columns of B.
  const uint32_t gx = gridDim.x, gy = gridDim.y, n_tiles = gx * gy;
  uint32_t tile = blockIdx.y * gx + blockIdx.x;
  tile = tile % 8 * (n_tiles / 8) + min(tile % 8, n_tiles % 8) + tile / 8;
  const uint32_t g0 = tile / (4 * gx) * 4, rows = min(4u, gy - g0);
  const uint32_t in = tile - g0 * gx;
  const int64_t m0 = int64_t(g0 + in % rows) * TS, n0 = int64_t(in / rows) * TS;
  const T *A = g.A;
  const T *B = g.B;
  T *C = g.C;
  uint32_t rem = blockIdx.z;
  for (int d = g.nb - 1; d >= 0; --d) {
    const uint32_t sz = uint32_t(g.bshape[d]);
    const uint32_t q = rem / sz;
    const int64_t c = rem - q * sz;
    rem = q;
    A += c * g.bsA[d];
    B += c * g.bsB[d];
    C += c * g.bsC[d];
  }
  // consecutive work-items along the axis with the smaller stride
  const bool a_mn = g.sAm < g.sAk, b_mn = g.sBn < g.sBk;
  T va[E], vb[E];
  auto load = [&](int64_t k0) {
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const int f = t + 256 * e;
      const int64_t ma = m0 + (a_mn ? f % TS : f / BK), ka = k0 + (a_mn ? f / TS : f % BK);
      const int64_t nb = n0 + (b_mn ? f % TS : f / BK), kb = k0 + (b_mn ? f / TS : f % BK);
      va[e] = ma < g.M && ka < g.K ? A[ma * g.sAm + ka * g.sAk] : T(0);
      vb[e] = nb < g.N && kb < g.K ? B[nb * g.sBn + kb * g.sBk] : T(0);
    }
  };
  auto store = [&](int s) {
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const int f = t + 256 * e;
      As[s][a_mn ? f / TS : f % BK][a_mn ? f % TS : f / BK] = va[e];
      Bs[s][b_mn ? f / TS : f % BK][b_mn ? f % TS : f / BK] = vb[e];
    }
  };
  // Output i of an axis: pairs of neighbours, 32 apart (a wave's reads of 16
  // bytes per work-item are then contiguous).
  auto at = [](int i, int q) { return TM == 1 ? q : (i / 2) * 32 + q * 2 + (i & 1); };
  T acc[TM][TM];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TM; ++j)
      acc[i][j] = T(0);
  load(0);
  store(0);
  __syncthreads();
  int s = 0;
  for (int64_t k0 = 0; k0 < g.K; k0 += BK, s ^= 1) {
    if (k0 + BK < g.K)
      load(k0 + BK);
    if (k0 + BK <= g.K) {
      // Groups of U k's, each group's LDS reads issued before the previous
      // group's arithmetic: a tile alone on its CU has one wave per SIMD,
      // and nothing else would hide their latency.
      constexpr int U = 4 / TM;
      T a[2][U][TM], b[2][U][TM];
      auto read = [&](int p, int k) {
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
          for (int i = 0; i < TM; ++i) {
            a[p][u][i] = As[s][k + u][at(i, ty)];
            b[p][u][i] = Bs[s][k + u][at(i, tx)];
          }
      };
      read(0, 0);
#pragma unroll
      for (int k = 0; k < BK; k += U) {
        const int p = k / U & 1;
        if (k + U < BK)
          read(p ^ 1, k + U);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < U; ++u) {
          T c[TM][TM];
#pragma unroll
          for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TM; ++j)
              c[i][j] = a[p][u][i] * b[p][u][j];
#pragma unroll
          for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TM; ++j)
              acc[i][j] = acc[i][j] + c[i][j];
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    } else { // no term past K (a zero operand times another is not always 0)
#pragma unroll 1
      for (int k = 0; k < int(g.K - k0); ++k)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TM; ++j)
            acc[i][j] = acc[i][j] + As[s][k][at(i, ty)] * Bs[s][k][at(j, tx)];
    }
    if (k0 + BK < g.K)
      store(s ^ 1);
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TM; ++j) {
      const int64_t row = m0 + at(i, ty), col = n0 + at(j, tx);
      if (row < g.M && col < g.N) {
        T *dst = C + row * g.sCm + col * g.sCn;
        *dst = g.accumulate ? T(*dst + acc[i][j]) : acc[i][j];
      }
    }
}

namespace {

int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

bool aligned16(const void *p) {
  return reinterpret_cast<uintptr_t>(p) % 16 == 0;
}

// Adds the S slices in a.part into C.
void launch_sum(const MMArgs &a, int S) {
  const int64_t outs = int64_t(a.nbatch) * a.M * a.N;
  bool vec = a.N % 4 == 0 && a.sCn == 1 && a.sCm % 4 == 0 && aligned16(a.C);
  for (int d = 0; d < a.nb; ++d)
    vec = vec && a.bsC[d] % 4 == 0;
  const FastDivU32 fdn{uint32_t(vec ? a.N / 4 : a.N)}, fdm{uint32_t(a.M)};
  const int64_t items = vec ? outs / 4 : outs;
  const dim3 grid{unsigned(ceil_div(items, 256)), 1u, 1u};
  auto sum = [&]<int SS>() {
    if (vec)
      mm_splitk_sum_kernel<SS, 4>
          <<<grid, 256, 0, stream()>>>(a, fdn, fdm, uint32_t(items));
    else
      mm_splitk_sum_kernel<SS, 1>
          <<<grid, 256, 0, stream()>>>(a, fdn, fdm, uint32_t(items));
  };
  switch (S) {
  case 2:
    return sum.template operator()<2>();
  case 3:
    return sum.template operator()<3>();
  case 4:
    return sum.template operator()<4>();
  case 6:
    return sum.template operator()<6>();
  case 8:
    return sum.template operator()<8>();
  case 12:
    return sum.template operator()<12>();
  case 16:
    return sum.template operator()<16>();
  default:
    fail(NT_ERR_RUNTIME, "matmul: no split-K sum for this slice count");
  }
}

// Runs `launch(args)` over S slices of K (each kslice long) into scratch and
// adds them up; over one slice straight into C.  A split that the device
// memory has no room for is not made.
template <class F> void run_split(const MMArgs &a, int S, int64_t kslice, F launch) {
  MMArgs w = a;
  w.kslice = a.K;
  w.part = nullptr;
  const int64_t outs = int64_t(a.nbatch) * a.M * a.N;
  if (S == 1 || outs >= (int64_t(1) << 32)) {
    launch(w, 1);
    return;
  }
  void *part = nullptr;
  try {
    part = device_alloc(size_t(S) * size_t(outs) * sizeof(float));
  } catch (const Error &e) {
    if (e.code != NT_ERR_OOM)
      throw;
    launch(w, 1);
    return;
  }
  struct Free {
    void *p;
    ~Free() { device_free(p); }
  } owner{part};
  w.kslice = kslice;
  w.part = static_cast<float *>(part);
  launch(w, S);
  NT_LAUNCH_CHECK();
  launch_sum(w, S);
}

// Tile shape and slices of K of mm_f32_tile_kernel for one product: the
// lowest estimated time.  The estimate, in us, is the k-tiles of one slice
// times the larger of the MFMA time of the workgroups that share a CU and
// the latency of a k-tile's loads (which up to 4 resident workgroups, or 2 of
// the 128x128 tile, hide for each other), plus an epilogue per workgroup and
// the pass that adds the slices.  The constants were fitted to 1700 timings:
// 80 products from 16x16x10 to 8192x4096x1000, single and batched, in every
// tile shape and split; over those products the choice is 1.0% slower than
// the best one on average and 13% at worst (a 9 us product).  Before, one
// 128x128 tile per workgroup and no split: 64x784x256 59 us, now 10; 8x4096
// x4096 259 -> 19; 1000x784x1000 59 -> 20; 1537x1023x777 (odd rows) 174 ->
// 35; 4000^3 1035 -> 951 (the 32-bit offsets of the staging loads).
struct TileChoice {
  int bm, bn, S;
  int64_t kslice;
  double us; // the estimate
};

TileChoice choose_tile(int64_t M, int64_t N, int64_t K, int64_t nbatch, bool only64 = false) {
  constexpr double TK128 = 2.3, TK = 1.8; // us per 128x128x32 of MFMAs on a CU
  constexpr double LAT128 = 0.65, LAT = 0.49, EPI = 1.07;
  constexpr double SUM = 2.2, SUM_BYTES = 8.8e6; // us, bytes per us
  constexpr double SCRATCH = 64 << 20; // a split's partial results
  constexpr int SPLITS[] = {1, 2, 3, 4, 6, 8, 12, 16}; // as in run_split
  const int64_t cus = device_cu_count();
  const double outs = double(M) * double(N) * double(nbatch);
  const int64_t kt = ceil_div(K, MM_BK);
  int64_t kts[8]; // k-tiles of a slice, 0: no such split
  double sum[8];  // the pass that adds the slices
  for (int i = 0; i < 8; ++i) {
    const int S = SPLITS[i];
    const int64_t n = ceil_div(kt, S);
    const bool ok = S == 1 || (n * (S - 1) < kt && S * outs * sizeof(float) <= SCRATCH);
    kts[i] = ok ? n : 0;
    sum[i] = S == 1 ? 0 : SUM + (S + 1) * outs * (sizeof(float) / SUM_BYTES);
  }
  static constexpr int SHAPES[][2] = {{128, 128}, {64, 64}, {32, 128}, {128, 32}};
  TileChoice best{128, 128, 1, K, 0};
  double best_t = std::numeric_limits<double>::infinity();
  for (const auto &sh : SHAPES) {
    const int bm = sh[0], bn = sh[1];
    if (only64 && (bm != 64 || bn != 64))
      continue;
    const bool big = bm == 128 && bn == 128;
    const double area = bm * bn / (128. * 128.);
    const int64_t tiles = ceil_div(M, bm) * ceil_div(N, bn) * nbatch;
    for (int i = 0; i < 8; ++i) {
      if (kts[i] == 0)
        continue;
      const int64_t per_cu = ceil_div(tiles * SPLITS[i], cus);
      const double mfma = double(per_cu) * (big ? TK128 : TK) * area;
      const double lat = double(big ? (per_cu + 1) / 2 : (per_cu + 3) / 4) *
                         (big ? LAT128 : LAT);
      const double t =
          double(kts[i]) * std::max(mfma, lat) + double(per_cu) * EPI * area + sum[i];
      if (t < best_t) {
        best_t = t;
        best = {bm, bn, SPLITS[i], i == 0 ? K : kts[i] * MM_BK, t};
      }
    }
  }
  return best;
}

template <int SA, int SB, int BM, int BN, bool FAR = false>
void launch_tile(const MMArgs &a, const TileChoice &c) {
  run_split(a, c.S, c.kslice, [](MMArgs w, int S) {
    w.tiles_m = ceil_div(w.M, BM);
    w.tiles_n = ceil_div(w.N, BN);
    const int64_t blocks = w.tiles_m * w.tiles_n * w.nbatch * S;
    if (blocks >= (int64_t(1) << 31))
      fail(NT_ERR_RUNTIME, "matmul: problem too large");
    mm_f32_tile_kernel<SA, SB, BM, BN, FAR>
        <<<dim3(unsigned(blocks)), MM_THREADS, 0, stream()>>>(w);
  });
}

template <int SA, int SB> void launch_stages(const MMArgs &a, bool far) {
  // Far strides: 64x64 only (64-bit offsets of a 128x128 tile's stages would
  // spill).  [64, 8M] times its transpose 743 ms (one element at a time through
  // registers, K unsplit) -> 17, its transpose times [64, 64] 3.2 -> 1.2.
  if (far)
    return launch_tile<SA, SB, 64, 64, true>(a, choose_tile(a.M, a.N, a.K, a.nbatch, true));
  const TileChoice c = choose_tile(a.M, a.N, a.K, a.nbatch);
  if (c.bm == 64)
    launch_tile<SA, SB, 64, 64>(a, c);
  else if (c.bm == 32)
    launch_tile<SA, SB, 32, 128>(a, c);
  else if (c.bn == 32)
    launch_tile<SA, SB, 128, 32>(a, c);
  else
    launch_tile<SA, SB, 128, 128>(a, c);
}

// Outputs per work-item and axis of mm_simt_kernel: a k step of a tile costs
// about TM units of LDS time (2 TM reads per work-item) for TM^2 outputs, so
// the larger tile wins unless it leaves CUs without one.
int simt_tile(int64_t M, int64_t N, int64_t nbatch) {
  int best = 1;
  int64_t best_t = std::numeric_limits<int64_t>::max();
  for (int tm : {4, 2, 1}) {
    const int64_t tiles = ceil_div(M, 16 * tm) * ceil_div(N, 16 * tm) * nbatch;
    const int64_t t = ceil_div(tiles, device_cu_count()) * tm;
    if (t < best_t) {
      best_t = t;
      best = tm;
    }
  }
  return best;
}

template <int LA, int LB> bool launch_wide(const MMArgs &a) {
  // 256x256 tiles when they (or, for one product, they times a split of
  // K into 2, 4 or 8 slices of at least 1024) give every CU one
  if (a.M % WD_BM != 0 || a.N % WD_BN != 0 || a.K % 64 != 0)
    return false;
  const int64_t tiles = a.M / WD_BM * (a.N / WD_BN) * a.nbatch;
  const int64_t cus = device_cu_count();
  int S = 1;
  while (tiles * S < cus && a.nbatch == 1 && S < 8 && a.K % (64 * 2 * S) == 0 &&
         a.K / (2 * S) >= 1024)
    S *= 2;
  if (tiles * S < cus)
    return false;
  run_split(a, S, a.K / S, [](MMArgs w, int slices) {
    w.tiles_m = w.M / WD_BM;
    w.tiles_n = w.N / WD_BN;
    mm_f32_mfma_wide_kernel<LA, LB>
        <<<dim3(unsigned(w.tiles_m * w.tiles_n * w.nbatch * slices)), WD_THREADS,
           0, stream()>>>(w);
  });
  return true;
}

// The product through packed bf16 planes (mm_split_kernel), where that is
// estimated to take no longer than the fp32 kernels, f32_us; false: not taken.
// A k step of a tile takes 0.8 us with few CUs at work and 1.12 with all (the
// clock falls with the power), packing 10 bytes per value at 5 TB/s and the
// three small launches 12 us; measured / estimated / fp32 measured, in us:
// 4000^3 630 / 660 / 1021, 8192x4096x1000 367 / 383 / 529, 1024x8192x4096
// 401 / 404 / 505, 6112x868x3912 229 / 245 / 365, 4096x320x4096 78 / 80 / 101.
// Over 32 products that take the planes they were 1.13 to 1.70 times as fast as
// the fp32 kernels, 1.34 in the mean.  ak, bk: the operand has 16-byte aligned
// rows along k.
template <class FB>
bool launch_split(const MMArgs &a, double f32_us, bool ak, bool bk, FB fallback) {
  if (f32_us < 40 || a.K >= (int64_t(1) << 27))
    return false;
  const int64_t tm = ceil_div(a.M, SP_B), tn = ceil_div(a.N, SP_B);
  const int64_t ksteps = ceil_div(a.K, 4 * SP_K) * 4; // in fours, see the kernel
  const int64_t tiles = tm * ceil_div(a.N, SP_BN);
  const int64_t cus = device_cu_count();
  const double outs = double(a.M) * double(a.N);
  double best_t = std::numeric_limits<double>::infinity();
  int S = 1;
  for (int s : {1, 2, 3, 4, 6, 8}) {
    const int64_t per = ceil_div(ksteps, 4 * s) * 4;
    if (ceil_div(ksteps, per) != s)
      continue;
    const double busy = std::min(1.0, double(tiles * s) / double(cus));
    double t = double(ceil_div(tiles * s, cus)) * (double(per) * (0.8 + 0.32 * busy) + 9);
    if (s > 1)
      t += 4 + (s + 1) * outs * 4 / 6e6;
    if (t < best_t) {
      best_t = t;
      S = s;
    }
  }
  const double pack = 12 + double(tm + tn) * SP_B * double(a.K) * 10 / 5e6;
  if (best_t + pack > f32_us)
    return false;
  const size_t abytes = size_t(tm * ksteps) * SP_STEP, bbytes = size_t(tn * ksteps) * SP_STEP;
  const size_t pbytes = S > 1 ? size_t(S) * size_t(outs) * sizeof(float) : 0;
  if (outs >= 4294967296. || tiles * S >= (int64_t(1) << 31) ||
      (tm + tn) * 8 * ceil_div(ksteps, 4) >= (int64_t(1) << 31))
    return false;
  void *scratch = nullptr;
  try {
    scratch = device_alloc(256 + abytes + bbytes + pbytes);
  } catch (const Error &e) {
    if (e.code != NT_ERR_OOM)
      throw;
    return false;
  }
  struct Free {
    void *p;
    ~Free() { device_free(p); }
  } owner{scratch};
  uint32_t *flags = static_cast<uint32_t *>(scratch);
  char *pa = static_cast<char *>(scratch) + 256, *pb = pa + abytes;
  mm_split_flags_kernel<<<1, 64, 0, stream()>>>(flags);
  NT_LAUNCH_CHECK();
  const uint32_t kgroups = uint32_t(ceil_div(ksteps, 4));
  const SplitOperand oa{a.A, a.M, a.sAm, a.sAk, pa, uint32_t(tm * 8) * kgroups, ak};
  const SplitOperand ob{a.B, a.N, a.sBn, a.sBk, pb, uint32_t(tn * 8) * kgroups, bk};
  mm_split_pack_kernel<<<oa.blocks + ob.blocks, 256, 0, stream()>>>(
      oa, ob, a.K, uint32_t(ksteps), flags);
  NT_LAUNCH_CHECK();
  MMArgs w = a;
  w.tiles_m = tm;
  w.tiles_n = ceil_div(a.N, SP_BN);
  w.part = S > 1 ? reinterpret_cast<float *>(pb + bbytes) : nullptr;
  mm_split_kernel<<<unsigned(tiles * S), 512, 0, stream()>>>(
      w, pa, pb, uint32_t(ksteps), uint32_t(ceil_div(ksteps, 4 * S) * 4), flags);
  NT_LAUNCH_CHECK();
  w.flags = flags;
  if (S > 1) {
    w.run_if = true;
    launch_sum(w, S);
    NT_LAUNCH_CHECK();
  }
  w.part = nullptr;
  w.run_if = false;
  fallback(w);
  NT_LAUNCH_CHECK();
  return true;
}

// fp32 product; al: both operands' bases and batch strides are 16-byte
// aligned; planes: large single products may run on bf16 planes.
void launch_f32(const MMArgs &a, bool al, bool planes) {
  // 16-byte loads need the unit-stride extent and the other stride to be
  // multiples of 4 elements.
  const bool ak = al && a.sAk == 1 && a.sAm % 4 == 0 && a.K % 4 == 0;
  const bool am = al && a.sAm == 1 && a.sAk % 4 == 0 && a.M % 4 == 0;
  const bool bn = al && a.sBn == 1 && a.sBk % 4 == 0 && a.N % 4 == 0;
  const bool bk = al && a.sBk == 1 && a.sBn % 4 == 0 && a.K % 4 == 0;
  const bool wide = (ak || am) && (bn || bk);
  const bool a_mn = wide ? !ak : a.sAm < a.sAk;
  const bool b_mn = wide ? bn : a.sBn < a.sBk;
  constexpr int64_t FAR = int64_t(1) << 22;
  const bool far = a.sAm > FAR || a.sAk > FAR || a.sBn > FAR || a.sBk > FAR;
  auto tiles = [&](const MMArgs &g) {
    if (wide) {
      if (a_mn)
        b_mn ? launch_stages<ST_MN16, ST_MN16>(g, far) : launch_stages<ST_MN16, ST_K16>(g, far);
      else
        b_mn ? launch_stages<ST_K16, ST_MN16>(g, far) : launch_stages<ST_K16, ST_K16>(g, far);
    } else {
      if (a_mn)
        b_mn ? launch_stages<ST_MN4, ST_MN4>(g, far) : launch_stages<ST_MN4, ST_K4>(g, far);
      else
        b_mn ? launch_stages<ST_K4, ST_MN4>(g, far) : launch_stages<ST_K4, ST_K4>(g, far);
    }
  };
  auto large = [&](const MMArgs &g) {
    return wide && (a_mn ? (b_mn ? launch_wide<LAY_MN, LAY_MN>(g)
                                 : launch_wide<LAY_MN, LAY_K>(g))
                         : (b_mn ? launch_wide<LAY_K, LAY_MN>(g)
                                 : launch_wide<LAY_K, LAY_K>(g)));
  };
  if (planes && !far && a.nbatch == 1) {
    // What the fp32 kernels take: large tiles at 131 TFLOP/s or the tile
    // kernel's estimate, of which 0.96 to 1.5 were measured (4-byte loads:
    // 1.09 to 1.3; medians 1.1 and 1.2 over 100 products).
    const double flops_us = 2. * double(a.M) * double(a.N) * double(a.K) / 131e6;
    if (flops_us > 20) {
      const double us = std::max(flops_us, choose_tile(a.M, a.N, a.K, 1).us);
      if (launch_split(a, (wide ? 1.08 : 1.15) * us, ak, bk, [&](const MMArgs &g) {
            if (!large(g))
              tiles(g);
          }))
        return;
    }
  }
  if (large(a))
    return;
  tiles(a);
}

} // namespace
} // namespace nt

using namespace nt;

namespace {

// C (+)= A . B, or C = A . B + bias (bias: one value per column of C,
// fp32 only, never with accumulate).  planes: see launch_f32.
void matmul_run(const nt_view *a, const nt_view *b, const nt_view *c,
                int32_t accumulate, const nt_view *bias, bool planes) {
  {
    check_view(a, "matmul");
    check_view(b, "matmul");
    check_view(c, "matmul");
    if (a->dtype != b->dtype || a->dtype != c->dtype)
      fail(NT_ERR_RUNTIME, "matmul: dtype mismatch");
    if (a->ndim != b->ndim || a->ndim != c->ndim)
      fail(NT_ERR_VALUE, "matmul: x1 and x2 have different ndim.");
    if (a->ndim < 2)
      fail(NT_ERR_VALUE, "matmul: kernel should be called with >=2d tensors.");
    const int nd = a->ndim, nb = nd - 2;
    for (int d = 0; d < nb; ++d)
      if (a->shape[d] != b->shape[d] || a->shape[d] != c->shape[d])
        fail(NT_ERR_VALUE, "Invalid broacast shapes.");
    const int64_t M = a->shape[nd - 2], K = a->shape[nd - 1];
    const int64_t N = b->shape[nd - 1];
    if (b->shape[nd - 2] != K)
      fail(NT_ERR_VALUE, "Invalid matmul shape.");
    if (c->shape[nd - 2] != M || c->shape[nd - 1] != N)
      fail(NT_ERR_RUNTIME, "matmul: output shape mismatch");
    if (a->dtype == NT_BOOL)
      fail(NT_ERR_VALUE, "Invalid dtype.");
    int64_t nbatch = 1;
    for (int d = 0; d < nb; ++d)
      nbatch *= a->shape[d];
    if (bias) {
      check_view(bias, "matmul_bias");
      if (a->dtype != NT_FLOAT32 || bias->dtype != NT_FLOAT32)
        fail(NT_ERR_VALUE, "matmul_bias: float32 operands only");
      if (accumulate)
        fail(NT_ERR_RUNTIME, "matmul_bias: no accumulate form");
      if (bias->ndim != 1 || bias->shape[0] != N)
        fail(NT_ERR_RUNTIME, "matmul_bias: bias must be 1-D with one value per column");
    }
    if (M == 0 || N == 0 || nbatch == 0)
      return;
    if (K == 0 && bias) {
      // C = fl(0 + bias), the bias broadcast over the rows (and batches), as
      // the empty product followed by the add gives (a -0.0 bias gives +0.0)
      DeviceScratch zero_buf(sizeof(float));
      if (nt_fill(zero_buf.get(), NT_FLOAT32, 1, 0.0) != NT_OK)
        fail(NT_ERR_RUNTIME, nt_last_error());
      nt_view zv = *c, bv = *c;
      zv.data = zero_buf.get();
      zv.offset = 0;
      bv.data = bias->data;
      bv.offset = bias->offset;
      for (int d = 0; d < nd; ++d)
        zv.strides[d] = bv.strides[d] = 0;
      bv.strides[nd - 1] = bias->strides[0];
      const int rc = nt_binary(NT_ADD, &zv, &bv, c);
      if (rc != NT_OK)
        fail(rc, nt_last_error());
      return;
    }
    if (K == 0) {
      if (!accumulate) {
        dispatch_arith(c->dtype, [&]<class T>() {
          // C = 0 through the copy kernel from a broadcast zero.
          DeviceScratch zero_buf(sizeof(T));
          T *zero = zero_buf.get<T>();
          if (nt_fill(zero, c->dtype, 1, 0.0) != NT_OK)
            fail(NT_ERR_RUNTIME, nt_last_error());
          nt_view zv = *c;
          zv.data = zero;
          zv.offset = 0;
          for (int d = 0; d < zv.ndim; ++d)
            zv.strides[d] = 0;
          const int rc = nt_copy(&zv, c);
          if (rc != NT_OK)
            fail(rc, nt_last_error());
        });
      }
      return;
    }
    // Size-1 dims carry no stride information; normalise them to 0.
    auto st = [](const nt_view *v, int d) {
      return v->shape[d] == 1 ? int64_t(0) : v->strides[d];
    };
    const int64_t sAm = st(a, nd - 2), sAk = st(a, nd - 1);
    const int64_t sBk = st(b, nd - 2), sBn = st(b, nd - 1);
    const int64_t sCm = c->strides[nd - 2], sCn = c->strides[nd - 1];

    if (a->dtype == NT_FLOAT32) {
      MMArgs g{};
      g.A = typed_ptr<const float>(a);
      g.B = typed_ptr<const float>(b);
      g.C = typed_ptr<float>(c);
      g.M = M;
      g.N = N;
      g.K = K;
      g.sAm = sAm;
      g.sAk = sAk;
      g.sBk = sBk;
      g.sBn = sBn;
      g.sCm = sCm;
      g.sCn = sCn;
      g.nb = nb;
      bool al = aligned16(g.A) && aligned16(g.B);
      for (int d = 0; d < nb; ++d) {
        g.bshape[d] = a->shape[d];
        g.bsA[d] = st(a, d);
        g.bsB[d] = st(b, d);
        g.bsC[d] = st(c, d);
        if (g.bsA[d] % 4 != 0 || g.bsB[d] % 4 != 0)
          al = false;
      }
      if (nbatch >= (int64_t(1) << 31))
        fail(NT_ERR_RUNTIME, "matmul: problem too large");
      g.nbatch = uint32_t(nbatch);
      g.accumulate = accumulate ? 1 : 0;
      g.kslice = K;
      g.part = nullptr;
      g.bias = bias ? typed_ptr<const float>(bias) : nullptr;
      g.sBias = bias ? bias->strides[0] : 0;
      launch_f32(g, al, planes);
      NT_LAUNCH_CHECK();
      return;
    }

    dispatch_arith(a->dtype, [&]<class T>() {
      MMArgsT<T> g{};
      g.A = typed_ptr<const T>(a);
      g.B = typed_ptr<const T>(b);
      g.C = typed_ptr<T>(c);
      g.M = M;
      g.N = N;
      g.K = K;
      g.sAm = sAm;
      g.sAk = sAk;
      g.sBk = sBk;
      g.sBn = sBn;
      g.sCm = sCm;
      g.sCn = sCn;
      g.nb = nb;
      for (int d = 0; d < nb; ++d) {
        g.bshape[d] = a->shape[d];
        g.bsA[d] = st(a, d);
        g.bsB[d] = st(b, d);
        g.bsC[d] = st(c, d);
      }
      g.accumulate = accumulate ? 1 : 0;
      if (nbatch > 65535)
        fail(NT_ERR_RUNTIME, "matmul: too many batches for the SIMT path");
      auto run = [&]<int TM>() {
        const dim3 grid{unsigned(ceil_div(N, 16 * TM)), unsigned(ceil_div(M, 16 * TM)),
                        unsigned(nbatch)};
        mm_simt_kernel<T, TM><<<grid, 256, 0, stream()>>>(g);
      };
      switch (simt_tile(M, N, nbatch)) {
      case 4:
        run.template operator()<4>();
        break;
      case 2:
        run.template operator()<2>();
        break;
      default:
        run.template operator()<1>();
      }
      NT_LAUNCH_CHECK();
    });
  }
}

} // namespace

extern "C" {

int nt_matmul(const nt_view *a, const nt_view *b, const nt_view *c,
              int32_t accumulate) {
  return guard([&] { matmul_run(a, b, c, accumulate, nullptr, true); });
}

int nt_matmul_bias(const nt_view *a, const nt_view *b, const nt_view *bias,
                   const nt_view *c) {
  return guard([&] { matmul_run(a, b, c, 0, bias, true); });
}

// A layer's forward keeps the fp32 unit's rounding at every size: whether a
// pre-activation near a ReLU's corner is kept is decided by its last bits,
// and one value on the other side moves a whole term of every gradient before
// it (the 4-layer MLP at batch 8192, 3e7 values: gradients 8e-4 away from
// those of the fp32 kernels, with products that were themselves as exact).
int nt_linear(const nt_view *x, const nt_view *w, const nt_view *bias,
              const nt_view *y) {
  return guard([&] { matmul_run(x, w, y, 0, bias, false); });
}

} // extern "C"
