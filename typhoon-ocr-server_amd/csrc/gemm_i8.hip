// gemm_i8.hip -- int8 GEMMs of prefill: per-token codes (W8A8) or the four
// int8 planes of fp32 tokens (W8A32) x int8 weights on v_mfma_i32_16x16x64_i8
// with K stages staged through an LDS ring.  Two kernels: the LDS-staged one
// below for few tiles of codes, the quadrant one further down for the rest.
//
// Reference: kernel/w8a8_kernel.c:259-268 (w8a8_gemm dequantizes both
// operands and calls cblas_sgemm).  Here the int32 sum is exact and the fp32
// epilogue is y = fl(fl(fl(acc) * ws[n]) * xs[m]) (+ bias[n] as its own
// rounding), ~4e-7 relative L2 from the reference's dequant-then-SGEMM.
//
// Both operands are stored as 16x64 int8 tiles (tl_common.h), so a K stage
// of the work-group's A rows and B columns is a list of whole 1 KiB tiles:
// each is copied global -> LDS directly (global_load_lds_dwordx4, no staging
// registers), and every MFMA operand is read back with one ds_read_b128 per
// lane at consecutive addresses (no bank conflicts, no swizzle needed).
// NST stage buffers form a ring, so NST-1 stages of copies are in flight while
// a stage's MFMAs run; one barrier per stage.
//
// Work-group tile (16 MT) x (16 NT); waves WM x WN each own a
// (16 MT/WM) x (16 NT/WN) block of 16x16 accumulators, each computed as the
// transposed product (weights as the MFMA's first operand) so that a lane ends
// up with 4 consecutive columns of one output row (16-byte stores).  Tiles are ordered so
// that the work-groups placed on one XCD (dispatch is round-robin over the 8
// XCDs) share a band of B columns and all of A, which then stays in that
// XCD's 4 MB L2.
#include <algorithm>
#include <atomic>

#include "gemm_common.h"
#include "tl_kernels.h"

namespace tl {

struct GemmI8Args {
  const uint8_t* At;    // activation code tiles [KB][MG]
  const uint8_t* Bt;    // weight tiles [KB][NG]
  const float* ws;      // [N]
  const float* xs;      // [M]
  const int* xe;        // OUT_F32_X4: per-token exponents [M / 4]
  const float* xraw;    // OUT_F32_X4: the fp32 token rows (null: NaN for a non-finite row)
  int ldxr;
  const float* bias;    // [N] or null
  void* Y;              // fp32 [M][ldy] or int32 (OUT_I32)
  int ldy;
  int M, N, K, KB, MG, NG;
  int ntm, ntn;         // work-group tiles along M and N
  int out;
  const uint8_t* zero_tile;  // 1 KiB of zeros (source of k-blocks past K)
  int S;                // K slices per tile
  int32_t* part;        // S > 1: int32 partial tiles [tiles][S][16 MT x 16 NT]
  uint32_t* cnt;        // S > 1: zeroed arrival counters [tiles]
  int xa;               // 2: each XCD owns a block of half the tile rows (tile_of)
};

// Work-group -> tile.  Dispatch is round-robin over the 8 XCDs: work-group b
// runs on XCD b % 8 as that XCD's (b / 8)-th.  When the tile columns divide
// over the XCDs, XCD x owns a band of ntn / 8 columns and walks it in groups
// of 4 tile rows x the whole band, so the ~32 work-groups an XCD runs at once
// share 4 A panels and the band's B panels, which fit its 4 MB L2 (one column
// at a time keeps ~32 A panels live at once: past the L2 once A exceeds it,
// e.g. the 4800 plane rows of a 1200-token fp32 batch).  Otherwise each XCD
// takes a run of consecutive tiles (columns of tm).
// With xa = 2 (one tile per CU, ntm even, ntn a multiple of 4, set by the
// launcher where it fills fewer L2 lines) XCD x owns rows (x % 2) ntm / 2 ..
// and columns (x / 2) ntn / 4 .., so it fills half of A and a quarter of the
// weights into its L2 instead of all of A and an eighth of the weights:
// 20 % fewer fills at M = 1024, N = 2048, K = 6144 (50 against 63 MB), and
// 23.2-23.9 -> 22.2-22.4 us for the LDS-staged kernel in a same-run A/B.
__device__ __forceinline__ void tile_of(int b, int ntm, int ntn, int& tm, int& tn, int xa = 1) {
  if (xa == 2) {
    const int x = b % 8, j = b / 8, bm = ntm / 2, bn = ntn / 4;
    tm = (x % 2) * bm + j % bm;
    tn = (x / 2) * bn + j / bm;
    return;
  }
  if (ntn % 8 == 0) {
    const int x = b % 8, j = b / 8, bw = ntn / 8;
    const int grp = j / (4 * bw), r = j - grp * 4 * bw;
    const int rows = min(4, ntm - 4 * grp);
    tm = 4 * grp + r % rows;
    tn = x * bw + r / rows;
  } else {
    const int ntiles = ntm * ntn;
    int t = b;
    if (ntiles % 8 == 0) t = (b % 8) * (ntiles / 8) + b / 8;
    tn = t / ntm;
    tm = t - tn * ntm;
  }
}

// K slices (a.S > 1): every work-group of the tile stores its int32 sums
// (16-byte write-through stores), waits for their acknowledgement and counts
// in; the last to arrive adds the S slices into its accumulators (exact integer
// sums, so any order gives the same bits; slice order here) and returns true.
// flag: a word of the stage ring, which no copy or read uses any more (an LDS
// word of its own would push the 80 KiB rings past two work-groups per CU).
template <int NW, int FM, int FN>
__device__ __forceinline__ bool merge_slices(const GemmI8Args& a, v4i (&acc)[FM][FN], int wv, int lane, int bt, int ks,
                                             int* flag) {
  constexpr int TF = NW * FM * FN * 256;        // sums per partial tile
  int32_t* mine = a.part + ((size_t)bt * a.S + ks) * TF;
#pragma unroll
  for (int i = 0; i < FM; i++)
#pragma unroll
    for (int j = 0; j < FN; j++)
      st_agent4(reinterpret_cast<float*>(mine) + (((wv * FM + i) * FN + j) * 64 + lane) * 4,
                __builtin_bit_cast(v4f, acc[i][j]));
  asm volatile("" ::: "memory");
  wait_vm<0>();                               // this thread's partial stores are acknowledged
  asm volatile("" ::: "memory");
  __syncthreads();
  if (threadIdx.x == 0)
    *flag = __hip_atomic_fetch_add(a.cnt + bt, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (uint32_t)(a.S - 1);
  __syncthreads();
  if (!*flag) return false;
  // the merger's acquire: the slices are read after the counter showed them
  // all arrived (agent scope, once per tile; plain 16-byte loads after it)
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
  constexpr int QB = FM * FN <= 8 ? 4 : (FM * FN <= 16 ? 2 : 1);   // slices in flight together
  const int32_t* slices = a.part + (size_t)bt * a.S * TF;
  for (int q0 = 0; q0 < a.S; q0 += QB) {
    v4i pv[QB][FM][FN];
#pragma unroll
    for (int u = 0; u < QB; u++)
#pragma unroll
      for (int i = 0; i < FM; i++)
#pragma unroll
        for (int j = 0; j < FN; j++)
          pv[u][i][j] = *reinterpret_cast<const v4i*>(slices + (size_t)min(q0 + u, a.S - 1) * TF +
                                                      (((wv * FM + i) * FN + j) * 64 + lane) * 4);
#pragma unroll
    for (int u = 0; u < QB; u++) {
      if (q0 + u >= a.S) break;
#pragma unroll
      for (int i = 0; i < FM; i++)
#pragma unroll
        for (int j = 0; j < FN; j++)
#pragma unroll
          for (int r = 0; r < 4; r++) acc[i][j][r] = q0 + u == 0 ? pv[u][i][j][r] : acc[i][j][r] + pv[u][i][j][r];
    }
  }
  if (threadIdx.x == 0) __hip_atomic_store(a.cnt + bt, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return true;
}

// Stage ring of NST buffers.  Every K stage is NW*PW whole 1 KiB tiles, each
// copied global -> LDS by one wave with one global_load_lds_dwordx4 (lane l
// writes bytes 16l..16l+15 of the tile, i.e. the tile layout itself).  Stage s
// lives in buffer s % NST; the ring is unrolled so every buffer is a distinct
// LDS object and the compiler keeps only the explicit waits in `step`.  The
// MFMA fragments of a stage are read from LDS one step before its MFMAs run.
template <int MT, int NT, int KT, int NST, int WM, int WN>
__global__ __launch_bounds__(64 * WM * WN) void gemm_i8_lds_kernel(GemmI8Args a) {
  constexpr int NW = WM * WN;
  constexpr int TA = MT * KT, TB = NT * KT, TS = TA + TB;  // tiles per stage
  static_assert(TS % NW == 0, "stage tiles must divide evenly over the waves");
  constexpr int PW = TS / NW;                              // tiles copied per wave per stage
  constexpr int FM = MT / WM, FN = NT / WN;                // 16x16 accumulators per wave
  static_assert(MT % WM == 0 && NT % WN == 0, "wave grid must divide the tile");
  static_assert(NST >= 2 && NST <= 8 && NST % 2 == 0, "2, 4, 6 or 8 stage buffers");
  static_assert(KT == 1, "one k-block per stage");
  static_assert(PW * (NST - 1) < 64, "vmcnt range");

  // one distinct LDS object per ring slot (unused slots are 16 bytes)
  __shared__ uint4 s0[TS * 64];
  __shared__ uint4 s1[TS * 64];
  __shared__ uint4 s2[NST > 2 ? TS * 64 : 1];
  __shared__ uint4 s3[NST > 3 ? TS * 64 : 1];
  __shared__ uint4 s4[NST > 4 ? TS * 64 : 1];
  __shared__ uint4 s5[NST > 5 ? TS * 64 : 1];
  __shared__ uint4 s6[NST > 6 ? TS * 64 : 1];
  __shared__ uint4 s7[NST > 7 ? TS * 64 : 1];
  uint4* const ring[8] = {s0, s1, s2, s3, s4, s5, s6, s7};

  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wv / WN, wn = wv % WN;

  // XCD-aware tile order: work-group b runs on XCD b % 8; the work-groups of
  // one XCD walk M fastest within a band of N tiles.  With K slices,
  // work-group b takes slice b / tiles of tile b % tiles.
  const int ntiles = a.ntm * a.ntn;
  const int ks = blockIdx.x / ntiles;
  const int bt = blockIdx.x - ks * ntiles;
  int tm, tn;
  tile_of(bt, a.ntm, a.ntn, tm, tn, a.xa);
  const int mg0 = tm * MT, ng0 = tn * NT;

  const uint4* A4 = reinterpret_cast<const uint4*>(a.At) + lane;
  const uint4* B4 = reinterpret_cast<const uint4*>(a.Bt) + lane;
  const uint4* Z4 = reinterpret_cast<const uint4*>(a.zero_tile) + lane;
  const int kb0 = (ks * a.KB) / a.S;                  // this work-group's k-blocks [kb0, kb0 + KB)
  const int KB = ((ks + 1) * a.KB) / a.S - kb0;
  const int nst = cdiv(KB, KT);

  // Copy source of each tile this wave copies, fixed except for the K offset:
  // rows/columns past the matrix edge re-read a valid tile (their
  // accumulators are never stored); k-blocks past K read the zero tile.
  const uint4* qsrc[PW];
  size_t qstride[PW];          // uint4 between consecutive stages
  uint32_t qlds[PW];           // byte offset of the tile inside a stage buffer
  int qk[PW];                  // k-block offset of the tile inside a stage
#pragma unroll
  for (int p = 0; p < PW; p++) {
    const int q = wv + NW * p;
    qk[p] = q % KT;
    qlds[p] = (uint32_t)q * 1024u;
    if (q < TA) {
      const int mg = min(mg0 + q / KT, a.MG - 1);
      qsrc[p] = A4 + ((size_t)(kb0 + qk[p]) * a.MG + mg) * 64;
      qstride[p] = (size_t)KT * a.MG * 64;
    } else {
      const int ng = min(ng0 + (q - TA) / KT, a.NG - 1);
      qsrc[p] = B4 + ((size_t)(kb0 + qk[p]) * a.NG + ng) * 64;
      qstride[p] = (size_t)KT * a.NG * 64;
    }
  }
  // copy p (of PW) of stage st into ring buffer buf; stages past the end of K
  // copy the zero tile, so every step issues exactly PW copies and the
  // explicit wait counts stay exact
  auto copy = [&](int st, uint32_t base, int p) {
    const uint4* g = (st * KT + qk[p] < KB) ? qsrc[p] + (size_t)st * qstride[p] : Z4;
    dma_tile(g, base + qlds[p]);
  };
  auto issue = [&](int st, uint4* buf) {
    const uint32_t base = lds_addr(buf);
#pragma unroll
    for (int p = 0; p < PW; p++) copy(st, base, p);
  };

  // Accumulator tile (i, j) is computed transposed (B fragment as the MFMA's
  // first operand): lane l holds Y[m][n .. n+3] with m = 16 mg + (l & 15) and
  // n = 16 ng + 4 (l >> 4), so the epilogue stores 16 contiguous bytes per lane.
  // Its operands are loaded first: they are older than every tile copy, so
  // the first copy wait below also covers them.
  const int mrow = lane & 15;
  const int ncol = (lane >> 4) * 4;
  float4 e_ws[FN], e_b[FN];
  float e_xs[FM];
#pragma unroll
  for (int j = 0; j < FN; j++) {
    const int n = (ng0 + wn * FN + j) * 16 + ncol;
    float w4[4], b4[4];
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int nn = min(n + r, a.N - 1);
      w4[r] = a.ws[nn];
      b4[r] = a.bias ? a.bias[nn] : 0.0f;
    }
    e_ws[j] = make_float4(w4[0], w4[1], w4[2], w4[3]);
    e_b[j] = make_float4(b4[0], b4[1], b4[2], b4[3]);
  }
#pragma unroll
  for (int i = 0; i < FM; i++) {
    const int m = min((mg0 + wm * FM + i) * 16 + mrow, a.M - 1);
    e_xs[i] = a.out == OUT_I32 ? 0.0f : a.xs[m];
  }

  v4i acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; i++)
#pragma unroll
    for (int j = 0; j < FN; j++) acc[i][j] = v4i{0, 0, 0, 0};

  // Fragments of a stage are read one step ahead of their MFMAs (two
  // register sets), so LDS latency hides behind the previous stage's MFMAs.
  uint4 fa[2][FM], fb[2][FN];
  auto read_frags = [&](const uint4* buf, int c) {
#pragma unroll
    for (int i = 0; i < FM; i++) fa[c][i] = buf[(wm * FM + i) * 64 + lane];
#pragma unroll
    for (int j = 0; j < FN; j++) fb[c][j] = buf[(TA + wn * FN + j) * 64 + lane];
  };


  // Step s: stage s's fragments are in registers (set s & 1).
  //   wait until this wave's copies of stage s+1 landed (later stages may
  //   still be in flight), and until its reads of stage s completed;
  //   barrier: stage s+1 is visible, every wave is done reading stage s;
  //   MFMAs of stage s, with the reads of stage s+1's fragments and the
  //   copies of stage s+NST (into stage s's buffer) interleaved one after
  //   each MFMA, so LDS, copy and matrix pipes work at the same time.
  auto step = [&](int st, uint4* cur, const uint4* nxt, int c) {
    wait_vm<PW * (NST - 2)>();
    wait_lgkm0();
    stage_barrier();
    const uint32_t cbase = lds_addr(cur);
    constexpr int NMEM = FM + FN + PW;
    auto mem_op = [&](int q) {
      if (q < FM) fa[c ^ 1][q] = nxt[(wm * FM + q) * 64 + lane];
      else if (q < FM + FN) fb[c ^ 1][q - FM] = nxt[(TA + wn * FN + q - FM) * 64 + lane];
      else copy(st + NST, cbase, q - FM - FN);
    };
    // (steps past the last stage multiply fragments of zero-tile stages and
    // add nothing)
#pragma unroll
    for (int m = 0; m < FM * FN; m++) {
      {
        const int i = m / FN, j = m % FN;
        acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(v4i, fb[c][j]),
                                                          __builtin_bit_cast(v4i, fa[c][i]), acc[i][j], 0, 0, 0);
      }
      // keep the source order: one MFMA, then one memory operation
      __builtin_amdgcn_sched_barrier(0);
      if (m < NMEM) mem_op(m);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int q = FM * FN; q < NMEM; q++) mem_op(q);
    __builtin_amdgcn_sched_barrier(0);
  };

  // prologue: stages 0 .. NST-1 in flight, stage 0's fragments read
#pragma unroll
  for (int b = 0; b < NST; b++) issue(b, ring[b]);
  wait_vm<PW * (NST - 1)>();
  stage_barrier();
  read_frags(ring[0], 0);
  // ring unrolled NST times (NST even, so the fragment set of every step is
  // a compile-time constant too)
  for (int st = 0; st < nst; st += NST) {
#pragma unroll
    for (int b = 0; b < NST; b++) step(st + b, ring[b], ring[(b + 1) % NST], b & 1);
  }

  wait_vm<0>();   // no copy may still be landing in LDS when the work-group exits

  if (a.S > 1 && !merge_slices<NW, FM, FN>(a, acc, wv, lane, bt, ks, reinterpret_cast<int*>(s0))) return;

  // epilogue: y = fl(fl(fl(acc) * ws[n]) * xs[m]) (+ bias[n]); 16-byte
  // streaming stores when the 4 columns are inside N and the row is 16-byte
  // aligned (the output passes the caches: 25 MB of fp32 at M = 1024,
  // N = 6144, whose write-back from L2 otherwise trails the last MFMA;
  // 23.5 -> 22.5 us per launch)
  const bool vec_ok = ((a.ldy & 3) == 0) && ((((uintptr_t)a.Y) & 15) == 0);
#pragma unroll
  for (int i = 0; i < FM; i++) {
    const int m = (mg0 + wm * FM + i) * 16 + mrow;
    if (m >= a.M) continue;
#pragma unroll
    for (int j = 0; j < FN; j++) {
      const int n = (ng0 + wn * FN + j) * 16 + ncol;
      if (n >= a.N) continue;
      const v4i c = acc[i][j];
      if (a.out == OUT_I32) {
        int32_t* yp = reinterpret_cast<int32_t*>(a.Y) + (size_t)m * a.ldy + n;
        if (vec_ok && n + 4 <= a.N) {
          st_stream(yp, make_int4(c[0], c[1], c[2], c[3]));
        } else {
          for (int r = 0; r < 4 && n + r < a.N; r++) yp[r] = c[r];
        }
        continue;
      }
      const float ws4[4] = {e_ws[j].x, e_ws[j].y, e_ws[j].z, e_ws[j].w};
      const float b4[4] = {e_b[j].x, e_b[j].y, e_b[j].z, e_b[j].w};
      float y[4];
#pragma unroll
      for (int r = 0; r < 4; r++) {
        y[r] = __fmul_rn(__fmul_rn((float)c[r], ws4[r]), e_xs[i]);
        if (a.bias) y[r] = __fadd_rn(y[r], b4[r]);
      }
      float* yp = reinterpret_cast<float*>(a.Y) + (size_t)m * a.ldy + n;
      if (vec_ok && n + 4 <= a.N) {
        st_stream(yp, make_float4(y[0], y[1], y[2], y[3]));
      } else {
        for (int r = 0; r < 4 && n + r < a.N; r++) yp[r] = y[r];
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Quadrant kernel: tiles of 16 WM FM x 32 FN outputs, WM x 2 waves, each holding
// a (16 FM) x (16 FN) block in its accumulators.  What bounds small tiles is the
// movement of operands: per 64-wide K stage a wave reads FM + FN fragments (1 KiB
// each) for FM FN MFMAs of 16 cycles, and a 256 x 256 tile pulls 32 B/clk per CU
// from L2 where 64 x 128 tiles need 96.  Two waves per SIMD keep the matrix pipe
// fed through each other's reads, copies and barriers: 8 waves on 256 x 256 tiles
// (4 waves of twice the block, in 512 registers: 116 -> 109 us at 1200 tokens of planes
// over N = 12288, K = 2048), two work-groups per CU on 128-row ones.  Few tokens of
// planes leave CUs without a 128-row tile: 64 x 128 ones, of 2 waves, are two and more
// work-groups where those are one (32 tokens, weights from HBM: N = 12288, K = 2048
// 12.8 -> 10.7 us, N = 2048, K = 6144 in 4 slices 15.6 -> 13.4).  256 x 192
// tiles keep 4 waves (8 waves: 54 -> 57 us at N = 2048, K = 6144).  Against the
// kernels before it (64 x 128 tiles with weights straight to registers): 2048
// tokens of planes over N = 12288, K = 2048 (split included) 313 -> 173 us (2.4
// POP/s), 1200 x 12288 x 2048 codes (128 x 128 LDS-staged tiles) 59 -> 45 us.  A
// stage of 256 x 256 takes 0.43 us at the MFMA rate, 0.58 on 152 CUs, 0.67 on all
// (the clock gives way).
//
// Stage s lives in ring slot s % NST.  Step s waits until stage s + 1 has
// landed, one barrier makes it visible and frees slot s % NST; the MFMAs of
// stage s run with the fragment reads of stage s + 1 and the copies of stage
// s + NST spread between them, one every MPO MFMAs.  Sources are uniform 64-bit
// bases plus one per-lane offset; stages past K re-read the last k-block
// (branch-free, so the wait counts are exact), and nothing reads what they bring in.
//
// QUAD_PLANES: grouped planes (GemmLaunch::planes_grouped): row group 4T + p holds
// plane p of tokens 16T .. 16T + 15, so the four sums of one output are the same
// lane's accumulators 4T .. 4T + 3 and fold without any exchange of lanes
// (with rows 4t + p the sums of an output lie in four lanes: 12 cross-lane moves per
// accumulator, a third of a 64 x 128 kernel's time at K = 2048).
// Accumulators and fragments are left to the register allocator.  Tiles of 8 row
// groups a wave (512 registers) need MFMAs with accumulators in the vector
// registers (a compiler option of this file, see the Makefile): it then keeps
// the fragments, which LDS reads can write there, in the accumulation registers,
// about ten moves per 96 MFMAs, where with accumulators in those it made 320.
enum { QUAD_F32, QUAD_PLANES, QUAD_I32 };   // outputs: scaled codes, folded planes, the sums
template <int WM, int FM, int FN, int NST, int MODE>
__global__ __launch_bounds__(128 * WM, FM == 8 || WM == 1 ? 1 : 2) void gemm_i8_quad_kernel(GemmI8Args a) {
  constexpr int NW = 2 * WM;                              // waves: WM x 2
  constexpr int MT = WM * FM, NT = 2 * FN, TS = MT + NT;  // row groups, column groups, tiles per stage
  constexpr int PA = MT / NW, PW = (TS + NW - 1) / NW;    // copies per wave per stage (PA of them activations)
  constexpr int NMEM = FM + FN + PW;                      // memory operations per wave per stage
  constexpr int MPO = FM * FN >= 2 * NMEM ? 2 : 1;        // MFMAs per memory operation
  static_assert(MT % NW == 0, "activation copies must divide over the waves");
  static_assert(MODE != QUAD_PLANES || FM % 4 == 0, "a wave holds whole plane groups");
  static_assert(NST >= 3 && NST * TS <= 160 && PW * (NST - 1) < 64, "LDS size, vmcnt range");
  constexpr uint32_t SB = TS * 1024;                      // bytes per stage
  __shared__ uint4 sS[NST * TS * 64];

  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wv >> 1, wn = wv & 1;
  // with K slices, work-group b takes slice b / tiles of tile b % tiles
  constexpr bool SLICES = MODE == QUAD_PLANES && FM * FN <= 16;
  const int ks = SLICES ? blockIdx.x / (a.ntm * a.ntn) : 0;
  const int bt = blockIdx.x - ks * a.ntm * a.ntn;
  int tm, tn;
  tile_patch(bt, a.ntm, a.ntn, MT == 16 ? 4 : 8, tm, tn);
  const int mg0 = tm * MT, ng0 = tn * NT;
  const int kb0 = SLICES ? (ks * a.KB) / a.S : 0;         // this work-group's k-blocks [kb0, kb0 + KB)
  const int KB = SLICES ? ((ks + 1) * a.KB) / a.S - kb0 : a.KB;
  const size_t astep = (size_t)a.MG * 1024, bstep = (size_t)a.NG * 1024;

  // copy p of a stage: tile wv + NW p of its A then B tiles (where NW does not
  // divide them the last waves have one copy less); rows / columns past the
  // matrix edge re-read a valid tile (never stored)
  const uint8_t* src[PW];
#pragma unroll
  for (int p = 0; p < PW; p++)
    src[p] = p < PA ? a.At + kb0 * astep + (size_t)min(mg0 + wv + NW * p, a.MG - 1) * 1024
                    : a.Bt + kb0 * bstep + (size_t)min(ng0 + wv + NW * (p - PA), a.NG - 1) * 1024;
  constexpr bool EVEN = TS % NW == 0;
  const bool last = EVEN || wv < TS % NW;                 // this wave has copy PW - 1
  const uint32_t lane16 = lane * 16;
  const uint32_t sbase = lds_addr(sS);
  auto copy = [&](size_t oa, size_t ob, uint32_t slot, int p) {
    if (EVEN || p < PW - 1 || last)
      dma_tile_s(lane16, src[p] + (p < PA ? oa : ob), sbase + slot + (uint32_t)(wv + NW * p) * 1024u);
  };
  auto wait_stages = [&](auto n) {                        // all but the latest n stages' copies landed
    if (EVEN || last) wait_vm<PW * n()>();
    else wait_vm<(PW - 1) * n()>();
  };

  v4i acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; i++)
#pragma unroll
    for (int j = 0; j < FN; j++) acc[i][j] = v4i{0, 0, 0, 0};

  uint4 fa[2][FM], fb[2][FN];
  const uint4* ra = sS + wm * FM * 64 + lane;             // this lane's A and B fragments in slot 0
  const uint4* rb = sS + (MT + wn * FN) * 64 + lane;

  // prologue: stages 0 .. NST-1 in flight, stage 0's fragments read
#pragma unroll
  for (int b = 0; b < NST; b++) {
    const size_t sc = min(b, KB - 1);
#pragma unroll
    for (int p = 0; p < PW; p++) copy(sc * astep, sc * bstep, b * SB, p);
  }
  wait_stages([]() constexpr { return NST - 1; });
  stage_barrier();
#pragma unroll
  for (int i = 0; i < FM; i++) fa[0][i] = ra[i * 64];
#pragma unroll
  for (int j = 0; j < FN; j++) fb[0][j] = rb[j * 64];

  uint32_t slot = 0;                                      // slot of stage s (bytes)
  auto step = [&](int st, int c) {
    wait_stages([]() constexpr { return NST - 2; });      // stage s + 1 landed (this wave's part)
    wait_lgkm0();                                         // this wave's reads of stage s are done
    stage_barrier();                                      // stage s + 1 visible; slot of stage s free
    const uint32_t nxt = slot + SB == NST * SB ? 0u : slot + SB;
    const uint4* na = ra + nxt / 16;
    const uint4* nb = rb + nxt / 16;
    const size_t sc = min(st + NST, KB - 1);
    const size_t oa = sc * astep, ob = sc * bstep;
    auto mem_op = [&](int q) {
      if (q < FN) fb[c ^ 1][q] = nb[q * 64];
      else if (q < FN + FM) fa[c ^ 1][q - FN] = na[(q - FN) * 64];
      else copy(oa, ob, slot, q - FN - FM);
    };
#pragma unroll
    for (int m = 0; m < FM * FN; m++) {
      const int i = m / FN, j = m % FN;
      acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(v4i, fb[c][j]),
                                                        __builtin_bit_cast(v4i, fa[c][i]), acc[i][j], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      if (m % MPO == 0 && m / MPO < NMEM) mem_op(m / MPO);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int q = (FM * FN + MPO - 1) / MPO; q < NMEM; q++) mem_op(q);
    __builtin_amdgcn_sched_barrier(0);
    slot = nxt;
  };
  // two steps a round, so that the fragment set is a compile-time constant
  int st = 0;
  for (; st + 2 <= KB; st += 2) {
    step(st, 0);
    step(st + 1, 1);
  }
  if (st < KB) step(st, 0);
  wait_vm<0>();   // no copy may still be landing in LDS when the work-group exits
  if constexpr (SLICES) {
    if (a.S > 1 && !merge_slices<NW, FM, FN>(a, acc, wv, lane, bt, ks, reinterpret_cast<int*>(sS))) return;
  }

  // Epilogue.  Every operand is loaded before the first store: memory
  // operations retire in order, so a load behind stores waits for their
  // acknowledgements (bias and scales loaded where they are used cost 25 us at
  // 64 accumulators).  No bias is -0, which added changes nothing.
  const int mrow = lane & 15, ncol = (lane >> 4) * 4;
  const int c0 = ng0 + wn * FN;                           // the wave's first column group
  float4 e_ws[FN], e_b[FN];
#pragma unroll
  for (int j = 0; j < FN; j++) {
    const int n = (c0 + j) * 16 + ncol;
    e_ws[j] = *reinterpret_cast<const float4*>(a.ws + min(c0 + j, a.NG - 1) * 16 + ncol);   // padded to 16 NG
    e_b[j] = make_float4(-0.0f, -0.0f, -0.0f, -0.0f);
    if (a.bias)
      e_b[j] = make_float4(a.bias[min(n, a.N - 1)], a.bias[min(n + 1, a.N - 1)], a.bias[min(n + 2, a.N - 1)],
                           a.bias[min(n + 3, a.N - 1)]);
  }
  // the lane's row of accumulator row group i: a token per 4 groups of planes,
  // or a token; its exponent or scale
  constexpr int RI = MODE == QUAD_PLANES ? 4 : 1;
  const int rows = MODE == QUAD_PLANES ? a.M >> 2 : a.M;
  const int r0 = (mg0 + wm * FM) * (16 / RI) + mrow;
  int e_xe[FM / RI];
  float e_xs[FM / RI];
#pragma unroll
  for (int i = 0; i < FM / RI; i++) {
    const int row = min(r0 + 16 * i, rows - 1);
    e_xe[i] = MODE == QUAD_PLANES ? a.xe[row] : 0;
    e_xs[i] = MODE == QUAD_F32 ? a.xs[row] : 0.0f;
  }
  auto value = [&](int i, int j) {                        // the 4 outputs of row i, column group j
    const float w[4] = {e_ws[j].x, e_ws[j].y, e_ws[j].z, e_ws[j].w};
    const float b[4] = {e_b[j].x, e_b[j].y, e_b[j].z, e_b[j].w};
    v4f y;
#pragma unroll
    for (int r = 0; r < 4; r++) {
      if constexpr (MODE == QUAD_I32) {
        y[r] = __int_as_float(acc[i][j][r]);
      } else {
        if constexpr (MODE == QUAD_PLANES)
          y[r] = planes_scale(planes_sum(acc[RI * i][j][r], acc[RI * i + 1][j][r], acc[RI * i + 2][j][r],
                                         acc[RI * i + 3][j][r]), w[r], e_xe[i]);
        else
          y[r] = __fmul_rn(__fmul_rn((float)acc[i][j][r], w[r]), e_xs[i]);
        y[r] = __fadd_rn(y[r], b[r]);
      }
    }
    return y;
  };
  float* Y = reinterpret_cast<float*>(a.Y);               // int32 bits with QUAD_I32
  if ((c0 + FN) * 16 <= a.N && (a.ldy & 3) == 0 && (((uintptr_t)a.Y) & 15) == 0) {
    // whole columns, 16-byte aligned rows: streaming stores
#pragma unroll
    for (int i = 0; i < FM / RI; i++) {
      const int row = r0 + 16 * i;
      if (row >= rows) continue;
#pragma unroll
      for (int j = 0; j < FN; j++)
        __builtin_nontemporal_store(value(i, j), reinterpret_cast<v4f*>(Y + (size_t)row * a.ldy + (c0 + j) * 16 + ncol));
    }
  } else {
#pragma unroll
    for (int i = 0; i < FM / RI; i++) {
      const int row = r0 + 16 * i;
      if (row >= rows) continue;
#pragma unroll
      for (int j = 0; j < FN; j++) {
        const v4f y = value(i, j);
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const int n = (c0 + j) * 16 + ncol + r;
          if (n < a.N) Y[(size_t)row * a.ldy + n] = y[r];
        }
      }
    }
  }
  if constexpr (MODE == QUAD_PLANES) {
    // tokens flagged kXeNonFinite: the same lane stores their outputs again
    // with the reference's fp32 value
    bool bad = false;
#pragma unroll
    for (int i = 0; i < FM / RI; i++) bad |= e_xe[i] == kXeNonFinite;
    if (bad && a.xraw) {
#pragma unroll 1
      for (int i = 0; i < FM / RI; i++) {
        const int t = r0 + 16 * i;
        if (t >= rows || a.xe[t] != kXeNonFinite) continue;
#pragma unroll 1
        for (int q = 0; q < 4 * FN; q++) {
          const int n = (c0 + (q >> 2)) * 16 + ncol + (q & 3);
          if (n >= a.N) continue;
          float y = nonfinite_dot(a.xraw, 0, (size_t)t * a.ldxr, 0, a.K, a.Bt, a.NG, n);
          if (a.bias) y = __fadd_rn(y, a.bias[n]);
          Y[(size_t)t * a.ldy + n] = y;
        }
      }
    }
  }
}

// ---------------------------------------------------------------------------
// planning and launch
// ---------------------------------------------------------------------------
// cfg 1: LDS-staged kernel, 64 x 128 tiles (8 stage buffers), of codes only
// cfg 3..7: quadrant kernel, 256 x 256, 256 x 192, 128 x 192, 128 x 128, 64 x 128 tiles
static void i8_cfg(int cfg, int& mt, int& nt) {
  static const int dims[8][2] = {{0, 0}, {4, 8}, {0, 0}, {16, 16}, {16, 12}, {8, 12}, {8, 8}, {4, 8}};
  mt = dims[cfg][0];
  nt = dims[cfg][1];
}

// tuning overrides; atomic, since a setter may run while other threads plan launches
static std::atomic<int> g_i8_force_cfg{-1};
static std::atomic<int> g_i8_force_split{0};
void gemm_i8_set_cfg(int cfg) { g_i8_force_cfg.store(cfg, std::memory_order_relaxed); }
void gemm_i8_set_split(int s) { g_i8_force_split.store(s > 0 ? s : 0, std::memory_order_relaxed); }

// the configuration that runs where `cfg` (0..7) is forced: planes have quadrant tiles
// other than 128 x 192, codes the LDS-staged 64 x 128 ones and quadrant tiles of 128 rows
static int i8_resolve(int cfg, bool planes) {
  static const int of_planes[8] = {6, 6, 6, 3, 4, 6, 6, 7}, of_codes[8] = {5, 1, 6, 5, 5, 5, 6, 6};
  return planes ? of_planes[cfg] : of_codes[cfg];
}

// Plan: the configuration and K slices of least estimated time.  The constants are
// fitted to launches whose weights come from HBM (more copies of them than the
// caches hold, as in a model of many layers) and, at lower weight, to repeated ones,
// of every configuration and 1..8 slices: 16 x 22 shapes of 17..2048 tokens of codes
// and 16 x 27 of 5..2048 tokens of planes, N = 1024 .. 12288, K = 1000..6144.  The
// kernel chosen (the small-M kernel among them) is on average 0.5 % (codes) and 0.4 %
// (planes) slower than the best of its shape with weights from HBM (1.0 % with limits
// fitted to repeated weights alone), 0.8 % and 0.4 % with repeated ones; over 99 shapes
// outside that range (N = 256 .. 151936, K = 512 .. 6144) 1.4 % and 1.1 %.
//   Codes over 256 x 192 or 256 x 256 tiles were the best at none: their fp32 outputs
// (64 KiB per 128 x 128) drain under the next work-group's loop only where two share a
// CU.  K slices cost a merge of three dependent memory round trips, about 3 us, so they
// pay only where the tiles leave most CUs idle and K is long; more than 4 were at most
// 3 % faster than 4 (64 x 5000 x 5000 codes 21.6 us on the small-M kernel, 15.5 with 4
// slices; 32 tokens of planes, 2048 x 6144: 22.2 us whole, 13.4 with 4).
struct I8Plan {
  int cfg, split;
  float us;
};
static I8Plan i8_best(bool planes, int M, int N, int K, bool whole = false) {
  const int MG = planes ? planes_groups(M / 4, true) : cdiv(M, 16), NG = cdiv(N, 16), KB = cdiv(K, 64);
  I8Plan best{planes ? 6 : 1, 1, 3.0e38f};
  auto tiles = [&](int c) {
    int mt, nt;
    i8_cfg(c, mt, nt);
    return cdiv(MG, mt) * cdiv(NG, nt);
  };
  auto offer = [&](int c, int s, float us) {
    if (us < best.us) best = I8Plan{c, s, us};
  };
  auto slices = [&](int c) { return tiles(c) <= 128 && !whole ? std::min(4, KB) : 1; };
  // one work-group per CU: rounds of 256
  auto rounds = [&](int c, float fixed, float kb, float fill) {
    offer(c, 1, cdiv(tiles(c), 256) * (fixed + kb * KB) + fill * tiles(c) / 256.0f);
  };
  // two work-groups share a CU: rounds of 512, a last one of up to 256 one per CU;
  // K slices and their merge
  auto paired = [&](int c, int s, float fixed, float fill, float full, float full_kb, float alone, float alone_kb,
                    float merge = 0.0f, float part = 0.0f) {
    const int t = tiles(c) * s, n = t / 512, rem = t % 512;
    const float kb = (float)KB / s, round = full + full_kb * kb;
    offer(c, s, fixed + fill * std::min(t, 256) / 256.0f + n * round +
                    (rem == 0 ? 0.0f : (rem <= 256 ? alone + alone_kb * kb : round)) + (s > 1 ? merge + part * t : 0.0f));
  };
  if (planes) {
    rounds(3, 1.6f, 0.612f, 8.04f);
    rounds(4, 5.56f, 0.463f, 2.66f);
    for (int s = 1; s <= slices(6); s++)
      paired(6, s, 0.159f, 1.23f, 4.11f, 0.425f, 3.41f, 0.205f, 3.76f, 0.0192f);
    for (int s = 1; s <= slices(7); s++)
      paired(7, s, 0.323f, 0.481f, 3.68f, 0.26f, 3.31f, 0.176f, 3.15f, 0.00935f);
  } else {
    // 64 x 128 tiles: as one round
    for (int s = 1; s <= slices(1); s++) {
      const int t = tiles(1) * s;
      if (t <= 256) offer(1, s, 5.71f + 0.634f * t / 256.0f + 0.138f * KB / s + (s > 1 ? 3.11f + 0.0109f * t : 0.0f));
    }
    paired(5, 1, 0.0553f, 2.57f, 21.4f, 0.335f, 5.91f, 0.273f);
    paired(6, 1, 0.222f, 0.103f, 11.8f, 0.361f, 4.99f, 0.207f);
  }
  return best;
}
// estimated us of the tiled kernels' plan, for code or plane rows (OUT_F32_X4)
float gemm_i8_us(int out, int M, int N, int K) { return i8_best(out == OUT_F32_X4, M, N, K).us; }

static void gemm_i8_plan(const GemmLaunch& L, int& cfg, int& split) {
  const bool planes = L.out == OUT_F32_X4;
  const int KB = cdiv(L.K, 64);
  const I8Plan best = i8_best(planes, L.M, L.N, L.K, L.whole);
  cfg = best.cfg;
  split = best.split;
  const int fc = g_i8_force_cfg.load(std::memory_order_relaxed);
  if (fc >= 0) {
    cfg = i8_resolve(fc, planes);
    split = 1;
  }
  const int fs = g_i8_force_split.load(std::memory_order_relaxed);
  if (fs > 0) {
    split = std::min(fs, KB);
    if (split > 1 && cfg >= 3 && !(planes && cfg == 7)) cfg = planes ? 6 : 1;   // the kernels that take slices
  }
}

void gemm_i8_resolve(GemmLaunch& L, size_t* part_bytes, size_t* counters) {
  int mt, nt;
  gemm_i8_plan(L, L.cfg, L.split);
  i8_cfg(L.cfg, mt, nt);
  const int MG = L.out == OUT_F32_X4 ? planes_groups(L.M / 4, true) : cdiv(L.M, 16);
  const size_t tiles = (size_t)cdiv(MG, mt) * cdiv(cdiv(L.N, 16), nt);
  *part_bytes = L.split > 1 ? tiles * L.split * (size_t)(256 * mt * nt) * sizeof(int32_t) : 0;
  *counters = L.split > 1 ? tiles : 0;
}

// planes on 256 x 256, 256 x 192, 128 x 128 and 64 x 128 tiles, codes on 128 x 192
// and 128 x 128 (i8_resolve)
template <int WM, int FM, int FN, int NST>
static void launch_quad(const GemmI8Args& a, int blocks, hipStream_t st) {
  const dim3 grid(blocks), block(128 * WM);
  if constexpr (FM == 8 || FN != 6) {
    if (a.out == OUT_F32_X4) {
      hipLaunchKernelGGL((gemm_i8_quad_kernel<WM, FM, FN, NST, QUAD_PLANES>), grid, block, 0, st, a);
      return;
    }
  }
  if constexpr (WM == 2 && FM == 4) {
    if (a.out == OUT_I32) hipLaunchKernelGGL((gemm_i8_quad_kernel<WM, FM, FN, NST, QUAD_I32>), grid, block, 0, st, a);
    else hipLaunchKernelGGL((gemm_i8_quad_kernel<WM, FM, FN, NST, QUAD_F32>), grid, block, 0, st, a);
  }
}

hipError_t launch_gemm_i8(const GemmLaunch& L, hipStream_t st) {
  GemmI8Args a;
  a.At = static_cast<const uint8_t*>(L.A);
  a.Bt = L.Bt;
  a.ws = L.ws;
  a.xs = L.xs;
  a.xe = L.xe;
  a.xraw = L.xraw;
  a.ldxr = L.ldxr;
  a.bias = L.bias;
  a.Y = L.Y;
  a.ldy = L.ldy;
  a.M = L.M;
  a.N = L.N;
  a.K = L.K;
  a.KB = cdiv(L.K, 64);
  a.MG = L.planes_grouped ? planes_groups(L.M / 4, true) : cdiv(L.M, 16);
  a.NG = cdiv(L.N, 16);
  a.out = L.out;
  a.zero_tile = L.zero_tile;
  if (L.out == OUT_F32_X4 && (!L.xe || L.M % 4 != 0)) return hipErrorInvalidValue;
  if (L.out != OUT_I32 && L.out != OUT_F32_X4 && !L.xs) return hipErrorInvalidValue;
  if (!L.zero_tile) return hipErrorInvalidValue;
  // planes come grouped (gemm_planes_grouped)
  if (L.out == OUT_F32_X4 && !L.planes_grouped) return hipErrorInvalidValue;
  const int sp = L.split;
  int mt, nt;
  i8_cfg(L.cfg, mt, nt);
  a.ntm = cdiv(a.MG, mt);
  a.ntn = cdiv(a.NG, nt);
  a.S = sp;
  // XCD blocks of half the tile rows x a quarter of the columns where they
  // fill fewer L2 lines (rows of A plus rows of weights per XCD)
  a.xa = 1;
  if ((long long)a.ntm * a.ntn <= 256 && a.ntm % 2 == 0 && a.ntn % 4 == 0 &&
      a.ntm * mt / 2 + a.ntn * nt / 4 < a.ntm * mt + a.ntn * nt / 8)
    a.xa = 2;
  a.part = static_cast<int32_t*>(L.part);
  a.cnt = L.cnt;
  if (sp > 1 && (!a.part || !a.cnt)) return hipErrorInvalidValue;
  const long long blocks_ll = (long long)a.ntm * a.ntn * sp;
  if (blocks_ll > 0x7fffffffLL) return hipErrorInvalidValue;
  const int blocks = (int)blocks_ll;
  switch (L.cfg) {
    case 1: hipLaunchKernelGGL((gemm_i8_lds_kernel<4, 8, 1, 8, 2, 2>), dim3(blocks), dim3(256), 0, st, a); break;
    case 3: launch_quad<4, 4, 8, 5>(a, blocks, st); break;
    case 4: launch_quad<2, 8, 6, 5>(a, blocks, st); break;
    case 5: launch_quad<2, 4, 6, 4>(a, blocks, st); break;
    case 7: launch_quad<1, 4, 4, 5>(a, blocks, st); break;
    default: launch_quad<2, 4, 4, 5>(a, blocks, st); break;
  }
  return hipGetLastError();
}

}  // namespace tl

extern "C" void tlk_gemm_i8_set_cfg(int cfg) { tl::gemm_i8_set_cfg(cfg); }
extern "C" void tlk_gemm_i8_set_split(int s) { tl::gemm_i8_set_split(s); }
