// gemm_b16.hip -- prefill GEMMs with 16-bit MFMAs over int8 weight tiles:
//   A_BF16  W8A16 (kernel/w8a16_kernel.c:203-216): bf16 X x int8 W (exact in
//           bf16) on v_mfma_f32_*_bf16, fp32 accumulation, fp32 scale
//           after the sum, fp32 / bf16 (RNE) / fp16 output.
//   A_F16   the same with fp16 X on v_mfma_f32_*_f16.
//
// Two kernels: the wave-grid one for every X under 4 GiB, the LDS-staged one
// (64-bit addresses) past that.  Both are a ring of LDS stage buffers filled by
// direct global -> LDS copies (one 16-byte piece per lane per copy), one
// barrier per 64-wide K stage, transposed accumulators (weights as the MFMA's
// first operand) so each lane holds 4 consecutive output columns.
//
// X (row-major in memory) is copied a whole 128-byte row segment per 8 lanes
// into a swizzled row-major LDS tile (xtile_* below: 2 copies per 16-row group
// and K block), and a wave reads each MFMA operand with one conflict-free
// ds_read_b128.  (Copies in MFMA operand order, lane l reading 16 bytes of row
// l & 15, spread every copy over 16 half-used lines: about 10 B/clk per CU
// against the int8 GEMM's 22-38.)  Weight tiles stay int8 and are widened to
// bf16/fp16 in registers after the read.  Lanes whose k is past K copy 16 bytes
// of zeros.
#include <algorithm>
#include <atomic>

#include "gemm_common.h"
#include "tl_kernels.h"

typedef _Float16 v8h_t __attribute__((ext_vector_type(8)));

namespace tl {

struct GemmB16Args {
  const void* X;         // row-major [M][lda], element type per AMODE
  int lda;
  const uint8_t* Bt;     // weight tiles [KB][NG]
  const float* ws;       // [N]
  const float* bias;     // [N] or null
  void* Y;
  int ldy;
  int M, N, K, KB, MG, NG;
  int ntm, ntn;
  int out;
  const uint8_t* zero_tile;
  int S;                 // K slices per tile (work-groups per tile)
  float* part;           // S > 1: fp32 partial tiles [tiles][S][MT*16 x NT*16]
  uint32_t* cnt;         // S > 1: zeroed arrival counters [tiles]
};

__device__ inline v8bf as_bf(uint4 u) { return __builtin_bit_cast(v8bf, u); }
__device__ inline v8h_t as_h(uint4 u) { return __builtin_bit_cast(v8h_t, u); }

// int8 weight lane (16 values) -> two 8-wide 16-bit operands (exact)
template <int AMODE>
__device__ inline void widen(uint4 w, uint4& h0, uint4& h1) {
  const uint32_t d[4] = {w.x, w.y, w.z, w.w};
  uint32_t o[8];
#pragma unroll
  for (int q = 0; q < 4; q++) {
    const float f0 = (float)(int8_t)(d[q] & 0xff), f1 = (float)(int8_t)((d[q] >> 8) & 0xff);
    const float f2 = (float)(int8_t)((d[q] >> 16) & 0xff), f3 = (float)(int8_t)(d[q] >> 24);
    if constexpr (AMODE == A_F16) {
      const _Float16 h0f = (_Float16)f0, h1f = (_Float16)f1, h2f = (_Float16)f2, h3f = (_Float16)f3;
      o[2 * q] = (uint32_t)__builtin_bit_cast(uint16_t, h0f) | ((uint32_t)__builtin_bit_cast(uint16_t, h1f) << 16);
      o[2 * q + 1] = (uint32_t)__builtin_bit_cast(uint16_t, h2f) | ((uint32_t)__builtin_bit_cast(uint16_t, h3f) << 16);
    } else {
      // |w| <= 127 is exact in bf16: the high halves of the floats, paired by
      // one byte permute (bytes 2, 3 of f0 then bytes 2, 3 of f1)
      o[2 * q] = __builtin_amdgcn_perm(__float_as_uint(f1), __float_as_uint(f0), 0x07060302u);
      o[2 * q + 1] = __builtin_amdgcn_perm(__float_as_uint(f3), __float_as_uint(f2), 0x07060302u);
    }
  }
  h0 = make_uint4(o[0], o[1], o[2], o[3]);
  h1 = make_uint4(o[4], o[5], o[6], o[7]);
}


template <int AMODE>
__device__ inline v4f mfma16(uint4 w, uint4 x, v4f c) {
  if constexpr (AMODE == A_F16) return __builtin_amdgcn_mfma_f32_16x16x32_f16(as_h(w), as_h(x), c, 0, 0, 0);
  else return __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf(w), as_bf(x), c, 0, 0, 0);
}

// X tiles in LDS.  A row group's 64-wide K block of X (16 rows x 128 bytes)
// is two 1 KiB copies, rows 0-7 and 8-15.  Copy half j: lane l fetches row
// 8 j + (l >> 3), 16-byte chunk (l & 7) ^ (l >> 3) ^ j of the row (so every
// 8 lanes read one whole 128-byte line of X), and its 16 bytes land at
// 16 l.  The XOR swizzle spreads the chunks that one MFMA operand read takes
// from 16 rows (lane l: row l & 15, chunk 2 (l >> 4) + h) over distinct
// bank groups.  Both functions are per-lane constants.
__device__ __forceinline__ int xtile_row(int lane, int j) { return 8 * j + (lane >> 3); }
__device__ __forceinline__ int xtile_chunk(int lane, int j) { return (lane & 7) ^ (lane >> 3) ^ j; }
// uint4 index, within a row group's two copies, of lane's operand for K half h
// (X[row lane & 15][16 (lane >> 4) + 8 h .. + 7])
__device__ __forceinline__ int xtile_frag(int lane, int h) {
  const int rr = lane & 15, j = rr >> 3, r8 = rr & 7;
  const int kc = 2 * (lane >> 4) + h;
  return j * 64 + r8 * 8 + (kc ^ r8 ^ j);
}

// K slices (a.S > 1): merges a tile's partial sums; true in the work-group that
// holds the whole sums afterwards.  acc[i][j] is this wave's fragment in slot
// slot0 + i of the partial tile (the slots of the waves of a work-group do not
// overlap).  flag: a word of the stage ring, which no copy or read uses any more
// (an LDS word of its own would push an 80 KiB ring past two work-groups per CU).
template <int FM, int FN>
__device__ __forceinline__ bool b16_merge(const GemmB16Args& a, v4f (&acc)[FM][FN], int slot0, int bt, int ks, int* flag) {
  const int lane = threadIdx.x & 63;
  // K slices: every work-group of the tile stores its fp32 sums, waits for
  // the stores' acknowledgement and counts in; the last to arrive adds the
  // S slices in slice order (its own from registers, the same sums and
  // order whichever work-group merges), then runs the epilogue below
  constexpr int TF = 4 * FM * FN * 256;         // floats per partial tile: 4 waves x FM x FN fragments
  float* mine = a.part + ((size_t)bt * a.S + ks) * TF;
#pragma unroll
  for (int i = 0; i < FM; i++)
#pragma unroll
    for (int j = 0; j < FN; j++) st_agent4(mine + (((slot0 + i) * FN + j) * 64 + lane) * 4, acc[i][j]);
  asm volatile("" ::: "memory");
  wait_vm<0>();                               // this thread's partial stores are acknowledged
  asm volatile("" ::: "memory");
  __syncthreads();
  if (threadIdx.x == 0)
    *flag = __hip_atomic_fetch_add(a.cnt + bt, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (uint32_t)(a.S - 1);
  __syncthreads();
  if (!*flag) return false;
  // the merger's acquire: the slices are read after the counter showed
  // them all arrived (agent scope, once per tile: it invalidates this
  // CU's caches, so the plain 16-byte loads below fetch what the stores
  // wrote through).  All S slices come from memory, this work-group's own
  // too (the values it stored), one slice's loads in flight at a time and
  // added in slice order.
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
  // QB slices' loads are in flight together (indices past S re-read the
  // last slice and are not added)
  constexpr int QB = FM * FN <= 2 ? 8 : (FM * FN <= 8 ? 4 : 1);
  const float* slices = a.part + (size_t)bt * a.S * TF;
  for (int q0 = 0; q0 < a.S; q0 += QB) {
    v4f p[QB][FM][FN];
#pragma unroll
    for (int u = 0; u < QB; u++)
#pragma unroll
      for (int i = 0; i < FM; i++)
#pragma unroll
        for (int j = 0; j < FN; j++)
          p[u][i][j] = *reinterpret_cast<const v4f*>(slices + (size_t)min(q0 + u, a.S - 1) * TF +
                                                    (((slot0 + i) * FN + j) * 64 + lane) * 4);
#pragma unroll
    for (int u = 0; u < QB; u++) {
      if (q0 + u >= a.S) break;
#pragma unroll
      for (int i = 0; i < FM; i++)
#pragma unroll
        for (int j = 0; j < FN; j++)
#pragma unroll
          for (int r = 0; r < 4; r++)
            acc[i][j][r] = q0 + u == 0 ? p[u][i][j][r] : __fadd_rn(acc[i][j][r], p[u][i][j][r]);
    }
  }
  if (threadIdx.x == 0) __hip_atomic_store(a.cnt + bt, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return true;
}

// Epilogue of the LDS-staged kernel: scale, bias, conversion, stores.  acc[i][j]
// holds row group rg0 + i (lane: row lane & 15) and column group cg0 + j (lane:
// columns 4 (lane >> 4) .. + 3).
template <int FM, int FN>
__device__ __forceinline__ void b16_finish(const GemmB16Args& a, v4f (&acc)[FM][FN], int rg0, int cg0,
                                           const float (&e_ws)[FN][4], const float (&e_b)[FN][4]) {
  const int lane = threadIdx.x & 63;
  const int mrow = lane & 15;
  const int ncol = (lane >> 4) * 4;
  const bool vec_ok = ((a.ldy & 3) == 0) &&
                      ((((uintptr_t)a.Y) & (a.out == OUT_F32 ? 15 : 7)) == 0);
#pragma unroll
  for (int i = 0; i < FM; i++) {
    const int m = (rg0 + i) * 16 + mrow;
    if (m >= a.M) continue;
#pragma unroll
    for (int j = 0; j < FN; j++) {
      const int n = (cg0 + j) * 16 + ncol;
      if (n >= a.N) continue;
      float y[4];
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const float c = acc[i][j][r];
        y[r] = __fmul_rn(c, e_ws[j][r]);
        if (a.bias) y[r] = __fadd_rn(y[r], e_b[j][r]);
      }
      const size_t o = (size_t)m * a.ldy + n;
      const bool full = vec_ok && n + 4 <= a.N;
      if (a.out == OUT_F32) {
        float* yp = reinterpret_cast<float*>(a.Y) + o;
        if (full) st_stream(yp, make_float4(y[0], y[1], y[2], y[3]));   // streaming, as the int8 GEMM's
        else for (int r = 0; r < 4 && n + r < a.N; r++) yp[r] = y[r];
      } else {
        uint16_t hv[4];
#pragma unroll
        for (int r = 0; r < 4; r++) {
          if (a.out == OUT_BF16) {
            hv[r] = (uint16_t)f32_to_bf16_rne(y[r]);
          } else {
            const _Float16 h = (_Float16)y[r];
            hv[r] = __builtin_bit_cast(uint16_t, h);
          }
        }
        uint16_t* yp = reinterpret_cast<uint16_t*>(a.Y) + o;
        if (full) *reinterpret_cast<uint2*>(yp) = make_uint2(hv[0] | ((uint32_t)hv[1] << 16), hv[2] | ((uint32_t)hv[3] << 16));
        else for (int r = 0; r < 4 && n + r < a.N; r++) yp[r] = hv[r];
      }
    }
  }
}

template <int AMODE, int MT, int NT, int NST, int WM, int WN>
__global__ __launch_bounds__(64 * WM * WN) void gemm_b16_lds_kernel(GemmB16Args a) {
  constexpr int NW = WM * WN;
  constexpr int AP = 2;                                // A copies per (row group, K block)
  constexpr int ESZ = 2;                               // bytes per X element
  constexpr int EPC = 16 / ESZ;                        // X elements per copy per lane
  constexpr int TA = MT * AP, TB = NT, TS = TA + TB;
  static_assert(TS % NW == 0, "stage copies must divide evenly over the waves");
  constexpr int PW = TS / NW;
  constexpr int FM = MT / WM, FN = NT / WN;
  static_assert(MT % WM == 0 && NT % WN == 0, "wave grid must divide the tile");
  static_assert(NST >= 2 && NST <= 8 && NST % 2 == 0, "2, 4, 6 or 8 stage buffers");
  static_assert(PW * (NST - 1) < 64, "vmcnt range");

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

  // work-group b: K slice b / ntiles of tile b % ntiles; with ntiles a
  // multiple of 8 the tiles are grouped per XCD (b % 8) as ntiles / 8
  // consecutive tile indices
  const int ntiles = a.ntm * a.ntn;
  const int ks = blockIdx.x / ntiles;
  const int bt = blockIdx.x - ks * ntiles;
  int t = bt;
  if (ntiles % 8 == 0) t = (bt % 8) * (ntiles / 8) + bt / 8;
  const int tn = t / a.ntm, tm = t - (t / a.ntm) * a.ntm;
  const int mg0 = tm * MT, ng0 = tn * NT;

  const uint4* B4 = reinterpret_cast<const uint4*>(a.Bt) + lane;
  const uint4* Z4 = reinterpret_cast<const uint4*>(a.zero_tile);   // any 16 zero bytes
  const char* Xb = static_cast<const char*>(a.X);
  const int KB = a.KB;
  const int kb0 = (ks * KB) / a.S;                     // this work-group's K blocks [kb0, kb0 + nst)
  const int nst = ((ks + 1) * KB) / a.S - kb0;

  // per copy: source for stage 0 and its advance per stage
  const char* qsrc[PW];
  int qkoff[PW];                // X column of this lane's piece at stage 0 (A copies), -1 for B
  bool qrow_ok[PW];
  uint32_t qlds[PW];
#pragma unroll
  for (int p = 0; p < PW; p++) {
    const int q = wv + NW * p;
    qlds[p] = (uint32_t)q * 1024u;
    if (q < TA) {
      const int i = q / AP, j = q % AP;
      const int row = (mg0 + i) * 16 + xtile_row(lane, j);
      const int koff = EPC * xtile_chunk(lane, j);
      qrow_ok[p] = row < a.M;
      qkoff[p] = koff;
      qsrc[p] = Xb + ((size_t)min(row, a.M - 1) * a.lda + koff) * ESZ;
    } else {
      const int ng = min(ng0 + (q - TA), a.NG - 1);
      qrow_ok[p] = true;
      qkoff[p] = -1;
      qsrc[p] = reinterpret_cast<const char*>(B4 + (size_t)ng * 64);
    }
  }
  const size_t bstride = (size_t)a.NG * 1024;   // bytes between K blocks of the weights
  // Every call issues exactly PW copies, so the explicit vmcnt waits in `step`
  // count exactly: stages past the end of the work-group's K range re-read its
  // last K block into a buffer that no step reads again.  (Skipping those
  // copies would let the last NST-2 steps' waits return before their own
  // stage had landed; waiting for every copy there instead measured 7% slower
  // at M = 64..256.)
  auto issue = [&](int st, uint4* buf) {
    const int sc = kb0 + min(st, nst - 1);
    const uint32_t base = lds_addr(buf);
#pragma unroll
    for (int p = 0; p < PW; p++) {
      const uint4* g;
      if (qkoff[p] >= 0) {
        const int k = sc * 64 + qkoff[p];
        g = (qrow_ok[p] && k < a.K) ? reinterpret_cast<const uint4*>(qsrc[p] + (size_t)sc * 64 * ESZ) : Z4;
      } else {
        g = reinterpret_cast<const uint4*>(qsrc[p] + (size_t)sc * bstride);
      }
      dma_tile(g, base + qlds[p]);
    }
  };

  // prologue: stages 0 .. NST-1 in flight first
#pragma unroll
  for (int b = 0; b < NST; b++) issue(b, ring[b]);
  // epilogue operands (transposed accumulators: lane holds row m, cols
  // n..n+3), loaded behind the first copies: the stage waits below then
  // also cover them (loads complete in issue order, so the extra loads only
  // make the first waits stricter), and the loop's last wait leaves them done
  const int ncol = (lane >> 4) * 4;
  float e_ws[FN][4], e_b[FN][4];
#pragma unroll
  for (int j = 0; j < FN; j++)
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int n = min((ng0 + wn * FN + j) * 16 + ncol + r, a.N - 1);
      e_ws[j][r] = a.ws[n];
      e_b[j][r] = a.bias ? a.bias[n] : 0.0f;
    }

  v4f acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; i++)
#pragma unroll
    for (int j = 0; j < FN; j++) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};

  // A stage's fragments are read from LDS into a register set one step ahead
  // of their MFMAs (two sets, so the read latency hides behind the previous
  // stage's MFMAs): set c holds the stage's A copies of this wave's row
  // groups and its raw int8 weight tiles.
  uint4 fa[2][FM * AP], fb[2][FN];
  const int xf[AP] = {xtile_frag(lane, 0), xtile_frag(lane, 1)};
  auto read_frags = [&](const uint4* buf, int c) {
#pragma unroll
    for (int i = 0; i < FM; i++)
#pragma unroll
      for (int h = 0; h < AP; h++) fa[c][i * AP + h] = buf[(wm * FM + i) * AP * 64 + xf[h]];
#pragma unroll
    for (int j = 0; j < FN; j++) fb[c][j] = buf[(TA + wn * FN + j) * 64 + lane];
  };

  // Column by column: the MFMAs of weight column j (both K halves of every
  // row group) run interleaved with the widening of column j + 1, so the
  // VALU work of the int8 -> 16-bit conversion hides under the matrix pipe
  // (all widening first, then all MFMAs, left them back to back).
  auto compute = [&](int c) {
    uint4 wcur[2], wnxt[2];
    widen<AMODE>(fb[c][0], wcur[0], wcur[1]);
#pragma unroll
    for (int j = 0; j < FN; j++) {
      if (j + 1 < FN) widen<AMODE>(fb[c][j + 1], wnxt[0], wnxt[1]);
#pragma unroll
      for (int h = 0; h < 2; h++)
#pragma unroll
        for (int i = 0; i < FM; i++) acc[i][j] = mfma16<AMODE>(wcur[h], fa[c][i * AP + h], acc[i][j]);
      if (j + 1 < FN) {
#pragma unroll
        for (int q = 0; q < 2 * FM; q++) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);   // one MFMA
          __builtin_amdgcn_sched_group_barrier(0x002, 3, 0);   // then three VALU
        }
      }
      __builtin_amdgcn_sched_barrier(0);
      wcur[0] = wnxt[0];
      wcur[1] = wnxt[1];
    }
  };

  // Step s (register set c = s & 1 holds stage s):
  //   wait until this wave's copies of stage s+1 landed (later stages may
  //   still fly) and its reads of stage s completed; barrier: stage s+1 is
  //   visible and every wave is done reading stage s's buffer;
  //   read stage s+1's fragments, refill stage s's buffer with stage s+NST,
  //   then widen and multiply stage s from registers (steps past the last
  //   stage only keep the copy count exact).
  auto step = [&](int st, uint4* cur, const uint4* nxt, int c) {
    wait_vm<PW * (NST - 2)>();
    wait_lgkm0();
    stage_barrier();
    read_frags(nxt, c ^ 1);
    issue(st + NST, cur);
    __builtin_amdgcn_sched_barrier(0);
    if (st < nst) compute(c);
    __builtin_amdgcn_sched_barrier(0);
  };

  // stage 0 landed (and the epilogue operands), its fragments read
  wait_vm<PW * (NST - 1)>();
  stage_barrier();
  read_frags(ring[0], 0);
  // ring unrolled NST times (NST even: every step's register set is a
  // compile-time constant)
  for (int st = 0; st < nst; st += NST) {
#pragma unroll
    for (int b = 0; b < NST; b++) step(st + b, ring[b], ring[(b + 1) % NST], b & 1);
  }
  wait_vm<0>();   // no copy may still be landing in LDS when the work-group exits

  if (a.S > 1 && !b16_merge<FM, FN>(a, acc, wv * FM, bt, ks, reinterpret_cast<int*>(s0))) return;
  b16_finish<FM, FN>(a, acc, mg0 + wm * FM, ng0 + wn * FN, e_ws, e_b);
}

// One output dword of the widening: int8 elements 2p, 2p + 1 of a lane's 16
// (dword p / 2, bytes 2 (p % 2), + 1) as two 16-bit values, exact
template <int AMODE>
__device__ __forceinline__ uint32_t widen_pair(uint4 w, int p) {
  const uint32_t d = (p >> 1) == 0 ? w.x : ((p >> 1) == 1 ? w.y : ((p >> 1) == 2 ? w.z : w.w));
  const int sh = (p & 1) * 16;
  const float f0 = (float)(int8_t)((d >> sh) & 0xff), f1 = (float)(int8_t)((d >> (sh + 8)) & 0xff);
  if constexpr (AMODE == A_F16) {
    return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(f0, f1));
  } else {
    return __builtin_amdgcn_perm(__float_as_uint(f1), __float_as_uint(f0), 0x07060302u);
  }
}
__device__ __forceinline__ void set_dword(uint4& u, int c, uint32_t v) {
  if (c == 0) u.x = v;
  else if (c == 1) u.y = v;
  else if (c == 2) u.z = v;
  else u.w = v;
}

// ---------------------------------------------------------------------------
// Wave-grid kernel: WM x WN waves, each holding a (32 RM) x (32 CN) block of the tile
// in its accumulation registers (RM x CN accumulators of 32 x 32).  X (swizzled
// row-major tiles, xtile_*) and the int8 weight tiles of a 64-wide K stage pass
// through one LDS ring; a wave widens the weights it reads.
//
// What bounds it is instruction issue beside the matrix pipe: a wave issues an
// instruction of the widening every 5.8 cycles at most, two waves on a SIMD one every
// 4.7; an MFMA with 6 of them takes 41.7 cycles of a SIMD with one wave, 33.4 with two.
// A widened dword (two weights) costs
// 3 vector instructions, so a 16 x 16 tile of weights costs 24 and feeds four
// 32 x 32 x 16 MFMAs (32 cycles each) per 64 rows of X.  Hence 32 x 32 MFMAs
// (half the instructions of 16 x 16 ones), and two waves per SIMD: 8 waves on the
// large tiles, two work-groups per CU on the small ones (one, and so one wave per
// SIMD, where a launch has no more than 256 of those).  A small
// tile's waves split its columns only (WM = 1), so that each weight is widened
// once.  The outputs leave through LDS for the same reason: unrolled over the
// accumulators, scaling and storing took 17 us per 256 x 192 work-group, now 5.
// Measured against the column-split kernel before it (bf16 out): 1024 x 12288 x
// 2048 65 -> 52 us, 333 x 2048 x 6144 40 -> 23 us, 400 x 2048 x 2048 17 -> 14 us.
// Accumulators are left to the register allocator (at most 256 registers, it
// keeps them in place; with asm MFMAs pinned to the accumulation registers it
// copied operands right in front of their use, without the wait states).
//
// Stage s lives in ring slot s % NST.  Step s waits until stage s + 1 has
// landed, one barrier makes it visible and frees slot s % NST; the 8 CN MFMAs
// of stage s run with the widening of the next operand, the fragment reads of
// stage s + 1 and the copies of stage s + NST spread between them.  Stages past
// the work-group's K range re-read its last K block (branch-free, so the wait
// counts are exact), and nothing reads what they bring in.
//
// KF: K is a multiple of 64.  Otherwise the lanes whose 8 columns of X lie past K
// copy 16 bytes of zeros (the next row's values there could be Inf or NaN, which
// the weight tile's zero padding would not cancel).
typedef float v16f __attribute__((ext_vector_type(16)));
template <int AMODE>
__device__ __forceinline__ void mfma32_acc(v16f& c, uint4 w, uint4 x) {
  if constexpr (AMODE == A_F16) c = __builtin_amdgcn_mfma_f32_32x32x16_f16(as_h(w), as_h(x), c, 0, 0, 0);
  else c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf(w), as_bf(x), c, 0, 0, 0);
}
template <int AMODE, int WM, int WN, int RM, int CN, int NST, bool KF>
__global__ __launch_bounds__(64 * WM * WN, 2) void gemm_b16_wave_kernel(GemmB16Args a) {
  constexpr int NW = WM * WN;
  constexpr int MT = 2 * RM * WM, NT = 2 * CN * WN;            // row groups, column groups
  constexpr int TA = 2 * MT, TS = TA + NT;                // X copies, copies per stage (1 KiB each)
  constexpr int PA = TA / NW, PW = (TS + NW - 1) / NW;    // copies per wave per stage (PA of them X)
  constexpr int NMEM = 4 * RM + 2 * CN + PW;                 // memory operations per wave per stage
  constexpr int NM = 4 * RM * CN;                         // MFMAs per wave per stage
  constexpr int MO = (NMEM + NM - 1) / NM;                // memory operations behind an MFMA
  static_assert(TA % NW == 0, "X copies must divide over the waves");
  static_assert(NST >= 3 && NST * TS <= 160 && PW * (NST - 1) < 64, "LDS size, vmcnt range");
  constexpr uint32_t SB = TS * 1024;                      // bytes per stage
  __shared__ uint4 sS[NST * TS * 64];

  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wv / WN, wn = wv % WN;
  // with K slices, work-group b takes slice b / tiles of tile b % tiles
  constexpr bool SLICES = NW == 4;
  const int ks = SLICES ? blockIdx.x / (a.ntm * a.ntn) : 0;
  const int bt = blockIdx.x - ks * a.ntm * a.ntn;
  int tm, tn;
  tile_patch(bt, a.ntm, a.ntn, MT >= 16 ? 4 : 8, tm, tn);
  const int mg0 = tm * MT, ng0 = tn * NT;
  // this work-group's k-blocks [kb0, kb0 + KB) (divisions run on the vector unit)
  const int kb0 = SLICES ? __builtin_amdgcn_readfirstlane((ks * a.KB) / a.S) : 0;
  const int KB = SLICES ? __builtin_amdgcn_readfirstlane(((ks + 1) * a.KB) / a.S) - kb0 : a.KB;
  const size_t bstep = (size_t)a.NG * 1024;

  // Copy p of a stage is q = wv + NW p: X copies first (q < TA; rows 8 (q % 2) ..
  // + 7 of row group q / 2; q % 2 = wv % 2, so a lane's 16-byte chunk of the row
  // is the same in all of them), then weight tiles; where NW does not divide TS
  // the last waves have one copy less.  Rows / columns past the matrix edge
  // re-read a valid one (never stored).
  const char* Xb = static_cast<const char*>(a.X) + (size_t)kb0 * 128;
  const int chunk = xtile_chunk(lane, wv & 1);
  uint32_t xo[PA];
#pragma unroll
  for (int p = 0; p < PA; p++) {
    const int row = min((mg0 + (wv >> 1) + NW / 2 * p) * 16 + xtile_row(lane, wv & 1), a.M - 1);
    xo[p] = (uint32_t)row * (uint32_t)(a.lda * 2) + 16u * chunk;
  }
  const int kroom = a.K - kb0 * 64 - 8 * chunk;           // stage st's chunk lies inside K while 64 st < kroom
  const uint8_t* bs[PW - PA];
#pragma unroll
  for (int p = 0; p < PW - PA; p++)
    bs[p] = a.Bt + kb0 * bstep + (size_t)min(ng0 + wv + NW * p, a.NG - 1) * 1024;
  constexpr bool EVEN = TS % NW == 0;
  const bool last = EVEN || wv < TS % NW;                 // this wave has copy PW - 1
  const uint32_t lane16 = lane * 16;
  const uint32_t sbase = lds_addr(sS);
  auto copy = [&](int sc, uint32_t slot, int p) {
    const uint32_t dst = sbase + slot + (uint32_t)(wv + NW * p) * 1024u;
    if (p >= PA) {
      if (EVEN || p < PW - 1 || last) dma_tile_s(lane16, bs[p - PA] + (size_t)sc * bstep, dst);
    } else if (KF) {
      dma_tile_s(xo[p], Xb + (size_t)sc * 128, dst);
    } else {
      uint32_t o = xo[p];
      asm volatile("" : "+v"(o));                         // no 64-bit address is kept per copy
      const char* g = Xb + (size_t)sc * 128 + o;
      if (sc * 64 >= kroom) g = reinterpret_cast<const char*>(a.zero_tile);
      dma_tile(reinterpret_cast<const uint4*>(g), dst);
    }
  };
  auto wait_stages = [&](auto n) {                        // all but the latest n stages' copies landed
    if (EVEN || last) wait_vm<PW * n()>();
    else wait_vm<(PW - 1) * n()>();
  };

  v16f acc[RM][CN];
#pragma unroll
  for (int i = 0; i < RM; i++)
#pragma unroll
    for (int j = 0; j < CN; j++)
#pragma unroll
      for (int r = 0; r < 16; r++) acc[i][j][r] = 0.0f;

  // Operands of a 32 x 32 x 16 MFMA: lane l holds row l & 31 of its matrix and 8
  // values of K.  MFMA (u, h) of a stage takes k = 32 u + 16 (l >> 5) + 8 h + 0..7,
  // so a lane's 16 weight bytes (k = 32 u + 16 (l >> 5) + 0..15) are its operands
  // for h = 0 and 1.
  uint4 fa[2][RM][4], fb[2][CN][2], wc[2];                 // X operands, int8 weights, widened operands
  const int half = (lane >> 4) & 1;                       // which of a block's two 16-row groups
  const uint4* ra[4];
#pragma unroll
  for (int t = 0; t < 4; t++) {
    const int rr = lane & 15, j = rr >> 3, r8 = rr & 7, kc = 4 * (t >> 1) + 2 * (lane >> 5) + (t & 1);
    ra[t] = sS + (wm * 2 * RM + half) * 128 + j * 64 + r8 * 8 + (kc ^ r8 ^ j);   // xtile layout
  }
  const uint4* rb = sS + (TA + wn * 2 * CN + half) * 64 + (lane & 15) + 16 * (lane >> 5);

  // prologue: stages 0 .. NST-1 in flight, stage 0's fragments read
#pragma unroll
  for (int b = 0; b < NST; b++)
#pragma unroll
    for (int p = 0; p < PW; p++) copy(min(b, KB - 1), b * SB, p);
  wait_stages([]() constexpr { return NST - 1; });
  stage_barrier();
#pragma unroll
  for (int q = 0; q < 2 * CN; q++) fb[0][q >> 1][q & 1] = rb[(q >> 1) * 128 + (q & 1) * 32];
#pragma unroll
  for (int q = 0; q < 4 * RM; q++) fa[0][q >> 2][q & 3] = ra[q & 3][(q >> 2) * 256];

  uint32_t slot = 0;                                      // slot of stage s (bytes)
  auto step = [&](int st, int c) {
    wait_stages([]() constexpr { return NST - 2; });      // stage s + 1 landed (this wave's part)
    wait_lgkm0();                                         // this wave's reads of stage s are done
#pragma unroll
    for (int q = 0; q < 4; q++) set_dword(wc[0], q, widen_pair<AMODE>(fb[c][0][0], q));
    __builtin_amdgcn_sched_barrier(0);
    stage_barrier();                                      // stage s + 1 visible; slot of stage s free
    const uint32_t nxt = slot + SB == NST * SB ? 0u : slot + SB;
    const int sc = min(st + NST, KB - 1);
    auto mem_op = [&](int q) {
      if (q < 2 * CN) fb[c ^ 1][q >> 1][q & 1] = rb[nxt / 16 + (q >> 1) * 128 + (q & 1) * 32];
      else if (q < 2 * CN + 4 * RM) {
        const int f = q - 2 * CN;
        fa[c ^ 1][f >> 2][f & 3] = ra[f & 3][nxt / 16 + (f >> 2) * 256];
      } else {
        copy(sc, slot, q - 2 * CN - 4 * RM);
      }
    };
#pragma unroll
    for (int m = 0; m < NM; m++) {
      const int ph = m / RM, i = m % RM, j = ph >> 2, t = ph & 3;   // phase ph: K part t = 2 u + h of column j
      // the next phase's operand, spread before this phase's MFMAs
      if (ph + 1 < 4 * CN) {
        const int nj = (ph + 1) >> 2, nt = (ph + 1) & 3;
#pragma unroll
        for (int q = 4 / RM * i; q < 4 / RM * (i + 1); q++)
          set_dword(wc[(ph + 1) & 1], q, widen_pair<AMODE>(fb[c][nj][nt >> 1], 4 * (nt & 1) + q));
      }
      __builtin_amdgcn_sched_barrier(0);
      mfma32_acc<AMODE>(acc[i][j], wc[ph & 1], fa[c][i][t]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int q = m * MO; q < (m + 1) * MO; q++)
        if (q < NMEM) mem_op(q);
      __builtin_amdgcn_sched_barrier(0);
    }
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

  // the sums as 4-column pieces: piece g of block (i, j) is row 32 i + (lane & 31),
  // columns 32 j + 8 g + 4 (lane >> 5) .. + 3 of the wave's block
  v4f sum[RM][4 * CN];
#pragma unroll
  for (int i = 0; i < RM; i++)
#pragma unroll
    for (int q = 0; q < 4 * CN; q++)
#pragma unroll
      for (int r = 0; r < 4; r++) sum[i][q][r] = acc[i][q >> 2][4 * (q & 3) + r];
  if constexpr (SLICES) {
    if (a.S > 1 && !b16_merge<RM, 4 * CN>(a, sum, wv * RM, bt, ks, reinterpret_cast<int*>(sS))) return;
  }

  // Epilogue.  A wave's outputs go through its own part of LDS, 32 rows at a time,
  // already scaled and in the output type, and leave as 16 bytes per lane of
  // consecutive columns (stored straight from the accumulators a store covers 16
  // or 32 bytes of each of 32 rows).
  constexpr int COLS = 32 * CN;
  constexpr int LD4 = 4 * COLS + 16, LD2 = 2 * COLS + 16;  // bytes per LDS row of fp32 and of 16-bit outputs
  static_assert(LD4 % 16 == 0 && LD2 % 16 == 0, "rows are read in aligned 16-byte pieces");
  static_assert(NW * 32 * LD4 <= NST * TS * 1024, "rows of a pass fit the ring");
  uint8_t* const lw = reinterpret_cast<uint8_t*>(sS) + wv * (32 * LD4);
  const int n0 = (ng0 + wn * 2 * CN) * 16;
  const int lrow = lane & 31, lcol = 4 * (lane >> 5);
  const bool wide = a.out == OUT_F32;
  const int esz = wide ? 4 : 2;
  const bool vec = (a.ldy * esz) % 16 == 0 && (((uintptr_t)a.Y) & 15) == 0;
  const int room = min(COLS, a.N - n0);                   // the wave's columns inside N
  v4f ws[4 * CN], b[4 * CN];
#pragma unroll
  for (int q = 0; q < 4 * CN; q++) {
    // scales are padded with zeros to 16 NG
    ws[q] = *reinterpret_cast<const v4f*>(a.ws + min(n0 + 8 * q + lcol, a.NG * 16 - 4));
#pragma unroll
    for (int r = 0; r < 4; r++) b[q][r] = a.bias ? a.bias[min(n0 + 8 * q + lcol + r, a.N - 1)] : 0.0f;
  }
  __syncthreads();                                        // every wave's fragment reads are done
#pragma unroll
  for (int i = 0; i < RM; i++) {
    const int m0 = (mg0 + wm * 2 * RM + 2 * i) * 16;
#pragma unroll
    for (int q = 0; q < 4 * CN; q++) {
      v4f y;
#pragma unroll
      for (int r = 0; r < 4; r++) y[r] = __fmul_rn(sum[i][q][r], ws[q][r]);
      if (a.bias) {
#pragma unroll
        for (int r = 0; r < 4; r++) y[r] = __fadd_rn(y[r], b[q][r]);
      }
      if (wide) {
        *reinterpret_cast<v4f*>(lw + lrow * LD4 + (8 * q + lcol) * 4) = y;
      } else {
        uint2 h;
        if (a.out == OUT_BF16) {
          h = make_uint2(pack_bf16x2(y[0], y[1]), pack_bf16x2(y[2], y[3]));
        } else {
          h = make_uint2(pack_f16x2(y[0], y[1]), pack_f16x2(y[2], y[3]));
        }
        *reinterpret_cast<uint2*>(lw + lrow * LD2 + (8 * q + lcol) * 2) = h;
      }
    }
    wave_lds_fence();                                     // lanes read what other lanes wrote
    auto rows_out = [&](auto width) {
      constexpr int E = width(), PC = 16 / E, CPR = COLS / PC;   // bytes per output, outputs per piece, pieces per row
#pragma unroll 4
      for (int t = 0; t < 32 * CPR / 64; t++) {
        const int c = t * 64 + lane, r = c / CPR, col = (c - r * CPR) * PC;
        const v4i v = *reinterpret_cast<const v4i*>(lw + r * (E == 4 ? LD4 : LD2) + col * E);
        uint8_t* yp = static_cast<uint8_t*>(a.Y) + ((size_t)(m0 + r) * a.ldy + n0 + col) * E;
        if (m0 + r >= a.M) continue;
        if (vec && col + PC <= room) {
          if (E == 4) __builtin_nontemporal_store(v, reinterpret_cast<v4i*>(yp));   // streaming, as the int8 GEMM's
          else *reinterpret_cast<v4i*>(yp) = v;
        } else {
#pragma unroll
          for (int k = 0; k < PC; k++) {
            if (col + k >= room) continue;
            if (E == 4) reinterpret_cast<int*>(yp)[k] = v[k];
            else reinterpret_cast<uint16_t*>(yp)[k] = (uint16_t)((uint32_t)v[k >> 1] >> (16 * (k & 1)));
          }
        }
      }
    };
    if (wide) rows_out([]() constexpr { return 4; });
    else rows_out([]() constexpr { return 2; });
    wave_lds_fence();                                     // the next rows overwrite these
  }
}

// ---------------------------------------------------------------------------
// planning and launch
// ---------------------------------------------------------------------------
// cfg 0: LDS-staged kernel, 128 x 192 tiles
// cfg 4..8: wave-grid kernel, 256 x 192 and 256 x 128 (8 waves), 128 x 128 (two
//   work-groups per CU), 64 x 128 tiles with a 4-deep (two per CU) or 3-deep
//   ring (three per CU).  A 5-deep ring of those took as long as the 4-deep one
//   with weights from HBM and up to 3 % longer with repeated ones
static void b16_cfg(int cfg, int& mt, int& nt) {
  static const int dims[9][2] = {{8, 12}, {0, 0}, {0, 0}, {0, 0}, {16, 12}, {16, 8}, {8, 8}, {4, 8}, {4, 8}};
  mt = dims[cfg][0];
  nt = dims[cfg][1];
}

// tuning overrides; atomic, since a setter may run while other threads plan launches
static std::atomic<int> g_b16_force_cfg{-1};
static std::atomic<int> g_b16_force_split{0};
void gemm_b16_set_plan(int cfg, int split) {
  g_b16_force_cfg.store(cfg >= 0 && cfg <= 8 ? cfg : -1, std::memory_order_relaxed);
  // with cfg 3, split (when > 64) picks the small-M kernel's work-group shape
  gemm_small_set_b16_shape(cfg == 3 && split > 64 ? split : 0);
  if (cfg == 3) split = 0;
  g_b16_force_split.store(split > 0 ? split : 0, std::memory_order_relaxed);
}

// -1 planner, 0..2 and 4..8 a forced tile configuration of this file's
// kernels, 3 the streamed small-M kernel
int gemm_b16_forced_cfg() { return g_b16_force_cfg.load(std::memory_order_relaxed); }

static int b16_tiles(int cfg, int MG, int NG) {
  int mt, nt;
  b16_cfg(cfg, mt, nt);
  return cdiv(MG, mt) * cdiv(NG, nt);
}

// Plan: the configuration and K slices of least estimated time, rounds of
// work-groups times the time of one over KB k-blocks.  The constants are fitted
// to launches whose weights come from HBM (more copies of them than the caches
// hold, as in a model of many layers) and, at lower weight, to repeated ones, of
// every configuration and 1..4 slices: 16 x 22 shapes of 17..2048 rows, N = 1024
// .. 12288, K = 1000..6144.  The kernel chosen (the small-M kernel among them, up
// to 256 rows) is on average 0.3 % and at most 8 % slower than the best of its
// shape with weights from HBM, 0.6 % and 13 % with repeated ones.  (Constants from
// repeated launches alone had picked the 3-deep ring for single rounds of 64 x 128
// tiles: 17-18 us at 64 x 12288 and 256 x 4096, K = 2048, where 4 stages take
// 13.5-14.5; repeated, both take 13.3.)  K slices (the 4-wave configurations take
// them) cost a merge of three dependent memory round trips, so they pay only where
// the tiles leave most CUs idle: offered up to 128 tiles (333 x 2048 x 6144: 30.6
// us unsplit, 23.3 with 4 slices of 128 x 128).
struct B16Plan {
  int cfg, split;
  float us;
};
static B16Plan b16_best(int MG, int NG, int KB, bool whole = false) {
  B16Plan best{0, 1, 3.0e38f};
  auto offer = [&](int c, int s, float us) {
    if (us < best.us) best = B16Plan{c, s, us};
  };
  // 8 waves, one work-group per CU
  offer(4, 1, cdiv(b16_tiles(4, MG, NG), 256) * (10.3f + 1.1f * KB));
  offer(5, 1, cdiv(b16_tiles(5, MG, NG), 256) * (6.71f + 0.638f * KB));
  // 4 waves, work-groups share CUs: the time of a k-block grows with each half
  // round of 256 (and part of the later ones' fixed time runs under others' loops)
  static const float fixed[3] = {5.9f, 5.3f, 4.92f}, alone[3] = {0.416f, 0.256f, 0.362f},
                     shared[3] = {0.483f, 0.282f, 0.306f}, later[3] = {-1.06f, 0.954f, -0.197f},
                     merge[2] = {2.23f, 3.0f}, part[2] = {0.0267f, 0.0139f};
  for (int c = 6; c <= 8; c++) {
    const int i = c - 6, tiles = b16_tiles(c, MG, NG);
    for (int s = 1; s <= (c < 8 && tiles <= 128 && !whole ? 4 : 1) && s <= KB; s++) {
      const float half = 0.5f * (float)cdiv(tiles * s, 128), kb = (float)KB / s;
      offer(c, s, fixed[i] + (tiles * s <= 256 ? kb * alone[i] : kb * shared[i] * half + later[i] * (half - 1.0f)) +
                      (s > 1 ? merge[i] + part[i] * tiles * s : 0.0f));
    }
  }
  return best;
}
// estimated us of the wave-grid kernel's plan
float gemm_b16_us(int M, int N, int K) { return b16_best(cdiv(M, 16), cdiv(N, 16), cdiv(K, 64)).us; }

static void b16_plan(int MG, int NG, int KB, bool off32, bool whole, int& cfg_out, int& split_out) {
  int cfg = 0, split = 1;
  if (off32) {
    const B16Plan best = b16_best(MG, NG, KB, whole);
    cfg = best.cfg;
    split = best.split;
  }
  const int fc = g_b16_force_cfg.load(std::memory_order_relaxed);
  const int fs = g_b16_force_split.load(std::memory_order_relaxed);
  if (fc >= 0 && fc != 3) {
    cfg = fc >= 4 && off32 ? fc : 0;
    split = 1;
  }
  if (fs > 0) split = std::min(fs, std::max(1, KB));
  if (split > 1 && (cfg == 4 || cfg == 5)) cfg = 6;   // the 4-wave configurations take slices
  cfg_out = cfg;
  split_out = split;
}

// the wave-grid kernel where every X byte offset fits 32 bits, else the LDS-staged
// one with its 64-bit addresses
void gemm_b16_resolve(GemmLaunch& L, size_t* part_bytes, size_t* counters) {
  const int MG = cdiv(L.M, 16), NG = cdiv(L.N, 16);
  const bool off32 = (size_t)L.M * (size_t)L.lda * 2 < ((size_t)1 << 32);
  int mt, nt;
  b16_plan(MG, NG, cdiv(L.K, 64), off32, L.whole, L.cfg, L.split);
  b16_cfg(L.cfg, mt, nt);
  const size_t tiles = (size_t)cdiv(MG, mt) * cdiv(NG, nt);
  *part_bytes = L.split > 1 ? tiles * L.split * (size_t)(256 * mt * nt) * sizeof(float) : 0;
  *counters = L.split > 1 ? tiles : 0;
}

template <int AMODE, int WM, int WN, int RM, int CN, int NST>
static void launch_b16_wave(const GemmB16Args& a, int blocks, hipStream_t st) {
  const dim3 grid(blocks), block(64 * WM * WN);
  if (a.K % 64 == 0) hipLaunchKernelGGL((gemm_b16_wave_kernel<AMODE, WM, WN, RM, CN, NST, true>), grid, block, 0, st, a);
  else hipLaunchKernelGGL((gemm_b16_wave_kernel<AMODE, WM, WN, RM, CN, NST, false>), grid, block, 0, st, a);
}
template <int AMODE>
static void launch_b16(const GemmB16Args& a, int cfg, int blocks, hipStream_t st) {
  switch (cfg) {
    case 0: hipLaunchKernelGGL((gemm_b16_lds_kernel<AMODE, 8, 12, 4, 2, 2>), dim3(blocks), dim3(256), 0, st, a); break;
    case 4: launch_b16_wave<AMODE, 4, 2, 2, 3, 3>(a, blocks, st); break;
    case 5: launch_b16_wave<AMODE, 2, 4, 4, 1, 4>(a, blocks, st); break;
    case 6: launch_b16_wave<AMODE, 1, 4, 4, 1, 3>(a, blocks, st); break;
    case 7: launch_b16_wave<AMODE, 1, 4, 2, 1, 4>(a, blocks, st); break;
    default: launch_b16_wave<AMODE, 1, 4, 2, 1, 3>(a, blocks, st); break;
  }
}

bool gemm_b16_supported(const GemmLaunch& L) {
  if (L.amode != A_BF16 && L.amode != A_F16) return false;
  if (L.K % 8 != 0 || L.lda % 8 != 0) return false;   // 8 elements per 16-byte copy
  if ((((uintptr_t)L.A) & 15) != 0) return false;
  return L.zero_tile != nullptr;
}

hipError_t launch_gemm_b16(const GemmLaunch& L, hipStream_t st) {
  if (!gemm_b16_supported(L) || L.ep != EP_SCALE) return hipErrorInvalidValue;
  GemmB16Args a;
  a.X = L.A;
  a.lda = L.lda;
  a.Bt = L.Bt;
  a.ws = L.ws;
  a.bias = L.bias;
  a.Y = L.Y;
  a.ldy = L.ldy;
  a.M = L.M;
  a.N = L.N;
  a.K = L.K;
  a.KB = cdiv(L.K, 64);
  a.MG = cdiv(L.M, 16);
  a.NG = cdiv(L.N, 16);
  a.out = L.out;
  a.zero_tile = L.zero_tile;
  const int sp = L.split;
  int mt, nt;
  b16_cfg(L.cfg, mt, nt);
  a.ntm = cdiv(a.MG, mt);
  a.ntn = cdiv(a.NG, nt);
  a.S = sp;
  a.part = static_cast<float*>(L.part);
  a.cnt = L.cnt;
  if (sp > 1 && (!a.part || !a.cnt)) return hipErrorInvalidValue;
  const long long blocks_ll = (long long)a.ntm * a.ntn * sp;
  if (blocks_ll > 0x7fffffffLL) return hipErrorInvalidValue;
  const int blocks = (int)blocks_ll;
  if (L.amode == A_BF16) launch_b16<A_BF16>(a, L.cfg, blocks, st);
  else launch_b16<A_F16>(a, L.cfg, blocks, st);
  return hipGetLastError();
}

}  // namespace tl
