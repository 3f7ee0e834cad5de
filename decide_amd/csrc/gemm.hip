// Projection GEMMs: C[M x N] = A[M x K] . B[N x K]^T on MFMA (fp32 accumulate).
//
// Replaces the reference's linearFwd -> blas.Sgemm(false, true, ...)
// (internal/nn/forward.go:122-124, internal/blas/gemm.go:61-138) for the four
// per-layer projections, with the elementwise work that follows each of them
// fused into the epilogue:
//   EPI_STORE : store in the operand type (qkv; RoPE is applied by the
//               attention kernel as it loads q and k)
//   EPI_F32   : store fp32, optionally C += (the residual adds, forward.go:318-322, 338-342)
//   EPI_GEGLU : act = gelu(value) * gate (forward.go:327-336); the Wi rows are
//               interleaved at upload so each 64-column group holds 32 value
//               rows followed by the 32 matching gate rows
//
// Design (gfx950):
//   * Both operands are K-contiguous (token-major activations, (out,in)
//     weights): every MFMA operand is one contiguous 16-byte LDS read.
//   * K is staged 128 bytes at a time through an NSTAGE-deep ring of LDS
//     buffers filled by direct global->LDS loads (global_load_lds_dwordx4), so
//     NSTAGE-1 stages are in flight while one is consumed and no registers are
//     spent on staging. Each wave-wide load writes 1 KB = 8 tile rows.
//   * LDS rows are 128 bytes with the 16-byte chunks XOR-swizzled by
//     (row >> 1) & 7, so the 16 rows read by a quarter-wave fall in distinct
//     banks (the swizzle is applied on the global side of the DMA).
//   * Workgroup -> tile order is XCD-aware: consecutive workgroup ids go
//     round-robin over the 8 XCDs; up to a B of 12 MB each XCD owns a
//     contiguous range of the tiles in row order, so an A panel is read into
//     one XCD's L2 (two at a range's ends). A B of up to ~2 MB stays there too;
//     a larger one is read again for every few panels, out of the memory-side
//     cache (32,768 x 2304 x 768: 293 MB fetched against 224 with the N tiles
//     in groups of 2 MB of B, both 142 to 144 us).
//   * The epilogue stages the finished tile through LDS so global stores are
//     full 16-byte-per-lane rows.
#include <type_traits>

#include "common.hpp"

namespace {


// XOR swizzle of the 16-byte chunks of an LDS tile row: with RB-byte rows,
// the 16 rows read by a quarter-wave at one logical chunk land in 16
// distinct 4-bank groups.
template <int RB>
__device__ __forceinline__ int swz(int row) {
  return RB == 128 ? (row >> 1) & 7 : (row >> 2) & 3;
}

typedef __attribute__((address_space(3))) void lds_void;
typedef const __attribute__((address_space(1))) void gbl_void;

// s_waitcnt vmcnt(n) with the other counters left alone (gfx9 encoding:
// vmcnt[3:0] in bits 3:0, vmcnt[5:4] in bits 15:14, expcnt 6:4, lgkmcnt 11:8).
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (15 << 8) | ((N >> 4) << 14));
}

// Eight 16-byte LDS reads and the wait for them (s_waitcnt lgkmcnt(0)) in
// one statement, so the outputs hold the data when the statement ends (an
// asm output counts as written at the end of its statement; were the wait a
// separate statement, a register copy the compiler placed in between would
// read a value not yet landed). The compiler does not see these as reads of
// memory that global->LDS DMA writes, so it adds no vmcnt wait of its own:
// the caller waits for the DMA explicitly.
__device__ __forceinline__ void lds_read8x16(const char *const (&p)[8], uint4 (&o)[8]) {
  typedef int i32x4 __attribute__((ext_vector_type(4)));
  uint32_t a[8];
#pragma unroll
  for (int i = 0; i < 8; i++) a[i] = (uint32_t)(size_t)(const __attribute__((address_space(3))) char *)p[i];
  i32x4 v0, v1, v2, v3, v4, v5, v6, v7;
  asm volatile(
      "ds_read_b128 %0, %8\n\t"
      "ds_read_b128 %1, %9\n\t"
      "ds_read_b128 %2, %10\n\t"
      "ds_read_b128 %3, %11\n\t"
      "ds_read_b128 %4, %12\n\t"
      "ds_read_b128 %5, %13\n\t"
      "ds_read_b128 %6, %14\n\t"
      "ds_read_b128 %7, %15\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(v0), "=&v"(v1), "=&v"(v2), "=&v"(v3), "=&v"(v4), "=&v"(v5), "=&v"(v6), "=&v"(v7)
      : "v"(a[0]), "v"(a[1]), "v"(a[2]), "v"(a[3]), "v"(a[4]), "v"(a[5]), "v"(a[6]), "v"(a[7])
      : "memory");
  o[0] = __builtin_bit_cast(uint4, v0), o[1] = __builtin_bit_cast(uint4, v1);
  o[2] = __builtin_bit_cast(uint4, v2), o[3] = __builtin_bit_cast(uint4, v3);
  o[4] = __builtin_bit_cast(uint4, v4), o[5] = __builtin_bit_cast(uint4, v5);
  o[6] = __builtin_bit_cast(uint4, v6), o[7] = __builtin_bit_cast(uint4, v7);
}

// The same with four reads.
__device__ __forceinline__ void lds_read4x16(const char *const (&p)[4], uint4 (&o)[4]) {
  typedef int i32x4 __attribute__((ext_vector_type(4)));
  uint32_t a[4];
#pragma unroll
  for (int i = 0; i < 4; i++) a[i] = (uint32_t)(size_t)(const __attribute__((address_space(3))) char *)p[i];
  i32x4 v0, v1, v2, v3;
  asm volatile(
      "ds_read_b128 %0, %4\n\t"
      "ds_read_b128 %1, %5\n\t"
      "ds_read_b128 %2, %6\n\t"
      "ds_read_b128 %3, %7\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(v0), "=&v"(v1), "=&v"(v2), "=&v"(v3)
      : "v"(a[0]), "v"(a[1]), "v"(a[2]), "v"(a[3])
      : "memory");
  o[0] = __builtin_bit_cast(uint4, v0), o[1] = __builtin_bit_cast(uint4, v1);
  o[2] = __builtin_bit_cast(uint4, v2), o[3] = __builtin_bit_cast(uint4, v3);
}

// Workgroup -> tile: XCD x (workgroup ids congruent to x mod 8) takes the x-th
// of eight contiguous ranges of the row-ordered tiles, for any tile count.
// Row order over all workgroups, which ragged row counts took before, spread
// each A panel over every XCD (3,840 x 768 x 2304, 128 x 128 tiles: 25.9 ->
// 23.4 us; 3,840 x 2304 x 768: 25.7 -> 24.3 us).
// A wide and large B would stream through every XCD's L2 for each of its
// panels: from kRowOrderB bytes and kRowOrderN columns on, the grid is one row
// of tiles after the other (blockIdx.y), whose column tiles go to the XCDs by
// ranges, so an XCD sees an eighth of B (bf16, us, ranges over the whole grid /
// this: 20,000 x 8192 x 1024, B 16 MB, 396 / 383; 8,192 x 4096 x 4096 into fp32,
// 383 / 344; 20,000 x 4096 x 4096 725 / 679; 20,000 x 8192 x 8192 2,770 / 2,590;
// 20,000 x 6144 x 1024, B 12 MB, 296 / 292; smaller or narrower B in row order
// lose or gain nothing: 20,000 x 5248 x 1024, B 10.2 MB, 248 / 259; 20,000 x
// 1024 x 8192 400 / 533; 20,000 x 2048 x 4096 356 / 355).
// The order is the grid's shape: as a word of the arguments, or computed from
// N and K, it cost every launch 0.1 to 0.25 us (a 512-token forward 932 -> 937
// and 938 -> 960 us).
constexpr size_t kRowOrderB = (size_t)12 << 20;
constexpr int kRowOrderN = 4096;
template <int BM, int BN>
struct TileOrder {
  int m0, n0;
  __device__ __forceinline__ explicit TileOrder(int tiles_n) {
    const int bid = blockIdx.x, nt = (int)gridDim.x, q = nt >> 3, r = nt & 7, xcd = bid & 7;
    const int t = (int)blockIdx.y * nt + xcd * q + min(xcd, r) + (bid >> 3);
    m0 = (t / tiles_n) * BM;
    n0 = (t % tiles_n) * BN;
  }
};

// Copies a staged tile (BM rows of V 16-byte vectors, LD elements apart in
// LDS) to rows m0.. of C (row stride ldc, from column c0), rows past M
// skipped. The LDS reads go in batches of eight ahead of their stores, so a
// thread waits for LDS once per batch rather than once per vector.
template <class T, int BM, int V, int NT, int LD>
__device__ __forceinline__ void store_staged(const T *st, T *C, int ldc, int m0, int c0, int M, int tid) {
  constexpr int EPV = 16 / sizeof(T), ITER = BM * V / NT;
  static_assert(ITER * NT == BM * V, "staged tile shape");
  if constexpr (ITER % 8 == 0) {
    // One asm statement reads the batch and waits for it (lds_read8x16), so
    // the compiler cannot sink each read into its store's row guard.
#pragma unroll
    for (int b0 = 0; b0 < ITER; b0 += 8) {
      const char *p[8];
      uint4 v[8];
#pragma unroll
      for (int u = 0; u < 8; u++) {
        const int c = tid + (b0 + u) * NT;
        p[u] = (const char *)(st + (c / V) * LD + (c % V) * EPV);
      }
      lds_read8x16(p, v);
#pragma unroll
      for (int u = 0; u < 8; u++) {
        const int c = tid + (b0 + u) * NT, row = m0 + c / V;
        if (row < M) *(uint4 *)(C + (size_t)row * ldc + c0 + (c % V) * EPV) = v[u];
      }
    }
  } else {
#pragma unroll
    for (int u = 0; u < ITER; u++) {
      const int c = tid + u * NT, row = m0 + c / V;
      if (row < M) *(uint4 *)(C + (size_t)row * ldc + c0 + (c % V) * EPV) = *(const uint4 *)(st + (c / V) * LD + (c % V) * EPV);
    }
  }
}

// Folded LayerNorm, consumer side. ln_fold_load fetches row `row`'s
// per-part (mean, M2) pairs (fp32: each of a row block's N-tiles reads
// them, so their bytes pass the memory path many times) and mprev (issued
// before the first stages' DMA,
// whose issue is not delayed by them); ln_fold_merge combines the pairs by
// the pairwise update of Chan, Golub and LeVeque for equal counts (the mean
// of the part means; M2 = the parts' M2 plus the count times the squared
// deviations of the part means), in fp64 like the LayerNorm kernel's
// two-pass statistics, and returns (rstd, mean - mprev) with mean and rstd
// rounded to float as that kernel rounds them; write_mean also stores the
// row's mean.
// NP parts of PC columns (launch_gemm checks lparts == NP, NP PC == K).
template <int NP>
__device__ __forceinline__ void ln_fold_load(const GemmArgs &g, const LnFold &lf, int row, float2 (&v)[NP], float &mp) {
  const int rr = min(row, g.M - 1);
  const float2 *pp = (const float2 *)lf.lpart + (size_t)rr * NP;
#pragma unroll
  for (int t = 0; t < NP; t++) v[t] = pp[t];
  mp = lf.mprev ? lf.mprev[rr] : 0.0f;
}
template <int NP, int PC>
__device__ __forceinline__ float2 ln_fold_merge(const GemmArgs &g, const LnFold &lf, int row, const float2 (&v)[NP],
                                                float mp, bool write_mean) {
  double sum = 0;
#pragma unroll
  for (int t = 0; t < NP; t++) sum += (double)v[t].x;
  const double mu = sum / NP;
  double m2 = 0;
#pragma unroll
  for (int t = 0; t < NP; t++) {
    const double d = (double)v[t].x - mu;
    m2 += (double)v[t].y + (double)PC * d * d;
  }
  const float mean = (float)mu;
  if (write_mean && row < g.M) lf.mean_out[row] = mean;
  return make_float2((float)(1.0 / sqrt(m2 / (double)g.K + (double)lf.eps)), mean - mp);
}

// WGM x WGN waves tile the BM x BN block; each wave owns a WM x WN sub-tile.
// The body of gemm_nt_kernel and gemm_nt_ln_kernel (lf: the folded
// LayerNorm's arguments, used by the EPI_*_LN forms only; PC: its statistics'
// columns per part). PF: the main loop for small wave tiles (below).
// SEG: the product is the sum of K / (seg stages) partial products, each
// summed from zero and added in K order, to the bit what a split over
// workgroups and a reduction in split order give.
template <class T, int BM, int BN, int RB, int NSTAGE, int EPI, int WPE, int WGM, int WGN, bool PF, int PC, bool SEG = false>
__device__ __forceinline__ void gemm_nt_tile(const GemmArgs &g, const LnFold &lf, int seg = 0) {
  static_assert(!SEG || PF, "segments are summed in the operand-resident loop");
  using MF = Mfma<T>;
  typedef typename MF::frag frag;
  constexpr int NW = WGM * WGN, NT = 64 * NW;
  constexpr int KT = RB / sizeof(T);   // K elements per stage (RB-byte rows)
  constexpr int CPR = RB / 16;         // 16-byte chunks per row
  constexpr int RPI = 1024 / RB;       // rows per wave-wide DMA instruction
  constexpr int WM = BM / WGM, WN = BN / WGN;
  constexpr int TM = WM / 32, TN = WN / 32;
  constexpr int STAGE = (BM + BN) * RB;
  constexpr int LOADS = (BM + BN) * CPR / NT;  // 16-byte DMA loads per thread per stage
  constexpr bool LNC = EPI == EPI_STORE_LN || EPI == EPI_GEGLU_LN;  // folded LayerNorm consumer
  static_assert(LOADS * NT == (BM + BN) * CPR, "tile rows must fill whole DMA instructions");
  static_assert(!LNC || (BM <= NT && BN <= NT), "one thread per row and column of the folded LayerNorm's terms");
  static_assert(EPI == EPI_F32 || EPI == EPI_F32_LN || EPI == EPI_GEGLU_BWD || TN % 2 == 0,
                "paired epilogues need 64-column wave tiles");
  constexpr bool F32OUT = EPI == EPI_F32 || EPI == EPI_F32_LN;
  constexpr bool GATED = EPI == EPI_GEGLU || EPI == EPI_GEGLU_LN;
  static_assert(NSTAGE >= 2 && LOADS * (NSTAGE - 2) < 64, "pipeline depth");
  // fp32 epilogue staged in WGM passes of WM rows; the others in one pass.
  constexpr int EPI_BYTES = (F32OUT || EPI == EPI_GEGLU_BWD) ? WM * (BN + 4) * 4
                                                            : BM * ((GATED ? BN / 2 : BN) + 8) * (int)sizeof(T);
  constexpr int SMEM_RING = NSTAGE * STAGE > EPI_BYTES ? NSTAGE * STAGE : EPI_BYTES;
  // The folded LayerNorm consumer's row statistics and column sums follow
  // the ring in the same array: a second LDS object would make the compiler
  // wait for every DMA (vmcnt(0)) before the main loop's fragment reads.
  constexpr int LN_BYTES = LNC ? BM * 8 + BN * 4 : 0;
  __shared__ __attribute__((aligned(1024))) char smem[SMEM_RING + LN_BYTES];

  // The wave index is uniform: readfirstlane keeps it (and every LDS-DMA
  // destination, which goes through M0) in scalar registers.
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WGN, wn = wave % WGN;
  const int lr = lane & 31, lh = lane >> 5;

  const TileOrder<BM, BN> to(g.N / BN);
  const int m0 = to.m0, n0 = to.n0;
  // Folded LayerNorm consumer: thread t < BM takes block row t's statistics
  // and thread t < BN column n0 + t's lcs (loaded here; merged after the
  // main loop, when they have landed with the last stage, so the first
  // stages start without waiting for them); the epilogue reads (rstd, mean -
  // mprev) of its rows from ln_st and its columns' lcs from ln_cs.
  float2 *const ln_st = (float2 *)(smem + SMEM_RING);
  float *const ln_cs = (float *)(smem + SMEM_RING + BM * 8);
  constexpr int NP = LNC ? kLnHidden / PC : 1;
  float2 ln_v[NP];
  float ln_mp = 0.0f, ln_c = 0.0f;
  if constexpr (LNC) {
    if (threadIdx.x < BM) ln_fold_load<NP>(g, lf, m0 + (int)threadIdx.x, ln_v, ln_mp);
    if (threadIdx.x < BN) ln_c = lf.lcs[n0 + threadIdx.x];
  }
  // Split-K: blockIdx.z takes K elements [z*K, (z+1)*K) of A and B and writes
  // its own partial output.
  const size_t koff = (size_t)blockIdx.z * g.K;
  const T *gA = (const T *)g.A + koff, *gB = (const T *)g.B + koff;
  char *gC = (char *)g.C + (size_t)blockIdx.z * g.c_split * (F32OUT ? 4 : sizeof(T));

  // DMA sources: load i of this wave fills tile rows RPI*(wave + NW*i) .. +RPI-1;
  // lane l writes row RPI*(wave+NW*i) + l/CPR, LDS chunk slot l%CPR, which
  // holds the row's logical 16-byte chunk (l%CPR) ^ swz(row).
  const char *src[LOADS];
#pragma unroll
  for (int i = 0; i < LOADS; i++) {
    const int r = RPI * (wave + NW * i) + lane / CPR;
    const int c = (lane % CPR) ^ swz<RB>(r);
    if (r < BM)
      src[i] = (const char *)gA + (size_t)min(m0 + r, g.M - 1) * g.lda * sizeof(T) + c * 16;
    else
      src[i] = (const char *)gB + (size_t)(n0 + r - BM) * g.ldb * sizeof(T) + c * 16;
  }
  auto issue_part = [&](int stage, int k0, int i0, int i1) {
    char *dst = smem + stage * STAGE + wave * 1024;
    const size_t kb = (size_t)k0 * sizeof(T);
#pragma unroll
    for (int i = i0; i < i1; i++)
      __builtin_amdgcn_global_load_lds((gbl_void *)(src[i] + kb), (lds_void *)(dst + i * NW * 1024), 16, 0, 0);
  };
  auto issue = [&](int stage, int k0) { issue_part(stage, k0, 0, LOADS); };

  f32x16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; i++)
#pragma unroll
    for (int j = 0; j < TN; j++)
#pragma unroll
      for (int e = 0; e < 16; e++) acc[i][j][e] = 0.0f;

  const int rw = wm * WM, cw = wn * WN;  // wave tile origin inside the block tile

  // Every stage issues the same number of DMA loads (past the end of K the
  // last stage is re-read into a ring slot nothing reads again), so the
  // vmcnt arithmetic below is exact and no branch surrounds a DMA issue.
  const int nk = g.K / KT;
#pragma unroll
  for (int s = 0; s < NSTAGE - 1; s++) issue(s, min(s, nk - 1) * KT);

  constexpr int NKS = KT / MF::KSTEP;                  // MFMA k steps per stage
  constexpr int PER_KS = (LOADS + NKS - 1) / NKS;      // next-stage loads issued per k step
  static_assert(NKS % 2 == 0, "operand double buffering alternates per k step");

  if constexpr (PF) {
    // Small wave tiles (one or two MFMAs a k step, fewer cycles than an LDS
    // read takes): a stage's operands are all in registers before its first
    // MFMA, and each k step's fragments are replaced by the next stage's right
    // after the MFMAs that used them. The loop below with its one k step of
    // lookahead spends ~550 cycles a stage on LDS latency there, this one about
    // half (512 x 768 x 768 on 64 x 64 tiles 6.9 -> 5.9 us, K = 2304 13.2 ->
    // 10.2 us; the same MFMAs in the same order). A stage is read into
    // registers one stage ahead, so one DMA stage fewer is in flight; past the
    // last one nothing is issued, and the last NSTAGE - 1 stages run unrolled
    // with their own waits.
    frag fa[NKS][TM], fb[NKS][TN];
    auto load_step = [&](int slot, int ks) {
      const char *sa = smem + slot * STAGE;
      const char *sb = sa + BM * RB;
      const int ke = ks * MF::KSTEP + lh * MF::SLOTS;
      const int chunk = ke * (int)sizeof(T) / 16, within = ke * (int)sizeof(T) % 16;
#pragma unroll
      for (int i = 0; i < TM; i++) {
        const int r = wm * WM + i * 32 + lr;
        fa[ks][i] = *(const frag *)(sa + r * RB + ((chunk ^ swz<RB>(r)) << 4) + within);
      }
#pragma unroll
      for (int j = 0; j < TN; j++) {
        const int r = wn * WN + j * 32 + lr;
        fb[ks][j] = *(const frag *)(sb + r * RB + ((chunk ^ swz<RB>(r)) << 4) + within);
      }
    };
    auto mfmas = [&](int ks) {
#pragma unroll
      for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) acc[i][j] = MF::mma(fb[ks][j], fa[ks][i], acc[i][j]);
    };
    wait_vmcnt<LOADS * (NSTAGE - 2)>();
    __builtin_amdgcn_s_barrier();
#pragma unroll
    for (int ks = 0; ks < NKS; ks++) load_step(0, ks);
    // No scalar load in flight past here, so the compiler's waits in the loop
    // count LDS reads exactly.
    __builtin_amdgcn_s_waitcnt(0xc07f);
    f32x16 total[SEG ? TM : 1][SEG ? TN : 1];
    int left = seg;  // stages to the segment's end
    if constexpr (SEG)
#pragma unroll
      for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
          for (int e = 0; e < 16; e++) total[i][j][e] = 0.0f;
    auto end_stage = [&]() {
      if constexpr (SEG)
        if (--left == 0) {
          left = seg;
#pragma unroll
          for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++)
#pragma unroll
              for (int e = 0; e < 16; e++) {
                total[i][j][e] += acc[i][j][e];
                acc[i][j][e] = 0.0f;
              }
        }
    };
    int kt = 0, slot = 0;
    for (; kt + NSTAGE - 1 < nk; kt++) {
      const int nslot = slot + 1 == NSTAGE ? 0 : slot + 1, pslot = slot == 0 ? NSTAGE - 1 : slot - 1;
      wait_vmcnt<LOADS * (NSTAGE - 3)>();
      __builtin_amdgcn_s_barrier();
#pragma unroll
      for (int ks = 0; ks < NKS; ks++) {
        mfmas(ks);
        load_step(nslot, ks);
        const int i0 = ks * PER_KS < LOADS ? ks * PER_KS : LOADS;
        const int i1 = (ks + 1) * PER_KS < LOADS ? (ks + 1) * PER_KS : LOADS;
        issue_part(pslot, (kt + NSTAGE - 1) * KT, i0, i1);
        __builtin_amdgcn_sched_group_barrier(0x008, TM * TN, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, TM + TN, 0);
        __builtin_amdgcn_sched_group_barrier(0x020, PER_KS, 0);
      }
      end_stage();
      slot = nslot;
    }
    auto tail = [&](auto tc) {
      constexpr int TT = decltype(tc)::value;  // 0 .. NSTAGE - 2
      if (kt + NSTAGE - 1 - TT == nk) {
        const int nslot = slot + 1 == NSTAGE ? 0 : slot + 1;
        if constexpr (TT < NSTAGE - 2) {
          wait_vmcnt<LOADS * (NSTAGE - 3 - TT > 0 ? NSTAGE - 3 - TT : 0)>();
          __builtin_amdgcn_s_barrier();
        }
#pragma unroll
        for (int ks = 0; ks < NKS; ks++) {
          mfmas(ks);
          if constexpr (TT < NSTAGE - 2) load_step(nslot, ks);
        }
        end_stage();
        slot = nslot;
        kt++;
      }
    };
    static_assert(NSTAGE >= 3 && NSTAGE <= 5, "unrolled tail");
    tail(std::integral_constant<int, 0>{});
    tail(std::integral_constant<int, 1>{});
    if constexpr (NSTAGE > 3) tail(std::integral_constant<int, 2>{});
    if constexpr (NSTAGE > 4) tail(std::integral_constant<int, 3>{});
    if constexpr (SEG)
#pragma unroll
      for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) acc[i][j] = total[i][j];
  } else {
    // MFMA operands are double buffered across k steps: the fragments of step
    // ks+1 (or of the next stage's step 0) are read from LDS while the MFMAs of
    // step ks run. The next stage's readiness (vmcnt + barrier) is established
    // at the end of each stage, after the last MFMAs of the stage are issued.
    frag fa[2][TM], fb[2][TN];
    auto load_frags = [&](int buf, int stage, int ks) {
      const char *sa = smem + stage * STAGE;
      const char *sb = sa + BM * RB;
      const int ke = ks * MF::KSTEP + lh * MF::SLOTS;  // first k element of this lane's operand
      const int chunk = ke * (int)sizeof(T) / 16, within = ke * (int)sizeof(T) % 16;
#pragma unroll
      for (int i = 0; i < TM; i++) {
        const int r = wm * WM + i * 32 + lr;
        fa[buf][i] = *(const frag *)(sa + r * RB + ((chunk ^ swz<RB>(r)) << 4) + within);
      }
#pragma unroll
      for (int j = 0; j < TN; j++) {
        const int r = wn * WN + j * 32 + lr;
        fb[buf][j] = *(const frag *)(sb + r * RB + ((chunk ^ swz<RB>(r)) << 4) + within);
      }
    };
    // Waits until stage kt has landed for every wave: NSTAGE-2 later stages'
    // loads may still be in flight.
    auto stage_ready = [&]() {
      wait_vmcnt<LOADS * (NSTAGE - 2)>();
      __builtin_amdgcn_s_barrier();
    };

    stage_ready();
    load_frags(0, 0, 0);
    for (int kt = 0; kt < nk; kt++) {
      // Refill the buffer of stage kt-1 (every wave finished reading it before
      // the barrier that made stage kt visible) with stage kt + NSTAGE - 1.
      const int rstage = (kt + NSTAGE - 1) % NSTAGE, rk = min(kt + NSTAGE - 1, nk - 1) * KT;
#pragma unroll
      for (int ks = 0; ks < NKS; ks++) {
        const int cur = ks & 1;
        // Program order: next step's operand reads, this step's share of the
        // DMA refill (the DMA writes LDS, so reads placed after it could not be
        // hoisted above it), then this step's MFMAs.
        if (ks + 1 < NKS) load_frags(cur ^ 1, kt % NSTAGE, ks + 1);
        {
          const int i0 = ks * PER_KS < LOADS ? ks * PER_KS : LOADS;
          const int i1 = (ks + 1) * PER_KS < LOADS ? (ks + 1) * PER_KS : LOADS;
          issue_part(rstage, rk, i0, i1);
        }
        // B is the MFMA's first operand: acc[i][j] holds the transposed
        // 32x32 block, so lane l owns token row l%32 and four runs of four
        // consecutive output columns (vector stores in the epilogue).
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
          for (int j = 0; j < TN; j++) acc[i][j] = MF::mma(fb[cur][j], fa[cur][i], acc[i][j]);
        // One MFMA, then all of the next step's operand reads (they get the
        // rest of the step to land), then the DMA issues, then the MFMAs.
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        if (ks + 1 < NKS) __builtin_amdgcn_sched_group_barrier(0x100, TM + TN, 0);
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x020, PER_KS, 0);
        __builtin_amdgcn_sched_group_barrier(0x008, TM * TN - 2, 0);
        if (ks + 1 == NKS && kt + 1 < nk) {
          stage_ready();
          load_frags(cur ^ 1, (kt + 1) % NSTAGE, 0);
        }
      }
    }
  }
  // All waves done with the ring and every DMA landed: reuse it for the epilogue.
  wait_vmcnt<0>();
  if constexpr (LNC) {
    // The folded LayerNorm's row statistics (loaded at the start, landed
    // with the last stage) and column sums, for every wave's epilogue: the
    // barrier must also wait for these LDS writes.
    if (threadIdx.x < BM) ln_st[threadIdx.x] = ln_fold_merge<NP, PC>(g, lf, m0 + (int)threadIdx.x, ln_v, ln_mp, n0 == 0);
    if (threadIdx.x < BN) ln_cs[threadIdx.x] = ln_c;
    __syncthreads();
  } else {
    __builtin_amdgcn_s_barrier();
  }
  // fp32 staging of the rows of wave row `pass` (LD floats per row).
  auto stage_f32 = [&](float *st, int LD, int pass) {
    if (wm == pass) {
#pragma unroll
      for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
          for (int q = 0; q < 4; q++)
            *(float4 *)(st + (i * 32 + lr) * LD + cw + j * 32 + mfma_row(4 * q, lane)) =
                make_float4(acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]);
    }
  };
  if constexpr (EPI == EPI_GEGLU_BWD) {
    // The product is dact (the GeGLU output's gradient, fp32, as the
    // reference's backward holds it); each thread takes 8 consecutive
    // columns of one row (inside one 32-column group), reads the matching
    // value and gate inputs and writes their gradients (backward.go:49-61).
    // Output column n of the product is value column 64*(n/32) + n%32 of the
    // interleaved layout, so the tile's outputs are 2*BN contiguous columns.
    constexpr int LD = BN + 4, HM = WM, U = BN / 8;
    constexpr int ITER = HM * U / NT;
    constexpr int BATCH = ITER <= 4 ? ITER : ITER % 4 == 0 ? 4 : ITER % 3 == 0 ? 3 : 2;
    static_assert(ITER * NT == HM * U && ITER % BATCH == 0, "GeGLU backward epilogue shape");
    float *st = (float *)smem;
    const T *Wg = (const T *)g.gin;
    T *D = (T *)gC;
#pragma unroll
    for (int pass = 0; pass < WGM; pass++) {
      stage_f32(st, LD, pass);
      __syncthreads();
      for (int b0 = 0; b0 < ITER; b0 += BATCH) {
        float a[BATCH][8], gt[BATCH][8];
#pragma unroll
        for (int u = 0; u < BATCH; u++) {
          const int c = tid + (b0 + u) * NT, r = c / U, cu = (c % U) * 8;
          const int row = min(m0 + pass * HM + r, g.M - 1);
          const size_t o = (size_t)row * g.ldc + 2 * n0 + 64 * (cu >> 5) + (cu & 31);
          Vec8<T>::load(Wg + o, a[u]);
          Vec8<T>::load(Wg + o + 32, gt[u]);
        }
#pragma unroll
        for (int u = 0; u < BATCH; u++) {
          const int c = tid + (b0 + u) * NT, r = c / U, cu = (c % U) * 8;
          const int row = m0 + pass * HM + r;
          if (row >= g.M) continue;
          const size_t o = (size_t)row * g.ldc + 2 * n0 + 64 * (cu >> 5) + (cu & 31);
          const float4 d0 = *(const float4 *)(st + r * LD + cu), d1 = *(const float4 *)(st + r * LD + cu + 4);
          const float da[8] = {d0.x, d0.y, d0.z, d0.w, d1.x, d1.y, d1.z, d1.w};
          float dv[8], dg[8];
#pragma unroll
          for (int e = 0; e < 8; e++) {
            dv[e] = da[e] * gt[u][e] * gelu_grad<T>(a[u][e]);
            dg[e] = da[e] * gelu_erf<T>(a[u][e]);
          }
          Vec8<T>::store(D + o, dv);
          Vec8<T>::store(D + o + 32, dg);
        }
      }
      if (pass + 1 < WGM) __syncthreads();
    }
  } else if constexpr (F32OUT) {
    constexpr bool LN = EPI == EPI_F32_LN;  // also the folded LayerNorm's operand and statistics
    constexpr int LD = BN + 4;  // floats per staged row
    constexpr int HM = WM;      // rows per pass: the waves with wm == pass stage theirs
    float *st = (float *)smem;
    float *C = (float *)gC;
    const float *R = g.res ? g.res : C;  // residual input of the accumulate
    constexpr int V = BN / 4;  // float4 per row
    constexpr int ITER = HM * V / NT;
    static_assert(ITER * NT == HM * V, "epilogue shape");
    // Folded LayerNorm: TPR threads per row of a pass, TPP per row and part
    // of PC columns. The sums of a part are associated as eight lanes' sums
    // whatever TPP is (16: a lane's chunks are split over two threads), so
    // the statistics do not depend on the tile.
    constexpr int TPR = NT / HM, PCC = LN ? PC : BN, TPP = TPR / (BN / PCC), CW = 4 * TPP;
    static_assert(!LN || (BN % PCC == 0 && TPR * HM == NT && TPP * (BN / PCC) == TPR && (TPP == 8 || TPP == 16) &&
                          PCC % CW == 0),
                  "LayerNorm statistics: 8 or 16 threads per row and part");
    const bool vec = (g.ldc & 3) == 0;
    // The residual loads of a pass are issued together (one HBM round trip
    // per pass): pass 0's before its staging, so that their latency overlaps
    // it; each later pass's right after the previous pass's stores, before
    // its staging barrier. Loads and stores of an element are made by the
    // same thread; the rows of different passes are disjoint.
    float4 old[ITER];
    auto load_old = [&](int pass) {
#pragma unroll
      for (int u = 0; u < ITER; u++) {
        const int c = tid + u * NT, r = c / V, c4 = (c % V) * 4;
        const int row = m0 + pass * HM + r, col = n0 + c4;
        old[u] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (g.accumulate && vec && row < g.M && col + 4 <= g.n_store)
          old[u] = *(const float4 *)(R + (size_t)row * g.ldc + col);
      }
    };
    load_old(0);
    // Folded LayerNorm: thread (row tid / TPR of the pass, thread tid % TPP of
    // part tid % TPR / TPP) takes the 4-column chunks CW q (q < NQ) after
    // column lnc, so that the TPP threads of a row and part store 8 TPP
    // contiguous bytes of the 16-bit operand per instruction; the LayerNorm
    // weight at them.
    constexpr int NQ = PCC / CW;
    const int lnc = tid % TPR / TPP * PCC + 4 * (tid % TPP);
    float4 lw4[LN ? NQ : 1];
    if constexpr (LN) {
#pragma unroll
      for (int q = 0; q < NQ; q++) lw4[q] = *(const float4 *)(lf.lw + n0 + lnc + CW * q);
    }
#pragma unroll
    for (int pass = 0; pass < WGM; pass++) {
      float ln_mp = 0.0f;
      if constexpr (LN)
        if (lf.mprev) ln_mp = lf.mprev[min(m0 + pass * HM + tid / TPR, g.M - 1)];
      stage_f32(st, LD, pass);
      __syncthreads();
#pragma unroll
      for (int u = 0; u < ITER; u++) {
        const int c = tid + u * NT, r = c / V, c4 = (c % V) * 4;
        const int row = m0 + pass * HM + r, col = n0 + c4;
        if (row >= g.M || col >= g.n_store) continue;
        const float4 v = *(const float4 *)(st + r * LD + c4);
        float *p = C + (size_t)row * g.ldc + col;
        if (vec && col + 4 <= g.n_store) {
          const float4 x = make_float4(v.x + old[u].x, v.y + old[u].y, v.z + old[u].z, v.w + old[u].w);
          *(float4 *)p = x;
          if constexpr (LN)  // read back below (launch_gemm guarantees vec and n_store == N for this form)
            *(float4 *)(st + r * LD + c4) = x;
        } else {
          const float vv[4] = {v.x, v.y, v.z, v.w};
          const float *pr = R + (size_t)row * g.ldc + col;
          for (int q = 0; q < 4 && col + q < g.n_store; q++) p[q] = g.accumulate ? pr[q] + vv[q] : vv[q];
        }
      }
      if constexpr (LN) {
        // The pass's rows from the staging area, the chunks above. The next
        // LayerNorm's operand (x - mprev) * w in T, one 8-byte store per chunk;
        // the statistics over each part's PC columns: fp32 sums of eight
        // lanes (lane v: the 4-column chunks 32 q + 4 v, in order), the eight
        // reduced in fp64 in a fixed order, then the squared deviations from
        // the part's mean the same way, stored as an fp32 pair (their fp32
        // rounding, ~1e-6 relative, is far below the 16-bit operand's).
        __syncthreads();
        const int r = tid / TPR;
        float4 xv[NQ];
#pragma unroll
        for (int q = 0; q < NQ; q++) xv[q] = *(const float4 *)(st + r * LD + lnc + CW * q);
        {
          const int row = m0 + pass * HM + r;
          if (row < g.M) {
            T *f = (T *)lf.fx + (size_t)row * g.ldc + n0 + lnc;
#pragma unroll
            for (int q = 0; q < NQ; q++) {
              const float4 a = xv[q], wa = lw4[q];
              *(uint2 *)(f + CW * q) = make_uint2(pack16<T>((a.x - ln_mp) * wa.x, (a.y - ln_mp) * wa.y),
                                                  pack16<T>((a.z - ln_mp) * wa.z, (a.w - ln_mp) * wa.w));
            }
          }
        }
        // A lane's chunk sums, added in column order: with 16 threads the
        // chunks alternate between threads v (even) and v + 8 (odd).
        const bool odd = TPP == 16 && (tid & 8);
        auto lane_sum = [&](const float (&c)[NQ]) {
          float t = 0.0f;
#pragma unroll
          for (int q = 0; q < NQ; q++) {
            if constexpr (TPP == 16) {
              const float o = __uint_as_float(dpp_u32<0x128>(__float_as_uint(c[q])));  // row_ror:8
              t += odd ? o : c[q];
              t += odd ? c[q] : o;
            } else {
              t += c[q];
            }
          }
          return t;
        };
        float cs[NQ];
#pragma unroll
        for (int q = 0; q < NQ; q++) cs[q] = (xv[q].x + xv[q].y) + (xv[q].z + xv[q].w);
        // Over eight lanes: lane ^ 1, lane ^ 2 and, the quads' lanes now being
        // equal, the half row mirrored for lane ^ 4.
        auto sum8 = [](double v) {
          v += dpp_f64<0xB1>(v);
          v += dpp_f64<0x4E>(v);
          v += dpp_f64<0x141>(v);
          return v;
        };
        const double sum = sum8(lane_sum(cs));
        const double mu = sum / PCC;
        const float muf = (float)mu;
#pragma unroll
        for (int q = 0; q < NQ; q++) {
          const float a = xv[q].x - muf, b = xv[q].y - muf, c = xv[q].z - muf, d = xv[q].w - muf;
          cs[q] = (a * a + b * b) + (c * c + d * d);
        }
        const double m2 = sum8(lane_sum(cs));
        const int row = m0 + pass * HM + r;
        if (tid % TPP == 0 && row < g.M)
          ((float2 *)lf.lpart)[(size_t)row * lf.lparts + (n0 + lnc) / PCC] = make_float2((float)mu, (float)m2);
      }
      if (pass + 1 < WGM) {
        load_old(pass + 1);
        __syncthreads();
      }
    }
  } else {
    // Operand-type epilogue: the plain product (gated false) or the GeGLU of
    // each value/gate column pair (gated true), staged in LDS and stored as
    // 16-byte rows. EPI_GEGLU_KEEP writes both (training keeps the Wi output).
    auto emit = [&](auto gated, T *Cout, int ldo) {
      constexpr bool G = decltype(gated)::value;
      constexpr int OC = G ? BN / 2 : BN;  // output columns of the block tile
      constexpr int LD = OC + 8;           // staged row length (elements)
      typedef T T4 __attribute__((ext_vector_type(4)));
      T *st = (T *)smem;
      // Folded LayerNorm consumer: lcs at this lane's columns (block j, run
      // q: the 4 columns from cw + 32 j + mfma_row(4 q)).
      float cs[LNC ? TN : 1][16];
      if constexpr (LNC) {
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
          for (int q = 0; q < 4; q++) {
            const float4 c4 = *(const float4 *)(ln_cs + cw + j * 32 + mfma_row(4 * q, lane));
            cs[j][4 * q] = c4.x, cs[j][4 * q + 1] = c4.y, cs[j][4 * q + 2] = c4.z, cs[j][4 * q + 3] = c4.w;
          }
      }
      // rstd * (product - (mean - mprev) * lcs) for the folded LayerNorm
      // (ln_st and ln_cs were written before the epilogue's barrier).
      float ln_rs[LNC ? TM : 1], ln_dm[LNC ? TM : 1];
      if constexpr (LNC) {
#pragma unroll
        for (int i = 0; i < TM; i++) {
          const float2 t = ln_st[rw + 32 * i + lr];
          ln_rs[i] = t.x, ln_dm[i] = t.y;
        }
      }
      auto fin = [&](float v, int i, int j, int e) -> float {
        if constexpr (LNC) {
          float r = __builtin_fmaf(-ln_dm[i], cs[j][e], v) * ln_rs[i];
          // fp16: the compiler would fuse this product into the conversion
          // for some outputs (v_fma_mixlo_f16, one rounding instead of two)
          // and not others, so results would depend on the tile shape; the
          // empty asm keeps every output a rounded fp32 product.
          if constexpr (std::is_same<T, f16>::value) asm("" : "+v"(r));
          return r;
        } else {
          return v;
        }
      };
#pragma unroll
      for (int i = 0; i < TM; i++) {
#pragma unroll
        for (int jp = 0; jp < TN / 2; jp++)
#pragma unroll
          for (int q = 0; q < 4; q++) {
            const int r = rw + i * 32 + lr, c = mfma_row(4 * q, lane);  // 4 consecutive columns from c
            const f32x16 &a = acc[i][2 * jp], &b = acc[i][2 * jp + 1];
            const int ja = 2 * jp, jb = 2 * jp + 1;
            if constexpr (!G) {
              *(T4 *)(st + r * LD + cw + jp * 64 + c) =
                  T4{to_elem<T>(fin(a[4 * q], i, ja, 4 * q)), to_elem<T>(fin(a[4 * q + 1], i, ja, 4 * q + 1)),
                     to_elem<T>(fin(a[4 * q + 2], i, ja, 4 * q + 2)), to_elem<T>(fin(a[4 * q + 3], i, ja, 4 * q + 3))};
              *(T4 *)(st + r * LD + cw + jp * 64 + 32 + c) =
                  T4{to_elem<T>(fin(b[4 * q], i, jb, 4 * q)), to_elem<T>(fin(b[4 * q + 1], i, jb, 4 * q + 1)),
                     to_elem<T>(fin(b[4 * q + 2], i, jb, 4 * q + 2)), to_elem<T>(fin(b[4 * q + 3], i, jb, 4 * q + 3))};
            } else {
              T4 o;
#pragma unroll
              for (int t = 0; t < 4; t++)
                o[t] = to_elem<T>(gelu_erf<T>(fin(a[4 * q + t], i, ja, 4 * q + t)) * fin(b[4 * q + t], i, jb, 4 * q + t));
              *(T4 *)(st + r * LD + (cw + jp * 64) / 2 + c) = o;
            }
          }
      }
      __syncthreads();
      const int oc0 = G ? n0 / 2 : n0;
      constexpr int EPV = 16 / sizeof(T);  // elements per 16-byte vector
      constexpr int V = OC / EPV;
      store_staged<T, BM, V, NT, LD>(st, Cout, ldo, m0, oc0, g.M, tid);
    };
    if constexpr (EPI == EPI_STORE || EPI == EPI_STORE_LN) {
      emit(std::false_type{}, (T *)gC, g.ldc);
    } else if constexpr (GATED) {
      emit(std::true_type{}, (T *)gC, g.ldc);
    } else {
      emit(std::false_type{}, (T *)gC, g.ldc);
      __syncthreads();  // the staging area is reused
      emit(std::true_type{}, (T *)g.C2, g.ldc2);
    }
  }
}

template <class T, int BM, int BN, int RB, int NSTAGE, int EPI, int WPE, int WGM, int WGN, bool PF>
__global__ __launch_bounds__(64 * WGM * WGN) __attribute__((amdgpu_waves_per_eu(WPE))) void gemm_nt_kernel(GemmArgs g) {
  static_assert(EPI < EPI_F32_LN, "the folded-LayerNorm forms run as gemm_nt_ln_kernel");
  gemm_nt_tile<T, BM, BN, RB, NSTAGE, EPI, WPE, WGM, WGN, PF, 0>(g, LnFold{});
}
template <class T, int BM, int BN, int RB, int NSTAGE, int WPE, int WGM, int WGN>
__global__ __launch_bounds__(64 * WGM * WGN) __attribute__((amdgpu_waves_per_eu(WPE))) void gemm_nt_seg_kernel(GemmArgs g,
                                                                                                             int seg) {
  gemm_nt_tile<T, BM, BN, RB, NSTAGE, EPI_F32, WPE, WGM, WGN, true, 0, true>(g, LnFold{}, seg);
}
template <class T, int BM, int BN, int RB, int NSTAGE, int EPI, int WPE, int WGM, int WGN, bool PF, int PC>
__global__ __launch_bounds__(64 * WGM * WGN) __attribute__((amdgpu_waves_per_eu(WPE))) void gemm_nt_ln_kernel(GemmArgs g,
                                                                                                            LnFold lf) {
  static_assert(EPI >= EPI_F32_LN, "plain forms run as gemm_nt_kernel");
  gemm_nt_tile<T, BM, BN, RB, NSTAGE, EPI, WPE, WGM, WGN, PF, PC>(g, lf);
}

// A tile configuration: block tile, K stage bytes, stages, workgroups per CU
// (waves per SIMD), waves, and the small-wave-tile main loop.
template <int BM_, int BN_, int RB_, int NSTAGE_, int WPE_, int WGM_, int WGN_, bool PF_ = false>
struct Tile {
  static constexpr int BM = BM_, BN = BN_, RB = RB_, NSTAGE = NSTAGE_, WPE = WPE_, WGM = WGM_, WGN = WGN_;
  static constexpr bool PF = PF_;
  static int count(const GemmArgs &a) { return (a.M + BM - 1) / BM * (a.N / BN); }
};

template <class T, class C, int EPI, int PC = 0>
hipError_t launch_tile(const GemmArgs &a, hipStream_t s, const LnFold *ln = nullptr, int splits = 1) {
  if (a.N % C::BN || a.K % (C::RB / (int)sizeof(T))) return hipErrorInvalidValue;
  const int tiles_n = a.N / C::BN, tiles_m = C::count(a) / tiles_n;
  const bool rows = a.N >= kRowOrderN && (size_t)a.N * a.K * sizeof(T) >= kRowOrderB && tiles_m <= 65535;
  const dim3 grid(rows ? tiles_n : tiles_n * tiles_m, rows ? tiles_m : 1, splits), block(64 * C::WGM * C::WGN);
  if constexpr (EPI >= EPI_F32_LN)
    hipLaunchKernelGGL((gemm_nt_ln_kernel<T, C::BM, C::BN, C::RB, C::NSTAGE, EPI, C::WPE, C::WGM, C::WGN, C::PF, PC>),
                       grid, block, 0, s, a, *ln);
  else
    hipLaunchKernelGGL((gemm_nt_kernel<T, C::BM, C::BN, C::RB, C::NSTAGE, EPI, C::WPE, C::WGM, C::WGN, C::PF>), grid,
                       block, 0, s, a);
  return hipGetLastError();
}

// Workgroups of a launch that runs in one round on 256 CUs.
constexpr int kCUs = 256;

// Small-M GEMM (M <= 128 in 16 bits: one request; fp32: f32_small_tiles, among
// them the scorer's dense layer over every [MASK] row of a batch). Such
// launches are bound by streaming the weights and by latency, and the
// 128-wide tiles above would give only N/128 workgroups. Here a workgroup
// owns a TR x TC output tile (TR = 32*MB rows, TC = 32*NB columns) and all
// of K:
//   * K is walked in groups of GK elements (four 16-byte loads per lane and
//     operand row); the W waves take the groups round-robin, each through
//     LDS of its own (DMA: whole rows a load, since the CU's address unit
//     serialises loads that touch 32 rows) or, on the 64-row and 16-bit
//     64-column tiles, straight from global memory into registers,
//     prefetching the next group while the current one is multiplied.
//   * The waves' partial tiles are summed through LDS in a fixed order, so
//     results do not depend on timing, by the threads that store the
//     result (one barrier). Splitting K across workgroups of one launch
//     would need a device-scope release/acquire per workgroup (an L2
//     writeback + invalidate on gfx950); instead launch_gemm_small_split
//     gives each K slice its own fp32 partial tile and the kernel that
//     follows (the next LayerNorm, launch_ln_parts) sums the slices.
// Operand layout: in load j of a group, lane l reads the 16 bytes of row
// l%32 at group offset 2*VPL*j + VPL*(l/32); for bf16 that is exactly the
// k step j operand of v_mfma_f32_32x32x16_bf16, for fp32 the four values
// feed four v_mfma_f32_32x32x2f32 (A and B use the same k order).
template <int V>
using fvec = float __attribute__((ext_vector_type(V)));

// Sum of the NP partial tiles (TE floats apart) at float index idx (a
// multiple of V): (p0 + p4) + (p1 + p5) + (p2 + p6) + (p3 + p7) for eight,
// p0 + p1 + p2 + p3 for four.
template <int V, int NP, int TE>
__device__ __forceinline__ fvec<V> partial_sum(const float *red, int idx) {
  const fvec<V> *p = (const fvec<V> *)(red + idx);
  constexpr int S = TE / V;
  fvec<V> v;
  if constexpr (NP == 8) {
    v = p[0] + p[4 * S];
#pragma unroll
    for (int w = 1; w < 4; w++) v = v + (p[w * S] + p[(w + 4) * S]);
  } else {
    v = p[0];
#pragma unroll
    for (int w = 1; w < 4; w++) v = v + p[w * S];
  }
  return v;
}

template <class T, int MB, int NB, int EPI, int W, bool F16 = false, bool DMA = false>
__global__ __launch_bounds__(64 * W) void gemm_skinny_kernel(GemmArgs g) {
  using MF = Mfma<T>;
  typedef typename MF::frag frag;
  static_assert(!F16 || sizeof(T) == 2, "16 x 16 blocks: 16-bit operands");
  static_assert(!DMA || (W == 8 && (sizeof(T) == 4 || (F16 && MB == 1 && NB == 1))),
                "LDS operand path: 8 waves, fp32 or 16-bit 32 x 32 tiles");
  // DMA: each wave stages its K groups through a private LDS slab of two
  // slots, in fp32 one (a group's 16 MFMAs of 64 cycles cover the next one's
  // arrival, and at 64 KB two workgroups share a CU).
  // A group's 32 A rows and 32 B rows (128 bytes each) arrive by eight
  // wave-wide global->LDS loads, lane l carrying 16 bytes of row 8j + l/8, so
  // every row is read as one whole 128-byte segment (the register path's
  // lanes read 64-byte pieces of 16 rows per instruction); the fragments are
  // then read from LDS in the same layout the register path loads them in,
  // so both paths feed the MFMAs the same operands in the same order.
  constexpr int TR = 32 * MB, TC = 32 * NB, TE = TR * TC;
  constexpr int SLAB = (TR + TC) * 128;  // bytes of one group (its rows x 128 bytes)
  constexpr int SLOTS = sizeof(T) == 2 ? 2 : 1;
  // F16: the tile as 16 x 16 blocks of the 16 x 16 x 32 MFMA, whose operand
  // lanes read 64 contiguous bytes of a row (four lanes x 16 bytes) where the
  // 32 x 32 x 16 form reads 32 (two lanes): half the cache-line sectors per
  // load instruction.
  constexpr int BW = F16 ? 16 : 32;                  // block width
  constexpr int RB = 32 * MB / BW, CB = 32 * NB / BW;  // row / column blocks
  constexpr int NS = F16 ? 2 : 4;                    // MFMA k steps per 64-element group
  constexpr int NE = F16 ? 4 : 16;                   // accumulator elements per lane
  typedef float accv __attribute__((__vector_size__(NE * sizeof(float))));
  constexpr int NT = 64 * W;
  constexpr int VPL = 16 / (int)sizeof(T);  // elements per 16-byte load
  constexpr int GK = 8 * VPL;               // k elements per group
  static_assert(EPI != EPI_GEGLU_KEEP || NB == 2, "the kept pre-activation tile is 32 value + 32 gate columns");
  static_assert(EPI != EPI_GEGLU || NB <= 2, "GeGLU tiles");
  static_assert(W == 4 || W == 8, "wave count");
  // Partial tiles held in LDS at once: all W when they fit in 64 KB.
  constexpr bool FOLD = W == 8 && 8 * TE * 4 > 65536;
  constexpr int NP = FOLD ? 4 : W;
  // The fp32 epilogue works on items of FV floats, two when that gives every
  // thread one item; NQ items per thread.
  constexpr int FV = TE <= 2 * NT ? 2 : 4, TEV = TE / FV, NQ = (TEV + NT - 1) / NT;
  // The partial tiles; in DMA mode the same memory first holds the waves'
  // slabs (W x SLOTS groups), and a barrier separates the two uses.
  constexpr int RED = DMA && W * SLOTS * SLAB / 4 > NP * TE ? W * SLOTS * SLAB / 4 : NP * TE;
  __shared__ __attribute__((aligned(1024))) float red[RED];

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, lr = lane & 31, lh = lane >> 5;
  const int n0 = blockIdx.x * TC, m0 = blockIdx.y * TR;
  // Split-K (fp32 epilogue): blockIdx.z takes K elements [z*K, (z+1)*K) of A
  // and B and writes its own partial output, c_split elements further on.
  const int kz = blockIdx.z * g.K;

  // This lane's row (column) within a block and its first k element.
  const int brow = F16 ? (lane & 15) : lr, bk = F16 ? (lane >> 4) * VPL : lh * VPL;
  const T *ap[RB], *bp[CB];
#pragma unroll
  for (int i = 0; i < RB; i++) ap[i] = (const T *)g.A + (size_t)min(m0 + BW * i + brow, g.M - 1) * g.lda + kz + bk;
#pragma unroll
  for (int j = 0; j < CB; j++) {
    const int cc = BW * j + brow;  // tile column
    // GeGLU on 32-column tiles: the 64-row group n0 / 64 of the interleaved
    // weights holds 32 value rows then their 32 gate rows; tile half
    // (n0 / 32) % 2 takes value rows 16h .. 16h+15 as columns 0..15 and the
    // matching gate rows as columns 16..31, so the tile's outputs are the 16
    // columns n0 / 2 .. n0 / 2 + 15.
    const int row = (EPI == EPI_GEGLU && NB == 1)
                        ? (n0 & ~63) + (cc < 16 ? 0 : 32) + ((n0 >> 5) & 1) * 16 + (cc & 15)
                        : n0 + cc;
    bp[j] = (const T *)g.B + (size_t)row * g.ldb + kz + bk;
  }

  accv acc[RB][CB];
#pragma unroll
  for (int i = 0; i < RB; i++)
#pragma unroll
    for (int j = 0; j < CB; j++)
#pragma unroll
      for (int e = 0; e < NE; e++) acc[i][j][e] = 0.0f;
  // Tile element (row-major TR x TC) of accumulator element e of block (i, j).
  auto tile_at = [&](int i, int j, int e) {
    if constexpr (F16) return (BW * i + 4 * (lane >> 4) + e) * TC + BW * j + (lane & 15);
    else return (32 * i + mfma_row(e, lane)) * TC + 32 * j + lr;
  };

#define SKINNY_LOAD(XA, XB, GRP)                                                                   \
  do {                                                                                             \
    const int k_ = (GRP) * GK;                                                                     \
    _Pragma("unroll") for (int i = 0; i < RB; i++) _Pragma("unroll") for (int q = 0; q < NS; q++) \
        XA[i][q] = *(const uint4 *)(ap[i] + k_ + (GK / NS) * q);                                   \
    _Pragma("unroll") for (int j = 0; j < CB; j++) _Pragma("unroll") for (int q = 0; q < NS; q++) \
        XB[j][q] = *(const uint4 *)(bp[j] + k_ + (GK / NS) * q);                                   \
  } while (0)

  // One K group's MFMAs.
  auto mfma_group = [&](const uint4 (&la)[RB][NS], const uint4 (&lb)[CB][NS]) {
#pragma unroll
    for (int q = 0; q < NS; q++) {
      if constexpr (F16) {
#pragma unroll
        for (int i = 0; i < RB; i++)
#pragma unroll
          for (int j = 0; j < CB; j++)
            acc[i][j] = mma16x16<T>(__builtin_bit_cast(frag, la[i][q]), __builtin_bit_cast(frag, lb[j][q]), acc[i][j]);
      } else if constexpr (sizeof(T) == 2) {
#pragma unroll
        for (int i = 0; i < MB; i++)
#pragma unroll
          for (int j = 0; j < NB; j++)
            acc[i][j] = MF::mma(__builtin_bit_cast(frag, la[i][q]), __builtin_bit_cast(frag, lb[j][q]), acc[i][j]);
      } else {
#pragma unroll
        for (int e = 0; e < 4; e++)
#pragma unroll
          for (int i = 0; i < MB; i++)
#pragma unroll
            for (int j = 0; j < NB; j++) {
              const uint4 a4 = la[i][q], b4 = lb[j][q];
              const unsigned ua = e == 0 ? a4.x : e == 1 ? a4.y : e == 2 ? a4.z : a4.w;
              const unsigned ub = e == 0 ? b4.x : e == 1 ? b4.y : e == 2 ? b4.z : b4.w;
              acc[i][j] = MF::mma(__builtin_bit_cast(frag, ua), __builtin_bit_cast(frag, ub), acc[i][j]);
            }
      }
    }
  };

  const int ngrp = g.K / GK;
  uint4 la[RB][NS], lb[CB][NS];
  int grp = wave;
  if (!DMA && grp < ngrp) SKINNY_LOAD(la, lb, grp);
  // The fp32 epilogue's residual input, loaded now (behind the first operand
  // group) so its latency overlaps the main loop instead of following the
  // reduction; each element is read and then written by this thread only.
  fvec<FV> pre[NQ];
  const bool vec = (g.ldc & (FV - 1)) == 0;
  if constexpr (EPI == EPI_F32) {
    const float *R = g.res ? g.res : (const float *)g.C;
#pragma unroll
    for (int k = 0; k < NQ; k++) {
      pre[k] = 0.0f;
      const int q = tid + NT * k;
      const int r = q / (TC / FV), col = n0 + (q % (TC / FV)) * FV;
      if (g.accumulate && vec && q < TEV && m0 + r < g.M && col + FV <= g.n_store)
        pre[k] = *(const fvec<FV> *)(R + (size_t)(m0 + r) * g.ldc + col);
    }
  }
  if constexpr (DMA) {
    // Slab row r < TR is A row m0 + r, r >= TR the B row of tile column
    // r - TR (the mapping of bp above). DMA load j of a group fills slab
    // rows 8j .. 8j+7; lane l brings the 16-byte chunk (l % 8) ^ swz(row) of
    // row 8j + l / 8 into LDS slot l % 8 of that row, so a row's logical
    // chunk c sits in slot c ^ swz(row) (the XOR swizzle spreads the 16 rows
    // a quarter-wave reads over distinct banks).
    constexpr int LPG = (TR + TC) / 8;  // loads per group
    const int wv = __builtin_amdgcn_readfirstlane(wave);
    const char *dsrc[LPG];
#pragma unroll
    for (int j = 0; j < LPG; j++) {
      const int r = 8 * j + (lane >> 3);
      const int c = (lane & 7) ^ swz<128>(r);
      const T *row;
      if (r < TR) {
        row = (const T *)g.A + (size_t)min(m0 + r, g.M - 1) * g.lda;
      } else {
        const int cc = r - TR;
        const int br = (EPI == EPI_GEGLU && NB == 1)
                           ? (n0 & ~63) + (cc < 16 ? 0 : 32) + ((n0 >> 5) & 1) * 16 + (cc & 15)
                           : n0 + cc;
        row = (const T *)g.B + (size_t)br * g.ldb;
      }
      dsrc[j] = (const char *)(row + kz) + c * 16;
    }
    // The LDS reads are opaque to the compiler (lds_read8x16 / 4x16), so it
    // adds no waits of its own for the DMA: the vmcnt waits below are the only
    // ones.
    auto issue = [&](int gi, int slot) {
      char *dst = (char *)red + (wv * SLOTS + slot) * SLAB;
      const size_t kb = (size_t)gi * GK * sizeof(T);
#pragma unroll
      for (int j = 0; j < LPG; j++)
        __builtin_amdgcn_global_load_lds((gbl_void *)(dsrc[j] + kb), (lds_void *)(dst + j * 1024), 16, 0, 0);
    };
    // This wave's groups: wv, wv + W, ... (the register path's order).
    const int myn = wv < ngrp ? (ngrp - 1 - wv) / W + 1 : 0;
#pragma unroll
    for (int i = 0; i < SLOTS; i++)
      if (myn > i) issue(wv + i * W, i);
    for (int i = 0; i < myn; i++) {
      // Group i has landed once at most the next group's eight loads are
      // outstanding (the residual loads above are older and count as done).
      if (SLOTS == 2 && i + 1 < myn) wait_vmcnt<LPG>();
      else wait_vmcnt<0>();
      const char *sl = (const char *)red + (wv * SLOTS + i % SLOTS) * SLAB;
      // The register path's rows and k chunks for this lane. When the reads
      // return the fragments are in registers: the MFMAs may use them and the
      // slot can be refilled with group i + SLOTS.
      if constexpr (F16) {
        const char *fp[8];
        uint4 fr[8];
#pragma unroll
        for (int q = 0; q < NS; q++) {
          const int c = (lane >> 4) + 4 * q;
#pragma unroll
          for (int b = 0; b < 2; b++) {
            const int ra = 16 * b + (lane & 15), rb = 32 + ra;
            fp[4 * q + b] = sl + ra * 128 + ((c ^ swz<128>(ra)) << 4);
            fp[4 * q + 2 + b] = sl + rb * 128 + ((c ^ swz<128>(rb)) << 4);
          }
        }
        lds_read8x16(fp, fr);
#pragma unroll
        for (int q = 0; q < NS; q++)
#pragma unroll
          for (int b = 0; b < 2; b++) {
            la[b][q] = fr[4 * q + b];
            lb[b][q] = fr[4 * q + 2 + b];
          }
      } else {
#pragma unroll
        for (int b = 0; b < MB + NB; b++) {
          const int r = 32 * b + lr;
          const char *fp[4];
          uint4 fr[4];
#pragma unroll
          for (int q = 0; q < 4; q++) fp[q] = sl + r * 128 + (((lh + 2 * q) ^ swz<128>(r)) << 4);
          lds_read4x16(fp, fr);
#pragma unroll
          for (int q = 0; q < 4; q++) {
            if (b < MB) la[b < MB ? b : 0][q] = fr[q];
            else lb[b < MB ? 0 : b - MB][q] = fr[q];
          }
        }
      }
      if (i + SLOTS < myn) issue(wv + (i + SLOTS) * W, i % SLOTS);
      mfma_group(la, lb);
    }
    // Every load has landed and every wave is done with its slab before the
    // partial tiles reuse the memory.
    wait_vmcnt<0>();
    __syncthreads();
    grp = ngrp;  // the register loop below does nothing
  }
  for (; grp < ngrp; grp += W) {
    uint4 na[RB][NS], nb[CB][NS];
    const bool more = grp + W < ngrp;
    if (more) SKINNY_LOAD(na, nb, grp + W);
    mfma_group(la, lb);
    if (more) {
#pragma unroll
      for (int i = 0; i < RB; i++)
#pragma unroll
        for (int q = 0; q < NS; q++) la[i][q] = na[i][q];
#pragma unroll
      for (int j = 0; j < CB; j++)
#pragma unroll
        for (int q = 0; q < NS; q++) lb[j][q] = nb[j][q];
    }
  }
#undef SKINNY_LOAD

  // Reduce the W partial tiles (row-major TR x TC) in a fixed order:
  // (p0 + p4) + (p1 + p5) + (p2 + p6) + (p3 + p7) with 8 waves, p0 + p1 + p2 +
  // p3 with 4. When the eight partials fit in LDS every wave stores its own
  // and one barrier follows; otherwise waves 4..7 fold theirs into waves 0..3
  // first. Each epilogue thread then sums only the elements it stores.
  if constexpr (FOLD) {
    if (wave >= 4) {
      float *mine = red + (wave - 4) * TE;
#pragma unroll
      for (int i = 0; i < RB; i++)
#pragma unroll
        for (int j = 0; j < CB; j++)
#pragma unroll
          for (int e = 0; e < NE; e++) mine[tile_at(i, j, e)] = acc[i][j][e];
    }
    __syncthreads();
    if (wave < 4) {
      const float *theirs = red + wave * TE;
#pragma unroll
      for (int i = 0; i < RB; i++)
#pragma unroll
        for (int j = 0; j < CB; j++)
#pragma unroll
          for (int e = 0; e < NE; e++) acc[i][j][e] += theirs[tile_at(i, j, e)];
    }
    __syncthreads();
  }
  if (wave < NP) {
    float *mine = red + wave * TE;
#pragma unroll
    for (int i = 0; i < RB; i++)
#pragma unroll
      for (int j = 0; j < CB; j++)
#pragma unroll
        for (int e = 0; e < NE; e++) mine[tile_at(i, j, e)] = acc[i][j][e];
  }
  __syncthreads();
  if constexpr (EPI == EPI_F32) {
    float *C = (float *)g.C + blockIdx.z * g.c_split;
#pragma unroll
    for (int k = 0; k < NQ; k++) {
      const int q = tid + NT * k;
      if (q >= TEV) break;
      const int r = q / (TC / FV), c = (q % (TC / FV)) * FV, col = n0 + c;
      if (m0 + r >= g.M || col >= g.n_store) continue;
      const fvec<FV> v = partial_sum<FV, NP, TE>(red, r * TC + c);
      float *p = C + (size_t)(m0 + r) * g.ldc + col;
      if (vec && col + FV <= g.n_store) {
        *(fvec<FV> *)p = pre[k] + v;
      } else {
        const float *pr = (g.res ? g.res : C) + (size_t)(m0 + r) * g.ldc + col;  // residual input
        for (int u = 0; u < FV && col + u < g.n_store; u++) p[u] = g.accumulate ? pr[u] + v[u] : v[u];
      }
    }
  } else {
    auto emit = [&](auto gated, T *C, int ldo) {
      constexpr bool G = decltype(gated)::value;
      constexpr int OC = G ? TC / 2 : TC;  // output columns of the tile
      // Elements per thread item: 16-bit types down to 2 (a 4-byte store) so
      // that every thread has an item; fp32 4 (16 bytes).
      constexpr int EPV = sizeof(T) == 4 ? 4 : TR * OC >= 8 * NT ? 8 : TR * OC >= 4 * NT ? 4 : 2;
      constexpr int RV = EPV > 4 ? 4 : EPV;  // partial-sum vector width
      const int oc0 = G ? n0 / 2 : n0;
      for (int q = tid; q < TR * (OC / EPV); q += NT) {
        const int r = q / (OC / EPV), c = (q % (OC / EPV)) * EPV;
        if (m0 + r >= g.M) continue;
        float val[EPV], gate[EPV];
#pragma unroll
        for (int h = 0; h < EPV / RV; h++) {
          const fvec<RV> v = partial_sum<RV, NP, TE>(red, r * TC + c + RV * h);
#pragma unroll
          for (int u = 0; u < RV; u++) val[RV * h + u] = v[u];
          if constexpr (G) {
            const fvec<RV> x = partial_sum<RV, NP, TE>(red, r * TC + TC / 2 + c + RV * h);
#pragma unroll
            for (int u = 0; u < RV; u++) gate[RV * h + u] = x[u];
          }
        }
        float o[EPV];
#pragma unroll
        for (int u = 0; u < EPV; u++) {
          if constexpr (!G) {
            o[u] = val[u];
          } else {
            o[u] = gelu_erf<T>(val[u]) * gate[u];
          }
        }
        T *dst = C + (size_t)(m0 + r) * ldo + oc0 + c;
        if constexpr (sizeof(T) == 2) {
          unsigned w[EPV / 2];
#pragma unroll
          for (int u = 0; u < EPV / 2; u++) w[u] = pack16<T>(o[2 * u], o[2 * u + 1]);
          if constexpr (EPV == 8) *(uint4 *)dst = make_uint4(w[0], w[1], w[2], w[3]);
          else if constexpr (EPV == 4) *(uint2 *)dst = make_uint2(w[0], w[1]);
          else *(unsigned *)dst = w[0];
        } else {
          *(float4 *)dst = make_float4(o[0], o[1], o[2], o[3]);
        }
      }
    };
    if constexpr (EPI == EPI_STORE) {
      emit(std::false_type{}, (T *)g.C, g.ldc);
    } else if constexpr (EPI == EPI_GEGLU) {
      emit(std::true_type{}, (T *)g.C, g.ldc);
    } else {
      emit(std::false_type{}, (T *)g.C, g.ldc);
      emit(std::true_type{}, (T *)g.C2, g.ldc2);
    }
  }
}

// bf16 32 x 32 tiles run as 16 x 16 x 32 MFMA blocks (cfg5 0.7165 -> 0.7055
// ms); the 64-row and 64-column tiles of 112-row batches were slower that
// way (0.860 -> 0.868 ms) and keep 32 x 32 x 16.
template <class T, int MB, int NB, int W>
hipError_t launch_skinny_cfg(int epi, const GemmArgs &a, hipStream_t s, int splits = 1) {
  constexpr bool F = sizeof(T) == 2 && MB == 1 && NB == 1;
  // The LDS operand path exists for these tiles.
  constexpr bool D = W == 8 && (std::is_same<T, float>::value || (MB == 1 && NB == 1));
  dim3 grid(a.N / (32 * NB), (a.M + 32 * MB - 1) / (32 * MB), splits), block(64 * W);
  auto go = [&](auto e) {
    constexpr int E = decltype(e)::value;
    if constexpr (D && std::is_same<T, float>::value) {
      hipLaunchKernelGGL((gemm_skinny_kernel<T, MB, NB, E, W, F, true>), grid, block, 0, s, a);
    } else if constexpr (D) {
      if (a.skinny_regs) hipLaunchKernelGGL((gemm_skinny_kernel<T, MB, NB, E, W, F>), grid, block, 0, s, a);
      else hipLaunchKernelGGL((gemm_skinny_kernel<T, MB, NB, E, W, F, true>), grid, block, 0, s, a);
    } else {
      hipLaunchKernelGGL((gemm_skinny_kernel<T, MB, NB, E, W, F>), grid, block, 0, s, a);
    }
  };
  switch (epi) {
    case EPI_F32:
      if constexpr (NB == 1 || std::is_same<T, float>::value) go(std::integral_constant<int, EPI_F32>{});
      else return hipErrorInvalidValue;
      break;
    case EPI_STORE:
      if constexpr (NB == 1 || std::is_same<T, float>::value) go(std::integral_constant<int, EPI_STORE>{});
      else return hipErrorInvalidValue;
      break;
    case EPI_GEGLU:
      if constexpr (MB == 1 || std::is_same<T, float>::value) go(std::integral_constant<int, EPI_GEGLU>{});
      else return hipErrorInvalidValue;
      break;
    default:
      if constexpr (NB == 2 && !std::is_same<T, f16>::value) go(std::integral_constant<int, EPI_GEGLU_KEEP>{});
      else return hipErrorInvalidValue;
      break;
  }
  return hipGetLastError();
}

// Tile choice, 8 waves: 32-row tiles up to 128 rows while the grid fits one
// workgroup per CU (more workgroups for the few rows: cfg5 1.10 -> 0.92 ms,
// cfg2 1.18 -> 1.06 ms against 64-row tiles everywhere), 64-row tiles
// otherwise; 32 columns, or for GeGLU 32 (16 value + 16 gate rows) or 64
// (32 + 32; training's kept pre-activation always). fp32: 32 x 32 at any row
// count, operands through LDS.
template <class T>
hipError_t launch_skinny(int epi, const GemmArgs &a, hipStream_t s) {
  constexpr bool f32 = std::is_same<T, float>::value;
  if (epi == EPI_GEGLU_KEEP) {
    if (a.M <= 128) return launch_skinny_cfg<T, 1, 2, 8>(epi, a, s);
    return launch_skinny_cfg<T, 2, 2, 8>(epi, a, s);
  }
  // 32 x 32 tiles while their grid fits one workgroup per CU (MI355X: 256):
  // QKV at 112 rows as 144 workgroups of 64 rows instead of 288 took cfg2 0.917
  // -> 0.901 ms, GeGLU on 32-column tiles there 0.932 -> 0.951 ms (cfg5 0.809
  // -> 0.789 ms).
  if constexpr (f32) {
    // A CU's time is its 32 x 32 blocks of the busiest round; 32 x 64 tiles
    // read a third less for the same blocks, so they are taken where they do
    // not add any (K = 768, N = 2304, us, 32 x 32 / 32 x 64 / the register
    // path: 203 rows 15.3 / 13.7 / 15.7, 300 rows 20.8 / 22.7 / 20.8, 512 rows
    // 29.5 / 31.2 / 30.7; N = 768: 203 rows 7.4 / 12.0 / 13.2, 512 rows 13.8 /
    // 12.2 / 13.6, 1,472 rows 28.8 / 32.2 / 101.7 on 256 x 128 tiles).
    // Longer K past one round: workgroups that share a CU cover each other's
    // loads, and the operands go straight into registers, on 64 x 32 tiles where
    // those take half the rounds, else 32 x 32 (us, 32 x 32 and 32 x 64 through
    // LDS / 32 x 32 and 64 x 32 in registers: 512 x 768 x 1152 20.8, 20.2 / 20.1,
    // 17.8; 203 x 2304 x 1152 20.7, 20.2 / 20.2, 26.1; 1,000 x 768 x 1152 30.2,
    // 35.4 / 29.1, 33.5; 1,000 x 1024 x 2304 77.7, 70.8 / 67.7, 58.2; 777 x 2304 x
    // 2304 142, 129 / 125, 114; 900 x 768 x 4096 102, 116 / 89, 95), at K = 1024
    // only in one round of the 64 x 32 ones (512 x 1024 18.6, 16.9 / 18.3, 16.6;
    // 1,300 x 1024 44.8, 43.1 / 45.6, 46.1).
    const int c32 = (a.N / 32) * ((a.M + 31) / 32), c64 = c32 / 2;
    const int r32 = (c32 + kCUs - 1) / kCUs, r64 = (c64 + kCUs - 1) / kCUs;
    if (epi == EPI_F32 && a.K > 768 && r32 > 1) {
      const dim3 tall(a.N / 32, (a.M + 63) / 64), square(a.N / 32, (a.M + 31) / 32);
      const int rtall = ((int)(tall.x * tall.y) + kCUs - 1) / kCUs;
      if (2 * rtall <= r32 && (rtall == 1 || a.K >= 1152)) {
        hipLaunchKernelGGL((gemm_skinny_kernel<float, 2, 1, EPI_F32, 8>), tall, dim3(512), 0, s, a);
        return hipGetLastError();
      }
      if (a.K >= 1152) {
        hipLaunchKernelGGL((gemm_skinny_kernel<float, 1, 1, EPI_F32, 8>), square, dim3(512), 0, s, a);
        return hipGetLastError();
      }
    }
    if (2 * r64 <= r32) return launch_skinny_cfg<T, 1, 2, 8>(epi, a, s);
  }
  if (f32 || (a.N / 32) * ((a.M + 31) / 32) <= 256) return launch_skinny_cfg<T, 1, 1, 8>(epi, a, s);
  if constexpr (!f32) {
    if (epi == EPI_GEGLU) return launch_skinny_cfg<T, 1, 2, 8>(epi, a, s);
    return launch_skinny_cfg<T, 2, 1, 8>(epi, a, s);
  }
  return hipErrorInvalidValue;
}

// Small-M split-K: a workgroup's time grows with the K it streams (~3.4 ns
// per K element at M = 64 on top of ~2.1 us, whatever the grid), so K is
// split over `splits` workgroups per tile, each writing an fp32 partial tile
// into partial[z][M x N]; the consumer sums them.
template <class T>
hipError_t launch_skinny_split(const GemmArgs &a0, int splits, float *partial, hipStream_t s) {
  GemmArgs a = a0;
  a.K = a0.K / splits;
  a.C = partial;
  a.res = nullptr;
  a.ldc = a0.N;
  a.n_store = a0.N;
  a.accumulate = 0;
  a.c_split = (size_t)a0.M * a0.N;
  return launch_skinny_cfg<T, 1, 1, 8>(EPI_F32, a, s, splits);
}

// C (+)= sum over splits of part[s * n + i], in split order; four
// consecutive elements per thread (n % 4 == 0), every split's load issued
// before the sum.
__global__ void splitk_reduce_kernel(const float *part, int splits, size_t n, float *C, int accumulate) {
  const size_t i = ((size_t)blockIdx.x * blockDim.x + threadIdx.x) * 4;
  if (i >= n) return;
  constexpr int MAXS = 16;
  float4 p[MAXS];
#pragma unroll
  for (int s = 0; s < MAXS; s++)
    if (s < splits) p[s] = *(const float4 *)(part + (size_t)s * n + i);
  float4 acc = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll
  for (int s = 0; s < MAXS; s++)
    if (s < splits) acc = make_float4(acc.x + p[s].x, acc.y + p[s].y, acc.z + p[s].z, acc.w + p[s].w);
  if (accumulate) {
    const float4 c = *(const float4 *)(C + i);
    acc = make_float4(c.x + acc.x, c.y + acc.y, c.z + acc.z, c.w + acc.w);
  }
  *(float4 *)(C + i) = acc;
}

}  // namespace

hipError_t launch_gemm_small_split(int precision, const GemmArgs &a, int splits, float *partial, hipStream_t s) {
  if (a.M <= 0) return hipSuccess;
  const int kt = prec16(precision) ? 64 : 32;
  if (a.M > 128 || splits < 1 || a.K % (splits * kt) != 0 || a.N % 128 != 0) return hipErrorInvalidValue;
  return precision == PREC_BF16  ? launch_skinny_split<bf16>(a, splits, partial, s)
         : precision == PREC_F16 ? launch_skinny_split<f16>(a, splits, partial, s)
                                 : launch_skinny_split<float>(a, splits, partial, s);
}

// Rows of B come in 128s (every tile width used divides N or is chosen only
// where it does); K is staged 64 or 128 bytes per step.
bool gemm_shape_ok(int precision, int N, int K) {
  const int kt = prec16(precision) ? 64 : 32;
  return N > 0 && K > 0 && N % 128 == 0 && K % kt == 0;
}

bool gemm_epi_ok(int precision, int epi, int M) {
  if (epi >= EPI_F32_LN) return prec16(precision) && M > 128;
  if (epi != EPI_GEGLU_BWD) return true;
  return prec16(precision) ? M > 128 : M > 1024;
}

bool gemm_ln_fold_ok(int precision, int M, int hidden, int inter) {
  // fp16 folds above 1,024 rows only. (x - m) * w is not scaled by the row, so
  // it leaves fp16's range where a residual value times a norm weight does; the
  // normalised row (at most sqrt(768) |w|) does not. A single request keeps
  // that range: 512 tokens 991 us instead of 924.
  return prec16(precision) && M > (precision == PREC_F16 ? 1024 : 128) && hidden == kLnHidden && inter > 0 &&
         inter % 64 == 0;
}

// Any-shape GEMM (model geometries the MFMA kernels do not tile): thread n of
// block (x, m) computes output element (m, 256 x + n) as an fp32 dot product
// over K in order, then the epilogue. Performance is not its purpose.
template <class T, int EPI>
__global__ __launch_bounds__(256) void gemm_generic_kernel(GemmArgs g) {
  const int m = blockIdx.y, n = blockIdx.x * 256 + threadIdx.x;
  const int ncols = EPI == EPI_GEGLU ? g.N / 2 : g.N;
  if (m >= g.M || n >= ncols) return;
  const T *a = (const T *)g.A + (size_t)m * g.lda;
  auto dot = [&](int row) {
    const T *b = (const T *)g.B + (size_t)row * g.ldb;
    float acc = 0.0f;
    for (int k = 0; k < g.K; k++) acc = fmaf((float)a[k], (float)b[k], acc);
    return acc;
  };
  if constexpr (EPI == EPI_F32) {
    if (n >= g.n_store) return;
    const float v = dot(n);
    float *C = (float *)g.C + (size_t)m * g.ldc + n;
    const float *R = g.res ? g.res + (size_t)m * g.ldc + n : C;
    *C = g.accumulate ? *R + v : v;
  } else if constexpr (EPI == EPI_STORE) {
    ((T *)g.C)[(size_t)m * g.ldc + n] = to_elem<T>(dot(n));
  } else {
    const float v = dot(n), gate = dot(ncols + n);
    ((T *)g.C)[(size_t)m * g.ldc + n] = to_elem<T>(gelu_erf<T>(v) * gate);
  }
}

template <class T>
hipError_t launch_gemm_generic_t(int epi, const GemmArgs &a, hipStream_t s) {
  const int ncols = epi == EPI_GEGLU ? a.N / 2 : a.N;
  const dim3 grid((ncols + 255) / 256, a.M), block(256);
  switch (epi) {
    case EPI_F32: hipLaunchKernelGGL((gemm_generic_kernel<T, EPI_F32>), grid, block, 0, s, a); break;
    case EPI_STORE: hipLaunchKernelGGL((gemm_generic_kernel<T, EPI_STORE>), grid, block, 0, s, a); break;
    case EPI_GEGLU: hipLaunchKernelGGL((gemm_generic_kernel<T, EPI_GEGLU>), grid, block, 0, s, a); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_gemm_generic(int precision, int epi, const GemmArgs &a, hipStream_t s) {
  if (a.M <= 0) return hipSuccess;
  if (a.N <= 0 || a.K <= 0 || (epi == EPI_GEGLU && a.N % 2)) return hipErrorInvalidValue;
  return precision == PREC_BF16  ? launch_gemm_generic_t<bf16>(epi, a, s)
         : precision == PREC_F16 ? launch_gemm_generic_t<f16>(epi, a, s)
                                 : launch_gemm_generic_t<float>(epi, a, s);
}

// fp32-output tiles (the residual GEMMs, input and weight gradients): the
// smallest tile whose grid is one round of the 256 CUs, since a launch takes
// about as long as one workgroup and that is its K loop's length times its
// tile. Measured on isolated launches with weights rotated past L2 (us, K =
// 768 / 1152 / 2304, N = 768), each beside the tile it replaced there:
//   64 x 64   600 rows   5.8 /  7.1 / 10.2  (64 x 128, four waves:  8.2 /  9.6 / 14.4)
//   64 x 128  2,046      8.1 /  9.4 / 16.2  (64 x 192:             11.5 / 13.7 / 22.8)
//   128 x 128 3,840     11.6 / 13.7 / 23.4  (64 x 192:             12.8 / 15.3 / 24.7)
//   64 x 256  5,400     13.9 / 17.0 / 29.5  (256 x 192:            25.1 / 31.8 / 56.5)
//   128 x 192 8,192     18.6 / 22.6 / 36.0  (256 x 192:            26.2 / 33.2 / 60.2)
//   256 x 192 16,000    33.3 / 42.8 / 73.6  (128 x 192, two rounds: 34.3 / 45.7 / 74.8)
// The first four hold a stage's operands in registers (PF): without it 64 x
// 64 took 6.9 / 8.7 / 13.2 us at 512 rows. 256 x 192 (eight waves of 64 x 96,
// one workgroup per CU) stages the fewest operand bytes per output.
typedef Tile<64, 64, 128, 5, 2, 2, 2, true> F64x64;
typedef Tile<64, 128, 128, 5, 1, 2, 4, true> F64x128;
typedef Tile<128, 128, 128, 4, 1, 4, 2, true> F128x128;
typedef Tile<64, 256, 128, 4, 1, 2, 4, true> F64x256;
typedef Tile<128, 192, 128, 3, 1, 4, 2> F128x192;
typedef Tile<256, 192, 128, 2, 2, 4, 2> F256x192;
typedef Tile<128, 128, 64, 3, 3, 2, 2> F128x128s;  // large outputs of other widths

template <class T>
hipError_t launch_f32(const GemmArgs &a, hipStream_t s) {
  if (F64x64::count(a) <= kCUs) return launch_tile<T, F64x64, EPI_F32>(a, s);
  if (F64x128::count(a) <= kCUs) return launch_tile<T, F64x128, EPI_F32>(a, s);
  if (F128x128::count(a) <= kCUs) return launch_tile<T, F128x128, EPI_F32>(a, s);
  if (a.N % 256 == 0 && F64x256::count(a) <= kCUs) return launch_tile<T, F64x256, EPI_F32>(a, s);
  if (a.N % 192) return launch_tile<T, F128x128s, EPI_F32>(a, s);
  if (F128x192::count(a) <= kCUs) return launch_tile<T, F128x192, EPI_F32>(a, s);
  return launch_tile<T, F256x192, EPI_F32>(a, s);
}

// Operand-type outputs (store, GeGLU, its backward and the folded-LayerNorm
// forms), by the same rule; past the largest one-round tile, 256 x 128 tiles at
// two workgroups per CU, whose epilogues and DMA stalls overlap the other's
// MFMAs. N = 2304, K = 768, store / GeGLU, isolated launches as above (us):
//   64 x 64 (two waves)  208 rows  5.8 /  6.1  (64 x 128:  6.8 /  7.1)
//   128 x 64             600       7.0 /  7.4  (64 x 128:  8.1 /  8.5)
//   128 x 128, 8 waves 1,500       9.4 /  9.8  (128 x 128, 64-byte stages: 12.5 / 13.0)
//   192 x 128          2,046      12.6 / 13.3  (256 x 128, 8 waves: 14.4 / 15.6)
//   256 x 128, 8 waves 3,000      16.3 / 17.0  (128 x 128, 64-byte stages: 19.3 / 19.9)
//   192 x 256          3,840      21.8 / 23.7  (128 x 128, 64-byte stages: 26.1 / 26.5)
//                      5,376      24.0 / 25.6  (256 x 128, two per CU: 27.9 / 28.9)
//   256 x 256          7,000      30.4 / 31.0  (256 x 128, two per CU: 32.2 / 34.2)
// N = 768, store, K = 768 / 2304: 192 x 256 at 16,000 rows 23.2 / 55.2 (256 x 256
// 24.1 / 60.5, 128 x 128 with 64-byte stages 27.3 / 76.2), 256 x 256 at 21,000 rows
// 28.5 / 67.0 (35.8 / 93.2).
// At 64 x 64 the line lies at 224 workgroups (64 x 64 / 128 x 64: N = 2304, 317
// rows 6.1 / 6.5, 381 rows, 216 of them, 6.4 / 6.6, 448 rows, 252, 7.2 / 6.8; K =
// 1152, 381 rows 7.5 / 7.8; N = 1536, 573 rows 6.3 / 6.6; N = 768, 957 rows 5.7 /
// 6.5, K = 2304 10.1 / 12.7).
typedef Tile<64, 64, 128, 5, 1, 2, 1, true> S64x64;
typedef Tile<128, 64, 128, 4, 1, 4, 1, true> S128x64;
typedef Tile<128, 128, 128, 4, 1, 4, 2, true> S128x128;
typedef Tile<192, 128, 128, 3, 1, 2, 2> S192x128;
typedef Tile<256, 128, 128, 3, 1, 4, 2> S256x128;
typedef Tile<192, 256, 128, 2, 2, 2, 4> S192x256;
typedef Tile<256, 256, 64, 5, 2, 2, 4, true> S256x256;
typedef Tile<128, 128, 64, 3, 3, 2, 2> S128x128s;
typedef Tile<256, 128, 64, 3, 2, 2, 2> S256x128s;

template <class T, int EPI, int PC = 0>
hipError_t launch_store(const GemmArgs &a, hipStream_t s, const LnFold *ln = nullptr) {
  constexpr bool gated = EPI == EPI_GEGLU || EPI == EPI_GEGLU_KEEP || EPI == EPI_GEGLU_LN;
  if constexpr (PC != kLnPartWide) {
    if (S64x64::count(a) <= kCUs * 7 / 8) return launch_tile<T, S64x64, EPI, PC>(a, s, ln);
    if (S128x64::count(a) <= kCUs) return launch_tile<T, S128x64, EPI, PC>(a, s, ln);
    if (S128x128::count(a) <= kCUs) return launch_tile<T, S128x128, EPI, PC>(a, s, ln);
    if (S192x128::count(a) <= kCUs) return launch_tile<T, S192x128, EPI, PC>(a, s, ln);
    if (S256x128::count(a) <= kCUs) return launch_tile<T, S256x128, EPI, PC>(a, s, ln);
  }
  if (a.N % 256 == 0 && S192x256::count(a) <= kCUs) return launch_tile<T, S192x256, EPI, PC>(a, s, ln);
  if constexpr (EPI == EPI_STORE || EPI == EPI_GEGLU)
    if (a.N % 256 == 0 && S256x256::count(a) <= kCUs) return launch_tile<T, S256x256, EPI, PC>(a, s, ln);
  if (a.M <= (gated ? 8192 : 4096)) return launch_tile<T, S128x128s, EPI, PC>(a, s, ln);
  return launch_tile<T, S256x128s, EPI, PC>(a, s, ln);
}

// The folded-LayerNorm forms. The statistics' parts are kLnPartNarrow columns
// for forwards of up to kLnNarrowTokens tokens (the residual tiles of one
// round there are 64 and 128 columns wide), else kLnPartWide (192-column
// tiles, a third of the pairs for the consumers' 18 N-tiles to re-read).
template <class T>
hipError_t launch_fold(int epi, const GemmArgs &a, const LnFold *ln, hipStream_t s) {
  if (!ln || !ln->lpart) return hipErrorInvalidValue;
  const bool narrow = ln->lparts == kLnHidden / kLnPartNarrow;
  if (!narrow && ln->lparts != kLnHidden / kLnPartWide) return hipErrorInvalidValue;
  if (epi == EPI_F32_LN) {
    if (a.N != kLnHidden || !a.accumulate || a.ldc % 4 || a.n_store != a.N || !ln->fx || !ln->lw)
      return hipErrorInvalidValue;
    if (narrow) {
      if (F64x64::count(a) <= kCUs) return launch_tile<T, F64x64, EPI_F32_LN, kLnPartNarrow>(a, s, ln);
      if (F64x128::count(a) <= kCUs) return launch_tile<T, F64x128, EPI_F32_LN, kLnPartNarrow>(a, s, ln);
      return launch_tile<T, F128x128, EPI_F32_LN, kLnPartNarrow>(a, s, ln);
    }
    if (F128x192::count(a) <= kCUs) return launch_tile<T, F128x192, EPI_F32_LN, kLnPartWide>(a, s, ln);
    return launch_tile<T, F256x192, EPI_F32_LN, kLnPartWide>(a, s, ln);
  }
  if (a.K != kLnHidden || !ln->lcs || !ln->mean_out) return hipErrorInvalidValue;
  if (epi == EPI_STORE_LN)
    return narrow ? launch_store<T, EPI_STORE_LN, kLnPartNarrow>(a, s, ln)
                  : launch_store<T, EPI_STORE_LN, kLnPartWide>(a, s, ln);
  return narrow ? launch_store<T, EPI_GEGLU_LN, kLnPartNarrow>(a, s, ln)
                : launch_store<T, EPI_GEGLU_LN, kLnPartWide>(a, s, ln);
}

template <class T>
hipError_t launch_gemm16(int epi, const GemmArgs &a, hipStream_t s, const LnFold *ln) {
  switch (epi) {
    case EPI_F32: return launch_f32<T>(a, s);
    case EPI_STORE: return launch_store<T, EPI_STORE>(a, s);
    case EPI_GEGLU: return launch_store<T, EPI_GEGLU>(a, s);
    case EPI_F32_LN: case EPI_STORE_LN: case EPI_GEGLU_LN: return launch_fold<T>(epi, a, ln, s);
  }
  if constexpr (std::is_same<T, bf16>::value) {  // training: bf16 only
    if (epi == EPI_GEGLU_KEEP) return launch_store<T, EPI_GEGLU_KEEP>(a, s);
    if (epi == EPI_GEGLU_BWD) return launch_store<T, EPI_GEGLU_BWD>(a, s);
  }
  return hipErrorInvalidValue;
}

// fp32 on the whole-K kernel (32 x 32 tiles, K split over eight waves, also
// the smaller summation error: 1.8e-7 of the result against 5e-7) or on 256 x
// 128 tiles, of which a round takes about as long as 20 rounds of 32 x 32 ones
// on the 256 CUs (K = 768, N = 2304: 1,472 rows 70 against 104 us, 2,048 rows
// 95 / 105, 3,000 rows 135 / 105, 4,000 rows 178 / 205; N = 768, 4,000 rows 64 /
// 104), for longer K 18 (K = 1152, 1,700 rows 130 / 149, 2,200 rows 163 / 151; K =
// 1536, 2,200 rows 204 / 197). A forward of 8,192 tokens or more runs as two
// parts that share the CUs, where CU time counts and the large tiles take three
// fifths of the small ones' (N = 768 on small / large: 4 x 2,800 tokens 34.9 /
// 33.1 ms, 11 x 1,000 29.8 / 26.7, 26 x 512 31.4 / 29.2). The two sum in
// different orders, so a forward chooses by the whole batch's rows, in parts or
// not.
constexpr int kF32SharedRows = 8192;
bool f32_small_tiles(int epi, const GemmArgs &a) {
  if (epi == EPI_GEGLU_BWD) return false;
  if (epi == EPI_GEGLU_KEEP) return a.M <= 1024;
  if (a.rows >= kF32SharedRows) return false;
  const long long M = a.rows ? a.rows : a.M;
  const long long r32 = ((M + 31) / 32 * (a.N / 32) + kCUs - 1) / kCUs;
  const long long rt = ((M + 255) / 256 * (a.N / 128) + kCUs - 1) / kCUs;
  return M <= 1024 || r32 <= (a.K > 768 ? 18 : 20) * rt;
}

template <class C>
hipError_t launch_gemm_f32_tile(int epi, const GemmArgs &a, hipStream_t s) {
  switch (epi) {
    case EPI_F32: return launch_tile<float, C, EPI_F32>(a, s);
    case EPI_STORE: return launch_tile<float, C, EPI_STORE>(a, s);
    case EPI_GEGLU: return launch_tile<float, C, EPI_GEGLU>(a, s);
    case EPI_GEGLU_KEEP: return launch_tile<float, C, EPI_GEGLU_KEEP>(a, s);
    case EPI_GEGLU_BWD: return launch_tile<float, C, EPI_GEGLU_BWD>(a, s);
  }
  return hipErrorInvalidValue;
}

hipError_t launch_gemm(int precision, int epi, const GemmArgs &a, hipStream_t s, const LnFold *ln) {
  if (a.M <= 0) return hipSuccess;
  if (!gemm_epi_ok(precision, epi, a.M) || (epi == EPI_GEGLU_BWD && (!a.gin || a.ldc % 8))) return hipErrorInvalidValue;
  // Small M goes to the whole-K kernel.
  if (a.M <= 128)
    return precision == PREC_BF16  ? launch_skinny<bf16>(epi, a, s)
           : precision == PREC_F16 ? launch_skinny<f16>(epi, a, s)
                                   : launch_skinny<float>(epi, a, s);
  if (precision == PREC_BF16) return launch_gemm16<bf16>(epi, a, s, ln);
  if (precision == PREC_F16) return launch_gemm16<f16>(epi, a, s, ln);
  if (f32_small_tiles(epi, a)) return launch_skinny<float>(epi, a, s);
  return launch_gemm_f32_tile<Tile<256, 128, 128, 3, 1, 2, 2>>(epi, a, s);
}

// Weight gradients: C (+)= A . B^T over the tokens (K) in `splits` partial
// sums added in order. They run on the side stream beside the input-gradient
// chain, so what they cost is the CU time they hold, not their own latency:
// in bf16 a 128 x 128 tile walks its splits one after the other (half the
// operand bytes per output of 64 x 128 tiles, and no partial outputs to write
// and read; dWqkv at 3840 tokens: 108 workgroups for 25 us against 216 for 21
// us; the backward of a step of 32 x 384 tokens in four micro-batches over 22
// layers 22.7 -> 21.7 ms). Fewer than 32 such tiles (hidden sizes below 768)
// would leave the side stream behind the chain and stay split over workgroups.
static bool wgrad_walks_splits(int precision, int M, int N) {
  GemmArgs a{};
  a.M = M;
  a.N = N;
  return precision == PREC_BF16 && F128x128::count(a) >= 32;
}

size_t gemm_wgrad_partial(int precision, int M, int N, int splits) {
  return splits == 1 || wgrad_walks_splits(precision, M, N) ? 0 : (size_t)splits * M * N;
}

hipError_t launch_gemm_wgrad(int precision, const GemmArgs &a0, int splits, float *partial, hipStream_t s) {
  if (a0.M <= 0) return hipSuccess;
  if (precision == PREC_F16) return hipErrorInvalidValue;  // training only
  if (splits < 1 || splits > 16 || a0.K % (splits * 64) != 0 || a0.N % 128 != 0) return hipErrorInvalidValue;
  GemmArgs a = a0;
  a.ldc = a0.N;
  a.n_store = a0.N;
  if (wgrad_walks_splits(precision, a.M, a.N)) {
    typedef F128x128 C;
    if (splits == 1) return launch_tile<bf16, C, EPI_F32>(a, s);
    hipLaunchKernelGGL((gemm_nt_seg_kernel<bf16, C::BM, C::BN, C::RB, C::NSTAGE, C::WPE, C::WGM, C::WGN>),
                       dim3(C::count(a)), dim3(64 * C::WGM * C::WGN), 0, s, a, a.K / splits / 64);
    return hipGetLastError();
  }
  if (splits == 1) return launch_gemm(precision, EPI_F32, a, s);
  a.K = a0.K / splits;
  a.C = partial;
  a.accumulate = 0;
  a.c_split = (size_t)a0.M * a0.N;
  const hipError_t e = precision == PREC_BF16
                           ? launch_tile<bf16, F64x128, EPI_F32>(a, s, nullptr, splits)
                           : launch_tile<float, Tile<128, 128, 128, 3, 1, 2, 2>, EPI_F32>(a, s, nullptr, splits);
  if (e != hipSuccess) return e;
  const size_t n = (size_t)a0.M * a0.N;
  hipLaunchKernelGGL(splitk_reduce_kernel, dim3((unsigned)((n / 4 + 255) / 256)), dim3(256), 0, s, partial, splits,
                     n, (float *)a0.C, a0.accumulate);
  return hipGetLastError();
}
