// The outer-product MFMA pipeline shared by the full-weight kernels: operand
// tiles of G and X staged by buffer loads straight into a ring of LDS stages,
// consumed by bf16 MFMA 16x16x32 into per-wave accumulator blocks.
//
// Included inside an anonymous namespace by each kernel source, after
// odp_internal.h.  The tile shape comes from macros a source may set before
// the include: ODP_LIN_OM x ODP_LIN_ON output tile (default 256 x 256),
// ODP_LIN_WAVES waves (default 8), ODP_LIN_RING stages (default 4),
// ODP_LIN_OCC waves per SIMD (default 2).  Each source thereby compiles its
// own copy of the pipeline for its own tile.
#pragma once

typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
// The same 16 bytes read from memory last written as other types (a tile
// staged element by element in LDS): may_alias keeps the compiler from
// moving the read above those writes.
typedef u32x4_t u32x4_alias_t __attribute__((may_alias));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
typedef u32x2_t u32x2_alias_t __attribute__((may_alias));
typedef short v4i16_t __attribute__((ext_vector_type(4)));

#ifndef ODP_LIN_OCC
#define ODP_LIN_OCC 2  // waves per SIMD the outer-product kernels are compiled for
#endif

#define ODP_GLOBAL __attribute__((address_space(1)))
#define ODP_LDS __attribute__((address_space(3)))
#define ODP_CONST __attribute__((address_space(4)))
__device__ __forceinline__ v4i16_t lds_tr16(const uint16_t* p) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16((ODP_LDS v4i16_t*)(ODP_LDS void*)p);
}

// Whether local segment sg (len rows) of problem f may overflow float32 in
// the Gram or clipped-sum forms: with a = max|x| and b = max|g| over the
// segment's finite entries (odp_nonfinite_columns), a b max(L, sqrt(d_in
// d_out)) >= 2^60, d_in a^2 >= 2^124 or d_out b^2 >= 2^124.  False without
// the per-segment maxima (no check requested).
__device__ __forceinline__ bool lin_seg_at_risk(const int64_t* f, int sg, int32_t len, int64_t d_in,
                                                int64_t d_out) {
  const uint32_t* xa = (const uint32_t*)f[ODP_LN_XAMAX];
  const uint32_t* ga = (const uint32_t*)f[ODP_LN_GAMAX];
  if (xa == nullptr || ga == nullptr || len <= 0) return false;
  const double a = (double)__uint_as_float(xa[sg]), b = (double)__uint_as_float(ga[sg]);
  const double din = (double)d_in, dout = (double)d_out;
  const double w = fmax((double)len, sqrt(din * dout));
  return a * b * w >= 0x1p60 || din * a * a >= 0x1p124 || dout * b * b >= 0x1p124;
}

// Whether any segment of the problem is at risk.
__device__ __forceinline__ bool lin_problem_at_risk(const int64_t* f, const int32_t* slen, int seg_first,
                                                    int n_seg, int64_t d_in, int64_t d_out) {
  if (f[ODP_LN_XAMAX] == 0 || f[ODP_LN_GAMAX] == 0) return false;
  for (int sg = 0; sg < n_seg; ++sg)
    if (lin_seg_at_risk(f, sg, slen[seg_first + sg], d_in, d_out)) return true;
  return false;
}

struct LinProblem {
  const uint16_t* X;
  const uint16_t* G;
  int64_t ldx, ldg, d_in, d_out;
  int seg_first, n_seg;
};

__device__ __forceinline__ LinProblem read_problem(const int64_t* f) {
  LinProblem P;
  P.X = (const uint16_t*)f[ODP_LN_X];
  P.ldx = f[ODP_LN_LDX];
  P.G = (const uint16_t*)f[ODP_LN_G];
  P.ldg = f[ODP_LN_LDG];
  P.d_in = f[ODP_LN_DIN];
  P.d_out = f[ODP_LN_DOUT];
  P.seg_first = (int)f[ODP_LN_SEG_FIRST];
  P.n_seg = (int)f[ODP_LN_NSEG];
  return P;
}

// ---------------------------------------------------------------------------
// Outer-product main loop.  The workgroup's tile covers OM output rows (o,
// columns of G) by ON output columns (n, columns of X); NW waves in a
// 2 x (NW / 2) arrangement each own a WM x WN block as BI x BJ MFMA 16 x 16
// blocks.  A pipeline step stages OK tokens of both operands as token-major
// LDS tiles.  256 x 256 tiles of eight 128 x 64 waves (one workgroup and two
// waves per SIMD per CU) move a third less data from L2 into LDS per flop
// than 256 x 128 tiles of four, at the same registers per wave; the loads
// into LDS, not the MFMAs or the LDS reads, bound these kernels.
// ---------------------------------------------------------------------------
#ifndef ODP_LIN_OM
#define ODP_LIN_OM 256
#endif
#ifndef ODP_LIN_ON
#define ODP_LIN_ON 256
#endif
#ifndef ODP_LIN_WAVES
#define ODP_LIN_WAVES 8  // waves per workgroup, 2 x (NW / 2) over the tile
#endif
constexpr int OM = ODP_LIN_OM, ON = ODP_LIN_ON, OK = 32, NW = ODP_LIN_WAVES, OUTER_THREADS = 64 * NW;
constexpr int WM = OM / 2, WN = ON / (NW / 2), BI = WM / 16, BJ = WN / 16;
constexpr int A_TILE = OK * OM, B_TILE = OK * ON;  // elements
constexpr int OUTER_STAGE = A_TILE + B_TILE;


// Token-major tiles are unpadded and XOR-swizzled in 4-element (8-byte)
// chunks: chunk k of row r lives at chunk k ^ swz(r).  The 16 rows x 4
// chunks that one transposing operand read touches (rows 8g + j, j < 4,
// g < 4) then land on every LDS bank exactly twice, and a 16-byte piece
// (an aligned chunk pair) stays contiguous.
__device__ __forceinline__ int swz(int row) { return ((row & 3) | ((row >> 1) & 4)) << 2; }


// 16 columns col0.. of a token-major tile of row pitch `pitch`, tokens
// 8 (lane >> 4) + 0..7: the MFMA operand layout (lane & 15 = row of A /
// column of B).  Rows r and r + 4 share swz(), so the second read is
// 4 rows further on.
__device__ __forceinline__ bf16x8_t outer_frag(const uint16_t* tile, int pitch, int col0) {
  const int lane = threadIdx.x & 63, c = lane & 15;
  const int row = 8 * (lane >> 4) + (c >> 2);
  const int k = (col0 >> 2) + (c & 3);
  const uint16_t* src = tile + row * pitch + 4 * (k ^ swz(row));
  const v4i16_t t0 = lds_tr16(src), t1 = lds_tr16(src + 4 * pitch);
  const v4i16_t tt[2] = {t0, t1};
  return __builtin_bit_cast(bf16x8_t, tt);
}

typedef f32x4_t OuterAcc[BI][BJ];

// Where a lane's accumulator entries lie in the wave's WM x WN block: the
// MFMAs take X as their first operand, so entry e of block (i, j) is row
// 16 i + (lane & 15) (an output, column of G) and column 16 j + 4 (lane >>
// 4) + e (an input, column of X): 4 consecutive elements of a row of M.
__device__ __forceinline__ int acc_row(int i) { return 16 * i + (int)(threadIdx.x & 15); }
__device__ __forceinline__ int acc_col(int j) { return 16 * j + 4 * (int)((threadIdx.x & 63) >> 4); }

// The operands a step starts with, read during the step before it.
struct OuterHead {
  bf16x8_t b[BJ], a[2];
};

__device__ __forceinline__ uint32_t uniform32(uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); }
__device__ __forceinline__ uint64_t uniform64(uint64_t v) {
  return ((uint64_t)uniform32((uint32_t)(v >> 32)) << 32) | uniform32((uint32_t)v);
}

// One pipeline step: rows [t0, t0 + OK) clipped to its segment [tb, te).
// `fix`: the segment has non-finite columns inside the tile, which the step
// zeroes in LDS before its MFMAs.  Plain 32-bit fields (row counts stay
// below 2^31): a struct of mixed widths and a bool was kept in memory by
// the compiler when copied conditionally.
struct Step {
  int32_t t0, tb, te, seg, live, fix;
};

// Element (r, c) of a token-major tile of row pitch `pitch` (the XOR swizzle
// above).
__device__ __forceinline__ int tile_at(int r, int c, int pitch) {
  return r * pitch + 4 * ((c >> 2) ^ swz(r)) + (c & 3);
}

// Bit `c` of a segment's column mask (uint32 words, bit j of word w =
// column 32 w + j).
__device__ __forceinline__ bool mask_bit(const uint32_t* m, int64_t c) {
  return (m[c >> 5] >> (c & 31)) & 1u;
}

typedef float f32x8_t __attribute__((ext_vector_type(8)));

// c * v for 8 bf16 values: widened exactly, multiplied in fp32 and rounded
// to nearest-even bf16 (v_cvt_pk_bf16_f32).
__device__ __forceinline__ u32x4_t scale_bf16x8(u32x4_t v, float c) {
  f32x8_t f = __builtin_convertvector(__builtin_bit_cast(bf16x8_t, v), f32x8_t);
  f = f * c;
  return __builtin_bit_cast(u32x4_t, __builtin_convertvector(f, bf16x8_t));
}


// ---------------------------------------------------------------------------
// Outer-product main loop, buffer loads straight into LDS.  The step's G and
// X tiles (token-major rows, the XOR swizzle above) are fetched by
// buffer_load ... lds into a ring of RING LDS stages, RING - 1 steps ahead of
// the compute, with no staging registers; each step waits for the next
// step's loads with an explicit vmcnt and an LDS-only barrier.  The buffer resources
// cover only the rows of the step's segment, so rows outside it (and
// columns past the matrix, sent past the end) arrive as zeros.  A step never
// crosses a segment, so the clip factor is one scalar per step; it scales
// X's fragments after the LDS read (c * x rounded to bf16).
// ---------------------------------------------------------------------------
constexpr uint32_t LIN_BUF_DWORD3 = 0x00020000;  // raw 32-bit dwords (CDNA buffer resource)
constexpr uint32_t LIN_OOB = 0x80000000u;        // an offset past every buffer's end
constexpr int A_DMA = A_TILE * 2 / 1024 / NW;     // 1 KB loads per wave per step (G tile)
constexpr int B_DMA = B_TILE * 2 / 1024 / NW;     // (X tile)
constexpr int RPW = OK / NW;                      // tile rows each wave loads per step
#ifndef ODP_LIN_RING
#define ODP_LIN_RING 4  // LDS stages of the outer-form ring (RING - 1 steps in flight)
#endif
constexpr int RING = ODP_LIN_RING;
constexpr int UNROLL = RING % 2 ? 2 * RING : RING;  // steps per loop: stages and operand sets come out even
static_assert((RING == 4 || RING == 5) && (RING - 2) * (A_DMA + B_DMA) < 64, "ring depth");
constexpr int DMA_PER_STEP = A_DMA + B_DMA;
constexpr int B_LPR = ON / 8, B_RPI = 64 / B_LPR;  // X tile: lanes per row, rows per load
static_assert(OM == 256 && (ON == 128 || ON == 256), "G tile rows take 32 lanes; X tile rows 16 or 32");
static_assert((NW == 4 || NW == 8) && A_DMA * 2 == RPW && B_DMA * B_RPI == RPW && WN % 16 == 0,
              "each wave loads whole rows of both tiles");
static_assert(DMA_PER_STEP <= BI && BJ < BI, "a step's loads and the next step's operands go out one per block row");

// c times an X fragment, rounded to bf16.
__device__ __forceinline__ bf16x8_t scale_frag(bf16x8_t v, float c) {
  return __builtin_bit_cast(bf16x8_t, scale_bf16x8(__builtin_bit_cast(u32x4_t, v), c));
}

__device__ __forceinline__ void read_head(const uint16_t* st, OuterHead& H) {
  const int wave = threadIdx.x >> 6;
  const int wm = WM * (wave & 1), wn = WN * (wave >> 1);
#pragma unroll
  for (int j = 0; j < BJ; ++j) H.b[j] = outer_frag(st + A_TILE, ON, wn + 16 * j);
  H.a[0] = outer_frag(st, OM, wm);
  H.a[1] = outer_frag(st, OM, wm + 16);
}

// One ring step: its MFMAs from stage `cur` and the operands in `H`, the
// loads of a later step into stage `nxt` (issued one by one between the
// first MFMAs), and the first operands of the next step from stage `ahead`
// into `N` beside the last MFMAs, so that after the next barrier the MFMAs
// start at once instead of all eight waves first waiting for their operand
// reads together (Llama-3-8B-shaped layer, 8 x 4096 tokens: outer norms 1195
// -> 1270 TFLOP/s with the store and 1279 -> 1350 without, clipped sum 1170
// -> 1238, moments + 5 %; a fifth stage, one more step of loads in flight,
// measured + 4 % without the store, nothing with it, and spills in the sum).  The stages are restrict parameters of one inlined call,
// which gives the compiler the alias scopes that keep the reads from waiting
// for the loads into `nxt`.  SCALE: X's fragments times `c` (rounded to
// bf16) before use.  `tick` (the scalar bookkeeping of the step after) runs
// between the MFMAs, not between the steps, where nothing would cover it.
template <bool SCALE, typename Issue, typename Tick>
__device__ __forceinline__ void ring_step(uint16_t* __restrict__ nxt, const uint16_t* __restrict__ cur,
                                          const uint16_t* __restrict__ ahead, Issue issue, Tick tick, float c,
                                          OuterHead& H, OuterHead& N, OuterAcc& acc) {
  const int wave = threadIdx.x >> 6;
  const int wm = WM * (wave & 1), wn = WN * (wave >> 1);
  bf16x8_t a[3];
  a[0] = H.a[0];
  a[1] = H.a[1];
  if (SCALE) {
#pragma unroll
    for (int j = 0; j < BJ; ++j) H.b[j] = scale_frag(H.b[j], c);
  }
#pragma unroll
  for (int i = 0; i < BI; ++i) {
    if (i + 2 < BI) a[(i + 2) % 3] = outer_frag(cur, OM, wm + 16 * (i + 2));
    if (i < DMA_PER_STEP) issue(nxt, i);
    if (i >= BI - 1 - BJ && i < BI - 1)
      N.b[i - (BI - 1 - BJ)] = outer_frag(ahead + A_TILE, ON, wn + 16 * (i - (BI - 1 - BJ)));
    if (i >= BI - 2) N.a[i - (BI - 2)] = outer_frag(ahead, OM, wm + 16 * (i - (BI - 2)));
#pragma unroll
    for (int j = 0; j < BJ; ++j)
      acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(H.b[j], a[i % 3], acc[i][j], 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
    if (i == DMA_PER_STEP - 1) {
      tick();
      __builtin_amdgcn_sched_barrier(0);
    }
  }
}

// The ring: one array per stage, so that reads of one stage are not made to
// wait for the loads into the others.  Kernels may reuse it once the main
// loop has returned.
__shared__ __attribute__((aligned(16))) uint16_t lin_ring0[OUTER_STAGE];
__shared__ __attribute__((aligned(16))) uint16_t lin_ring1[OUTER_STAGE];
__shared__ __attribute__((aligned(16))) uint16_t lin_ring2[OUTER_STAGE];
__shared__ __attribute__((aligned(16))) uint16_t lin_ring3[OUTER_STAGE];
__shared__ __attribute__((aligned(16))) uint16_t lin_ring4[RING > 4 ? OUTER_STAGE : 64];
__device__ __forceinline__ uint16_t* lin_stage(int k) {
  return k == 0 ? lin_ring0 : k == 1 ? lin_ring1 : k == 2 ? lin_ring2 : k == 3 ? lin_ring3 : lin_ring4;
}

// FIX: a step whose `fix` is set has its stage changed by fixup(stage, step)
// once its loads have landed, before anything reads it.
template <bool SCALE, bool FIX, typename Next, typename Scale, typename Fixup>
__device__ __forceinline__ void dma_mainloop(const LinProblem& P, int64_t o0, int64_t n0, Step first,
                                             Next next, Scale scale, Fixup fixup, OuterAcc& acc) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // The problem and the steps are the same for every lane; where the compiler
  // cannot tell (vector loads), it is told.
  const uint64_t G = uniform64((uint64_t)P.G), X = uniform64((uint64_t)P.X);
  const uint32_t ldg = uniform32((uint32_t)P.ldg), ldx = uniform32((uint32_t)P.ldx);
  first = Step{(int32_t)uniform32(first.t0),  (int32_t)uniform32(first.tb),   (int32_t)uniform32(first.te),
               (int32_t)uniform32(first.seg), (int32_t)uniform32(first.live), (int32_t)uniform32(first.fix)};
  // Per lane: byte offset of each of its loads from the step's first row
  // (row within the step, column within the tile after undoing the swizzle;
  // columns past the matrix go past the end of every buffer).  The step only
  // moves the buffers' bases, on the scalar unit.
  uint32_t aoff[A_DMA], boff[B_DMA];
#pragma unroll
  for (int i = 0; i < A_DMA; ++i) {
    const int r = RPW * wave + 2 * i + (lane >> 5);
    const int32_t col = (int32_t)o0 + 8 * ((lane & 31) ^ (swz(r) >> 1));
    aoff[i] = col < (int32_t)P.d_out ? ((uint32_t)r * ldg + (uint32_t)col) * 2u : LIN_OOB;
  }
#pragma unroll
  for (int i = 0; i < B_DMA; ++i) {
    const int r = RPW * wave + B_RPI * i + (lane / B_LPR);
    const int32_t col = (int32_t)n0 + 8 * ((lane % B_LPR) ^ (swz(r) >> 1));
    boff[i] = col < (int32_t)P.d_in ? ((uint32_t)r * ldx + (uint32_t)col) * 2u : LIN_OOB;
  }

  // Where the loads of a step start: its first row of G and of X, and the
  // bytes from there to the segment's end (rows past it arrive as zeros; a
  // step past the last one has none).
  struct LoadAt {
    uint64_t g, x;
    uint32_t gbytes, xbytes;
  };
  auto load_at = [&](const Step& x) __attribute__((always_inline)) {
    const uint32_t rows = x.live ? (uint32_t)(x.te - x.t0) : 0u;
    return LoadAt{G + (uint64_t)x.t0 * ldg * 2u, X + (uint64_t)x.t0 * ldx * 2u, rows * ldg * 2u, rows * ldx * 2u};
  };
  // Load i of a step (i < A_DMA: rows of G, then X).
  auto issue = [&](uint16_t* st, const LoadAt& at, int i) __attribute__((always_inline)) {
    if (i < A_DMA) {
      const __amdgpu_buffer_rsrc_t gr =
          __builtin_amdgcn_make_buffer_rsrc((void*)at.g, (short)0, (int)at.gbytes, LIN_BUF_DWORD3);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(gr, (ODP_LDS void*)(st + (RPW * wave + 2 * i) * OM), 16, aoff[i], 0, 0,
                                               0);
    } else {
      const int k = i - A_DMA;
      const __amdgpu_buffer_rsrc_t xr =
          __builtin_amdgcn_make_buffer_rsrc((void*)at.x, (short)0, (int)at.xbytes, LIN_BUF_DWORD3);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(xr, (ODP_LDS void*)(st + A_TILE + (RPW * wave + B_RPI * k) * ON), 16,
                                               boff[k], 0, 0, 0);
    }
  };

  // Prologue: steps 0 .. RING - 2 in flight, then the operands step 0 starts
  // with.  Steps past the last one still issue (zero rows, so out of range)
  // to keep the wait counts constant.
  Step cur = first;
  Step ld = first;
  float c = 1.0f;  // of the step `cur`
#pragma unroll
  for (int q = 0; q < RING - 1; ++q) {
#pragma unroll
    for (int i = 0; i < DMA_PER_STEP; ++i) issue(lin_stage(q), load_at(ld), i);
    ld = next(ld);
  }
  LoadAt at = load_at(ld);
  Step nx = next(cur);
  // Opaque from here on: left as the constants they start with, the
  // accumulators of a loop with an exit at every step were kept twice.
#pragma unroll
  for (int i = 0; i < BI; ++i)
#pragma unroll
    for (int j = 0; j < BJ; ++j) __asm__ volatile("" : "+v"(acc[i][j]));
  OuterHead H[2];
  __builtin_amdgcn_s_waitcnt(vmcnt_imm((RING - 2) * DMA_PER_STEP));
  __asm__ volatile("s_barrier" ::: "memory");
  if (FIX && __builtin_expect(cur.fix, 0)) {
    fixup(lin_stage(0), cur);
    __syncthreads();
  }
  read_head(lin_stage(0), H[0]);
  if (SCALE && cur.live) c = scale(cur);
  while (cur.live) {
#pragma unroll
    for (int k = 0; k < UNROLL; ++k) {
      if (!cur.live) break;
      // The next step's loads have landed (this wave's; the barrier says so
      // for the others); the later RING - 3 steps' may fly.
      __builtin_amdgcn_s_waitcnt(vmcnt_imm((RING - 3) * DMA_PER_STEP));
      __asm__ volatile("s_barrier" ::: "memory");
      if (FIX && __builtin_expect(nx.fix, 0)) {
        fixup(lin_stage((k + 1) % RING), nx);
        __syncthreads();
      }
      // Loads of step ld go into the stage computed at the previous step.
      ring_step<SCALE>(lin_stage((k + RING - 1) % RING), lin_stage(k % RING), lin_stage((k + 1) % RING),
                       [&](uint16_t* st, int i) __attribute__((always_inline)) { issue(st, at, i); },
                       [&]() __attribute__((always_inline)) {
                         ld = next(ld);
                         at = load_at(ld);
                         cur = nx;
                         nx = next(nx);
                         // Computed here, not where they are used: worth
                         // 4 % of the clipped sum, whose steps cross
                         // segments (without FIX, a step is an addition
                         // and pinning it measured 1 % slower).
                         if (FIX) __asm__ volatile("" : "+s"(at.g), "+s"(at.x), "+s"(at.gbytes), "+s"(at.xbytes));
                       },
                       c, H[k & 1], H[(k + 1) & 1], acc);
      if (SCALE && cur.live) c = scale(cur);
    }
  }
  __builtin_amdgcn_s_waitcnt(0);  // no load into LDS may outlive the workgroup
  __asm__ volatile("s_barrier" ::: "memory");
}

// Compile-time loop: f(Idx<0>{}), ..., f(Idx<N - 1>{}).  Accumulator
// arrays indexed only through it stay in registers whatever their size
// (a plain loop the unroller declines leaves them in scratch memory).
template <int V>
struct Idx {
  static constexpr int value = V;
};
template <int N, int K = 0, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (K < N) {
    f(Idx<K>{});
    static_for<N, K + 1>(f);
  }
}

template <int I, int J>
__device__ __forceinline__ void zero_acc(f32x4_t (&acc)[I][J]) {
#pragma unroll
  for (int i = 0; i < I; ++i)
#pragma unroll
    for (int j = 0; j < J; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
}
