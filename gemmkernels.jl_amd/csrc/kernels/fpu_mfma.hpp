// Tiled GEMM of FPUOp (reference src/operator.jl:35-153) on the FP32 / FP64 matrix instructions.
//
// FPUOp.mma is one scalar fused multiply-add per k in ascending k, so every output is the fma chain
//   acc <- fma(a[k], b[k], acc),  k = 0, 1, ..., K - 1.
// v_mfma_f32_16x16x4_f32 and v_mfma_f64_16x16x4_f64 compute exactly that chain over their four k: checked on the
// device against fmaf / fma on 12 800 outputs per distribution (values spread over [-1, 1), over 40 binary orders of
// magnitude, sums in the subnormal range, subnormal factors) with no bit different, where the descending chain differs
// in a third to a half of them and a single rounding of the whole sum in as many.  A product on these instructions is
// therefore bit-identical to the vector-ALU kernel (fpu_gemm.hpp) and to a sequential loop on the host -- but for the sign of a
// zero where K is no multiple of four: the zeros behind K make +0 of a sum that underflowed to -0 -- at a higher rate:
// 148 TFLOP/s in FP32 from registers (v_fma_f32: 64), 77 in FP64 (v_fma_f64: 63; the packed FP32 fma that would
// double the vector ALUs' FP32 rate is not used in this library).
//
// What bounds it: the matrix cores.  An instruction takes 32 clocks (FP32; 64 in FP64) and reads one register per operand
// and 16 rows, so a wave tile of 64 x 64 reads 8 LDS words per lane for 512 clocks of matrix-core time: LDS and the
// vector-memory path are nearly idle, and the tiles go global -> registers -> LDS, which costs little here and leaves the
// values in a place where they are converted, scaled, moved and zeroed on their way.  What matters is that every SIMD has
// an MFMA to issue all the time.  An MFMA leaves room for seven other instructions of its wave, and an LDS read takes about
// four MFMAs to answer, so the instructions of a step are placed one behind each MFMA and the fragments are read LOOK
// steps ahead (1024^3, one 64 x 64 tile per CU: 27 us with reads in a group one step ahead, 23 so).  Most tiles use two
// LDS stages and leave the CU to several workgroups; the Float32 tiles of 128 x 128, and of 32 x 32 on four waves, three, with
// the first fragments of the next tile read in front of the barrier, because they often have a CU to themselves.
//
// Measured (beta = 0, one box; before, on the vector ALUs): Float32 256^3 12.2 -> 4.4 us, 1024^3 71 -> 23, 2048^3
// 293 -> 134, 3001 x 3003 x 2999 -> 461 (0.79 of the instruction's rate), 4096^3 1900 -> 1028 us (134 TFLOP/s, 0.90);
// Float64 1000^3 115 -> 41 us, 2048^3 -> 270 (64 TFLOP/s, 0.83).  What is left: the last round of tiles (2560^3 has 1600
// tiles of 64 x 64 for 256 CUs: 7 rounds where 6.25 would do), and the ends of a launch.
//
// A K tile of 32 x 32 x 32 is a few hundred clocks of work for the matrix cores (512 in FP64, 256 in FP32), less than a load
// takes from the last-level cache: on four waves these tiles have the loads of two K tiles in flight (DEPTH; the loop is
// written out for a pair of tiles, so that each finds its registers): Float32 1024^3 25.7 -> 24.7 us, 300 x 700 x 1500
// 17.2 -> 16.3, Float64 500 x 500 x 700 12.7 -> 12.1, 1024^3 44.9 -> 42.6.  Tiles of 64 x 64 that share a CU gain nothing from it (Float64
// 1024^3 41.1 -> 41.6, Float32 2048^3 142 -> 145): one in flight.
//
// Launches that have at most one workgroup per CU run instances of their own (fpu_mfma_deep.hip).
//
// Sizes, leading dimensions and addresses are free.  A vector load takes any address that is aligned to its elements; rows
// beyond the edge of an operand are clamped to the last ones (their products land in outputs that are not stored):
// where memory is contiguous along the rows the vector that reaches over the edge is fetched from 1 .. 3 elements further
// back and moved into place.  The last K tile, when it is partial, is fetched the same way along k with zeros beyond K,
// waits in registers for the end of the loop, and only its steps that hold values are multiplied (moved and zeroed inside
// the loop instead: 3001 x 3003 x 2999 557 us).
//
// Hooks.  What a BLAS-level call asks for -- a factor on A, one on C -- is a multiplication in the loads' way to LDS and one of C
// before the loop (level 1: the K loop of the plain kernel); lists of operations run over all vectors of a tile at once, in
// front of its first MFMA (level 2).  One instance for both, whose lists were indexed at run time per vector, had the
// argument block in scratch memory and up to 259 spilled registers.  From it to these: factors, Float64 1000^3 'T','N' 49.4 ->
// 42.9 us, Float32 512^3 8.9 -> 8.0, 4096^3 1215 -> 1126 (plain 1024); lists on A, B and D, Float32 4096^3 3774 -> 1653 (on the
// vector ALUs 1975), 512^3 21.4 -> 18.6 (26.8), Float64 2048^3 668 -> 386 (567).
#pragma once
#include "fpu_gemm.hpp"

namespace gk {

// One step of four k for a block of 16 x 16 outputs, of which a lane owns four: register r is row row(lane, r) of column
// col(lane, r).  FP32: the A fragment first, so a lane owns 4 consecutive rows of one column (16-byte stores); FP64, whose
// lanes own every fourth index of the first operand: the B fragment first, so that 16 lanes own 16 consecutive rows of a
// column (128 bytes per column and store).
template <typename T> struct ChainBlock;
template <> struct ChainBlock<float> {
  typedef float acc_t __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ acc_t mma(float a, float b, acc_t c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
  static __device__ __forceinline__ int row(int lane, int r) { return 4 * (lane >> 4) + r; }
  static __device__ __forceinline__ int col(int lane, int r) { (void)r; return lane & 15; }
};
template <> struct ChainBlock<double> {
  typedef double acc_t __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ acc_t mma(double a, double b, acc_t c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(b, a, c, 0, 0, 0); }
  static __device__ __forceinline__ int row(int lane, int r) { (void)r; return lane & 15; }
  static __device__ __forceinline__ int col(int lane, int r) { return 4 * r + (lane >> 4); }
};

template <int BM_, int BN_, int BK_, int WAVES_M_, int WAVES_N_, typename TIN_, bool A_KMAJOR_, bool B_KMAJOR_, typename TACC_, int FUSED_,
          int STAGES_, int RING_, int DEPTH_, bool SPLITK_ = false>
struct FpuMfmaConfig {
  static constexpr int BM = BM_, BN = BN_, BK = BK_, WAVES_M = WAVES_M_, WAVES_N = WAVES_N_, STAGES = STAGES_, RING = RING_, DEPTH = DEPTH_;
  static constexpr bool A_KMAJOR = A_KMAJOR_, B_KMAJOR = B_KMAJOR_;
  // a workgroup handles one slice of K (blockIdx.z); the slices of a tile meet in a workspace (splitk_reduce)
  static constexpr bool SPLITK = SPLITK_;
  // hooks: 0 none (no bias either); 1 at most one scale on A, on B and on C, any on D; 2 any
  static constexpr int FUSED = FUSED_;
  typedef TIN_ TIN;
  typedef TACC_ TACC;
  static constexpr int THREADS = WAVES_M * WAVES_N * kWaveSize;
  static constexpr int WTM = BM / WAVES_M, WTN = BN / WAVES_N, FM = WTM / 16, FN = WTN / 16, STEPS = BK / 4;
  static constexpr int V = sizeof(TIN) == 8 ? 2 : 4;               // elements per load: 16 bytes (8 of Float16)
  // LDS rows: k for an operand whose rows (m or n) are contiguous in memory, m or n for one that is contiguous along k.
  // Pitches that make the fragment reads free of bank conflicts (a read takes 16 rows at 2 k per half wave): 16
  // elements more than a multiple of 32, and 4 (FP64: 2) times an odd number.
  static constexpr int pitch(bool kmajor, int rows) { return kmajor ? BK + (sizeof(TACC) == 8 ? 2 : 4) : rows + 16; }
  static constexpr int PA = pitch(A_KMAJOR, BM), PB = pitch(B_KMAJOR, BN);
  static constexpr int A_ELEMS = (A_KMAJOR ? BM : BK) * PA, B_ELEMS = (B_KMAJOR ? BN : BK) * PB;
  static constexpr int LDS_BYTES = STAGES * (A_ELEMS + B_ELEMS) * (int)sizeof(TACC);
  static constexpr int A_PER_THREAD = BM * BK / V / THREADS, B_PER_THREAD = BN * BK / V / THREADS;
  // Hooks take registers: a wave may have all 512 of its SIMD where LDS leaves room for one workgroup of a tile anyway, and
  // where lists meet 64 accumulators (256 registers spill there).
  static constexpr int WAVES_PER_SIMD = FUSED != 0 && THREADS == 256 && (LDS_BYTES > 80 * 1024 || (FUSED == 2 && BM * BN >= 64 * THREADS)) ? 1 : 2;
  static_assert(BM % (16 * WAVES_M) == 0 && BN % (16 * WAVES_N) == 0 && BM % 32 == 0 && BN % 32 == 0 && BK % 8 == 0, "wave tiles are made of 16 x 16 blocks");
  static_assert(A_PER_THREAD * V * THREADS == BM * BK && B_PER_THREAD * V * THREADS == BN * BK, "tile loads divide evenly over the threads");
  static_assert(STAGES == 3 || (STAGES == 2 && RING == 2), "two stages, or three with the first fragments read ahead of the barrier");
  static_assert((RING & (RING - 1)) == 0 && STEPS % RING == 0, "a step finds its fragments in buffer s % RING in every tile");
};

// A list of operations in scalar registers, loaded from the kernel arguments where it is used.  (The address goes through a
// statement that the compiler cannot see through: loaded once, the lists would hold half of the scalar registers all
// through the K loop.  The arguments themselves, indexed at run time, would be copied to scratch memory as a whole.)
struct ListRegs {
  int n, kind[kMaxOps];
  float p0[kMaxOps], p1[kMaxOps];
  __device__ __forceinline__ explicit ListRegs(int hook) {
    typedef const __attribute__((address_space(4))) char* bytes;
    typedef const __attribute__((address_space(4))) OpList* list;
    bytes arguments = (bytes)__builtin_amdgcn_kernarg_segment_ptr();      // (GemmArgs is the kernel's only argument)
    asm volatile("" : "+s"(arguments));
    list t = (list)(arguments + __builtin_offsetof(GemmArgs, t) + hook * (int)sizeof(OpList));
    n = t->n;
#pragma unroll
    for (int i = 0; i < kMaxOps; ++i) { kind[i] = t->kind[i]; p0[i] = t->p0[i]; p1[i] = t->p1[i]; }
  }
};

// A list applied to COUNT values in registers, slot after slot in a loop that is not unrolled: with up to 64 accumulators the
// code of every op stands once per hook, not once per slot, and the switch is paid once per slot, not once per value.
// The loop always takes the first slot and moves the others up.
template <typename X, int COUNT>
__device__ __forceinline__ void apply_list_looped(ListRegs t, X (&x)[COUNT]) {
#pragma clang loop unroll(disable)
  for (int i = 0; i < t.n; ++i) {
    const int kind = t.kind[0];
    const float p0 = t.p0[0], p1 = t.p1[0];
#pragma unroll
    for (int j = 1; j < kMaxOps; ++j) { t.kind[j - 1] = t.kind[j]; t.p0[j - 1] = t.p0[j]; t.p1[j - 1] = t.p1[j]; }
    auto each = [&](auto kind_c) __attribute__((always_inline)) {
#pragma unroll
      for (int e = 0; e < COUNT; ++e) x[e] = apply_op_t<X>(decltype(kind_c)::value, p0, p1, x[e]);
    };
    switch (kind) {
      case T_SCALE: each(std::integral_constant<int, T_SCALE>{}); break;
      case T_ADD: each(std::integral_constant<int, T_ADD>{}); break;
      case T_RELU: each(std::integral_constant<int, T_RELU>{}); break;
      case T_NEG: each(std::integral_constant<int, T_NEG>{}); break;
      case T_ABS: each(std::integral_constant<int, T_ABS>{}); break;
      case T_CLAMP: each(std::integral_constant<int, T_CLAMP>{}); break;
      case T_SQUARE: each(std::integral_constant<int, T_SQUARE>{}); break;
      default: break;
    }
  }
}

// One operand of a workgroup: ROWS rows (m or n) from row r0 of a matrix with `limit` rows.
template <class Cfg, int ROWS, bool KMAJOR, int PITCH, int PER>
struct ChainOperand {
  typedef typename Cfg::TIN TIN;
  typedef typename Cfg::TACC TACC;
  typedef typename ArithOf<TIN>::type TAR;                             // arithmetic type of the hooks
  static constexpr int V = Cfg::V, BK = Cfg::BK;
  static constexpr int PER_LINE = KMAJOR ? BK / V : ROWS / V;          // vectors per LDS row
  static constexpr int LINES = Cfg::THREADS / PER_LINE;                // LDS rows that the threads fill at a time
  static_assert(Cfg::THREADS % PER_LINE == 0, "the threads fill whole LDS rows");
  // a vector at any address its elements may have
  typedef TIN vec __attribute__((ext_vector_type(V)));
  struct __attribute__((packed, aligned(sizeof(TIN)))) loose { vec v; };

  const TIN* base;
  long long ld;
  long long off[KMAJOR ? PER : 1];      // element offset of the thread's vectors in the operand at k = 0, rows clamped to the operand
  int line, within;       // LDS row of the thread's first vector, element in it
  int shift;              // rows by which the thread's vectors are fetched too early (memory contiguous along the rows)
  int r0, limit, K;
  TAR scale;              // FUSED == 1: the hooks of the operand are one multiplication (1: there are none)

  __device__ __forceinline__ void init(const void* p, long long ld_, int r0_, int limit_, int K_, int tid, float scale_) {
    base = (const TIN*)p; ld = ld_; r0 = r0_; limit = limit_; K = K_;
    line = tid / PER_LINE;
    within = (tid % PER_LINE) * V;
    shift = 0;
    if constexpr (KMAJOR) {
#pragma unroll
      for (int i = 0; i < PER; ++i) {
        const int r = r0 + line + i * LINES;
        off[i] = (long long)(r < limit ? r : limit - 1) * ld;
      }
    } else {
      int r = r0 + within;
      const int last = limit - V;
      if (r > last) { shift = r - last; r = last; }
      off[0] = r;
    }
    scale = (TAR)scale_;        // (x * 1 is x: a multiplication in the K loop costs no branch)
  }
  // no row or K is short of a whole vector (else every fetch of this workgroup is element by element)
  __device__ __forceinline__ bool vectors_fit() const { return (KMAJOR ? K : limit) >= V; }
  // vector i of the K tile from k0.  TAIL: the tile reaches over K (the vector is fetched further back, or from the
  // last k, and put right by settle)
  template <bool TAIL>
  __device__ __forceinline__ vec fetch(int i, int k0) const {
    const TIN* p;
    if constexpr (KMAJOR) {
      int k = k0 + within;
      if constexpr (TAIL) k = k < K - V ? k : K - V;
      p = base + (off[KMAJOR ? i : 0] + k);
    } else {
      int k = k0 + line + i * LINES;
      if constexpr (TAIL) k = k < K ? k : K - 1;
      p = base + ((long long)((unsigned long long)(unsigned)k * (unsigned)ld) + off[0]);       // (ld < 2^31: the host refuses more)
    }
    return ((const loose*)p)->v;
  }
  // moves the elements of a vector that was fetched `by` elements too early into place
  static __device__ __forceinline__ vec moved(vec y, int by) {
    const bool one = (by & 1) != 0;
    vec z = y;
#pragma unroll
    for (int e = 0; e + 1 < V; ++e) z[e] = one ? y[e + 1] : y[e];
    if constexpr (V == 4) {
      const bool two = (by & 2) != 0;
      y = z;
      z[0] = two ? y[2] : y[0];
      z[1] = two ? y[3] : y[1];
    }
    return z;
  }
  // puts a vector right.  MOVED: its rows may reach over the edge (those beyond it hold anything: their products are not
  // stored); TAIL: of a partial K tile, values beyond K are zero
  template <bool MOVED, bool TAIL>
  __device__ __forceinline__ vec settle(vec x, int i, int k0) const {
    if constexpr (MOVED && !KMAJOR) x = moved(x, shift);
    if constexpr (TAIL) {
      const int k = k0 + (KMAJOR ? within : line + i * LINES), early = k - (K - V);
      if constexpr (KMAJOR) x = moved(x, early > 0 ? early : 0);
      x = cut(x, i, k0);
    }
    return x;
  }
  // a vector element by element (beyond K: the last values)
  __device__ __forceinline__ vec fetch_slow(int i, int k0) const {
    vec x;
#pragma unroll
    for (int e = 0; e < V; ++e) {
      int r = r0 + (KMAJOR ? line + i * LINES : within + e);
      const int k = k0 + (KMAJOR ? within + e : line + i * LINES);
      r = r < limit ? r : limit - 1;
      const int kk = k < K ? k : K - 1;
      x[e] = base[KMAJOR ? (long long)r * ld + kk : (long long)kk * ld + r];
    }
    return x;
  }
  // The two load hooks, each rounded to the element type of its destination (the operand's own type): a scale of one
  // vector, or the lists over all vectors of a tile at once.  They come before settle: 0 times an infinite factor, or a
  // list, makes something of the zeros behind K.
  __device__ __forceinline__ vec scaled(vec x) const {
    if constexpr (Cfg::FUSED == 1) {
#pragma unroll
      for (int e = 0; e < V; ++e) x[e] = (TIN)((TAR)x[e] * scale);
    }
    return x;
  }
  static __device__ __forceinline__ void listed(vec (&x)[PER], int hook0, int hook1) {
    const ListRegs t0(hook0), t1(hook1);
    TAR w[PER * V];
#pragma unroll
    for (int i = 0; i < PER * V; ++i) w[i] = (TAR)x[i / V][i % V];
    if (t0.n > 0) {
      apply_list_looped<TAR, PER * V>(t0, w);
#pragma unroll
      for (int i = 0; i < PER * V; ++i) w[i] = (TAR)(TIN)w[i];
    }
    apply_list_looped<TAR, PER * V>(t1, w);
#pragma unroll
    for (int i = 0; i < PER * V; ++i) x[i / V][i % V] = (TIN)w[i];
  }
  // values beyond K are zero
  __device__ __forceinline__ vec cut(vec x, int i, int k0) const {
#pragma unroll
    for (int e = 0; e < V; ++e) x[e] = k0 + (KMAJOR ? within + e : line + i * LINES) < K ? x[e] : (TIN)0;
    return x;
  }
  // converted to the accumulator type for the fma
  __device__ __forceinline__ void store(TACC* lds, vec x, int i) const {
    typedef TACC accv __attribute__((ext_vector_type(V)));
    accv z;
#pragma unroll
    for (int e = 0; e < V; ++e) z[e] = (TACC)x[e];
    *(accv*)&lds[(line + i * LINES) * PITCH + within] = z;
  }
  // value of row `row` at k of an LDS stage
  static __device__ __forceinline__ TACC at(const TACC* lds, int row, int k) { return KMAJOR ? lds[row * PITCH + k] : lds[k * PITCH + row]; }
};

constexpr int min_of(int a, int b) { return a < b ? a : b; }

// waits until at most N LDS instructions are outstanding (the counter holds 15)
template <int N>
__device__ __forceinline__ void wait_lds() { asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(N < 15 ? N : 15) : "memory"); }

template <class Cfg>
__global__ void __launch_bounds__(Cfg::THREADS, Cfg::WAVES_PER_SIMD) fpu_mfma_kernel(const GemmArgs args) {
  typedef typename Cfg::TIN TIN;
  typedef typename Cfg::TACC TACC;
  constexpr int BM = Cfg::BM, BN = Cfg::BN, BK = Cfg::BK, FM = Cfg::FM, FN = Cfg::FN, STEPS = Cfg::STEPS, STAGES = Cfg::STAGES;
  typedef ChainBlock<TACC> Block;
  constexpr int COUNT = FM * FN * 4;
  typedef typename Block::acc_t acc_t;
  constexpr bool AHEAD = STAGES == 3;
  constexpr int FAR = AHEAD ? 2 : 1;             // a tile goes to LDS FAR tiles before it is multiplied, DEPTH tiles after its loads set out
  constexpr int DEPTH = Cfg::DEPTH;
  constexpr int STAGE = Cfg::A_ELEMS + Cfg::B_ELEMS, PA = Cfg::A_PER_THREAD, PB = Cfg::B_PER_THREAD;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  TACC* lds = (TACC*)smem;

  // what stands in front of the first load, read in one go (0.2 us for each group of arguments that is a trip of its own)
  asm volatile("" ::"s"(args.a), "s"(args.b), "s"(args.lda), "s"(args.ldb), "s"(args.M), "s"(args.N), "s"(args.K), "s"(args.nbm), "s"(args.nbn), "s"(args.swz_kind), "s"(args.swz_param));
  if constexpr (Cfg::SPLITK) asm volatile("" ::"s"(args.k_steps), "s"(args.k_slices));
  if constexpr (Cfg::FUSED == 1) asm volatile("" ::"s"(args.scale_a), "s"(args.scale_b), "s"(args.t[H_RF2SH_D].n), "s"(args.t[H_SH2GL_D].n));
  int ti, tj;
  cta_swizzle(args.swz_kind, args.swz_param, (int)blockIdx.x, (int)blockIdx.y, args.nbm, args.nbn, ti, tj);
  if (ti >= args.nbm || tj >= args.nbn) return;
  const int tid = (int)threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave % Cfg::WAVES_M, wn = wave / Cfg::WAVES_M;
  const int m0 = ti * BM, n0 = tj * BN;
  // (K-split instances: the slice's k values only, A and B seen from its first one)
  const int k_first = Cfg::SPLITK ? (int)blockIdx.z * args.k_steps * BK : 0;
  const int K = !Cfg::SPLITK ? args.K : (args.K - k_first < args.k_steps * BK ? args.K - k_first : args.k_steps * BK);
  if (Cfg::SPLITK && K <= 0) return;           // (the whole workgroup leaves together)
  const int KT = (K + BK - 1) / BK;
  const bool edge_m = m0 + BM > args.M, edge_n = n0 + BN > args.N;
  const bool zero_ab = args.a_kind == 0;         // Layout.Zero: alpha == 0 (reference src/matmul.jl:127-130)

  ChainOperand<Cfg, BM, Cfg::A_KMAJOR, Cfg::PA, PA> oa;
  ChainOperand<Cfg, BN, Cfg::B_KMAJOR, Cfg::PB, PB> ob;
  oa.init((const TIN*)args.a + (Cfg::A_KMAJOR ? (long long)k_first : k_first * args.lda), args.lda, m0, args.M, K, tid, Cfg::FUSED == 1 ? args.scale_a : 1.0f);
  ob.init((const TIN*)args.b + (Cfg::B_KMAJOR ? (long long)k_first : k_first * args.ldb), args.ldb, n0, args.N, K, tid, Cfg::FUSED == 1 ? args.scale_b : 1.0f);
  const bool with_c = args.c_mode != 0 && (!Cfg::SPLITK || blockIdx.z == 0);       // the first slice of K starts from C, the others from zero

  acc_t acc[FM][FN];
  auto row_of = [&](int fi, int r) { return m0 + wm * Cfg::WTM + fi * 16 + Block::row(lane, r); };
  auto col_of = [&](int fj, int r) { return n0 + wn * Cfg::WTN + fj * 16 + Block::col(lane, r); };
  constexpr bool WIDE = sizeof(TACC) == 4;            // a lane's four outputs of a block are consecutive rows
  struct __attribute__((packed, aligned(sizeof(TACC)))) loose_acc { acc_t v; };
  // one hook over all accumulators of the lane
  [[maybe_unused]] auto hook_acc = [&](int hook) __attribute__((always_inline)) {
    if (args.t[hook].n == 0) return;
    const ListRegs t(hook);
    TACC flat[COUNT];
#pragma unroll
    for (int x = 0; x < COUNT; ++x) flat[x] = acc[x / 4 % FM][x / 4 / FM][x % 4];
    apply_list_looped<TACC, COUNT>(t, flat);
#pragma unroll
    for (int x = 0; x < COUNT; ++x) acc[x / 4 % FM][x / 4 / FM][x % 4] = flat[x];
  };
  // accumulators start from C
  auto load_c = [&]() __attribute__((always_inline)) {
    const TACC* C = (const TACC*)args.c;
#pragma unroll
    for (int fi = 0; fi < FM; ++fi)
#pragma unroll
      for (int fj = 0; fj < FN; ++fj) {
        acc_t c = (TACC)0;
        if (with_c) {
          if (WIDE && !edge_m && !edge_n) {
            c = ((const loose_acc*)(C + row_of(fi, 0) + (long long)col_of(fj, 0) * args.ldc))->v;
          } else {
            // (rows and columns beyond the edge read the last ones: no branch, so all loads are in flight together)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              int rr = row_of(fi, r), cc = col_of(fj, r);
              rr = rr < args.M ? rr : args.M - 1;
              cc = cc < args.N ? cc : args.N - 1;
              c[r] = C[rr + (long long)cc * args.ldc];
            }
          }
        }
        acc[fi][fj] = c;
      }
    if constexpr (Cfg::FUSED == 1) {
      if (!Cfg::SPLITK || with_c) {            // (0 times an infinite factor would make something of the zeros)
#pragma unroll
        for (int fi = 0; fi < FM; ++fi)
#pragma unroll
          for (int fj = 0; fj < FN; ++fj) acc[fi][fj] *= (TACC)args.acc_pre_scale;
      }
    }
    if constexpr (Cfg::FUSED == 2) {
      if (args.c_mode != 0) {
        hook_acc(H_GL2SH_C);
        hook_acc(H_SH2RF_C);
      }
    }
  };

  constexpr int RING = Cfg::RING, LOOK = RING - 1;       // fragments are read LOOK steps ahead
  TACC fa[RING][FM], fb[RING][FN];
  const int row_a = wm * Cfg::WTM + (lane & 15), row_b = wn * Cfg::WTN + (lane & 15), q = lane >> 4;
  auto read = [&](int buf, const TACC* stage, int s) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < FM; ++i) fa[buf][i] = decltype(oa)::at(stage, row_a + 16 * i, 4 * s + q);
#pragma unroll
    for (int j = 0; j < FN; ++j) fb[buf][j] = decltype(ob)::at(stage + Cfg::A_ELEMS, row_b + 16 * j, 4 * s + q);
  };
  auto multiply = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int i = 0; i < FM; ++i) acc[i][j] = Block::mma(fa[buf][i], fb[buf][j], acc[i][j]);
  };

  // The order of the instructions of a step: behind every MFMA one LDS read of the next step's fragments and a few of the
  // instructions that bring a later tile in.  An MFMA leaves room for seven other instructions of its wave; read in a
  // group, the fragments of a step cost a lone wave a fifth of the rate (144 -> 117 TFLOP/s in a loop of reads and MFMAs).
  auto interleave = [&]() __attribute__((always_inline)) {
    fpu_static_for<0, FM * FN>([&](auto) __attribute__((always_inline)) {
      __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);          // MFMA
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);        // LDS read
      __builtin_amdgcn_sched_group_barrier(0x2, 3, 0);          // vector ALU
      __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);        // LDS write
      __builtin_amdgcn_sched_group_barrier(0x20, 1, 0);         // load from memory
    });
  };

  // The vectors of a tile go to LDS in the first steps of a tile.  The LDS answers in order, so the barrier that
  // publishes them need not wait for the fragment reads behind the last write: those of the QUIET steps that write nothing,
  // less the last step of two stages, which has no later step of its tile to read for.  (An instruction reads one or two
  // fragments: at least (FM + FN) / 2 of them a step.)
  constexpr int SHARE = (PA + PB + STEPS - 2) / (STEPS - 1), QUIET = STEPS - (PA + PB + SHARE - 1) / SHARE;
  constexpr int READS_BEHIND = (AHEAD ? QUIET : QUIET - 1) * ((FM + FN + 1) / 2);
  static_assert(QUIET >= 1, "the last step writes nothing");

  // FUSED == 2: the lists of both operands over the vectors of a tile
  auto lists = [&](auto& xa, auto& xb) __attribute__((always_inline)) {
    if constexpr (Cfg::FUSED == 2) {
      if (args.t[H_GL2SH_A].n + args.t[H_SH2RF_A].n > 0) decltype(oa)::listed(xa, H_GL2SH_A, H_SH2RF_A);
      if (args.t[H_GL2SH_B].n + args.t[H_SH2RF_B].n > 0) decltype(ob)::listed(xb, H_GL2SH_B, H_SH2RF_B);
    }
  };

  // The K loop over the whole tiles, written without a branch inside a tile: tiles beyond the last one are fetched and
  // stored like any other (from the addresses of the last, into stages that nobody reads), so that the loads, the moves and
  // the LDS writes of a later tile stand between the MFMAs of this one.  A partial last tile sets out before the loop
  // and waits in registers of its own for the end of it.  MOVED: the rows of an operand that is contiguous along them
  // reach over its edge.
  const int whole = K / BK, k_tail = whole * BK;
  // SCALE_B: B has a factor as well (a BLAS-level call has one on A alone; without the multiplication of every value of B by 1, with factors on A and C: 1000^3
  // 'T','N' Float64 40.9 -> 39.7 us, Float32 28.7 -> 27.4).
  auto pipeline = [&](auto moved_c, [[maybe_unused]] auto scale_b_c) __attribute__((always_inline)) {
    constexpr bool MOVED = decltype(moved_c)::value, SCALE_B = decltype(scale_b_c)::value;
    typename decltype(oa)::vec ra[FAR + DEPTH][PA], ta[PA];      // (tile t of the loop waits in slot FAR + (t - FAR) % DEPTH)
    typename decltype(ob)::vec rb[FAR + DEPTH][PB], tb[PB];
    auto k_of = [&](int t) { return (t < whole ? t : whole - 1) * BK; };      // a tile that exists
    if constexpr (Cfg::FUSED == 2) load_c();       // (its lists before the tiles set out: no registers for both)
    if (whole > 0)
      fpu_static_for<0, FAR + DEPTH>([&](auto t_c) __attribute__((always_inline)) {
        constexpr int t = decltype(t_c)::value;
#pragma unroll
        for (int i = 0; i < PA; ++i) ra[t][i] = oa.template fetch<false>(i, k_of(t));
#pragma unroll
        for (int i = 0; i < PB; ++i) rb[t][i] = ob.template fetch<false>(i, k_of(t));
      });
    if (k_tail < K) {
#pragma unroll
      for (int i = 0; i < PA; ++i) ta[i] = oa.template fetch<true>(i, k_tail);
#pragma unroll
      for (int i = 0; i < PB; ++i) tb[i] = ob.template fetch<true>(i, k_tail);
    }
    if constexpr (Cfg::FUSED != 2) load_c();
    auto stash_a = [&](TACC* stage, typename decltype(oa)::vec x, int i, int k0) __attribute__((always_inline)) {
      oa.store(stage, oa.template settle<MOVED, false>(oa.scaled(x), i, k0), i);
    };
    auto stash_b = [&](TACC* stage, typename decltype(ob)::vec x, int i, int k0) __attribute__((always_inline)) {
      if constexpr (SCALE_B) x = ob.scaled(x);
      ob.store(stage + Cfg::A_ELEMS, ob.template settle<MOVED, false>(x, i, k0), i);
    };
    int stage = 0;
    if (whole > 0) {
      fpu_static_for<0, FAR>([&](auto t_c) __attribute__((always_inline)) {
        constexpr int t = decltype(t_c)::value;
        lists(ra[t], rb[t]);
#pragma unroll
        for (int i = 0; i < PA; ++i) stash_a(lds + t * STAGE, ra[t][i], i, k_of(t));
#pragma unroll
        for (int i = 0; i < PB; ++i) stash_b(lds + t * STAGE, rb[t][i], i, k_of(t));
      });
      wait_lgkmcnt0();
      block_barrier();
      if constexpr (AHEAD)
        fpu_static_for<0, LOOK>([&](auto s_c) __attribute__((always_inline)) { read(decltype(s_c)::value, lds, decltype(s_c)::value); });
    }
    auto tile = [&](int kt, auto slot_c) __attribute__((always_inline)) {
      constexpr int SLOT = FAR + decltype(slot_c)::value;
      const TACC* here = lds + stage * STAGE;
      const int next = stage + 1 == STAGES ? 0 : stage + 1, after = next + 1 == STAGES ? 0 : next + 1;
      TACC* into = lds + (AHEAD ? after : next) * STAGE;
      const int k_in = k_of(kt + FAR), k_out = k_of(kt + FAR + DEPTH);
      lists(ra[SLOT], rb[SLOT]);
      if constexpr (!AHEAD) read(0, here, 0);
      fpu_static_for<0, STEPS>([&](auto s_c) __attribute__((always_inline)) {
        constexpr int s = decltype(s_c)::value;
        if constexpr (s + LOOK < STEPS) read((s + LOOK) % RING, here, s + LOOK);
        else if constexpr (AHEAD) read((s + LOOK) % RING, lds + next * STAGE, s + LOOK - STEPS);
        multiply(s % RING);
        // this step's share of the vectors of a tile: into LDS, and the next ones on their way
        constexpr int lo = min_of(PA + PB, s * SHARE), hi = min_of(PA + PB, (s + 1) * SHARE);
        fpu_static_for<lo, hi>([&](auto v_c) __attribute__((always_inline)) {
          constexpr int v = decltype(v_c)::value;
          if constexpr (v < PA) {
            stash_a(into, ra[SLOT][v], v, k_in);
            ra[SLOT][v] = oa.template fetch<false>(v, k_out);
          } else {
            stash_b(into, rb[SLOT][v - PA], v - PA, k_in);
            rb[SLOT][v - PA] = ob.template fetch<false>(v - PA, k_out);
          }
        });
        interleave();
        __builtin_amdgcn_sched_barrier(0);
      });
      wait_lds<READS_BEHIND>();
      block_barrier();
      stage = next;
    };
    // The accumulators that C filled have arrived when the loop begins: left open, the compiler waits for every load of the
    // next tile in front of the first MFMA of each tile (vmcnt(0) there; with this, one vector at a time where it goes to LDS).
    __builtin_amdgcn_s_waitcnt(0x0F70);         // vmcnt(0)
    for (int kt = 0; kt < whole; kt += DEPTH) {
      // (written out for DEPTH tiles: each finds the registers of its loads)
      fpu_static_for<0, DEPTH>([&](auto d_c) __attribute__((always_inline)) {
        constexpr int d = decltype(d_c)::value;
        if (d == 0 || kt + d < whole) tile(kt + d, d_c);
      });
    }
    if (k_tail < K) {
      // (the barrier above: everyone has read the last whole tile)
      wait_lgkmcnt0();
      block_barrier();
      lists(ta, tb);
#pragma unroll
      for (int i = 0; i < PA; ++i) oa.store(lds, oa.template settle<MOVED, true>(oa.scaled(ta[i]), i, k_tail), i);
#pragma unroll
      for (int i = 0; i < PB; ++i) ob.store(lds + Cfg::A_ELEMS, ob.template settle<MOVED, true>(ob.scaled(tb[i]), i, k_tail), i);
      wait_lgkmcnt0();
      block_barrier();
      const int steps = (K - k_tail + 3) / 4;            // the steps that hold values
      for (int s = 0; s < steps; ++s) {
        read(0, lds, s);
        multiply(0);
      }
    }
  };

  if (zero_ab) {
    load_c();
    if constexpr (Cfg::FUSED != 0) {
      // zeros through the hooks, as loaded values would go
      typedef typename ArithOf<TIN>::type TAR;
      TAR a[1] = {0}, b[1] = {0};
      for (const int h : {H_GL2SH_A, H_SH2RF_A}) { apply_list_looped<TAR, 1>(ListRegs(h), a); a[0] = (TIN)a[0]; }
      for (const int h : {H_GL2SH_B, H_SH2RF_B}) { apply_list_looped<TAR, 1>(ListRegs(h), b); b[0] = (TIN)b[0]; }
      if (!(a[0] == 0 || b[0] == 0))
        for (int k = 0; k < K; ++k)
#pragma unroll
          for (int x = 0; x < COUNT; ++x)
            acc[x / 4 % FM][x / 4 / FM][x % 4] = fpu_fma<TACC>((TACC)a[0], (TACC)b[0], acc[x / 4 % FM][x / 4 / FM][x % 4]);
    }
  } else if (!oa.vectors_fit() || !ob.vectors_fit()) {
    // an operand with fewer than V rows (or k) along its contiguous index: element by element, one tile ahead
    typename decltype(oa)::vec xa[PA];
    typename decltype(ob)::vec xb[PB];
    auto fetch = [&](int k0) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < PA; ++i) xa[i] = oa.fetch_slow(i, k0);
#pragma unroll
      for (int i = 0; i < PB; ++i) xb[i] = ob.fetch_slow(i, k0);
    };
    fetch(0);
    load_c();
    for (int kt = 0; kt < KT; ++kt) {
      block_barrier();
      lists(xa, xb);
#pragma unroll
      for (int i = 0; i < PA; ++i) oa.store(lds, oa.cut(oa.scaled(xa[i]), i, kt * BK), i);
#pragma unroll
      for (int i = 0; i < PB; ++i) ob.store(lds + Cfg::A_ELEMS, ob.cut(ob.scaled(xb[i]), i, kt * BK), i);
      wait_lgkmcnt0();
      block_barrier();
      if (kt + 1 < KT) fetch((kt + 1) * BK);
      const int left = (K - kt * BK + 3) / 4;
      for (int s = 0; s < (left < STEPS ? left : STEPS); ++s) {
        read(0, lds, s);
        multiply(0);
      }
      wait_lgkmcnt0();
    }
  } else if (Cfg::FUSED == 2 || (!Cfg::A_KMAJOR && edge_m) || (!Cfg::B_KMAJOR && edge_n)) {
    if (Cfg::FUSED == 1 && args.scale_b != 1.0f) pipeline(std::true_type{}, std::true_type{});
    else pipeline(std::true_type{}, std::false_type{});
  } else {
    if (Cfg::FUSED == 1 && args.scale_b != 1.0f) pipeline(std::false_type{}, std::true_type{});
    else pipeline(std::false_type{}, std::false_type{});
  }

  if constexpr (Cfg::SPLITK) {
    // every slice of K leaves its partial tile in the workspace; the last one to arrive adds them up in slice order
    // and goes on to the epilogue, the others are done
    block_barrier();         // every wave is done with the LDS tiles: the first word now carries the arrival count
    if (!splitk_reduce<Cfg::THREADS, TACC>(acc, args, ti + tj * args.nbm, (unsigned*)smem)) return;
  }

  // epilogue: transform, bias, transform, store; the bias of Epilogue.Bias is fp32 (reference src/epilogue.jl:44-52) and
  // only offered with fp32 accumulators
  TACC* D = (TACC*)args.d;
  // (one look at all three arguments: a wait for each, one behind another, is part of the end of every launch)
  if (Cfg::FUSED != 0 && (args.t[H_RF2SH_D].n | args.t[H_SH2GL_D].n | args.epi_kind) != 0) {
    hook_acc(H_RF2SH_D);
    if constexpr (std::is_same<TACC, float>::value) {
      if (args.epi_kind == 1) {
#pragma unroll
        for (int fj = 0; fj < FN; ++fj) {
          const int cc = col_of(fj, 0);
          const float bv = args.bias[cc < args.N ? cc : 0];
#pragma unroll
          for (int fi = 0; fi < FM; ++fi)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[fi][fj][r] += bv;
        }
      } else if (args.epi_kind == 2) {
#pragma unroll
        for (int fi = 0; fi < FM; ++fi)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int rr = row_of(fi, r);
            const float bv = args.bias[rr < args.M ? rr : 0];
#pragma unroll
            for (int fj = 0; fj < FN; ++fj) acc[fi][fj][r] += bv;
          }
      }
    }
    hook_acc(H_SH2GL_D);
  }
#pragma unroll
  for (int fj = 0; fj < FN; ++fj)
#pragma unroll
    for (int fi = 0; fi < FM; ++fi) {
      if (WIDE && !edge_m && !edge_n) {
        ((loose_acc*)(D + row_of(fi, 0) + (long long)col_of(fj, 0) * args.ldd))->v = acc[fi][fj];
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int rr = row_of(fi, r), cc = col_of(fj, r);
          if (rr < args.M && cc < args.N) D[rr + (long long)cc * args.ldd] = acc[fi][fj][r];
        }
      }
    }
}

}  // namespace gk
