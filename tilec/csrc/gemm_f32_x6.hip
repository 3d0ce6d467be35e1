// fp32 GEMM on the bf16 matrix cores, C[M,N] = A[M,K] · B[K,N] (each operand
// row- or column-major, read in place at any 4-byte alignment).
//
// Same tile semantics as the reference tile kernel `_matmul_tiled`
// (tilec/ext.py:13-24): zero accumulator, K steps over masked tiles with
// `other=0.0`, masked store.
//
// What bounds it: gfx950's fp32 MFMAs run at 1/16 of the bf16 rate, so a
// large fp32 product on them is bound by that unit (137 GFLOP at 4096^3 take
// 0.89 ms at its 157 TFLOP/s peak).  Here every fp32 value x is split exactly
// into three bf16 planes,
//   y = 2^16 x, hi = bf16(y), mid = bf16(y - hi), lo = bf16(y - hi - mid),  y = hi + mid + lo
// (8 significand bits each, round to nearest; both differences are exact; the
// split and its six products are a published method: Henry, Tang and Heinecke,
// "Leveraging the bfloat16 Artificial Intelligence Datatype For
// Higher-Precision Computations", ARITH 2019), and the product is the six
// plane products of relative size 2^-16 and up,
//   hi hi + (hi mid + mid hi) + (hi lo + mid mid + lo hi),
// each exact in fp32 and accumulated in fp32: 6 x the MFMA work at 16 x the
// rate.  The three dropped products are below 2^-24 of the term they belong
// to, half an ulp of it, and the MFMA adds 16 products per rounding of the
// accumulator where the fp32 MFMA adds 2, so from 3 products an output on the
// result is closer to the exact one than the fp32 MFMA's (1 or 2 products:
// 3.5e-8 and 2.6e-8, without and with LOW, against 2.5e-8 to 3.2e-8).
//
// Range.  bf16 has the exponents of fp32 and 16 bits less, so the low planes of
// a value under 2^-110 would fall below bf16's smallest subnormal, 2^-133.  The
// factor 2^16 lifts every fp32 value, subnormals too, far enough (the least bit
// of a subnormal, 2^-149, to 2^-133; the matrix cores keep bf16 and fp32
// subnormals), and a product that is a normal fp32 number lifts the terms of
// its plane products above 2^-142.  So the split is exact for every element on
// its own, whatever else its row or column holds.  The sums are 2^32 times the
// result and are multiplied by 2^-32 at the end.  What the factor takes is the
// other end: a value of 2^112 (5e33) or a sum of 2^96 (8e28) overflows, as an
// infinity or NaN would, into a sum that is not finite.  Each wave tests its
// sums after the K loop and multiplies the row blocks that hold such a one
// again on the fp32 MFMAs, which gives them the fp32 kernels' results.  On
// MI355X, 4096^3 in 256 x 256 tiles: 0.57 ms; one infinity in x1 0.71 ms
// (every column tile redoes one row block); every sum NaN or above 2^96 1.45
// to 1.54 ms.  The fp32 MFMA kernel takes 0.91 ms whatever the data.  (Without loads in
// flight, and the wave's whole part at a time: 2.05 and 2.77 ms.)
//
// Data movement.  A K step's tiles go global -> registers -> LDS: a thread
// loads 8 consecutive k of one row ("chunk"; two 16-byte loads of a
// k-contiguous operand, eight 4-byte loads along k of an r-contiguous one,
// coalesced over lanes), splits them (6.5 VALU operations a value, beside the
// other waves' MFMAs) and stores three 16-byte chunks, which are the MFMA
// operands as they are: LDS holds chunk (plane, kg, r) at
// (plane KG + kg) R + (r ^ swz(kg)), so reads of 32 consecutive rows and the
// stores of both thread mappings are free of bank conflicts.  Three LDS
// stages and PF register sets: loads run PF + 2 K steps ahead (PF = 4 on the
// 8-wave 128 x 128 tile, whose steps are short; the larger tiles' registers
// hold one set).  Splitting in the kernel
// reads each operand at 4 bytes a value; a pass that wrote three planes to
// memory first would move 10 bytes a value and the GEMM 6.
// A K step that is not whole is taken first, with loads masked one by one,
// so the loop has no edge in K.
//
// Measured on MI355X against the fp32 MFMA kernels: 4096^3 565 against 914 us
// (256 x 256, 8 waves; matrix cores 76 % busy at 1.77 GHz, the power limit;
// relative error 1.0e-6 against 1.1e-6), 2048^3 94 against 126 us (128 x 128,
// 8 waves; error 2.7e-7 against 8.1e-7), 1000 x 4097 x 3001 143 against 204 us
// (128 x 128, 4 waves, two workgroups a CU, K split 4; no padding copies).
// Those 128-tiles keep the matrix cores 48 and 51 % busy, with 5 VALU
// instructions an MFMA (2.4 in the 256-tile).
// The 128-tiles keep the five small products in sums of their own (LOW),
// which their registers allow; the 256-tile's do not.
#include <type_traits>

#include "common.h"
#include "../../include/tilec.h"

namespace tilec {

namespace {

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

constexpr float kScale = 0x1p16f, kUnscale = 0x1p-32f;

// 8 fp32 values -> three planes of 8 bf16 (hi, mid, lo) of kScale times them,
// rounded to nearest.
// (Splitting with integer adds and permutes, or with dot products by (-1, 0)
// for the differences, measured level and 5 % slower.)
__device__ __forceinline__ void split3(const float (&x)[8], u32x4 (&p)[3]) {
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    float a = kScale * x[2 * j], b = kScale * x[2 * j + 1];
#pragma unroll
    for (int s = 0; s < 3; ++s) {
      uint32_t w = __builtin_bit_cast(uint32_t, bf16x2{(__bf16)a, (__bf16)b});
      asm("" : "+v"(w));  // one conversion of the pair, not one more of each half
      p[s][j] = w;
      if (s < 2) {
        a -= __uint_as_float(w << 16);
        b -= __uint_as_float(w & 0xffff0000u);
      }
    }
  }
}

// One operand's tile of R rows (M of x1, N of x2) by BK of K.  KC: element
// (r, k) at X[r * ld + k]; otherwise at X[k * ld + r].
template <int R, int BK, int NT, bool KC>
struct Op6 {
  static constexpr int KG = BK / 8;         // 8-deep k groups per step
  static constexpr int Q = R * KG / NT;     // chunks per thread
  static constexpr int PLANE = R * KG;      // chunks per plane
  static constexpr int BYTES = 3 * PLANE * 16;
  static_assert(R * KG % NT == 0, "chunks must divide evenly");
  static_assert(KG == 2 || KG == 4 || KG == 8, "swizzle");
  typedef float Regs[Q][8];

  __device__ __forceinline__ static void coord(int tid, int q, int& r, int& kg) {
    const int e = tid + q * NT;
    if constexpr (KC) {
      r = e / KG;
      kg = e % KG;
    } else {
      r = e % R;
      kg = e / R;
    }
  }
  // LDS byte offset of chunk (plane 0, kg, r).
  __device__ __forceinline__ static uint32_t at(int kg, int r) { return 16u * (uint32_t)(kg * R + (r ^ (kg * (8 / KG)))); }
};

__device__ __forceinline__ float load_f32_s(BufRsrc r, uint32_t voff, uint32_t soff) {
  return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, (int)voff, (int)soff, 0));
}
// A wave-uniform value in a scalar register: a load whose scalar offset the
// compiler moved to a vector register sits in a waterfall loop.
__device__ __forceinline__ uint32_t to_scalar(uint32_t v) {
  asm("" : "+v"(v));
  return (uint32_t)__builtin_amdgcn_readfirstlane((int)v);
}
__device__ __forceinline__ f32x4 load_f32x4_s(BufRsrc r, uint32_t voff, uint32_t soff) {
  return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)voff, (int)soff, 0));
}

template <int BM, int BN, int BK, int WM, int WN, bool CA, bool CB>
struct Gemm6 {
  static constexpr int NT = WM * WN * 64;
  static constexpr int WTM = BM / WM, WTN = BN / WN;
  static constexpr int TM = WTM / 32, TN = WTN / 32;
  using OA = Op6<BM, BK, NT, !CA>;
  using OB = Op6<BN, BK, NT, CB>;
  static constexpr int STAGE = OA::BYTES + OB::BYTES;
  static_assert(WTM % 32 == 0 && WTN % 32 == 0, "wave tile must be whole 32x32 blocks");
  static_assert(3 * STAGE + 16 <= 160 * 1024, "LDS is 160 KiB");
};

// c = TN 32 x 32 blocks of products over `len` k on the fp32 MFMAs, operands
// straight from memory.  `a` and `b`: the tile's first row and column at the
// first k; this lane's row and columns are byte offsets from there (kOob past
// the end) of k = 4 half.  Eight k a step, half h of the wave takes
// 4 h .. 4 h + 3; SETS steps of loads in flight.  KA, KB: k contiguous.
template <int TN, bool KA, bool KB>
__device__ __forceinline__ void fp32_block(f32x16 (&c)[TN], const float* a, const float* b, int64_t lda, int64_t ldb,
                                           uint32_t off_a, const uint32_t (&off_b)[TN], int len, int half) {
  constexpr int SETS = 4;
  float xa[SETS][4], xb[SETS][TN][4];
  uint32_t k_a[4], k_b[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    k_a[e] = KA ? 4u * e : to_scalar(4u * e * (uint32_t)lda);
    k_b[e] = KB ? 4u * e : to_scalar(4u * e * (uint32_t)ldb);
  }
  auto four = [](auto kc, float (&x)[4], const BufRsrc& rs, uint32_t off, const uint32_t (&k)[4])
      __attribute__((always_inline)) {
    if constexpr (decltype(kc)::value) {
      const f32x4 v = load_f32x4_s(rs, off, 0);
#pragma unroll
      for (int e = 0; e < 4; ++e) x[e] = v[e];
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) x[e] = load_f32_s(rs, off, k[e]);
    }
  };
  auto mma = [&](const float (&x)[4], const float (&y)[TN][4]) __attribute__((always_inline)) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int j = 0; j < TN; ++j) c[j] = mfma32x32x2(x[e], y[j][e], c[j]);
  };
#pragma unroll
  for (int j = 0; j < TN; ++j)
#pragma unroll
    for (int r = 0; r < 16; ++r) c[j][r] = 0.f;
  const int64_t a_step = KA ? 8 : 8 * lda, b_step = KB ? 8 : 8 * ldb;
  int left = len;  // k not loaded yet; loads past the last whole step return zeros
  auto load = [&](int p) __attribute__((always_inline)) {
    const uint32_t recs = left >= 8 ? 0x7FFFFFFFu : 0u;
    const BufRsrc ra = make_rsrc_uniform(a, recs), rb = make_rsrc_uniform(b, recs);
    four(std::bool_constant<KA>{}, xa[p], ra, off_a, k_a);
#pragma unroll
    for (int j = 0; j < TN; ++j) four(std::bool_constant<KB>{}, xb[p][j], rb, off_b[j], k_b);
    if (left >= 8) {
      a += a_step;
      b += b_step;
      left -= 8;
    }
  };
#pragma unroll
  for (int p = 0; p < SETS; ++p) load(p);
#pragma unroll 1
  for (int s = 0; s < len / 8; s += SETS)
#pragma unroll
    for (int p = 0; p < SETS; ++p) {
      mma(xa[p], xb[p]);
      load(p);
    }
  if (left > 0) {
    const BufRsrc ra = make_rsrc_uniform(a, 0x7FFFFFFFu), rb = make_rsrc_uniform(b, 0x7FFFFFFFu);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const bool in = 4 * half + e < left;
      xa[0][e] = load_f32_s(ra, in ? off_a : kOob, k_a[e]);
#pragma unroll
      for (int j = 0; j < TN; ++j) xb[0][j][e] = load_f32_s(rb, in ? off_b[j] : kOob, k_b[e]);
    }
    mma(xa[0], xb[0]);
  }
}

// Scheduling of one row block: its NM MFMAs in order, the LDS reads of the
// next operands behind the first ones, and behind every MFMA a few of the
// VALU operations that split chunks.
template <int NM, int X = 0>
__device__ __forceinline__ void sched_block() {
  if constexpr (X < NM) {
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    if constexpr (X < NM / 2) __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
    __builtin_amdgcn_sched_group_barrier(0x002, 6, 0);
    if constexpr (X >= NM / 2) __builtin_amdgcn_sched_group_barrier(0x200, 2, 0);
    if constexpr (X >= NM / 2) __builtin_amdgcn_sched_group_barrier(0x020, 2, 0);
    sched_block<NM, X + 1>();
  }
}

template <int BM, int BN, int BK, int WM, int WN, int PF, bool CA, bool CB, int WPE, bool LOW>
__global__ __launch_bounds__(WM * WN * 64, WPE) void gemm_f32_x6_kernel(
    const float* __restrict__ A, const float* __restrict__ B, float* __restrict__ C, int M, int N, int K, int64_t lda,
    int64_t ldb, int64_t ldc, int group_m, int xcds, int split_steps, float* __restrict__ ws,
    unsigned* __restrict__ counters) {
  using P = Gemm6<BM, BN, BK, WM, WN, CA, CB>;
  using OA = typename P::OA;
  using OB = typename P::OB;
  constexpr int TM = P::TM, TN = P::TN;
  __shared__ int last_flag;
  __shared__ __align__(16) char lds[3 * P::STAGE];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WN, wn = wave % WN;
  const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
  int tm, tn;
  tile_of(blockIdx.x, xcds, tiles_m, tiles_n, group_m, tm, tn);
  const int m0 = tm * BM, n0 = tn * BN;
  // K steps [kt0, kt1) of this workgroup (grid y = K splits); the step past
  // the last whole one (if it is this workgroup's) is taken first.
  const int split = blockIdx.y, S = gridDim.y;
  const int kt0 = split * split_steps;
  const int kt1 = min((K + BK - 1) / BK, kt0 + split_steps);
  const int nk = max(0, kt1 - kt0);
  const bool tail = nk > 0 && kt1 * BK > K;
  const int whole = nk - (tail ? 1 : 0);

  uint32_t off_a[OA::Q], off_b[OB::Q];
#pragma unroll
  for (int q = 0; q < OA::Q; ++q) {
    int r, kg;
    OA::coord(tid, q, r, kg);
    const uint32_t o = 4u * (CA ? 8u * kg * (uint32_t)lda + r : (uint32_t)r * (uint32_t)lda + 8u * kg);
    off_a[q] = m0 + r < M ? o : kOob;
  }
#pragma unroll
  for (int q = 0; q < OB::Q; ++q) {
    int r, kg;
    OB::coord(tid, q, r, kg);
    const uint32_t o = 4u * (!CB ? 8u * kg * (uint32_t)ldb + r : (uint32_t)r * (uint32_t)ldb + 8u * kg);
    off_b[q] = n0 + r < N ? o : kOob;
  }
  const float* a_next = !CA ? A + (int64_t)m0 * lda + (int64_t)kt0 * BK : A + (int64_t)kt0 * BK * lda + m0;
  const float* b_next = CB ? B + (int64_t)n0 * ldb + (int64_t)kt0 * BK : B + (int64_t)kt0 * BK * ldb + n0;
  const int64_t a_step = !CA ? BK : (int64_t)BK * lda;
  const int64_t b_step = CB ? BK : (int64_t)BK * ldb;

  // Byte offsets of the 8 k of an r-contiguous chunk.
  uint32_t k_a[8], k_b[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    k_a[e] = CA ? to_scalar(4u * e * (uint32_t)lda) : 0u;
    k_b[e] = !CB ? to_scalar(4u * e * (uint32_t)ldb) : 0u;
  }

  typename OA::Regs xa[PF];
  typename OB::Regs xb[PF];
  // Resources of the next whole K step; past the last one (w >= whole) its
  // loads return zeros.
  BufRsrc sa = make_rsrc(A), sb = make_rsrc(B);
  int w = 0;
  auto next_step = [&]() __attribute__((always_inline)) {
    const uint32_t recs = w < whole ? 0x7FFFFFFFu : 0u;
    sa = make_rsrc_uniform(a_next, recs);
    sb = make_rsrc_uniform(b_next, recs);
    a_next += a_step;
    b_next += b_step;
    ++w;
  };
  auto load_chunk = [](auto kc, const BufRsrc& rs, float (&x)[8], uint32_t off, const uint32_t (&k)[8])
      __attribute__((always_inline)) {
    if constexpr (decltype(kc)::value) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const f32x4 v = load_f32x4_s(rs, off, 16 * h);
#pragma unroll
        for (int c = 0; c < 4; ++c) x[4 * h + c] = v[c];
      }
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] = load_f32_s(rs, off, k[e]);
    }
  };
  // Chunk c of the step (A's first, then B's) into register set p.
  constexpr int CH = OA::Q + OB::Q;
  auto load = [&](int p, int c) __attribute__((always_inline)) {
    if (c < OA::Q) load_chunk(std::bool_constant<!CA>{}, sa, xa[p][c], off_a[c], k_a);
    else load_chunk(std::bool_constant<CB>{}, sb, xb[p][c - OA::Q], off_b[c - OA::Q], k_b);
  };
  // The K step that is not whole, element by element.
  auto load_tail = [&]() __attribute__((always_inline)) {
    const int k0 = (kt1 - 1) * BK;
    const BufRsrc ta = make_rsrc_uniform(!CA ? A + (int64_t)m0 * lda + k0 : A + (int64_t)k0 * lda + m0, 0x7FFFFFFFu);
    const BufRsrc tb = make_rsrc_uniform(CB ? B + (int64_t)n0 * ldb + k0 : B + (int64_t)k0 * ldb + n0, 0x7FFFFFFFu);
#pragma unroll
    for (int q = 0; q < OA::Q; ++q) {
      int r, kg;
      OA::coord(tid, q, r, kg);
#pragma unroll
      for (int e = 0; e < 8; ++e)
        xa[0][q][e] = load_f32_s(ta, k0 + 8 * kg + e < K ? off_a[q] : kOob, !CA ? 4u * e : k_a[e]);
    }
#pragma unroll
    for (int q = 0; q < OB::Q; ++q) {
      int r, kg;
      OB::coord(tid, q, r, kg);
#pragma unroll
      for (int e = 0; e < 8; ++e)
        xb[0][q][e] = load_f32_s(tb, k0 + 8 * kg + e < K ? off_b[q] : kOob, CB ? 4u * e : k_b[e]);
    }
  };

  auto put = [&](auto op, const float (&x)[8], int q, char* area) __attribute__((always_inline)) {
    using O = decltype(op);
    int r, kg;
    O::coord(tid, q, r, kg);
    u32x4 p[3];
    split3(x, p);
    char* d = area + O::at(kg, r);
#pragma unroll
    for (int s = 0; s < 3; ++s) *reinterpret_cast<u32x4*>(d + 16 * O::PLANE * s) = p[s];
  };
  auto store = [&](int p, int c, char* st) __attribute__((always_inline)) {
    if (c < OA::Q) put(OA{}, xa[p][c], c, st);
    else put(OB{}, xb[p][c - OA::Q], c - OA::Q, st + OA::BYTES);
  };

  f32x16 acc[TM][TN], low[LOW ? TM : 1][TN];
  auto clear = [](auto& c) __attribute__((always_inline)) {
#pragma unroll
    for (auto& row : c)
#pragma unroll
      for (auto& blk : row)
#pragma unroll
        for (int r = 0; r < 16; ++r) blk[r] = 0.f;
  };
  clear(acc);
  clear(low);

  const int half = lane >> 5;
  const int a_r = wm * P::WTM + (lane & 31), b_r = wn * P::WTN + (lane & 31);
  struct Planes {
    bf16x8 p[3];
  };
  auto read = [&](auto op, const char* area, int r, int ks) __attribute__((always_inline)) -> Planes {
    using O = decltype(op);
    const char* d = area + O::at(2 * ks + half, r);
    Planes f;
#pragma unroll
    for (int s = 0; s < 3; ++s) f.p[s] = *reinterpret_cast<const bf16x8*>(d + 16 * O::PLANE * s);
    return f;
  };
  // The products of row block i, small ones first.  LOW: the five small ones
  // go to sums of their own, which meet the running sum after the K loop, so
  // that it is rounded once per 16 k and not six times.
  auto row_block = [&](int i, const Planes& a, const Planes (&b)[TN]) __attribute__((always_inline)) {
    constexpr int PA[6] = {2, 1, 0, 1, 0, 0}, PB[6] = {0, 1, 2, 0, 1, 0};
#pragma unroll
    for (int q = 0; q < 6; ++q)
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        f32x16& c = LOW && q < 5 ? low[LOW ? i : 0][j] : acc[i][j];
        c = mfma32x32x16bf16(a.p[PA[q]], b[j].p[PB[q]], c);
      }
  };
  auto barrier = [&]() __attribute__((always_inline)) {
    // lgkmcnt(0): this wave's LDS reads and writes are done; global loads stay in flight
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(15 | (3 << 14) | (7 << 4));
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };

  constexpr int KS = BK / 16;
  // Row block x of a step's KS * TM: the chunks it stores to `st` from
  // register set p, and whose registers it then loads PF steps further on.
  constexpr int NB = KS * TM, CPB = (CH + NB - 1) / NB;
  auto chunks = [&](int p, int x, char* st) __attribute__((always_inline)) {
    if (x == 0) next_step();
#pragma unroll
    for (int c = x * CPB; c < (x + 1) * CPB && c < CH; ++c) {
      store(p, c, st);
      load(p, c);
    }
  };
  // Three LDS stages (byte offsets, scalars): step s computes from one and,
  // before the barrier that ends it, reads the first operands of step s + 1
  // (stored a step before, so complete); step s + 2 is split into the third
  // stage; steps s + 3 .. s + PF + 2 are in flight to the PF register sets.
  int cur = 0, nxt = P::STAGE, nn = 2 * P::STAGE;
  if (nk > 0) {
#pragma unroll
    for (int p = 0; p < PF; ++p) {
      if (p == 0 && tail) {
        load_tail();
        continue;
      }
      next_step();
#pragma unroll
      for (int c = 0; c < CH; ++c) load(p, c);
    }
#pragma unroll
    for (int d = 0; d < 2; ++d) {
      next_step();
#pragma unroll
      for (int c = 0; c < CH; ++c) {
        store(d % PF, c, lds + d * P::STAGE);
        load(d % PF, c);
      }
    }
    barrier();
    Planes a[2], b[2][TN];
    a[0] = read(OA{}, lds, a_r, 0);
#pragma unroll
    for (int j = 0; j < TN; ++j) b[0][j] = read(OB{}, lds + OA::BYTES, b_r + 32 * j, 0);
    // Step s, I = s % U.  Operand sets alternate over the KS * TM row blocks
    // (A) and the KS k-slices (B) of a step, so the step's parity picks them
    // where those counts are odd.
    constexpr int U = PF % 2 == 0 ? PF : 2 * PF;
    auto step = [&](auto I) __attribute__((always_inline)) {
      constexpr int I0 = decltype(I)::value;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const bool last_k = ks + 1 == KS;
        const int bs = (I0 * KS + ks) & 1;
#pragma unroll
        for (int i = 0; i < TM; ++i) {
          const int as = (I0 * KS * TM + ks * TM + i) & 1;
          const bool last = i + 1 == TM;
          a[as ^ 1] = read(OA{}, lds + (last && last_k ? nxt : cur), a_r + (last ? 0 : 32 * (i + 1)),
                           last ? (last_k ? 0 : ks + 1) : ks);
          if (last) {
#pragma unroll
            for (int j = 0; j < TN; ++j)
              b[bs ^ 1][j] = read(OB{}, lds + (last_k ? nxt : cur) + OA::BYTES, b_r + 32 * j, last_k ? 0 : ks + 1);
          }
          chunks((I0 + 2) % PF, ks * TM + i, lds + nn);
          row_block(i, a[as], b[bs]);
          sched_block<6 * TN>();
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      barrier();
      const int t = cur;
      cur = nxt;
      nxt = nn;
      nn = t;
    };
    int s = 0;
#pragma unroll 1
    for (; s + U <= nk; s += U) {
      step(std::integral_constant<int, 0>{});
      step(std::integral_constant<int, 1>{});
      if constexpr (U > 2) {
        step(std::integral_constant<int, 2>{});
        step(std::integral_constant<int, 3>{});
      }
    }
    if (s < nk) step(std::integral_constant<int, 0>{});
    if constexpr (U > 2) {
      if (s + 1 < nk) step(std::integral_constant<int, 1>{});
      if (s + 2 < nk) step(std::integral_constant<int, 2>{});
    }
    if constexpr (LOW) {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
          for (int r = 0; r < 16; ++r) acc[i][j][r] += low[i][j][r];
    }
  }

  // Sums that are not finite (see above): their row blocks again.
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    bool bad = false;
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        bad |= !(fabsf(acc[i][j][r]) <= 3.402823466e38f);
        acc[i][j][r] *= kUnscale;
      }
    if (__ballot(bad) == 0) continue;
    const int ra = a_r + 32 * i;
    const uint32_t fa =
        m0 + ra < M ? 4u * (CA ? 4u * half * (uint32_t)lda + ra : (uint32_t)ra * (uint32_t)lda + 4u * half) : kOob;
    uint32_t fb[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int rb = b_r + 32 * j;
      fb[j] = n0 + rb < N ? 4u * (!CB ? 4u * half * (uint32_t)ldb + rb : (uint32_t)rb * (uint32_t)ldb + 4u * half) : kOob;
    }
    fp32_block<TN, !CA, CB>(acc[i], !CA ? A + (int64_t)m0 * lda + (int64_t)kt0 * BK : A + (int64_t)kt0 * BK * lda + m0,
                            CB ? B + (int64_t)n0 * ldb + (int64_t)kt0 * BK : B + (int64_t)kt0 * BK * ldb + n0, lda, ldb,
                            fa, fb, min(K, kt1 * BK) - kt0 * BK, half);
  }

  const bool interior = (m0 + BM <= M) && (n0 + BN <= N);
  const int row_base = m0 + wm * P::WTM + 4 * half;
  const int col_base = n0 + b_r;
  if (S > 1 && !splitk_tile<TM, TN, P::NT>(acc, split, S, blockIdx.x, gridDim.x, ws, counters, &last_flag, row_base,
                                           col_base, M, N))
    return;
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int gn = col_base + 32 * j;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int gm = row_base + 32 * i + 8 * (r >> 2) + (r & 3);
        if (interior || (gm < M && gn < N)) C[(int64_t)gm * ldc + gn] = acc[i][j][r];
      }
    }
}

// ---------------------------------------------------------------------------
// The same products with K shared out inside the workgroup, for outputs of too
// few tiles to keep the staged kernel's CUs busy: a workgroup owns a 64 x 64
// tile and its W waves share K, wave w taking the 16-deep steps w, w + W, ...
// of the workgroup's.  Every wave loads its own operands straight into
// registers (chunks of 8 consecutive k, which split into MFMA operands as
// they are), so the K loop has no barrier, no LDS traffic and no wait but for
// its own loads; the waves' sums meet in LDS in wave order.  A step
// issues 10 VALU instructions an MFMA.  On MI355X, 1024^3 back to back: 22 us
// (the direct-to-LDS 64 x 64 tile on the fp32 MFMAs 23), error 2.4e-7 against
// 5.7e-7; 512 x 1000 x 2048 20.2 us, 27.0 for a staged 64 x 64 x 32 tile of the
// kernel above.  A ring of direct-to-LDS copies in front of the registers
// measured no faster.
// ---------------------------------------------------------------------------
template <int NM, int X = 0>
__device__ __forceinline__ void sched_direct() {
  if constexpr (X < NM) {
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    __builtin_amdgcn_sched_group_barrier(0x002, 8, 0);
    sched_direct<NM, X + 1>();
  }
}

template <int W, bool CA, bool CB>
__global__ __launch_bounds__(W * 64, 2) void gemm_f32_x6_direct_kernel(
    const float* __restrict__ A, const float* __restrict__ B, float* __restrict__ C, int M, int N, int K, int64_t lda,
    int64_t ldb, int64_t ldc, int group_m, int xcds, int split_steps, float* __restrict__ ws,
    unsigned* __restrict__ counters) {
  constexpr int T = 64, NT = 64 * W;
  constexpr int RS = T + 4;              // row stride of a wave's sums in LDS
  constexpr int ITEMS = T * T / 4 / NT;  // float4 results per thread
  static_assert(T * T % (4 * NT) == 0 && W * T * RS * 4 + 64 <= 160 * 1024, "results divide, LDS fits");
  __shared__ __align__(16) float sums[W * T * RS];
  __shared__ int flag, last_flag;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int half = lane >> 5, l32 = lane & 31;
  const int tiles_m = (M + T - 1) / T, tiles_n = (N + T - 1) / T;
  int tm, tn;
  tile_of(blockIdx.x, xcds, tiles_m, tiles_n, group_m, tm, tn);
  const int m0 = tm * T, n0 = tn * T;
  const int split = blockIdx.y, S = gridDim.y;
  const int kt0 = split * split_steps;
  const int kt1 = min((K + 15) / 16, kt0 + split_steps);
  // This wave's steps kt0 + wave + i W; the one that is not whole, if it is
  // this wave's, is taken first.
  const int mine = kt1 - kt0 > wave ? (kt1 - kt0 - wave + W - 1) / W : 0;
  const bool tail = mine > 0 && kt1 * 16 > K && (kt1 - 1 - kt0) % W == wave;
  const int whole = mine - (tail ? 1 : 0);

  if (tid == 0) flag = 0;
  __syncthreads();

  // Chunk c of a step: rows 32 c + l32 of A (c < 2), then 32 (c - 2) + l32 of
  // B, k = 8 half .. + 7.
  uint32_t off[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const int r = 32 * (c & 1) + l32;
    const uint32_t ld = (uint32_t)(c < 2 ? lda : ldb);
    const bool kc = c < 2 ? !CA : CB;
    const uint32_t o = 4u * (kc ? (uint32_t)r * ld + 8u * half : 8u * half * ld + (uint32_t)r);
    off[c] = (c < 2 ? m0 + r < M : n0 + r < N) ? o : kOob;
  }
  uint32_t k_a[8], k_b[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    k_a[e] = CA ? to_scalar(4u * e * (uint32_t)lda) : 0u;
    k_b[e] = !CB ? to_scalar(4u * e * (uint32_t)ldb) : 0u;
  }
  auto base_a = [&](int step) {
    return !CA ? A + (int64_t)m0 * lda + (int64_t)step * 16 : A + (int64_t)step * 16 * lda + m0;
  };
  auto base_b = [&](int step) {
    return CB ? B + (int64_t)n0 * ldb + (int64_t)step * 16 : B + (int64_t)step * 16 * ldb + n0;
  };
  const float* a_next = base_a(kt0 + wave);
  const float* b_next = base_b(kt0 + wave);
  const int64_t a_step = !CA ? 16 * W : (int64_t)16 * W * lda;
  const int64_t b_step = CB ? 16 * W : (int64_t)16 * W * ldb;

  float x[2][4][8];
  int w = 0;
  auto load_step = [&](int p) __attribute__((always_inline)) {
    const uint32_t recs = w < whole ? 0x7FFFFFFFu : 0u;
    const BufRsrc sa = make_rsrc_uniform(a_next, recs), sb = make_rsrc_uniform(b_next, recs);
    a_next += a_step;
    b_next += b_step;
    ++w;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const BufRsrc& rs = c < 2 ? sa : sb;
      if (c < 2 ? !CA : CB) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const f32x4 v = load_f32x4_s(rs, off[c], 16 * h);
#pragma unroll
          for (int e = 0; e < 4; ++e) x[p][c][4 * h + e] = v[e];
        }
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) x[p][c][e] = load_f32_s(rs, off[c], c < 2 ? k_a[e] : k_b[e]);
      }
    }
  };

  // This wave's first step into set 0.
  auto first_step = [&]() __attribute__((always_inline)) {
    if (!tail) return load_step(0);
    const int k0 = (kt1 - 1) * 16;
    const BufRsrc sa = make_rsrc_uniform(base_a(kt1 - 1), 0x7FFFFFFFu);
    const BufRsrc sb = make_rsrc_uniform(base_b(kt1 - 1), 0x7FFFFFFFu);
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int e = 0; e < 8; ++e)
        x[0][c][e] = load_f32_s(c < 2 ? sa : sb, k0 + 8 * half + e < K ? off[c] : kOob,
                                (c < 2 ? !CA : CB) ? 4u * e : c < 2 ? k_a[e] : k_b[e]);
  };

  f32x16 acc[2][2];
  auto clear = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
  };
  clear();
  struct Planes {
    bf16x8 p[3];
  };
  Planes f[2][4];
  auto split_all = [&](int p, Planes (&d)[4]) __attribute__((always_inline)) {
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      u32x4 q[3];
      split3(x[p][c], q);
#pragma unroll
      for (int s = 0; s < 3; ++s) d[c].p[s] = __builtin_bit_cast(bf16x8, q[s]);
    }
  };
  auto multiply = [&](const Planes (&d)[4]) __attribute__((always_inline)) {
    // small products first
    constexpr int PA[6] = {2, 1, 0, 1, 0, 0}, PB[6] = {0, 1, 2, 0, 1, 0};
#pragma unroll
    for (int q = 0; q < 6; ++q)
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = mfma32x32x16bf16(d[i].p[PA[q]], d[2 + j].p[PB[q]], acc[i][j]);
  };

  if (mine > 0) {
    // Step s multiplies f[s & 1] while step s + 1 is split into the other set
    // and the registers it came from are loaded for step s + 3.
    first_step();
    load_step(1);
    split_all(0, f[0]);
    load_step(0);
    auto step = [&](auto I) __attribute__((always_inline)) {
      constexpr int i = decltype(I)::value;
      split_all(i ^ 1, f[i ^ 1]);
      multiply(f[i]);
      sched_direct<24>();
      __builtin_amdgcn_sched_barrier(0);
      load_step(i ^ 1);
      __builtin_amdgcn_sched_barrier(0);
    };
    int s = 0;
#pragma unroll 1
    for (; s + 2 <= mine; s += 2) {
      step(std::integral_constant<int, 0>{});
      step(std::integral_constant<int, 1>{});
    }
    if (s < mine) multiply(f[0]);
  }

  // Sums that are not finite: the whole workgroup's again on the fp32 MFMAs,
  // from the same loads (operand e of a chunk is k = e in one half of the wave
  // and 8 + e in the other).
  bool redo = false;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        redo |= !(fabsf(acc[i][j][r]) <= 3.402823466e38f);
        acc[i][j][r] *= kUnscale;
      }
  if (redo) flag = 1;
  __syncthreads();
  if (flag) {
    clear();
    if (mine > 0) {
      auto multiply32 = [&](int p) __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < 8; ++e)
#pragma unroll
          for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) acc[i][j] = mfma32x32x2(x[p][i][e], x[p][2 + j][e], acc[i][j]);
      };
      a_next = base_a(kt0 + wave);
      b_next = base_b(kt0 + wave);
      w = 0;
      first_step();
      load_step(1);
      int s = 0;
#pragma unroll 1
      for (; s + 2 <= mine; s += 2) {
        multiply32(0);
        load_step(0);
        multiply32(1);
        load_step(1);
      }
      if (s < mine) multiply32(0);
    }
  }

  // The waves' sums, in wave order: thread t takes float4 t + q NT.
  float* const own = sums + wave * T * RS;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) own[(32 * i + 8 * (r >> 2) + 4 * half + (r & 3)) * RS + 32 * j + l32] = acc[i][j][r];
  __syncthreads();
  f32x4 v[ITEMS];
  bool live[ITEMS];
#pragma unroll
  for (int q = 0; q < ITEMS; ++q) {
    const int it = tid + q * NT, row = it / (T / 4), col = 4 * (it % (T / 4));
    v[q] = *reinterpret_cast<const f32x4*>(sums + row * RS + col);
#pragma unroll
    for (int u = 1; u < W; ++u) v[q] += *reinterpret_cast<const f32x4*>(sums + (u * T + row) * RS + col);
    live[q] = (m0 + row < M) & (n0 + col < N);
  }
  if (S > 1 && !splitk_combine<NT, ITEMS>(v, live, split, S, blockIdx.x, gridDim.x, ws, counters, &last_flag)) return;
  const bool vec = ldc % 4 == 0 && reinterpret_cast<uintptr_t>(C) % 16 == 0;
#pragma unroll
  for (int q = 0; q < ITEMS; ++q) {
    const int it = tid + q * NT, row = it / (T / 4), col = 4 * (it % (T / 4));
    if (!live[q]) continue;
    float* const d = C + (int64_t)(m0 + row) * ldc + n0 + col;
    if (vec && n0 + col + 4 <= N) {
      *reinterpret_cast<f32x4*>(d) = v[q];
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (n0 + col + e < N) d[e] = v[q][e];
    }
  }
}

template <int BM, int BN, int BK, int WM, int WN, int PF, int WPE, bool LOW, bool CA, bool CB>
hipError_t launch_layout6(const MatmulArgs& a) {
  using P = Gemm6<BM, BN, BK, WM, WN, CA, CB>;
  const int64_t tiles = cdiv(a.M, BM) * cdiv(a.N, BN);
  if (tiles == 0) return hipSuccess;
  const SplitGeom g = gemm_split_geom(a.K, BK, a.split_k);
  if (g.splits > 1 && P::TM * P::TN * 16 > kSplitMaxAccPerThread) return hipErrorInvalidConfiguration;
  hipLaunchKernelGGL((gemm_f32_x6_kernel<BM, BN, BK, WM, WN, PF, CA, CB, WPE, LOW>), dim3((unsigned)tiles, (unsigned)g.splits),
                     dim3(P::NT), 0, a.stream, static_cast<const float*>(a.x1), static_cast<const float*>(a.x2), a.out,
                     (int)a.M, (int)a.N, (int)a.K, a.ldx1, a.ldx2, a.ldo, 4, device_xcds(), (int)g.steps,
                     g.splits > 1 ? static_cast<float*>(a.workspace) : nullptr, g.splits > 1 ? a.counters : nullptr);
  return hipGetLastError();
}

template <int W, bool CA, bool CB>
hipError_t launch_direct6(const MatmulArgs& a) {
  const int64_t tiles = cdiv(a.M, 64) * cdiv(a.N, 64);
  if (tiles == 0) return hipSuccess;
  const SplitGeom g = gemm_split_geom(a.K, 16, a.split_k);
  hipLaunchKernelGGL((gemm_f32_x6_direct_kernel<W, CA, CB>), dim3((unsigned)tiles, (unsigned)g.splits), dim3(64 * W), 0,
                     a.stream, static_cast<const float*>(a.x1), static_cast<const float*>(a.x2), a.out, (int)a.M,
                     (int)a.N, (int)a.K, a.ldx1, a.ldx2, a.ldo, 4, device_xcds(), (int)g.steps,
                     g.splits > 1 ? static_cast<float*>(a.workspace) : nullptr, g.splits > 1 ? a.counters : nullptr);
  return hipGetLastError();
}

}  // namespace

// Byte offsets within a K step take 31 bits: (rows of the tile along the
// stride) * ld * 4.
template <int BM, int BN, int BK, int WM, int WN, int PF, int WPE, bool LOW>
hipError_t launch_gemm_f32_x6(const MatmulArgs& a) {
  switch (a.layout & 3) {
    case 0: return launch_layout6<BM, BN, BK, WM, WN, PF, WPE, LOW, false, false>(a);
    case TILEC_X1_COL_MAJOR: return launch_layout6<BM, BN, BK, WM, WN, PF, WPE, LOW, true, false>(a);
    case TILEC_X2_COL_MAJOR: return launch_layout6<BM, BN, BK, WM, WN, PF, WPE, LOW, false, true>(a);
    default: return launch_layout6<BM, BN, BK, WM, WN, PF, WPE, LOW, true, true>(a);
  }
}

template hipError_t launch_gemm_f32_x6<256, 256, 16, 2, 4, 1, 1, false>(const MatmulArgs&);
template hipError_t launch_gemm_f32_x6<128, 128, 16, 2, 2, 1, 2, true>(const MatmulArgs&);
template hipError_t launch_gemm_f32_x6<128, 128, 32, 2, 4, 4, 1, true>(const MatmulArgs&);

template <int W>
hipError_t launch_gemm_f32_x6_direct(const MatmulArgs& a) {
  switch (a.layout & 3) {
    case 0: return launch_direct6<W, false, false>(a);
    case TILEC_X1_COL_MAJOR: return launch_direct6<W, true, false>(a);
    case TILEC_X2_COL_MAJOR: return launch_direct6<W, false, true>(a);
    default: return launch_direct6<W, true, true>(a);
  }
}
template hipError_t launch_gemm_f32_x6_direct<4>(const MatmulArgs&);

}  // namespace tilec
