// bf16 GEMM for operands of any element alignment, C[M,N] (fp32) = A[M,K] ·
// B[K,N] (bf16, each row- or column-major, read in place), fp32 accumulate, on
// v_mfma_f32_32x32x16_bf16.
//
// Same tile semantics as the reference tile kernel `_matmul_tiled`
// (tilec/ext.py:13-24).  Rows that are not whole 16-byte groups (an odd K or
// N, a column slice at an odd offset) cannot take the direct-to-LDS copies of
// gemm_bf16_lds.hip.  Copying both operands into padded rows first costs a
// pass over them and a launch, which small products feel most (on MI355X, pad
// variant against this kernel: 326 x 4758 x 501 26.2 and 14.5 us, 97 x 200 x
// 137 7.7 and 5.2); large ones repay the copy (1359 x 4447 x 1009 33.6 and
// 40.6 us row-major, 33.1 and 34.6 with x2 column-major).  Here a
// K step goes global -> registers -> LDS with loads at the operands' own
// alignment (gfx950 takes global loads at any byte): 16 bytes along k of a
// k-contiguous operand; dwords of two columns at each of 8 k of an
// r-contiguous one, which byte permutes turn into two chunks of 8 consecutive
// k.  Memory latency is what a register-staged step is bound by, so loads run
// PF register sets (steps) ahead of the LDS store, which itself is two steps
// ahead of the MFMAs (three LDS stages, one barrier a step; a step's first
// operands are read before the barrier that ends the step before it).
// LDS holds chunk (kg, r) (8 consecutive k of row r) at kg R + (r ^ kg), which
// spreads 32 consecutive rows over all banks (300 x 2051 x 1001 row-major: 2 %
// of the cycles in bank conflicts).
//
// Edges: rows past M or N are clamped to the last (their results are not
// stored); a pair of columns past the end is moved down to the last pair (the
// permute then takes the other half); the K step that is not whole is taken
// first, its straddling chunk loaded from the row's last 8 elements and
// shifted.  So every load lies inside the matrix.  Needs K >= 8 and, along an
// r-contiguous extent, two elements (the launcher checks).
#include <type_traits>

#include "common.h"
#include "../../include/tilec.h"

namespace tilec {

namespace {

typedef unsigned short u16;

template <int R, int NT, bool KC>
struct OpAny {
  static constexpr int KG = 8;                     // 8-deep k groups per 64-deep step
  static constexpr int Q = R * KG / NT;            // chunks per thread
  static constexpr int UNITS = KC ? Q : Q / 2;     // loads' units: a chunk, or two columns' chunks
  static constexpr int WORDS = KC ? 4 : 8;         // dwords per unit
  static constexpr int BYTES = R * KG * 16;
  static_assert(R * KG % NT == 0 && (KC || Q % 2 == 0), "chunks must divide evenly");
  typedef uint32_t Regs[UNITS][WORDS];
  // Row (first of two unless KC) and k group of unit u.
  __device__ __forceinline__ static void coord(int tid, int u, int& r, int& kg) {
    const int e = tid + u * NT;
    if constexpr (KC) {
      r = e / KG;
      kg = e % KG;
    } else {
      r = 2 * (e % (R / 2));
      kg = e / (R / 2);
    }
  }
  __device__ __forceinline__ static uint32_t at(int kg, int r) { return 16u * (uint32_t)(kg * R + (r ^ kg)); }
};

// Byte loads at any alignment from a wave-uniform base.
__device__ __forceinline__ u32x4 load16(const char* base, uint32_t off) {
  u32x4 v;
  __builtin_memcpy(&v, base + off, 16);
  return v;
}
__device__ __forceinline__ uint32_t load4(const char* base, uint32_t off) {
  uint32_t v;
  __builtin_memcpy(&v, base + off, 4);
  return v;
}

template <int BM, int BN, int WM, int WN, int PF, bool CA, bool CB, int WPE>
__global__ __launch_bounds__(WM * WN * 64, WPE) void gemm_bf16_any_kernel(
    const u16* __restrict__ A, const u16* __restrict__ B, float* __restrict__ C, int M, int N, int K, int64_t lda,
    int64_t ldb, int64_t ldc, int group_m, int xcds, int split_steps, float* __restrict__ ws,
    unsigned* __restrict__ counters) {
  constexpr int BK = 64, NT = WM * WN * 64;
  constexpr int WTM = BM / WM, WTN = BN / WN, TM = WTM / 32, TN = WTN / 32;
  using OA = OpAny<BM, NT, !CA>;
  using OB = OpAny<BN, NT, CB>;
  constexpr int STAGE = OA::BYTES + OB::BYTES;
  static_assert(3 * STAGE + 16 <= 160 * 1024, "LDS is 160 KiB");
  static_assert(PF == 2 || PF == 4, "register sets");
  __shared__ int last_flag;
  __shared__ __align__(16) char lds[3 * STAGE];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WN, wn = wave % WN;
  const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
  int tm, tn;
  tile_of(blockIdx.x, xcds, tiles_m, tiles_n, group_m, tm, tn);
  const int m0 = tm * BM, n0 = tn * BN;
  const int split = blockIdx.y, S = gridDim.y;
  const int kt0 = split * split_steps;
  const int kt1 = min((K + BK - 1) / BK, kt0 + split_steps);
  const int nk = max(0, kt1 - kt0);
  const bool tail = nk > 0 && kt1 * BK > K;
  const int whole = nk - (tail ? 1 : 0);

  // Byte offset of each unit from the step's base (the tile's first row and
  // the step's first k), edges clamped; `last[u]`: the unit's first column is
  // the operand's last, read as the upper half of the pair below it.
  auto place = [&](auto op, int u, int64_t ld, int r0, int extent, bool& last) __attribute__((always_inline)) -> uint32_t {
    using O = decltype(op);
    int r, kg;
    O::coord(tid, u, r, kg);
    last = false;
    if constexpr (O::WORDS == 4) {
      r = min(r, extent - 1 - r0);
      return 2u * ((uint32_t)r * (uint32_t)ld + 8u * kg);
    } else {
      last = r0 + r == extent - 1;
      r = min(r0 + r, extent - 2) - r0;  // below the tile's first column (-1) where that is the last one
      return 2u * (8u * kg * (uint32_t)ld) + 2u * (uint32_t)(r + 1);
    }
  };
  uint32_t off_a[OA::UNITS], off_b[OB::UNITS], sel_a[OA::UNITS], sel_b[OB::UNITS];
#pragma unroll
  for (int u = 0; u < OA::UNITS; ++u) {
    bool last;
    off_a[u] = place(OA{}, u, lda, m0, M, last);
    sel_a[u] = last ? 0x07060302u : 0x05040100u;
  }
#pragma unroll
  for (int u = 0; u < OB::UNITS; ++u) {
    bool last;
    off_b[u] = place(OB{}, u, ldb, n0, N, last);
    sel_b[u] = last ? 0x07060302u : 0x05040100u;
  }
  // Base of K step `step`; r-contiguous offsets count from one column below
  // the tile's first.
  auto base_a = [&](int step) {
    return reinterpret_cast<const char*>(!CA ? A + (int64_t)m0 * lda + (int64_t)step * BK
                                             : A + (int64_t)step * BK * lda + m0 - 1);
  };
  auto base_b = [&](int step) {
    return reinterpret_cast<const char*>(CB ? B + (int64_t)n0 * ldb + (int64_t)step * BK
                                            : B + (int64_t)step * BK * ldb + n0 - 1);
  };
  const char* a_next = base_a(kt0);
  const char* b_next = base_b(kt0);
  const int64_t a_step = 2 * (!CA ? BK : (int64_t)BK * lda), b_step = 2 * (CB ? BK : (int64_t)BK * ldb);
  const int64_t a_row = 2 * lda, b_row = 2 * ldb;  // bytes between k-rows of an r-contiguous operand

  typename OA::Regs xa[PF];
  typename OB::Regs xb[PF];
  auto load_op = [&](auto op, auto& x, const char* base, const auto& off, int64_t row) __attribute__((always_inline)) {
    using O = decltype(op);
#pragma unroll
    for (int u = 0; u < O::UNITS; ++u) {
      if constexpr (O::WORDS == 4) {
        const u32x4 v = load16(base, off[u]);
#pragma unroll
        for (int j = 0; j < 4; ++j) x[u][j] = v[j];
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) x[u][e] = load4(base + e * row, off[u]);
      }
    }
  };
  auto zero = [](auto& x) __attribute__((always_inline)) {
#pragma unroll
    for (auto& unit : x)
#pragma unroll
      for (auto& d : unit) d = 0u;
  };
  int w = 0;
  // The next whole K step into set p; past the last one zeros.
  auto load = [&](int p) __attribute__((always_inline)) {
    if (w < whole) {
      load_op(OA{}, xa[p], a_next, off_a, a_row);
      load_op(OB{}, xb[p], b_next, off_b, b_row);
      a_next += a_step;
      b_next += b_step;
    } else {
      zero(xa[p]);
      zero(xb[p]);
    }
    ++w;
  };
  // The K step that is not whole, into set 0.
  auto tail_op = [&](auto op, auto& x, const char* base, const auto& off, int64_t row) __attribute__((always_inline)) {
    using O = decltype(op);
    const int left = K - (kt1 - 1) * BK;  // k of this step inside the matrix
#pragma unroll
    for (int u = 0; u < O::UNITS; ++u) {
      int r, kg;
      O::coord(tid, u, r, kg);
      const int valid = left - 8 * kg;  // of the unit's 8 k
      if constexpr (O::WORDS == 4) {
        u32x4 v = {0u, 0u, 0u, 0u};
        if (valid > 0) v = load16(base - (valid < 8 ? 2 * (8 - valid) : 0), off[u]);  // K >= 8: inside the row
        if (valid > 0 && valid < 8) v = funnel16(v, u32x4{0u, 0u, 0u, 0u}, 2u * (uint32_t)(8 - valid));
#pragma unroll
        for (int j = 0; j < 4; ++j) x[u][j] = v[j];
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) x[u][e] = e < valid ? load4(base + e * row, off[u]) : 0u;
      }
    }
  };
  auto put = [&](auto op, const auto& x, const auto& sel, char* area) __attribute__((always_inline)) {
    using O = decltype(op);
#pragma unroll
    for (int u = 0; u < O::UNITS; ++u) {
      int r, kg;
      O::coord(tid, u, r, kg);
      if constexpr (O::WORDS == 4) {
        *reinterpret_cast<u32x4*>(area + O::at(kg, r)) = u32x4{x[u][0], x[u][1], x[u][2], x[u][3]};
      } else {
        u32x4 lo, hi;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          lo[j] = __builtin_amdgcn_perm(x[u][2 * j + 1], x[u][2 * j], sel[u]);
          hi[j] = __builtin_amdgcn_perm(x[u][2 * j + 1], x[u][2 * j], 0x07060302u);
        }
        *reinterpret_cast<u32x4*>(area + O::at(kg, r)) = lo;
        *reinterpret_cast<u32x4*>(area + O::at(kg, r + 1)) = hi;
      }
    }
  };
  auto store = [&](int p, char* st) __attribute__((always_inline)) {
    put(OA{}, xa[p], sel_a, st);
    put(OB{}, xb[p], sel_b, st + OA::BYTES);
  };

  f32x16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

  // The running sums move to a second set every 256 k, in the 64 x 64 tile every
  // 128 up to 2048 k (beyond, the second set's additions count for more): a
  // sum's rounding error grows as the root of the number of its additions, and
  // the tiles and streaming kernels with many K splits that this kernel takes
  // over from kept theirs short.  14 x 1538 x 1050 (x @ W.T, 4 splits): 9.3e-8
  // with folds of 256 k, 8.5e-8 with 128 (7.5 us both), 9.0e-8 on the streaming
  // kernel (11.5 us).  In the larger tiles folds of 128 k cost 4 to 5 % (300 x
  // 2051 x 1001 in 128 x 64: 20.8 and 21.7 us).
  const bool fine = BM == 64 && nk <= 32;
  f32x16 sum[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) sum[i][j] = acc[i][j];
  auto fold = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          sum[i][j][r] += acc[i][j][r];
          acc[i][j][r] = 0.f;
        }
  };

  const int half = lane >> 5;
  const int a_r = wm * WTM + (lane & 31), b_r = wn * WTN + (lane & 31);
  struct Frag {
    bf16x8 a[TM], b[TN];
  };
  auto read = [&](const char* st, int ks, Frag& f) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < TM; ++i) f.a[i] = *reinterpret_cast<const bf16x8*>(st + OA::at(2 * ks + half, a_r + 32 * i));
#pragma unroll
    for (int j = 0; j < TN; ++j)
      f.b[j] = *reinterpret_cast<const bf16x8*>(st + OA::BYTES + OB::at(2 * ks + half, b_r + 32 * j));
  };
  auto mma = [&](const Frag& f) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] = mfma32x32x16bf16(f.a[i], f.b[j], acc[i][j]);
  };
  auto barrier = [&]() __attribute__((always_inline)) {
    // lgkmcnt(0): this wave's LDS reads and writes are done; global loads stay in flight
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(15 | (3 << 14) | (7 << 4));
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };

  int cur = 0, nxt = STAGE, nn = 2 * STAGE;
  if (nk > 0) {
    if (tail) {
      tail_op(OA{}, xa[0], base_a(kt1 - 1), off_a, a_row);
      tail_op(OB{}, xb[0], base_b(kt1 - 1), off_b, b_row);
    } else {
      load(0);
    }
#pragma unroll
    for (int p = 1; p < PF; ++p) load(p);
    store(0, lds);
    load(0);
    store(1, lds + STAGE);
    load(1);
    barrier();
    Frag f[2];
    read(lds, 0, f[0]);
    // Step s (I = s % PF): its four k-slices, each read during the one before;
    // the last reads the next step's first.  Set (s + 2) % PF is stored to the
    // third stage and loaded again for step s + 2 + PF.
    auto step = [&](auto I) __attribute__((always_inline)) {
      constexpr int p = (decltype(I)::value + 2) % PF;
      read(lds + cur, 1, f[1]);
      mma(f[0]);
      store(p, lds + nn);
      load(p);
      read(lds + cur, 2, f[0]);
      mma(f[1]);
      read(lds + cur, 3, f[1]);
      mma(f[0]);
      read(lds + nxt, 0, f[0]);
      mma(f[1]);
      barrier();
      const int t = cur;
      cur = nxt;
      nxt = nn;
      nn = t;
    };
    int s = 0;
#pragma unroll 1
    for (; s + PF <= nk; s += PF) {
      step(std::integral_constant<int, 0>{});
      step(std::integral_constant<int, 1>{});
      if (fine) fold();
      if constexpr (PF > 2) {
        step(std::integral_constant<int, 2>{});
        step(std::integral_constant<int, 3>{});
      }
      if ((PF > 2 || !fine) && (s + PF) % 4 == 0) fold();
    }
    if (s < nk) step(std::integral_constant<int, 0>{});
    if constexpr (PF > 2) {
      if (s + 1 < nk) step(std::integral_constant<int, 1>{});
      if (s + 2 < nk) step(std::integral_constant<int, 2>{});
    }
  }

#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] += sum[i][j][r];

  const bool interior = (m0 + BM <= M) && (n0 + BN <= N);
  const int row_base = m0 + wm * WTM + 4 * half;
  const int col_base = n0 + b_r;
  if (S > 1 && !splitk_tile<TM, TN, NT>(acc, split, S, blockIdx.x, gridDim.x, ws, counters, &last_flag, row_base,
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

template <int BM, int BN, int WM, int WN, int PF, int WPE, bool CA, bool CB>
hipError_t launch_any(const MatmulArgs& a) {
  const int64_t tiles = cdiv(a.M, BM) * cdiv(a.N, BN);
  if (tiles == 0) return hipSuccess;
  const SplitGeom g = gemm_split_geom(a.K, 64, a.split_k);
  if (g.splits > 1 && BM * BN > kSplitMaxAccPerThread * WM * WN * 64) return hipErrorInvalidConfiguration;
  hipLaunchKernelGGL((gemm_bf16_any_kernel<BM, BN, WM, WN, PF, CA, CB, WPE>), dim3((unsigned)tiles, (unsigned)g.splits),
                     dim3(WM * WN * 64), 0, a.stream, static_cast<const u16*>(a.x1), static_cast<const u16*>(a.x2),
                     a.out, (int)a.M, (int)a.N, (int)a.K, a.ldx1, a.ldx2, a.ldo, 4, device_xcds(), (int)g.steps,
                     g.splits > 1 ? static_cast<float*>(a.workspace) : nullptr, g.splits > 1 ? a.counters : nullptr);
  return hipGetLastError();
}

}  // namespace

template <int BM, int BN, int WM, int WN, int PF, int WPE>
hipError_t launch_gemm_bf16_any(const MatmulArgs& a) {
  switch (a.layout & 3) {
    case 0: return launch_any<BM, BN, WM, WN, PF, WPE, false, false>(a);
    case TILEC_X1_COL_MAJOR: return launch_any<BM, BN, WM, WN, PF, WPE, true, false>(a);
    case TILEC_X2_COL_MAJOR: return launch_any<BM, BN, WM, WN, PF, WPE, false, true>(a);
    default: return launch_any<BM, BN, WM, WN, PF, WPE, true, true>(a);
  }
}
template hipError_t launch_gemm_bf16_any<64, 64, 2, 2, 4, 2>(const MatmulArgs&);
template hipError_t launch_gemm_bf16_any<128, 64, 2, 2, 2, 2>(const MatmulArgs&);
template hipError_t launch_gemm_bf16_any<128, 128, 2, 4, 4, 1>(const MatmulArgs&);

}  // namespace tilec
