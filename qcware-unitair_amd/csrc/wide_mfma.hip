// Dense 6- to 10-qubit complex gates on the matrix cores, in place or not, one
// operator or one per batch entry.
//
// unitair permutes the targets to the front and contracts with einsum
// (unitair/simulation/operations.py:151-186, 258-329): a (D x D) x (D x 2^(n-k))
// complex product, D = 2^k.  Here a workgroup owns the D x G block of it that
// lies in one tile of the state (the k targets plus the lowest LG other index
// bits, G = 2^LG groups), keeps the tile in LDS and streams U from the caches:
//   - the tile is loaded in ascending address order and stored in LDS as
//     [column][group] with a bank swizzle; gate index bits keep the caller's
//     qubit order, so U is read as it lies in memory, a 128-byte line of a row
//     at a time, one step ahead;
//   - every wavefront forms RTW x CTW tiles of 16 rows x 16 groups, real and
//     imaginary parts in accumulators of their own: four
//     v_mfma_f32_16x16x4f32 / v_mfma_f64_16x16x4f64 for each step of four
//     columns, with -Im x formed once per read of x;
//   - the results replace the inputs in LDS when all of them have been read,
//     and leave in the load's order.  All D rows of a group are in one
//     workgroup, so the kernel may run in place.
// Where that leaves compute units idle (few tiles) and the output does not
// overlap the input, the rows are split over workgroups (blockIdx.y) that each
// load the tile and store their rows straight from the accumulators.
//
// What bounds it: the matrix cores (8 D flop per amplitude, measured 88-117
// TFLOP/s in complex64 against 154 of a large library product, 43-58 in
// complex128 against 66), and the memory phases that the two to four
// workgroups of a CU do not hide.  Before, as a tiled vector kernel (complex128,
// 9 and 10 targets) and as row slices of the real block (complex64 7 and 8):
// 8 targets at 24 qubits 384 us (now 280), 10 at 23 qubits 2724 (620);
// complex128 7 targets at 22 qubits 310 (84), 8 at 21 qubits 433 (74).
#include "mfma_common.h"

namespace ua {
namespace {

constexpr int kThreads = 512;
constexpr int kWaves = kThreads / 64;
constexpr int kMaxTB = 14;
constexpr int kMaxGemmK = 10;

struct GemmPass {
  const void* op;          // D x D row-major in the caller's qubit order
  int64_t tiles;           // batch * 2^(n - TB)
  int64_t in_bstride;      // batch stride of the input (0: one state for every entry)
  int64_t bstride;         // batch stride of the output: 2^n
  int64_t op_bstride;      // 0 or D * D
  int log2_tiles;          // n - TB
  int xcd;                 // visit tiles in XCD-contiguous ranges (tiles % 8 == 0)
  int local[kMaxTB];       // ascending state bits of the tile
  int pcol[kMaxTB];        // LDS position of tile bit i
  int tbit[kMaxGemmK];     // state bit of gate-index bit m
  int gbit[8];             // state bit of group bit j
};

// LDS position of (column c, group g), linear over GF(2).  The bits of c are
// folded onto the bank bits: lanes that differ in low columns (targets on low
// index bits, while a tile is loaded) or in column bits 2 and 3 (B-operands)
// meet different banks.
template <typename T, int LG>
__host__ __device__ __forceinline__ constexpr int gemm_pos(int c, int g) {
  if constexpr (sizeof(T) == 8) {
    const int m = (c ^ (c >> 5)) & 31;
    return ((c << LG) | g) ^ (((m << 2) | (m >> 3)) & 31);
  } else {
    return ((c << LG) | g) ^ ((c ^ (c >> 4) ^ (c >> 8)) & 15);
  }
}

// RTW: row tiles of 16 per wavefront.  WR wavefronts (WR_, or as many as there
// are row tiles for) cover the rows of a workgroup, WC the groups, KS ranges of
// the columns.
template <typename T, int K, int LG, int RTW, int WR_ = 0, int KS = 1> struct GemmShape {
  static constexpr int D = 1 << K, G = 1 << LG, TB = K + LG;
  static constexpr int RT = D / 16, CT = G / 16;
  static constexpr int WR = WR_ ? WR_ : RT / RTW < kWaves ? RT / RTW : kWaves;
  static constexpr int WC = kWaves / WR / KS;
  static constexpr int CTW = CT / WC;
  static constexpr int S = RT / (WR * RTW);   // row slices (blockIdx.y)
  static constexpr int AC = 32 / sizeof(T);   // columns of U a lane reads a step: 32 bytes
  // workgroups per CU that the registers must leave room for (LDS: 160 KB; three or
  // four of 32 KB are within 1 % of each other, 6 and 7 targets, 18 to 24 qubits)
  static constexpr int kLds = sizeof(T) << TB;
  static constexpr int kPerCu = kLds <= 32768 ? (K == 7 ? 4 : 3) : kLds <= 65536 ? 2 : 1;
  // 8-qubit complex64 gates sum 512 real terms as four partial sums of 128 (error
  // of a random gate 2.1e-7; 4.1e-7 in one chain)
  static constexpr int NSUM = K == 8 && sizeof(T) == 8 ? 4 : 1;
  static_assert(WR * WC * KS == kWaves && CTW * WC == CT && S * WR * RTW == RT, "split");
  static_assert(KS == 1 || (KS == NSUM && S > 1), "a wavefront's columns are a partial sum");
};

template <typename T, int K, int LG, int RTW, int WR_ = 0, int KS = 1>
__global__ __launch_bounds__(kThreads)
__attribute__((amdgpu_waves_per_eu(2 * GemmShape<T, K, LG, RTW, WR_, KS>::kPerCu)))
void dense_gemm_kernel(T* out, const T* in, GemmPass p) {
  using Sh = GemmShape<T, K, LG, RTW, WR_, KS>;
  using R = typename RealOf<T>::type;
  using M = Mfma<R>;
  constexpr int D = Sh::D, TB = Sh::TB, CTW = Sh::CTW;
  constexpr int UPT = (1 << TB) / 2 / kThreads;  // element pairs per thread
  constexpr int AC = Sh::AC, KK = D / (4 * AC);  // steps of 4 * AC columns
  __shared__ __attribute__((aligned(16))) T xs[1 << TB];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int q = lane >> 4, l16 = lane & 15;

  int64_t tile = blockIdx.x;
  if (p.xcd) tile = (tile & 7) * (p.tiles >> 3) + (tile >> 3);
  const int64_t b = tile >> p.log2_tiles;
  const int64_t origin = int64_t(insert_zero_bits(
      uint64_t(tile) & ((uint64_t(1) << p.log2_tiles) - 1), p.local, TB));
  const T* U = static_cast<const T*>(p.op) + b * p.op_bstride;

  // ---- this wavefront's row and group tiles; its first columns of U
  const int wr = wave % Sh::WR, wc = KS > 1 ? wave / Sh::WR % Sh::WC : wave / Sh::WR;
  const int ks = KS > 1 ? wave / Sh::WR / Sh::WC : 0;
  constexpr int KW = KK / KS;            // steps of a wavefront, from kb on
  const int kb = ks * KW;
  const int t0 = (int(blockIdx.y) * Sh::WR + wr) * RTW;
  const int g0 = 16 * CTW * wc;
  const T* urow = U + int64_t(16 * t0 + l16) * D + AC * q;
  T a[RTW][AC];
  auto load_a = [&](T (&dst)[RTW][AC], int kk) {
#pragma unroll
    for (int i = 0; i < RTW; ++i)
#pragma unroll
      for (int h = 0; h < AC / 2; ++h) {
        const Pair<T> v = *reinterpret_cast<const Pair<T>*>(urow + int64_t(16 * i) * D +
                                                            4 * AC * kk + 2 * h);
        dst[i][2 * h] = v.v[0];
        dst[i][2 * h + 1] = v.v[1];
      }
  };
  load_a(a, kb);

  // ---- the tile: element pair e = 2 * (tid + kThreads * u), tile bit i = state bit local[i]
  int64_t dep_t = 0;
  int pos_t = 0;
#pragma unroll
  for (int i = 1; i < 10; ++i) {
    const int bit = ((2 * tid) >> i) & 1;
    dep_t |= int64_t(bit) << p.local[i];
    pos_t ^= bit ? p.pcol[i] : 0;
  }
  auto dep_u = [&](int u) {
    int64_t d = 0;
#pragma unroll
    for (int i = 10; i < TB; ++i) d |= int64_t((u >> (i - 10)) & 1) << p.local[i];
    return d;
  };
  auto pos_u = [&](int u) {
    int d = 0;
#pragma unroll
    for (int i = 10; i < TB; ++i) d ^= ((u >> (i - 10)) & 1) ? p.pcol[i] : 0;
    return d;
  };
  {
    const T* src = in + b * p.in_bstride + origin + dep_t;
    Pair<T> v[UPT];
#pragma unroll
    for (int u = 0; u < UPT; ++u) v[u] = *reinterpret_cast<const Pair<T>*>(src + dep_u(u));
#pragma unroll
    for (int u = 0; u < UPT; ++u) {
      const int e = pos_t ^ pos_u(u);
      xs[e] = v[u].v[0];
      xs[e ^ p.pcol[0]] = v[u].v[1];
    }
  }
  __syncthreads();

  // ---- products
  const int bl = gemm_pos<T, LG>(AC * q, g0 + l16);
  typename M::acc_t re[RTW][CTW], im[RTW][CTW];
#pragma unroll
  for (int i = 0; i < RTW; ++i)
#pragma unroll
    for (int c = 0; c < CTW; ++c) re[i][c] = im[i][c] = typename M::acc_t{0, 0, 0, 0};
  typename M::acc_t sre[RTW][CTW], sim[RTW][CTW];  // sums of the earlier partial sums
  auto step = [&](const T (&u)[RTW][AC], int kk) {  // columns 4 AC kk ...
#pragma unroll
    for (int s = 0; s < AC; ++s) {
      T x[CTW];
#pragma unroll
      for (int c = 0; c < CTW; ++c) x[c] = xs[bl ^ gemm_pos<T, LG>(4 * AC * kk + s, 16 * c)];
#pragma unroll
      for (int i = 0; i < RTW; ++i)
#pragma unroll
        for (int c = 0; c < CTW; ++c) {
          re[i][c] = M::mma(u[i][s].x, x[c].x, re[i][c]);
          im[i][c] = M::mma(u[i][s].y, x[c].x, im[i][c]);
        }
#pragma unroll
      for (int i = 0; i < RTW; ++i)
#pragma unroll
        for (int c = 0; c < CTW; ++c) {
          re[i][c] = M::mma(u[i][s].y, -x[c].y, re[i][c]);
          im[i][c] = M::mma(u[i][s].x, x[c].y, im[i][c]);
        }
    }
  };
  static_assert(KK % (2 * Sh::NSUM) == 0, "two steps a turn");
  T a1[RTW][AC];
#pragma unroll 1
  for (int k0 = kb; k0 < kb + KW; k0 += KK / Sh::NSUM) {
#pragma unroll 1
    for (int kk = k0; kk < k0 + KK / Sh::NSUM; kk += 2) {
      // each step's columns are requested a step ahead; the scheduler would
      // move the loads down to their use
      load_a(a1, kk + 1);
      __builtin_amdgcn_sched_barrier(0);
      step(a, kk);
      load_a(a, kk + 2 < kb + KW ? kk + 2 : kk);
      __builtin_amdgcn_sched_barrier(0);
      step(a1, kk + 1);
    }
    if constexpr (Sh::NSUM > 1 && KS == 1) {  // a partial sum is complete
      const bool start = k0 == 0, end = k0 + KK / Sh::NSUM == KK;
#pragma unroll
      for (int i = 0; i < RTW; ++i)
#pragma unroll
        for (int c = 0; c < CTW; ++c) {
          sre[i][c] = start ? re[i][c] : sre[i][c] + re[i][c];
          sim[i][c] = start ? im[i][c] : sim[i][c] + im[i][c];
          re[i][c] = end ? sre[i][c] : typename M::acc_t{0, 0, 0, 0};
          im[i][c] = end ? sim[i][c] : typename M::acc_t{0, 0, 0, 0};
        }
    }
  }

  T* dst = out + b * p.bstride + origin;
  if constexpr (KS > 1) {
    // ---- the wavefronts' partial sums meet in LDS, in the order of one chain
    constexpr int PART = RTW * CTW * 4 * 64;
    static_assert(Sh::WR * Sh::WC * KS * PART <= (1 << TB), "the tile's place holds them");
    T* const mine = xs + wave * PART + lane;
    __syncthreads();  // every input is read
#pragma unroll
    for (int i = 0; i < RTW; ++i)
#pragma unroll
      for (int c = 0; c < CTW; ++c)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          T v;
          v.x = re[i][c][r];
          v.y = im[i][c][r];
          mine[((i * CTW + c) * 4 + r) * 64] = v;
        }
    __syncthreads();
    if (ks > 0) return;  // no barrier follows
#pragma unroll
    for (int k = 1; k < KS; ++k)
#pragma unroll
      for (int i = 0; i < RTW; ++i)
#pragma unroll
        for (int c = 0; c < CTW; ++c)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const T v = mine[k * Sh::WR * Sh::WC * PART + ((i * CTW + c) * 4 + r) * 64];
            re[i][c][r] += v.x;
            im[i][c][r] += v.y;
          }
  }
  if constexpr (Sh::S > 1) {
    // ---- a slice of the rows, straight from the accumulators
    int64_t lane_off = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) lane_off |= int64_t((l16 >> j) & 1) << p.gbit[j];
#pragma unroll
    for (int i = 0; i < RTW; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = 16 * (t0 + i) + M::row(lane, r);
        int64_t row_off = 0;
#pragma unroll
        for (int m = 0; m < K; ++m) row_off |= int64_t((row >> m) & 1) << p.tbit[m];
#pragma unroll
        for (int c = 0; c < CTW; ++c) {
          int64_t g_off = 0;
#pragma unroll
          for (int j = 4; j < LG; ++j)
            g_off |= int64_t(((g0 + 16 * c) >> j) & 1) << p.gbit[j];
          T v;
          v.x = re[i][c][r];
          v.y = im[i][c][r];
          dst[lane_off + row_off + g_off] = v;
        }
      }
  } else {
    __syncthreads();  // every input is read: the results take their places
    const int wl = gemm_pos<T, LG>(M::row(lane, 0), g0 + l16);
#pragma unroll
    for (int i = 0; i < RTW; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int c = 0; c < CTW; ++c) {
          T v;
          v.x = re[i][c][r];
          v.y = im[i][c][r];
          xs[wl ^ gemm_pos<T, LG>(16 * (t0 + i) + M::row(0, r), 16 * c)] = v;
        }
    __syncthreads();
    dst += dep_t;
#pragma unroll
    for (int u = 0; u < UPT; ++u) {
      const int e = pos_t ^ pos_u(u);
      Pair<T> v;
      v.v[0] = xs[e];
      v.v[1] = xs[e ^ p.pcol[0]];
      *reinterpret_cast<Pair<T>*>(dst + dep_u(u)) = v;
    }
  }
}

struct GemmArgs {
  void* out;
  const void* in;
  const void* op;
  int n, k;
  const int* tb;  // target state bits, gate-index MSB first
  int64_t batch, in_bstride, op_bstride;
  hipStream_t s;
};

template <typename T, int K, int LG, int RTW, int WR_ = 0, int KS = 1>
int launch_gemm(const GemmArgs& a) {
  using Sh = GemmShape<T, K, LG, RTW, WR_, KS>;
  GemmPass p{};
  p.op = a.op;
  p.log2_tiles = a.n - Sh::TB;
  p.tiles = a.batch << p.log2_tiles;
  UA_CHECK_ARG(p.log2_tiles >= 0 && p.tiles <= 0x7fffffffLL, "internal: %lld tiles",
               (long long)p.tiles);
  p.in_bstride = a.in_bstride;
  p.bstride = int64_t(1) << a.n;
  p.op_bstride = a.op_bstride;
  p.xcd = p.tiles % 8 == 0;
  uint64_t tmask = 0;
  for (int m = 0; m < K; ++m) {
    p.tbit[m] = a.tb[K - 1 - m];
    tmask |= uint64_t(1) << p.tbit[m];
  }
  uint64_t lmask = tmask;
  for (int bit = 0, j = 0; j < LG; ++bit)  // the lowest other bits
    if (!((tmask >> bit) & 1)) {
      p.gbit[j++] = bit;
      lmask |= uint64_t(1) << bit;
    }
  for (int i = 0; i < Sh::TB; ++i) {
    const int bit = __builtin_ctzll(lmask);
    lmask &= lmask - 1;
    p.local[i] = bit;
    for (int m = 0; m < K; ++m)
      if (p.tbit[m] == bit) p.pcol[i] = gemm_pos<T, LG>(1 << m, 0);
    for (int j = 0; j < LG; ++j)
      if (p.gbit[j] == bit) p.pcol[i] = gemm_pos<T, LG>(0, 1 << j);
  }
  dense_gemm_kernel<T, K, LG, RTW, WR_, KS><<<dim3(unsigned(p.tiles), Sh::S), kThreads, 0, a.s>>>(
      static_cast<T*>(a.out), static_cast<const T*>(a.in), p);
  return check_launch("dense_gemm_kernel");
}

// log2 of the groups of a tile (0: the gate is not taken here).  Measured at 22
// to 24 qubits against tiles of half and twice the groups: 6 targets 98 us (111
// and 119), 7 158 (168 with twice), 8 304 (367 with half), 9 295 at 23 qubits
// (321 with half); complex128 6 targets 101 (113 with twice), 7 167 (176 with
// half), 8 158 at 22 qubits (170 with twice).
int gemm_groups(int dtype, int k) {
  if (dtype == UA_COMPLEX64) return k == 6 ? 6 : k <= 9 ? 5 : k == 10 ? 4 : 0;
  if (dtype == UA_COMPLEX128) return k <= 7 ? 5 : k <= 9 ? 4 : 0;
  return 0;
}

bool disjoint(const GemmArgs& a, size_t es) {
  const uintptr_t o0 = reinterpret_cast<uintptr_t>(a.out);
  const uintptr_t o1 = o0 + (uintptr_t(a.batch) << a.n) * es;
  const uintptr_t i0 = reinterpret_cast<uintptr_t>(a.in);
  const uintptr_t i1 =
      i0 + (uintptr_t(a.batch - 1) * a.in_bstride + (uintptr_t(1) << a.n)) * es;
  return o1 <= i0 || i1 <= o0;
}

}  // namespace

bool gemm_applies(int dtype, int n, int k, const void* out, const void* in, const void* op,
                  int64_t in_bstride) {
  if (k < 6 || k > kMaxGemmK || n < 12) return false;
  const int lg = gemm_groups(dtype, k);
  const size_t align = 2 * elem_size(dtype);
  return lg > 0 && n >= k + lg && reinterpret_cast<uintptr_t>(out) % align == 0 &&
         reinterpret_cast<uintptr_t>(in) % align == 0 &&
         reinterpret_cast<uintptr_t>(op) % align == 0 && in_bstride % 2 == 0;
}

// tb: target state bits in the caller's order (gate-index MSB first).
int apply_dense_gemm(void* out, const void* in, const void* op, int dtype, int n, int k,
                     const int* tb, int64_t batch, int64_t in_bstride, int64_t op_bstride,
                     hipStream_t s) {
  UA_CHECK_ARG(gemm_applies(dtype, n, k, out, in, op, in_bstride) && batch >= 1,
               "internal: matrix-core path for %d targets on %d qubits", k, n);
  const GemmArgs a{out, in, op, n, k, tb, batch, in_bstride, op_bstride, s};
  const int64_t tiles = batch << (n - k - gemm_groups(dtype, k));
  // Fewer tiles than CUs: the rows of a tile go to several workgroups (20
  // qubits, 9 targets: 134 -> 48 us; with 256 tiles or more the whole tile in
  // one workgroup is as fast or faster: 8 targets, 21 qubits 42 against 44 us)
  const bool split = tiles < 256 && disjoint(a, elem_size(dtype));
  if (dtype == UA_COMPLEX64) switch (k) {
    case 6: return split ? launch_gemm<float2, 6, 6, 1, 2>(a) : launch_gemm<float2, 6, 6, 1>(a);
    case 7: return split ? launch_gemm<float2, 7, 5, 1, 4>(a) : launch_gemm<float2, 7, 5, 1>(a);
    case 8:
      // Few tiles: the wavefronts of a workgroup split the columns too (the partial
      // sums are there anyway), and the rows of a tile go to 16 workgroups or to
      // 8 (14 qubits, 2 tiles 5.6 and 8.2 us, in rows alone 14; 32 tiles 8.9 and
      // 9.0, 64 tiles 13.8 and 12.0, 224 tiles 51 and 43, 40 in one piece).  Little more
      // than 256 tiles leave a second round nearly empty: 320 tiles 78 us in one
      // piece, 66 so; from 384 on one piece is faster (78 and 79).
      if (disjoint(a, 8) && (tiles <= 352 && tiles != 256)) {
        if (tiles <= 48) return launch_gemm<float2, 8, 5, 1, 1, 4>(a);
        return launch_gemm<float2, 8, 5, 1, 2, 4>(a);
      }
      return launch_gemm<float2, 8, 5, 2>(a);
    case 9: return split ? launch_gemm<float2, 9, 5, 1, 4>(a) : launch_gemm<float2, 9, 5, 4>(a);
    default: return split ? launch_gemm<float2, 10, 4, 1>(a) : launch_gemm<float2, 10, 4, 8>(a);
  }
  switch (k) {
    case 6: return launch_gemm<double2, 6, 5, 1>(a);  // 4 x 2 tiles: one for each wavefront
    case 7: return split ? launch_gemm<double2, 7, 5, 1, 4>(a) : launch_gemm<double2, 7, 5, 1>(a);
    case 8: return split ? launch_gemm<double2, 8, 4, 1>(a) : launch_gemm<double2, 8, 4, 2>(a);
    default: return split ? launch_gemm<double2, 9, 4, 1>(a) : launch_gemm<double2, 9, 4, 4>(a);
  }
}

}  // namespace ua
