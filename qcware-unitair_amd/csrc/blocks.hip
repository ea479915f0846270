// Runs of dense 4- and 5-qubit gates, several gates per pass over the state,
// on the matrix cores: ua_plan_dense_blocks / ua_run_dense_blocks.
//
// unitair applies each gate as its own contraction over the whole state
// (unitair/simulation/operations.py:151-186, 322), and so does
// ua_apply_operator (mfma.hip for these sizes): every 4/5-qubit gate reads and
// writes the state once, which at 28 qubits is ~4.3 GB of HBM traffic per
// gate for ~0.07 TFLOP of matrix work.  Here consecutive gates whose targets
// fit together in one 12-bit tile are applied in one pass:
//   - tile = 2^12 amplitudes spanning the union of the pass's targets, state
//     bits 0 and 1 (runs of at least 4 amplitudes), and the lowest other state
//     bits up to 12 ("local bits"); one workgroup and 32 KB (complex64) or 64 KB
//     (complex128) of LDS per tile, so that four (two) of them on a CU are in
//     different phases;
//   - per gate, the tile's 2^(12-k) groups are the GEMM columns: each
//     wavefront owns whole column tiles of 16 groups and all rows of them,
//     reads their B-operands from LDS and writes the results back in place, so
//     one barrier per gate suffices.  U comes from the caches into registers as
//     it lies in memory; real and imaginary parts have accumulators of their
//     own (mfma as in wide_mfma.hip).
// A pass holds up to 3 gates in complex64 and 2 in complex128; the union of two
// 5-qubit gates always fits (10 bits + 2).  Gates of other kinds or sizes,
// states below 14 qubits, and matrices off 16- (32-) byte alignment run one by
// one as ua_run_circuit runs them.
//
// What bounds it: matrix products and memory phases that overlap in part (26
// qubits complex64, 80 gates: 12.8 ms; products alone 10.3, loads and stores
// alone 7.4).  Before, persistent workgroups staged every gate's real block in
// LDS (80 to 128 KB, two or one to a CU) and prefetched the next tile: 13.0 ms
// there, 2.27 against 1.94 at 24 qubits and 50 gates, 0.37 against 0.17 at 18
// qubits and 40 gates; complex128 at 24 qubits 4.30 against 3.77 ms.  Also
// slower: lane-private products (mfma_common.h) with the matrix in registers
// (14.0 ms), next-tile prefetch in persistent workgroups (15.5), 13-bit tiles
// (13.4), 512-thread workgroups (13.9).
#include "mfma_common.h"

namespace ua {
int run_gate(const ua_gate& g, int index, void* dst, void* cur, int dtype, int n,
             int64_t batch, hipStream_t s);
int record_event(void* ev, hipStream_t s);

namespace {

constexpr int kTB = 12;
constexpr int kTile = 1 << kTB;
constexpr int kMaxPassGates = 3;
constexpr int kMinBlockQubits = 14;   // whole tiles and a few of them per state

struct BlockGate {
  const void* op;   // D x D matrix, row-major, in the caller's qubit order
  int k;            // 4 or 5
  int jcol[5];      // LDS position of gate-index bit m
  int gcol[8];      // LDS position of group bit j: lane bits 0..3, then column tiles
  int jbit[5];      // the same bits of the state's index
  int gbit[8];
};

struct BlockPass {
  int64_t tiles;        // batch * 2^(n - 12)
  int64_t bstride;      // batch stride: 2^n
  int log2_tiles;       // n - 12
  int group;            // neighbouring tiles that one XCD takes (0: no order)
  int reverse;          // walk the tiles from the last to the first
  int local[kTB];       // ascending state bits of the tile
  int num_gates;
  int direct_in;        // the first gate reads its groups from the state
  int direct_out;       // the last gate writes its results to it (complex128)
  BlockGate g[kMaxPassGates];
};

// LDS position of tile element e, linear over GF(2): the low five bits, which
// pick the bank column, take in the others.
__host__ __device__ __forceinline__ constexpr int block_pos(int e) {
  const int h = e >> 10;
  return e ^ ((e >> 5) & 31) ^ ((h | (h << 3)) & 31);
}

// Multiplies every group of the tile by gate g (K targets): a wavefront takes
// CTW column tiles of 16 groups and all D rows of them, so only it reads and
// writes their amplitudes.  U comes from the caches as it lies in memory, 32
// bytes of a row per lane and step, and stays in registers for the gate.
// IN / OUT: the amplitudes come from / go to the state (st: the tile's origin),
// the other way they are in LDS.
template <typename T, int THREADS, int K, bool IN, bool OUT>
__device__ __forceinline__ void apply_gate(T* tile, T* st, const BlockGate& g, int lane,
                                           int wave) {
  using R = typename RealOf<T>::type;
  using M = Mfma<R>;
  constexpr int D = 1 << K, RT = D / 16;
  constexpr int CTW = (kTile >> K) / 16 / (THREADS / 64);
  constexpr int AC = 32 / sizeof(T), AB = AC == 4 ? 2 : 1;  // columns of a lane's 32 bytes, log2
  constexpr int KK = D / (4 * AC);
  static_assert(CTW >= 1, "a column tile per wavefront");
  const int q = lane >> 4, l16 = lane & 15;
  const T* U = static_cast<const T*>(g.op) + l16 * D + AC * q;
  T a[RT][KK][AC];
#pragma unroll
  for (int kk = 0; kk < KK; ++kk)
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int h = 0; h < AC / 2; ++h) {
        const Pair<T> v = *reinterpret_cast<const Pair<T>*>(U + 16 * i * D + 4 * AC * kk + 2 * h);
        a[i][kk][2 * h] = v.v[0];
        a[i][kk][2 * h + 1] = v.v[1];
      }
  // the lane's group within a column tile, gate index j and column tile c of
  // this wavefront, as LDS positions (XOR) and state offsets (sum)
  int gl = 0;
#pragma unroll
  for (int j = 0; j < 4; ++j) gl ^= ((l16 >> j) & 1) ? g.gcol[j] : 0;
  auto entry = [&](int j) {
    int c = 0;
#pragma unroll
    for (int m = 0; m < K; ++m) c ^= ((j >> m) & 1) ? g.jcol[m] : 0;
    return c;
  };
  auto column = [&](int c) {
    int x = 0;
#pragma unroll
    for (int j = 4; j < kTB - K; ++j) x ^= (((wave * CTW + c) >> (j - 4)) & 1) ? g.gcol[j] : 0;
    return x;
  };
  int64_t go = 0;
#pragma unroll
  for (int j = 0; j < 4; ++j) go |= int64_t((l16 >> j) & 1) << g.gbit[j];
  auto entry_off = [&](int j) {
    int64_t o = 0;
#pragma unroll
    for (int m = 0; m < K; ++m) o |= int64_t((j >> m) & 1) << g.jbit[m];
    return o;
  };
  auto column_off = [&](int c) {
    int64_t o = 0;
#pragma unroll
    for (int j = 4; j < kTB - K; ++j)
      o |= int64_t(((wave * CTW + c) >> (j - 4)) & 1) << g.gbit[j];
    return o;
  };
  T xin[IN ? KK : 1][IN ? AC : 1][CTW];
  if constexpr (IN) {
    const T* src =
        st + go + (int64_t(q & 1) << g.jbit[AB]) + (int64_t(q >> 1) << g.jbit[AB + 1]);
#pragma unroll
    for (int kk = 0; kk < KK; ++kk)
#pragma unroll
      for (int s = 0; s < AC; ++s)
#pragma unroll
        for (int c = 0; c < CTW; ++c)
          xin[kk][s][c] = src[entry_off(4 * AC * kk + s) + column_off(c)];
  }
  const int bl = gl ^ ((q & 1) ? g.jcol[AB] : 0) ^ ((q & 2) ? g.jcol[AB + 1] : 0);
  typename M::acc_t re[RT][CTW], im[RT][CTW];
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int c = 0; c < CTW; ++c) re[i][c] = im[i][c] = typename M::acc_t{0, 0, 0, 0};
#pragma unroll
  for (int kk = 0; kk < KK; ++kk)
#pragma unroll
    for (int s = 0; s < AC; ++s) {
      T x[CTW];
#pragma unroll
      for (int c = 0; c < CTW; ++c) {
        if constexpr (IN) x[c] = xin[kk][s][c];
        else x[c] = tile[bl ^ entry(4 * AC * kk + s) ^ column(c)];
      }
#pragma unroll
      for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int c = 0; c < CTW; ++c) {
          re[i][c] = M::mma(a[i][kk][s].x, x[c].x, re[i][c]);
          im[i][c] = M::mma(a[i][kk][s].y, x[c].x, im[i][c]);
        }
#pragma unroll
      for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int c = 0; c < CTW; ++c) {
          re[i][c] = M::mma(a[i][kk][s].y, -x[c].y, re[i][c]);
          im[i][c] = M::mma(a[i][kk][s].x, x[c].y, im[i][c]);
        }
    }
  constexpr int RB = sizeof(R) == 4 ? 2 : 0;  // gate-index bits of a result's lane rows
  const int wl = gl ^ ((q & 1) ? g.jcol[RB] : 0) ^ ((q & 2) ? g.jcol[RB + 1] : 0);
  T* dst = st + go + (int64_t(q & 1) << g.jbit[RB]) + (int64_t(q >> 1) << g.jbit[RB + 1]);
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int c = 0; c < CTW; ++c) {
        T v;
        v.x = re[i][c][r];
        v.y = im[i][c][r];
        if constexpr (OUT) dst[entry_off(16 * i + M::row(0, r)) + column_off(c)] = v;
        else tile[wl ^ entry(16 * i + M::row(0, r)) ^ column(c)] = v;
      }
}

template <typename T, int THREADS>
__global__ __launch_bounds__(THREADS) __attribute__((amdgpu_waves_per_eu(sizeof(T) == 8 ? 5 : 2)))
void dense_blocks_kernel(T* state, BlockPass p) {
  constexpr int UPT = kTile / 2 / THREADS;  // element pairs per thread
  constexpr int EB = 9;                     // tile bits of 2 * thread
  static_assert(2 * THREADS == 1 << EB, "element pairs");
  constexpr bool kOut = sizeof(T) == 16;
  __shared__ T tile[kTile];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  int64_t t = blockIdx.x;
  if (p.group) {  // workgroup t runs on XCD t % 8
    const unsigned gr = p.group, i = blockIdx.x >> 3;
    const unsigned w = p.reverse ? unsigned(p.tiles >> 3) - 1 - i : i;
    t = (w / gr) * (8 * gr) + (blockIdx.x & 7) * gr + w % gr;
  } else if (p.reverse) {
    t = p.tiles - 1 - t;
  }
  T* const st = state + (t >> p.log2_tiles) * p.bstride +
                int64_t(insert_zero_bits(
                    uint64_t(t) & ((uint64_t(1) << p.log2_tiles) - 1), p.local, kTB));
  // element pair e = 2 * (tid + THREADS * u), tile bit i = state bit local[i]
  int64_t dep_t = 0;
#pragma unroll
  for (int i = 1; i < EB; ++i) dep_t |= int64_t(((2 * tid) >> i) & 1) << p.local[i];
  auto dep_u = [&](int u) {
    int64_t d = 0;
#pragma unroll
    for (int i = EB; i < kTB; ++i) d |= int64_t((u >> (i - EB)) & 1) << p.local[i];
    return d;
  };
  const int pos_t = block_pos(2 * tid);
  int first = 0, last = p.num_gates;
  if (p.direct_in) {
    first = 1;
    if (p.g[0].k == 5)
      apply_gate<T, THREADS, 5, true, false>(tile, st, p.g[0], lane, wave);
    else
      apply_gate<T, THREADS, 4, true, false>(tile, st, p.g[0], lane, wave);
  } else {
    Pair<T> v[UPT];
#pragma unroll
    for (int u = 0; u < UPT; ++u) v[u] = *reinterpret_cast<const Pair<T>*>(st + dep_t + dep_u(u));
#pragma unroll
    for (int u = 0; u < UPT; ++u) {
      const int e = pos_t ^ block_pos(2 * THREADS * u);
      tile[e] = v[u].v[0];
      tile[e ^ 1] = v[u].v[1];
    }
  }
  if (kOut && p.direct_out) --last;
  for (int gi = first; gi < last; ++gi) {
    __syncthreads();  // groups of this gate span the tile
    if (p.g[gi].k == 5)
      apply_gate<T, THREADS, 5, false, false>(tile, st, p.g[gi], lane, wave);
    else
      apply_gate<T, THREADS, 4, false, false>(tile, st, p.g[gi], lane, wave);
  }
  __syncthreads();
  if (kOut && p.direct_out) {
    const BlockGate& g = p.g[p.num_gates - 1];
    if (g.k == 5)
      apply_gate<T, THREADS, 5, false, kOut>(tile, st, g, lane, wave);
    else
      apply_gate<T, THREADS, 4, false, kOut>(tile, st, g, lane, wave);
    return;
  }
#pragma unroll
  for (int u = 0; u < UPT; ++u) {
    const int e = pos_t ^ block_pos(2 * THREADS * u);
    Pair<T> w;
    w.v[0] = tile[e];
    w.v[1] = tile[e ^ 1];
    *reinterpret_cast<Pair<T>*>(st + dep_t + dep_u(u)) = w;
  }
}

constexpr int kThreads64 = 256, kThreads128 = 256;
// gates of a pass: the plan that callers see (ua_plan_dense_blocks)
constexpr int kMaxGates64 = 3, kMaxGates128 = 2;

bool block_gate(const ua_gate& g, int dtype, int n) {
  return g.kind == UA_GATE_DENSE && (g.num_targets == 4 || g.num_targets == 5) &&
         (dtype == UA_COMPLEX64 || dtype == UA_COMPLEX128) && n >= kMinBlockQubits;
}

// Passes load pairs of elements, of the state and of U, as one access.
bool pass_aligned(const void* state, int dtype, const ua_gate* gates, int count) {
  const size_t align = 2 * elem_size(dtype);
  for (int i = 0; i < count; ++i)
    if (reinterpret_cast<uintptr_t>(gates[i].data) % align != 0) return false;
  return reinterpret_cast<uintptr_t>(state) % align == 0;
}

uint64_t target_mask(const ua_gate& g, int n) {
  uint64_t m = 0;
  for (int j = 0; j < g.num_targets; ++j) m |= uint64_t(1) << (n - 1 - g.qubits[j]);
  return m;
}

// Units of work in order: a pass of block gates [first, first + count) or a
// single other gate (count = 1, pass = false).
struct Unit {
  int first, count;
  bool pass;
};

int plan_units(int dtype, int n, const ua_gate* gates, int num_gates, Unit* units) {
  const int maxg = dtype == UA_COMPLEX64 ? kMaxGates64 : kMaxGates128;
  int nu = 0;
  uint64_t uni = 0;
  for (int i = 0; i < num_gates; ++i) {
    const ua_gate& g = gates[i];
    if (!block_gate(g, dtype, n)) {
      units[nu++] = {i, 1, false};
      uni = 0;
      continue;
    }
    const uint64_t m = target_mask(g, n);
    Unit* last = nu ? &units[nu - 1] : nullptr;
    if (last && last->pass && last->count < maxg &&
        __builtin_popcountll(uni | m | 3) <= kTB) {
      ++last->count;
      uni |= m;
    } else {
      units[nu++] = {i, 1, true};
      uni = m;
    }
  }
  return nu;
}

int check_gates(int n, const ua_gate* gates, int num_gates) {
  for (int i = 0; i < num_gates; ++i) {
    const ua_gate& g = gates[i];
    if (g.kind != UA_GATE_DENSE && g.kind != UA_GATE_CZ && g.kind != UA_GATE_CNOT &&
        g.kind != UA_GATE_PHASE) {
      set_error("gate %d: unknown kind %d", i, g.kind);
      return UA_ERR_INVALID_ARGUMENT;
    }
    if (g.kind == UA_GATE_PHASE) continue;
    const int k = g.kind == UA_GATE_DENSE ? g.num_targets : 2;
    if (k < 1 || k > UA_MAX_GATE_QUBITS) {
      set_error("gate %d: %d targets", i, k);
      return UA_ERR_INVALID_ARGUMENT;
    }
    uint64_t seen = 0;
    for (int j = 0; j < k; ++j) {
      const int q = g.qubits[j];
      if (q < 0 || q >= n || ((seen >> q) & 1)) {
        set_error("gate %d: qubit %d repeated or out of range for %d qubits", i, q, n);
        return UA_ERR_INVALID_ARGUMENT;
      }
      seen |= uint64_t(1) << q;
    }
    if (g.kind == UA_GATE_DENSE && !g.data) {
      set_error("gate %d: NULL matrix", i);
      return UA_ERR_INVALID_ARGUMENT;
    }
  }
  return UA_OK;
}

// A pass of one complex128 gate is the same work as the gate alone, whose kernel
// (mfma.hip) needs no tile: on 4 qubits it is the faster one (20 qubits 8.5 us,
// 22 qubits 23, 24 qubits 83; the pass 9..12, 27..39, 86..118), on 5 where both
// lowest bits are targets (24 qubits 109 and 136; others 112 and 110, 20 qubits 14
// and 10).
bool pass_pays(int dtype, int n, const ua_gate* gates, int count) {
  return count > 1 || dtype == UA_COMPLEX64 ||
         (gates[0].num_targets == 5 && (target_mask(gates[0], n) & 3) != 3);
}

// One pass of gates[0..count) (4/5-qubit gates) in place.
int launch_pass(void* state, int dtype, int n, int64_t batch, const ua_gate* gates, int count,
                bool reverse, hipStream_t s) {
  BlockPass p{};
  p.log2_tiles = n - kTB;
  p.tiles = batch << p.log2_tiles;
  p.bstride = int64_t(1) << n;
  // Tiles that share 128-byte lines are neighbours and meet in one XCD's L2; the
  // XCDs together walk through the state from one end, alternate passes from the
  // other, so that a pass begins with what the last one left in the Infinity
  // Cache (26 qubits complex64, 512 MiB, 80 gates: 13.1 -> 12.8 ms; groups of
  // 8 to 256 within 1 %, contiguous eighths of the state the slowest).  An XCD
  // keeps its tiles when the walk turns round: states that the L2s hold were
  // fetched from the other XCDs' otherwise (20 qubits complex128, 16 4-qubit
  // gates: 154 us, 88 so).
  p.group = p.tiles % 256 == 0 ? 32 : p.tiles % 8 == 0 ? int(p.tiles / 8) : 0;
  p.reverse = reverse;
  p.num_gates = count;
  UA_CHECK_ARG(p.tiles <= 0x7fffffffLL, "too many tiles");
  uint64_t uni = 3;
  for (int i = 0; i < count; ++i) uni |= target_mask(gates[i], n);
  UA_CHECK_ARG(__builtin_popcountll(uni) <= kTB, "internal: %d tile bits",
               __builtin_popcountll(uni));
  for (int bit = 0; __builtin_popcountll(uni) < kTB; ++bit) uni |= uint64_t(1) << bit;
  for (int i = 0; i < kTB; ++i) {
    p.local[i] = __builtin_ctzll(uni);
    uni &= uni - 1;
  }
  const bool c64 = dtype == UA_COMPLEX64;
  // The first gate of a pass can read its groups from the state, and the last one
  // write to it, which saves a trip through LDS and a barrier each.  Measured
  // (50 gates, 24 qubits): complex128 4.50 ms staged, 3.77 both ways direct (20
  // qubits 0.92 -> 0.59); complex64 1.97 staged, 1.94 direct in, 2.03 direct
  // out, and in only where the lanes keep runs of 32 bytes.
  // A single complex128 gate only writes directly (5 qubits at 20: 24 us the other
  // way round, 10 so).  Beyond the Infinity Cache a last gate with both lowest
  // bits among its targets, which leaves the lanes pieces of lines, goes through
  // LDS (24 qubits, 2 gates: 1.13 and 0.99 of 123 us).
  p.direct_in = c64 ? !(target_mask(gates[0], n) & 3) : count > 1;
  p.direct_out = !c64 && !((target_mask(gates[count - 1], n) & 3) == 3 && count > 1 &&
                           (batch << n) >= (int64_t(1) << 24));
  for (int gi = 0; gi < count; ++gi) {
    const ua_gate& g = gates[gi];
    BlockGate& b = p.g[gi];
    b.op = g.data;
    b.k = g.num_targets;
    const uint64_t tmask = target_mask(g, n);
    for (int m = 0; m < b.k; ++m) {  // gate-index bit m: qubits[k - 1 - m]
      const int bit = n - 1 - g.qubits[b.k - 1 - m];
      b.jbit[m] = bit;
      for (int i = 0; i < kTB; ++i)
        if (p.local[i] == bit) b.jcol[m] = block_pos(1 << i);
    }
    // The lanes of an access differ in two gate-index bits and four group bits.
    // In LDS those group bits come first whose bank columns are independent of
    // the others'; a gate that meets the state takes its lowest ones.
    const bool meets = (gi == 0 && p.direct_in) || (gi == count - 1 && p.direct_out);
    int basis[5] = {0, 0, 0, 0, 0};
    auto independent = [&](int v) {
      v &= 31;
      for (int k = 4; k >= 0 && v; --k) {
        if (!((v >> k) & 1)) continue;
        if (!basis[k]) {
          basis[k] = v;
          return true;
        }
        v ^= basis[k];
      }
      return false;
    };
    independent(b.jcol[c64 ? 2 : 1]);
    independent(b.jcol[c64 ? 3 : 2]);
    int order[8], rest[8], nf = 0, nr = 0;
    for (int i = 0; i < kTB; ++i) {
      if ((tmask >> p.local[i]) & 1) continue;
      if (meets || independent(block_pos(1 << i))) order[nf++] = i;
      else rest[nr++] = i;
    }
    for (int j = 0; j < nr; ++j) order[nf++] = rest[j];
    for (int j = 0; j < kTB - b.k; ++j) {
      b.gcol[j] = block_pos(1 << order[j]);
      b.gbit[j] = p.local[order[j]];
    }
  }
  if (c64)
    dense_blocks_kernel<float2, kThreads64>
        <<<unsigned(p.tiles), kThreads64, 0, s>>>(static_cast<float2*>(state), p);
  else
    dense_blocks_kernel<double2, kThreads128>
        <<<unsigned(p.tiles), kThreads128, 0, s>>>(static_cast<double2*>(state), p);
  return check_launch("dense_blocks_kernel");
}

}  // namespace

}  // namespace ua

extern "C" int ua_plan_dense_blocks(int dtype, int num_qubits, const ua_gate* gates,
                                    int num_gates, int* unit_of_gate, int* num_units) {
  using namespace ua;
  UA_CHECK_ARG(elem_size(dtype) != 0, "unsupported dtype code %d", dtype);
  UA_CHECK_ARG(num_qubits >= 1 && num_qubits <= 62, "num_qubits=%d out of range", num_qubits);
  UA_CHECK_ARG(num_gates >= 0 && (num_gates == 0 || gates), "bad gate list");
  UA_CHECK_ARG(num_units, "NULL num_units");
  const int rc = check_gates(num_qubits, gates, num_gates);
  if (rc) return rc;
  Unit* units = new Unit[num_gates > 0 ? num_gates : 1];
  const int nu = plan_units(dtype, num_qubits, gates, num_gates, units);
  if (unit_of_gate)
    for (int i = 0; i < nu; ++i)
      for (int j = 0; j < units[i].count; ++j) unit_of_gate[units[i].first + j] = i;
  delete[] units;
  *num_units = nu;
  return UA_OK;
}

extern "C" int ua_run_dense_blocks(void* state, int dtype, int num_qubits, int64_t batch,
                                   const ua_gate* gates, int num_gates, void* const* events,
                                   ua_stream_t stream) {
  using namespace ua;
  hipStream_t s = static_cast<hipStream_t>(stream);
  UA_CHECK_ARG(elem_size(dtype) != 0, "unsupported dtype code %d", dtype);
  UA_CHECK_ARG(num_qubits >= 1 && num_qubits <= 62, "num_qubits=%d out of range", num_qubits);
  UA_CHECK_ARG(num_gates >= 0 && (num_gates == 0 || gates), "bad gate list");
  UA_CHECK_ARG(batch >= 0, "negative batch");
  int rc = check_gates(num_qubits, gates, num_gates);
  if (rc) return rc;
  if (batch == 0 || num_gates == 0) return UA_OK;
  UA_CHECK_ARG(state, "NULL state");
  Unit* units = new Unit[num_gates];
  const int nu = plan_units(dtype, num_qubits, gates, num_gates, units);
  for (int i = 0; i < nu && rc == UA_OK; ++i) {
    // a start event that is the previous unit's end event is already recorded
    if (events && !(i > 0 && events[2 * i] == events[2 * i - 1])) rc = record_event(events[2 * i], s);
    if (rc) break;
    const Unit& u = units[i];
    if (u.pass && pass_aligned(state, dtype, gates + u.first, u.count) &&
        pass_pays(dtype, num_qubits, gates + u.first, u.count)) {
      rc = launch_pass(state, dtype, num_qubits, batch, gates + u.first, u.count, i & 1, s);
    } else {
      for (int j = 0; j < u.count && rc == UA_OK; ++j)
        rc = run_gate(gates[u.first + j], u.first + j, state, state, dtype, num_qubits, batch,
                      s);
    }
    if (rc) break;
    if (events) rc = record_event(events[2 * i + 1], s);
  }
  delete[] units;
  return rc;
}
