// Dense k-qubit gate application: ua_apply_operator.
//
// Replaces the reference's permute -> einsum -> inverse-permute sequence
// (unitair/simulation/operations.py:151-186 and :258-329), which moves the
// whole state three to five times per gate, with one streaming pass that
// addresses the target bits in place:
//
//   out[i] = sum_j U[r(i), j] * in[(i & ~targets) | scatter(j)]
//
// where r(i) gathers the target bits of i into a gate index whose most
// significant bit belongs to the first listed qubit (operations.py:78-86,
// unitair/utils.py:5-27).
//
// Fast path (k <= 5): one thread owns whole groups of 2**k amplitudes (the
// amplitudes that differ only in target bits), so a group is read once and
// written once and the kernel can run in place.  On the host the targets are
// sorted by state bit ("canonical" order) and the matrix is read through the
// matching index permutation, so the lowest target is always gate bit 0.
// That fixes the access pattern at compile time:
//   VEC  : lowest target bit >= 1 -> each thread takes two neighbouring groups
//          and moves 2 amplitudes per access (16 B for complex64);
//   PAIR : lowest target bit == 0 -> the two amplitudes that differ in bit 0
//          are adjacent and move as one 16 B access;
//   SCALAR: fallback for misaligned views.
// For k >= 3 the (permuted) matrix is staged in LDS once per workgroup.
#include "dense_kernels.h"
#include "fused_common.h"

namespace ua {

int g_unroll = 0;      // units per thread for single-operator launches (0 = auto)
extern bool g_use_mfma;  // 4/5-qubit complex gates on the matrix cores
int apply_dense_mfma(void* out, const void* in, const void* op, int dtype, int n, int k,
                     const int* tb, const int* gp, int64_t batch, int64_t in_bstride,
                     hipStream_t s);
bool g_use_xch = true; // lane-exchange path for 1-qubit gates on index bits 1..6

using namespace dense_detail;

namespace {

// One-qubit gate whose target is index bit b in [1, 6] (with 2 elements per
// lane: lane bit b-1).  Every lane moves one contiguous pair of amplitudes,
// so each wavefront access is one contiguous block; the partner amplitudes
// differ in lane bit b-1 and arrive by a cross-lane exchange.  The host
// guarantees 2**n >= 128, so every wavefront is full and inside one state.
template <typename T> __device__ __forceinline__ T shfl_xor_val(T v, int m);
template <> __device__ __forceinline__ float shfl_xor_val(float v, int m) { return __shfl_xor(v, m, 64); }
template <> __device__ __forceinline__ double shfl_xor_val(double v, int m) { return __shfl_xor(v, m, 64); }
template <> __device__ __forceinline__ float2 shfl_xor_val(float2 v, int m) {
  return make_float2(__shfl_xor(v.x, m, 64), __shfl_xor(v.y, m, 64));
}
template <> __device__ __forceinline__ double2 shfl_xor_val(double2 v, int m) {
  return make_double2(__shfl_xor(v.x, m, 64), __shfl_xor(v.y, m, 64));
}

struct XchParams {
  int64_t total;        // units (pairs of elements) over the whole batch
  int64_t in_bstride;   // elements between input states
  int64_t out_bstride;  // elements between output states
  int log2_ups;         // log2(units per state)
  int lane_mask;        // 1 << (b - 1)
};

template <typename T, int UNR>
__global__ __launch_bounds__(kBlock) void dense_xch_kernel(
    T* out, const T* in, const T* __restrict__ op, XchParams p) {
  using A = Num<T>;
  const T u00 = op[0], u01 = op[1], u10 = op[2], u11 = op[3];
  const int64_t first = int64_t(blockIdx.x) * (kBlock * UNR) + threadIdx.x;
  Pair<T> v[UNR];
  T* dst[UNR];
#pragma unroll
  for (int u = 0; u < UNR; ++u) {
    const int64_t unit = first + int64_t(u) * kBlock;
    dst[u] = nullptr;
    if (unit >= p.total) continue;   // uniform over a wavefront
    const int64_t b = unit >> p.log2_ups;
    const int64_t e = (unit & ((int64_t(1) << p.log2_ups) - 1)) * 2;
    v[u] = *reinterpret_cast<const Pair<T>*>(in + b * p.in_bstride + e);
    dst[u] = out + b * p.out_bstride + e;
  }
  const bool upper = (threadIdx.x & p.lane_mask) != 0;
  // row of the gate this lane produces and the coefficients for (own, partner)
  const T c_own = upper ? u11 : u00;
  const T c_par = upper ? u10 : u01;
#pragma unroll
  for (int u = 0; u < UNR; ++u) {
    if (dst[u] == nullptr) continue;
    Pair<T> w;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const T partner = shfl_xor_val(v[u].v[h], p.lane_mask);
      w.v[h] = A::mac(A::mac(A::zero(), c_own, v[u].v[h]), c_par, partner);
    }
    *reinterpret_cast<Pair<T>*>(dst[u]) = w;
  }
}

// 2- and 3-qubit gates with targets on low index bits.  A wavefront's 64 groups
// are taken as one block of 2^(6 + k) amplitudes, contiguous but for the
// targets beyond it, which are its highest bits: the block moves in whole
// lines and is exchanged in LDS, where each lane finds its group.  (With a
// thread reading its own group, targets on low bits make every access of a
// wavefront touch 64 different lines.)  The operator is read with scalar
// loads.  The products are those of dense_fast_kernel, in the same order.
// Bound by memory: 24 qubits complex64 41 us for 2 targets, 45 for 3 (6.5 and
// 6.0 TB/s) wherever they lie, 42..65 and 46..79 before.  low_pays_2 and
// low_pays_3 say where it is the faster one.
struct LowParams {
  int64_t total;        // wavefronts that own work
  int64_t in_bstride, out_bstride, op_bstride;
  int log2_wps;         // log2(wavefronts per state)
  int log2_run;         // log2(contiguous amplitudes): 6 + k - targets beyond
  int beyond;           // targets at log2_run and above ...
  int hb[2];            // ... and their state bits, ascending
  int tb[3];            // ascending target positions in the block
  int gpos[3];          // gate-index bit of canonical bit p
};

template <typename T, int K>
__global__ __launch_bounds__(kBlock) void dense_low_kernel(T* out, const T* in,
                                                           const T* __restrict__ op,
                                                           LowParams p) {
  using A = Num<T>;
  constexpr int D = 1 << K, C = 64 * D, V = sizeof(T) == 16 ? 1 : 2, M = D / V;
  // log2 of the elements that span the LDS banks: higher bits are XORed in
  constexpr int NB = sizeof(T) == 16 ? 4 : sizeof(T) == 8 ? 5 : 6;
  __shared__ T tiles[kBlock / 64][C];
  const int lane = threadIdx.x & 63;
  T* tile = tiles[threadIdx.x >> 6];
  const int64_t w = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6)) +
                    int64_t(blockIdx.x) * (kBlock / 64);
  if (w >= p.total) return;            // whole wavefronts; no workgroup barrier below
  const int64_t b = w >> p.log2_wps;
  const int64_t first = int64_t(insert_zero_bits(
      uint64_t(w & ((int64_t(1) << p.log2_wps) - 1)) << p.log2_run, p.hb, p.beyond));
  const T* src = in + b * p.in_bstride + first;
  T* dst = out + b * p.out_bstride + first;
  const T* u = op + b * p.op_bstride;
  auto pos = [](int e) { return e ^ ((e >> NB) & ((1 << NB) - 1)); };
  auto fence = []() {                  // LDS accesses of a wavefront complete in order
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  };
  // state offset of access m's first element: 64 V <= 128 <= 2^log2_run
  // elements lie in one run
  auto at = [&](int m) {
    const int e = m * 64 * V;
    uint64_t o = e & ((1 << p.log2_run) - 1);
#pragma unroll
    for (int i = 0; i < K - 1; ++i)
      if (i < p.beyond) o |= uint64_t((e >> (p.log2_run + i)) & 1) << p.hb[i];
    return o;
  };
  struct alignas(V * sizeof(T)) Unit { T v[V]; };
  Unit x[M];
#pragma unroll
  for (int m = 0; m < M; ++m)
    x[m] = *reinterpret_cast<const Unit*>(src + at(m) + lane * V);
#pragma unroll
  for (int m = 0; m < M; ++m)
#pragma unroll
    for (int h = 0; h < V; ++h) tile[pos((m * 64 + lane) * V + h)] = x[m].v[h];
  fence();
  int base = lane;
#pragma unroll
  for (int q = 0; q < K; ++q)
    base = ((base >> p.tb[q]) << (p.tb[q] + 1)) | (base & ((1 << p.tb[q]) - 1));
  int off[D], orig[D];                 // by canonical gate index
#pragma unroll
  for (int j = 0; j < D; ++j) {
    off[j] = orig[j] = 0;
#pragma unroll
    for (int q = 0; q < K; ++q)
      if ((j >> q) & 1) {
        off[j] |= 1 << p.tb[q];
        orig[j] |= 1 << p.gpos[q];
      }
  }
  const int pb = pos(base);            // pos is linear: pos(base | off) = pb ^ pos(off)
  T a[D];
#pragma unroll
  for (int j = 0; j < D; ++j) a[j] = tile[pb ^ pos(off[j])];
  fence();
#pragma unroll
  for (int r = 0; r < D; ++r) {
    T acc = A::zero();
#pragma unroll
    for (int j = 0; j < D; ++j) acc = A::mac(acc, u[orig[r] * D + orig[j]], a[j]);
    tile[pb ^ pos(off[r])] = acc;
  }
  fence();
#pragma unroll
  for (int m = 0; m < M; ++m) {
#pragma unroll
    for (int h = 0; h < V; ++h) x[m].v[h] = tile[pos((m * 64 + lane) * V + h)];
    *reinterpret_cast<Unit*>(dst + at(m) + lane * V) = x[m];
  }
}

// Any k (including 0 and k > 5): one thread per output amplitude, reading
// its group from memory.  Out of place only.
constexpr int kMaxQubits = 62;

struct GenericParams {
  int64_t total;  // batch * 2**n
  int64_t in_bstride, op_bstride;
  int n, k;
  uint64_t tmask;        // OR of all target bits
  int tbit[kMaxQubits];  // state bit of gate bit k-1-m, in `qubits` order
};

template <typename T>
__global__ __launch_bounds__(kBlock) void dense_generic_kernel(
    T* __restrict__ out, const T* __restrict__ in, const T* __restrict__ op,
    GenericParams p) {
  using A = Num<T>;
  const int64_t tid = int64_t(blockIdx.x) * kBlock + threadIdx.x;
  if (tid >= p.total) return;
  const int64_t b = tid >> p.n;
  const uint64_t x = uint64_t(tid) & ((uint64_t(1) << p.n) - 1);
  const int64_t D = int64_t(1) << p.k;
  int64_t r = 0;
  for (int m = 0; m < p.k; ++m) r = (r << 1) | int64_t((x >> p.tbit[m]) & 1);
  const uint64_t base = x & ~p.tmask;
  const T* src = in + b * p.in_bstride;
  const T* row = op + b * p.op_bstride + r * D;
  T acc = A::zero();
  for (int64_t j = 0; j < D; ++j) {
    uint64_t s = base;
    for (int m = 0; m < p.k; ++m)
      if ((j >> (p.k - 1 - m)) & 1) s |= uint64_t(1) << p.tbit[m];
    acc = A::mac(acc, row[j], src[s]);
  }
  out[tid] = acc;
}


template <typename T>
void launch_xch(void* out, const void* in, const void* op, const XchParams& p, int unr,
                hipStream_t s) {
  T* o = static_cast<T*>(out);
  const T* i = static_cast<const T*>(in);
  const T* m = static_cast<const T*>(op);
  switch (unr) {
    case 4: dense_xch_kernel<T, 4><<<grid_for(p.total, kBlock * 4), kBlock, 0, s>>>(o, i, m, p); break;
    case 2: dense_xch_kernel<T, 2><<<grid_for(p.total, kBlock * 2), kBlock, 0, s>>>(o, i, m, p); break;
    default: dense_xch_kernel<T, 1><<<grid_for(p.total, kBlock), kBlock, 0, s>>>(o, i, m, p);
  }
}

template <typename T>
void launch_low(int k, void* out, const void* in, const void* op, const LowParams& p,
                hipStream_t s) {
  T* o = static_cast<T*>(out);
  const T* i = static_cast<const T*>(in);
  const T* m = static_cast<const T*>(op);
  const unsigned grid = grid_for(p.total, kBlock / 64);
  if (k == 2) dense_low_kernel<T, 2><<<grid, kBlock, 0, s>>>(o, i, m, p);
  else dense_low_kernel<T, 3><<<grid, kBlock, 0, s>>>(o, i, m, p);
}

bool aligned(const void* ptr, int64_t stride_elems, size_t esize, size_t align) {
  return (reinterpret_cast<uintptr_t>(ptr) % align) == 0 &&
         ((stride_elems * int64_t(esize)) % int64_t(align)) == 0;
}

// Where dense_low_kernel beats the vector kernel: by ratios of times measured for
// 34 sets of targets from 2^10 to 2^28 amplitudes in each of the four types, with
// one operator and one per state; ratios of 1 and above stay out.  What it saves
// are the partial lines of targets on bits 1..3 ("lines"), so the wider the
// element the more; what it adds are two trips through LDS and, with an operator
// for each state, scalar loads that every wavefront waits for.  In between lies
// the size: small states wait for the vector kernel's longer chain of accesses,
// states beyond the Infinity Cache for their lines, those that it holds for
// neither.  Measurements in us (vector kernel -> this one) are of complex64 states
// of 24 qubits unless said otherwise, ratios are the range over the sizes.
struct LowCase {
  size_t es;       // bytes of an element
  const int* tb;   // ascending targets, the first `near` of them inside the block
  int near;
  int64_t amps;    // all states together
  bool per;        // an operator for each state
  bool staged;     // the vector kernel would keep that in LDS (k = 3)
  bool from(int e) const { return amps >= (int64_t(1) << e); }
  bool up_to(int e) const { return amps < (int64_t(3) << e) / 2; }
  bool beyond() const { return amps * int64_t(es) >= (int64_t(1) << 28); }
};

bool low_pays_2(const LowCase& c) {
  const int* tb = c.tb;
  const size_t es = c.es;
  const bool near = c.near == 2;
  int lines = 0, first = 4;
  for (int m = 1; m >= 0; --m)
    if (tb[m] >= 1 && tb[m] <= 3) ++lines, first = tb[m];
  // float32: 1 2 0.79..0.95 (0.68 beyond the cache; per state up to 1.17 there); 1 5
  // and 0 1 up to 1.21, 0.91 beyond
  if (es == 4) {
    if (c.per) return lines == 2 && c.from(18) && !c.beyond();
    return lines == 2 || (lines && near && c.beyond());
  }
  if (tb[0] != 0) {
    // 1 2 65 -> 42, 2 3 55 -> 41; bit 3 as the lowest 0.92 up to 2^18, then up to
    // 1.15, 0.96 beyond (complex128 0.75..0.98 throughout).  Targets beyond the
    // block: h 1 at 22 qubits 13.9 -> 14.0, with an operator per state 48 -> 46,
    // complex128 at 23 qubits 61 -> 43
    if (!near && !c.per && es == 8) return false;
    return lines && (first < 3 || es == 16 || c.beyond() || (!c.per && c.up_to(18)));
  }
  // bit 0, which the vector kernel pairs: 0 1 and 0 2 0.94..0.98 from 2^19 (1.02
  // below), 0 3 up to 1.12 within the cache; per state 10 qubits 0.80..0.93 from
  // 2^19, 1.10 below.  complex128: 0 1 0.64..0.94, others 1.04 below 2^19
  if (es == 16 && tb[1] == 1) return true;
  if (!c.from(19)) return false;
  if (c.per) return es == 8 || lines || c.up_to(21);
  return near && tb[1] <= (es == 16 || c.beyond() ? 3 : 2);
}

// Where the vector kernel keeps each state's operator in LDS that beats the scalar
// loads unless lines are saved (0 1 5 with 12 qubits x 64: 1.57); where it reads
// the operator from memory (10 qubits x 8192: 0.36..0.9) nearly everything gains.
bool low_pays_3(const LowCase& c) {
  const int* tb = c.tb;
  const bool near = c.near == 3, per = c.per, staged = c.staged;
  int lines = 0, first = 4;
  for (int m = 2; m >= 0; --m)
    if (tb[m] >= 1 && tb[m] <= 3) ++lines, first = tb[m];
  const bool bit0 = tb[0] == 0, one_two = tb[0] == 1 && tb[1] == 2;
  if (c.es == 4) {
    // 1 2 3 0.50..0.76; others without bit 0 0.91 up to 2^19, from there up to 1.36;
    // with it 1.06..1.53; beyond the cache two on lines 0.75, 1 4 6 0.80
    if (lines == 3) return !staged || c.from(18);
    if (staged) return false;
    if (c.beyond()) return lines == 2 || (near && (bit0 ? per : first == 1));
    return !bit0 && c.up_to(19) && (lines == 2 || (near && (!per || first < 4)));
  }
  if (c.es == 8) {
    if (bit0) {
      // 0 1 2 61 -> 52 (1.03 below 2^20); others 1.05..1.15 with one operator
      if (tb[2] == 2) return per ? !staged || c.from(21) : c.from(20);
      return near && per && !staged && c.from(20);
    }
    // 1 2 3 79 -> 50, h 1 2 64 -> 50; staged 1.10 below 2^19 and 1.20 below 2^20
    if (lines == 3) return !staged || c.from(19);
    if (one_two) return !staged || c.from(20);
    // h 1 3, h 2 3: 0.74..0.87 up to 2^20, 0.72..0.95 from 2^24, 1.03 between
    if (lines == 2) return staged ? c.beyond() : per || c.up_to(20) || c.from(24);
    // 4 5 6: 0.81..0.94 up to 2^20, 0.90 beyond the cache, 1.04..1.13 between
    if (staged || !near) return false;
    return per ? first < 3 || (first == 3 && c.from(21)) : c.up_to(20) || c.beyond();
  }
  if (bit0) {
    // 0 1 2 0.57..0.78, 0 1 5 0.64..0.84, h 0 1 0.66..0.93; 0 3 6 0.78 up to 2^19,
    // 1.09 above; h 0 2 0.79..0.95 up to 2^20, 0.80 from 2^24, 1.18 between
    if (tb[2] == 2) return !staged || c.from(19);
    if (tb[1] == 1) return !staged || (near && c.from(20));
    if (staged) return false;
    if (!near) return tb[1] == 2 && (per ? c.from(20) : c.up_to(20) || c.from(24));
    return per ? c.from(20) : c.up_to(19);
  }
  // 1 2 6 0.46..0.68, 1 4 6 0.57..0.85, h 1 3 0.62..0.85; staged 1.14 below 2^19
  if (first == 1) return one_two || !staged || c.from(near ? 18 : 19);
  // 2 5 7 0.57..0.96; h 2 3, h 2 6 0.63..0.84 up to 2^20, 0.80 from 2^24, 1.18 between
  if (first == 2 && near && lines == 1) return !staged || c.from(21);
  if (staged) return false;
  if (first == 2) return c.up_to(20) || c.from(per ? 23 : 24);
  // 4 5 6: 0.63..0.94 up to 2^21, 1.03..1.10 above
  return near && (per ? first == 3 && (c.up_to(20) || c.from(23)) : c.up_to(21));
}

}  // namespace

// Complex gates on 6..10 qubits on the matrix cores (wide_mfma.hip).
bool gemm_applies(int dtype, int n, int k, const void* out, const void* in, const void* op,
                  int64_t in_bstride);
int apply_dense_gemm(void* out, const void* in, const void* op, int dtype, int n, int k,
                     const int* tb, int64_t batch, int64_t in_bstride, int64_t op_bstride,
                     hipStream_t s);

// Tiled dense gates on 6..kMaxWideGateK qubits (wide.hip).
constexpr int kMaxWideGateK = 10;
bool wide_applies(int n, int k);
int apply_dense_wide(void* out, const void* in, const void* op, int dtype, int n, int k,
                     const int* tb, int64_t batch, int64_t in_bstride, int64_t out_bstride,
                     int64_t op_bstride, hipStream_t s);

// Validated entry used by ua_apply_operator and by other host code.
int apply_operator_impl(void* out, const void* state, const void* op, int dtype,
                        int n, int k, const int* qubits, int64_t batch,
                        int64_t state_bstride, int64_t op_bstride, hipStream_t s) {
  const size_t es = elem_size(dtype);
  UA_CHECK_ARG(es != 0, "unsupported dtype code %d", dtype);
  UA_CHECK_ARG(n >= 0 && n <= kMaxQubits, "num_qubits=%d out of range", n);
  UA_CHECK_ARG(k >= 0 && k <= n, "cannot apply a %d-qubit operator to %d qubit(s)", k, n);
  UA_CHECK_ARG(batch >= 0, "batch=%lld is negative", (long long)batch);
  UA_CHECK_ARG(state_bstride >= 0 && op_bstride >= 0, "negative batch stride");
  UA_CHECK_ARG(k == 0 || qubits != nullptr, "qubits is NULL");
  if (batch == 0) return UA_OK;
  UA_CHECK_ARG(out && state && op, "NULL data pointer");

  uint64_t seen = 0;
  for (int m = 0; m < k; ++m) {
    UA_CHECK_ARG(qubits[m] >= 0 && qubits[m] < n,
                 "qubit %d is not in range for a %d-qubit state", qubits[m], n);
    const uint64_t bit = uint64_t(1) << qubits[m];
    UA_CHECK_ARG(!(seen & bit), "qubit %d appears more than once", qubits[m]);
    seen |= bit;
  }
  const int64_t N = int64_t(1) << n;
  const bool in_place = (out == state);
  UA_CHECK_ARG(!in_place || state_bstride == N || batch == 1,
               "in-place application needs one state per batch entry");

  if (k >= 1 && k <= kMaxFastK) {
    FastParams p{};
    // canonical order: ascending state bit; gpos = caller's gate-index bit
    int tb[kMaxFastK], gp[kMaxFastK];
    for (int m = 0; m < k; ++m) {
      tb[m] = n - 1 - qubits[m];
      gp[m] = k - 1 - m;
    }
    for (int i = 1; i < k; ++i)  // insertion sort by tb
      for (int j = i; j > 0 && tb[j - 1] > tb[j]; --j) {
        int t0 = tb[j]; tb[j] = tb[j - 1]; tb[j - 1] = t0;
        int g0 = gp[j]; gp[j] = gp[j - 1]; gp[j - 1] = g0;
      }
    for (int m = 0; m < k; ++m) { p.tb[m] = tb[m]; p.gpos[m] = gp[m]; }
    // Matrix cores for the fused-block sizes where they measured faster on
    // MI355X (28-qubit complex64 / 27-qubit complex128 states): every 5-qubit
    // gate; complex128 4-qubit gates; complex64 4-qubit gates when all targets
    // lie in the low 6 bits (the vector kernel streams the others at HBM
    // speed: 26 qubits 208..225 us, matrix cores 222..235) or the states stay
    // in the caches, where the vector kernel waits for LDS and the matrix: 16
    // qubits 8.6..12.9 -> 3.0 us, 22 qubits 16.6..20 -> 14.5..16.8 (23 qubits
    // with several states in turn: 28..40 and 26..45, by the targets).  With a
    // target on bit 0, which the vector kernel pairs, the line is 2^21 amplitudes
    // (22 qubits 16.8 and 18.2).
    const bool mfma_shape =
        (k == 5 && dtype != UA_FLOAT32 && dtype != UA_FLOAT64) ||
        (k == 4 && dtype == UA_COMPLEX128) || (k == 4 && dtype == UA_COMPLEX64 &&
         (tb[k - 1] < 6 || batch <= ((int64_t(1) << (tb[0] == 0 ? 21 : 22)) >> n)));
    if (g_use_mfma && mfma_shape && op_bstride == 0 && n - k >= 6)
      return apply_dense_mfma(out, state, op, dtype, n, k, tb, gp, batch, state_bstride, s);

    const size_t pair_align = 2 * es;
    const bool io_aligned = aligned(state, state_bstride, es, pair_align) &&
                            aligned(out, N, es, pair_align);
    // measured on MI355X: 1-qubit gates stream best with one group pair per
    // thread, wider gates with two units per thread
    const int unr = (op_bstride != 0) ? 1 : (g_unroll ? g_unroll : (k == 1 ? 1 : 2));
    if (g_use_xch && k == 1 && io_aligned && op_bstride == 0 && n >= 7 && tb[0] >= 1 &&
        tb[0] <= 6) {
      XchParams x{};
      x.log2_ups = n - 1;
      x.total = batch << x.log2_ups;
      x.in_bstride = state_bstride;
      x.out_bstride = N;
      x.lane_mask = 1 << (tb[0] - 1);
      switch (dtype) {
        case UA_FLOAT32: launch_xch<float>(out, state, op, x, unr, s); break;
        case UA_FLOAT64: launch_xch<double>(out, state, op, x, unr, s); break;
        case UA_COMPLEX64: launch_xch<float2>(out, state, op, x, unr, s); break;
        case UA_COMPLEX128: launch_xch<double2>(out, state, op, x, unr, s); break;
      }
      return check_launch("dense_xch_kernel");
    }
    if ((k == 2 || k == 3) && io_aligned && n >= k + 6) {
      LowParams l{};
      int near = 0;                  // targets inside the contiguous run
      while (near < k && tb[near] < 6 + near + 1) ++near;
      LowCase c{es, tb, near, batch << n, op_bstride != 0, false};
      c.staged = k == 3 && c.per && n - k - (tb[0] == 0 ? 0 : 1) >= 8;
      const bool low = near > 0 && (batch << (n - k - 6)) >= (k == 3 ? 64 : 16) &&
                       (k == 2 ? low_pays_2(c) : low_pays_3(c));
      if (low) {
        l.beyond = k - near;
        l.log2_run = 6 + near;
        l.log2_wps = n - k - 6;
        l.total = batch << l.log2_wps;
        l.in_bstride = state_bstride;
        l.out_bstride = N;
        l.op_bstride = op_bstride;
        for (int m = 0; m < k; ++m) {
          l.tb[m] = m < near ? tb[m] : 6 + m;
          l.gpos[m] = gp[m];
          if (m >= near) l.hb[m - near] = tb[m];
        }
        switch (dtype) {
          case UA_FLOAT32: launch_low<float>(k, out, state, op, l, s); break;
          case UA_FLOAT64: launch_low<double>(k, out, state, op, l, s); break;
          case UA_COMPLEX64: launch_low<float2>(k, out, state, op, l, s); break;
          case UA_COMPLEX128: launch_low<double2>(k, out, state, op, l, s); break;
        }
        return check_launch("dense_low_kernel");
      }
    }
    int mode = SCALAR;
    if (io_aligned) mode = (tb[0] == 0) ? PAIR : VEC;
    const int log2_groups = n - k;  // groups per state
    const int log2_tps = log2_groups - (mode == VEC ? 1 : 0);
    p.log2_tps = log2_tps;
    p.total = batch << log2_tps;
    p.in_bstride = state_bstride;
    p.out_bstride = N;
    p.op_bstride = op_bstride;
    const bool lds = (k >= 3) && (op_bstride == 0 || log2_tps >= 8);
    switch (dtype) {
      case UA_FLOAT32: launch_fast_k_f32(k, mode, lds, out, state, op, p, unr, s); break;
      case UA_FLOAT64: launch_fast_k_f64(k, mode, lds, out, state, op, p, unr, s); break;
      case UA_COMPLEX64: launch_fast_k_c64(k, mode, lds, out, state, op, p, unr, s); break;
      case UA_COMPLEX128: launch_fast_k_c128(k, mode, lds, out, state, op, p, unr, s); break;
    }
    return check_launch("dense_fast_kernel");
  }

  // 7- and 8-qubit complex64 gates with one operator keep the vector kernel when
  // they run in place.  Not for speed (22 qubits 86 and 294 us; out of place on the
  // matrix cores 43 and 80): their in-place results have always been the vector
  // kernel's to the bit, and tests/test_gpu_parity.py holds them to that.
  const bool vector_in_place =
      in_place && op_bstride == 0 && dtype == UA_COMPLEX64 && (k == 7 || k == 8);
  if (g_use_mfma && !vector_in_place &&
      gemm_applies(dtype, n, k, out, state, op, state_bstride)) {
    int tbc[kMaxWideGateK];
    for (int m = 0; m < k; ++m) tbc[m] = n - 1 - qubits[m];
    return apply_dense_gemm(out, state, op, dtype, n, k, tbc, batch, state_bstride, op_bstride,
                            s);
  }
  if (wide_applies(n, k)) {  // 6..10 targets: tiled, in place or not
    int tbc[kMaxWideGateK];
    for (int m = 0; m < k; ++m) tbc[m] = n - 1 - qubits[m];
    return apply_dense_wide(out, state, op, dtype, n, k, tbc, batch, state_bstride, N,
                            op_bstride, s);
  }
  UA_CHECK_ARG(!in_place,
               "in-place application supports operators on 1..%d qubits (6..%d with at "
               "least 12 qubits)", kMaxFastK, kMaxWideGateK);
  UA_CHECK_ARG(k <= 20, "operators on more than 20 qubits are not supported");
  GenericParams g{};
  g.total = batch * N;
  g.in_bstride = state_bstride;
  g.op_bstride = op_bstride;
  g.n = n;
  g.k = k;
  g.tmask = 0;
  for (int m = 0; m < k; ++m) {
    g.tbit[m] = n - 1 - qubits[m];
    g.tmask |= uint64_t(1) << g.tbit[m];
  }
  const unsigned grid = grid_for(g.total);
  switch (dtype) {
    case UA_FLOAT32:
      dense_generic_kernel<float><<<grid, kBlock, 0, s>>>(
          (float*)out, (const float*)state, (const float*)op, g);
      break;
    case UA_FLOAT64:
      dense_generic_kernel<double><<<grid, kBlock, 0, s>>>(
          (double*)out, (const double*)state, (const double*)op, g);
      break;
    case UA_COMPLEX64:
      dense_generic_kernel<float2><<<grid, kBlock, 0, s>>>(
          (float2*)out, (const float2*)state, (const float2*)op, g);
      break;
    case UA_COMPLEX128:
      dense_generic_kernel<double2><<<grid, kBlock, 0, s>>>(
          (double2*)out, (const double2*)state, (const double2*)op, g);
      break;
  }
  return check_launch("dense_generic_kernel");
}

}  // namespace ua

extern "C" int ua_set_tuning(int key, int value) {
  switch (key) {
    case UA_TUNE_UNROLL:
      UA_CHECK_ARG(value == 0 || value == 1 || value == 2 || value == 4,
                   "unroll must be 0 (auto), 1, 2 or 4");
      ua::g_unroll = value;
      return UA_OK;
    case UA_TUNE_LANE_EXCHANGE:
      ua::g_use_xch = value != 0;
      return UA_OK;
    case UA_TUNE_MFMA:
      ua::g_use_mfma = value != 0;
      return UA_OK;
    case UA_TUNE_COMPILED_WAVES:
      return ua::set_compiled_waves(value);
  }
  ua::set_error("unknown tuning key %d", key);
  return UA_ERR_INVALID_ARGUMENT;
}

extern "C" int ua_apply_operator(void* out, const void* state, const void* op,
                                 int dtype, int num_qubits, int op_num_qubits,
                                 const int* qubits, int64_t batch,
                                 int64_t state_batch_stride,
                                 int64_t op_batch_stride, ua_stream_t stream) {
  return ua::apply_operator_impl(out, state, op, dtype, num_qubits, op_num_qubits,
                                 qubits, batch, state_batch_stride, op_batch_stride,
                                 static_cast<hipStream_t>(stream));
}
