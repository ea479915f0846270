// Kernels for adjoint differentiation of Pauli-rotation circuits with the
// observable H = sum_i Z_i.
//
// unitair has no gradient code: its circuits are differentiated by torch
// autograd through apply_operator / apply_phase (unitair/simulation/
// operations.py:41-42,322), the gate builders (unitair/gates/gates.py:35-91)
// and the loss diag_expectation_value (unitair/states/innerprod.py:49-59),
// which keeps one saved state per gate.  The adjoint method keeps two states
// (psi and the co-state lambda = H psi pulled back through the gates) and
// needs, per rotation exp(-i t/2 P_q):
//     dL/dt = Im <lambda| P_q |psi>
// evaluated at the point right after that gate.  Same-kind rotations on
// different qubits commute, so one (lambda, psi) point serves every qubit of a
// layer: ua_pauli_gradients returns all n values of a layer in one call.
#include <algorithm>

#include "mfma_common.h"
#include "ua_common.h"

namespace ua {
namespace {

constexpr int kLowBits = 12;
constexpr int kLowTile = 1 << kLowBits;
constexpr int kMaxN = 40;
constexpr int kZChunkConst = 4096;

template <typename T> struct D2;
template <> struct D2<float2> {
  __device__ static double2 get(float2 v) { return make_double2(v.x, v.y); }
};
template <> struct D2<double2> {
  __device__ static double2 get(double2 v) { return v; }
};

// Re(conj(a) * b)
__device__ __forceinline__ double re_cj(double2 a, double2 b) { return a.x * b.x + a.y * b.y; }
// Im(conj(a) * b)
__device__ __forceinline__ double im_cj(double2 a, double2 b) { return a.x * b.y - a.y * b.x; }

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
  return v;
}

// Sums of 16 values over a wavefront at once: at each of the first four steps a
// lane hands half of its values to its partner and keeps the sums of the other
// half, the last two steps add what is left (17 exchanges; 16 sums one after
// another take 96).  Returns the sum of value `which`, the lane's top four bits.
__device__ __forceinline__ double wave_sums(double (&v)[16], int& which) {
  const int lane = threadIdx.x & 63;
  int cnt = 16;
  which = 0;
#pragma unroll
  for (int m = 32; m >= 4; m >>= 1) {
    cnt >>= 1;
    const bool upper = lane & m;
#pragma unroll
    for (int i = 0; i < cnt; ++i)
      v[i] = (upper ? v[i + cnt] : v[i]) + __shfl_xor(upper ? v[i] : v[i + cnt], m, 64);
    which += upper ? cnt : 0;
  }
  v[0] += __shfl_xor(v[0], 2, 64);
  v[0] += __shfl_xor(v[0], 1, 64);
  return v[0];
}

// Sums v over the workgroup (256 threads); result in thread 0.
__device__ double block_sum(double v, double* scratch) {
  v = wave_sum(v);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  __syncthreads();
  if (lane == 0) scratch[wave] = v;
  __syncthreads();
  double r = 0.0;
  if (threadIdx.x == 0)
    for (int w = 0; w < kBlock / 64; ++w) r += scratch[w];
  return r;
}

// Im <lambda| P_b |psi> summed over one amplitude pair (x0 with bit b clear,
// x1 = x0 | 2^b), for P = X or Y:
//   X: (P psi)_x = psi_{x^b}             -> Im(l0* p1) + Im(l1* p0)
//   Y: (P psi)_{x0} = -i psi_{x1},
//      (P psi)_{x1} =  i psi_{x0}        -> Re(l1* p0) - Re(l0* p1)
template <int P>
__device__ __forceinline__ double pair_term(double2 l0, double2 l1, double2 p0, double2 p1) {
  if constexpr (P == UA_PAULI_X) return im_cj(l0, p1) + im_cj(l1, p0);
  else return re_cj(l1, p0) - re_cj(l0, p1);
}

// X / Y gradients for index bits 0..min(n,12)-1.  One workgroup per (state,
// tile of 2^m contiguous amplitudes); lambda and psi tiles sit in LDS.
// partial[(b * tiles + tile) * n + bit] = sum over the tile's pairs.
template <typename T, int P>
__global__ __launch_bounds__(kBlock) void grad_low_kernel(
    double* __restrict__ partial, const T* __restrict__ lam, const T* __restrict__ psi,
    int n, int m, int64_t tiles_per_state) {
  __shared__ T sl[kLowTile];
  __shared__ T sp[kLowTile];
  __shared__ double scratch[kBlock / 64];
  const int64_t tile = blockIdx.x;
  const int64_t b = tile / tiles_per_state;
  const int64_t t = tile % tiles_per_state;
  const int64_t N = int64_t(1) << n;
  const int size = 1 << m;
  const T* L = lam + b * N + t * size;
  const T* Ps = psi + b * N + t * size;
  for (int i = threadIdx.x; i < size; i += kBlock) {
    sl[i] = L[i];
    sp[i] = Ps[i];
  }
  __syncthreads();
  for (int bit = 0; bit < m; ++bit) {
    double acc = 0.0;
    const int half = size >> 1;
    for (int pidx = threadIdx.x; pidx < half; pidx += kBlock) {
      const int x0 = ((pidx >> bit) << (bit + 1)) | (pidx & ((1 << bit) - 1));
      const int x1 = x0 | (1 << bit);
      acc += pair_term<P>(D2<T>::get(sl[x0]), D2<T>::get(sl[x1]), D2<T>::get(sp[x0]),
                          D2<T>::get(sp[x1]));
    }
    const double s = block_sum(acc, scratch);
    if (threadIdx.x == 0) partial[(b * tiles_per_state + t) * n + bit] = s;
  }
}

// pair_term in the state's precision, returned as double (the sums are
// float64): complex64 terms are formed in float32 (relative rounding 6e-8
// per term, far inside complex64 state error), complex128 in double.
template <int P>
__device__ __forceinline__ double pair_term_of(float2 l0, float2 l1, float2 p0, float2 p1) {
  float r;
  if constexpr (P == UA_PAULI_X)
    r = (l0.x * p1.y - l0.y * p1.x) + (l1.x * p0.y - l1.y * p0.x);
  else
    r = (l1.x * p0.x + l1.y * p0.y) - (l0.x * p1.x + l0.y * p1.y);
  return double(r);
}
template <int P>
__device__ __forceinline__ double pair_term_of(double2 l0, double2 l1, double2 p0, double2 p1) {
  return pair_term<P>(l0, l1, p0, p1);
}

// The same sums for full 4096-amplitude tiles (m = 12, every state of 12 or more
// qubits) with the work in registers: a thread's 16 loads of either state are the
// cube of tile bits 8..11; both tiles go to LDS, from where it reads the cubes of
// bits 0..3 and 4..7, and it adds the pair terms of each cube's 4 bits.  The sums
// stay in registers over all tiles of the workgroup until one reduction.  LDS
// position of element e: e ^ ((e >> 4) & 15), so the copy and both cube reads
// touch distinct banks across 16 lanes.
//
// 16 qubits x 1024 states, complex64 (1 GiB of both states): 262 us with Z, where
// X / Y took 295 and Z another 264.  What it cost was the reduction, 12 sums of
// every wavefront for each tile; one for a run of tiles and 17 exchanges for 16
// sums leave the reads (4.1 TB/s) and LDS.  More wavefronts with smaller cubes
// were slower (504 us), the next tile's loads ahead too (385, spilled registers).
__device__ __forceinline__ int low_swz(int e) { return e ^ ((e >> 4) & 15); }

constexpr int kMaxRun = 16;  // tiles of a workgroup

template <int P, int B0, typename T>
__device__ __forceinline__ void cube_terms(double (&acc)[16], const T (&l)[16], const T (&p)[16]) {
#pragma unroll
  for (int k = 0; k < 4; ++k)
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      if (j & (1 << k)) continue;
      const int j1 = j | (1 << k);
      acc[B0 + k] += pair_term_of<P>(l[j], l[j1], p[j], p[j1]);
    }
}

template <int P, int B0, typename T>
__device__ __forceinline__ void low_cube(double (&acc)[16], const T* sl, const T* sp, int e0) {
  T l[16], p[16];
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    l[j] = sl[low_swz(e0 | (j << B0))];
    p[j] = sp[low_swz(e0 | (j << B0))];
  }
  cube_terms<P, B0>(acc, l, p);
}

// A workgroup takes `run` (a power of two, at most 16) consecutive tiles of a
// state: partial[(b * runs + r) * n + bit].
// Z: also the Z gradients, in zpartial[(b * runs + r) * n + qubit].  The thread
// that copies elements tid + 256 k has the cube of bits 8..11 in registers, so
// those bits and Z need no read of LDS.
template <typename T, int P, bool Z>
__global__ __launch_bounds__(kBlock)
__attribute__((amdgpu_waves_per_eu(sizeof(T) == 8 ? 2 : 1))) void grad_low_full_kernel(
    double* __restrict__ partial, double* __restrict__ zpartial, const T* __restrict__ lam,
    const T* __restrict__ psi, int n, int64_t runs_per_state, int run) {
  __shared__ T sl[kLowTile];
  __shared__ T sp[kLowTile];
  __shared__ double red[kBlock / 64][16];
  __shared__ double zred[kBlock / 64][16];
  const int64_t b = blockIdx.x / runs_per_state;
  const int64_t r0 = blockIdx.x % runs_per_state;
  const int64_t N = int64_t(1) << n;
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const T* L = lam + b * N + r0 * run * kLowTile + tid;
  const T* Ps = psi + b * N + r0 * run * kLowTile + tid;
  double acc[16];
  // signed sums of Z: bits 8..11 (0..3), bits 12..15 within the run (4..7), the total (8)
  double z[Z ? 9 : 1];
#pragma unroll
  for (int i = 0; i < 16; ++i) acc[i] = 0.0;
#pragma unroll
  for (int i = 0; i < (Z ? 9 : 1); ++i) z[i] = 0.0;
  for (int t = 0; t < run; ++t, L += kLowTile, Ps += kLowTile) {
    T l[16], p[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      l[k] = L[k * kBlock];
      p[k] = Ps[k * kBlock];
    }
    if (t > 0) __syncthreads();  // the tile before is read
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      sl[low_swz(tid + k * kBlock)] = l[k];
      sp[low_swz(tid + k * kBlock)] = p[k];
    }
    __syncthreads();
    cube_terms<P, 8>(acc, l, p);
    if constexpr (Z) {
      double total = 0.0;
#pragma unroll
      for (int k = 0; k < 16; ++k) {
        const double v = im_cj(D2<T>::get(l[k]), D2<T>::get(p[k]));
        total += v;
#pragma unroll
        for (int bit = 0; bit < 4; ++bit) z[bit] += ((k >> bit) & 1) ? -v : v;
      }
#pragma unroll
      for (int bit = 0; bit < 4; ++bit) z[4 + bit] += ((t >> bit) & 1) ? -total : total;
      z[8] += total;
    }
    // the empty asm keeps the LDS reads of each part after the arithmetic of the
    // one before: all hoisted, the registers overflow
    asm volatile("" ::: "memory");
    // thread tid's cube entry 0: tid's 8 bits around the cube's 4
    low_cube<P, 0>(acc, sl, sp, tid << 4);
    asm volatile("" ::: "memory");
    low_cube<P, 4>(acc, sl, sp, (tid & 15) | ((tid >> 4) << 8));
  }
  int which;
  const double sum = wave_sums(acc, which);
  if ((lane & 3) == 0) red[wave][which] = sum;
  if constexpr (Z) {
    double v[16];  // z as it is, then bits 0..5 as 9..14
#pragma unroll
    for (int i = 0; i < 9; ++i) v[i] = z[i];
#pragma unroll
    for (int bit = 0; bit < 6; ++bit) v[9 + bit] = ((tid >> bit) & 1) ? -z[8] : z[8];
    v[15] = 0.0;
    const double zs = wave_sums(v, which);
    if ((lane & 3) == 0) zred[wave][which] = zs;
  }
  __syncthreads();
  if (tid < kLowBits) {
    double r = 0.0;
#pragma unroll
    for (int w = 0; w < kBlock / 64; ++w) r += red[w][tid];
    partial[(b * runs_per_state + r0) * n + tid] = r;
  }
  if constexpr (Z) {
    if (tid < n) {
      const int bit = tid;  // index bit: of the lanes, the wavefronts, the cube, the run or above
      const bool in_run = bit >= kLowBits && bit < kLowBits + 4 && (run >> (bit - kLowBits)) > 1;
      double r = 0.0;
#pragma unroll
      for (int w = 0; w < kBlock / 64; ++w) {
        const double total = zred[w][8];
        if (bit < 6) r += zred[w][9 + bit];
        else if (bit < 8) r += ((w >> (bit - 6)) & 1) ? -total : total;
        else if (bit < kLowBits) r += zred[w][bit - 8];
        else if (in_run) r += zred[w][4 + bit - kLowBits];
        else r += (((r0 * run) >> (bit - kLowBits)) & 1) ? -total : total;
      }
      zpartial[(b * runs_per_state + r0) * n + (n - 1 - bit)] = r;
    }
  }
}

// X / Y gradients for a window of H index bits w0..w0+H-1 (w0 >= 12).  Each
// thread owns one low index (bits 0..11: 256 consecutive per workgroup, so
// every load is coalesced) and, for each value r of the other high bits in
// its block's range, the 2^H amplitudes over the window.  A workgroup takes
// `chunks` neighbouring chunks of 256 low indices, so that one reduction serves
// them all (16 qubits x 1024 states: 238 -> 214 us, 5.0 TB/s).
// partial[((b * gridDim.y + blockIdx.y) * gridDim.z + blockIdx.z) * n + bit].
template <typename T, int P, int H>
__global__ __launch_bounds__(kBlock) void grad_high_kernel(
    double* __restrict__ partial, const T* __restrict__ lam, const T* __restrict__ psi, int n,
    int w0, int64_t rest_per_block, int chunks) {
  __shared__ double red[kBlock / 64][16];
  constexpr int HN = 1 << H;
  const int64_t b = blockIdx.x;
  const int64_t N = int64_t(1) << n;
  const int below = w0 - kLowBits;                    // other high bits under the window
  double acc[16];
#pragma unroll
  for (int hb = 0; hb < 16; ++hb) acc[hb] = 0.0;
  const int64_t r0 = int64_t(blockIdx.z) * rest_per_block;
  for (int64_t r = r0; r < r0 + rest_per_block; ++r) {
    const uint64_t rest = ((uint64_t(r) & ((uint64_t(1) << below) - 1)) << kLowBits) |
                          ((uint64_t(r) >> below) << (w0 + H));
    for (int c = 0; c < chunks; ++c) {
      const int low = (int(blockIdx.y) * chunks + c) * kBlock + threadIdx.x;  // < 4096
      const int64_t base = b * N + int64_t(rest) + low;
      T l[HN], p[HN];
#pragma unroll
      for (int h = 0; h < HN; ++h) {
        l[h] = lam[base + (int64_t(h) << w0)];
        p[h] = psi[base + (int64_t(h) << w0)];
      }
#pragma unroll
      for (int hb = 0; hb < H; ++hb) {
        // the amplitudes stay in the state's own type: as float64 for all bits at
        // once they take twice the registers (230, two wavefronts per SIMD)
#pragma unroll
        for (int h = 0; h < HN; ++h)
          asm volatile("" : "+v"(l[h].x), "+v"(l[h].y), "+v"(p[h].x), "+v"(p[h].y));
#pragma unroll
        for (int h = 0; h < HN; ++h) {
          if (h & (1 << hb)) continue;
          const int h1 = h | (1 << hb);
          acc[hb] += pair_term<P>(D2<T>::get(l[h]), D2<T>::get(l[h1]), D2<T>::get(p[h]),
                                  D2<T>::get(p[h1]));
        }
      }
    }
  }
  const int64_t part = (b * gridDim.y + blockIdx.y) * gridDim.z + blockIdx.z;
  int which;
  const double sum = wave_sums(acc, which);
  if ((threadIdx.x & 3) == 0) red[threadIdx.x >> 6][which] = sum;
  __syncthreads();
  if (threadIdx.x < H) {
    double t = 0.0;
#pragma unroll
    for (int w = 0; w < kBlock / 64; ++w) t += red[w][threadIdx.x];
    partial[part * n + w0 + threadIdx.x] = t;
  }
}

// Z gradients (and, with want_loss, the loss sum_x |psi_x|^2 (n-2 popcount x)).
// A workgroup covers a chunk of 4096 amplitudes of one state (or the whole
// state when it is smaller); thread t visits i = chunk_base + t + 256*k.
// Index bits 0..7 of i are fixed per thread, bits 8..11 follow k and bits
// >= 12 are fixed per chunk, so each thread keeps 16 partial sums (one per k)
// and the per-qubit signs are applied afterwards.
// partial[(b * chunks + c) * (n + 1) + q]; slot n holds the loss part.
template <typename T>
__global__ __launch_bounds__(kBlock) void grad_z_kernel(
    double* __restrict__ partial, const T* __restrict__ lam, const T* __restrict__ psi, int n,
    int64_t chunks, int want_loss) {
  constexpr int K = kZChunkConst / kBlock;  // 16
  const int64_t b = blockIdx.x / chunks;
  const int64_t c = blockIdx.x % chunks;
  const int64_t N = int64_t(1) << n;
  const int64_t base = c * kZChunkConst;
  double vk[K];
  double loss = 0.0;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    vk[k] = 0.0;
    const int64_t i = base + threadIdx.x + int64_t(k) * kBlock;
    if (i < N) {
      const double2 pv = D2<T>::get(psi[b * N + i]);
      if (want_loss) {
        const double w = pv.x * pv.x + pv.y * pv.y;
        loss += w * double(n - 2 * int(__popcll(uint64_t(i))));
      }
      if (lam) vk[k] = im_cj(D2<T>::get(lam[b * N + i]), pv);
    }
  }
  double total = 0.0;
#pragma unroll
  for (int k = 0; k < K; ++k) total += vk[k];
  // this thread's share of each low bit's signed sum (bits >= 12 are fixed
  // per chunk: plus or minus the chunk's total), the total and the loss,
  // reduced together once
  constexpr int kVals = kLowBits + 2;
  double vals[kVals];
#pragma unroll
  for (int bit = 0; bit < 8; ++bit) vals[bit] = ((threadIdx.x >> bit) & 1) ? -total : total;
#pragma unroll
  for (int bit = 8; bit < kLowBits; ++bit) {
    double v = 0.0;
#pragma unroll
    for (int k = 0; k < K; ++k) v += ((k >> (bit - 8)) & 1) ? -vk[k] : vk[k];
    vals[bit] = v;
  }
  vals[kLowBits] = total;
  vals[kLowBits + 1] = loss;
  __shared__ double red[kBlock / 64][kVals];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int i = 0; i < kVals; ++i) {
    const double v = wave_sum(vals[i]);
    if (lane == 0) red[wave][i] = v;
  }
  __syncthreads();
  if (threadIdx.x < kVals) {
    double r = 0.0;
#pragma unroll
    for (int w = 0; w < kBlock / 64; ++w) r += red[w][threadIdx.x];
    red[0][threadIdx.x] = r;  // each thread reads and writes only its own column
  }
  __syncthreads();
  double* out = partial + (b * chunks + c) * (n + 1);
  if (want_loss && threadIdx.x == 0) out[n] = red[0][kLowBits + 1];
  if (!lam) return;
  for (int bit = threadIdx.x; bit < n; bit += kBlock) {
    const double sum = bit < kLowBits ? red[0][bit]
                                      : (((base >> bit) & 1) ? -red[0][kLowBits]
                                                             : red[0][kLowBits]);
    out[n - 1 - bit] = sum;
  }
}

// out[b * out_stride + out_q0 + out_dir * q] = sum over `parts` rows of
// partial[(b*parts + r)*stride + q0 + q], q < n_out (out_dir -1: index bit
// q0 + q is qubit out_q0 - q)
__global__ __launch_bounds__(kBlock) void sum_parts_kernel(
    double* __restrict__ out, const double* __restrict__ partial, int64_t batch, int64_t parts,
    int stride, int q0, int n_out, int out_stride, int out_q0, int accumulate, int out_dir) {
  const int64_t idx = int64_t(blockIdx.x) * kBlock + threadIdx.x;
  if (idx >= batch * n_out) return;
  const int64_t b = idx / n_out;
  const int q = int(idx % n_out);
  double s = 0.0;
  for (int64_t r = 0; r < parts; ++r) s += partial[(b * parts + r) * stride + q0 + q];
  double* o = out + b * out_stride + out_q0 + out_dir * q;
  *o = accumulate ? *o + s : s;
}

// lambda_x = (n - 2 popcount(x)) psi_x
template <typename T>
__global__ __launch_bounds__(kBlock) void sum_z_apply_kernel(T* __restrict__ out,
                                                             const T* __restrict__ psi, int n,
                                                             int64_t total) {
  const int64_t stride = int64_t(gridDim.x) * kBlock;
  const uint64_t mask = (uint64_t(1) << n) - 1;
  for (int64_t i = int64_t(blockIdx.x) * kBlock + threadIdx.x; i < total; i += stride) {
    const auto w = decltype(psi[0].x)(n - 2 * int(__popcll(uint64_t(i) & mask)));
    T v = psi[i];
    v.x *= w;
    v.y *= w;
    out[i] = v;
  }
}

int64_t y_low_parts(int n) { return n > kLowBits ? (int64_t(1) << (n - kLowBits)) : 1; }
constexpr int64_t kHighParts = kLowTile / kBlock;  // 16 low chunks per state
constexpr int kHighWindow = 4;                      // index bits per high-bit launch
// Splits of the other high bits of a window launch across blockIdx.z: enough
// workgroups to fill the GPU (about 2048 per launch) with at least one value
// of the other bits each.
int64_t high_z(int n, int64_t batch) {
  const int rest_bits = n - kLowBits - kHighWindow;
  if (rest_bits <= 0) return 1;
  int64_t z = (2048 + batch * kHighParts - 1) / (batch * kHighParts);
  const int64_t rest = int64_t(1) << rest_bits;
  if (z > rest) z = rest;
  int64_t p2 = 1;
  while (p2 * 2 <= z) p2 *= 2;   // a power of two divides the rest count
  return p2;
}
int64_t z_parts(int n) {
  return ((int64_t(1) << n) + kZChunkConst - 1) / kZChunkConst;
}

}  // namespace
}  // namespace ua

using namespace ua;

extern "C" int64_t ua_pauli_gradients_workspace(int num_qubits, int64_t batch) {
  const int n = num_qubits;
  if (n < 1 || n > kMaxN || batch < 0) return -1;
  int64_t a = y_low_parts(n) * n;
  const int64_t h = kHighParts * high_z(n, batch < 1 ? 1 : batch) * n;
  const int64_t z = z_parts(n) * (n + 1);
  if (h > a) a = h;
  if (z > a) a = z;
  if (n >= kLowBits && 2 * y_low_parts(n) * n > a) a = 2 * y_low_parts(n) * n;  // X / Y and Z
  return (batch < 1 ? 1 : batch) * a * int64_t(sizeof(double));
}

namespace ua {
namespace {
// z_out: NULL, or where the Z gradients go as well (X / Y on at least 12 qubits;
// their partials follow the others' in the workspace).
int pauli_gradients(double* out, double* z_out, const void* lambda, const void* psi, int dtype,
                    int n, int64_t batch, int pauli, void* workspace, ua_stream_t stream) {
  hipStream_t s = static_cast<hipStream_t>(stream);
  UA_CHECK_ARG(dtype == UA_COMPLEX64 || dtype == UA_COMPLEX128, "complex states only");
  UA_CHECK_ARG(n >= 1 && n <= kMaxN, "num_qubits=%d out of range", n);
  UA_CHECK_ARG(pauli == UA_PAULI_X || pauli == UA_PAULI_Y || pauli == UA_PAULI_Z,
               "pauli must be X, Y or Z");
  UA_CHECK_ARG(batch >= 0, "negative batch");
  if (batch == 0) return UA_OK;
  UA_CHECK_ARG(out && lambda && psi && workspace, "NULL pointer");
  double* part = static_cast<double*>(workspace);
  const bool c64 = dtype == UA_COMPLEX64;
  if (pauli == UA_PAULI_Z) {
    const int64_t chunks = z_parts(n);
    UA_CHECK_ARG(batch * chunks <= 0x7fffffffLL, "grid too large");
    const unsigned g = unsigned(batch * chunks);
    if (c64)
      grad_z_kernel<float2><<<g, kBlock, 0, s>>>(part, (const float2*)lambda, (const float2*)psi,
                                                 n, chunks, 0);
    else
      grad_z_kernel<double2><<<g, kBlock, 0, s>>>(part, (const double2*)lambda,
                                                  (const double2*)psi, n, chunks, 0);
    int rc = check_launch("grad_z_kernel");
    if (rc) return rc;
    // out[b*n + q] = sum over chunks (partials are stored by qubit)
    sum_parts_kernel<<<grid_for(batch * n), kBlock, 0, s>>>(out, part, batch, chunks, n + 1, 0, n,
                                                            n, 0, 0, 1);
    return check_launch("sum_parts_kernel");
  }
  // X / Y: index bit i belongs to qubit n-1-i; partials are kept per index
  // bit and mapped to qubits when summed.
  const int m = n < kLowBits ? n : kLowBits;
  const int64_t tiles = y_low_parts(n);
  UA_CHECK_ARG(batch * tiles <= 0x7fffffffLL, "grid too large");
  // full tiles: runs of them for a workgroup, as long as 2048 workgroups are left
  int run = 1;
  if (m == kLowBits)
    while (run < kMaxRun && run < tiles && batch * (tiles / (2 * run)) >= 2048) run *= 2;
  const int64_t runs = tiles / run;
  const unsigned glow = unsigned(batch * runs);
  double* const zpart = part + batch * tiles * n;
#define UA_LOW(TT, PP)                                                                   \
  do {                                                                                   \
    if (m == kLowBits && z_out)                                                          \
      grad_low_full_kernel<TT, PP, true><<<glow, kBlock, 0, s>>>(                        \
          part, zpart, (const TT*)lambda, (const TT*)psi, n, runs, run);                     \
    else if (m == kLowBits)                                                              \
      grad_low_full_kernel<TT, PP, false><<<glow, kBlock, 0, s>>>(                       \
          part, nullptr, (const TT*)lambda, (const TT*)psi, n, runs, run);                   \
    else                                                                                 \
      grad_low_kernel<TT, PP><<<glow, kBlock, 0, s>>>(part, (const TT*)lambda,           \
                                                      (const TT*)psi, n, m, tiles);       \
  } while (0)
  if (pauli == UA_PAULI_X) {
    if (c64) UA_LOW(float2, UA_PAULI_X); else UA_LOW(double2, UA_PAULI_X);
  } else {
    if (c64) UA_LOW(float2, UA_PAULI_Y); else UA_LOW(double2, UA_PAULI_Y);
  }
#undef UA_LOW
  int rc = check_launch("grad_low_kernel");
  if (rc) return rc;
  if (z_out) {  // stored by qubit
    sum_parts_kernel<<<grid_for(batch * n), kBlock, 0, s>>>(z_out, zpart, batch, runs, n, 0, n, n,
                                                            0, 0, 1);
    rc = check_launch("sum_parts_kernel");
    if (rc) return rc;
  }
  // bits 0..m-1 -> qubits n-1 .. n-m, one launch
  sum_parts_kernel<<<grid_for(batch * m), kBlock, 0, s>>>(out, part, batch, runs, n, 0, m, n,
                                                          n - 1, 0, -1);
  rc = check_launch("sum_parts_kernel");
  if (rc) return rc;
  // high bits, kHighWindow at a time; each launch reads both states once
  UA_CHECK_ARG(batch <= 0x7fffffffLL, "grid too large");
  const int64_t z = high_z(n, batch);
  for (int w0 = kLowBits; w0 < n; w0 += kHighWindow) {
    const int H = (n - w0) < kHighWindow ? (n - w0) : kHighWindow;
    const int rest_bits = n - kLowBits - H;
    const int64_t zz = rest_bits > 0 ? z : 1;
    const int64_t per_block = (int64_t(1) << (rest_bits > 0 ? rest_bits : 0)) / zz;
    int chunks = 1;  // of low indices, as long as 2048 workgroups are left
    while (chunks < kHighParts && batch * zz * (kHighParts / (2 * chunks)) >= 2048) chunks *= 2;
    const int64_t parts = kHighParts / chunks;
    const dim3 grid = dim3(unsigned(batch), unsigned(parts), unsigned(zz));
#define UA_HIGH(HH)                                                                             \
  if (H == HH) {                                                                               \
    if (pauli == UA_PAULI_X) {                                                                 \
      if (c64)                                                                                 \
        grad_high_kernel<float2, UA_PAULI_X, HH><<<grid, kBlock, 0, s>>>(                      \
            part, (const float2*)lambda, (const float2*)psi, n, w0, per_block, chunks);        \
      else                                                                                     \
        grad_high_kernel<double2, UA_PAULI_X, HH><<<grid, kBlock, 0, s>>>(                     \
            part, (const double2*)lambda, (const double2*)psi, n, w0, per_block, chunks);      \
    } else {                                                                                   \
      if (c64)                                                                                 \
        grad_high_kernel<float2, UA_PAULI_Y, HH><<<grid, kBlock, 0, s>>>(                      \
            part, (const float2*)lambda, (const float2*)psi, n, w0, per_block, chunks);        \
      else                                                                                     \
        grad_high_kernel<double2, UA_PAULI_Y, HH><<<grid, kBlock, 0, s>>>(                     \
            part, (const double2*)lambda, (const double2*)psi, n, w0, per_block, chunks);      \
    }                                                                                          \
  }
    UA_HIGH(1) UA_HIGH(2) UA_HIGH(3) UA_HIGH(4)
#undef UA_HIGH
    rc = check_launch("grad_high_kernel");
    if (rc) return rc;
    // bits w0..w0+H-1 -> qubits n-1-w0 .. n-w0-H, one launch
    sum_parts_kernel<<<grid_for(batch * H), kBlock, 0, s>>>(out, part, batch, parts * zz, n,
                                                            w0, H, n, n - 1 - w0, 0, -1);
    rc = check_launch("sum_parts_kernel");
    if (rc) return rc;
  }
  return UA_OK;
}

// whether one launch can give the Z gradients beside the X / Y ones
bool z_beside(int n) { return n >= kLowBits; }
}  // namespace
}  // namespace ua

extern "C" int ua_pauli_gradients(double* out, const void* lambda, const void* psi, int dtype,
                                  int num_qubits, int64_t batch, int pauli, void* workspace,
                                  ua_stream_t stream) {
  return pauli_gradients(out, nullptr, lambda, psi, dtype, num_qubits, batch, pauli, workspace,
                         stream);
}

extern "C" int ua_pauli_gradients_z(double* out, double* z_out, const void* lambda,
                                    const void* psi, int dtype, int num_qubits, int64_t batch,
                                    int pauli, void* workspace, ua_stream_t stream) {
  UA_CHECK_ARG(pauli == UA_PAULI_X || pauli == UA_PAULI_Y, "pauli must be X or Y");
  UA_CHECK_ARG(batch <= 0 || z_out, "NULL pointer");
  if (num_qubits >= 1 && num_qubits <= kMaxN && !z_beside(num_qubits)) {
    const int rc = pauli_gradients(z_out, nullptr, lambda, psi, dtype, num_qubits, batch,
                                   UA_PAULI_Z, workspace, stream);
    if (rc) return rc;
    z_out = nullptr;
  }
  return pauli_gradients(out, z_out, lambda, psi, dtype, num_qubits, batch, pauli, workspace,
                         stream);
}

namespace ua {
namespace {
// out_x = d_x psi_x with a real diagonal d (one row, or one row per state)
template <typename T, typename D>
__global__ __launch_bounds__(kBlock) void diag_scale_kernel(T* __restrict__ out,
                                                            const T* __restrict__ psi,
                                                            const D* __restrict__ diag, int n,
                                                            int64_t total, int64_t dstride) {
  const int64_t stride = int64_t(gridDim.x) * kBlock;
  const uint64_t mask = (uint64_t(1) << n) - 1;
  for (int64_t i = int64_t(blockIdx.x) * kBlock + threadIdx.x; i < total; i += stride) {
    const auto w = decltype(psi[0].x)(diag[(i >> n) * dstride + int64_t(uint64_t(i) & mask)]);
    T v = psi[i];
    v.x *= w;
    v.y *= w;
    out[i] = v;
  }
}
}  // namespace
}  // namespace ua

extern "C" int ua_apply_diagonal(void* out, const void* psi, int dtype, const void* diag,
                                 int diag_dtype, int64_t diag_batch_stride, int num_qubits,
                                 int64_t batch, ua_stream_t stream) {
  const int n = num_qubits;
  UA_CHECK_ARG(dtype == UA_COMPLEX64 || dtype == UA_COMPLEX128, "complex states only");
  UA_CHECK_ARG(diag_dtype == UA_FLOAT32 || diag_dtype == UA_FLOAT64, "real diagonal only");
  UA_CHECK_ARG(n >= 0 && n <= 62 && batch >= 0 && diag_batch_stride >= 0, "bad sizes");
  if (batch == 0) return UA_OK;
  UA_CHECK_ARG(out && psi && diag, "NULL pointer");
  const int64_t total = batch << n;
  int64_t blocks = (total + kBlock - 1) / kBlock;
  if (blocks > 65536) blocks = 65536;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const unsigned g = unsigned(blocks);
#define UA_DS(T, D)                                                                     \
  diag_scale_kernel<T, D><<<g, kBlock, 0, s>>>((T*)out, (const T*)psi, (const D*)diag, n, \
                                               total, diag_batch_stride)
  if (dtype == UA_COMPLEX64) {
    if (diag_dtype == UA_FLOAT32) UA_DS(float2, float); else UA_DS(float2, double);
  } else {
    if (diag_dtype == UA_FLOAT32) UA_DS(double2, float); else UA_DS(double2, double);
  }
#undef UA_DS
  return check_launch("diag_scale_kernel");
}

extern "C" int ua_apply_sum_z(void* out, const void* psi, int dtype, int num_qubits,
                              int64_t batch, ua_stream_t stream) {
  const int n = num_qubits;
  UA_CHECK_ARG(dtype == UA_COMPLEX64 || dtype == UA_COMPLEX128, "complex states only");
  UA_CHECK_ARG(n >= 1 && n <= 62 && batch >= 0, "bad sizes");
  if (batch == 0) return UA_OK;
  UA_CHECK_ARG(out && psi, "NULL pointer");
  const int64_t total = batch << n;
  int64_t blocks = (total + kBlock - 1) / kBlock;
  if (blocks > 65536) blocks = 65536;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (dtype == UA_COMPLEX64)
    sum_z_apply_kernel<float2><<<unsigned(blocks), kBlock, 0, s>>>((float2*)out,
                                                                   (const float2*)psi, n, total);
  else
    sum_z_apply_kernel<double2><<<unsigned(blocks), kBlock, 0, s>>>((double2*)out,
                                                                    (const double2*)psi, n, total);
  return check_launch("sum_z_apply_kernel");
}

extern "C" int ua_expect_sum_z(double* out, const void* psi, int dtype, int num_qubits,
                               int64_t batch, void* workspace, ua_stream_t stream) {
  const int n = num_qubits;
  hipStream_t s = static_cast<hipStream_t>(stream);
  UA_CHECK_ARG(dtype == UA_COMPLEX64 || dtype == UA_COMPLEX128, "complex states only");
  UA_CHECK_ARG(n >= 1 && n <= kMaxN && batch >= 0, "bad sizes");
  if (batch == 0) return UA_OK;
  UA_CHECK_ARG(out && psi && workspace, "NULL pointer");
  double* part = static_cast<double*>(workspace);
  const int64_t chunks = z_parts(n);
  UA_CHECK_ARG(batch * chunks <= 0x7fffffffLL, "grid too large");
  const unsigned g = unsigned(batch * chunks);
  if (dtype == UA_COMPLEX64)
    grad_z_kernel<float2><<<g, kBlock, 0, s>>>(part, nullptr, (const float2*)psi, n, chunks, 1);
  else
    grad_z_kernel<double2><<<g, kBlock, 0, s>>>(part, nullptr, (const double2*)psi, n, chunks, 1);
  int rc = check_launch("grad_z_kernel");
  if (rc) return rc;
  sum_parts_kernel<<<grid_for(batch), kBlock, 0, s>>>(out, part, batch, chunks, n + 1, n, 1, 1, 0,
                                                      0, 1);
  return check_launch("sum_parts_kernel");
}

// ---------------------------------------------------------------------------
// Gradient of apply_operator with respect to the operator (backward of
// unitair/simulation/operations.py:322, out = U @ in on the target bits):
//   grad_U[o][r][c] = sum over batch entries b using operator o, and over
//                     groups g:  grad_out[b][g|off(r)] * conj(in[b][g|off(c)])
// i.e. grad_U = G^T conj(X) with G, X the (groups x 2^k) views of grad_out
// and in: a tall-skinny product whose reduction runs over 2^(n-k) groups.
//
// op_grad_partial_kernel: a workgroup owns one operator o, one slice ("part")
// of that operator's groups and one RB x CB block of the 2^k x 2^k result.
// Each thread walks the slice with stride 256 (consecutive threads take
// consecutive groups, so every load is coalesced), keeps the block's RB*CB
// products in float64 registers, and the workgroup reduces them with
// wavefront shuffles and LDS.  With one part the sums go straight to grad_op;
// otherwise to the float64 workspace, and op_grad_finish_kernel adds the
// parts (one workgroup per result entry).  k = 1, 2 take the whole result in
// one block (each amplitude read once); larger k tile it 4 x 4, unless
// op_grad_on_mfma prefers op_grad_mfma_kernel.
//
// GS (k = 1, 2): the thread holds whole groups of grad_out, so it also forms the
// state's gradient U^H grad_out of them: one read of grad_out less, and no
// adjoint operator to make first (22 qubits x 3 states, k = 2, forward and
// backward: 195 -> 153 us, of which the kernels are about 100).  In complex128 with
// a target on bit 0 and 2^15 to 2^18 amplitudes the one kernel takes longer than the
// two it replaces (16 qubits, bits 0 and 1: 25.4 and 21.9 us with what makes the
// adjoint operator), but its call less on the host (89 and 111 us for the whole
// backward there).
namespace ua {
namespace {

struct OpGradParams {
  int n, k;
  int64_t batch, op_count;   // op_count: distinct operators (1 or batch)
  int64_t in_bstride;        // 0 when one input state serves the whole batch
  int64_t parts;             // slices of each operator's groups
  int64_t units;             // groups per operator: (batch / op_count) << (n - k)
  int64_t units_per_part;
  int nblk_c;                // column blocks: 2^k / CB
  int tbit[UA_MAX_GRAD_QUBITS];    // state bit of gate-index bit k-1-m (qubits order)
  int sorted[UA_MAX_GRAD_QUBITS];  // target state bits, ascending
};

template <typename T> __device__ __forceinline__ double2 as_d2(T v);
template <> __device__ __forceinline__ double2 as_d2(float v) { return make_double2(v, 0.0); }
template <> __device__ __forceinline__ double2 as_d2(double v) { return make_double2(v, 0.0); }
template <> __device__ __forceinline__ double2 as_d2(float2 v) { return make_double2(v.x, v.y); }
template <> __device__ __forceinline__ double2 as_d2(double2 v) { return v; }

template <typename T> __device__ __forceinline__ T from_d2(double2 v);
template <> __device__ __forceinline__ float from_d2(double2 v) { return float(v.x); }
template <> __device__ __forceinline__ double from_d2(double2 v) { return v.x; }
template <> __device__ __forceinline__ float2 from_d2(double2 v) { return make_float2(float(v.x), float(v.y)); }
template <> __device__ __forceinline__ double2 from_d2(double2 v) { return v; }

__device__ __forceinline__ uint64_t gate_offset(int idx, const OpGradParams& p) {
  uint64_t o = 0;
  for (int m = 0; m < p.k; ++m)
    if ((idx >> (p.k - 1 - m)) & 1) o |= uint64_t(1) << p.tbit[m];
  return o;
}

// acc + conj(u) * a
__device__ __forceinline__ float cj_mac(float acc, float u, float a) { return fmaf(u, a, acc); }
__device__ __forceinline__ double cj_mac(double acc, double u, double a) { return fma(u, a, acc); }
template <typename T>
__device__ __forceinline__ T cj_mac(T acc, T u, T a) {
  acc.x = fma(u.x, a.x, acc.x);
  acc.x = fma(u.y, a.y, acc.x);
  acc.y = fma(u.x, a.y, acc.y);
  acc.y = fma(-u.y, a.x, acc.y);
  return acc;
}

template <typename T, int RB, int CB, int UNR, bool GS>
__global__ __launch_bounds__(kBlock) void op_grad_partial_kernel(
    T* __restrict__ grad_op, double* __restrict__ part_out, const T* __restrict__ gout,
    const T* __restrict__ in, T* __restrict__ grad_state, const T* __restrict__ op,
    OpGradParams p) {
  __shared__ double2 red[kBlock / 64][RB * CB];
  const int64_t D = int64_t(1) << p.k;
  const int blk = int(blockIdx.x % unsigned(p.nblk_c * (D / RB)));
  const int64_t rest = int64_t(blockIdx.x) / (p.nblk_c * (D / RB));
  const int64_t part = rest % p.parts;
  const int64_t o = rest / p.parts;
  const int r0 = (blk / p.nblk_c) * RB, c0 = (blk % p.nblk_c) * CB;
  uint64_t offr[RB], offc[CB];
#pragma unroll
  for (int i = 0; i < RB; ++i) offr[i] = gate_offset(r0 + i, p);
#pragma unroll
  for (int j = 0; j < CB; ++j) offc[j] = gate_offset(c0 + j, p);

  const int gbits = p.n - p.k;
  const int64_t N = int64_t(1) << p.n;
  const int64_t u_begin = part * p.units_per_part;
  int64_t u_end = u_begin + p.units_per_part;
  if (u_end > p.units) u_end = p.units;
  T um[GS ? RB : 1][GS ? CB : 1];  // the whole operator
  if constexpr (GS) {
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
      for (int j = 0; j < CB; ++j) um[i][j] = op[(o * RB + i) * CB + j];
  }
  double2 acc[RB][CB];
#pragma unroll
  for (int i = 0; i < RB; ++i)
#pragma unroll
    for (int j = 0; j < CB; ++j) acc[i][j] = make_double2(0.0, 0.0);
  // UNR groups per iteration, all their loads issued before any product
  for (int64_t u0 = u_begin + threadIdx.x; u0 < u_end; u0 += UNR * kBlock) {
    T gr[UNR][RB], xr[UNR][CB];
#pragma unroll
    for (int q = 0; q < UNR; ++q) {
      const int64_t u = u0 + q * kBlock;
      if (u >= u_end) continue;
      const int64_t b = (p.op_count == 1) ? (u >> gbits) : o;
      const uint64_t gi = uint64_t(u) & ((uint64_t(1) << gbits) - 1);
      const uint64_t base = insert_zero_bits(gi, p.sorted, p.k);
      const T* gb = gout + b * N + base;
      const T* xb = in + b * p.in_bstride + base;
#pragma unroll
      for (int i = 0; i < RB; ++i) gr[q][i] = gb[offr[i]];
#pragma unroll
      for (int j = 0; j < CB; ++j) xr[q][j] = xb[offc[j]];
    }
#pragma unroll
    for (int q = 0; q < UNR; ++q) {
      if (u0 + q * kBlock >= u_end) continue;
      if constexpr (GS) {
        const int64_t u = u0 + q * kBlock;
        const int64_t b = (p.op_count == 1) ? (u >> gbits) : o;
        T* sb = grad_state + b * N +
                insert_zero_bits(uint64_t(u) & ((uint64_t(1) << gbits) - 1), p.sorted, p.k);
#pragma unroll
        for (int j = 0; j < CB; ++j) {
          T v{};
#pragma unroll
          for (int i = 0; i < RB; ++i) v = cj_mac(v, um[i][j], gr[q][i]);
          sb[offc[j]] = v;
        }
      }
#pragma unroll
      for (int i = 0; i < RB; ++i)
#pragma unroll
        for (int j = 0; j < CB; ++j) {
          // g * conj(x)
          const double2 g = as_d2(gr[q][i]), x = as_d2(xr[q][j]);
          acc[i][j].x = fma(g.x, x.x, fma(g.y, x.y, acc[i][j].x));
          acc[i][j].y = fma(g.y, x.x, fma(-g.x, x.y, acc[i][j].y));
        }
    }
  }
  // workgroup reduction: shuffles inside each wavefront, then LDS
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int i = 0; i < RB; ++i)
#pragma unroll
    for (int j = 0; j < CB; ++j) {
      double vr = acc[i][j].x, vi = acc[i][j].y;
#pragma unroll
      for (int d = 32; d > 0; d >>= 1) {
        vr += __shfl_xor(vr, d, 64);
        vi += __shfl_xor(vi, d, 64);
      }
      if (lane == 0) red[wave][i * CB + j] = make_double2(vr, vi);
    }
  __syncthreads();
  if (threadIdx.x < RB * CB) {
    double2 t = red[0][threadIdx.x];
#pragma unroll
    for (int w = 1; w < kBlock / 64; ++w) {
      t.x += red[w][threadIdx.x].x;
      t.y += red[w][threadIdx.x].y;
    }
    const int64_t e = int64_t(r0 + threadIdx.x / CB) * D + (c0 + threadIdx.x % CB);
    if (p.parts == 1) {
      grad_op[o * D * D + e] = from_d2<T>(t);
    } else {
      double* dst = part_out + ((o * p.parts + part) * D * D + e) * 2;
      dst[0] = t.x;
      dst[1] = t.y;
    }
  }
}

// The same for operators on 4 qubits (complex) and 5 (complex64), 16 A = 2^k rows:
// the whole result in one workgroup, on the matrix cores.  Four groups are the depth of a
// v_mfma_f64_16x16x4f64: lane l holds row l % 16 (+ 16 a) of group l / 16 of G
// and of X, as loaded, and G^T conj(X) is four real products for each pair of
// 16-row blocks.  Every amplitude is read once (the 4 x 4 blocks above read it
// 2^k / 4 times and convert it each time); products are float64 and exact for
// complex64, as there.  Bound by memory and the float64 products together: 22
// qubits x 3 states complex64, 4 targets 105..331 -> 47..62 us by the targets, 5
// targets 169..784 -> 78..92; 21 qubits complex128, 4 targets 97..291 -> 57..68; 10
// qubits x 301 operators of their own 84 -> 7.1.  (complex128 on 5 qubits would
// take too many registers for sums as short as the ones it has.)
// A lane takes UNR neighbouring groups, one for each step: with no target on
// the lowest index bits (RUN) they are neighbours in memory too.
template <typename T, int A, bool RUN>
__global__ __launch_bounds__(kBlock) void op_grad_mfma_kernel(
    T* __restrict__ grad_op, double* __restrict__ part_out, const T* __restrict__ gout,
    const T* __restrict__ in, OpGradParams p) {
  constexpr int D = 16 * A, K = 3 + A, kWaves = kBlock / 64, UNR = 4;
  // complex128: sums of their own for each step of a run and each of the two
  // products.  One long chain had twice the rounding error of the many short
  // ones of the kernel above (7e-16 against 3.4e-16); so it is no larger (18
  // qubits x 3: 2.2e-16 against 2.6e-16).
  constexpr int S = sizeof(T) == 16 ? 2 * UNR : 1;
  using M = Mfma<double>;
  __shared__ double2 red[D * D];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
  const int64_t part = int64_t(blockIdx.x) % p.parts, o = int64_t(blockIdx.x) / p.parts;
  uint64_t off[A];
#pragma unroll
  for (int a = 0; a < A; ++a) off[a] = gate_offset(16 * a + (lane & 15), p);
  const int gbits = p.n - p.k;
  const int64_t N = int64_t(1) << p.n;
  const int64_t u_begin = part * p.units_per_part;
  int64_t u_end = u_begin + p.units_per_part;
  if (u_end > p.units) u_end = p.units;
  M::acc_t re[S][A][A], im[S][A][A];
#pragma unroll
  for (int s = 0; s < S; ++s)
#pragma unroll
    for (int a = 0; a < A; ++a)
#pragma unroll
      for (int c = 0; c < A; ++c) re[s][a][c] = im[s][a][c] = M::acc_t{0.0, 0.0, 0.0, 0.0};
  struct alignas(16) Run { T v[UNR]; };
  for (int64_t u0 = u_begin + 4 * UNR * wave; u0 < u_end; u0 += 4 * UNR * kWaves) {  // wave-uniform
    Run g[A], x[A];
    const int64_t u = u0 + UNR * (lane >> 4);
#pragma unroll
    for (int q = 0; q < (RUN ? 1 : UNR); ++q) {
      const bool ok = u + q < u_end;            // RUN: for all UNR of them
      const int64_t v = ok ? u + q : u_begin;   // past the end: zeros count for nothing
      const int64_t b = (p.op_count == 1) ? (v >> gbits) : o;
      const uint64_t base =
          insert_zero_bits(uint64_t(v) & ((uint64_t(1) << gbits) - 1), p.sorted, K);
#pragma unroll
      for (int a = 0; a < A; ++a) {
        const T* gp = gout + b * N + base + off[a];
        const T* xp = in + b * p.in_bstride + base + off[a];
        if constexpr (RUN) {
          g[a] = *reinterpret_cast<const Run*>(gp);
          x[a] = *reinterpret_cast<const Run*>(xp);
          if (!ok) g[a] = x[a] = Run{};
        } else {
          g[a].v[q] = ok ? *gp : T{};
          x[a].v[q] = ok ? *xp : T{};
        }
      }
    }
#pragma unroll
    for (int q = 0; q < UNR; ++q)
#pragma unroll
      for (int a = 0; a < A; ++a)
#pragma unroll
        for (int c = 0; c < A; ++c) {            // g * conj(x)
          const double2 gv = as_d2(g[a].v[q]), xv = as_d2(x[c].v[q]);
          const int s0 = q % S, s1 = (q + UNR) % S;
          re[s0][a][c] = M::mma(gv.x, xv.x, re[s0][a][c]);
          im[s0][a][c] = M::mma(gv.y, xv.x, im[s0][a][c]);
          re[s1][a][c] = M::mma(gv.y, xv.y, re[s1][a][c]);
          im[s1][a][c] = M::mma(-gv.x, xv.y, im[s1][a][c]);
        }
  }
#pragma unroll
  for (int h = S / 2; h > 0; h /= 2)
#pragma unroll
    for (int s = 0; s < h; ++s)
#pragma unroll
      for (int a = 0; a < A; ++a)
#pragma unroll
        for (int c = 0; c < A; ++c) {
          re[s][a][c] += re[s + h][a][c];
          im[s][a][c] += im[s + h][a][c];
        }
  for (int w = 0; w < kWaves; ++w) {
    if (wave == w) {
#pragma unroll
      for (int a = 0; a < A; ++a)
#pragma unroll
        for (int c = 0; c < A; ++c)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            double2& e = red[(16 * a + M::row(lane, i)) * D + 16 * c + (lane & 15)];
            e.x = (w ? e.x : 0.0) + re[0][a][c][i];
            e.y = (w ? e.y : 0.0) + im[0][a][c][i];
          }
    }
    __syncthreads();
  }
  for (int e = threadIdx.x; e < D * D; e += kBlock) {
    if (p.parts == 1) {
      grad_op[o * D * D + e] = from_d2<T>(red[e]);
    } else {
      double* dst = part_out + ((o * p.parts + part) * D * D + e) * 2;
      dst[0] = red[e].x;
      dst[1] = red[e].y;
    }
  }
}

// One workgroup per (operator, entry): the threads split the parts, then
// reduce with wavefront shuffles and LDS.
template <typename T>
__global__ __launch_bounds__(kBlock) void op_grad_finish_kernel(T* __restrict__ grad_op,
                                                                const double* __restrict__ part,
                                                                int64_t parts, int64_t DD) {
  __shared__ double2 red[kBlock / 64];
  const int64_t t = blockIdx.x;  // o * DD + e
  const int64_t o = t / DD, e = t % DD;
  double vr = 0.0, vi = 0.0;
  for (int64_t q = threadIdx.x; q < parts; q += kBlock) {
    const double* src = part + ((o * parts + q) * DD + e) * 2;
    vr += src[0];
    vi += src[1];
  }
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) {
    vr += __shfl_xor(vr, d, 64);
    vi += __shfl_xor(vi, d, 64);
  }
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = make_double2(vr, vi);
  __syncthreads();
  if (threadIdx.x == 0) {
    double2 sum = red[0];
#pragma unroll
    for (int w = 1; w < kBlock / 64; ++w) {
      sum.x += red[w].x;
      sum.y += red[w].y;
    }
    grad_op[t] = from_d2<T>(sum);
  }
}

// Launch shape shared by the workspace query and the entry point.
struct OpGradShape {
  int rb, cb;
  int64_t nblk, parts, units, units_per_part;
};

// Complex operators on 4 qubits and complex64 ones on 5: whether the matrix cores
// (op_grad_mfma_kernel) are faster than the 4 x 4 blocks.  They are where one
// workgroup does an operator (up to 128 groups of 4 qubits, 64 of 5; 256 operators
// of 64 groups 71 -> 4 and 272 -> 8 us) and where the groups are many (5 qubits,
// 4096: 17.5 -> 13.2); between, several operators wait for their parts' whole
// results to be written and added (16 of 4 qubits, 256 groups each: 9.2 -> 10.7 in
// complex64, 9.1 -> 12.7 in complex128; one of 5, 512 groups: 9.8 -> 12.8).  With
// low targets, which the blocks read worst, the line lies lower (16 of 4 qubits,
// 1024 groups: complex64 13.7 -> 11.7, complex128 19.7 -> 12.6; one of 5, 2048:
// 16.5 -> 13.3).  sorted: ascending target bits; groups: of one operator.
bool op_grad_on_mfma(int dtype, int k, const int* sorted, int64_t groups, int64_t op_count) {
  const bool c64 = dtype == UA_COMPLEX64, several = op_count >= 8;
  const bool low = c64 ? sorted[k - 1] < 6 : sorted[0] == 0;
  if (k == 4 && (c64 || dtype == UA_COMPLEX128))
    return !several || groups <= 128 || groups >= (c64 ? 2048 : 4096) || (low && groups >= 1024);
  if (k == 5 && c64)
    return groups <= (several ? 128 : 64) || groups >= 4096 ||
           (low && groups >= (several ? 1024 : 2048));
  return false;
}

OpGradShape op_grad_shape(int n, int k, int64_t batch, int64_t op_count, bool mfma) {
  OpGradShape sh{};
  const int64_t D = int64_t(1) << k;
  sh.rb = sh.cb = int(D < 4 ? D : 4);
  sh.nblk = (D / sh.rb) * (D / sh.cb);
  sh.units = (batch / op_count) << (n - k);
  // about 4096 workgroups in all, each thread with at least 16 groups
  const int64_t want = (4096 + op_count * sh.nblk - 1) / (op_count * sh.nblk);
  const int64_t most = (sh.units + kBlock * 16 - 1) / (kBlock * 16);
  sh.parts = want < most ? want : most;
  if (mfma) {
    // one workgroup a part (op_grad_mfma_kernel): four per CU for 4 qubits, two
    // for 5 (half as many: complex64 6 % slower, complex128 chains of twice the
    // length), each with at least 128 groups (with 256: 14 qubits 14 -> 20 us)
    const int64_t fill = ((k == 4 ? 1024 : 512) + op_count - 1) / op_count;
    const int64_t full = (sh.units + 127) / 128;
    sh.parts = fill < full ? fill : full;
  }
  if (sh.parts < 1) sh.parts = 1;
  sh.units_per_part = (sh.units + sh.parts - 1) / sh.parts;
  if (mfma) {                        // whole runs of neighbouring groups in a part
    sh.units_per_part = (sh.units_per_part + 15) / 16 * 16;
    sh.parts = (sh.units + sh.units_per_part - 1) / sh.units_per_part;
  }
  return sh;
}

template <typename T>
void launch_op_grad(int rb, unsigned grid, T* grad, double* part, const T* g, const T* x, T* gs,
                    const T* op, const OpGradParams& p, hipStream_t s) {
  if (rb == 1)
    op_grad_partial_kernel<T, 1, 1, 4, false><<<grid, kBlock, 0, s>>>(grad, part, g, x, gs, op, p);
  else if (rb == 2 && gs)
    op_grad_partial_kernel<T, 2, 2, 4, true><<<grid, kBlock, 0, s>>>(grad, part, g, x, gs, op, p);
  else if (rb == 2)
    op_grad_partial_kernel<T, 2, 2, 4, false><<<grid, kBlock, 0, s>>>(grad, part, g, x, gs, op, p);
  else if (gs)
    op_grad_partial_kernel<T, 4, 4, 2, true><<<grid, kBlock, 0, s>>>(grad, part, g, x, gs, op, p);
  else
    op_grad_partial_kernel<T, 4, 4, 2, false><<<grid, kBlock, 0, s>>>(grad, part, g, x, gs, op, p);
}

template <typename T, int A>
void launch_op_grad_mfma(unsigned grid, T* grad, double* part, const T* g, const T* x,
                         const OpGradParams& p, hipStream_t s) {
  // a lane's four neighbouring groups as one run
  const bool run = p.sorted[0] >= 2 && reinterpret_cast<uintptr_t>(g) % 16 == 0 &&
                   reinterpret_cast<uintptr_t>(x) % 16 == 0 && p.in_bstride % 2 == 0;
  if (run) op_grad_mfma_kernel<T, A, true><<<grid, kBlock, 0, s>>>(grad, part, g, x, p);
  else op_grad_mfma_kernel<T, A, false><<<grid, kBlock, 0, s>>>(grad, part, g, x, p);
}

}  // namespace
}  // namespace ua

extern "C" int64_t ua_operator_gradient_workspace_bytes(int num_qubits, int op_num_qubits,
                                                       int64_t batch, int64_t op_count) {
  const int n = num_qubits, k = op_num_qubits;
  if (n < 1 || n > 62 || k < 0 || k > n || k > UA_MAX_GRAD_QUBITS || batch < 0 ||
      !(op_count == 1 || op_count == batch))
    return -1;
  if (batch == 0) return 0;
  // for whichever type: complex ones take the matrix cores
  int64_t parts = ua::op_grad_shape(n, k, batch, op_count, false).parts;
  if (k == 4 || k == 5)
    parts = std::max(parts, ua::op_grad_shape(n, k, batch, op_count, true).parts);
  if (parts == 1) return 0;
  return op_count * parts * (int64_t(1) << (2 * k)) * 2 * int64_t(sizeof(double));
}

namespace ua {
namespace {
// grad_state / op: NULL, or the state's gradient to form as well and the operators
int operator_gradient(void* grad_op, void* grad_state, const void* grad_out, const void* state,
                      const void* op, int dtype, int n, int k, const int* qubits, int64_t batch,
                      int64_t op_count, int64_t state_batch_stride, void* workspace,
                      ua_stream_t stream) {
  UA_CHECK_ARG(elem_size(dtype) != 0, "bad dtype");
  UA_CHECK_ARG(n >= 1 && n <= 62 && k >= 0 && k <= n && k <= UA_MAX_GRAD_QUBITS,
               "bad qubit counts (n=%d, k=%d)", n, k);
  UA_CHECK_ARG(batch >= 0 && (op_count == 1 || op_count == batch), "op_count must be 1 or batch");
  if (batch == 0) return UA_OK;
  UA_CHECK_ARG(grad_op && grad_out && state, "NULL pointer");
  OpGradParams p{};
  p.n = n;
  p.k = k;
  p.batch = batch;
  p.op_count = op_count;
  p.in_bstride = state_batch_stride;
  uint64_t seen = 0;
  for (int m = 0; m < k; ++m) {
    UA_CHECK_ARG(qubits[m] >= 0 && qubits[m] < n, "qubit out of range");
    p.tbit[m] = n - 1 - qubits[m];
    UA_CHECK_ARG(!((seen >> p.tbit[m]) & 1), "duplicate qubit");
    seen |= uint64_t(1) << p.tbit[m];
  }
  for (int b = 0, m = 0; b < n; ++b)
    if ((seen >> b) & 1) p.sorted[m++] = b;
  const bool mfma = op_grad_on_mfma(dtype, k, p.sorted,
                                    op_count == 1 ? batch << (n - k) : int64_t(1) << (n - k),
                                    op_count);
  const OpGradShape sh = op_grad_shape(n, k, batch, op_count, mfma);
  p.parts = sh.parts;
  p.units = sh.units;
  p.units_per_part = sh.units_per_part;
  p.nblk_c = int((int64_t(1) << k) / sh.cb);
  const int64_t blocks = op_count * sh.parts * sh.nblk;
  UA_CHECK_ARG(blocks <= 0x7fffffffLL, "grid too large");
  UA_CHECK_ARG(sh.parts == 1 || (workspace && reinterpret_cast<uintptr_t>(workspace) % 8 == 0),
               "workspace (ua_operator_gradient_workspace_bytes) missing or misaligned");
  hipStream_t s = static_cast<hipStream_t>(stream);
  double* part = static_cast<double*>(workspace);
  const unsigned grid = unsigned(blocks);
  if (mfma) {
    const unsigned mgrid = unsigned(op_count * sh.parts);
    if (dtype == UA_COMPLEX128)
      launch_op_grad_mfma<double2, 1>(mgrid, (double2*)grad_op, part, (const double2*)grad_out,
                                      (const double2*)state, p, s);
    else if (k == 4)
      launch_op_grad_mfma<float2, 1>(mgrid, (float2*)grad_op, part, (const float2*)grad_out,
                                     (const float2*)state, p, s);
    else
      launch_op_grad_mfma<float2, 2>(mgrid, (float2*)grad_op, part, (const float2*)grad_out,
                                     (const float2*)state, p, s);
  } else switch (dtype) {
    case UA_FLOAT32:
      launch_op_grad(sh.rb, grid, (float*)grad_op, part, (const float*)grad_out, (const float*)state,
                     (float*)grad_state, (const float*)op, p, s);
      break;
    case UA_FLOAT64:
      launch_op_grad(sh.rb, grid, (double*)grad_op, part, (const double*)grad_out, (const double*)state,
                     (double*)grad_state, (const double*)op, p, s);
      break;
    case UA_COMPLEX64:
      launch_op_grad(sh.rb, grid, (float2*)grad_op, part, (const float2*)grad_out, (const float2*)state,
                     (float2*)grad_state, (const float2*)op, p, s);
      break;
    case UA_COMPLEX128:
      launch_op_grad(sh.rb, grid, (double2*)grad_op, part, (const double2*)grad_out, (const double2*)state,
                     (double2*)grad_state, (const double2*)op, p, s);
      break;
  }
  if (int rc = check_launch("op_grad_partial_kernel")) return rc;
  if (sh.parts == 1) return UA_OK;
  const int64_t DD = int64_t(1) << (2 * k);
  UA_CHECK_ARG(op_count * DD <= 0x7fffffffLL, "grid too large");
  const unsigned fgrid = unsigned(op_count * DD);
  switch (dtype) {
    case UA_FLOAT32: op_grad_finish_kernel<float><<<fgrid, kBlock, 0, s>>>((float*)grad_op, part, sh.parts, DD); break;
    case UA_FLOAT64: op_grad_finish_kernel<double><<<fgrid, kBlock, 0, s>>>((double*)grad_op, part, sh.parts, DD); break;
    case UA_COMPLEX64: op_grad_finish_kernel<float2><<<fgrid, kBlock, 0, s>>>((float2*)grad_op, part, sh.parts, DD); break;
    case UA_COMPLEX128: op_grad_finish_kernel<double2><<<fgrid, kBlock, 0, s>>>((double2*)grad_op, part, sh.parts, DD); break;
  }
  return check_launch("op_grad_finish_kernel");
}
}  // namespace
}  // namespace ua

extern "C" int ua_operator_gradient(void* grad_op, const void* grad_out, const void* state,
                                    int dtype, int num_qubits, int op_num_qubits,
                                    const int* qubits, int64_t batch, int64_t op_count,
                                    int64_t state_batch_stride, void* workspace,
                                    ua_stream_t stream) {
  return ua::operator_gradient(grad_op, nullptr, grad_out, state, nullptr, dtype, num_qubits,
                               op_num_qubits, qubits, batch, op_count, state_batch_stride,
                               workspace, stream);
}

extern "C" int ua_operator_backward(void* grad_op, void* grad_state, const void* grad_out,
                                    const void* state, const void* op, int dtype,
                                    int num_qubits, int op_num_qubits, const int* qubits,
                                    int64_t batch, int64_t op_count, void* workspace,
                                    ua_stream_t stream) {
  using namespace ua;
  UA_CHECK_ARG(op_num_qubits == 1 || op_num_qubits == 2,
               "ua_operator_backward takes operators on 1 or 2 qubits (got %d)", op_num_qubits);
  UA_CHECK_ARG(num_qubits >= 1 && num_qubits <= 62, "num_qubits=%d out of range", num_qubits);
  UA_CHECK_ARG(batch <= 0 || (grad_state && op), "NULL pointer");
  UA_CHECK_ARG(batch <= 0 || (grad_state != grad_out && grad_state != state),
               "grad_state must not alias an input");
  return operator_gradient(grad_op, grad_state, grad_out, state, op, dtype, num_qubits,
                           op_num_qubits, qubits, batch, op_count, int64_t(1) << num_qubits,
                           workspace, stream);
}
