// The Chebyshev solve of one local/global pass in a single launch: every
// workgroup owns a tile of rows, keeps their M^2 entries in registers for all
// the sweeps and exchanges only the iterates with the tiles around it.
//
// What bounds it: the streamed sweeps (k_solve.hip) read the whole matrix once
// per sweep (5 to 10 bytes per entry) and pay a kernel boundary per sweep;
// below about 100 k rows both are larger than the arithmetic.  The registers
// of the chip (512 KB per compute unit) hold such a matrix, so here it is read
// once per solve, and a sweep is LDS reads and FMAs on the tile plus one
// exchange of the iterate over the Infinity Cache.  Per sweep of a 256^2
// cloth (256 tiles of 256 rows): about 1 us of LDS reads and 1 us of exchange
// against 4.7 us (FP32) and 8.6 us (FP64) for the streamed kernels.
//
// Tiles: compact in space (recursive bisection of the rest positions, model by
// model), at most one per compute unit, so that all of them are resident
// together and the waits below end.  Thread (row, part) holds the entries of
// 8 / TPR of the row's 8 SELL lanes and sums each lane's entries in the
// streamed kernels' order; the lane sums are combined in the order of their
// shuffle tree, so every iterate is bit-identical to the streamed sweeps'.
// Rows are consecutive across a wavefront's lanes: at one step the lanes read
// nearly consecutive LDS rows (the streamed kernels' 8 lanes per row read 8
// scattered ones).
//
// Exchange: an iterate's row is published as 8-byte words (FP32: (x, y) and
// (z, 0); FP64: x, y, z) by relaxed agent-scope atomic stores, and read by the
// neighbours with relaxed agent-scope atomic loads that repeat until the word
// is no longer kTileEmpty, a NaN no iterate can hold.  The data are their own
// flag: no fence and no barrier between workgroups.  Publication j of a launch
// goes to slot j % 4.  After publishing j a thread empties its words of
// publication j - 2: it has staged publication j - 1 of all neighbours, who had
// staged j - 2 before publishing it (the neighbour relation is symmetric).  It
// waits for that store before it publishes j + 1 (a whole sweep later, so the
// wait is over when it begins); a reader reaches publication j + 2, the same
// slot as j - 2, only after it has staged this thread's publication j + 1, and
// so finds the emptied word or the new value.  The last two publications of a
// launch stay; launches alternate between two sets of slots, each emptying the
// other set.
//
// Every wait is bounded (kTileWaitTicks): a tile whose neighbours do not
// arrive -- another process's kernels hold compute units for good -- raises
// the abort flag, every tile leaves, X keeps a finite value, and the host
// repeats the outer iteration with the streamed kernels.
#include "device.hpp"

namespace pdipc {
namespace {

constexpr unsigned long long kTileEmpty = 0xfff5a5a5fff5a5a5ull;
constexpr unsigned long long kTileWaitTicks = 1000000ull;  // 10 ms of the 100 MHz wall clock
constexpr int kPollBatch = 6;  // words per thread polled together

__device__ __forceinline__ void publish(unsigned long long* p, unsigned long long v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned long long peek(const unsigned long long* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template <class T> struct TileWords;
template <> struct TileWords<float> {
  using V2 = float2;
  static constexpr int N = 2;  // words per row
  static __device__ __forceinline__ unsigned long long word(const float (&d)[3], int w) {
    return w == 0 ? ((unsigned long long)__float_as_uint(d[1]) << 32) | __float_as_uint(d[0])
                  : (unsigned long long)__float_as_uint(d[2]);
  }
  static __device__ __forceinline__ void unpack(unsigned long long v, int w, float2* xy, float* z, int u) {
    if (w == 0) xy[u] = make_float2(__uint_as_float((unsigned)v), __uint_as_float((unsigned)(v >> 32)));
    else z[u] = __uint_as_float((unsigned)v);
  }
};
template <> struct TileWords<double> {
  using V2 = double2;
  static constexpr int N = 3;
  static __device__ __forceinline__ unsigned long long word(const double (&d)[3], int w) {
    return (unsigned long long)__double_as_longlong(w == 0 ? d[0] : (w == 1 ? d[1] : d[2]));
  }
  static __device__ __forceinline__ void unpack(unsigned long long v, int w, double2* xy, double* z, int u) {
    const double x = __longlong_as_double((long long)v);
    if (w == 0) xy[u].x = x;
    else if (w == 1) xy[u].y = x;
    else z[u] = x;
  }
};

// The sum of a row's 8 lane sums in the order of the streamed kernels' shuffle
// tree (xor 4, 2, 1): thread `part` of TPR holds lanes part, part + TPR, ...
template <int TPR, class T>
__device__ __forceinline__ T lane_tree(const T (&s)[8 / TPR]) {
  if constexpr (TPR == 1) return ((s[0] + s[4]) + (s[2] + s[6])) + ((s[1] + s[5]) + (s[3] + s[7]));
  if constexpr (TPR == 2) {
    const T a = (s[0] + s[2]) + (s[1] + s[3]);
    return a + __shfl_xor(a, 32, kWave);
  }
  if constexpr (TPR == 4) {
    T a = s[0] + s[1];
    a += __shfl_xor(a, 32, kWave);
    return a + __shfl_xor(a, 16, kWave);
  }
}

struct TileShape {  // what one launch works on (device pointers of DeviceMesh)
  int n, ld, R, uCap;
  const int4* rows;     // [tile][R]: row (-1 past the last), its first SELL entry, entries per lane
  const int* haloOff;   // [tile + 1]
  const int* halo;      // rows of other tiles that the tile's entries read
  const uint16_t* loc;  // [tile][chunk of 8 entries][thread][8]: LDS index per entry
  unsigned long long* slots;  // this launch's four publication slots
  unsigned long long* other;  // the other set, emptied here
  size_t slotStride;          // words per slot
  int* abort;
  const double* cheb;         // W_1 .. W_{iters-1}
  int iters;
};

template <class T, int BT, int TPR, int W, bool LM>
struct TileState {
  static constexpr int SUBS = 8 / TPR, E = SUBS * W, RW = kWave / TPR, NW = TileWords<T>::N;
  using V2 = typename TileWords<T>::V2;
  T v[E];
  unsigned li[E / 2];
  int rl, part, row;  // row < 0: this thread holds no row
  int nHalo;
  const int* halo;
  V2* xy;  // LDS: the staged iterate, (x, y) pairs and z values, own rows first, then the halo
  T* z;
  double* cheb;        // LDS: the sweeps' weights
  int hw[kPollBatch];  // word offset of the thread's first polled words (-1: none)

  __device__ __forceinline__ void init(const TileShape& a, const T* __restrict__ val, char* lds) {
    const int t = threadIdx.x, tile = blockIdx.x;
    xy = (V2*)lds;
    z = (T*)(lds + (size_t)a.uCap * sizeof(V2));
    cheb = (double*)(lds + (size_t)a.uCap * 3 * sizeof(T));
    for (int k = t; k < a.iters - 1; k += BT) cheb[k] = a.cheb[k];
    const int ln = t % kWave;
    rl = (t / kWave) * RW + ln % RW;
    part = ln / RW;
    const int4 ri = rl < a.R ? a.rows[(size_t)tile * a.R + rl] : make_int4(-1, 0, 0, 0);
    row = ri.x;
    halo = a.halo + a.haloOff[tile];
    nHalo = a.haloOff[tile + 1] - a.haloOff[tile];
    const uint4* lp = (const uint4*)a.loc + (size_t)tile * (E / 8) * BT + t;
#pragma unroll
    for (int c = 0; c < E / 8; c++) {
      const uint4 q = lp[(size_t)c * BT];
      li[4 * c] = q.x;
      li[4 * c + 1] = q.y;
      li[4 * c + 2] = q.z;
      li[4 * c + 3] = q.w;
    }
    if constexpr (LM) {  // lane-major, width 8: a lane's entries are one aligned run
      const T* p = val + ri.y + part * 8;
#pragma unroll
      for (int g = 0; g < SUBS; g++)
#pragma unroll
        for (int c = 0; c < 8; c += (int)(16 / sizeof(T))) {
          if constexpr (sizeof(T) == 4) {
            const float4 q = *(const float4*)(p + g * TPR * 8 + c);
            v[g * 8 + c] = q.x;
            v[g * 8 + c + 1] = q.y;
            v[g * 8 + c + 2] = q.z;
            v[g * 8 + c + 3] = q.w;
          } else {
            const double2 q = *(const double2*)(p + g * TPR * 8 + c);
            v[g * 8 + c] = q.x;
            v[g * 8 + c + 1] = q.y;
          }
        }
    } else {
      const T* p = val + ri.y + part;
#pragma unroll
      for (int g = 0; g < SUBS; g++)
#pragma unroll
        for (int c = 0; c < W; c++) v[g * W + c] = c < ri.z ? p[(int64_t)c * kWave + g * TPR] : T(0);
    }
    if (row < 0)
#pragma unroll
      for (int e = 0; e < E; e++) v[e] = T(0);
#pragma unroll
    for (int q = 0; q < kPollBatch; q++) {
      const int i = t + q * BT;
      hw[q] = i < nHalo * NW ? halo[i / NW] * NW + i % NW : -1;
    }
    // empty the other set's slots for the next launch
    if (row >= 0 && nHalo > 0)
      for (int w = part; w < NW; w += TPR)
#pragma unroll
        for (int s = 0; s < 4; s++) publish(a.other + s * a.slotStride + (size_t)row * NW + w, kTileEmpty);
  }

  // Keeps the compiler from unpacking the LDS indices once for all sweeps where
  // the unpacked ones would not fit the registers beside the entries.
  // (unpacked: an address for the pair and one for z per entry)
  static constexpr bool kLean = E * (2 + (int)sizeof(T) / 4) > 100;

  // M^2 times the staged iterate, at the thread's row (in all its parts)
  __device__ __forceinline__ void apply(T (&acc)[3]) {
    if constexpr (kLean)
#pragma unroll
      for (int e = 0; e < E / 2; e++) asm volatile("" : "+v"(li[e]));
    T s[3][SUBS];
#pragma unroll
    for (int g = 0; g < SUBS; g++) s[0][g] = s[1][g] = s[2][g] = T(0);
    // the lanes' sums advance together, one entry of each per step: their
    // additions are independent, and the steps' LDS reads overlap them
#pragma unroll
    for (int c = 0; c < W; c++) {
      V2 p[SUBS];
      T zz[SUBS];
#pragma unroll
      for (int g = 0; g < SUBS; g++) {
        const int e = g * W + c;
        const unsigned l = (e & 1) ? li[e / 2] >> 16 : li[e / 2] & 0xffffu;
        p[g] = xy[l];
        zz[g] = z[l];
      }
#pragma unroll
      for (int g = 0; g < SUBS; g++) {
        const int e = g * W + c;
        s[0][g] += v[e] * p[g].x;
        s[1][g] += v[e] * p[g].y;
        s[2][g] += v[e] * zz[g];
      }
    }
#pragma unroll
    for (int k = 0; k < 3; k++) acc[k] = lane_tree<TPR, T>(s[k]);
  }

  // publication j of the row
  __device__ __forceinline__ void send(const TileShape& a, int j, const T (&d)[3]) const {
    if (row < 0 || nHalo == 0) return;  // without a halo nobody reads this tile's rows
    unsigned long long* s = a.slots + (size_t)row * NW;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the words emptied a sweep ago have reached memory
    for (int w = part; w < NW; w += TPR) publish(s + (size_t)(j & 3) * a.slotStride + w, TileWords<T>::word(d, w));
    if (j >= 2)
      for (int w = part; w < NW; w += TPR) publish(s + (size_t)((j + 2) & 3) * a.slotStride + w, kTileEmpty);
  }
  __device__ __forceinline__ void stage_own(T x, T y, T w) const {
    if (row < 0 || part != 0) return;
    xy[rl] = V2{x, y};
    z[rl] = w;
  }
  // polls the words at off[] (-1: none) until all have arrived, then stages them
  __device__ __forceinline__ bool poll(const TileShape& a, const unsigned long long* s, const int (&off)[kPollBatch],
                                       int i0, unsigned long long t0) const {
    unsigned long long w[kPollBatch];
    for (int spin = 1;; spin++) {
      bool ready = true;
#pragma unroll
      for (int q = 0; q < kPollBatch; q++) w[q] = off[q] >= 0 ? peek(s + off[q]) : 0ull;
#pragma unroll
      for (int q = 0; q < kPollBatch; q++) ready = ready && w[q] != kTileEmpty;
      if (ready) break;
      if ((spin & 63) == 0 && (wall_clock64() - t0 > kTileWaitTicks ||
                               __hip_atomic_load(a.abort, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)))
        return false;
    }
#pragma unroll
    for (int q = 0; q < kPollBatch; q++) {
      const int i = i0 + q * BT;
      if (off[q] >= 0) TileWords<T>::unpack(w[q], i % NW, xy, z, a.R + i / NW);
    }
    return true;
  }
  // stages publication j of the neighbours' rows; false: gave up waiting
  __device__ __forceinline__ bool receive(const TileShape& a, int j, unsigned long long t0) const {
    const int items = nHalo * NW;
    if (items == 0) return true;
    const unsigned long long* s = a.slots + (size_t)(j & 3) * a.slotStride;
    // the neighbours finish at about the same time and a store takes about 0.4 us
    // to arrive: polling at once only delays it (256^2 cloth, per sweep: 2.7 us
    // without this pause, 2.3 us with it)
    __builtin_amdgcn_s_sleep(6);
    bool ok = poll(a, s, hw, threadIdx.x, t0);
    for (int i0 = threadIdx.x + kPollBatch * BT; i0 < items; i0 += kPollBatch * BT) {
      int off[kPollBatch];
#pragma unroll
      for (int q = 0; q < kPollBatch; q++) {
        const int i = i0 + q * BT;
        off[q] = i < items ? halo[i / NW] * NW + i % NW : -1;
      }
      ok = poll(a, s, off, i0, t0) && ok;
    }
    return ok;
  }
  // ends sweep j: the row's new iterate to the neighbours and into LDS, theirs
  // into LDS; false (for the whole workgroup): some wait was given up
  __device__ __forceinline__ bool exchange(const TileShape& a, int j, const T (&d)[3], int* flag,
                                           unsigned long long t0) const {
    send(a, j, d);
    __syncthreads();  // every row of the tile has read the old iterate
    stage_own(d[0], d[1], d[2]);
    if (!receive(a, j, t0)) {
      *flag = 1;
      __hip_atomic_store(a.abort, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    return *flag == 0;
  }
};

// LDS: uCap staged rows, (x, y) pairs then z values, then the sweeps' weights
// (uCap is a multiple of 8, so the weights are aligned)
template <class T>
constexpr size_t tile_lds_bytes(int uCap, int iters) {
  return (size_t)uCap * 3 * sizeof(T) + (size_t)iters * sizeof(double);
}

// leaves the kernel at its start when an earlier launch gave up (the same
// answer for the whole workgroup)
__device__ __forceinline__ bool tile_aborted(const int* abort, int* flag) {
  if (threadIdx.x == 0) *flag = __hip_atomic_load(abort, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  return *flag != 0;
}

// FP32-split: delta_1 = r0 (global, from the residual pass), then
// delta_{k+1} = W_k (M^2 delta_k + r0 - delta_{k-1}) + delta_{k-1}; X += the last.
template <int BT, int TPR, int W, bool LM>
__global__ void __launch_bounds__(BT) k_tile_solve32(TileShape a, const float* __restrict__ val,
                                                     const float4* __restrict__ r0, double* __restrict__ X) {
  extern __shared__ __attribute__((aligned(16))) char tileLds[];
  __shared__ int flag;
  if (tile_aborted(a.abort, &flag)) return;
  TileState<float, BT, TPR, W, LM> st;
  st.init(a, val, tileLds);
  for (int u = threadIdx.x; u < st.nHalo; u += BT) {
    const float4 q = r0[st.halo[u]];
    st.xy[a.R + u] = make_float2(q.x, q.y);
    st.z[a.R + u] = q.z;
  }
  float r[3] = {0.f, 0.f, 0.f}, pre[3] = {0.f, 0.f, 0.f}, cur[3] = {0.f, 0.f, 0.f};
  if (st.row >= 0) {
    const float4 q = r0[st.row];
    r[0] = cur[0] = q.x;
    r[1] = cur[1] = q.y;
    r[2] = cur[2] = q.z;
    st.stage_own(q.x, q.y, q.z);
  }
  __syncthreads();
  const unsigned long long t0 = wall_clock64();
  for (int it = 1; it < a.iters; it++) {
    const float Wc = (float)st.cheb[it - 1];
    float acc[3];
    st.apply(acc);
    float d[3];
#pragma unroll
    for (int k = 0; k < 3; k++) {
      d[k] = Wc * (acc[k] + r[k] - pre[k]) + pre[k];
      pre[k] = cur[k];
      cur[k] = d[k];
    }
    if (it < a.iters - 1 && !st.exchange(a, it - 1, d, &flag, t0)) return;
  }
  if (st.row >= 0 && st.part == 0)
#pragma unroll
    for (int k = 0; k < 3; k++) X[k * a.ld + st.row] += (double)cur[k];
}

// FP64: x_0 = X, c computed here from R1, D and b (as k_first64), x_1 = M^2 x_0 + c,
// x_{k+1} = W_k (M^2 x_k + c - x_{k-1}) + x_{k-1}; the last to X.  With `out`
// every iterate x_k also goes to out + (k - 1) outStride (SoA).
struct TileFirst {
  const int* off;
  const int* col;
  const double* val;
  const double* D;
  const double* b;
  double w;
};
template <int BT, int TPR, int W, bool LM>
__global__ void __launch_bounds__(BT) k_tile_solve64(TileShape a, const double* __restrict__ val, TileFirst ft,
                                                     double* X, double* __restrict__ out, int64_t outStride) {
  extern __shared__ __attribute__((aligned(16))) char tileLds[];
  __shared__ int flag;
  if (tile_aborted(a.abort, &flag)) return;
  using State = TileState<double, BT, TPR, W, LM>;
  constexpr int SUBS = State::SUBS;
  State st;
  st.init(a, val, tileLds);
  for (int u = threadIdx.x; u < st.nHalo; u += BT) {
    const int h = st.halo[u];
    st.xy[a.R + u] = make_double2(X[h], X[a.ld + h]);
    st.z[a.R + u] = X[2 * a.ld + h];
  }
  double pre[3] = {0.0, 0.0, 0.0}, cur[3] = {0.0, 0.0, 0.0}, c[3] = {0.0, 0.0, 0.0};
  {
    const int rr = st.row >= 0 ? st.row : 0;
    const int q0 = ft.off[rr], q1 = st.row >= 0 ? ft.off[rr + 1] : q0;
    double di = ft.D[rr], bi[3];
#pragma unroll
    for (int k = 0; k < 3; k++) {
      bi[k] = ft.b[k * a.ld + rr];
      cur[k] = X[k * a.ld + rr];
    }
    st.stage_own(cur[0], cur[1], cur[2]);
    // lane s of the row sums the R1 entries s, s + 8, ...
    double s[3][SUBS];
#pragma unroll
    for (int g = 0; g < SUBS; g++) s[0][g] = s[1][g] = s[2][g] = 0.0;
    for (int q = q0; q < q1; q += 8) {
      int jj[SUBS];
      double f[SUBS];
#pragma unroll
      for (int g = 0; g < SUBS; g++) {
        const int e = q + st.part + TPR * g;
        jj[g] = e < q1 ? ft.col[e] : rr;
        f[g] = e < q1 ? ft.val[e] : 0.0;
      }
#pragma unroll
      for (int g = 0; g < SUBS; g++) {
        const bool in = q + st.part + TPR * g < q1;
        f[g] = f[g] / ft.D[jj[g]];
#pragma unroll
        for (int k = 0; k < 3; k++) {
          const double bj = ft.b[k * a.ld + jj[g]];
          if (in) s[k][g] += f[g] * bj;
        }
      }
    }
#pragma unroll
    for (int k = 0; k < 3; k++) {
      c[k] = first_term(ft.w, lane_tree<TPR, double>(s[k]), bi[k], di);
    }
  }
  __syncthreads();
  const unsigned long long t0 = wall_clock64();
  for (int it = 0; it < a.iters; it++) {
    const double Wc = it > 0 ? st.cheb[it - 1] : 0.0;
    double acc[3], d[3];
    st.apply(acc);
    if (it == 0) {
#pragma unroll
      for (int k = 0; k < 3; k++) d[k] = acc[k] + c[k];
    } else {
#pragma unroll
      for (int k = 0; k < 3; k++) d[k] = Wc * (acc[k] + c[k] - pre[k]) + pre[k];
    }
#pragma unroll
    for (int k = 0; k < 3; k++) {
      pre[k] = cur[k];
      cur[k] = d[k];
    }
    if (it < a.iters - 1 && !st.exchange(a, it, d, &flag, t0)) return;
    if (out && st.row >= 0 && st.part == 0)
#pragma unroll
      for (int k = 0; k < 3; k++) out[it * outStride + k * a.ld + st.row] = d[k];
  }
  if (st.row >= 0 && st.part == 0)
#pragma unroll
    for (int k = 0; k < 3; k++) X[k * a.ld + st.row] = cur[k];
}

__global__ void k_tile_reset(size_t n, unsigned long long* __restrict__ slots) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) slots[i] = kTileEmpty;
}

using Solve32 = void (*)(TileShape, const float*, const float4*, double*);
using Solve64 = void (*)(TileShape, const double*, TileFirst, double*, double*, int64_t);

// The kernel of a tiling's shape (null: none).  FP64 rows of width 12 and more at one
// thread per row would need more registers than a thread has.
Solve32 solve32_kernel(const TileConfig& c) {
#define PICK(BT, TPR)                                            \
  if (c.threads == BT && c.tpr == TPR) {                         \
    if (c.laneMajor) return k_tile_solve32<BT, TPR, 8, true>;    \
    if (c.width == 8) return k_tile_solve32<BT, TPR, 8, false>;  \
    if (c.width == 12) return k_tile_solve32<BT, TPR, 12, false>; \
  }
  PICK(256, 4)
  PICK(512, 4)
  PICK(512, 2)
  PICK(512, 1)
#undef PICK
  return nullptr;
}
Solve64 solve64_kernel(const TileConfig& c) {
#define PICK(BT, TPR)                                            \
  if (c.threads == BT && c.tpr == TPR) {                         \
    if (c.laneMajor) return k_tile_solve64<BT, TPR, 8, true>;    \
    if (c.width == 8) return k_tile_solve64<BT, TPR, 8, false>;  \
    if (c.width == 12 && TPR > 1) return k_tile_solve64<BT, TPR, (TPR > 1 ? 12 : 8), false>; \
  }
  PICK(256, 4)
  PICK(512, 4)
  PICK(512, 2)
  PICK(512, 1)
#undef PICK
  return nullptr;
}

TileShape shape_of(const DeviceMesh& m, int parity, int words, int iters) {
  TileShape a;
  a.n = m.nSim;
  a.ld = m.ld;
  a.R = m.tile.rowsPerTile;
  a.uCap = m.tile.uCap;
  a.rows = m.tile.rows;
  a.haloOff = m.tile.haloOff;
  a.halo = m.tile.halo;
  a.loc = m.tile.loc;
  a.slotStride = (size_t)m.ld * words;
  const size_t set = 4 * (size_t)m.ld * 3;  // words per set, sized for FP64
  a.slots = m.tile.slots + (parity ? set : 0);
  a.other = m.tile.slots + (parity ? 0 : set);
  a.abort = m.tile.abort;
  a.cheb = m.tile.cheb;
  a.iters = iters;
  return a;
}

template <class K>
bool fits(K kernel, int threads, size_t lds, int tiles, int cus) {
  if (!kernel) return false;
  if (lds > (64 << 10) &&
      hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  int occ = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, kernel, threads, lds) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  return occ >= 1 && tiles <= cus;
}

}  // namespace

void tile_check(DeviceMesh& m, int cus, int iters) {
  TileConfig& c = m.tile.cfg;
  m.tile.ok32 = fits(solve32_kernel(c), c.threads, tile_lds_bytes<float>(m.tile.uCap, iters), m.tile.nTiles, cus);
  m.tile.ok64 = fits(solve64_kernel(c), c.threads, tile_lds_bytes<double>(m.tile.uCap, iters), m.tile.nTiles, cus);
}

void launch_tile_reset(const DeviceMesh& m, hipStream_t s) {
  const size_t n = 4 * (size_t)m.ld * 3;
  hipLaunchKernelGGL(k_tile_reset, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, n, m.tile.slots);
}

void launch_tile_solve32(const DeviceMesh& m, int iters, int parity, hipStream_t s) {
  launch_t(m.timer, TC_SWEEP32, solve32_kernel(m.tile.cfg), dim3(m.tile.nTiles), dim3(m.tile.cfg.threads),
           (uint32_t)tile_lds_bytes<float>(m.tile.uCap, iters), s, shape_of(m, parity, 2, iters), (const float*)m.m2ValF,
           (const float4*)m.r0, m.X);
  if (m.timer) m.timer->weigh(iters - 1);
}

void launch_tile_solve64(const DeviceMesh& m, double w, int iters, int parity, double* out, int64_t outStride,
                         hipStream_t s) {
  const TileFirst ft{m.r1Off, m.r1Col, m.r1Val, m.sysDiag, m.sysRhs, w};
  launch_t(m.timer, TC_SWEEP64, solve64_kernel(m.tile.cfg), dim3(m.tile.nTiles), dim3(m.tile.cfg.threads),
           (uint32_t)tile_lds_bytes<double>(m.tile.uCap, iters), s, shape_of(m, parity, 3, iters), (const double*)m.m2Val, ft,
           m.X, out, outStride);
  if (m.timer) m.timer->weigh(iters - 1);
}

}  // namespace pdipc
