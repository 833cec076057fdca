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
// cloth (256 tiles of 256 rows), loads and launch included: 2.8 us (FP32) and
// 5.1 (FP64) against 4.7 and 8.6 for the streamed kernels.
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
// is no longer kTileEmpty, a NaN no iterate can hold.  Only rows that other
// tiles read are published (512^2 cloth, all rows: 8.6 us per sweep, 6.5 with
// the 44 % that are read).  The data are their own flag: no fence and no
// barrier between workgroups.  Publication j of a launch goes to slot j % 4.
// After publishing j a thread empties its words of
// publication j - 2: it has staged publication j - 1 of all neighbours, who had
// staged j - 2 before publishing it (the neighbour relation is symmetric).  It
// waits for that store before it publishes j + 1 (a whole sweep later, so the
// wait is over when it begins); a reader reaches publication j + 2, the same
// slot as j - 2, only after it has staged this thread's publication j + 1, and
// so finds the emptied word or the new value.  The last two publications of a
// launch stay; launches alternate between two sets of slots, each emptying the
// other set.
//
// Every wait is bounded (kTileWaitRounds of polling): a tile whose
// neighbours do not arrive -- other kernels hold compute units for long --
// raises the abort flag, every tile leaves, and the host, which restores X,
// repeats the outer iteration with the streamed kernels.
#include <algorithm>

#include "device.hpp"
#include "local_ops.hpp"

namespace pdipc {
namespace {

constexpr unsigned long long kTileEmpty = 0xfff5a5a5fff5a5a5ull;
// polling rounds per wait: about 10 ms (2^14 rounds of a 40^2 to 300^2 cloth's
// solve took 3.8); counted, so that a wait takes no registers for the clock
constexpr int kTileWaitRounds = 44 << 10;
constexpr int kRowWords = 3;   // words per row in a publication slot (FP32 vectors use two)

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
  const int4* rows;     // [tile][R]: row (-1 past the last), its first SELL entry, entries per lane, read by other tiles
  const int* haloOff;   // [tile + 1]
  const int* halo;      // rows of other tiles that the tile's entries read
  const uint16_t* loc;  // [tile][chunk of 8 entries][thread][8]: LDS index per entry
  unsigned long long* slots;  // this launch's four publication slots
  unsigned long long* other;  // the other set, emptied here
  size_t slotStride;          // words per slot
  int* abort;                 // and, two words on, where tile 0 gives up (tests): a publication + 1
  const double* cheb;         // W_1 .. W_{iters-1}
  int iters;
};

// PB: words per thread polled together; LEAN: keep the LDS indices packed
template <class T, int BT, int TPR, int W, bool LM, int PB, bool LEAN>
struct TileState {
  static constexpr int SUBS = 8 / TPR, E = SUBS * W, RW = kWave / TPR, NW = TileWords<T>::N;
  using V2 = typename TileWords<T>::V2;
  using Words = TileWords<T>;
  T v[E];
  unsigned li[E / 2];
  int rl, part, row;  // row < 0: this thread holds no row
  bool pub;           // other tiles read the row
  int nHalo;
  const int* halo;
  V2* xy;  // LDS: the staged iterate, (x, y) pairs and z values, own rows first, then the halo
  T* z;
  double* cheb;        // LDS: the sweeps' weights
  int hw[PB];  // word offset of the thread's first polled words (-1: none)
  int stop;    // this tile gives up at that publication (-1: none)

  // a row's LDS indices (tables of `threads` threads per tile, here thread t's)
  static __device__ __forceinline__ void load_loc(const TileShape& a, int threads, int t, unsigned (&li)[E / 2]) {
    const uint4* lp = (const uint4*)a.loc + (size_t)blockIdx.x * (E / 8) * threads + t;
#pragma unroll
    for (int c = 0; c < E / 8; c++) {
      const uint4 q = lp[(size_t)c * threads];
      li[4 * c] = q.x;
      li[4 * c + 1] = q.y;
      li[4 * c + 2] = q.z;
      li[4 * c + 3] = q.w;
    }
  }
  // the entries of a row in lanes part, part + TPR, ... (threads without a row: some row's)
  static __device__ __forceinline__ void load_val(const int4& ri, int part, const T* __restrict__ val, T (&v)[E]) {
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
  }
  // LDS pointers, weights, halo and the first polled words
  __device__ __forceinline__ void setup(const TileShape& a, char* lds, int stopAt) {
    stop = __builtin_amdgcn_readfirstlane(stopAt);
    const int t = threadIdx.x, tile = blockIdx.x;
    xy = (V2*)lds;
    z = (T*)(lds + (size_t)a.uCap * sizeof(V2));
    cheb = (double*)(lds + (size_t)a.uCap * 3 * sizeof(T));
    for (int k = t; k < a.iters - 1; k += BT) cheb[k] = a.cheb[k];
    halo = a.halo + a.haloOff[tile];
    nHalo = a.haloOff[tile + 1] - a.haloOff[tile];
#pragma unroll
    for (int q = 0; q < PB; q++) {
      const int i = t + q * BT;
      hw[q] = i < nHalo * NW ? halo[i / NW] * kRowWords + i % NW : -1;
    }
  }
  // empties the other set's words of a published row, for the next launch
  __device__ __forceinline__ void empty_other(const TileShape& a, int r) const {
    for (int w = part; w < NW; w += TPR)
#pragma unroll
      for (int s = 0; s < 4; s++) publish(a.other + s * a.slotStride + (size_t)r * kRowWords + w, kTileEmpty);
  }

  __device__ __forceinline__ void load(const TileShape& a, const int4& ri, const T* __restrict__ val) {
    load_loc(a, BT, threadIdx.x, li);
    load_val(ri, part, val, v);
  }
  template <bool EMPTY_OTHER, bool LOAD = true>
  __device__ __forceinline__ int4 init(const TileShape& a, const T* __restrict__ val, char* lds, int stopAt) {
    setup(a, lds, stopAt);
    const int t = threadIdx.x, ln = t % kWave;
    rl = (t / kWave) * RW + ln % RW;
    part = ln / RW;
    const int4 ri = rl < a.R ? a.rows[(size_t)blockIdx.x * a.R + rl] : make_int4(-1, 0, 0, 0);
    row = ri.x;
    pub = ri.w != 0;
    if constexpr (LOAD) load(a, ri, val);
    if (EMPTY_OTHER && pub) empty_other(a, row);
    return ri;
  }

  // M^2 times the staged iterate at one row, lanes G0, G0 + STEP, ... of the
  // thread's: the lanes' sums advance together, one entry of each per step, so
  // their additions are independent and the steps' LDS reads overlap them
  template <int G0, int STEP, int N>
  __device__ __forceinline__ void lanes(const T (&v)[E], const unsigned (&li)[E / 2], T (&s)[3][N]) const {
#pragma unroll
    for (int g = 0; g < N; g++) s[0][g] = s[1][g] = s[2][g] = T(0);
#pragma unroll
    for (int c = 0; c < W; c++) {
      V2 p[N];
      T zz[N];
#pragma unroll
      for (int g = 0; g < N; g++) {
        const int e = (G0 + g * STEP) * W + c;
        const unsigned l = (e & 1) ? li[e / 2] >> 16 : li[e / 2] & 0xffffu;
        p[g] = xy[l];
        zz[g] = z[l];
      }
#pragma unroll
      for (int g = 0; g < N; g++) {
        const int e = (G0 + g * STEP) * W + c;
        s[0][g] += v[e] * p[g].x;
        s[1][g] += v[e] * p[g].y;
        s[2][g] += v[e] * zz[g];
      }
      if constexpr (STEP > 1) __builtin_amdgcn_sched_barrier(0);
    }
  }
  // the thread's row (in all its parts)
  __device__ __forceinline__ void apply(T (&acc)[3]) {
    if constexpr (LEAN)  // (opaque per sweep: the compiler would unpack them once for all sweeps)
#pragma unroll
      for (int e = 0; e < E / 2; e++) asm volatile("" : "+v"(li[e]));
    if constexpr (TPR == 1 && LEAN) {
      apply_halves(v, li, acc);
    } else {
      T s[3][SUBS];
      lanes<0, 1, SUBS>(v, li, s);
#pragma unroll
      for (int k = 0; k < 3; k++) acc[k] = lane_tree<TPR, T>(s[k]);
    }
  }
  // one thread per row with few registers left: the even lanes, then the odd
  // ones (the two sides of the lane tree's last addition)
  __device__ __forceinline__ void apply_halves(const T (&v)[E], const unsigned (&li)[E / 2], T (&acc)[3]) const {
    T s[3][4], even[3];
    lanes<0, 2, 4>(v, li, s);
#pragma unroll
    for (int k = 0; k < 3; k++) even[k] = (s[k][0] + s[k][2]) + (s[k][1] + s[k][3]);
    lanes<1, 2, 4>(v, li, s);
#pragma unroll
    for (int k = 0; k < 3; k++) acc[k] = even[k] + ((s[k][0] + s[k][2]) + (s[k][1] + s[k][3]));
  }

  // publication j of the row (values of type U), emptying `old` words of
  // publication j - 2
  template <class U>
  __device__ __forceinline__ void send(const TileShape& a, int j, const U (&d)[3], int old) const {
    if (!pub) return;
    unsigned long long* s = a.slots + (size_t)row * kRowWords;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the words emptied a sweep ago have reached memory
    for (int w = part; w < TileWords<U>::N; w += TPR)
      publish(s + (size_t)(j & 3) * a.slotStride + w, TileWords<U>::word(d, w));
    if (j >= 2)
      for (int w = part; w < old; w += TPR) publish(s + (size_t)((j + 2) & 3) * a.slotStride + w, kTileEmpty);
  }
  template <class U, class U2>
  __device__ __forceinline__ void stage_own(U2* pxy, U* pz, U x, U y, U w) const {
    if (row < 0 || part != 0) return;
    pxy[rl] = U2{x, y};
    pz[rl] = w;
  }
  // polls the words at off[] (-1: none) until all have arrived, then stages them
  template <class U, class U2>
  __device__ __forceinline__ bool poll(const TileShape& a, const unsigned long long* s, const int (&off)[PB],
                                       int i0, U2* pxy, U* pz) const {
    constexpr int N = TileWords<U>::N;
    unsigned long long w[PB];
    for (int spin = 1;; spin++) {
      bool ready = true;
#pragma unroll
      for (int q = 0; q < PB; q++) w[q] = off[q] >= 0 ? peek(s + off[q]) : 0ull;
#pragma unroll
      for (int q = 0; q < PB; q++) ready = ready && w[q] != kTileEmpty;
      if (ready) break;
      if ((spin & 63) == 0 && (spin >= kTileWaitRounds ||
                               __hip_atomic_load(a.abort, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)))
        return false;
    }
#pragma unroll
    for (int q = 0; q < PB; q++) {
      const int i = i0 + q * BT;
      if (off[q] >= 0) TileWords<U>::unpack(w[q], i % N, pxy, pz, a.R + i / N);
    }
    return true;
  }
  // stages publication j of the neighbours' rows; false: gave up waiting
  template <class U, class U2>
  __device__ __forceinline__ bool receive(const TileShape& a, int j, U2* pxy, U* pz) const {
    constexpr int N = TileWords<U>::N;
    const int items = nHalo * N;
    if (items == 0) return true;
    const unsigned long long* s = a.slots + (size_t)(j & 3) * a.slotStride;
    // the neighbours finish at about the same time and a store takes about 0.4 us
    // to arrive: polling at once only delays it (256^2 cloth, per sweep: 2.7 us
    // without this pause, 2.3 us with it)
    __builtin_amdgcn_s_sleep(6);
    bool ok = true;
    int i0 = threadIdx.x;
    if constexpr (N == NW) {  // the words of the solve's own type are listed at the start
      ok = poll(a, s, hw, i0, pxy, pz);
      i0 += PB * BT;
    }
    for (; i0 < items; i0 += PB * BT) {
      int off[PB];
#pragma unroll
      for (int q = 0; q < PB; q++) {
        const int i = i0 + q * BT;
        off[q] = i < items ? halo[i / N] * kRowWords + i % N : -1;
      }
      ok = poll(a, s, off, i0, pxy, pz) && ok;
    }
    return ok;
  }
  // publication j: the row's new vector to the neighbours and into LDS, theirs
  // into LDS; false (for the whole workgroup): some wait was given up
  template <class U, class U2>
  __device__ __forceinline__ bool exchange(const TileShape& a, int j, const U (&d)[3], int old, int* flag,
                                           U2* pxy, U* pz) const {
    send(a, j, d, old);
    __syncthreads();  // every row of the tile has read the old vector
    stage_own(pxy, pz, d[0], d[1], d[2]);
    if (!receive(a, j, pxy, pz) || j == stop) {
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

// The unpacked LDS indices (an address for the pair and one for z per entry)
// are kept where they fit the registers beside the entries.
template <class T, int TPR, int W>
constexpr bool tile_lean() { return 8 / TPR * W * (2 + (int)sizeof(T) / 4) > 100; }

// leaves the kernel at its start when an earlier launch gave up (the same
// answer for the whole workgroup); stop: the publication at which this tile does
__device__ __forceinline__ bool tile_aborted(const int* abort, int* flag, int* stop) {
  if (threadIdx.x == 0) {
    const int f = __hip_atomic_load(abort, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    *stop = (blockIdx.x == 0 ? __hip_atomic_load(abort + 2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0) - 1;
    *flag = f;
  }
  __syncthreads();
  return *flag != 0;
}

// FP32-split: delta_1 = r0 (global, from the residual pass), then
// delta_{k+1} = W_k (M^2 delta_k + r0 - delta_{k-1}) + delta_{k-1}; X += the last.
template <int BT, int TPR, int W, bool LM>
__global__ void __launch_bounds__(BT) k_tile_solve32(TileShape a, const float* __restrict__ val,
                                                     const float4* __restrict__ r0, double* __restrict__ X) {
  extern __shared__ __attribute__((aligned(16))) char tileLds[];
  __shared__ int flag, stop;
  if (tile_aborted(a.abort, &flag, &stop)) return;
  TileState<float, BT, TPR, W, LM, 6, tile_lean<float, TPR, W>()> st;
  st.template init<true>(a, val, tileLds, stop);
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
    st.stage_own(st.xy, st.z, q.x, q.y, q.z);
  }
  __syncthreads();
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
    if (it < a.iters - 1 && !st.exchange(a, it - 1, d, 2, &flag, st.xy, st.z)) return;
  }
  if (st.row >= 0 && st.part == 0)
#pragma unroll
    for (int k = 0; k < 3; k++) X[k * a.ld + st.row] += (double)cur[k];
}

// The same with two rows per thread (t and t + BT of tables laid out for 2 BT
// threads), for tiles of 513 to 1024 rows of width 8: entries and LDS indices
// take 192 of a thread's 256 registers, so r0 and delta_{k-1} are kept in LDS
// and a row's lanes advance in two halves (even lanes, then odd ones: the two
// sides of the lane tree's last addition).  512^2 cloth: 117 us per solve (24
// to load 100 MB of entries and indices, then 6.5 per sweep: 3.4 LDS reads and
// FMAs, 3.1 exchange) against 270 us streamed (18 per sweep at 5.6 TB/s).
constexpr int kTwoThreads = 512;
constexpr size_t tile_two_lds_bytes(int uCap, int iters) {
  return tile_lds_bytes<float>(uCap, iters) + 2 * (size_t)(2 * kTwoThreads) * 3 * sizeof(float);
}
template <bool LM>
__global__ void __launch_bounds__(kTwoThreads) k_tile_solve32_two(TileShape a, const float* __restrict__ val,
                                                                  const float4* __restrict__ r0,
                                                                  double* __restrict__ X) {
  constexpr int BT = kTwoThreads;
  using St = TileState<float, BT, 1, 8, LM, 4, true>;
  extern __shared__ __attribute__((aligned(16))) char tileLds[];
  __shared__ int flag, stop;
  if (tile_aborted(a.abort, &flag, &stop)) return;
  St st;
  st.setup(a, tileLds, stop);
  st.part = 0;
  float* rs = (float*)(tileLds + tile_lds_bytes<float>(a.uCap, a.iters));  // r0, then delta_{k-1}, of the own rows
  float* ps = rs + 3 * 2 * BT;
  float v[2][St::E];
  unsigned li[2][St::E / 2];
  int row[2], rl[2];
  bool pub[2];
#pragma unroll
  for (int q = 0; q < 2; q++) {
    rl[q] = threadIdx.x + q * BT;
    const int4 ri = rl[q] < a.R ? a.rows[(size_t)blockIdx.x * a.R + rl[q]] : make_int4(-1, 0, 0, 0);
    row[q] = ri.x;
    St::load_loc(a, 2 * BT, rl[q], li[q]);
    St::load_val(ri, 0, val, v[q]);
    pub[q] = ri.w != 0;
    if (pub[q]) st.empty_other(a, row[q]);
    const float4 r = row[q] >= 0 ? r0[row[q]] : make_float4(0.f, 0.f, 0.f, 0.f);
    if (row[q] >= 0) {
      st.xy[rl[q]] = make_float2(r.x, r.y);
      st.z[rl[q]] = r.z;
    }
    rs[3 * rl[q]] = r.x;
    rs[3 * rl[q] + 1] = r.y;
    rs[3 * rl[q] + 2] = r.z;
    ps[3 * rl[q]] = ps[3 * rl[q] + 1] = ps[3 * rl[q] + 2] = 0.f;
  }
  for (int u = threadIdx.x; u < st.nHalo; u += BT) {
    const float4 q = r0[st.halo[u]];
    st.xy[a.R + u] = make_float2(q.x, q.y);
    st.z[a.R + u] = q.z;
  }
  __syncthreads();
  for (int it = 1; it < a.iters; it++) {
    const float Wc = (float)st.cheb[it - 1];
    float d[2][3];
#pragma unroll
    for (int q = 0; q < 2; q++) {
#pragma unroll
      for (int e = 0; e < St::E / 2; e++) asm volatile("" : "+v"(li[q][e]));  // (not unpacked for all sweeps)
      float acc[3];
      st.apply_halves(v[q], li[q], acc);
#pragma unroll
      for (int k = 0; k < 3; k++) {
        const float pre = ps[3 * rl[q] + k];
        d[q][k] = Wc * (acc[k] + rs[3 * rl[q] + k] - pre) + pre;
      }
    }
    if (it == a.iters - 1) {
#pragma unroll
      for (int q = 0; q < 2; q++)
        if (row[q] >= 0)
#pragma unroll
          for (int k = 0; k < 3; k++) X[k * a.ld + row[q]] += (double)d[q][k];
      return;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the words emptied a sweep ago have reached memory
    const int j = it - 1;
    const size_t now = (size_t)(j & 3) * a.slotStride, old = (size_t)((j + 2) & 3) * a.slotStride;
#pragma unroll
    for (int q = 0; q < 2; q++)
      if (pub[q])
#pragma unroll
        for (int w = 0; w < 2; w++)
          publish(a.slots + now + (size_t)row[q] * kRowWords + w, TileWords<float>::word(d[q], w));
    if (j >= 2)
#pragma unroll
      for (int q = 0; q < 2; q++)
        if (pub[q])
#pragma unroll
          for (int w = 0; w < 2; w++) publish(a.slots + old + (size_t)row[q] * kRowWords + w, kTileEmpty);
    __syncthreads();  // every row of the tile has read the old iterate
#pragma unroll
    for (int q = 0; q < 2; q++)
      if (row[q] >= 0) {
        const int r = rl[q];
        const float2 c = st.xy[r];
        ps[3 * r] = c.x;
        ps[3 * r + 1] = c.y;
        ps[3 * r + 2] = st.z[r];
        st.xy[r] = make_float2(d[q][0], d[q][1]);
        st.z[r] = d[q][2];
      }
    if (!st.receive(a, j, st.xy, st.z) || j == st.stop) {
      flag = 1;
      __hip_atomic_store(a.abort, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    if (flag != 0) return;
  }
  // one sweep only: delta_1 = r0
#pragma unroll
  for (int q = 0; q < 2; q++)
    if (row[q] >= 0)
#pragma unroll
      for (int k = 0; k < 3; k++) X[k * a.ld + row[q]] += (double)rs[3 * rl[q] + k];
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
  __shared__ int flag, stop;
  if (tile_aborted(a.abort, &flag, &stop)) return;
  using State = TileState<double, BT, TPR, W, LM, 6, tile_lean<double, TPR, W>()>;
  constexpr int SUBS = State::SUBS;
  State st;
  // (one thread per row: the entries' registers are not free before c is formed)
  const int4 ri = st.template init<true, (TPR > 1)>(a, val, tileLds, stop);
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
    st.stage_own(st.xy, st.z, cur[0], cur[1], cur[2]);
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
  if constexpr (TPR == 1) st.load(a, ri, val);
  __syncthreads();
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
    // (a single sweep's iterate is exchanged too: a tile writes its rows of X only
    // when its neighbours have staged their halos from it)
    if ((it == 0 || it < a.iters - 1) && !st.exchange(a, it, d, 3, &flag, st.xy, st.z)) return;
    if (out && st.row >= 0 && st.part == 0)
#pragma unroll
      for (int k = 0; k < 3; k++) out[it * outStride + k * a.ld + st.row] = d[k];
  }
  if (st.row >= 0 && st.part == 0)
#pragma unroll
    for (int k = 0; k < 3; k++) X[k * a.ld + st.row] = cur[k];
}

// The reverse sweeps of one pass (the adjoint's recurrence on u = D^{-1} xbar,
// k_solve.hip): from u_K, u_k = W_k M^2 u_{k+1} + b_k u_{k+2} for k = K - 1 .. 0
// with b_k = 1 - W_{k+1} (none at K - 1), every u_k stored and
// uc += W_k u_{k+1}.  128^2 cloth, 15 sweeps: 37.5 us, about 80 as
// streamed sweeps with their boundaries (4.6 each).
template <int BT, int TPR, int W, bool LM>
__global__ void __launch_bounds__(BT) k_tile_adj(TileShape a, const double* __restrict__ val, TileAdj g) {
  extern __shared__ __attribute__((aligned(16))) char tileLds[];
  __shared__ int flag, stop;
  if (tile_aborted(a.abort, &flag, &stop)) return;
  TileState<double, BT, TPR, W, LM, 6, tile_lean<double, TPR, W>()> st;
  st.template init<true>(a, val, tileLds, stop);
  const double* u0 = g.u[g.K];
  for (int q = threadIdx.x; q < st.nHalo; q += BT) {
    const int h = st.halo[q];
    st.xy[a.R + q] = make_double2(u0[h], u0[a.ld + h]);
    st.z[a.R + q] = u0[2 * a.ld + h];
  }
  double oth[3] = {0.0, 0.0, 0.0}, cur[3] = {0.0, 0.0, 0.0}, uc[3] = {0.0, 0.0, 0.0};
  if (st.row >= 0) {
#pragma unroll
    for (int k = 0; k < 3; k++) {
      cur[k] = u0[k * a.ld + st.row];
      uc[k] = g.uc[k * a.ld + st.row];
    }
    st.stage_own(st.xy, st.z, cur[0], cur[1], cur[2]);
  }
  __syncthreads();
  for (int k = g.K - 1; k >= 0; k--) {
    const double w = g.w[k], b = k + 1 <= g.K - 1 ? 1.0 - g.w[k + 1] : 0.0;
    double acc[3], d[3];
    st.apply(acc);
#pragma unroll
    for (int q = 0; q < 3; q++) {
      const double o = b != 0.0 ? b * oth[q] : 0.0;
      d[q] = fmad(w, acc[q], o);
      uc[q] = fmad(w, cur[q], uc[q]);
      oth[q] = cur[q];
      cur[q] = d[q];
    }
    if (k > 0 && !st.exchange(a, g.K - 1 - k, d, 3, &flag, st.xy, st.z)) return;
    if (st.row >= 0 && st.part == 0)
#pragma unroll
      for (int q = 0; q < 3; q++) g.u[k][q * a.ld + st.row] = d[q];
  }
  if (st.row >= 0 && st.part == 0)
#pragma unroll
    for (int q = 0; q < 3; q++) g.uc[q * a.ld + st.row] = uc[q];
}

// ---- the whole local/global loop of an outer iteration
//
// For scenes of cloths only, one launch runs every local/global pass: the
// matrix stays in the registers through all of them, positions and the
// intermediate vectors stay in LDS, and the curvature, right-hand-side and
// residual kernels with their boundaries (26 us per pass of a 256^2 cloth,
// 10 us of a 64^2 one, beside solves of 38 and 26) become phases between
// exchanges.  A pass:
//   curvature   a_i of the tile's rows and, again, of the neighbouring rows
//               their bending sums read (no exchange)
//   rhs         springs, bending, collision and position terms of each row; in
//               FP32-split also the first residual pass (v and its pointwise part)
//   exchange    v (FP32-split) or the rhs (FP64)
//   residual    delta_1 = r0 (FP32-split), or the first term c (FP64)
//   sweeps      as in the solves above, every iterate exchanged; the last one
//               moves the staged positions, own and neighbours'
// The sums over a point's ring and R1 entries are dealt to 4 lanes (first
// term: 8) and combined as k_rhs, k_res_b and k_first64 do, with the same
// rounding sequences (local_ops.hpp): the results are theirs bit for bit.
// Measured per pass, separate kernels -> one launch: FP32 256^2 cloth 66 -> 49
// us (sweeps 36, the rest 13), 64^2 38 -> 29; FP64 64^2 50 -> 32.
struct TileLoop {
  const int4* curvItems;     // [tile][curvCap]: first ring slot, slots, index of the first LDS place, cloth vertex
  int curvCap;               // per tile: its rows' items (R of them), then the neighbours'
  const uint16_t* curvLoc;   // LDS places of the items' ring slots
  const uint16_t* ringLoc;   // per ring slot: LDS place of its point in the owner's tile
  const uint16_t* ringItem;  // per ring slot: its point's curvature item there
  const uint16_t* r1Loc;     // per R1 entry: LDS place of its column in the row's tile
  const int2* ringRange;
  const double *cRest, *cStrain, *cBendIn, *cLbo, *cH0;
  const int* r1Off;
  const double *r1Val, *D;
  const double *initRhs, *colRhs, *fixK, *Xrest;
  int withCol, passes;
  double w;
  double* X;
  double* rhsOut;  // recorded steps: every pass's rhs and iterates (SoA, at these strides)
  int64_t rhsStride;
  double* itOut;
  int64_t itStride;
};

// lanes l, l + TPR, ... of 4 held by a thread, combined as xor 2, 1
template <int TPR, class T>
__device__ __forceinline__ T quad_tree(const T (&s)[4 / TPR]) {
  if constexpr (TPR == 1) return (s[0] + s[2]) + (s[1] + s[3]);
  if constexpr (TPR == 2) {
    const T a = s[0] + s[1];
    return a + __shfl_xor(a, 32, kWave);
  }
  if constexpr (TPR == 4) {
    T a = s[0];
    a += __shfl_xor(a, 32, kWave);
    return a + __shfl_xor(a, 16, kWave);
  }
}

template <class T>
constexpr size_t tile_loop_lds(int uCap, int aCap, int iters) {
  // the iterate and the weights; the positions (FP32-split: the iterate is a
  // correction); v or the rhs; D (FP64, for the first term); the curvature vectors
  return ((tile_lds_bytes<T>(uCap, iters) + 15) & ~(size_t)15) + (size_t)uCap * (sizeof(T) == 4 ? 48 : 32) +
         (size_t)aCap * 24;
}

template <class T, int BT, int TPR, int W, bool LM>
__global__ void __launch_bounds__(BT) k_tile_loop(TileShape a, TileLoop g, const T* __restrict__ val) {
  extern __shared__ __attribute__((aligned(16))) char tileLds[];
  __shared__ int flag, stop;
  if (tile_aborted(a.abort, &flag, &stop)) return;
  constexpr bool F32 = sizeof(T) == 4;
  using State = TileState<T, BT, TPR, W, LM, 3, tile_lean<T, TPR, W>()>;
  constexpr int SUBS = State::SUBS, QL = 4 / TPR;
  State st;
  st.template init<false>(a, val, tileLds, stop);
  const int t = threadIdx.x, U = a.uCap, ld = a.ld;
  // LDS arrays after the iterate and the weights
  char* p = tileLds + ((tile_lds_bytes<T>(U, a.iters) + 15) & ~(size_t)15);
  double2* Vxy = (double2*)p;  // v (FP32-split) or the rhs (FP64)
  double2* Pxy = Vxy + U;      // positions (FP32-split)
  double2* Axy = F32 ? Pxy + U : Vxy + U;
  double* Vz = (double*)(Axy + g.curvCap);
  double* Pz = Vz + U;  // positions' z (FP32-split) or D (FP64)
  double* Az = Pz + U;
  if constexpr (!F32) {  // FP64: the iterate is the position
    Pxy = (double2*)st.xy;
    Pz = (double*)st.z;
  }
  double* Dl = Vz + U;  // FP64
  for (int u = t; u < st.nHalo; u += BT) {
    const int h = st.halo[u];
    Pxy[a.R + u] = make_double2(g.X[h], g.X[ld + h]);
    Pz[a.R + u] = g.X[2 * ld + h];
    if constexpr (!F32) Dl[a.R + u] = g.D[h];
  }
  // the row's own constants
  const int rr = st.row >= 0 ? st.row : 0;
  const bool live = st.row >= 0;
  const int2 ring = live ? g.ringRange[rr] : make_int2(0, 0);
  const int q0 = live ? g.r1Off[rr] : 0, q1 = live ? g.r1Off[rr + 1] : 0;
  const double di = g.D[rr], kf = g.fixK[rr];
  double xi[3];
#pragma unroll
  for (int k = 0; k < 3; k++) xi[k] = g.X[k * ld + rr];
  st.stage_own(Pxy, Pz, xi[0], xi[1], xi[2]);
  if constexpr (!F32)
    if (live && st.part == 0) Dl[st.rl] = di;
  __syncthreads();
  int j = 0;  // publications so far
  for (int pass = 0; pass < g.passes; pass++) {
    const bool last = pass == g.passes - 1;
      // curvature
    for (int i = t; i < g.curvCap; i += BT) {
      const int4 it = g.curvItems[(size_t)blockIdx.x * g.curvCap + i];
      if (it.y == 0) continue;
      const uint16_t* loc = g.curvLoc + it.z;
      const int me = loc[0];
      const double x[3] = {Pxy[me].x, Pxy[me].y, Pz[me]};
      double lsum = g.cLbo[it.x];
      T s[3] = {T(0), T(0), T(0)};
      for (int q = 1; q < it.y; q++) {
        const int u = loc[q];
        const double lq = g.cLbo[it.x + q];
        const T l = (T)lq;
        lsum += lq;
        const double2 pu = Pxy[u];
        s[0] = fmad(l, (T)(pu.x - x[0]), s[0]);
        s[1] = fmad(l, (T)(pu.y - x[1]), s[1]);
        s[2] = fmad(l, (T)(Pz[u] - x[2]), s[2]);
      }
      double ad[3];
      curvature_rescale(s, lsum, x, g.cH0[it.w], ad);
      Axy[i] = make_double2(ad[0], ad[1]);
      Az[i] = ad[2];
    }
    __syncthreads();
    // rhs
    double r[3];
    {
      T sp[3][QL];
      double bd[3][QL], sx[3][QL];
#pragma unroll
      for (int q = 0; q < QL; q++)
#pragma unroll
        for (int k = 0; k < 3; k++) {
          sp[k][q] = T(0);
          bd[k][q] = sx[k][q] = 0.0;
        }
      for (int s0 = ring.x; s0 < ring.y; s0 += 4)
#pragma unroll
        for (int q = 0; q < QL; q++) {
          const int s = s0 + st.part + TPR * q;
          if (s >= ring.y) continue;
          const double2 pu = Pxy[g.ringLoc[s]];
          const double pz = Pz[g.ringLoc[s]];
          const int ai = g.ringItem[s];
          const double bw = g.cBendIn[s];
          if (s > ring.x) {
            const T d[3] = {(T)(xi[0] - pu.x), (T)(xi[1] - pu.y), (T)(xi[2] - pz)};
            T f[3] = {sp[0][q], sp[1][q], sp[2][q]};
            add_spring(d, g.cStrain[s], g.cRest[s], f);
#pragma unroll
            for (int k = 0; k < 3; k++) sp[k][q] = f[k];
          }
          const double2 au = Axy[ai];
          bd[0][q] = fmad(bw, au.x, bd[0][q]);
          bd[1][q] = fmad(bw, au.y, bd[1][q]);
          bd[2][q] = fmad(bw, Az[ai], bd[2][q]);
        }
      if constexpr (F32)
        for (int e0 = q0; e0 < q1; e0 += 4)
#pragma unroll
          for (int q = 0; q < QL; q++) {
            const int e = e0 + st.part + TPR * q;
            if (e >= q1) continue;
            const int u = g.r1Loc[e];
            const double av = g.r1Val[e];
            const double2 pu = Pxy[u];
            sx[0][q] = fmad(av, pu.x, sx[0][q]);
            sx[1][q] = fmad(av, pu.y, sx[1][q]);
            sx[2][q] = fmad(av, Pz[u], sx[2][q]);
          }
      double vv[3], pt[3];
#pragma unroll
      for (int k = 0; k < 3; k++) {
        const T spk = quad_tree<TPR, T>(sp[k]);
        const double bdk = quad_tree<TPR, double>(bd[k]);
        r[k] = g.initRhs[k * ld + rr];
        if (ring.y > ring.x) r[k] += (double)spk + bdk;
        if (g.withCol) r[k] += g.colRhs[k * ld + rr];
        if (kf != 0.0) r[k] = fmad(kf, g.Xrest[k * ld + rr], r[k]);
        if constexpr (F32) {
          const double sxk = quad_tree<TPR, double>(sx[k]);
          residual_first(g.w, xi[k], sxk, r[k], di, &vv[k], &pt[k]);
        }
      }
      if constexpr (F32) {
        // (publication j - 2: a correction of two words, or with one sweep the last pass's v)
        if (!st.exchange(a, j, vv, a.iters == 1 ? 3 : 2, &flag, Vxy, Vz)) return;
        j++;
#pragma unroll
        for (int k = 0; k < 3; k++) r[k] = pt[k];
      } else {
        if (!st.exchange(a, j, r, 3, &flag, Vxy, Vz)) return;
        j++;
        if (g.rhsOut && live && st.part == 0)
#pragma unroll
          for (int k = 0; k < 3; k++) g.rhsOut[pass * g.rhsStride + k * ld + st.row] = r[k];
      }
    }
    if constexpr (F32) {
      // second residual pass: delta_1 = r0 = pt + (w / D) R1 v
      double sv[3][QL];
#pragma unroll
      for (int q = 0; q < QL; q++) sv[0][q] = sv[1][q] = sv[2][q] = 0.0;
      for (int e0 = q0; e0 < q1; e0 += 4)
#pragma unroll
        for (int q = 0; q < QL; q++) {
          const int e = e0 + st.part + TPR * q;
          if (e >= q1) continue;
          const int u = g.r1Loc[e];
          const double av = g.r1Val[e];
          const double2 vu = Vxy[u];
          sv[0][q] = fmad(av, vu.x, sv[0][q]);
          sv[1][q] = fmad(av, vu.y, sv[1][q]);
          sv[2][q] = fmad(av, Vz[u], sv[2][q]);
        }
      const double f = g.w / di;
      float r0[3], pre[3] = {0.f, 0.f, 0.f}, cur[3];
#pragma unroll
      for (int k = 0; k < 3; k++) r0[k] = cur[k] = (float)fmad(f, quad_tree<TPR, double>(sv[k]), r[k]);
      for (int it = 0;; it++) {  // cur = delta_{it + 1}
        const bool done = it == a.iters - 1;
        if (done && last) break;
        // (publication j - 2 was v, of three words, at it = 1)
        if (!st.exchange(a, j, cur, it == 1 ? 3 : 2, &flag, (float2*)st.xy, (float*)st.z)) return;
        j++;
        if (done) break;
        const float Wc = (float)st.cheb[it];
        float acc[3];
        st.apply(acc);
#pragma unroll
        for (int k = 0; k < 3; k++) {
          const float d = fmad(Wc, acc[k] + r0[k] - pre[k], pre[k]);
          pre[k] = cur[k];
          cur[k] = d;
        }
      }
#pragma unroll
      for (int k = 0; k < 3; k++) xi[k] += (double)cur[k];
      if (!last) {  // the staged positions move with the last correction
        for (int u = t; u < a.R + st.nHalo; u += BT) {
          const float2 d = ((float2*)st.xy)[u];
          Pxy[u].x += (double)d.x;
          Pxy[u].y += (double)d.y;
          Pz[u] += (double)((float*)st.z)[u];
        }
        __syncthreads();
      }
    } else {
      // the first term c from the staged rhs (8 lanes, as k_first64)
      double s[3][SUBS], c[3];
#pragma unroll
      for (int q = 0; q < SUBS; q++) s[0][q] = s[1][q] = s[2][q] = 0.0;
      for (int e0 = q0; e0 < q1; e0 += 8)
#pragma unroll
        for (int q = 0; q < SUBS; q++) {
          const int e = e0 + st.part + TPR * q;
          if (e >= q1) continue;
          const int u = g.r1Loc[e];
          const double f = g.r1Val[e] / Dl[u];
          const double2 bu = Vxy[u];
          s[0][q] = fmad(f, bu.x, s[0][q]);
          s[1][q] = fmad(f, bu.y, s[1][q]);
          s[2][q] = fmad(f, Vz[u], s[2][q]);
        }
#pragma unroll
      for (int k = 0; k < 3; k++) c[k] = first_term(g.w, lane_tree<TPR, double>(s[k]), r[k], di);
      double pre[3] = {0.0, 0.0, 0.0};
      for (int it = 0; it < a.iters; it++) {
        const double Wc = it > 0 ? st.cheb[it - 1] : 0.0;
        double acc[3], d[3];
        st.apply((T(&)[3])acc);
#pragma unroll
        for (int k = 0; k < 3; k++) {
          d[k] = it == 0 ? acc[k] + c[k] : fmad(Wc, acc[k] + c[k] - pre[k], pre[k]);
          pre[k] = xi[k];
          xi[k] = d[k];
        }
        if (!(last && it == a.iters - 1)) {
          if (!st.exchange(a, j, d, 3, &flag, (double2*)st.xy, (double*)st.z)) return;
          j++;
        }
        if (g.itOut && live && st.part == 0)
#pragma unroll
          for (int k = 0; k < 3; k++) g.itOut[(pass * (int64_t)a.iters + it) * g.itStride + k * ld + st.row] = d[k];
      }
    }
  }
  if (live && st.part == 0)
#pragma unroll
    for (int k = 0; k < 3; k++) g.X[k * ld + st.row] = xi[k];
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
  if (c.threads == 2 * kTwoThreads && c.width == 8)
    return c.laneMajor ? k_tile_solve32_two<true> : k_tile_solve32_two<false>;
  return nullptr;
}
// launched threads and LDS of an FP32 solve
int solve32_threads(const TileConfig& c) { return std::min(c.threads, 512); }
size_t solve32_lds(const TileMesh& t, int iters) {
  return t.cfg.threads == 2 * kTwoThreads ? tile_two_lds_bytes(t.uCap, iters)
                                          : tile_lds_bytes<float>(t.uCap, iters);
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

using Adj = void (*)(TileShape, const double*, TileAdj);
Adj adj_kernel(const TileConfig& c) {
#define PICK(BT, TPR)                                            \
  if (c.threads == BT && c.tpr == TPR) {                         \
    if (c.laneMajor) return k_tile_adj<BT, TPR, 8, true>;        \
    if (c.width == 8) return k_tile_adj<BT, TPR, 8, false>;      \
    if (c.width == 12 && TPR > 1) return k_tile_adj<BT, TPR, (TPR > 1 ? 12 : 8), false>; \
  }
  PICK(256, 4)
  PICK(512, 4)
  PICK(512, 2)
  PICK(512, 1)
#undef PICK
  return nullptr;
}

// Not with one thread per row, nor in FP64 with two: the entries and the passes'
// other phases would need more registers than a thread has (FP64, 256 rows per
// tile: 124 us per pass with 100 registers spilled, 92 as separate kernels).
template <class T>
auto loop_kernel(const TileConfig& c) -> void (*)(TileShape, TileLoop, const T*) {
#define PICK(BT, TPR)                                              \
  if (c.threads == BT && c.tpr == TPR) {                           \
    if (c.laneMajor) return k_tile_loop<T, BT, TPR, 8, true>;      \
    if (c.width == 8) return k_tile_loop<T, BT, TPR, 8, false>;    \
  }
  PICK(256, 4)
  PICK(512, 4)
  if constexpr (sizeof(T) == 4) {
    PICK(512, 2)
  }
#undef PICK
  return nullptr;
}

TileShape shape_of(const DeviceMesh& m, int parity, int iters) {
  TileShape a;
  a.n = m.nSim;
  a.ld = m.ld;
  a.R = m.tile.rowsPerTile;
  a.uCap = m.tile.uCap;
  a.rows = m.tile.rows;
  a.haloOff = m.tile.haloOff;
  a.halo = m.tile.halo;
  a.loc = m.tile.loc;
  a.slotStride = (size_t)m.ld * kRowWords;
  const size_t set = 4 * a.slotStride;  // words per set
  a.slots = m.tile.slots + (parity ? set : 0);
  a.other = m.tile.slots + (parity ? 0 : set);
  a.abort = m.tile.abort;
  a.cheb = m.tile.cheb;
  a.iters = iters;
  return a;
}

// A kernel's dynamic LDS limit belongs to the process, and handles of other
// tilings share the kernels: always the whole of what its static LDS leaves of
// a compute unit's 160 KB, so that no handle lowers it under another one.
constexpr size_t kLdsBytes = 160 << 10;
bool allow_lds(const void* kernel, size_t lds) {
  hipFuncAttributes at;
  return hipFuncGetAttributes(&at, kernel) == hipSuccess && at.sharedSizeBytes + lds <= kLdsBytes &&
         hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                             (int)(kLdsBytes - at.sharedSizeBytes)) == hipSuccess;
}

template <class K>
bool fits(K kernel, int threads, size_t lds, int tiles, int cus) {
  if (!kernel) return false;
  if (lds > (64 << 10) && !allow_lds((const void*)kernel, lds)) {
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
  m.tile.ok32 = fits(solve32_kernel(c), solve32_threads(c), solve32_lds(m.tile, iters), m.tile.nTiles, cus);
  m.tile.ok64 = fits(solve64_kernel(c), c.threads, tile_lds_bytes<double>(m.tile.uCap, iters), m.tile.nTiles, cus);
  m.tile.adj = m.tile.ok64 &&
               fits(adj_kernel(c), c.threads, tile_lds_bytes<double>(m.tile.uCap, iters), m.tile.nTiles, cus);
  if (m.tile.curvCap == 0) return;
  m.tile.loop32 = m.tile.ok32 && fits(loop_kernel<float>(c), c.threads,
                                      tile_loop_lds<float>(m.tile.uCap, m.tile.curvCap, iters), m.tile.nTiles, cus);
  m.tile.loop64 = m.tile.ok64 && fits(loop_kernel<double>(c), c.threads,
                                      tile_loop_lds<double>(m.tile.uCap, m.tile.curvCap, iters), m.tile.nTiles, cus);
}

void launch_tile_reset(const DeviceMesh& m, hipStream_t s) {
  const size_t n = 4 * (size_t)m.ld * kRowWords;
  hipLaunchKernelGGL(k_tile_reset, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, n, m.tile.slots);
}

void launch_tile_solve32(const DeviceMesh& m, int iters, int parity, hipStream_t s) {
  launch_n(m.timer, TC_SWEEP32, iters - 1, solve32_kernel(m.tile.cfg), dim3(m.tile.nTiles),
           dim3(solve32_threads(m.tile.cfg)), (uint32_t)solve32_lds(m.tile, iters), s, shape_of(m, parity, iters), (const float*)m.m2ValF,
           (const float4*)m.r0, m.X);
}

void launch_tile_solve64(const DeviceMesh& m, double w, int iters, int parity, double* out, int64_t outStride,
                         hipStream_t s) {
  const TileFirst ft{m.r1Off, m.r1Col, m.r1Val, m.sysDiag, m.sysRhs, w};
  launch_n(m.timer, TC_SWEEP64, iters - 1, solve64_kernel(m.tile.cfg), dim3(m.tile.nTiles), dim3(m.tile.cfg.threads),
           (uint32_t)tile_lds_bytes<double>(m.tile.uCap, iters), s, shape_of(m, parity, iters), (const double*)m.m2Val, ft,
           m.X, out, outStride);
}

void launch_tile_adj(const DeviceMesh& m, const TileAdj& g, int parity, hipStream_t s) {
  TileShape a = shape_of(m, parity, g.K);
  a.abort = m.tile.abort + 1;  // the forward passes' flag has the host repeat an outer iteration
  hipLaunchKernelGGL(adj_kernel(m.tile.cfg), dim3(m.tile.nTiles), dim3(m.tile.cfg.threads),
                     tile_lds_bytes<double>(m.tile.uCap, g.K), s, a, (const double*)m.m2Val, g);
}

void launch_tile_loop(const DeviceMesh& m, int precision, double w, int passes, int iters, int withCol,
                      double* rhsOut, int64_t rhsStride, double* itOut, int64_t itStride, hipStream_t s) {
  const TileMesh& t = m.tile;
  TileLoop g;
  g.curvItems = t.curvItems;
  g.curvCap = t.curvCap;
  g.curvLoc = t.curvLoc;
  g.ringLoc = t.ringLoc;
  g.ringItem = t.ringItem;
  g.r1Loc = t.r1Loc;
  g.ringRange = m.ringRange;
  g.cRest = m.cRest;
  g.cStrain = m.cStrain;
  g.cBendIn = m.cBendIn;
  g.cLbo = m.cLbo;
  g.cH0 = m.cH0;
  g.r1Off = m.r1Off;
  g.r1Val = m.r1Val;
  g.D = m.sysDiag;
  g.initRhs = m.initRhs;
  g.colRhs = m.colRhs;
  g.fixK = m.fixK;
  g.Xrest = m.Xrest;
  g.withCol = withCol;
  g.passes = passes;
  g.w = w;
  g.X = m.X;
  g.rhsOut = rhsOut;
  g.rhsStride = rhsStride;
  g.itOut = itOut;
  g.itStride = itStride;
  const TileShape a = shape_of(m, 0, iters);
  if (precision == 0)
    launch_t(m.timer, TC_LOOP, loop_kernel<double>(t.cfg), dim3(t.nTiles), dim3(t.cfg.threads),
             (uint32_t)tile_loop_lds<double>(t.uCap, t.curvCap, iters), s, a, g, (const double*)m.m2Val);
  else
    launch_t(m.timer, TC_LOOP, loop_kernel<float>(t.cfg), dim3(t.nTiles), dim3(t.cfg.threads),
             (uint32_t)tile_loop_lds<float>(t.uCap, t.curvCap, iters), s, a, g, (const float*)m.m2ValF);
}

}  // namespace pdipc
