// What follows a reduction's second stage: the solver's state on the device, and the values the host
// waits for, left in pinned memory.
//
// Included by wl_kernels.h before the kernels that use it.
#ifndef WL_FINISH_H
#define WL_FINISH_H

namespace wl {

// ω of solver!(ml) kept on the device (src/MultiLevelPoisson.jl:110,117-121): st[3] = ω,
// st[4] = r₂ (both in T).  Init sets ω = 1 and r₂ = Σr² after residual!; control takes the new
// Σr² (the value stored in dsc[1], passed in: the fused finish must not read it back through
// another pointer), adapts ω, stores r₂ and keeps the old r₂ in dsc[6].
template <class T>
__device__ __forceinline__ void mg_init_state(double r2sum, T* __restrict__ st) {
  st[3] = T(1);
  st[4] = (T)r2sum;
}
template <class T>
__device__ __forceinline__ void mg_control_state(double r2sum, double* __restrict__ dsc, T* __restrict__ st) {
  const T rnew = (T)r2sum;
  T w = st[3];
  const T r2 = st[4];
  if (rnew >= r2) w = (T)fmax(0.2, 0.9 * (double)w);
  else if (rnew < r2) w = (T)fmin(1.0, 1.02 * (double)w);
  st[3] = w;
  st[4] = rnew;
  dsc[6] = (double)r2;
}

// Values the host waits for (three per step): it writes HOST_UNSET (a NaN no arithmetic here forms)
// before the launch and reads until another value is there.  A copy and a stream synchronisation
// instead cost a launch and the wait for their packets, 15 to 20 us each with the GPU idle: step of
// 64x64 187 -> 139 us, 192x128 205 -> 162, 1024x512 283 -> 262.
// (Second stages in the block that ends last save nothing: its fence, counter and reads of the other
// blocks' partials take what the launch takes, 139 -> 143 us at 64x64; with thousands of blocks the
// fences' cache write-backs cost more than the pass, 870 -> 1610 us at 256x128x128.)
constexpr unsigned long long HOST_UNSET = 0xfff8a5a5a5a5a5a5ull;
enum HostSlot { HOST_R2 = 0, HOST_R2_OLD = 1, HOST_MAX = 2, HOST_ROWS = 3, HOST_DONE = 4, HOST_ROW0 = 8, HOST_SLOTS = 20 };
__device__ __forceinline__ void host_post(double* __restrict__ host, int slot, double v) {
  unsigned long long b = (unsigned long long)__double_as_longlong(v);
  if (b == HOST_UNSET) b = 0x7ff8000000000000ull;
  __hip_atomic_store((unsigned long long*)host + slot, b, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

__global__ void k_post_done(double* __restrict__ host) { host_post(host, HOST_DONE, 1.0); }
// What a control decides besides ω: whether another iteration follows (the host's own tests, with its
// tolerance; last: the iteration limit is reached).  A launch that is issued before the host has read
// Σr² carries a Gate and ends at once where the decision was the other one.
struct Next {
  int* go;
  double tol;
  int last;
};
struct Gate {
  const int* go;  // nullptr: no condition
  int want;
  __device__ __forceinline__ bool closed() const { return go != nullptr && *go != want; }
};
enum FinMode { FIN_SUM = 0, FIN_MEAN = 1, FIN_INIT = 2, FIN_CONTROL = 3 };
// what follows from the sum s: FIN_MEAN (residual!): the mean in T and whether it is removed (st[0..1]);
// FIN_INIT, FIN_CONTROL: the solver's state, the host then told of a control's Σr²
template <class T>
__device__ __forceinline__ void fin_apply(int mode, double s, double* __restrict__ outd, T* __restrict__ st, double ninside,
                                          double* __restrict__ dsc, double* __restrict__ host,
                                          Next next = Next{nullptr, 0, 0}) {
  outd[0] = s;
  if (mode == FIN_MEAN) {
    const T sm = (T)s / (T)ninside;
    st[0] = sm;
    st[1] = fabs(sm) <= T(2) * eps_t<T>() ? T(0) : T(1);
  }
  if (mode == FIN_INIT) mg_init_state<T>(s, st);
  if (mode == FIN_CONTROL) {
    mg_control_state<T>(s, dsc, st);
    if (next.go) *next.go = !((double)(T)s < next.tol) && isfinite((T)s) && !next.last;
    if (host) {
      host[HOST_R2_OLD] = dsc[6];
      host_post(host, HOST_R2, s);
    }
  }
}

__device__ __forceinline__ int fin_tid() { return (int)(threadIdx.x + blockDim.x * threadIdx.y); }
// Whether this block ends last of nb, with the others' partials (each written by its thread 0 before)
// visible to all of its threads
__device__ __forceinline__ bool fin_last(unsigned* cnt, unsigned nb) {
  __shared__ unsigned last;
  if (fin_tid() == 0) {
    __threadfence();
    last = atomicAdd(cnt, 1u) == nb - 1 ? 1u : 0u;
    if (last) atomicExch(cnt, 0u);
  }
  __syncthreads();
  const bool l = last != 0u;
  if (l) __threadfence();
  return l;
}
// N sums Σ partial[k·stride .. k·stride + np) as 1024 threads and block_sum add them (k_finish_sum), by a
// block of 256: each thread stands for four, whose loads and adds run side by side.  Valid in every
// thread of the first wave.
template <int N>
__device__ __forceinline__ void fin_total(const double* partial, int64_t np, int64_t stride, double* out) {
  __shared__ double sh[N][16];
  const int t = fin_tid();
  double a[N][4];
#pragma unroll
  for (int k = 0; k < N; ++k)
#pragma unroll
    for (int j = 0; j < 4; ++j) a[k][j] = 0;
#pragma unroll 4
  for (int64_t q = t; q < np; q += 1024)
#pragma unroll
    for (int k = 0; k < N; ++k)
#pragma unroll
      for (int j = 0; j < 4; ++j) {  // no branch between the loads: one beyond np reads slot 0 and adds 0
        const bool in = q + 256 * j < np;
        const double v = partial[k * stride + (in ? q + 256 * j : 0)];
        a[k][j] += in ? v : 0.0;
      }
#pragma unroll
  for (int k = 0; k < N; ++k)
#pragma unroll
    for (int j = 0; j < 4; ++j) a[k][j] = wave_sum(a[k][j]);
  if ((t & 63) == 0)
#pragma unroll
    for (int k = 0; k < N; ++k)
#pragma unroll
      for (int j = 0; j < 4; ++j) sh[k][4 * j + (t >> 6)] = a[k][j];
  __syncthreads();
#pragma unroll
  for (int k = 0; k < N; ++k) out[k] = wave_sum((t & 63) < 16 ? sh[k][t & 15] : 0.0);
  __syncthreads();
}

}  // namespace wl
#endif
