// Scan in one pass over the data (decoupled look-back across workgroups).
//
// A workgroup takes a tile of 256 * ITEMS elements: every thread takes ITEMS consecutive ones, the tile is scanned
// through registers, wave shuffles and LDS, the workgroup publishes the tile's aggregate in a status word,
// and its first wave looks back over the status words of the preceding tiles, 64 at a time, until it meets
// one that already knows its inclusive prefix.  Workgroups number themselves by a ticket, so every
// predecessor of a workgroup is already running and the look-back cannot wait for a workgroup that has not
// been scheduled.  The state (ticket + one 64-bit word per tile: flag in the two top bits, value in the low
// 62) is cleared by a kernel in front of the scan.  In-place (out == in) is allowed.
#pragma once
#include <cstdint>
#include <hip/hip_runtime.h>

namespace sph_scan {

constexpr int kThreads = 256;
constexpr int kItems = 8; // elements per thread of a scan over an array
constexpr int kTile = kThreads * kItems;
constexpr int kWaveSize = 64;
constexpr unsigned long long kAggregate = 1ull << 62; // value = the tile's own aggregate
constexpr unsigned long long kInclusive = 2ull << 62; // value = aggregate of everything up to and including the tile

// sums of int, or of 64-bit words that hold two 30-bit numbers
struct Plus {
    typedef int value;
    static __device__ __forceinline__ unsigned long long to_word(int v) { return (unsigned)v; }
    static __device__ __forceinline__ int from_word(unsigned long long w) { return (int)(unsigned)w; }
};
struct PlusPair {
    typedef unsigned long long value;
    static __device__ __forceinline__ unsigned long long to_word(unsigned long long v) { return v; }
    static __device__ __forceinline__ unsigned long long from_word(unsigned long long w) { return w & (kAggregate - 1); }
};

inline int tiles(long n, int items = kItems) { return (int)((n + kThreads * items - 1) / (kThreads * items)); }
// ints of the state that must be zero when the scan kernel starts
inline int state_ints(long n, int items = kItems) { return 2 + 2 * tiles(n > 0 ? n : 1, items); }
// bytes of state a scan of n elements needs (a multiple of 256)
inline size_t state_bytes(long n, int items = kItems) { return ((size_t)state_ints(n, items) * 4 + 255) & ~(size_t)255; }

static __global__ void clear_state_kernel(int *state, int nints)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < nints) state[i] = 0;
}

// What is scanned: an array in memory (16-byte loads where it is aligned), or any function object load(i) that makes
// element i on the fly (an intermediate array less to write and read).
struct FromArray {
    const int32_t *in;
    template <int ITEMS> __device__ __forceinline__ void tile(long base, long n, int (&v)[ITEMS]) const
    {
        static_assert(ITEMS == 8, "two 16-byte loads");
        if (base + ITEMS <= n && ((uintptr_t)in & 15) == 0) {
            const int4 a = *(const int4 *)(in + base), b = *(const int4 *)(in + base + 4);
            v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
        } else {
#pragma unroll
            for (int i = 0; i < ITEMS; i++) v[i] = base + i < n ? in[base + i] : 0;
        }
    }
};
template <class F> struct FromFunction {
    F load;
    template <class V, int ITEMS> __device__ __forceinline__ void tile(long base, long n, V (&v)[ITEMS]) const
    {
#pragma unroll
        for (int i = 0; i < ITEMS; i++) v[i] = base + i < n ? load(base + i) : 0;
    }
};

// Where the sums go: to an array of inclusive sums, the sum of all n to *total (may be null; any address the GPU can
// write, e.g. pinned host memory); or to any function object with the same two members.
struct ToArray {
    int32_t *out, *total;
    template <int ITEMS> __device__ __forceinline__ void tile(long base, long n, int, const int (&incl)[ITEMS]) const
    {
        if (ITEMS == 8 && base + ITEMS <= n && ((uintptr_t)out & 15) == 0) {
            *(int4 *)(out + base) = make_int4(incl[0], incl[1 % ITEMS], incl[2 % ITEMS], incl[3 % ITEMS]);
            *(int4 *)(out + base + 4) = make_int4(incl[4 % ITEMS], incl[5 % ITEMS], incl[6 % ITEMS], incl[7 % ITEMS]);
        } else {
#pragma unroll
            for (int i = 0; i < ITEMS; i++)
                if (base + i < n) out[base + i] = incl[i];
        }
    }
    __device__ __forceinline__ void all(int sum) const
    {
        if (total) *total = sum;
    }
};

template <class OP, int ITEMS, class IN, class OUT>
__global__ __launch_bounds__(kThreads) void scan_kernel(IN in, OUT out, long n, int *state)
{
    typedef typename OP::value V;
    __shared__ int s_ticket;
    __shared__ V s_wave[kThreads / kWaveSize];
    __shared__ V s_prefix;
    unsigned long long *status = (unsigned long long *)(state + 2);
    const int tid = threadIdx.x, lane = tid & (kWaveSize - 1), wave = tid / kWaveSize;
    if (tid == 0) s_ticket = atomicAdd(&state[0], 1);
    __syncthreads();
    const int t = s_ticket;
    const long base = (long)t * (kThreads * ITEMS) + (long)tid * ITEMS;

    V v[ITEMS];
    in.tile(base, n, v);
    // inclusive scan of the thread's items, then of the threads' totals over the wave
#pragma unroll
    for (int i = 1; i < ITEMS; i++) v[i] += v[i - 1];
    V incl = v[ITEMS - 1];
#pragma unroll
    for (int off = 1; off < kWaveSize; off <<= 1) {
        const V u = __shfl_up(incl, off, kWaveSize);
        if (lane >= off) incl += u;
    }
    if (lane == kWaveSize - 1) s_wave[wave] = incl;
    __syncthreads();
    V wave_excl = 0, agg = 0;
#pragma unroll
    for (int w = 0; w < kThreads / kWaveSize; w++) {
        if (w < wave) wave_excl += s_wave[w];
        agg += s_wave[w];
    }

    if (wave == 0) {
        V excl = 0;
        if (t > 0) {
            if (lane == 0)
                __hip_atomic_store(&status[t], kAggregate | OP::to_word(agg), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            for (int b = t - 1;;) {
                const int idx = b - lane; // lane 0 looks at the nearest predecessor
                const unsigned long long w =
                    idx >= 0 ? __hip_atomic_load(&status[idx], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0ull;
                const unsigned long long flag = idx >= 0 ? w >> 62 : 3ull; // 3: before the first tile
                const unsigned long long done = __ballot(flag >= 2), empty = __ballot(flag == 0);
                const int fi = done ? __ffsll((long long)done) - 1 : kWaveSize; // nearest tile that ends the look-back
                const unsigned long long need = fi >= kWaveSize - 1 ? ~0ull : (2ull << fi) - 1ull;
                if (empty & need) { // a predecessor on the way has not published yet
                    __builtin_amdgcn_s_sleep(1);
                    continue;
                }
                V x = (lane <= fi && flag != 3ull) ? OP::from_word(w) : 0;
#pragma unroll
                for (int off = 1; off < kWaveSize; off <<= 1) {
                    const V u = __shfl_down(x, off, kWaveSize);
                    if (lane + off < kWaveSize) x += u;
                }
                excl += __shfl(x, 0, kWaveSize);
                if (fi < kWaveSize) break;
                b -= kWaveSize;
            }
        }
        if (lane == 0) {
            __hip_atomic_store(&status[t], kInclusive | OP::to_word(excl + agg), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            s_prefix = excl;
            if (t == (int)gridDim.x - 1) out.all(excl + agg);
        }
    }
    __syncthreads();
    // what precedes this thread's first item
    V before = s_prefix + wave_excl;
    const V up = __shfl_up(incl, 1, kWaveSize);
    if (lane > 0) before += up;
#pragma unroll
    for (int i = 0; i < ITEMS; i++) v[i] += before;
    out.tile(base, n, before, v);
}

// Enqueues the scan of n elements on st; state: state_bytes(n, ITEMS) bytes of device memory, 8-byte aligned.
// clear_state = false: a kernel enqueued before on the same stream has already zeroed the first state_ints(n, ITEMS) ints.
template <class OP, int ITEMS, class IN, class OUT>
inline hipError_t launch_from(const IN &in, const OUT &out, long n, void *state, hipStream_t st, bool clear_state = true)
{
    if (n <= 0) return hipSuccess;
    const int nints = state_ints(n, ITEMS);
    if (clear_state)
        hipLaunchKernelGGL(clear_state_kernel, dim3((nints + 255) / 256), dim3(256), 0, st, (int *)state, nints);
    hipLaunchKernelGGL((scan_kernel<OP, ITEMS, IN, OUT>), dim3(tiles(n, ITEMS)), dim3(kThreads), 0, st, in, out, n, (int *)state);
    return hipGetLastError();
}
// out[i] = in[0] + ... + in[i]
inline hipError_t launch(const int32_t *in, int32_t *out, long n, void *state, hipStream_t st, int32_t *total = nullptr,
                         bool clear_state = true)
{
    return launch_from<Plus, kItems>(FromArray{in}, ToArray{out, total}, n, state, st, clear_state);
}

} // namespace sph_scan
