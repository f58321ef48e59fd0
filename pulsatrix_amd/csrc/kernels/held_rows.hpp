// Row kernels that hold their row in registers between a reduction over it and the pass that uses
// the reduction: T threads own one row (a wave64 or a workgroup), thread t the V-float vectors
// t, t + T, ... of it, at most NV of them. Every input is read from memory once, with all its loads
// in flight before the reduction, where a wave that walks the row twice waits out the memory latency
// of each pass (cols / 64 dependent steps) and reads the row again from L2. Bound by HBM: at 4096 x
// 2048 the softmax takes 13.0 us against 35.3 by such a wave, its backward 15.8 (6.4 TB/s) against 26.6,
// RMSNorm's backward 22.0 (6.1 TB/s) against 48.4, the log-sum-exp 8.1 against 19.1.
#pragma once

#include "common.hpp"

namespace pxk {

constexpr int kHeldThreads = 256;

template <int T_, int V_, int NV_>
struct HeldShape {
    static constexpr int T = T_, V = V_, NV = NV_;
};

// Calls f with the shape for rows of `cols` floats; false (f not called) for rows that no shape holds.
// vec: every operand is 16-byte aligned (a ragged width then still takes single floats). Up to 64
// columns a row is one step of the walking wave, which loses nothing by it (RMSNorm's backward at 16384
// x 64: 5.5 us, 7.1 held). Up to 128 a float4 a thread would leave half the wave idle (16384 x 128: 7.8 us
// walked, 8.6 so, 6.5 by single floats). One wave a row up to 1024 columns, where a workgroup a row would leave most
// of its threads a float4 or less; above, a workgroup, which keeps a thread's share under 32 floats an
// operand up to 8192 columns. RMSNorm's backward, walked and held: 16384 x 500 32.6 and 20.4 us, 4096 x
// 1001 20.7 and 11.4, 2048 x 8191 117 and 47, 8 x 576 5.6 and 3.4, 1 x 4096 27.3 and 3.5. The single-float
// shapes are the finer ones: a place that holds no column costs its exponential and store all the same
// (log-sum-exp, walked and held in twice the places or more: 16384 x 257 9.0 and 10.3 us, 16384 x 2049 51
// and 63; as below 7.0 and 29).
// A launch has fewer than 2^32 threads: 2^24 rows and more of a workgroup each are left to the walk.
template <class F>
bool with_held_shape(int64_t rows, int64_t cols, bool vec, F&& f) {
    if (cols <= kWave || (cols > 1024 && rows >= (int64_t{1} << 24))) return false;
    if (cols <= 128) {
        f(HeldShape<64, 1, 2>{});
    } else if (vec && cols % 4 == 0) {
        if (cols <= 256) f(HeldShape<64, 4, 1>{});
        else if (cols <= 512) f(HeldShape<64, 4, 2>{});
        else if (cols <= 1024) f(HeldShape<64, 4, 4>{});
        else if (cols <= 2048) f(HeldShape<256, 4, 2>{});
        else if (cols <= 4096) f(HeldShape<256, 4, 4>{});
        else if (cols <= 8192) f(HeldShape<256, 4, 8>{});
        else return false;
    } else {
        if (cols <= 256) f(HeldShape<64, 1, 4>{});
        else if (cols <= 512) f(HeldShape<64, 1, 8>{});
        else if (cols <= 1024) f(HeldShape<64, 1, 16>{});
        else if (cols <= 1536) f(HeldShape<256, 1, 6>{});
        else if (cols <= 2048) f(HeldShape<256, 1, 8>{});
        else if (cols <= 3072) f(HeldShape<256, 1, 12>{});
        else if (cols <= 4096) f(HeldShape<256, 1, 16>{});
        else if (cols <= 6144) f(HeldShape<256, 1, 24>{});
        else if (cols <= 8192) f(HeldShape<256, 1, 32>{});
        else return false;
    }
    return true;
}

template <class Shape>
dim3 held_grid(int64_t rows) {
    return dim3(static_cast<unsigned>(cdiv(rows, kHeldThreads / Shape::T)));
}

// A thread's place in its row. The loads clamp their column instead of branching around it (a lane
// past the row reads its last vector again), so they issue back to back; `live` says what counts.
template <class Shape>
struct HeldRow {
    typedef float vec __attribute__((ext_vector_type(Shape::V)));
    int64_t row;
    int t, n;  // thread of the row, vectors of the row (>= 1)

    __device__ HeldRow(int64_t cols)
        : row(static_cast<int64_t>(blockIdx.x) * (kHeldThreads / Shape::T) + threadIdx.x / Shape::T),
          t(threadIdx.x % Shape::T),
          n(static_cast<int>(cols / Shape::V)) {}
    __device__ int column(int j) const { return t + j * Shape::T; }
    __device__ bool live(int j) const { return column(j) < n; }
    __device__ void load(const float* base, vec (&v)[Shape::NV]) const {
        const vec* p = reinterpret_cast<const vec*>(base);
#pragma unroll
        for (int j = 0; j < Shape::NV; ++j) v[j] = p[live(j) ? column(j) : n - 1];
    }
    __device__ void store(float* base, int j, vec v) const { reinterpret_cast<vec*>(base)[column(j)] = v; }
};

// The sum (largest) over a row's threads, the same in each, in a fixed order. With a workgroup to a
// row these hold a barrier that all of it reaches, and each is called once by a kernel.
template <int T>
__device__ __forceinline__ float held_sum(float v) {
    v = wave_sum(v);
    if constexpr (T > kWave) {
        __shared__ float part[T / kWave];
        if (threadIdx.x % kWave == 0) part[threadIdx.x / kWave] = v;
        __syncthreads();
        v = part[0];
#pragma unroll
        for (int w = 1; w < T / kWave; ++w) v += part[w];
    }
    return v;
}

template <int T>
__device__ __forceinline__ float held_max(float v) {
    v = wave_max(v);
    if constexpr (T > kWave) {
        __shared__ float part[T / kWave];
        if (threadIdx.x % kWave == 0) part[threadIdx.x / kWave] = v;
        __syncthreads();
        v = part[0];
#pragma unroll
        for (int w = 1; w < T / kWave; ++w) v = fmaxf(v, part[w]);
    }
    return v;
}

}  // namespace pxk
