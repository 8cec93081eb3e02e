// Device buffers set to constants, all of a reset in one launch.
//
// A reset sets every field, memory variable, auxiliary and output of a run.
// From host vectors that was a fill in host memory and a copy over the bus at
// some 20 GB/s; on the device it is bound by writing, at the 6.8 TB/s of a
// large fill (16 bytes a lane, consecutive lanes).  Measured, reset and run: 60
// RK3 steps on 6,006 tets (N = 5, attenuation, PML) 59.9 -> 27.2 ms, 300 steps of
// 4 FP32 shots on 3,000 tets (N = 4) 47.0 -> 38.7 ms, 1,000 RK4 steps on 3,072
// tets (N = 3) 64.4 -> 63.3 ms.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <vector>

namespace nexd {

struct FillSegment {
    unsigned *p;          // 16-byte aligned
    size_t words;         // of 4 bytes
    unsigned even, odd;   // the words' values
};
constexpr int kFillSegments = 32;
struct FillList {
    FillSegment s[kFillSegments];
    int n;
};

static __global__ void __launch_bounds__(256) fill_kernel(FillList l) {
    typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
    const size_t id = (size_t)blockIdx.x * blockDim.x + threadIdx.x, step = (size_t)gridDim.x * blockDim.x;
    for (int k = 0; k < l.n; ++k) {
        const FillSegment s = l.s[k];
        const u32x4 v = {s.even, s.odd, s.even, s.odd};
        const size_t quads = s.words / 4;
        u32x4 *q = reinterpret_cast<u32x4 *>(s.p);
        for (size_t i = id; i < quads; i += step) q[i] = v;
        if (id < s.words % 4) s.p[4 * quads + id] = id % 2 ? s.odd : s.even;
    }
}

// Collects the buffers, run() sets them and waits.  On the null stream, as the
// copies were: after everything queued on the device's streams.
class Fill {
public:
    template <typename T>
    void add(T *p, size_t n, T value) {
        static_assert(sizeof(T) == 4 || sizeof(T) == 8, "words");
        unsigned w[2];
        std::memcpy(w, &value, sizeof(T));
        if (sizeof(T) == 4) w[1] = w[0];
        if (p && n) seg_.push_back({reinterpret_cast<unsigned *>(p), n * (sizeof(T) / 4), w[0], w[1]});
    }
    hipError_t run(int device) {
        int before = device;
        hipError_t e = hipGetDevice(&before);
        if (e == hipSuccess && before != device) e = hipSetDevice(device);
        if (e != hipSuccess) return e;
        for (size_t at = 0; at < seg_.size(); at += kFillSegments) {
            FillList l{};
            size_t most = 0;
            for (; l.n < kFillSegments && at + l.n < seg_.size(); ++l.n) {
                l.s[l.n] = seg_[at + l.n];
                most = std::max(most, l.s[l.n].words);
            }
            // four blocks of four waves a CU, fewer for small buffers
            const unsigned grid = (unsigned)std::min<size_t>(2048, most / 1024 + 1);
            hipLaunchKernelGGL(fill_kernel, dim3(grid), dim3(256), 0, nullptr, l);
        }
        e = hipGetLastError();
        if (e == hipSuccess) e = hipStreamSynchronize(nullptr);
        if (before != device) (void)hipSetDevice(before);
        return e;
    }

private:
    std::vector<FillSegment> seg_;
};

}  // namespace nexd
