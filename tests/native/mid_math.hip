// The helpers of device_math.hpp element by element, for the test that compares them with IEEE operations.
#include "../../alien_amd/csrc/device_math.hpp"

namespace {
template <class F> __global__ void apply(const float* in, float* out, int n, F f) {
    const int i = int(blockIdx.x * blockDim.x + threadIdx.x);
    if (i < n) out[i] = f(in[i]);
}
// in, out: n floats of host memory
template <class F> int run(const float* in, float* out, int n, F f) {
    if (n <= 0) return 0;
    const size_t bytes = sizeof(float) * size_t(n);
    float* d = nullptr;
    hipError_t e = hipMalloc(reinterpret_cast<void**>(&d), 2 * bytes);
    if (e != hipSuccess) return int(e);
    e = hipMemcpy(d, in, bytes, hipMemcpyHostToDevice);
    if (e == hipSuccess) {
        apply<<<(n + 255) / 256, 256>>>(d, d + n, n, f);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipMemcpy(out, d + n, bytes, hipMemcpyDeviceToHost);
    (void)hipFree(d);
    return int(e);
}
}  // namespace

extern "C" int mid_apply(int op, const float* in, float* out, int n) {
    using namespace alien;
    switch (op) {
        case 0: return run(in, out, n, [] __device__(float x) { return mid_rcp(x); });
        case 1: return run(in, out, n, [] __device__(float x) { return mid_sqrt(x); });
        case 2: return run(in, out, n, [] __device__(float x) { return mid_div<5>(x); });
        case 3: return run(in, out, n, [] __device__(float x) { return mid_div<6>(x); });
        case 4: return run(in, out, n, [] __device__(float x) { return mid_range(x) ? 1.0f : 0.0f; });
    }
    return -1;
}
