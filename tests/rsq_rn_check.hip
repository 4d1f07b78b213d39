// Device check of dist_rn (liquidsimulation_amd/csrc/lps_kernels.hip): distance
// and reciprocal distance from one hardware reciprocal square root, against
// the IEEE square root and division for every float in [2^-96, 2^80).  The
// expressions are those of dist_rn.  Prints the number of floats, of wrong
// roots, of wrong reciprocals that dist_rn accepts, and of floats it refuses.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstdio>

__global__ void k_check(uint32_t u0, uint32_t u1, unsigned long long* out) {
    unsigned long long root = 0, rcp = 0, refused = 0;
    for (uint64_t u = (uint64_t)u0 + blockIdx.x * blockDim.x + threadIdx.x; u < u1; u += gridDim.x * blockDim.x) {
        const float s = __uint_as_float((uint32_t)u);
        const float y0 = __builtin_amdgcn_rsqf(s);
        const float g = s * y0;
        const float d = __builtin_fmaf(__builtin_fmaf(-g, g, s), 0.5f * y0, g);
        const float e = __builtin_fmaf(-d, y0, 1.f);
        const float y = __builtin_fmaf(e, y0, y0);
        const float ref = __builtin_sqrtf(s);
        if (!(s >= 0x1p-96f && e != 0x1p-24f)) {
            refused++;
            continue;
        }
        if (__float_as_uint(d) != __float_as_uint(ref)) root++;
        if (__float_as_uint(y) != __float_as_uint(1.f / ref)) rcp++;
    }
    if (root) atomicAdd(&out[0], root);
    if (rcp) atomicAdd(&out[1], rcp);
    if (refused) atomicAdd(&out[2], refused);
}

int main() {
    unsigned long long *dev, h[3];
    if (hipMalloc((void**)&dev, sizeof(h)) != hipSuccess || hipMemset(dev, 0, sizeof(h)) != hipSuccess) return 2;
    const uint32_t u0 = (uint32_t)(127 - 96) << 23, u1 = (uint32_t)(127 + 80) << 23;
    k_check<<<2048, 256>>>(u0, u1, dev);
    if (hipMemcpy(h, dev, sizeof(h), hipMemcpyDeviceToHost) != hipSuccess) return 2;
    std::printf("%u floats, %llu wrong roots, %llu wrong reciprocals, %llu refused\n", u1 - u0, h[0], h[1], h[2]);
    return h[0] == 0 && h[1] == 0 ? 0 : 1;
}
