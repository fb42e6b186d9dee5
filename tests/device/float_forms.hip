/*
 * The float helpers of include/blackframe_math.h that have a form of their own on the device, item by item
 * on the device (float_forms_device) and in their bit forms on the host (float_forms_host).
 */
#include <hip/hip_runtime.h>

#include "../../include/blackframe_math.h"

struct float_forms {
    uint32_t classes; /* bit 0: NaN, bit 1: finite */
    uint32_t mantissa;
    int32_t exponent;
    uint32_t scaled;
};

static __host__ __device__ float_forms forms_of(uint32_t bits, int32_t n) {
    const float x = bf_bits_float(bits);
    float_forms f;
    int e = 0;
    f.classes = (bf_isnan(x) ? 1u : 0u) | (bf_isfinite(x) ? 2u : 0u);
    f.mantissa = bf_float_bits(bf_frexpf(x, &e));
    f.exponent = e;
    f.scaled = bf_float_bits(bf_ldexpf(x, n));
    return f;
}

__global__ void k_float_forms(const uint32_t* bits, const int32_t* exponents, uint32_t count, float_forms* out) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < count) out[i] = forms_of(bits[i], exponents[i]);
}

extern "C" int float_forms_device(const uint32_t* bits, const int32_t* exponents, uint32_t count, float_forms* out) {
    if (count == 0u) return 0;
    hipLaunchKernelGGL(k_float_forms, dim3((count - 1u) / 256u + 1u), dim3(256), 0, nullptr, bits, exponents, count, out);
    return (int)hipGetLastError();
}

extern "C" void float_forms_host(const uint32_t* bits, const int32_t* exponents, uint32_t count, float_forms* out) {
    for (uint32_t i = 0; i < count; ++i) out[i] = forms_of(bits[i], exponents[i]);
}
