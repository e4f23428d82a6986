// Row-wise element-wise kernels for gfx950: RMSNorm, fused add+RMSNorm, SiLU-gate and residual
// add.  Replace src/kernel/norm.cu, activation.cu and add.cu of the BlitzScale worker.  All of
// them move 16 bytes per lane and reduce in fp32, within a wave through the vector ALU's lane permutes.
#include "bz_common.hpp"

namespace bz {

// sum over the workgroup, wave by wave; every lane gets the result (called once per kernel: smem is not handed back)
__device__ __forceinline__ float block_sum(float v, float (&smem)[16]) {
    v = wave_sum(v);
    const int wave = threadIdx.x / 64, lane = threadIdx.x % 64, nw = (blockDim.x + 63) / 64;
    if (lane == 0) smem[wave] = v;
    __syncthreads();
    float part[8], t = 0.f; // (eight asked for at once; a loop over the waves that there are waits for each)
    for (int w0 = 0; w0 < nw; w0 += 8) {
#pragma unroll
        for (int w = 0; w < 8; w += 4) *reinterpret_cast<float4*>(&part[w]) = *reinterpret_cast<const float4*>(&smem[w0 + w]);
#pragma unroll
        for (int w = 0; w < 8; ++w) t += w0 + w < nw ? part[w] : 0.f;
    }
    return t;
}

// out[n,:] = x[n,:] * rsqrt(mean(x^2)+eps) * w.  ADD: residual += input first (rounded to storage),
// x is the rounded residual and the result overwrites input.
// WHOLE: a lane has at most one vector of eight (rows of up to 8 192, the workgroup is made that wide): the row stays in
// registers between the sum and the scaling and the weights are asked for with it, one memory round trip where the other
// form has two, which is what bounds the kernel at a few rows and half of it at a thousand.  Same sums, same bits.
template <typename T, bool ADD, bool WHOLE>
__global__ __launch_bounds__(1024) void rms_norm_kernel(T* input, T* residual, const T* weight, T* output,
                                                         uint32_t h, float eps) {
    __shared__ __attribute__((aligned(16))) float smem[16];
    const size_t row = (size_t)blockIdx.x * h;
    const uint32_t nvec = h / 8;
    float ss = 0.f;
    float x[8];
    Vec8<T> w;
    for (uint32_t i = threadIdx.x; i < nvec; i += blockDim.x) {
        Vec8<T> v, r;
        v.load(input + row + i * 8);
        if (ADD) r.load(residual + row + i * 8);
        if (WHOLE) w.load(weight + i * 8);
        v.to_float(x);
        if (ADD) {
            float y[8];
            r.to_float(y);
#pragma unroll
            for (int e = 0; e < 8; ++e) x[e] += y[e];
            r.from_float(x);
            r.store(residual + row + i * 8);
            r.to_float(x); // the rounded residual is what gets normalised
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) ss += x[e] * x[e];
        if (WHOLE) break;
    }
    ss = block_sum(ss, smem);
    const float rr = rsqrtf(ss / (float)h + eps);
    const T* src = ADD ? residual : input;
    for (uint32_t i = threadIdx.x; i < nvec; i += blockDim.x) {
        Vec8<T> v;
        float g[8];
        if (!WHOLE) {
            v.load(src + row + i * 8);
            w.load(weight + i * 8);
            v.to_float(x);
        }
        w.to_float(g);
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = x[e] * rr * g[e];
        v.from_float(x);
        v.store(output + row + i * 8);
        if (WHOLE) break;
    }
}

// out[n,i] = silu(in[n,i]) * in[n,I+i]
template <typename T>
__global__ __launch_bounds__(256) void silu_and_mul_kernel(const T* in, T* out, uint32_t I) {
    const size_t n = blockIdx.y;
    const uint32_t i = (blockIdx.x * blockDim.x + threadIdx.x) * 8;
    if (i >= I) return;
    Vec8<T> g, u;
    float gf[8], uf[8];
    g.load(in + n * 2 * I + i);
    u.load(in + n * 2 * I + I + i);
    g.to_float(gf);
    u.to_float(uf);
#pragma unroll
    for (int e = 0; e < 8; ++e) gf[e] = gf[e] / (1.0f + __expf(-gf[e])) * uf[e];
    g.from_float(gf);
    g.store(out + n * I + i);
}

// residual += input, exactly one rounding per element
template <typename T> __device__ __forceinline__ void add8(Vec8<T>& r, const Vec8<T>& x);
template <> __device__ __forceinline__ void add8<f16_t>(Vec8<f16_t>& r, const Vec8<f16_t>& x) {
    // native packed f16 add rounds the exact sum once
    uint32_t a[4] = {r.raw.x, r.raw.y, r.raw.z, r.raw.w};
    const uint32_t b[4] = {x.raw.x, x.raw.y, x.raw.z, x.raw.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        __half2 ha = *reinterpret_cast<__half2*>(&a[i]);
        const __half2 hb = *reinterpret_cast<const __half2*>(&b[i]);
        ha = __hadd2(ha, hb);
        a[i] = *reinterpret_cast<uint32_t*>(&ha);
    }
    r.raw = make_uint4(a[0], a[1], a[2], a[3]);
}
template <> __device__ __forceinline__ void add8<bf16_t>(Vec8<bf16_t>& r, const Vec8<bf16_t>& x) {
    // the fp32 sum of two bf16 values is exact whenever it can matter for the bf16 rounding
    float a[8], b[8];
    r.to_float(a);
    x.to_float(b);
#pragma unroll
    for (int e = 0; e < 8; ++e) a[e] += b[e];
    r.from_float(a);
}

template <typename T>
__global__ __launch_bounds__(256) void add_residual_kernel(const T* input, T* residual, size_t nvec) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nvec) return;
    Vec8<T> r, x;
    r.load(residual + i * 8);
    x.load(input + i * 8);
    add8<T>(r, x);
    r.store(residual + i * 8);
}

template <typename T, bool ADD>
static void launch_rms_norm(void* input, void* residual, const void* weight, void* output, uint32_t rows, uint32_t h, float eps,
                            hipStream_t s) {
    uint32_t t = (h / 8 + 63) / 64 * 64;
    t = t > 1024 ? 1024 : (t < 64 ? 64 : t);
    if (h / 8 <= t)
        launch_kernel((rms_norm_kernel<T, ADD, true>), dim3(rows), dim3(t), 0, s, (T*)input, (T*)residual, (const T*)weight,
                           (T*)output, h, eps);
    else
        launch_kernel((rms_norm_kernel<T, ADD, false>), dim3(rows), dim3(t), 0, s, (T*)input, (T*)residual, (const T*)weight,
                           (T*)output, h, eps);
}

} // namespace bz

using namespace bz;

extern "C" int bz_rms_norm(const void* input, const void* weight, void* output, int dtype, uint32_t num_tokens,
                           uint32_t hidden_size, float eps, void* stream) {
    if (!input || !weight || !output) return BZ_ERR_BAD_ARG;
    if (hidden_size % 8) return BZ_ERR_UNSUPPORTED;
    if (num_tokens == 0) return 0;
    void* in = const_cast<void*>(input);
    if (dtype == BZ_F16) launch_rms_norm<f16_t, false>(in, nullptr, weight, output, num_tokens, hidden_size, eps, (hipStream_t)stream);
    else if (dtype == BZ_BF16) launch_rms_norm<bf16_t, false>(in, nullptr, weight, output, num_tokens, hidden_size, eps, (hipStream_t)stream);
    else return BZ_ERR_UNSUPPORTED;
    BZ_LAUNCH_CHECK();
    return 0;
}

extern "C" int bz_add_rms_norm(void* input, void* residual, const void* weight, int dtype, uint32_t num_tokens,
                               uint32_t hidden_size, float eps, void* stream) {
    if (!input || !weight || !residual) return BZ_ERR_BAD_ARG;
    if (hidden_size % 8) return BZ_ERR_UNSUPPORTED;
    if (num_tokens == 0) return 0;
    if (dtype == BZ_F16) launch_rms_norm<f16_t, true>(input, residual, weight, input, num_tokens, hidden_size, eps, (hipStream_t)stream);
    else if (dtype == BZ_BF16) launch_rms_norm<bf16_t, true>(input, residual, weight, input, num_tokens, hidden_size, eps, (hipStream_t)stream);
    else return BZ_ERR_UNSUPPORTED;
    BZ_LAUNCH_CHECK();
    return 0;
}

extern "C" int bz_silu_and_mul(const void* input, void* output, int dtype, uint32_t num_tokens, uint32_t inter_size,
                               void* stream) {
    if (!input || !output) return BZ_ERR_BAD_ARG;
    if (inter_size % 8) return BZ_ERR_UNSUPPORTED;
    if (num_tokens == 0 || inter_size == 0) return 0;
    hipStream_t s = (hipStream_t)stream;
    const dim3 block(256), grid((inter_size / 8 + 255) / 256, num_tokens);
    if (dtype == BZ_F16)
        launch_kernel((silu_and_mul_kernel<f16_t>), grid, block, 0, s, (const f16_t*)input, (f16_t*)output, inter_size);
    else if (dtype == BZ_BF16)
        launch_kernel((silu_and_mul_kernel<bf16_t>), grid, block, 0, s, (const bf16_t*)input, (bf16_t*)output, inter_size);
    else return BZ_ERR_UNSUPPORTED;
    BZ_LAUNCH_CHECK();
    return 0;
}

extern "C" int bz_add_residual(const void* input, void* residual, int dtype, uint32_t num_tokens, uint32_t dim,
                               void* stream) {
    if (!input || !residual) return BZ_ERR_BAD_ARG;
    const size_t n = (size_t)num_tokens * dim;
    if (n % 8) return BZ_ERR_UNSUPPORTED;
    if (n == 0) return 0;
    hipStream_t s = (hipStream_t)stream;
    const size_t nvec = n / 8;
    const dim3 block(256), grid((unsigned)((nvec + 255) / 256));
    if (dtype == BZ_F16)
        launch_kernel((add_residual_kernel<f16_t>), grid, block, 0, s, (const f16_t*)input, (f16_t*)residual, nvec);
    else if (dtype == BZ_BF16)
        launch_kernel((add_residual_kernel<bf16_t>), grid, block, 0, s, (const bf16_t*)input, (bf16_t*)residual, nvec);
    else return BZ_ERR_UNSUPPORTED;
    BZ_LAUNCH_CHECK();
    return 0;
}
