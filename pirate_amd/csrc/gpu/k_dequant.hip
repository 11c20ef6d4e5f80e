// Dequantization of packed int4 input on gfx950.
// Reference semantics: ReferenceDequantizationKernel::apply (src_lib/GpuDequantizationKernel.cu:326-380),
// format in include/pirate/GpuDequantizationKernel.hpp:17-43:
//   data (nbeams, nfreq, ntime) int4, two per byte, low nibble = even sample;
//   scales_offsets (nbeams, nfreq, ntime/256, 2) float16 {scale, offset}, converted to float
//   before any arithmetic;  out = (value == -8) ? 0 : scale * value + offset.
// The product of a float16 scale and a 4-bit integer is exact in float32, so the single
// rounding of fmaf equals the reference's multiply-then-add. 16-bit outputs round that float32
// value to the storage type.
//
// HBM-bound (0.5 B read, 2-4 B written per sample). One thread per 16 bytes of output (4 float32
// or 8 16-bit samples), so that each store instruction of a wave writes 1 KB without gaps: with
// 8 samples per thread, float32 took two stores, each of every other 16 bytes (16 beams x 16384
// channels x 2048 samples, float32: 0.85 -> 0.42 ms, 5.8 TB/s; float16 0.25 -> 0.23 ms). 64 or 32 consecutive threads share one (scale,
// offset) pair.

#include "device_common.hpp"
#include "kernels.hpp"

#include <algorithm>

namespace pirate_amd {

template<typename Tout>
__global__ void __launch_bounds__(256)
k_dequant(const void *data, const uint32_t *scoff, Tout *out, long nthreads)
{
    constexpr int V = 16 / int(sizeof(Tout));                          // samples per thread
    using Word = typename std::conditional<V == 4, uint16_t, uint32_t>::type;
    const long w = long(blockIdx.x) * 256 + threadIdx.x;
    if (w >= nthreads)
        return;
    const uint32_t word = static_cast<const Word *>(data)[w];
    const uint32_t so = scoff[w / (256 / V)];                          // one pair per 256 samples
    const float scale = __half2float(__ushort_as_half((unsigned short) (so & 0xffffu)));
    const float offset = __half2float(__ushort_as_half((unsigned short) (so >> 16)));
    float x[V];
#pragma unroll
    for (int k = 0; k < V; k++) {
        const int nib = int((word >> (4 * k)) & 0xfu);
        const float v = float((nib ^ 8) - 8);
        x[k] = (nib == 8) ? 0.0f : fmaf(scale, v, offset);
    }
    stv_st<Tout, V>(out + V * w, x);
}

template<typename Tout>
static void launch_dequant_t(const void *data, const void *scoff, void *out, long nsamples, hipStream_t st)
{
    constexpr long V = 16 / long(sizeof(Tout));
    // A launch takes less than 2^32 threads (of more, HIP runs the low 32 bits' worth, without an error).
    for (long s0 = 0; s0 < nsamples; s0 += V << 30) {
        const long nthreads = std::min(nsamples - s0, V << 30) / V;
        hipLaunchKernelGGL(k_dequant<Tout>, dim3((nthreads + 255) / 256), dim3(256), 0, st, (const char *) data + s0 / 2,
                           (const uint32_t *) scoff + s0 / 256, (Tout *) out + s0, nthreads);
    }
}

void launch_dequant(Dtype dt, const void *data, const void *scoff, void *out, long nsamples, hipStream_t st)
{
    switch (dt) {
        case Dtype::float32: launch_dequant_t<float>(data, scoff, out, nsamples, st); break;
        case Dtype::float16: launch_dequant_t<__half>(data, scoff, out, nsamples, st); break;
        case Dtype::bfloat16: launch_dequant_t<__hip_bfloat16>(data, scoff, out, nsamples, st); break;
    }
}

}  // namespace pirate_amd
