// aos.hip -- gplum_particle arrays <-> one device array per field.
//
// Bound by the host link: one transfer of the caller's array per direction, where one
// transfer and one strided host loop per field took 89 ms up and 90 ms down for 1M particles (312
// MB; now 14 and 18 ms) and 6.4 and 7.3 ms for 100k (now 1.3 and 1.9 ms).  The kernels
// touch each word once: consecutive lanes take consecutive words of the particle array
// (coalesced), whose field arrays are read in whole cache lines by a workgroup.
#include "aos.hpp"

namespace gplum {

template <bool PACK>
__global__ __launch_bounds__(256) void k_aos(AosTable table, int i0, int n, unsigned long long *__restrict__ aos) {
    __shared__ AosWord s_w[AOS_WORDS];
    if (threadIdx.x < AOS_WORDS) s_w[threadIdx.x] = table.w[threadIdx.x];
    __syncthreads();
    const size_t words = (size_t)n * AOS_WORDS, step = (size_t)gridDim.x * blockDim.x;
    for (size_t k = (size_t)blockIdx.x * blockDim.x + threadIdx.x; k < words; k += step) {
        const size_t p = k / AOS_WORDS, i = i0 + p;
        const AosWord q = s_w[k - p * AOS_WORDS];
        if (!q.pair) {
            if (!q.a) continue;
            unsigned long long *f = static_cast<unsigned long long *>(q.a) + (size_t)q.stride * i;
            if (PACK) aos[k] = *f;
            else *f = aos[k];
        } else {
            int32_t *half = reinterpret_cast<int32_t *>(aos + k);
            int32_t *a = static_cast<int32_t *>(q.a), *b = static_cast<int32_t *>(q.b);
            if (PACK) {
                if (a) half[0] = a[i];
                if (b) half[1] = b[i];
            } else {
                if (a) a[i] = half[0];
                if (b) b[i] = half[1];
            }
        }
    }
}

template <bool PACK>
static int launch_aos(const AosTable &t, int i0, int n, gplum_particle *aos, hipStream_t st) {
    if (n <= 0) return GPLUM_OK;
    const size_t words = (size_t)n * AOS_WORDS;
    const int grid = (int)std::min<size_t>((words + 255) / 256, 8192);
    hipLaunchKernelGGL(k_aos<PACK>, dim3(grid), dim3(256), 0, st, t, i0, n, reinterpret_cast<unsigned long long *>(aos));
    GPLUM_HIP(hipGetLastError());
    return GPLUM_OK;
}
int aos_pack(const AosTable &t, int i0, int n, gplum_particle *aos, hipStream_t st) {
    return launch_aos<true>(t, i0, n, aos, st);
}
int aos_unpack(const AosTable &t, int i0, int n, const gplum_particle *aos, hipStream_t st) {
    return launch_aos<false>(t, i0, n, const_cast<gplum_particle *>(aos), st);
}

}  // namespace gplum
