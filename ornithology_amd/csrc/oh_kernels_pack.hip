// oh_kernels_pack.hip - the translation unit of the planes -> GGUF byte order copy.
#include "oh_common.h"
#include "oh_launch.h"

namespace {

// Two bytes of the GGUF blocks of super-blocks [b0, b0 + n) per thread: every
// piece of a block starts and ends at an even byte. The host's loop over the
// blocks' pieces took longer than the copy from the device (encoding 4 M
// values to Q4_K, a whole call: 954 us, 877 with this).
__global__ void __launch_bounds__(256) oh_k_gguf_pack(const uint8_t *A, const uint8_t *B, const uint8_t *C, int type, int size,
                                                      int64_t b0, int64_t n, uint16_t *out) {
    const int64_t w = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (w >= n * (size / 2)) return;
    const int64_t i = b0 + w / (size / 2);
    const int o = 2 * (int)(w % (size / 2));
    const uint8_t *src;
    if (type == OH_Q4_K) {
        src = o < 16 ? B + 16 * i + o : A + oh_a_off(OH_Q4_K, i, o - 16);
    } else if (type == OH_Q6_K) {
        src = o < 192 ? A + oh_a_off(OH_Q6_K, i, o) : o < 208 ? B + 16 * i + o - 192 : C + 2 * i;
    } else if (type == OH_Q8_0) {
        const int k = o / 34, p = o % 34;
        src = p < 2 ? B + 16 * i + 2 * k : A + oh_a_off(OH_Q8_0, i, 32 * k + p - 2);
    } else {
        src = o < 2 ? C + 2 * i : A + 64 * i + o - 2;
    }
    stg(out + w, ldg((const uint16_t *)src));
}

} // namespace

extern "C" hipError_t oh_launch_gguf_pack(const uint8_t *A, const uint8_t *B, const uint8_t *C, int type, int size,
                                          int64_t b0, int64_t n, void *out, hipStream_t st) {
    if (n <= 0) return hipSuccess;
    const int64_t words = n * (size / 2);
    hipLaunchKernelGGL(oh_k_gguf_pack, dim3((unsigned)((words + 255) / 256)), dim3(256), 0, st, A, B, C, type, size, b0, n,
                       (uint16_t *)out);
    return hipGetLastError();
}
