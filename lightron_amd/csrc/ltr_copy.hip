// Strided view -> contiguous tensor for MI355X (gfx950): the data movement of the Ulysses exchange (parallel/parallel_cp.py:49-96 of the
// reference, split / all_to_all / cat) on one GPU, where the exchange is an index permutation of whole runs of heads.
#include <hip/hip_runtime.h>
#include <atomic>
#include <stdint.h>
#include "ltr_attn.h"

namespace {

typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

// Division by a run-time constant as a multiplication: floor(n / d) = (n * mul) >> shift for n < 2^31, with
// mul = ceil(2^(31 + bits) / d), bits = ceil(log2 d) (round-up method; the 64-bit product does not overflow).
struct FastDiv {
    unsigned d, shift;
    unsigned long long mul;
};

struct CopyParams {
    const char *src;
    char *dst;
    unsigned n_vec;              // 16-byte vectors in all
    int n_outer;                 // outer dimensions, innermost first in div / stride
    FastDiv run;                 // vectors per contiguous run
    FastDiv div[LTR_COPY_DIMS];
    long long stride[LTR_COPY_DIMS];   // bytes
};

__device__ __forceinline__ unsigned divide(unsigned n, const FastDiv &f) { return (unsigned)((n * f.mul) >> f.shift); }

// Bound: HBM (each byte read and written once).  A thread moves UNROLL vectors of 16 bytes a block's width apart, all loads
// before the stores: four outstanding loads per thread keep the memory pipe full with 32-bit index arithmetic beside it (the
// run-time divisions are multiplications).  Measured on 64 MB of bf16 [4, 8, 1024, 16, 64] (sequence -> head exchange, runs of
// 512 bytes): 24.4 us = 5.5 TB/s, the elementwise copy of a strided view that it replaces 46 us, a plain contiguous copy 26 us.
constexpr int UNROLL = 4;
__global__ __launch_bounds__(256) void copy_strided_kernel(const CopyParams p) {
    const unsigned first = blockIdx.x * (256 * UNROLL) + threadIdx.x;
    u32x4 v[UNROLL];
#pragma unroll
    for (int u = 0; u < UNROLL; u++) {
        const unsigned i = first + u * 256;
        if (i >= p.n_vec) break;
        unsigned o = divide(i, p.run);
        long long off = (long long)(i - o * p.run.d) * 16;
        for (int k = 0; k < p.n_outer; k++) {
            const unsigned q = divide(o, p.div[k]);
            off += (long long)(o - q * p.div[k].d) * p.stride[k];
            o = q;
        }
        v[u] = *(const u32x4 *)(p.src + off);
    }
#pragma unroll
    for (int u = 0; u < UNROLL; u++) {
        const unsigned i = first + u * 256;
        if (i >= p.n_vec) break;
        *(u32x4 *)(p.dst + (long long)i * 16) = v[u];
    }
}

FastDiv fast_div(unsigned d) {
    unsigned bits = 0;
    while (bits < 31 && (1u << bits) < d) bits++;
    FastDiv f;
    f.d = d;
    f.shift = 31 + bits;
    f.mul = ((1ull << f.shift) + d - 1) / d;
    return f;
}

bool on_gfx950() {   // see ltr_rope.hip
    constexpr int MAX_DEVICES = 64;
    static std::atomic<int> arch[MAX_DEVICES];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= MAX_DEVICES) return false;
    int known = arch[dev].load(std::memory_order_acquire);
    if (known == 0) {
        hipDeviceProp_t prop;
        if (hipGetDeviceProperties(&prop, dev) != hipSuccess) return false;
        const char *a = prop.gcnArchName;
        known = (a[0] == 'g' && a[1] == 'f' && a[2] == 'x' && a[3] == '9' && a[4] == '5' && a[5] == '0') ? 1 : -1;
        arch[dev].store(known, std::memory_order_release);
    }
    return known == 1;
}

}  // namespace

extern "C" int ltr_copy_strided(const ltr_copy_args *a, void *stream) {
    if (!a || !a->src || !a->dst || a->n_outer < 0 || a->n_outer > LTR_COPY_DIMS || a->run_bytes < 0) return LTR_EINVAL;
    if (((uintptr_t)a->src | (uintptr_t)a->dst) & 15 || a->run_bytes % 16) return LTR_EALIGN;
    long long total = a->run_bytes / 16;
    for (int i = 0; i < a->n_outer; i++) {
        if (a->size[i] < 0) return LTR_EINVAL;
        if (a->stride_bytes[i] % 16) return LTR_EALIGN;
        if (a->size[i] > 0x7fffffffLL || (a->size[i] > 0 && total > 0x7fffffffLL / a->size[i])) return LTR_EINVAL;   // 32-bit vector index
        total *= a->size[i];
    }
    if (total == 0) return LTR_OK;
    if (total > 0x7fffffffLL - 256 * UNROLL) return LTR_EINVAL;
    if (!on_gfx950()) return LTR_EDEVICE;
    CopyParams p;
    p.src = (const char *)a->src;
    p.dst = (char *)a->dst;
    p.n_vec = (unsigned)total;
    p.n_outer = a->n_outer;
    p.run = fast_div((unsigned)(a->run_bytes / 16));
    for (int i = 0; i < a->n_outer; i++) {
        p.div[i] = fast_div((unsigned)a->size[a->n_outer - 1 - i]);
        p.stride[i] = a->stride_bytes[a->n_outer - 1 - i];
    }
    void *args[] = {(void *)&p};
    const unsigned grid = (unsigned)((total + 256 * UNROLL - 1) / (256 * UNROLL));
    return hipLaunchKernel((const void *)copy_strided_kernel, dim3(grid), dim3(256), args, 0, (hipStream_t)stream) == hipSuccess ? LTR_OK : LTR_ELAUNCH;
}
