// A HIP runtime on the host, for checking which addresses kernels touch: a
// launch runs its threads one after another on one CPU thread (fibers that
// switch at barriers and matrix instructions), and every device allocation ends
// at a page without access, so that a read or write past its end is a
// segmentation fault.  New memory holds 0xFF bytes (NaN, index -1).
#pragma once

#include <sys/mman.h>
#include <ucontext.h>

#include <cmath>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <memory>
#include <vector>

#define __global__
#define __device__
#define __forceinline__ inline
#define __launch_bounds__(...)
#define __shared__ thread_local

typedef int hipError_t;
typedef void* hipStream_t;
typedef void* hipEvent_t;
enum { hipSuccess = 0 };
enum { hipMemcpyHostToDevice, hipMemcpyDeviceToHost, hipMemcpyDeviceToDevice, hipHostMallocDefault = 0 };

struct dim3 {
    unsigned x, y = 1, z = 1;
    dim3(unsigned x_ = 1) : x(x_) {}
};
inline thread_local dim3 threadIdx, blockIdx, blockDim, gridDim;

inline const char* hipGetErrorString(hipError_t) { return ""; }
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
template <class T> hipError_t hipMalloc(T** p, size_t n) {
    const size_t page = 4096, len = (n + page - 1) / page * page;
    char* b = static_cast<char*>(mmap(nullptr, len + page, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0));
    if (b == MAP_FAILED || mprotect(b + len, page, PROT_NONE)) std::abort();
    std::memset(b, 0xFF, len);
    *p = reinterpret_cast<T*>(b + len - n);
    return hipSuccess;
}
template <class T> hipError_t hipHostMalloc(T** p, size_t n, int) { return hipMalloc(p, n); }
inline hipError_t hipFree(void*) { return hipSuccess; }
inline hipError_t hipHostFree(void*) { return hipSuccess; }
inline hipError_t hipMemcpy(void* d, const void* s, size_t n, int) { std::memcpy(d, s, n); return hipSuccess; }
inline hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, int, hipStream_t) { return hipMemcpy(d, s, n, 0); }
inline hipError_t hipMemset(void* d, int v, size_t n) { std::memset(d, v, n); return hipSuccess; }
inline hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) { return hipMemset(d, v, n); }

inline uint32_t __float_as_uint(float x) { uint32_t u; std::memcpy(&u, &x, 4); return u; }
inline float __uint_as_float(uint32_t u) { float x; std::memcpy(&x, &u, 4); return x; }
template <class T> T min(T a, T b) { return a < b ? a : b; }

namespace host_hip {

struct Fiber {
    ucontext_t ctx;
    std::unique_ptr<char[]> stack;
    long waves = 0, blocks = 0;   // barriers passed
    bool done = false;
};
constexpr size_t STACK = 64 * 1024;
inline std::vector<Fiber> fibers;
inline ucontext_t sched;
inline std::vector<long> wave_here;   // arrivals per wavefront
inline long block_here = 0;
inline std::function<void()>* body = nullptr;
inline unsigned self = 0;

inline void yield() { swapcontext(&fibers[self].ctx, &sched); }
inline void entry() {
    (*body)();
    fibers[self].done = true;
    yield();
}
inline void wave_barrier() {
    Fiber& f = fibers[self];
    const unsigned w = self / 64;
    ++wave_here[w];
    ++f.waves;
    while (wave_here[w] < 64 * f.waves) yield();
}
inline void block_barrier() {
    Fiber& f = fibers[self];
    ++block_here;
    ++f.blocks;
    while (block_here < long(fibers.size()) * f.blocks) yield();
}
inline void launch(dim3 grid, dim3 block, std::function<void()> kernel) {
    const unsigned n = block.x;
    if (fibers.size() != n) {
        fibers = std::vector<Fiber>(n);
        for (Fiber& f : fibers) f.stack.reset(new char[STACK]);
    }
    body = &kernel;
    gridDim = grid;
    blockDim = block;
    for (unsigned b = 0; b < grid.x; ++b) {
        blockIdx = dim3(b);
        wave_here.assign((n + 63) / 64, 0);
        block_here = 0;
        for (Fiber& f : fibers) {
            f.waves = f.blocks = 0;
            f.done = false;
            getcontext(&f.ctx);
            f.ctx.uc_stack.ss_sp = f.stack.get();
            f.ctx.uc_stack.ss_size = STACK;
            f.ctx.uc_link = nullptr;
            makecontext(&f.ctx, entry, 0);
        }
        for (bool left = true; left;) {
            left = false;
            for (self = 0; self < n; ++self)
                if (!fibers[self].done) {
                    threadIdx = dim3(self);
                    swapcontext(&sched, &fibers[self].ctx);
                    left |= !fibers[self].done;
                }
        }
    }
}

typedef short s4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));
inline s4 op_a[2][64 * 16], op_b[2][64 * 16];

// D = A B + C over 16x16x16: lane l holds A[l % 16][4 (l / 16) ..], B[4 (l / 16) ..][l % 16]
// and D[4 (l / 16) ..][l % 16]
inline f4 mfma_16x16x16_bf16(s4 a, s4 b, f4 c, int, int, int) {
    const unsigned w0 = self / 64 * 64, l = self % 64;
    const long p = fibers[self].waves & 1;
    op_a[p][self] = a;
    op_b[p][self] = b;
    wave_barrier();
    auto val = [](short x) { return __uint_as_float(uint32_t(uint16_t(x)) << 16); };
    for (unsigned i = 0; i < 4; ++i)
        for (unsigned k = 0; k < 16; ++k)
            c[i] += val(op_a[p][w0 + 16 * (k / 4) + 4 * (l / 16) + i][k % 4]) * val(op_b[p][w0 + 16 * (k / 4) + l % 16][k % 4]);
    return c;
}

}  // namespace host_hip

inline void __syncthreads() { host_hip::block_barrier(); }
#define __builtin_amdgcn_mfma_f32_16x16x16bf16_1k host_hip::mfma_16x16x16_bf16
#define hipLaunchKernelGGL(k, grid, block, lds, stream, ...) host_hip::launch(grid, block, [&] { k(__VA_ARGS__); })
