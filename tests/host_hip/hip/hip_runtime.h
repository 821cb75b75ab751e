// A HIP runtime on the host, for checking what kernels and the code around
// them do: a launch runs its workgroups on a few CPU threads, a workgroup's
// threads as fibers that switch at barriers, matrix instructions, lane
// reads and while they poll.  Every device allocation ends at a page without
// access, so that a read or write past its end is a segmentation fault, as is
// one through a null pointer.  New memory holds 0xFF bytes (NaN, index -1).
#pragma once

#include <sched.h>
#include <sys/mman.h>

#include <atomic>
#include <cmath>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <memory>
#include <mutex>
#include <thread>
#include <vector>

#define __global__
#define __device__
#define __forceinline__ inline
#define __launch_bounds__(...)
#define __shared__ thread_local

typedef int hipError_t;
typedef void* hipStream_t;
typedef void* hipEvent_t;
enum { hipSuccess = 0, hipErrorOutOfMemory = 2 };
enum { hipMemcpyHostToDevice, hipMemcpyDeviceToHost, hipMemcpyDeviceToDevice, hipHostMallocDefault = 0 };
enum { hipDeviceAttributeMultiprocessorCount };

struct dim3 {
    unsigned x, y = 1, z = 1;
    dim3(unsigned x_ = 1) : x(x_) {}
};
inline thread_local dim3 threadIdx, blockIdx, blockDim, gridDim;

namespace host_hip {
inline long fail_at = -1;   // this many device allocations succeed, the next one fails (-1: none fails)
}
inline const char* hipGetErrorString(hipError_t) { return ""; }
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
inline hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
inline hipError_t hipDeviceGetAttribute(int* v, int, int) { *v = 256; return hipSuccess; }
inline hipError_t hipEventCreate(hipEvent_t*) { return hipSuccess; }
inline hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
inline hipError_t hipEventElapsedTime(float* t, hipEvent_t, hipEvent_t) { *t = 1.0f; return hipSuccess; }
template <class T> hipError_t hipMalloc(T** p, size_t n) {
    if (host_hip::fail_at == 0) { host_hip::fail_at = -1; return hipErrorOutOfMemory; }
    if (host_hip::fail_at > 0) --host_hip::fail_at;
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
template <class T> T max(T a, T b) { return a > b ? a : b; }

namespace host_hip {

// ---- fibers: the threads of the workgroup that this CPU thread runs ----------
struct Fiber {
    void* sp = nullptr;
    std::unique_ptr<char[]> stack;
    long waves = 0, blocks = 0;   // barriers passed
    bool done = false;
};
constexpr size_t STACK = 64 * 1024;
inline thread_local std::vector<Fiber> fibers;
inline thread_local void* sched_sp;
inline thread_local std::vector<long> wave_here;   // arrivals per wavefront
inline thread_local long block_here;
inline thread_local const std::function<void()>* body;
inline thread_local unsigned self;

// saves the callee-saved registers on the stack and continues on another one
extern "C" void host_hip_switch(void** from, void* to);
__asm__(R"(
.weak host_hip_switch
host_hip_switch:
    push %rbp
    push %rbx
    push %r12
    push %r13
    push %r14
    push %r15
    mov %rsp, (%rdi)
    mov %rsi, %rsp
    pop %r15
    pop %r14
    pop %r13
    pop %r12
    pop %rbx
    pop %rbp
    ret
)");

inline void yield() { host_hip_switch(&fibers[self].sp, sched_sp); }
inline void entry() {
    (*body)();
    fibers[self].done = true;
    for (;;) yield();
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
inline void wait_stores() {   // the stores of the whole wavefront
    wave_barrier();
    std::atomic_thread_fence(std::memory_order_seq_cst);
}
inline void poll_pause() {
    if (self % 64 == 0) sched_yield();
    yield();
}
inline void run_block(unsigned b, unsigned grid, unsigned n, const std::function<void()>& kernel) {
    if (fibers.size() != n) {
        fibers = std::vector<Fiber>(n);
        for (Fiber& f : fibers) f.stack.reset(new char[STACK]);
    }
    body = &kernel;
    gridDim = dim3(grid);
    blockDim = dim3(n);
    blockIdx = dim3(b);
    wave_here.assign((n + 63) / 64, 0);
    block_here = 0;
    for (Fiber& f : fibers) {
        f.waves = f.blocks = 0;
        f.done = false;
        void** top = reinterpret_cast<void**>((reinterpret_cast<uintptr_t>(f.stack.get()) + STACK) & ~uintptr_t(15));
        *--top = nullptr;                                // keeps the stack aligned as after a call
        *--top = reinterpret_cast<void*>(&entry);
        for (int i = 0; i < 6; ++i) *--top = nullptr;
        f.sp = top;
    }
    for (bool left = true; left;) {
        left = false;
        for (self = 0; self < n; ++self)
            if (!fibers[self].done) {
                threadIdx = dim3(self);
                host_hip_switch(&sched_sp, fibers[self].sp);
                left |= !fibers[self].done;
            }
    }
}

// ---- dispatch ----------------------------------------------------------------
// Workgroup i of a launch belongs to XCD i mod xcds, which starts its
// workgroups in order, `slots` at a time.  With two launches at once XCD x
// starts those of launch x mod 2 first.
inline int xcds = 4, slots = 2;
struct Launch {
    unsigned grid, block;
    std::function<void()> kernel;
};
inline void run(const std::vector<Launch>& launches) {
    const int nx = xcds;
    std::vector<std::vector<unsigned>> next(launches.size(), std::vector<unsigned>(size_t(nx), 0));
    std::mutex m;
    auto worker = [&](int x) {
        for (;;) {
            const Launch* l = nullptr;
            unsigned b = 0;
            {
                std::lock_guard<std::mutex> g(m);
                for (size_t k = 0; k < launches.size() && !l; ++k) {
                    const size_t i = (size_t(x) + k) % launches.size();
                    b = next[i][size_t(x)] * unsigned(nx) + unsigned(x);
                    if (b < launches[i].grid) {
                        l = &launches[i];
                        ++next[i][size_t(x)];
                    }
                }
            }
            if (!l) return;
            run_block(b, l->grid, l->block, l->kernel);
        }
    };
    std::vector<std::thread> ts;
    for (int w = 0; w < nx * slots; ++w) ts.emplace_back(worker, w % nx);
    for (std::thread& t : ts) t.join();
}
// while set, launches are collected here instead of run
inline std::vector<Launch>* held = nullptr;

// ---- what lanes of a wavefront hand to each other ---------------------------------
template <class T> struct Lanes { static inline thread_local T at[2][1024]; };
template <class T> T* exchange(T v) {   // the wavefront's values by lane
    const long p = fibers[self].waves & 1;
    Lanes<T>::at[p][self] = v;
    wave_barrier();
    return &Lanes<T>::at[p][self / 64 * 64];
}
inline unsigned readlane(unsigned v, int lane) { return exchange(v)[lane]; }
inline int readfirstlane(int v) { return exchange(v)[0]; }

typedef short s4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef double d4 __attribute__((ext_vector_type(4)));
typedef int i4 __attribute__((ext_vector_type(4)));
struct Bf16Ops { s4 a, b; };
struct F64Ops { double a, b; };

// D = A B + C over 16x16x16: lane l holds A[l % 16][4 (l / 16) ..], B[4 (l / 16) ..][l % 16]
// and D[4 (l / 16) ..][l % 16]
inline f4 mfma_16x16x16_bf16(s4 a, s4 b, f4 c, int, int, int) {
    const unsigned l = self % 64;
    const Bf16Ops* o = exchange(Bf16Ops{a, b});
    auto val = [](short x) { return __uint_as_float(uint32_t(uint16_t(x)) << 16); };
    for (unsigned i = 0; i < 4; ++i)
        for (unsigned k = 0; k < 16; ++k)
            c[i] += val(o[16 * (k / 4) + 4 * (l / 16) + i].a[k % 4]) * val(o[16 * (k / 4) + l % 16].b[k % 4]);
    return c;
}
// D = A B + C over 16x16x4: lane l holds A[l % 16][l / 16], B[l / 16][l % 16] and D[l / 16 + 4 e][l % 16]
inline d4 mfma_16x16x4_f64(double a, double b, d4 c, int, int, int) {
    const unsigned l = self % 64;
    const F64Ops* o = exchange(F64Ops{a, b});
    for (unsigned e = 0; e < 4; ++e)
        for (unsigned k = 0; k < 4; ++k) c[e] = std::fma(o[16 * k + l / 16 + 4 * e].a, o[16 * k + l % 16].b, c[e]);
    return c;
}

struct Buffer { char* p; size_t n; };
inline void buffer_store(i4 v, Buffer b, size_t off) {
    if (off + 16 > b.n) std::abort();
    std::memcpy(b.p + off, &v, 16);
}
template <class T> T load(const T* p) { T v; __atomic_load(const_cast<T*>(p), &v, __ATOMIC_SEQ_CST); return v; }
template <class T> void store(T* p, T v) { __atomic_store(p, &v, __ATOMIC_SEQ_CST); }

inline void launch(dim3 grid, dim3 block, std::function<void()> kernel) {
    if (held) held->push_back({grid.x, block.x, kernel});
    else run({{grid.x, block.x, kernel}});
}

}  // namespace host_hip

inline void __syncthreads() { host_hip::block_barrier(); }
inline int atomicAdd(int* p, int v) { return __atomic_fetch_add(p, v, __ATOMIC_SEQ_CST); }
inline int atomicOr(int* p, int v) { return __atomic_fetch_or(p, v, __ATOMIC_SEQ_CST); }
#define __HIP_MEMORY_SCOPE_SYSTEM 5
#define __hip_atomic_load(p, order, scope) host_hip::load(p)
#define __hip_atomic_store(p, v, order, scope) host_hip::store(p, v)
#define __builtin_amdgcn_mfma_f32_16x16x16bf16_1k host_hip::mfma_16x16x16_bf16
#define __builtin_amdgcn_mfma_f64_16x16x4f64 host_hip::mfma_16x16x4_f64
#define __builtin_amdgcn_readlane host_hip::readlane
#define __builtin_amdgcn_readfirstlane host_hip::readfirstlane
#define __builtin_amdgcn_wave_barrier host_hip::wave_barrier
#define __builtin_amdgcn_s_sleep(n) host_hip::poll_pause()
#define __builtin_amdgcn_s_waitcnt(n) host_hip::wait_stores()
#define __builtin_amdgcn_rcp(x) (1.0 / (x))
#define __builtin_amdgcn_make_buffer_rsrc(p, stride, n, flags) host_hip::Buffer{reinterpret_cast<char*>(p), size_t(n)}
#define __builtin_amdgcn_raw_buffer_store_b128(v, b, off, soff, aux) host_hip::buffer_store(v, b, size_t(off))
#define hipLaunchKernelGGL(k, grid, block, lds, stream, ...) host_hip::launch(grid, block, [=] { k(__VA_ARGS__); })
