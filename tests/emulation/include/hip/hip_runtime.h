// The part of the HIP language and runtime that the library's Fock, gradient,
// one-electron and work-list code uses, on the CPU (see ../../emulator.cpp): the
// blocks of a launch run one after another, the lanes of a block as fibers that
// meet at wavefront operations and barriers.  For tests without a device.
#pragma once
#include <algorithm>
#include <climits>
#include <cmath>
#include <cstddef>
#include <cstdint>
#include <cstring>
#include <functional>

#define __global__
#define __device__
#define __host__
#define __constant__
#define __forceinline__ inline
#define __launch_bounds__(...)
#define __align__(n) __attribute__((aligned(n)))
#define __shared__ static   // one block at a time
#define HIP_SYMBOL(x) (x)

struct int2 { int x, y; };
struct alignas(16) int4 { int x, y, z, w; };
struct alignas(16) uint4 { unsigned x, y, z, w; };
struct alignas(16) double2 { double x, y; };
inline int2 make_int2(int x, int y) { return {x, y}; }
inline int4 make_int4(int x, int y, int z, int w) { return {x, y, z, w}; }
inline uint4 make_uint4(unsigned x, unsigned y, unsigned z, unsigned w) { return {x, y, z, w}; }
struct dim3 {
    unsigned x, y, z;
    dim3(unsigned x_ = 1, unsigned y_ = 1, unsigned z_ = 1) : x(x_), y(y_), z(z_) {}
};

// ---- runtime
enum hipError_t { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorOutOfMemory = 2, hipErrorInvalidDevice = 101,
                  hipErrorLaunchFailure = 719 };
enum hipMemcpyKind { hipMemcpyHostToDevice, hipMemcpyDeviceToHost, hipMemcpyDeviceToDevice };
enum hipFuncAttribute { hipFuncAttributeMaxDynamicSharedMemorySize };
enum { hipStreamNonBlocking = 1, hipEventDisableTiming = 2 };
struct EmuStream;
struct EmuEvent;
using hipStream_t = EmuStream*;
using hipEvent_t = EmuEvent*;
struct hipFuncAttributes { size_t localSizeBytes, sharedSizeBytes; int numRegs; };
struct hipDeviceProp_t {
    char name[256], gcnArchName[256];
    size_t totalGlobalMem;
    int multiProcessorCount, clockRate, major, minor;
};
const char* hipGetErrorString(hipError_t);
hipError_t hipGetLastError();
hipError_t hipMalloc(void** p, size_t n);
template <class T>
hipError_t hipMalloc(T** p, size_t n) { return hipMalloc((void**)p, n); }
hipError_t hipFree(void* p);
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind);
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t);
hipError_t hipGetDeviceCount(int* n);
hipError_t hipGetDevice(int* d);
hipError_t hipSetDevice(int d);
hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int d);
hipError_t hipDeviceSynchronize();
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned flags);
hipError_t hipStreamDestroy(hipStream_t s);
hipError_t hipStreamSynchronize(hipStream_t s);
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned flags);
hipError_t hipEventCreate(hipEvent_t* e);
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned flags);
hipError_t hipEventDestroy(hipEvent_t e);
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s = nullptr);
hipError_t hipEventSynchronize(hipEvent_t e);
hipError_t hipEventElapsedTime(float* ms, hipEvent_t a, hipEvent_t b);
hipError_t hipFuncGetAttributes(hipFuncAttributes* a, const void* f);
hipError_t hipFuncSetAttribute(const void* f, hipFuncAttribute a, int v);
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void* f, int threads, size_t lds);
template <class T>
hipError_t hipGetSymbolAddress(void** p, T& sym) { *p = (void*)&sym; return hipSuccess; }

// ---- launches
namespace emu {
struct Idx { unsigned x, y, z; };
extern Idx g_block, g_thread, g_block_dim, g_grid_dim;
void* dynamic_lds();
// runs `body` for every thread of the grid (kernel: its address, for the record)
void launch(const void* kernel, dim3 grid, dim3 block, size_t lds, hipStream_t s, const std::function<void()>& body);
// what the lanes of the caller's wavefront that reached this operation passed to it
struct Wave {
    uint64_t v[64];
    uint64_t active;   // lanes that take part
};
const Wave& wave_op(uint64_t mine, const char* what);
void block_barrier();
unsigned lane();
template <class T>
uint64_t bits(T v) { uint64_t b = 0; std::memcpy(&b, &v, sizeof(T)); return b; }
template <class T>
T value(uint64_t b) { T v; std::memcpy(&v, &b, sizeof(T)); return v; }
}  // namespace emu
#define blockIdx emu::g_block
#define threadIdx emu::g_thread
#define blockDim emu::g_block_dim
#define gridDim emu::g_grid_dim
template <class... P, class... A>
void emu_launch_kernel(void (*k)(P...), dim3 grid, dim3 block, size_t lds, hipStream_t s, A... a) {
    emu::launch((const void*)k, grid, block, lds, s, [=] { k(a...); });
}
#define hipLaunchKernelGGL(k, grid, block, lds, s, ...) emu_launch_kernel(k, grid, block, lds, s, __VA_ARGS__)

// ---- device functions (g++ leaves names that begin with __builtin_ unmangled)
#define __builtin_amdgcn_fence emu_amdgcn_fence
#define __builtin_amdgcn_ldexp emu_amdgcn_ldexp
#define __builtin_amdgcn_rcp emu_amdgcn_rcp
#define __builtin_amdgcn_rcpf emu_amdgcn_rcpf
#define __builtin_amdgcn_readfirstlane emu_amdgcn_readfirstlane
#define __builtin_amdgcn_rsq emu_amdgcn_rsq
#define __builtin_amdgcn_rsqf emu_amdgcn_rsqf
#define __builtin_amdgcn_update_dpp emu_amdgcn_update_dpp
#define __builtin_amdgcn_wave_barrier emu_amdgcn_wave_barrier
inline void __syncthreads() { emu::block_barrier(); }
template <class T>
T __shfl_xor(T v, int m, int = 64) {
    const emu::Wave& w = emu::wave_op(emu::bits(v), "shfl_xor");
    const unsigned src = emu::lane() ^ m;
    return (w.active >> src) & 1 ? emu::value<T>(w.v[src]) : v;
}
inline unsigned long long __ballot(int p) {
    const emu::Wave& w = emu::wave_op(p != 0, "ballot");
    unsigned long long m = 0;
    for (int l = 0; l < 64; ++l)
        if ((w.active >> l) & 1 && w.v[l]) m |= 1ull << l;
    return m;
}
inline int __any(int p) { return __ballot(p) != 0; }
template <class T>
T emu_amdgcn_readfirstlane(T v) {
    const emu::Wave& w = emu::wave_op(emu::bits(v), "readfirstlane");
    return emu::value<T>(w.v[__builtin_ctzll(w.active)]);
}
inline void emu_amdgcn_wave_barrier() { emu::wave_op(0, "wave_barrier"); }
inline void emu_amdgcn_fence(int, const char*) {}
// the data-parallel moves in use: row_shr:n, row_bcast:15, row_bcast:31
inline int emu_amdgcn_update_dpp(int old, int src, int ctl, int row_mask, int, bool) {
    const emu::Wave& w = emu::wave_op((uint32_t)src, "dpp");
    const int l = (int)emu::lane(), row = l >> 4;
    if (!((row_mask >> row) & 1)) return old;
    int from = -1;
    if (ctl > 0x110 && ctl <= 0x11f) from = (l & 15) >= (ctl & 15) ? l - (ctl & 15) : -1;
    else if (ctl == 0x142) from = row ? 16 * row - 1 : -1;
    else if (ctl == 0x143) from = row >= 2 ? 31 : -1;
    else __builtin_trap();
    return from >= 0 && (w.active >> from) & 1 ? (int)(uint32_t)w.v[from] : old;
}
inline double emu_amdgcn_rcp(double x) { return 1.0 / x; }
inline double emu_amdgcn_rsq(double x) { return 1.0 / std::sqrt(x); }
inline float emu_amdgcn_rcpf(float x) { return 1.0f / x; }
inline float emu_amdgcn_rsqf(float x) { return 1.0f / std::sqrt(x); }
inline double emu_amdgcn_ldexp(double x, int k) { return std::ldexp(x, k); }
inline long long __double2ll_rn(double x) { return (long long)std::nearbyint(x); }
inline int __float2int_rn(float x) { return (int)std::nearbyint(x); }
inline int __float2int_rz(float x) { return (int)x; }
inline int __double2loint(double x) { return (int)(uint32_t)emu::bits(x); }
inline int __double2hiint(double x) { return (int)(uint32_t)(emu::bits(x) >> 32); }
inline double __hiloint2double(int h, int l) { return emu::value<double>((uint64_t)(uint32_t)h << 32 | (uint32_t)l); }
inline int __popcll(unsigned long long x) { return __builtin_popcountll(x); }
inline float __expf(float x) { return std::exp(x); }
inline unsigned long long atomicAdd(unsigned long long* p, unsigned long long v) { const auto o = *p; *p += v; return o; }
inline unsigned long long atomicOr(unsigned long long* p, unsigned long long v) { const auto o = *p; *p |= v; return o; }
inline int min(int a, int b) { return a < b ? a : b; }
inline int max(int a, int b) { return a > b ? a : b; }
