// The HIP names that the resident kernels use, for running their source on the
// CPU (tests only): every lane is a fibre, the lanes of a wave meet at each
// cross-lane operation, and a workgroup runs until all its lanes wait, then the
// next one runs.  An adversarial schedule of workgroups, and every buffer
// access checked against its bounds.
#pragma once
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <algorithm>

#define __global__
#define __device__
#define __host__
#define __forceinline__ inline
#define __launch_bounds__(...)
#define __shared__ static thread_local   // a workgroup is a thread

using std::max;
using std::min;
typedef int hipError_t;
typedef void *hipStream_t;

namespace wavefront {
struct Index { unsigned x; };
const Index &thread_index();
extern thread_local Index block;
void workgroup_barrier();
// Meets the wave's other lanes with a value; the values of all lanes.
const int *meet(int value);
void pause();                 // nothing to do until another workgroup has run
[[noreturn]] void fail(const char *what);
inline int lane() { return (int)(thread_index().x & 63u); }
}

#define threadIdx wavefront::thread_index()
#define blockIdx wavefront::block
struct GridDim { unsigned x; };
extern GridDim gridDim;
inline void __syncthreads() { wavefront::workgroup_barrier(); }

inline long long __double_as_longlong(double v) { long long b; memcpy(&b, &v, 8); return b; }
inline double __longlong_as_double(long long b) { double v; memcpy(&v, &b, 8); return v; }
inline int __float_as_int(float v) { int b; memcpy(&b, &v, 4); return b; }
inline unsigned __float_as_uint(float v) { unsigned b; memcpy(&b, &v, 4); return b; }
inline float __int_as_float(int b) { float v; memcpy(&v, &b, 4); return v; }
inline float __uint_as_float(unsigned b) { float v; memcpy(&v, &b, 4); return v; }
inline double __shfl_xor(double v, int, int) { return v; }   // (not used by these kernels)

inline int dpp_source(int lane, int ctrl)   // -1: none
{
    if (ctrl >= 0x111 && ctrl <= 0x11f) return (lane & 15) >= ctrl - 0x110 ? lane - (ctrl - 0x110) : -1;   // row_shr
    if (ctrl == 0x138) return lane - 1;                          // wave_shr:1
    if (ctrl == 0x130) return lane < 63 ? lane + 1 : -1;         // wave_shl:1
    if (ctrl == 0x142) return lane < 16 ? -1 : (lane & ~15) - 1; // row_bcast:15
    if (ctrl == 0x143) return lane < 32 ? -1 : 31;               // row_bcast:31
    wavefront::fail("a DPP control this does not know");
}
inline int __builtin_amdgcn_update_dpp(int old, int v, int ctrl, int rows, int, bool zero)
{
    const int *all = wavefront::meet(v), l = wavefront::lane(), from = dpp_source(l, ctrl);
    if (!(rows >> (l / 16) & 1)) return old;
    return from < 0 ? (zero ? 0 : old) : all[from];
}
inline int __builtin_amdgcn_mov_dpp(int v, int ctrl, int rows, int banks, bool zero)
{
    return __builtin_amdgcn_update_dpp(v, v, ctrl, rows, banks, zero);
}
inline int __builtin_amdgcn_readlane(int v, int lane) { return wavefront::meet(v)[lane]; }
inline int __builtin_amdgcn_readfirstlane(int v) { return wavefront::meet(v)[0]; }
inline bool __all(bool p)
{
    const int *all = wavefront::meet(p);
    return std::all_of(all, all + 64, [](int v) { return v != 0; });
}
inline void __builtin_amdgcn_fence(int, const char *) {}
inline void __builtin_amdgcn_wave_barrier() { wavefront::meet(0); }
inline void __builtin_amdgcn_s_sleep(int) { wavefront::pause(); }
inline long long wall_clock64() { wavefront::pause(); return 0; }

#define __HIP_MEMORY_SCOPE_AGENT 0
#define __HIP_MEMORY_SCOPE_WORKGROUP 0
#define __HIP_MEMORY_SCOPE_SYSTEM 0
#define __hip_atomic_load(p, order, scope) __atomic_load_n(p, order)
#define __hip_atomic_store(p, v, order, scope) __atomic_store_n(p, v, order)
#define __hip_atomic_fetch_add(p, v, order, scope) __atomic_fetch_add(p, v, order)
#define __hip_atomic_compare_exchange_strong(p, expected, v, good, bad, scope) \
    __atomic_compare_exchange_n(p, expected, v, false, good, bad)

// Raw buffers: a lane offset at or beyond the size less the uniform offset reads 0 and writes nothing.
struct __amdgpu_buffer_rsrc_t {
    char *base;
    unsigned bytes;
};
struct Words2 { unsigned w[2]; };
inline __amdgpu_buffer_rsrc_t __builtin_amdgcn_make_buffer_rsrc(void *base, short, int bytes, int)
{
    return {(char *)base, (unsigned)bytes};
}
inline char *buffer_at(const __amdgpu_buffer_rsrc_t &r, int lane_offset, int uniform, unsigned size)
{
    const unsigned long long o = (unsigned)lane_offset, u = (unsigned)uniform;
    if (o + u >= r.bytes) return nullptr;
    if (o + u + size > r.bytes) wavefront::fail("a buffer access across the end");
    return r.base + o + u;
}
inline unsigned __builtin_amdgcn_raw_buffer_load_b32(__amdgpu_buffer_rsrc_t r, int o, int u, int)
{
    unsigned v = 0;
    if (const char *p = buffer_at(r, o, u, 4)) memcpy(&v, p, 4);
    return v;
}
inline Words2 __builtin_amdgcn_raw_buffer_load_b64(__amdgpu_buffer_rsrc_t r, int o, int u, int)
{
    Words2 v{};
    if (const char *p = buffer_at(r, o, u, 8)) memcpy(&v, p, 8);
    return v;
}
inline void __builtin_amdgcn_raw_buffer_store_b32(unsigned v, __amdgpu_buffer_rsrc_t r, int o, int u, int)
{
    if (char *p = buffer_at(r, o, u, 4)) memcpy(p, &v, 4);
}
inline void __builtin_amdgcn_raw_buffer_store_b64(Words2 v, __amdgpu_buffer_rsrc_t r, int o, int u, int)
{
    if (char *p = buffer_at(r, o, u, 8)) memcpy(p, &v, 8);
}
