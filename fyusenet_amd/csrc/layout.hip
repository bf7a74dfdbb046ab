// Layout converters between host buffers and device tensors.
//
// The host side of a transfer is page-locked memory that the kernels read and write in place, over PCIe: conversion and
// transfer are one launch, where a copy into a device buffer followed by a conversion kernel (or the reverse) costs a
// second launch and a round trip through the runtime's copy queue -- 10 us on a small frame.  What bounds them is the
// link (about 55 GB/s each way), so a thread moves sixteen bytes per access and few workgroups are enough: measured on
// 25 MB, 64 to 256 workgroups of such loads 448 us = 55 GB/s, 1024 workgroups 488 us, the copy engine alone 439 us.
// From the host 48 take a frame (below), to the host 128.
// The same kernels serve buffers in device memory.
#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include <algorithm>

#include "kernels.h"
#include "range.h"

namespace fynhip {

namespace {
constexpr unsigned kMaxBlocks = 128;          // buffers behind the link
// Buffers in device memory: few workgroups of 1024 threads.  At a launch's end its workgroups meet in one word (the value range
// of what was uploaded, the host's word), one after the other (15 ns each, twice): 936 workgroups of 256 threads took 26.5
// us for 3.8 MB of interleaved pixels, 78 of 1024 take 8; the result's 5 MB 10 -> 8.6.  A stream of 512x624 frames through
// the sample's style net 2897 -> 2663 us for twelve.
constexpr unsigned kMaxDeviceBlocks = 128;
constexpr int kDeviceThreads = 1024;
// Frames from the host: the workgroups keep pace with the host's copy, and each one's looks at its progress (HostFeed) and
// its arrival at the end cost the others time.  A segmentation frame (3.7 MB) from call to launch complete, with 24, 32,
// 40, 48, 64 and 80 workgroups: 106, 98, 92, 93, 96, 97 us (111 with 128 that ended with a fence each); 25 MB: 566, 492,
// 489, 490, 497, 534.  (Two sizes, one host with a 55 GB/s link: elsewhere the number is a guess; what depends on it is how
// close to the link's rate an upload runs, not what arrives.)
constexpr unsigned kMaxUploadBlocks = 48;
unsigned blocks_for(size_t items, unsigned most, int threads) { return (unsigned)std::min<size_t>(most, (items + threads - 1) / threads); }

// The host may still be copying the frame when the launch runs (HostFeed): before a workgroup reads pixels it looks, where
// it has to, whether they are there.  The launch's own latency (8 us) and the host's copy then overlap the transfer
// instead of preceding it.  Every thread of the workgroup calls this with the workgroup's largest pixel; `seen` holds what
// the last look said.  The wait ends after HostFeed::give_up ticks in any case, and the host is told (FeedWord::late): it
// looks at that word when the frame is complete and has the frame converted again.  It cannot miss it: the word is set
// before the last look at the progress, and looked at behind the last progress.
__device__ __forceinline__ void await_feed(const HostFeed& f, unsigned need, unsigned& seen) {
    if (!f.word || seen >= need) return;   // (the same for all threads)
    __shared__ unsigned box;
    if (threadIdx.x == 0) {
        const unsigned long long t0 = wall_clock64();
        unsigned r;
        while ((int)((r = __hip_atomic_load(&f.word->ready, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_SYSTEM) - f.base) - need) < 0) {
            if (wall_clock64() - t0 >= f.give_up) {
                __hip_atomic_store(&f.word->late, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // (also before the workgroup counts as arrived, below)
                __threadfence_system();
                r = __hip_atomic_load(&f.word->ready, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_SYSTEM) - f.base;
                if ((int)(r - need) < 0) r = 0x7fffffffu;
                break;
            }
            // (not before the host can have come so far: a look takes the word's line from the core that is copying, and
            // the link from the copy; 1.3 us at least)
            const unsigned long long t1 = wall_clock64(), ticks = min(10000u, 130u + (unsigned)((float)(need - r) * f.ticks_per_pixel));
            while (wall_clock64() - t1 < ticks) __builtin_amdgcn_s_sleep(8);
        }
        box = r;
    }
    __syncthreads();
    seen = box;
    __syncthreads();
}

// The value range of an uploaded tensor.  Its record is written, not raised, so that no launch has to clear it first: the
// workgroups meet in a word of the network's (device scope: they sit on different XCDs), and the one that arrives last
// moves the maximum into the record and leaves the words as they were found.
template <int NT>
__device__ __forceinline__ void publish_range(const UploadRange& u, float m) {
    if (!u.record) return;
    __shared__ float wave_max[NT / 64];
    __shared__ unsigned last;
    m = range_wave_max(m);
    if ((threadIdx.x & 63) == 0) wave_max[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
        for (int w = 0; w < NT / 64; w++) m = fmaxf(m, wave_max[w]);
        (void)__hip_atomic_fetch_max(&u.words[0], __float_as_uint(m), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // (the maximum has been taken before the arrival counts)
        unsigned all = 0u;
        if (__hip_atomic_fetch_add(&u.words[1], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == gridDim.x - 1) {
            all = __hip_atomic_exchange(&u.words[0], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) | 0x80000000u;   // (the sign bit marks the last workgroup)
            __hip_atomic_store(&u.words[1], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        last = all;
    }
    __syncthreads();
    if (last && threadIdx.x < RANGE_SLOTS) u.record[threadIdx.x * RANGE_STRIDE] = threadIdx.x == 0 ? last & 0x7fffffffu : 0u;
}

// Stores of the workgroup's threads, then -- by the workgroup that arrives last -- the host's word: when the host reads
// `value` there, everything the launch has written lies in memory.  A host that polls the word sees the result 5 us
// earlier than one that waits for the stream (10.8 against 5.9 us around an empty kernel), because the stream's
// completion signal is a packet of its own behind the kernel.
__device__ __forceinline__ void tell_host(const HostDone& d) {
    if (!d.flag) return;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0) {
        __threadfence_system();
        if (__hip_atomic_fetch_add(d.counter, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) == gridDim.x - 1) {
            __hip_atomic_store(d.counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);   // for the next launch on this stream
            __threadfence_system();
            __hip_atomic_store(d.flag, d.value, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
        }
    }
}

// The same for a launch that has read the host's memory.  What it tells is that nothing reads it any more, so nothing has to
// be made visible first: the fence above is a write-back, 0.2 us for every workgroup and one after the other.
__device__ __forceinline__ void tell_host_read(const HostDone& d) {
    if (!d.flag) return;
    __syncthreads();   // (the values read have all been used)
    if (threadIdx.x == 0 && __hip_atomic_fetch_add(d.counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == gridDim.x - 1) {
        __hip_atomic_store(d.counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __hip_atomic_store(d.flag, d.value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

template <typename T>
__device__ __forceinline__ float4 load4(const T* p) {
    if constexpr (sizeof(T) == 2) {
        typedef _Float16 h4 __attribute__((ext_vector_type(4)));
        const h4 h = *reinterpret_cast<const h4*>(p);
        return make_float4((float)h[0], (float)h[1], (float)h[2], (float)h[3]);
    } else {
        return *reinterpret_cast<const float4*>(p);
    }
}
template <typename T>
__device__ __forceinline__ void store4(T* p, float a, float b, float c, float d) {
    if constexpr (sizeof(T) == 2) {
        typedef _Float16 h4 __attribute__((ext_vector_type(4)));
        h4 h;
        h[0] = (_Float16)a; h[1] = (_Float16)b; h[2] = (_Float16)c; h[3] = (_Float16)d;
        *reinterpret_cast<h4*>(p) = h;
    } else {
        *reinterpret_cast<float4*>(p) = make_float4(a, b, c, d);
    }
}
}  // namespace

// Planes `plane` floats apart (a multiple of four, as is the planes' address in units of four floats): a thread takes four
// pixels of four channels.  Channels beyond the tensor's read as zero.
template <typename T, int NT>
__global__ __launch_bounds__(NT) void chw_to_tensor_kernel(const float* chw, size_t plane, const TView t, const UploadRange range, const HostFeed feed, const HostDone done) {
    const unsigned npix = (unsigned)t.h * t.w, quads = (npix + 3) >> 2;
    const size_t n = (size_t)quads * (t.cp >> 2);
    float vmax = 0.f;
    unsigned seen = 0;
    for (size_t i0 = (size_t)blockIdx.x * NT; i0 < n; i0 += (size_t)gridDim.x * NT) {
        const unsigned q0 = (unsigned)(i0 % quads);
        await_feed(feed, q0 + NT >= quads ? npix : (q0 + NT) * 4, seen);
        const size_t i = i0 + threadIdx.x;
        if (i >= n) break;
        const unsigned pix = (unsigned)(i % quads) * 4;
        const int c = (int)(i / quads) * 4;
        float4 v[4];
#pragma unroll
        for (int k = 0; k < 4; k++) v[k] = c + k < t.c ? *reinterpret_cast<const float4*>(chw + (size_t)(c + k) * plane + pix) : make_float4(0.f, 0.f, 0.f, 0.f);
        unsigned y = pix / (unsigned)t.w, x = pix - y * (unsigned)t.w;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            if (pix + j < npix) {
                float e[4];
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    e[k] = j == 0 ? v[k].x : j == 1 ? v[k].y : j == 2 ? v[k].z : v[k].w;
                    vmax = fmaxf(vmax, fabsf(e[k]));
                }
                store4<T>(reinterpret_cast<T*>(t.ptr) + ((size_t)(y + t.pad) * t.wp() + x + t.pad) * t.cp + c, e[0], e[1], e[2], e[3]);
            }
            if (++x == (unsigned)t.w) {
                x = 0;
                y++;
            }
        }
    }
    publish_range<NT>(range, vmax);
    tell_host_read(done);
}
void launch_chw_to_tensor(const float* chw, size_t plane, const TView& t, const UploadRange& range, const HostFeed& feed, const HostDone& done, bool device, hipStream_t s) {
    const size_t items = ((size_t)t.h * t.w + 3) / 4 * (t.cp >> 2);
    auto go = [&](auto kernel, unsigned most, int threads) {
        hipLaunchKernelGGL(kernel, dim3(blocks_for(items, most, threads)), dim3(threads), 0, s, chw, plane, t, range, feed, done);
    };
    if (device && t.f16) go(chw_to_tensor_kernel<_Float16, kDeviceThreads>, kMaxDeviceBlocks, kDeviceThreads);
    else if (device) go(chw_to_tensor_kernel<float, kDeviceThreads>, kMaxDeviceBlocks, kDeviceThreads);
    else if (t.f16) go(chw_to_tensor_kernel<_Float16, 256>, kMaxUploadBlocks, 256);
    else go(chw_to_tensor_kernel<float, 256>, kMaxUploadBlocks, 256);
}

// Interleaved pixels of t.c floats: the buffer is read as one run of sixteen-byte pieces (an element's pixel and channel
// follow from its index), the tensor's pad channels keep the zeros they were allocated with.  The last piece may reach
// up to three floats behind the buffer's end.
template <typename T, int NT>
__global__ __launch_bounds__(NT) void hwc_to_tensor_kernel(const float* hwc, const TView t, const UploadRange range, const HostFeed feed, const HostDone done) {
    const size_t npix = (size_t)t.h * t.w, e1 = npix * t.c, q1 = (e1 + 3) >> 2;
    float vmax = 0.f;
    unsigned seen = 0;
    for (size_t q0 = (size_t)blockIdx.x * NT; q0 < q1; q0 += (size_t)gridDim.x * NT) {
        await_feed(feed, q0 + NT >= q1 ? (unsigned)npix : (unsigned)((q0 + NT) * 4 / t.c + 1), seen);
        const size_t q = q0 + threadIdx.x;
        if (q >= q1) break;
        const float4 v = *reinterpret_cast<const float4*>(hwc + q * 4);
        const float e[4] = {v.x, v.y, v.z, v.w};
        unsigned pix = (unsigned)(q * 4 / t.c), c = (unsigned)(q * 4 - (size_t)pix * t.c);
        unsigned y = pix / (unsigned)t.w, x = pix - y * (unsigned)t.w;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            if (q * 4 + k < e1) {
                reinterpret_cast<T*>(t.ptr)[((size_t)(y + t.pad) * t.wp() + x + t.pad) * t.cp + c] = (T)e[k];
                vmax = fmaxf(vmax, fabsf(e[k]));
            }
            if (++c == (unsigned)t.c) {
                c = 0;
                if (++x == (unsigned)t.w) {
                    x = 0;
                    y++;
                }
            }
        }
    }
    publish_range<NT>(range, vmax);
    tell_host_read(done);
}
// The same for images of three channels in device memory: a thread takes four pixels, three loads and four whole-pixel
// stores of sixteen bytes (fp32 tensors), instead of one load and four stores of a channel each.
template <typename T>
__global__ __launch_bounds__(kDeviceThreads) void hwc3_to_tensor_kernel(const float* hwc, const TView t, const UploadRange range, const HostDone done) {
    const unsigned npix = (unsigned)t.h * t.w, quads = (npix + 3) >> 2;
    float vmax = 0.f;
    for (unsigned q = blockIdx.x * kDeviceThreads + threadIdx.x; q < quads; q += gridDim.x * kDeviceThreads) {
        float e[12];
#pragma unroll
        for (int k = 0; k < 3; k++) {
            // (the last pixels' piece: no further behind the buffer's end than the kernel above reads)
            const bool there = (size_t)q * 12 + k * 4 < (size_t)npix * 3;
            const float4 v = there ? *reinterpret_cast<const float4*>(hwc + (size_t)q * 12 + k * 4) : make_float4(0.f, 0.f, 0.f, 0.f);
            e[4 * k] = v.x; e[4 * k + 1] = v.y; e[4 * k + 2] = v.z; e[4 * k + 3] = v.w;
        }
        unsigned y = q * 4 / (unsigned)t.w, x = q * 4 - y * (unsigned)t.w;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            if (q * 4 + j < npix) {
                store4<T>(reinterpret_cast<T*>(t.ptr) + ((size_t)(y + t.pad) * t.wp() + x + t.pad) * 4, e[3 * j], e[3 * j + 1], e[3 * j + 2], 0.f);
                vmax = fmaxf(fmaxf(vmax, fabsf(e[3 * j])), fmaxf(fabsf(e[3 * j + 1]), fabsf(e[3 * j + 2])));
            }
            if (++x == (unsigned)t.w) {
                x = 0;
                y++;
            }
        }
    }
    publish_range<kDeviceThreads>(range, vmax);
    tell_host_read(done);
}
void launch_hwc_to_tensor(const float* hwc, const TView& t, const UploadRange& range, const HostFeed& feed, const HostDone& done, bool device, hipStream_t s) {
    const size_t items = ((size_t)t.h * t.w * t.c + 3) / 4;
    auto go = [&](auto kernel, unsigned most, int threads) {
        hipLaunchKernelGGL(kernel, dim3(blocks_for(items, most, threads)), dim3(threads), 0, s, hwc, t, range, feed, done);
    };
    if (device && t.c == 3 && t.cp == 4) {
        const dim3 grid(blocks_for(((size_t)t.h * t.w + 3) / 4, kMaxDeviceBlocks, kDeviceThreads));
        if (t.f16) hipLaunchKernelGGL(hwc3_to_tensor_kernel<_Float16>, grid, dim3(kDeviceThreads), 0, s, hwc, t, range, done);
        else hipLaunchKernelGGL(hwc3_to_tensor_kernel<float>, grid, dim3(kDeviceThreads), 0, s, hwc, t, range, done);
    } else if (device && t.f16) go(hwc_to_tensor_kernel<_Float16, kDeviceThreads>, kMaxDeviceBlocks, kDeviceThreads);
    else if (device) go(hwc_to_tensor_kernel<float, kDeviceThreads>, kMaxDeviceBlocks, kDeviceThreads);
    else if (t.f16) go(hwc_to_tensor_kernel<_Float16, 256>, kMaxUploadBlocks, 256);
    else go(hwc_to_tensor_kernel<float, 256>, kMaxUploadBlocks, 256);
}

// Pixels [p0, p1) of the net area (keep_pad: of the area with its halo) to planes `plane` floats apart.  Q = 4: a thread
// takes four pixels of four channels, planes on sixteen-byte boundaries (p0 a multiple of four, the last piece may
// reach up to three floats behind a plane); Q = 1: one pixel of four channels, any planes.
template <typename T, int Q>
__global__ __launch_bounds__(kDeviceThreads) void tensor_to_chw_kernel(const TView t, float* chw, size_t plane, int keep_pad, unsigned p0, unsigned p1, const HostDone done) {
    const unsigned ow = (unsigned)(keep_pad ? t.wp() : t.w);
    const int off = keep_pad ? 0 : t.pad;
    const unsigned groups = (p1 - p0 + Q - 1) / Q;
    const size_t n = (size_t)groups * ((t.c + 3) >> 2);
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
        const unsigned pix = p0 + (unsigned)(i % groups) * Q;
        const int c = (int)(i / groups) * 4;
        unsigned y = pix / ow, x = pix - y * ow;
        float4 v[Q];
#pragma unroll
        for (int j = 0; j < Q; j++) {
            v[j] = pix + j < p1 ? load4<T>(reinterpret_cast<const T*>(t.ptr) + ((size_t)(y + off) * t.wp() + x + off) * t.cp + c) : make_float4(0.f, 0.f, 0.f, 0.f);
            if (++x == ow) {
                x = 0;
                y++;
            }
        }
#pragma unroll
        for (int k = 0; k < 4; k++) {
            float e[Q];
#pragma unroll
            for (int j = 0; j < Q; j++) e[j] = k == 0 ? v[j].x : k == 1 ? v[j].y : k == 2 ? v[j].z : v[j].w;
            if (c + k < t.c) {
                float* dst = chw + (size_t)(c + k) * plane + pix;
                if constexpr (Q == 4) *reinterpret_cast<float4*>(dst) = make_float4(e[0], e[1], e[2], e[3]);
                else *dst = e[0];
            }
        }
    }
    tell_host(done);
}
// All planes of a small or odd area, one behind the other without gaps: the buffer is written as one run of sixteen-byte
// pieces, whatever planes they fall into (46 KB in planes of 36 floats, one float per store: 14 us; this way 4).
template <typename T>
__global__ __launch_bounds__(256) void tensor_to_run_kernel(const TView t, float* chw, unsigned npix, int keep_pad, const HostDone done) {
    const unsigned ow = (unsigned)(keep_pad ? t.wp() : t.w);
    const int off = keep_pad ? 0 : t.pad;
    const size_t n = (size_t)npix * t.c;
    for (size_t i = ((size_t)blockIdx.x * 256 + threadIdx.x) * 4; i < n; i += (size_t)gridDim.x * 1024) {
        unsigned c = (unsigned)(i / npix), pix = (unsigned)(i - (size_t)c * npix);
        unsigned y = pix / ow, x = pix - y * ow;
        float e[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k = 0; k < 4; k++) {
            if (i + k < n) e[k] = (float)reinterpret_cast<const T*>(t.ptr)[((size_t)(y + off) * t.wp() + x + off) * t.cp + c];
            if (++x == ow) {
                x = 0;
                y++;
            }
            if (++pix == npix) {
                pix = x = y = 0;
                c++;
            }
        }
        if (i + 4 <= n) *reinterpret_cast<float4*>(chw + i) = make_float4(e[0], e[1], e[2], e[3]);
        else
            for (int k = 0; i + k < n; k++) chw[i + k] = e[k];
    }
    tell_host(done);
}
void launch_tensor_to_chw(const TView& t, float* chw, size_t plane, int include_padding, size_t p0, size_t p1, const HostDone& done, bool device, hipStream_t s) {
    const size_t npix = include_padding ? (size_t)t.hp() * t.wp() : (size_t)t.h * t.w;
    if (plane == npix && p0 == 0 && p1 == npix && (plane % 4 != 0 || plane < 256) && (reinterpret_cast<size_t>(chw) & 15) == 0 && t.c > 1) {
        const dim3 grid((unsigned)std::min<size_t>(kMaxBlocks, ((npix * t.c + 3) / 4 + 255) / 256));
        if (t.f16) hipLaunchKernelGGL(tensor_to_run_kernel<_Float16>, grid, dim3(256), 0, s, t, chw, (unsigned)npix, include_padding, done);
        else hipLaunchKernelGGL(tensor_to_run_kernel<float>, grid, dim3(256), 0, s, t, chw, (unsigned)npix, include_padding, done);
        return;
    }
    const bool quad = plane % 4 == 0 && (reinterpret_cast<size_t>(chw) & 15) == 0 && p0 % 4 == 0;
    const size_t items = (p1 - p0 + (quad ? 3 : 0)) / (quad ? 4 : 1) * ((t.c + 3) >> 2);
    const int threads = device ? kDeviceThreads : 256;
    const dim3 grid(blocks_for(items, device ? kMaxDeviceBlocks : kMaxBlocks, threads));
    const unsigned a = (unsigned)p0, b = (unsigned)p1;
    if (t.f16) {
        if (quad) hipLaunchKernelGGL((tensor_to_chw_kernel<_Float16, 4>), grid, dim3(threads), 0, s, t, chw, plane, include_padding, a, b, done);
        else hipLaunchKernelGGL((tensor_to_chw_kernel<_Float16, 1>), grid, dim3(threads), 0, s, t, chw, plane, include_padding, a, b, done);
    } else {
        if (quad) hipLaunchKernelGGL((tensor_to_chw_kernel<float, 4>), grid, dim3(threads), 0, s, t, chw, plane, include_padding, a, b, done);
        else hipLaunchKernelGGL((tensor_to_chw_kernel<float, 1>), grid, dim3(threads), 0, s, t, chw, plane, include_padding, a, b, done);
    }
}

// Interleaved pixels of PC = 1, 2 or 4 floats: a pixel per thread, one store each.
template <typename T, int PC>
__global__ __launch_bounds__(kDeviceThreads) void tensor_to_hwc_kernel(const TView t, float* hwc, size_t p0, size_t p1, const HostDone done) {
    for (size_t pix = p0 + (size_t)blockIdx.x * blockDim.x + threadIdx.x; pix < p1; pix += (size_t)gridDim.x * blockDim.x) {
        const unsigned y = (unsigned)pix / (unsigned)t.w, x = (unsigned)pix - y * (unsigned)t.w;
        const float4 v = load4<T>(reinterpret_cast<const T*>(t.ptr) + ((size_t)(y + t.pad) * t.wp() + x + t.pad) * t.cp);
        if constexpr (PC == 4) *reinterpret_cast<float4*>(hwc + pix * 4) = make_float4(v.x, v.y, v.z, t.c > 3 ? v.w : 0.f);
        else if constexpr (PC == 2) *reinterpret_cast<float2*>(hwc + pix * 2) = make_float2(v.x, v.y);
        else hwc[pix] = v.x;
    }
    tell_host(done);
}
template <typename T>
static void launch_hwc_out(const TView& t, float* hwc, int pc, size_t p0, size_t p1, const HostDone& done, bool device, hipStream_t s) {
    const int threads = device ? kDeviceThreads : 256;
    const dim3 grid(blocks_for(p1 - p0, device ? kMaxDeviceBlocks : kMaxBlocks, threads));
    if (pc == 4) hipLaunchKernelGGL((tensor_to_hwc_kernel<T, 4>), grid, dim3(threads), 0, s, t, hwc, p0, p1, done);
    else if (pc == 2) hipLaunchKernelGGL((tensor_to_hwc_kernel<T, 2>), grid, dim3(threads), 0, s, t, hwc, p0, p1, done);
    else hipLaunchKernelGGL((tensor_to_hwc_kernel<T, 1>), grid, dim3(threads), 0, s, t, hwc, p0, p1, done);
}
void launch_tensor_to_hwc(const TView& t, float* hwc, int pc, size_t p0, size_t p1, const HostDone& done, bool device, hipStream_t s) {
    if (t.f16) launch_hwc_out<_Float16>(t, hwc, pc, p0, p1, done, device, s);
    else launch_hwc_out<float>(t, hwc, pc, p0, p1, done, device, s);
}

// An arg-max layer's two results: the exact indices it keeps beside its tensor, and the tensor's second channel.
template <typename T>
__global__ __launch_bounds__(256) void argmax_to_host_kernel(const int* idx, const TView t, int* idx_out, float* val_out, size_t p0, size_t p1, const HostDone done) {
    for (size_t pix = p0 + (size_t)blockIdx.x * 256 + threadIdx.x; pix < p1; pix += (size_t)gridDim.x * 256) {
        const unsigned y = (unsigned)pix / (unsigned)t.w, x = (unsigned)pix - y * (unsigned)t.w;
        if (idx_out) idx_out[pix] = idx[pix];
        if (val_out) val_out[pix] = (float)reinterpret_cast<const T*>(t.ptr)[((size_t)(y + t.pad) * t.wp() + x + t.pad) * t.cp + 1];
    }
    tell_host(done);
}
void launch_argmax_to_host(const int* idx, const TView& t, int* idx_out, float* val_out, size_t p0, size_t p1, const HostDone& done, hipStream_t s) {
    const dim3 grid((unsigned)std::min<size_t>(kMaxBlocks, (p1 - p0 + 255) / 256));
    if (t.f16) hipLaunchKernelGGL(argmax_to_host_kernel<_Float16>, grid, dim3(256), 0, s, idx, t, idx_out, val_out, p0, p1, done);
    else hipLaunchKernelGGL(argmax_to_host_kernel<float>, grid, dim3(256), 0, s, idx, t, idx_out, val_out, p0, p1, done);
}

__global__ void await_feed_kernel(const HostFeed feed, unsigned npix) {
    unsigned seen = 0;
    await_feed(feed, npix, seen);
}
void launch_await_feed(const HostFeed& feed, size_t npix, hipStream_t s) { hipLaunchKernelGGL(await_feed_kernel, dim3(1), dim3(64), 0, s, feed, (unsigned)npix); }

__global__ void tell_host_kernel(const HostDone done) { tell_host(done); }
void launch_tell_host(const HostDone& done, hipStream_t s) { hipLaunchKernelGGL(tell_host_kernel, dim3(1), dim3(64), 0, s, done); }

__global__ __launch_bounds__(256) void fill_zero_kernel(uint4* p, size_t n16, unsigned char* tail, size_t ntail) {
    const size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;
    const size_t stride = (size_t)gridDim.x * 256;
    for (size_t i = idx; i < n16; i += stride) p[i] = make_uint4(0, 0, 0, 0);
    if (idx < ntail) tail[idx] = 0;
}
void launch_fill_zero(void* ptr, size_t bytes, hipStream_t s) {
    const size_t n16 = bytes / 16;
    size_t blocks = (n16 + 255) / 256;
    if (blocks > 4096) blocks = 4096;
    if (blocks == 0) blocks = 1;
    hipLaunchKernelGGL(fill_zero_kernel, dim3((unsigned)blocks), dim3(256), 0, s, reinterpret_cast<uint4*>(ptr), n16,
                       reinterpret_cast<unsigned char*>(ptr) + n16 * 16, bytes - n16 * 16);
}

}  // namespace fynhip
