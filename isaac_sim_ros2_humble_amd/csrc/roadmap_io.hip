// The two ends of a roadmap's life on the device: its start and goal states spread over the arrays, and
// the finished roadmap laid out as the caller reads it.  Both go through host memory that the device
// maps, so each takes one launch (one per megabyte of a large roadmap).  Copied array by array (18 and 17 copies of a few hundred bytes to a
// few KB, 10 to 30 us each) they took most of a small roadmap's time; the figures stand at Storage in
// roadmap.cpp.
#include <hip/hip_runtime.h>

#include "mp_plan.h"

namespace {

__global__ void __launch_bounds__(256) start_kernel(mp::RoadmapStart a) {
    const long long step = (long long)gridDim.x * blockDim.x, t0 = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    for (long long t = t0; t < (long long)a.count * a.dof; t += step) {
        const long long r = t / a.dof, j = t - r * a.dof, v = a.first + r;
        const float x = a.states[t];
        a.node[j * a.vcap + v] = x;
        if (v < a.ns)
            a.gq[0][j * a.vcap + v] = x;
        else
            a.gq[1][j * a.vcap + v - a.ns] = x;
    }
    for (long long v = a.first + t0; v < (long long)a.first + a.count; v += step) {
        a.vgroup[v] = v < a.ns ? 1 : 2;
        if (v < a.ns)
            a.gv[0][v] = (int)v;
        else
            a.gv[1][v - a.ns] = (int)v;
    }
    if (t0 < a.nctl) a.ctl[t0] = a.state[t0];
}

__global__ void __launch_bounds__(256) pack_kernel(mp::RoadmapPack a) {
    const long long step = (long long)gridDim.x * blockDim.x;
    for (long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x; t < a.count; t += step) {
        const long long w = a.first + t;
        unsigned x;
        if (w < a.at[1]) {
            const long long v = w / a.dof, j = w - v * a.dof;
            x = __float_as_uint(a.node[j * a.vcap + v]);
        } else if (w < a.at[2]) {
            x = (unsigned)a.vgroup[w - a.at[1]];
        } else if (w < a.at[3]) {
            const long long e = w - a.at[2];
            x = (unsigned)((e & 1) ? a.eb[e >> 1] : a.ea[e >> 1]);
        } else if (w < a.at[4]) {
            x = __float_as_uint(a.ew[w - a.at[3]]);
        } else {
            x = (unsigned)(w < a.at[5] ? a.gv[0][w - a.at[4]] : a.gv[1][w - a.at[5]]);
        }
        a.out[t] = x;
    }
}

// one thread per element up to a fill of the chip; the loops take the rest
unsigned blocks(long long elements) {
    const long long b = (elements + 255) / 256;
    return (unsigned)(b < 1 ? 1 : (b > 1024 ? 1024 : b));
}

// Launches kernel(a).  The launch's own status is what counts: hipGetLastError also reports what an
// earlier call of the caller's left behind (an allocation that was refused, say).
template <class A>
void launch_one(void (*kernel)(A), A a, long long elements, hipStream_t s) {
    void* args[] = {&a};
    MP_HIP(hipLaunchKernel(reinterpret_cast<const void*>(kernel), dim3(blocks(elements)), dim3(256), args, 0, s));
}

}  // namespace

namespace mp {

void roadmap_start(const RoadmapStart& a, hipStream_t s) {
    launch_one(start_kernel, a, (long long)a.count * a.dof, s);
}

void roadmap_pack(const RoadmapPack& a, hipStream_t s) {
    launch_one(pack_kernel, a, a.count, s);
}

}  // namespace mp
