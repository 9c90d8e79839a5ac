// The two ends of a roadmap's life on the device: its start and goal states spread over the arrays, and
// the finished roadmap laid out as the caller reads it.  Both go through host memory that the device
// maps, so each takes one launch.  Copied array by array (18 and 17 copies of a few hundred bytes to a
// few KB, 10 to 30 us each) they took most of a small roadmap's time; the figures stand at Storage in
// roadmap.cpp.
#include <hip/hip_runtime.h>

#include "mp_plan.h"

namespace {

__global__ void __launch_bounds__(256) start_kernel(mp::RoadmapStart a) {
    const long long step = (long long)gridDim.x * blockDim.x, t0 = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    const long long nv = (long long)a.ns + a.ng;
    for (long long t = t0; t < nv * a.dof; t += step) {
        const long long v = t / a.dof, j = t - v * a.dof;
        const float x = a.states[t];
        a.node[j * a.vcap + v] = x;
        if (v < a.ns)
            a.gq[0][j * a.vcap + v] = x;
        else
            a.gq[1][j * a.vcap + v - a.ns] = x;
    }
    for (long long v = t0; v < nv; v += step) {
        a.vgroup[v] = v < a.ns ? 1 : 2;
        if (v < a.ns)
            a.gv[0][v] = (int)v;
        else
            a.gv[1][v - a.ns] = (int)v;
    }
    if (t0 < a.nctl) a.ctl[t0] = a.state[t0];
}

__global__ void __launch_bounds__(256) pack_kernel(mp::RoadmapPack a) {
    const long long step = (long long)gridDim.x * blockDim.x, t0 = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    for (long long t = t0; t < (long long)a.nv * a.dof; t += step) {
        const long long v = t / a.dof, j = t - v * a.dof;
        a.vertices[t] = a.node[j * a.vcap + v];
    }
    for (long long v = t0; v < a.nv; v += step) a.groups[v] = a.vgroup[v];
    for (long long t = t0; t < 2ll * a.ne; t += step) a.edges[t] = (t & 1) ? a.eb[t >> 1] : a.ea[t >> 1];
    for (long long e = t0; e < a.ne; e += step) a.weights[e] = a.ew[e];
    for (int s = 0; s < 2; ++s)
        for (long long i = t0; i < a.n[s]; i += step) a.members[s][i] = a.gv[s][i];
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
    launch_one(start_kernel, a, ((long long)a.ns + a.ng) * a.dof, s);
}

void roadmap_pack(const RoadmapPack& a, hipStream_t s) {
    launch_one(pack_kernel, a, (long long)a.nv * a.dof, s);
}

}  // namespace mp
