// Device-resident roadmap planner (the extend-connect loop of CUDAMPLib::RRG::solve,
// cudampl/CUDAMPLib/src/planners/RRG.cpp:241-424): the roadmap's vertices, group members and
// edges live in device memory; every loop pass is three launches on the library stream (sample,
// motions, commit) with no host round trip.  The host keeps a few passes in flight, watches a
// host-mapped copy of the loop state for the solution, and grows the buffers before a pass could
// run out of room.
#include <algorithm>
#include <cstring>
#include <mutex>
#include <vector>

#include "mp_plan.h"

using mp::Error;

namespace {

constexpr int kNctl = 16;      // MP_RM_NCTL
constexpr int kMaxK = 256;     // MP_RM_MAX_K
constexpr int kDepth = 3;      // passes in flight
enum { T = 0, SOLVED = 1, NV = 2, NE = 3, G1 = 4, G2 = 5, PASS = 6, FULL = 7, TRAVEL1 = 8, TRAVEL2 = 9 };

// Host mirror of the kernels' RoadmapDev (layout must match the kernel template).
struct RoadmapDevHost {
    float* node;
    int* vgroup;
    float* gq[2];
    int* gv[2];
    int* ea;
    int* eb;
    float* ew;
    float* smp;
    int* nn;
    unsigned char* ok;
    float* len;
    unsigned char* freed;
    int* ctl;
    int* mirror;
    uint64_t seed, offset;
    int k, vcap, ecap, dof;
    float res, max_travel;
};

int f2i(float f) {
    int i;
    std::memcpy(&i, &f, 4);
    return i;
}
float i2f(int i) {
    float f;
    std::memcpy(&f, &i, 4);
    return f;
}

// What a roadmap lives in: one device allocation with its arrays, one host allocation that the device maps
// (loop state, then the start and goal states or the roadmap being read out) and its events.  Destroyed
// roadmaps leave it to the next one.  With 15 allocations, 18 copies to fill the arrays and 17 to read them,
// a roadmap of three passes (FR3, 60 samples each, 20 spheres) took 135 us to create, 755 us to read (the
// passes' own 150 us among them) and 87 us to destroy; four such from creation to the graph read
// back: 2.50 -> 0.93 ms.
struct Storage {
    int device = -1;
    char* dev = nullptr;
    size_t dev_bytes = 0;
    char* host = nullptr;
    char* host_dev = nullptr;  // the device's address of host
    size_t host_bytes = 0;
    hipEvent_t ev[kDepth] = {};
};
constexpr size_t kStateBytes = 256;             // loop state at the head of the host allocation
constexpr size_t kHostBytes = 256 << 10;        // host allocation of a new roadmap, unless it needs more
constexpr size_t kHostMost = 1 << 20;           // what does not fit this goes through it in pieces
constexpr size_t kKeep = 4, kKeepBytes = 8 << 20;  // storage kept: so many, each allocation up to so large
std::mutex g_mu;                                // guards g_kept
std::vector<Storage> g_kept;

bool smaller(const Storage& a, const Storage& b) {
    return a.dev_bytes != b.dev_bytes ? a.dev_bytes < b.dev_bytes : a.host_bytes < b.host_bytes;
}

void host_alloc(Storage& st, size_t bytes) {
    MP_HIP(hipHostMalloc((void**)&st.host, bytes, hipHostMallocMapped | hipHostMallocCoherent));
    st.host_bytes = bytes;
    MP_HIP(hipHostGetDevicePointer((void**)&st.host_dev, st.host, 0));
}

void free_storage(Storage& st) {
    if (st.dev) hipFree(st.dev);
    if (st.host) hipHostFree(st.host);
    for (auto& e : st.ev)
        if (e) hipEventDestroy(e);
    st = Storage();
}

// The smallest kept storage with room for the sizes, else new.  `st` is the caller's to free also when
// this throws.
void take_storage(Storage& st, size_t dev_bytes, size_t host_bytes) {
    int device = 0;
    MP_HIP(hipGetDevice(&device));
    {
        std::lock_guard<std::mutex> g(g_mu);
        auto best = g_kept.end();
        for (auto it = g_kept.begin(); it != g_kept.end(); ++it)
            if (it->device == device && it->dev_bytes >= dev_bytes && it->host_bytes >= host_bytes &&
                (best == g_kept.end() || smaller(*it, *best)))
                best = it;
        if (best != g_kept.end()) {
            st = *best;
            g_kept.erase(best);
            return;
        }
    }
    st.device = device;
    MP_HIP(hipMalloc((void**)&st.dev, dev_bytes));
    st.dev_bytes = dev_bytes;
    host_alloc(st, std::max(host_bytes, kHostBytes));
    for (auto& e : st.ev) MP_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
}

// Keeps whole storage that no work uses any more (the caller has waited for the stream), in the place of
// the smallest kept when there are enough, or frees it.
void give_back(Storage& st) {
    if (st.dev && st.host_dev && st.ev[kDepth - 1] && st.dev_bytes <= kKeepBytes && st.host_bytes <= kKeepBytes) {
        std::lock_guard<std::mutex> g(g_mu);
        if (g_kept.size() < kKeep) {
            g_kept.push_back(st);
            st = Storage();
        } else {
            auto least = std::min_element(g_kept.begin(), g_kept.end(), smaller);
            if (smaller(*least, st)) std::swap(*least, st);
        }
    }
    free_storage(st);
}

// Bytes of a roadmap's arrays; sets g's pointers into `base` when there is one.  Every array starts at a
// multiple of 256 bytes.
size_t place(RoadmapDevHost& g, char* base, size_t vcap, size_t ecap) {
    size_t at = 0;
    auto put = [&](auto*& p, size_t n) {
        if (base) p = reinterpret_cast<std::remove_reference_t<decltype(p)>>(base + at);
        at += (n * sizeof(*p) + 255) & ~(size_t)255;
    };
    const size_t dof = (size_t)g.dof, k = (size_t)g.k;
    put(g.ctl, kNctl);
    put(g.smp, k * dof);
    put(g.nn, 3 * k);
    put(g.ok, 2 * k);
    put(g.len, 2 * k);
    put(g.freed, k);
    put(g.node, dof * vcap);
    for (int s = 0; s < 2; s++) {
        put(g.gq[s], dof * vcap);
        put(g.gv[s], vcap);
    }
    put(g.vgroup, vcap);
    put(g.ea, ecap);
    put(g.eb, ecap);
    put(g.ew, ecap);
    if (base) {
        g.vcap = (int)vcap;
        g.ecap = (int)ecap;
    }
    return at;
}

}  // namespace

namespace mp {

void roadmap_release_storage() {
    std::lock_guard<std::mutex> g(g_mu);
    for (Storage& st : g_kept) free_storage(st);
    g_kept.clear();
}

}  // namespace mp

struct mp_roadmap {
    mp_robot* robot = nullptr;
    const mp_scene* scene = nullptr;
    RoadmapDevHost g{};
    Storage mem;
    int* mirror_h = nullptr;   // host-mapped loop state: equal to ctl when no pass is in flight
    long long enqueued = 0, completed = 0;  // passes enqueued / known finished
    hipFunction_t f_sample = nullptr, f_edges = nullptr, f_commit = nullptr;

    void grow(int need_v, int need_e);
    void wait_all();
};

void mp_roadmap::wait_all() {
    MP_HIP(hipStreamSynchronize(mp::lib_stream()));
    completed = enqueued;
}

// Doubles the capacities until need_v vertices and need_e edges fit, copying the roadmap (the
// structure-of-arrays rows move to the new stride).
void mp_roadmap::grow(int need_v, int need_e) {
    int vcap = g.vcap, ecap = g.ecap;
    while (vcap < need_v) vcap *= 2;
    while (ecap < need_e) ecap *= 2;
    if (vcap == g.vcap && ecap == g.ecap) return;
    wait_all();
    hipStream_t s = mp::lib_stream();
    const volatile int* ctl = mirror_h;
    const RoadmapDevHost old = g;
    const size_t bytes = place(g, nullptr, vcap, ecap);
    char* block = nullptr;
    MP_HIP(hipMalloc((void**)&block, bytes));
    place(g, block, vcap, ecap);
    char* const old_block = mem.dev;
    mem.dev = block;
    mem.dev_bytes = bytes;
    const int dof = g.dof, nv = ctl[NV], ne = ctl[NE], n1 = ctl[G1], n2 = ctl[G2];
    auto copy = [&](void* to, const void* from, int n) {
        MP_HIP(hipMemcpyAsync(to, from, (size_t)n * 4, hipMemcpyDeviceToDevice, s));
    };
    try {
        copy(g.ctl, old.ctl, kNctl);
        for (int j = 0; j < dof; j++) {
            copy(g.node + (size_t)j * vcap, old.node + (size_t)j * old.vcap, nv);
            copy(g.gq[0] + (size_t)j * vcap, old.gq[0] + (size_t)j * old.vcap, n1);
            copy(g.gq[1] + (size_t)j * vcap, old.gq[1] + (size_t)j * old.vcap, n2);
        }
        copy(g.vgroup, old.vgroup, nv);
        copy(g.gv[0], old.gv[0], n1);
        copy(g.gv[1], old.gv[1], n2);
        copy(g.ea, old.ea, ne);
        copy(g.eb, old.eb, ne);
        copy(g.ew, old.ew, ne);
        MP_HIP(hipStreamSynchronize(s));
    } catch (...) {
        hipStreamSynchronize(s);
        hipFree(old_block);
        throw;
    }
    hipFree(old_block);
}

extern "C" {

int mp_roadmap_create(mp_robot* robot, const mp_scene* scene, const float* starts, int ns, const float* goals, int ng,
                      int samples_per_iteration, float max_travel_distance, float resolution, uint64_t seed,
                      uint64_t sample_offset, mp_roadmap** out) {
    return mp::guard_call([&] {
        if (mp::lib_stream() == nullptr) throw Error(MP_E_STATE, "mp_init() has not been called");
        if (!robot || !scene || !out || ns < 1 || ng < 1 || !starts || !goals) throw Error(MP_E_INVALID, "bad roadmap arguments");
        if (samples_per_iteration < 1 || samples_per_iteration > kMaxK)
            throw Error(MP_E_INVALID, "samples per iteration must be in [1, 256]");
        if (!(max_travel_distance > 0.0f) || !(resolution > 0.0f)) throw Error(MP_E_INVALID, "bad travel distance or resolution");
        auto rm = std::make_unique<mp_roadmap>();
        rm->robot = robot;
        rm->scene = scene;
        const int dof = robot->model.dof;
        RoadmapDevHost& g = rm->g;
        g.dof = dof;
        g.k = samples_per_iteration;
        g.seed = seed;
        g.offset = sample_offset;
        g.res = resolution;
        g.max_travel = max_travel_distance;
        const int nv0 = ns + ng;
        int vcap = 4096;
        while (vcap < nv0 + kDepth * 2 * g.k) vcap *= 2;
        try {
            const size_t row = (size_t)dof * sizeof(float);
            take_storage(rm->mem, place(g, nullptr, vcap, 2 * vcap), std::min(kStateBytes + (size_t)nv0 * row, kHostMost));
            place(g, rm->mem.dev, vcap, 2 * vcap);
            rm->mirror_h = reinterpret_cast<int*>(rm->mem.host);
            g.mirror = reinterpret_cast<int*>(rm->mem.host_dev);
            int ctl[kNctl] = {0};
            ctl[NV] = nv0;
            ctl[G1] = ns;
            ctl[G2] = ng;
            ctl[TRAVEL1] = ctl[TRAVEL2] = f2i(max_travel_distance);
            std::memcpy(rm->mirror_h, ctl, sizeof(ctl));
            // the start and goal states: vertices, and the first members of their groups
            hipStream_t s = mp::lib_stream();
            const int rows = (int)std::min((size_t)nv0, (rm->mem.host_bytes - kStateBytes) / row);
            for (int v = 0; v < nv0; v += rows) {
                const int n = std::min(rows, nv0 - v), n_starts = std::max(0, std::min(n, ns - v));
                char* const states = rm->mem.host + kStateBytes;
                if (v > 0) MP_HIP(hipStreamSynchronize(s));  // the rows before have been read
                if (n_starts > 0) std::memcpy(states, starts + (size_t)v * dof, n_starts * row);
                if (n > n_starts)
                    std::memcpy(states + n_starts * row, goals + (size_t)(v + n_starts - ns) * dof, (n - n_starts) * row);
                mp::roadmap_start({reinterpret_cast<const float*>(rm->mem.host_dev + kStateBytes), g.mirror, g.node,
                                   {g.gq[0], g.gq[1]}, {g.gv[0], g.gv[1]}, g.vgroup, g.ctl, ns, v, n, dof, vcap, kNctl}, s);
            }
            mp::Module& mod = *robot->module;
            rm->f_sample = mod.fn("mp_rm_sample_0");
            rm->f_edges = mod.fn("mp_rm_edges_0");
            rm->f_commit = mod.fn("mp_rm_commit_0");
        } catch (...) {
            mp_roadmap_destroy(rm.release());
            throw;
        }
        *out = rm.release();
    });
}

int mp_roadmap_iterate(mp_roadmap* rm, int* solved) {
    return mp::guard_call([&] {
        if (!rm || !solved) throw Error(MP_E_INVALID, "bad arguments");
        RoadmapDevHost& g = rm->g;
        hipStream_t s = mp::lib_stream();
        if (rm->enqueued - rm->completed >= kDepth) {  // keep at most kDepth passes in flight
            MP_HIP(hipEventSynchronize(rm->mem.ev[rm->completed % kDepth]));
            rm->completed++;
        }
        volatile int* m = rm->mirror_h;
        if (m[SOLVED]) {
            *solved = 1;
            return;
        }
        if (m[FULL]) {  // a pass found no room: grow, then run it again
            rm->wait_all();
            rm->grow(2 * g.vcap, 2 * g.ecap);
            const int zero = 0;
            MP_HIP(hipMemcpy(g.ctl + FULL, &zero, sizeof(int), hipMemcpyHostToDevice));
            m[FULL] = 0;
        }
        // the mirror holds at least every finished pass; the passes in flight and this one add
        // at most k vertices, 2k edges and k members each
        const int pending = (int)(rm->enqueued - rm->completed) + 1;
        const int need_v = std::max(m[NV], std::max(m[G1], m[G2])) + pending * g.k;
        const int need_e = m[NE] + pending * 2 * g.k;
        if (need_v > g.vcap || need_e > g.ecap) rm->grow(need_v, need_e);
        mp::SceneDevHost sv = mp::scene_view(rm->scene);
        unsigned long long* work = mp::lib_work_counter();
        void* a1[] = {&g, &sv};
        void* a2[] = {&g, &sv, &work};
        void* a3[] = {&g};
        mp::launch(rm->f_sample, (unsigned)g.k, 64, s, a1, nullptr);
        mp::launch(rm->f_edges, (unsigned)((2 * g.k + 3) / 4), 256, s, a2, "rrg");
        mp::launch(rm->f_commit, 1, 64, s, a3, nullptr);
        MP_HIP(hipEventRecord(rm->mem.ev[rm->enqueued % kDepth], s));
        rm->enqueued++;
        *solved = 0;
    });
}

int mp_roadmap_info_get(mp_roadmap* rm, mp_roadmap_info* info) {
    return mp::guard_call([&] {
        if (!rm || !info) throw Error(MP_E_INVALID, "bad arguments");
        rm->wait_all();
        const volatile int* c = rm->mirror_h;
        info->solved = c[SOLVED];
        info->passes = c[PASS];
        info->loop_index = c[T];
        info->vertices = c[NV];
        info->edges = c[NE];
        info->start_group = c[G1];
        info->goal_group = c[G2];
        info->travel_start = i2f(c[TRAVEL1]);
        info->travel_goal = i2f(c[TRAVEL2]);
    });
}

int mp_roadmap_read(mp_roadmap* rm, float* vertices, int* groups, int* edges, float* weights, int* start_members,
                    int* goal_members) {
    return mp::guard_call([&] {
        if (!rm) throw Error(MP_E_INVALID, "null roadmap");
        rm->wait_all();
        const RoadmapDevHost& g = rm->g;
        const volatile int* c = rm->mirror_h;
        const size_t nv = (size_t)c[NV], ne = (size_t)c[NE], n1 = (size_t)c[G1], n2 = (size_t)c[G2], dof = (size_t)g.dof;
        void* const to[6] = {vertices, groups, edges, weights, start_members, goal_members};
        const size_t words[6] = {nv * dof, nv, 2 * ne, ne, n1, n2};
        mp::RoadmapPack p{g.node, g.vgroup, g.ea, g.eb, g.ew, {g.gv[0], g.gv[1]}, g.dof, g.vcap, {0}, 0, 0, nullptr};
        for (int i = 0; i < 6; i++) p.at[i + 1] = p.at[i] + (to[i] ? (long long)words[i] : 0);
        const long long total = p.at[6];
        if (kStateBytes + (size_t)total * 4 > rm->mem.host_bytes && rm->mem.host_bytes < kHostMost) {
            Storage more;  // the loop state moves along; without the memory the roadmap goes in smaller pieces
            try {
                host_alloc(more, kHostMost);
                std::memcpy(more.host, rm->mem.host, kStateBytes);
                std::swap(more.host, rm->mem.host);
                std::swap(more.host_dev, rm->mem.host_dev);
                std::swap(more.host_bytes, rm->mem.host_bytes);
                rm->mirror_h = reinterpret_cast<int*>(rm->mem.host);
                rm->g.mirror = reinterpret_cast<int*>(rm->mem.host_dev);
            } catch (const Error&) {
            }
            free_storage(more);
        }
        const long long room = (long long)(rm->mem.host_bytes - kStateBytes) / 4;
        const char* const got = rm->mem.host + kStateBytes;
        p.out = reinterpret_cast<unsigned*>(rm->mem.host_dev + kStateBytes);
        for (p.first = 0; p.first < total; p.first += room) {
            p.count = std::min(room, total - p.first);
            mp::roadmap_pack(p, mp::lib_stream());
            MP_HIP(hipStreamSynchronize(mp::lib_stream()));
            for (int i = 0; i < 6; i++) {
                const long long lo = std::max(p.first, p.at[i]), hi = std::min(p.first + p.count, p.at[i + 1]);
                if (lo < hi) std::memcpy((char*)to[i] + (lo - p.at[i]) * 4, got + (lo - p.first) * 4, (size_t)(hi - lo) * 4);
            }
        }
    });
}

int mp_roadmap_destroy(mp_roadmap* rm) {
    return mp::guard_call([&] {
        if (!rm) return;
        if (mp::lib_stream() && hipStreamSynchronize(mp::lib_stream()) == hipSuccess)
            give_back(rm->mem);
        else
            free_storage(rm->mem);
        delete rm;
    });
}

}  // extern "C"
