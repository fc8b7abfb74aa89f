// ekg_engine.cpp -- host side of the plain and batched simulation paths:
// heart upload, excitation-sequence driver, ECG layout, batch planning and
// the kernel launch sequence.  All validation happens here, before any
// launch, so that every kernel runs on extents it was sized for.
#include "ekg_engine.hpp"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <numeric>
#include <type_traits>
#include <unordered_map>

namespace ekg {

// Default launch shape of the matrix-core path (measured on MI355X at 128^3 x
// 256 requests: 128-voxel chunks in 2-wave blocks keep eight blocks per CU;
// larger blocks leave waves idle in the transition tiles while holding LDS).
constexpr int DEFAULT_CHUNK = 128;
constexpr int DEFAULT_WAVES = 2;


[[noreturn]] void fail(int code, const std::string& msg) { throw Error{code, msg}; }

void hip_check(hipError_t e, const char* what)
{
    if (e != hipSuccess) fail(EKG_EDEVICE, std::string(what) + ": " + hipGetErrorString(e));
}

void DevBuf::reserve(size_t n)
{
    if (n <= bytes) return;
    release();
    if (n == 0) return;
    void* q = nullptr;
    hipError_t e = hipMalloc(&q, n);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        fail(EKG_ENOMEM, "device allocation of " + std::to_string(n) + " bytes failed: " +
                             hipGetErrorString(e));
    }
    p = q;
    bytes = n;
}

void DevBuf::adopt(void* q, size_t n)
{
    release();
    p = q;
    bytes = n;
    owned = false;
}

void DevBuf::release()
{
    if (p && owned) (void)hipFree(p);
    p = nullptr;
    bytes = 0;
    owned = true;
}

void Workspace::need(DevBuf& b, size_t n)
{
    if (!arena) {
        // grow by at least half the current size: a workspace that serves
        // groups of varying size reallocates (and synchronises the device
        // in hipFree) a few times, not at every larger group
        if (n > b.bytes) b.reserve(std::max(n, b.bytes + b.bytes / 2));
        return;
    }
    const size_t at = (arena_used + 255) & ~(size_t)255;
    if (at > arena_bytes || n > arena_bytes - at) full();
    b.adopt(arena + at, n);
    arena_used = at + n;
}

void Workspace::full() const
{
    fail(EKG_ENOMEM, "the group needs more than the " + std::to_string(arena_bytes >> 20) +
                             " MiB static device workspace of the allocation-free entry point; use fewer "
                             "requests per call or ekg_simulate_batch_device");
}

void Ctx::bind() const { hip_check(hipSetDevice(device), "hipSetDevice"); }

Workspace::~Workspace()
{
    if (graph) (void)hipGraphExecDestroy(graph);
    if (side) {
        (void)hipStreamSynchronize(side);
        (void)hipStreamDestroy(side);
    }
    if (ev_fork) (void)hipEventDestroy(ev_fork);
    if (ev_join) (void)hipEventDestroy(ev_join);
}

void Workspace::ensure_side()
{
    if (side) return;
    hip_check(hipStreamCreateWithFlags(&side, hipStreamNonBlocking), "hipStreamCreate");
    hip_check(hipEventCreateWithFlags(&ev_fork, hipEventDisableTiming), "hipEventCreate");
    hip_check(hipEventCreateWithFlags(&ev_join, hipEventDisableTiming), "hipEventCreate");
}

hipEvent_t Ctx::get_event()
{
    if (!free_events.empty()) {
        hipEvent_t e = free_events.back();
        free_events.pop_back();
        return e;
    }
    hipEvent_t e;
    hip_check(hipEventCreate(&e), "hipEventCreate");
    return e;
}

void Ctx::collect_timings()
{
    for (auto& pr : pending) {
        hip_check(hipEventSynchronize(pr.second), "hipEventSynchronize");
        float ms = 0.f;
        hip_check(hipEventElapsedTime(&ms, pr.first, pr.second), "hipEventElapsedTime");
        fused_ms += ms;
        fused_launches += pr.counts;
        free_events.push_back(pr.first);
        free_events.push_back(pr.second);
    }
    pending.clear();
}

// Neighbourhood::create + callbacks (simulator.h:325-390): offsets in the
// order of active over {0,1,2}^3 with active[0] outermost.
int nhood_offsets(int type, int8_t dif[26][3])
{
    int n = 0;
    for (int a0 = 0; a0 < 3; ++a0)
        for (int a1 = 0; a1 < 3; ++a1)
            for (int a2 = 0; a2 < 3; ++a2) {
                const int d0 = std::abs(a0 - 1), d1 = std::abs(a1 - 1), d2 = std::abs(a2 - 1);
                const int mn12 = std::min(d1, d2), mx12 = std::max(d1, d2);
                const int mn = std::min(d0, mn12), mx = std::max(d0, mx12);
                bool take = false;
                switch (type) {
                case EKG_NHOOD_2D4: take = mn12 == 1 && mx12 == 1 && d0 == 0; break;
                case EKG_NHOOD_2D8: take = mx12 == 1 && d0 == 0; break;
                case EKG_NHOOD_3D4: take = mn == 1 && mx == 1; break;
                case EKG_NHOOD_3D8: take = mx == 1; break;
                default: return -1;
                }
                if (take) {
                    dif[n][0] = (int8_t)(a0 - 1);
                    dif[n][1] = (int8_t)(a1 - 1);
                    dif[n][2] = (int8_t)(a2 - 1);
                    ++n;
                }
            }
    return n;
}

int64_t num_steps(double length, double dt)
{
    if (!(dt > 0) || !std::isfinite(dt) || !std::isfinite(length) || length <= 0) return 0;
    const double s = std::ceil(length / dt);  // simulator.cpp:470
    if (!(s < 1e9)) return -1;
    return (int64_t)s;
}

// Iterations of the neighbour loop `for (simTime = start; simTime < start +
// length; simTime += dt)` (simulator.cpp:481, 519).  It can differ from T
// for steps like 1/3; samples at or beyond it receive no dipole.
static int64_t neighbour_steps(double start, double length, double dt, int64_t cap)
{
    const double total = length + start;
    int64_t n = 0;
    for (double st = start; st < total; st += dt) {
        if (++n > cap) break;
    }
    return n;
}

ReqSpec make_spec(Heart& h, const ekg_sim_desc& d, bool host_values)
{
    ReqSpec r;
    r.h = &h;
    r.L = d.n_leads;
    r.nl = d.n_layers;
    r.nhood = d.nhood;
    r.start = d.start;
    r.length = d.length;
    r.dt = d.dt;
    if (r.L < 1 || r.L > EKG_MAX_LEADS)
        fail(EKG_EINVAL, "n_leads must be in 1.." + std::to_string(EKG_MAX_LEADS));
    if (r.nhood < EKG_NHOOD_2D4 || r.nhood > EKG_NHOOD_3D8)
        fail(EKG_EINVAL, "unknown neighbourhood (only know of these: 2D4, 3D4, 2D8, 3D8 (cube))");
    if (r.nl < h.max_layer || r.nl < 1 || r.nl > 255)
        fail(EKG_EINVAL, "the heart has " + std::to_string(h.max_layer) + " layers but " +
                             std::to_string(r.nl) + " layer APs were given");
    if (!(r.dt > 0) || !std::isfinite(r.dt) || !std::isfinite(r.start) || !std::isfinite(r.length))
        fail(EKG_EINVAL, "time step must be positive and times finite");
    r.T = num_steps(r.length, r.dt);
    if (r.T < 0 || r.T > (1 << 24)) fail(EKG_EINVAL, "too many time steps");
    r.Tp = std::max<int64_t>(64, ((r.T + 63) / 64) * 64);
    r.n_tiles = (int)(r.Tp / 64);
    r.Tn = neighbour_steps(r.start, r.length, r.dt, r.T + 1);
    if (r.Tn > r.T)
        fail(EKG_EINVAL, "time step makes the neighbour loop of the reference run past the "
                         "sample buffer (simulator.cpp:519); choose another time step");
    if (host_values) {
        if (!d.layer_k || !d.lead_pos) fail(EKG_EINVAL, "layer_k and lead_pos are required");
        for (int i = 0; i < 9 * r.nl; ++i)
            if (!std::isfinite(d.layer_k[i])) fail(EKG_EINVAL, "non-finite AP coefficient");
        for (int i = 0; i < 3 * r.L; ++i)
            if (!std::isfinite(d.lead_pos[i])) fail(EKG_EINVAL, "non-finite lead position");
        r.k = d.layer_k;
        r.pos = d.lead_pos;
    }
    return r;
}

bool heart_mfma(const Ctx& ctx, const Heart& h)
{
    int kernel = h.tune_kernel ? h.tune_kernel : ctx.kernel;
    if (ctx.kernel != EKG_KERNEL_AUTO) kernel = ctx.kernel;  // as in plan_group
    return kernel != EKG_KERNEL_VALU;
}

GroupPlan plan_group(Ctx& ctx, std::vector<ReqSpec> reqs)
{
    if (reqs.empty()) fail(EKG_EINVAL, "empty group");
    GroupPlan g;
    g.nhood = reqs[0].nhood;
    int L = 1, kernel = ctx.kernel, waves = 0, phase = 0;
    const bool path0 = heart_mfma(ctx, *reqs[0].h);
    for (const ReqSpec& r : reqs) {
        if (r.nhood != g.nhood) fail(EKG_EINVAL, "all requests of a launch group must share the neighbourhood");
        // each heart's layout is the one of its own contraction path
        if (heart_mfma(ctx, *r.h) != path0)
            fail(EKG_EINVAL, "all requests of a launch group must take the same contraction path");
        L = std::max(L, r.L);
        if (r.h->tune_kernel) kernel = r.h->tune_kernel;
        if (r.h->tune_waves) waves = std::max(waves, r.h->tune_waves);
        if (r.h->tune_phase && !phase) phase = r.h->tune_phase;
    }
    if (ctx.kernel != EKG_KERNEL_AUTO) kernel = ctx.kernel;  // an explicit context choice wins
    g.LP = L <= 4 ? 4 : L <= 8 ? 8 : L <= 12 ? 12 : 16;
    g.mfma = kernel != EKG_KERNEL_VALU;
    g.waves = waves ? waves : DEFAULT_WAVES;
    g.lf_phase = phase ? phase : 2;
    g.reqs = std::move(reqs);
    return g;
}

// Largest activation-time span inside one chunk (ms).  The saturated AP path
// scales exponentials by e^{(k4+k5)(a - t_ref)} per voxel; a bounded span
// keeps that factor far from FP32 overflow for any realistic k4, k5.
constexpr double CHUNK_SPAN_MS = 16.0;
// Smallest activation class by default: a run of at least this many voxels of
// one layer with one activation time takes the class path.
constexpr int DEFAULT_CLASS_MIN = 64;
// Largest class chunk (voxels): a class is kept as a run of class chunks
// (layout bookkeeping; the class-box kernel takes whole classes).
constexpr int64_t CLASS_CHUNK = 4096;
// Windows of six classes and pieces of 1024 groups of 16 window entries: the
// units in which layout_info states a layout's size, and the fixed workspace
// its share of class sums.
constexpr int CLASS_WINDOW = 6;
constexpr int64_t CLASS_PIECE = 1024;
// Class boxes: 4 x 8 x 8 cells (z, y, x) in four sub-bricks of 4^3.
constexpr int BOX_Z = 4, BOX_Y = 8, BOX_X = 8;
constexpr int CB_SLOTS = ekgk::CB_SLOTS;
constexpr int LONG_RANGES = 512;        // chunks from which the reduction sums in parts
constexpr size_t BOX_CLASSES = 64;  // classes of one listing of a box (16 tiles)
// Most bytes of class sums per launch; a larger group runs its rows in
// several launches.
constexpr int64_t GSUM_BYTES = (int64_t)256 << 20;
constexpr int64_t LINE_BYTES = 16 * 8;

namespace {
// Chunk size: DEFAULT_CHUNK voxels unless the heart is tuned.  Chunks are
// layer-pure and span at most CHUNK_SPAN_MS of activation time.
int64_t chunk_target_of(const Heart& h) { return h.tune_chunk ? h.tune_chunk : DEFAULT_CHUNK; }
// Activation classes (matrix-core path only): runs of one layer and one
// activation time with at least this many voxels (0: none).
int class_min_of(const Heart& h, bool mfma)
{
    return (!mfma || h.tune_class < 0) ? 0 : (h.tune_class > 0 ? h.tune_class : DEFAULT_CLASS_MIN);
}
}  // namespace

bool layout_ready(const Heart& h, bool mfma, int nhood)
{
    const EcgLayout& L = h.layout;
    if (!(h.excited && L.valid && L.chunk_target == chunk_target_of(h) && L.class_min == class_min_of(h, mfma)))
        return false;
    return !mfma || (nhood >= 0 && nhood < 4 && L.cells_built[nhood]);
}

void ensure_layout(Heart& h, bool mfma)
{
    if (!h.excited) fail(EKG_ESTATE, "excitation sequence not computed or loaded");
    EcgLayout& L = h.layout;
    const int64_t target = chunk_target_of(h);
    const int cmin = class_min_of(h, mfma);
    if (L.valid && L.chunk_target == target && L.class_min == cmin) return;
    // The layout's device buffers are rewritten in place: kernels still
    // reading the old layout on any stream (a server's slots) finish first.
    if (L.valid) {
        h.ctx->bind();
        hip_check(hipDeviceSynchronize(), "hipDeviceSynchronize");
    }
    L.valid = false;
    std::vector<int64_t> idx;
    idx.reserve(h.n_myo);
    for (int64_t i = 0; i < h.nvox; ++i)
        if (h.h_layer[i]) idx.push_back(i);
    std::stable_sort(idx.begin(), idx.end(), [&](int64_t a, int64_t b) {
        if (h.h_layer[a] != h.h_layer[b]) return h.h_layer[a] < h.h_layer[b];
        return h.h_act[a] < h.h_act[b];
    });
    const int64_t V = (int64_t)idx.size();
    L.V = V;
    L.max_layer = h.max_layer;
    L.a_last = 0.0;
    for (int64_t i : idx) L.a_last = std::max(L.a_last, h.h_act[i]);
    L.h_chunks.clear();
    L.h_cchunks.clear();
    L.h_classes.clear();
    L.h_class_a.clear();
    L.chunk_target = (int)target;
    L.class_min = cmin;
    for (bool& b : L.cells_built) b = false;
    // reference time of layer l: its earliest activation time, rounded to FP32
    L.h_layer_t0.assign(h.max_layer + 1, 0.0);
    std::vector<int64_t> order;  // the layout's voxel order
    order.reserve(V);
    auto tbits_of = [](double a) {
        const float t = (float)a;
        int b;
        std::memcpy(&b, &t, 4);
        return b;
    };
    int64_t v = 0;
    while (v < V) {
        const int lay = h.h_layer[idx[v]];
        int64_t e = v;
        while (e < V && h.h_layer[idx[e]] == lay) ++e;
        L.h_layer_t0[lay] = (double)(float)h.h_act[idx[v]];
        // voxels outside classes first, then the classes' runs
        std::vector<std::pair<int64_t, int64_t>> runs;
        const int64_t m0 = (int64_t)order.size();
        for (int64_t s0 = v; s0 < e;) {
            int64_t s1 = s0 + 1;
            while (s1 < e && h.h_act[idx[s1]] == h.h_act[idx[s0]]) ++s1;
            if (cmin > 0 && s1 - s0 >= cmin)
                runs.push_back({s0, s1});
            else
                order.insert(order.end(), idx.begin() + s0, idx.begin() + s1);
            s0 = s1;
        }
        const int64_t m1 = (int64_t)order.size();
        // chunks: k near-equal pieces of at most `target`, each further cut
        // where the activation span would exceed CHUNK_SPAN_MS
        const int64_t n = m1 - m0;
        const int64_t k = (n + target - 1) / target;
        for (int64_t c = 0; c < k; ++c) {
            int64_t b0 = m0 + n * c / k;
            const int64_t b1 = m0 + n * (c + 1) / k;
            while (b0 < b1) {
                const float tref = (float)h.h_act[order[b0]];
                int64_t b2 = b0 + 1;
                while (b2 < b1 && h.h_act[order[b2]] - (double)tref <= CHUNK_SPAN_MS) ++b2;
                L.h_chunks.push_back(int4{lay, (int)b0, (int)b2, tbits_of(h.h_act[order[b0]])});
                b0 = b2;
            }
        }
        // class chunks: near-equal pieces of at most CLASS_CHUNK per class
        for (const auto& rr : runs) {
            const int64_t c0 = (int64_t)order.size(), nc = rr.second - rr.first;
            order.insert(order.end(), idx.begin() + rr.first, idx.begin() + rr.second);
            const int64_t kc = (nc + CLASS_CHUNK - 1) / CLASS_CHUNK;
            const int first = (int)L.h_cchunks.size();
            const double a = h.h_act[idx[rr.first]];
            for (int64_t c = 0; c < kc; ++c)
                L.h_cchunks.push_back(int4{lay, (int)(c0 + nc * c / kc), (int)(c0 + nc * (c + 1) / kc), tbits_of(a)});
            L.h_classes.push_back(int4{lay, first, (int)L.h_cchunks.size(), 0});
            L.h_class_a.push_back(a);
        }
        v = e;
    }
    idx.swap(order);
    L.n_chunks = (int)L.h_chunks.size();
    L.n_cchunks = (int)L.h_cchunks.size();
    L.n_classes = (int)L.h_classes.size();
    // chunks of layer l: [layer_chunk[l], layer_chunk[l+1])
    L.h_layer_chunk.assign(h.max_layer + 2, L.n_chunks);
    for (int c = L.n_chunks - 1; c >= 0; --c) L.h_layer_chunk[L.h_chunks[c].x] = c;
    L.h_layer_chunk[0] = 0;
    for (int l = h.max_layer; l >= 1; --l)
        if (L.h_layer_chunk[l] > L.h_layer_chunk[l + 1]) L.h_layer_chunk[l] = L.h_layer_chunk[l + 1];
    // per sorted voxel: chunk index and activation time (FP64 and hi/lo FP32)
    std::vector<int> vchunk(V ? V : 1);
    for (int c = 0; c < L.n_chunks; ++c)
        for (int v2 = L.h_chunks[c].y; v2 < L.h_chunks[c].z; ++v2) vchunk[v2] = c;
    std::vector<double> a64(V ? V : 1);
    std::vector<float2> af(V ? V : 1);
    std::vector<uint2> geo(V ? V : 1);
    if (h.n0 > 1024 || h.n1 > 1024 || h.n2 > 1024) fail(EKG_EINVAL, "grid dimensions above 1024");
    for (int64_t i = 0; i < V; ++i) {
        const double a = h.h_act[idx[i]];
        a64[i] = a;
        const float hi = (float)a;
        af[i] = float2{hi, (float)(a - (double)hi)};
        // grid coordinates and the 3x3x3 myocardium mask of the voxel
        const int64_t x = idx[i];
        const int i2 = (int)(x % h.n2);
        const int i1 = (int)((x / h.n2) % h.n1), i0 = (int)(x / ((int64_t)h.n2 * h.n1));
        uint32_t mask = 0;
        for (int d0 = -1; d0 <= 1; ++d0)
            for (int d1 = -1; d1 <= 1; ++d1)
                for (int d2 = -1; d2 <= 1; ++d2) {
                    const int z = i0 + d0, y = i1 + d1, xx = i2 + d2;
                    if (z < 0 || z >= h.n0 || y < 0 || y >= h.n1 || xx < 0 || xx >= h.n2) continue;
                    if (h.h_layer[((int64_t)z * h.n1 + y) * h.n2 + xx])
                        mask |= 1u << ((d0 + 1) * 9 + (d1 + 1) * 3 + (d2 + 1));
                }
        geo[i] = make_uint2((uint32_t)i0 | ((uint32_t)i1 << 10) | ((uint32_t)i2 << 20), mask);
    }
    // 8^3 bricks of the grid that hold myocardium, with their voxels
    // {sorted index, local cell} grouped by brick (counting sort)
    const int nb0 = (h.n0 + 7) / 8, nb1 = (h.n1 + 7) / 8, nb2 = (h.n2 + 7) / 8;
    std::vector<int> cnt((size_t)nb0 * nb1 * nb2 + 1, 0);
    std::vector<int> vbrick(V ? V : 1);
    for (int64_t i = 0; i < V; ++i) {
        const int64_t x = idx[i];
        const int i2 = (int)(x % h.n2);
        const int64_t r = x / h.n2;
        const int i1 = (int)(r % h.n1), i0 = (int)(r / h.n1);
        vbrick[i] = ((i0 / 8) * nb1 + i1 / 8) * nb2 + i2 / 8;
        ++cnt[vbrick[i]];
    }
    std::vector<int4> bricks;
    std::vector<int> boff;
    std::vector<int> bslot(cnt.size(), -1);
    for (int bq = 0; bq < nb0 * nb1 * nb2; ++bq)
        if (cnt[bq]) {
            bslot[bq] = (int)bricks.size();
            bricks.push_back(int4{(bq / (nb1 * nb2)) * 8, ((bq / nb2) % nb1) * 8, (bq % nb2) * 8, 0});
        }
    boff.assign(bricks.size() + 1, 0);
    for (int bq = 0; bq < nb0 * nb1 * nb2; ++bq)
        if (cnt[bq]) boff[bslot[bq] + 1] = cnt[bq];
    for (size_t q = 1; q < boff.size(); ++q) boff[q] += boff[q - 1];
    std::vector<int2> bvox(V ? V : 1);
    std::vector<int> fill(boff.begin(), boff.end() - 1);
    for (int64_t i = 0; i < V; ++i) {
        const int64_t x = idx[i];
        const int i2 = (int)(x % h.n2);
        const int64_t r = x / h.n2;
        const int i1 = (int)(r % h.n1), i0 = (int)(r / h.n1);
        const int cell = ((i0 % 8) * 8 + (i1 % 8)) * 8 + (i2 % 8);
        bvox[fill[bslot[vbrick[i]]]++] = int2{(int)i, cell};
    }
    // cell order inside each brick: a wave's stencil gathers then touch
    // neighbouring LDS words (few bank conflicts)
    for (size_t q = 0; q + 1 < boff.size(); ++q)
        std::sort(bvox.begin() + boff[q], bvox.begin() + boff[q + 1],
                  [](const int2& x, const int2& y) { return x.y < y.y; });
    L.n_bricks = (int)bricks.size();
    // myocardial cells of each brick's 10^3 box (brick + 1-voxel halo)
    std::vector<int> hoff(bricks.size() + 1, 0);
    std::vector<uint16_t> hcells;
    for (size_t q = 0; q < bricks.size(); ++q) {
        const int4 bq = bricks[q];
        for (int c = 0; c < 1000; ++c) {
            const int gz = bq.x - 1 + c / 100, gy = bq.y - 1 + (c / 10) % 10, gx = bq.z - 1 + c % 10;
            if (gz < 0 || gz >= h.n0 || gy < 0 || gy >= h.n1 || gx < 0 || gx >= h.n2) continue;
            if (h.h_layer[((int64_t)gz * h.n1 + gy) * h.n2 + gx]) hcells.push_back((uint16_t)c);
        }
        hoff[q + 1] = (int)hcells.size();
    }
    if (hcells.empty()) hcells.push_back(0);
    h.ctx->bind();
    L.vox_chunk.reserve(vchunk.size() * sizeof(int));
    L.bricks.reserve(std::max<size_t>(1, bricks.size()) * sizeof(int4));
    L.brick_off.reserve(boff.size() * sizeof(int));
    L.brick_vox.reserve(bvox.size() * sizeof(int2));
    L.vox_a64.reserve(a64.size() * sizeof(double));
    L.vox_a.reserve(af.size() * sizeof(float2));
    L.vox_geo.reserve(geo.size() * sizeof(uint2));
    L.chunks.reserve(std::max<size_t>(1, L.h_chunks.size()) * sizeof(int4));
    hip_check(hipMemcpy(L.vox_chunk.p, vchunk.data(), vchunk.size() * sizeof(int), hipMemcpyHostToDevice),
              "upload voxel chunks");
    if (!bricks.empty())
        hip_check(hipMemcpy(L.bricks.p, bricks.data(), bricks.size() * sizeof(int4), hipMemcpyHostToDevice),
                  "upload bricks");
    hip_check(hipMemcpy(L.brick_off.p, boff.data(), boff.size() * sizeof(int), hipMemcpyHostToDevice),
              "upload brick offsets");
    hip_check(hipMemcpy(L.brick_vox.p, bvox.data(), bvox.size() * sizeof(int2), hipMemcpyHostToDevice),
              "upload brick voxels");
    L.halo_off.reserve(hoff.size() * sizeof(int));
    L.halo_cells.reserve(hcells.size() * sizeof(uint16_t));
    hip_check(hipMemcpy(L.halo_off.p, hoff.data(), hoff.size() * sizeof(int), hipMemcpyHostToDevice),
              "upload halo offsets");
    hip_check(hipMemcpy(L.halo_cells.p, hcells.data(), hcells.size() * sizeof(uint16_t),
                        hipMemcpyHostToDevice),
              "upload halo cells");
    hip_check(hipMemcpy(L.vox_a64.p, a64.data(), a64.size() * sizeof(double), hipMemcpyHostToDevice),
              "upload activation times");
    hip_check(hipMemcpy(L.vox_a.p, af.data(), af.size() * sizeof(float2), hipMemcpyHostToDevice),
              "upload activation times");
    hip_check(hipMemcpy(L.vox_geo.p, geo.data(), geo.size() * sizeof(uint2), hipMemcpyHostToDevice),
              "upload voxel geometry");
    L.h_geo.swap(geo);
    if (!L.h_chunks.empty())
        hip_check(hipMemcpy(L.chunks.p, L.h_chunks.data(), L.h_chunks.size() * sizeof(int4),
                            hipMemcpyHostToDevice),
                  "upload chunks");
    L.classes.reserve(std::max<size_t>(1, L.h_classes.size()) * sizeof(int4));
    L.class_a.reserve(std::max<size_t>(1, L.h_class_a.size()) * sizeof(double));
    if (!L.h_cchunks.empty()) {
        hip_check(hipMemcpy(L.classes.p, L.h_classes.data(), L.h_classes.size() * sizeof(int4),
                            hipMemcpyHostToDevice),
                  "upload classes");
        hip_check(hipMemcpy(L.class_a.p, L.h_class_a.data(), L.h_class_a.size() * sizeof(double),
                            hipMemcpyHostToDevice),
                  "upload class times");
    }
    L.layer_chunk.reserve(L.h_layer_chunk.size() * sizeof(int));
    L.layer_t0.reserve(L.h_layer_t0.size() * sizeof(double));
    hip_check(hipMemcpy(L.layer_chunk.p, L.h_layer_chunk.data(), L.h_layer_chunk.size() * sizeof(int),
                        hipMemcpyHostToDevice),
              "upload layer chunks");
    hip_check(hipMemcpy(L.layer_t0.p, L.h_layer_t0.data(), L.h_layer_t0.size() * sizeof(double),
                        hipMemcpyHostToDevice),
              "upload layer times");
    ekgk::HeartDev& d = L.dev;
    d.grid_layer = h.d_layer.as<uint8_t>();
    d.bricks = L.bricks.as<int4>();
    d.brick_off = L.brick_off.as<int>();
    d.brick_vox = L.brick_vox.as<int2>();
    d.halo_off = L.halo_off.as<int>();
    d.halo_cells = L.halo_cells.as<uint16_t>();
    d.vox_chunk = L.vox_chunk.as<int>();
    d.vox_a64 = L.vox_a64.as<double>();
    d.vox_a = L.vox_a.as<float2>();
    d.vox_geo = L.vox_geo.as<uint2>();
    d.chunks = L.chunks.as<int4>();
    d.layer_chunk = L.layer_chunk.as<int>();
    d.layer_t0 = L.layer_t0.as<double>();
    d.classes = L.classes.as<int4>();
    d.class_a = L.class_a.as<double>();
    d.n0 = h.n0;
    d.n1 = h.n1;
    d.n2 = h.n2;
    d.V = (int)V;
    d.n_chunks = L.n_chunks;
    d.n_bricks = L.n_bricks;
    d.max_layer = h.max_layer;
    d.n_classes = L.n_classes;
    L.valid = true;
}

// The sum of the G rows of a set of voxels S, regrouped by cell: a voxel u
// contributes m(u) . s_u (s_u = sum of the d in N with u + d myocardial) and
// m(u + d) . d for each such d, so
//   sum_{u in S} G(u) = sum_w m(w) . D(w),
//   D(w) = [w in S] s_w + sum_{d in N, w - d in S, w myocardial} d,
// an integer vector per cell; cells inside S cancel (D = 0).  With S an
// activation class, every voxel of S has the same AP, so the class needs only
// this sum; a cell w has grid coordinates + 1 (the reference's voxel centre)
// c(w), D(w) and its moment K(w) = -D(w) . c(w), all integers.
//
// The class-box kernel evaluates a cell's weight once and adds it to every
// class with a non-zero D there.  Layout, per neighbourhood:
//  * The cells are taken in boxes of 4 x 8 x 8 (aligned in the grid, in Morton
//    order), each in four sub-bricks of 4^3 cells.
//  * A box's classes, in order, are cut into tiles of 4; for each sub-brick with
//    cells of a tile's classes there is one coefficient block, the int8 operand of
//    v_mfma_i32_16x16x64_i8: lane 16 z + 4 class + coefficient, byte 4 y + x holds
//    D_z, D_y, D_x or K = -D . (c - c0) of the cell, c0 the box's first cell
//    (|D| <= 9 and, for any set of neighbours, |K| <= 93).  The kernel
//    feeds each byte of a weight less 128, so a tile's accumulators start at 128
//    times the sum of their coefficients.
//  * Consecutive boxes form regions, whose class sums a block keeps in LDS: at
//    most CB_SLOTS classes, or on hearts with many classes to a box CB_SLOTS for each
//    of 2 parts or CB_SLOTS4 of 4 that the waves divide (class_cut); a box with more classes is
//    listed again with the rest.  With parts, a box is listed once a part, with the
//    part's classes.
//    Each (region, class) has a line of sums, listed per class in order.
// The cut depends on the heart only, so a request's ECG does not depend on
// the batch it runs in.
namespace {

// Parts of a region's classes, and its boxes, from the mean number of classes of a box.
// With few classes to a box a region holds boxes enough for its block's four
// waves, each for all of the classes.  With many, one or two boxes fill the region's
// slots, which leaves waves idle and a line of sums for almost every class of a
// box; so the waves divide the classes, and the region holds as many times the
// classes.  In two parts each wave forms the weights of its boxes, so a box's weights
// are formed twice; in four all waves take the same box and share its weights.  Measured on
// integer-delay hearts, us for 1 / 64 / 256 requests of 12 leads and 64 steps:
//   classes a box   1 part                 2 parts              4 parts
//   112^3, 27       100 / 330 / 1,165       89 / 368 / 1,288     87 / 401 / 1,358
//   112^3, 37       100 / 482 / 1,786      100 / 422 / 1,474     94 / 460 / 1,663
//   144^3, 43       145 / 1,245 / 4,816    123 / 795 / 2,909    113 / 925 / 3,330
//   112^3, 62       120 / 1,151 / 4,426    119 / 691 / 2,432    114 / 666 / 2,393
//   144^3, 73       201 / 3,710 / 14,434   161 / 1,568 / 5,981  147 / 1,421 / 5,301
// (34 classes at 144^3: 124 / 889 / - in one part, 104 / 758 / - in two).  Larger
// regions have fewer lines, smaller ones more blocks for a lone request: 80^3 with
// 50 classes a box and two parts, 92 / 281 / 921 us with 8 boxes, 92 / 277 / 898 with 12,
// 98 / 267 / 830 with 16; 112^3 with 78 and four parts 125 / 900 / 3,334 with 4, 125 / 872 /
// 3,116 with 8, 140 / 916 / 3,292 with 16.
struct Cut {
    int split, boxes;
};

Cut class_cut(int64_t pairs, int64_t boxes)
{
    if (pairs <= 33 * boxes) return {1, (int)std::min<int64_t>(64, std::max<int64_t>(4, (boxes / 64 + 3) / 4 * 4))};
    if (pairs <= 60 * boxes) return {2, (int)std::min<int64_t>(16, std::max<int64_t>(12, boxes / 192))};
    return {4, 8};
}

}  // namespace

void ensure_cells(Heart& h, int nhood)
{
    EcgLayout& L = h.layout;
    if (nhood < 0 || nhood > 3) fail(EKG_EINVAL, "unknown neighbourhood");
    if (L.cells_built[nhood]) return;
    int8_t dif[26][3];
    const int nd = nhood_offsets(nhood, dif);
    // cell -> index among the current class's cells (-1: none): a dense array
    // over the grid, or a hash map for grids above 2^27 cells (the array would
    // exceed 512 MB)
    const bool dense = h.nvox <= ((int64_t)1 << 27);
    std::vector<int64_t> touched;   // cells of the current class, first-touch order
    std::vector<int> acc;           // D per touched cell, three ints
    std::vector<int> tslot(dense && L.n_classes > 0 ? (size_t)h.nvox : 0, -1);
    std::unordered_map<int64_t, int> tslot_map;
    struct Rec {  // a cell with a non-zero D for a class
        int box, cls;
        uint8_t cell;  // 64 sub-brick + 16 z + 4 y + x within the box
        int8_t d[3];
    };
    std::vector<Rec> recs;
    const int nb1 = (h.n1 + BOX_Y - 1) / BOX_Y, nb2 = (h.n2 + BOX_X - 1) / BOX_X;
    std::vector<int64_t> box_begin((size_t)((h.n0 + BOX_Z - 1) / BOX_Z) * nb1 * nb2 + 1, 0);
    auto bit = [](int d0, int d1, int d2) { return (d0 + 1) * 9 + (d1 + 1) * 3 + (d2 + 1); };
    auto add = [&](int z, int y, int x, int d0, int d1, int d2) {
        const int64_t gi = ((int64_t)z * h.n1 + y) * h.n2 + x;
        int sl;
        if (dense) {
            sl = tslot[gi];
            if (sl < 0) sl = tslot[gi] = (int)touched.size();
        } else {
            sl = tslot_map.emplace(gi, (int)touched.size()).first->second;
        }
        if (sl == (int)touched.size()) {
            touched.push_back(gi);
            acc.insert(acc.end(), {0, 0, 0});
        }
        acc[3 * sl] += d0;
        acc[3 * sl + 1] += d1;
        acc[3 * sl + 2] += d2;
    };
    for (int k = 0; k < L.n_classes; ++k) {
        // the class's voxels: those of its class chunks, which are consecutive
        const int4 cl = L.h_classes[k];
        const int v_begin = L.h_cchunks[cl.y].y, v_end = L.h_cchunks[cl.z - 1].z;
        touched.clear();
        acc.clear();
        for (int v = v_begin; v < v_end; ++v) {
            const uint2 g = L.h_geo[v];
            const int z = (int)(g.x & 1023u), y = (int)((g.x >> 10) & 1023u), x = (int)(g.x >> 20);
            int s0 = 0, s1 = 0, s2 = 0;
            for (int q = 0; q < nd; ++q) {
                if (!((g.y >> bit(dif[q][0], dif[q][1], dif[q][2])) & 1u)) continue;
                add(z + dif[q][0], y + dif[q][1], x + dif[q][2], dif[q][0], dif[q][1], dif[q][2]);
                s0 += dif[q][0];
                s1 += dif[q][1];
                s2 += dif[q][2];
            }
            add(z, y, x, s0, s1, s2);
        }
        tslot_map.clear();
        for (size_t t = 0; t < touched.size(); ++t) {
            const int64_t gi = touched[t];
            if (dense) tslot[gi] = -1;
            const int D0 = acc[3 * t], D1 = acc[3 * t + 1], D2 = acc[3 * t + 2];
            if (!(D0 || D1 || D2)) continue;
            if (std::abs(D0) > 9 || std::abs(D1) > 9 || std::abs(D2) > 9) fail(EKG_EINVAL, "dipole vector out of range");
            const int x = (int)(gi % h.n2), y = (int)((gi / h.n2) % h.n1), z = (int)(gi / ((int64_t)h.n2 * h.n1));
            const int box = ((z / BOX_Z) * nb1 + y / BOX_Y) * nb2 + x / BOX_X;
            const int sub = 2 * ((y / 4) & 1) + ((x / 4) & 1);
            recs.push_back(Rec{box, k, (uint8_t)(64 * sub + 16 * (z & 3) + 4 * (y & 3) + (x & 3)),
                               {(int8_t)D0, (int8_t)D1, (int8_t)D2}});
            ++box_begin[box + 1];
        }
    }
    // records by box, each box's by class (counting sort, stable)
    std::vector<std::pair<uint64_t, int>> order;  // used boxes in Morton order
    for (size_t q = 0; q + 1 < box_begin.size(); ++q) {
        if (box_begin[q + 1]) {
            const uint32_t bx = (uint32_t)(q % nb2), by = (uint32_t)((q / nb2) % nb1), bz = (uint32_t)(q / nb2 / nb1);
            uint64_t code = 0;
            for (int i = 0; i < 12; ++i)
                code |= (uint64_t)((bx >> i) & 1) << (3 * i + 1) | (uint64_t)((by >> i) & 1) << (3 * i + 2) |
                        (uint64_t)((bz >> (i + 1)) & 1) << (3 * i + 3);
            order.push_back({code | (bz & 1), (int)q});
        }
        box_begin[q + 1] += box_begin[q];
    }
    std::sort(order.begin(), order.end());
    std::vector<Rec> sorted(recs.size());
    {
        std::vector<int64_t> at(box_begin.begin(), box_begin.end() - 1);
        for (const Rec& r : recs) sorted[at[r.box]++] = r;
        std::vector<Rec>().swap(recs);
    }
    int64_t n_entries = 0;
    std::vector<int64_t> win_entries((L.n_classes + CLASS_WINDOW - 1) / CLASS_WINDOW, 0);
    std::vector<int4> regions, ext;           // ext: a region's first and last cells + 1 per axis
    int n_box = 0;                            // listed boxes
    std::vector<int4> pkt;                    // 64 per listed box: its tiles' records, its own
    std::vector<int> init;                    // 256 per listed box: 16 per tile
    std::vector<int8_t> coef;                 // 1024 per block
    std::vector<uint64_t> mask;               // 4 per listed box
    std::vector<std::pair<int, int>> lines;   // (class, line)
    // A region's classes are divided over `split` parts with CB_SLOTS (or CB_SLOTS4) slots each:
    // wave w of a block adds the classes of part w % split, of every
    // (CB_WAVES / split)-th box.
    int64_t pairs = 0;  // (box, class)
    for (size_t q = 0; q < sorted.size(); ++q)
        pairs += q == 0 || sorted[q].box != sorted[q - 1].box || sorted[q].cls != sorted[q - 1].cls;
    const Cut cut = class_cut(pairs, (int64_t)order.size());
    const int split = cut.split, target = cut.boxes;
    const int groups = ekgk::CB_WAVES / split;
    const int slots_part = split == 4 ? ekgk::CB_SLOTS4 : CB_SLOTS;
    std::vector<int> slot_of(L.n_classes, -1);     // part << 8 | slot in the current region
    std::vector<std::vector<int>> slot_cls(split);  // the region's classes by part and slot
    std::vector<int> cost;  // per item (box listing, one packet a part) of the current region
    auto close = [&]() {
        int4& r = regions.back();
        r.y = n_box;
        // Group g of the block's waves takes items g, g + groups, ...: order
        // them so that the groups' work is about equal (largest first, each to
        // the group with least so far that still has a place).
        const int n = (r.y - r.x) / split;
        std::vector<int> by(n), at(n);
        std::iota(by.begin(), by.end(), 0);
        std::stable_sort(by.begin(), by.end(), [&](int x, int y) { return cost[x] > cost[y]; });
        std::vector<int64_t> load(groups, 0);
        std::vector<int> cnt(groups, 0);
        for (int i : by) {
            int w = -1;
            for (int q = 0; q < groups; ++q)
                if (cnt[q] * groups + q < n && (w < 0 || load[q] < load[w])) w = q;
            at[i] = cnt[w]++ * groups + w;
            load[w] += cost[i];
        }
        cost.clear();
        auto reorder = [&](auto& v, size_t per) {
            std::remove_reference_t<decltype(v)> tmp(v.begin() + (std::ptrdiff_t)(per * r.x), v.end());
            per *= split;
            for (int i = 0; i < n; ++i)
                std::copy_n(tmp.begin() + (std::ptrdiff_t)(per * i), per,
                            v.begin() + (std::ptrdiff_t)(per / split * r.x + per * at[i]));
        };
        reorder(pkt, 64);
        reorder(init, 256);
        reorder(mask, 4);
        // the parts' lines one after the other; the first line of parts 1 to 3 (or past the region's)
        int base = 0, first = 0;
        for (int p = 0; p < ekgk::CB_WAVES; ++p) {
            if (p > 0) first |= (p < split ? base : 511) << (9 * (p - 1));  // at most 3 CB_SLOTS: 9 bits
            if (p >= split) continue;
            for (size_t i = 0; i < slot_cls[p].size(); ++i) {
                lines.push_back({slot_cls[p][i], r.z + base + (int)i});
                slot_of[slot_cls[p][i]] = -1;
            }
            base += (int)slot_cls[p].size();
            slot_cls[p].clear();
        }
        r.w = base | split << 16;
        ext.back().w = first;
    };
    std::vector<int> cls;                         // the box's classes
    std::vector<const Rec*> cls_rec;              // their records: [cls_rec[c], cls_rec[c + 1])
    std::vector<int> cls_sub;                     // and the sub-bricks of their cells
    std::vector<std::vector<size_t>> part(split);  // of an item: indexes into cls by part
    std::vector<size_t> fresh;                    // the item's classes new to the region
    // takes classes from c0 on into the item's parts, at most BOX_CLASSES a part; false when the
    // region has no slot left for one
    auto take = [&](size_t c0, size_t& c1) {
        for (auto& q : part) q.clear();
        fresh.clear();
        for (c1 = c0; c1 < cls.size(); ++c1) {
            int p = slot_of[cls[c1]] >> 8;
            if (slot_of[cls[c1]] < 0) {
                p = -1;
                for (int q = 0; q < split; ++q)
                    if (slot_cls[q].size() < (size_t)slots_part && (p < 0 || part[q].size() < part[p].size())) p = q;
            }
            if (p >= 0 && part[p].size() == BOX_CLASSES) break;
            if (p < 0) {
                for (size_t c : fresh) {
                    slot_cls[slot_of[cls[c]] >> 8].pop_back();
                    slot_of[cls[c]] = -1;
                }
                return false;
            }
            if (slot_of[cls[c1]] < 0) {
                slot_of[cls[c1]] = p << 8 | (int)slot_cls[p].size();
                slot_cls[p].push_back(cls[c1]);
                fresh.push_back(c1);
            }
            part[p].push_back(c1);
        }
        return true;
    };
    for (const auto& ob : order) {
        const Rec* r0 = sorted.data() + box_begin[ob.second];
        const Rec* r1 = sorted.data() + box_begin[ob.second + 1];
        const int bx = ob.second % nb2, by = (ob.second / nb2) % nb1, bz = ob.second / nb2 / nb1;
        int last_win[256];
        std::fill(last_win, last_win + 256, -1);
        cls.clear();
        cls_rec.clear();
        cls_sub.clear();
        for (const Rec* r = r0; r < r1; ++r) {
            if (cls.empty() || cls.back() != r->cls) {
                cls.push_back(r->cls);
                cls_rec.push_back(r);
                cls_sub.push_back(0);
            }
            cls_sub.back() |= 1 << (r->cell >> 6);
            const int w = r->cls / CLASS_WINDOW;
            if (last_win[r->cell] != w) {
                last_win[r->cell] = w;
                ++win_entries[w];
                ++n_entries;
            }
        }
        cls_rec.push_back(r1);
        for (size_t c0 = 0, c1; c0 < cls.size(); c0 = c1) {
            if (regions.empty() || n_box - regions.back().x >= target * split || !take(c0, c1)) {
                if (!regions.empty()) close();
                regions.push_back(int4{n_box, 0, (int)lines.size(), 0});
                ext.push_back(int4{0xffff, 0xffff, 0xffff, 0});
                take(c0, c1);
            }
            int item_cost = 0, item_rows = 0;
            const size_t item = pkt.size();
            const int o[3] = {bz * BOX_Z + 1, by * BOX_Y + 1, bx * BOX_X + 1};
            for (const std::vector<size_t>& pc : part) {
                const size_t blk0 = coef.size() / 1024;
                const int n_tile = std::max(1, (int)((pc.size() + 3) / 4));  // none: an empty tile
                const size_t pk = 64 * (size_t)n_box;
                pkt.resize(pk + 64, int4{0, 0, 0, 0});
                init.resize(256 * (size_t)n_box + 256, 0);
                int used = 0;
                uint64_t bm[4] = {0, 0, 0, 0};
                for (int t = 0; t < n_tile; ++t) {
                    const size_t q0 = 4 * t, q1 = std::min(pc.size(), q0 + 4);
                    unsigned slots = 0;
                    int subs = 0;
                    for (size_t q = q0; q < q0 + 4; ++q) {
                        slots |= (unsigned)(q < q1 ? slot_of[cls[pc[q]]] & 255 : slots_part) << (8 * (q - q0));
                        if (q < q1) subs |= cls_sub[pc[q]];
                    }
                    if (coef.size() / 1024 > 0x7ffffff0u) fail(EKG_EINVAL, "too many class cells");
                    const size_t base = coef.size(), ib = 256 * (size_t)n_box + 16 * t;
                    pkt[pk + t] = int4{subs, (int)slots, (int)(base / 1024), 0};
                    coef.resize(base + 1024 * (size_t)__builtin_popcount((unsigned)subs), 0);
                    for (size_t q = q0; q < q1; ++q)
                        for (const Rec* r = cls_rec[pc[q]]; r < cls_rec[pc[q] + 1]; ++r) {
                            const int sub = r->cell >> 6, z = (r->cell >> 4) & 3, y = (r->cell >> 2) & 3, x = r->cell & 3;
                            const int dz = z, dy = y + 4 * (sub >> 1), dx = x + 4 * (sub & 1);
                            const int K = -(r->d[0] * dz + r->d[1] * dy + r->d[2] * dx);
                            if (K < -127 || K > 127) fail(EKG_EINVAL, "dipole moment out of range");
                            const int row = 4 * (int)(q - q0);
                            const int co[4] = {r->d[0], r->d[1], r->d[2], K};
                            const size_t blk = base + 1024 * (size_t)__builtin_popcount((unsigned)(subs & ((1 << sub) - 1)));
                            bm[sub] |= (uint64_t)1 << (r->cell & 63);
                            used |= 1 << (4 * sub + y);
                            for (int i = 0; i < 4; ++i) {
                                coef[blk + 16 * (16 * z + row + i) + 4 * y + x] = (int8_t)co[i];
                                init[ib + row + i] += 128 * co[i];
                            }
                        }
                }
                pkt[pk + 16] = int4{n_tile, used, 0, 0};
                item_rows |= used;
                pkt[pk + 17] = int4{o[0], o[1], o[2], 0};
                // cycles of a box, roughly: 34 a weight of 64 lanes, 64 a block's
                // four products, 180 a tile's flush
                item_cost = std::max(item_cost, 500 + 136 * __builtin_popcount((unsigned)used) +
                                                    64 * (int)(coef.size() / 1024 - blk0) + 180 * n_tile);
                ++n_box;
                mask.insert(mask.end(), bm, bm + 4);
            }
            for (int p = 0; p < split; ++p) pkt[item + 64 * p + 16].z = item_rows;
            cost.push_back(item_cost);
            const int len[3] = {BOX_Z, BOX_Y, BOX_X};
            int* e = &ext.back().x;
            for (int i = 0; i < 3; ++i)
                e[i] = std::min(e[i] & 0xffff, o[i]) | std::max(e[i] >> 16, o[i] + len[i] - 1) << 16;
        }
    }
    if (!regions.empty()) close();
    int64_t n_pieces = 0;
    for (int64_t ne : win_entries) {
        const int64_t groups = (ne + 15) / 16, pc = std::max<int64_t>(1, (groups + CLASS_PIECE - 1) / CLASS_PIECE);
        const int64_t size = std::max<int64_t>(1, (groups + pc - 1) / pc);
        n_pieces += std::max<int64_t>(1, (groups + size - 1) / size);
    }
    // lines per class, in region order
    std::vector<int> cs_off(L.n_classes + 1, 0), cs_line(lines.size());
    for (const auto& l : lines) ++cs_off[l.first + 1];
    for (int k = 0; k < L.n_classes; ++k) cs_off[k + 1] += cs_off[k];
    {
        std::vector<int> at(cs_off.begin(), cs_off.end() - 1);
        for (const auto& l : lines) cs_line[at[l.first]++] = l.second;
    }
    h.ctx->bind();
    auto upload = [&](DevBuf& b, const void* p, size_t n, const char* what) {
        b.reserve(std::max<size_t>(n, 16));
        if (n) hip_check(hipMemcpy(b.p, p, n, hipMemcpyHostToDevice), what);
    };
    std::vector<int4> reg2;
    for (size_t i = 0; i < regions.size(); ++i) {
        reg2.push_back(regions[i]);
        reg2.push_back(ext[i]);
    }
    upload(L.cregion[nhood], reg2.data(), reg2.size() * sizeof(int4), "upload class regions");
    upload(L.cbox[nhood], pkt.data(), pkt.size() * sizeof(int4), "upload class boxes");
    upload(L.cinit[nhood], init.data(), init.size() * sizeof(int), "upload class tile starts");
    upload(L.ccoef[nhood], coef.data(), coef.size(), "upload class coefficients");
    upload(L.cmask[nhood], mask.data(), mask.size() * sizeof(uint64_t), "upload class cell masks");
    upload(L.cs_off[nhood], cs_off.data(), cs_off.size() * sizeof(int), "upload class lines");
    upload(L.cs_line[nhood], cs_line.data(), cs_line.size() * sizeof(int), "upload class lines");
    L.n_ccells[nhood] = (int64_t)sorted.size();
    L.n_centries[nhood] = n_entries;
    L.n_cpieces[nhood] = (int)n_pieces;
    L.n_lines[nhood] = (int)lines.size();
    L.class_parts[nhood] = split;
    L.h_region_line[nhood].clear();
    for (const int4& r : regions) L.h_region_line[nhood].push_back(r.z);
    L.h_region_line[nhood].push_back((int)lines.size());
    L.n_regions[nhood] = (int)regions.size();
    L.cells_built[nhood] = true;
}

namespace {

// Per-request sizes of a group's packed arrays.
struct ReqSizes {
    int64_t rows, chunks, bricks, classes;
};

ReqSizes req_sizes(const ReqSpec& r, bool mfma)
{
    const EcgLayout& L = r.h->layout;
    // the chunk kernel (matrix-core path) keeps G rows on chip: no records
    return ReqSizes{mfma ? 0 : L.V + ekgk::MFMA_PAD, L.n_chunks, L.n_bricks, L.n_classes};
}

// Least share of a request in the fixed workspace for its class sums and their
// tables: a row per window piece and class of the window, three sums per lead
// slot.  The batch that fits depends on it; the class sums take all that the
// group's other buffers leave.
int64_t fixed_class_bytes(const ReqSpec& r, int LP)
{
    const EcgLayout& L = r.h->layout;
    return L.n_classes > 0 ? (int64_t)L.n_cpieces[r.nhood] * CLASS_WINDOW * (3 * LP * 8 + 8) : 0;
}

template <class T>
void append(std::vector<char>& buf, const T* p, size_t n)
{
    const char* c = reinterpret_cast<const char*>(p);
    buf.insert(buf.end(), c, c + n * sizeof(T));
}

// Lines of a group's class sums: the leads of each run of consecutive requests
// of one heart fill rows of 16, a row has a line per (region, class) of the
// heart.  Before the cells are built, a class counts eight lines (2 to 45 on hearts
// measured: a guess, which a launch is held to by class_bytes); a heart that is one class as a
// whole (no lines: its cells cancel) counts one.
struct ClassLines {
    int64_t all = 0, rows = 0, runs = 0;
    // most bytes of the rows' tables: row and position of 16 leads, segment
    // of each row, and a segment per run and launch
    int64_t table_bytes(int64_t cap) const
    {
        return rows * (16 * 8 + 4) + std::min(rows, runs + 1 + 2 * all / cap) * (int64_t)sizeof(ekgk::ClassSeg);
    }
};

ClassLines class_lines(const GroupPlan& g)
{
    ClassLines c;
    for (size_t r = 0; r < g.reqs.size();) {
        const Heart* h = g.reqs[r].h;
        const EcgLayout& L = h->layout;
        int64_t leads = 0;
        for (; r < g.reqs.size() && g.reqs[r].h == h; ++r) leads += g.reqs[r].L;
        // a layout for the other path is sized as one without classes
        if (!(g.mfma && L.valid && L.n_classes > 0)) continue;
        const int64_t lines = L.cells_built[g.nhood] ? std::max(1, L.n_lines[g.nhood]) : (int64_t)8 * L.n_classes;
        c.all += (leads + 15) / 16 * lines;
        c.rows += (leads + 15) / 16;
        ++c.runs;
    }
    return c;
}

}  // namespace

size_t group_device_bytes(GroupPlan& g, size_t budget)
{
    size_t s = 0;
    const int LP = g.LP;
    for (const ReqSpec& r : g.reqs) {
        const EcgLayout& L = r.h->layout;
        const int64_t V = L.valid ? L.V : r.h->n_myo;
        // a layout for the other path is sized as one without classes
        const bool fits = L.valid && (L.class_min == 0 || g.mfma);
        const int64_t est = std::max<int64_t>(1, V / 64 + r.h->max_layer + 4);
        const int64_t nmix = fits ? L.n_chunks : est;
        const int64_t ncls = fits ? L.n_classes : 0;
        const int64_t rows = g.mfma ? 0 : V + ekgk::MFMA_PAD;
        s += (size_t)r.nl * 9 * 8 + (size_t)r.L * 3 * 8 + (size_t)r.Tp * 16;
        s += (size_t)r.nl * (sizeof(ekgk::LayerConst) + r.Tp * 16);
        s += (size_t)rows * (16 * 8 + 16);
        s += (size_t)nmix * (3 * LP * 8 + 8) + (size_t)ncls * 3 * LP * 8;
        s += (size_t)r.nl * ((r.Tp >> (g.mfma ? ekgk::BT_SHIFT_MFMA : ekgk::BT_SHIFT_VALU)) + 1) *
             (8 + 2 * LP * 8);
        s += (size_t)nmix * LP * r.Tp * 8;
        s += (size_t)r.L * r.T * 8;
        // record, heart, seven start tables
        s += sizeof(ekgk::ReqDev) + sizeof(ekgk::HeartDev) + 7 * 8;
    }
    const ClassLines c = class_lines(g);
    g.class_bytes = std::min(c.all * LINE_BYTES, GSUM_BYTES);
    if (c.all == 0) return s;
    // a row of class sums is cut into as many launches as its share asks for, down to a line each
    const int64_t tables = c.table_bytes(1);
    if (s + (size_t)(tables + g.class_bytes) > budget)
        g.class_bytes = std::max<int64_t>(LINE_BYTES, (int64_t)budget - (int64_t)s - tables) / LINE_BYTES * LINE_BYTES;
    return s + (size_t)(tables + g.class_bytes);
}

void enqueue_group(Ctx& ctx, GroupPlan& g, Workspace& ws, hipStream_t stream, const double* d_k,
                   const double* d_pos, double* d_ecg, bool time_fused, bool allow_graph)
{
    const int B = (int)g.reqs.size();
    // the launches below report hipGetLastError: drop an error that an
    // unchecked call (a destroy, a best-effort synchronise) left before them
    (void)hipGetLastError();
    if (ws.arena) {
        // a fixed workspace is shared by every call on the device: nothing of
        // an earlier group (tables, time grids) can be assumed still there
        ws.arena_used = 0;
        ws.h_tables.clear();
        ws.h_grids.clear();
    }
    const int LP = g.LP;
    const bool dev_in = d_k != nullptr;
    // hearts of the group
    std::vector<Heart*> hs;
    std::vector<ekgk::HeartDev> hdev;
    std::vector<ekgk::ReqDev> rd(B);
    // time grids shared by requests with the same start, step and length:
    // t_j = start + j*dt by repeated addition (simulator.cpp:496-500),
    // continued over the padding so the last tile stays monotone
    ws.h_tgrid.clear();
    ws.h_thl.clear();
    std::vector<std::pair<std::pair<double, double>, std::pair<int64_t, int64_t>>> grids;  // (start, dt) -> (Tp, off)
    std::vector<int64_t> st_red(B + 1, 0), st_redp(B + 1, 0);
    std::vector<int64_t> st_lf(B + 1, 0), st_ch(B + 1, 0), st_xy(B + 1, 0), st_lay(B + 1, 0), st_out(B + 1, 0),
        st_cs(B + 1, 0), st_cl(B + 1, 0);
    int64_t k_off = 0, pos_off = 0, rows = 0, c_off = 0, p_off = 0, pre_off = 0;
    if (!dev_in) {
        ws.h_k.clear();
        ws.h_pos.clear();
    }
    for (int r = 0; r < B; ++r) {
        ReqSpec& q = g.reqs[r];
        Heart& h = *q.h;
        ensure_layout(h, g.mfma);
        if (g.mfma) ensure_cells(h, g.nhood);
        int hi = -1;
        for (size_t i = 0; i < hs.size(); ++i)
            if (hs[i] == &h) hi = (int)i;
        if (hi < 0) {
            hi = (int)hs.size();
            hs.push_back(&h);
            ekgk::HeartDev d = h.layout.dev;
            if (g.mfma) {
                const EcgLayout& hl = h.layout;
                d.cregion = hl.cregion[g.nhood].as<int4>();
                d.cbox = hl.cbox[g.nhood].as<int4>();
                d.cinit = hl.cinit[g.nhood].as<int4>();
                d.ccoef = hl.ccoef[g.nhood].as<int4>();
                d.cmask = hl.cmask[g.nhood].as<uint64_t>();
                d.cs_off = hl.cs_off[g.nhood].as<int>();
                d.cs_line = hl.cs_line[g.nhood].as<int>();
                d.n_lines = hl.n_lines[g.nhood];
                d.n_regions = hl.n_regions[g.nhood];
            }
            hdev.push_back(d);
        }
        int64_t t_off = -1;
        for (auto& gr : grids)
            if (gr.first.first == q.start && gr.first.second == q.dt && gr.second.first >= q.Tp) t_off = gr.second.second;
        if (t_off < 0) {
            t_off = (int64_t)ws.h_tgrid.size();
            grids.push_back({{q.start, q.dt}, {q.Tp, t_off}});
            double st = q.start;
            for (int64_t j = 0; j < q.Tp; ++j) {
                ws.h_tgrid.push_back(st);
                const float hi32 = (float)st;
                ws.h_thl.push_back(hi32);
                ws.h_thl.push_back((float)(st - (double)hi32));
                st += q.dt;
            }
        }
        const ReqSizes z = req_sizes(q, g.mfma);
        ekgk::ReqDev& R = rd[r];
        R.heart = hi;
        R.L = q.L;
        R.nl = q.nl;
        R.T = (int)q.T;
        R.Tn = (int)q.Tn;
        R.Tp = (int)q.Tp;
        R.n_tiles = q.n_tiles;
        R.bt_shift = g.mfma ? ekgk::BT_SHIFT_MFMA : ekgk::BT_SHIFT_VALU;
        R.k_off = dev_in ? (int64_t)r * q.nl * 9 : k_off;
        R.pos_off = dev_in ? (int64_t)r * q.L * 3 : pos_off;
        R.ecg_off = st_out[r];
        R.t_off = t_off;
        R.lay_off = st_lay[r];
        R.xy_off = st_xy[r];
        R.g_off = rows;
        R.c_off = c_off;
        R.p_off = p_off;
        R.pre_off = pre_off;
        R.cls_off = st_cs[r];
        if (!dev_in) {
            ws.h_k.insert(ws.h_k.end(), q.k, q.k + 9 * q.nl);
            ws.h_pos.insert(ws.h_pos.end(), q.pos, q.pos + 3 * q.L);
            k_off += 9 * q.nl;
            pos_off += 3 * q.L;
        }
        rows += z.rows;
        c_off += z.chunks;
        p_off += z.chunks * LP * q.Tp;
        pre_off += (int64_t)q.nl * ((q.Tp >> R.bt_shift) + 1);
        st_lf[r + 1] = st_lf[r] + z.bricks;
        st_ch[r + 1] = st_ch[r] + z.chunks;
        st_xy[r + 1] = st_xy[r] + (int64_t)q.nl * q.Tp;
        st_lay[r + 1] = st_lay[r] + q.nl;
        st_out[r + 1] = st_out[r] + (int64_t)q.L * q.T;
        const int64_t tiles = ((int64_t)q.T + (1 << R.bt_shift) - 1) >> R.bt_shift;
        // Long ranges of chunks in transition: a heart of many chunks, from before
        // its last activation on (a request that starts later meets every
        // chunk saturated).  512 chunks put about 170 into a range of the upstroke,
        // where the sums in parts begin to pay (48^3: 157 chunks, 12 us either way;
        // one 12-lead request on the 80^3, 96^3 and 128^3 conduction-matrix hearts
        // 104, 98 and 137 us, 140, 152 and 224 without).  On the vector-ALU path a
        // tile has 64 steps, so that from 8 leads on its sums fill a block without
        // parts: 12 leads on 128^3 404 us, 510 in parts; 2 leads 338 and 226.
        const bool parts = (g.mfma || LP == 4) && h.layout.n_chunks >= LONG_RANGES && q.start < h.layout.a_last;
        st_red[r + 1] = st_red[r] + (parts ? 0 : (q.L * tiles) << R.bt_shift);
        st_redp[r + 1] = st_redp[r] + (parts ? tiles : 0);
        st_cs[r + 1] = st_cs[r] + z.classes;
        st_cl[r + 1] = st_cl[r] + (z.classes > 0 ? q.n_tiles : 0);
    }
    const int64_t pos_max = rd[B - 1].pos_off + 3 * 16;
    if (st_lf[B] > 0x7fffffffLL || st_ch[B] > 0x7fffffffLL || st_lay[B] > 0x7fffffffLL ||
        st_redp[B] > 0x7fffffffLL || st_cl[B] > 0x7fffffffLL || pos_max > 0x7fffffffLL)
        fail(EKG_EINVAL, "launch group too large");
    // device buffers (grow-only)
    ws.need(ws.lc, (size_t)st_lay[B] * sizeof(ekgk::LayerConst));
    ws.need(ws.xy, (size_t)std::max<int64_t>(1, st_xy[B]) * 16);
    ws.need(ws.G, (size_t)std::max<int64_t>(1, rows) * 16 * 8);
    ws.need(ws.aux, (size_t)std::max<int64_t>(1, rows) * sizeof(float4));
    ws.need(ws.sums, (size_t)std::max<int64_t>(1, c_off) * 3 * LP * 8);
    ws.need(ws.bnd, (size_t)std::max<int64_t>(1, c_off) * sizeof(int2));
    ws.need(ws.pre_rng, (size_t)std::max<int64_t>(1, pre_off) * sizeof(int2));
    ws.need(ws.pre_ab, (size_t)std::max<int64_t>(1, pre_off) * 2 * LP * 8);
    ws.need(ws.partial, (size_t)std::max<int64_t>(1, p_off) * 8);
    ws.need(ws.csums, (size_t)std::max<int64_t>(1, st_cs[B]) * 3 * LP * 8);
    if (!d_ecg) {
        ws.need(ws.ecg, (size_t)std::max<int64_t>(1, st_out[B]) * 8);
        d_ecg = ws.ecg.as<double>();
    }
    // Class boxes: the leads of consecutive requests of one heart (a server
    // group is ordered by heart) fill rows of 16, those of a heart's run cut into
    // segments whose sums fit gsum, and the segments into launches.
    std::vector<ekgk::ClassSeg> segs;
    std::vector<ekgk::ClassLaunch> launches;
    std::vector<int> rowtab, rowpos, rgseg;
    if (g.mfma && st_cs[B] > 0) {
        const ClassLines cl = class_lines(g);
        int64_t fixed = 0;
        for (const ReqSpec& r : g.reqs) fixed += fixed_class_bytes(r, LP);
        int64_t cap = std::min(cl.all, GSUM_BYTES / LINE_BYTES);
        if (ws.arena) {
            // what is left of it after the tables and time grids below, each aligned
            const size_t others = rd.size() * sizeof rd[0] + hdev.size() * sizeof hdev[0] + 7 * (B + 1) * 8 +
                                  ws.h_tgrid.size() * 8 + ws.h_thl.size() * 4 + 3 * 256;
            const int64_t room = (int64_t)ws.arena_bytes - (int64_t)((ws.arena_used + 255) & ~(size_t)255) - (int64_t)others;
            if (room < fixed) ws.full();
            cap = std::min(cap, (room - cl.table_bytes(1)) / LINE_BYTES);
        }
        if (g.class_bytes >= 0) cap = std::min(cap, g.class_bytes / LINE_BYTES);
        cap = std::max<int64_t>(1, cap);
        ws.need(ws.gsum, (size_t)(cap * LINE_BYTES));
        int64_t block0 = 0, used = cap;  // lines taken in the current launch
        for (int r = 0; r < B;) {
            const EcgLayout& hl = g.reqs[r].h->layout;
            int r1 = r;
            const int rg_first = (int)rgseg.size();
            size_t at = rowtab.size(), leads = 0;
            for (; r1 < B && g.reqs[r1].h == g.reqs[r].h; ++r1)
                if (hl.n_classes > 0) leads += g.reqs[r1].L;
            rowtab.resize(at + ((leads + 15) & ~(size_t)15));
            rowpos.resize(rowtab.size());
            for (int q = r; q < r1 && leads > 0; ++q)
                for (int i = 0; i < g.reqs[q].L; ++i, ++at) {
                    rowtab[at] = q << 5 | i;
                    rowpos[at] = (int)rd[q].pos_off + 3 * i;
                }
            for (; at < rowtab.size(); ++at) {
                rowtab[at] = rowtab[at - 1] | (int)0x80000000u;
                rowpos[at] = rowpos[at - 1];
            }
            const int64_t lines = std::max(1, hl.n_lines[g.nhood]);
            const int rg_end = (int)(rowtab.size() / 16);
            for (int rg = rg_first; rg < rg_end;) {
                if (lines > cap) {  // not even one row fits: its lines in turn, cut at regions where that leaves half
                    const std::vector<int>& rl = hl.h_region_line[g.nhood];
                    for (int64_t l0 = 0, l1; l0 < lines; l0 = l1) {
                        l1 = std::min(lines, l0 + cap);
                        const int cut = *(std::upper_bound(rl.begin(), rl.end(), (int)l1) - 1);
                        if (cut - l0 >= cap / 2 && cut > l0) l1 = cut;
                        const int reg0 = (int)(std::upper_bound(rl.begin(), rl.end(), (int)l0) - rl.begin()) - 1;
                        const int reg1 = (int)(std::lower_bound(rl.begin(), rl.end(), (int)l1) - rl.begin());
                        launches.push_back({(int)segs.size(), 1, rg, 1, (int)l0, (int)l1, reg0, reg1 - reg0, reg1 - reg0,
                                            hl.class_parts[g.nhood] == 4 ? 2 : 1});
                    }
                    segs.push_back(ekgk::ClassSeg{rg, 1, hl.n_regions[g.nhood], rd[r].heart, 1, 0, block0, 0});
                    rgseg.push_back((int)segs.size() - 1);
                    block0 += hl.n_regions[g.nhood];
                    used = cap;
                    ++rg;
                    continue;
                }
                const bool four = hl.class_parts[g.nhood] == 4;  // a kernel instance of its own
                if (used + lines > cap || launches.back().n_rg >= 65535 || four != (launches.back().parts == 2)) {
                    launches.push_back({(int)segs.size(), 0, rg, 0});
                    used = 0;
                }
                ekgk::ClassLaunch& la = launches.back();
                const int n = (int)std::min<int64_t>({rg_end - rg, (cap - used) / lines, 65535 - la.n_rg});
                const int nr = hl.n_regions[g.nhood];
                // rows a block: as many as leave about six rounds of blocks on
                // the chip (three a CU), at most 8
                const int per = (int)std::max<int64_t>(1, std::min<int64_t>(8, (int64_t)n * nr / (6 * 768)));
                segs.push_back(ekgk::ClassSeg{rg, n, nr, rd[r].heart, per, 0, block0, used});
                for (int i = 0; i < n; ++i) rgseg.push_back((int)segs.size() - 1);
                const int64_t nblk = (int64_t)nr * ((n + per - 1) / per);
                block0 += nblk;
                la.blocks += nblk;
                ++la.n_segs;
                if (hl.class_parts[g.nhood] > 1) la.parts = four ? 2 : 1;
                la.n_rg += n;
                used += n * lines;
                rg += n;
            }
            r = r1;
        }
    }
    // tables: uploaded only when they changed since the last group on this
    // workspace (a repeated group replays without host traffic)
    std::vector<char> tables;
    tables.reserve(hdev.size() * sizeof hdev[0] + rd.size() * sizeof rd[0] + 7 * (B + 1) * 8 +
                   segs.size() * sizeof(ekgk::ClassSeg) + (rgseg.size() + rowtab.size() + rowpos.size()) * 4);
    append(tables, hdev.data(), hdev.size());
    const size_t o_req = tables.size();
    append(tables, rd.data(), rd.size());
    const size_t o_st = tables.size();
    for (auto* st : {&st_lf, &st_ch, &st_xy, &st_lay, &st_cl, &st_red, &st_redp})
        append(tables, st->data(), st->size());
    const size_t o_seg = tables.size();
    append(tables, segs.data(), segs.size());
    const size_t o_rgseg = tables.size();
    append(tables, rgseg.data(), rgseg.size());
    const size_t o_row = tables.size();
    append(tables, rowtab.data(), rowtab.size());
    const size_t o_pos = tables.size();
    append(tables, rowpos.data(), rowpos.size());
    void* before = ws.hearts.p;
    ws.need(ws.hearts, tables.size());
    if (ws.hearts.p != before) ws.h_tables.clear();
    if (tables != ws.h_tables) {
        hip_check(hipMemcpyAsync(ws.hearts.p, tables.data(), tables.size(), hipMemcpyHostToDevice, stream),
                  "upload group tables");
        ws.h_tables.swap(tables);
    }
    std::vector<char> grid_bytes;
    append(grid_bytes, ws.h_tgrid.data(), ws.h_tgrid.size());
    append(grid_bytes, ws.h_thl.data(), ws.h_thl.size());
    before = ws.tgrid.p;
    ws.need(ws.tgrid, grid_bytes.size());
    if (ws.tgrid.p != before) ws.h_grids.clear();
    if (grid_bytes != ws.h_grids) {
        hip_check(hipMemcpyAsync(ws.tgrid.p, grid_bytes.data(), grid_bytes.size(), hipMemcpyHostToDevice, stream),
                  "upload time grids");
        ws.h_grids.swap(grid_bytes);
    }
    if (!dev_in) {
        // coefficients and positions in one upload: each is about 10 us of host
        // and copy engine before the group's first kernel
        const size_t nk = ws.h_k.size();
        ws.h_k.insert(ws.h_k.end(), ws.h_pos.begin(), ws.h_pos.end());
        ws.need(ws.layer_k, ws.h_k.size() * 8);
        hip_check(hipMemcpyAsync(ws.layer_k.p, ws.h_k.data(), ws.h_k.size() * 8, hipMemcpyHostToDevice, stream),
                  "upload AP coefficients and lead positions");
        d_k = ws.layer_k.as<double>();
        d_pos = d_k + nk;
    }
    const char* tb = static_cast<const char*>(ws.hearts.p);
    const int64_t* stp = reinterpret_cast<const int64_t*>(tb + o_st);
    ekgk::GroupArgs a{};
    a.hearts = reinterpret_cast<const ekgk::HeartDev*>(tb);
    a.reqs = reinterpret_cast<const ekgk::ReqDev*>(tb + o_req);
    a.B = B;
    a.LP = LP;
    a.nhood = g.nhood;
    a.mfma = g.mfma ? 1 : 0;
    a.mfma_waves = g.waves;
    a.lf_phase = g.lf_phase;
    a.chunk_max = 0;
    for (Heart* hp : hs) a.chunk_max = std::max(a.chunk_max, hp->layout.chunk_target);
    a.lf_start = stp;
    a.ch_start = stp + (B + 1);
    a.xy_start = stp + 2 * (B + 1);
    a.lay_start = stp + 3 * (B + 1);
    a.cl_start = stp + 4 * (B + 1);
    a.red_start = stp + 5 * (B + 1);
    a.redp_start = stp + 6 * (B + 1);
    a.cs_max = 0;
    for (int r = 0; r < B; ++r) a.cs_max = std::max<int>(a.cs_max, (int)(st_cs[r + 1] - st_cs[r]));
    a.n_cl = st_cl[B];
    a.n_lf = st_lf[B];
    a.n_ch = st_ch[B];
    // every request with the same chunk count: the chunk kernel runs chunk-major
    a.ch_uniform = B > 0 ? (int)(st_ch[1] - st_ch[0]) : 0;
    for (int r = 1; r < B && a.ch_uniform; ++r)
        if (st_ch[r + 1] - st_ch[r] != a.ch_uniform) a.ch_uniform = 0;
    a.one_heart = hs.size() == 1 ? 1 : 0;
    a.segs = reinterpret_cast<const ekgk::ClassSeg*>(tb + o_seg);
    a.rgseg = reinterpret_cast<const int*>(tb + o_rgseg);
    a.rowtab = reinterpret_cast<const int*>(tb + o_row);
    a.rowpos = reinterpret_cast<const int*>(tb + o_pos);
    // class-kernel blocks: XCD-aware order when every request has the same count
    a.cl_per_req = (B > 0 && B % 8 == 0) ? (int)(st_cl[1] - st_cl[0]) : 0;
    for (int r = 1; r < B && a.cl_per_req; ++r)
        if (st_cl[r + 1] - st_cl[r] != a.cl_per_req) a.cl_per_req = 0;
    a.n_xy = st_xy[B];
    a.n_lay = st_lay[B];
    a.n_red = st_red[B];
    a.n_redp = st_redp[B];
    a.red_items = std::min(128, LP << (g.mfma ? ekgk::BT_SHIFT_MFMA : ekgk::BT_SHIFT_VALU));
    // a prefix block sums a layer's chunks: wide where there are many (64 requests with
    // about 1,000 a layer: 10 us less than 256 threads; 128 requests with 130 a layer: 22 us more)
    int64_t nc_max = 0;
    for (Heart* hp : hs)
        for (int l = 1; l <= hp->max_layer; ++l)
            nc_max = std::max<int64_t>(nc_max, hp->layout.h_layer_chunk[l + 1] - hp->layout.h_layer_chunk[l]);
    a.pre_threads = nc_max > 512 ? 1024 : 256;
    a.layer_k = d_k;
    a.lead_pos = d_pos;
    a.tgrid = ws.tgrid.as<double>();
    a.thl = reinterpret_cast<const float2*>(static_cast<const char*>(ws.tgrid.p) + ws.h_tgrid.size() * 8);
    a.lc = ws.lc.as<ekgk::LayerConst>();
    a.xy = ws.xy.as<double2>();
    a.rec = ws.G.as<double>();
    a.aux = ws.aux.as<float4>();
    a.sums = ws.sums.as<double>();
    a.bnd = ws.bnd.as<int2>();
    a.pre_rng = ws.pre_rng.as<int2>();
    a.pre_ab = ws.pre_ab.as<double>();
    a.partial = ws.partial.as<double>();
    a.gsum = ws.gsum.as<double>();
    a.csums = ws.csums.as<double>();
    a.ecg = d_ecg;
    int64_t w_class = 0, w_chunk = 0;  // chunks of classes and of other voxels, times leads
    for (const ReqSpec& r : g.reqs) {
        w_class += (int64_t)r.L * r.h->layout.n_cchunks;
        w_chunk += (int64_t)r.L * r.h->layout.n_chunks;
    }
    const bool classes_lead = w_class > w_chunk;
    auto launch_all = [&](bool timed) {
        // The timed kernel is the dominant one of each path: the class-box
        // kernel, or without classes the chunk kernel (matrix-core path), or
        // the fused transition-tile kernel (vector ALUs).
        hipEvent_t e0 = nullptr, e1 = nullptr;
        bool counts = true;
        auto tic = [&]() {
            if (!timed) return;
            e0 = ctx.get_event();
            e1 = ctx.get_event();
            hip_check(hipEventRecord(e0, stream), "hipEventRecord");
        };
        auto toc = [&]() {
            if (!timed) return;
            hip_check(hipEventRecord(e1, stream), "hipEventRecord");
            ctx.pending.push_back({e0, e1, counts});
            counts = false;
        };
        auto classes = [&]() {
            for (const ekgk::ClassLaunch& c : launches) {
                tic();
                hip_check(ekgk::launch_class_boxes(a, c, stream), "class_box launch");
                toc();
                hip_check(ekgk::launch_class_sums(a, c, stream), "class_sums launch");
            }
        };
        if (g.mfma && !launches.empty() && ws.side) {
            // Two branches: the class-box kernel and the class sums on
            // `stream`, beside the AP tables, chunk, prefix and reduction
            // kernels on the side stream (they share no buffer); the
            // class ECG kernel adds to the reduction's output after both.
            // The branch with more of the voxels is launched first; a small
            // class branch goes out while the chunk kernel runs.  One 12-lead
            // request on a 128^3 heart, classes mostly: 167 us with the whole side
            // branch first, 142 after the AP tables, 126 ahead of all.
            // One on a 24-layer heart, classes few: 124 us with the side branch
            // first, 121 after the AP tables, 114 after the chunk
            // kernel; 128 such requests 578, 573, 573, and 582 us ahead of all.
            hip_check(hipEventRecord(ws.ev_fork, stream), "hipEventRecord");
            if (classes_lead) classes();
            hip_check(hipStreamWaitEvent(ws.side, ws.ev_fork, 0), "hipStreamWaitEvent");
            hip_check(ekgk::launch_ap_tables(a, ws.side), "ap_tables launch");
            hip_check(ekgk::launch_ecg_chunk(a, ws.side), "ecg_chunk launch");
            if (!classes_lead) classes();
            hip_check(ekgk::launch_layer_prefix(a, ws.side), "layer_prefix launch");
            hip_check(ekgk::launch_ecg_reduce(a, ws.side), "ecg_reduce launch");
            hip_check(hipEventRecord(ws.ev_join, ws.side), "hipEventRecord");
            hip_check(hipStreamWaitEvent(stream, ws.ev_join, 0), "hipStreamWaitEvent");
            hip_check(ekgk::launch_ecg_class(a, stream), "ecg_class launch");
            return;
        }
        hip_check(ekgk::launch_ap_tables(a, stream), "ap_tables launch");
        if (g.mfma) {
            // the class-box kernel is timed when the group has classes
            if (launches.empty()) tic();
            hip_check(ekgk::launch_ecg_chunk(a, stream), "ecg_chunk launch");
            if (launches.empty()) toc();
            classes();
            hip_check(ekgk::launch_layer_prefix(a, stream), "layer_prefix launch");
        } else {
            hip_check(ekgk::launch_lead_field(a, stream), "lead_field launch");
            hip_check(ekgk::launch_chunk_sums(a, stream), "chunk_sums launch");
            hip_check(ekgk::launch_layer_prefix(a, stream), "layer_prefix launch");
            tic();
            hip_check(ekgk::launch_ecg_fused(a, stream), "ecg_fused launch");
            toc();
        }
        hip_check(ekgk::launch_ecg_reduce(a, stream), "ecg_reduce launch");
        hip_check(ekgk::launch_ecg_class(a, stream), "ecg_class launch");
    };
    if (!ctx.graphs || time_fused || !allow_graph) {
        launch_all(time_fused);
        return;
    }
    // Graph mode: the launches of a group are captured once and replayed
    // while the kernel arguments (buffers, counts, shapes) stay the same; the
    // per-request values live in device tables and buffers, so new inputs
    // in the same places need no recapture.  The graph holds kernels only.
    std::vector<char> key(reinterpret_cast<const char*>(&a), reinterpret_cast<const char*>(&a) + sizeof a);
    append(key, launches.data(), launches.size());
    if (!ws.graph || key != ws.graph_key) {
        if (ws.graph) {
            (void)hipGraphExecDestroy(ws.graph);
            ws.graph = nullptr;
        }
        ws.graph_key.clear();
        hip_check(hipStreamBeginCapture(stream, hipStreamCaptureModeThreadLocal), "hipStreamBeginCapture");
        hipGraph_t graph = nullptr;
        try {
            launch_all(false);
        } catch (...) {
            (void)hipStreamEndCapture(stream, &graph);
            if (graph) (void)hipGraphDestroy(graph);
            throw;
        }
        hip_check(hipStreamEndCapture(stream, &graph), "hipStreamEndCapture");
        const hipError_t e = hipGraphInstantiate(&ws.graph, graph, nullptr, nullptr, 0);
        (void)hipGraphDestroy(graph);
        hip_check(e, "hipGraphInstantiate");
        ws.graph_key.swap(key);
        ++ctx.graph_captures;
    }
    hip_check(hipGraphLaunch(ws.graph, stream), "hipGraphLaunch");
    ++ctx.graph_launches;
}

void simulate(Heart& h, int batch, const ekg_sim_desc* descs, double* ecg)
{
    Ctx& ctx = *h.ctx;
    std::lock_guard<std::mutex> g1(ctx.mu);
    std::lock_guard<std::mutex> g2(h.mu);
    if (!ecg) fail(EKG_EINVAL, "ecg output buffer is required");
    if (batch < 1 || !descs) fail(EKG_EINVAL, "batch must hold at least one descriptor");
    std::vector<ReqSpec> specs;
    for (int b = 0; b < batch; ++b) specs.push_back(make_spec(h, descs[b], true));
    int64_t n_out = 0;
    for (const ReqSpec& r : specs) n_out += (int64_t)r.L * r.T;
    if (n_out == 0) return;
    ctx.bind();
    GroupPlan g = plan_group(ctx, std::move(specs));
    enqueue_group(ctx, g, ctx.ws, ctx.stream, nullptr, nullptr, nullptr, ctx.profiling);
    hip_check(hipMemcpyAsync(ecg, ctx.ws.ecg.p, (size_t)n_out * 8, hipMemcpyDeviceToHost, ctx.stream),
              "download ECG");
    hip_check(hipStreamSynchronize(ctx.stream), "hipStreamSynchronize");
    if (ctx.profiling) ctx.collect_timings();
}

void simulate_device(Heart& h, const ekg_batch_dev& d)
{
    Ctx& ctx = *h.ctx;
    std::lock_guard<std::mutex> g1(ctx.mu);
    std::lock_guard<std::mutex> g2(h.mu);
    if (!d.layer_k_dev || !d.lead_pos_dev || !d.ecg_dev) fail(EKG_EINVAL, "device pointers are required");
    if (d.batch < 1 || d.batch > (1 << 20)) fail(EKG_EINVAL, "batch must hold 1..2^20 simulations");
    ekg_sim_desc s{};
    s.n_layers = d.n_layers;
    s.n_leads = d.n_leads;
    s.nhood = d.nhood;
    s.start = d.start;
    s.length = d.length;
    s.dt = d.dt;
    const ReqSpec one = make_spec(h, s, false);
    if (one.T == 0) return;
    ctx.bind();
    GroupPlan g = plan_group(ctx, std::vector<ReqSpec>(d.batch, one));
    enqueue_group(ctx, g, ctx.ws, ctx.stream, d.layer_k_dev, d.lead_pos_dev, d.ecg_dev, ctx.profiling);
}

void simulate_device_fixed(Heart& h, const ekg_batch_dev& d)
{
    Ctx& ctx = *h.ctx;
    std::lock_guard<std::mutex> g1(ctx.mu);
    std::lock_guard<std::mutex> g2(h.mu);
    if (!d.layer_k_dev || !d.lead_pos_dev || !d.ecg_dev) fail(EKG_EINVAL, "device pointers are required");
    if (d.batch < 1 || d.batch > (1 << 20)) fail(EKG_EINVAL, "batch must hold 1..2^20 simulations");
    if (!ctx.ws_fixed.arena) fail(EKG_ESTATE, "the device's static workspace is not resolved");
    ekg_sim_desc s{};
    s.n_layers = d.n_layers;
    s.n_leads = d.n_leads;
    s.nhood = d.nhood;
    s.start = d.start;
    s.length = d.length;
    s.dt = d.dt;
    const ReqSpec one = make_spec(h, s, false);
    if (one.T == 0) return;
    GroupPlan g = plan_group(ctx, std::vector<ReqSpec>(d.batch, one));
    // the per-heart layout is device memory built on first use: it must exist
    if (!layout_ready(h, g.mfma, g.nhood))
        fail(EKG_ESTATE, "the heart's layout for this neighbourhood and tuning is not built; call "
                         "ekg_heart_layout_info (or any simulation of the heart) first");
    ctx.bind();
    enqueue_group(ctx, g, ctx.ws_fixed, ctx.stream, d.layer_k_dev, d.lead_pos_dev, d.ecg_dev, false, false);
}

ekg_tune autotune(Heart& h, const ekg_sim_desc& sample, int batch)
{
    Ctx& ctx = *h.ctx;
    std::lock_guard<std::mutex> g1(ctx.mu);
    std::lock_guard<std::mutex> g2(h.mu);
    if (batch < 1 || batch > 4096) fail(EKG_EINVAL, "autotune batch must be 1..4096");
    const ReqSpec one = make_spec(h, sample, true);
    if (one.T == 0) fail(EKG_EINVAL, "the sample simulation has no time steps");
    if (!h.excited) fail(EKG_ESTATE, "excitation sequence not computed or loaded");
    ctx.bind();
    const int saved_kernel = ctx.kernel;
    const int def_chunk = DEFAULT_CHUNK;
    ekg_tune best{def_chunk, DEFAULT_WAVES, 2, EKG_KERNEL_MFMA, h.tune_class, 0.0};
    Workspace ws;
    hipStream_t st = ctx.stream;
    hipEvent_t e0 = ctx.get_event(), e1 = ctx.get_event();
    // time one configuration: one warm-up group, then the best of two
    auto trial = [&](const ekg_tune& c) {
        h.tune_chunk = c.chunk_voxels;
        h.tune_waves = c.mfma_waves;
        h.tune_phase = c.lead_phase;
        h.tune_kernel = c.kernel;
        h.tune_class = c.class_min;
        ctx.kernel = EKG_KERNEL_AUTO;
        GroupPlan g = plan_group(ctx, std::vector<ReqSpec>(batch, one));
        double best_ms = 1e30;
        for (int it = 0; it < 3; ++it) {
            hip_check(hipEventRecord(e0, st), "hipEventRecord");
            enqueue_group(ctx, g, ws, st, nullptr, nullptr, nullptr, false);
            hip_check(hipEventRecord(e1, st), "hipEventRecord");
            hip_check(hipEventSynchronize(e1), "hipEventSynchronize");
            float ms = 0.f;
            hip_check(hipEventElapsedTime(&ms, e0, e1), "hipEventElapsedTime");
            if (it > 0) best_ms = std::min(best_ms, (double)ms);
        }
        return best_ms;
    };
    try {
        best.ms_per_batch = trial(best);
        auto sweep = [&](int ekg_tune::*field, std::vector<int> values) {
            for (int v : values) {
                if (v == best.*field) continue;
                ekg_tune c = best;
                c.*field = v;
                const double ms = trial(c);
                if (ms < best.ms_per_batch) {
                    best = c;
                    best.ms_per_batch = ms;
                }
            }
        };
        sweep(&ekg_tune::kernel, {EKG_KERNEL_MFMA, EKG_KERNEL_VALU});
        if (best.kernel == EKG_KERNEL_MFMA) {
            // chunk size and block size interact (LDS rows per block against
            // blocks per CU): every pair
            const ekg_tune base = best;
            for (int chunk : {64, 128, 256, 512})
                for (int waves : {2, 4, 8}) {
                    if (chunk == base.chunk_voxels && waves == base.mfma_waves) continue;
                    ekg_tune c = base;
                    c.chunk_voxels = chunk;
                    c.mfma_waves = waves;
                    const double ms = trial(c);
                    if (ms < best.ms_per_batch) {
                        best = c;
                        best.ms_per_batch = ms;
                    }
                }
            // every voxel in a class (no chunks outside classes) when the
            // default threshold already leaves at most 1% of the voxels out:
            // the few extra classes are cheaper than the chunk path for them
            if (best.class_min == 0 && h.layout.valid && h.layout.n_classes > 0) {
                int64_t cv = 0;
                for (const int4& cc : h.layout.h_cchunks) cv += cc.z - cc.y;
                if (h.layout.V - cv <= h.layout.V / 100) sweep(&ekg_tune::class_min, {1});
            }
        } else {
            std::vector<int> chunks{64, 128, 256, 512};
            chunks.erase(std::remove(chunks.begin(), chunks.end(), def_chunk), chunks.end());
            sweep(&ekg_tune::chunk_voxels, chunks);
            sweep(&ekg_tune::lead_phase, {2, 4});
        }
    } catch (...) {
        ctx.kernel = saved_kernel;
        h.tune_chunk = h.tune_waves = h.tune_phase = h.tune_kernel = 0;
        ctx.free_events.push_back(e0);
        ctx.free_events.push_back(e1);
        throw;
    }
    ctx.kernel = saved_kernel;
    ctx.free_events.push_back(e0);
    ctx.free_events.push_back(e1);
    h.tune_chunk = best.chunk_voxels;
    h.tune_waves = best.mfma_waves;
    h.tune_phase = best.lead_phase;
    h.tune_kernel = best.kernel;
    h.tune_class = best.class_min;
    ensure_layout(h, best.kernel != EKG_KERNEL_VALU);
    hip_check(hipStreamSynchronize(st), "hipStreamSynchronize");
    return best;
}

namespace {

int crit_count(const ekg_criteria_desc& c, int n_leads)
{
    if (c.mode < EKG_CMP_RMS || c.mode > EKG_CMP_VECTOR_CORRELATION) fail(EKG_EINVAL, "unknown comparison mode");
    if (c.n_targets < 1 || c.target_len < 1 || !c.targets || !c.target_offsets)
        fail(EKG_EINVAL, "criteria need at least one non-empty target and its offset");
    return std::min(n_leads, c.n_targets);
}

// Targets and offsets into the context's buffers on its stream, and their
// statistics over the comparison length for ECGs of n_steps samples -- only
// when these differ from the last call (an optimiser keeps its targets).
void prepare_targets(Ctx& ctx, const ekg_criteria_desc& c, int64_t n_steps)
{
    const size_t nt = (size_t)c.n_targets * (size_t)c.target_len;
    const int64_t len = std::min<int64_t>(n_steps, c.target_len);
    std::vector<double> h(c.targets, c.targets + nt);
    h.insert(h.end(), c.target_offsets, c.target_offsets + c.n_targets);
    h.push_back((double)c.n_targets);
    h.push_back((double)len);
    void* b0 = ctx.crit_tg.p;
    void* b1 = ctx.crit_off.p;
    void* b2 = ctx.crit_stats.p;
    ctx.crit_tg.reserve(nt * 8);
    ctx.crit_off.reserve((size_t)c.n_targets * 8);
    ctx.crit_stats.reserve((size_t)c.n_targets * 4 * 8);
    if (ctx.crit_tg.p != b0 || ctx.crit_off.p != b1 || ctx.crit_stats.p != b2) ctx.crit_h.clear();
    if (h == ctx.crit_h) return;
    hip_check(hipMemcpyAsync(ctx.crit_tg.p, c.targets, nt * 8, hipMemcpyHostToDevice, ctx.stream), "upload targets");
    hip_check(hipMemcpyAsync(ctx.crit_off.p, c.target_offsets, (size_t)c.n_targets * 8, hipMemcpyHostToDevice,
                             ctx.stream),
              "upload target offsets");
    hip_check(ekgk::launch_target_stats(ctx.crit_tg.as<double>(), c.n_targets, c.target_len, len,
                                        ctx.crit_stats.as<double>(), ctx.stream),
              "target statistics launch");
    ctx.crit_h.swap(h);
}

}  // namespace

void criteria_device(Ctx& ctx, const ekg_criteria_desc& c, const double* d_ecg, int batch, int n_leads,
                     int64_t n_steps, double* d_out)
{
    std::lock_guard<std::mutex> g(ctx.mu);
    if (batch < 0 || n_leads < 1 || n_steps < 1) fail(EKG_EINVAL, "bad batch shape");
    if (!d_ecg || !d_out) fail(EKG_EINVAL, "NULL device buffer");
    const int n_crit = crit_count(c, n_leads);
    if (batch == 0) return;
    ctx.bind();
    prepare_targets(ctx, c, n_steps);
    hip_check(ekgk::launch_criteria(c.mode, c.peaks ? 1 : 0, c.raw ? 1 : 0, d_ecg, batch, n_leads, n_steps,
                                    ctx.crit_tg.as<double>(), ctx.crit_off.as<double>(), ctx.crit_stats.as<double>(),
                                    n_crit, c.target_len, d_out, ctx.stream),
              "criteria launch");
}

void simulate_criteria(Heart& h, int batch, const ekg_sim_desc* descs, const ekg_criteria_desc& c,
                       double* criteria)
{
    Ctx& ctx = *h.ctx;
    std::lock_guard<std::mutex> g1(ctx.mu);
    std::lock_guard<std::mutex> g2(h.mu);
    if (!criteria) fail(EKG_EINVAL, "criteria output buffer is required");
    if (batch < 1 || !descs) fail(EKG_EINVAL, "batch must hold at least one descriptor");
    std::vector<ReqSpec> specs;
    for (int b = 0; b < batch; ++b) specs.push_back(make_spec(h, descs[b], true));
    const int L = specs[0].L;
    const int64_t T = specs[0].T;
    for (const ReqSpec& r : specs)
        if (r.L != L || r.T != T) fail(EKG_EINVAL, "every request of a criteria batch needs the same leads and steps");
    if (T < 1) fail(EKG_EINVAL, "no time steps");
    const int n_crit = crit_count(c, L);
    const size_t per = (size_t)n_crit * (c.peaks ? 2 : 1);
    ctx.bind();
    GroupPlan g = plan_group(ctx, std::move(specs));
    enqueue_group(ctx, g, ctx.ws, ctx.stream, nullptr, nullptr, nullptr, ctx.profiling);
    prepare_targets(ctx, c, T);
    ctx.crit_out.reserve((size_t)batch * per * 8);
    hip_check(ekgk::launch_criteria(c.mode, c.peaks ? 1 : 0, c.raw ? 1 : 0, ctx.ws.ecg.as<double>(), batch, L, T,
                                    ctx.crit_tg.as<double>(), ctx.crit_off.as<double>(), ctx.crit_stats.as<double>(),
                                    n_crit, c.target_len, ctx.crit_out.as<double>(), ctx.stream),
              "criteria launch");
    hip_check(hipMemcpyAsync(criteria, ctx.crit_out.p, (size_t)batch * per * 8, hipMemcpyDeviceToHost, ctx.stream),
              "download criteria");
    hip_check(hipStreamSynchronize(ctx.stream), "hipStreamSynchronize");
    if (ctx.profiling) ctx.collect_timings();
}

void excite(Heart& h, bool is_int, const double* transfer, int rows, int cols, const uint8_t* delay)
{
    Ctx& ctx = *h.ctx;
    std::lock_guard<std::mutex> g1(ctx.mu);
    std::lock_guard<std::mutex> g2(h.mu);
    if (h.h_seed.empty()) fail(EKG_ENOSEED, "Could not find starting point for excitation sequence");
    int64_t nseeds = 0;
    for (int64_t i = 0; i < h.nvox; ++i)
        if (h.h_seed[i]) {
            if (!h.h_layer[i]) fail(EKG_EINVAL, "excitation starting point on an empty voxel");
            ++nseeds;
        }
    if (nseeds == 0) fail(EKG_ENOSEED, "Could not find starting point for excitation sequence");
    std::vector<double> wtab;
    if (!is_int) {
        if (!transfer || rows < 1 || cols < 1) fail(EKG_EINVAL, "transfer matrix required");
        if (h.max_layer >= cols || h.max_layer >= rows)
            fail(EKG_ETRANSFER, "transfer (conduction) matrix does not define layer " +
                                    std::to_string(h.max_layer));
        for (int a = 1; a <= h.max_layer; ++a)
            for (int b = 1; b <= h.max_layer; ++b) {
                const double t = transfer[a * cols + b];
                if (!(t >= 0) || !std::isfinite(t))
                    fail(EKG_ETRANSFER, "conduction matrix entries between tissue layers must be "
                                        "finite and >= 0");
            }
        // lag = transfer[lu][lv] * sqrt(|d|^2), FP64 (simulator.cpp:239-240)
        wtab.assign((size_t)rows * cols * 4, 0.0);
        for (int a = 0; a < rows; ++a)
            for (int b = 0; b < cols; ++b)
                for (int k = 1; k <= 3; ++k) {
                    double lag = transfer[a * cols + b];
                    lag *= std::sqrt((double)k);
                    wtab[((size_t)a * cols + b) * 4 + k] = lag;
                }
    } else if (!delay) {
        fail(EKG_EINVAL, "delay grid required");
    }
    ctx.bind();
    const int nb0 = (h.n0 + 7) / 8, nb1 = (h.n1 + 7) / 8, nb2 = (h.n2 + 7) / 8;
    const int nbricks = nb0 * nb1 * nb2;
    // Sweeps are enqueued in rounds of growing length (4, 8, 16, ... up to
    // 64) with one flag per sweep; the host reads the flags once per round.
    // A sweep after convergence finds no active brick and changes nothing.
    constexpr int MAX_ROUND = 64;
    DevBuf d_dist, d_wtab, d_delay, d_flags, d_any;
    d_dist.reserve((size_t)h.nvox * (is_int ? 4 : 8));
    d_flags.reserve((size_t)nbricks * 2);
    d_any.reserve(MAX_ROUND * sizeof(int));
    if (!is_int) {
        d_wtab.reserve(wtab.size() * 8);
        hip_check(hipMemcpy(d_wtab.p, wtab.data(), wtab.size() * 8, hipMemcpyHostToDevice),
                  "upload lag table");
    } else {
        d_delay.reserve(h.nvox);
        hip_check(hipMemcpy(d_delay.p, delay, h.nvox, hipMemcpyHostToDevice), "upload delays");
    }
    uint8_t* fa = d_flags.as<uint8_t>();
    uint8_t* fb = fa + nbricks;
    hipStream_t s = ctx.stream;
    hip_check(hipMemsetAsync(fa, 0, (size_t)nbricks * 2, s), "hipMemsetAsync");
    hip_check(ekgk::launch_ca_init(is_int, h.d_layer.as<uint8_t>(), h.d_seed.as<uint8_t>(), d_dist.p,
                                   fa, h.n0, h.n1, h.n2, nb1, nb2, s),
              "ca_init launch");
    int64_t sweeps = 0;
    const int64_t max_sweeps = 64 + 8 * (int64_t)h.nvox;
    int flags[MAX_ROUND];
    for (int round = 4;; round = std::min(2 * round, MAX_ROUND)) {
        hip_check(hipMemsetAsync(d_any.p, 0, (size_t)round * sizeof(int), s), "hipMemsetAsync");
        for (int q = 0; q < round; ++q) {
            hip_check(ekgk::launch_ca_sweep(is_int, h.d_layer.as<uint8_t>(), d_delay.as<uint8_t>(),
                                            d_wtab.as<double>(), cols, d_dist.p, h.n0, h.n1, h.n2, nb0,
                                            nb1, nb2, fa, fb, d_any.as<int>() + q, s),
                      "ca_sweep launch");
            std::swap(fa, fb);
        }
        hip_check(hipMemcpyAsync(flags, d_any.p, (size_t)round * sizeof(int), hipMemcpyDeviceToHost, s),
                  "read flags");
        hip_check(hipStreamSynchronize(s), "hipStreamSynchronize");
        sweeps += round;
        if (!flags[round - 1]) break;  // the round's last sweep marked no brick: converged
        if (sweeps > max_sweeps) fail(EKG_EDEVICE, "excitation relaxation did not converge");
    }
    h.d_act.reserve((size_t)h.nvox * 8);
    hip_check(ekgk::launch_ca_finalize(is_int, d_dist.p, h.d_act.as<double>(), h.nvox, s),
              "ca_finalize launch");
    h.h_act.resize(h.nvox);
    hip_check(hipMemcpyAsync(h.h_act.data(), h.d_act.p, (size_t)h.nvox * 8, hipMemcpyDeviceToHost, s),
              "download activation");
    hip_check(hipStreamSynchronize(s), "hipStreamSynchronize");
    h.excited = true;
    h.layout.valid = false;
}

}  // namespace ekg
