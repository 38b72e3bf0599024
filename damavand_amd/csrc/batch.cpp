// Batched forward + adjoint of many small circuits in common launches.
#include <algorithm>
#include <atomic>
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <memory>
#include <mutex>
#include <string>
#include <system_error>
#include <thread>
#include <unordered_map>
#include <vector>

#include "device.hpp"
#include "kernels.hpp"
#include "runtime.hpp"

namespace dmv {

// The batched kernels' tile shape (tile qubits k, log2 threads): from the
// caller's choice `pin`, else the tunables batch_tile_qubits /
// batch_threads_log2, else the tuning table for (qubits of the largest circuit,
// dtype), else k = 11 on 256 threads.  The workgroups per CU of earlier tuning
// files and of the tunable batch_wgs_per_cu are checked and have no effect: the
// grid is the circuits' tiles.
static void batch_shape(int nmax, int dtype, const TuneChoice *pin, int *k, int *tlog, int *wgs)
{
    *k = 11;
    *tlog = 8;
    *wgs = 3;
    TuneChoice t;
    if (tune_lookup(tune_key(nmax, dtype, "batch"), &t) && t.set()) {
        *k = t.k;
        *tlog = t.tlog > 0 ? t.tlog : *tlog;
        *wgs = t.wgs > 0 ? t.wgs : *wgs;
    }
    *k = (int)tune_value("batch_tile_qubits", *k);
    *tlog = (int)tune_value("batch_threads_log2", *tlog);
    *wgs = (int)tune_value("batch_wgs_per_cu", *wgs);
    if (pin && pin->set()) {
        *k = pin->k;
        *tlog = pin->tlog > 0 ? pin->tlog : *tlog;
        *wgs = pin->wgs > 0 ? pin->wgs : *wgs;
    }
}

// One device buffer a call, cut into parts of 256 bytes' alignment, and a host
// buffer for what goes into the first parts.  Both are kept for the next call up
// to kKeptBytes each (the host buffer is pinned then); calls from other threads
// meanwhile allocate their own.
class Arena {
public:
    static constexpr uint64_t kKeptBytes = uint64_t(64) << 20;
    ~Arena()
    {
        if (copying_)  // an error came between the copy and the call's last wait
            (void)hipStreamSynchronize(stream());
        {
            std::lock_guard<std::mutex> lk(mu());
            Bufs &K = kept();
            if (b_.cap <= kKeptBytes && !K.dev)
                std::swap(K.dev, b_.dev), std::swap(K.cap, b_.cap);
            if (!K.host)
                std::swap(K.host, b_.host), std::swap(K.host_cap, b_.host_cap);
        }
        release(b_.dev);
        if (b_.host)
            (void)hipHostFree(b_.host);
    }
    static bool give_back()
    {
        void *dev = nullptr;
        {
            std::lock_guard<std::mutex> lk(mu());
            std::swap(dev, kept().dev);
            kept().cap = 0;
        }
        release(dev);
        return dev != nullptr;
    }
    uint64_t part(uint64_t bytes)
    {
        const uint64_t at = size_;
        size_ += (std::max<uint64_t>(bytes, 1) + 255) & ~uint64_t(255);
        return at;
    }
    // The buffers, the host's of `filled` bytes.
    int get(uint64_t filled)
    {
        {
            std::lock_guard<std::mutex> lk(mu());
            std::swap(b_, kept());
        }
        if (b_.cap < size_) {
            release(b_.dev);
            b_.dev = nullptr;
            b_.cap = 0;
            DMV_TRY(alloc(&b_.dev, size_));
            b_.cap = size_;
        }
        filled_ = filled;
        if (filled > kKeptBytes) {
            own_.reset(new char[filled]);
        } else if (b_.host_cap < filled) {
            if (b_.host)
                (void)hipHostFree(b_.host);
            b_.host = nullptr;
            b_.host_cap = 0;
            const uint64_t want = std::min(kKeptBytes, filled + filled / 4);
            if (hipHostMalloc(&b_.host, want, hipHostMallocDefault) == hipSuccess) {
                b_.host_cap = want;
            } else {
                (void)hipGetLastError();
                b_.host = nullptr;
                own_.reset(new char[filled]);
            }
        }
        return DMV_OK;
    }
    char *host() const { return own_ ? own_.get() : (char *)b_.host; }
    int send()
    {
        if (own_)
            return copy_h2d(b_.dev, own_.get(), filled_);
        if (hipMemcpyAsync(b_.dev, b_.host, filled_, hipMemcpyHostToDevice, stream()) != hipSuccess) {
            set_error("batch upload failed");
            return DMV_ERR_HIP;
        }
        copying_ = true;
        return DMV_OK;
    }
    void sent() { copying_ = false; }  // the stream has been waited for since
    template <class T> T *at(uint64_t offset) const { return (T *)((char *)b_.dev + offset); }

private:
    struct Bufs {
        void *dev = nullptr, *host = nullptr;
        uint64_t cap = 0, host_cap = 0;
    };
    static Bufs &kept()
    {
        static Bufs b;
        return b;
    }
    static std::mutex &mu()
    {
        static std::mutex *m = new std::mutex();
        return *m;
    }
    Bufs b_;
    std::unique_ptr<char[]> own_;
    uint64_t size_ = 0, filled_ = 0;
    bool copying_ = false;
};

bool give_back_batch() { return Arena::give_back(); }

int batch_forward_adjoint(int count, int dtype, const int *n, const int *gate_offset, const int *gate_kind,
                          const int *gate_control, const int *gate_target, const double *gate_param,
                          const int *coef_offset, const double *coef, const int *param_offset, double *energy,
                          double *grad, const TuneChoice *pin, double *kernel_ms)
{
    DMV_CHECK_ARG(count >= 1, "empty batch");
    DMV_CHECK_ARG(dtype == DMV_C128 || dtype == DMV_C64, "bad dtype");
    DMV_CHECK_ARG(n && gate_offset && gate_kind && gate_control && gate_target && gate_param && coef_offset && coef &&
                      param_offset && energy && grad,
                  "null batch array");
    // the offsets index host arrays here and device buffers in the kernel:
    // gate ranges must be ordered, coefficient ranges non-negative, and the
    // gradient offsets the exclusive prefix sum of the parameter counts
    // (checked once the counts are known, below)
    DMV_CHECK_ARG(gate_offset[0] >= 0, "gate_offset[0] is negative");
    for (int i = 0; i < count; i++) {
        DMV_CHECK_ARG(gate_offset[i + 1] >= gate_offset[i], "gate_offset decreases at circuit %d", i);
        DMV_CHECK_ARG(coef_offset[i] >= 0, "coef_offset[%d] is negative", i);
    }
    int nmax_all = 0;
    for (int i = 0; i < count; i++)
        nmax_all = std::max(nmax_all, n[i]);
    int K, tlog, per_cu;
    batch_shape(nmax_all, dtype, pin, &K, &tlog, &per_cu);
    const int rlog = K - tlog;
    DMV_CHECK_ARG(batch_kernel_exists(dtype, rlog, tlog), "no batched kernel for %d tile qubits on %d threads", K,
                  1 << tlog);
    DMV_CHECK_ARG(per_cu >= 1 && per_cu <= 16, "batch_wgs_per_cu must be in [1, 16], got %d", per_cu);

    // Circuits with the same gates on the same qubits share one plan: their
    // ops differ in matrices only.  Lowering (matrices), planning and filling
    // in run on host threads; the result does not depend on threading.
    struct Built {
        int rc = DMV_OK;
        std::string err;
        int np = 0;
        uint64_t key = 0;              // of its structure
        int like = -1;                 // the first circuit of the same structure (perhaps itself)
        std::vector<HostOp> f, a;      // merged ops
        std::shared_ptr<const Plan> pf, pa;  // where like is the circuit itself
        uint32_t fwd = 0, adj = 0;     // ... its first passes among all
        uint32_t slots = 0;            // ... and its slots in the slot table
    };
    std::vector<Built> built(count);
    PlanParams pp0;
    pp0.k = K;
    pp0.rlog = rlog;
    pp0.tlog = tlog;
    pp0.low_bits = coalesce_bits(dtype);
    pp0.swz_bits = dtype == DMV_C64 ? 4 : 3;
    const int64_t gen = tune_value("max_gen_per_pass", -1);
    pp0.max_gen_per_pass = gen > 0 ? (int)gen : 8;
    pp0.gen_auto = gen > 0 ? 0 : 1;
    auto lower = [&](int i, Built &B) -> int {
        const int ni = n[i];
        DMV_CHECK_ARG(ni >= 2 && ni <= 24, "batch circuit %d: qubits must be in [2, 24], got %d", i, ni);
        std::vector<Gate> gates;
        gates.reserve((size_t)(gate_offset[i + 1] - gate_offset[i]));
        for (int g = gate_offset[i]; g < gate_offset[i + 1]; g++) {
            Gate G;
            G.kind = gate_kind[g];
            G.control = gate_control[g];
            G.target = gate_target[g];
            G.p[0] = gate_param[3 * (int64_t)g];
            G.p[1] = gate_param[3 * (int64_t)g + 1];
            G.p[2] = gate_param[3 * (int64_t)g + 2];
            G.observable = false;
            DMV_CHECK_ARG(G.kind >= DMV_GATE_H && G.kind <= DMV_GATE_CZ, "batch circuit %d: bad gate kind", i);
            DMV_CHECK_ARG(G.target >= 0 && G.target < ni, "batch circuit %d: target out of range", i);
            const bool ctl = G.kind == DMV_GATE_CNOT || G.kind == DMV_GATE_CZ;
            DMV_CHECK_ARG(!ctl || (G.control >= 0 && G.control < ni && G.control != G.target),
                          "batch circuit %d: bad control", i);
            if (!ctl)
                G.control = -1;
            gates.push_back(G);
        }
        for (const Gate &G : gates)
            if (gate_is_parametric(G.kind))
                B.np++;
        B.f = merge_ops(forward_ops(gates));
        B.a = merge_ops(adjoint_ops(gates));
        if (B.f.empty()) {
            // the first forward pass also writes |0>: a circuit without gates
            // gets an identity
            HostOp id{OP_DIAG, 0, 0, {1, 0, 0, 0, 0, 0, 1, 0}, -1, false};
            B.f.push_back(id);
        }
        B.key = (uint64_t)ni;
        for (const std::vector<HostOp> *v : {&B.f, &B.a})
            for (const HostOp &op : *v)
                B.key = (B.key ^ (op.kind + 16 * (uint64_t)op.target + 1024 * (op.ctrl + 1))) * 0x9E3779B97F4A7C15ull;
        return DMV_OK;
    };
    auto plan_one = [&](int i, Built &B) -> int {
        PlanParams pp = pp0;
        pp.n = std::max(n[i], K);  // a circuit smaller than a tile leaves qubits idle
        pp.max_ip_per_pass = n[i] >= K ? (int)kBatchMaxIp : pp.max_ip_per_pass;
        DMV_TRY(shared_plan(B.f, pp, &B.pf));
        DMV_TRY(shared_plan(B.a, pp, &B.pa));
        const std::vector<uint32_t> &ip = B.pa->ip_begin;
        for (size_t p = 0; p + 1 < ip.size() && n[i] >= K; p++)
            DMV_CHECK_ARG(ip[p + 1] - ip[p] <= kBatchMaxIp,
                          "batch circuit %d: %u parameters in one reverse pass (at most %u)", i, ip[p + 1] - ip[p],
                          kBatchMaxIp);
        return DMV_OK;
    };
    // fn(i) for i < total, on up to 16 threads with `grain` of them each or more
    auto on_threads = [](int total, int grain, const std::function<void(int)> &fn) {
        const int hw = (int)std::max(1u, std::thread::hardware_concurrency());
        const int nthreads = std::max(1, std::min({hw, 16, total / grain}));
        std::atomic<int> next{0};
        auto worker = [&]() {
            for (int i = next.fetch_add(1); i < total; i = next.fetch_add(1))
                fn(i);
        };
        std::vector<std::thread> pool;
        try {
            for (int t = 1; t < nthreads; t++)
                pool.emplace_back(worker);
        } catch (const std::system_error &) {
            // no more threads to be had: the work is shared by those there are
        }
        worker();
        for (std::thread &t : pool)
            t.join();
    };
    on_threads(count, 16, [&](int i) {
        built[i].rc = lower(i, built[i]);
        if (built[i].rc != DMV_OK)
            built[i].err = last_error();
    });
    for (int i = 0; i < count; i++)
        if (built[i].rc != DMV_OK) {
            set_error("%s", built[i].err.c_str());
            return built[i].rc;
        }
    std::vector<int> firsts;  // circuits of a new structure
    {
        std::unordered_map<uint64_t, int> seen;
        for (int i = 0; i < count; i++)
            built[i].like = seen.emplace(built[i].key, i).first->second;
        on_threads(count, 16, [&](int i) {  // a circuit whose key another structure has goes on its own
            Built &B = built[i];
            const Built &O = built[B.like];
            if (B.like != i &&
                !(n[B.like] == n[i] && same_structure(O.f, B.f) && same_structure(O.a, B.a)))
                B.like = i;
        });
        for (int i = 0; i < count; i++)
            if (built[i].like == i)
                firsts.push_back(i);
    }
    on_threads((int)firsts.size(), 2, [&](int j) {
        Built &B = built[firsts[(size_t)j]];
        B.rc = plan_one(firsts[(size_t)j], B);
        if (B.rc != DMV_OK)
            B.err = last_error();
    });

    std::vector<BatchCircuit> circ(count);
    std::vector<DevPass> passes;
    std::vector<DevPhase> phases;
    std::vector<int> slots;
    int64_t total_params = 0;
    uint64_t n_ops = 0;
    for (int i = 0; i < count; i++) {
        Built &B = built[i];
        if (B.rc != DMV_OK) {
            set_error("%s", B.err.c_str());
            return B.rc;
        }
        if (param_offset[i] != total_params) {
            set_error("param_offset[%d] is %d; it must be the number of parameters of the circuits before it (%lld)", i,
                      param_offset[i], (long long)total_params);
            return DMV_ERR_ARG;
        }
        total_params += B.np;
        if (B.like == i) {
            for (int which = 0; which < 2; which++) {
                const Plan &plan = which == 0 ? *B.pf : *B.pa;
                (which == 0 ? B.fwd : B.adj) = (uint32_t)passes.size();
                const uint32_t phbase = (uint32_t)phases.size();
                for (DevPass P : plan.passes) {
                    P.phase_begin += phbase;
                    P.phase_end += phbase;
                    passes.push_back(P);
                }
                phases.insert(phases.end(), plan.phases.begin(), plan.phases.end());
            }
            B.slots = (uint32_t)slots.size();
            slots.insert(slots.end(), B.pa->ip_slots.begin(), B.pa->ip_slots.end());
        }
        const Built &T = built[B.like];
        BatchCircuit &C = circ[i];
        C.n = (uint32_t)n[i];
        C.index = (uint32_t)i;
        C.coef = (uint32_t)coef_offset[i];
        C.grad = (uint32_t)param_offset[i];
        C.fwd_begin = T.fwd;
        C.adj_begin = T.adj;
        C.n_ip = (uint32_t)T.pa->ip_slots.size();
        C.slots = T.slots;
        C.amps = uint64_t(1) << std::max(n[i], K);
        C.tiles = (uint32_t)(C.amps >> K);
        C.fwd_ops = n_ops;
        C.adj_ops = n_ops + T.pf->ops.size();
        n_ops += T.pf->ops.size() + T.pa->ops.size();
    }
    // Circuits run in groups whose states and partials fit `limit` bytes (one
    // circuit at least): 16 GiB, or tunable batch_pool_mib, and half of what a
    // group took where the device has no room for it.  With the default tiles the
    // 4096-circuit 12-18 qubit batch in complex128 takes 9.8 + 1.3 GB and is
    // one group.
    const int64_t pool_mib = tune_value("batch_pool_mib", 0);
    uint64_t limit = pool_mib > 0 ? (uint64_t)pool_mib << 20 : uint64_t(16) << 30;
    const uint32_t waves = (1u << tlog) / 64;
    struct Group {
        uint32_t first, count;
        uint64_t tile_at;            // first entry in by_fwd / by_adj
        std::vector<uint32_t> fwd_tiles, adj_tiles;
        uint32_t tiles;
    };
    std::vector<Group> groups;
    std::vector<BatchTile> by_fwd, by_adj;
    uint64_t pool_amps = 0, pool_parts = 0, pool_tiles = 0;
    auto make_groups = [&]() -> int {
        groups.clear();
        by_fwd.clear();
        by_adj.clear();
        pool_amps = pool_parts = pool_tiles = 0;
        for (int i = 0; i < count;) {
            Group G{(uint32_t)i, 0, by_fwd.size(), {}, {}, 0};
            uint64_t amps = 0, parts = 0, tiles = 0;
            for (; i < count; i++) {
                BatchCircuit &C = circ[i];
                const uint64_t a2 = amps + 2 * C.amps, p2 = parts + (uint64_t)C.n_ip * C.tiles * waves;
                if (G.count > 0 && a2 * amp_bytes(dtype) + p2 * 8 > limit)
                    break;
                C.state = amps;
                C.parts = parts;
                C.tile0 = (uint32_t)tiles;
                amps = a2;
                parts = p2;
                tiles += C.tiles;
                G.count++;
            }
            DMV_CHECK_ARG(tiles <= 0x7FFFFFFFull, "batch too large");
            G.tiles = (uint32_t)tiles;
            pool_amps = std::max(pool_amps, amps);
            pool_parts = std::max(pool_parts, parts);
            pool_tiles = std::max(pool_tiles, tiles);
            for (int which = 0; which < 2; which++) {
                auto levels = [&](uint32_t c) {
                    const Built &T = built[built[c].like];
                    return (which == 0 ? *T.pf : *T.pa).passes.size();
                };
                std::vector<uint32_t> order(G.count);
                for (uint32_t j = 0; j < G.count; j++)
                    order[j] = G.first + j;
                std::stable_sort(order.begin(), order.end(), [&](uint32_t x, uint32_t y) { return levels(x) > levels(y); });
                std::vector<BatchTile> &list = which == 0 ? by_fwd : by_adj;
                std::vector<uint32_t> &per_level = which == 0 ? G.fwd_tiles : G.adj_tiles;
                per_level.assign(levels(order[0]), 0);
                for (uint32_t c : order) {
                    for (uint32_t t = 0; t < circ[c].tiles; t++)
                        list.push_back({c, t});
                    for (size_t p = 0; p < levels(c); p++)
                        per_level[p] += circ[c].tiles;
                }
            }
            groups.push_back(std::move(G));
        }
        return DMV_OK;
    };
    DMV_TRY(make_groups());

    // host work and argument checks are done: only now touch the device
    DMV_TRY(ensure_device());
    int64_t coef_len = 0;
    for (int i = 0; i < count; i++)
        coef_len = std::max<int64_t>(coef_len, (int64_t)coef_offset[i] + 2 * n[i] - 1);

    // One device buffer: what the host fills in first, so that it goes over in
    // one copy, then the results, partials and states.
    std::unique_ptr<Arena> arena;
    uint64_t o_circ, o_fwd, o_adj, o_passes, o_phases, o_ops, o_slots, o_coef, o_energy, o_grad, o_eparts, o_parts, o_pool;
    for (;;) {
        arena.reset();
        arena.reset(new Arena);
        Arena &A = *arena;
        o_circ = A.part(circ.size() * sizeof(BatchCircuit));
        o_fwd = A.part(by_fwd.size() * sizeof(BatchTile));
        o_adj = A.part(by_adj.size() * sizeof(BatchTile));
        o_passes = A.part(passes.size() * sizeof(DevPass));
        o_phases = A.part(phases.size() * sizeof(DevPhase));
        o_ops = A.part(n_ops * sizeof(DevOp));
        o_slots = A.part(slots.size() * sizeof(int));
        o_coef = A.part((uint64_t)coef_len * sizeof(double));
        o_energy = A.part((uint64_t)count * sizeof(double) + (uint64_t)total_params * sizeof(double));
        o_grad = o_energy + (uint64_t)count * sizeof(double);
        o_eparts = A.part(pool_tiles * sizeof(double));
        o_parts = A.part(pool_parts * sizeof(double));
        o_pool = A.part(pool_amps * (uint64_t)amp_bytes(dtype));
        const int rc = A.get(o_energy);
        if (rc == DMV_OK)
            break;
        if (rc != DMV_ERR_MEMORY || groups.size() == (size_t)count)
            return rc;
        limit = std::min(limit, pool_amps * (uint64_t)amp_bytes(dtype) + pool_parts * sizeof(double)) / 2;
        DMV_TRY(make_groups());
    }
    Arena &A = *arena;
    char *filled = A.host();
    std::memcpy(filled + o_circ, circ.data(), circ.size() * sizeof(BatchCircuit));
    std::memcpy(filled + o_fwd, by_fwd.data(), by_fwd.size() * sizeof(BatchTile));
    std::memcpy(filled + o_adj, by_adj.data(), by_adj.size() * sizeof(BatchTile));
    std::memcpy(filled + o_passes, passes.data(), passes.size() * sizeof(DevPass));
    std::memcpy(filled + o_phases, phases.data(), phases.size() * sizeof(DevPhase));
    std::memcpy(filled + o_slots, slots.data(), slots.size() * sizeof(int));
    std::memcpy(filled + o_coef, coef, (size_t)coef_len * sizeof(double));
    DevOp *ops = (DevOp *)(filled + o_ops);
    on_threads(count, 16, [&](int i) {
        const Built &B = built[i], &T = built[B.like];
        std::vector<DevOp> dev = T.pf->ops;
        refresh_ops(B.f, false, T.pf->op_src, &dev);
        std::copy(dev.begin(), dev.end(), ops + circ[i].fwd_ops);
        dev = T.pa->ops;
        refresh_ops(B.a, false, T.pa->op_src, &dev);
        std::copy(dev.begin(), dev.end(), ops + circ[i].adj_ops);
    });
    DMV_TRY(A.send());

    BatchLaunch L;
    L.circ = A.at<BatchCircuit>(o_circ);
    L.passes = A.at<DevPass>(o_passes);
    L.phases = A.at<DevPhase>(o_phases);
    L.ops = A.at<DevOp>(o_ops);
    L.slots = A.at<int>(o_slots);
    L.coef = A.at<double>(o_coef);
    L.pool = A.at<void>(o_pool);
    L.parts = A.at<double>(o_parts);
    L.energy_parts = A.at<double>(o_eparts);
    L.energy = A.at<double>(o_energy);
    L.grad = A.at<double>(o_grad);
    L.rlog = rlog;
    L.tlog = tlog;
    // streaming loads and stores once the states take twice the last-level
    // cache (512 MiB)
    L.nt = tune_value("nontemporal", pool_amps * amp_bytes(dtype) >= (uint64_t(512) << 20) ? 1 : 0) != 0;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    if (kernel_ms && (hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess)) {
        if (e0)
            (void)hipEventDestroy(e0);
        set_error("hipEventCreate failed");
        return DMV_ERR_HIP;
    }
    if (kernel_ms)
        (void)hipEventRecord(e0, stream());
    prof_begin(DMV_KC_BATCH);
    int rc = DMV_OK;
    for (const Group &G : groups) {
        L.first = G.first;
        L.count = G.count;
        L.by_fwd = A.at<BatchTile>(o_fwd) + G.tile_at;
        L.by_adj = A.at<BatchTile>(o_adj) + G.tile_at;
        L.all_tiles = G.tiles;
        L.fwd_levels = (uint32_t)G.fwd_tiles.size();
        L.adj_levels = (uint32_t)G.adj_tiles.size();
        L.fwd_tiles = G.fwd_tiles.data();
        L.adj_tiles = G.adj_tiles.data();
        if (rc == DMV_OK)
            rc = launch_batch(dtype, L);
    }
    if (kernel_ms) {
        (void)hipEventRecord(e1, stream());
        float ms = 0.f;
        if (rc == DMV_OK && hipEventSynchronize(e1) == hipSuccess)
            (void)hipEventElapsedTime(&ms, e0, e1);
        *kernel_ms = ms;
        (void)hipEventDestroy(e0);
        (void)hipEventDestroy(e1);
    }
    DMV_TRY(rc);
    double bytes = 0.0;
    for (int i = 0; i < count; i++) {
        const double sb = (double)circ[i].amps * amp_bytes(dtype);
        const Built &T = built[built[i].like];
        bytes += 2.0 * sb * T.pf->passes.size() + 4.0 * sb * T.pa->passes.size() + 3.0 * sb;
    }
    prof_end(DMV_KC_BATCH, bytes);
    std::vector<double> out((size_t)count + (size_t)total_params);
    DMV_TRY(copy_d2h(out.data(), A.at<void>(o_energy), out.size() * sizeof(double)));
    A.sent();
    std::copy(out.begin(), out.begin() + count, energy);
    std::copy(out.begin() + count, out.end(), grad);
    return DMV_OK;
}

}  // namespace dmv
