// Batched circuits: every launch runs one pass of all circuits that have it, a
// workgroup per tile, so the whole chip works on whatever circuits are left.
// (One persistent launch whose workgroups each took whole circuits left the
// chip to the last large ones: a workgroup takes about 70 ms for an 18-qubit
// circuit.  1024 circuits of 12-18 qubits, complex128: 102 ms there,
// 34 ms here.)
// Circuits smaller than a tile run as one tile, their idle qubits at zero.
#include "kernels.hpp"
#include "tile_ops.hpp"

namespace dmv {

// The pass `level` of a circuit's forward, over its tiles.  Level 0 starts from
// |0> in registers instead of reading it.  complex64 (S = float) is computed in
// FP64, as in reverse sweeps (see tile_body).
template <class S, int RLOG, int TLOG, bool STREAM>
__global__ void __launch_bounds__(1 << TLOG)
k_batch_forward(const BatchCircuit *__restrict__ circ, const BatchTile *__restrict__ tiles, uint32_t level,
                const DevPass *__restrict__ passes, const DevPhase *__restrict__ phases,
                const DevOp *__restrict__ ops, typename Cplx<S>::T *__restrict__ pool)
{
    constexpr int NR = 1 << RLOG, K = RLOG + TLOG;
    __shared__ c128 lds[1 << K];
    const uint32_t tid = threadIdx.x;
    const BatchTile T = tiles[blockIdx.x];
    const BatchCircuit *C = circ + T.circuit;
    const DevPass *P = passes + C->fwd_begin + level;
    typename Cplx<S>::T *psi = pool + C->state;
    const uint64_t g = tile_base<K>(P, T.tile);
    const uint64_t gl = g | thread_global_offset<TLOG>(P->gthr_ld, tid);
    c128 v[NR];
    if (level == 0) {
#pragma unroll
        for (int r = 0; r < NR; r++)
            v[r] = c128{(gl ^ P->greg_ld[r]) == 0 ? 1.0 : 0.0, 0.0};
    } else {
        load_tile<STREAM>(v, psi, gl, P->greg_ld, kPlainLayout);
    }
    process_tile<S, double, RLOG, TLOG, false>(v, P, phases, ops + C->fwd_ops, lds);
    store_tile<STREAM>(v, psi, g | thread_global_offset<TLOG>(P->gthr_st, tid), P->greg_st, kPlainLayout);
}

// lambda = h psi for the chain observable h(x) = sum_q a_q z_q + sum_{q<n-1} b_q
// z_q z_{q+1}, and each tile's part of the energy (a tile here: 2^K amplitudes
// in a row).  The terms of the tile's high bits are summed once.
template <class S, int K>
__global__ void __launch_bounds__(256)
k_batch_obs(const BatchCircuit *__restrict__ circ, const BatchTile *__restrict__ tiles, const double *__restrict__ coef,
            typename Cplx<S>::T *__restrict__ pool, double *__restrict__ energy_parts)
{
    using ST = typename Cplx<S>::T;
    __shared__ double red[4];
    const BatchTile T = tiles[blockIdx.x];
    const BatchCircuit *C = circ + T.circuit;
    const uint32_t n = C->n, low = n < (uint32_t)K ? n : (uint32_t)K;
    const double *a = coef + C->coef, *b = a + n;
    const ST *psi = pool + C->state + ((uint64_t)T.tile << K);
    ST *lam = pool + C->state + C->amps + ((uint64_t)T.tile << K);
    double hi = 0.0;
    for (uint32_t q = low; q < n; q++) {
        const uint32_t bq = (T.tile >> (q - K)) & 1u;
        hi += bq ? -a[q] : a[q];
        if (q + 1 < n)
            hi += (bq ^ ((T.tile >> (q + 1 - K)) & 1u)) ? -b[q] : b[q];
    }
    const double edge = low < n ? ((T.tile & 1u) ? -b[low - 1] : b[low - 1]) : 0.0;  // b z of the first high bit
    double acc = 0.0;
    for (uint32_t i = threadIdx.x; i < (1u << K); i += 256) {
        double h = hi;
        for (uint32_t q = 0; q < low; q++) {
            const uint32_t bq = (i >> q) & 1u;
            h += bq ? -a[q] : a[q];
            const double bb = q + 1 < low ? (((i >> (q + 1)) & 1u) ? -b[q] : b[q]) : edge;
            h += bq ? -bb : bb;
        }
        const ST v = psi[i];
        acc += h * norm2(v);
        ST w;
        w.x = v.x * h;
        w.y = v.y * h;
        lam[i] = w;
    }
    acc = block_sum<256>(acc, red);
    if (threadIdx.x == 0)
        energy_parts[C->tile0 + T.tile] = acc;
}

// One partial per (IP op of the circuit, tile, wave).
struct BatchSink {
    double *parts;  // of the pass's first IP op, at this tile
    uint64_t per_ip;
    __device__ void operator()(const DevOp *op, double v, uint32_t wave) const
    {
        parts[(uint64_t)op->aux * per_ip + wave] = v;
    }
};

// The pass `level` of a circuit's reverse sweep.
template <class S, int RLOG, int TLOG, bool STREAM>
__global__ void __launch_bounds__(1 << TLOG)
k_batch_reverse(const BatchCircuit *__restrict__ circ, const BatchTile *__restrict__ tiles, uint32_t level,
                const DevPass *__restrict__ passes, const DevPhase *__restrict__ phases,
                const DevOp *__restrict__ ops, typename Cplx<S>::T *__restrict__ pool, double *__restrict__ parts)
{
    constexpr uint32_t W = (1u << TLOG) / 64;
    __shared__ c128 lds[1 << (RLOG + TLOG)];
    const BatchTile T = tiles[blockIdx.x];
    const BatchCircuit *C = circ + T.circuit;
    const DevPass *P = passes + C->adj_begin + level;
    const uint64_t per_ip = (uint64_t)C->tiles * W;
    BatchSink sink{parts + C->parts + P->ip_begin * per_ip + (uint64_t)T.tile * W, per_ip};
    typename Cplx<S>::T *psi = pool + C->state;
    tile_body_adjoint<S, double, RLOG, TLOG, STREAM>(psi, psi + C->amps, P, phases, ops + C->adj_ops, T.tile, lds, sink,
                                                     kPlainLayout);
}

// A circuit's gradient entries and energy: a wave per IP op, in a fixed order.
constexpr int kSumThreads = 1024;
__global__ void __launch_bounds__(kSumThreads)
k_batch_sums(const BatchCircuit *__restrict__ circ, uint32_t first, const int *__restrict__ slots, uint32_t waves,
             const double *__restrict__ parts, const double *__restrict__ energy_parts, double *__restrict__ energy,
             double *__restrict__ grad)
{
    const BatchCircuit *C = circ + first + blockIdx.x;
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t per_ip = C->tiles * waves;
    for (uint32_t i = threadIdx.x >> 6; i <= C->n_ip; i += kSumThreads / 64) {
        const bool is_energy = i == C->n_ip;
        const double *p = is_energy ? energy_parts + C->tile0 : parts + C->parts + (uint64_t)i * per_ip;
        const uint32_t count = is_energy ? C->tiles : per_ip;
        double s = 0.0;
        for (uint32_t t = lane; t < count; t += 64)
            s += p[t];
        s = wave_sum_rows(s);
        if (lane == 0) {
            if (is_energy)
                energy[C->index] = s;
            else
                grad[C->grad + (uint32_t)slots[C->slots + i]] = s;
        }
    }
}

template <class S, int RLOG, int TLOG, bool STREAM = false>
static int run_batch(const BatchLaunch &L)
{
    using ST = typename Cplx<S>::T;
    ST *pool = (ST *)L.pool;
    for (uint32_t p = 0; p < L.fwd_levels; p++) {
        hipLaunchKernelGGL((k_batch_forward<S, RLOG, TLOG, STREAM>), dim3(L.fwd_tiles[p]), dim3(1 << TLOG), 0, stream(),
                           L.circ, L.by_fwd, p, L.passes, L.phases, L.ops, pool);
        DMV_TRY(check_launch("batch forward"));
    }
    hipLaunchKernelGGL((k_batch_obs<S, RLOG + TLOG>), dim3(L.all_tiles), dim3(256), 0, stream(), L.circ, L.by_fwd, L.coef,
                       pool, L.energy_parts);
    DMV_TRY(check_launch("batch observable"));
    for (uint32_t p = 0; p < L.adj_levels; p++) {
        hipLaunchKernelGGL((k_batch_reverse<S, RLOG, TLOG, STREAM>), dim3(L.adj_tiles[p]), dim3(1 << TLOG), 0, stream(),
                           L.circ, L.by_adj, p, L.passes, L.phases, L.ops, pool, L.parts);
        DMV_TRY(check_launch("batch reverse sweep"));
    }
    hipLaunchKernelGGL(k_batch_sums, dim3(L.count), dim3(kSumThreads), 0, stream(), L.circ, L.first, L.slots,
                       (1u << TLOG) / 64, L.parts, L.energy_parts, L.energy, L.grad);
    return check_launch("batch sums");
}

// Tile shapes (log2 amplitudes per thread and state, log2 threads) of the
// batched kernels: 8 amplitudes per thread and state at most, since the
// reverse sweep holds psi and lambda in registers together.
#define DMV_BATCH_SHAPES(X) X(3, 8) X(2, 8) X(3, 7) X(3, 9)

bool batch_kernel_exists(int dtype, int rlog, int tlog)
{
    (void)dtype;
#define DMV_BATCH_HAS(R, T)                                                                        \
    if (rlog == R && tlog == T)                                                                    \
        return true;
    DMV_BATCH_SHAPES(DMV_BATCH_HAS)
#undef DMV_BATCH_HAS
    return false;
}

int launch_batch(int dtype, const BatchLaunch &L)
{
    DMV_CHECK_ARG(L.count >= 1 && L.all_tiles >= 1, "empty batch");
    // the default shape also comes with streaming loads and stores; the
    // other shapes (tunables) take the hint as a no-op
    if (L.nt && L.rlog == 3 && L.tlog == 8)
        return dtype == DMV_C64 ? run_batch<float, 3, 8, true>(L) : run_batch<double, 3, 8, true>(L);
#define DMV_BATCH_RUN(R, T)                                                                        \
    if (L.rlog == R && L.tlog == T)                                                                \
        return dtype == DMV_C64 ? run_batch<float, R, T>(L) : run_batch<double, R, T>(L);
    DMV_BATCH_SHAPES(DMV_BATCH_RUN)
#undef DMV_BATCH_RUN
    set_error("no batched kernel for rlog %d tlog %d", L.rlog, L.tlog);
    return DMV_ERR_ARG;
}

}  // namespace dmv
