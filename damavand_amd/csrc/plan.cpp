// Circuit lowering and the fused-pass scheduler.  Host C++ only.
#include "plan.hpp"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <functional>
#include <mutex>
#include <unordered_map>

namespace dmv {

bool gate_is_parametric(int kind)
{
    return kind == DMV_GATE_RX || kind == DMV_GATE_RY || kind == DMV_GATE_RZ;
}

int gate_num_params(int kind)
{
    if (gate_is_parametric(kind))
        return 1;
    if (kind == DMV_GATE_U3)
        return 3;
    return 0;
}

// Matrices of src/qubit_backend/gates.rs (H :98-119, CNOT :170-174,
// X :224-233, Y :289-298, Z :353-362, RX :418-439, RY :490-511, RZ :562-577,
// S :627-636, T :685-697, Identity :40-49).  U3 and CZ are additions.
int gate_matrix(int kind, const double *p, double m[8])
{
    const double t = p ? p[0] : 0.0;
    for (int i = 0; i < 8; i++)
        m[i] = 0.0;
    switch (kind) {
    case DMV_GATE_ID:
        m[0] = 1.0; m[6] = 1.0;
        return DMV_OK;
    case DMV_GATE_H:
        m[0] = 1.0 / std::sqrt(2.0); m[2] = 1.0 / std::sqrt(2.0);
        m[4] = 1.0 / std::sqrt(2.0); m[6] = -1.0 / std::sqrt(2.0);
        return DMV_OK;
    case DMV_GATE_X:
    case DMV_GATE_CNOT:
        m[2] = 1.0; m[4] = 1.0;
        return DMV_OK;
    case DMV_GATE_Y:
        m[3] = -1.0; m[5] = 1.0;
        return DMV_OK;
    case DMV_GATE_Z:
    case DMV_GATE_CZ:
        m[0] = 1.0; m[6] = -1.0;
        return DMV_OK;
    case DMV_GATE_RX:
        m[0] = std::cos(t / 2.0); m[3] = -std::sin(t / 2.0);
        m[5] = -std::sin(t / 2.0); m[6] = std::cos(t / 2.0);
        return DMV_OK;
    case DMV_GATE_RY:
        m[0] = std::cos(t / 2.0); m[2] = -std::sin(t / 2.0);
        m[4] = std::sin(t / 2.0); m[6] = std::cos(t / 2.0);
        return DMV_OK;
    case DMV_GATE_RZ:
        m[0] = std::cos(-t / 2.0); m[1] = std::sin(-t / 2.0);
        m[6] = std::cos(t / 2.0); m[7] = std::sin(t / 2.0);
        return DMV_OK;
    case DMV_GATE_S:
        m[0] = 1.0; m[7] = 1.0;
        return DMV_OK;
    case DMV_GATE_T:
        m[0] = 1.0; m[6] = std::sqrt(2.0) / 2.0; m[7] = std::sqrt(2.0) / 2.0;
        return DMV_OK;
    case DMV_GATE_U3: {
        const double th = p[0], ph = p[1], la = p[2];
        const double c = std::cos(th / 2.0), s = std::sin(th / 2.0);
        m[0] = c;
        m[2] = -std::cos(la) * s; m[3] = -std::sin(la) * s;
        m[4] = std::cos(ph) * s; m[5] = std::sin(ph) * s;
        m[6] = std::cos(ph + la) * c; m[7] = std::sin(ph + la) * c;
        return DMV_OK;
    }
    default:
        set_error("unknown gate kind %d", kind);
        return DMV_ERR_ARG;
    }
}

uint32_t gate_class(int kind)
{
    switch (kind) {
    case DMV_GATE_X:
    case DMV_GATE_CNOT:
        return OP_SWAP;
    case DMV_GATE_Z:
    case DMV_GATE_CZ:
    case DMV_GATE_RZ:
    case DMV_GATE_S:
    case DMV_GATE_T:
    case DMV_GATE_ID:
        return OP_DIAG;
    default:
        return OP_GEN;
    }
}

static HostOp gate_op(const Gate &g)
{
    HostOp op;
    op.kind = gate_class(g.kind);
    op.target = g.target;
    op.ctrl = g.control >= 0 ? (uint64_t(1) << g.control) : 0;
    gate_matrix(g.kind, g.p, op.m);
    op.slot = -1;
    return op;
}

std::vector<HostOp> forward_ops(const std::vector<Gate> &gates)
{
    std::vector<HostOp> out;
    out.reserve(gates.size());
    for (const Gate &g : gates)
        if (!g.observable)
            out.push_back(gate_op(g));
    return out;
}

// Conjugate transpose of a 2x2 stored as m00 m01 m10 m11 (re, im).
static void dagger(const double m[8], double d[8])
{
    d[0] = m[0]; d[1] = -m[1];   // d00 = conj(m00)
    d[2] = m[4]; d[3] = -m[5];   // d01 = conj(m10)
    d[4] = m[2]; d[5] = -m[3];   // d10 = conj(m01)
    d[6] = m[6]; d[7] = -m[7];   // d11 = conj(m11)
}

static void matmul2(const double a[8], const double b[8], double c[8]);

// Reverse sweep with every IP op moved to the start of its qubit's run of
// uncontrolled one-qubit ops.  Within such a run the state at the IP's own
// place is U psi, U the product of the run's ops before it (both psi and
// lambda carry it), so Im<U lambda|P|U psi> = Im<lambda|U^dag P U|psi> with
// U^dag P U = ax X + ay Y + az Z (Hermitian, traceless, real coefficients).
// Ops on other qubits commute with all of this.  The run's ops then merge
// into one 2x2 (merge_ops) and the run's IP ops share one pass over the
// registers: an RY/RZ layer's reverse step is one GEN and one IP group
// instead of two IP ops, a GEN and a diagonal.
static std::vector<HostOp> hoist_ips(const std::vector<HostOp> &ops, int n)
{
    struct Run {
        bool open = false;
        double U[8];
        int group = -1;
    };
    struct Group {
        int first = -1, last = -1;  // its IP ops, a list in `ips`
        bool general = false;       // one of them has an X or Y part
    };
    std::vector<Run> run(n);
    std::vector<Group> groups;
    std::vector<HostOp> ips;
    std::vector<int> next;   // of each entry of ips
    std::vector<int> where;  // per output entry: -1 - group, or the index of an op
    ips.reserve(ops.size() / 2);
    next.reserve(ops.size() / 2);
    where.reserve(ops.size() + (size_t)n);
    auto open_run = [&](int q) {
        Run &R = run[q];
        if (R.open)
            return;
        R.open = true;
        const double I[8] = {1, 0, 0, 0, 0, 0, 1, 0};
        std::memcpy(R.U, I, sizeof(I));
        R.group = (int)groups.size();
        groups.emplace_back();
        where.push_back(-1 - R.group);
    };
    for (size_t i = 0; i < ops.size(); i++) {
        const HostOp &op = ops[i];
        const int q = op.target;
        if (op_is_ip(op.kind)) {
            open_run(q);
            Run &R = run[q];
            // A = U^dag P U with P = ax X + ay Y + az Z from op.m[0..2]
            const double P[8] = {op.m[2], 0.0, op.m[0], -op.m[1], op.m[0], op.m[1], -op.m[2], 0.0};
            double Ud[8], t[8], A[8];
            Ud[0] = R.U[0]; Ud[1] = -R.U[1]; Ud[2] = R.U[4]; Ud[3] = -R.U[5];
            Ud[4] = R.U[2]; Ud[5] = -R.U[3]; Ud[6] = R.U[6]; Ud[7] = -R.U[7];
            matmul2(P, R.U, t);
            matmul2(Ud, t, A);
            HostOp ip = op;
            std::memset(ip.m, 0, sizeof(ip.m));
            ip.m[0] = A[4];  // A10 = ax + i ay
            ip.m[1] = A[5];
            ip.m[2] = A[0];  // A00 = az
            Group &G = groups[(size_t)R.group];
            G.general = G.general || ip.m[0] != 0.0 || ip.m[1] != 0.0;
            (G.last >= 0 ? next[(size_t)G.last] : G.first) = (int)ips.size();
            G.last = (int)ips.size();
            ips.push_back(ip);
            next.push_back(-1);
            continue;
        }
        if (op.ctrl == 0) {
            open_run(q);
            Run &R = run[q];
            double nu[8];
            matmul2(op.m, R.U, nu);  // op acts after the run so far
            std::memcpy(R.U, nu, sizeof(nu));
        } else {
            run[q].open = false;
            for (uint64_t m = op.ctrl; m; m &= m - 1)
                run[__builtin_ctzll(m)].open = false;
        }
        where.push_back((int)i);
    }
    std::vector<HostOp> out;
    out.reserve(ops.size());
    for (int w : where) {
        if (w >= 0) {
            out.push_back(ops[(size_t)w]);
            continue;
        }
        // one kind per group, so that the kernel computes its sums once
        const Group &G = groups[(size_t)(-1 - w)];
        for (int i = G.first; i >= 0; i = next[(size_t)i]) {
            ips[(size_t)i].kind = G.general ? OP_IPG : OP_IPZ;
            out.push_back(ips[(size_t)i]);
        }
    }
    return out;
}

std::vector<HostOp> adjoint_ops(const std::vector<Gate> &gates)
{
    // parameter index of every gate
    std::vector<int> pidx(gates.size(), -1);
    int np = 0, n = 1;
    for (size_t i = 0; i < gates.size(); i++) {
        if (gate_is_parametric(gates[i].kind))
            pidx[i] = np++;
        n = std::max(n, std::max(gates[i].target, gates[i].control) + 1);
    }
    std::vector<HostOp> out;
    out.reserve(2 * gates.size());
    for (size_t j = gates.size(); j-- > 0;) {
        const Gate &g = gates[j];
        if (g.observable)
            continue;
        if (pidx[j] >= 0) {
            // dE/dtheta = Im<lambda|P|psi> for e^{-i theta P / 2}, P on the target
            HostOp ip;
            ip.kind = g.kind == DMV_GATE_RZ ? OP_IPZ : OP_IPG;
            ip.target = g.target;
            ip.ctrl = 0;
            std::memset(ip.m, 0, sizeof(ip.m));
            ip.m[g.kind == DMV_GATE_RX ? 0 : (g.kind == DMV_GATE_RY ? 1 : 2)] = 1.0;
            ip.slot = pidx[j];
            out.push_back(ip);
        }
        HostOp op = gate_op(g);
        double d[8];
        dagger(op.m, d);
        std::memcpy(op.m, d, sizeof(d));
        out.push_back(op);
    }
    return tune_value("adjoint_hoist", 1) ? hoist_ips(out, n) : out;
}

// c = a * b for 2x2 complex matrices.
static void matmul2(const double a[8], const double b[8], double c[8])
{
    for (int i = 0; i < 2; i++)
        for (int j = 0; j < 2; j++) {
            double re = 0.0, im = 0.0;
            for (int l = 0; l < 2; l++) {
                const double ar = a[2 * (2 * i + l)], ai = a[2 * (2 * i + l) + 1];
                const double br = b[2 * (2 * l + j)], bi = b[2 * (2 * l + j) + 1];
                re += ar * br - ai * bi;
                im += ar * bi + ai * br;
            }
            c[2 * (2 * i + j)] = re;
            c[2 * (2 * i + j) + 1] = im;
        }
}

static uint32_t merged_class(uint32_t earlier, uint32_t later)
{
    if (earlier == OP_DIAG && later == OP_DIAG)
        return OP_DIAG;
    if (earlier == OP_SWAP && later == OP_SWAP)
        return OP_DIAG;  // X * X = I exactly
    return OP_GEN;
}

std::vector<HostOp> merge_ops(const std::vector<HostOp> &ops)
{
    std::vector<HostOp> out;
    out.reserve(ops.size());
    int pending[64];
    for (int &p : pending)
        p = -1;
    for (const HostOp &op : ops) {
        const bool one_qubit = op.ctrl == 0 && !op_is_ip(op.kind);
        if (one_qubit) {
            const int pi = pending[op.target];
            if (pi >= 0) {
                HostOp &prev = out[pi];
                double c[8];
                matmul2(op.m, prev.m, c);
                std::memcpy(prev.m, c, sizeof(c));
                prev.kind = merged_class(prev.kind, op.kind);
                continue;
            }
            out.push_back(op);
            pending[op.target] = (int)out.size() - 1;
        } else {
            out.push_back(op);
            pending[op.target] = -1;
            for (uint64_t m = op.ctrl; m; m &= m - 1)
                pending[__builtin_ctzll(m)] = -1;
        }
    }
    return out;
}

// Writes m / p as special unitary, the mean of what m00 and m11*, m10 and -m01*
// say (equal up to rounding), and returns the phase that the mean drops (about
// the rounding of p).
template <class R> static R su2_mean(double *m, R pr, R pi)
{
    auto over = [&](R x, R y, R *re, R *im) {
        *re = x * pr + y * pi;
        *im = y * pr - x * pi;
    };
    R ar, ai, cr, ci, br, bi, er, ei;
    over(m[0], m[1], &ar, &ai);
    over(m[6], m[7], &cr, &ci);
    over(m[4], m[5], &br, &bi);
    over(m[2], m[3], &er, &ei);
    m[0] = (double)((ar + cr) / 2);
    m[1] = (double)((ai - ci) / 2);
    m[4] = (double)((br - er) / 2);
    m[5] = (double)((bi + ei) / 2);
    m[2] = -m[4];
    m[3] = m[5];
    m[6] = m[0];
    m[7] = -m[1];
    return (m[0] * (ai + ci) + m[1] * (cr - ar) + m[4] * (bi - ei) - m[5] * (br + er)) / 2;
}

// Determinants other than 1 are taken out in 80 bits: in 64 the matrices would
// be rounded twice more than the gates are (9 to 12 qubits, U3 and CNOT: 13% more
// error in the amplitudes than without, and now 13% less).
void special_unitary(std::vector<HostOp> *ops)
{
    using R = long double;
    R gr = 1, gi = 0;  // product of the phases taken out
    R drop = 0;        // ... and the sum of the small ones, apart from it: it would round them away
    HostOp *general = nullptr;
    for (HostOp &op : *ops) {
        if (op.kind != OP_GEN || op.ctrl)
            continue;
        double *m = op.m;
        const double dr = m[0] * m[6] - m[1] * m[7] - m[2] * m[4] + m[3] * m[5];
        const double di = m[0] * m[7] + m[1] * m[6] - m[2] * m[5] - m[3] * m[4];
        if (!(std::abs(std::hypot(dr, di) - 1.0) < 1e-12))
            continue;  // not unitary: stays as it is
        op.su2 = true;
        if (std::abs(dr - 1.0) < 1e-13 && std::abs(di) < 1e-13) {
            drop += su2_mean<double>(m, 1.0, 0.0);
            if (!general)
                general = &op;
            continue;
        }
        // p = sqrt(det) by half angles (no cancellation), m / p is special unitary
        R er = (R)m[0] * m[6] - (R)m[1] * m[7] - (R)m[2] * m[4] + (R)m[3] * m[5];
        R ei = (R)m[0] * m[7] + (R)m[1] * m[6] - (R)m[2] * m[5] - (R)m[3] * m[4];
        const R abs = std::sqrt(er * er + ei * ei);
        er /= abs;
        ei /= abs;
        R pr, pi;
        if (er >= 0) {
            pr = std::sqrt((1 + er) / 2);
            pi = ei / (2 * pr);
        } else {
            pi = std::sqrt((1 - er) / 2);
            pr = ei / (2 * pi);
        }
        drop += su2_mean<R>(m, pr, pi);
        const R t = gr * pr - gi * pi;
        gi = gr * pi + gi * pr;
        gr = t;
        general = &op;
    }
    if (!general || (gr == 1 && gi == 0 && std::abs(drop) < 1e-16L))
        return;
    const R t = gr - gi * drop;
    gi += gr * drop;
    gr = t;
    general->su2 = false;
    for (int i = 0; i < 4; i++) {
        const R x = general->m[2 * i], y = general->m[2 * i + 1];
        general->m[2 * i] = (double)(x * gr - y * gi);
        general->m[2 * i + 1] = (double)(x * gi + y * gr);
    }
}

static uint64_t op_qubits(const HostOp &op) { return (uint64_t(1) << op.target) | op.ctrl; }

static uint64_t deposit(uint64_t x, const uint32_t *pos, int nbits)
{
    uint64_t r = 0;
    for (int j = 0; j < nbits; j++)
        if ((x >> j) & 1)
            r |= uint64_t(1) << pos[j];
    return r;
}

// Builds the register/thread layout of a phase whose register bits are `rs`.
// coalesced: thread bits 0..low_bits-1 are local bits 0..low_bits-1 (they
// must not be register bits); otherwise thread bits 0..swz_bits-1 get local
// bits with distinct residues mod swz_bits, which keeps 128-bit LDS accesses
// of consecutive lanes in distinct banks under the swizzle of the kernels.
// top >= 0: local bit `top` (not in rs) takes the highest thread bit.
static DevLayout make_layout(uint32_t rs, const PlanParams &pp, bool coalesced, int top)
{
    DevLayout L;
    std::memset(&L, 0, sizeof(L));
    uint32_t regbits[kMaxRegs];
    int nr = 0;
    for (int b = 0; b < pp.k; b++)
        if ((rs >> b) & 1)
            regbits[nr++] = (uint32_t)b;
    for (int r = 0; r < (1 << pp.rlog); r++)
        L.lreg[r] = (uint32_t)deposit((uint64_t)r, regbits, nr);
    std::vector<int> tb;
    for (int b = 0; b < pp.k; b++)
        if (!((rs >> b) & 1) && b != top)
            tb.push_back(b);
    std::vector<int> order;
    if (coalesced) {
        for (int b = 0; b < pp.low_bits; b++)
            order.push_back(b);
    } else {
        for (int c = 0; c < pp.swz_bits && (int)order.size() < (int)tb.size(); c++)
            for (int b : tb)
                if (b % pp.swz_bits == c && std::find(order.begin(), order.end(), b) == order.end()) {
                    order.push_back(b);
                    break;
                }
    }
    for (int b : tb)
        if (std::find(order.begin(), order.end(), b) == order.end())
            order.push_back(b);
    if (top >= 0)
        order.push_back(top);
    for (int j = 0; j < pp.tlog; j++)
        L.thr[j] = (uint32_t)order[j];
    const uint32_t elem = pp.swz_bits == 3 ? 16u : 8u;
    for (int r = 0; r < (1 << pp.rlog); r++)
        L.lswz[r] = (pp.swz_bits == 3 ? swz_index<3>(L.lreg[r]) : swz_index<4>(L.lreg[r])) * elem;
    return L;
}

// Register bit of a local bit in a layout, or kNoReg.
static uint32_t register_bit(const DevLayout &L, const PlanParams &pp, uint32_t lbit)
{
    for (int j = 0; j < pp.rlog; j++)
        if (L.lreg[1 << j] == (1u << lbit))
            return (uint32_t)j;
    return kNoReg;
}

// Thread bit of a local bit in a layout, or kNoReg.
static uint32_t thread_bit(const DevLayout &L, const PlanParams &pp, uint32_t lbit)
{
    for (int j = 0; j < pp.tlog; j++)
        if (L.thr[j] == lbit)
            return (uint32_t)j;
    return kNoReg;
}

static bool layouts_equal(const DevLayout &a, const DevLayout &b, const PlanParams &pp)
{
    for (int r = 0; r < (1 << pp.rlog); r++)
        if (a.lreg[r] != b.lreg[r])
            return false;
    for (int j = 0; j < pp.tlog; j++)
        if (a.thr[j] != b.thr[j])
            return false;
    return true;
}

// Pads a register set to rlog bits, preferring the highest local bits that
// are not kept in lanes for coalescing, and never taking the bits of `avoid`.
static uint32_t pad_regs(uint32_t rs, const PlanParams &pp, uint32_t avoid)
{
    for (int b = pp.k - 1; b >= pp.low_bits && popcount64(rs) < pp.rlog; b--)
        if (!((avoid >> b) & 1))
            rs |= 1u << b;
    for (int b = 0; b < pp.k && popcount64(rs) < pp.rlog; b++)
        if (!((avoid >> b) & 1))
            rs |= 1u << b;
    return rs;
}

// Registers p with the highest set bit of partner mask m clear: the first
// member of each pair (p, p ^ m) as the kernels enumerate pairs.
static uint32_t first_members(uint32_t m, int nr)
{
    uint32_t hb = 1;
    while ((hb << 1) <= m)
        hb <<= 1;
    uint32_t f = 0;
    for (int p = 0; p < nr; p++)
        if (!(p & hb))
            f |= 1u << p;
    return f;
}

// ------------------------------------------------------------- scheduling --
// Ops as the scheduler sees them: which bits an op touches, and which bit must
// be in registers.  Two ops that share a bit keep their order; ops on
// disjoint bits commute.
struct SchedOp {
    uint64_t bits;     // target and controls
    uint64_t ctrl;     // controls
    int target;
    uint32_t kind;
    int weight;        // progress that running it counts for
    int group;         // an IP op: how many its run of IP ops on the target has from here on
};

// Every bit's ops in order, and how far each bit has got.  An op can run once
// it is the next one of all its bits.
struct Frontier {
    const std::vector<SchedOp> *ops;
    std::vector<int> list;      // op indices, bit after bit
    int begin[kMaxQubits], end[kMaxQubits];  // each bit's range in `list`
    int at[kMaxQubits];                      // ... and its next op

    void build(const std::vector<SchedOp> &o, int n)
    {
        ops = &o;
        int count[kMaxQubits] = {};
        for (const SchedOp &op : o)
            for (uint64_t m = op.bits; m; m &= m - 1)
                count[__builtin_ctzll(m)]++;
        int total = 0;
        for (int q = 0; q < kMaxQubits; q++) {
            begin[q] = end[q] = at[q] = total;
            total += q < n ? count[q] : 0;
        }
        list.resize((size_t)total);
        for (size_t i = 0; i < o.size(); i++)
            for (uint64_t m = o[i].bits; m; m &= m - 1)
                list[(size_t)end[__builtin_ctzll(m)]++] = (int)i;
    }
    int next(const int *pos, int q) const { return pos[q] < end[q] ? list[(size_t)pos[q]] : -1; }
};

// What a pass or phase may hold.
struct SchedLimits {
    int max_gen = 1 << 30;      // general 2x2 ops
    int max_ip = 1 << 30;       // IP ops (an op of a run is counted with the rest of its run)
    int max_high_targets = 64;  // register targets outside `low`
    uint64_t low = 0;
};

// A trial: the bits it may use, how far it has got, and what it holds.
struct Trial {
    uint64_t bits = 0;      // pass: the tile's qubits; phase: the register bits
    int pos[kMaxQubits];
    int score = 0, gen = 0, ip = 0;
    uint64_t targets = 0;   // bits that need a register
};

// Whether op i, the next one of bit q, can run now.  Passes: all its bits must
// be in the tile.  Phases: the target of a pair op must be a register bit, and
// with `renames_only` an X or CNOT also needs its control in registers (it
// then only relabels registers).
template <bool PHASE>
static bool can_run(const Frontier &F, const SchedLimits &lim, bool renames_only, const Trial &t, int i)
{
    const SchedOp &op = (*F.ops)[(size_t)i];
    if constexpr (PHASE) {
        if (op_needs_register(op.kind) &&
            (!((t.bits >> op.target) & 1) || (renames_only && op.kind == OP_SWAP && (op.ctrl & ~t.bits))))
            return false;
    } else {
        if (op.bits & ~t.bits)
            return false;
    }
    for (uint64_t m = op.bits; m; m &= m - 1)
        if (F.next(t.pos, __builtin_ctzll(m)) != i)
            return false;
    if constexpr (!PHASE) {
        const uint64_t targets = op_needs_register(op.kind) ? t.targets | (uint64_t(1) << op.target) : t.targets;
        return !(op.kind == OP_GEN && t.gen >= lim.max_gen) &&
               !(op.group > 0 && t.ip > 0 && t.ip + op.group > lim.max_ip) &&
               popcount64(targets & ~lim.low) <= lim.max_high_targets;
    }
    return true;
}

// Runs every op that the trial's bits allow.  `dirty`: the bits to look at first.
template <bool PHASE>
static void run_trial(const Frontier &F, const SchedLimits &lim, bool renames_only, uint64_t dirty, Trial &t,
                      std::vector<int> *taken)
{
    while (dirty) {
        const int q = __builtin_ctzll(dirty);
        const int i = F.next(t.pos, q);
        if (i < 0 || !can_run<PHASE>(F, lim, renames_only, t, i)) {
            dirty &= dirty - 1;
            continue;
        }
        const SchedOp &op = (*F.ops)[(size_t)i];
        for (uint64_t m = op.bits; m; m &= m - 1)
            t.pos[__builtin_ctzll(m)]++;
        t.score += op.weight;
        t.gen += op.kind == OP_GEN;
        t.ip += op_is_ip(op.kind);
        if (op_needs_register(op.kind))
            t.targets |= uint64_t(1) << op.target;
        if (taken)
            taken->push_back(i);
        dirty |= op.bits;
    }
}

// Grows a trial by one bit at a time, each time by the bit that lets it run
// the most; where none lets it run anything, by the bit whose next op is the
// oldest.  `width`: how many bits it may have; `allowed`: which.
template <bool PHASE>
static void grow_trial(const Frontier &F, const SchedLimits &lim, bool renames_only, int n, uint64_t allowed, int width,
                       Trial &t)
{
    run_trial<PHASE>(F, lim, renames_only, PHASE ? ((uint64_t(1) << n) - 1) : t.bits, t, nullptr);
    Trial best, u;
    while (popcount64(t.bits) < width) {
        int best_gain = -1, best_old = 0;
        uint64_t best_bit = 0;
        for (uint64_t m = allowed & ~t.bits; m; m &= m - 1) {
            const uint64_t bit = m & -m;
            const int q = __builtin_ctzll(m);
            const int first = F.next(t.pos, q);
            if (first < 0)
                continue;
            // whatever the new bit lets run starts with its own next op
            t.bits |= bit;
            const bool runs = can_run<PHASE>(F, lim, renames_only, t, first);
            int gain = 0;
            if (runs) {
                u = t;
                run_trial<PHASE>(F, lim, renames_only, bit, u, nullptr);
                gain = u.score - t.score;
            }
            t.bits &= ~bit;
            if (gain > best_gain || (gain == best_gain && first < best_old)) {
                if (runs)
                    best = u;
                best_gain = gain;
                best_old = first;
                best_bit = bit;
            }
        }
        if (best_gain < 0 || (PHASE && best_gain == 0))
            break;
        if (best_gain > 0)
            t = best;
        else
            t.bits |= best_bit;
    }
}

// The bits of the next pass (PHASE = false) or phase: trials grown from
// `start` alone and from the bits of the next few two-bit ops, the one that
// gets furthest.
template <bool PHASE>
static Trial pick_bits(const Frontier &F, const SchedLimits &lim, bool renames_only, int n, uint64_t start,
                       uint64_t allowed, int width)
{
    constexpr int kSeeds = PHASE ? 2 : 4;
    uint64_t seeds[kSeeds + 1] = {0};
    int n_seeds = 1;
    const std::vector<SchedOp> &ops = *F.ops;
    int cand[kMaxQubits], nc = 0;
    for (int q = 0; q < n; q++)
        for (int p = F.at[q]; p < F.end[q]; p++) {
            const int i = F.list[(size_t)p];
            if (ops[(size_t)i].ctrl) {
                cand[nc++] = i;
                break;
            }
        }
    std::sort(cand, cand + nc);
    for (int c = 0; c < nc && n_seeds <= kSeeds; c++) {
        const uint64_t b = ops[(size_t)cand[c]].bits & allowed & ~start;
        bool fresh = b != 0 && popcount64(start | b) <= width;
        for (int j = 0; j < n_seeds && fresh; j++)
            fresh = seeds[j] != b;
        if (fresh)
            seeds[n_seeds++] = b;
    }
    Trial best;
    for (int j = 0; j < n_seeds; j++) {
        Trial t;
        t.bits = start | seeds[j];
        std::memcpy(t.pos, F.at, sizeof(t.pos));
        grow_trial<PHASE>(F, lim, renames_only, n, allowed, width, t);
        if (j == 0 || t.score > best.score)
            best = t;
    }
    return best;
}

static int op_weight(const HostOp &op) { return op.kind == OP_GEN ? 2 : 1; }

// A register phase of a pass: its register bits and its ops in order.
struct Ph {
    uint32_t rs;
    std::vector<int> ops;
};

// Cost of a pass's phases in hundredths of an HBM pass (see plan_cost): each
// phase, a load or store transpose where the low qubits must leave the
// registers, and an X or CNOT whose control is a thread bit (per-lane selects
// of every register).
constexpr int kPhaseCost = 13, kTransposeCost = 13, kFarSwapCost = 6;

static int phase_cost(const Ph &ph, const std::vector<SchedOp> &ops)
{
    int c = kPhaseCost;
    for (int i : ph.ops)
        if (ops[(size_t)i].kind == OP_SWAP && (ops[(size_t)i].ctrl & ~(uint64_t)ph.rs))
            c += kFarSwapCost;
    return c;
}

static int phases_cost(const std::vector<Ph> &phs, const std::vector<SchedOp> &ops, uint32_t lowmask)
{
    int c = 0;
    for (const Ph &ph : phs)
        c += phase_cost(ph, ops);
    if (phs.front().rs & lowmask)
        c += kTransposeCost;
    if (phs.back().rs & lowmask)
        c += kTransposeCost;
    return c;
}

// Phases in op order: registers go to the first targets that come along.  A
// phase looks only at the next op of every bit (the oldest first): what lies behind one that
// does not fit cannot run either.  (A walk over all ops left, once per phase,
// took 0.5 s for a 10-qubit circuit of 98000 gates, which is one pass.)
static void first_fit_phases(Frontier F, const PlanParams &pp, std::vector<Ph> *out)
{
    const std::vector<SchedOp> &ops = *F.ops;
    auto ready = [&](int i) {
        for (uint64_t m = ops[(size_t)i].bits; m; m &= m - 1)
            if (F.next(F.at, __builtin_ctzll(m)) != i)
                return false;
        return true;
    };
    out->clear();
    std::vector<int> heap;  // ops that come next on all their bits
    auto offer = [&](uint64_t bits) {
        for (uint64_t m = bits; m; m &= m - 1) {
            const int q = __builtin_ctzll(m), i = F.next(F.at, q);
            if (i >= 0 && (ops[(size_t)i].bits & bits & ((uint64_t(1) << q) - 1)) == 0 && ready(i)) {
                heap.push_back(i);
                std::push_heap(heap.begin(), heap.end(), std::greater<int>());
            }
        }
    };
    for (size_t left = ops.size(); left > 0;) {
        Ph ph{0u, {}};
        offer((uint64_t(1) << pp.k) - 1);
        while (!heap.empty()) {
            std::pop_heap(heap.begin(), heap.end(), std::greater<int>());
            const int i = heap.back();
            heap.pop_back();
            const SchedOp &op = ops[(size_t)i];
            if (op_needs_register(op.kind)) {
                const uint32_t tb = 1u << op.target;
                if (!(ph.rs & tb) && popcount64(ph.rs) >= pp.rlog)
                    continue;
                ph.rs |= tb;
            }
            ph.ops.push_back(i);
            left--;
            for (uint64_t m = op.bits; m; m &= m - 1)
                F.at[__builtin_ctzll(m)]++;
            offer(op.bits);
        }
        out->push_back(std::move(ph));
    }
}

// Phases searched for (false: there are none, or they cost `limit` or more).
static bool split_phases(Frontier F, const PlanParams &pp, bool renames_only, bool high_first, int limit,
                         std::vector<Ph> *out)
{
    const std::vector<SchedOp> &so = *F.ops;
    const SchedLimits none;
    const uint64_t all = (uint64_t(1) << pp.k) - 1, low = (uint64_t(1) << pp.low_bits) - 1;
    size_t left = so.size();
    int cost = 0;
    out->clear();
    while (left > 0) {
        const uint64_t allowed = out->empty() && high_first ? all & ~low : all;
        Trial t = pick_bits<true>(F, none, renames_only, pp.k, 0, allowed, pp.rlog);
        bool only = renames_only;
        if (t.score == 0 && only) {
            only = false;  // only swaps with controls far away are left to run
            t = pick_bits<true>(F, none, false, pp.k, 0, allowed, pp.rlog);
        }
        if (t.score == 0)
            return false;  // nothing runs without the bits that are not allowed
        Ph ph{(uint32_t)t.bits, {}};
        Trial done;
        done.bits = t.bits;
        std::memcpy(done.pos, F.at, sizeof(done.pos));
        run_trial<true>(F, none, only, all, done, &ph.ops);
        std::memcpy(F.at, done.pos, sizeof(F.at));
        left -= ph.ops.size();
        // register bits that no pair op of the phase needs are free again
        uint32_t used = 0;
        for (int i : ph.ops)
            if (op_needs_register(so[(size_t)i].kind))
                used |= (uint32_t)(so[(size_t)i].bits & t.bits);
        ph.rs = used;
        cost += phase_cost(ph, so) + (out->empty() && (used & low) ? kTransposeCost : 0);
        if (cost >= limit)
            return false;
        out->push_back(std::move(ph));
    }
    return true;
}

// One HBM pass: its qubits, its ops on tile bits in order, and its phases.
struct PassCut {
    uint32_t qpos[16];
    std::vector<HostOp> loc;
    std::vector<int> src;  // which op of the circuit each is
    std::vector<Ph> phs;
    int cost = 0;  // of the phases
};

static int cut_pass(uint64_t Q, const std::vector<HostOp> &ops, const std::vector<int> &order, const PlanParams &pp,
                    bool first_fit, std::vector<PassCut> *out)
{
    out->emplace_back();
    PassCut &C = out->back();
    int nq = 0, local[64];
    for (int q = 0; q < pp.n; q++)
        if ((Q >> q) & 1) {
            if (nq < 16)
                C.qpos[nq] = (uint32_t)q;
            local[q] = nq++;
        }
    if (nq != pp.k) {
        set_error("internal: pass has %d qubits, expected %d", nq, pp.k);
        return DMV_ERR_STATE;
    }
    C.loc.reserve(order.size());
    for (int i : order) {
        HostOp op = ops[(size_t)i];
        op.target = local[op.target];
        uint64_t ctrl = 0;
        for (uint64_t m = op.ctrl; m; m &= m - 1)
            ctrl |= uint64_t(1) << local[__builtin_ctzll(m)];
        op.ctrl = ctrl;
        C.loc.push_back(op);
    }
    C.src = order;
    // Register phases: the cheapest of the ways to cut the pass into them: in
    // op order, or searched for (swaps with thread-bit controls kept until
    // they only relabel, or done in place; the first phase's registers off the
    // low bits, which saves the load's transpose, or anywhere).
    const uint32_t lowmask = (1u << pp.low_bits) - 1;
    std::vector<SchedOp> so(C.loc.size());
    bool far_swaps = false;
    for (size_t i = 0; i < C.loc.size(); i++) {
        so[i] = SchedOp{op_qubits(C.loc[i]), C.loc[i].ctrl, C.loc[i].target, C.loc[i].kind, op_weight(C.loc[i]), 0};
        far_swaps = far_swaps || (so[i].kind == OP_SWAP && so[i].ctrl);
    }
    Frontier F;
    F.build(so, pp.k);
    first_fit_phases(F, pp, &C.phs);
    C.cost = phases_cost(C.phs, so, lowmask);
    std::vector<Ph> trial;
    for (int way = 0; way < 4 && !first_fit; way++) {
        if ((way & 1) && !far_swaps)
            continue;  // without such swaps this is the way before
        if (!split_phases(F, pp, (way & 1) == 0, (way & 2) != 0, C.cost, &trial))
            continue;
        const int c = phases_cost(trial, so, lowmask);
        if (c < C.cost) {
            C.cost = c;
            C.phs.swap(trial);
        }
    }
    return DMV_OK;
}

static void set_values(const HostOp &h, DevOp *op);

static int make_pass(const PassCut &C, const PlanParams &pp, Plan *plan)
{
    DevPass P;
    std::memset(&P, 0, sizeof(P));
    P.k = (uint32_t)pp.k;
    for (int j = 0; j < pp.k; j++)
        P.qpos[j] = C.qpos[j];
    const std::vector<HostOp> &loc = C.loc;
    std::vector<Ph> phs = C.phs;
    const uint32_t lowmask = (1u << pp.low_bits) - 1;
    // Split transposes: the highest local bit above the lane-coalesced and
    // swizzle-group bits that no op of the pass needs in a register stays a
    // thread bit, at the top, in every layout of the pass (wave-uniform halves).
    int top = -1;
    if (pp.half_lds && pp.tlog >= 7) {
        uint32_t targets = 0;
        for (const Ph &ph : phs)
            targets |= ph.rs;
        for (int b = pp.k - 1; b >= std::max(pp.low_bits, pp.swz_bits) && top < 0; b--)
            if (!((targets >> b) & 1))
                top = b;
    }
    const uint32_t avoid = top >= 0 ? 1u << top : 0u;
    for (Ph &ph : phs)
        ph.rs = pad_regs(ph.rs, pp, avoid);

    // Layouts: load/store layouts keep the low qubits in lanes.  By default
    // the first/last phase's layout is reused when it keeps the low qubits in
    // lanes.  With memory-ordered layouts (tunable) they are always the
    // canonical layout: lanes and waves take the tile's lowest qubits in
    // ascending order and registers its highest, and a phase whose register
    // set differs pays an LDS transpose instead (measured slower overall on
    // the gapped state layout).
    const uint32_t default_rs = pad_regs(0u, pp, avoid);
    const bool mem_order = tune_value("memory_layouts", 0) != 0;
    const bool renaming = tune_value("register_renaming", 1) != 0;
    const bool first_coalesced = (phs.front().rs & lowmask) == 0;
    const bool last_coalesced = (phs.back().rs & lowmask) == 0;
    P.lay_ld = make_layout(first_coalesced && !mem_order ? phs.front().rs : default_rs, pp, true, top);
    const uint32_t elem_log2 = pp.swz_bits == 3 ? 4u : 3u;
    P.split = top >= 0 ? (uint32_t)top + elem_log2 : 0u;
    auto lds_off = [&](uint32_t y) { return P.split ? drop_bit(y, P.split) : y; };
    P.phase_begin = (uint32_t)plan->phases.size();
    const int pass_index = (int)plan->passes.size();
    const int NR = 1 << pp.rlog;
    const uint32_t all_regs = NR >= 32 ? 0xFFFFFFFFu : ((1u << NR) - 1);

    // Register renaming: physical register p holds logical register tab[p]
    // (an affine map over GF(2)).  X gates and CNOTs between register bits
    // only update the map; every later op addresses physical registers
    // through it, and the next transpose or store writes register p to the
    // place of logical register tab[p].
    uint32_t tab[kMaxRegs], inv[kMaxRegs];
    auto reset_tab = [&]() {
        for (int q = 0; q < NR; q++)
            tab[q] = (uint32_t)q;
    };
    auto invert = [&]() {
        for (int q = 0; q < NR; q++)
            inv[tab[q]] = (uint32_t)q;
    };
    reset_tab();
    DevLayout prev = P.lay_ld;
    for (size_t p = 0; p < phs.size(); p++) {
        DevPhase D;
        std::memset(&D, 0, sizeof(D));
        const bool coal = (p == 0 && first_coalesced) ||
                          (p + 1 == phs.size() && last_coalesced && !(p == 0 && !first_coalesced));
        D.lay = make_layout(phs[p].rs, pp, coal && (phs[p].rs & lowmask) == 0, top);
        D.transpose_in = layouts_equal(D.lay, prev, pp) ? 0u : 1u;
        if (D.transpose_in) {
            for (int q = 0; q < NR; q++) {
                D.src_lswz[q] = lds_off(prev.lswz[tab[q]]);
                D.dst_lswz[q] = lds_off(D.lay.lswz[q]);
            }
            reset_tab();
        }
        D.op_begin = (uint32_t)plan->ops.size();
        for (int i : phs[p].ops) {
            const HostOp &h = loc[i];
            {
                HostOp g = h;
                g.target = (int)P.qpos[h.target];
                g.ctrl = deposit(h.ctrl, P.qpos, pp.k);
                plan->logical.push_back(g);
                plan->logical_pass.push_back(pass_index);
            }
            const uint32_t J = register_bit(D.lay, pp, (uint32_t)h.target);
            uint32_t creg = 0, cthr = 0;
            for (int b = 0; b < pp.k; b++) {
                if (!((h.ctrl >> b) & 1))
                    continue;
                const uint32_t rb = register_bit(D.lay, pp, (uint32_t)b);
                if (rb != kNoReg)
                    creg |= 1u << rb;
                else
                    cthr |= 1u << thread_bit(D.lay, pp, (uint32_t)b);
            }
            if (op_needs_register(h.kind) && J == kNoReg) {
                set_error("internal: op target not a register bit");
                return DMV_ERR_STATE;
            }
            // relabel-only X / CNOT: the map stays affine with at most one register control
            if (h.kind == OP_SWAP && cthr == 0 && popcount64(creg) <= 1 && renaming) {
                for (int q = 0; q < NR; q++)
                    if ((tab[q] & creg) == creg)
                        tab[q] ^= 1u << J;
                continue;
            }
            invert();
            DevOp op;
            std::memset(&op, 0, sizeof(op));
            op.kind = h.kind;
            op.target = (uint32_t)h.target;
            op.ctrl = h.ctrl;
            op.slot = h.slot;
            op.ctrl_thr = cthr;
            set_values(h, &op);
            op.tbit = J == kNoReg ? thread_bit(D.lay, pp, (uint32_t)h.target) : kNoReg;
            op.en = 0;
            for (int q = 0; q < NR; q++)
                if ((tab[q] & creg) == creg)
                    op.en |= 1u << q;
            if (J != kNoReg) {
                op.fl = 0;
                for (int q = 0; q < NR; q++)
                    if ((tab[q] >> J) & 1)
                        op.fl |= 1u << q;
                // partner of physical q: the physical register of logical tab[q] ^ e_J
                op.rmask = inv[tab[0] ^ (1u << J)] ^ inv[tab[0]];
                if (!op_needs_register(h.kind))
                    op.rmask = op.fl;  // register-target diagonal: registers whose target bit is 1
            } else {
                op.rmask = 0;
                op.fl = 0;
            }
            if (h.kind == OP_GEN && J != kNoReg)
                op.plain = (op.en == all_regs && (op.fl & first_members(op.rmask, NR)) == 0) ? 1u : 0u;
            if (op_is_ip(h.kind) && h.slot + 1 > plan->n_slots)
                plan->n_slots = h.slot + 1;
            if (op_is_ip(h.kind) && plan->ops.size() > D.op_begin) {
                // an IP op right after one of the same kind and masks reuses its sums
                const DevOp &prev = plan->ops.back();
                op.plain = prev.kind == op.kind && prev.target == op.target && prev.tbit == op.tbit &&
                                   prev.rmask == op.rmask && prev.fl == op.fl
                               ? 1u
                               : 0u;
            }
            plan->ops.push_back(op);
            plan->op_pass.push_back(pass_index);
            plan->op_src.push_back(C.src[(size_t)i]);
        }
        D.op_end = (uint32_t)plan->ops.size();
        plan->phases.push_back(D);
        prev = D.lay;
    }
    P.phase_end = (uint32_t)plan->phases.size();
    const DevLayout last = prev;
    const bool store_direct = mem_order ? layouts_equal(last, make_layout(default_rs, pp, true, top), pp)
                                        : last_coalesced &&
                                              layouts_equal(last, make_layout(phs.back().rs, pp, true, top), pp);
    P.lay_st = store_direct ? last : make_layout(default_rs, pp, true, top);
    P.transpose_st = layouts_equal(P.lay_st, last, pp) ? 0u : 1u;
    if (P.transpose_st) {
        for (int q = 0; q < NR; q++) {
            P.st_src_lswz[q] = lds_off(last.lswz[tab[q]]);
            P.st_dst_lswz[q] = lds_off(P.lay_st.lswz[q]);
        }
        reset_tab();
    }
    // a pass without transposes needs no LDS at all
    bool any_transpose = P.transpose_st != 0;
    for (uint32_t p = P.phase_begin; p < (uint32_t)plan->phases.size(); p++)
        any_transpose = any_transpose || plan->phases[p].transpose_in;
    P.lds_half = (P.split || !any_transpose) && pp.half_lds ? 1u : 0u;
    // global offsets of the load/store layouts (the store through the final map)
    for (int r = 0; r < NR; r++) {
        // element offsets: the kernels add them to the element of tile base | thread offset
        P.greg_ld[r] = elem(deposit(P.lay_ld.lreg[r], P.qpos, pp.k), pp.layout);
        P.greg_st[r] = elem(deposit(P.lay_st.lreg[tab[r]], P.qpos, pp.k), pp.layout);
    }
    for (int j = 0; j < pp.tlog; j++) {
        P.gthr_ld[j] = P.qpos[P.lay_ld.thr[j]];
        P.gthr_st[j] = P.qpos[P.lay_st.thr[j]];
    }
    plan->passes.push_back(P);
    return DMV_OK;
}

// Cost of a plan in hundredths of an HBM pass.  Fitted to the 30-qubit layered
// circuit in complex128 (745 gates, 6 to 19 passes, 35 to 48 phases): 2.6 ms a
// pass plus 0.33 ms a phase on top of the ops' own time.
static int plan_cost(const std::vector<PassCut> &cuts)
{
    int c = 0;
    for (const PassCut &C : cuts)
        c += 100 + C.cost;
    return c;
}

// Passes in op order: a pass takes every op that still fits, and what it
// cannot take blocks its qubits.
static int first_fit_passes(const std::vector<HostOp> &ops, const std::vector<SchedOp> &so, const SchedLimits &lim,
                            const PlanParams &pp, std::vector<PassCut> *out)
{
    const uint64_t all = (uint64_t(1) << pp.n) - 1, lowmask = (uint64_t(1) << pp.low_bits) - 1;
    std::vector<char> done(ops.size(), 0);
    std::vector<int> order;
    size_t first = 0;
    while (first < ops.size()) {
        uint64_t Q = lowmask, blocked = 0, treg = 0;
        int gen = 0, ip = 0;
        order.clear();
        for (size_t i = first; i < ops.size(); i++) {
            if (done[i])
                continue;
            const SchedOp &op = so[i];
            const uint64_t nt = op_needs_register(op.kind) ? treg | (uint64_t(1) << op.target) : treg;
            if (!(op.bits & blocked) && popcount64(Q | op.bits) <= pp.k && (op.kind != OP_GEN || gen < lim.max_gen) &&
                popcount64(nt & ~lim.low) <= lim.max_high_targets &&
                !(op.group > 0 && ip > 0 && ip + op.group > lim.max_ip)) {
                Q |= op.bits;
                treg = nt;
                order.push_back((int)i);
                done[i] = 1;
                gen += op.kind == OP_GEN;
                ip += op_is_ip(op.kind);
            } else {
                blocked |= op.bits;
                if ((blocked & all) == all)
                    break;
            }
        }
        while (first < ops.size() && done[first])
            first++;
        // fill the tile up to k qubits with the lowest unused qubits
        for (int q = 0; q < pp.n && popcount64(Q) < pp.k; q++)
            Q |= uint64_t(1) << q;
        DMV_TRY(cut_pass(Q, ops, order, pp, true, out));
    }
    return DMV_OK;
}

// Passes searched for: each takes the qubits that let it run the most ops
// (pick_bits), whatever layer of the circuit they are in.
static int searched_passes(const std::vector<HostOp> &ops, const std::vector<SchedOp> &so, const SchedLimits &lim,
                           const PlanParams &pp, std::vector<PassCut> *out)
{
    const uint64_t all = (uint64_t(1) << pp.n) - 1, lowmask = (uint64_t(1) << pp.low_bits) - 1;
    Frontier F;
    F.build(so, pp.n);
    size_t left = ops.size();
    std::vector<int> order;
    while (left > 0) {
        uint64_t Q = pick_bits<false>(F, lim, false, pp.n, lowmask, all, pp.k).bits;
        for (int q = 0; q < pp.n && popcount64(Q) < pp.k; q++)
            Q |= uint64_t(1) << q;
        Trial done;
        done.bits = Q;
        std::memcpy(done.pos, F.at, sizeof(done.pos));
        order.clear();
        run_trial<false>(F, lim, false, Q, done, &order);
        if (order.empty()) {
            set_error("internal: scheduler made no progress");
            return DMV_ERR_STATE;
        }
        std::memcpy(F.at, done.pos, sizeof(F.at));
        left -= order.size();
        DMV_TRY(cut_pass(Q, ops, order, pp, false, out));
    }
    return DMV_OK;
}

// The scheduler's view of the ops and what a pass may hold.
static std::vector<SchedOp> sched_ops(const std::vector<HostOp> &ops, const PlanParams &pp, SchedLimits *lim)
{
    std::vector<SchedOp> so(ops.size());
    int run[64] = {}, head[64] = {};  // each qubit's open run of IP ops, counted at its first op
    for (size_t i = ops.size(); i-- > 0;) {
        so[i] = SchedOp{op_qubits(ops[i]), ops[i].ctrl, ops[i].target, ops[i].kind, op_weight(ops[i]), 0};
        if (op_is_ip(ops[i].kind)) {
            const int q = ops[i].target;
            if (run[q] > 0)
                so[(size_t)head[q]].group = 0;
            head[q] = (int)i;
            so[i].group = ++run[q];
        } else {
            for (uint64_t m = so[i].bits; m; m &= m - 1)
                run[__builtin_ctzll(m)] = 0;
        }
    }
    // With split transposes, a pass keeps one of its qubits above the lane
    // and swizzle-group bits free of register targets (the split bit): an op
    // that would make every such qubit a register target waits for the next
    // pass.  The lowest qubits are always in the tile, so those candidates
    // are the tile's qubits outside the lowest max(low_bits, swz_bits).
    const int kept = std::max(pp.low_bits, pp.swz_bits);
    lim->max_gen = pp.max_gen_per_pass;
    lim->max_ip = pp.max_ip_per_pass;
    lim->max_high_targets = pp.half_lds && pp.tlog >= 7 ? pp.k - kept - 1 : 64;
    lim->low = (uint64_t(1) << kept) - 1;
    return so;
}

bool same_structure(const std::vector<HostOp> &a, const std::vector<HostOp> &b)
{
    if (a.size() != b.size())
        return false;
    for (size_t i = 0; i < a.size(); i++)
        if (a[i].kind != b[i].kind || a[i].target != b[i].target || a[i].ctrl != b[i].ctrl || a[i].slot != b[i].slot)
            return false;
    return true;
}

// What a device op takes from its op's values.
static void set_values(const HostOp &h, DevOp *op)
{
    std::memcpy(op->m, h.m, sizeof(op->m));
    if (h.kind == OP_GEN)
        op->aux = h.su2 ? 1u : 0u;
    if (h.kind == OP_DIAG)
        op->plain = diag_is_sign_flip(op->m) ? 1u : 0u;
}

void refresh_ops(const std::vector<HostOp> &given, bool fp32, const std::vector<int> &op_src, std::vector<DevOp> *dev)
{
    std::vector<HostOp> ops = given;
    if (!fp32)
        special_unitary(&ops);
    for (size_t i = 0; i < dev->size(); i++)
        set_values(ops[(size_t)op_src[i]], &(*dev)[i]);
}

namespace {
struct KeptPlan {
    PlanParams pp;
    int renaming, mem_order;  // the tunables that make_pass reads
    std::vector<HostOp> source;
    std::shared_ptr<const Plan> plan;
};

struct PlanCache {
    std::mutex mu;
    std::unordered_multimap<uint64_t, KeptPlan> kept;
    size_t ops = 0;
};

PlanCache &plan_cache()
{
    static PlanCache *c = new PlanCache();  // never destroyed: outlives static destructors
    return *c;
}

bool same_params(const PlanParams &a, const PlanParams &b)
{
    return a.n == b.n && a.k == b.k && a.rlog == b.rlog && a.tlog == b.tlog && a.low_bits == b.low_bits &&
           a.swz_bits == b.swz_bits && a.max_gen_per_pass == b.max_gen_per_pass && a.half_lds == b.half_lds &&
           a.max_ip_per_pass == b.max_ip_per_pass && a.gen_auto == b.gen_auto && a.fp32 == b.fp32 && same_layout(a.layout, b.layout);
}
}  // namespace

int shared_plan(const std::vector<HostOp> &ops, const PlanParams &pp, std::shared_ptr<const Plan> *out)
{
    const int renaming = tune_value("register_renaming", 1) != 0, mem_order = tune_value("memory_layouts", 0) != 0;
    uint64_t key = (uint64_t)pp.n + 64 * ((uint64_t)pp.k + 16 * ((uint64_t)pp.tlog + 16 * (uint64_t)pp.swz_bits));
    for (const HostOp &op : ops)
        key = (key ^ (op.kind + 16 * (uint64_t)op.target + 1024 * (op.ctrl + 1))) * 0x9E3779B97F4A7C15ull;
    PlanCache &C = plan_cache();
    {
        std::lock_guard<std::mutex> lk(C.mu);
        const auto range = C.kept.equal_range(key);
        for (auto it = range.first; it != range.second; ++it) {
            const KeptPlan &P = it->second;
            if (P.renaming == renaming && P.mem_order == mem_order && same_params(P.pp, pp) &&
                same_structure(P.source, ops)) {
                *out = P.plan;
                return DMV_OK;
            }
        }
    }
    auto made = std::make_shared<Plan>();
    DMV_TRY(build_plan(ops, pp, made.get()));
    made->logical = {};
    made->logical_pass = {};
    made->op_pass = {};
    *out = made;
    std::lock_guard<std::mutex> lk(C.mu);
    const size_t size = ops.size() + made->ops.size();
    if (size > kKeptOps)
        return DMV_OK;
    if (C.ops + size > kKeptOps) {
        C.kept.clear();
        C.ops = 0;
    }
    C.kept.emplace(key, KeptPlan{pp, renaming, mem_order, ops, made});
    C.ops += size;
    return DMV_OK;
}

int in_order_budget(const std::vector<HostOp> &ops, const PlanParams &pp, int *budget)
{
    SchedLimits lim;
    const std::vector<SchedOp> so = sched_ops(ops, pp, &lim);
    size_t cost[2];
    const int budgets[2] = {8, 12};
    for (int i = 0; i < 2; i++) {
        lim.max_gen = budgets[i];
        std::vector<PassCut> cuts;
        DMV_TRY(first_fit_passes(ops, so, lim, pp, &cuts));
        cost[i] = 4 * cuts.size();
        for (const PassCut &C : cuts)
            cost[i] += 6 * C.phs.size();
    }
    *budget = budgets[cost[1] < cost[0]];
    return DMV_OK;
}

int build_plan(const std::vector<HostOp> &given, const PlanParams &pp, Plan *out)
{
    std::vector<HostOp> ops = given;
    if (!pp.fp32)
        special_unitary(&ops);
    DMV_CHECK_ARG(pp.k == pp.rlog + pp.tlog, "tile qubits %d != %d + %d", pp.k, pp.rlog, pp.tlog);
    DMV_CHECK_ARG(pp.n >= pp.k && pp.k <= kMaxTileQubits && pp.rlog >= 1 &&
                      (1 << pp.rlog) <= kMaxRegs && pp.tlog <= kMaxThreadBits &&
                      pp.low_bits <= pp.tlog && pp.low_bits + pp.rlog <= pp.k,
                  "invalid tile shape n=%d k=%d rlog=%d tlog=%d", pp.n, pp.k, pp.rlog, pp.tlog);
    Plan plan;
    const uint64_t all = (pp.n >= 64) ? ~uint64_t(0) : ((uint64_t(1) << pp.n) - 1);
    for (const HostOp &op : ops) {
        DMV_CHECK_ARG(op.target >= 0 && op.target < pp.n, "target %d out of range", op.target);
        DMV_CHECK_ARG((op.ctrl & ~all) == 0 && !((op.ctrl >> op.target) & 1), "bad control mask");
    }
    SchedLimits lim;
    const std::vector<SchedOp> so = sched_ops(ops, pp, &lim);
    // A budget of eight GENs a pass (the caller's, or tried here) is filled in
    // op order: measured on the 30-qubit layered circuit, both ways take 19
    // passes, but searched ones 48 phases for 38 (114 against 109 ms).
    // Without a budget the search is tried too and the cheaper plan kept: 6
    // passes of that circuit (70 ms), 9 for 25 at 20 qubits and 10 layers (328
    // against 532 us).  A CNOT ring, whose next layer waits for the whole ring,
    // takes as many passes either way.
    constexpr int kInOrder = 8;
    const auto gens = std::count_if(so.begin(), so.end(), [](const SchedOp &op) { return op.kind == OP_GEN; });
    std::vector<PassCut> cuts;
    if (pp.fp32) {
        if (pp.gen_auto)
            DMV_TRY(in_order_budget(ops, pp, &lim.max_gen));
        DMV_TRY(first_fit_passes(ops, so, lim, pp, &cuts));
    } else if (pp.gen_auto ? pp.n > pp.k || gens <= kInOrder : pp.max_gen_per_pass <= kInOrder) {
        // (not for a state of one tile if it takes passes in order: searched, it is one)
        if (pp.gen_auto)
            lim.max_gen = kInOrder;
        DMV_TRY(first_fit_passes(ops, so, lim, pp, &cuts));
    }
    if (!pp.fp32 && (pp.gen_auto || pp.max_gen_per_pass > kInOrder)) {
        if (pp.gen_auto)
            lim.max_gen = 1 << 30;
        std::vector<PassCut> more;
        DMV_TRY(searched_passes(ops, so, lim, pp, &more));
        if (cuts.empty() || plan_cost(more) < plan_cost(cuts))
            cuts.swap(more);
        // Passes that need not split their transposes: those that do not go through
        // LDS by parts, three workgroups a CU all the same.  24 qubits: 52 passes
        // for 60 of a CNOT ring ansatz (6.15 -> 5.48 ms), 12 for 13 of a random circuit
        // (1.85 -> 1.73 ms); 30 qubits, layered: 8 for 6 (85 against 72 ms).
        if (pp.gen_auto && pp.half_lds) {
            lim.max_high_targets = 64;
            more.clear();
            DMV_TRY(searched_passes(ops, so, lim, pp, &more));
            if (plan_cost(more) < plan_cost(cuts))
                cuts.swap(more);
        }
    }
    for (const PassCut &C : cuts)
        DMV_TRY(make_pass(C, pp, &plan));
    // number the IP ops of every pass: pass p's gradient partials are rows
    // ip_begin[p] .. ip_begin[p+1] of the per-pass partial buffer
    plan.ip_begin.assign(plan.passes.size() + 1, 0);
    plan.ip_slots.clear();
    for (size_t p = 0; p < plan.passes.size(); p++) {
        plan.ip_begin[p] = plan.passes[p].ip_begin = (uint32_t)plan.ip_slots.size();
        for (uint32_t ph = plan.passes[p].phase_begin; ph < plan.passes[p].phase_end; ph++)
            for (uint32_t o = plan.phases[ph].op_begin; o < plan.phases[ph].op_end; o++)
                if (op_is_ip(plan.ops[o].kind)) {
                    plan.ops[o].aux = (uint32_t)plan.ip_slots.size() - plan.ip_begin[p];
                    plan.ip_slots.push_back(plan.ops[o].slot);
                }
    }
    plan.ip_begin[plan.passes.size()] = (uint32_t)plan.ip_slots.size();
    DMV_TRY(validate_plan(plan, pp));
    *out = std::move(plan);
    return DMV_OK;
}

static int check_layout(const DevLayout &L, const PlanParams &pp, const char *what)
{
    uint32_t seen = 0;
    for (int j = 0; j < pp.tlog; j++) {
        if (L.thr[j] >= (uint32_t)pp.k || ((seen >> L.thr[j]) & 1)) {
            set_error("internal: %s thread bit %d invalid", what, j);
            return DMV_ERR_STATE;
        }
        seen |= 1u << L.thr[j];
    }
    uint32_t regmask = 0;
    for (int j = 0; j < pp.rlog; j++)
        regmask |= L.lreg[1 << j];
    if ((regmask & seen) != 0 || popcount64(regmask) != pp.rlog || ((regmask | seen) + 1) != (1u << pp.k)) {
        set_error("internal: %s register bits invalid", what);
        return DMV_ERR_STATE;
    }
    const uint32_t elem = pp.swz_bits == 3 ? 16u : 8u;
    for (int r = 0; r < (1 << pp.rlog); r++) {
        uint32_t expect = 0;
        for (int j = 0; j < pp.rlog; j++)
            if ((r >> j) & 1)
                expect |= L.lreg[1 << j];
        const uint32_t sw = (pp.swz_bits == 3 ? swz_index<3>(L.lreg[r]) : swz_index<4>(L.lreg[r])) * elem;
        if (L.lreg[r] != expect || L.lswz[r] != sw || L.lswz[r] >= (elem << pp.k)) {
            set_error("internal: %s register offsets inconsistent", what);
            return DMV_ERR_STATE;
        }
    }
    return DMV_OK;
}

// A transpose's write offsets must be a permutation of its source layout's
// and its read offsets its destination layout's, with the split bit removed
// in a split pass.  There, the split local bit must be the top thread bit of
// both layouts (so each half of the threads exchanges amplitudes only within
// itself) and the offsets must fit half a tile.
static int check_offsets(const uint32_t *src, const DevLayout &A, const uint32_t *dst, const DevLayout &B,
                         uint32_t split, const PlanParams &pp, const char *what)
{
    const int NR = 1 << pp.rlog;
    const uint32_t elem_log2 = pp.swz_bits == 3 ? 4u : 3u;
    const uint32_t limit = (1u << (pp.k + (int)elem_log2)) >> (split ? 1 : 0);
    std::vector<uint32_t> a(src, src + NR), b(NR), c(dst, dst + NR), d(NR);
    for (int r = 0; r < NR; r++) {
        b[r] = split ? drop_bit(A.lswz[r], split) : A.lswz[r];
        d[r] = split ? drop_bit(B.lswz[r], split) : B.lswz[r];
        if (d[r] != c[r] || a[r] >= limit) {
            set_error("internal: %s read offsets inconsistent", what);
            return DMV_ERR_STATE;
        }
    }
    std::sort(a.begin(), a.end());
    std::sort(b.begin(), b.end());
    if (a != b) {
        set_error("internal: %s offsets are not a permutation of the layout", what);
        return DMV_ERR_STATE;
    }
    if (split) {
        const uint32_t w = split - elem_log2;
        if (split < elem_log2 || (int)w < pp.swz_bits || (int)w >= pp.k || pp.tlog < 7 ||
            A.thr[pp.tlog - 1] != w || B.thr[pp.tlog - 1] != w) {
            set_error("internal: %s split bit is not the top thread bit of both layouts", what);
            return DMV_ERR_STATE;
        }
    }
    return DMV_OK;
}

int validate_plan(const Plan &plan, const PlanParams &pp)
{
    const uint64_t n_amp = uint64_t(1) << pp.n;
    for (const DevPass &P : plan.passes) {
        if ((int)P.k != pp.k) {
            set_error("internal: pass k mismatch");
            return DMV_ERR_STATE;
        }
        for (int j = 0; j < pp.k; j++)
            if (P.qpos[j] >= (uint32_t)pp.n || (j > 0 && P.qpos[j] <= P.qpos[j - 1])) {
                set_error("internal: pass qubit list invalid");
                return DMV_ERR_STATE;
            }
        DMV_TRY(check_layout(P.lay_ld, pp, "load layout"));
        DMV_TRY(check_layout(P.lay_st, pp, "store layout"));
        for (int j = 0; j < pp.low_bits; j++)
            if (P.lay_ld.thr[j] != (uint32_t)j || P.lay_st.thr[j] != (uint32_t)j) {
                set_error("internal: load/store layout not coalesced");
                return DMV_ERR_STATE;
            }
        for (int r = 0; r < (1 << pp.rlog); r++)
            if (P.greg_ld[r] >= n_amp || P.greg_st[r] >= n_amp) {
                set_error("internal: register offset out of range");
                return DMV_ERR_STATE;
            }
        for (int j = 0; j < pp.tlog; j++)
            if (P.gthr_ld[j] >= (uint32_t)pp.n || P.gthr_st[j] >= (uint32_t)pp.n) {
                set_error("internal: thread bit position out of range");
                return DMV_ERR_STATE;
            }
        if (P.phase_begin >= P.phase_end || P.phase_end > plan.phases.size()) {
            set_error("internal: phase range invalid");
            return DMV_ERR_STATE;
        }
        for (uint32_t p = P.phase_begin; p < P.phase_end; p++) {
            const DevPhase &D = plan.phases[p];
            DMV_TRY(check_layout(D.lay, pp, "phase layout"));
            if (D.op_begin > D.op_end || D.op_end > plan.ops.size()) {
                set_error("internal: op range invalid");
                return DMV_ERR_STATE;
            }
            if (D.transpose_in)
                DMV_TRY(check_offsets(D.src_lswz, p == P.phase_begin ? P.lay_ld : plan.phases[p - 1].lay,
                                      D.dst_lswz, D.lay, P.split, pp, "phase transpose"));
            for (uint32_t o = D.op_begin; o < D.op_end; o++) {
                const DevOp &op = plan.ops[o];
                const int NR = 1 << pp.rlog;
                const uint32_t regs = NR >= 32 ? 0xFFFFFFFFu : ((1u << NR) - 1);
                if (op.target >= (uint32_t)pp.k || (op.ctrl >> pp.k) != 0 || ((op.ctrl >> op.target) & 1)) {
                    set_error("internal: op bits out of range");
                    return DMV_ERR_STATE;
                }
                if (op.kind != OP_GEN && op.kind != OP_DIAG && op.kind != OP_SWAP && !op_is_ip(op.kind)) {
                    set_error("internal: op kind invalid");
                    return DMV_ERR_STATE;
                }
                if ((op.en & ~regs) || (op.fl & ~regs) || (op.ctrl_thr >> pp.tlog) != 0) {
                    set_error("internal: op masks out of range");
                    return DMV_ERR_STATE;
                }
                // GENs come from uncontrolled gates only; the reverse sweep's
                // kernels apply them to every pair of every lane
                if (op.kind == OP_GEN && (op.ctrl != 0 || op.ctrl_thr != 0 || op.en != regs)) {
                    set_error("internal: controlled GEN op");
                    return DMV_ERR_STATE;
                }
                if (op.kind == OP_GEN && op.aux &&
                    (op.m[6] != op.m[0] || op.m[7] != -op.m[1] || op.m[2] != -op.m[4] || op.m[3] != op.m[5])) {
                    set_error("internal: special-unitary flag on a general matrix");
                    return DMV_ERR_STATE;
                }
                if (op_is_ip(op.kind)) {
                    const DevOp *prev = o > D.op_begin ? &plan.ops[o - 1] : nullptr;
                    if (op.plain && !(prev && prev->kind == op.kind && prev->target == op.target &&
                                      prev->tbit == op.tbit && prev->rmask == op.rmask && prev->fl == op.fl)) {
                        set_error("internal: IP op reuses sums it has no predecessor for");
                        return DMV_ERR_STATE;
                    }
                } else if (op.plain && op.kind == OP_DIAG) {
                    if (!diag_is_sign_flip(op.m)) {
                        set_error("internal: plain flag on a diagonal other than diag(1, -1)");
                        return DMV_ERR_STATE;
                    }
                } else if (op.plain &&
                           (op.kind != OP_GEN || op.en != regs || (op.fl & first_members(op.rmask, NR)) != 0)) {
                    set_error("internal: plain flag on an op that needs selects");
                    return DMV_ERR_STATE;
                }
                const bool target_reg = register_bit(D.lay, pp, op.target) != kNoReg;
                if (op_needs_register(op.kind)) {
                    if (!target_reg || op.rmask == 0 || op.rmask >= (uint32_t)NR || op.tbit != kNoReg) {
                        set_error("internal: pair op without a register partner");
                        return DMV_ERR_STATE;
                    }
                } else if (target_reg) {
                    if ((op.rmask & ~regs) || op.tbit != kNoReg) {
                        set_error("internal: register diagonal masks out of range");
                        return DMV_ERR_STATE;
                    }
                } else if (op.tbit >= (uint32_t)pp.tlog || D.lay.thr[op.tbit] != op.target) {
                    set_error("internal: thread-bit target inconsistent");
                    return DMV_ERR_STATE;
                }
                for (int j = 0; j < pp.tlog; j++)
                    if (((op.ctrl_thr >> j) & 1) && !((op.ctrl >> D.lay.thr[j]) & 1)) {
                        set_error("internal: thread control not in the control mask");
                        return DMV_ERR_STATE;
                    }
            }
        }
        if (P.transpose_st)
            DMV_TRY(check_offsets(P.st_src_lswz, plan.phases[P.phase_end - 1].lay, P.st_dst_lswz, P.lay_st, P.split,
                                  pp, "store transpose"));
        bool any_transpose = P.transpose_st != 0;
        for (uint32_t p = P.phase_begin; p < P.phase_end; p++)
            any_transpose = any_transpose || plan.phases[p].transpose_in;
        if ((P.lds_half || P.split) && !pp.half_lds) {
            set_error("internal: split transposes in a plan for full-LDS kernels");
            return DMV_ERR_STATE;
        }
        if (P.lds_half && any_transpose && !P.split) {
            set_error("internal: half-LDS pass with a full transpose");
            return DMV_ERR_STATE;
        }
    }
    return DMV_OK;
}

std::vector<HostOp> plan_global_ops(const Plan &plan, std::vector<int> *pass_of_op)
{
    if (pass_of_op)
        *pass_of_op = plan.logical_pass;
    return plan.logical;
}

std::vector<DevOp> global_dev_ops(const std::vector<HostOp> &ops)
{
    std::vector<DevOp> out(ops.size());
    for (size_t i = 0; i < ops.size(); i++) {
        std::memset(&out[i], 0, sizeof(DevOp));
        out[i].kind = ops[i].kind;
        out[i].target = (uint32_t)ops[i].target;
        out[i].ctrl = ops[i].ctrl;
        out[i].slot = ops[i].slot;
        std::memcpy(out[i].m, ops[i].m, sizeof(out[i].m));
    }
    return out;
}

}  // namespace dmv
