// pergate.hip -- the plain method: gates one after another, without a plan.
//
// Replaces kernelExecSimple and its 19 gate kernels (src/kernelSimple.cu:40-446).
// Differences by design: one templated kernel per update form instead of one
// per gate type; threads enumerate only the pairs whose controls are set
// (the reference launches 2^(n-1) threads and idles the others); 64-bit
// indexing so n >= 33 works; consecutive gates share a pass over the state
// where the tile of one thread and its wave holds their targets.

#include "hq_ops.h"

#include <algorithm>
#include <cmath>
#include <new>

namespace hq {

bool gate_is_diagonal_type(int type)
{
    // Gate::isDiagonal, src/gate.h:27-29
    switch (type) {
    case HQ_CZ: case HQ_CU1: case HQ_CRZ: case HQ_U1: case HQ_Z:
    case HQ_S: case HQ_SDG: case HQ_T: case HQ_TDG: case HQ_RZ:
        return true;
    default:
        return false;
    }
}

int gate_num_controls(int type)
{
    switch (type) {
    case HQ_CCX: return 2;
    case HQ_CNOT: case HQ_CY: case HQ_CZ: case HQ_CRX: case HQ_CRY: case HQ_CU1: case HQ_CRZ: return 1;
    default: return 0;
    }
}

hq_status validate_gate(const hq_gate& g, int n)
{
    HQ_CHECK(g.type >= 0 && g.type <= HQ_GCC && g.type != HQ_TOTAL, HQ_ERR_ARG, "gate: unknown type");
    HQ_CHECK(g.target >= 0 && g.target < n, HQ_ERR_ARG, "gate: target out of range");
    int nc = gate_num_controls(g.type);
    if (nc >= 1) {
        HQ_CHECK(g.control >= 0 && g.control < n && g.control != g.target, HQ_ERR_ARG,
                 "gate: control missing, out of range or equal to the target");
    } else {
        HQ_CHECK(g.control == -1, HQ_ERR_ARG, "gate: this gate type takes no control");
    }
    if (nc == 2) {
        HQ_CHECK(g.control2 >= 0 && g.control2 < n && g.control2 != g.target && g.control2 != g.control,
                 HQ_ERR_ARG, "gate: second control missing, out of range or repeated");
    } else {
        HQ_CHECK(g.control2 == -1, HQ_ERR_ARG, "gate: this gate type takes no second control");
    }
    for (int i = 0; i < 8; i++)
        HQ_CHECK(std::isfinite(g.mat[i]), HQ_ERR_ARG, "gate: matrix entry is not finite");
    return HQ_OK;
}

int classify_gate(const hq_gate& g)
{
    const double* m = g.mat;
    bool offdiag_zero = m[2] == 0 && m[3] == 0 && m[4] == 0 && m[5] == 0;
    if (gate_is_diagonal_type(g.type) || offdiag_zero) {
        if (m[0] == 1 && m[1] == 0) return SHM_PHASE;
        return SHM_DIAG;
    }
    bool diag_zero = m[0] == 0 && m[1] == 0 && m[6] == 0 && m[7] == 0;
    if (diag_zero && m[2] == 1 && m[3] == 0 && m[4] == 1 && m[5] == 0) return SHM_SWAP;
    if (diag_zero && m[2] == 0 && m[3] == -1 && m[4] == 0 && m[5] == 1) return SHM_Y;
    if (m[1] == 0 && m[3] == 0 && m[5] == 0 && m[7] == 0) return SHM_REAL;
    if (m[1] == 0 && m[7] == 0 && m[2] == 0 && m[4] == 0) return SHM_RX;
    return SHM_GEN;
}

// Insert bits into a pair index: `nins` positions (ascending) get the values
// in `vals` (0 for the target, 1 for each control).
struct Inserts {
    int pos[3];
    int val[3];
    int n;
};

template <int CLS, typename R>
__global__ __launch_bounds__(256) void k_plain(cplx<R>* __restrict__ a, uint64_t work, Inserts ins, int t,
                                               Coef<R> c)
{
    uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < work; i += stride) {
        uint64_t lo = i;
#pragma unroll
        for (int k = 0; k < 3; k++) {
            if (k < ins.n) {
                int p = ins.pos[k];
                lo = ((lo >> p) << (p + 1)) | (lo & (((uint64_t)1 << p) - 1)) | ((uint64_t)ins.val[k] << p);
            }
        }
        uint64_t hi = lo | ((uint64_t)1 << t);
        cplx<R> x = a[lo], y = a[hi];
        pair_update<CLS, R>(x, y, c.m);
        if constexpr (CLS != SHM_PHASE) a[lo] = x;
        a[hi] = y;
    }
}

template <typename R>
static hq_status launch_plain_gate(hq_state s, const hq_gate& g)
{
    int cls = classify_gate(g);
    Inserts ins{};
    ins.n = 0;
    int ps[3], vs[3], np = 0;
    ps[np] = g.target; vs[np++] = 0;
    if (g.control >= 0) { ps[np] = g.control; vs[np++] = 1; }
    if (g.control2 >= 0) { ps[np] = g.control2; vs[np++] = 1; }
    // ascending insertion order
    for (int i = 0; i < np; i++)
        for (int j = i + 1; j < np; j++)
            if (ps[j] < ps[i]) { std::swap(ps[i], ps[j]); std::swap(vs[i], vs[j]); }
    for (int i = 0; i < np; i++) { ins.pos[i] = ps[i]; ins.val[i] = vs[i]; }
    ins.n = np;
    uint64_t work = s->amps >> np;
    Coef<R> c;
    for (int i = 0; i < 8; i++) c.m[i] = (R)g.mat[i];
    unsigned threads = 256;
    uint64_t blocks = (work + threads - 1) / threads;
    if (blocks > 1u << 20) blocks = 1u << 20;
    cplx<R>* a = (cplx<R>*)s->data;
    switch (cls) {
#define HQ_PLAIN_CASE(C) \
    case C: hipLaunchKernelGGL((k_plain<C, R>), dim3((unsigned)blocks), dim3(threads), 0, s->stream, a, work, ins, g.target, c); break;
        HQ_PLAIN_CASE(SHM_SWAP)
        HQ_PLAIN_CASE(SHM_Y)
        HQ_PLAIN_CASE(SHM_REAL)
        HQ_PLAIN_CASE(SHM_RX)
        HQ_PLAIN_CASE(SHM_GEN)
        HQ_PLAIN_CASE(SHM_DIAG)
        HQ_PLAIN_CASE(SHM_PHASE)
#undef HQ_PLAIN_CASE
    default: break;
    }
    HQ_HIP(hipGetLastError());
    return HQ_OK;
}

// ---- runs of gates in one pass -------------------------------------------------------------
// One gate a pass is bound by HBM (20 qubits and less: by launches, 4 to 6 us each).
// Here a thread holds 16 amplitudes, four register bits of the index above the
// wave's six lane bits (index bits 0 to 5, so that every access is a whole run
// of 64 amplitudes), and a run of gates whose targets are among those ten bits
// is applied in order; diagonal gates and controls may sit anywhere.  Register
// targets are pair updates, lane targets one exchange with the partner lane.
// Branches are on the run's fields and uniform, but for the lanes a diagonal
// gate skips; controls select.  Random layers, a gate on average, one by one and
// in runs: 10 qubits (20 layers) 3.1 and 0.66 us, 20 qubits complex128 (20) 6.2 and
// 1.34, 25 qubits (8) 147 and 15.5 (complex64 62 and 7.1), 30 qubits (30 layers) 4 890
// and 507.  Those 1350 gates of 30 qubits are 88 runs of 15 gates on average, 7.7 ms
// each (4.5 TB/s), and two single gates; a state of few waves is bound by the
// chain of a run's gates (20 qubits: 26 us for 21).
constexpr int RUN_MAX_RB = 4, RUN_LANES = 6, RUN_GATES = 32;
constexpr int RUN_MIN_QUBITS = RUN_MAX_RB + RUN_LANES;
// Up to here 8 amplitudes a thread: fewer gates fit a pass, but a pass is a
// chain of its gates by one wave or none per SIMD (600 to 300 gates of random
// layers, us, 8 against 16 amplitudes: 10 qubits 213 / 284, 17 qubits
// complex64 365 / 434, 20 qubits complex128 840 / 783, 28 qubits 35 600 / 27 400).
constexpr int RUN_SMALL_QUBITS = 18;

// Passes over the state that gates must cost one by one to share a pass: one
// of 16 strided runs takes 1.0 to 1.35 of a plain pass, by the strides (28
// qubits complex128: one H 1.58 ms, two in a run 1.61 to 2.11; two CNOTs, half
// a pass each, 1.59 one by one and 2.12 in a run, three 2.39 and 2.14).
constexpr double RUN_MIN_SHARE = 1.35;

enum RunForm : uint32_t {
    RUN_SWAP, RUN_REAL, RUN_RX, RUN_GEN, RUN_Y, RUN_LSWAP, RUN_LREAL, RUN_LRX, RUN_LGEN, RUN_LY,
    RUN_DIAG,       // complex factors on every amplitude, or all with a register target set
    RUN_DIAG_REAL,  // real factors on some (Z, CZ)
    RUN_DIAG_SOME   // complex factors on some
};

struct RunFields {
    uint64_t omask;      // controls outside the register bits
    uint64_t tbit;       // RUN_DIAG: target outside the register bits; lane forms: the lane's target bit
    uint32_t form;       // RunForm
    uint32_t pos;        // register bit of the target; lane forms: its lane bit
    uint32_t rmask;      // controls among the register bits
    uint32_t rbit : 31;  // RUN_DIAG: target among the register bits
    uint32_t phase : 1;  // RUN_DIAG: the factor is 1 where the target is clear

    __device__ __forceinline__ RunFields uniform() const
    {
        struct Words { uint32_t w[8]; };
        Words u = __builtin_bit_cast(Words, *this);
#pragma unroll
        for (int i = 0; i < 8; i++) u.w[i] = (uint32_t)__builtin_amdgcn_readfirstlane((int)u.w[i]);
        return __builtin_bit_cast(RunFields, u);
    }
};
static_assert(sizeof(RunFields) == 32, "RunFields layout");

template <typename R>
struct alignas(16) RunGate {
    R m[8];
    RunFields f;
};

template <typename R>
struct Run {
    RunGate<R> g[RUN_GATES + 1];   // (the last is only read ahead)
    int num;
    int pos[RUN_MAX_RB];     // index bit of each register bit, ascending
};
static_assert(sizeof(Run<double>) < 4000, "kernel arguments");

template <typename R>
__device__ __forceinline__ cplx<R> pick(bool c, cplx<R> a, cplx<R> b)
{
    cplx<R> r;
    r.x = c ? a.x : b.x;
    r.y = c ? a.y : b.y;
    return r;
}

// register target P; lane: the lane's controls hold
template <int CLS, int P, bool CTRL, int RB, typename R>
__device__ __forceinline__ void run_pairs(cplx<R> (&a)[1 << RB], const R* m, bool lane, uint32_t rmask)
{
#pragma unroll
    for (int j = 0; j < (1 << RB); j++) {
        if (j & (1 << P)) continue;
        cplx<R> x = a[j], y = a[j | (1 << P)];
        pair_update<CLS, R>(x, y, m);
        const bool on = !CTRL || (lane && ((uint32_t)j & rmask) == rmask);
        a[j] = pick(on, x, a[j]);
        a[j | (1 << P)] = pick(on, y, a[j | (1 << P)]);
    }
}

template <int P, bool CTRL, int RB, typename R>
__device__ __forceinline__ void run_reg(cplx<R> (&a)[1 << RB], uint32_t form, const R* m, bool lane, uint32_t rmask)
{
    if constexpr (P < RB) {
    if (form == RUN_SWAP) run_pairs<SHM_SWAP, P, CTRL, RB, R>(a, m, lane, rmask);
    else if (form == RUN_REAL) run_pairs<SHM_REAL, P, CTRL, RB, R>(a, m, lane, rmask);
    else if (form == RUN_RX) run_pairs<SHM_RX, P, CTRL, RB, R>(a, m, lane, rmask);
    else if (form == RUN_GEN) run_pairs<SHM_GEN, P, CTRL, RB, R>(a, m, lane, rmask);
    else run_pairs<SHM_Y, P, CTRL, RB, R>(a, m, lane, rmask);
    }
}

// amplitudes with register bit P clear *= l, set *= h (P < 0: all *= l); phase: l is 1
template <int RB, int P, typename R>
__device__ __forceinline__ void run_scale(cplx<R> (&a)[1 << RB], R lr, R li, R hr, R hi, bool phase)
{
    if constexpr (P < RB) {
#pragma unroll
        for (int half = 0; half < 2; half++) {
            if (half == 0 && phase) continue;
#pragma unroll
            for (int j = 0; j < (1 << RB); j++) {
                if (P < 0 ? half != 0 : ((j >> (P < 0 ? 0 : P)) & 1) != half) continue;
                const R x = a[j].x, y = a[j].y, fr = half ? hr : lr, fi = half ? hi : li;
                a[j].x = fr * x - fi * y;
                a[j].y = fr * y + fi * x;
            }
        }
    }
}

// x of the lane whose index differs in bit BIT; hi: the lane's bit
template <int BIT>
__device__ __forceinline__ uint32_t partner32(uint32_t x, bool hi)
{
    if constexpr (BIT == 0) return (uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0xB1, 0xf, 0xf, true);   // quad 1 0 3 2
    if constexpr (BIT == 1) return (uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0x4E, 0xf, 0xf, true);   // quad 2 3 0 1
    if constexpr (BIT == 2)   // half rows mirrored (xor 7), then quads (xor 3)
        return (uint32_t)__builtin_amdgcn_mov_dpp(__builtin_amdgcn_mov_dpp((int)x, 0x141, 0xf, 0xf, true), 0x1B, 0xf,
                                                  0xf, true);
    if constexpr (BIT == 3) return (uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0x128, 0xf, 0xf, true);  // row rotated by 8
    // (first: every lane's value at bit clear, second: at bit set)
    if constexpr (BIT == 4) {
        const auto r = __builtin_amdgcn_permlane16_swap(x, x, false, false);
        return hi ? r[0] : r[1];
    }
    if constexpr (BIT == 5) {
        const auto r = __builtin_amdgcn_permlane32_swap(x, x, false, false);
        return hi ? r[0] : r[1];
    }
}
template <int BIT>
__device__ __forceinline__ float partner(float x, bool hi)
{
    return __uint_as_float(partner32<BIT>(__float_as_uint(x), hi));
}
template <int BIT>
__device__ __forceinline__ double partner(double x, bool hi)
{
    return __hiloint2double((int)partner32<BIT>((uint32_t)__double2hiint(x), hi),
                            (int)partner32<BIT>((uint32_t)__double2loint(x), hi));
}
template <int BIT, int N, typename R>
__device__ __forceinline__ void partners(const cplx<R>* a, cplx<R>* p, bool hi)
{
#pragma unroll
    for (int j = 0; j < N; j++) {
        p[j].x = partner<BIT>(a[j].x, hi);
        p[j].y = partner<BIT>(a[j].y, hi);
    }
}

template <int RB, typename R>
__global__ __launch_bounds__(256) void k_run(cplx<R>* __restrict__ psi, const Run<R> run)
{
    constexpr int NR = 1 << RB;
    uint64_t base = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
#pragma unroll
    for (int k = 0; k < RB; k++) {
        const int p = run.pos[k];
        base = ((base >> p) << (p + 1)) | (base & (((uint64_t)1 << p) - 1));
    }
    cplx<R>* const at = psi + base;
    uint64_t off[NR];
    cplx<R> a[NR];
#pragma unroll
    for (int j = 0; j < NR; j++) {
        off[j] = 0;
#pragma unroll
        for (int k = 0; k < RB; k++) if ((j >> k) & 1) off[j] |= (uint64_t)1 << run.pos[k];
        a[j] = at[off[j]];
    }
    auto apply = [&](const R* m, const RunFields& g) {
        const uint32_t rmask = g.rmask;
        const bool lane = (base & g.omask) == g.omask;
        if (g.form <= RUN_Y) {
            if ((g.omask | rmask) != 0) {
                switch (g.pos) {
                case 0: run_reg<0, true, RB, R>(a, g.form, m, lane, rmask); break;
                case 1: run_reg<1, true, RB, R>(a, g.form, m, lane, rmask); break;
                case 2: run_reg<2, true, RB, R>(a, g.form, m, lane, rmask); break;
                default: run_reg<3, true, RB, R>(a, g.form, m, lane, rmask); break;
                }
            } else {
                switch (g.pos) {
                case 0: run_reg<0, false, RB, R>(a, g.form, m, lane, rmask); break;
                case 1: run_reg<1, false, RB, R>(a, g.form, m, lane, rmask); break;
                case 2: run_reg<2, false, RB, R>(a, g.form, m, lane, rmask); break;
                default: run_reg<3, false, RB, R>(a, g.form, m, lane, rmask); break;
                }
            }
        } else if (g.form == RUN_DIAG) {
            // factor of the lane's amplitudes with the register target clear and set
            const bool hi = (base & g.tbit) != 0;
            const R lr = hi ? m[6] : m[0], li = hi ? m[7] : m[1], hr = m[6], hi_i = m[7];
            switch (g.rbit) {
            case 0: run_scale<RB, -1>(a, lr, li, hr, hi_i, false); break;
            case 1: run_scale<RB, 0>(a, lr, li, hr, hi_i, g.phase != 0); break;
            case 2: run_scale<RB, 1>(a, lr, li, hr, hi_i, g.phase != 0); break;
            case 4: run_scale<RB, 2>(a, lr, li, hr, hi_i, g.phase != 0); break;
            default: run_scale<RB, 3>(a, lr, li, hr, hi_i, g.phase != 0); break;
            }
        } else if (g.form >= RUN_DIAG_REAL) {
            // Amplitudes the gate leaves alone keep their value, as in a pass
            // of the gate alone: multiplied by 1 + 0i, an infinite part would
            // become NaN.  Signs multiply by a real 1; other factors skip the
            // lanes, and select under register controls (64 controlled phases
            // on 26 qubits complex128: 1.36 ms by 1 + 0i, 1.56; random layers
            // within 1 %).
            const bool hi = (base & g.tbit) != 0, act = lane && (hi || g.tbit == 0 || !g.phase);
            const uint32_t need = g.phase ? rmask | g.rbit : rmask;
            if (g.form == RUN_DIAG_REAL) {
                const R lr = act ? (hi ? m[6] : m[0]) : R(1), hr = act ? m[6] : R(1);
#pragma unroll
                for (int j = 0; j < NR; j++) {
                    const R f = ((uint32_t)j & need) != need ? R(1) : ((uint32_t)j & g.rbit) != 0 ? hr : lr;
                    a[j].x *= f;
                    a[j].y *= f;
                }
            } else if (rmask == 0) {
                const R lr = hi ? m[6] : m[0], li = hi ? m[7] : m[1], hr = m[6], hi_i = m[7];
                if (act) {
                    switch (g.rbit) {
                    case 0: run_scale<RB, -1>(a, lr, li, hr, hi_i, false); break;
                    case 1: run_scale<RB, 0>(a, lr, li, hr, hi_i, g.phase != 0); break;
                    case 2: run_scale<RB, 1>(a, lr, li, hr, hi_i, g.phase != 0); break;
                    case 4: run_scale<RB, 2>(a, lr, li, hr, hi_i, g.phase != 0); break;
                    default: run_scale<RB, 3>(a, lr, li, hr, hi_i, g.phase != 0); break;
                    }
                }
            } else {
                const R lr = hi ? m[6] : m[0], li = hi ? m[7] : m[1], hr = m[6], hi_i = m[7];
#pragma unroll
                for (int j = 0; j < NR; j++) {
                    const bool set = ((uint32_t)j & g.rbit) != 0, on = act && ((uint32_t)j & need) == need;
                    const R fr = set ? hr : lr, fi = set ? hi_i : li, x = a[j].x, y = a[j].y;
                    cplx<R> v;
                    v.x = fr * x - fi * y;
                    v.y = fr * y + fi * x;
                    a[j] = pick(on, v, a[j]);
                }
            }
        } else {
            // a lane's amplitude and its partner's, in the order (own, other)
            const bool hi = (base & g.tbit) != 0;
            const R or_ = hi ? m[6] : m[0], oi = hi ? m[7] : m[1], pr = hi ? m[4] : m[2], pi = hi ? m[5] : m[3];
#pragma unroll
            for (int h = 0; h < NR; h += NR / 2) {
                cplx<R> p[NR / 2];
                switch (g.pos) {
                case 0: partners<0, NR / 2>(a + h, p, hi); break;
                case 1: partners<1, NR / 2>(a + h, p, hi); break;
                case 2: partners<2, NR / 2>(a + h, p, hi); break;
                case 3: partners<3, NR / 2>(a + h, p, hi); break;
                case 4: partners<4, NR / 2>(a + h, p, hi); break;
                default: partners<5, NR / 2>(a + h, p, hi); break;
                }
                if (g.form == RUN_LREAL) {
#pragma unroll
                    for (int j = 0; j < NR / 2; j++) {
                        p[j].x = or_ * a[h + j].x + pr * p[j].x;
                        p[j].y = or_ * a[h + j].y + pr * p[j].y;
                    }
                } else if (g.form == RUN_LRX) {
#pragma unroll
                    for (int j = 0; j < NR / 2; j++) {
                        const cplx<R> t = p[j];
                        p[j].x = or_ * a[h + j].x - pi * t.y;
                        p[j].y = or_ * a[h + j].y + pi * t.x;
                    }
                } else if (g.form == RUN_LGEN) {
#pragma unroll
                    for (int j = 0; j < NR / 2; j++) {
                        const cplx<R> o = a[h + j], t = p[j];
                        p[j].x = or_ * o.x - oi * o.y + (pr * t.x - pi * t.y);
                        p[j].y = or_ * o.y + oi * o.x + (pr * t.y + pi * t.x);
                    }
                } else if (g.form == RUN_LY) {
#pragma unroll
                    for (int j = 0; j < NR / 2; j++) {
                        const cplx<R> t = p[j];
                        p[j].x = hi ? -t.y : t.y;
                        p[j].y = hi ? t.x : -t.x;
                    }
                }
                if ((g.omask | rmask) == 0) {
#pragma unroll
                    for (int j = 0; j < NR / 2; j++) a[h + j] = p[j];
                } else {
#pragma unroll
                    for (int j = 0; j < NR / 2; j++) {
                        const bool on = lane && ((uint32_t)(h + j) & rmask) == rmask;
                        a[h + j] = pick(on, p[j], a[h + j]);
                    }
                }
            }
        }
    };
    if constexpr (RB < RUN_MAX_RB) {
        // Few waves: the gates go to LDS in one latency instead of one per
        // gate.  (With 16 amplitudes a thread the barrier costs more than
        // that at size: 30 qubits 7.9 against 7.5 ms a pass.)
        __shared__ RunGate<R> gates[RUN_GATES];
        for (uint32_t t = threadIdx.x; t < (uint32_t)run.num * (sizeof(RunGate<R>) / 16); t += blockDim.x)
            __builtin_memcpy((char*)gates + 16 * t, (const char*)run.g + 16 * t, 16);
        __syncthreads();
        for (int q = 0; q < run.num; q++) apply(gates[q].m, gates[q].f.uniform());
    } else {
        RunGate<R> next = run.g[0];
        for (int q = 0; q < run.num; q++) {
            const RunGate<R> g = next;
            next = run.g[q + 1];     // read while this one is applied
            apply(g.m, g.f);
        }
    }
#pragma unroll
    for (int j = 0; j < NR; j++) at[off[j]] = a[j];
}

// Share of the state that k_plain moves for a gate: the pairs whose controls
// are set, half of each for a phase
static double plain_share(const hq_gate& g)
{
    double f = classify_gate(g) == SHM_PHASE ? 0.5 : 1.0;
    if (g.control >= 0) f *= 0.5;
    if (g.control2 >= 0) f *= 0.5;
    return f;
}

static bool run_diagonal(int cls) { return cls == SHM_DIAG || cls == SHM_PHASE; }

struct PlainGate {
    int index;           // in the call's array
    bool done;
    uint64_t qubits;     // target and controls
    uint64_t reg;        // the register bit it needs, 0 for lane targets and diagonal gates
    double share;
};

// The gates of the next pass, in order: those among the next RUN_AHEAD that
// share no qubit with a gate left out before them (so that they commute with
// it) and whose targets fit.  1350 gates of random layers on 30 qubits need 90
// passes, 190 without looking past the first gate that does not fit.
constexpr size_t RUN_AHEAD = 256;

static void next_run(int rb, std::vector<PlainGate>& list, size_t first, uint64_t all, std::vector<int>* members,
                     uint64_t* regs, double* share)
{
    members->clear();
    *regs = 0;
    *share = 0;
    uint64_t blocked = 0;
    const size_t end = std::min(list.size(), first + RUN_AHEAD);
    for (size_t i = first; i < end && blocked != all && (int)members->size() < RUN_GATES; i++) {
        PlainGate& g = list[i];
        if (g.done) continue;
        if ((g.qubits & blocked) || __builtin_popcountll(*regs | g.reg) > rb) {
            blocked |= g.qubits;
            continue;
        }
        *regs |= g.reg;
        g.done = true;
        members->push_back(g.index);
        *share += g.share;
    }
}

template <int RB, typename R>
static hq_status launch_run(hq_state s, const hq_gate* gates, const std::vector<int>& members, uint64_t regs)
{
    // register bits without a target: the highest free ones
    for (int q = s->n - 1; __builtin_popcountll(regs) < RB; q--) regs |= (uint64_t)1 << q;
    Run<R> run = {};
    int bit_of[64], k = 0;
    for (int q = 0; q < s->n; q++) {
        bit_of[q] = -1;
        if (regs >> q & 1) { run.pos[k] = q; bit_of[q] = k++; }
    }
    run.num = 0;
    for (int i : members) {
        const hq_gate& g = gates[i];
        const int cls = classify_gate(g);
        RunGate<R>& rg = run.g[run.num++];
        RunFields& o = rg.f;
        for (int j = 0; j < 8; j++) rg.m[j] = (R)g.mat[j];
        o.omask = o.tbit = 0;
        o.pos = o.rmask = o.rbit = o.phase = 0;
        for (int c : {g.control, g.control2}) {
            if (c < 0) continue;
            if (bit_of[c] >= 0) o.rmask |= 1u << bit_of[c];
            else o.omask |= (uint64_t)1 << c;
        }
        const int rb = bit_of[g.target];
        if (run_diagonal(cls)) {
            if (cls == SHM_PHASE) { rg.m[0] = R(1); rg.m[1] = R(0); o.phase = 1; }
            if (rb >= 0) o.rbit = 1u << rb;
            else o.tbit = (uint64_t)1 << g.target;
            const bool some = o.omask || o.rmask || (o.phase && o.tbit);
            o.form = !some ? RUN_DIAG : rg.m[1] == R(0) && rg.m[7] == R(0) ? RUN_DIAG_REAL : RUN_DIAG_SOME;
        } else if (rb >= 0) {
            o.form = cls == SHM_SWAP ? RUN_SWAP : cls == SHM_Y ? RUN_Y : cls == SHM_REAL ? RUN_REAL
                     : cls == SHM_RX ? RUN_RX : RUN_GEN;
            o.pos = (uint32_t)rb;
        } else {
            o.form = cls == SHM_SWAP ? RUN_LSWAP : cls == SHM_Y ? RUN_LY : cls == SHM_REAL ? RUN_LREAL
                     : cls == SHM_RX ? RUN_LRX : RUN_LGEN;
            o.pos = (uint32_t)g.target;
            o.tbit = (uint64_t)1 << g.target;
        }
    }
    const uint64_t threads = s->amps >> RB, block = std::min<uint64_t>(threads, 256);
    hipLaunchKernelGGL((k_run<RB, R>), dim3((unsigned)(threads / block)), dim3((unsigned)block), 0, s->stream,
                       (cplx<R>*)s->data, run);
    HQ_HIP(hipGetLastError());
    return HQ_OK;
}

template <typename R>
static hq_status apply_plain(hq_state s, const hq_gate* gates, int num)
{
    if (s->n < RUN_MIN_QUBITS || num == 1) {
        for (int i = 0; i < num; i++) {
            if (gates[i].type == HQ_ID) continue;
            hq_status st = launch_plain_gate<R>(s, gates[i]);
            if (st != HQ_OK) return st;
        }
        return HQ_OK;
    }
    std::vector<PlainGate> list;
    list.reserve((size_t)num);
    for (int i = 0; i < num; i++) {
        const hq_gate& g = gates[i];
        if (g.type == HQ_ID) continue;
        PlainGate p{i, false, (uint64_t)1 << g.target, 0, plain_share(g)};
        for (int c : {g.control, g.control2})
            if (c >= 0) p.qubits |= (uint64_t)1 << c;
        if (g.target >= RUN_LANES && !run_diagonal(classify_gate(g))) p.reg = (uint64_t)1 << g.target;
        list.push_back(p);
    }
    const uint64_t all = ((uint64_t)1 << s->n) - 1;
    // a launch costs what 20 MB of traffic do, in passes over the state
    const double launch = 20e6 / (2.0 * (double)s->amps * sizeof(cplx<R>));
    const int rb = s->n <= RUN_SMALL_QUBITS ? 3 : 4;
    std::vector<int> members;
    for (size_t first = 0;;) {
        while (first < list.size() && list[first].done) first++;
        if (first == list.size()) return HQ_OK;
        uint64_t regs;
        double share;
        next_run(rb, list, first, all, &members, &regs, &share);
        hq_status st = HQ_OK;
        if (members.size() > 1 && share + (double)(members.size() - 1) * launch > RUN_MIN_SHARE) {
            st = rb == 3 ? launch_run<3, R>(s, gates, members, regs) : launch_run<4, R>(s, gates, members, regs);
        } else {
            for (size_t k = 0; k < members.size() && st == HQ_OK; k++) st = launch_plain_gate<R>(s, gates[members[k]]);
        }
        if (st != HQ_OK) return st;
    }
}

}  // namespace hq

using namespace hq;

extern "C" hq_status hq_apply_gates_plain(hq_state s, const hq_gate* gates, int num_gates)
{
    HQ_CHECK(s, HQ_ERR_ARG, "hq_apply_gates_plain: null state");
    HQ_CHECK(num_gates >= 0 && (num_gates == 0 || gates), HQ_ERR_ARG, "hq_apply_gates_plain: bad gate array");
    for (int i = 0; i < num_gates; i++) {
        hq_status st = validate_gate(gates[i], s->n);
        if (st != HQ_OK) return st;
    }
    int slot;
    hq_status st = prof_begin(s, 0, &slot);
    if (st != HQ_OK) return st;
    try {
        st = s->precision == HQ_C128 ? apply_plain<double>(s, gates, num_gates)
                                     : apply_plain<float>(s, gates, num_gates);
    } catch (const std::bad_alloc&) {
        set_error("hq_apply_gates_plain: out of host memory");
        return HQ_ERR_OOM;
    }
    if (st != HQ_OK) return st;
    return prof_end(s, slot);
}
