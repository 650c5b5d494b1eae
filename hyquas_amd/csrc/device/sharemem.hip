// sharemem.hip -- OShareMem: one HBM pass applies a whole gate group.
//
// Reference behaviour (src/kernelOpt.cu:388-433, src/executor.cpp:462-493,
// 585-632): each block owns the 2^k amplitudes that differ only in the k
// "shared" qubits, loads them, applies every gate of the group, stores them.
// Gates whose target is outside the tile must be diagonal; controls and
// diagonal targets may sit on block bits.
//
// MI355X design (not the reference's): the tile lives in REGISTERS, not in
// shared memory.  Each thread holds 2^RB amplitudes; the tile bits are split
// per stage into RB register bits and TB thread bits (k = RB + TB).  Every
// non-diagonal gate of a stage targets a register bit, so it is a pure
// register update; diagonal gates and controls on thread or block bits are
// per-lane / per-block predicates.  Between stages the tile is re-split by
// one LDS exchange (write, barrier, read).  The first stage reads HBM directly
// and the last writes HBM directly, so a group with s stages costs one HBM
// read + write and s-1 LDS round trips instead of one LDS round trip per gate.
// LDS addresses are XOR-swizzled (tile bits >= 3 fold into bits 0..2) and
// the host picks lane bits 0..2 so that 8-lane groups hit distinct 16-byte
// bank groups.

#include "sharemem_dev.h"

#include <algorithm>
#include <cmath>
#include <complex>
#include <cstdlib>
#include <cstring>

namespace hq {

// ---- device side ----------------------------------------------------------------------

template <typename R, int RB, int TB>
__global__ __launch_bounds__(1 << TB) void k_sharemem(cplx<R>* __restrict__ psi, const char* __restrict__ prog,
                                                     uint32_t mode)
{
    __shared__ cplx<R> lds[1 << (RB + TB)];
    __shared__ __align__(16) char win[SHM_WINDOW_LDS];
    tile_pass<R, RB, TB, sizeof(R) == 4>(psi, prog, blockIdx.x, lds, win, mode, 0, nullptr);
}

// ---- launch table -------------------------------------------------------------------------

template <typename R, int RB, int TB>
static hq_status launch_variant(hq_state s, hq_program p)
{
    uint64_t blocks = (uint64_t)1 << (p->n - p->tile);
    const uint32_t mode = p->plan && p->plan->init ? TILE_INIT : 0u;
    hipLaunchKernelGGL((k_sharemem<R, RB, TB>), dim3((unsigned)blocks), dim3(1 << TB), 0, s->stream,
                       (cplx<R>*)s->data, (const char*)p->d_prog, mode);
    HQ_HIP(hipGetLastError());
    return HQ_OK;
}

template <typename R>
static hq_status launch_by_shape(hq_state s, hq_program p)
{
    const int rb = p->rb, tb = p->tb;
#define HQ_SHM_CASE(RBV, TBV) \
    if (rb == RBV && tb == TBV) return launch_variant<R, RBV, TBV>(s, p);
    HQ_SHM_CASE(1, 6) HQ_SHM_CASE(2, 6) HQ_SHM_CASE(3, 6) HQ_SHM_CASE(4, 6) HQ_SHM_CASE(5, 6)
    HQ_SHM_CASE(2, 7) HQ_SHM_CASE(3, 7) HQ_SHM_CASE(4, 7) HQ_SHM_CASE(5, 7)
    HQ_SHM_CASE(3, 8) HQ_SHM_CASE(4, 8) HQ_SHM_CASE(5, 8) HQ_SHM_CASE(3, 9) HQ_SHM_CASE(4, 9)
    if constexpr (sizeof(R) == 4) { HQ_SHM_CASE(6, 8) }   // 14-qubit complex64 tiles
#undef HQ_SHM_CASE
    set_error("sharemem: no kernel for this register/thread split");
    return HQ_ERR_UNSUPPORTED;
}

static bool shape_supported(int rb, int tb, int precision)
{
    static const int shapes[][2] = {{1, 6}, {2, 6}, {3, 6}, {4, 6}, {5, 6}, {2, 7}, {3, 7},
                                    {4, 7}, {5, 7}, {3, 8}, {4, 8}, {5, 8}, {3, 9}, {4, 9}};
    for (auto& sh : shapes)
        if (sh[0] == rb && sh[1] == tb) return true;
    return precision == HQ_C64 && rb == 6 && tb == 8;
}

hq_status launch_sharemem(hq_state s, hq_program p)
{
    return s->precision == HQ_C128 ? launch_by_shape<double>(s, p) : launch_by_shape<float>(s, p);
}

int sharemem_default_rb(int precision, int tile)
{
    // tile = RB + TB; 256-thread blocks with 16 (complex128) or 32 (complex64)
    // amplitudes per thread at the default 12/13-qubit tiles
    if (tile <= 10) return std::max(1, tile - 6);
    if (precision == HQ_C128) return tile >= 13 ? 5 : 4;
    // complex64: 256 threads x 16 amplitudes at 12 qubits measured fastest;
    // 14-qubit tiles hold 64 amplitudes per thread (the register bytes of a
    // 13-qubit complex128 tile)
    return tile >= 14 ? 6 : tile == 13 ? 5 : tile == 12 ? 4 : tile - 6;
}

int interpreter_rb(int precision, int tile, int n)
{
    // Up to a block or two per CU a pass is a chain of ops whose latency shows:
    // 8 amplitudes on twice the threads take less of it per op than 16 and one
    // more exchange per stage costs.  12-qubit tiles, 16 random layers, 16 and
    // 8 amplitudes: complex64 17 qubits 212 and 165 us, 20 qubits 367 and 235,
    // 21 qubits (512 blocks) 407 and 339; complex128 17 qubits 210 and 186, 20
    // qubits 334 and 306, but 21 qubits 413 and 515.  10 qubits in one block: 103 and 87.
    if (tile >= 10 && tile <= 12 && n - tile <= (precision == HQ_C128 ? 8 : 9)) return 3;
    // 13-qubit complex64 blocks: 512 threads x 16 instead of 256 x 32 (100
    // ansatz circuits of 10 to 14 qubits: 0.93 and 1.16 ms)
    if (tile == 13 && precision == HQ_C64) return 4;
    return sharemem_default_rb(precision, tile);
}

// ---- host side: lowering + register-stage planning -------------------------------------------

namespace {

struct Lowered {
    int cls;
    bool needs_reg;       // non-diagonal update: target must be a register bit
    int t_tile, t_block;  // target as tile bit or block bit (-1 if not)
    int c_tile[2], c_block[2];
    double m[8];
    std::complex<double> scale{1.0, 0.0};   // factored out of m (applied later in the pass)
};

// Rotation [[c, -s], [s, c]] (c >= 0 after the sign is moved into the
// scalar) as three shears: [[1, a], [0, 1]] [[1, 0], [b, 1]] [[1, a], [0, 1]]
// with a = -tan(phi / 2) = -s / (1 + c), b = s = sin(phi); |a|, |b| <= 1 and
// no division by a small number, for every angle.
void shear_form(double c, double s, double* a, double* b, std::complex<double>* S)
{
    const double r = std::hypot(c, s);
    c /= r;
    s /= r;
    double sigma = 1.0;
    if (c < 0) { c = -c; s = -s; sigma = -1.0; }
    *S *= sigma * r;
    *a = -s / (1.0 + c);
    *b = s;
}

// Factor a scalar out of an uncontrolled gate so that its pair update needs
// half the multiplies: H = r [[1, 1], [1, -1]]; a rotation [[c, -s], [s, c]]
// = c [[1, -t], [t, 1]] (t = s/c) or s [[u, -1], [1, u]] (u = c/s), whichever
// keeps |t|, |u| <= 1; RX-type [[a, ib], [ib, a]] likewise; a unit diagonal
// diag(d0, d1) = d0 diag(1, d1/d0).  Other gates are left as they are.
// True when the gate was rewritten (its scalar multiplied into S).
bool factor_scalar(Lowered& L, std::complex<double>* S, bool shared_code)
{
    double* m = L.m;
    // shared_code: only factorings whose op class does not depend on the
    // angle, so groups that differ only in angles emit the same specialised
    // kernel source: H, unit diagonals, and rotations as three shears
    if (shared_code && L.cls == SHM_REAL && m[0] == m[6] && m[2] == -m[4] && (m[0] != 0 || m[4] != 0)) {
        double a, b;
        shear_form(m[0], m[4], &a, &b, S);
        L.cls = SHM_SHEAR;
        memset(m, 0, sizeof(L.m));
        m[0] = a;
        m[2] = b;
        return true;
    }
    if (shared_code && L.cls == SHM_RX && m[0] == m[6] && m[3] == m[5] && (m[0] != 0 || m[3] != 0)) {
        // [[c, -i s], [-i s, c]] = diag(1, -i) [[c, -s], [s, c]] diag(1, i)
        double a, b;
        shear_form(m[0], -m[3], &a, &b, S);
        L.cls = SHM_SHEARX;
        memset(m, 0, sizeof(L.m));
        m[0] = a;
        m[2] = b;
        return true;
    }
    if (shared_code && (L.cls == SHM_RX || (L.cls == SHM_REAL && !(m[0] == m[2] && m[0] == m[4] && m[0] == -m[6]))))
        return false;
    const int cls_in = L.cls;
    if (L.cls == SHM_REAL) {
        if (m[0] == m[2] && m[0] == m[4] && m[0] == -m[6] && m[0] != 0) {
            *S *= m[0];
            L.cls = SHM_HADD;
            memset(m, 0, sizeof(L.m));
        } else if (m[0] == m[6] && m[2] == -m[4] && (m[0] != 0 || m[4] != 0)) {
            const double c = m[0], s = m[4];
            if (std::fabs(c) >= std::fabs(s)) { *S *= c; L.cls = SHM_ROTA; memset(m, 0, sizeof(L.m)); m[0] = s / c; }
            else { *S *= s; L.cls = SHM_ROTB; memset(m, 0, sizeof(L.m)); m[0] = c / s; }
        }
    } else if (L.cls == SHM_RX) {
        // lo' = a lo + i b hi, hi' = i c lo + d hi with a = d, b = c
        const double a = m[0], b = m[3];
        if (a == m[6] && b == m[5] && (a != 0 || b != 0)) {
            if (std::fabs(a) >= std::fabs(b)) { *S *= a; L.cls = SHM_RXA; memset(m, 0, sizeof(L.m)); m[0] = b / a; }
            else { *S *= b; L.cls = SHM_RXB; memset(m, 0, sizeof(L.m)); m[0] = a / b; }
        }
    } else if (L.cls == SHM_DIAG) {
        const std::complex<double> d0(m[0], m[1]), d1(m[6], m[7]);
        if (std::fabs(std::abs(d0) - 1.0) < 1e-12) {
            const std::complex<double> q = d1 / d0;
            *S *= d0;
            L.cls = SHM_PHASE;
            memset(m, 0, sizeof(L.m));
            m[0] = 1.0;
            m[6] = q.real();
            m[7] = q.imag();
        }
    }
    return L.cls != cls_in;
}

// swizzle column of tile bit i (bits >= 3 fold into the low 3 bits)
uint32_t swz_column(int i)
{
    static const uint32_t cyc[7] = {3, 5, 6, 7, 1, 2, 4};
    return i < 3 ? (1u << i) : cyc[(i - 3) % 7];
}

// GF(2) rank of a set of 3-bit vectors
int rank3(const std::vector<uint32_t>& v)
{
    uint32_t basis[3] = {0, 0, 0};
    int r = 0;
    for (uint32_t x : v) {
        for (int b = 2; b >= 0; b--) {
            if (!((x >> b) & 1)) continue;
            if (!basis[b]) { basis[b] = x; r++; break; }
            x ^= basis[b];
        }
    }
    return r;
}

// Turns the gates of the register stages into ops.  Diagonal gates are not
// emitted where they stand: each is one or two factors ("terms") on the
// amplitudes whose bits match, and a term commutes with every other term and
// with every gate whose target is not one of its bits.  Terms stay pending
// until a gate mixes one of their bits (or the pass ends) and are then applied
// together:
//   terms on register bits alone       one table over the register index
//   terms on thread and block bits     one factor per lane, commuting with all
//                                      of a stage's ops; in the last stage it
//                                      carries the scale of the factored gates
//   terms on both                      SHM_MIX, only if still mixed when forced
// Register-controlled X permutes a pending table instead of forcing it.  One
// table or lane factor costs 4 operations per amplitude whatever it merges; a
// diagonal gate by itself costs 2 (register bit) or 4 (thread or block bit).
class StageLowering {
public:
    StageLowering(const std::vector<Lowered>& low, const std::vector<int>& type, int precision, int rb, int tb,
                  bool shared, bool precise, bool merge)
        : low_(low), type_(type), rb_(rb), tb_(tb), nr_(1 << rb), shared_(shared), precise_(precise),
          merge_(merge),          limit_(precision == HQ_C128 ? 480.0 : 48.0)
    {
    }

    void stage(const ShmStage& st, const ShmStage* next, const std::vector<int>& gates, bool factored,
               std::vector<ShmOp>* ops, std::vector<double>* tabs)
    {
        ops_ = ops;
        tabs_ = tabs;
        regset_ = set_of(st.reg_bits, rb_);
        for (int i = 0; i < SHM_MAX_TILE; i++) reg_[i] = thr_[i] = -1;
        for (int i = 0; i < rb_; i++) reg_[st.reg_bits[i]] = i;
        for (int i = 0; i < tb_; i++) thr_[st.thr_bits[i]] = i;
        reset_table();
        for (int idx : gates) {
            const Lowered& L = low_[idx];
            if (L.needs_reg) mixing(L, type_[idx]);
            else diagonal(L, type_[idx]);
            add_scale(L);
        }
        std::vector<Term> lane;
        if (!next) {
            take([&](const Term& t) { return !(t.tmask & regset_); }, &lane);
            take_mixed(~0u);
            flush_table();
            if (!lane.empty() || factored) emit_lane(lane, true, factored);
            return;
        }
        // terms of one bit stay pending; terms of several are applied in the
        // form they have if they would be mixed in the next stage
        const uint32_t nreg = set_of(next->reg_bits, rb_);
        auto mixed_next = [&](const Term& t) { return (t.tmask & nreg) && ((t.tmask & ~nreg) || t.bmask); };
        std::vector<Term> now;
        take([&](const Term& t) { return reg_only(t) && mixed_next(t); }, &now);
        for (auto& t : now) table_add(t);
        if (tactive_) flush_table();
        bool need = false;
        for (auto& t : pend_) need = need || (!(t.tmask & regset_) && mixed_next(t));
        if (need) {
            take([&](const Term& t) { return !(t.tmask & regset_); }, &lane);
            emit_lane(lane, false, false);
        }
    }

private:
    struct Term {
        uint32_t tmask, tval;   // tile bits
        uint32_t bmask, bval;   // block bits
        std::complex<double> f;
        bool konst, real;
        int gates;              // factors multiplied into f
    };

    // a gate's factor as one float: what the gate alone would multiply by
    std::complex<double> rounded(const std::complex<double>& f) const
    {
        return precise_ ? std::complex<double>((float)f.real(), (float)f.imag()) : f;
    }

    static uint32_t set_of(const uint32_t* bits, int n)
    {
        uint32_t s = 0;
        for (int i = 0; i < n; i++) s |= 1u << bits[i];
        return s;
    }
    static bool const_type(int type)
    {
        switch (type) {
        case HQ_CCX: case HQ_CNOT: case HQ_CY: case HQ_CZ: case HQ_H: case HQ_X: case HQ_Y: case HQ_Z:
        case HQ_S: case HQ_SDG: case HQ_T: case HQ_TDG: case HQ_ID: case HQ_GII: case HQ_GZZ:
            return true;
        default:
            return false;
        }
    }
    bool reg_only(const Term& t) const { return !t.bmask && !(t.tmask & ~regset_) && t.tmask; }

    // masks of tile bits over the stage's register / thread index
    uint32_t to_reg(uint32_t tile) const
    {
        uint32_t r = 0;
        for (int b = 0; b < SHM_MAX_TILE; b++)
            if (((tile >> b) & 1) && reg_[b] >= 0) r |= 1u << reg_[b];
        return r;
    }
    uint32_t to_thr(uint32_t tile) const
    {
        uint32_t r = 0;
        for (int b = 0; b < SHM_MAX_TILE; b++)
            if (((tile >> b) & 1) && thr_[b] >= 0) r |= 1u << thr_[b];
        return r;
    }

    template <typename Pred>
    void take(Pred pred, std::vector<Term>* out)
    {
        std::vector<Term> keep;
        for (auto& t : pend_) (pred(t) ? *out : keep).push_back(t);
        pend_.swap(keep);
    }

    void diagonal(const Lowered& L, int type)
    {
        for (int v = 0; v < 2; v++) {
            const std::complex<double> f(v ? L.m[6] : L.m[0], v ? L.m[7] : L.m[1]);
            // the |0> half of a phase is 1 by the gate's form
            if (!v && L.cls == SHM_PHASE) continue;
            Term t{0, 0, 0, 0, rounded(f), const_type(type), type == HQ_Z || type == HQ_CZ, 1};
            if (L.t_tile >= 0) { t.tmask |= 1u << L.t_tile; t.tval |= (uint32_t)v << L.t_tile; }
            else { t.bmask |= 1u << L.t_block; t.bval |= (uint32_t)v << L.t_block; }
            for (int c = 0; c < 2; c++) {
                if (L.c_tile[c] >= 0) { t.tmask |= 1u << L.c_tile[c]; t.tval |= 1u << L.c_tile[c]; }
                if (L.c_block[c] >= 0) { t.bmask |= 1u << L.c_block[c]; t.bval |= 1u << L.c_block[c]; }
            }
            if (!merge_) {
                push_mix(t);
                continue;
            }
            bool merged = false;
            for (auto& p : pend_) {
                if (precise_) break;   // a product would be rounded once more
                if (p.tmask != t.tmask || p.tval != t.tval || p.bmask != t.bmask || p.bval != t.bval) continue;
                p.f *= t.f;
                p.gates++;
                p.konst = p.konst && t.konst;
                p.real = p.real && t.real;
                merged = true;
                break;
            }
            if (!merged) pend_.push_back(t);
        }
    }

    void mixing(const Lowered& L, int type)
    {
        const uint32_t pbit = 1u << L.t_tile;
        const int P = reg_[L.t_tile];
        uint32_t ct = 0, cb = 0;
        for (int c = 0; c < 2; c++) {
            if (L.c_tile[c] >= 0) ct |= 1u << L.c_tile[c];
            if (L.c_block[c] >= 0) cb |= 1u << L.c_block[c];
        }
        ShmOp o;
        o.cls = (uint8_t)L.cls;
        o.tpos = (uint8_t)P;
        o.creg = o.cregv = (uint8_t)to_reg(ct);
        o.cthr = o.cthrv = (uint16_t)to_thr(ct);
        o.cblk = o.cblkv = cb;
        memcpy(o.m, L.m, sizeof(o.m));
        // a thread-bit control makes the op the identity on some lanes: Y
        // takes an update form whose coefficients can express the identity
        if (o.cthr && o.cls == SHM_Y) o.cls = SHM_RX;
        if (const_type(type)) o.flags |= SHM_FLAG_CONST;
        const bool perm = L.cls == SHM_SWAP && !o.cthr && !cb;
        if (perm && !ct) {
            // X: the value a term asks of this bit flips
            for (auto& t : pend_) t.tval ^= t.tmask & pbit;
        } else {
            take_mixed(pbit);
            std::vector<Term> now;
            if (perm) {
                take([&](const Term& t) { return (t.tmask & pbit) != 0; }, &now);
                for (auto& t : now) table_add(t);
            } else {
                bool need = tactive_ && ((tdep_ >> P) & 1);
                for (auto& t : pend_) need = need || (t.tmask & pbit);
                if (need) flush_table();
            }
        }
        if (perm && tactive_) {
            for (int j = 0; j < nr_; j++) {
                if ((j >> P) & 1 || (j & o.creg) != o.creg) continue;
                std::swap(table_[j], table_[j | (1 << P)]);
                std::swap(used_[j], used_[j | (1 << P)]);
            }
            if ((tdep_ >> P) & 1) tdep_ |= o.creg;
        }
        ops_->push_back(o);
    }

    // applies the mixed terms on any of `bits` now
    void take_mixed(uint32_t bits)
    {
        std::vector<Term> now;
        take([&](const Term& t) { return (t.tmask & bits) && (t.tmask & regset_) && !reg_only(t); }, &now);
        for (auto& t : now) push_mix(t);
    }
    void push_mix(const Term& t)
    {
        ShmOp o;
        o.cls = SHM_MIX;
        o.creg = (uint8_t)to_reg(t.tmask);
        o.cregv = (uint8_t)to_reg(t.tval);
        lane_cond(t, &o);
        ops_->push_back(o);
    }

    void lane_cond(const Term& t, ShmOp* o) const
    {
        o->cthr = (uint16_t)to_thr(t.tmask);
        o->cthrv = (uint16_t)to_thr(t.tval);
        o->cblk = t.bmask;
        o->cblkv = t.bval;
        o->m[0] = t.f.real();
        o->m[1] = t.real ? 0.0 : t.f.imag();
        if (t.konst) o->flags |= SHM_FLAG_CONST;
        if (t.real) o->flags |= SHM_FLAG_REAL;
    }

    void reset_table()
    {
        table_.assign(nr_, 1.0);
        used_.assign(nr_, 0);
        tdep_ = 0;
        tactive_ = false;
    }
    void table_add(const Term& t)
    {
        const uint32_t m = to_reg(t.tmask), v = to_reg(t.tval);
        for (int j = 0; j < nr_; j++)
            if ((j & m) == v) { table_[j] *= t.f; used_[j] += t.real ? SIGN : (uint64_t)t.gates; }
        tdep_ |= m;
        tactive_ = true;
    }
    // applies the table, every pending term on register bits alone with it
    void flush_table()
    {
        std::vector<Term> now;
        take([&](const Term& t) { return reg_only(t); }, &now);
        for (auto& t : now) table_add(t);
        if (!tactive_) return;
        ShmOp o;
        o.cls = SHM_TAB;
        o.tab = (uint32_t)(tabs_->size() / 2);
        o.jdep = tdep_;
        for (int j = 0; j < nr_; j++) {
            if (used_[j]) o.jmask |= 1ull << j;
            if (precise_ && (used_[j] & (SIGN - 1)) > 1) o.jprod |= 1ull << j;
            tabs_->push_back(table_[j].real());
            tabs_->push_back(table_[j].imag());
        }
        ops_->push_back(o);
        reset_table();
    }

    void emit_lane(const std::vector<Term>& lane, bool scale, bool factored)
    {
        bool real = true;
        for (auto& t : lane) {
            ShmOp o;
            o.cls = SHM_LANE;
            lane_cond(t, &o);
            ops_->push_back(o);
            real = real && t.real;
        }
        push_scale(scale && factored, lane.empty(), real);
    }
    void push_scale(bool scale, bool nolane, bool real)
    {
        ShmOp o;
        o.cls = SHM_LANEMUL;
        o.m[0] = 1.0;
        if (nolane) o.flags |= SHM_FLAG_NOLANE;
        if (scale) {
            const std::complex<double> f = rounded(scale_);
            o.m[0] = f.real();
            o.m[1] = f.imag();
            scale_ = 1.0;
            logs_ = 0.0;
        } else {
            o.flags |= SHM_FLAG_UNIT;
            if (real) o.flags |= SHM_FLAG_REAL;
        }
        // nothing to multiply by: unless same-structure groups share the code
        if (nolane && !shared_ && o.m[0] == 1.0 && o.m[1] == 0.0) return;
        ops_->push_back(o);
    }
    // The amplitudes grow by 1 / |scale| until the scale is applied: a group of
    // hundreds of factored gates would leave float's range, so the scale is
    // also applied whenever that growth reaches 2^48 (2^480 in double).  Shared
    // code counts what the gates' types alone imply: 2^(1/2) per H.
    void add_scale(const Lowered& L)
    {
        if (L.scale == std::complex<double>(1.0, 0.0)) return;
        scale_ *= L.scale;
        logs_ += shared_ ? (L.cls == SHM_HADD ? -0.5 : 0.0) : std::log2(std::abs(L.scale));
        if (std::fabs(logs_) >= limit_) push_scale(true, true, false);
    }

    const std::vector<Lowered>& low_;
    const std::vector<int>& type_;
    const int rb_, tb_, nr_;
    const bool shared_, precise_, merge_;
    const double limit_;
    std::vector<Term> pend_;
    std::vector<ShmOp>* ops_ = nullptr;
    std::vector<double>* tabs_ = nullptr;
    uint32_t regset_ = 0;
    int reg_[SHM_MAX_TILE], thr_[SHM_MAX_TILE];
    std::vector<std::complex<double>> table_;
    static constexpr uint64_t SIGN = 1ull << 32;
    std::vector<uint64_t> used_;   // gates in each entry, signs counted in the upper half
    uint32_t tdep_ = 0;
    bool tactive_ = false;
    std::complex<double> scale_{1.0, 0.0};
    double logs_ = 0.0;
};

}  // namespace

hq_status plan_sharemem(int n, int precision, const hq_gate* gates, int num_gates, uint64_t shared_mask, int rb_req,
                        ShmPlan* plan, bool init, int io, bool shared_code, DiagMode diag)
{
    HQ_CHECK(num_gates >= 0 && (num_gates == 0 || gates), HQ_ERR_ARG, "sharemem: bad gate array");
    const size_t amp_bytes = precision == HQ_C128 ? 16 : 8;
    const uint64_t all = n >= 64 ? ~0ull : ((1ull << n) - 1);
    HQ_CHECK((shared_mask & ~all) == 0, HQ_ERR_ARG, "sharemem: shared mask has bits beyond the state");
    const int k = __builtin_popcountll(shared_mask);
    HQ_CHECK(k >= 7 && k <= SHM_MAX_TILE, HQ_ERR_ARG, "sharemem: tile must have 7..14 qubits");
    HQ_CHECK(((size_t)1 << k) * amp_bytes <= 160 * 1024, HQ_ERR_ARG, "sharemem: tile exceeds the 160 KiB LDS");
    const int rb = rb_req > 0 ? rb_req : sharemem_default_rb(precision, k);
    const int tb = k - rb;
    HQ_CHECK(shape_supported(rb, tb, precision), HQ_ERR_UNSUPPORTED, "sharemem: unsupported register/thread split");

    int tile_of[64], block_of[64];
    std::vector<int> tile_pos, block_pos;
    for (int q = 0; q < n; q++) {
        if ((shared_mask >> q) & 1) { tile_of[q] = (int)tile_pos.size(); block_of[q] = -1; tile_pos.push_back(q); }
        else { block_of[q] = (int)block_pos.size(); tile_of[q] = -1; block_pos.push_back(q); }
    }

    std::vector<Lowered> low;
    std::vector<int> low_type;
    low.reserve(num_gates);
    // uncontrolled H, RX, RY and unit diagonals lose a scalar factor; the
    // factors' product is applied at the end of the pass (HQ_SHM_FACTOR=0: off)
    static const bool factor = !getenv("HQ_SHM_FACTOR") || atoi(getenv("HQ_SHM_FACTOR")) != 0;
    bool factored = false;
    for (int i = 0; i < num_gates; i++) {
        const hq_gate& g = gates[i];
        hq_status st = validate_gate(g, n);
        if (st != HQ_OK) return st;
        if (g.type == HQ_ID) continue;
        Lowered L;
        L.cls = classify_gate(g);
        L.needs_reg = !(L.cls == SHM_DIAG || L.cls == SHM_PHASE);
        L.t_tile = tile_of[g.target];
        L.t_block = block_of[g.target];
        if (L.needs_reg && L.t_tile < 0) {
            set_error("sharemem: gate " + std::to_string(i) + " is not diagonal but its target is outside the tile");
            return HQ_ERR_ARG;
        }
        int cs[2] = {g.control, g.control2};
        for (int c = 0; c < 2; c++) {
            L.c_tile[c] = cs[c] >= 0 ? tile_of[cs[c]] : -1;
            L.c_block[c] = cs[c] >= 0 ? block_of[cs[c]] : -1;
        }
        memcpy(L.m, g.mat, sizeof(L.m));
        if (factor && g.control < 0 && g.control2 < 0 && factor_scalar(L, &L.scale, shared_code)) factored = true;
        low.push_back(L);
        low_type.push_back(g.type);
    }

    // greedy stage planning: take gates in order; a stage has at most RB
    // distinct register targets; a gate that cannot join blocks its qubits
    struct Stage {
        std::vector<int> reg_bits, thr_bits;
        std::vector<int> ops;
    };
    std::vector<Stage> stages;
    // thread bits: lanes 0..2 get three bits with independent swizzle
    // columns (lowest first), the rest follow in ascending order
    auto assign_lanes = [&](Stage& S, uint32_t regset) {
        std::vector<int> free_bits;
        for (int b = 0; b < k; b++)
            if (!((regset >> b) & 1)) free_bits.push_back(b);
        std::vector<int> lane3;
        std::vector<uint32_t> cols;
        for (int b : free_bits) {
            if (lane3.size() == 3) break;
            cols.push_back(swz_column(b));
            if (rank3(cols) == (int)cols.size()) lane3.push_back(b);
            else cols.pop_back();
        }
        for (int b : lane3) S.thr_bits.push_back(b);
        for (int b : free_bits)
            if (std::find(lane3.begin(), lane3.end(), b) == lane3.end()) S.thr_bits.push_back(b);
    };
    std::vector<int> pending(low.size());
    for (size_t i = 0; i < low.size(); i++) pending[i] = (int)i;
    // a tile above 64 KiB is exchanged in two LDS halves by the specialised
    // kernel, split on a register bit that consecutive stages share: keep one
    const bool split_lds = ((size_t)1 << k) * amp_bytes > 64 * 1024;
    uint32_t prev_reg = 0;
    do {
        Stage S;
        uint32_t regset = 0;
        int cnt = 0;
        uint32_t blk_tile = 0;
        uint64_t blk_block = 0;
        std::vector<int> rest;
        for (int idx : pending) {
            const Lowered& L = low[idx];
            uint32_t tt = L.t_tile >= 0 ? 1u << L.t_tile : 0;
            uint64_t tbk = L.t_block >= 0 ? 1ull << L.t_block : 0;
            for (int c = 0; c < 2; c++) {
                if (L.c_tile[c] >= 0) tt |= 1u << L.c_tile[c];
                if (L.c_block[c] >= 0) tbk |= 1ull << L.c_block[c];
            }
            bool ok = !(tt & blk_tile) && !(tbk & blk_block);
            if (ok && L.needs_reg) {
                uint32_t tb1 = 1u << L.t_tile;
                if (!(regset & tb1)) {
                    const bool keep = split_lds && !stages.empty() && !((regset | tb1) & prev_reg);
                    if (cnt < (keep ? rb - 1 : rb)) { regset |= tb1; cnt++; }
                    else ok = false;
                }
            }
            if (ok) S.ops.push_back(idx);
            else { blk_tile |= tt; blk_block |= tbk; rest.push_back(idx); }
        }
        if (split_lds && !stages.empty() && !(regset & prev_reg) && cnt < rb) {
            for (int b = k - 1; b >= 0; b--)
                if ((prev_reg >> b) & 1) { regset |= 1u << b; cnt++; break; }
        }
        // fill the register set with the highest remaining tile bits, so the
        // lanes cover the low (contiguous) tile bits
        for (int b = k - 1; b >= 0 && cnt < rb; b--)
            if (!((regset >> b) & 1)) { regset |= 1u << b; cnt++; }
        for (int b = 0; b < k; b++)
            if ((regset >> b) & 1) S.reg_bits.push_back(b);
        assign_lanes(S, regset);
        prev_reg = regset;
        stages.push_back(std::move(S));
        pending.swap(rest);
    } while (!pending.empty());

    // HBM-facing stages: the first stage's lanes load the tile and the last
    // stage's lanes store it.  When one of them holds one of the lowest tile
    // bits of a 128-byte line (3 for complex128, 4 for complex64) in
    // registers, a wave's access covers each line in pieces; an added stage
    // without gates (register bits = highest tile bits, plus the neighbour's
    // highest register bit for split exchanges) moves the HBM access to
    // whole-line lanes at the cost of one LDS exchange.  complex64 tiles that
    // hold the lowest state qubit keep it as a register bit in such a stage:
    // a lane then moves two neighbouring amplitudes as one 16-byte access and
    // 8 lanes cover a 128-byte line.
    const bool pair64 = amp_bytes == 8 && tile_pos[0] == 0;
    auto short_runs = [&](const Stage& st) {
        uint32_t regs = 0;
        for (int b : st.reg_bits) regs |= 1u << b;
        return (regs & ((1u << (amp_bytes == 16 ? 3 : 4)) - 1)) != 0;
    };
    auto make_io = [&](const Stage& nb) {
        Stage S;
        uint32_t regset = 0;
        int cnt = 0;
        if (pair64) { regset |= 1u; cnt++; }
        if (split_lds && !((regset >> nb.reg_bits.back()) & 1)) { regset |= 1u << nb.reg_bits.back(); cnt++; }
        for (int b = k - 1; b >= 0 && cnt < rb; b--)
            if (!((regset >> b) & 1)) { regset |= 1u << b; cnt++; }
        for (int b = 0; b < k; b++)
            if ((regset >> b) & 1) S.reg_bits.push_back(b);
        assign_lanes(S, regset);
        return S;
    };
    if ((io & 1) && !init && short_runs(stages.front())) stages.insert(stages.begin(), make_io(stages.front()));
    if ((io & 2) && short_runs(stages.back())) stages.push_back(make_io(stages.back()));

    // lower the stages' gates to ops, diagonal gates merged (StageLowering)
    std::vector<ShmStage> dst;
    const bool precise = precision == HQ_C64 && diag == DiagMode::PRECISE;
    StageLowering lo(low, low_type, precision, rb, tb, shared_code, precise, diag != DiagMode::APART);
    for (auto& S : stages) {
        ShmStage d;
        memset(&d, 0, sizeof(d));
        for (int i = 0; i < rb; i++) d.reg_bits[i] = S.reg_bits[i];
        for (int i = 0; i < tb; i++) d.thr_bits[i] = S.thr_bits[i];
        dst.push_back(d);
    }
    std::vector<ShmOp> ops;
    std::vector<double> tabs;
    for (size_t s = 0; s < dst.size(); s++) {
        dst[s].op_begin = (uint32_t)ops.size();
        lo.stage(dst[s], s + 1 < dst.size() ? &dst[s + 1] : nullptr, stages[s].ops, factored, &ops, &tabs);
        dst[s].op_end = (uint32_t)ops.size();
    }

    ShmHeader hdr;
    memset(&hdr, 0, sizeof(hdr));
    for (size_t j = 0; j < block_pos.size(); j++) hdr.block_phys[j] = 1ull << block_pos[j];
    for (int i = 0; i < k; i++) { hdr.tile_phys[i] = 1ull << tile_pos[i]; hdr.swz_col[i] = swz_column(i); }
    hdr.num_block_bits = (uint32_t)block_pos.size();
    hdr.num_stages = (uint32_t)dst.size();
    // lowered gates, plus the final scale when a gate was factored
    hdr.num_ops = (uint32_t)(low.size() + (factored ? 1 : 0));

    plan->n = n;
    plan->precision = precision;
    plan->k = k;
    plan->rb = rb;
    plan->tb = tb;
    plan->shared_mask = shared_mask;
    plan->hdr = hdr;
    plan->stages = std::move(dst);
    plan->ops = std::move(ops);
    plan->tabs = std::move(tabs);
    plan->precise = precise;
    return HQ_OK;
}

// ---- the interpreter's program ------------------------------------------------------------

namespace {

template <typename R, bool PRECISE>
struct Encoder {
    const ShmPlan& P;
    std::vector<char> slots;
    std::vector<Factor<R, PRECISE>> lanes;   // 2^tb entries per lane table
    static constexpr int SLOT = shm_slot_bytes<R>();
    static_assert(SHM_WINDOW_BYTES % SLOT == 0, "windows hold whole slots");

    size_t count() const { return slots.size() / SLOT; }

    // room for `need` consecutive slots before the window's last one, which
    // is kept for the refill
    void room(size_t need)
    {
        const size_t W = (size_t)shm_window_slots<R>();
        if (count() % W + need <= W - 1) return;
        ShmSlot none{};
        none.kind = SLOT_END;       // never reached: a refill comes first
        ShmSlot refill{};
        refill.kind = SLOT_REFILL;
        put(refill, nullptr, 0);
        while (count() % W) put(none, nullptr, 0);
    }
    void put(const ShmSlot& h, const void* payload, size_t bytes)
    {
        const size_t at = slots.size();
        slots.resize(at + SLOT, 0);
        memcpy(slots.data() + at, &h, sizeof(h));
        if (bytes) memcpy(slots.data() + at + sizeof(h), payload, bytes);
    }
    void op(const ShmSlot& h, const double* m, int nm)
    {
        R c[8] = {};
        // a matrix: real parts first (real updates read half of the slot)
        for (int i = 0; i < nm; i++) c[nm == 8 ? (i & 1) * 4 + i / 2 : i] = (R)m[i];
        room(1);
        put(h, c, sizeof(c));
    }
    static ShmSlot head(const ShmOp& o, int kind)
    {
        ShmSlot h{};
        h.kind = (uint8_t)kind;
        h.aux = o.tpos;
        h.creg = o.creg; h.cregv = o.cregv;
        h.cthr = o.cthr; h.cthrv = o.cthrv;
        h.cblk = o.cblk; h.cblkv = o.cblkv;
        return h;
    }

    ShmXchg xchg(const ShmStage& st) const
    {
        ShmXchg x{};
        auto swz = [&](uint32_t bit) { return (uint16_t)(bit < 3 ? 1u << bit : (1u << bit) ^ P.hdr.swz_col[bit]); };
        for (int i = 0; i < P.tb; i++) x.thr[i] = swz(st.thr_bits[i]);
        for (int i = 0; i < P.rb; i++) x.reg[i] = swz(st.reg_bits[i]);
        return x;
    }

    void stage(const ShmStage& st)
    {
        // the lane factor of the stage: what depends on the thread bits alone
        // (and the scale) as a table, loaded before the stage's ops
        const int NT = 1 << P.tb;
        bool table = false;
        std::vector<std::complex<double>> f;
        const ShmOp* mul = nullptr;
        for (uint32_t i = st.op_begin; i < st.op_end; i++) {
            const ShmOp& o = P.ops[i];
            if (o.cls == SHM_LANEMUL && !(o.flags & SHM_FLAG_NOLANE)) mul = &o;
            if (o.cls != SHM_LANE || o.cblk) continue;
            if (!table) { f.assign(NT, 1.0); table = true; }
            for (int t = 0; t < NT; t++)
                if ((t & o.cthr) == o.cthrv) f[t] *= std::complex<double>(o.m[0], o.m[1]);
        }
        if (table) {
            const std::complex<double> S(mul->m[0], mul->m[1]);
            ShmSlot h{};
            h.kind = SLOT_LANETAB;
            h.cblk = (uint32_t)(lanes.size() / NT);
            for (int t = 0; t < NT; t++) {
                const std::complex<double> v = f[t] * S;
                lanes.push_back(Factor<R, PRECISE>::of(v.real(), v.imag()));
            }
            op(h, nullptr, 0);
        }
        for (uint32_t i = st.op_begin; i < st.op_end; i++) {
            const ShmOp& o = P.ops[i];
            switch (o.cls) {
            case SHM_TAB: {
                // factors on the |1> half of one register bit
                const uint32_t d = o.jdep;
                if (!(d & (d - 1)) && !(o.jmask & 1) && !((o.jprod >> d) & 1)) {
                    ShmSlot h{};
                    h.kind = (uint8_t)(8 * __builtin_ctz(d) + DIRECT_PHASE);
                    op(h, &P.tabs[2 * (o.tab + d)], 2);
                    break;
                }
                const size_t bytes = ((size_t)1 << P.rb) * sizeof(Factor<R, PRECISE>);
                const size_t more = (bytes + SLOT - 1) / SLOT;
                std::vector<Factor<R, PRECISE>> t((size_t)1 << P.rb);
                for (size_t j = 0; j < t.size(); j++)
                    t[j] = Factor<R, PRECISE>::of(P.tabs[2 * (o.tab + j)], P.tabs[2 * (o.tab + j) + 1]);
                ShmSlot h{};
                h.kind = SLOT_TAB;
                h.aux = (uint8_t)more;
                room(1 + more);
                put(h, nullptr, 0);
                const size_t at = slots.size();
                slots.resize(at + more * SLOT, 0);
                memcpy(slots.data() + at, t.data(), bytes);
                break;
            }
            case SHM_MIX:
                // (a factor on no register bit is every amplitude's)
                if (!o.cblk && o.creg && o.creg == o.cregv && !(o.creg & (o.creg - 1)))
                    op(head(o, 8 * __builtin_ctz(o.creg) + DIRECT_LPHASE), o.m, 2);
                else
                    op(head(o, (o.flags & SHM_FLAG_REAL) && o.m[0] == -1.0 ? SLOT_MIXSIGN : SLOT_MIX), o.m, 2);
                break;
            case SHM_LANE:
                if (o.cblk) op(head(o, SLOT_LANE), o.m, 2);
                break;
            case SHM_LANEMUL:
                if (o.flags & SHM_FLAG_NOLANE) {
                    op(head(o, SLOT_SCALE), o.m, 2);
                } else {
                    if (!table && !(o.flags & SHM_FLAG_UNIT)) op(head(o, SLOT_LANE), o.m, 2);
                    op(head(o, SLOT_LANEMUL), nullptr, 0);
                }
                break;
            case SHM_SWAP:
                if (o.cthr && !o.creg && !o.cblk) op(head(o, 8 * o.tpos + DIRECT_LSWAP), nullptr, 0);
                else op(head(o, o.cthr ? (int)SLOT_CSWAP : SLOT_PAIR + SHM_SWAP), nullptr, 0);
                break;
            // the factored forms come from uncontrolled gates
            case SHM_HADD: op(head(o, 8 * o.tpos + DIRECT_HADD), nullptr, 0); break;
            case SHM_ROTA: op(head(o, 8 * o.tpos + DIRECT_ROTA), o.m, 1); break;
            case SHM_ROTB: op(head(o, 8 * o.tpos + DIRECT_ROTB), o.m, 1); break;
            case SHM_RXA: op(head(o, 8 * o.tpos + DIRECT_RXA), o.m, 1); break;
            case SHM_RXB: op(head(o, 8 * o.tpos + DIRECT_RXB), o.m, 1); break;
            default:
                op(head(o, SLOT_PAIR + o.cls), o.m, 8);
                break;
            }
        }
    }

    std::vector<char> run()
    {
        ShmProg H{};
        for (size_t s = 0; s < P.stages.size(); s++) {
            if (s > 0) {
                ShmSlot h{};
                h.kind = SLOT_XCHG;
                const ShmXchg x = xchg(P.stages[s]);
                room(1);
                put(h, &x, sizeof(x));
            }
            stage(P.stages[s]);
        }
        ShmSlot end{};
        end.kind = SLOT_END;
        room(1);
        put(end, nullptr, 0);
        // runs of consecutive block positions
        const uint32_t nb = P.hdr.num_block_bits;
        for (uint32_t j = 0; j < nb;) {
            const int p = __builtin_ctzll(P.hdr.block_phys[j]);
            uint32_t len = 1;
            while (j + len < nb && __builtin_ctzll(P.hdr.block_phys[j + len]) == p + (int)len) len++;
            H.run[H.num_runs++] = ShmRun{j, (uint32_t)p, (1ull << len) - 1};
            j += len;
        }
        H.num_slots = (uint32_t)count();
        H.zero_mask = P.hdr.zero_mask;
        auto pos = [&](uint32_t tile) { return (uint8_t)__builtin_ctzll(P.hdr.tile_phys[tile]); };
        const ShmStage &f = P.stages.front(), &l = P.stages.back();
        for (int i = 0; i < P.tb; i++) { H.ld_thr[i] = pos(f.thr_bits[i]); H.st_thr[i] = pos(l.thr_bits[i]); }
        for (int i = 0; i < P.rb; i++) { H.ld_reg[i] = pos(f.reg_bits[i]); H.st_reg[i] = pos(l.reg_bits[i]); }
        H.first = xchg(f);
        // the last window is copied whole
        const size_t tail = slots.size() - slots.size() % (size_t)SHM_WINDOW_BYTES + SHM_WINDOW_COPY;
        const size_t lane_off = (SHM_PROG_HEADER + tail + 255) & ~(size_t)255;
        H.lane_off = (uint32_t)lane_off;
        std::vector<char> out(lane_off + lanes.size() * sizeof(Factor<R, PRECISE>), 0);
        memcpy(out.data(), &H, sizeof(H));
        memcpy(out.data() + SHM_PROG_HEADER, slots.data(), slots.size());
        if (!lanes.empty()) memcpy(out.data() + lane_off, lanes.data(), lanes.size() * sizeof(Factor<R, PRECISE>));
        return out;
    }
};

}  // namespace

std::vector<char> encode_program(const ShmPlan& plan)
{
    if (plan.precision == HQ_C128) return Encoder<double, false>{plan, {}, {}}.run();
    if (plan.precise) return Encoder<float, true>{plan, {}, {}}.run();
    return Encoder<float, false>{plan, {}, {}}.run();
}

hq_status build_sharemem_program(hq_state s, const hq_gate* gates, int num_gates, uint64_t shared_mask, int rb_req,
                                 hq_program* out, bool init, int variant, uint64_t zero_mask, bool apart)
{
    HQ_CHECK(s && out, HQ_ERR_ARG, "sharemem: null argument");
    *out = nullptr;
    ShmPlan plan;
    const DiagMode diag = apart ? DiagMode::APART : DiagMode::PRECISE;
    // variant bit 0: whole-line stages; bit 1: non-temporal stores; bit 2:
    // non-temporal loads
    const bool whole_line = variant & 1;
    hq_status st = plan_sharemem(s->n, s->precision, gates, num_gates, shared_mask, rb_req, &plan, init,
                                 whole_line ? 3 : 0, false, diag);
    if (st != HQ_OK) return st;
    plan.init = init;
    plan.whole_line = whole_line;
    plan.nt_store = (variant & 2) != 0;
    plan.nt_load = (variant & 4) != 0;
    plan.hdr.zero_mask = init ? 0 : zero_mask;
    const std::vector<char> blob = encode_program(plan);
    const size_t bytes = blob.size();

    hq_program p = new hq_program_s();
    p->kind = 1;
    p->n = plan.n;
    p->precision = s->precision;
    p->tile = plan.k;
    p->rb = plan.rb;
    p->tb = plan.tb;
    p->num_stages = (int)plan.stages.size();
    p->num_ops = (int)plan.hdr.num_ops;
    p->shared_mask = shared_mask;
    p->prog_bytes = bytes;
    p->plan = new ShmPlan(std::move(plan));
    hipError_t e = hipMalloc(&p->d_prog, bytes);
    if (e != hipSuccess) {
        set_error(std::string("sharemem: hipMalloc: ") + hipGetErrorString(e));
        delete p->plan;
        delete p;
        return HQ_ERR_OOM;
    }
    e = hipMemcpy(p->d_prog, blob.data(), bytes, hipMemcpyHostToDevice);
    if (e != hipSuccess) {
        set_error(std::string("sharemem: hipMemcpy: ") + hipGetErrorString(e));
        (void)hipFree(p->d_prog);
        delete p->plan;
        delete p;
        return HQ_ERR_HIP;
    }
    *out = p;
    return HQ_OK;
}

}  // namespace hq
