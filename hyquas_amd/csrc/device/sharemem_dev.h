// sharemem_dev.h -- device body of the register-tiled OShareMem pass, shared by
// the single-state kernel (sharemem.hip) and the batched kernels (engine.hip).
//
// Reference behaviour (src/kernelOpt.cu:388-433): a block owns the 2^k
// amplitudes that differ only in the k tile ("shared") qubits, applies every
// gate of the group to them and writes them back.  Here the tile lives in
// registers (2^RB per thread, 2^TB threads); stages of gates on register bits
// are separated by one LDS exchange each.
#pragma once

#include "hq_ops.h"

namespace hq {

// Global-memory pointers.  The batched kernel reads its program and state
// pointers from an item table, which makes them generic (flat) pointers; the
// compiler takes every flat load for a per-lane value, so the op dispatch
// below would compile to divergent branches.  Casting to the global address
// space keeps the program's fields uniform (scalar loads, scalar branches).
// (The host pass of a HIP file sees the same templates: no address space there.)
#if defined(__HIP_DEVICE_COMPILE__)
#define HQ_GLOBAL __attribute__((address_space(1)))
#else
#define HQ_GLOBAL
#endif
template <typename T> __device__ __forceinline__ HQ_GLOBAL T* to_global(T* p) { return (HQ_GLOBAL T*)p; }

// tile_pass modes (bit set)
constexpr uint32_t TILE_INIT = 1;     // start from |0...0> instead of loading the tile
constexpr uint32_t TILE_NOSTORE = 2;  // do not write the tile back
constexpr uint32_t TILE_READ = 4;     // write {sum p, sum p*Z, sum p*ZZ} of the tile to part[3*blk]

template <typename R, int RB, int CLS, int P>
__device__ __forceinline__ void reg_pairs(cplx<R> (&a)[1 << RB], uint32_t creg, const R* m)
{
    // without register controls every pair is updated: no per-pair branch
    // (a branch per pair makes the compiler copy both amplitudes for the
    // path that skips the update)
    if (creg == 0) {
#pragma unroll
        for (int j = 0; j < (1 << RB); j++) {
            if (j & (1 << P)) continue;
            pair_update<CLS, R>(a[j], a[j | (1 << P)], m);
        }
        return;
    }
#pragma unroll
    for (int j = 0; j < (1 << RB); j++) {
        if (j & (1 << P)) continue;
        if ((j & creg) != creg) continue;
        pair_update<CLS, R>(a[j], a[j | (1 << P)], m);
    }
}

// X where the lane's thread-bit controls are set: selects, no arithmetic
template <typename R, int RB, int P>
__device__ __forceinline__ void lane_swap(cplx<R> (&a)[1 << RB], uint32_t creg, bool on)
{
#pragma unroll
    for (int j = 0; j < (1 << RB); j++) {
        if (j & (1 << P)) continue;
        if ((j & creg) != creg) continue;
        const cplx<R> lo = a[j], hi = a[j | (1 << P)];
        a[j].x = on ? hi.x : lo.x;
        a[j].y = on ? hi.y : lo.y;
        a[j | (1 << P)].x = on ? lo.x : hi.x;
        a[j | (1 << P)].y = on ? lo.y : hi.y;
    }
}

// SlotDirect updates of register bit P; `on`: the lane's thread-bit condition
template <typename R, int RB, int P>
__device__ __forceinline__ void direct_op(cplx<R> (&a)[1 << RB], int op, bool on, R c0, R c1)
{
    R m[8];
    m[0] = c0;
    m[6] = c0;
    m[7] = c1;
    switch (op) {
    case DIRECT_HADD: reg_pairs<R, RB, SHM_HADD, P>(a, 0, m); break;
    case DIRECT_ROTA: reg_pairs<R, RB, SHM_ROTA, P>(a, 0, m); break;
    case DIRECT_ROTB: reg_pairs<R, RB, SHM_ROTB, P>(a, 0, m); break;
    case DIRECT_RXA: reg_pairs<R, RB, SHM_RXA, P>(a, 0, m); break;
    case DIRECT_RXB: reg_pairs<R, RB, SHM_RXB, P>(a, 0, m); break;
    case DIRECT_PHASE: reg_pairs<R, RB, SHM_PHASE, P>(a, 0, m); break;
    case DIRECT_LPHASE:
        m[6] = on ? c0 : R(1);
        m[7] = on ? c1 : R(0);
        reg_pairs<R, RB, SHM_PHASE, P>(a, 0, m);
        break;
    default: lane_swap<R, RB, P>(a, 0, on); break;
    }
}

// the other pair updates; coef: the matrix's real parts, then its imaginary
// ones, in LDS; lane: some thread-bit control, `on` where it holds
template <typename R, int RB, int P>
__device__ __forceinline__ void reg_op(cplx<R> (&a)[1 << RB], int kind, uint32_t creg, bool lane, bool on,
                                       const R* coef)
{
    R m[8];
    auto matrix = [&](bool imag) {
#pragma unroll
        for (int i = 0; i < 4; i++) { m[2 * i] = coef[i]; m[2 * i + 1] = imag ? coef[4 + i] : R(0); }
        if (lane) {
#pragma unroll
            for (int i = 0; i < 8; i++)
                if (imag || !(i & 1)) m[i] = on ? m[i] : (i == 0 || i == 6) ? R(1) : R(0);
        }
    };
    switch (kind) {
    case SLOT_PAIR + SHM_SWAP: reg_pairs<R, RB, SHM_SWAP, P>(a, creg, m); break;
    case SLOT_PAIR + SHM_Y: reg_pairs<R, RB, SHM_Y, P>(a, creg, m); break;
    case SLOT_PAIR + SHM_REAL: matrix(false); reg_pairs<R, RB, SHM_REAL, P>(a, creg, m); break;
    case SLOT_PAIR + SHM_RX: matrix(true); reg_pairs<R, RB, SHM_RX, P>(a, creg, m); break;
    case SLOT_PAIR + SHM_GEN: matrix(true); reg_pairs<R, RB, SHM_GEN, P>(a, creg, m); break;
    default: lane_swap<R, RB, P>(a, creg, on); break;
    }
}

__device__ __forceinline__ uint32_t uniform(uint32_t x) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)x); }

// Z-sum and nearest-neighbour ZZ-sum eigenvalues of basis state idx over n qubits:
// sum_q (1 - 2 b_q) and sum_{q<n-1} (1 - 2 (b_q xor b_{q+1})).
__device__ __forceinline__ void zsums(uint64_t idx, int n, double* z, double* zz)
{
    // __popcll returns unsigned: keep the arithmetic signed
    *z = (double)(n - 2 * (int)__popcll(idx));
    const uint64_t m = n >= 2 ? ((1ull << (n - 1)) - 1) : 0;
    *zz = (double)((n - 1) - 2 * (int)__popcll((idx ^ (idx >> 1)) & m));
}

// One OShareMem pass of tile `blk` of the group program `prog` over `psi`.
// `mode` is uniform over the grid; the single-state kernel passes 0.
//
// The program is a list of slots executed in order.  A pass over a small state
// is a chain of ops run by one wave per SIMD, so what an op costs is its fetch
// and dispatch: read from HBM through the scalar cache, each op's fields were
// three dependent misses.  Slots are copied to
// LDS a window at a time, together with the tile's loads, and the next slot is
// read while one executes.  With diagonal gates merged, uniform branches, one
// switch for the frequent updates and 8 amplitudes a thread on top, passes of
// the 17-qubit complex64 and 20-qubit complex128 random circuits (32 and 256
// blocks) went from 61 and 67.5 us to 24 and 31 us, the 174 gates of a
// 10-qubit ansatz from 132 to 34.5 us.
template <typename R, int RB, int TB, bool PRECISE>
__device__ __forceinline__ void tile_pass(cplx<R>* __restrict__ psi_any, const char* __restrict__ prog_any,
                                          uint64_t blk, cplx<R>* __restrict__ lds, char* __restrict__ win,
                                          uint32_t mode, int n, double* __restrict__ part_any)
{
    HQ_GLOBAL cplx<R>* __restrict__ psi = to_global(psi_any);
    const HQ_GLOBAL char* __restrict__ prog = to_global(prog_any);
    HQ_GLOBAL double* __restrict__ part = to_global(part_any);
    constexpr int NR = 1 << RB;
    constexpr int NT = 1 << TB;
    constexpr int SLOT = shm_slot_bytes<R>();

    const HQ_GLOBAL ShmProg* __restrict__ H = (const HQ_GLOBAL ShmProg*)prog;
    const uint32_t tid = threadIdx.x;

    // block base address: the block index scattered to the block bits
    // (the first runs without a branch, so that their loads go out together;
    // unused runs have an empty mask)
    uint64_t base = 0;
#pragma unroll
    for (uint32_t j = 0; j < 4; j++) base |= ((blk >> H->run[j].src) & H->run[j].mask) << H->run[j].dst;
    const uint32_t nruns = H->num_runs;
    for (uint32_t j = 4; j < nruns; j++) base |= ((blk >> H->run[j].src) & H->run[j].mask) << H->run[j].dst;
    // a tile known to be zero stays zero (uniform over the block)
    if (!(mode & TILE_READ) && (base & H->zero_mask)) return;

    // a window of slots, global -> registers -> LDS, in pieces of 16 bytes a
    // thread (every window is readable to SHM_WINDOW_COPY bytes).  No branch
    // here or in the loop below depends on the lane: one that did would make
    // the compiler rebuild the whole loop with copies of every amplitude at
    // its joins (17 qubits complex64: 12 200 VALU instructions per wave and
    // pass instead of 6 200).
    const uint32_t nbytes = H->num_slots * SLOT;
    constexpr int WIN_BYTES = shm_window_slots<R>() * SLOT;
    constexpr int PIECES = SHM_WINDOW_COPY / (16 * NT);
    const HQ_GLOBAL char* __restrict__ slots = prog + SHM_PROG_HEADER;
    // (a native vector: uint4's copies of unread pieces went to scratch memory in half of the shapes)
    typedef uint32_t Piece __attribute__((ext_vector_type(4)));
    Piece piece[PIECES];
    auto fetch = [&](uint32_t from) {
#pragma unroll
        for (int i = 0; i < PIECES; i++)
            if (i == 0 || from + (uint32_t)(i * NT) * 16u < nbytes)
                piece[i] = *(const HQ_GLOBAL Piece*)(slots + from + (uint32_t)(i * NT + tid) * 16u);
    };
    auto fill = [&]() {
#pragma unroll
        for (int i = 0; i < PIECES; i++) *(Piece*)(win + (uint32_t)(i * NT + tid) * 16u) = piece[i];
    };

    cplx<R> a[NR];
    uint64_t rphys[RB];
    if (mode == TILE_INIT && base != 0) {
        // first pass of a run: a tile other than the origin's starts at zero
        // and stays zero under the group's linear gates
        uint64_t pt = 0;
#pragma unroll
        for (int i = 0; i < TB; i++) pt |= (uint64_t)((tid >> i) & 1u) << H->st_thr[i];
#pragma unroll
        for (int i = 0; i < RB; i++) rphys[i] = (uint64_t)1 << H->st_reg[i];
        HQ_GLOBAL cplx<R>* __restrict__ dst = psi + (base | pt);
        cplx<R> z;
        z.x = R(0);
        z.y = R(0);
#pragma unroll
        for (int j = 0; j < NR; j++) {
            uint64_t off = 0;
#pragma unroll
            for (int i = 0; i < RB; i++) if ((j >> i) & 1) off |= rphys[i];
            dst[off] = z;
        }
        return;
    }
    // issued before the tile's loads, so that it can be stored while they are in flight
    fetch(0);
    {
        uint64_t pt = 0;
#pragma unroll
        for (int i = 0; i < TB; i++) pt |= (uint64_t)((tid >> i) & 1u) << H->ld_thr[i];
        if (mode & TILE_INIT) {
            const bool origin = (base | pt) == 0;
#pragma unroll
            for (int j = 0; j < NR; j++) {
                a[j].x = (origin && j == 0) ? R(1) : R(0);
                a[j].y = R(0);
            }
        } else {
#pragma unroll
            for (int i = 0; i < RB; i++) rphys[i] = (uint64_t)1 << H->ld_reg[i];
            const HQ_GLOBAL cplx<R>* __restrict__ src = psi + (base | pt);
#pragma unroll
            for (int j = 0; j < NR; j++) {
                uint64_t off = 0;
#pragma unroll
                for (int i = 0; i < RB; i++) if ((j >> i) & 1) off |= rphys[i];
                a[j] = src[off];
            }
        }
    }
    fill();
    // LDS addresses (bytes) of the current stage
    uint32_t at, reg_at[RB];
    {
        uint32_t r = 0;
#pragma unroll
        for (int i = 0; i < TB; i++) r ^= (0u - ((tid >> i) & 1u)) & (uint32_t)H->first.thr[i];
        at = r * (uint32_t)sizeof(cplx<R>);
#pragma unroll
        for (int i = 0; i < RB; i++) reg_at[i] = H->first.reg[i] * (uint32_t)sizeof(cplx<R>);
    }
    __syncthreads();

    double lx = 1, ly = 0;    // the lane's factor
    uint32_t window = 0;      // bytes of the current window's start in the program
    const char* pc = win;
    // fields and first two coefficients of the next slot: all that most ops
    // have (the rest is read when it is used)
    uint4 next = *(const uint4*)pc;
    R next0 = ((const R*)(pc + 16))[0], next1 = ((const R*)(pc + 16))[1];
    auto read_next = [&]() {
        next = *(const uint4*)pc;     // (behind the last slot of a window: unused)
        next0 = ((const R*)(pc + 16))[0];
        next1 = ((const R*)(pc + 16))[1];
    };
    char* const xlds = (char*)lds;
    for (;;) {
        const uint32_t w0 = uniform(next.x), w1 = uniform(next.y);
        const uint32_t cb = uniform(next.z), cbv = uniform(next.w);
        const R* const coef = (const R*)(pc + 16);
        const R c0 = next0, c1 = next1;
        pc += SLOT;
        read_next();
        const int kind = (int)(w0 & 255u), aux = (int)((w0 >> 8) & 255u);
        const uint32_t creg = (w0 >> 16) & 255u, cregv = w0 >> 24;
        const uint32_t cthr = w1 & 0xffffu, cthrv = w1 >> 16;
        const bool on = (tid & cthr) == cthrv;
        // Every branch below is uniform over the block: a lane whose
        // thread-bit condition does not hold gets the identity's coefficients
        // or keeps its values by selects instead of leaving the op.
        if (kind < SLOT_DIRECT_END) {
            switch (kind) {
#define HQ_DIRECT(PV)                                                                          \
    case 8 * PV + 0: case 8 * PV + 1: case 8 * PV + 2: case 8 * PV + 3: case 8 * PV + 4:        \
    case 8 * PV + 5: case 8 * PV + 6: case 8 * PV + 7:                                          \
        if constexpr (RB > PV) direct_op<R, RB, PV>(a, kind & 7, on, c0, c1);                   \
        break;
                HQ_DIRECT(0) HQ_DIRECT(1) HQ_DIRECT(2) HQ_DIRECT(3) HQ_DIRECT(4)
            default:
                if constexpr (RB > 5) direct_op<R, RB, 5>(a, kind & 7, on, c0, c1);
                break;
#undef HQ_DIRECT
            }
            static_assert(RB <= 6, "register positions above 5 are not dispatched");
            continue;
        }
        if (kind <= SLOT_CSWAP) {
            if (((uint32_t)blk & cb) != cbv) continue;
            const bool lane = cthr != 0;
            switch (aux) {
            case 0: reg_op<R, RB, 0>(a, kind, creg, lane, on, coef); break;
            case 1: if constexpr (RB > 1) reg_op<R, RB, 1>(a, kind, creg, lane, on, coef); break;
            case 2: if constexpr (RB > 2) reg_op<R, RB, 2>(a, kind, creg, lane, on, coef); break;
            case 3: if constexpr (RB > 3) reg_op<R, RB, 3>(a, kind, creg, lane, on, coef); break;
            case 4: if constexpr (RB > 4) reg_op<R, RB, 4>(a, kind, creg, lane, on, coef); break;
            default: if constexpr (RB > 5) reg_op<R, RB, 5>(a, kind, creg, lane, on, coef); break;
            }
            static_assert(RB <= 6, "register positions above 5 are not dispatched");
            continue;
        }
        if (kind == SLOT_XCHG) {
            // write under the old split, read under the new one; a register's
            // LDS address is the lane's xor its register bits' entries (all
            // kept in bytes: one xor per access)
#pragma unroll
            for (int j = 0; j < NR; j++) {
                uint32_t so = 0;
#pragma unroll
                for (int i = 0; i < RB; i++) if ((j >> i) & 1) so ^= reg_at[i];
                *(cplx<R>*)(xlds + (at ^ so)) = a[j];
            }
            const ShmXchg* const x = (const ShmXchg*)coef;
            uint32_t e[(SHM_MAX_TB + SHM_MAX_RB + 1) / 2];   // two 16-bit entries each
#pragma unroll
            for (int i = 0; i < (int)(sizeof(e) / 4); i++) e[i] = ((const uint32_t*)x)[i];
            auto entry = [&](int i) { return (i & 1) ? e[i / 2] >> 16 : e[i / 2] & 0xffffu; };
            at = 0;
#pragma unroll
            for (int i = 0; i < TB; i++) at ^= (0u - ((tid >> i) & 1u)) & entry(i);
            at *= (uint32_t)sizeof(cplx<R>);
#pragma unroll
            for (int i = 0; i < RB; i++) reg_at[i] = uniform(entry(SHM_MAX_TB + i)) * (uint32_t)sizeof(cplx<R>);
            __syncthreads();
#pragma unroll
            for (int j = 0; j < NR; j++) {
                uint32_t so = 0;
#pragma unroll
                for (int i = 0; i < RB; i++) if ((j >> i) & 1) so ^= reg_at[i];
                a[j] = *(const cplx<R>*)(xlds + (at ^ so));
            }
            // the next exchange overwrites lds: every lane must have read first
            __syncthreads();
            continue;
        }
        if (kind == SLOT_TAB) {
            const Factor<R, PRECISE>* __restrict__ tab = (const Factor<R, PRECISE>*)pc;
#pragma unroll
            for (int j = 0; j < NR; j++) scale(a[j], tab[j]);
            pc += aux * SLOT;
            read_next();
            continue;
        }
        if (kind == SLOT_SCALE) {
#pragma unroll
            for (int j = 0; j < NR; j++) scale(a[j], c0, c1);
            continue;
        }
        if (kind == SLOT_LANEMUL) {
            const Factor<R, PRECISE> f = Factor<R, PRECISE>::of(lx, ly);
#pragma unroll
            for (int j = 0; j < NR; j++) scale(a[j], f);
            lx = 1;
            ly = 0;
            continue;
        }
        if (kind == SLOT_LANETAB) {
            const HQ_GLOBAL Factor<R, PRECISE>* __restrict__ t =
                (const HQ_GLOBAL Factor<R, PRECISE>*)(prog + H->lane_off) + (size_t)cb * NT;
            const Factor<R, PRECISE> f = t[tid];
            lx = f.x;
            ly = f.y;
            if constexpr (PRECISE) { lx += f.lx; ly += f.ly; }
            continue;
        }
        if (kind == SLOT_REFILL) {
            window += (uint32_t)WIN_BYTES;
            __syncthreads();   // every lane has read this window's last slot
            fetch(window);
            fill();
            __syncthreads();
            pc = win;
            read_next();
            continue;
        }
        if (kind == SLOT_END) break;
        if (((uint32_t)blk & cb) != cbv) continue;
        if (kind == SLOT_LANE) {
            const double fr = on ? (double)c0 : 1.0, fi = on ? (double)c1 : 0.0;
            const double x = lx, y = ly;
            lx = fr * x - fi * y;
            ly = fr * y + fi * x;
        } else if (kind == SLOT_MIXSIGN) {
            const R f = on ? R(-1) : R(1);
#pragma unroll
            for (int j = 0; j < NR; j++)
                if ((j & creg) == cregv) { a[j].x *= f; a[j].y *= f; }
        } else {   // SLOT_MIX
            const R fr = on ? c0 : R(1), fi = on ? c1 : R(0);
#pragma unroll
            for (int j = 0; j < NR; j++)
                if ((j & creg) == cregv) scale(a[j], fr, fi);
        }
    }

    // mapping of the last stage
    uint64_t pt = 0;
#pragma unroll
    for (int i = 0; i < TB; i++) pt |= (uint64_t)((tid >> i) & 1u) << H->st_thr[i];
#pragma unroll
    for (int i = 0; i < RB; i++) rphys[i] = (uint64_t)1 << H->st_reg[i];

    if (mode & TILE_READ) {
        double s0 = 0, s1 = 0, s2 = 0;
#pragma unroll
        for (int j = 0; j < NR; j++) {
            uint64_t off = 0;
#pragma unroll
            for (int i = 0; i < RB; i++) if ((j >> i) & 1) off |= rphys[i];
            const double re = (double)a[j].x, im = (double)a[j].y;
            const double p = re * re + im * im;
            double z, zz;
            zsums(base | pt | off, n, &z, &zz);
            s0 += p;
            s1 += p * z;
            s2 += p * zz;
        }
        // fixed-order block reduction: xor butterfly in the wave, then waves in order
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) {
            s0 += __shfl_xor(s0, o);
            s1 += __shfl_xor(s1, o);
            s2 += __shfl_xor(s2, o);
        }
        __shared__ double red[3][(1 << SHM_MAX_TB) / 64];
        const uint32_t w = tid >> 6;
        if ((tid & 63) == 0) { red[0][w] = s0; red[1][w] = s1; red[2][w] = s2; }
        __syncthreads();
        if (tid == 0) {
            double t0 = 0, t1 = 0, t2 = 0;
            for (uint32_t i = 0; i < ((1u << TB) >> 6); i++) { t0 += red[0][i]; t1 += red[1][i]; t2 += red[2][i]; }
            part[3 * blk + 0] = t0;
            part[3 * blk + 1] = t1;
            part[3 * blk + 2] = t2;
        }
    }

    if (!(mode & TILE_NOSTORE)) {
        HQ_GLOBAL cplx<R>* __restrict__ dst = psi + (base | pt);
#pragma unroll
        for (int j = 0; j < NR; j++) {
            uint64_t off = 0;
#pragma unroll
            for (int i = 0; i < RB; i++) if ((j >> i) & 1) off |= rphys[i];
            dst[off] = a[j];
        }
    }
}

}  // namespace hq
