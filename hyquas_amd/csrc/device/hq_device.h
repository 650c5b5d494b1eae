// hq_device.h -- internal types of the HIP device layer (not part of the ABI).
#pragma once

#include <hip/hip_runtime.h>
#include <cstdint>
#include <mutex>
#include <string>
#include <vector>

#include "hyquas_amd.h"
#include "hq_internal.h"

namespace hq {

// ---- errors ------------------------------------------------------------------
void set_error(const std::string& msg);
const char* get_error();

#define HQ_HIP(call)                                                               \
    do {                                                                           \
        hipError_t e_ = (call);                                                    \
        if (e_ != hipSuccess) {                                                    \
            ::hq::set_error(std::string(#call) + ": " + hipGetErrorString(e_));    \
            return HQ_ERR_HIP;                                                     \
        }                                                                          \
    } while (0)

#define HQ_CHECK(cond, code, msg)                                                  \
    do {                                                                           \
        if (!(cond)) { ::hq::set_error(msg); return (code); }                      \
    } while (0)

// ---- complex amplitude -----------------------------------------------------------
template <typename R>
struct alignas(2 * sizeof(R)) cplx {
    R x, y;
};

// ---- state -------------------------------------------------------------------------
struct ProfileEntry {
    int kind;
    hipEvent_t start, stop;
};

}  // namespace hq

struct hq_state_s {
    int n = 0;
    int precision = HQ_C128;
    int device = 0;
    uint64_t amps = 0;
    size_t amp_bytes = 16;
    void* data = nullptr;     // current state vector
    void* buf = nullptr;      // work buffer (TransMM), may be null
    hipStream_t stream = nullptr;
    double* d_red = nullptr;  // reduction scratch (device)
    double* h_red = nullptr;  // reduction scratch (pinned host)
    size_t red_cap = 0;       // doubles
    char* d_ws = nullptr;     // readout workspace (device, pinned host), see ensure_ws
    char* h_ws = nullptr;
    size_t ws_dev = 0, ws_host = 0;   // bytes
    std::mutex ws_mu;         // held by a readout from its use of d_red, h_red or the workspace until it has its results
    bool profiling = false;
    std::vector<hq::ProfileEntry> prof;
    std::vector<hipEvent_t> free_events;
};

namespace hq {

// Profiling helpers: bracket one launch with events when enabled.
hq_status prof_begin(hq_state s, int kind, int* slot);
hq_status prof_end(hq_state s, int slot);

// Room for a readout in the state's workspace (grown on demand, freed with
// the state); contents do not outlive a call, which holds ws_mu.
hq_status ensure_ws(hq_state s, size_t dev, size_t host);
// Gives back workspace beyond `keep` bytes (no work of the state may use it).
void trim_ws(hq_state s, size_t keep);

// ---- OShareMem program (device-resident) ---------------------------------------------
// Op classes of the register kernel.
enum ShmClass : uint8_t {
    SHM_SWAP = 0,   // lo <-> hi                       (X, CNOT, CCX)
    SHM_Y = 1,      // lo' = -i hi, hi' = i lo         (Y, CY)
    SHM_REAL = 2,   // real 2x2                        (H, RY, CRY, ...)
    SHM_RX = 3,     // real diagonal, imaginary off-diagonal (RX, CRX)
    SHM_GEN = 4,    // complex 2x2                     (U2, U3, ...)
    SHM_DIAG = 5,   // lo *= d0, hi *= d1              (RZ, CRZ, ...)
    SHM_PHASE = 6,  // hi *= d1                        (T, S, Z, U1, CZ, CU1, ...)
    // uncontrolled gates with a scalar factored out (the group's product of
    // factors is applied by a later SHM_LANEMUL op); t, u = m[0]
    SHM_HADD = 7,   // lo' = lo + hi, hi' = lo - hi               (H / r)
    SHM_ROTA = 8,   // lo' = lo - t hi, hi' = t lo + hi           (RY / cos)
    SHM_ROTB = 9,   // lo' = u lo - hi, hi' = lo + u hi           (RY / sin)
    SHM_RXA = 10,   // lo' = lo + i t hi, hi' = i t lo + hi       (RX / cos)
    SHM_RXB = 11,   // lo' = u lo + i hi, hi' = i lo + u hi       (RX / sin)
    // rotations in specialised kernels shared by same-structure groups (one
    // form for every angle; the scalar factor goes to SHM_LANEMUL): three
    // shears, a = m[0], b = m[2], |a|, |b| <= 1
    SHM_SHEAR = 13,  // lo += a hi, hi += b lo, lo += a hi        (RY)
    SHM_SHEARX = 14, // lo += i a hi, hi -= i b lo, lo += i a hi  (RX)
    // diagonal factors of a stage, merged by the planner (SHM_DIAG and
    // SHM_PHASE are gate classes only: no op of a plan carries them)
    SHM_TAB = 15,    // amplitude of register index j *= table[j]
    SHM_MIX = 16,    // (m[0], m[1]) where register, thread and block bits match
    SHM_LANE = 17,   // the lane's factor *= (m[0], m[1]) where thread and block bits match
    SHM_LANEMUL = 18 // every amplitude *= the lane's factor * (m[0], m[1]); the factor is 1 again
};

// One op of a stage.  A condition is a mask and the value the masked bits
// must have; pair updates (SHM_SWAP..SHM_RXB and the shears, target register
// bit tpos) take all-ones values: their controls.
struct ShmOp {
    uint8_t cls = 0;
    uint8_t tpos = 0;        // pair updates: register-index bit of the target
    uint8_t creg = 0, cregv = 0;     // over register-index bits
    uint16_t cthr = 0, cthrv = 0;    // over thread-index bits
    uint32_t cblk = 0, cblkv = 0;    // over block-index bits (at most 29)
    uint32_t flags = 0;      // SHM_FLAG_*
    uint32_t tab = 0;        // SHM_TAB: first entry in ShmPlan::tabs (2^rb entries)
    uint64_t jmask = 0;      // SHM_TAB: register indices whose entry is not 1 by structure
    uint64_t jprod = 0;      // SHM_TAB, precise plans: entries that are products of several gates' factors
    uint32_t jdep = 0;       // SHM_TAB: register-index bits the table depends on
    double m[8] = {0, 0, 0, 0, 0, 0, 0, 0};   // re/im interleaved, row-major 2x2
};

// the op's coefficients are fixed by its gate type (H, T, CNOT, ...), so a
// specialised kernel may embed them as constants
constexpr uint32_t SHM_FLAG_CONST = 1;
// SHM_MIX, SHM_LANE, SHM_LANEMUL: the factor is real by structure (Z, CZ signs)
constexpr uint32_t SHM_FLAG_REAL = 2;
// SHM_LANEMUL: (m[0], m[1]) is exactly 1 by structure
constexpr uint32_t SHM_FLAG_UNIT = 4;
// SHM_LANEMUL: no SHM_LANE op before it (the lane's factor is 1)
constexpr uint32_t SHM_FLAG_NOLANE = 8;

constexpr int SHM_MAX_TILE = 14;
constexpr int SHM_MAX_TB = 9;
constexpr int SHM_MAX_RB = 6;   // 6 only for complex64 (64 amplitudes = 128 VGPRs per thread)

struct ShmStage {
    uint32_t reg_bits[SHM_MAX_RB];  // tile bit of register-index bit i (RB used)
    uint32_t thr_bits[SHM_MAX_TB];  // tile bit of thread-index bit i (TB used)
    uint32_t op_begin, op_end;
};

struct ShmHeader {
    uint64_t block_phys[64];   // physical bit (as a mask) of block-index bit j
    uint64_t tile_phys[SHM_MAX_TILE];  // physical bit (as a mask) of tile bit i
    uint32_t swz_col[SHM_MAX_TILE];    // LDS swizzle column of tile bit i
    uint32_t num_block_bits;
    uint32_t num_stages;
    uint32_t num_ops;          // lowered gates and the final scale (before diagonal factors are merged)
    uint32_t pad;
    // tiles whose block address has a bit in zero_mask hold only zeros before
    // the pass (the run started from |0...0> and no earlier group reached
    // those qubits) and keep them: the pass skips them
    uint64_t zero_mask;
};

// ---- the interpreter's program: header, op slots, lane tables ---------------------------
// A slot is 16 bytes of decoded fields and eight coefficients in the state's
// precision; the coefficients of a pair update are its 2x2 matrix's real parts,
// then the imaginary ones.  The kernel copies slots to LDS a window at a time (one memory
// latency per window instead of several per op) and reads the next slot while
// it executes one.
struct ShmSlot {
    uint8_t kind, aux;           // SlotKind; target register bit, or table slots that follow
    uint8_t creg, cregv;
    uint16_t cthr, cthrv;
    uint32_t cblk, cblkv;
};
static_assert(sizeof(ShmSlot) == 16, "ShmSlot layout");

// Kinds below SLOT_DIRECT_END are 8 P + SlotDirect for register bit P: the
// frequent updates, without register or block conditions, reached by one
// switch.  A dispatch step is a compare and a branch, some 40 cycles of a lone
// wave; the general path takes twice as many of them.
enum SlotDirect : uint8_t {
    DIRECT_HADD, DIRECT_ROTA, DIRECT_ROTB, DIRECT_RXA, DIRECT_RXB,
    DIRECT_PHASE,        // |1> half *= (m[0], m[1])
    DIRECT_LPHASE,       // the same where the thread-bit condition holds
    DIRECT_LSWAP,        // X where it holds
};
enum SlotKind : uint8_t {
    SLOT_DIRECT_END = 48,
    SLOT_PAIR = 64,      // + ShmClass (SHM_SWAP..SHM_GEN): pair update under any controls, target bit aux
    SLOT_CSWAP = 95,     // SHM_SWAP under a thread-bit control and others
    SLOT_SCALE,          // every amplitude *= (m[0], m[1])
    SLOT_TAB,            // complex table of the 2^RB register indices in the next `aux` slots
    SLOT_MIX,
    SLOT_MIXSIGN,        // factor -1
    SLOT_LANE,
    SLOT_LANETAB,        // the lane's factor = thread's entry of the lane table cblk (of this program)
    SLOT_LANEMUL,        // every amplitude *= the lane's factor
    SLOT_XCHG,           // LDS exchange into the next stage's split
    SLOT_REFILL,         // copy the next window of slots to LDS
    SLOT_END,
};

constexpr int SHM_WINDOW_BYTES = 7680;   // 96 slots of complex128, 160 of complex64
template <typename R> constexpr int shm_slot_bytes() { return 16 + 8 * (int)sizeof(R); }
template <typename R> constexpr int shm_window_slots() { return SHM_WINDOW_BYTES / shm_slot_bytes<R>(); }
constexpr int SHM_WINDOW_COPY = 8192;    // copied at a time, in whole 16-byte pieces of 64 to 512 threads
constexpr int SHM_WINDOW_LDS = SHM_WINDOW_COPY;
static_assert(SHM_WINDOW_COPY >= SHM_WINDOW_BYTES + 80, "the slot behind a window's last one is read ahead");

// exchange slots: swizzled LDS index of each thread and register bit of the
// stage they lead to
struct ShmXchg {
    uint16_t thr[SHM_MAX_TB];
    uint16_t reg[SHM_MAX_RB];
};
static_assert(sizeof(ShmXchg) <= 32, "an exchange fits the coefficients of a complex64 slot");

struct ShmRun {                // base |= ((block >> src) & mask) << dst
    uint32_t src, dst;
    uint64_t mask;
};

struct ShmProg {
    uint32_t num_runs, num_slots;
    uint32_t lane_off;         // lane tables, bytes from the program's start
    uint32_t pad;
    uint64_t zero_mask;
    uint8_t ld_thr[SHM_MAX_TB + 1], ld_reg[SHM_MAX_RB];   // physical position of each bit, first stage
    uint8_t st_thr[SHM_MAX_TB + 1], st_reg[SHM_MAX_RB];   // last stage
    ShmXchg first;             // the first stage's LDS indices
    uint16_t pad2;
    ShmRun run[SHM_MAX_TILE + 1];   // block bits in runs of consecutive positions
};
constexpr size_t SHM_PROG_HEADER = 512;
static_assert(sizeof(ShmProg) <= SHM_PROG_HEADER, "ShmProg header size");

// Host-side result of lowering + register-stage planning of one group.
struct ShmPlan {
    int n = 0, precision = 0, k = 0, rb = 0, tb = 0;
    bool init = false;        // start from |0...0> instead of loading (first group of a run)
    bool nt_load = false;     // specialised kernel: non-temporal HBM loads
    bool nt_store = false;    // specialised kernel: non-temporal HBM stores
    // complex64: a merged diagonal factor is held and applied as a sum of two
    // floats.  Rounded to one float, the moduli of its entries are each off by
    // up to 2^-24 in a pattern over the index bits, the same in every tile, and
    // <Z_q> of a large state (of order 2^(-n/2)) reads that pattern: at 31
    // qubits it moved <Z> by 4e-4 of its size.  Gate by gate the rounded
    // products average out over the amplitudes.
    bool precise = false;
    bool whole_line = false;  // planned with the whole-line HBM stages (io = 3)
    uint64_t shared_mask = 0;
    ShmHeader hdr;
    std::vector<ShmStage> stages;
    std::vector<ShmOp> ops;
    std::vector<double> tabs;  // SHM_TAB entries, re/im interleaved
};

}  // namespace hq

struct hq_program_s {
    int kind = 0;            // 1 sharemem, 2 blas (transpose + GEMM), 3 dense in place
    int n = 0;
    int precision = HQ_C128;
    // sharemem
    void* d_prog = nullptr;
    size_t prog_bytes = 0;
    int tile = 0, rb = 0, tb = 0, num_stages = 0, num_ops = 0;
    uint64_t shared_mask = 0;
    // blas
    bool identity_perm = true;
    std::vector<int> perm;
    void* d_targs = nullptr; // transpose launch arguments (device)
    void* d_mat = nullptr;   // K x K, column-major, split planes re | im, in state precision
    int mat_qubits = 0;
    uint64_t rows_mask = 0;  // dense in place: the qubits U acts on (row bit j = j-th lowest)
    // specialised (JIT) OShareMem kernel; null when the interpreter runs the group
    hipModule_t jit_module = nullptr;
    hipFunction_t jit_fn = nullptr;
    void* d_coef = nullptr;  // runtime coefficients of the specialised kernel
    hq::ShmPlan* plan = nullptr;  // kept for specialisation (owned)
};

namespace hq {
// How a plan applies diagonal gates: gate by gate; merged across the stage; or
// merged with complex64 factors kept as two floats (ShmPlan::precise).
enum class DiagMode { APART, MERGED, PRECISE };

// Launchers implemented in the .hip files.
hq_status launch_sharemem(hq_state s, hq_program p);
hq_status transpose_prepare(hq_state s, const int* perm, void** dev_args);
hq_status transpose_launch(hq_state s, const void* dev_args, void* in, void* out);
hq_status launch_dense(hq_state s, const void* d_mat, int mat_qubits, void* in, void* out);
// U (rows in the order of the set bits of `rows`) on those qubits, in place.
hq_status launch_dense_at(hq_state s, const void* d_mat, int mat_qubits, uint64_t rows);
int sharemem_default_rb(int precision, int tile);
// Register qubits of the interpreter's kernel on one n-qubit state.
int interpreter_rb(int precision, int tile, int n);
// io: bit 0 adds a leading, bit 1 a trailing stage without gates where the
// first / last stage holds one of the three lowest tile bits in registers
// (the HBM access then covers whole 128-byte lines per wave instruction).
// shared_code: op classes that do not depend on gate angles (rotations keep
// their full 2x2 form), so same-structure groups share a specialised kernel.
hq_status plan_sharemem(int n, int precision, const hq_gate* gates, int num_gates, uint64_t shared_mask,
                        int rb, ShmPlan* out, bool init = false, int io = 0, bool shared_code = false,
                        DiagMode diag = DiagMode::PRECISE);
// The interpreter's program of a plan (ShmProg header, slots, lane tables).
std::vector<char> encode_program(const ShmPlan& plan);
// Specialised kernel for a planned group: generate, compile (cached), load.
hq_status jit_sharemem(const ShmPlan& plan, hq_program p);
hq_status launch_sharemem_jit(hq_state s, hq_program p);
hq_status jit_sharemem_many(const std::vector<const ShmPlan*>& plans, const std::vector<hq_program>& progs,
                            int threads);
// batch: the batched form hq_group_batch(const BatchItem* items, unsigned count)
// (blocks map to (circuit, tile) by the items' first_block, the item's prog
// field holds the group's coefficient array); readout: it also folds the
// tile's sum p, p Z, p ZZ into the item's partials (the circuit's last group).
std::string jit_source(const ShmPlan& plan, std::vector<double>* coef, bool batch = false, bool readout = false);
// Compile a generated source (cached like every specialised kernel) and load
// its kernel `name` as a module of the current device.
hq_status jit_compile_load(const std::string& src, const char* name, hipModule_t* mod, hipFunction_t* fn);
}  // namespace hq
