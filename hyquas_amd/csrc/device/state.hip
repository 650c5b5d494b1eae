// state.hip -- state vectors, readout reductions and profiling of the device layer.
//
// Replaces kernelInit / kernelDestroy / kernelGetAmp / kernelDeviceToHost /
// kernelMeasure (src/kernelSimple.cu:9-37, 448-529).  Allocation is 64-bit
// throughout (the reference's int nVec overflows at n >= 33).

#include "hq_device.h"
#include "reduce_dev.h"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <mutex>

namespace hq {

static thread_local std::string g_error;

void set_error(const std::string& msg) { g_error = msg; }
const char* get_error() { return g_error.c_str(); }

// ---- kernels -------------------------------------------------------------------------

// |0...0>: a fill kernel rather than hipMemsetAsync so the reset can be
// captured in a HIP graph.
template <typename R>
__global__ void k_reset(cplx<R>* __restrict__ a, uint64_t n_amps)
{
    uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (; i < n_amps; i += stride) {
        cplx<R> v;
        v.x = (i == 0) ? R(1) : R(0);
        v.y = R(0);
        a[i] = v;
    }
}

constexpr int RED_BLOCKS = 1024;
constexpr int RED_THREADS = 256;
constexpr int RED_MAXQ = 36;

__device__ inline double block_sum(double v, double* sh)
{
    // wave64 shuffle reduction, then across the 4 waves through LDS
    for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
    int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    __syncthreads();
    if (lane == 0) sh[wave] = v;
    __syncthreads();
    double r = 0;
    if (threadIdx.x == 0)
        for (int w = 0; w < (int)(blockDim.x >> 6); w++) r += sh[w];
    return r;
}

// Kahan-compensated FP64 accumulation of |a_i|^2 over a subset (bit `target`
// clear when target >= 0: the subset's elements are numbered, nothing of the
// rest is read), one partial per block (measure<>/reduce<>,
// kernelSimple.cu:448-495).  Bound by HBM: independent 16-byte loads per thread and
// step.  Complex64 takes four (one 8-byte load at a time read a 2 GiB state in 0.65
// ms, this in 0.42), complex128 two (26 and 28 qubits: one load 206 and 866 us,
// two 197 and 774, four 217 and 836; 24 qubits 53, 54.5 and 56).
template <typename R>
__global__ __launch_bounds__(RED_THREADS) void k_norm(const cplx<R>* __restrict__ a, uint64_t n_amps, int target,
                                                      double* __restrict__ out)
{
    constexpr int E = 16 / (2 * (int)sizeof(R));   // amplitudes per 16-byte element
    constexpr int U = E == 2 ? 4 : 2;              // loads per thread and step
    struct alignas(16) Elem { cplx<R> v[E]; };
    __shared__ double sh[16];
    double s = 0, c = 0;
    auto add = [&](cplx<R> v) {
        const double p = (double)v.x * (double)v.x + (double)v.y * (double)v.y;
        const double y = p - c;
        const double t = s + y;
        c = (t - s) - y;
        s = t;
    };
    // a target inside an element (complex64 qubit 0) drops its second amplitude
    const bool inside = E == 2 && target == 0;
    const int tb = target < 0 || inside ? -1 : target - (E == 2 ? 1 : 0);
    const uint64_t elems = n_amps / E >> (tb >= 0 ? 1 : 0);
    const Elem* __restrict__ src = (const Elem*)a;
    auto at = [&](uint64_t i) { return tb < 0 ? i : (i >> tb) << (tb + 1) | (i & (((uint64_t)1 << tb) - 1)); };
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    for (; i + (U - 1) * stride < elems; i += U * stride) {
        Elem v[U];
#pragma unroll
        for (int k = 0; k < U; k++) v[k] = src[at(i + (uint64_t)k * stride)];
#pragma unroll
        for (int k = 0; k < U; k++) {
            add(v[k].v[0]);
            if constexpr (E == 2) { if (!inside) add(v[k].v[1]); }
        }
    }
    for (; i < elems; i += stride) {
        const Elem v = src[at(i)];
        add(v.v[0]);
        if constexpr (E == 2) { if (!inside) add(v.v[1]); }
    }
    double r = block_sum(s, sh);
    if (threadIdx.x == 0) out[blockIdx.x] = r;
}

// ---- <Z_q>, <Z_q Z_{q+1}> -------------------------------------------------------------
// Row layout of a block's partials: sum p, sum p bit_q (RED_MAXQ columns),
// sum p (bit_q xor bit_{q+1}) (RED_MAXQ columns); columns of absent qubits
// hold zeros.
constexpr int RED_Z_BLOCKS = 256;
constexpr int RED_Z_STRIDE = 1 + 2 * RED_MAXQ;
constexpr int EZ_THREADS = 1024;
constexpr int EZ_CHUNK_BITS = 13;   // 1024 threads x 8 amplitudes

// One row of partials per block, one read of the state.  HBM-bound by
// construction: an index bit's weight is a constant of the place that holds
// it, so per amplitude only p is formed and added to one of the thread's
// eight accumulators; nothing is added per qubit and amplitude (that form
// spent 2 n additions on every amplitude: 64.6 ms at 30 qubits complex128,
// 129 ms at 31 qubits complex64; this one 2.92 ms = 5.9 TB/s and 3.22 ms =
// 5.3 TB/s).
//   index bits   held by
//   0..12        lane (6), register (3), wave (4): weighted once at the end
//   13..12+l     the block's loop over its 2^l consecutive chunks (l <= LB):
//                one conditional add per chunk, thread and bit
//   above        the block index: weighted in the row
// A lane moves 16 bytes per load: one complex128 amplitude, or two
// neighbouring complex64 ones (bit 0 is then a register bit).
template <typename R, int LB>
__global__ __launch_bounds__(EZ_THREADS) void k_expect_z(const cplx<R>* __restrict__ a, int n, int l,
                                                         double* __restrict__ out)
{
    constexpr bool PAIR = sizeof(R) == 4;
    constexpr int NCOL = 20 + 2 * LB;
    __shared__ double sh[EZ_THREADS / 64][NCOL];
    const uint64_t amps = (uint64_t)1 << n;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint64_t blk = blockIdx.x;
    double acc[8];
#pragma unroll
    for (int j = 0; j < 8; j++) acc[j] = 0;
    double s[LB > 0 ? LB : 1], zz[LB > 0 ? LB : 1], zw = 0;
#pragma unroll
    for (int b = 0; b < LB; b++) { s[b] = 0; zz[b] = 0; }
    const uint64_t c0 = blk << l, c1 = c0 + ((uint64_t)1 << l);
    for (uint64_t c = c0; c < c1; c++) {
        double p[8];
        const uint64_t base = (c << EZ_CHUNK_BITS) | ((uint64_t)wave << 9);
        if constexpr (PAIR) {
            struct alignas(16) Two { cplx<R> v[2]; };
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const uint64_t i = base | (uint64_t)(k << 7 | lane << 1);
                Two t = {};
                if (i < amps) t = *(const Two*)(a + i);
#pragma unroll
                for (int h = 0; h < 2; h++)
                    p[2 * k + h] = (double)t.v[h].x * (double)t.v[h].x + (double)t.v[h].y * (double)t.v[h].y;
            }
        } else {
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const uint64_t i = base | (uint64_t)(j << 6 | lane);
                cplx<R> t = {};
                if (i < amps) t = a[i];
                p[j] = (double)t.x * (double)t.x + (double)t.y * (double)t.y;
            }
        }
#pragma unroll
        for (int j = 0; j < 8; j++) acc[j] += p[j];
        const double t = ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
        // uniform conditions: scalar branches
        const uint64_t x = c ^ (c >> 1);
        if (((uint64_t)(wave >> 3) ^ c) & 1) zw += t;
#pragma unroll
        for (int b = 0; b < LB; b++) {
            if ((c >> b) & 1) s[b] += t;
            if ((x >> b) & 1) zz[b] += t;
        }
    }
    // thread columns: 0 total; 1..6 lane bits; 7..11 neighbouring lane bits;
    // 12..14 register bits; 15 register bits 1,2; 16, 17 the two pairs between
    // lane and register bits (complex128: register bits 0,1 take 16); 18 the
    // last register and the first wave bit; 19 the last wave bit and chunk bit
    // 0; then the chunk bits and their pairs
    {
        double v[NCOL];
        double half[3][2];
#pragma unroll
        for (int r = 0; r < 3; r++)
#pragma unroll
            for (int h = 0; h < 2; h++) {
                double t = 0;
#pragma unroll
                for (int j = 0; j < 8; j++)
                    if (((j >> r) & 1) == h) t += acc[j];
                half[r][h] = t;
            }
        auto cross = [&](int r0, int r1) {
            double t = 0;
#pragma unroll
            for (int j = 0; j < 8; j++)
                if (((j >> r0) ^ (j >> r1)) & 1) t += acc[j];
            return t;
        };
        const double T = half[0][0] + half[0][1];
        v[0] = T;
#pragma unroll
        for (int k = 0; k < 6; k++) v[1 + k] = ((lane >> k) & 1) ? T : 0.0;
#pragma unroll
        for (int k = 0; k < 5; k++) v[7 + k] = (((lane ^ (lane >> 1)) >> k) & 1) ? T : 0.0;
#pragma unroll
        for (int r = 0; r < 3; r++) v[12 + r] = half[r][1];
        v[15] = cross(1, 2);
        if constexpr (PAIR) {
            v[16] = (lane & 1) ? half[0][0] : half[0][1];
            v[17] = (lane >> 5) ? half[1][0] : half[1][1];
        } else {
            v[16] = cross(0, 1);
            v[17] = (lane >> 5) ? half[0][0] : half[0][1];
        }
        v[18] = (wave & 1) ? half[2][0] : half[2][1];
        v[19] = zw;
#pragma unroll
        for (int b = 0; b < LB; b++) { v[20 + b] = s[b]; v[20 + LB + b] = zz[b]; }
        const double r = wave_columns<NCOL, 32>(v, lane);
        const int col = (int)(__brev((unsigned)lane) >> 26);
        if (col < NCOL) sh[wave][col] = r;
    }
    __syncthreads();
    const int waves = (int)(blockDim.x >> 6);
    for (int o = threadIdx.x; o < RED_Z_STRIDE; o += (int)blockDim.x) {
        // row column o: qubit q's bit (pair = 0) or the pair q, q+1
        const bool pair = o > RED_MAXQ;
        const int q = o == 0 ? -1 : pair ? o - 1 - RED_MAXQ : o - 1;
        int col = 0;            // thread column summed over the waves with weight 1 ...
        int wmask = -1;         // ... or, >= 0: over the waves whose index has odd parity under it
        bool zero = false;
        constexpr int LANE0 = PAIR ? 1 : 0;   // qubit of lane bit 0
        if (q < 0) {
            col = 0;
        } else if (q + (pair ? 1 : 0) >= n) {
            zero = true;
        } else if (q >= EZ_CHUNK_BITS + LB) {
            const uint64_t c = blk << l;      // constant over the block
            const uint64_t y = pair ? c ^ (c >> 1) : c;
            zero = !((y >> (q - EZ_CHUNK_BITS)) & 1);
        } else if (q >= EZ_CHUNK_BITS) {
            col = 20 + (pair ? LB : 0) + (q - EZ_CHUNK_BITS);
        } else if (!pair) {
            if (q >= 9) wmask = 1 << (q - 9);
            else if (q >= 7) col = 12 + (q - 6);
            else if (PAIR && q == 0) col = 12;
            else if (!PAIR && q == 6) col = 12;
            else col = 1 + (q - LANE0);
        } else {
            if (q == 12) col = 19;
            else if (q >= 9) wmask = 3 << (q - 9);
            else if (q == 8) col = 18;
            else if (q == 7) col = 15;
            else if (PAIR) col = q == 6 ? 17 : q == 0 ? 16 : 7 + (q - 1);
            else col = q == 6 ? 16 : q == 5 ? 17 : 7 + q;
        }
        double r = 0;
        if (!zero)
            for (int w = 0; w < waves; w++)
                if (wmask < 0 || (__popc(w & wmask) & 1)) r += sh[w][col];
        out[blk * RED_Z_STRIDE + o] = r;
    }
}

template <typename RA, typename RB>
__global__ void k_inner(const cplx<RA>* __restrict__ a, const cplx<RB>* __restrict__ b, uint64_t n_amps,
                        double* __restrict__ out)
{
    __shared__ double sh[16];
    double sr = 0, si = 0;
    uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n_amps; i += stride) {
        cplx<RA> x = a[i];
        cplx<RB> y = b[i];
        double xr = x.x, xi = x.y, yr = y.x, yi = y.y;
        sr += xr * yr + xi * yi;   // conj(x) * y
        si += xr * yi - xi * yr;
    }
    double r1 = block_sum(sr, sh);
    if (threadIdx.x == 0) out[2 * blockIdx.x] = r1;
    double r2 = block_sum(si, sh);
    if (threadIdx.x == 0) out[2 * blockIdx.x + 1] = r2;
}

// Column sums of `count` rows (row stride `stride`) into fin, one wave per
// column: lane i takes rows i, i + 64, ... with a Kahan sum, then a fixed tree
// over the lanes.  fin may be host memory the device can write.
__global__ __launch_bounds__(64) void k_sum_columns(const double* __restrict__ part, int count, int stride,
                                                    double* __restrict__ fin)
{
    const int c = blockIdx.x;
    double sum = 0, comp = 0;
#pragma unroll 4
    for (int b = threadIdx.x; b < count; b += 64) {
        double y = part[(size_t)b * stride + c] - comp;
        double t = sum + y;
        comp = (t - sum) - y;
        sum = t;
    }
#pragma unroll
    for (int m = 32; m > 0; m >>= 1) sum += __shfl_xor(sum, m);
    if (threadIdx.x == 0) fin[c] = sum;
}

// ---- allocation-free readout -----------------------------------------------------------
// Scratch of hq_expect_z_noalloc: the per-block partials of k_expect_z (at
// most RED_Z_BLOCKS rows of 1 + 2 * RED_MAXQ doubles) followed by one row of
// column sums.  One copy per device, held until the process ends; host code
// addresses it only through the pointer hipGetSymbolAddress returns for the
// device (noalloc_scratch below).
constexpr size_t NOALLOC_SCRATCH_DOUBLES = (size_t)(RED_Z_BLOCKS + 1) * RED_Z_STRIDE;   // 147 KiB
static __device__ __align__(256) double scratch[NOALLOC_SCRATCH_DOUBLES];

constexpr int NOALLOC_MAX_DEVICES = 64;
static std::mutex g_scratch_mu;
static double* g_scratch_ptr[NOALLOC_MAX_DEVICES] = {};

// Device address of `scratch` on `device`, looked up once per device with that
// device current (each device holds its own copy at its own address).
static hq_status noalloc_scratch(int device, double** out)
{
    HQ_CHECK(device >= 0 && device < NOALLOC_MAX_DEVICES, HQ_ERR_UNSUPPORTED,
             "hq_expect_z_noalloc: device index beyond the supported 64");
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[device]) {
        int cur = 0;
        HQ_HIP(hipGetDevice(&cur));
        if (cur != device) HQ_HIP(hipSetDevice(device));
        void* ptr = nullptr;
        hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (cur != device) (void)hipSetDevice(cur);
        if (e != hipSuccess || !ptr) {
            set_error(std::string("hq_expect_z_noalloc: hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
            return HQ_ERR_HIP;
        }
        g_scratch_ptr[device] = (double*)ptr;
    }
    *out = g_scratch_ptr[device];
    return HQ_OK;
}

// Room in the state's reduction buffers; the caller holds ws_mu until it has read
// its results out of h_red (growing frees the buffers, and every readout writes
// to their start).
static hq_status ensure_red(hq_state s, size_t doubles)
{
    if (s->red_cap >= doubles) return HQ_OK;
    if (s->d_red) { (void)hipFree(s->d_red); s->d_red = nullptr; }
    if (s->h_red) { (void)hipHostFree(s->h_red); s->h_red = nullptr; }
    s->red_cap = 0;
    HQ_HIP(hipMalloc(&s->d_red, doubles * sizeof(double)));
    HQ_HIP(hipHostMalloc(&s->h_red, doubles * sizeof(double), hipHostMallocDefault));
    s->red_cap = doubles;
    return HQ_OK;
}

// The state's readout workspace: at least `dev` bytes of device and `host` bytes
// of pinned memory, kept for the next readout.
hq_status ensure_ws(hq_state s, size_t dev, size_t host)
{
    if (s->ws_dev < dev) {
        if (s->d_ws) (void)hipFree(s->d_ws);
        s->d_ws = nullptr;
        s->ws_dev = 0;
        HQ_HIP(hipMalloc((void**)&s->d_ws, dev));
        s->ws_dev = dev;
    }
    if (s->ws_host < host) {
        if (s->h_ws) (void)hipHostFree(s->h_ws);
        s->h_ws = nullptr;
        s->ws_host = 0;
        HQ_HIP(hipHostMalloc((void**)&s->h_ws, host, hipHostMallocDefault));
        s->ws_host = host;
    }
    return HQ_OK;
}

void trim_ws(hq_state s, size_t keep)
{
    if (s->ws_dev > keep) { (void)hipFree(s->d_ws); s->d_ws = nullptr; s->ws_dev = 0; }
    if (s->ws_host > keep) { (void)hipHostFree(s->h_ws); s->h_ws = nullptr; s->ws_host = 0; }
}

static unsigned grid_for(uint64_t work, unsigned threads, unsigned cap)
{
    uint64_t g = (work + threads - 1) / threads;
    if (g > cap) g = cap;
    if (g < 1) g = 1;
    return (unsigned)g;
}

hq_status prof_begin(hq_state s, int kind, int* slot)
{
    *slot = -1;
    if (!s->profiling) return HQ_OK;
    ProfileEntry e;
    e.kind = kind;
    for (hipEvent_t* ev : {&e.start, &e.stop}) {
        if (!s->free_events.empty()) { *ev = s->free_events.back(); s->free_events.pop_back(); }
        else HQ_HIP(hipEventCreate(ev));
    }
    HQ_HIP(hipEventRecord(e.start, s->stream));
    s->prof.push_back(e);
    *slot = (int)s->prof.size() - 1;
    return HQ_OK;
}

hq_status prof_end(hq_state s, int slot)
{
    if (slot < 0) return HQ_OK;
    HQ_HIP(hipEventRecord(s->prof[slot].stop, s->stream));
    return HQ_OK;
}

}  // namespace hq

using namespace hq;

extern "C" {

const char* hq_last_error(void) { return hq::get_error(); }

hq_status hq_device_count(int* count)
{
    HQ_CHECK(count, HQ_ERR_ARG, "hq_device_count: null pointer");
    int c = 0;
    hipError_t e = hipGetDeviceCount(&c);
    if (e != hipSuccess || c == 0) {
        *count = 0;
        set_error(std::string("no HIP device visible: ") + hipGetErrorString(e));
        return HQ_ERR_NO_DEVICE;
    }
    *count = c;
    return HQ_OK;
}

hq_status hq_state_create(int num_qubits, int precision, int with_buffer, hq_state* out)
{
    HQ_CHECK(out, HQ_ERR_ARG, "hq_state_create: null output");
    *out = nullptr;
    HQ_CHECK(num_qubits >= 1 && num_qubits <= 36, HQ_ERR_ARG, "hq_state_create: num_qubits must be in [1, 36]");
    HQ_CHECK(precision == HQ_C128 || precision == HQ_C64, HQ_ERR_ARG, "hq_state_create: bad precision");
    int ndev = 0;
    hq_status st = hq_device_count(&ndev);
    if (st != HQ_OK) return st;
    hq_state s = new hq_state_s();
    s->n = num_qubits;
    s->precision = precision;
    s->amps = (uint64_t)1 << num_qubits;
    s->amp_bytes = precision == HQ_C128 ? 16 : 8;
    if (hipGetDevice(&s->device) != hipSuccess) s->device = 0;
    size_t bytes = s->amps * s->amp_bytes;
    hipError_t e = hipMalloc(&s->data, bytes);
    if (e != hipSuccess) {
        set_error("hq_state_create: hipMalloc of " + std::to_string(bytes) + " B failed: " + hipGetErrorString(e));
        delete s;
        return HQ_ERR_OOM;
    }
    if (with_buffer) {
        e = hipMalloc(&s->buf, bytes);
        if (e != hipSuccess) {
            set_error("hq_state_create: hipMalloc of the work buffer failed: " + std::string(hipGetErrorString(e)));
            (void)hipFree(s->data);
            delete s;
            return HQ_ERR_OOM;
        }
    }
    e = hipStreamCreateWithFlags(&s->stream, hipStreamNonBlocking);
    if (e != hipSuccess) {
        set_error(std::string("hipStreamCreate: ") + hipGetErrorString(e));
        (void)hipFree(s->data);
        if (s->buf) (void)hipFree(s->buf);
        delete s;
        return HQ_ERR_HIP;
    }
    *out = s;
    return hq_state_reset(s);
}

hq_status hq_state_destroy(hq_state s)
{
    if (!s) return HQ_OK;
    if (s->stream) (void)hipStreamSynchronize(s->stream);
    if (s->data) (void)hipFree(s->data);
    if (s->buf) (void)hipFree(s->buf);
    if (s->d_red) (void)hipFree(s->d_red);
    if (s->h_red) (void)hipHostFree(s->h_red);
    if (s->d_ws) (void)hipFree(s->d_ws);
    if (s->h_ws) (void)hipHostFree(s->h_ws);
    for (auto& e : s->prof) { (void)hipEventDestroy(e.start); (void)hipEventDestroy(e.stop); }
    for (auto& e : s->free_events) (void)hipEventDestroy(e);
    if (s->stream) (void)hipStreamDestroy(s->stream);
    delete s;
    return HQ_OK;
}

hq_status hq_state_reset(hq_state s)
{
    HQ_CHECK(s, HQ_ERR_ARG, "hq_state_reset: null state");
    unsigned g = grid_for(s->amps, 256, 65536);
    if (s->precision == HQ_C128)
        hipLaunchKernelGGL(k_reset<double>, dim3(g), dim3(256), 0, s->stream, (cplx<double>*)s->data, s->amps);
    else
        hipLaunchKernelGGL(k_reset<float>, dim3(g), dim3(256), 0, s->stream, (cplx<float>*)s->data, s->amps);
    HQ_HIP(hipGetLastError());
    return HQ_OK;
}

hq_status hq_state_info(hq_state s, int* num_qubits, int* precision)
{
    HQ_CHECK(s, HQ_ERR_ARG, "hq_state_info: null state");
    if (num_qubits) *num_qubits = s->n;
    if (precision) *precision = s->precision;
    return HQ_OK;
}

hq_status hq_state_has_buffer(hq_state s, int* has_buffer)
{
    HQ_CHECK(s && has_buffer, HQ_ERR_ARG, "hq_state_has_buffer: null argument");
    *has_buffer = s->buf ? 1 : 0;
    return HQ_OK;
}

hq_status hq_state_sync(hq_state s)
{
    HQ_CHECK(s, HQ_ERR_ARG, "hq_state_sync: null state");
    HQ_HIP(hipStreamSynchronize(s->stream));
    return HQ_OK;
}

hq_status hq_state_download(hq_state s, void* host, uint64_t count)
{
    HQ_CHECK(s && host, HQ_ERR_ARG, "hq_state_download: null argument");
    HQ_CHECK(count == s->amps, HQ_ERR_ARG, "hq_state_download: count must be 2^n");
    HQ_HIP(hipMemcpyAsync(host, s->data, s->amps * s->amp_bytes, hipMemcpyDeviceToHost, s->stream));
    HQ_HIP(hipStreamSynchronize(s->stream));
    return HQ_OK;
}

hq_status hq_state_upload(hq_state s, const void* host, uint64_t count)
{
    HQ_CHECK(s && host, HQ_ERR_ARG, "hq_state_upload: null argument");
    HQ_CHECK(count == s->amps, HQ_ERR_ARG, "hq_state_upload: count must be 2^n");
    HQ_HIP(hipMemcpyAsync(s->data, host, s->amps * s->amp_bytes, hipMemcpyHostToDevice, s->stream));
    HQ_HIP(hipStreamSynchronize(s->stream));
    return HQ_OK;
}

hq_status hq_state_get_amp(hq_state s, uint64_t index, double* re, double* im)
{
    HQ_CHECK(s && re && im, HQ_ERR_ARG, "hq_state_get_amp: null argument");
    HQ_CHECK(index < s->amps, HQ_ERR_ARG, "hq_state_get_amp: index out of range");
    std::lock_guard<std::mutex> lock(s->ws_mu);
    hq_status st = ensure_red(s, 2);
    if (st != HQ_OK) return st;
    HQ_HIP(hipMemcpyAsync(s->h_red, (char*)s->data + index * s->amp_bytes, s->amp_bytes,
                          hipMemcpyDeviceToHost, s->stream));
    HQ_HIP(hipStreamSynchronize(s->stream));
    if (s->precision == HQ_C128) { *re = s->h_red[0]; *im = s->h_red[1]; }
    else { float* f = (float*)s->h_red; *re = f[0]; *im = f[1]; }
    return HQ_OK;
}

static hq_status sum_partials(hq_state s, int count, int stride, int offset, double* out)
{
    // Kahan sum of the per-block partials on the host, in FP64.
    double sum = 0, c = 0;
    for (int b = 0; b < count; b++) {
        double y = s->h_red[b * stride + offset] - c;
        double t = sum + y;
        c = (t - sum) - y;
        sum = t;
    }
    *out = sum;
    return HQ_OK;
}

static hq_status run_norm(hq_state s, int target, double* out)
{
    std::lock_guard<std::mutex> lock(s->ws_mu);
    hq_status st = ensure_red(s, RED_BLOCKS);
    if (st != HQ_OK) return st;
    unsigned g = grid_for(s->amps, RED_THREADS, RED_BLOCKS);
    if (s->precision == HQ_C128)
        hipLaunchKernelGGL(k_norm<double>, dim3(g), dim3(RED_THREADS), 0, s->stream,
                           (const cplx<double>*)s->data, s->amps, target, s->d_red);
    else
        hipLaunchKernelGGL(k_norm<float>, dim3(g), dim3(RED_THREADS), 0, s->stream,
                           (const cplx<float>*)s->data, s->amps, target, s->d_red);
    HQ_HIP(hipGetLastError());
    HQ_HIP(hipMemcpyAsync(s->h_red, s->d_red, g * sizeof(double), hipMemcpyDeviceToHost, s->stream));
    HQ_HIP(hipStreamSynchronize(s->stream));
    return sum_partials(s, (int)g, 1, 0, out);
}

hq_status hq_state_norm(hq_state s, double* norm2)
{
    HQ_CHECK(s && norm2, HQ_ERR_ARG, "hq_state_norm: null argument");
    return run_norm(s, -1, norm2);
}

hq_status hq_measure_zero(hq_state s, int target, double* p0)
{
    HQ_CHECK(s && p0, HQ_ERR_ARG, "hq_measure_zero: null argument");
    HQ_CHECK(target >= 0 && target < s->n, HQ_ERR_ARG, "hq_measure_zero: target out of range");
    return run_norm(s, target, p0);
}

// Column sums of the state (the layout of a k_expect_z row) into fin, device
// or device-writable host memory; rows: RED_Z_BLOCKS rows of device scratch,
// unused by a state of one chunk.  Asynchronous.
static hq_status launch_expect_z(hq_state s, double* rows, double* fin)
{
    // one chunk per block up to RED_Z_BLOCKS blocks (2^21 amplitudes), then
    // 2^l consecutive chunks per block: 16 waves on every CU, and at most
    // RED_Z_BLOCKS rows.  LB, the loop bits a kernel has columns for, costs
    // registers (two doubles a thread each) and reduction steps, so it is
    // 0, 10 or 15 by size
    const int cb = std::max(0, s->n - EZ_CHUNK_BITS);
    const int l = std::max(0, cb - 8);
    const unsigned g = 1u << (cb - l);
    static_assert(RED_Z_BLOCKS == 1 << 8, "block bits");
    double* part = g > 1 ? rows : fin;
    // states below one chunk: a wave per 512 amplitudes
    const unsigned threads = s->n >= EZ_CHUNK_BITS ? EZ_THREADS : 64u << std::max(0, s->n - 9);
#define HQ_EZ(RV, LBV)                                                                                          \
    hipLaunchKernelGGL((k_expect_z<RV, LBV>), dim3(g), dim3(threads), 0, s->stream, (const cplx<RV>*)s->data, \
                       s->n, l, part)
    if (s->precision == HQ_C128) {
        if (l == 0) HQ_EZ(double, 0);
        else if (l <= 10) HQ_EZ(double, 10);
        else HQ_EZ(double, 15);
    } else {
        if (l == 0) HQ_EZ(float, 0);
        else if (l <= 10) HQ_EZ(float, 10);
        else HQ_EZ(float, 15);
    }
#undef HQ_EZ
    HQ_HIP(hipGetLastError());
    if (g > 1) {
        hipLaunchKernelGGL(k_sum_columns, dim3(RED_Z_STRIDE), dim3(64), 0, s->stream, (const double*)rows, (int)g,
                           RED_Z_STRIDE, fin);
        HQ_HIP(hipGetLastError());
    }
    return HQ_OK;
}

// z[q] = <Z_q>, zz[q] = <Z_q Z_{q+1}> from the column sums of k_expect_z
// (tot, sum p bit_q, sum p (bit_q xor bit_{q+1})).
static void finish_expect_z(int n, const double* col, double* z, double* zz)
{
    const double tot = col[0];
    for (int q = 0; q < n; q++) {
        if (z) z[q] = tot - 2 * col[1 + q];
        if (zz && q + 1 < n) zz[q] = tot - 2 * col[1 + RED_MAXQ + q];
    }
}

hq_status hq_expect_z(hq_state s, double* z, double* zz)
{
    HQ_CHECK(s, HQ_ERR_ARG, "hq_expect_z: null state");
    HQ_CHECK(s->n <= RED_MAXQ, HQ_ERR_UNSUPPORTED, "hq_expect_z: at most 36 qubits");
    std::lock_guard<std::mutex> lock(s->ws_mu);
    hq_status st = ensure_red(s, (size_t)RED_Z_BLOCKS * RED_Z_STRIDE);
    if (st != HQ_OK) return st;
    // the sums go straight to the pinned buffer: no copy to wait for
    st = launch_expect_z(s, s->d_red, s->h_red);
    if (st != HQ_OK) return st;
    HQ_HIP(hipStreamSynchronize(s->stream));
    finish_expect_z(s->n, s->h_red, z, zz);
    return HQ_OK;
}

hq_status hq_expect_z_noalloc(hq_state s, double* z, double* zz)
{
    HQ_CHECK(s, HQ_ERR_ARG, "hq_expect_z_noalloc: null state");
    HQ_CHECK(s->n <= RED_MAXQ, HQ_ERR_UNSUPPORTED, "hq_expect_z_noalloc: at most 36 qubits");
    double* ptr = nullptr;
    hq_status st = noalloc_scratch(s->device, &ptr);
    if (st != HQ_OK) return st;
    // every partial row and the column-sum row are written before they are
    // read: nothing in the scratch has to start at zero
    double* fin = ptr + (size_t)RED_Z_BLOCKS * RED_Z_STRIDE;
    st = launch_expect_z(s, ptr, fin);
    if (st != HQ_OK) return st;
    double col[RED_Z_STRIDE];
    HQ_HIP(hipMemcpyAsync(col, fin, RED_Z_STRIDE * sizeof(double), hipMemcpyDeviceToHost, s->stream));
    HQ_HIP(hipStreamSynchronize(s->stream));
    finish_expect_z(s->n, col, z, zz);
    return HQ_OK;
}

hq_status hq_state_inner(hq_state a, hq_state b, double* re, double* im)
{
    HQ_CHECK(a && b && re && im, HQ_ERR_ARG, "hq_state_inner: null argument");
    HQ_CHECK(a->n == b->n, HQ_ERR_ARG, "hq_state_inner: qubit counts differ");
    HQ_HIP(hipStreamSynchronize(b->stream));
    unsigned g = grid_for(a->amps, RED_THREADS, RED_BLOCKS);
    std::lock_guard<std::mutex> lock(a->ws_mu);
    hq_status st = ensure_red(a, 2 * (size_t)g);
    if (st != HQ_OK) return st;
    if (a->precision == HQ_C128 && b->precision == HQ_C128)
        hipLaunchKernelGGL((k_inner<double, double>), dim3(g), dim3(RED_THREADS), 0, a->stream,
                           (const cplx<double>*)a->data, (const cplx<double>*)b->data, a->amps, a->d_red);
    else if (a->precision == HQ_C128)
        hipLaunchKernelGGL((k_inner<double, float>), dim3(g), dim3(RED_THREADS), 0, a->stream,
                           (const cplx<double>*)a->data, (const cplx<float>*)b->data, a->amps, a->d_red);
    else if (b->precision == HQ_C128)
        hipLaunchKernelGGL((k_inner<float, double>), dim3(g), dim3(RED_THREADS), 0, a->stream,
                           (const cplx<float>*)a->data, (const cplx<double>*)b->data, a->amps, a->d_red);
    else
        hipLaunchKernelGGL((k_inner<float, float>), dim3(g), dim3(RED_THREADS), 0, a->stream,
                           (const cplx<float>*)a->data, (const cplx<float>*)b->data, a->amps, a->d_red);
    HQ_HIP(hipGetLastError());
    HQ_HIP(hipMemcpyAsync(a->h_red, a->d_red, 2 * (size_t)g * sizeof(double), hipMemcpyDeviceToHost, a->stream));
    HQ_HIP(hipStreamSynchronize(a->stream));
    sum_partials(a, (int)g, 2, 0, re);
    sum_partials(a, (int)g, 2, 1, im);
    return HQ_OK;
}

hq_status hq_profile_enable(hq_state s, int enable)
{
    HQ_CHECK(s, HQ_ERR_ARG, "hq_profile_enable: null state");
    s->profiling = enable != 0;
    return HQ_OK;
}

hq_status hq_profile_read(hq_state s, int* kinds, double* ms, int cap, int* count)
{
    HQ_CHECK(s && count, HQ_ERR_ARG, "hq_profile_read: null argument");
    HQ_HIP(hipStreamSynchronize(s->stream));
    int k = 0;
    for (auto& e : s->prof) {
        float t = 0;
        HQ_HIP(hipEventElapsedTime(&t, e.start, e.stop));
        if (k < cap) {
            if (kinds) kinds[k] = e.kind;
            if (ms) ms[k] = t;
        }
        k++;
        s->free_events.push_back(e.start);
        s->free_events.push_back(e.stop);
    }
    s->prof.clear();
    *count = k;
    return HQ_OK;
}

}  // extern "C"
