// readout.hip -- measurement sampling of a device state.
//
// The reference reads a state through kernelMeasure (P(qubit = 0),
// src/kernelSimple.cu:497-516) and full copies; drawing measurement shots
// is the step after it.  A shot is the smallest basis index i whose
// cumulative probability exceeds u * total, u uniform in [0, 1) from the
// portable generator (xoshiro256** seeded by SplitMix64, u = (x >> 11) 2^-53).
//
// Device work: one pass computes the probability sum of every 4096-amplitude
// chunk (fixed order) and of its 64 parts; the host forms the chunk prefix
// (FP64, in order); one wave per shot then searches the prefix, the chunk's
// parts and the part's amplitudes.  A thread walking its chunk amplitude by
// amplitude took 1.56 ms for 100 000 shots of 25 qubits (and 0.8 ms for 4096,
// the latency of one walk), beside 5 ms of searches on the host; this search
// reads 512 B of part sums, one part (1 KiB in complex128) and three probes of
// the prefix a lane and shot, one dependent step after another: 58 us and 6.4 us,
// after 128 us for the sums (87 without the part sums, 512 MiB).

#include "hq_device.h"
#include "reduce_dev.h"

#include <algorithm>
#include <vector>

#include "gate.h"

namespace hq {

constexpr int SAMPLE_CHUNK = 4096;
constexpr int SAMPLE_PART = 64;
constexpr int SAMPLE_PARTS = SAMPLE_CHUNK / SAMPLE_PART;
constexpr int SAMPLE_BATCH = 1 << 18;   // shots per launch
// Part sums take an eighth of a byte per amplitude: kept up to 64 MiB (29
// qubits); a wave of a larger state sums the parts of its chunk itself (64 KiB
// read per shot, little beside the pass over the state).
constexpr uint64_t SAMPLE_MAX_PARTS = 1ull << 23;
constexpr size_t SAMPLE_KEEP = (size_t)128 << 20;   // workspace kept between calls

template <typename R>
__device__ __forceinline__ double prob(const cplx<R>* __restrict__ a, uint64_t i, uint64_t amps)
{
    if (i >= amps) return 0;
    const double re = (double)a[i].x, im = (double)a[i].y;
    return re * re + im * im;
}

// parts may be null
template <typename R>
__global__ __launch_bounds__(256) void k_chunk_sums(const cplx<R>* __restrict__ a, uint64_t amps,
                                                     double* __restrict__ sums, double* __restrict__ parts)
{
    const uint64_t c = blockIdx.x;
    const uint32_t t = threadIdx.x;
    double p[SAMPLE_CHUNK / 256];
    double s = 0;
#pragma unroll
    for (int j = 0; j < SAMPLE_CHUNK / 256; j++) {
        p[j] = prob(a, c * SAMPLE_CHUNK + (uint64_t)j * 256 + t, amps);
        s += p[j];
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) s += __shfl_xor(s, o);
    __shared__ double red[4];
    if ((t & 63) == 0) red[t >> 6] = s;
    __syncthreads();
    if (t == 0) sums[c] = (red[0] + red[1]) + (red[2] + red[3]);
    if (!parts) return;
    // wave w's j-th load is part 4 j + w
    const int lane = (int)(t & 63);
    const double r = wave_columns<SAMPLE_CHUNK / 256, 32>(p, lane);
    const uint32_t j = __brev((uint32_t)lane) >> 26 & 15u;
    if ((lane & 3) == 0) parts[c * SAMPLE_PARTS + 4 * j + (t >> 6)] = r;
}

// One wave per shot; out[k] for the k-th uniform u[k].
template <typename R>
__global__ __launch_bounds__(256) void k_sample(const cplx<R>* __restrict__ a, uint64_t amps,
                                                 const double* __restrict__ prefix, uint64_t chunks,
                                                 const double* __restrict__ parts, const double* __restrict__ u,
                                                 uint32_t shots, uint64_t* __restrict__ out)
{
    const uint32_t k = blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = (int)(threadIdx.x & 63);
    if (k >= shots) return;
    const double t = u[k] * prefix[chunks - 1];
    // first chunk whose prefix exceeds t, 64 probes a step
    uint64_t lo = 0, hi = chunks;      // it is in [lo, hi], hi = chunks: none
    while (hi > lo) {
        const uint64_t step = (hi - lo + 63) / 64;
        const uint64_t i = lo + (uint64_t)lane * step + step - 1;   // last of the lane's stretch
        const bool in = i < hi;
        const uint64_t m = __ballot(in && prefix[in ? i : lo] > t);
        const uint64_t valid = __ballot(in);
        if (m) {
            const int f = __builtin_ctzll(m);
            hi = lo + (uint64_t)f * step + step - 1;
            lo += (uint64_t)f * step;
        } else {
            lo += (uint64_t)__popcll(valid) * step;
        }
    }
    const uint64_t c = lo < chunks ? lo : chunks - 1;
    const double r = t - (c ? prefix[c - 1] : 0.0);
    const uint64_t base = c * SAMPLE_CHUNK;
    // the chunk's part sums, one per lane
    double part;
    if (parts) {
        part = parts[c * SAMPLE_PARTS + lane];
    } else {
        part = 0;
        for (int q = 0; q < SAMPLE_PARTS; q++) {
            double p = prob(a, base + (uint64_t)(q * SAMPLE_PART + lane), amps);
#pragma unroll
            for (int o = 32; o >= 1; o >>= 1) p += __shfl_xor(p, o);
            if (lane == q) part = p;
        }
    }
    const double acc = wave_scan(part, lane);
    // an index of probability 0 is never drawn; where rounding leaves no sum
    // above r, the last index of nonzero probability is
    const uint64_t some = __ballot(part > 0);
    const uint64_t over = __ballot(part > 0 && acc > r);
    uint64_t pick = base;
    if (some) {
        const int q = over ? __builtin_ctzll(over) : 63 - __builtin_clzll(some);
        const double before = q ? __shfl(acc, q - 1) : 0.0;
        const double p = prob(a, base + (uint64_t)(q * SAMPLE_PART + lane), amps);
        const double in = before + wave_scan(p, lane);
        const uint64_t psome = __ballot(p > 0);
        const uint64_t pover = __ballot(p > 0 && in > r);
        const int l = over && pover ? __builtin_ctzll(pover) : psome ? 63 - __builtin_clzll(psome) : 0;
        pick = base + (uint64_t)(q * SAMPLE_PART + l);
    }
    if (lane == 0) out[k] = pick;
}

static void launch_sums(hq_state s, uint64_t chunks, double* sums, double* parts)
{
    if (s->precision == HQ_C128)
        hipLaunchKernelGGL(k_chunk_sums<double>, dim3((unsigned)chunks), dim3(256), 0, s->stream,
                           (const cplx<double>*)s->data, s->amps, sums, parts);
    else
        hipLaunchKernelGGL(k_chunk_sums<float>, dim3((unsigned)chunks), dim3(256), 0, s->stream,
                           (const cplx<float>*)s->data, s->amps, sums, parts);
}

static void launch_shots(hq_state s, uint64_t chunks, const double* prefix, const double* parts, const double* u,
                         uint32_t shots, uint64_t* out)
{
    const unsigned blocks = (shots + 3) / 4;
    if (s->precision == HQ_C128)
        hipLaunchKernelGGL(k_sample<double>, dim3(blocks), dim3(256), 0, s->stream, (const cplx<double>*)s->data,
                           s->amps, prefix, chunks, parts, u, shots, out);
    else
        hipLaunchKernelGGL(k_sample<float>, dim3(blocks), dim3(256), 0, s->stream, (const cplx<float>*)s->data,
                           s->amps, prefix, chunks, parts, u, shots, out);
}

static hq_status sample(hq_state s, int shots, uint64_t seed, uint64_t* out)
{
    const uint64_t chunks = (s->amps + SAMPLE_CHUNK - 1) / SAMPLE_CHUNK;
    const size_t batch = (size_t)std::min(shots, SAMPLE_BATCH);
    bool with_parts = chunks * SAMPLE_PARTS <= SAMPLE_MAX_PARTS;
    // device: prefix, uniforms, shots, part sums; pinned: uniforms, shots, prefix
    const size_t dev = (chunks + 2 * batch) * 8, host = dev;
    hq_status st = ensure_ws(s, dev + (with_parts ? chunks * SAMPLE_PARTS * 8 : 0), host);
    if (st != HQ_OK && with_parts) {   // no room beside the state: the waves sum the parts themselves
        (void)hipGetLastError();
        with_parts = false;
        st = ensure_ws(s, dev, host);
    }
    if (st != HQ_OK) return st;
    double* d_prefix = (double*)s->d_ws;
    double* d_u = d_prefix + chunks;
    uint64_t* d_out = (uint64_t*)(d_u + batch);
    double* d_parts = with_parts ? (double*)(d_out + batch) : nullptr;
    double* h_u = (double*)s->h_ws;
    uint64_t* h_out = (uint64_t*)(h_u + batch);
    double* prefix = (double*)(h_out + batch);
    launch_sums(s, chunks, d_prefix, d_parts);
    HQ_HIP(hipGetLastError());
    HQ_HIP(hipMemcpyAsync(prefix, d_prefix, chunks * 8, hipMemcpyDeviceToHost, s->stream));
    Rng rng(seed);
    for (size_t k = 0; k < batch; k++) h_u[k] = rng.uniform();   // while the sums run
    HQ_HIP(hipStreamSynchronize(s->stream));
    for (uint64_t c = 1; c < chunks; c++) prefix[c] += prefix[c - 1];
    if (!(prefix[chunks - 1] > 0)) {
        set_error("hq_state_sample: the state has zero norm");
        return HQ_ERR_STATE;
    }
    HQ_HIP(hipMemcpyAsync(d_prefix, prefix, chunks * 8, hipMemcpyHostToDevice, s->stream));
    for (size_t done = 0; done < (size_t)shots;) {
        const size_t m = std::min(batch, (size_t)shots - done);
        if (done)
            for (size_t k = 0; k < m; k++) h_u[k] = rng.uniform();
        HQ_HIP(hipMemcpyAsync(d_u, h_u, m * 8, hipMemcpyHostToDevice, s->stream));
        launch_shots(s, chunks, d_prefix, d_parts, d_u, (uint32_t)m, d_out);
        HQ_HIP(hipGetLastError());
        HQ_HIP(hipMemcpyAsync(h_out, d_out, m * 8, hipMemcpyDeviceToHost, s->stream));
        HQ_HIP(hipStreamSynchronize(s->stream));
        std::copy(h_out, h_out + m, out + done);
        done += m;
    }
    return HQ_OK;
}

}  // namespace hq

using namespace hq;

extern "C" hq_status hq_state_sample(hq_state s, int shots, uint64_t seed, uint64_t* out)
{
    HQ_CHECK(s && (out || shots == 0), HQ_ERR_ARG, "hq_state_sample: null argument");
    HQ_CHECK(shots >= 0 && shots <= (1 << 24), HQ_ERR_ARG, "hq_state_sample: shots must be in [0, 2^24]");
    if (shots == 0) return HQ_OK;
    std::lock_guard<std::mutex> lock(s->ws_mu);
    const hq_status st = sample(s, shots, seed, out);
    // after an error some of the call's work may still be queued
    if (st != HQ_OK && st != HQ_ERR_STATE) (void)hipStreamSynchronize(s->stream);
    trim_ws(s, SAMPLE_KEEP);
    return st;
}
