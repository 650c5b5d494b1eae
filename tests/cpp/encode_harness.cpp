// The interpreter's program of a group of diagonal gates, executed on the CPU
// (test infrastructure): the factor each amplitude of the state is multiplied
// by, as the slots say.  Links the library for its planner and encoder.
// usage: encode_harness n precision shared_mask diag_mode gates.bin out.bin
//   gates.bin: hq_gate array; out.bin: 2^n complex doubles
#include <complex>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <vector>

#include "hq_device.h"

using namespace hq;

template <typename R>
static int run(const ShmPlan& plan, const std::vector<char>& prog, std::vector<std::complex<double>>& out)
{
    ShmProg H;
    memcpy(&H, prog.data(), sizeof(H));
    const int tb = plan.tb, rb = plan.rb, blocks = 1 << (plan.n - plan.k), SLOT = shm_slot_bytes<R>();
    if (plan.stages.size() != 1) return 2;
    for (int b = 0; b < blocks; b++)
        for (int t = 0; t < (1 << tb); t++)
            for (int j = 0; j < (1 << rb); j++) {
                size_t idx = 0;
                for (uint32_t r = 0; r < H.num_runs; r++) idx |= (((uint64_t)b >> H.run[r].src) & H.run[r].mask) << H.run[r].dst;
                for (int i = 0; i < tb; i++) if ((t >> i) & 1) idx |= (size_t)1 << H.ld_thr[i];
                for (int i = 0; i < rb; i++) if ((j >> i) & 1) idx |= (size_t)1 << H.ld_reg[i];
                std::complex<double> f = 1;
                for (uint32_t q = 0; q < H.num_slots; q++) {
                    ShmSlot s;
                    const char* at = prog.data() + SHM_PROG_HEADER + (size_t)q * SLOT;
                    memcpy(&s, at, sizeof(s));
                    R c[2];
                    memcpy(c, at + sizeof(s), sizeof(c));
                    const std::complex<double> m(c[0], c[1]);
                    const bool on = (t & s.cthr) == s.cthrv, blk = ((uint32_t)b & s.cblk) == s.cblkv;
                    const bool reg = (j & s.creg) == s.cregv;
                    if (s.kind < SLOT_DIRECT_END) {
                        const int op = s.kind & 7, bit = s.kind >> 3;
                        if (op != DIRECT_PHASE && op != DIRECT_LPHASE) return 3;
                        if (((j >> bit) & 1) && (op == DIRECT_PHASE || on)) f *= m;
                    } else if (s.kind == SLOT_SCALE) {
                        f *= m;
                    } else if (s.kind == SLOT_MIX) {
                        if (blk && on && reg) f *= m;
                    } else if (s.kind == SLOT_MIXSIGN) {
                        if (blk && on && reg) f = -f;
                    } else if (s.kind == SLOT_REFILL) {
                        q += shm_window_slots<R>() - 1 - q % shm_window_slots<R>();
                    } else if (s.kind == SLOT_END) {
                        break;
                    } else {
                        return 4;   // forms of merged plans
                    }
                }
                out[idx] = f;
            }
    return 0;
}

int main(int argc, char** argv)
{
    if (argc != 7) return 1;
    const int n = atoi(argv[1]), precision = atoi(argv[2]);
    std::vector<hq_gate> gates;
    FILE* f = fopen(argv[5], "rb");
    hq_gate g;
    while (f && fread(&g, sizeof(g), 1, f) == 1) gates.push_back(g);
    if (f) fclose(f);
    ShmPlan plan;
    if (plan_sharemem(n, precision, gates.data(), (int)gates.size(), strtoull(argv[3], nullptr, 0), 0, &plan, false, 0,
                      false, (DiagMode)atoi(argv[4])) != HQ_OK)
        return 5;
    const std::vector<char> prog = encode_program(plan);
    std::vector<std::complex<double>> out((size_t)1 << n);
    const int rc = precision == HQ_C128 ? run<double>(plan, prog, out) : run<float>(plan, prog, out);
    if (rc) return rc;
    f = fopen(argv[6], "wb");
    if (!f || fwrite(out.data(), sizeof(out[0]), out.size(), f) != out.size()) return 6;
    return fclose(f);
}
