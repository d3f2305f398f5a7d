// Which step kernel an on-chip plan gets, for every block size and several LDS
// sizes: host build of plb_onchip.hip, nothing is launched (tests/test_host_onchip.py).
#include "plb_onchip.hip"

namespace plb {

// Named by the host code, never called here.
StepArgs make_args(plb_ctx*, int64_t, bool) { return StepArgs(); }
static std::vector<size_t> asked;
hipError_t dev_alloc(void** p, size_t n)
{
    asked.push_back(n);
    if (asked.size() > 1) return hipErrorOutOfMemory;   // the plan's own arrays, then its scratch
    *p = malloc(64);
    return hipSuccess;
}
void dev_free(void*) {}

struct Kernel {
    const void* f;
    int elem, K;
    bool twice;
    int threads;
};
template <typename S, int K, bool TWICE, int MAXT>
static Kernel entry()
{
    return {(const void*)k_onchip<S, K, TWICE, MAXT>, (int)sizeof(S), K, TWICE, MAXT};
}

static int run()
{
    const Kernel all[] = {entry<double, 1, true, 512>(), entry<double, 1, false, 1024>(), entry<float, 2, false, 1024>(),
                          entry<float, 1, true, 512>(), entry<float, 1, true, 1024>(), entry<__half, 2, true, 1024>(),
                          entry<__half, 1, true, 512>(), entry<__half, 1, true, 1024>()};
    int fails = 0, plans = 0;
    plb_ctx c;
    for (int precision : {PLB_FP64, PLB_FP32, PLB_FP16})
        for (int kb = 16; kb <= 256; kb += 8) {
            c.cfg.precision = precision;
            c.elem = precision == PLB_FP64 ? 8 : precision == PLB_FP32 ? 4 : 2;
            c.lds_per_cu = kb * 1024;
            for (int nodes = 1; nodes <= 4096; nodes++) {
                if (!fits(&c, nodes)) continue;
                plans++;
                OnchipPlan p;
                shape(&c, &p, nodes);
                const void* f = nullptr;
                with_kernel(&c, &p, [&](auto* kern) { f = (const void*)kern; });
                bool ok = false;
                for (const Kernel& k : all)
                    ok |= k.f == f && k.elem == (int)c.elem && k.K == p.K && k.twice == p.twice && p.T <= k.threads;
                ok = ok && p.T * p.K == p.NS && p.NS >= nodes && p.T % 64 == 0 && lds_bytes(&c, p.NS, p.twice) + 64 <= (size_t)c.lds_per_cu;
                if (!ok && fails++ < 5)
                    fprintf(stderr, "precision %d, %d KB, %d nodes: K %d, T %d, NS %d, twice %d\n", precision, kb, nodes, p.K, p.T, p.NS, (int)p.twice);
            }
        }
    // A plan's scratch does not grow with samples that do not fit the chip.
    size_t scratch[2];
    for (int with = 0; with < 2; with++) {
        plb_ctx b;
        b.cfg.precision = PLB_FP32;
        b.elem = 4;
        b.lds_per_cu = 160 * 1024;
        std::vector<OnchipSample> samples(1 + with);
        samples[0].n = 20000;
        samples[0].nblocks = 20;
        for (OnchipSample& s : samples) s.d[0] = s.d[1] = s.d[2] = 30;
        if (with) {
            samples[1].off = 20032;
            samples[1].n = 100000000;
            samples[1].block0 = 20;
        }
        b.N = samples.back().off + samples.back().n;
        asked.clear();
        build_onchip(&b, samples, 20, 1024);
        scratch[with] = asked.size() == 2 ? asked[1] : 0;
    }
    if (!scratch[0] || scratch[1] > scratch[0] + 4096) {
        fprintf(stderr, "scratch: %zu bytes, with a large sample beside it %zu\n", scratch[0], scratch[1]);
        fails++;
    }
    printf("%d plans, %d failed\n", plans, fails);
    return fails || !plans;
}

}  // namespace plb

// There is no device code in this program.
extern "C" {
void** __hipRegisterFatBinary(const void*) { return nullptr; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void*, char*, const char*, unsigned, void*, void*, void*, void*, int*) {}
}
void plb_set_hip_error(hipError_t, const char*, const char*, int) {}
int main() { return plb::run(); }
