// Walks the lanes of the paired tiles that end a real forward transform (SplitCfg) and checks that
// every index a lane makes into the pass-twiddle tables lies inside them, also for the lanes
// that have no sequence.  Host code only.
#include <cstdio>

#include "../../gfft_amd/csrc/tile_kernel.h"

using namespace gfftx;

template <class C> int walk(long long S, long long ns)
{
    // the tables of M = ns L roots, as upload_root_tables sizes them
    const long long M = ns * C::L;
    int b = 0;
    while ((1LL << (2 * b)) < M) ++b;
    const long long nlo = 1LL << b, nhi = (M + nlo - 1) / nlo + 1;
    const long long pairs = (S - 1) / 2, h = C::NB / 2, tiles = 1 + (pairs + h - 1) / h;
    const int LR = C::L / C::R[0];
    int bad = 0;
    for (long long tile = 0; tile < tiles; ++tile)
        for (int t = 0; t < C::NB; ++t) {
            const long long tg = split_seq<C>(S, (unsigned)tile, t);
            const long long kp = pass_phase(tg >= 0, tg, ns);
            for (long long j = 0; j <= LR; ++j) {  // (j = LR: the step's index)
                const long long m = kp * j;
                if (m < 0 || (m & (nlo - 1)) >= nlo || (m >> b) < 0 || (m >> b) >= nhi) {
                    if (!bad++) printf("S=%lld ns=%lld tile=%lld lane=%d: sequence %lld, index %lld of %lld\n", S, ns, tile, t, tg, m >> b, nhi);
                }
            }
        }
    return bad;
}

int main()
{
    using A = SplitCfg<TileCfg<float, 1024, 8, 512, true, true, 16, 16, 4>>;
    using B = SplitCfg<TileCfg<float, 16, 64, 64, true, true, 16>>;
    using D = SplitCfg<TileCfg<double, 320, 12, 240, true, true, 16, 4, 5>>;
    int bad = 0;
    for (long long S : {2LL, 3LL, 16LL, 257LL, 1536LL}) {
        bad += walk<A>(S, S) + walk<B>(S, S) + walk<D>(S, S);
        if (S % 16 == 0) bad += walk<A>(S, S / 16);
    }
    printf(bad ? "%d indexes out of range\n" : "ok\n", bad);
    return bad != 0;
}
