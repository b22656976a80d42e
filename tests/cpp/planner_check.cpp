// planner_check.cpp -- the planner's choices, on the CPU.
//
//   - the split an untuned plan takes is one of those measured within 15% of the fastest of its
//     length on an MI355X (back to back, three pairs of arrays), complex and real transforms;
//   - the search for the best few splits finds what listing them all would;
//   - the splits a tuned plan times include those;
//   - passes store the way that was measured fastest for their kind, rows and size;
//   - the autotuner's repeated in-place transforms stay in the range of their numbers;
//   - the lanes of one LDS cycle meet distinct banks in the pass tiles;
//   - describe() names a tuned choice in full;
//   - twiddle tables and the table of an unfused real split hold the roots, bit for bit;
//   - a length runs natively exactly where a tile or a split exists.
#include <cstdio>
#include <functional>

#include "../../gfft_amd/csrc/plan_internal.h"

static int fails = 0;

typedef std::vector<std::vector<int>> Splits;

static std::string text(const std::vector<int>& v)
{
    std::string s;
    for (int x : v) s += (s.empty() ? "" : "*") + std::to_string(x);
    return s;
}

static const RealPart kComplex{}, kForward{REAL_POST, false}, kInverse{REAL_PRE, true};

static void fast(RealPart real, int prec, unsigned long long n, const Splits& good)
{
    std::vector<int> l;
    if (!choose_passes(prec, n, l, 1, 256, real) || std::find(good.begin(), good.end(), l) == good.end()) {
        printf("FAIL real %d prec %d n %llu: %s is not among the fast splits\n", real.kind, prec, n, text(l).c_str());
        ++fails;
    }
}

// Store kind of pass i of the split `lens` for n points, one item.
static void store(int want, RealPart real, int prec, unsigned long long n, const std::vector<int>& lens, size_t i, bool nt = false)
{
    unsigned long long ns = 1;
    for (size_t j = 0; j < i; ++j) ns *= (unsigned long long)lens[j];
    Pass ps;
    ps.k = pass_tile(prec, lens[i], ns, n, 1, 256);
    if (real.kind == REAL_POST ? i + 1 == lens.size() : real.kind == REAL_PRE && i == 0) ps.k = find_real_tile(ps.k, real.kind);
    ps.ns_pass = (long long)ns;
    const int got = !ps.k ? -1 : pass_store(true, nt, i, lens.size(), (size_t)n * elem_bytes(prec), ps, (size_t)n, 1);
    if (got != want || (ps.k && pass_store(false, false, i, lens.size(), (size_t)n * elem_bytes(prec), ps, (size_t)n, 1) != STORE_PLAIN)) {
        printf("FAIL real %d prec %d n %llu %s pass %zu: store %d, not %d\n", real.kind, prec, n, text(lens).c_str(), i, got, want);
        ++fails;
    }
}

// LDS cycles of a T-mode pass tile: `lanes` lanes in a row (one cycle's: 128 bytes), NB of them on one element of
// NB sequences, the next ones on the element `step` further; their places modulo the banks differ.
static bool spread(int prec, int nb, unsigned ts, const std::function<unsigned(unsigned)>& place, unsigned step)
{
    const unsigned lanes = prec == PREC_F64 ? 8 : 16;
    for (unsigned j0 = 0; j0 < 4; ++j0) {
        std::vector<char> hit(lanes, 0);
        for (unsigned l = 0; l < lanes; ++l) {
            const unsigned lane = j0 * lanes + l, p = lane % nb * ts + place(lane / nb * step);
            if (hit[p % lanes]++) return false;
        }
    }
    return true;
}

template <class C> static void spread_tile()
{
    auto place = [](unsigned e) { return e + (e >> C::PADSH); };
    if (!spread(sizeof(typename C::T) == 8 ? PREC_F64 : PREC_F32, C::NB, C::TS, place, 1) ||
        !spread(sizeof(typename C::T) == 8 ? PREC_F64 : PREC_F32, C::NB, C::TS, place, C::R[0])) {
        printf("FAIL banks of L %d nb %d ts %d\n", C::L, C::NB, C::TS);
        ++fails;
    }
}

static bool smooth(unsigned long long n)
{
    for (int f : {2, 3, 5, 7})
        while (n % f == 0) n /= f;
    return n == 1;
}

int main()
{
    unsetenv("GFFTX_PASSES");
    const int F64 = PREC_F64, F32 = PREC_F32;
    // (the fastest time, and a slow split for comparison)
    fast(kComplex, F64, 32768, {{128, 16, 16}, {256, 16, 8}, {256, 128}, {1024, 32}});       // 11.1 us; 32*32*32 16.8
    fast(kComplex, F32, 32768, {{128, 16, 16}, {256, 16, 8}, {256, 128}});                   // 9.8; 32*32*32 16.6
    fast(kComplex, F64, 65536, {{256, 16, 16}, {256, 256}, {1024, 64}});                     // 11.4; 2048*32 16.3
    fast(kComplex, F64, 262144, {{256, 64, 16}, {1024, 16, 16}, {1024, 256}});               // 13.2; 512*512 18.9
    fast(kComplex, F32, 262144, {{128, 128, 16}, {256, 64, 16}, {256, 256, 4}, {1024, 16, 16}, {1024, 256}});  // 12.4; 512*512 15.2
    fast(kComplex, F64, 393216, {{192, 128, 16}, {256, 96, 16}, {768, 512}, {1024, 384}, {1536, 256}});  // 16.4; 384*32*32 23.0
    fast(kForward, F64, 32768, {{128, 16, 16}, {256, 16, 8}, {1024, 32}, {2048, 16}});       // 14.3; 32*32*32 19.3
    fast(kForward, F32, 32768, {{128, 16, 16}, {256, 16, 8}, {256, 128}, {1024, 32}});       // 13.2; 32*32*32 19.0
    fast(kForward, F64, 65536, {{256, 16, 16}, {256, 256}, {1024, 64}, {4096, 16}});         // 15.2; 2048*32 19.0
    fast(kForward, F64, 262144, {{128, 128, 16}, {256, 64, 16}, {1024, 16, 16}, {1024, 256}});  // 17.0; 512*512 22.3
    fast(kForward, F64, 196608, {{192, 64, 16}, {256, 96, 8}, {768, 256}, {1024, 192}, {1536, 128}});  // 17.5; 512*384 21.7
    fast(kForward, F32, 1572864, {{192, 128, 64}, {256, 96, 64}, {256, 128, 48}, {384, 256, 16}, {1536, 64, 16}, {1536, 1024}});  // 25.0; 256*128*48 31.0
    fast(kInverse, F64, 32768, {{128, 16, 16}, {256, 16, 8}, {256, 128}, {512, 64}, {1024, 32}});  // 16.1; 32*32*32 21.5
    fast(kInverse, F32, 32768, {{128, 16, 16}, {256, 16, 8}, {256, 128}, {512, 64}});        // 14.3; 32*32*32 21.1
    fast(kInverse, F64, 65536, {{256, 16, 16}, {256, 256}, {512, 128}, {1024, 64}});         // 16.3; 2048*32 23.0
    fast(kInverse, F32, 65536, {{256, 16, 16}, {256, 256}, {512, 128}, {1024, 64}});         // 14.7; 4096*16 21.0
    fast(kInverse, F64, 262144, {{256, 64, 16}, {256, 256, 4}, {1024, 16, 16}, {1024, 256}});  // 21.5; 512*512 27.0
    fast(kInverse, F64, 393216, {{128, 64, 48}, {256, 96, 16}, {256, 192, 8}, {1024, 384}});  // 24.0; 384*32*32 33.5
    // the split's own pass is part of the price: where the array is large, it rides in a pass
    for (int prec : {F64, F32})
        for (unsigned long long n = 1 << 20; n <= 1 << 24; n *= 2)
            for (const RealPart& real : {kForward, kInverse}) {
                std::vector<int> l;
                choose_passes(prec, n, l, 1, 256, real);
                const bool post = real.kind == REAL_POST;
                const TileEntry* k = l.empty() ? nullptr : pass_tile(prec, post ? l.back() : l[0], post ? n / l.back() : 1, n, 1, 256);
                if (!k || !find_real_tile(k, real.kind)) {
                    printf("FAIL real %d prec %d n %llu: %s leaves the split to a kernel of its own\n", real.kind, prec, n, text(l).c_str());
                    ++fails;
                }
            }
    // the autotuner gets to time the splits that are fast with tiles other than the default ones, the ones
    // of few passes and, of a real transform, those of its passes alone
    const struct {
        RealPart real;
        unsigned long long n;
        std::vector<int> split;
    } timed[] = {{kComplex, 32768, {4096, 8}}, {kComplex, 12288, {4096, 3}}, {kComplex, 393216, {1536, 256}}, {kComplex, 480000, {1280, 375}},
                 {kForward, 131072, {1024, 128}}, {kForward, 262144, {1024, 256}}, {kForward, 393216, {1536, 256}}, {kInverse, 393216, {1536, 256}}};
    for (const auto& x : timed) {
        const Splits v = tuned_splits(F32, x.n, 5, 1, 256, x.real);
        if (std::find(v.begin(), v.end(), x.split) == v.end()) {
            printf("FAIL real %d n %llu: %s is not timed\n", x.real.kind, x.n, text(x.split).c_str());
            ++fails;
        }
    }
    // forward splits: half rows of 128 bytes and more through the L2 to 64 MiB, of 64 to 16, shorter ones never
    store(STORE_THROUGH, kForward, F32, 3 << 19, {256, 96, 64}, 2);
    store(STORE_THROUGH, kForward, F32, 1 << 22, {256, 256, 64}, 2);
    store(STORE_THROUGH, kForward, F64, 1 << 21, {128, 128, 128}, 2);
    store(STORE_THROUGH, kForward, F32, 1 << 18, {1024, 256}, 1);
    store(STORE_PLAIN, kForward, F32, 1 << 17, {1024, 128}, 1);
    store(STORE_PLAIN, kForward, F32, 1 << 24, {256, 256, 256}, 2);
    store(STORE_PLAIN, kForward, F64, 1 << 20, {1024, 1024}, 1);
    // at the end of a call above the Infinity Cache: non-temporally with half rows of 256 bytes
    store(STORE_PLAIN, kForward, F64, 1 << 24, {256, 256, 256}, 2, true);
    store(STORE_PLAIN, kForward, F32, 1 << 26, {1024, 512, 128}, 2, true);
    store(STORE_NT, kForward, F64, 1 << 25, {1024, 256, 128}, 2, true);
    store(STORE_NT, kForward, F32, 1 << 26, {1024, 1024, 64}, 2, true);
    store(STORE_NT, kComplex, F32, 1 << 26, {1024, 512, 128}, 2, true);
    // inverse splits: from 12 (FP64 16) to 32 MiB
    store(STORE_PLAIN, kInverse, F32, 1 << 18, {1024, 256}, 0);
    store(STORE_PLAIN, kInverse, F64, 1 << 17, {1024, 128}, 0);
    store(STORE_PLAIN, kInverse, F32, 1 << 20, {256, 64, 64}, 0);
    store(STORE_THROUGH, kInverse, F32, 3 << 19, {256, 96, 64}, 0);
    store(STORE_THROUGH, kInverse, F32, 1 << 22, {256, 256, 64}, 0);
    store(STORE_PLAIN, kInverse, F32, 1 << 23, {256, 256, 128}, 0);
    store(STORE_PLAIN, kInverse, F64, 1 << 19, {256, 128, 16}, 0);
    store(STORE_THROUGH, kInverse, F64, 1 << 21, {256, 128, 64}, 0);
    store(STORE_PLAIN, kInverse, F64, 1 << 22, {256, 256, 64}, 0);
    store(STORE_THROUGH, kInverse, F64, 1 << 21, {256, 128, 64}, 1);
    // complex passes: from 2 MiB, rows below 64 bytes from 8, whole lines to 64 MiB
    store(STORE_THROUGH, kComplex, F64, 1 << 17, {1024, 128}, 0);
    store(STORE_PLAIN, kComplex, F32, 1 << 17, {1024, 128}, 0);
    store(STORE_THROUGH, kComplex, F32, 1 << 23, {256, 256, 128}, 2);
    store(STORE_PLAIN, kComplex, F64, 1 << 23, {256, 256, 128}, 2);
    store(STORE_PLAIN, kComplex, F32, 3 << 20, {256, 192, 64}, 1);
    // in-place timing stays in the range of its numbers (27 bits of FP32's, 123 of FP64's kept clear)
    for (unsigned long long n = 2; n <= 1ull << 28; n = n * 5 / 3 + 1)
        for (int prec : {F64, F32}) {
            const int r = fill_reps(prec, n);
            if (r < 1 || r * std::log2(2.0 * (double)n) / 2 > (prec == F64 ? 900 : 100)) {
                printf("FAIL prec %d n %llu: %d transforms in place\n", prec, n, r);
                ++fails;
            }
        }
    // a choice keeps the run-time tiles it was timed with: the default one changes with the items
    {
        const std::vector<int> one = with_tiles(F32, 40000, 1, 256, {200, 200}), many = with_tiles(F32, 40000, 256, 256, {200, 200});
        const TileEntry *a = pass_tile(F32, 200, 1, 40000, 1, 256), *b = pass_tile(F32, 200, 1, 40000, 256, 256);
        if (one.size() != 7 || one[2] != 0 || one[3] != a->nb || one[4] != a->wg || many[3] != b->nb || many[4] != b->wg || a == b ||
            with_tiles(F32, 1 << 18, 1, 256, {1024, 256}) != std::vector<int>({1024, 256, 0, 0, 0, 0, 0}) ||
            with_tiles(F32, 1000, 1, 256, {1000, 1, 0, 2, 256}) != std::vector<int>({1000, 1, 0, 2, 256}) ||
            with_tiles(F32, 1000000, 1, 256, {1000, 1000, 0, 8, 832, 4, 448}) != std::vector<int>({1000, 1000, 0, 8, 832, 4, 448})) {
            printf("FAIL with_tiles\n");
            ++fails;
        }
    }
    // choices of a cache file that are no split of n
    if (!passes_fit({512, 256}, 1 << 17) || passes_fit({512, 256}, 1 << 18) || passes_fit({1 << 17, 1}, 1 << 17) || passes_fit({1 << 17}, 1 << 17) ||
        passes_fit({}, 1) || passes_fit({65536, 65536, 65536, 65536, 65536}, 1 << 16)) {
        printf("FAIL passes_fit\n");
        ++fails;
    }
    // a cycle's lanes of a pass tile meet distinct banks
    spread_tile<TileCfg<float, 256, 16, 256, true, true, 16, 16>>();
    spread_tile<TileCfg<float, 256, 8, 128, true, true, 16, 16>>();
    spread_tile<TileCfg<float, 192, 16, 192, true, true, 16, 4, 3>>();
    spread_tile<TileCfg<float, 128, 32, 256, true, true, 16, 8>>();
    spread_tile<TileCfg<float, 1024, 8, 512, true, true, 16, 16, 4>>();
    spread_tile<TileCfg<float, 1024, 8, 1024, true, true, 8, 8, 8, 2>>();
    spread_tile<TileCfg<float, 1024, 4, 256, true, false, 16, 16, 4>>();
    spread_tile<TileCfg<float, 1536, 4, 768, true, false, 8, 8, 8, 3>>();
    spread_tile<TileCfg<float, 4096, 2, 512, true, false, 16, 16, 16>>();
    spread_tile<TileCfg<float, 4096, 4, 1024, true, false, 16, 16, 16>>();
    spread_tile<TileCfg<double, 1024, 4, 256, true, true, 16, 16, 4>>();
    spread_tile<TileCfg<double, 256, 16, 256, true, true, 16, 16>>();
    spread_tile<TileCfg<double, 4096, 2, 512, true, false, 16, 16, 16>>();
    for (int L : {96, 250, 384, 500, 512, 1000, 1250})
        for (const TileEntry* k : mix_tiles(F64, L, true, true))
            if ((size_t)k->nb * k->mix->ts * elem_bytes(F64) <= 150 * 1024 &&
                !spread(F64, k->nb, k->mix->ts, [](unsigned e) { return e; }, 1)) {
                printf("FAIL banks of %s ts %u\n", k->name, k->mix->ts);
                ++fails;
            }
    // a choice's name shows every pass with its own tile
    const struct {
        std::vector<int> c;
        bool chirp;
        const char* want;
    } names[] = {{{1000, 1, 0, 2, 256}, false, "single/2-256"},
                 {{512, 256}, false, "512x256"},
                 {{512, 256, 0, 4, 128, 0, 0}, false, "512/4-128x256"},
                 {{2048, 1, 0, 1, 128}, true, "2048: single/1-128"},
                 {{131220, 324, 405, 0, 2, 128, 4, 64, 2, 192}, true, "131220: 324/2-128x405/4-64x324/2-192"},
                 {{8388608, 128, 256, 256, 0, 16, 128, 16, 256, 8, 129, 16, 512, 32, 64}, true,
                  "8388608: 128/16-128x256/16-256x256/8-129x256/16-512x128/32-64"}};
    for (const auto& x : names)
        if (choice_label(x.c, x.chirp) != x.want) {
            printf("FAIL label %s, not %s\n", choice_label(x.c, x.chirp).c_str(), x.want);
            ++fails;
        }
    // the roots of a table, folded out of the first octant or not, are the evaluated ones
    for (long long N : {1ll, 2ll, 6ll, 8ll, 15ll, 16ll, 24ll, 40ll, 100ll, 256ll, 1000ll, 1536ll, 4096ll, 10000ll, 16384ll}) {
        const auto w = all_roots(N);
        bool ok = w.size() == (size_t)N;
        for (long long m = 0; ok && m < N; ++m) {
            long double c, s, c2, s2;
            root_ld(m, N, &c, &s);
            root_ld(m * 64, N * 64, &c2, &s2);  // (and a power of two scales out)
            ok = w[m].first == c && w[m].second == s && c2 == c && s2 == s;
        }
        if (!ok) {
            printf("FAIL roots of order %lld\n", N);
            ++fails;
        }
    }
    // the split table's mirrored and shared-out entries are the roots themselves
    for (long long n : {2ll, 4ll, 6ll, 10ll, 12ll, 98ll, 1000ll, 4096ll, 200000ll, 524290ll}) {
        const std::vector<float> f = split_roots<float>(n);
        const std::vector<double> d = split_roots<double>(n);
        bool ok = f.size() == (size_t)n + 2 && d.size() == (size_t)n + 2;
        for (long long k = 0; ok && k <= n / 2; ++k) {
            long double c, s;
            root_ld(k, 2 * n, &c, &s);
            ok = f[2 * k] == (float)c && f[2 * k + 1] == (float)s && d[2 * k] == (double)c && d[2 * k + 1] == (double)s;
        }
        if (!ok) {
            printf("FAIL split table of %lld\n", n);
            ++fails;
        }
    }
    // pruned search against the full list
    for (unsigned long long n : {4096ull, 20000ull, 44100ull, 362880ull, 1ull << 20, 3628800ull, 12700800ull})
        for (int prec : {F64, F32})
            for (const RealPart& real : {kComplex, kForward, kInverse}) {
                Splits all = candidate_passes(prec, n, 1000000, 1, 256, true, real), some = candidate_passes(prec, n, 5, 1, 256, true, real);
                all.resize(std::min<size_t>(all.size(), 5));
                if (all != some) {
                    printf("FAIL prec %d n %llu: the best five differ\n", prec, n);
                    ++fails;
                }
            }
    for (int prec : {F64, F32}) {
        for (unsigned long long n = 1; n <= 4000; ++n) {
            const bool want = find_tile(prec, (int)n, false, false) || !candidate_passes(prec, n, 1).empty();
            if (native_length(prec, n) != want || (n > 1 && want != smooth(n))) {
                printf("FAIL prec %d n %llu: native %d\n", prec, n, (int)native_length(prec, n));
                ++fails;
            }
        }
        for (unsigned long long n : {1ull << 28, 203212800ull, 127008000ull, 1000000ull, 1000003ull, 2097143ull, 282475249ull, 11ull << 20})
            if (native_length(prec, n) != !candidate_passes(prec, n, 1).empty()) {
                printf("FAIL prec %d n %llu: native %d\n", prec, n, (int)native_length(prec, n));
                ++fails;
            }
    }
    printf("%d failures\n", fails);
    return fails != 0;
}
