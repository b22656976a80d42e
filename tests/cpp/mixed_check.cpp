// mixed_check.cpp -- the shapes of the run-time mixed-radix tiles, walked on the CPU.
//
// For every length with the factors 2, 3, 5 and 7 up to a tile's limit, both precisions, every
// mode and width: the stages of mixed_kernel.h with the shape's own reciprocals, strides and
// twiddle offsets on an array of the shape's LDS size.  Checked: every index inside its array,
// every element written once per stage and by the threads there are, the workgroup and LDS
// limits, and the transform of three impulses against its closed form.
#include <cmath>
#include <complex>
#include <cstdio>
#include <vector>

#include "../../gfft_amd/csrc/plan_internal.h"

typedef std::complex<double> cd;

static int fails = 0;
#define CHECK(c)                                                                                          \
    do {                                                                                                  \
        if (!(c) && ++fails < 20) printf("FAIL %s: %s (line %d)\n", e.name, #c, __LINE__);                \
    } while (0)

static cd root(long long m, long long n)
{
    const double t = -2.0 * M_PI * (double)(m % n) / (double)n;
    return cd(std::cos(t), std::sin(t));
}

static void check(const TileEntry& e)
{
    const MixShape& m = *e.mix;
    const unsigned L = m.L, tpt = m.tpt;
    CHECK((int)L == e.L && m.nb == (unsigned)e.nb && m.wg == (unsigned)e.wg && m.wg <= 1024 && m.wg % 64 == 0);
    CHECK(m.nb * tpt <= m.wg && e.lds_bytes <= 160 * 1024 && m.nst <= MIX_STAGES && m.nb * L < (1u << 15));
    for (const Div& d : {m.dtpt, m.dr0, m.dl}) CHECK(d.m < (1u << 17));
    for (unsigned x = 0; x < (1u << 15); x += 7) CHECK(m.dl(x) == x / L && m.dr0(x) == x / m.st[0].R);
    CHECK(m.nst == 1 || (size_t)e.lds_bytes == (size_t)m.nb * m.ts * (e.prec == PREC_F64 ? 16 : 8));
    CHECK(!e.loadT || (m.nb & (m.nb - 1)) == 0);
    CHECK(!(e.loadT || e.real) || m.nst >= 2);
    CHECK((e.real != CHIRP_ALL && e.real != CHIRP_TURN) || m.st[0].R == m.st[m.nst - 1].R);
    if (!e.loadT)
        for (unsigned tid = 0; tid < m.wg; ++tid)
            CHECK(m.dtpt(tid) == tid / tpt);
    if (e.loadT && !e.storeT)
        for (unsigned lin = 0; lin < m.nb * L; ++lin) CHECK(m.dl(lin) == lin / L);
    std::vector<cd> in(L, 0), lds(m.ts), out(L);
    const unsigned at[3] = {0, L / 3, L - 1};
    for (int i = 0; i < 3; ++i) in[at[i]] += cd(1.0 + i, 0.5 * i);
    unsigned tw = 0, ns = 1;
    for (unsigned s = 0; s < m.nst; ++s) {
        const MixStage& st = m.st[s];
        const unsigned R = st.R, lr = st.lr, B = MIX_POINTS / R;
        const bool last = s + 1 == m.nst;
        CHECK(R * lr == L && st.ns == ns && (s == 0 || st.tw == tw) && R >= 2 && R <= 16);
        CHECK(B * tpt >= lr);
        std::vector<cd> next(m.ts);
        std::vector<char> hit(m.ts, 0), done(lr, 0);
        for (unsigned jt = 0; jt < tpt; ++jt)
            for (unsigned b = 0; b < B; ++b) {
                const unsigned j = jt + b * tpt;
                if (j >= lr) continue;
                CHECK(!done[j]);
                done[j] = 1;
                CHECK(m.dr0(j) == j / m.st[0].R && st.dns(j) == j / ns && j < (1u << 15));
                const unsigned p = j + (m.dr0(j) & (0u - m.pad)), q = s == 0 ? j : last ? 0 : st.dns(j);
                CHECK(q == j / ns);
                const unsigned k = j - q * ns;
                std::vector<cd> v(R), y(R);
                for (unsigned r = 0; r < R; ++r) {
                    if (s == 0) {
                        v[r] = in[j + r * lr];
                    } else {
                        CHECK(p + r * st.rst < m.ts);
                        CHECK(p + r * st.rst == j + r * lr + m.pad * ((j + r * lr) / m.st[0].R));
                        v[r] = lds[p + r * st.rst] * root((long long)k * r, (long long)ns * R);
                    }
                }
                for (unsigned f = 0; f < R; ++f) {
                    y[f] = 0;
                    for (unsigned r = 0; r < R; ++r) y[f] += v[r] * root(f * r, R);
                }
                for (unsigned r = 0; r < R; ++r) {
                    if (last) {
                        CHECK(j + r * lr < L);
                        out[j + r * lr] = y[r];
                    }
                    if (m.nst == 1) continue;
                    const unsigned w = s == 0 ? j * (R + m.pad) + r : p + q * st.wq + r * st.wst;
                    CHECK(w < m.ts && !hit[w]);
                    const unsigned el = q * ns * R + k + r * ns;  // the Stockham rule
                    CHECK(w == el + m.pad * (el / m.st[0].R));
                    hit[w] = 1;
                    next[w] = y[r];
                }
            }
        for (unsigned j = 0; j < lr; ++j) CHECK(done[j]);
        lds = next;
        if (s) tw += e.prec == PREC_F64 ? ns * (R - 1) : ns;
        ns *= R;
    }
    CHECK(ns == L);
    double worst = 0;
    for (unsigned k = 0; k < L; ++k) {
        cd want = 0;
        for (int i = 0; i < 3; ++i) want += cd(1.0 + i, 0.5 * i) * root((long long)at[i] * k, L);
        worst = std::max(worst, std::abs(out[k] - want));
    }
    CHECK(worst < 1e-11);
}

int main()
{
    size_t tiles = 0, lengths = 0;
    for (int prec = 0; prec < 2; ++prec)
        for (int L = 2; L <= 16384; ++L) {
            bool any = false;
            for (int mode = 0; mode < 9; ++mode) {
                static const int kinds[9] = {REAL_NONE, REAL_NONE, REAL_NONE, REAL_POST, REAL_PRE,
                                             CHIRP_ALL, CHIRP_IN, CHIRP_TURN, CHIRP_OUT};
                const bool storeT = mode == 2 || mode == 8, loadT = storeT || mode == 1 || mode == 6 || mode == 7;
                const int real = kinds[mode];
                if ((real == REAL_POST || real == REAL_PRE) && L % 2) continue;
                for (const TileEntry* e : mix_tiles(prec, L, loadT, storeT, real)) {
                    check(*e);
                    ++tiles;
                    any = true;
                }
            }
            lengths += any;
        }
    printf("%zu tiles of %zu lengths, %d failures\n", tiles, lengths, fails);
    return fails != 0;
}
