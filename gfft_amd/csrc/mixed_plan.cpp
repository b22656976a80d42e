// mixed_plan.cpp -- run-time mixed-radix tiles (mixed_kernel.h): radices and shape of a length,
// and the table entries plans use.
#include "plan_internal.h"

namespace gfftx {
namespace detail {

namespace {

constexpr int kMixRadix[] = {16, 15, 14, 12, 10, 9, 8, 7, 6, 5, 4, 3, 2};

// Instructions of one butterfly of radix R, next to those of its loads, stores and twiddles.
double dft_cost(int R)
{
    switch (R) {
        case 2: return 4;
        case 3: return 14;
        case 4: return 16;
        case 5: return 40;
        case 6: return 40;
        case 7: return 78;
        case 8: return 56;
        case 9: return 84;
        case 10: return 100;
        case 12: return 104;
        case 14: return 184;
        case 15: return 190;
        default: return 168;
    }
}

// Threads per sequence for radices `r`: every stage's butterflies fit the registers.
int threads_for(int L, const std::vector<int>& r)
{
    int tpt = 1;
    for (int R : r) {
        const int b = MIX_POINTS / R;
        tpt = std::max(tpt, (L / R + b - 1) / b);
    }
    return tpt;
}

// Modelled time of a sequence: thread slots of every stage, idle ones included, times the
// instructions of a butterfly (about 17 per point for the LDS, the addresses and the FP64
// twiddle), and 40 per thread for a stage's barriers.
double shape_cost(int L, const std::vector<int>& r)
{
    const int tpt = threads_for(L, r);
    double c = 0;
    for (size_t s = 0; s < r.size(); ++s) {
        const int nb = (L / r[s] + tpt - 1) / tpt;
        c += (double)tpt * (nb * (dft_cost(r[s]) + (s ? 17.0 : 8.0) * r[s]) + 40.0);
    }
    return c;
}

// The radices of length L with the lowest modelled time, at least `least` of them, the largest
// first; empty when L has another prime factor than 2, 3, 5 and 7.
std::vector<int> mix_radices(int L, size_t least)
{
    std::vector<int> best, cur;
    double best_cost = 0;
    std::function<void(int, int)> rec = [&](int rem, int from) {
        if (rem == 1) {
            if (cur.size() < least) return;
            const double c = shape_cost(L, cur);
            if (best.empty() || c < best_cost) {
                best = cur;
                best_cost = c;
            }
            return;
        }
        if (cur.size() == (size_t)MIX_STAGES) return;
        if (!best.empty() && cur.size() > best.size()) return;  // at most one stage more than the best so far
        for (int i = from; i < (int)(sizeof(kMixRadix) / sizeof(int)); ++i) {
            if (rem % kMixRadix[i]) continue;
            cur.push_back(kMixRadix[i]);
            rec(rem / kMixRadix[i], i);
            cur.pop_back();
        }
    };
    rec(L, 0);
    return best;
}

// The same for a chirp-z turn: the first radix and the last one alike.
std::vector<int> turn_radices(int L)
{
    std::vector<int> best;
    double best_cost = 0;
    for (int R : kMixRadix) {
        if (L % (R * R)) continue;
        std::vector<int> r = L == R * R ? std::vector<int>() : mix_radices(L / (R * R), 1);
        if (L != R * R && r.empty()) continue;
        r.insert(r.begin(), R);
        r.push_back(R);
        const double c = shape_cost(L, r);
        if (best.empty() || c < best_cost) {
            best = r;
            best_cost = c;
        }
    }
    return best;
}

Div divisor(unsigned d)
{
    unsigned s = 15;
    while ((1u << (s - 15)) < d) ++s;
    return Div{(unsigned)((1ull << s) / d) + 1, s};
}

struct MixTile {
    TileEntry e;
    MixShape m;
    std::vector<int> radices;
    std::string name;
};

// Fills a tile of `nb` sequences of length L; false when it does not fit a workgroup.
bool fill(MixTile& t, int prec, int L, bool loadT, bool storeT, int real, int nb, const std::vector<int>& r)
{
    const size_t eb = elem_bytes(prec);
    MixShape& m = t.m;
    m = MixShape{};
    t.radices = r;
    m.L = L;
    m.nb = nb;
    m.tpt = threads_for(L, r);
    const unsigned wg = (m.tpt * nb + 63) / 64 * 64;
    if (wg > 1024) return false;
    m.wg = wg;
    m.dtpt = divisor(m.tpt);
    m.pad = r[0] % 2 == 0 ? 1 : 0;  // an odd distance between the runs the first stage writes
    m.dr0 = divisor(r[0]);
    m.dl = divisor(L);
    m.nst = (unsigned)r.size();
    m.ts = L + m.pad * (L / r[0]);
    // lanes that walk sequences are spread over the banks where the LDS has room (8 / nb modulo 8 in FP64,
    // TileCfg::lds_distance).  FP32 keeps 32 / nb modulo 32: 16 / nb modulo 16, the better spread, takes the
    // same time here (15625 to 1440000 points in the same tiles, 0.99 to 1.02 of it)
    const unsigned banks = prec == PREC_F64 ? 8 : 32, odd = m.ts | 1;
    if (loadT && nb >= 2 && (unsigned)nb < banks)
        while (m.ts % banks != banks / nb) ++m.ts;
    else
        m.ts = odd;
    if ((size_t)nb * m.ts * eb > 160 * 1024) m.ts = odd;
    unsigned ns = 1, tw = 0;
    for (size_t s = 0; s < r.size(); ++s) {
        MixStage& st = m.st[s];
        st.R = r[s];
        st.lr = L / r[s];
        st.ns = ns;
        st.dns = divisor(ns);
        st.rst = st.lr + (s ? m.pad * st.lr / r[0] : 0);
        st.wst = s ? ns + m.pad * ns / r[0] : 1;
        st.wq = (st.R - 1) * st.wst;
        st.tw = tw;
        if (s) tw += prec == PREC_F64 ? ns * (r[s] - 1) : ns;
        ns *= r[s];
    }
    // (a CHIRP_ALL tile's L is the convolution length, its input rows are shorter.  Whole lines are not what
    // decides there: non-temporal against plain loads, 8192 x 1009 FP32 on rotating arrays above the
    // Infinity Cache 63.2 and 65.4 us, 32768 x 1009 230 and 238, the same for 1012 and its half lines;
    // with the input in that cache 8192 x 1104, whole lines, 76.6 and 72.9, 8192 x 1009 FP64 129 and 121)
    const size_t row = (loadT ? (size_t)nb : (size_t)nb * L) * eb;
    m.nt_in = row % 128 == 0 ? 1 : 0;
    const size_t lds = r.size() > 1 ? (size_t)nb * m.ts * eb : 0;
    if (lds > 160 * 1024) return false;
    t.e = TileEntry{};
    t.e.prec = prec;
    t.e.L = L;
    t.e.nb = nb;
    t.e.wg = (int)wg;
    t.e.loadT = loadT;
    t.e.storeT = storeT;
    t.e.nrad = (int)r.size();
    t.e.lds_bytes = (int)lds;
    t.e.real = real;
    return true;
}

// Sequences per tile worth trying, the default first.  E->E: workgroups near 256 threads with
// few idle ones, then smaller ones.  T modes: rows of whole 128-byte lines and workgroups of 128
// to 512 threads, then narrower and wider rows.
std::vector<int> tile_widths(int prec, int L, bool loadT, const std::vector<int>& r)
{
    const int tpt = threads_for(L, r);
    std::vector<int> out;
    auto add = [&](int nb) {
        if (nb >= 1 && std::find(out.begin(), out.end(), nb) == out.end()) out.push_back(nb);
    };
    if (!loadT) {
        for (int most : {256, 128, 512}) {
            // the fullest workgroup of at most `most` threads (a single sequence may need more)
            int best = 1;
            double eff = 0;
            for (int nb = std::max(1, most / tpt); nb >= 1 && nb * tpt * 2 > most; --nb) {
                const int th = nb * tpt;
                const double e = (double)th / ((th + 63) / 64 * 64);
                if (e > eff + 0.02) {
                    eff = e;
                    best = nb;
                }
            }
            add(best);
        }
        return out;
    }
    const int line = 128 / (int)elem_bytes(prec);
    int nb = line;
    while (nb * tpt < 128) nb *= 2;
    while (nb > line / 4 && (nb * tpt > 1024 || (size_t)nb * (L + L / r[0] + 1) * elem_bytes(prec) > 160 * 1024)) nb /= 2;
    add(nb);
    if (nb * 2 * tpt <= 512) add(nb * 2);
    if (nb / 2 >= line / 4) add(nb / 2);  // narrower: more workgroups for transforms of a few points
    if (nb / 4 >= line / 4) add(nb / 4);
    return out;
}

std::mutex g_mix_mu;
// Every tile made so far; entries live as long as the library (plans point to them), one list
// for each of the lengths, modes and precisions used.
std::map<std::vector<int>, std::vector<MixTile*>> g_mix;

const std::vector<MixTile*>& tiles_locked(int prec, int L, bool loadT, bool storeT, int real)
{
    const std::vector<int> key = {prec, L, loadT, storeT, real};
    auto it = g_mix.find(key);
    if (it != g_mix.end()) return it->second;
    std::vector<MixTile*> v;
    const std::vector<int> r = real == CHIRP_ALL || real == CHIRP_TURN ? turn_radices(L)
                                                                       : mix_radices(L, loadT || real != REAL_NONE ? 2 : 1);
    if (!r.empty())
        for (int nb : tile_widths(prec, L, loadT, r)) {
            MixTile* t = new MixTile();
            if (!fill(*t, prec, L, loadT, storeT, real, nb, r)) {
                delete t;
                continue;
            }
            char buf[96];
            snprintf(buf, sizeof(buf), "mixed_%s_L%d_nb%d_wg%d_%s", prec == PREC_F64 ? "double" : "float", L, nb, t->e.wg,
                     real == CHIRP_ALL    ? "chirp"
                     : real == CHIRP_IN   ? "chirp_in"
                     : real == CHIRP_TURN ? "chirp_turn"
                     : real == CHIRP_OUT  ? "chirp_out"
                     : loadT              ? (storeT ? "truetrue" : "truefalse")
                     : real == REAL_POST  ? "e_split"
                     : real == REAL_PRE   ? "e_presplit"
                                          : "falsefalse");
            t->name = buf;
            t->e.name = t->name.c_str();
            t->e.radices = t->radices.data();
            t->e.mix = &t->m;
            v.push_back(t);
        }
    return g_mix[key] = v;
}

}  // namespace

// Largest length of a run-time tile: 16 points for each of 1024 threads and the LDS for a single
// pass; as a pass, rows of at least 32 bytes.
int mix_max(int prec, bool loadT) { return prec == PREC_F64 ? (loadT ? 2048 : 8192) : (loadT ? 4096 : 16384); }

std::vector<const TileEntry*> mix_tiles(int prec, int L, bool loadT, bool storeT, int real)
{
    std::vector<const TileEntry*> out;
    if (L < 2 || L > mix_max(prec, loadT) || (storeT && !loadT)) return out;
    if (loadT && (real == REAL_POST || real == REAL_PRE)) return out;
    int rest = L;
    for (int f : {2, 3, 5, 7})
        while (rest % f == 0) rest /= f;
    if (rest != 1) return out;
    std::lock_guard<std::mutex> lk(g_mix_mu);
    for (MixTile* t : tiles_locked(prec, L, loadT, storeT, real)) out.push_back(&t->e);
    return out;
}

// Modelled time of one of a tile's sequences (shape_cost).
double mix_cost(const TileEntry& e) { return shape_cost(e.L, std::vector<int>(e.radices, e.radices + e.nrad)); }

// Stage twiddles of a run-time tile: FP32 the FP64 roots W_{Ns R}^k (k < Ns) of every later
// stage, FP64 the rows W_{Ns R}^{k r}, r = 1..R-1, each contiguous in k.
int upload_mix_table(std::vector<void*>& owned, const TileEntry& k, void** out)
{
    *out = nullptr;
    std::vector<double> t;
    long long ns = k.radices[0];
    for (int s = 1; s < k.nrad; ++s) {
        const long long R = k.radices[s];
        const auto w = all_roots(ns * R);
        for (long long r = 1; r < (k.prec == PREC_F64 ? R : 2); ++r)
            for (long long kk = 0; kk < ns; ++kk) {
                t.push_back((double)w[kk * r].first);
                t.push_back((double)w[kk * r].second);
            }
        ns *= R;
    }
    if (t.empty()) return GFFTX_SUCCESS;
    const int rc = dev_alloc_list(owned, out, t.size() * sizeof(double));
    if (rc) return rc;
    HIP_TRY(hipMemcpy(*out, t.data(), t.size() * sizeof(double), hipMemcpyHostToDevice));
    return GFFTX_SUCCESS;
}

// Stage twiddles of any tile, and the launch limits of a run-time one.
int upload_tile_table(std::vector<void*>& owned, const TileEntry* k, void** out)
{
    if (!k->mix) return upload_stage_table_r(owned, k->prec, k->nrad, k->radices, out);
    HIP_TRY(mixed_prepare(*k));
    return upload_mix_table(owned, *k, out);
}

}  // namespace detail
}  // namespace gfftx
