// chirp_plan.cpp -- chirp-z (Bluestein) transforms: convolution length, passes, tables and
// execution, for lengths with a prime factor above 7.
//
// With c_j = W_{2n}^{j^2}, X_k = c_k sum_j (x_j c_j) conj(c_{k-j}): a linear convolution, computed
// as a circular one of length m >= 2n - 1.  The products by the chirp and by the filter's spectrum
// ride in the passes of the two length-m transforms (mixed_kernel.h, CHIRP_*): up to 8192 points
// one kernel does it all in the LDS; longer ones take 2k - 1 passes for a split of m into k, the
// last forward pass and the first backward one being one kernel.
#include "plan_internal.h"

namespace gfftx {
namespace detail {

namespace {

// Longest convolution one tile takes.
constexpr unsigned long long kChirpTile = 8192;

// The products of 2, 3, 5 and 7 in [lo, hi], ascending.
std::vector<unsigned long long> smooth_between(unsigned long long lo, unsigned long long hi)
{
    std::vector<unsigned long long> v;
    for (unsigned long long a = 1; a <= hi; a *= 2)
        for (unsigned long long b = a; b <= hi; b *= 3)
            for (unsigned long long c = b; c <= hi; c *= 5)
                for (unsigned long long d = c; d <= hi; d *= 7)
                    if (d >= lo) v.push_back(d);
    std::sort(v.begin(), v.end());
    return v;
}

struct Choice {
    unsigned long long m = 0;
    std::vector<const TileEntry*> tiles;  // one CHIRP_ALL tile, or the 2k - 1 passes in order
    double cost = 0;                      // modelled
};

// The kind of pass i of np, and the tiles it can take for length L.
std::vector<const TileEntry*> pass_tiles(int prec, int L, size_t i, size_t np)
{
    if (np == 1) return mix_tiles(prec, L, false, false, CHIRP_ALL);
    if (i == 0) return mix_tiles(prec, L, true, false, CHIRP_IN);
    if (i + 1 == np) return mix_tiles(prec, L, true, true, CHIRP_OUT);
    if (i == np / 2) return mix_tiles(prec, L, true, false, CHIRP_TURN);
    return tile_shapes(prec, L, true, true);
}

// One-tile choices, by the modelled work per sequence (two transforms of m points, idle threads
// included; where the tiles leave CUs idle, narrow ones first).
void one_tile(int prec, unsigned long long n, unsigned long long batch, int cus, std::vector<Choice>& out)
{
    const unsigned long long lo = 2 * n - 1;
    for (unsigned long long m : smooth_between(lo, std::min(kChirpTile, 2 * lo)))
        for (const TileEntry* e : pass_tiles(prec, (int)m, 0, 1)) {
            const double used = std::min<double>((double)batch, e->nb);
            const bool few = (double)batch <= (double)e->nb * cus;
            Choice c;
            c.m = m;
            c.tiles = {e};
            c.cost = mix_cost(*e) * (double)e->wg / (used * e->mix->tpt) * (few ? 1.0 + 0.05 * e->nb : 1.0);
            out.push_back(c);
        }
}

// Modelled time (us) of one chirp-z pass by tile `k` over `batch` items of m points: 2.5 us of launch,
// and either the bytes at the bandwidth the tile reaches (less for a run-time tile and for rows below a
// 128-byte line) or, when there is little to move, the time of one tile, 1.5 us and 0.12 us per KB, for
// each round of tiles the device holds at once.  (The chirp's and the filter's loads weigh on a
// tile as its own bytes do, which the fit of pass_cost() to plain passes does not know.)
double chirp_cost(const TileEntry* k, unsigned long long m, unsigned long long batch, int cus)
{
    const int by_lds = k->lds_bytes > 0 ? (160 * 1024) / k->lds_bytes : 8;
    const int per_cu = std::max(1, std::min(by_lds, 2048 / k->wg));
    const double tiles = std::ceil((double)(m / (unsigned long long)k->L) / k->nb) * (double)batch;
    const double rounds = std::ceil(tiles / ((double)cus * per_cu));
    const double kb = (double)k->nb * k->L * elem_bytes(k->prec) / 1024.0;
    const double row = (double)k->nb * elem_bytes(k->prec);
    const double bw = pass_bandwidth(k->prec, k->L) * (k->mix ? 0.9 : 1.0) * (row >= 128 ? 1.0 : row >= 64 ? 0.9 : 0.7);
    const double move = 2.0 * (double)m * (double)batch * elem_bytes(k->prec) / (bw * 1e6);
    return 2.5 + std::max(move, rounds * (1.5 + 0.12 * kb));
}

// Splits of m into two or three passes.
void splits(int prec, unsigned long long m, unsigned long long batch, int cus, std::vector<Choice>& out)
{
    struct Len {
        int L;
        const TileEntry* t[4];  // in, middle, turn, out: the cheapest of each kind (or null)
        double c[4];
    };
    std::vector<Len> len;
    for (unsigned long long d : smooth_between(17, (unsigned long long)mix_max(prec, true))) {
        if (m % d) continue;
        Len l{};
        l.L = (int)d;
        for (int kind = 0; kind < 4; ++kind) {
            for (const TileEntry* k : pass_tiles(prec, l.L, kind == 3 ? 4 : kind, 5)) {
                const double c = chirp_cost(k, m, batch, cus) * (kind == 2 ? 1.5 : 1.0);  // the turn: two transforms
                if (l.t[kind] && c >= l.c[kind]) continue;
                l.t[kind] = k;
                l.c[kind] = c;
            }
        }
        len.push_back(l);
    }
    for (const Len& a : len) {
        if (!a.t[0] || !a.t[3]) continue;
        for (const Len& z : len) {
            if (!z.t[2] || (m / a.L) % z.L) continue;
            const unsigned long long rest = m / a.L / z.L;
            Choice c;
            c.m = m;
            c.cost = a.c[0] + a.c[3] + z.c[2];
            if (rest == 1) {
                c.tiles = {a.t[0], z.t[2], a.t[3]};
                out.push_back(c);
                continue;
            }
            for (const Len& b : len)
                if (b.t[1] && (unsigned long long)b.L == rest) {
                    c.cost += 2 * b.c[1];
                    c.tiles = {a.t[0], b.t[1], z.t[2], b.t[1], a.t[3]};
                    out.push_back(c);
                }
        }
    }
}

// The `k` cheapest choices by the model.
std::vector<Choice> choices(int prec, unsigned long long n, unsigned long long batch, int cus, size_t k)
{
    const unsigned long long lo = 2 * n - 1, maxm = bluestein_max_m(prec);
    std::vector<Choice> v;
    if (lo <= kChirpTile) one_tile(prec, n, batch, cus, v);
    // lengths well above the shortest only where nothing nearer splits
    if (v.empty())
        for (unsigned long long hi : {lo + lo / 24, lo + lo / 4, 2 * lo}) {
            for (unsigned long long m : smooth_between(lo, std::min(hi, maxm))) splits(prec, m, batch, cus, v);
            if (!v.empty()) break;
        }
    std::stable_sort(v.begin(), v.end(), [](const Choice& x, const Choice& y) { return x.cost < y.cost; });
    if (v.size() > k) v.resize(k);
    return v;
}

// A choice as the tuning cache keeps it: [m, 1, 0, nb, wg] for one tile, else
// [m, P_0, .., P_k-1, 0, nb, wg of every pass].
std::vector<int> encode(const Choice& c)
{
    std::vector<int> v = {(int)c.m};
    const size_t np = c.tiles.size();
    if (np == 1) v.push_back(1);
    else
        for (size_t i = 0; i <= np / 2; ++i) v.push_back(c.tiles[i]->L);
    v.push_back(0);
    for (const TileEntry* k : c.tiles) {
        v.push_back(k->nb);
        v.push_back(k->wg);
    }
    return v;
}

// The choice a cache entry names; m is 0 when it does not fit n or has no such tiles.
Choice decode(int prec, unsigned long long n, const std::vector<int>& v)
{
    std::vector<int> lens;
    std::vector<std::pair<int, int>> shape;
    split_choice(v, lens, shape);
    Choice c;
    if (lens.size() < 2 || (unsigned long long)lens[0] < 2 * n - 1) return c;
    const bool one = lens.size() == 2 && lens[1] == 1;
    const size_t k = lens.size() - 1, np = one ? 1 : 2 * k - 1;
    if (shape.size() != np || (!one && (k < 2 || k > 3))) return c;
    unsigned long long prod = 1;
    for (size_t i = 0; i < np; ++i) {
        const int L = one ? lens[0] : lens[1 + (i < k ? i : 2 * k - 2 - i)];
        if (i < k) prod *= (unsigned long long)L;
        const TileEntry* t = nullptr;
        for (const TileEntry* e : pass_tiles(prec, L, i, np))
            if (e->nb == shape[i].first && e->wg == shape[i].second) t = e;
        if (!t) return Choice();
        c.tiles.push_back(t);
    }
    if (prod == (unsigned long long)lens[0]) c.m = prod;
    return c;
}

}  // namespace

// Choices for the autotuner to time, the model's favourite first.
std::vector<std::vector<int>> chirp_candidates(int prec, unsigned long long n, unsigned long long batch, int cus, size_t k)
{
    std::vector<std::vector<int>> out;
    for (const Choice& c : choices(prec, n, batch, cus, k)) out.push_back(encode(c));
    return out;
}

// A choice of several passes with every other tile shape at pass `i`.
std::vector<std::vector<int>> chirp_variants(int prec, unsigned long long n, const std::vector<int>& v, size_t i)
{
    std::vector<std::vector<int>> out;
    const Choice c = decode(prec, n, v);
    if (!c.m || i >= c.tiles.size() || c.tiles.size() == 1) return out;
    for (const TileEntry* e : pass_tiles(prec, c.tiles[i]->L, i, c.tiles.size())) {
        if (e == c.tiles[i]) continue;
        Choice d = c;
        d.tiles[i] = e;
        out.push_back(encode(d));
    }
    return out;
}

// Largest convolution length of the chirp-z path: the multi-pass limit of the precision.
unsigned long long bluestein_max_m(int prec) { return prec == PREC_F64 ? (1ull << 26) : (1ull << 28); }

int build_bluestein(gfftx_plan_s* p)
{
    const unsigned long long n = p->n;
    if (p->flags & GFFTX_FLAG_SPLIT_MFMA)
        return fail(GFFTX_ERR_UNSUPPORTED, "split-precision MFMA path: FP32 C2C of length 256 or 4096 only (n=%llu)", n);
    if (n < 2 || 2 * n - 1 > bluestein_max_m(p->prec))
        return fail(GFFTX_ERR_UNSUPPORTED, "length %llu with a prime factor above 7: the chirp-z path takes 2 <= n <= %llu",
                    n, (bluestein_max_m(p->prec) + 1) / 2);
    Choice ch;
    if (!p->forced_lens.empty()) ch = decode(p->prec, n, p->forced_lens);
    if (!ch.m) {
        const std::vector<Choice> v = choices(p->prec, n, p->batch, device_cus(p->device), 1);
        if (!v.empty()) ch = v[0];
    }
    if (!ch.m) return fail(GFFTX_ERR_UNSUPPORTED, "no convolution length for n=%llu", n);
    const unsigned long long m = p->blue_m = ch.m;
    const size_t eb = elem_bytes(p->prec), np = ch.tiles.size();
    int rc = GFFTX_SUCCESS;
    std::string names;
    long long ns = 1;
    for (size_t i = 0; i < np; ++i) {
        const TileEntry* k = ch.tiles[i];
        Pass ps;
        ps.k = k;
        ps.real = k->real;
        if (np == 1) {
            ps.items_in_ntrans = true;
            ps.ntrans = (long long)p->batch;
            ps.its = (long long)p->dist;
            ps.ies = 1;
            ps.ns_pass = 1;
        } else {
            ps.xcd = xcd_remap(k, p->prec);
            ps.ntrans = (long long)(m / k->L);
            ps.its = 1;
            ps.ies = ps.ntrans;
            ps.ns_pass = ns;
            ps.bdist = (long long)m;
        }
        rc = upload_tile_table(p->allocs, k, &ps.stage_tw);
        if (!rc && ps.ns_pass > 1) {
            ps.ptw_m = ns * k->L;
            rc = upload_root_tables(p->allocs, ps.ptw_m, &ps.ptw_lo, &ps.ptw_hi, &ps.ptw_shift);
        }
        if (rc) return rc;
        ns = i == np / 2 ? k->L : ns * k->L;  // the turn ends the forward transform and starts the other
        // a launch profile shows where the three products of the chirp-z formula happen
        ps.slot = np == 1 ? k->name : i == 0 ? "bluestein_pre" : i + 1 == np ? "bluestein_post" : i == np / 2 ? "bluestein_mul" : k->name;
        names += std::string(i ? "," : "") + "{\"kernel\":\"" + k->name + "\"}";
        p->blue.push_back(ps);
    }
    for (size_t b = 0; b < (np == 1 ? 0u : 2u); ++b) {
        rc = dev_alloc(p, &p->blue_work[b], (size_t)m * p->batch * eb);
        if (rc) return rc;
    }
    rc = dev_alloc(p, &p->blue_chirp, (size_t)n * eb);
    if (rc) return rc;
    rc = dev_alloc(p, &p->blue_filter, (size_t)m * eb);
    if (rc) return rc;
    // the chirp from the two-level root table of order 2n; the filter's spectrum over m, from a
    // transform in FP64 (up to 2^24 points) that is rounded to the working precision once
    const int fp = m <= (1ull << 24) ? PREC_F64 : p->prec;
    const size_t fb = elem_bytes(fp);
    std::vector<void*> tmp;
    struct Free {
        std::vector<void*>& v;
        ~Free()
        {
            for (void* q : v) (void)hipFree(q);
        }
    } free_tmp{tmp};
    ChirpTableArgs ca;
    memset(&ca, 0, sizeof(ca));
    ca.n = (long long)n;
    rc = upload_root_tables(tmp, (long long)(2 * n), const_cast<double2**>(&ca.lo), const_cast<double2**>(&ca.hi), &ca.shift);
    if (rc) return rc;
    ca.chirp = p->blue_chirp;
    hipError_t e = launch_chirp_table(p->prec, ca, nullptr);
    void *fc = p->blue_chirp, *b = nullptr, *spec = nullptr;
    if (fp != p->prec) {
        rc = dev_alloc_list(tmp, &fc, (size_t)n * fb);
        if (rc) return rc;
        ca.chirp = fc;
        if (e == hipSuccess) e = launch_chirp_table(fp, ca, nullptr);
    }
    if (e != hipSuccess) return fail(GFFTX_ERR_LAUNCH, "chirp table: %s", hipGetErrorString(e));
    rc = dev_alloc_list(tmp, &b, (size_t)m * fb);
    if (!rc) rc = dev_alloc_list(tmp, &spec, (size_t)m * fb);
    if (rc) return rc;
    e = launch_chirp_filter(fp, fc, b, (long long)n, (long long)m, nullptr);
    if (e != hipSuccess) return fail(GFFTX_ERR_LAUNCH, "chirp filter: %s", hipGetErrorString(e));
    gfftx_plan f = nullptr;
    rc = create_plan_impl(&f, m, 1, fp == PREC_F64 ? GFFTX_COMPLEX_DOUBLE : GFFTX_COMPLEX_FLOAT, GFFTX_DFT,
                          GFFTX_OUT_OF_PLACE, p->device, 0, {}, "");
    if (rc) return rc;
    rc = exec_device(f, b, spec, nullptr);
    if (!rc) {
        e = launch_chirp_spectrum(fp, p->prec, spec, p->blue_filter, (long long)m, nullptr);
        if (e != hipSuccess) rc = fail(GFFTX_ERR_LAUNCH, "chirp spectrum: %s", hipGetErrorString(e));
    }
    const hipError_t se = hipStreamSynchronize(nullptr);  // before the temporary arrays go
    gfftx_plan_destroy(f);
    if (rc) return rc;
    if (se != hipSuccess) return fail(GFFTX_ERR_DEVICE, "filter transform: %s", hipGetErrorString(se));
    p->desc = "{\"n\":" + std::to_string(n) + ",\"batch\":" + std::to_string(p->batch) + ",\"precision\":\"" +
              (p->prec == PREC_F64 ? "f64" : "f32") + "\",\"passes\":[],\"bluestein\":{\"m\":" + std::to_string(m) +
              ",\"passes\":[" + names + "]}" + p->tune_note + "}";
    return GFFTX_SUCCESS;
}

// Runs the passes on batch items `r` of `in` and `out` (base pointers of the whole batch).  `boff`
// (optional) gives the element offset of every batch item in `in` and `out`; the range must then
// cover the whole batch.
int run_bluestein(gfftx_plan_s* p, const void* in, void* out, hipStream_t s, Range r, const long long* boff)
{
    if (!r.nb) r.nb = p->batch;
    const size_t eb = elem_bytes(p->prec), np = p->blue.size();
    // passes over several items take them from the grid's y dimension, at most 65535 a launch
    const unsigned long long most = np == 1 ? r.nb : 65535;
    for (unsigned long long b0 = r.b0; b0 < r.b0 + r.nb; b0 += most) {
        const unsigned long long nb = std::min(most, r.b0 + r.nb - b0);
        const size_t off = boff ? 0 : (size_t)b0 * p->dist * eb;
        const long long* bo = boff ? boff + b0 : nullptr;
        const size_t woff = (size_t)b0 * p->blue_m * eb;
        const void* src = (const char*)in + off;
        for (size_t i = 0; i < np; ++i) {
            const Pass& ps = p->blue[i];
            const bool first = i == 0, last = i + 1 == np;
            void* dst = last ? (char*)out + off : (char*)p->blue_work[i % 2] + woff;
            TileArgs a;
            memset(&a, 0, sizeof(a));
            a.in = src;
            a.out = dst;
            a.ntrans = np == 1 ? (long long)nb : ps.ntrans;
            a.its = ps.its;
            a.ies = ps.ies;
            a.ns_pass = ps.ns_pass;
            a.bdist = np == 1 ? 0 : first || last ? (long long)p->dist : ps.bdist;
            a.tw = ps.stage_tw;
            a.ptw_lo = ps.ptw_lo;
            a.ptw_hi = ps.ptw_hi;
            a.ptw_shift = ps.ptw_shift;
            a.conj_in = first && p->inverse ? 1 : 0;
            a.conj_out = last && p->inverse ? 1 : 0;
            a.scale = last && p->inverse ? 1.0 / (double)p->n : 1.0;
            a.xcd = ps.xcd;
            const size_t odist = last ? p->dist : p->blue_m;
            a.store = pass_store(p->through, r.nt, i, np, odist * nb * eb, ps, odist, nb);
            if (np == 1) a.seq_off = bo;
            else if (first || last) a.boff = bo;
            ChirpArgs c;
            c.chirp = p->blue_chirp;
            c.filter = p->blue_filter;
            c.n = (unsigned)p->n;
            c.mdist = (long long)p->blue_m;
            const dim3 grid((unsigned)((a.ntrans + ps.k->nb - 1) / ps.k->nb), np == 1 ? 1u : (unsigned)nb);
            std::pair<hipEvent_t, hipEvent_t> ev;
            const bool on = prof_begin(p, i, ps.slot, s, &ev, true);
            const hipEvent_t t0 = on ? ev.first : nullptr, t1 = on ? ev.second : nullptr;
            const hipError_t e = ps.k->mix ? launch_mixed(*ps.k, a, grid, s, t0, t1, &c) : launch_entry(ps.k, a, grid, s, t0, t1);
            if (on) prof_end(p, i, s, ev, true);
            if (e != hipSuccess) return fail(GFFTX_ERR_LAUNCH, "%s: %s", ps.k->name, hipGetErrorString(e));
            src = dst;
        }
    }
    return GFFTX_SUCCESS;
}

}  // namespace detail
}  // namespace gfftx
