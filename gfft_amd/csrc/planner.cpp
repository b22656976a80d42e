// planner.cpp -- twiddle roots, tile lookup, the pass cost model and pass splits, and the device
// tables plans upload.
#include "plan_internal.h"

#include <cstring>
#include "roots.h"

namespace gfftx {
namespace detail {

void root_ld(long long m, long long N, long double* c, long double* s) { root_ld_eval(m, N, c, s); }

// Every tile of (prec, L, modes), the default first: the compiled ones in table order, or,
// where there is none, the run-time mixed-radix tiles.
std::vector<const TileEntry*> tile_shapes(int prec, int L, bool loadT, bool storeT)
{
    std::vector<const TileEntry*> out;
    for (int i = 0; i < kNumTiles; ++i) {
        const TileEntry& e = kTiles[i];
        if (e.prec == prec && e.L == L && e.loadT == loadT && e.storeT == storeT) out.push_back(&e);
    }
    return out.empty() ? mix_tiles(prec, L, loadT, storeT) : out;
}

// First tile for (prec, L, modes), or the first one with nb == want_nb and wg == want_wg (each
// when nonzero) when there is one.
const TileEntry* find_tile(int prec, int L, bool loadT, bool storeT, int want_nb, int want_wg)
{
    const std::vector<const TileEntry*> v = tile_shapes(prec, L, loadT, storeT);
    if (want_nb || want_wg)
        for (const TileEntry* e : v)
            if ((!want_nb || e->nb == want_nb) && (!want_wg || e->wg == want_wg)) return e;
    return v.empty() ? nullptr : v[0];
}

// The variant of tile k (same length, shape, radices and access modes) with the real-transform
// split `kind` (REAL_POST, REAL_PRE) fused in, or null.
const TileEntry* find_real_tile(const TileEntry* k, int kind)
{
    if (k->mix) {
        // same shape, or, beside a one-butterfly tile, a shape of its own (two stages or more)
        const std::vector<const TileEntry*> v = mix_tiles(k->prec, k->L, k->loadT, k->storeT, kind);
        for (const TileEntry* e : v)
            if (e->nb == k->nb && e->wg == k->wg) return e;
        return k->nrad == 1 && !v.empty() ? v[0] : nullptr;
    }
    for (int i = 0; i < kNumRealTiles; ++i) {
        const TileEntry& e = kRealTiles[i];
        if (e.real != kind || e.prec != k->prec || e.L != k->L || e.nb != k->nb || e.wg != k->wg ||
            e.loadT != k->loadT || e.storeT != k->storeT || e.nrad != k->nrad)
            continue;
        bool same = true;
        for (int r = 0; r < e.nrad; ++r) same = same && e.radices[r] == k->radices[r];
        if (same) return &e;
    }
    return nullptr;
}

int env_int(const char* name, int dflt)
{
    const char* v = getenv(name);
    return v ? atoi(v) : dflt;
}

// Compute units of a device (256 on MI355X when the query fails).
int device_cus(int device)
{
    static int cached[64] = {0};
    if (device >= 0 && device < 64 && cached[device]) return cached[device];
    hipDeviceProp_t prop;
    int cus = 256;
    if (hipGetDeviceProperties(&prop, device) == hipSuccess) cus = prop.multiProcessorCount;
    else (void)hipGetLastError();
    if (device >= 0 && device < 64) cached[device] = cus;
    return cus;
}

// Bandwidth (TB/s) a multi-pass tile of length L reaches on MI355X with XCD remapping,
// measured over N = 2^24 passes; lengths not listed are interpolated by size class.  (The price of a
// chirp-z pass, chirp_plan.cpp.)
double pass_bandwidth(int prec, int L)
{
    const bool f32 = prec == PREC_F32;
    if (L < 16) return 5.0;  // one extra pass over the data for a leftover factor
    if (L <= 16) return f32 ? 5.5 : 5.6;
    if (L <= 64) return f32 ? 4.6 : 4.7;
    if (L <= 256) return f32 ? 4.2 : 4.6;
    if (L <= 1536) return f32 ? 3.1 : 3.5;
    return f32 ? 2.6 : 2.5;
}

// Modelled time (us) of one pass by tile `k` after passes of `ns` points in all (1: the first pass),
// over `batch` items of n points: the launch (a later pass also looks its twiddles up), and the
// bytes at the bandwidth the tile reaches next to the time of the tiles, one round after the other
// where the device does not hold them all (LDS and threads limit a CU to 160 KB and 2048 threads).
// The bandwidth falls with rows below a 128-byte line, with rows that begin anywhere in one, and in a
// run-time tile.  Fitted to 2193 splits of 69 lengths (16384 to 2^25 points, both precisions, 1 to
// 300 items, back to back): 8% rms, and the split it ranks first takes 4% more than the fastest
// of its length.  With one time a KB for every tile, and no stages, the first ranked one took 15%
// more (262144 FP64 in 512 * 512, rows of 32 bytes, 18.9 us; in 1024 * 256, 13.2).
double pass_cost(const TileEntry* k, unsigned long long ns, unsigned long long n, unsigned long long batch, int cus)
{
    const int by_lds = k->lds_bytes > 0 ? (160 * 1024) / k->lds_bytes : 8;
    const int per_cu = std::max(1, std::min(by_lds, 2048 / k->wg));
    const unsigned long long eb = elem_bytes(k->prec), pitch = n / (unsigned long long)k->L;
    const double tiles = std::ceil((double)pitch / k->nb) * (double)batch;
    const double rounds = std::ceil(tiles / ((double)cus * per_cu));
    const double kb = (double)k->nb * k->L * (double)eb / 1024.0;
    const bool f64 = k->prec == PREC_F64;
    const double tile = k->mix ? -0.4 + 1.7 * k->nrad + (f64 ? 0.061 : 0.056) * kb
                               : -2.4 + 1.7 * k->nrad + (f64 ? 0.048 : 0.063) * kb;
    const double bytes = (double)n * (double)batch * (double)eb;
    const bool cached = bytes <= 64.0 * 1048576;  // the pass's arrays stay in the Infinity Cache
    const unsigned long long row = (unsigned long long)k->nb * eb;
    const double bw = 7.0 * (k->mix ? 0.78 : 1.0) *
                      (row >= 128 ? 1.0 : row >= 64 ? (cached ? 0.85 : 0.65) : (cached ? 0.48 : 0.35)) *
                      (pitch * eb % 128 ? 0.73 : 1.0) * (ns > 1 && ns * eb % 128 ? 0.88 : 1.0);
    return (ns > 1 ? 3.0 : 0.4) + std::hypot(2.0 * bytes / (bw * 1e6), rounds * std::max(tile, 1.0));
}

// Modelled time (us) that a real transform's split adds to the passes when tile `k` is the one it can
// ride in: the last pass of a forward transform, the first of an inverse one.  Measured against the
// complex transform in the same passes: as a kernel of its own 2 us and 0.34 us a MB (an out-of-place
// inverse copies its input as well, the same again); fused 4.5 us and, by the length of the half
// rows it reads or writes, 0.15 (256 bytes, forward) to 1 us a MB (134 MB FP32 forward: 31 us in half
// rows of 256 bytes, 49 of 64; 33 MB FP32 inverse: 15 us in half rows of 32 bytes, 42 of 16).
double split_cost(const RealPart& real, const TileEntry* k, unsigned long long n, unsigned long long batch)
{
    if (real.kind == REAL_NONE) return 0;
    const double mb = (double)n * (double)batch * elem_bytes(k->prec) / 1e6;
    if (!find_real_tile(k, real.kind)) return (2.0 + 0.34 * mb) * (real.copy ? 2.0 : 1.0);
    const size_t half = (size_t)k->nb / 2 * elem_bytes(k->prec);
    const double us = real.kind == REAL_PRE ? (half >= 128 ? 0.2 : half >= 32 ? 0.3 : 0.9)
                                            : (half >= 256 ? 0.15 : half >= 128 ? 0.28 : half >= 64 ? 0.4 : 1.0);
    return 4.5 + us * mb;
}

// The tile a pass of length L takes after passes of `ns` points unless one is named: the default one
// of a compiled length, the one with the lowest modelled time of a run-time length; null when there is
// none.  *cost is that tile's modelled time or, with `any`, the lowest of the length's tiles.
const TileEntry* pass_tile(int prec, int L, unsigned long long ns, unsigned long long n, unsigned long long batch, int cus,
                           double* cost, bool any)
{
    const TileEntry* best = nullptr;
    double bc = 0, least = 0;
    for (const TileEntry* k : tile_shapes(prec, L, true, ns > 1)) {
        const double c = pass_cost(k, ns, n, batch, cus);
        if (!best || c < least) least = c;
        if (best && (!k->mix || c >= bc)) continue;
        best = k;
        bc = c;
    }
    if (cost) *cost = any ? least : bc;
    return best;
}

// Lengths of the pass tiles that divide n: the compiled ones and, with `mixed`, every other divisor
// with the factors 2, 3, 5 and 7 from 17 up to the run-time tiles' limit.  Ascending.
static std::vector<int> pass_lengths(int prec, unsigned long long n, bool mixed)
{
    std::vector<int> lens;
    for (int i = 0; i < kNumTiles; ++i)
        if (kTiles[i].prec == prec && kTiles[i].loadT && kTiles[i].storeT && n % (unsigned long long)kTiles[i].L == 0)
            lens.push_back(kTiles[i].L);
    std::sort(lens.begin(), lens.end());
    lens.erase(std::unique(lens.begin(), lens.end()), lens.end());
    if (mixed) {
        std::vector<int> more;
        const int most = mix_max(prec, true);
        for (long long a = 1; a <= most; a *= 2)
            for (long long b = a; b <= most; b *= 3)
                for (long long c = b; c <= most; c *= 5)
                    for (long long d = c; d <= most; d *= 7)
                        if (d > 16 && n % (unsigned long long)d == 0 && !std::binary_search(lens.begin(), lens.end(), (int)d))
                            more.push_back((int)d);
        lens.insert(lens.end(), more.begin(), more.end());
        std::sort(lens.begin(), lens.end());
    }
    return lens;
}

// Pass splits of n into T-mode tile lengths (2..4 passes), best `k` by the cost model (pass_cost(),
// and split_cost() of a real transform).  The first length of every split has a T->E tile.  A length
// counts with the tile it runs with by default or, with `any`, with its cheapest one (the autotuner
// times them all: 4096 * 8 of 32768 points FP32 takes 14.0 us by default and 9.2 with its best tiles).
std::vector<std::vector<int>> candidate_passes(int prec, unsigned long long n, size_t k, unsigned long long batch,
                                               int cus, bool mixed, RealPart real, bool any)
{
    const std::vector<int> lens = pass_lengths(prec, n, mixed);
    // cost of each length as the first pass, after passes of a multiple of 16 points (whole lines in
    // both precisions) and after others (negative: no such tile), and of the split of a real transform
    static const unsigned long long kNs[3] = {1, 16, 17};
    struct Cost {
        double pass[3] = {-1, -1, -1}, split[3] = {0, 0, 0};
    };
    std::vector<Cost> cost(lens.size());
    for (size_t i = 0; i < lens.size(); ++i)
        for (int j = 0; j < 3; ++j) {
            const TileEntry* t = pass_tile(prec, lens[i], kNs[j], n, batch, cus, &cost[i].pass[j], any);
            if (!t) cost[i].pass[j] = -1;
            else if ((j == 0) == (real.kind == REAL_PRE)) cost[i].split[j] = split_cost(real, t, n, batch);
        }
    auto kind = [&](unsigned long long ns) { return ns == 1 ? 0 : ns * elem_bytes(prec) % 128 == 0 ? 1 : 2; };
    std::vector<std::pair<double, std::vector<int>>> found;  // the best k so far, in the order met where equal
    std::vector<int> cur;                                    // indices into lens, largest first
    std::function<void(unsigned long long, int, double)> rec = [&](unsigned long long rem, int maxi, double least) {
        if (found.size() == k && (k == 0 || least >= found.back().first)) return;  // no better than the best k
        if (rem == 1) {
            if (cur.size() < 2) return;
            std::vector<int> order = cur;
            for (size_t i = 0; i < order.size(); ++i)
                if (cost[order[i]].pass[0] >= 0) {
                    std::swap(order[0], order[i]);
                    break;
                }
            double sum = 0;
            std::vector<int> l;
            unsigned long long ns = 1;
            for (size_t i = 0; i < order.size(); ++i) {
                const Cost& c = cost[order[i]];
                const int j = kind(ns);
                if (c.pass[j] < 0) return;
                sum += c.pass[j];
                if (real.kind == REAL_PRE ? i == 0 : i + 1 == order.size()) sum += c.split[j];
                l.push_back(lens[order[i]]);
                ns *= (unsigned long long)lens[order[i]];
            }
            auto at = std::upper_bound(found.begin(), found.end(), sum,
                                       [](double c, const std::pair<double, std::vector<int>>& f) { return c < f.first; });
            found.insert(at, {sum, l});
            if (found.size() > k) found.pop_back();
            return;
        }
        if (cur.size() == 4) return;
        for (int i = maxi; i >= 0; --i) {
            if (rem % (unsigned long long)lens[i]) continue;
            double c = -1;  // the least this length costs anywhere
            for (double x : cost[i].pass)
                if (x >= 0 && (c < 0 || x < c)) c = x;
            cur.push_back(i);
            rec(rem / lens[i], i, least + std::max(c, 0.0));
            cur.pop_back();
        }
    };
    rec(n, (int)lens.size() - 1, 0.0);
    std::vector<std::vector<int>> out;
    for (const auto& f : found) out.push_back(f.second);
    return out;
}

// A plan choice is the pass lengths, optionally followed by 0 and one (nb, wg) pair per
// pass naming the tile to use ((0, 0): the default tile of that length and mode).
void split_choice(const std::vector<int>& c, std::vector<int>& lens, std::vector<std::pair<int, int>>& tiles)
{
    lens.clear();
    tiles.clear();
    size_t i = 0;
    while (i < c.size() && c[i] != 0) lens.push_back(c[i++]);
    if (i < c.size()) ++i;
    while (i + 1 < c.size()) {
        tiles.push_back({c[i], c[i + 1]});
        i += 2;
    }
}

// Whether the pass lengths of a choice, which may come from a cache file, multiply to n.
bool passes_fit(const std::vector<int>& lens, unsigned long long n)
{
    unsigned long long prod = 1;
    for (int L : lens) {
        if (L < 2 || prod > n / (unsigned long long)L) return false;
        prod *= (unsigned long long)L;
    }
    return lens.size() >= 2 && prod == n;
}

// XCD-aware tile order for a pass tile (GFFTX_XCD overrides): on when the tile's rows are not
// whole 128-byte lines, so that the neighbouring tiles that share the lines at their ends run
// on one XCD and meet in its L2.  Tiles with whole-line rows share no lines; they load their
// inputs non-temporally and run fastest in dispatch order.
int xcd_remap(const TileEntry* k, int prec)
{
    const int forced = env_int("GFFTX_XCD", -1);
    if (forced >= 0) return forced ? 1 : 0;
    return (size_t)k->nb * elem_bytes(prec) % 128 != 0 ? 1 : 0;
}

// Whether n runs natively: one single-pass tile, or a split into pass tiles (lengths with the
// factors 2, 3, 5 and 7).  Any other n runs as a chirp-z convolution.  (Every plan asks, so the
// search ends at the first split: listing them all took 17 ms at 203212800.)
bool native_length(int prec, unsigned long long n)
{
    if (n <= (1ull << 30) && find_tile(prec, (int)n, false, false)) return true;
    const std::vector<int> lens = pass_lengths(prec, n, true);
    std::function<bool(unsigned long long, int, int, bool)> rec = [&](unsigned long long rem, int maxi, int passes, bool first) {
        if (rem == 1) return passes >= 2 && first;
        if (passes == 4) return false;
        for (int i = maxi; i >= 0; --i)
            if (rem % (unsigned long long)lens[i] == 0 &&
                rec(rem / lens[i], i, passes + 1, first || find_tile(prec, lens[i], true, false) != nullptr))
                return true;
        return false;
    };
    return rec(n, (int)lens.size() - 1, 0, false);
}

// The pass split GFFTX_PASSES="a,b,c" names, when it multiplies to n and every length has a tile.
bool env_passes(int prec, unsigned long long n, std::vector<int>& out)
{
    const char* env = getenv("GFFTX_PASSES");
    if (!env) return false;
    std::vector<int> v;
    unsigned long long prod = 1;
    const char* p = env;
    while (*p) {
        const long x = strtol(p, const_cast<char**>(&p), 10);
        if (x <= 1) break;
        v.push_back((int)x);
        prod *= (unsigned long long)x;
        if (*p == ',') ++p;
        else break;
    }
    bool ok = prod == n && v.size() >= 2;
    for (size_t i = 0; ok && i < v.size(); ++i)
        ok = find_tile(prec, v[i], true, i == 0 ? false : true) != nullptr;
    if (ok) out = v;
    return ok;
}

// The single-pass tile of n, or null where n runs in passes: no tile of that length, or a
// run-time one and a split named by GFFTX_PASSES.
const TileEntry* single_tile(int prec, unsigned long long n, int want_nb, int want_wg)
{
    if (n > (1ull << 30)) return nullptr;
    const TileEntry* k = find_tile(prec, (int)n, false, false, want_nb, want_wg);
    std::vector<int> v;
    return k && k->mix && env_passes(prec, n, v) ? nullptr : k;
}

// Split n into pass lengths available as T-mode tiles (largest first), or the override list.
bool choose_passes(int prec, unsigned long long n, std::vector<int>& out, unsigned long long batch, int cus, RealPart real)
{
    out.clear();
    if (env_passes(prec, n, out)) return true;
    std::vector<std::vector<int>> c = candidate_passes(prec, n, 1, batch, cus, true, real);
    if (c.empty()) return false;
    out = c[0];
    return true;
}

// W_N^m = first + i second, m = 0..N-1.  Where N is a multiple of 8 the first octant is evaluated and
// the others follow from it by the folds of root_ld: the same bits with an eighth of the evaluations
// (0.1 us each: the 1552 of a 1024-point tile were most of the 0.2 ms its plan took to make).
std::vector<std::pair<long double, long double>> all_roots(long long N)
{
    std::vector<std::pair<long double, long double>> w(N);
    const long long o8 = N % 8 == 0 ? N / 8 : 0;
    if (!o8) {
        for (long long m = 0; m < N; ++m) root_ld(m, N, &w[m].first, &w[m].second);
        return w;
    }
    std::vector<long double> co(o8 + 1), si(o8 + 1);  // cosine and sine, 0 to pi/4
    for (long long j = 0; j <= o8; ++j) {
        long double c, s;
        root_ld(j, N, &c, &s);
        co[j] = j < o8 ? c : -s;
        si[j] = j < o8 ? -s : c;
    }
    for (long long m = 0; m < N; ++m) {
        const long long o = m / o8, j = o % 2 ? o8 - m % o8 : m % o8;
        const bool swap = o == 1 || o == 2 || o == 5 || o == 6;
        const long double c = swap ? si[j] : co[j], s = swap ? co[j] : si[j];
        w[m] = {o >= 2 && o <= 5 ? -c : c, o < 4 ? -s : s};
    }
    return w;
}

template <typename T> void pack_stage_table(int nrad, const int* radices, std::vector<T>& out)
{
    // stage s >= 1: rows k in [0, Ns), entries r in [0, R): W_{Ns*R}^{k*r}
    out.clear();
    long long ns = radices[0];
    for (int s = 1; s < nrad; ++s) {
        const long long R = radices[s];
        const auto w = all_roots(ns * R);
        for (long long kk = 0; kk < ns; ++kk)
            for (long long r = 0; r < R; ++r) {
                out.push_back((T)w[kk * r].first);
                out.push_back((T)w[kk * r].second);
            }
        ns *= R;
    }
}

// Device allocation recorded in an owner's list (plans and ragged plans).
int dev_alloc_list(std::vector<void*>& owned, void** out, size_t bytes)
{
    if (bytes == 0) bytes = 16;
    hipError_t e = hipMalloc(out, bytes);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        return fail(GFFTX_ERR_ALLOC, "hipMalloc(%zu) failed: %s", bytes, hipGetErrorString(e));
    }
    owned.push_back(*out);
    return GFFTX_SUCCESS;
}

int upload_stage_table_r(std::vector<void*>& owned, int prec, int nrad, const int* radices, void** out,
                         double scale)
{
    *out = nullptr;
    if (nrad <= 1) return GFFTX_SUCCESS;
    // the rows in the working precision, then, 16-byte aligned, the FP64 roots W_{Ns R}^k
    // (k < Ns) of every stage s >= 1, from which the tiles form their twiddles
    // (TileCfg::TW_POW)
    std::vector<double> roots;
    long long ns = radices[0];
    for (int st = 1; st < nrad; ++st) {
        const auto w = all_roots(ns * radices[st]);
        for (long long kk = 0; kk < ns; ++kk) {
            roots.push_back((double)w[kk].first);
            roots.push_back((double)w[kk].second);
        }
        ns *= radices[st];
    }
    std::vector<unsigned char> bytes;
    if (prec == PREC_F64) {
        std::vector<double> t;
        pack_stage_table(nrad, radices, t);
        for (double& v : t) v *= scale;
        bytes.resize(t.size() * sizeof(double));
        memcpy(bytes.data(), t.data(), bytes.size());
    } else {
        std::vector<float> t;
        pack_stage_table(nrad, radices, t);
        for (float& v : t) v = (float)(v * scale);
        while (t.size() % 4) t.push_back(0.f);
        bytes.resize(t.size() * sizeof(float));
        memcpy(bytes.data(), t.data(), bytes.size());
    }
    const size_t rows = bytes.size();
    bytes.resize(rows + roots.size() * sizeof(double));
    memcpy(bytes.data() + rows, roots.data(), roots.size() * sizeof(double));
    int rc = dev_alloc_list(owned, out, bytes.size());
    if (rc) return rc;
    HIP_TRY(hipMemcpy(*out, bytes.data(), bytes.size(), hipMemcpyHostToDevice));
    return GFFTX_SUCCESS;
}

// FP64 two-level table for W_M^m: lo[m mod 2^b], hi[m >> b], 2^b ~ sqrt(M).
int upload_root_tables(std::vector<void*>& owned, long long M, double2** lo_out, double2** hi_out, int* shift)
{
    int b = 0;
    while ((1LL << (2 * b)) < M) ++b;
    const long long nlo = 1LL << b, nhi = (M + nlo - 1) / nlo + 1;
    std::vector<double> lo(2 * nlo), hi(2 * nhi);
    for (long long m = 0; m < nlo; ++m) {
        long double c, s;
        root_ld(m, M, &c, &s);
        lo[2 * m] = (double)c;
        lo[2 * m + 1] = (double)s;
    }
    // where 2^b divides M, W_M^{h 2^b} is a root of order M / 2^b (a power of two scales out of the angle)
    const auto w = M % nlo == 0 ? all_roots(M / nlo) : std::vector<std::pair<long double, long double>>();
    for (long long h = 0; h < nhi; ++h) {
        long double c, s;
        if (!w.empty()) {
            c = w[h % (long long)w.size()].first;
            s = w[h % (long long)w.size()].second;
        } else {
            root_ld(h * nlo, M, &c, &s);
        }
        hi[2 * h] = (double)c;
        hi[2 * h + 1] = (double)s;
    }
    void* dlo = nullptr;
    void* dhi = nullptr;
    int rc = dev_alloc_list(owned, &dlo, lo.size() * sizeof(double));
    if (rc) return rc;
    rc = dev_alloc_list(owned, &dhi, hi.size() * sizeof(double));
    if (rc) return rc;
    HIP_TRY(hipMemcpy(dlo, lo.data(), lo.size() * sizeof(double), hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(dhi, hi.data(), hi.size() * sizeof(double), hipMemcpyHostToDevice));
    *lo_out = (double2*)dlo;
    *hi_out = (double2*)dhi;
    *shift = b;
    return GFFTX_SUCCESS;
}

// Twiddles of the MFMA kernel (MfmaArgs::tw): W_256^m times `scale` (the per-stage 2^-4 or 1),
// then W_4096^m, m < 256.
int upload_mfma_twiddles(std::vector<void*>& owned, double scale, void** out)
{
    std::vector<float> t;
    for (int m = 0; m < 256; ++m) {
        long double c, si;
        root_ld(m, 256, &c, &si);
        t.push_back((float)((double)c * scale));
        t.push_back((float)((double)si * scale));
    }
    for (int m = 0; m < 256; ++m) {
        long double c, si;
        root_ld(m, 4096, &c, &si);
        t.push_back((float)c);
        t.push_back((float)si);
    }
    int rc = dev_alloc_list(owned, out, t.size() * sizeof(float));
    if (rc) return rc;
    HIP_TRY(hipMemcpy(*out, t.data(), t.size() * sizeof(float), hipMemcpyHostToDevice));
    return GFFTX_SUCCESS;
}

// A operands of the MFMA radix-16 stage (mfma_kernel.h): [mt][hi/lo][lane][8] halves.
int upload_mfma_matrix(std::vector<void*>& owned, void** out)
{
    std::vector<_Float16> h(MFMA_A_HALFS);
    for (int mt = 0; mt < 2; ++mt)
        for (int lane = 0; lane < 64; ++lane)
            for (int i = 0; i < 8; ++i) {
                const int q = lane % 16, k = 8 * (lane / 16) + i, r = k / 2, im = k % 2;
                long double c, sn;
                root_ld((long long)q * r, 16, &c, &sn);  // F[q][r] = W16^{qr} = c + i sn
                long double val;
                if (mt == 0) val = im ? -sn : c;   // Re Y row: Re F, -Im F
                else val = im ? c : sn;            // Im Y row: Im F,  Re F
                const _Float16 hi = (_Float16)(double)val;
                const _Float16 lo = (_Float16)(double)(val - (long double)(double)hi);
                h[((mt * 2 + 0) * 64 + lane) * 8 + i] = hi;
                h[((mt * 2 + 1) * 64 + lane) * 8 + i] = lo;
            }
    int rc = dev_alloc_list(owned, out, h.size() * sizeof(_Float16));
    if (rc) return rc;
    HIP_TRY(hipMemcpy(*out, h.data(), h.size() * sizeof(_Float16), hipMemcpyHostToDevice));
    return GFFTX_SUCCESS;
}

}  // namespace detail
}  // namespace gfftx
