// tuner.cpp -- plan creation with the measured autotuner and its versioned JSON cache.
#include "plan_internal.h"

#include <fcntl.h>
#include <sys/file.h>

namespace gfftx {
namespace detail {

// ---------------------------------------------------------------------------------------
// Autotuner: for a multi-pass plan, time the best few pass splits of the cost model on this
// device and keep the fastest.  Results are cached per (device, kernel revision, precision, n,
// batch, kind, place) in memory and in a versioned JSON file ($GFFTX_TUNE_CACHE, default
// ~/.cache/gfftx/tune.json).
std::mutex g_tune_mu;
std::map<std::string, std::vector<int>> g_tune;
std::string g_tune_loaded;  // cache file the in-memory entries belong to

std::string tune_path()
{
    if (const char* e = getenv("GFFTX_TUNE_CACHE")) return e;
    const char* h = getenv("HOME");
    return std::string(h ? h : "/tmp") + "/.cache/gfftx/tune.json";
}

// One entry per line: "key": [pass lengths..., 0, nb, wg per pass] (version 1 files hold
// the pass lengths only, which still load)
void read_entries(const std::string& path, std::map<std::string, std::vector<int>>& out)
{
    FILE* f = fopen(path.c_str(), "r");
    if (!f) return;
    char line[512];
    while (fgets(line, sizeof(line), f)) {
        char* q1 = strchr(line, '"');
        if (!q1) continue;
        char* q2 = strchr(q1 + 1, '"');
        char* lb = q2 ? strchr(q2, '[') : nullptr;
        if (!lb) continue;
        const std::string key(q1 + 1, q2);
        if (key == "version" || key == "entries") continue;
        std::vector<int> v;
        char* p = lb + 1;
        while (*p && *p != ']') {
            const long x = strtol(p, &p, 10);
            if (x < 0) break;
            v.push_back((int)x);
            while (*p == ',' || *p == ' ') ++p;
            if (!isdigit((unsigned char)*p) && *p != ']') break;
        }
        std::vector<int> lens;
        std::vector<std::pair<int, int>> tiles;
        split_choice(v, lens, tiles);
        // plan entries hold two pass lengths or more; a ragged batch's entry one limit
        const bool ragged = key.find("|ragged|") != std::string::npos;
        if (lens.size() >= 2 || (ragged && v.size() == 1)) out[key] = v;
    }
    fclose(f);
}

void tune_load()
{
    const std::string path = tune_path();
    if (g_tune_loaded == path) return;
    g_tune_loaded = path;
    g_tune.clear();
    read_entries(path, g_tune);
}

// Writes the in-memory entries merged with what the file holds now: another process may have
// stored entries since this one read it.  An exclusive lock on "<file>.lock" serialises the
// read-merge-rename of concurrent writers; entries of this process win on equal keys.
void tune_store()
{
    const std::string path = tune_path();
    const size_t slash = path.find_last_of('/');
    if (slash != std::string::npos) {
        std::string dir = path.substr(0, slash);
        for (size_t i = 1; i <= dir.size(); ++i)
            if (i == dir.size() || dir[i] == '/') (void)mkdir(dir.substr(0, i).c_str(), 0755);
    }
    const int lk = open((path + ".lock").c_str(), O_CREAT | O_RDWR, 0644);
    if (lk >= 0) (void)flock(lk, LOCK_EX);
    std::map<std::string, std::vector<int>> disk;
    read_entries(path, disk);
    for (const auto& kv : disk) g_tune.insert(kv);  // keeps this process's entry on equal keys
    const std::string tmp = path + ".tmp" + std::to_string((long)getpid());
    FILE* f = fopen(tmp.c_str(), "w");
    if (!f) {
        if (lk >= 0) close(lk);
        return;
    }
    fprintf(f, "{\"version\": 2, \"entries\": {\n");
    size_t i = 0;
    for (const auto& kv : g_tune) {
        fprintf(f, "\"%s\": [", kv.first.c_str());
        for (size_t j = 0; j < kv.second.size(); ++j) fprintf(f, "%s%d", j ? ", " : "", kv.second[j]);
        fprintf(f, "]%s\n", ++i < g_tune.size() ? "," : "");
    }
    fprintf(f, "}}\n");
    fclose(f);
    (void)rename(tmp.c_str(), path.c_str());
    if (lk >= 0) close(lk);  // releases the lock
}

std::string tune_key(int device, int prec, uint64_t n, uint64_t batch);

// Key of a ragged batch's choice: the device, the precision, the point and transform counts
// and an FNV-1a hash of the (length, count) classes in increasing length.
std::string ragged_tune_key(int device, int prec, const uint64_t* lengths, uint64_t count)
{
    std::map<uint64_t, uint64_t> classes;
    uint64_t points = 0;
    for (uint64_t i = 0; i < count; ++i) {
        ++classes[lengths[i]];
        points += lengths[i];
    }
    uint64_t h = 1469598103934665603ull;
    auto mix = [&h](uint64_t v) {
        for (int b = 0; b < 8; ++b) {
            h ^= (v >> (8 * b)) & 0xff;
            h *= 1099511628211ull;
        }
    };
    for (const auto& kv : classes) {
        mix(kv.first);
        mix(kv.second);
    }
    char hex[24];
    snprintf(hex, sizeof(hex), "%016llx", (unsigned long long)h);
    return tune_key(device, prec, points, count) + "|ragged|h=" + hex;
}

bool tune_get(const std::string& key, std::vector<int>* v)
{
    std::lock_guard<std::mutex> lk(g_tune_mu);
    tune_load();
    auto it = g_tune.find(key);
    if (it == g_tune.end()) return false;
    *v = it->second;
    return true;
}

void tune_put(const std::string& key, const std::vector<int>& v)
{
    std::lock_guard<std::mutex> lk(g_tune_mu);
    tune_load();
    g_tune[key] = v;
    tune_store();
}

// Revision of the kernels the cached choices were measured with: part of every key, so that a
// cache file written by a library with other tiles is measured afresh, not taken over.
static constexpr int kTuneRevision = 5;

std::string tune_key(int device, int prec, uint64_t n, uint64_t batch)
{
    hipDeviceProp_t prop;
    std::string dev = "dev";
    if (hipGetDeviceProperties(&prop, device) == hipSuccess) dev = std::string(prop.gcnArchName) + ":" + std::to_string(prop.multiProcessorCount) + "cu";
    else (void)hipGetLastError();
    return dev + ":r" + std::to_string(kTuneRevision) + "|" + (prec == PREC_F64 ? "f64" : "f32") + "|n=" + std::to_string(n) + "|b=" + std::to_string(batch);
}

// Transforms of n points that may run in place one after the other from numbers around 1: each
// forward one multiplies their rms by sqrt(n) (a real one of 2n points by sqrt(2n)), each inverse one
// divides it.  Up to 2^100 FP32 and 2^900 FP64 either way: a chirp-z transform's convolution goes up to 2^14
// higher, and single numbers 2^3.  At least one.
int fill_reps(int prec, unsigned long long n)
{
    return std::max(1, (int)((prec == PREC_F64 ? 1800.0 : 200.0) / std::log2(2.0 * (double)n)));
}

// Time (ms) of one execution of a plan on scratch buffers, as a throughput: three groups of at
// least `reps` executions issued back to back between two events, the median of the group means.
// Back-to-back calls are what a batch loop issues; a call timed alone after a synchronisation
// also carries the start of an idle device.
// The calls walk over `sets` pairs of arrays, `stride` bytes apart, as a program's successive
// inputs do: on one pair a transform of a few MB runs from the L2 caches, and the choice between
// two splits can come out the other way.  With `alt` (2 (sets - 1) more arrays) the passes'
// intermediate arrays change with them, as where a program's plans take turns: 3 * 2^20 reals FP32
// in 1536 * 1024 take 28.6 us on one pair of them and 24.9 on three, in 256 * 96 * 64 26.0 and 25.0.
// With `fill`, `a` is set to it before every group, which then has at most fill_reps() executions: a
// transform that runs in place would leave the range of its numbers.
int time_plan(gfftx_plan_s* p, void* a, void* b, hipStream_t s, int reps, float* ms_out, int sets = 1, size_t stride = 0,
              void* alt = nullptr, const void* fill = nullptr, size_t fill_bytes = 0)
{
    const int most = fill ? fill_reps(p->prec, p->n) : 1 << 30;
    reps = std::min(reps, most);
    int call = 0;
    auto exec = [&]() {
        const size_t set = (size_t)(call++ % sets), off = set * stride;
        if (alt && set && p->scratch[0]) {
            p->call_scratch[0] = (char*)alt + 2 * (set - 1) * stride;
            p->call_scratch[1] = (char*)alt + (2 * (set - 1) + 1) * stride;
        }
        const int rc = exec_device(p, (char*)a + off, (char*)b + off, s);
        p->call_scratch[0] = p->call_scratch[1] = nullptr;
        return rc;
    };
    for (int i = 0; i < 2; ++i) {
        int rc = exec();
        if (rc) return rc;
    }
    std::vector<float> t;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    if (hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess) {
        if (e0) (void)hipEventDestroy(e0);
        (void)hipGetLastError();
        return fail(GFFTX_ERR_DEVICE, "cannot create timing events");
    }
    // a first group that does not count gives the repetitions: at least 0.4 ms in a group
    for (int g = -1; g < 3; ++g) {
        if (fill) (void)hipMemcpyAsync(a, fill, fill_bytes, hipMemcpyDeviceToDevice, s);
        (void)hipEventRecord(e0, s);
        int rc = GFFTX_SUCCESS;
        for (int i = 0; i < reps && !rc; ++i) rc = exec();
        (void)hipEventRecord(e1, s);
        (void)hipEventSynchronize(e1);
        if (rc) {
            (void)hipEventDestroy(e0);
            (void)hipEventDestroy(e1);
            return rc;
        }
        float ms = 0;
        (void)hipEventElapsedTime(&ms, e0, e1);
        if (g >= 0) {
            t.push_back(ms / reps);
            continue;
        }
        reps = std::min(most, std::max(reps, (int)(0.4f / std::max(ms / reps, 0.002f))));
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    std::sort(t.begin(), t.end());
    *ms_out = t[t.size() / 2];
    return GFFTX_SUCCESS;
}

// Numbers between -1 and 1 (a multiplicative generator, repeated every MiB), written on stream s.
static bool fill_numbers(int prec, void* dst, size_t bytes, hipStream_t s)
{
    const size_t block = std::min<size_t>(bytes, (size_t)1 << 20);
    std::vector<double> d(prec == PREC_F64 ? block / 8 : 0);
    std::vector<float> f(prec == PREC_F64 ? 0 : block / 4);
    uint64_t x = 88172645463325252ull;
    auto next = [&x]() {
        x = x * 6364136223846793005ull + 1442695040888963407ull;
        return (double)(int64_t)x / 9223372036854775808.0;
    };
    for (double& v : d) v = next();
    for (float& v : f) v = (float)next();
    const void* src = prec == PREC_F64 ? (const void*)d.data() : (const void*)f.data();
    bool ok = hipMemcpyAsync(dst, src, block, hipMemcpyHostToDevice, s) == hipSuccess;
    for (size_t n = block; ok && n < bytes; n *= 2)
        ok = hipMemcpyAsync((char*)dst + n, dst, std::min(n, bytes - n), hipMemcpyDeviceToDevice, s) == hipSuccess;
    return hipStreamSynchronize(s) == hipSuccess && ok;  // before the host arrays go
}

// Arrays and stream the candidates of one choice run on: up to 64 MiB three pairs of arrays that the
// calls walk over (time_plan) and, with `passes`, three sets of intermediate ones; above, one pair of
// numbers.  A large transform is bound by memory and by the power it takes, and on zeros it takes
// less power (65536 x 1024 FP64, four sequences a workgroup against one: 363 and 366 us on zeros, 369
// and 364 on numbers).
struct TuneArrays {
    void *a = nullptr, *b = nullptr, *alt = nullptr;
    hipStream_t s = nullptr;
    size_t bytes = 0;
    int sets = 1;
    const void* fill = nullptr;

    // false: no room for the arrays a call needs
    bool make(int prec, size_t want, bool inplace, bool passes)
    {
        bytes = (want + 255) / 256 * 256;
        sets = bytes <= (64u << 20) ? 3 : 1;
        if (hipStreamCreateWithFlags(&s, hipStreamNonBlocking) != hipSuccess || hipMalloc(&a, bytes * sets) != hipSuccess ||
            (!inplace && hipMalloc(&b, bytes * sets) != hipSuccess)) {
            (void)hipGetLastError();
            return false;
        }
        if (sets > 1 && passes && hipMalloc(&alt, bytes * 2 * (sets - 1)) != hipSuccess) alt = nullptr;
        if (sets == 1 && inplace && hipMalloc(&b, bytes) != hipSuccess) b = nullptr;  // (then on zeros)
        // all of it on `s`: that stream does not wait for the null stream
        (void)hipMemsetAsync(a, 0, bytes * sets, s);
        if (sets == 1 && b && fill_numbers(prec, b, bytes, s) &&
            hipMemcpyAsync(a, b, bytes, hipMemcpyDeviceToDevice, s) == hipSuccess)
            fill = inplace ? b : nullptr;
        (void)hipGetLastError();
        return true;
    }
    int time(gfftx_plan_s* p, int reps, float* ms) const
    {
        return time_plan(p, a, p->place == GFFTX_IN_PLACE ? a : b, s, reps, ms, sets, bytes, alt, fill, bytes);
    }
    ~TuneArrays()
    {
        if (s) {
            (void)hipStreamSynchronize(s);
            (void)hipStreamDestroy(s);
        }
        for (void* p : {a, b, alt})
            if (p) (void)hipFree(p);
        (void)hipGetLastError();
    }
};

// The candidates of one choice, timed on `arrays`; `make` builds one (null: it cannot be built).
struct TuneRun {
    const TuneArrays& arrays;
    std::function<gfftx_plan(const std::vector<int>&)> make;
    std::vector<std::pair<float, std::vector<int>>> timed;
    std::vector<int> chosen;  // the fastest so far
    float best = 1e30f;

    // ms of one execution, or -1
    float time(const std::vector<int>& c)
    {
        gfftx_plan p = make(c);
        if (!p) return -1.f;
        float ms = 0;
        const int rc = arrays.time(p, 5, &ms);
        gfftx_plan_destroy(p);
        if (rc) return -1.f;
        timed.push_back({ms, c});
        if (ms < best) {
            best = ms;
            chosen = c;
        }
        return ms;
    }
    // the fastest few once more, in turn, on plans that stay: a single timing of a short transform
    // moves by more than the candidates differ
    void again(size_t few)
    {
        std::vector<std::pair<float, std::vector<int>>> top = timed;
        std::stable_sort(top.begin(), top.end(), [](const auto& x, const auto& y) { return x.first < y.first; });
        top.resize(std::min<size_t>(top.size(), arrays.bytes <= (64u << 20) ? few : 2));
        if (top.size() < 2) return;
        std::vector<gfftx_plan> tp;
        std::vector<float> tms(top.size(), 1e30f);
        for (const auto& t : top) tp.push_back(make(t.second));
        for (int rep = 0; rep < 3; ++rep)
            for (size_t i = 0; i < top.size(); ++i) {
                float ms = 0;
                if (tp[i] && arrays.time(tp[i], 10, &ms) == GFFTX_SUCCESS) tms[i] = std::min(tms[i], ms);
            }
        const size_t w = std::min_element(tms.begin(), tms.end()) - tms.begin();
        if (tms[w] < 1e30f) chosen = top[w].second;
        for (gfftx_plan q : tp) gfftx_plan_destroy(q);
    }
};

// The splits to time: the cost model's best `k` and its best three of compiled tiles alone, each length
// counted with its cheapest tile; the best two of the fewest passes, which the model's price of a
// stage can put behind (480000 FP32: 960 * 500 15.5 us, 768 * 25 * 25 16.4); of a real transform also the best three of its passes alone (the
// price of a fused split is the model's least certain part: 393216 FP32 forward, 1536 * 256 fused
// 17.1 us, the best with its split priced 19.0); and the one an untuned plan takes.
std::vector<std::vector<int>> tuned_splits(int prec, unsigned long long n, size_t k, unsigned long long batch, int cus, RealPart real)
{
    std::vector<std::vector<int>> v = candidate_passes(prec, n, k, batch, cus, true, real, true);
    auto add = [&v](const std::vector<std::vector<int>>& more) {
        for (const std::vector<int>& c : more)
            if (std::find(v.begin(), v.end(), c) == v.end()) v.push_back(c);
    };
    add(candidate_passes(prec, n, 3, batch, cus, false, real, true));
    std::vector<std::vector<int>> few = candidate_passes(prec, n, 40, batch, cus, true, real, true);
    std::stable_sort(few.begin(), few.end(), [](const auto& x, const auto& y) { return x.size() < y.size(); });
    if (few.size() > 1 && few[1].size() > few[0].size()) few.resize(1);
    few.resize(std::min<size_t>(few.size(), 2));
    add(few);
    if (real.kind != REAL_NONE) add(candidate_passes(prec, n, 3, batch, cus, false, RealPart(), true));
    add(candidate_passes(prec, n, 1, batch, cus, true, real));
    return v;
}

// Tuning candidates from pass splits: each split with its default tiles, then with every
// other compiled tile shape of its first pass (T->E) and of each length it uses after the
// first pass (T->T), one position at a time ([lens..., 0, nb, wg per pass], 0 = default).
static std::vector<std::vector<int>> split_variants(int prec, unsigned long long n, unsigned long long batch, int cus,
                                                    const std::vector<std::vector<int>>& splits)
{
    std::vector<std::vector<int>> cands;
    for (const std::vector<int>& sp : splits) {
        cands.push_back(sp);
        std::vector<int> seen;
        unsigned long long ns = 1;
        for (size_t i = 0; i < sp.size(); ++i) {
            const int L = sp[i];
            const bool later = i > 0;
            const unsigned long long before = ns;
            ns *= (unsigned long long)L;
            if (later && std::find(seen.begin(), seen.end(), L) != seen.end()) continue;
            if (later) seen.push_back(L);
            const TileEntry* def = pass_tile(prec, L, before, n, batch, cus);
            for (const TileEntry* t : tile_shapes(prec, L, true, later)) {
                if (t == def) continue;
                const TileEntry& e = *t;
                std::vector<int> c = sp;
                c.push_back(0);
                for (size_t j = 0; j < sp.size(); ++j) {
                    const bool alt = later ? (j > 0 && sp[j] == L) : j == 0;
                    c.push_back(alt ? e.nb : 0);
                    c.push_back(alt ? e.wg : 0);
                }
                cands.push_back(c);
            }
        }
    }
    return cands;
}

// The candidates vary one pass position at a time around the default tiles.  For the split of
// `chosen`, the fastest variant timed at each position combined (ms[i] < 0: candidate i failed);
// empty when that is no new candidate.
static std::vector<int> best_combination(const std::vector<int>& chosen, const std::vector<std::vector<int>>& cands,
                                         const std::vector<float>& ms)
{
    std::vector<int> wl;
    std::vector<std::pair<int, int>> wt;
    split_choice(chosen, wl, wt);
    std::vector<std::pair<int, int>> bt(wl.size(), {0, 0});
    std::vector<float> bms(wl.size(), 1e30f);
    for (size_t i = 0; i < cands.size(); ++i) {
        if (ms[i] < 0) continue;
        std::vector<int> cl;
        std::vector<std::pair<int, int>> ct;
        split_choice(cands[i], cl, ct);
        if (cl != wl) continue;
        for (size_t j = 0; j < ct.size() && j < wl.size(); ++j)
            if (ct[j].first && ms[i] < bms[j]) {
                bms[j] = ms[i];
                bt[j] = ct[j];
            }
    }
    std::vector<int> combo = wl;
    combo.push_back(0);
    for (const auto& t : bt) {
        combo.push_back(t.first);
        combo.push_back(t.second);
    }
    const bool varied = std::any_of(bt.begin(), bt.end(), [](const std::pair<int, int>& t) { return t.first != 0; });
    if (!varied || combo == chosen || std::find(cands.begin(), cands.end(), combo) != cands.end()) return {};
    return combo;
}

// A choice with the run-time tiles its lengths ran with: which one is the default depends on the number of
// items, and the candidates of a batch above 1 GiB run on fewer than the plan has.
std::vector<int> with_tiles(int prec, unsigned long long n, unsigned long long batch, int cus, const std::vector<int>& c)
{
    std::vector<int> l;
    std::vector<std::pair<int, int>> t;
    split_choice(c, l, t);
    if (!passes_fit(l, n) || getenv("GFFTX_TNB") || getenv("GFFTX_TWG")) return c;
    t.resize(l.size(), {0, 0});
    unsigned long long ns = 1;
    for (size_t i = 0; i < l.size(); ++i) {
        const TileEntry* k = t[i].first ? nullptr : pass_tile(prec, l[i], ns, n, batch, cus);
        if (k && k->mix) t[i] = {k->nb, k->wg};
        ns *= (unsigned long long)l[i];
    }
    l.push_back(0);
    for (const auto& x : t) {
        l.push_back(x.first);
        l.push_back(x.second);
    }
    return l;
}

// A choice as describe() names it: the pass lengths, each with /nb-wg where the choice names the tile,
// or single/nb-wg; for a chirp-z plan the convolution length m first, then all of its passes (a split of
// m into k lengths runs in 2k - 1).
std::string choice_label(const std::vector<int>& c, bool chirp)
{
    std::vector<int> l;
    std::vector<std::pair<int, int>> t;
    split_choice(c, l, t);
    std::string s;
    if (chirp && l.size() > 1) {
        s = std::to_string(l[0]) + ": ";
        l.erase(l.begin());
        if (l.size() > 1)
            for (size_t i = l.size() - 1; i-- > 0;) l.push_back(l[i]);
    } else if (l.size() == 2 && l[1] == 1) {
        l.erase(l.begin());
    }
    for (size_t j = 0; j < l.size(); ++j) {
        s += (j ? "x" : "") + (l.size() == 1 && l[0] == 1 ? std::string("single") : std::to_string(l[j]));
        if (j < t.size() && t[j].first) s += "/" + std::to_string(t[j].first) + "-" + std::to_string(t[j].second);
    }
    return s;
}

// The candidates timed, for describe(): the fastest 32, fastest first (a length with many divisors
// has over a hundred, more than describe()'s callers have room for).
static std::string tune_note(std::vector<std::pair<float, std::vector<int>>> timed, bool chirp)
{
    std::stable_sort(timed.begin(), timed.end(), [](const auto& x, const auto& y) { return x.first < y.first; });
    timed.resize(std::min<size_t>(timed.size(), 32));
    std::string s = ",\"tuned\":[";
    for (size_t i = 0; i < timed.size(); ++i) {
        char ms[32];
        snprintf(ms, sizeof(ms), "%.4f", timed[i].first);
        s += std::string(i ? "," : "") + "{\"split\":\"" + choice_label(timed[i].second, chirp) + "\",\"ms\":" + ms + "}";
    }
    return s + "]";
}

int create_plan(gfftx_plan* out, uint64_t n, uint64_t batch, int vtype, int ttype, int place, int device,
                uint32_t flags)
{
    // a real plan is timed with the split fused into its last (forward) or first (inverse)
    // pass, and every candidate runs with the plan's own placement (one buffer or two), so
    // the choice is kept per transform kind and place; forward and inverse complex transforms
    // share it
    const bool tune = !(flags & (GFFTX_FLAG_NO_AUTOTUNE | GFFTX_FLAG_SPLIT_MFMA)) && env_int("GFFTX_AUTOTUNE", 1) != 0 &&
                      !getenv("GFFTX_PASSES");
    std::string key;
    std::vector<int> chosen;
    std::string note;
    if (tune) {
        const int prec = (vtype == GFFTX_DOUBLE || vtype == GFFTX_COMPLEX_DOUBLE) ? PREC_F64 : PREC_F32;
        key = tune_key(device, prec, n, batch) +
              (ttype == GFFTX_RDFT ? "|rdft" : ttype == GFFTX_IRDFT ? "|irdft" : "") +
              (place == GFFTX_IN_PLACE ? "|ip" : "|oop");
        // a measured choice: the plan is built with it at once (a plan that cannot be built this
        // way, or at all, is built by the cost model below, which says why not)
        if (tune_get(key, &chosen)) {
            if (create_plan_impl(out, n, batch, vtype, ttype, place, device, flags, chosen, ",\"tuned\":\"cache\"") ==
                GFFTX_SUCCESS)
                return GFFTX_SUCCESS;
            return create_plan_impl(out, n, batch, vtype, ttype, place, device, flags, {}, "");
        }
    }
    int rc = create_plan_impl(out, n, batch, vtype, ttype, place, device, flags, {}, "");
    if (rc != GFFTX_SUCCESS) return rc;
    gfftx_plan_s* p = *out;
    // a batched single-pass plan is tuned over the tiles of its length (shape and radices), a
    // multi-pass plan over pass splits and tile shapes
    const bool single_pass = p->passes.size() == 1 && p->passes[0].k && p->passes[0].items_in_ntrans;
    const bool chirp = p->blue_m != 0;  // convolution lengths, their splits and the passes' shapes
    if (!tune || (p->passes.size() < 2 && !single_pass && !chirp)) return GFFTX_SUCCESS;
    {
        std::vector<std::vector<int>> splits;
        // a single-pass plan is timed against pass splits where its workgroups leave most of
        // the device idle: no more than the CUs for a run-time tile, 8 (one per XCD) for a
        // compiled one of a complex transform, from 2048 points up
        const uint64_t tiles = single_pass ? (batch + p->passes[0].k->nb - 1) / p->passes[0].k->nb : 0;
        const uint64_t few = single_pass ? (p->passes[0].k->mix ? device_cus(device) : p->real ? 0 : 8) : 0;
        if (!chirp && (!single_pass || (n >= 2048 && tiles <= few)))
            splits = tuned_splits(p->prec, n, (size_t)env_int("GFFTX_TUNE_CANDIDATES", 5), batch, device_cus(device), p->real_part());
        // an inverse real transform's first pass carries the C2R pre-split, which halves the runs of
        // its rows: its two-pass splits are timed in the other order too
        if (p->real && p->inverse)
            for (size_t i = splits.size(); i-- > 0;)
                if (splits[i].size() == 2 && splits[i][0] != splits[i][1] && find_tile(p->prec, splits[i][1], true, false))
                    splits.push_back({splits[i][1], splits[i][0]});
        std::vector<std::vector<int>> cands = split_variants(p->prec, n, batch, device_cus(device), splits);
        if (single_pass)
            for (const TileEntry* e : tile_shapes(p->prec, (int)n, false, false)) cands.push_back({(int)n, 1, 0, e->nb, e->wg});
        if (chirp) cands = chirp_candidates(p->prec, n, batch, device_cus(device), 6);
        if (cands.size() < 2) return GFFTX_SUCCESS;
        DeviceGuard g(device);
        // the candidates run on at most 1 GiB of data (a larger batch is timed on a prefix of
        // its items), so tuning never doubles a large plan's memory; the prefix still exceeds
        // the 256 MB Infinity Cache, so the timings see HBM as the plan will
        const size_t item_bytes = (size_t)p->dist * elem_bytes(p->prec);
        const uint64_t tbatch = std::min<uint64_t>(batch, std::max<uint64_t>(1, (1ull << 30) / item_bytes));
        TuneArrays arrays;
        // no room to tune: keep the cost-model plan
        if (!arrays.make(p->prec, item_bytes * tbatch, place == GFFTX_IN_PLACE, !single_pass && !chirp)) return GFFTX_SUCCESS;
        // the candidates are the plan's own transform (a real forward plan times its last pass with the
        // R2C split fused in) with its own placement: an in-place plan runs on one buffer, which the caches
        // treat differently from two; the arrays cover the bins layout
        SplitTable split;
        split.tw = p->split_tw;
        TuneRun run{arrays, [&](const std::vector<int>& c) {
            gfftx_plan cp = nullptr;
            (void)create_plan_impl(&cp, n, tbatch, vtype, ttype, place, device, flags & GFFTX_FLAG_R2C_BINS, c, "", &split);
            return cp;
        }};
        std::vector<float> cms(cands.size(), -1.f);  // time of each candidate (-1: failed)
        for (size_t i = 0; i < cands.size(); ++i) cms[i] = run.time(cands[i]);
        if (chirp && !run.chosen.empty()) {
            for (size_t i = 0; i < 5; ++i)
                for (const std::vector<int>& c : chirp_variants(p->prec, n, run.chosen, i)) run.time(c);
        } else if (!run.chosen.empty() && run.chosen[1] != 1) {
            // the combination of the fastest variants, for each of the three fastest splits
            std::vector<size_t> order(cands.size());
            for (size_t i = 0; i < order.size(); ++i) order[i] = i;
            std::stable_sort(order.begin(), order.end(), [&](size_t x, size_t y) { return cms[x] < cms[y]; });
            std::vector<std::vector<int>> seen;
            for (size_t i : order) {
                std::vector<int> l;
                std::vector<std::pair<int, int>> t;
                split_choice(cands[i], l, t);
                if (cms[i] < 0 || (l.size() == 2 && l[1] == 1) || std::find(seen.begin(), seen.end(), l) != seen.end()) continue;
                seen.push_back(l);
                const std::vector<int> combo = best_combination(cands[i], cands, cms);
                if (!combo.empty()) run.time(combo);
                if (seen.size() == 3) break;
            }
        }
        note = tune_note(run.timed, chirp);
        run.again(6);
        if (run.chosen.empty()) return GFFTX_SUCCESS;
        chosen = chirp ? run.chosen : with_tiles(p->prec, n, tbatch, device_cus(device), run.chosen);
        std::lock_guard<std::mutex> lk(g_tune_mu);
        g_tune[key] = chosen;
        tune_store();
    }
    gfftx_plan q = nullptr;
    rc = create_plan_impl(&q, n, batch, vtype, ttype, place, device, flags, chosen, note);
    if (rc != GFFTX_SUCCESS) return GFFTX_SUCCESS;  // keep the cost-model plan
    gfftx_plan_destroy(p);
    *out = q;
    return GFFTX_SUCCESS;
}

// Plan choice for one length class of a ragged batch (count transforms of length L): every
// compiled single-pass tile of the length against the cost model's best three pass splits,
// each timed on a contiguous batch of the class's size, stored the way the class stores: plainly, and
// non-temporally at the end where the whole batch is (`nt`).  Returns false when nothing was
// measured (autotuning off, or no buffers), and the caller keeps its built-in rule.  Cached
// like plans, under the class's own key; a single-pass choice is stored as [L, 1, 0, nb, wg]
// and returned with *single set and the tile's shape in *nb, *wg.
bool tune_length_class(int device, int prec, long long L, long long count, bool inverse, bool nt, bool* single,
                       std::vector<int>* lens, std::vector<std::pair<int, int>>* tiles)
{
    if (env_int("GFFTX_AUTOTUNE", 1) == 0) return false;
    const bool has_single = L <= (1 << 30) && find_tile(prec, (int)L, false, false) != nullptr;
    const std::vector<std::vector<int>> splits = tuned_splits(prec, (unsigned long long)L, 3, (unsigned long long)count,
                                                              device_cus(device));
    if ((has_single ? 1 : 0) + splits.size() < 2) return false;
    const std::string key = tune_key(device, prec, (uint64_t)L, (uint64_t)count) + (nt ? "|class|nt" : "|class");
    std::vector<int> chosen;
    {
        std::lock_guard<std::mutex> lk(g_tune_mu);
        tune_load();
        auto it = g_tune.find(key);
        if (it != g_tune.end()) chosen = it->second;
    }
    if (chosen.empty()) {
        std::vector<std::vector<int>> cands;
        if (has_single)
            for (const TileEntry* e : tile_shapes(prec, (int)L, false, false)) cands.push_back({(int)L, 1, 0, e->nb, e->wg});
        for (const std::vector<int>& sp : split_variants(prec, (unsigned long long)L, (unsigned long long)count,
                                                         device_cus(device), splits))
            cands.push_back(sp);
        DeviceGuard g(device);
        // at most 1 GiB of data, like plan tuning
        const uint64_t tcount = std::min<uint64_t>((uint64_t)count,
                                                   std::max<uint64_t>(1, (1ull << 30) / ((size_t)L * elem_bytes(prec))));
        TuneArrays arrays;
        // (in place, as the classes of a ragged batch run)
        if (!arrays.make(prec, (size_t)L * tcount * elem_bytes(prec), true, true)) return false;
        const int cvt = prec == PREC_F64 ? GFFTX_COMPLEX_DOUBLE : GFFTX_COMPLEX_FLOAT;
        TuneRun run{arrays, [&](const std::vector<int>& c) {
            gfftx_plan cp = nullptr;
            if (create_plan_impl(&cp, (uint64_t)L, tcount, cvt, inverse ? GFFTX_IDFT : GFFTX_DFT, GFFTX_IN_PLACE, device,
                                 GFFTX_FLAG_NO_AUTOTUNE, c, "") == GFFTX_SUCCESS) {
                cp->through = false;
                cp->nt = nt ? 1 : 0;
            }
            return cp;
        }};
        std::vector<float> cms(cands.size(), -1.f);
        for (size_t i = 0; i < cands.size(); ++i) cms[i] = run.time(cands[i]);
        if (run.chosen.empty()) return false;
        if (!(run.chosen[1] == 1 && run.chosen[0] == (int)L)) {
            const std::vector<int> combo = best_combination(run.chosen, cands, cms);
            if (!combo.empty()) run.time(combo);
        }
        run.again(3);  // (a batch may have dozens of classes)
        chosen = with_tiles(prec, (unsigned long long)L, tcount, device_cus(device), run.chosen);
        std::lock_guard<std::mutex> lk(g_tune_mu);
        g_tune[key] = chosen;
        tune_store();
    }
    split_choice(chosen, *lens, *tiles);
    *single = lens->size() == 2 && (*lens)[1] == 1;
    if (*single) lens->clear();
    return true;
}

}  // namespace detail
}  // namespace gfftx
