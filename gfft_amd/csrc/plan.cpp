// plan.cpp -- plans of the gfx950 FFT engine: construction, execution and C ABI.
//
// A plan is a list of passes over device buffers.  A transform whose length fits one LDS
// tile is one batched pass; a longer one is a Stockham decomposition into "super radices"
// N = P_0 * P_1 * ... each executed as one pass of the tile kernel (see tile_kernel.h).
// Twiddles are generated here once per plan from long-double evaluations with octant
// argument reduction and stored in the working precision (stage tables) or FP64 (pass
// tables).  GFFT evaluates the same roots W_N = exp(-2 pi i/N) at compile time to 18
// digits (src/metaroot.h:104-120) and then runs a recurrence at run time
// (src/gfftalg.h:249-261); tables avoid the recurrence's error growth.
#include "plan_internal.h"

#include <system_error>

namespace gfftx {
namespace detail {

thread_local std::string g_last_error;

}  // namespace detail
}  // namespace gfftx

namespace gfftx {
namespace detail {

int fail(int code, const char* fmt, ...)
{
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof(buf), fmt, ap);
    va_end(ap);
    g_last_error = buf;
    return code;
}

bool nt_output(size_t bytes)
{
    const long long mib = env_int("GFFTX_NT_STORE_MIB", 256);
    return mib >= 0 && bytes > (size_t)mib << 20;
}

// How pass `ps`, number i of m, stores its `bytes` of output (STORE_*, tile_kernel.h): non-temporally at
// the end of a large call, through the L2 where that pays, else plainly.
//
// Through the L2 from 2 MiB (below, the shorter way of a plain store counts more: 59049 FP64, 0.9 MiB,
// 12.2 us plain, 12.7 through) to 64 MiB (2^23 FP32, 74.0 us plain, 69.4 through; 2^20 x 16 FP32, 128 MiB,
// 143-147 plain, 148 through) where the tile writes whole 128-byte lines.  Parts of lines are written by
// themselves, so with them the gain ends at 16 MiB (823543 x 5 FP32, 31 MiB, 49.5 -> 51.9 and 3000000
// FP64, 46 MiB, 67.8 -> 74.2), and with rows below 64 bytes it begins at 8 (524288 FP32 ending in 512,
// 4 MiB, 16.0 -> 16.5 us; 2^20 FP32, 17.4 -> 15.9).
//
// The pass of a real transform's split, plain -> through, us:
//   forward (rows half as long, beginning anywhere): half rows of 256 bytes 28.4 -> 27.1 (2^21 FP32, 16 MiB),
//   81.8 -> 80.3 (2^22 FP64, 64 MiB); of 128 bytes 17.9 -> 17.4 (2^18 FP64), 47.5 -> 44.5 (2^21 FP64, 32 MiB),
//   84.6 -> 83.7 (2^23 FP32, 64 MiB); of 64 bytes 16.2 -> 15.8 (2^18 FP32, 2 MiB), 161.5 -> 167.9 (2^24 FP32,
//   128 MiB); of 32 bytes 25.6 -> 26.3 (2^20 FP32), 32.7 -> 34.6 (FP64);
//   inverse (whole sequences, a pair's elements side by side): FP32 17.7 -> 21.5 (2^18, 2 MiB), 26.5 -> 27.3
//   (2^20, 8 MiB), 34.6 -> 32.3 (3 * 2^19, 12 MiB), 38.2 -> 34.7 (2^21), 53.9 -> 53.8 (2^22, 32 MiB), 85.5 ->
//   89.8 (2^23); FP64 17.5 -> 20.4 (2^17, 2 MiB), 27.7 -> 29.3 (2^19, 8 MiB), 36.3 -> 36.1 (2^20, 16 MiB), with the
//   passes behind it through as well 55.6 -> 51.8 (2^21, 32 MiB), 83.7 -> 88.5 (2^22).
// Non-temporally, the forward split's pass wants half rows of 256 bytes: 2^25 FP64 811 -> 778 us, 2^26 FP32 897
// -> 855, but 2^24 FP64 (128 bytes) 336 -> 389 and 2^25 FP32 (128 bytes) 424 -> 433.
// GFFTX_THROUGH_STORE=0 (when the plan is made): never through.
int pass_store(bool through, bool nt, size_t i, size_t m, size_t bytes, const Pass& ps, size_t dist, size_t items)
{
    const TileEntry& k = *ps.k;
    const size_t eb = elem_bytes(k.prec), half = (size_t)k.nb / 2 * eb;
    const bool post = k.real == REAL_POST && k.loadT;
    if (nt && i + 1 == m) return post && half < 256 ? STORE_PLAIN : STORE_NT;
    if (m < 2 || !through) return STORE_PLAIN;
    auto lines = [&](size_t elems) { return elems * eb % 128 == 0; };
    size_t least = 2, most;  // MiB
    if (post) most = half >= 128 ? 64 : half >= 64 ? 16 : 0;
    else if (items > 1 && !lines(dist)) most = 16;
    else if (k.storeT) most = lines(k.nb) && lines(ps.ns_pass) ? 64 : 16;
    else if (k.real == REAL_PRE) most = lines(k.L) ? 32 : 16;
    else most = lines((size_t)k.nb * k.L) ? 64 : 16;
    if (k.real == REAL_PRE) least = k.prec == PREC_F64 ? 16 : 12;
    else if (k.storeT && !post && (size_t)k.nb * eb < 64) least = 8;
    return bytes >= least << 20 && bytes <= most << 20 ? STORE_THROUGH : STORE_PLAIN;
}

int dev_alloc(gfftx_plan_s* p, void** out, size_t bytes)
{
    if (bytes == 0) bytes = 16;
    hipError_t e = hipMalloc(out, bytes);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        return fail(GFFTX_ERR_ALLOC, "hipMalloc(%zu) failed: %s", bytes, hipGetErrorString(e));
    }
    p->allocs.push_back(*out);
    return GFFTX_SUCCESS;
}

int upload_stage_table(gfftx_plan_s* p, const TileEntry* k, void** out)
{
    return upload_tile_table(p->allocs, k, out);
}

int upload_pass_table(gfftx_plan_s* p, Pass& ps, long long M)
{
    ps.ptw_m = M;
    return upload_root_tables(p->allocs, M, &ps.ptw_lo, &ps.ptw_hi, &ps.ptw_shift);
}

int build_c2c_passes(gfftx_plan_s* p)
{
    const unsigned long long n = p->n;
    char buf[256];
    p->desc = "{\"n\":" + std::to_string(n) + ",\"batch\":" + std::to_string(p->batch) +
              ",\"precision\":\"" + (p->prec == PREC_F64 ? "f64" : "f32") + "\",\"passes\":[";
    if (p->flags & GFFTX_FLAG_SPLIT_MFMA) {
        const MfmaEntry* me = nullptr;
        const char* sm = getenv("GFFTX_MFMA_SCALE");
        const int want = (sm && !strcmp(sm, "column")) ? MFMA_SCALE_COLUMN : MFMA_SCALE_STAGE;
        for (int i = 0; i < kNumMfma && !me; ++i)
            if ((unsigned long long)kMfma[i].L == n && kMfma[i].scale == want) me = &kMfma[i];
        if (p->prec != PREC_F32 || p->real || !me)
            return fail(GFFTX_ERR_UNSUPPORTED, "split-precision MFMA path: FP32 C2C of length 256 or 4096 only (n=%llu)", n);
        Pass ps;
        ps.mfma = me;
        ps.items_in_ntrans = true;
        ps.ntrans = (long long)p->batch;
        // per-stage scaling: each stage after the first takes its input times 2^-4 through
        // the twiddles (exact: a power of two)
        int rc = upload_mfma_twiddles(p->allocs, me->scale == MFMA_SCALE_STAGE ? 0.0625 : 1.0, &ps.stage_tw);
        if (rc) return rc;
        rc = upload_mfma_matrix(p->allocs, &ps.amat);
        if (rc) return rc;
        p->passes.push_back(ps);
        snprintf(buf, sizeof(buf), "{\"kernel\":\"%s\",\"L\":%d,\"ntrans\":%lld}", me->name, me->L, ps.ntrans);
        p->desc += buf;
        p->desc += "]}";
        return GFFTX_SUCCESS;
    }
    // a forced choice (autotuner candidates, tuning cache): [n, 1, 0, nb, wg] names a
    // single-pass tile; any other list is a pass split, which overrides the single-pass tile
    const bool forced_single = p->forced_lens.size() >= 2 && p->forced_lens[0] == (int)n && p->forced_lens[1] == 1;
    const TileEntry* single = nullptr;
    if (p->forced_lens.empty() || forced_single) {
        std::vector<int> fl;
        std::vector<std::pair<int, int>> ft;
        split_choice(p->forced_lens, fl, ft);
        single = single_tile(p->prec, n, ft.empty() ? 0 : ft[0].first, ft.empty() ? 0 : ft[0].second);
    }
    if (single) {
        const TileEntry* k = single;
        Pass ps;
        ps.k = k;
        ps.items_in_ntrans = true;
        ps.ntrans = (long long)p->batch;
        ps.its = (long long)p->dist;
        ps.ies = 1;
        ps.ns_pass = 1;
        ps.bdist = 0;
        ps.batch = 1;
        int rc = upload_stage_table(p, k, &ps.stage_tw);
        if (rc) return rc;
        // real transform: the split runs inside the tile (after the last stage forward, before
        // the first stage inverse) when the tile has such a variant
        if (p->real && env_int("GFFTX_FUSED_SPLIT", 1)) {
            if (const TileEntry* kr = find_real_tile(k, p->inverse ? REAL_PRE : REAL_POST)) {
                if (kr->mix) rc = upload_tile_table(p->allocs, kr, &ps.stage_tw);  // its own stages
                if (rc) return rc;
                ps.k = kr;
                ps.real = kr->real;
                rc = upload_root_tables(p->allocs, (long long)(2 * n), &ps.sp_lo, &ps.sp_hi, &ps.sp_shift);
                if (rc) return rc;
                p->split_fused = true;
            }
        }
        p->passes.push_back(ps);
        snprintf(buf, sizeof(buf), "{\"kernel\":\"%s\",\"L\":%d,\"ntrans\":%lld}", ps.k->name, k->L, ps.ntrans);
        p->desc += buf;
    } else {
        std::vector<int> lens;
        std::vector<std::pair<int, int>> tiles;
        split_choice(p->forced_lens, lens, tiles);
        if (lens.empty() && !choose_passes(p->prec, n, lens, p->batch, device_cus(p->device), p->real_part()))
            return fail(GFFTX_ERR_UNSUPPORTED, "no multi-pass decomposition for n=%llu", n);
        if (!passes_fit(lens, n)) return fail(GFFTX_ERR_UNSUPPORTED, "passes that do not multiply to n=%llu", n);
        long long ns = 1;
        for (size_t i = 0; i < lens.size(); ++i) {
            const int L = lens[i];
            const int want_nb = i < tiles.size() && tiles[i].first ? tiles[i].first : env_int("GFFTX_TNB", 0);
            const int want_wg = i < tiles.size() && tiles[i].first ? tiles[i].second : env_int("GFFTX_TWG", 0);
            const TileEntry* k = want_nb || want_wg ? find_tile(p->prec, L, true, i > 0, want_nb, want_wg)
                                                    : pass_tile(p->prec, L, (unsigned long long)ns, n, p->batch, device_cus(p->device));
            if (!k) return fail(GFFTX_ERR_UNSUPPORTED, "no pass kernel L=%d", L);
            Pass ps;
            ps.k = k;
            ps.xcd = xcd_remap(k, p->prec);
            ps.ntrans = (long long)(n / L);
            ps.its = 1;
            ps.ies = (long long)(n / L);
            ps.ns_pass = ns;
            ps.bdist = (long long)p->dist;
            ps.batch = (unsigned)p->batch;
            int rc = upload_stage_table(p, k, &ps.stage_tw);
            if (rc) return rc;
            if (ns > 1) {
                rc = upload_pass_table(p, ps, ns * L);
                if (rc) return rc;
            }
            p->passes.push_back(ps);
            // real transform: the last pass of a forward transform computes the R2C split, the
            // first pass of an inverse one the C2R pre-pass, when the tile has a fused variant
            const bool fuse_here = p->inverse ? i == 0 : i + 1 == lens.size();
            if (fuse_here && p->real && env_int("GFFTX_FUSED_SPLIT", 1)) {
                if (const TileEntry* ks = find_real_tile(k, p->inverse ? REAL_PRE : REAL_POST)) {
                    Pass& pr = p->passes.back();
                    pr.k = ks;
                    pr.real = ks->real;
                    rc = upload_root_tables(p->allocs, (long long)(2 * n), &pr.sp_lo, &pr.sp_hi, &pr.sp_shift);
                    if (rc) return rc;
                    p->split_fused = true;
                }
            }
            snprintf(buf, sizeof(buf), "%s{\"kernel\":\"%s\",\"L\":%d,\"ns\":%lld,\"ntrans\":%lld,\"xcd\":%d}",
                     i ? "," : "", p->passes.back().k->name, L, ns, ps.ntrans, ps.xcd);
            p->desc += buf;
            ns *= L;
        }
    }
    p->desc += "]" + p->tune_note + "}";
    return GFFTX_SUCCESS;
}

// W_{2n}^k, k = 0..n/2 (n even), in the working precision.  Entries above n/4 mirror those below
// (root_ld folds an angle to the first octant, so the bits are those of an evaluation), and the
// others are shared out to up to 8 threads: 2^24 + 1 entries took one thread 3.8 s.
template <typename T> std::vector<T> split_roots(long long n)
{
    std::vector<T> t(2 * (n / 2 + 1));
    const long long direct = n / 4 + 1;  // k <= n/4
    auto part = [&](long long lo, long long hi) {
        for (long long k = lo; k < hi; ++k) {
            long double c, s;
            root_ld(k, 2 * n, &c, &s);
            t[2 * k] = (T)c;
            t[2 * k + 1] = (T)s;
        }
    };
    const long long want = std::min<long long>({8, std::max(1u, std::thread::hardware_concurrency()), direct >> 15});
    std::vector<std::thread> th;
    long long done = 0;
    for (long long i = 1; i < want; ++i) {
        const long long hi = direct * i / want;
        try {
            th.emplace_back(part, done, hi);
        } catch (const std::system_error&) {
            break;  // no more threads: the rest below
        }
        done = hi;
    }
    part(done, direct);
    for (auto& x : th) x.join();
    for (long long k = direct; k <= n / 2; ++k) {
        t[2 * k] = -t[2 * (n / 2 - k) + 1];
        t[2 * k + 1] = -t[2 * (n / 2 - k)];
    }
    return t;
}
template std::vector<float> split_roots<float>(long long n);
template std::vector<double> split_roots<double>(long long n);

int upload_split_table(std::vector<void*>& owned, int prec, long long n, void** out)
{
    auto up = [&](const auto& t) -> int {
        const size_t bytes = t.size() * sizeof(t[0]);
        const int rc = dev_alloc_list(owned, out, bytes);
        if (rc) return rc;
        HIP_TRY(hipMemcpy(*out, t.data(), bytes, hipMemcpyHostToDevice));
        return GFFTX_SUCCESS;
    };
    return prec == PREC_F64 ? up(split_roots<double>(n)) : up(split_roots<float>(n));
}

bool is_device_ptr(const void* ptr)
{
    hipPointerAttribute_t attr;
    hipError_t e = hipPointerGetAttributes(&attr, ptr);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    return attr.type == hipMemoryTypeDevice || attr.type == hipMemoryTypeManaged;
}

// Event pair for launch slot `slot` (GFFTX_FLAG_PROFILE); returns false when not profiling.
// With `attached` the pair goes to the launch itself (hipExtLaunchKernel stamps the kernel's
// start and end); otherwise the events are recorded on s around the launch.
bool prof_begin(gfftx_plan_s* p, size_t slot, const char* name, hipStream_t s, std::pair<hipEvent_t, hipEvent_t>* ev,
                bool attached)
{
    if (!(p->flags & GFFTX_FLAG_PROFILE) || p->capturing || p->no_events) return false;
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;  // a capture the caller runs
    if (hipStreamIsCapturing(s, &cs) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    if (cs != hipStreamCaptureStatusNone) return false;
    if (p->slots.size() <= slot) p->slots.resize(slot + 1);
    gfftx_plan_s::Slot& sl = p->slots[slot];
    sl.name = name;
    if (sl.pool.empty()) {
        hipEvent_t a, b;
        if (hipEventCreate(&a) != hipSuccess || hipEventCreate(&b) != hipSuccess) {
            (void)hipGetLastError();
            return false;
        }
        sl.pool.push_back({a, b});
    }
    *ev = sl.pool.back();
    sl.pool.pop_back();
    if (!attached) (void)hipEventRecord(ev->first, s);
    return true;
}

void prof_end(gfftx_plan_s* p, size_t slot, hipStream_t s, const std::pair<hipEvent_t, hipEvent_t>& ev, bool attached)
{
    if (!attached) (void)hipEventRecord(ev.second, s);
    p->slots[slot].pending.push_back(ev);
}

// Runs the pass list of `p` on batch items `r` of the arrays `in`/`out` (base pointers of
// the whole batch).
int run_passes(gfftx_plan_s* p, const void* in, void* out, hipStream_t s, Range r)
{
    if (!r.nb) r.nb = p->batch;
    const size_t off = (size_t)r.b0 * p->dist * elem_bytes(p->prec);
    auto at = [off](const void* q) { return (void*)((char*)const_cast<void*>(q) + off); };
    const size_t m = p->passes.size();
    // buffer for the output of pass i (i < m-1): alternate so that no pass is in place and
    // the caller's input is never written unless it is also the output
    void* const s0 = p->call_scratch[0] ? p->call_scratch[0] : p->scratch[0];
    void* const s1 = p->call_scratch[0] ? p->call_scratch[1] : p->scratch[1];
    void* dst[32];
    if (m == 0 || m > 32) return fail(GFFTX_ERR_INVALID_ARG, "plan with %zu passes", m);
    dst[m - 1] = out;
    for (size_t i = m - 1; i-- > 0;) {
        void* next_src_dst = dst[i + 1];
        void* cand = (next_src_dst == s0) ? out : s0;
        if (cand == in || cand == next_src_dst) cand = s1;
        dst[i] = cand;
    }
    const void* src = in;
    for (size_t i = 0; i < m; ++i) {
        const Pass& ps = p->passes[i];
        if (ps.mfma) {
            MfmaArgs ma;
            ma.in = (const float2*)at(src);
            ma.out = (float2*)at(dst[i]);
            ma.ntrans = (long long)r.nb;
            ma.tw = (const float2*)ps.stage_tw;
            ma.amat = (const _Float16*)ps.amat;
            ma.conj_in = p->inverse ? 1 : 0;
            ma.conj_out = p->inverse ? 1 : 0;
            ma.scale = p->inverse ? (float)(1.0 / (double)p->n) : 1.0f;
            ma.nt_out = (r.nt && i == m - 1) ? 1 : 0;
            dim3 grid((unsigned)((ma.ntrans + ps.mfma->nb - 1) / ps.mfma->nb));
            std::pair<hipEvent_t, hipEvent_t> ev;
            const bool on = prof_begin(p, i, ps.mfma->name, s, &ev, true);
            hipError_t e = ps.mfma->launch(ma, grid, s, on ? ev.first : nullptr, on ? ev.second : nullptr);
            if (on) prof_end(p, i, s, ev, true);
            if (e != hipSuccess) return fail(GFFTX_ERR_LAUNCH, "%s: %s", ps.mfma->name, hipGetErrorString(e));
            src = dst[i];
            continue;
        }
        TileArgs a;
        memset(&a, 0, sizeof(a));
        a.in = at(src);
        a.out = at(dst[i]);
        a.ntrans = ps.items_in_ntrans ? (long long)r.nb : ps.ntrans;
        a.its = ps.its;
        a.ies = ps.ies;
        a.ns_pass = ps.ns_pass;
        a.bdist = ps.bdist;
        a.tw = ps.stage_tw;
        a.ptw_lo = ps.ptw_lo;
        a.ptw_hi = ps.ptw_hi;
        a.ptw_shift = ps.ptw_shift;
        a.conj_in = (p->inverse && i == 0) ? 1 : 0;
        a.conj_out = (p->inverse && i == m - 1) ? 1 : 0;
        a.scale = (p->inverse && i == m - 1) ? 1.0 / (double)p->n : 1.0;
        a.xcd = ps.xcd;
        a.store = pass_store(p->through, r.nt, i, m, (size_t)p->dist * r.nb * elem_bytes(p->prec), ps, p->dist, r.nb);
        const long long nb = ps.k->nb;
        unsigned ntiles = (unsigned)((a.ntrans + nb - 1) / nb);
        if (ps.real) {
            a.sp_lo = ps.sp_lo;
            a.sp_hi = ps.sp_hi;
            a.sp_shift = ps.sp_shift;
            a.split_bins = (p->flags & GFFTX_FLAG_R2C_BINS) ? 1 : 0;
            a.nfull = (long long)p->n;
            if (ps.k->loadT) {
                // paired T-mode tiles: tile 0 takes sequences 0 and S/2, then nb/2 pairs
                // (p, S - p), 1 <= p <= (S-1)/2
                const long long pairs = (a.ntrans - 1) / 2, h = nb / 2;
                ntiles = (unsigned)(1 + (pairs + h - 1) / h);
            }
        }
        dim3 grid(ntiles, ps.items_in_ntrans ? 1u : (unsigned)r.nb);
        std::pair<hipEvent_t, hipEvent_t> ev;
        const bool on = prof_begin(p, i, ps.k->name, s, &ev, true);
        hipError_t e = launch_entry(ps.k, a, grid, s, on ? ev.first : nullptr, on ? ev.second : nullptr);
        if (on) prof_end(p, i, s, ev, true);
        if (e != hipSuccess) return fail(GFFTX_ERR_LAUNCH, "%s: %s", ps.k->name, hipGetErrorString(e));
        src = dst[i];
    }
    return GFFTX_SUCCESS;
}

// Launch slots the complex transform of `p` uses (profiling); the split pass comes next.
size_t c2c_slots(const gfftx_plan_s* p)
{
    return p->blue_m ? p->blue.size() : p->passes.size();
}

int run_c2c(gfftx_plan_s* p, const void* in, void* out, hipStream_t s, Range r)
{
    return p->blue_m ? run_bluestein(p, in, out, s, r) : run_passes(p, in, out, s, r);
}

int run_split(gfftx_plan_s* p, void* data, hipStream_t s, Range r)
{
    if (!r.nb) r.nb = p->batch;
    SplitArgs a;
    a.data = (char*)data + (size_t)r.b0 * p->dist * elem_bytes(p->prec);
    a.n = (long long)p->n;
    a.bdist = (long long)p->dist;
    a.nbatch = (long long)r.nb;
    a.tw = p->split_tw;
    a.inverse = p->inverse ? 1 : 0;
    a.bins = (p->flags & GFFTX_FLAG_R2C_BINS) ? 1 : 0;
    std::pair<hipEvent_t, hipEvent_t> ev;
    const size_t slot = c2c_slots(p);
    const bool prof = prof_begin(p, slot, "split_kernel", s, &ev, false);
    hipError_t e = launch_split(p->prec, a, s);
    if (prof) prof_end(p, slot, s, ev, false);
    if (e != hipSuccess) return fail(GFFTX_ERR_LAUNCH, "split: %s", hipGetErrorString(e));
    return GFFTX_SUCCESS;
}

// Full transform on device pointers.  Real forward: complex FFT then split on the output.
// Real inverse: split on a copy of the input (the input of an out-of-place call is left
// unchanged), then the inverse complex FFT.  A plan whose split is fused into one of its
// passes runs the complex passes only.
// `r` selects batch items (all by default); in and out are the base pointers of the batch.
int exec_device(gfftx_plan_s* p, const void* in, void* out, hipStream_t s, Range r)
{
    if (!r.nb) {
        // a call over the whole batch on device arrays: nothing in the call reads its output
        // back, so a large one is stored non-temporally (the host path's staged chunks are
        // copied out right after, and stay cached)
        r.nb = p->batch;
        r.nt = p->nt < 0 ? nt_output((size_t)p->dist * p->batch * elem_bytes(p->prec)) : p->nt != 0;
    }
    if (!p->real || p->split_fused) return run_c2c(p, in, out, s, r);
    if (!p->inverse) {
        Range rt = r;
        rt.nt = false;  // the split kernel reads the transform's output
        int rc = run_c2c(p, in, out, s, rt);
        if (rc) return rc;
        return run_split(p, out, s, r);
    }
    void* work = out;
    if (in != out) {
        work = p->real_work;
        const size_t eb = elem_bytes(p->prec), off = (size_t)r.b0 * p->dist * eb;
        HIP_TRY(hipMemcpyAsync((char*)work + off, (const char*)in + off, (size_t)p->dist * r.nb * eb,
                               hipMemcpyDeviceToDevice, s));
    }
    int rc = run_split(p, work, s, r);
    if (rc) return rc;
    return run_c2c(p, work, out, s, r);
}

// Replays the plan's launches as one captured hipGraph, one per (in, out) pair (the last
// eight kept).  Capture happens on a plan-owned stream; the graph is launched on the caller's.
int exec_graph(gfftx_plan_s* p, const void* in, void* out, hipStream_t s)
{
    GraphCache::Entry* g = p->graphs.find(in, out);
    if (!g) {
        if (!p->graphs.cap_stream) HIP_TRY(hipStreamCreateWithFlags(&p->graphs.cap_stream, hipStreamNonBlocking));
        HIP_TRY(hipStreamBeginCapture(p->graphs.cap_stream, hipStreamCaptureModeThreadLocal));
        p->capturing = true;
        const int rc = exec_device(p, in, out, p->graphs.cap_stream);
        p->capturing = false;
        hipGraph_t gr = nullptr;
        const hipError_t ce = hipStreamEndCapture(p->graphs.cap_stream, &gr);
        if (rc) {
            if (gr) (void)hipGraphDestroy(gr);
            return rc;
        }
        if (ce != hipSuccess) return fail(GFFTX_ERR_DEVICE, "end capture: %s", hipGetErrorString(ce));
        g = p->graphs.take();
        g->graph = gr;
        const hipError_t ie = hipGraphInstantiate(&g->exec, gr, nullptr, nullptr, 0);
        if (ie != hipSuccess) {
            GraphCache::release(*g);
            return fail(GFFTX_ERR_DEVICE, "graph instantiate: %s", hipGetErrorString(ie));
        }
        g->in = in;
        g->out = out;
        g->used = ++p->graphs.tick;
    }
    HIP_TRY(GraphCache::launch(*g, s));
    return GFFTX_SUCCESS;
}

int exec_dispatch(gfftx_plan_s* p, const void* in, void* out, hipStream_t s)
{
    // one pointer query per distinct array (an in-place call asks once)
    const bool din = is_device_ptr(in), dout = out == in ? din : is_device_ptr(out);
    if (din && dout && (p->flags & GFFTX_FLAG_GRAPH)) return exec_graph(p, in, out, s);
    // complex elements the caller's arrays hold: the real side of a real transform has n
    // per item, the complex side dist (n, or n+1 with the bins layout)
    const size_t full = (size_t)p->dist * p->batch, real_side = (size_t)p->dist * (p->batch - 1) + p->n;
    const size_t eb = elem_bytes(p->prec);
    size_t in_bytes = full * eb, out_bytes = full * eb;
    if (p->real && in != out) {
        if (p->inverse) out_bytes = real_side * eb;
        else in_bytes = real_side * eb;
    }
    if (din && dout) return exec_device(p, in, out, s);
    return exec_host(p, in, out, s, din, dout, in_bytes, out_bytes);
}

// One call of the plan: calls from several threads run one at a time, and a call on another
// stream than the previous call's waits until that call's work is done when the calls share
// device arrays (scratch, chirp-z work, graphs).
int exec_any(gfftx_plan_s* p, const void* in, void* out, hipStream_t s)
{
    std::lock_guard<std::mutex> lk(p->mu);
    DeviceGuard g(p->device);
    if (!g.ok) return fail(GFFTX_ERR_DEVICE, "cannot select device %d", p->device);
    if (p->shared_state) HIP_TRY(p->order.before(s));
    return exec_dispatch(p, in, out, s);
}

int create_plan_impl(gfftx_plan* out, uint64_t n, uint64_t batch, int vtype, int ttype, int place, int device,
                     uint32_t flags, const std::vector<int>& forced, const std::string& note, SplitTable* lent)
{
    if (!out) return fail(GFFTX_ERR_INVALID_ARG, "plan pointer is NULL");
    *out = nullptr;
    if (n == 0 || batch == 0) return fail(GFFTX_ERR_INVALID_ARG, "n and batch must be positive");
    if (vtype < 0 || vtype > 3) return fail(GFFTX_ERR_INVALID_ARG, "unknown value type %d", vtype);
    if (ttype < 0 || ttype > 3) return fail(GFFTX_ERR_INVALID_ARG, "unknown transform type %d", ttype);
    if (place != GFFTX_IN_PLACE && place != GFFTX_OUT_OF_PLACE)
        return fail(GFFTX_ERR_INVALID_ARG, "unknown place %d", place);
    if (flags & ~(GFFTX_FLAG_R2C_BINS | GFFTX_FLAG_SPLIT_MFMA | GFFTX_FLAG_NO_AUTOTUNE | GFFTX_FLAG_GRAPH |
                  GFFTX_FLAG_PROFILE))
        return fail(GFFTX_ERR_INVALID_ARG, "unknown flags 0x%x", flags);
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0) {
        (void)hipGetLastError();
        return fail(GFFTX_ERR_DEVICE, "no HIP device available");
    }
    if (device < 0 || device >= ndev) return fail(GFFTX_ERR_DEVICE, "device %d out of range (%d)", device, ndev);
    const bool real = ttype == GFFTX_RDFT || ttype == GFFTX_IRDFT;
    if (real && (n % 2))
        return fail(GFFTX_ERR_UNSUPPORTED, "real transforms need an even complex length (n=%llu)",
                    (unsigned long long)n);
    if ((flags & GFFTX_FLAG_R2C_BINS) && !real)
        return fail(GFFTX_ERR_INVALID_ARG, "GFFTX_FLAG_R2C_BINS applies to RDFT/IRDFT only");
    if ((flags & GFFTX_FLAG_R2C_BINS) && batch != 1)
        return fail(GFFTX_ERR_UNSUPPORTED, "the bins layout is available for batch 1 only");

    DeviceGuard g(device);
    if (!g.ok) return fail(GFFTX_ERR_DEVICE, "cannot select device %d", device);
    gfftx_plan_s* p = new (std::nothrow) gfftx_plan_s();
    if (!p) return fail(GFFTX_ERR_ALLOC, "host allocation failed");
    p->device = device;
    p->n = n;
    p->batch = batch;
    p->vtype = vtype;
    p->ttype = ttype;
    p->place = place;
    p->flags = flags;
    p->prec = (vtype == GFFTX_DOUBLE || vtype == GFFTX_COMPLEX_DOUBLE) ? PREC_F64 : PREC_F32;
    p->real = real;
    p->inverse = ttype == GFFTX_IDFT || ttype == GFFTX_IRDFT;
    p->dist = n + ((real && (flags & GFFTX_FLAG_R2C_BINS)) ? 1 : 0);
    p->forced_lens = forced;
    p->through = env_int("GFFTX_THROUGH_STORE", 1) != 0;
    p->tune_note = note;
    int rc = native_length(p->prec, n) ? build_c2c_passes(p) : build_bluestein(p);
    // an unfused split runs as a kernel of its own with a table; that of an out-of-place
    // IRDFT works on a copy of the input
    if (rc == GFFTX_SUCCESS && real && !p->split_fused) {
        if (!lent) {
            rc = upload_split_table(p->allocs, p->prec, (long long)n, &p->split_tw);
        } else {
            if (!lent->tw) rc = upload_split_table(lent->owned, p->prec, (long long)n, &lent->tw);
            p->split_tw = lent->tw;
        }
    }
    if (rc == GFFTX_SUCCESS && real && p->inverse && !p->split_fused)
        rc = dev_alloc(p, &p->real_work, (size_t)p->dist * batch * elem_bytes(p->prec));
    if (rc == GFFTX_SUCCESS && p->passes.size() > 1) {
        const size_t bytes = (size_t)p->dist * batch * elem_bytes(p->prec);
        rc = dev_alloc(p, &p->scratch[0], bytes);
        if (rc == GFFTX_SUCCESS && p->passes.size() > 2) rc = dev_alloc(p, &p->scratch[1], bytes);
    }
    if (rc != GFFTX_SUCCESS) {
        gfftx_plan_destroy(p);  // frees inner plans too; leaves the error message alone
        return rc;
    }
    // device arrays that every call writes: calls from different streams must not overlap
    p->shared_state = p->scratch[0] || p->blue_work[0] || p->real_work || (flags & GFFTX_FLAG_GRAPH);
    *out = p;
    return GFFTX_SUCCESS;
}

}  // namespace detail
}  // namespace gfftx

extern "C" {

int gfftx_plan_create(gfftx_plan* plan, uint64_t n, int vtype, int ttype, int place, int device, uint32_t flags)
{
    return create_plan(plan, n, 1, vtype, ttype, place, device, flags);
}

int gfftx_plan_create_batched(gfftx_plan* plan, uint64_t n, uint64_t batch, int vtype, int ttype, int place,
                              int device, uint32_t flags)
{
    return create_plan(plan, n, batch, vtype, ttype, place, device, flags);
}

int gfftx_exec_inplace(gfftx_plan plan, void* data, void* stream)
{
    if (!plan) return fail(GFFTX_ERR_INVALID_ARG, "plan is NULL");
    if (!data) return fail(GFFTX_ERR_INVALID_ARG, "data is NULL");
    if (plan->place != GFFTX_IN_PLACE) return fail(GFFTX_ERR_INVALID_ARG, "plan is out-of-place");
    return exec_any(plan, data, data, (hipStream_t)stream);
}

int gfftx_exec_oop(gfftx_plan plan, const void* src, void* dst, void* stream)
{
    if (!plan) return fail(GFFTX_ERR_INVALID_ARG, "plan is NULL");
    if (!src || !dst) return fail(GFFTX_ERR_INVALID_ARG, "src/dst is NULL");
    if (plan->place != GFFTX_OUT_OF_PLACE) return fail(GFFTX_ERR_INVALID_ARG, "plan is in-place");
    if (src == dst) return fail(GFFTX_ERR_ALIAS, "out-of-place transform with src == dst");
    return exec_any(plan, src, dst, (hipStream_t)stream);
}

int gfftx_exec_batch(const gfftx_plan* plans, void* const* data, size_t count, void* stream)
{
    if (count == 0) return GFFTX_SUCCESS;
    if (!plans || !data) return fail(GFFTX_ERR_INVALID_ARG, "plans/data is NULL");
    for (size_t i = 0; i < count; ++i) {
        if (!plans[i]) return fail(GFFTX_ERR_INVALID_ARG, "plans[%zu] is NULL", i);
        if (!data[i]) return fail(GFFTX_ERR_INVALID_ARG, "data[%zu] is NULL", i);
        if (plans[i]->place != GFFTX_IN_PLACE) return fail(GFFTX_ERR_INVALID_ARG, "plans[%zu] is out-of-place", i);
    }
    for (size_t i = 0; i < count; ++i) {
        const int rc = exec_any(plans[i], data[i], data[i], (hipStream_t)stream);
        if (rc) {
            const std::string msg = g_last_error;
            return fail(rc, "exec_batch item %zu: %s", i, msg.c_str());
        }
    }
    return GFFTX_SUCCESS;
}

int gfftx_stream_synchronize(void* stream)
{
    const hipError_t e = hipStreamSynchronize((hipStream_t)stream);
    if (e != hipSuccess) return fail(GFFTX_ERR_DEVICE, "stream synchronize: %s", hipGetErrorString(e));
    return GFFTX_SUCCESS;
}

int gfftx_plan_profile(gfftx_plan plan, double* total_ms, uint64_t* count, const char** names, int max,
                       int* nslots)
{
    if (!plan || !total_ms || !count || max < 0) return fail(GFFTX_ERR_INVALID_ARG, "bad arguments");
    if (!(plan->flags & GFFTX_FLAG_PROFILE)) return fail(GFFTX_ERR_INVALID_ARG, "plan was not created with GFFTX_FLAG_PROFILE");
    std::lock_guard<std::mutex> lk(plan->mu);
    DeviceGuard g(plan->device);
    const int n = (int)plan->slots.size();
    if (nslots) *nslots = n;
    for (int i = 0; i < n; ++i) {
        gfftx_plan_s::Slot& sl = plan->slots[i];
        double tot = 0;
        for (auto& ev : sl.pending) {
            HIP_TRY(hipEventSynchronize(ev.second));
            float ms = 0;
            HIP_TRY(hipEventElapsedTime(&ms, ev.first, ev.second));
            tot += ms;
            sl.pool.push_back(ev);
        }
        if (i < max) {
            total_ms[i] = tot;
            count[i] = sl.pending.size();
            if (names) names[i] = sl.name.c_str();
        }
        sl.pending.clear();
    }
    return GFFTX_SUCCESS;
}

int gfftx_plan_destroy(gfftx_plan plan)
{
    if (!plan) return GFFTX_SUCCESS;
    DeviceGuard g(plan->device);
    plan->graphs.clear();
    for (int k = 0; k < 2; ++k) {
        if (plan->pin_in[k]) (void)hipHostFree(plan->pin_in[k]);
        if (plan->pin_out[k]) (void)hipHostFree(plan->pin_out[k]);
        if (plan->pin_in_ev[k]) (void)hipEventDestroy(plan->pin_in_ev[k]);
        if (plan->pin_out_ev[k]) (void)hipEventDestroy(plan->pin_out_ev[k]);
    }
    if (plan->h2d_ev) (void)hipEventDestroy(plan->h2d_ev);
    if (plan->done_ev) (void)hipEventDestroy(plan->done_ev);
    if (plan->h2d_stream) (void)hipStreamDestroy(plan->h2d_stream);
    if (plan->d2h_stream) (void)hipStreamDestroy(plan->d2h_stream);
    for (auto& sl : plan->slots) {
        for (auto& ev : sl.pending) { (void)hipEventDestroy(ev.first); (void)hipEventDestroy(ev.second); }
        for (auto& ev : sl.pool) { (void)hipEventDestroy(ev.first); (void)hipEventDestroy(ev.second); }
    }
    for (void* a : plan->allocs) (void)hipFree(a);
    delete plan;
    return GFFTX_SUCCESS;
}

int gfftx_plan_describe(gfftx_plan plan, char* buf, size_t len)
{
    if (!plan || !buf || len == 0) return fail(GFFTX_ERR_INVALID_ARG, "bad arguments");
    snprintf(buf, len, "%s", plan->desc.c_str());
    return plan->desc.size() < len ? GFFTX_SUCCESS : fail(GFFTX_ERR_INVALID_ARG, "buffer too small");
}

int gfftx_digit_reverse(const void* src, void* dst, uint64_t radix, uint32_t digits, int vtype, void* stream)
{
    if (!src || !dst || src == dst) return fail(GFFTX_ERR_INVALID_ARG, "src/dst NULL or aliased");
    if (radix < 2 || digits == 0) return fail(GFFTX_ERR_INVALID_ARG, "radix >= 2 and digits >= 1 required");
    long double nn = 1;
    for (uint32_t i = 0; i < digits; ++i) nn *= (long double)radix;
    if (nn > 9.0e15L) return fail(GFFTX_ERR_INVALID_ARG, "radix^digits too large");
    if (vtype < 0 || vtype > 3) return fail(GFFTX_ERR_INVALID_ARG, "unknown value type %d", vtype);
    if (!is_device_ptr(src) || !is_device_ptr(dst))
        return fail(GFFTX_ERR_INVALID_ARG, "gfftx_digit_reverse takes device pointers");
    const int prec = (vtype == GFFTX_DOUBLE || vtype == GFFTX_COMPLEX_DOUBLE) ? PREC_F64 : PREC_F32;
    hipError_t e = launch_digit_reverse(prec, src, dst, (long long)radix, (int)digits, (long long)nn,
                                        (hipStream_t)stream);
    if (e != hipSuccess) return fail(GFFTX_ERR_LAUNCH, "digit_reverse: %s", hipGetErrorString(e));
    return GFFTX_SUCCESS;
}

const char* gfftx_strerror(int status)
{
    switch (status) {
        case GFFTX_SUCCESS: return "success";
        case GFFTX_ERR_INVALID_ARG: return "invalid argument";
        case GFFTX_ERR_UNSUPPORTED: return "Requested transform is not compiled! (unsupported length/type/place)";
        case GFFTX_ERR_ALLOC: return "allocation failed";
        case GFFTX_ERR_DEVICE: return "HIP device error";
        case GFFTX_ERR_ALIAS: return "out-of-place transform with src == dst";
        case GFFTX_ERR_LAUNCH: return "kernel launch failed";
        default: return "unknown status";
    }
}

const char* gfftx_last_error(void) { return g_last_error.c_str(); }

}  // extern "C"
