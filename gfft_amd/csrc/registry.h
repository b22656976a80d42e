// registry.h -- host-visible table of compiled FFT kernels.
#pragma once
#include <hip/hip_runtime.h>

#include "mfma_kernel.h"
#include "mixed_kernel.h"
#include "tile_kernel.h"

namespace gfftx {

enum Prec { PREC_F64 = 0, PREC_F32 = 1 };

// Launchers take an optional event pair (both null or both created): when given, the
// launch goes through hipExtLaunchKernel, which stamps the events with the kernel's own
// start and end instead of recording them as separate stream commands.
typedef hipError_t (*TileLaunch)(const TileArgs&, dim3, hipStream_t, hipEvent_t, hipEvent_t);

struct TileEntry {
    int prec;
    int L;
    int nb;
    int wg;
    bool loadT;
    bool storeT;
    int nrad;
    const int* radices;
    int lds_bytes;
    TileLaunch launch;
    const char* name;
    int real;  // REAL_NONE, or the real-transform split fused in (REAL_POST, REAL_PRE: RealCfg)
    const MixShape* mix = nullptr;  // run-time mixed-radix tile (mixed.cpp; `launch` is null)
};

// Run-time mixed-radix tiles (mixed.cpp).  mixed_prepare lifts the kernel's limit on dynamic
// LDS; it is called once per shape, when a plan is made.
hipError_t mixed_prepare(const TileEntry& k);
hipError_t launch_mixed(const TileEntry& k, const TileArgs& a, dim3 grid, hipStream_t s, hipEvent_t t0, hipEvent_t t1,
                        const ChirpArgs* c = nullptr);

inline hipError_t launch_entry(const TileEntry* k, const TileArgs& a, dim3 grid, hipStream_t s, hipEvent_t t0 = nullptr,
                               hipEvent_t t1 = nullptr)
{
    return k->mix ? launch_mixed(*k, a, grid, s, t0, t1) : k->launch(a, grid, s, t0, t1);
}

// Complex tiles (kernels.hip) and tiles with a real-transform split fused in (real_tiles.hip).
extern TileEntry kTiles[];
extern const int kNumTiles;
extern TileEntry kRealTiles[];
extern const int kNumRealTiles;

// Split-precision MFMA kernels (FP32, lengths 16^S).
typedef hipError_t (*MfmaLaunch)(const MfmaArgs&, dim3, hipStream_t, hipEvent_t, hipEvent_t);
struct MfmaEntry {
    int L;
    int nb;
    int scale;  // MFMA_SCALE_STAGE (stage twiddles carry 2^-4) or MFMA_SCALE_COLUMN
    int wg;     // threads per workgroup
    MfmaLaunch launch;
    const char* name;
};
extern MfmaEntry kMfma[];
extern const int kNumMfma;

// Real-transform split pass (Separate, src/gfftswap.h:239-336) as one kernel.
struct SplitArgs {
    void* data;            // n complex (+1 when bins)
    long long n;           // complex half length
    long long bdist;       // distance between batch items, complex elements
    long long nbatch;
    const void* tw;        // n/2+1 entries W_{2n}^k in working precision (forward sign)
    int inverse;           // 0: post-pass of RDFT, 1: pre-pass of IRDFT
    int bins;              // 1: n+1 bins layout, 0: NR packing
};
hipError_t launch_split(int prec, const SplitArgs& a, hipStream_t s);

// Tables of the chirp-z (Bluestein) path for lengths with a prime factor above 7 (bluestein.hip).
struct ChirpTableArgs {
    void* chirp;            // n entries c_j = W_{2n}^{j^2}, working precision
    long long n;
    const double2* lo;      // two-level FP64 root table of order 2n
    const double2* hi;
    int shift;
};
hipError_t launch_chirp_table(int prec, const ChirpTableArgs& a, hipStream_t s);
// b over length m: conj(c_j) at j < n and at m - j for 0 < j < n, zero elsewhere
hipError_t launch_chirp_filter(int prec, const void* chirp, void* b, long long n, long long m, hipStream_t s);
// filter[i] = spec[i] / m, from precision `from` to `to`
hipError_t launch_chirp_spectrum(int from, int to, const void* spec, void* filter, long long m, hipStream_t s);

// Digit reversal dst[rev(k)] = src[k] over radix^digits elements.
hipError_t launch_digit_reverse(int prec, const void* src, void* dst, long long radix, int digits,
                                long long n, hipStream_t s);

}  // namespace gfftx
