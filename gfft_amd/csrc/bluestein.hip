// bluestein.hip -- tables of the chirp-z (Bluestein) path for lengths with a prime factor above 7:
// the chirp c_j = W_{2n}^{j^2} = exp(-i pi j^2 / n), the filter
//     b_j = conj(c_j) (0 <= j < n),  b_{m-j} = conj(c_j) (0 < j < n),  0 elsewhere,
// and its spectrum in the working precision.  The transform itself runs in the passes of
// mixed_kernel.h (CHIRP_*).
//
// All kernels are streaming: one complex element per thread and iteration.
#include "registry.h"

namespace gfftx {

namespace {

// c_j = W_{2n}^{j^2 mod 2n} from the two-level FP64 root table of order 2n.
template <class T> __global__ __launch_bounds__(256) void chirp_table_kernel(ChirpTableArgs a)
{
    V2<T>* c = (V2<T>*)a.chirp;
    const unsigned long long two_n = 2ull * (unsigned long long)a.n;
    const unsigned long long mask = (1ull << a.shift) - 1;
    for (unsigned long long j = blockIdx.x * 256ull + threadIdx.x; j < (unsigned long long)a.n;
         j += (unsigned long long)gridDim.x * 256ull) {
        const unsigned long long m = (j * j) % two_n;  // j < 2^32: j^2 is exact in 64 bits
        const double2 lo = a.lo[m & mask], hi = a.hi[m >> a.shift];
        const double2 w = cmul(lo, hi);
        c[j] = V2<T>{(T)w.x, (T)w.y};
    }
}

// b over length m: conj(c_j) at j < n and at m - j for 0 < j < n, zero elsewhere.
template <class T> __global__ __launch_bounds__(256) void chirp_filter_kernel(const V2<T>* c, V2<T>* b, unsigned long long n, unsigned long long m)
{
    for (unsigned long long j = blockIdx.x * 256ull + threadIdx.x; j < m; j += (unsigned long long)gridDim.x * 256ull) {
        V2<T> v{0, 0};
        if (j < n) v = cconj(c[j]);
        else if (j > m - n) v = cconj(c[m - j]);
        b[j] = v;
    }
}

// The filter's spectrum over m, divided in FP64 and rounded once.
template <class F, class T> __global__ __launch_bounds__(256) void chirp_spectrum_kernel(const V2<F>* s, V2<T>* f, unsigned long long m)
{
    for (unsigned long long j = blockIdx.x * 256ull + threadIdx.x; j < m; j += (unsigned long long)gridDim.x * 256ull)
        f[j] = V2<T>{(T)((double)s[j].x / (double)m), (T)((double)s[j].y / (double)m)};
}

dim3 stream_grid(long long len)
{
    // up to 16K workgroups (every CU many times over); the kernels stride over the rest
    const long long g = (len + 255) / 256;
    return dim3((unsigned)(g < 16384 ? g : 16384));
}

}  // namespace

hipError_t launch_chirp_table(int prec, const ChirpTableArgs& a, hipStream_t s)
{
    const dim3 g = stream_grid(a.n);
    if (prec == PREC_F64) chirp_table_kernel<double><<<g, 256, 0, s>>>(a);
    else chirp_table_kernel<float><<<g, 256, 0, s>>>(a);
    return hipGetLastError();
}

hipError_t launch_chirp_filter(int prec, const void* chirp, void* b, long long n, long long m, hipStream_t s)
{
    const dim3 g = stream_grid(m);
    if (prec == PREC_F64) chirp_filter_kernel<double><<<g, 256, 0, s>>>((const double2*)chirp, (double2*)b, n, m);
    else chirp_filter_kernel<float><<<g, 256, 0, s>>>((const float2*)chirp, (float2*)b, n, m);
    return hipGetLastError();
}

hipError_t launch_chirp_spectrum(int from, int to, const void* spec, void* filter, long long m, hipStream_t s)
{
    const dim3 g = stream_grid(m);
    if (from == PREC_F64 && to == PREC_F64)
        chirp_spectrum_kernel<double, double><<<g, 256, 0, s>>>((const double2*)spec, (double2*)filter, m);
    else if (from == PREC_F64)
        chirp_spectrum_kernel<double, float><<<g, 256, 0, s>>>((const double2*)spec, (float2*)filter, m);
    else
        chirp_spectrum_kernel<float, float><<<g, 256, 0, s>>>((const float2*)spec, (float2*)filter, m);
    return hipGetLastError();
}

}  // namespace gfftx
