// mixed_kernel.h -- batched Stockham FFT of any length with the factors 2, 3, 5 and 7 that
// fits the LDS, its radices and shape given at run time (gfx950).
//
// The tiles of tile_kernel.h are compiled per length.  A length without one used to be split
// into passes of small compiled tiles (1000 = 25*8*5: three passes over HBM); this kernel runs
// it in one.  The stages are the ones of tile_kernel.h, with
//   - radices up to 16, composite ones included (6, 9, 10, 12, 14, 15), so that a length has few
//     stages and a thread holds at most MIX_POINTS points;
//   - a stage's radix chosen by a branch that is uniform over the launch: every radix is a
//     register butterfly of its own, nothing is indexed at run time inside it;
//   - division by a stage's Ns as a 24-bit multiplication and a shift (Div; 32-bit products run at
//     a quarter of the rate and took a fifth of a stage's issue slots), and an LDS layout (pad
//     elements after every R_0) in which the elements of a butterfly lie at a constant distance,
//     so that an element costs one address addition.
// Access modes as in tile_kernel.h: E->E (single pass), T->E (first pass), T->T (later passes).
#pragma once
#include <cstddef>

#include "tile_kernel.h"

namespace gfftx {

constexpr int MIX_POINTS = 16;    // most points of a sequence one thread holds
constexpr int MIX_STAGES = 10;    // more than any length takes (16384 = 16*16*8*8)
#define GFFTX_MIX_RADICES(X) X(2) X(3) X(4) X(5) X(6) X(7) X(8) X(9) X(10) X(12) X(14) X(15) X(16)

// Product of a 16-bit and a 24-bit number, the ranges spelled out: one full-rate instruction.
__host__ __device__ __forceinline__ unsigned mul24(unsigned a, unsigned b) { return (a & 0xffffu) * (b & 0xffffffu); }

// x / d = (x * m) >> s for x < 2^15, m < 2^17: s = 15 + ceil(log2 d), m = floor(2^s / d) + 1
// (x * (m d - 2^s) < 2^s, since 0 < m d - 2^s <= d <= 2^(s - 15)).
struct Div {
    unsigned m, s;
    __host__ __device__ __forceinline__ unsigned operator()(unsigned x) const
    {
        return mul24(x, m) >> s;
    }
};

struct MixStage {
    unsigned R;     // radix
    unsigned lr;    // L / R: butterflies per sequence
    unsigned ns;    // product of the earlier radices
    Div dns;        // j / ns
    unsigned rst;   // LDS distance of the elements j, j + L/R, .. a butterfly reads
    unsigned wst;   // LDS distance of the elements it writes (ns apart)
    unsigned wq;    // (R - 1) wst
    unsigned tw;    // first entry of the stage's twiddles (FP32: ns FP64 roots; FP64: rows r = 1..R-1 of ns entries)
};

struct MixShape {
    unsigned L, nb, tpt, wg;  // nb sequences of tpt threads each; wg >= nb * tpt threads
    Div dtpt, dr0, dl;        // x / tpt, x / R_0, x / L
    unsigned ts;              // LDS distance between sequences
    unsigned pad;             // LDS pad elements after every R_0 elements: 0 or 1
    unsigned nst;
    int nt_in;                // 1: rows of L (T modes: nb) elements are whole 128-byte lines, the input is loaded non-temporally
    MixStage st[MIX_STAGES];
};

// Chirp-z kinds of a tile, beside the real-transform ones (REAL_NONE, REAL_POST, REAL_PRE).  The
// convolution of length m runs in passes P_0 .. P_k forward and P_k .. P_0 backward:
//   CHIRP_IN    first pass (T->E): x[e] c[e] for e < n, zero beyond, in the loads;
//   CHIRP_TURN  last forward pass and first backward pass in one (T->E).  The forward one leaves
//               element q of sequence t at t + q S (S = m / L), which is what the backward one
//               takes as element q of its sequence t: the filter is multiplied in between, in
//               registers, and the conjugate goes on (the inverse FFT is conj FFT conj);
//   CHIRP_OUT   last backward pass (T->T): conj and c[k] in the stores of k < n;
//   CHIRP_ALL   all of it in one tile (E->E) where m points fit: HBM holds nothing but x and X.
// The turn needs the same radix first and last: a thread's outputs of the last stage are then
// its inputs of the first one.
enum { CHIRP_ALL = 3, CHIRP_IN = 4, CHIRP_TURN = 5, CHIRP_OUT = 6 };

struct ChirpArgs {
    const void* chirp;   // n entries c_j = W_{2n}^{j^2}
    const void* filter;  // m entries: FFT_m of the chirp filter, over m
    unsigned n;
    long long mdist;     // distance between the work array's batch items
};

struct MixArgs {
    TileArgs a;
    MixShape m;
    ChirpArgs c;
};

enum { MIX_EE = 0, MIX_TE = 1, MIX_TT = 2 };

// Good-Thomas butterfly of A*B points, A and B coprime: an A x B two-dimensional DFT between
// two index maps, without twiddles.  Input n = (B n1 + A n2) mod AB, output
// k = (B (B^-1 mod A) k1 + A (A^-1 mod B) k2) mod AB (I. J. Good, 1958).
template <int A, int B> struct PfaDft {
    static constexpr int N = A * B;
    static constexpr int inv(int x, int m)
    {
        for (int i = 1; i < m; ++i)
            if (x * i % m == 1) return i;
        return 1;
    }
    template <typename V> __device__ __forceinline__ static void run(V* v)
    {
        V w[A][B];
#pragma unroll
        for (int i = 0; i < A; ++i) {
#pragma unroll
            for (int k = 0; k < B; ++k) w[i][k] = v[(B * i + A * k) % N];
            Dft<B>::run(w[i]);
        }
#pragma unroll
        for (int k = 0; k < B; ++k) {
            V c[A];
#pragma unroll
            for (int i = 0; i < A; ++i) c[i] = w[i][k];
            Dft<A>::run(c);
#pragma unroll
            for (int i = 0; i < A; ++i) v[(B * inv(B % A, A) * i + A * inv(A % B, B) * k) % N] = c[i];
        }
    }
};
template <> struct Dft<6> : PfaDft<2, 3> {};
template <> struct Dft<10> : PfaDft<2, 5> {};
template <> struct Dft<12> : PfaDft<4, 3> {};
template <> struct Dft<14> : PfaDft<2, 7> {};
template <> struct Dft<15> : PfaDft<3, 5> {};

// 9 = 3 * 3: n = i + 3 m, k = q + 3 p, twiddles W_9^{iq}
template <> struct Dft<9> {
    template <typename V> __device__ __forceinline__ static void run(V* v)
    {
        using S = decltype(v[0].x);
        const V w1{(S)0.76604444311897803520239265055541667394, (S)-0.64278760968653932632264340990726343291};
        const V w2{(S)0.17364817766693034885171662676931479600, (S)-0.98480775301220805936674302458952301367};
        const V w4{(S)-0.93969262078590838405410927732473146994, (S)-0.34202014332566873304409961468225958076};
        V a[3][3];
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            a[i][0] = v[i];
            a[i][1] = v[i + 3];
            a[i][2] = v[i + 6];
            Dft<3>::run(a[i]);
        }
        a[1][1] = cmul(a[1][1], w1);
        a[1][2] = cmul(a[1][2], w2);
        a[2][1] = cmul(a[2][1], w2);
        a[2][2] = cmul(a[2][2], w4);
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            V b[3] = {a[0][q], a[1][q], a[2][q]};
            Dft<3>::run(b);
            v[q] = b[0];
            v[q + 3] = b[1];
            v[q + 6] = b[2];
        }
    }
};

// Thread context of one tile.
template <typename T> struct MixCtx {
    using V = V2<T>;
    V* lds;        // this sequence's LDS region
    const V* in;   // element e of the sequence at in[e * ies]
    V* out;        // output q of the sequence at out[q * ns]
    unsigned jt;   // thread within the sequence; beyond every butterfly for idle threads
    unsigned ies, ons;
    long long tg;  // sequence within the batch item
    long long bo;  // element offset of the batch item in the output
    double2 rw;    // FP32: root of the next stage's first butterfly, in flight (see fetch_roots, tile_kernel.h)
};

// Whether the roots are fetched one stage ahead.  Not in plain single passes: they run at the rate
// of memory with six waves per SIMD, whose 80 registers have no room for it (16384 x 1000: 51 us
// without, 56 us with it and five waves, 67 us with it and six, spilling).
template <int MODE, int REAL> constexpr bool mix_ahead() { return MODE != MIX_EE || REAL != REAL_NONE; }

template <typename T> __device__ __forceinline__ void mix_fetch(MixCtx<T>& c, const void* tw, const MixStage& st)
{
    if constexpr (sizeof(T) == 4) {
        if (c.jt < st.lr) c.rw = reinterpret_cast<const double2*>(tw)[st.tw + c.jt - mul24(st.dns(c.jt), st.ns)];
    }
}

// Stage s of the launch's shape, read from the kernel arguments where they lie (MixArgs is the only
// argument): indexing the by-value struct at run time makes the compiler copy all of it to scratch
// memory (616 bytes a thread; the chirp-z tile then ran three times as long).
__device__ __forceinline__ MixStage mix_stage_args(unsigned s)
{
    typedef const __attribute__((address_space(4))) unsigned char* Bytes;
    typedef const __attribute__((address_space(4))) MixStage* Stages;
    const Bytes k = (Bytes)__builtin_amdgcn_kernarg_segment_ptr();
    const Stages st = (Stages)(k + offsetof(MixArgs, m) + offsetof(MixShape, st)) + s;
    return MixStage{st->R, st->lr, st->ns, Div{st->dns.m, st->dns.s}, st->rst, st->wst, st->wq, st->tw};
}

// LDS index of element e (pad is 0 or 1).
__device__ __forceinline__ unsigned mix_pos(const MixShape& m, unsigned e) { return e + (m.dr0(e) & (0u - m.pad)); }

// Twiddles W^{k r}, r = 1..R-1, of one butterfly.  FP32: FP64 powers of the FP64 root, rounded
// once (as in tile_kernel.h); FP64: the table's rows, row r contiguous in k.
template <typename T, int R>
__device__ __forceinline__ void mix_twiddle(V2<T>* v, const void* tw, const MixStage& st, unsigned k, const double2* root = nullptr)
{
    using V = V2<T>;
    if constexpr (sizeof(T) == 4) {
        const double2 w1 = root ? *root : reinterpret_cast<const double2*>(tw)[st.tw + k];
        v[1] = cmul(v[1], to_v<V>(w1));
        if constexpr (R > 2) {
            const double2 w2 = dmul(w1, w1);
            v[2] = cmul(v[2], to_v<V>(w2));
            if constexpr (R > 3) {
                const double2 w3 = dmul(w2, w1);
                v[3] = cmul(v[3], to_v<V>(w3));
                if constexpr (R > 4) {
                    // W^{4a + c} = (W^4)^a W^c: at most five products from the root
                    const double2 w4 = dmul(w2, w2);
                    double2 wa = w4;
#pragma unroll
                    for (int r = 4; r < R; ++r) {
                        if (r % 4 == 0) {
                            if (r > 4) wa = dmul(wa, w4);
                            v[r] = cmul(v[r], to_v<V>(wa));
                        } else {
                            v[r] = cmul(v[r], to_v<V>(dmul(wa, r % 4 == 1 ? w1 : r % 4 == 2 ? w2 : w3)));
                        }
                    }
                }
            }
        }
    } else {
        const V* row = reinterpret_cast<const V*>(tw) + st.tw + k;
#pragma unroll
        for (int r = 1; r < R; ++r) {
            v[r] = cmul(v[r], row[(unsigned)(r - 1) * st.ns]);
            if (r % 4 == 0) __builtin_amdgcn_sched_barrier(0);  // four rows in flight: the registers hold no more
        }
    }
}

// Butterflies a thread runs per stage: as many as MIX_POINTS points hold (the host chooses tpt
// so that they cover the sequence).
template <int R> constexpr int mix_b() { return MIX_POINTS / R; }

// First stage: global memory to registers (pass twiddle of a later pass, conjugation of an
// inverse transform, C2R pre-pass of a real one), butterfly, LDS.
template <typename T, int MODE, int REAL, int R, bool ONLY>
__device__ __forceinline__ void mix_first(const MixArgs& x, MixCtx<T>& c)
{
    using V = V2<T>;
    using S_ = T;
    constexpr int B = mix_b<R>();
    const TileArgs& a = x.a;
    const unsigned lr = x.m.st[0].lr, tpt = x.m.tpt;
    const unsigned cn = x.c.n, e0 = REAL == CHIRP_IN ? (unsigned)c.tg : 0u;  // chirp-z: element e0 + i
    const unsigned istep = MODE == MIX_EE ? lr : lr * c.ies;  // between the elements of a butterfly
    // chirp-z: n <= (m + 1) / 2, so the elements r lr + j with 2 r >= R lie in the zero padding
    constexpr int RN = REAL == CHIRP_ALL || REAL == CHIRP_IN ? (R + 1) / 2 : R;
    V v[B][R];
    if constexpr (RN < R) {
#pragma unroll
        for (int b = 0; b < B; ++b)
#pragma unroll
            for (int r = RN; r < R; ++r) v[b][r] = V{0, 0};
    }
    with_nt(x.m.nt_in != 0, [&](auto ntc) {
#pragma unroll
        for (int b = 0; b < B; ++b) {
            const unsigned j = c.jt + b * tpt;
            if (j >= lr) continue;
            const unsigned i0 = MODE == MIX_EE ? j : j * c.ies;
#pragma unroll
            for (int r = 0; r < RN; ++r) {
                const unsigned i = i0 + r * istep;
                const V* p = &c.in[i];
                if constexpr (REAL == CHIRP_ALL || REAL == CHIRP_IN) {
                    v[b][r] = V{0, 0};
                    if (e0 + i >= cn) continue;
                }
                if constexpr (decltype(ntc)::value) v[b][r] = nt_load(p);
                else v[b][r] = *p;
            }
        }
    });
    if constexpr (!ONLY && mix_ahead<MODE, REAL>()) mix_fetch(c, a.tw, mix_stage_args(1));
    if constexpr (REAL == REAL_PRE) {
        // Z[e] from X[e] and X[N - e] of the same sequence (see pre_split, tile_kernel.h); the
        // exchange uses a plain layout, element e at e
#pragma unroll
        for (int b = 0; b < B; ++b) {
            const unsigned j = c.jt + b * tpt;
            if (j >= lr) continue;
#pragma unroll
            for (int r = 0; r < R; ++r) c.lds[j + r * lr] = v[b][r];
        }
        __syncthreads();
        const S_ half = (S_)0.5;
        const unsigned N = x.m.L;
        const long long mask = (1LL << a.sp_shift) - 1;
        const double2 step = dmul(a.sp_lo[lr & mask], a.sp_hi[lr >> a.sp_shift]);
#pragma unroll
        for (int b = 0; b < B; ++b) {
            const unsigned j = c.jt + b * tpt;
            if (j >= lr) continue;
            double2 w = dmul(a.sp_lo[j & mask], a.sp_hi[j >> a.sp_shift]);
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const unsigned e = j + r * lr;
                const V xe = v[b][r], xp = c.lds[e == 0 ? 0 : N - e];
                V z;
                if (e == 0) {
                    const S_ x0 = xe.x, xn = a.split_bins ? c.in[N].x : xe.y;
                    z = V{half * (x0 + xn), half * (x0 - xn)};
                } else {
                    const bool lo = e <= N - e;
                    const V A = lo ? xe : xp, Bv = lo ? xp : xe;
                    // conj(W^k) for k = min(e, N - e): conj(W^{N-e}) = -W^e
                    const V cw = to_v<V>(lo ? double2{w.x, -w.y} : double2{-w.x, -w.y});
                    const V h1 = V{half * (A.x + Bv.x), half * (A.y - Bv.y)};
                    const V dd = V{half * (A.x - Bv.x), half * (A.y + Bv.y)};
                    const V t = cmul(cw, dd);
                    const V p = V{-t.y, t.x};  // i conj(W^k) d
                    z = lo ? V{h1.x + p.x, h1.y + p.y} : V{h1.x - p.x, p.y - h1.y};
                }
                v[b][r] = z;
                w = dmul(w, step);
            }
        }
        __syncthreads();
    }
    const unsigned flip = a.conj_in ? 0x80000000u : 0u;
    constexpr bool PTW = MODE == MIX_TT || REAL == CHIRP_TURN;
    const long long kp = (PTW && a.ptw_lo != nullptr) ? c.tg % a.ns_pass : 0;
#pragma unroll
    for (int b = 0; b < B; ++b) {
        const unsigned j = c.jt + b * tpt;
        if (j >= lr) continue;
#pragma unroll
        for (int r = 0; r < RN; ++r)
            if (flip) v[b][r].y = -v[b][r].y;
        if constexpr (REAL == CHIRP_ALL || REAL == CHIRP_IN) {
            const V* ch = reinterpret_cast<const V*>(x.c.chirp) + e0;
            const unsigned i0 = MODE == MIX_EE ? j : j * c.ies;
#pragma unroll
            for (int r = 0; r < RN; ++r) {
                const unsigned i = i0 + r * istep;
                if (e0 + i < cn) v[b][r] = cmul(v[b][r], ch[i]);
            }
        }
        if constexpr (PTW) {
            if (kp != 0) {
                // W_M^{kp e}, e = j + r lr: base W^{kp j} times step^r, step = W^{kp lr}
                const long long pm = (1LL << a.ptw_shift) - 1, m0 = kp * j, ms = kp * lr;
                const double2 step = dmul(a.ptw_lo[ms & pm], a.ptw_hi[ms >> a.ptw_shift]);
                double2 w = dmul(a.ptw_lo[m0 & pm], a.ptw_hi[m0 >> a.ptw_shift]);
                v[b][0] = cmul(v[b][0], to_v<V>(w));
#pragma unroll
                for (int r = 1; r < R; ++r) {
                    w = dmul(w, step);
                    v[b][r] = cmul(v[b][r], to_v<V>(w));
                }
            }
        }
        Dft<R>::run(v[b]);
        if constexpr (!ONLY) {
            V* w = c.lds + mul24(j, R + x.m.pad);
#pragma unroll
            for (int r = 0; r < R; ++r) w[r] = v[b][r];
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (ONLY) {
        // a length that is one butterfly: straight to the output
        const unsigned fo = a.conj_out ? 0x80000000u : 0u;
        const T sc = (T)a.scale;
        with_store<MODE != MIX_EE>(a.store, [&](auto kind) {
#pragma unroll
            for (int b = 0; b < B; ++b) {
                if (c.jt + b * tpt >= lr) continue;
#pragma unroll
                for (int r = 0; r < R; ++r)
                    put<decltype(kind)::value>(&c.out[r * c.ons], flip_im(a.scale == 1.0 ? v[b][r] : cscale(v[b][r], sc), fo));
            }
        });
    } else {
        __syncthreads();
    }
}

// A later stage: LDS to registers, twiddles, butterfly, and back to the LDS or, after the last
// stage of a mode whose stores match its lanes, to the output.
template <typename T, int MODE, int REAL, int R, bool LAST>
__device__ __forceinline__ void mix_stage(const MixArgs& x, MixCtx<T>& c, const MixStage& st, const MixStage& next)
{
    using V = V2<T>;
    constexpr int B = mix_b<R>();
    constexpr bool DIRECT = LAST && MODE != MIX_TE && REAL != REAL_POST;
    const TileArgs& a = x.a;
    const unsigned lr = st.lr, tpt = x.m.tpt, rst = st.rst;
    V v[B][R];
    // j / ns (the last stage has ns = lr > j)
    auto quot = [&](unsigned j) { return LAST ? 0u : st.dns(j); };
#pragma unroll
    for (int b = 0; b < B; ++b) {
        const unsigned j = c.jt + b * tpt;
        if (j >= lr) continue;
        const V* rd = c.lds + mix_pos(x.m, j);
#pragma unroll
        for (int r = 0; r < R; ++r, rd += rst) v[b][r] = *rd;
    }
    const double2 w1 = c.rw;
    if constexpr (!LAST && mix_ahead<MODE, REAL>()) mix_fetch(c, a.tw, next);  // (by every thread: it may take part in the next stage alone)
#pragma unroll
    for (int b = 0; b < B; ++b) {
        const unsigned j = c.jt + b * tpt;
        if (j < lr) {
            const unsigned k = j - mul24(quot(j), st.ns);
            if (mix_ahead<MODE, REAL>() && b == 0) mix_twiddle<T, R>(v[b], a.tw, st, k, &w1);
            else mix_twiddle<T, R>(v[b], a.tw, st, k);
            Dft<R>::run(v[b]);
        }
        __builtin_amdgcn_sched_barrier(0);  // one butterfly's twiddles at a time (registers)
    }
    if constexpr (DIRECT) {
        const unsigned fo = a.conj_out ? 0x80000000u : 0u;
        const T sc = (T)a.scale;
        const bool one = a.scale == 1.0;
        constexpr int RN = REAL == CHIRP_ALL || REAL == CHIRP_OUT ? (R + 1) / 2 : R;  // the others are k >= n
        const V* chirp = reinterpret_cast<const V*>(x.c.chirp);  // (copies: the lambda would take x's address)
        if constexpr (REAL != CHIRP_ALL && REAL != CHIRP_OUT) {
            if (a.conj_out || !one) {  // inverse transforms
#pragma unroll
                for (int b = 0; b < B; ++b)
#pragma unroll
                    for (int r = 0; r < R; ++r) v[b][r] = flip_im(cscale(v[b][r], sc), fo);
            }
        }
        const unsigned cn = x.c.n, ostep = MODE == MIX_EE ? lr : lr * c.ons;
        with_store<MODE != MIX_EE>(a.store, [&](auto kind) {
#pragma unroll
            for (int b = 0; b < B; ++b) {
                const unsigned j = c.jt + b * tpt;
                if (j >= lr) continue;
                const unsigned i0 = MODE == MIX_EE ? j : j * c.ons;
#pragma unroll
                for (int r = 0; r < RN; ++r) {
                    const unsigned i = i0 + r * ostep;
                    if constexpr (REAL == CHIRP_ALL || REAL == CHIRP_OUT) {
                        const unsigned k = (REAL == CHIRP_OUT ? (unsigned)c.tg : 0u) + i;
                        if (k < cn) {
                            const V u = cmul(chirp[k], V{v[b][r].x, -v[b][r].y});
                            put<decltype(kind)::value>(&c.out[i], flip_im(one ? u : cscale(u, sc), fo));
                        }
                    } else {
                        put<decltype(kind)::value>(&c.out[i], v[b][r]);
                    }
                }
            }
        });
    } else {
        __syncthreads();
#pragma unroll
        for (int b = 0; b < B; ++b) {
            const unsigned j = c.jt + b * tpt;
            if (j >= lr) continue;
            V* wr = c.lds + mix_pos(x.m, j) + mul24(quot(j), st.wq);
#pragma unroll
            for (int r = 0; r < R; ++r, wr += st.wst) *wr = v[b][r];
        }
        __syncthreads();
    }
}

// The turn of a chirp-z tile: last stage of the forward transform, filter, conjugate, first stage
// of the backward one (the same radix), back to the LDS.
template <typename T, int REAL, int R>
__device__ __forceinline__ void mix_turn(const MixArgs& x, MixCtx<T>& c, const MixStage& st)
{
    using V = V2<T>;
    constexpr int B = mix_b<R>();
    const unsigned lr = st.lr, tpt = x.m.tpt, rst = st.rst;
    V v[B][R];
#pragma unroll
    for (int b = 0; b < B; ++b) {
        const unsigned j = c.jt + b * tpt;
        if (j >= lr) continue;
        const V* rd = c.lds + mix_pos(x.m, j);
#pragma unroll
        for (int r = 0; r < R; ++r, rd += rst) v[b][r] = *rd;
    }
    const double2 w1 = c.rw;
    mix_fetch(c, x.a.tw, mix_stage_args(1));  // the backward transform's second stage
    const unsigned istep = REAL == CHIRP_TURN ? lr * c.ies : lr;
    const V* filter = reinterpret_cast<const V*>(x.c.filter) + (REAL == CHIRP_TURN ? (unsigned)c.tg : 0u);
#pragma unroll
    for (int b = 0; b < B; ++b) {
        const unsigned j = c.jt + b * tpt;
        if (j < lr) {
            if (b == 0) mix_twiddle<T, R>(v[b], x.a.tw, st, j, &w1);
            else mix_twiddle<T, R>(v[b], x.a.tw, st, j);
            Dft<R>::run(v[b]);
            const unsigned i0 = REAL == CHIRP_TURN ? j * c.ies : j;
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const unsigned i = i0 + r * istep;
                v[b][r] = cmul(v[b][r], filter[i]);
                v[b][r].y = -v[b][r].y;
                if (sizeof(T) == 8 && r % 4 == 3) __builtin_amdgcn_sched_barrier(0);
            }
            Dft<R>::run(v[b]);
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    __syncthreads();
#pragma unroll
    for (int b = 0; b < B; ++b) {
        const unsigned j = c.jt + b * tpt;
        if (j >= lr) continue;
        V* w = c.lds + mul24(j, R + x.m.pad);
#pragma unroll
        for (int r = 0; r < R; ++r) w[r] = v[b][r];
    }
    __syncthreads();
}

// T->E store: the tile's nb * L outputs are one contiguous run (first pass, Ns = 1).
template <typename T> __device__ __forceinline__ void mix_finish_te(const MixArgs& x, const V2<T>* lds, long long bo, unsigned tile)
{
    using V = V2<T>;
    const TileArgs& a = x.a;
    const unsigned L = x.m.L;
    V* o = reinterpret_cast<V*>(a.out) + bo + (long long)tile * x.m.nb * L;
    const long long left = a.ntrans - (long long)tile * x.m.nb;
    const unsigned total = (left < (long long)x.m.nb ? (unsigned)left : x.m.nb) * L;
    const unsigned fo = a.conj_out ? 0x80000000u : 0u;
    const T sc = (T)a.scale;
    const bool one = a.scale == 1.0;
    with_store<true>(a.store, [&](auto kind) {
#pragma unroll 4
        for (unsigned lin = threadIdx.x; lin < total; lin += x.m.wg) {
            const unsigned t = x.m.dl(lin), q = lin - mul24(t, L);
            const V u = lds[mul24(t, x.m.ts) + mix_pos(x.m, q)];
            put<decltype(kind)::value>(&o[lin], flip_im(one ? u : cscale(u, sc), fo));
        }
    });
}

// R2C post-pass of a single-pass real transform (see split_finish_e, tile_kernel.h).
template <typename T> __device__ __forceinline__ void mix_split(const MixArgs& x, const MixCtx<T>& c)
{
    using V = V2<T>;
    const TileArgs& a = x.a;
    const unsigned L = x.m.L, tpt = x.m.tpt;
    if (c.jt >= tpt) return;
    const T half = (T)0.5;
    const long long mask = (1LL << a.sp_shift) - 1;
    double2 w = dmul(a.sp_lo[c.jt & mask], a.sp_hi[c.jt >> a.sp_shift]);
    const double2 step = dmul(a.sp_lo[tpt & mask], a.sp_hi[tpt >> a.sp_shift]);
    auto at = [&](unsigned e) { return c.lds[mix_pos(x.m, e)]; };
#pragma unroll 4
    for (unsigned k = c.jt; k < L; k += tpt) {
        const V zk = at(k), zp = at(k == 0 ? 0 : L - k);
        if (k == 0) {
            const T x0 = zk.x + zk.y, xn = zk.x - zk.y;
            if (a.split_bins) {
                c.out[0] = V{x0, 0};
                c.out[L] = V{xn, 0};
            } else {
                c.out[0] = V{x0, xn};
            }
        } else {
            const bool lo = k <= L - k;
            const V A = lo ? zk : zp, B = lo ? zp : zk;
            const V wv = to_v<V>(lo ? w : double2{-w.x, w.y});  // W^k, or W^{N-k} = -conj(W^k)
            const V h1 = V{half * (A.x + B.x), half * (A.y - B.y)};
            const V dd = V{half * (A.x - B.x), half * (A.y + B.y)};
            const V p = cmul(wv, V{dd.y, -dd.x});
            c.out[k] = lo ? V{h1.x + p.x, h1.y + p.y} : V{h1.x - p.x, p.y - h1.y};
        }
        w = dmul(w, step);
    }
}

// The stages between the first and the last one.
template <typename T, int MODE, int REAL> __device__ __forceinline__ void mix_middle(const MixArgs& x, MixCtx<T>& c)
{
    MixStage next = mix_stage_args(1);
    for (unsigned s = 1; s + 1 < x.m.nst; ++s) {
        const MixStage st = next;
        next = mix_stage_args(s + 1);
        switch (st.R) {
#define X(R_) \
    case R_: mix_stage<T, MODE, REAL, R_, false>(x, c, st, next); break;
            GFFTX_MIX_RADICES(X)
#undef X
            default: break;
        }
    }
}

// Waves per SIMD the registers are allotted for (128, 96 or 80 of them).
template <typename T, int MODE, int REAL> struct MixWaves {
    static constexpr int value = sizeof(T) == 8 ? 4 : mix_ahead<MODE, REAL>() ? 5 : 6;
};

template <typename T, int MODE, int REAL>
__global__ __launch_bounds__(1024, (MixWaves<T, MODE, REAL>::value)) void mixed_kernel(MixArgs x)
{
    using V = V2<T>;
    extern __shared__ __align__(16) unsigned char mix_lds[];
    V* lds = reinterpret_cast<V*>(mix_lds);
    const TileArgs& a = x.a;
    const unsigned tile = tile_index(blockIdx.x, gridDim.x, a.xcd), tid = threadIdx.x;
    unsigned t;
    MixCtx<T> c;
    if constexpr (MODE == MIX_EE) {
        t = x.m.dtpt(tid);
        c.jt = tid - t * x.m.tpt;
    } else {
        t = tid & (x.m.nb - 1);  // nb is a power of two in the T modes
        c.jt = tid >> __builtin_ctz(x.m.nb);
        if (c.jt >= x.m.tpt) c.jt = 1u << 20;
    }
    c.tg = (long long)tile * x.m.nb + t;
    const bool valid = t < x.m.nb && c.tg < a.ntrans;
    if (!valid) {  // beyond every loop bound: takes part in the barriers only
        c.jt = 1u << 20;
        c.tg = 0;
        t = 0;
    }
    const long long bo = batch_offset(a, blockIdx.y);
    c.bo = REAL == CHIRP_IN ? (long long)blockIdx.y * x.c.mdist : bo;
    c.lds = lds + t * x.m.ts;
    const long long so = a.seq_off ? a.seq_off[c.tg] : 0;
    c.in = reinterpret_cast<const V*>(a.in) + (REAL == CHIRP_OUT ? (long long)blockIdx.y * x.c.mdist : bo) +
           (a.seq_off ? so : c.tg * a.its);
    c.ies = (unsigned)a.ies;
    c.ons = (unsigned)a.ns_pass;
    long long ob = so;
    if (!a.seq_off) {
        const unsigned ns = (unsigned)a.ns_pass, t32 = (unsigned)c.tg;
        if (MODE == MIX_EE) ob = c.tg * a.its;
        else ob = ns == 1 ? c.tg * x.m.L : (long long)(t32 / ns) * ns * x.m.L + (t32 % ns);
    }
    c.out = reinterpret_cast<V*>(a.out) + c.bo + ob;
    const unsigned nst = x.m.nst;
    if (MODE == MIX_EE && REAL == REAL_NONE && nst == 1) {
        switch (x.m.st[0].R) {
#define X(R_) \
    case R_: mix_first<T, MODE, REAL, R_, true>(x, c); break;
            GFFTX_MIX_RADICES(X)
#undef X
            default: break;
        }
        return;
    }
    switch (x.m.st[0].R) {
#define X(R_) \
    case R_: mix_first<T, MODE, REAL, R_, false>(x, c); break;
        GFFTX_MIX_RADICES(X)
#undef X
        default: break;
    }
    mix_middle<T, MODE, REAL>(x, c);
    const MixStage sl = mix_stage_args(nst - 1);
    if constexpr (REAL == CHIRP_ALL || REAL == CHIRP_TURN) {
        switch (sl.R) {
#define X(R_) \
    case R_: mix_turn<T, REAL, R_>(x, c, sl); break;
            GFFTX_MIX_RADICES(X)
#undef X
            default: break;
        }
        mix_middle<T, MODE, REAL>(x, c);
    }
    switch (sl.R) {
#define X(R_) \
    case R_: mix_stage<T, MODE, REAL, R_, true>(x, c, sl, sl); break;
        GFFTX_MIX_RADICES(X)
#undef X
        default: break;
    }
    if constexpr (MODE == MIX_TE) mix_finish_te<T>(x, lds, c.bo, tile);
    if constexpr (REAL == REAL_POST) mix_split<T>(x, c);
}

}  // namespace gfftx
