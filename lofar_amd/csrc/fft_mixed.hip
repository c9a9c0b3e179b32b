// Mixed-radix transforms for gfx950: lines of any length up to 8192 whose prime factors
// are at most 13 (the sides fftw_data() plans that are not powers of two,
// fourier_transform.c:25-27), as rows or as strided columns of [w][v][u] planes.
//
// A workgroup transforms L lines: L adjacent columns (so that each row access is a run of
// L cells) or L rows.  Stockham stages of composite radices up to 16, chosen per length so
// that the stages are few: the first stage reads its butterflies straight from memory and
// the last one stores straight to it, the stages between go through one LDS buffer in
// place (every thread reads its butterflies into registers, a barrier, then they are
// written back), so a line of 3000 (10*10*6*5) crosses LDS three times.  Butterfly j (k = j
// mod Ns, Ns the product of the radices before this stage) takes x[j + q*N/P], q < P, times
// exp(2 pi i q k / (Ns P)), DFT over q, and gives y[(j - k)*P + k + r*Ns].  Each stage's
// twiddles are laid out [q-1][k], so that a wave's butterflies read runs of the table
// (stage_twiddle_order; read from an N-entry table in order, every lane took a cache line of
// its own); the small DFTs have their roots as constants
// (odd primes by the even and odd parts of their inputs, half the products of the
// definition).  Inverse signs swap the real and imaginary parts on the way in and out.
//
// Bound: the load - stages - store sequence of the one or two workgroups a CU holds; rows
// are near the copy rate, columns longer than 2048 complex doubles get runs of only 32
// bytes (64-byte runs do not fit LDS).  16 planes of 3000 x 3000 complex doubles, row-major:
// columns 1.92 ms, rows 1.15 ms (2.4 and 4.0 TB/s); in strips of 4 columns ([nx/4][ny][4], the
// images' cubes: strip_log in capi.cpp) 1.42 and 1.36, of 2 1.20 and 1.77, of 8 1.77 and 1.24.
// One line per 256-thread workgroup with 128 KiB of LDS and radices 8, 3, 5, 5, 5 took 12.5 ms
// for both.
#include <algorithm>

#include "fft_kernels.h"

namespace lofar {

constexpr int kMixMaxN = 8192;  // longest line
constexpr int kMixMaxT = 1024;
constexpr int kMixMaxStages = 8;

// Stages of one length; magic = floor(2^32/ns) + 1: j / ns = umulhi(j, magic) for j < 2^13.
struct MixPlan {
    int n, nstages;
    int radix[kMixMaxStages], ns[kMixMaxStages];
    unsigned magic[kMixMaxStages];
};

// cos and sin of 2 pi m / N
template <int N>
struct Root;
#define LOFAR_ROOTS(N_, C_, S_)                          \
    template <>                                          \
    struct Root<N_> {                                    \
        static constexpr double c[N_] = C_, s[N_] = S_;  \
    };
#define V_(...) {__VA_ARGS__}
LOFAR_ROOTS(3, V_(1.0, -0.5, -0.5), V_(0.0, 0.8660254037844386, -0.8660254037844386))
LOFAR_ROOTS(5, V_(1.0, 0.30901699437494745, -0.8090169943749475, -0.8090169943749475,
                  0.30901699437494745),
            V_(0.0, 0.9510565162951535, 0.5877852522924731, -0.5877852522924731,
               -0.9510565162951535))
LOFAR_ROOTS(6, V_(1.0, 0.5, -0.5, -1.0, -0.5, 0.5),
            V_(0.0, 0.8660254037844386, 0.8660254037844386, 0.0, -0.8660254037844386,
               -0.8660254037844386))
LOFAR_ROOTS(7, V_(1.0, 0.6234898018587335, -0.2225209339563144, -0.9009688679024191,
                  -0.9009688679024191, -0.2225209339563144, 0.6234898018587335),
            V_(0.0, 0.7818314824680298, 0.9749279121818236, 0.4338837391175581,
               -0.4338837391175581, -0.9749279121818236, -0.7818314824680298))
LOFAR_ROOTS(9, V_(1.0, 0.766044443118978, 0.17364817766693036, -0.5, -0.9396926207859084,
                  -0.9396926207859084, -0.5, 0.17364817766693036, 0.766044443118978),
            V_(0.0, 0.6427876096865394, 0.984807753012208, 0.8660254037844386,
               0.3420201433256687, -0.3420201433256687, -0.8660254037844386,
               -0.984807753012208, -0.6427876096865394))
LOFAR_ROOTS(10, V_(1.0, 0.8090169943749475, 0.30901699437494745, -0.30901699437494745,
                   -0.8090169943749475, -1.0, -0.8090169943749475, -0.30901699437494745,
                   0.30901699437494745, 0.8090169943749475),
            V_(0.0, 0.5877852522924731, 0.9510565162951535, 0.9510565162951535,
               0.5877852522924731, 0.0, -0.5877852522924731, -0.9510565162951535,
               -0.9510565162951535, -0.5877852522924731))
LOFAR_ROOTS(11, V_(1.0, 0.8412535328311812, 0.41541501300188644, -0.14231483827328514,
                   -0.6548607339452851, -0.9594929736144974, -0.9594929736144974,
                   -0.6548607339452851, -0.14231483827328514, 0.41541501300188644,
                   0.8412535328311812),
            V_(0.0, 0.5406408174555976, 0.9096319953545183, 0.9898214418809327,
               0.7557495743542583, 0.28173255684142967, -0.28173255684142967,
               -0.7557495743542583, -0.9898214418809327, -0.9096319953545183,
               -0.5406408174555976))
LOFAR_ROOTS(12, V_(1.0, 0.8660254037844386, 0.5, 0.0, -0.5, -0.8660254037844386, -1.0,
                   -0.8660254037844386, -0.5, 0.0, 0.5, 0.8660254037844386),
            V_(0.0, 0.5, 0.8660254037844386, 1.0, 0.8660254037844386, 0.5, 0.0, -0.5,
               -0.8660254037844386, -1.0, -0.8660254037844386, -0.5))
LOFAR_ROOTS(13, V_(1.0, 0.8854560256532099, 0.5680647467311558, 0.12053668025532305,
                   -0.3546048870425356, -0.7485107481711011, -0.970941817426052,
                   -0.970941817426052, -0.7485107481711011, -0.3546048870425356,
                   0.12053668025532305, 0.5680647467311558, 0.8854560256532099),
            V_(0.0, 0.46472317204376856, 0.8229838658936564, 0.992708874098054,
               0.9350162426854148, 0.6631226582407952, 0.23931566428755777,
               -0.23931566428755777, -0.6631226582407952, -0.9350162426854148,
               -0.992708874098054, -0.8229838658936564, -0.46472317204376856))
LOFAR_ROOTS(15, V_(1.0, 0.9135454576426009, 0.6691306063588582, 0.30901699437494745,
                   -0.10452846326765347, -0.5, -0.8090169943749475, -0.9781476007338057,
                   -0.9781476007338057, -0.8090169943749475, -0.5, -0.10452846326765347,
                   0.30901699437494745, 0.6691306063588582, 0.9135454576426009),
            V_(0.0, 0.4067366430758002, 0.7431448254773942, 0.9510565162951535,
               0.9945218953682733, 0.8660254037844386, 0.5877852522924731, 0.20791169081775934,
               -0.20791169081775934, -0.5877852522924731, -0.8660254037844386,
               -0.9945218953682733, -0.9510565162951535, -0.7431448254773942,
               -0.4067366430758002))
#undef V_
#undef LOFAR_ROOTS

// x * exp(2 pi i M / N)
template <int N, int M, typename T2>
__device__ __forceinline__ T2 mul_root(T2 x)
{
    using R = decltype(x.x);
    constexpr int m = M % N;
    if constexpr (m == 0) {
        return x;
    } else {
        constexpr R c = (R)Root<N>::c[m], s = (R)Root<N>::s[m];
        return T2{x.x * c - x.y * s, x.x * s + x.y * c};
    }
}

// DFT over an odd prime P, in place: with t_q = x_q + x_{P-q}, d_q = x_q - x_{P-q}, outputs r
// and P-r are x_0 + sum cos(2 pi q r/P) t_q +- i sum sin(2 pi q r/P) d_q.
template <int P, typename T2>
__device__ __forceinline__ void dft_odd(T2* v)
{
    using R = decltype(v[0].x);
    constexpr int H = (P - 1) / 2;
    T2 t[H], d[H], o[P];
    const T2 x0 = v[0];
    o[0] = x0;
#pragma unroll
    for (int q = 1; q <= H; q++) {
        t[q - 1] = c_add(v[q], v[P - q]);
        d[q - 1] = c_sub(v[q], v[P - q]);
        o[0] = c_add(o[0], t[q - 1]);
    }
#pragma unroll
    for (int r = 1; r <= H; r++) {
        T2 a = x0, b = T2{0, 0};
#pragma unroll
        for (int q = 1; q <= H; q++) {
            const R c = (R)Root<P>::c[q * r % P], s = (R)Root<P>::s[q * r % P];
            a.x += c * t[q - 1].x;
            a.y += c * t[q - 1].y;
            b.x += s * d[q - 1].x;
            b.y += s * d[q - 1].y;
        }
        o[r] = T2{a.x - b.y, a.y + b.x};
        o[P - r] = T2{a.x + b.y, a.y - b.x};
    }
#pragma unroll
    for (int r = 0; r < P; r++) v[r] = o[r];
}

template <int P, typename T2>
__device__ __forceinline__ void dft_mixed(T2* v);

// column n2 of an A x B DFT: the A-point DFT of x[B*n1 + n2], times exp(2 pi i n2 k1 / (A B))
template <int A, int B, int N2, int K1, typename T2>
__device__ __forceinline__ void pair_roots(const T2* a, T2* m)
{
    if constexpr (K1 < A) {
        m[K1 * B + N2] = mul_root<A * B, N2 * K1>(a[K1]);
        pair_roots<A, B, N2, K1 + 1>(a, m);
    }
}
template <int A, int B, int N2, typename T2>
__device__ __forceinline__ void pair_cols(const T2* v, T2* m)
{
    if constexpr (N2 < B) {
        T2 a[A];
#pragma unroll
        for (int n1 = 0; n1 < A; n1++) a[n1] = v[B * n1 + N2];
        dft_mixed<A>(a);
        pair_roots<A, B, N2, 0>(a, m);
        pair_cols<A, B, N2 + 1>(v, m);
    }
}
template <int A, int B, typename T2>
__device__ __forceinline__ void dft_pair(T2* v)
{
    T2 m[A * B];
    pair_cols<A, B, 0>(v, m);
#pragma unroll
    for (int k1 = 0; k1 < A; k1++) {
        dft_mixed<B>(&m[k1 * B]);
#pragma unroll
        for (int k2 = 0; k2 < B; k2++) v[k1 + A * k2] = m[k1 * B + k2];
    }
}

// DFT over A*B, A and B coprime (Good's mapping): x[B*n1 + A*n2 mod AB] as an A x B array has
// no factors between its two DFTs, and output k is element (k mod A, k mod B).  Against
// dft_pair it rounds less: transforms of 3000 x 3000 complex floats 1.97e-7 -> 1.84e-7 from 64
// bits, of 1000 x 1000 1.85e-7 -> 1.63e-7.
template <int A, int B, typename T2>
__device__ __forceinline__ void dft_coprime(T2* v)
{
    T2 m[A * B];
#pragma unroll
    for (int n2 = 0; n2 < B; n2++) {
        T2 a[A];
#pragma unroll
        for (int n1 = 0; n1 < A; n1++) a[n1] = v[(B * n1 + A * n2) % (A * B)];
        dft_mixed<A>(a);
#pragma unroll
        for (int k1 = 0; k1 < A; k1++) m[k1 * B + n2] = a[k1];
    }
#pragma unroll
    for (int k1 = 0; k1 < A; k1++) dft_mixed<B>(&m[k1 * B]);
#pragma unroll
    for (int k = 0; k < A * B; k++) v[k] = m[(k % A) * B + k % B];
}

// complex doubles keep dft_pair: with dft_coprime the column kernel's 1024-thread register
// allocation comes out worse (16 planes of 3000 columns of 3000, 1.43 -> 1.56 ms)
template <int A, int B, typename T2>
__device__ __forceinline__ void dft_product(T2* v)
{
    if constexpr (sizeof(T2) == 16)
        dft_pair<A, B>(v);
    else
        dft_coprime<A, B>(v);
}

template <int P, typename T2>
__device__ __forceinline__ void dft_mixed(T2* v)
{
    if constexpr (P == 2 || P == 4 || P == 8 || P == 16)
        dft<P, 1>(v);
    else if constexpr (P == 6)
        dft_product<2, 3>(v);
    else if constexpr (P == 9)
        dft_pair<3, 3>(v);
    else if constexpr (P == 10)
        dft_product<2, 5>(v);
    else if constexpr (P == 12)
        dft_product<4, 3>(v);
    else if constexpr (P == 15)
        dft_product<3, 5>(v);
    else
        dft_odd<P>(v);
}

// Elements one thread holds between a stage's reads and writes, at most (64 VGPRs).
template <typename Real>
constexpr int kMixElems = 128 / (2 * (int)sizeof(Real)) * 2;
// butterflies of radix p per thread, at most
__host__ __device__ constexpr int mix_nb(int elems, int p) { return elems / p > 1 ? elems / p : 1; }

// Lines of a launch: line l starts at (l / per) * plane + (l % per) * lstride.  Element e is at
// e * estride of a column and at (e >> sm) * strip + e % 2^sm of a row: strips of 2^sm columns,
// strip cells apart (one strip for row-major planes: sm = 30, strip 0).
struct MixLines {
    long long count, per, plane, lstride;
    int estride, sm, strip;
    int llog;     // 2^llog lines per workgroup
    int swap;     // inverse sign: parts swapped on the way in and out
};

// LDS slot of element i of the workgroup's lines: one pad slot every 8 keeps a butterfly's
// outputs (a radix apart in the first stages) off each other's banks
__device__ __forceinline__ int mix_pad(int i) { return i + (i >> 3); }

template <typename Real, bool ROWS>
struct MixThread {
    using T2 = typename cplx<Real>::type;
    const T2* in;   // this thread's line
    T2* out;
    T2* buf;
    const T2* tw;
    int n, r0, l, j0, tpl, llog, estride, sm, strip;
    bool active, swap;
    Real scale;
    __device__ __forceinline__ int slot(int e) const
    {
        return mix_pad(ROWS ? l * n + e : (e << llog) + l);
    }
    __device__ __forceinline__ long long at(int e) const
    {
        return ROWS ? (e >> sm) * strip + (e & ((1 << sm) - 1)) : (long long)e * estride;
    }
};

// Inputs of butterfly j into a: from memory (FIRST) or the LDS buffer.
template <int P, bool FIRST, typename Real, bool ROWS, typename T2>
__device__ __forceinline__ void mix_read(const MixThread<Real, ROWS>& m, int j, int nb, T2* a)
{
#pragma unroll
    for (int q = 0; q < P; q++) {
        if constexpr (FIRST) {
            const T2 x = m.in[m.at(j + q * nb)];
            a[q] = m.swap ? T2{x.y, x.x} : x;
        } else {
            a[q] = m.buf[m.slot(j + q * nb)];
        }
    }
}

// Butterfly j: twiddles (all but the first stage; tw: this stage's part of the table), DFT,
// outputs to LDS or memory (LAST).
template <int P, bool FIRST, bool LAST, typename Real, bool ROWS, typename T2>
__device__ __forceinline__ void mix_butterfly(const MixThread<Real, ROWS>& m, const T2* tw, int j,
                                              int ns, unsigned magic, T2* a)
{
    int k = 0, hi = j;  // j mod ns, j - j mod ns
    if constexpr (!FIRST) {
        hi = (int)__umulhi((unsigned)j, magic) * ns;
        k = j - hi;
#pragma unroll
        for (int q = 1; q < P; q++) a[q] = c_mul_tw<1>(a[q], tw[(q - 1) * ns + k]);
    }
    dft_mixed<P>(a);
    const int base = hi * P + k;
#pragma unroll
    for (int r = 0; r < P; r++) {
        if constexpr (LAST) {
            T2 x = a[r];
            x.x *= m.scale;
            x.y *= m.scale;
            m.out[m.at(base + r * ns)] = m.swap ? T2{x.y, x.x} : x;
        } else {
            m.buf[m.slot(base + r * ns)] = a[r];
        }
    }
}

// One stage of radix P with spans ns; FIRST reads memory, LAST stores to it.  Those two take
// one butterfly at a time; a stage between reads all of a thread's butterflies, waits for
// the other threads' reads, and writes them back in place.
template <int P, bool FIRST, bool LAST, typename Real, bool ROWS>
__device__ __forceinline__ void mix_stage(MixThread<Real, ROWS> m, int ns, unsigned magic)
{
    using T2 = typename cplx<Real>::type;
    // opaque per radix: the compiler otherwise computes the addresses of all radices ahead
    // of the switch that picks one (170-350 spilled registers)
    asm volatile("" : "+v"(m.j0), "+v"(m.l));
    const int nb = m.n / P;
    const T2* tw = m.tw + (FIRST ? 0 : ns - m.r0);  // stage_twiddle_order
    if constexpr (FIRST || LAST) {
        if (m.active) {
#pragma unroll 1
            for (int j = m.j0; j < nb; j += m.tpl) {
                T2 a[P];
                mix_read<P, FIRST>(m, j, nb, a);
                mix_butterfly<P, FIRST, LAST>(m, tw, j, ns, magic, a);
            }
        }
    } else {
        constexpr int NB = mix_nb(kMixElems<Real>, P);
        T2 a[NB][P];
#pragma unroll
        for (int i = 0; i < NB; i++) {
            const int j = m.j0 + i * m.tpl;
            if (j < nb) mix_read<P, false>(m, j, nb, a[i]);
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < NB; i++) {
            const int j = m.j0 + i * m.tpl;
            if (j < nb) mix_butterfly<P, false, false>(m, tw, j, ns, magic, a[i]);
        }
    }
    if constexpr (!LAST) __syncthreads();
}

template <bool FIRST, bool LAST, typename Real, bool ROWS>
__device__ __forceinline__ void mix_radix(const MixThread<Real, ROWS>& m, int p, int ns,
                                          unsigned magic)
{
    switch (p) {
        case 2: return mix_stage<2, FIRST, LAST>(m, ns, magic);
        case 3: return mix_stage<3, FIRST, LAST>(m, ns, magic);
        case 4: return mix_stage<4, FIRST, LAST>(m, ns, magic);
        case 5: return mix_stage<5, FIRST, LAST>(m, ns, magic);
        case 6: return mix_stage<6, FIRST, LAST>(m, ns, magic);
        case 7: return mix_stage<7, FIRST, LAST>(m, ns, magic);
        case 8: return mix_stage<8, FIRST, LAST>(m, ns, magic);
        case 9: return mix_stage<9, FIRST, LAST>(m, ns, magic);
        case 10: return mix_stage<10, FIRST, LAST>(m, ns, magic);
        case 11: return mix_stage<11, FIRST, LAST>(m, ns, magic);
        case 12: return mix_stage<12, FIRST, LAST>(m, ns, magic);
        case 13: return mix_stage<13, FIRST, LAST>(m, ns, magic);
        case 15: return mix_stage<15, FIRST, LAST>(m, ns, magic);
        default: return mix_stage<16, FIRST, LAST>(m, ns, magic);
    }
}

template <typename Real, bool ROWS>
__global__ __launch_bounds__(kMixMaxT) void k_fft_mixed(const typename cplx<Real>::type* in,
                                                        typename cplx<Real>::type* out,
                                                        const typename cplx<Real>::type* tw,
                                                        MixPlan plan, MixLines ln, Real scale)
{
    using T2 = typename cplx<Real>::type;
    extern __shared__ __align__(16) char mix_lds[];
    MixThread<Real, ROWS> m;
    const int tid = threadIdx.x;
    m.n = plan.n;
    m.r0 = plan.radix[0];
    m.llog = ln.llog;
    m.tpl = blockDim.x >> ln.llog;
    if constexpr (ROWS) {
        m.l = tid / m.tpl;
        m.j0 = tid % m.tpl;
    } else {  // consecutive lanes on the columns of one row
        m.l = tid & ((1 << ln.llog) - 1);
        m.j0 = tid >> ln.llog;
    }
    const long long line = (xcd_remap(blockIdx.x, gridDim.x) << ln.llog) + m.l;
    m.active = line < ln.count;
    const long long base = m.active ? (line / ln.per) * ln.plane + (line % ln.per) * ln.lstride : 0;
    m.in = in + base;
    m.out = out + base;
    m.buf = (T2*)mix_lds;
    m.tw = tw;
    m.estride = ln.estride;
    m.sm = ln.sm;
    m.strip = ln.strip;
    m.swap = ln.swap != 0;
    m.scale = scale;
    const int last = plan.nstages - 1;
    if (last == 0) {
        mix_radix<true, true>(m, plan.radix[0], 1, 0u);
        return;
    }
    mix_radix<true, false>(m, plan.radix[0], 1, 0u);
    for (int s = 1; s < last; s++)
        mix_radix<false, false>(m, plan.radix[s], plan.ns[s], plan.magic[s]);
    mix_radix<false, true>(m, plan.radix[last], plan.ns[last], plan.magic[last]);
}

// ---------------------------------------------------------------------------
// host dispatch

// Radices of n in descending order with the fewest stages, then the smallest sum (the
// most even split); the stages' cost is their LDS crossing far more than their arithmetic.
static void mix_search(int n, int limit, int depth, int sum, int* cur, int& best_d, int& best_s,
                       int* best)
{
    static const int radices[] = {16, 15, 13, 12, 11, 10, 9, 8, 7, 6, 5, 4, 3, 2};
    if (n == 1) {
        if (depth < best_d || (depth == best_d && sum < best_s)) {
            best_d = depth;
            best_s = sum;
            std::copy(cur, cur + depth, best);
        }
        return;
    }
    if (depth >= best_d || depth >= kMixMaxStages) return;
    for (int r : radices) {
        if (r > limit || n % r) continue;
        cur[depth] = r;
        mix_search(n / r, r, depth + 1, sum + r, cur, best_d, best_s, best);
    }
}

bool mixed_plan(int n, MixPlan& p)
{
    if (n < 2 || n > kMixMaxN) return false;
    int cur[kMixMaxStages], best[kMixMaxStages], d = kMixMaxStages + 1, s = 1 << 30;
    mix_search(n, 16, 0, 0, cur, d, s, best);
    if (d > kMixMaxStages) return false;
    // the two largest radices first and last (one butterfly at a time), the others between
    std::rotate(best + std::min(1, d), best + std::min(2, d), best + d);
    p.n = n;
    p.nstages = d;
    int ns = 1;
    for (int i = 0; i < d; i++) {
        p.radix[i] = best[i];
        p.ns[i] = ns;
        p.magic[i] = ns > 1 ? (unsigned)((1ull << 32) / (unsigned)ns) + 1u : 0u;
        ns *= best[i];
    }
    return true;
}

// stages of a table: the mixed-radix plan (rx 0), or radix rx and the remainder of a power of
// two (Plan in fft_kernels.h)
static bool table_plan(int n, int rx, MixPlan& p)
{
    if (rx == 0) return mixed_plan(n, p);
    if (n < 2 || n > kMixMaxN || (n & (n - 1))) return false;
    p.n = n;
    p.nstages = 0;
    for (int ns = 1; ns < n; ns *= p.radix[p.nstages++]) {
        p.ns[p.nstages] = ns;
        p.radix[p.nstages] = std::min(rx, n / ns);
        p.magic[p.nstages] = 0u;
    }
    return true;
}

bool stage_twiddle_order(int n, int rx, int* order)
{
    MixPlan p;
    if (!table_plan(n, rx, p)) return false;
    std::fill(order, order + n, 0);
    for (int s = 1; s < p.nstages; s++) {
        const int ns = p.ns[s], turn = n / (ns * p.radix[s]);
        for (int q = 1; q < p.radix[s]; q++)
            for (int k = 0; k < ns; k++)
                order[ns - p.radix[0] + (q - 1) * ns + k] = q * k * turn;
    }
    return true;
}

template <typename Real>
__global__ __launch_bounds__(256) void k_stage_twiddles(typename cplx<Real>::type* tw, MixPlan p)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= p.n) return;
    int m = 0;
    for (int s = 1; s < p.nstages; s++) {
        const int ns = p.ns[s], r = i + p.radix[0] - ns;  // q-1, k of stage s
        if (r >= 0 && r < ns * (p.radix[s] - 1))
            m = (r / ns + 1) * (r % ns) * (p.n / (ns * p.radix[s]));
    }
    double sn, cs;
    sincospi(2.0 * (double)m / (double)p.n, &sn, &cs);
    tw[i] = typename cplx<Real>::type{(Real)cs, (Real)sn};
}

hipError_t fill_stage_twiddles(int precision, int n, int rx, void* tw, hipStream_t st)
{
    MixPlan p;
    if (!table_plan(n, rx, p)) return hipErrorInvalidValue;
    const dim3 blocks((unsigned)((n + 255) / 256));
    if (precision == LOFAR_FP64)
        hipLaunchKernelGGL(k_stage_twiddles<double>, blocks, dim3(256), 0, st, (double2*)tw, p);
    else
        hipLaunchKernelGGL(k_stage_twiddles<float>, blocks, dim3(256), 0, st, (float2*)tw, p);
    return hipGetLastError();
}

bool fft_size_ok(int n)
{
    if (n >= 2 && n <= 8192 && (n & (n - 1)) == 0) return true;
    MixPlan p;
    return mixed_plan(n, p);
}

template <typename Real>
hipError_t fft_generic(int sign, const void* in, void* out, const void* tw, int n, long long lines,
                       long long per, long long plane, long long lstride, long long estride,
                       double scale, hipStream_t st, int sm, long long strip)
{
    using T2 = typename cplx<Real>::type;
    MixPlan p;
    if (!mixed_plan(n, p)) return hipErrorInvalidValue;
    if (lines <= 0) return hipSuccess;
    const bool rows = estride == 1;
    const int elems = kMixElems<Real>;
    // Lines per workgroup.  Columns: 64-byte runs, as far as the lines fit 144 KiB of LDS
    // (8192 complex doubles with padding).  Rows are contiguous: one a workgroup, more
    // of short ones so that a workgroup has whole waves.
    const int cap = elems * 512;
    int llog = 0;
    if (rows)
        while ((n << (llog + 1)) <= 1024 && llog < 6) llog++;
    else
        while ((2 * sizeof(T2) << llog) <= 64 && (n << (llog + 1)) <= cap) llog++;
    // Threads: the middle stages' butterflies within their registers, and about 10
    // (complex double) or 16 (complex float) elements a thread.  Fewer waves a line leave
    // room for other lines on the CU: rows of 2400 x 2000 x 16 complex doubles take 606 us
    // at 10 and 711 at 6, rows of 3000 x 16 x 3000 complex floats 609 us at 16 and 759 at 6.
    const int want = sizeof(Real) == 8 ? 10 : 16;
    int tpl = 1;
    for (int s = 1; s + 1 < p.nstages; s++) {
        const int nb = n / p.radix[s], per_thread = mix_nb(elems, p.radix[s]);
        tpl = std::max(tpl, (nb + per_thread - 1) / per_thread);
    }
    const int need = tpl << llog;
    int threads = std::max(need, ((n << llog) + want - 1) / want);
    threads = std::min(kMixMaxT, (threads + 63) / 64 * 64);
    if (threads < need) return hipErrorInvalidValue;
    MixLines ln;
    ln.count = lines;
    ln.per = per;
    ln.plane = plane;
    ln.lstride = lstride;
    ln.estride = (int)estride;
    ln.sm = sm;
    ln.strip = (int)strip;
    ln.llog = llog;
    ln.swap = sign < 0;
    const long long blocks = (lines + (1LL << llog) - 1) >> llog;
    const int slots = n << llog;
    const size_t lds = (size_t)(slots + slots / 8 + 1) * sizeof(T2);
    auto k = rows ? k_fft_mixed<Real, true> : k_fft_mixed<Real, false>;
    hipLaunchKernelGGL(k, dim3((unsigned)blocks), dim3(threads), lds, st, (const T2*)in, (T2*)out,
                       (const T2*)tw, p, ln, (Real)scale);
    return hipGetLastError();
}

template hipError_t fft_generic<double>(int, const void*, void*, const void*, int, long long,
                                        long long, long long, long long, long long, double,
                                        hipStream_t, int, long long);
template hipError_t fft_generic<float>(int, const void*, void*, const void*, int, long long,
                                       long long, long long, long long, long long, double,
                                       hipStream_t, int, long long);

}  // namespace lofar
