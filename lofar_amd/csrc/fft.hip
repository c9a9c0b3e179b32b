// Batched per-plane 2D FFT for gfx950: Stockham autosort, radix-E stages
// (E = 8 or 16 elements per thread) with a smaller remainder stage, lines
// staged in LDS between stages.
//
// Semantics follow fftw_data() (fourier_transform.c:7-74): per w-plane an
// unnormalised FFTW_BACKWARD transform over dims (n0=ny, n1=nx) of the [v][u]
// plane, scaled by 1/(nx*ny).  Column transforms run first, then rows, so the
// last pass (rows, contiguous) fuses the w-phase screen and the plane sum of
// phase_correction() (phase_correction.cu:151-210) and the image is written once.
#include <algorithm>
#include <cstdlib>

#include "fft_kernels.h"

namespace lofar {

template <typename Real>
using C2 = typename cplx<Real>::type;

// Raw buffer load of one complex value at byte offset voff + soff (soff
// wave-uniform, held in a scalar register).
template <typename T2>
__device__ __forceinline__ T2 load_soff(__amdgpu_buffer_rsrc_t r, unsigned voff, unsigned soff)
{
    if constexpr (sizeof(T2) == 16)
        return __builtin_bit_cast(T2, __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0));
    else
        return __builtin_bit_cast(T2, __builtin_amdgcn_raw_buffer_load_b64(r, voff, soff, 0));
}

// Raw buffer store of one complex value at byte offset voff + soff.  The whole
// offset goes in the vector register and the scalar offset field is 0: with a
// scalar register there, the compiler does not keep the next VALU instruction
// from overwriting the data registers of a 128-bit store before the store has
// read them, and complex-double stores wrote the following element's value.
template <typename T2>
__device__ __forceinline__ void store_at(T2 x, __amdgpu_buffer_rsrc_t r, unsigned voff,
                                           unsigned soff)
{
    using U4 = unsigned __attribute__((ext_vector_type(4)));
    using U2 = unsigned __attribute__((ext_vector_type(2)));
    if constexpr (sizeof(T2) == 16)
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(U4, x), r, voff + soff, 0, 0);
    else
        __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(U2, x), r, voff + soff, 0, 0);
}

// ---------------------------------------------------------------------------
// standalone passes

// Row transforms: one line (row) per workgroup.  STRIP: rows of strip-major planes
// ([N/L][ny][L], L = 2^sm_log at most TPL; in and out alike), line l row l%ny of plane l/ny.
template <typename Real, int N, int E, int SIGN, bool STRIP>
__global__ __launch_bounds__((Plan<N, E>::TPL)) void k_fft_rows(const C2<Real>* in, C2<Real>* out,
                                                              const C2<Real>* tw, Real scale,
                                                              int ny, int sm_log)
{
    using T2 = C2<Real>;
    using P = Plan<N, E>;
    __shared__ T2 lds[P::LDS];
    const long long line = blockIdx.x;
    const int t = threadIdx.x;
    // element t + d of the row, d a multiple of TPL (whole strips): d*per_u from element t
    const long long base =
        STRIP ? (line / ny) * ny * N + ((((long long)(t >> sm_log) * ny + line % ny) << sm_log) |
                                        (t & ((1 << sm_log) - 1)))
              : line * N + t;
    const int per_u = STRIP ? ny : 1;
    const T2* src = in + base;
    T2* dst = out + base;
    T2 v[P::E];
#pragma unroll
    for (int q = 0; q < P::E; q++) v[q] = src[P::in_index(0, q) * (long long)per_u];
    stages<T2, N, E, SIGN, 1>(v, lds, 1, t, tw);
#pragma unroll
    for (int e = 0; e < P::E; e++) {
        T2 x = v[e];
        x.x *= scale;
        x.y *= scale;
        dst[P::out_index(0, e) * (long long)per_u] = x;
    }
}

// Column transforms: one strip of W adjacent columns per workgroup (W*16 or
// W*8 bytes contiguous per row access), LDS laid out [slot][W].  Workgroups
// are numbered so that the strips one XCD runs at a time are adjacent in
// memory and share its L2 lines.
// OCC: `occ` holds the forward path's occupancy bits (rows of empty tiles read as
// zeros).  NEED: `occ` holds the tiles a degridding reads (same indexing); rows of
// other tiles are not stored, and a strip whose tile column holds none is skipped.
template <typename Real, int N, int E, int W, int ROUNDS, int SIGN, bool OCC, bool NEED = false>
__global__ __launch_bounds__((W * Plan<N, E>::TPL)) void k_fft_cols(const C2<Real>* in,
                                                                 C2<Real>* out,
                                                                 const C2<Real>* tw, int nx,
                                                                 int strips_per_plane,
                                                                 long long nstrips, Real scale,
                                                                 const unsigned long long* occ,
                                                                 int sm_log)
{
    using T2 = C2<Real>;
    using P = Plan<N, E>;
    // complex doubles are stored through a buffer resource (one vector offset per
    // thread, no 64-bit address arithmetic per element), complex floats with
    // global stores (measured as fast, with fewer instructions around them)
    constexpr bool kBufStore = sizeof(T2) >= 16;
    constexpr int WR = W / ROUNDS;  // columns sharing the LDS buffer in one round
    __shared__ T2 lds[P::LDS * WR];
    const long long s = xcd_remap(blockIdx.x, gridDim.x);
    const long long plane = s / strips_per_plane;
    const int u0 = (int)(s % strips_per_plane) * W;
    const int c = threadIdx.x % W;
    const int t = threadIdx.x / W;
    const bool active = u0 + c < nx;  // the last strip of a plane may be partial
    // row-major planes: rows nx apart; strip-major planes ([nx/L][N][L], L = 2^sm_log,
    // a multiple of W): rows L apart inside the strip holding these columns
    const long long rs = sm_log >= 0 ? (1LL << sm_log) : nx;
    const long long plane0 = plane * (long long)N * nx;
    const long long base =
        plane0 +
        (sm_log >= 0 ? ((long long)(u0 >> sm_log) * N << sm_log) + (u0 & ((1 << sm_log) - 1)) + c
                     : (active ? u0 + c : 0));
    // Element q sits dq = in_index(t, q) - t rows below the thread's first row, and
    // output e at out_index(t, e) - t, the same for every thread: buffer accesses
    // are one per-thread byte offset into the plane plus a per-element offset
    // (planes are below 2 GiB, launch_cols_cfg checks: 32-bit offsets).
    const int plane_bytes = (int)((long long)N * nx * (long long)sizeof(T2));
    const unsigned row_step = (unsigned)(rs * (long long)sizeof(T2));
    const unsigned vbase =
        (unsigned)((base - plane0) * (long long)sizeof(T2)) + (unsigned)t * row_step;
    // complex doubles: the stages' twiddles as powers of roots loaded here, ahead
    // of the column data
    constexpr int NWD = ((N + kTile - 1) / kTile + 63) / 64;  // mask words per tile column
    static_assert(NWD <= 2, "tile masks cover at most 128 tile rows");
    unsigned long long need0 = ~0ull, need1 = ~0ull;
    if constexpr (NEED) {
        const int ntu = (nx + kTile - 1) / kTile;
        const unsigned long long* nm = occ + (plane * ntu + u0 / kTile) * NWD;
        need0 = nm[0];
        need1 = NWD > 1 ? nm[1] : 0ull;
        if ((need0 | need1) == 0ull) return;  // nothing of this tile column is read
    }
    constexpr bool kRoots = sizeof(T2) >= 16 && W * P::TPL <= 512;  // not at the 128-VGPR cap
    constexpr int NRT = kRoots ? root_count<N, E>(1) : 0;
    T2 rt[NRT > 0 ? NRT : 1];
    if constexpr (NRT > 0) load_roots<T2, N, E, 1>(rt, t, tw);
    // complex floats: the second stage's twiddles (each row's are shared by the W columns and
    // recur every 16 rows) from LDS, written ahead of the first exchange's barrier
    constexpr int kTwSpan = !kRoots && sizeof(T2) < 16 && N > 256 ? 256 : 0;
    constexpr int NTL = kTwSpan ? kTwSpan - P::R0 : 0;
    __shared__ T2 twl[NTL > 0 ? NTL : 1];
    for (int i = threadIdx.x; i < NTL; i += W * P::TPL) twl[i] = tw[i];
    T2 v[P::E];
    if constexpr (OCC) {
        // An offset past the plane (rows of tiles without samples, columns past the
        // grid) reads zeros without a memory access.
        const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
            (void*)(in + plane0), (short)0, plane_bytes, 0x00020000);  // raw, range-checked
        // bit tv of word tv/64: tile row tv of this strip's tile column holds samples
        const int ntu = (nx + kTile - 1) / kTile;
        const unsigned long long* om = occ + (plane * ntu + u0 / kTile) * NWD;
        const unsigned long long live0 = om[0], live1 = NWD > 1 ? om[1] : 0ull;
        if ((live0 | live1) == 0ull) {
            // no samples anywhere in this strip's tile column: its transform is
            // zero, stored without loads or arithmetic
            if (active) {
                const __amdgpu_buffer_rsrc_t wsrc = __builtin_amdgcn_make_buffer_rsrc(
                    (void*)(out + plane0), (short)0, plane_bytes, 0x00020000);
#pragma unroll
                for (int e = 0; e < P::E; e++)
                    store_at(T2{0, 0}, wsrc, vbase,
                               (unsigned)(P::out_index(0, e)) * row_step);
            }
            return;
        }
#pragma unroll
        for (int q = 0; q < P::E; q++) {
            const int dq = P::in_index(0, q);
            const int tv = (t + dq) / kTile;
            const bool live = active && ((((tv < 64) ? live0 : live1) >> (tv & 63)) & 1ull);
            // offsets of live rows are below 2^31; dead rows read past the plane
            const unsigned voff = live ? vbase : 0x80000000u;
            v[q] = load_soff<T2>(rsrc, voff, (unsigned)dq * row_step);
        }
    } else {
#pragma unroll
        for (int q = 0; q < P::E; q++)
            v[q] = active ? in[base + (long long)P::in_index(t, q) * rs] : T2{0, 0};
    }
    stages<T2, N, E, SIGN, 1, ROUNDS, (NRT > 0), kTwSpan>(v, lds + c % WR, WR, t, tw, c / WR, rt,
                                                          twl);
    if (active) {
        const __amdgpu_buffer_rsrc_t wsrc = __builtin_amdgcn_make_buffer_rsrc(
            (void*)(out + plane0), (short)0, plane_bytes, 0x00020000);
#pragma unroll
        for (int e = 0; e < P::E; e++) {
            if constexpr (NEED) {
                const int tv = (t + P::out_index(0, e)) / kTile;
                if (!((((tv < 64) ? need0 : need1) >> (tv & 63)) & 1ull)) continue;
            }
            T2 x = v[e];
            x.x *= scale;
            x.y *= scale;
            if constexpr (kBufStore)
                store_at(x, wsrc, vbase, (unsigned)(P::out_index(0, e)) * row_step);
            else
                out[base + (long long)P::out_index(t, e) * rs] = x;
        }
    }
}

// ---------------------------------------------------------------------------
// fused passes

// Per-pixel factor sqrt(1-l^2-m^2) (phase_correction.cu:164-172); 1 without the phase.
__device__ __forceinline__ double pixel_fac(const PhaseParams& pp, int iu, double ycoord)
{
    if (!pp.phase_on) return 1.0;
    const double xcoord = pp.coord(iu, pp.xtot);
    const double radius2 = (xcoord * xcoord + ycoord * ycoord);
    return sqrt(1 - radius2);
}

// Row transforms of every plane of one image row, summed over the planes with their w-phase
// factors z0*step^w (phase_start, phase_step; phase_correction.cu:160,182-183,193-195) in registers,
// last plane first: acc = acc*step + v, and the row written once is acc*z0 (Horner: no
// running factor per pixel, a third less state and half the products).  The last
// stage's twiddles stay in registers and the others' in LDS, since every plane's row uses
// the same ones.  FP64 phase and accumulation in both precision modes.
// Row prefetch for k_rows_phase: row iv of plane psrc goes straight into
// pbuf[0, N) with 16-byte direct-to-LDS loads (global_load_lds_dwordx4); wave
// instruction c of the row writes 1 KiB, elements [c*K, (c+1)*K) with K = 1024 /
// sizeof(T2): one run of a row-major row, or a run of each of K/L strips of a strip-major
// plane (every lane has an address of its own).
template <typename T2, int N, int TPL>
__device__ __forceinline__ void prefetch_row(const T2* psrc, T2* pbuf, int t, int iv, int ny,
                                             int sm_log)
{
    constexpr int PER = 16 / (int)sizeof(T2);  // elements per lane
    constexpr int K = 64 * PER;                 // elements per wave instruction
    constexpr int NWAVE = TPL / 64;
    static_assert(NWAVE >= 1 && N % K == 0, "whole waves, whole 1 KiB runs");
    const int lane = t & 63, wave = t >> 6;
    constexpr int ITER = (N / K + NWAVE - 1) / NWAVE;
    // wave-uniform part (scalar registers) plus a per-lane offset: with L <= K columns a
    // strip, element u + k of a wave's K is in strip u/L + k/L
    const int wave_u = __builtin_amdgcn_readfirstlane(wave);
    const int k = lane * PER;
    const T2* lane_src =
        psrc + (sm_log < 0 ? (long long)iv * N + k
                           : ((((long long)(k >> sm_log) * ny + iv) << sm_log) |
                              (k & ((1 << sm_log) - 1))));
    const long long per_u = sm_log < 0 ? 1 : ny;
#pragma unroll
    for (int i = 0; i < ITER; i++) {
        const int c = wave_u + i * NWAVE;
        if (c >= N / K) break;
        const int u = c * K;
        const long long o = u * per_u;
        __builtin_amdgcn_global_load_lds((const void*)(lane_src + o),
                                         (__attribute__((address_space(3))) void*)(pbuf + u), 16,
                                         0, 0);
    }
}

// The fused row passes of complex floats from 2048 on are compiled for two workgroups of
// 4096 a CU (capped at 128 VGPRs, 72 KiB of LDS), which overlap each other's loads, exchanges
// and arithmetic: the last stage's twiddles in registers, the others' in LDS.  The cap costs
// spilled registers, 8 at 4096, 14 at 2048 and 20 in the adjoint, and is a gain with them
// (32 planes of 4096 x 4096: 1.50 -> 1.17 ms).  Shorter rows have
// several workgroups a CU either way, and complex doubles (172-256 VGPRs) one: theirs are
// all in registers, since LDS is what bounds them (1024 rows of 1024 complex doubles and 8
// planes: 48 us, 73 with the early stages' twiddles in LDS).
template <typename Real, int N>
constexpr bool kRowPair = sizeof(Real) == 4 && N >= 2048;
template <typename Real, int N, int E>
constexpr int row_tw_from()
{
    return kRowPair<Real, N> ? last_span<N, E>() : 1;
}

// LDS bytes of k_rows_phase with the row prefetch buffer
template <typename Real, int N, int E>
constexpr bool rows_prefetch_fits()
{
    return (Plan<N, E>::LDS + N + tw_lds<N, E>(row_tw_from<Real, N, E>())) * (int)sizeof(C2<Real>) <= 160 * 1024;
}

// x, hidden from the compiler: what is computed from it again is not kept in registers
__device__ __forceinline__ int opaque(int x)
{
    asm volatile("" : "+v"(x));
    return x;
}

// Groups of threads of a workgroup that share an image row's planes (launch_rows_phase_n);
// rows of short images, whose few workgroups would wait out one plane after the other.
constexpr int kRowGroups = 4;

// G: groups of Plan::TPL threads, group g takes planes [g*ceil(nw/G), ...); their sums meet in
// LDS and group 0 writes the row.
template <typename Real, int N, int E, bool PF, int G>
__global__ __launch_bounds__((G * Plan<N, E>::TPL), (kRowPair<Real, N> ? 4 : 1)) void k_rows_phase(
    const C2<Real>* cube, const C2<Real>* tw, int ny, int nw, PhaseParams pp, double scale,
    double* img_re, double* img_im, int accumulate, int sm_log)
{
    using T2 = C2<Real>;
    using P = Plan<N, E>;
    static_assert(G == 1 || !PF, "the prefetch buffer is one group's");
    constexpr int FROM = row_tw_from<Real, N, E>();
    constexpr int NTW = tw_regs<N, E>(FROM), NTL = tw_lds<N, E>(FROM);
    __shared__ T2 lds_all[G * P::LDS];
    __shared__ T2 twl[NTL > 0 ? NTL : 1];
    // PF: plane iw-1's row is loaded into pbuf while plane iw is transformed
    __shared__ __align__(16) T2 pbuf[PF ? N : 1];
    __shared__ double2 sums[G > 1 ? (G - 1) * N : 1];
    // rows of one XCD are adjacent (strips may be narrower than a cache line of its L2)
    const int iv = (int)xcd_remap(blockIdx.x, gridDim.x);
    const int grp = G > 1 ? threadIdx.x / P::TPL : 0;
    const int t = G > 1 ? threadIdx.x % P::TPL : threadIdx.x;
    T2* lds = lds_all + grp * P::LDS;
    const int per = (nw + G - 1) / G, first = grp * per;
    const long long img_row = (long long)iv * N;
    const long long plane_stride = (long long)ny * N;
    const T2* plane = cube + (long long)(first + per - 1) * plane_stride;
    if constexpr (PF) prefetch_row<T2, N, P::TPL>(plane, pbuf, t, iv, ny, sm_log);
    pp.wmin += first * pp.dw;
    const double ycoord = pp.phase_on ? pp.coord(iv, pp.ytot) : 0.0;
    for (int i = threadIdx.x; i < NTL; i += G * P::TPL) twl[i] = tw[i];  // read after barriers
    T2 twr[NTW > 0 ? NTW : 1];
    if constexpr (NTW > 0) load_twiddles<T2, N, E, FROM>(twr, t, tw);
    double2 acc[P::E], step[P::E];
    double fac[P::E];  // kept where there are registers, else computed again at the end
#pragma unroll
    for (int e = 0; e < P::E; e++) {
        fac[e] = pixel_fac(pp, P::out_index(t, e), ycoord);
        step[e] = phase_step(pp, fac[e]);
        acc[e] = double2{0.0, 0.0};
    }
    T2 v[P::E];
    for (int iw = per - 1; iw >= 0; iw--, plane -= plane_stride) {
        if constexpr (PF) {
            wait_loads();
            lds_barrier();  // every wave's part of the row is in pbuf
#pragma unroll
            for (int q = 0; q < P::E; q++) v[q] = pbuf[P::in_index(t, q)];
            lds_barrier();  // pbuf read by every wave: free for the next plane
            if (iw > 0)
                prefetch_row<T2, N, P::TPL>(plane - plane_stride, pbuf, t, iv, ny, sm_log);
        } else {
            // element u of the row: at u (row-major planes) or, in strip-major planes
            // ([N/L][ny][L], L = 2^sm_log), at (u/L)*ny*L + iv*L + u%L
            const bool there = G == 1 || first + iw < nw;
#pragma unroll
            for (int q = 0; q < P::E; q++) {
                const int u = P::in_index(t, q);
                const long long o = sm_log < 0
                                        ? img_row + u
                                        : ((((long long)(u >> sm_log) * ny + iv) << sm_log) |
                                           (u & ((1 << sm_log) - 1)));
                v[q] = there ? plane[o] : T2{0, 0};
            }
        }
        stages_rt<T2, N, E, 1, FROM, PF>(v, lds, t, twr, twl);
#pragma unroll
        for (int e = 0; e < P::E; e++) {
            const double2 a = acc[e], s = step[e];
            acc[e].x = fma(a.x, s.x, fma(-a.y, s.y, (double)v[e].x));
            acc[e].y = fma(a.x, s.y, fma(a.y, s.x, (double)v[e].y));
        }
    }
#pragma unroll
    for (int e = 0; e < P::E; e++) {
        const int u = P::out_index(t, e);
        double2 z0 = phase_start(pp, kRowPair<Real, N> ? pixel_fac(pp, opaque(u), ycoord) : fac[e]);
        z0.x *= scale;  // the transform's 1/(nx*ny), a power of two: exact
        z0.y *= scale;
        acc[e] = cmul(acc[e], z0);
        if (G > 1 && grp > 0) sums[(grp - 1) * N + u] = acc[e];
    }
    if constexpr (G > 1) {
        __syncthreads();
        if (grp > 0) return;
    }
#pragma unroll
    for (int e = 0; e < P::E; e++) {
        const int u = P::out_index(t, e);
        double2 x = acc[e];
#pragma unroll
        for (int g = 1; g < G; g++) {
            const double2 y = sums[(g - 1) * N + u];
            x.x += y.x;
            x.y += y.y;
        }
        const long long o = img_row + u;
        if (accumulate) {
            img_re[o] += x.x;
            img_im[o] += x.y;
        } else {
            img_re[o] = x.x;
            img_im[o] = x.y;
        }
    }
}

// Adjoint of k_rows_phase: for every plane, the image row times the conjugate
// w-phase factor (the row times conj(z0), turned by conj(step) from plane to plane), forward
// row transform, plane row written out.
template <typename Real, int N, int E>
__global__ __launch_bounds__((Plan<N, E>::TPL), (kRowPair<Real, N> ? 4 : 1)) void k_rows_phase_adj(
    C2<Real>* cube, const C2<Real>* tw, int ny, int nw, PhaseParams pp, double scale,
    const double* img_re, const double* img_im)
{
    using T2 = C2<Real>;
    using P = Plan<N, E>;
    constexpr int FROM = row_tw_from<Real, N, E>();
    constexpr int NTW = tw_regs<N, E>(FROM), NTL = tw_lds<N, E>(FROM);
    __shared__ T2 lds[P::LDS];
    __shared__ T2 twl[NTL > 0 ? NTL : 1];
    const int iv = blockIdx.x;
    const int t = threadIdx.x;
    const long long img_row = (long long)iv * N;
    const int per = (nw + gridDim.y - 1) / gridDim.y, first = blockIdx.y * per;
    const int last = min(nw, first + per);
    pp.wmin += first * pp.dw;
    const double ycoord = pp.phase_on ? pp.coord(iv, pp.ytot) : 0.0;
    for (int i = t; i < NTL; i += P::TPL) twl[i] = tw[i];  // read after a stage's barriers
    T2 twr[NTW > 0 ? NTW : 1];
    if constexpr (NTW > 0) load_twiddles<T2, N, E, FROM>(twr, t, tw);
    double2 a[P::E], step[P::E];
#pragma unroll
    for (int q = 0; q < P::E; q++) {
        const int iu = P::in_index(t, q);
        const double fac = pixel_fac(pp, iu, ycoord);
        const double2 z0 = phase_start(pp, fac);
        step[q] = phase_step(pp, fac);
        a[q] = cmul_conj(double2{img_re[img_row + iu], img_im[img_row + iu]}, z0);
    }
    const long long plane_stride = (long long)ny * N;
    for (int iw = first; iw < last; iw++) {
        T2 v[P::E];
#pragma unroll
        for (int q = 0; q < P::E; q++) {
            v[q] = T2{(Real)a[q].x, (Real)a[q].y};
            a[q] = cmul_conj(a[q], step[q]);
        }
        stages_rt<T2, N, E, -1, FROM, true>(v, lds, t, twr, twl);
        T2* dst = cube + (long long)iw * plane_stride + img_row;
#pragma unroll
        for (int e = 0; e < P::E; e++) {
            T2 x = v[e];
            x.x = (Real)(x.x * scale);
            x.y = (Real)(x.y * scale);
            dst[P::out_index(t, e)] = x;
        }
    }
}

// ---------------------------------------------------------------------------
// host-side dispatch

// elements per thread of the fused row passes and of the column pass, and
// columns per strip; LOFAR_FFT_CFG overrides the column configuration (tuning)
constexpr int kRowE = 16;
constexpr int kPhaseE = 8;

static int col_cfg()
{
    static int cfg = -1;
    if (cfg < 0) {
        const char* s = getenv("LOFAR_FFT_CFG");
        cfg = s ? atoi(s) : 0;
    }
    return cfg;
}

template <typename Real, int N>
static hipError_t launch_rows_n(int sign, const void* in, void* out, const void* tw,
                                long long lines, double scale, hipStream_t st, int ny, int sm_log)
{
    using T2 = C2<Real>;
    constexpr int TPL = Plan<N, kRowE>::TPL;
    if (lines <= 0) return hipSuccess;
    auto k = sign > 0 ? k_fft_rows<Real, N, kRowE, 1, false> : k_fft_rows<Real, N, kRowE, -1, false>;
    if (sm_log >= 0) {
        // the images' two-pass rows; shorter rows of strips run in the fused pass
        if (N <= 4096 || sign < 0 || (1 << sm_log) > TPL || ny < 1 || lines % ny)
            return hipErrorInvalidValue;
        if constexpr (N > 4096) k = k_fft_rows<Real, N, kRowE, 1, true>;
    }
    hipLaunchKernelGGL(k, dim3((unsigned)lines), dim3(TPL), 0, st, (const T2*)in, (T2*)out,
                       (const T2*)tw, (Real)scale, ny, sm_log);
    return hipGetLastError();
}

template <typename Real, int N, int E, int WREQ, int RREQ>
static hipError_t launch_cols_cfg(int sign, const void* in, void* out, const void* tw, int nx,
                                  int nw, double scale, const unsigned long long* occ, int sm_log,
                                  hipStream_t st)
{
    using T2 = C2<Real>;
    constexpr int TPL = Plan<N, E>::TPL;
    // at most 1024 threads per workgroup; ROUNDS divides W (both powers of two)
    // and is large enough that one round's columns fit 140 KiB of LDS
    constexpr int W = WREQ * TPL <= 1024 ? WREQ : 1024 / TPL;
    constexpr int COL = Plan<N, E>::LDS * 2 * (int)sizeof(Real);
    constexpr int RMIN = (W * COL + 143359) / 143360;
    constexpr int RMIN2 = RMIN <= 1 ? 1 : RMIN <= 2 ? 2 : RMIN <= 4 ? 4 : RMIN <= 8 ? 8 : 16;
    constexpr int R1 = RREQ > RMIN2 ? RREQ : RMIN2;
    constexpr int ROUNDS = R1 < W ? R1 : W;
    const int strips = (nx + W - 1) / W;
    const long long nstrips = (long long)strips * nw;
    // the kernel addresses a plane with 32-bit byte offsets
    if ((long long)N * nx * (long long)sizeof(T2) >= (1LL << 31)) return hipErrorInvalidValue;
    // forward transforms read `occ` as occupancy, inverse ones as the tiles to store
    auto k = sign > 0 ? (occ ? k_fft_cols<Real, N, E, W, ROUNDS, 1, true>
                             : k_fft_cols<Real, N, E, W, ROUNDS, 1, false>)
                      : (occ ? k_fft_cols<Real, N, E, W, ROUNDS, -1, false, true>
                             : k_fft_cols<Real, N, E, W, ROUNDS, -1, false>);
    // strip-major planes: whole strips of a power-of-two width that W divides
    if (sm_log >= 0 && ((1 << sm_log) % W != 0 || nx % (1 << sm_log) != 0))
        return hipErrorInvalidValue;
    hipLaunchKernelGGL(k, dim3((unsigned)nstrips), dim3(W * TPL), 0, st, (const T2*)in, (T2*)out,
                       (const T2*)tw, nx, strips, nstrips, (Real)scale, occ, sm_log);
    return hipGetLastError();
}

// Column-pass configurations; entry 0 is the default.  W2: strip width whose
// LDS fits ~128 KiB in one round; W64: 64-byte row segments.
template <typename Real, int N>
static hipError_t launch_cols_n(int sign, const void* in, void* out, const void* tw, int nx,
                                int nw, double scale, const unsigned long long* occ, int sm_log,
                                hipStream_t st)
{
    constexpr int B = Plan<N, 16>::LDS * 2 * (int)sizeof(Real);
    constexpr int W2 = 140000 / B >= 1 ? (140000 / B > 16 ? 16 : 140000 / B) : 1;
    constexpr int W64 = 64 / (2 * (int)sizeof(Real));
    // 8192-long complex-double columns at 32 elements a thread would need 128 VGPRs
    // of data alone at 1024 threads (they spilled: 0.74 TB/s); 16 elements, 2 columns
    // and 2 LDS rounds run without spills (2.5 TB/s).  Columns up to 1024 complex doubles
    // also take 16: twice the waves for a strip (54 -> 46 us for 8 planes of 1024 x 1024);
    // 2048 measured the same at 16 and 32, 4096 3.55 ms at 16 and 3.44 at 32.
    if constexpr (sizeof(Real) == 8 && (N >= 8192 || N <= 1024))
        if (col_cfg() == 0 || sm_log >= 0)
            return launch_cols_cfg<Real, N, 16, W64, 2>(sign, in, out, tw, nx, nw, scale, occ, sm_log, st);
    if (sm_log >= 0)
        return launch_cols_cfg<Real, N, 32, W64, 2>(sign, in, out, tw, nx, nw, scale, occ, sm_log, st);
    switch (col_cfg()) {
        case 1: return launch_cols_cfg<Real, N, 16, W2, 1>(sign, in, out, tw, nx, nw, scale, occ, sm_log, st);
        case 2: return launch_cols_cfg<Real, N, 32, W64, 4>(sign, in, out, tw, nx, nw, scale, occ, sm_log, st);
        case 3: return launch_cols_cfg<Real, N, 16, W64, 2>(sign, in, out, tw, nx, nw, scale, occ, sm_log, st);
        default: return launch_cols_cfg<Real, N, 32, W64, 2>(sign, in, out, tw, nx, nw, scale, occ, sm_log, st);
    }
}

// Parts an image row's planes are split into: kRowGroups where one workgroup per row is at
// most 4 waves a CU (rows up to 512 of images as tall) and there are as many planes.
static int row_groups(int tpl, int ny, int nw)
{
    return (long long)ny * std::max(tpl, 64) <= 4 * 64 * 256 && nw >= kRowGroups ? kRowGroups : 1;
}

// the fused row pass: 8 elements per thread, the next row prefetched into LDS where it fits
// and strips are of whole 16-byte loads and no wider than a wave's 1 KiB
template <typename Real, int N>
static hipError_t launch_rows_phase_n(const void* cube, const void* tw, int ny, int nw,
                                      const PhaseParams& pp, double scale, double* re, double* im,
                                      int accumulate, int sm_log, hipStream_t st)
{
    using T2 = C2<Real>;
    constexpr int E = kPhaseE;
    constexpr int K = 1024 / (int)sizeof(T2);
    constexpr bool fits = Plan<N, E>::TPL >= 64 && rows_prefetch_fits<Real, N, E>();
    constexpr int TPL = Plan<N, E>::TPL;
    if constexpr (N <= 512) {
        if (row_groups(TPL, ny, nw) > 1) {
            hipLaunchKernelGGL((k_rows_phase<Real, N, E, false, kRowGroups>), dim3(ny),
                               dim3(kRowGroups * TPL), 0, st, (const T2*)cube, (const T2*)tw, ny,
                               nw, pp, scale, re, im, accumulate, sm_log);
            return hipGetLastError();
        }
    }
    constexpr int PER = 16 / (int)sizeof(T2);
    auto k = fits && (sm_log < 0 || ((1 << sm_log) >= PER && (1 << sm_log) <= K))
                 ? k_rows_phase<Real, N, E, fits, 1>
                 : k_rows_phase<Real, N, E, false, 1>;
    hipLaunchKernelGGL(k, dim3(ny), dim3(TPL), 0, st, (const T2*)cube, (const T2*)tw, ny, nw, pp,
                       scale, re, im, accumulate, sm_log);
    return hipGetLastError();
}

template <typename Real, int N>
static hipError_t launch_rows_phase_adj_n(void* cube, const void* tw, int ny, int nw,
                                          const PhaseParams& pp, double scale, const double* re,
                                          const double* im, hipStream_t st)
{
    using T2 = C2<Real>;
    constexpr int TPL = Plan<N, kPhaseE>::TPL;
    hipLaunchKernelGGL((k_rows_phase_adj<Real, N, kPhaseE>), dim3(ny, row_groups(TPL, ny, nw)),
                       dim3(TPL), 0, st, (T2*)cube, (const T2*)tw, ny, nw, pp,
                       scale, re, im);
    return hipGetLastError();
}

// sides up to 4096 (the fused row passes), and up to 8192
#define LOFAR_FFT_CASES(CALL)     \
    case 2: return CALL(2);       \
    case 4: return CALL(4);       \
    case 8: return CALL(8);       \
    case 16: return CALL(16);     \
    case 32: return CALL(32);     \
    case 64: return CALL(64);     \
    case 128: return CALL(128);   \
    case 256: return CALL(256);   \
    case 512: return CALL(512);   \
    case 1024: return CALL(1024); \
    case 2048: return CALL(2048); \
    case 4096: return CALL(4096);
#define LOFAR_FFT_SWITCH_4096(N_, CALL)       \
    switch (N_) {                             \
        LOFAR_FFT_CASES(CALL)                 \
        default: return hipErrorInvalidValue; \
    }
#define LOFAR_FFT_SWITCH(N_, CALL)            \
    switch (N_) {                             \
        LOFAR_FFT_CASES(CALL)                 \
        case 8192: return CALL(8192);         \
        default: return hipErrorInvalidValue; \
    }

template <typename Real>
hipError_t fft_rows(int sign, const void* in, void* out, const void* tw, int nx, long long lines,
                    double scale, hipStream_t st, int ny, int sm_log)
{
#define CALL_(n) launch_rows_n<Real, n>(sign, in, out, tw, lines, scale, st, ny, sm_log)
    LOFAR_FFT_SWITCH(nx, CALL_)
#undef CALL_
}

template <typename Real>
hipError_t fft_cols(int sign, const void* in, void* out, const void* tw, int nx, int ny, int nw,
                    double scale, hipStream_t st, const unsigned long long* occ, int sm_log)
{
#define CALL_(n) launch_cols_n<Real, n>(sign, in, out, tw, nx, nw, scale, occ, sm_log, st)
    LOFAR_FFT_SWITCH(ny, CALL_)
#undef CALL_
}

template <typename Real>
hipError_t rows_phase(const void* cube, const void* tw, int nx, int ny, int nw,
                      const PhaseParams& pp, double scale, double* re, double* im, int accumulate,
                      hipStream_t st, int sm_log)
{
#define CALL_(n) launch_rows_phase_n<Real, n>(cube, tw, ny, nw, pp, scale, re, im, accumulate, sm_log, st)
    LOFAR_FFT_SWITCH_4096(nx, CALL_)
#undef CALL_
}

template <typename Real>
hipError_t rows_phase_adj(void* cube, const void* tw, int nx, int ny, int nw,
                          const PhaseParams& pp, double scale, const double* re, const double* im,
                          hipStream_t st)
{
#define CALL_(n) launch_rows_phase_adj_n<Real, n>(cube, tw, ny, nw, pp, scale, re, im, st)
    LOFAR_FFT_SWITCH_4096(nx, CALL_)
#undef CALL_
}

int device_cus()
{
    static int cus = 0;
    if (cus == 0) {
        int dev = 0;
        hipDeviceProp_t p;
        if (hipGetDevice(&dev) == hipSuccess && hipGetDeviceProperties(&p, dev) == hipSuccess)
            cus = p.multiProcessorCount;
        if (cus <= 0) cus = 256;
    }
    return cus;
}

template hipError_t fft_rows<double>(int, const void*, void*, const void*, int, long long, double,
                                     hipStream_t, int, int);
template hipError_t fft_rows<float>(int, const void*, void*, const void*, int, long long, double,
                                    hipStream_t, int, int);
template hipError_t fft_cols<double>(int, const void*, void*, const void*, int, int, int, double,
                                     hipStream_t, const unsigned long long*, int);
template hipError_t fft_cols<float>(int, const void*, void*, const void*, int, int, int, double,
                                    hipStream_t, const unsigned long long*, int);
template hipError_t rows_phase<double>(const void*, const void*, int, int, int, const PhaseParams&,
                                       double, double*, double*, int, hipStream_t, int);
template hipError_t rows_phase<float>(const void*, const void*, int, int, int, const PhaseParams&,
                                      double, double*, double*, int, hipStream_t, int);
template hipError_t rows_phase_adj<double>(void*, const void*, int, int, int, const PhaseParams&,
                                           double, const double*, const double*, hipStream_t);
template hipError_t rows_phase_adj<float>(void*, const void*, int, int, int, const PhaseParams&,
                                          double, const double*, const double*, hipStream_t);

}  // namespace lofar
