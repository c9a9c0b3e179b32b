// Bucketing of the samples into (w-plane, uv tile) buckets for gfx950: a
// two-level counting sort whose histograms live in LDS.
//
// Level 1 groups the samples by super-tile (sst x sst tiles of one w-plane):
// one record (position and channel/polarisation-summed visibility,
// w-stacking_omp.c:85-90,116-133; 32 bytes in FP64 mode, 16 in FP32 mode, Rec32)
// per super-tile the sample's window touches,
// which is one record for almost every sample.  Every workgroup takes a
// contiguous chunk of samples, counts its records (and the tile entries they
// will expand into) per super-tile in LDS histograms, reserves its range in
// each super-tile with one global atomic per non-empty bin, and after the scan
// places its records with LDS cursors.
//
// Level 2 splits every super-tile's records into blocks of at most l2_block
// records, so that the work spreads over many workgroups even when the w
// distribution piles samples into a few planes: a per-block LDS count of the
// entries per tile, a per-super-tile scan over its blocks (which also yields
// the bucket offsets), then a per-block scatter with LDS cursors that expands
// every record into one entry per tile of its window (w-stacking_omp.c:93-96).
// Entries are self-contained (no side arrays), so every scattered write is one
// aligned 16- or 32-byte store.
//
// A plan of few tiles (kStageMaxBins in all) is sorted by level 1 alone, with tiles for
// super-tiles.
//
// Both scatters run staged where their bins fit one per thread (level 1 up to
// kStageMaxBins super-tiles, level 2 always): a round's records are counted, scanned
// and placed in an LDS buffer in bin order, then stored with consecutive lanes on
// consecutive slots, so each bin's records leave as a run instead of one lane per bin
// (the scattered 16-byte stores cost two 32-byte writes each).
#include <type_traits>

#include "grid_kernels.h"

namespace lofar {

constexpr int kMaxFine = 256;     // sst <= 16
constexpr int kUnroll = 4;        // samples or records per thread per round

// n words of p and m words of q
__global__ __launch_bounds__(256) void k_fill_u32(unsigned* p, long long n, unsigned* q,
                                                  long long m, unsigned v)
{
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
    else if (i - n < m) q[i - n] = v;
}

// Tiles [tu_a, tu_b] x [tv_a, tv_b] of a non-empty window.
struct TileSpan {
    int tu_a, tu_b, tv_a, tv_b;
};
__device__ __forceinline__ TileSpan tiles_of(const Window& s)
{
    return TileSpan{s.j0 / kTile, s.j1 / kTile, s.k0 / kTile, s.k1 / kTile};
}

// ---------------------------------------------------------------------------
// level 1: count

// GLOBAL: more super-tiles than the LDS histograms hold; the counts go straight to
// count1/count1e with global atomics (no per-workgroup bases).
template <bool GLOBAL>
__global__ __launch_bounds__(256) void k_l1_count(int mode, long long n, const double* uu,
                                                  const double* vv, const double* ww, Geometry g,
                                                  TileMap tm, long long chunk, unsigned* count1,
                                                  unsigned* count1e, unsigned* base1, int* err)
{
    extern __shared__ unsigned hist_lds[];  // [nk1] records, then [nk1] entries
    unsigned* hist = GLOBAL ? count1 : hist_lds;
    unsigned* hent = GLOBAL ? count1e : hist_lds + tm.nk1;
    const int tid = threadIdx.x;
    if constexpr (!GLOBAL) {
        for (long long k = tid; k < 2 * tm.nk1; k += 256) hist[k] = 0u;
        __syncthreads();
    }
    const long long beg = (long long)blockIdx.x * chunk;
    const long long end = min(n, beg + chunk);
    bool bad = false;
    for (long long i0 = beg + tid; i0 < end; i0 += 256 * kUnroll) {
#pragma unroll
      for (int u = 0; u < kUnroll; u++) {
        const long long i = i0 + (long long)u * 256;
        if (i >= end) break;
        SampleWin s;
        if (!sample_window(uu[i], vv[i], ww[i], g, s)) {
            bad = true;
            continue;
        }
        if (mode == kBucketHome) {
            int cu, cv;
            home_cell(s, g, cu, cv);
            const long long k = tm.key1(s.gw, cv / kTile, cu / kTile);
            atomicAdd(&hist[k], 1u);
            atomicAdd(&hent[k], 1u);
            continue;
        }
        if (s.j0 > s.j1 || s.k0 > s.k1) continue;
        const TileSpan t = tiles_of(s);
        for (int sv = t.tv_a >> tm.lsst; sv <= t.tv_b >> tm.lsst; sv++) {
            const int nv = min(t.tv_b, (sv << tm.lsst) + tm.sst - 1) - max(t.tv_a, sv << tm.lsst) + 1;
            for (int su = t.tu_a >> tm.lsst; su <= t.tu_b >> tm.lsst; su++) {
                const int nu =
                    min(t.tu_b, (su << tm.lsst) + tm.sst - 1) - max(t.tu_a, su << tm.lsst) + 1;
                const long long k = tm.key_st(s.gw, sv, su);
                atomicAdd(&hist[k], 1u);
                atomicAdd(&hent[k], (unsigned)(nu * nv));
            }
        }
      }
    }
    if (bad) atomicOr(err, 1);
    if constexpr (GLOBAL) return;
    __syncthreads();
    unsigned* my_base = base1 + (long long)blockIdx.x * tm.nk1;
    for (long long k = tid; k < tm.nk1; k += 256) {
        const unsigned c = hist[k], ce = hent[k];
        my_base[k] = c ? atomicAdd(&count1[k], c) : 0u;
        if (ce) atomicAdd(&count1e[k], ce);
    }
}

// ---------------------------------------------------------------------------
// scans over the super-tiles

// Exclusive scan of one value per thread over the workgroup; the sum to total.
// Ends with every wave past the barrier that publishes the wave sums.
template <int NT, typename T>
__device__ __forceinline__ T block_exscan(T v, T* wsum, T& total)
{
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    T x = v;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const T y = __shfl_up(x, d, 64);
        if (lane >= d) x += y;
    }
    if (lane == 63) wsum[wid] = x;
    __syncthreads();
    T pre = 0, tot = 0;
#pragma unroll NT <= 512 ? NT / 64 : 1
    for (int w = 0; w < NT / 64; w++) {
        const T s = wsum[w];
        pre += w < wid ? s : (T)0;
        tot += s;
    }
    total = tot;
    return pre + x - v;
}

// Lists a dense tile and its pieces; the tile's place in the list is left in slots.
__device__ __forceinline__ void list_heavy(const Heavy& h, long long bkt, long long beg,
                                           long long n, int* slots, int* nslots)
{
    const int np = (int)((n + h.piece - 1) / h.piece);
    const int t = atomicAdd(&h.count[0], 1), p0 = atomicAdd(&h.count[1], np);
    HeavyTile d;
    d.bkt = bkt;
    d.beg = beg;
    d.end = beg + n;
    d.np = np;
    d.pad = 0;
    h.tile[t] = d;
    for (int i = 0; i < np; i++) h.piece_of[p0 + i] = int2{t, i};
    slots[atomicAdd(nslots, 1)] = t;
}

// Clears the states of the workgroup's listed tiles.
template <int NT>
__device__ __forceinline__ void clear_heavy(const Heavy& h, const int* slots, int nslots)
{
    if (!h.state) return;
    constexpr int W = sizeof(HeavyState) / 4;
    for (int i = threadIdx.x; i < nslots * W; i += NT)
        ((unsigned*)&h.state[slots[i / W]])[i % W] = 0u;
}

// One workgroup: record, entry and level-2 block offsets of every super-tile, the block
// table, and the call's status (entry total, validation flag, then seq, which the host waits
// for) straight into host memory.  Nine scan launches and a copy took 45 us of a small
// image's 220; this takes 11 at 64 bins, 18 for 16M samples and 37 for 64M on 512 super-tiles:
// the status's stores wait for host memory one after the other, and the block table's binary
// searches grow with the blocks.  boff null: one level, the super-tiles are the tiles; dense
// ones are listed here, and the largest count goes to the host.
__global__ __launch_bounds__(1024) void k_l1_scan(long long nk1, const unsigned* count1,
                                                  const unsigned* count1e, long long* off1,
                                                  long long* eoff1, long long bs, long long* boff,
                                                  L2Block* blk, const int* err,
                                                  volatile long long* status, long long seq,
                                                  Heavy h)
{
    __shared__ long long ws[3][1024 / 64];
    __shared__ int hslot[1024], hn;
    __shared__ unsigned top;
    const int tid = threadIdx.x;
    if (tid == 0) {
        top = 0u;
        hn = 0;
    }
    long long crec = 0, cent = 0, cblk = 0;
    for (long long c0 = 0; c0 < nk1; c0 += 1024) {
        const long long k = c0 + tid;
        const long long r = k < nk1 ? (long long)count1[k] : 0;
        const long long e = k < nk1 ? (long long)count1e[k] : 0;
        const long long nb = (r + bs - 1) / bs;
        long long tr, te, tb;
        const long long rec = crec + block_exscan<1024>(r, ws[0], tr);
        const long long ent = cent + block_exscan<1024>(e, ws[1], te);
        const long long b0 = cblk + block_exscan<1024>(nb, ws[2], tb);
        if (k < nk1) {
            off1[k] = rec;
            eoff1[k] = ent;
            if (boff) boff[k] = b0;
        }
        if (!boff) {
            if (e > 0) atomicMax(&top, (unsigned)e);
            if (e > h.min) list_heavy(h, k, ent, e, hslot, &hn);
        }
        crec += tr;
        cent += te;
        cblk += tb;
        __syncthreads();  // the wave sums are read: free for the next round
    }
    // the status first: the host prepares the next launches while the rest is written
    if (tid == 0) {
        off1[nk1] = crec;
        eoff1[nk1] = cent;
        if (boff) boff[nk1] = cblk;
        status[0] = cent;
        status[1] = *err;
        status[3] = top;
        __threadfence_system();
        status[2] = seq;
    }
    if (!boff) {
        clear_heavy<1024>(h, hslot, hn);
        return;
    }
    // block descriptors, one thread each: its segment is the last that starts at or before it.
    // off1[nk1] is not read: no barrier stands between its store above and here, and every
    // thread holds the total (crec).
    for (long long j = tid; j < cblk; j += 1024) {
        long long lo = 0, hi = nk1;  // boff[lo] <= j < boff[hi]
        while (hi - lo > 1) {
            const long long mid = (lo + hi) >> 1;
            if (boff[mid] <= j)
                lo = mid;
            else
                hi = mid;
        }
        L2Block d;
        d.k1 = lo;
        d.beg = off1[lo] + (j - boff[lo]) * bs;
        d.end = min(lo + 1 < nk1 ? off1[lo + 1] : crec, d.beg + bs);
        d.pad = 0;
        blk[j] = d;
    }
}

// ---------------------------------------------------------------------------
// level 1: scatter records into super-tile order

// The record of sample i (position e.pu, e.pv and summed visibility e.vr, e.vi) in
// super-tile (sv, su); IDX: the sample's index in the real part's slot instead.
template <typename Rec, bool IDX>
__device__ __forceinline__ Rec make_record(const Entry64& e, const TileMap& tm, int sv, int su,
                                           long long i)
{
    if constexpr (std::is_same<Rec, Rec32>::value) {
        Rec32 r;
        r.u = rec_axis(e.pu, (su << tm.lsst) * kTile, tm.rfb);
        r.v = rec_axis(e.pv, (sv << tm.lsst) * kTile, tm.rfb);
        r.vr = IDX ? __uint_as_float((unsigned)i) : (float)e.vr;
        r.vi = (float)e.vi;
        return r;
    } else if constexpr (std::is_same<Rec, Entry32>::value) {
        // one level: the entry of tile (sv, su), through the record's rounded position, so
        // that both sorts give the same bits
        const int u0 = su * kTile, v0 = sv * kTile;
        const double pu = rec_pos(rec_axis(e.pu, u0, tm.rfb), u0, tm.rfb);
        const double pv = rec_pos(rec_axis(e.pv, v0, tm.rfb), v0, tm.rfb);
        Entry32 r;
        r.wu = pack_cell((int)pu - u0, pu - (double)(int)pu);
        r.wv = pack_cell((int)pv - v0, pv - (double)(int)pv);
        r.vr = IDX ? __uint_as_float((unsigned)i) : (float)e.vr;
        r.vi = (float)e.vi;
        return r;
    } else {
        Entry64 r = e;
        if constexpr (IDX) r.vr = __longlong_as_double(i);
        return r;
    }
}

// Rec: Entry64 (FP64 mode), Rec32 (FP32 mode, position relative to the super-tile,
// rec_axis) or Entry32 (FP32 mode, one level)
// GLOBAL: base1 is one global cursor per super-tile (zeroed), taken with global atomics.
// IDX: the records carry the sample's index (bits of the real part's slot, entry_index)
// instead of its visibility, for a sort kept across calls (plan_fill).
template <typename Rec, bool GLOBAL, bool IDX>
__global__ __launch_bounds__(256) void k_l1_scatter_grid(long long n, long long F, long long P,
                                                         const double* uu, const double* vv,
                                                         const double* ww, const float* vr,
                                                         const float* vi, const float* wt,
                                                         Geometry g, TileMap tm, long long chunk,
                                                         const long long* off1,
                                                         unsigned* base1, Rec* rec)
{
    extern __shared__ unsigned cur_lds[];
    unsigned* cur = GLOBAL ? base1 : cur_lds;
    const int tid = threadIdx.x;
    if constexpr (!GLOBAL) {
        const unsigned* my_base = base1 + (long long)blockIdx.x * tm.nk1;
        for (long long k = tid; k < tm.nk1; k += 256) cur[k] = my_base[k];
        __syncthreads();
    }
    const long long beg = (long long)blockIdx.x * chunk;
    const long long end = min(n, beg + chunk);
    // kUnroll samples per thread per round, their loads issued together
    for (long long i0 = beg + tid; i0 < end; i0 += 256 * kUnroll) {
        SampleWin s[kUnroll];
        Entry64 e[kUnroll];
        bool ok[kUnroll];
#pragma unroll
        for (int u = 0; u < kUnroll; u++) {
            const long long i = min(i0 + (long long)u * 256, end - 1);
            ok[u] = i0 + (long long)u * 256 < end && sample_window(uu[i], vv[i], ww[i], g, s[u]) &&
                    s[u].j0 <= s[u].j1 && s[u].k0 <= s[u].k1;
            if constexpr (IDX) {
                e[u].vr = 0.0;
                e[u].vi = 0.0;
            } else {
                sample_vis(i, F, P, vr, vi, wt, e[u].vr, e[u].vi);
            }
            e[u].pu = s[u].pu;
            e[u].pv = s[u].pv;
        }
#pragma unroll
        for (int u = 0; u < kUnroll; u++) {
            if (!ok[u]) continue;
            const TileSpan t = tiles_of(s[u]);
            for (int sv = t.tv_a >> tm.lsst; sv <= t.tv_b >> tm.lsst; sv++)
                for (int su = t.tu_a >> tm.lsst; su <= t.tu_b >> tm.lsst; su++) {
                    const long long k = tm.key_st(s[u].gw, sv, su);
                    const long long at = off1[k] + atomicAdd(&cur[k], 1u);
                    rec[at] = make_record<Rec, IDX>(e[u], tm, sv, su, i0 + u * 256);
                }
        }
    }
}

// ---------------------------------------------------------------------------
// staged scatters: a 512-thread workgroup takes its items in rounds, counts the
// round's records per bin in LDS, scans, places them in an LDS buffer in bin order
// and then stores the buffer with consecutive lanes on consecutive slots of a bin,
// so that a bin's records leave in runs instead of one lane per bin.  A round's
// records beyond the buffer are stored directly (same slots).  One bin per thread.

constexpr int kStageThreads = 512;  // two workgroups per CU overlap their rounds' phases
constexpr int kStageBytes = 65536;  // LDS buffer of one round's entries (level 2)
static_assert(kStageMaxBins <= kStageThreads && kStageMaxBins <= 65536, "one bin per thread");

// Level 1: buffer capacity (records) and samples per thread and round, so that
// buffer, keys and bins stay within half a CU's 160 KiB of LDS (two workgroups per
// CU) and a round's records (about 1.02 per sample on 16x16-tile super-tiles)
// mostly fit.
template <typename Rec>
struct L1Stage {
    static constexpr int CAP = sizeof(Rec) == sizeof(Rec32) ? 4032 : 2144;
    static constexpr int U = 4;
    static_assert(CAP * (sizeof(Rec) + 2) + kStageMaxBins * 16 + 64 <= 81920, "LDS");
};

// Per-round bin bookkeeping of a staged scatter.  gnext (thread tid's register, bin
// tid): global slot of the bin's next record.  After open(): dst[k] + p is the
// global slot of staged position p of bin k, pos[k] the bin's first staged position.
template <int NT>
struct StageBins {
    long long* dst;
    unsigned *cnt, *pos, *wsum;
    // after the counting pass (and a barrier): the round's layout; zeroes the counts
    __device__ __forceinline__ unsigned open(long long nbins, long long& gnext)
    {
        const int tid = threadIdx.x;
        const unsigned c = tid < nbins ? cnt[tid] : 0u;
        unsigned total;
        const unsigned ex = block_exscan<NT>(c, wsum, total);
        if (tid < nbins) {
            dst[tid] = gnext - (long long)ex;
            pos[tid] = ex;
            cnt[tid] = 0u;
            gnext += c;
        }
        __syncthreads();
        return total;
    }
};

template <typename Rec, bool IDX>
__global__ __launch_bounds__(kStageThreads) __attribute__((amdgpu_waves_per_eu(4)))
void k_l1_scatter_staged(
    long long n, long long F, long long P, const double* uu, const double* vv, const double* ww,
    const float* vr, const float* vi, const float* wt, Geometry g, TileMap tm, long long chunk,
    const long long* off1, const unsigned* base1, Rec* rec)
{
    constexpr int NT = kStageThreads;
    constexpr int CAP = L1Stage<Rec>::CAP;
    constexpr int U = L1Stage<Rec>::U;  // samples per thread and round
    // visibility sum as the record keeps it (float for Rec32: the same bits as rounding later)
    using V = typename std::conditional<sizeof(Rec) == sizeof(Rec32), float, double>::type;
    __shared__ Rec stage[CAP];
    __shared__ unsigned short skey[CAP];
    __shared__ long long dst[kStageMaxBins];
    __shared__ unsigned cnt[kStageMaxBins], pos[kStageMaxBins], wsum[NT / 64];
    StageBins<NT> sb{dst, cnt, pos, wsum};
    const int tid = threadIdx.x;
    long long gnext = 0;
    if (tid < tm.nk1) {
        gnext = off1[tid] + base1[(long long)blockIdx.x * tm.nk1 + tid];
        cnt[tid] = 0u;
    }
    __syncthreads();
    const long long beg = (long long)blockIdx.x * chunk;
    const long long end = min(n, beg + chunk);
    for (long long r0 = beg; r0 < end; r0 += (long long)NT * U) {
        // per sample only the position, plane (-1: no record) and visibility; the
        // window is re-derived from the position in each pass
        double pu[U], pv[U];
        int gw[U];
        V sr[U], si[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const long long i0 = r0 + (long long)u * NT + tid;
            const long long i = min(i0, end - 1);
            SampleWin s;
            const bool ok = i0 < end && sample_window(uu[i], vv[i], ww[i], g, s) &&
                            s.j0 <= s.j1 && s.k0 <= s.k1;
            pu[u] = ok ? s.pu : 0.0;
            pv[u] = ok ? s.pv : 0.0;
            gw[u] = ok ? s.gw : -1;
            if constexpr (IDX) {
                sr[u] = si[u] = (V)0;
            } else {
                double a, b;
                sample_vis(i, F, P, vr, vi, wt, a, b);
                sr[u] = (V)a;
                si[u] = (V)b;
            }
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            if (gw[u] < 0) continue;
            const TileSpan t = tiles_of(window_of(pu[u], pv[u], g));
            for (int sv = t.tv_a >> tm.lsst; sv <= t.tv_b >> tm.lsst; sv++)
                for (int su = t.tu_a >> tm.lsst; su <= t.tu_b >> tm.lsst; su++)
                    atomicAdd(&cnt[tm.key_st(gw[u], sv, su)], 1u);
        }
        __syncthreads();
        const unsigned total = sb.open(tm.nk1, gnext);
#pragma unroll
        for (int u = 0; u < U; u++) {
            if (gw[u] < 0) continue;
            const TileSpan t = tiles_of(window_of(pu[u], pv[u], g));
            const Entry64 e{pu[u], pv[u], (double)sr[u], (double)si[u]};
            for (int sv = t.tv_a >> tm.lsst; sv <= t.tv_b >> tm.lsst; sv++)
                for (int su = t.tu_a >> tm.lsst; su <= t.tu_b >> tm.lsst; su++) {
                    const int k = (int)tm.key_st(gw[u], sv, su);
                    const unsigned p = atomicAdd(&pos[k], 1u);
                    const Rec r = make_record<Rec, IDX>(e, tm, sv, su,
                                                        r0 + (long long)u * NT + tid);
                    if (p < (unsigned)CAP) {
                        stage[p] = r;
                        skey[p] = (unsigned short)k;
                    } else {
                        rec[dst[k] + p] = r;
                    }
                }
        }
        __syncthreads();
        const unsigned m = min(total, (unsigned)CAP);
        for (unsigned j = tid; j < m; j += NT) rec[dst[skey[j]] + j] = stage[j];
        __syncthreads();
    }
}

// wt1: the samples' weights when there is one polarisation (each entry then carries its
// sample's weight, so the degridder reads no weight array in the caller's order), else null.
template <bool GLOBAL>
__global__ __launch_bounds__(256) void k_l1_scatter_home(long long n, const double* uu,
                                                         const double* vv, const double* ww,
                                                         const float* wt1, Geometry g,
                                                         TileMap tm, long long chunk,
                                                         const long long* off1,
                                                         unsigned* base1, DEntry* rec)
{
    extern __shared__ unsigned cur_lds[];
    unsigned* cur = GLOBAL ? base1 : cur_lds;
    const int tid = threadIdx.x;
    if constexpr (!GLOBAL) {
        const unsigned* my_base = base1 + (long long)blockIdx.x * tm.nk1;
        for (long long k = tid; k < tm.nk1; k += 256) cur[k] = my_base[k];
        __syncthreads();
    }
    const long long beg = (long long)blockIdx.x * chunk;
    const long long end = min(n, beg + chunk);
    for (long long i = beg + tid; i < end; i += 256) {
        SampleWin s;
        if (!sample_window(uu[i], vv[i], ww[i], g, s)) continue;
        int cu, cv;
        home_cell(s, g, cu, cv);
        const long long k = tm.key1(s.gw, cv / kTile, cu / kTile);
        DEntry e;
        e.pu = s.pu;
        e.pv = s.pv;
        e.idx = i;
        e.pad = wt1 ? (long long)__float_as_uint(wt1[i]) : 0;
        rec[off1[k] + atomicAdd(&cur[k], 1u)] = e;
    }
}

// Staged form of k_l1_scatter_home (see k_l1_scatter_staged): one record per valid
// sample, in its home tile's super-tile.
__global__ __launch_bounds__(kStageThreads) __attribute__((amdgpu_waves_per_eu(4)))
void k_l1_scatter_home_staged(long long n, const double* uu, const double* vv,
                              const double* ww, const float* wt1, Geometry g, TileMap tm,
                              long long chunk, const long long* off1, const unsigned* base1,
                              DEntry* rec)
{
    constexpr int NT = kStageThreads;
    constexpr int CAP = L1Stage<DEntry>::CAP;
    constexpr int U = L1Stage<DEntry>::U;
    static_assert(U * NT <= CAP, "one record per sample: a round always fits the buffer");
    __shared__ DEntry stage[CAP];
    __shared__ unsigned short skey[CAP];
    __shared__ long long dst[kStageMaxBins];
    __shared__ unsigned cnt[kStageMaxBins], pos[kStageMaxBins], wsum[NT / 64];
    StageBins<NT> sb{dst, cnt, pos, wsum};
    const int tid = threadIdx.x;
    long long gnext = 0;
    if (tid < tm.nk1) {
        gnext = off1[tid] + base1[(long long)blockIdx.x * tm.nk1 + tid];
        cnt[tid] = 0u;
    }
    __syncthreads();
    const long long beg = (long long)blockIdx.x * chunk;
    const long long end = min(n, beg + chunk);
    for (long long r0 = beg; r0 < end; r0 += (long long)NT * U) {
        DEntry e[U];
        int key[U];  // -1: no record
#pragma unroll
        for (int u = 0; u < U; u++) {
            const long long i0 = r0 + (long long)u * NT + tid;
            const long long i = min(i0, end - 1);
            SampleWin s;
            key[u] = -1;
            if (i0 < end && sample_window(uu[i], vv[i], ww[i], g, s)) {
                int cu, cv;
                home_cell(s, g, cu, cv);
                key[u] = (int)tm.key1(s.gw, cv / kTile, cu / kTile);
                e[u].pu = s.pu;
                e[u].pv = s.pv;
                e[u].idx = i;
                e[u].pad = wt1 ? (long long)__float_as_uint(wt1[i]) : 0;
                atomicAdd(&cnt[key[u]], 1u);
            }
        }
        __syncthreads();
        const unsigned total = sb.open(tm.nk1, gnext);
#pragma unroll
        for (int u = 0; u < U; u++) {
            if (key[u] < 0) continue;
            const unsigned p = atomicAdd(&pos[key[u]], 1u);
            stage[p] = e[u];
            skey[p] = (unsigned short)key[u];
        }
        __syncthreads();
        for (unsigned j = tid; j < total; j += NT) rec[dst[skey[j]] + j] = stage[j];
        __syncthreads();
    }
}

// ---------------------------------------------------------------------------
// level 2

enum { kOutFp64 = 0, kOutFp32 = 1, kOutHome = 2 };

// Tiles of the record's window inside super-tile (sv, su), as inclusive ranges
// of fine coordinates; for the home mode the single home tile.
template <typename Rec>
__device__ __forceinline__ void record_pos(const Rec& r, const TileMap&, int, int, double& pu,
                                           double& pv)
{
    pu = r.pu;
    pv = r.pv;
}
__device__ __forceinline__ void record_pos(const Rec32& r, const TileMap& tm, int sv, int su,
                                           double& pu, double& pv)
{
    pu = rec_pos(r.u, (su << tm.lsst) * kTile, tm.rfb);
    pv = rec_pos(r.v, (sv << tm.lsst) * kTile, tm.rfb);
}

template <int OUT, typename Rec>
__device__ __forceinline__ bool record_tiles(const Rec& r, const Geometry& g, const TileMap& tm,
                                             int sv, int su, int& fu_a, int& fu_b, int& fv_a,
                                             int& fv_b, Window& s)
{
    double pu, pv;
    record_pos(r, tm, sv, su, pu, pv);
    s = window_of(pu, pv, g);
    if constexpr (OUT == kOutHome) {
        int cu, cv;
        home_cell(s, g, cu, cv);
        fu_a = fu_b = (cu / kTile) - (su << tm.lsst);
        fv_a = fv_b = (cv / kTile) - (sv << tm.lsst);
        return true;
    } else {
        const TileSpan t = tiles_of(s);
        fu_a = max(t.tu_a - (su << tm.lsst), 0);
        fu_b = min(t.tu_b - (su << tm.lsst), tm.sst - 1);
        fv_a = max(t.tv_a - (sv << tm.lsst), 0);
        fv_b = min(t.tv_b - (sv << tm.lsst), tm.sst - 1);
        return fu_a <= fu_b && fv_a <= fv_b;
    }
}

template <int OUT, typename Rec>
__global__ __launch_bounds__(256) void k_l2_count(Geometry g, TileMap tm, const long long* nblocks,
                                                  const L2Block* blk, const Rec* rec,
                                                  unsigned* cnt2)
{
    __shared__ unsigned cnt[kMaxFine];
    const long long b = blockIdx.x;
    if (b >= *nblocks) return;  // the grid is sized from an upper bound
    const int tid = threadIdx.x;
    const int nf = tm.sst * tm.sst;
    for (int f = tid; f < nf; f += 256) cnt[f] = 0u;
    __syncthreads();
    const L2Block d = blk[b];
    int sv, su;
    tm.super_of(d.k1, sv, su);
    for (long long r0 = d.beg + tid; r0 < d.end; r0 += 256 * kUnroll) {
        Rec xs[kUnroll];
#pragma unroll
        for (int u = 0; u < kUnroll; u++) xs[u] = rec[min(r0 + (long long)u * 256, d.end - 1)];
#pragma unroll
        for (int u = 0; u < kUnroll; u++) {
            if (r0 + (long long)u * 256 >= d.end) break;
            int fu_a, fu_b, fv_a, fv_b;
            Window s;
            if (!record_tiles<OUT>(xs[u], g, tm, sv, su, fu_a, fu_b, fv_a, fv_b, s)) continue;
            for (int fv = fv_a; fv <= fv_b; fv++)
                for (int fu = fu_a; fu <= fu_b; fu++) atomicAdd(&cnt[(fv << tm.lsst) | fu], 1u);
        }
    }
    __syncthreads();
    for (int f = tid; f < nf; f += 256) cnt2[b * nf + f] = cnt[f];
}

// One workgroup per segment: per fine tile, running sums over the segment's blocks (replacing
// the counts by block bases relative to the segment's first entry); the exclusive scan over
// fine tiles gives the bucket offsets.  Four groups of threads, a tile per thread, take a
// quarter of the blocks each and read G blocks' counts at a time (kept for the write where
// they are all): few segments with many blocks were 16 serial round trips, 25 us of a
// 1M-sample image.  Dense tiles are listed on the way (Heavy).
__global__ __launch_bounds__(4 * kMaxFine) void k_l2_scan(TileMap tm, const long long* eoff1,
                                                          const long long* boff, unsigned* cnt2,
                                                          long long* offsets, Heavy h)
{
    __shared__ unsigned part[4][kMaxFine], tile0[kMaxFine], ws[4 * kMaxFine / 64];
    __shared__ int hslot[kMaxFine], hn;
    constexpr int G = 16;
    const int f = threadIdx.x % kMaxFine, grp = threadIdx.x / kMaxFine;
    const int nf = tm.sst * tm.sst;
    const long long k1 = blockIdx.x;
    const long long s0 = boff[k1], s1 = boff[k1 + 1], q = (s1 - s0 + 3) / 4;
    const long long b0 = min(s1, s0 + grp * q), b1 = min(s1, b0 + q);
    const bool on = f < nf;
    const bool whole = q <= G;  // one read of the counts
    unsigned c[G], tot = 0;
    for (long long j = b0; j < b1; j += G) {
#pragma unroll
        for (int i = 0; i < G; i++) c[i] = on && j + i < b1 ? cnt2[(j + i) * nf + f] : 0u;
#pragma unroll
        for (int i = 0; i < G; i++) tot += c[i];
    }
    part[grp][f] = tot;
    if (threadIdx.x == 0) hn = 0;
    __syncthreads();
    unsigned all = 0, before = 0;  // the tile's entries, and those of the groups before
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const unsigned x = part[i][f];
        before += i < grp ? x : 0u;
        all += x;
    }
    unsigned sum;
    const unsigned run0 = block_exscan<4 * kMaxFine>(grp == 0 ? all : 0u, ws, sum);
    if (grp == 0) {
        tile0[f] = run0;
        if (on) offsets[k1 * nf + f] = eoff1[k1] + run0;
        if (on && (long long)all > h.min)
            list_heavy(h, k1 * nf + f, eoff1[k1] + run0, all, hslot, &hn);
    }
    __syncthreads();
    clear_heavy<4 * kMaxFine>(h, hslot, hn);
    unsigned run = tile0[f] + before;
    for (long long j = b0; j < b1; j += G) {
        if (!whole) {
#pragma unroll
            for (int i = 0; i < G; i++) c[i] = on && j + i < b1 ? cnt2[(j + i) * nf + f] : 0u;
        }
#pragma unroll
        for (int i = 0; i < G; i++) {
            if (on && j + i < b1) cnt2[(j + i) * nf + f] = run;
            run += c[i];
        }
    }
    if (k1 == 0 && threadIdx.x == 0) offsets[tm.nk1 * nf] = eoff1[tm.nk1];
}

// The entry of record x (window s) for fine tile (fv, fu) of super-tile (sv, su).
template <int OUT, typename Rec, typename Out>
__device__ __forceinline__ Out make_entry(const Rec& x, const Window& s, const TileMap& tm, int sv,
                                          int su, int fv, int fu)
{
    if constexpr (OUT == kOutFp32) {
        const int u0 = ((su << tm.lsst) + fu) * kTile;
        const int v0 = ((sv << tm.lsst) + fv) * kTile;
        double pu, pv;
        record_pos(x, tm, sv, su, pu, pv);
        Entry32 e;
        e.wu = pack_cell(s.gu - u0, pu - (double)s.gu);
        e.wv = pack_cell(s.gv - v0, pv - (double)s.gv);
        e.vr = x.vr;  // bit for bit (a plan's index, see k_l1_scatter_grid)
        e.vi = x.vi;
        return e;
    } else {
        return x;
    }
}

template <int OUT, typename Rec, typename Out>
__global__ __launch_bounds__(256) void k_l2_scatter(Geometry g, TileMap tm, const long long* eoff1,
                                                    const long long* nblocks, const L2Block* blk,
                                                    const unsigned* cnt2, const Rec* rec,
                                                    Out* ent)
{
    __shared__ unsigned cur[kMaxFine];
    const long long b = blockIdx.x;
    if (b >= *nblocks) return;
    const int tid = threadIdx.x;
    const int nf = tm.sst * tm.sst;
    for (int f = tid; f < nf; f += 256) cur[f] = cnt2[b * nf + f];
    __syncthreads();
    const L2Block d = blk[b];
    int sv, su;
    tm.super_of(d.k1, sv, su);
    const long long beg = eoff1[d.k1];
    for (long long r0 = d.beg + tid; r0 < d.end; r0 += 256 * kUnroll) {
      Rec xs[kUnroll];
#pragma unroll
      for (int u = 0; u < kUnroll; u++) xs[u] = rec[min(r0 + (long long)u * 256, d.end - 1)];
#pragma unroll
      for (int u = 0; u < kUnroll; u++) {
        if (r0 + (long long)u * 256 >= d.end) break;
        const Rec& x = xs[u];
        int fu_a, fu_b, fv_a, fv_b;
        Window s;
        if (!record_tiles<OUT>(x, g, tm, sv, su, fu_a, fu_b, fv_a, fv_b, s)) continue;
        for (int fv = fv_a; fv <= fv_b; fv++) {
            for (int fu = fu_a; fu <= fu_b; fu++) {
                const long long p = beg + atomicAdd(&cur[(fv << tm.lsst) | fu], 1u);
                ent[p] = make_entry<OUT, Rec, Out>(x, s, tm, sv, su, fv, fu);
            }
        }
      }
    }
}

// Level-2 scatter of one block, staged (see k_l1_scatter_staged): rounds of U records
// per thread, the round's entries placed in LDS in fine-tile order, then stored in runs.
template <int OUT, typename Rec, typename Out>
__global__ __launch_bounds__(kStageThreads) void k_l2_scatter_staged(
    Geometry g, TileMap tm, const long long* eoff1, const long long* nblocks, const L2Block* blk,
    const unsigned* cnt2, const Rec* rec, Out* ent)
{
    constexpr int NT = kStageThreads;
    constexpr int CAP = kStageBytes / (int)sizeof(Out);
    constexpr int U = sizeof(Out) == sizeof(Entry32) ? 4 : 2;  // records per thread and round
    __shared__ Out stage[CAP];
    __shared__ unsigned char skey[CAP];
    __shared__ long long dst[kMaxFine];
    __shared__ unsigned cnt[kMaxFine], pos[kMaxFine], wsum[NT / 64];
    StageBins<NT> sb{dst, cnt, pos, wsum};
    const long long b = blockIdx.x;
    if (b >= *nblocks) return;  // the grid is sized from an upper bound
    const int tid = threadIdx.x;
    const int nf = tm.sst * tm.sst;
    const L2Block d = blk[b];
    int sv, su;
    tm.super_of(d.k1, sv, su);
    long long gnext = 0;
    if (tid < nf) {
        gnext = eoff1[d.k1] + cnt2[b * nf + tid];
        cnt[tid] = 0u;
    }
    __syncthreads();
    for (long long r0 = d.beg; r0 < d.end; r0 += (long long)NT * U) {
        Rec xs[U];
        Window s[U];
        int fu_a[U], fu_b[U], fv_a[U], fv_b[U];
        bool ok[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const long long r = r0 + (long long)u * NT + tid;
            xs[u] = rec[min(r, d.end - 1)];
            ok[u] = r < d.end && record_tiles<OUT>(xs[u], g, tm, sv, su, fu_a[u], fu_b[u],
                                                   fv_a[u], fv_b[u], s[u]);
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            if (!ok[u]) continue;
            for (int fv = fv_a[u]; fv <= fv_b[u]; fv++)
                for (int fu = fu_a[u]; fu <= fu_b[u]; fu++)
                    atomicAdd(&cnt[(fv << tm.lsst) | fu], 1u);
        }
        __syncthreads();
        const unsigned total = sb.open(nf, gnext);
#pragma unroll
        for (int u = 0; u < U; u++) {
            if (!ok[u]) continue;
            for (int fv = fv_a[u]; fv <= fv_b[u]; fv++)
                for (int fu = fu_a[u]; fu <= fu_b[u]; fu++) {
                    const int f = (fv << tm.lsst) | fu;
                    const unsigned p = atomicAdd(&pos[f], 1u);
                    const Out e = make_entry<OUT, Rec, Out>(xs[u], s[u], tm, sv, su, fv, fu);
                    if (p < (unsigned)CAP) {
                        stage[p] = e;
                        skey[p] = (unsigned char)f;
                    } else {
                        ent[dst[f] + p] = e;
                    }
                }
        }
        __syncthreads();
        const unsigned m = min(total, (unsigned)CAP);
        for (unsigned j = tid; j < m; j += NT) ent[dst[skey[j]] + j] = stage[j];
        __syncthreads();
    }
}

// ---------------------------------------------------------------------------
// host dispatch

static inline unsigned blocks_for(long long n, int t) { return (unsigned)((n + t - 1) / t); }

hipError_t fill_u32(unsigned* p, long long n, unsigned v, hipStream_t st)
{
    if (n > 0)
        hipLaunchKernelGGL(k_fill_u32, dim3(blocks_for(n, 256)), dim3(256), 0, st, p, n,
                           (unsigned*)nullptr, 0LL, v);
    return hipGetLastError();
}

hipError_t bucket_count(int mode, long long n, const double* uu, const double* vv, const double* ww,
                        const Geometry& g, const Buckets& b, unsigned* zero2, long long nzero2,
                        hipStream_t st)
{
    hipLaunchKernelGGL(k_fill_u32, dim3(blocks_for(b.nzero + nzero2, 256)), dim3(256), 0, st,
                       (unsigned*)b.zero, b.nzero, zero2, nzero2, 0u);
    if (n > 0 && b.global_l1)
        hipLaunchKernelGGL(k_l1_count<true>, dim3((unsigned)b.nwg), dim3(256), 0, st, mode, n, uu,
                           vv, ww, g, b.map, b.chunk, b.count1, b.count1e, b.base1, b.err);
    else if (n > 0)
        hipLaunchKernelGGL(k_l1_count<false>, dim3((unsigned)b.nwg), dim3(256),
                           2 * (size_t)b.map.nk1 * sizeof(unsigned), st, mode, n, uu, vv, ww, g,
                           b.map, b.chunk, b.count1, b.count1e, b.base1, b.err);
    return hipGetLastError();
}

hipError_t bucket_scan(const Buckets& b, long long seq, hipStream_t st)
{
    hipLaunchKernelGGL(k_l1_scan, dim3(1), dim3(1024), 0, st, b.map.nk1, b.count1, b.count1e,
                       b.off1, b.eoff1, b.l2_block, b.one_level ? nullptr : b.l2_boff, b.l2_blk,
                       b.err, b.status, seq, b.one_level ? b.heavy : Heavy());
    return hipGetLastError();
}

template <int OUT, typename Rec, typename Out>
static hipError_t level2(const Geometry& g, const Buckets& b, const Rec* rec, Out* ent,
                         hipStream_t st)
{
    const long long nk1 = b.map.nk1;
    const unsigned grid = (unsigned)b.l2_max_blocks;
    const long long* nblocks = b.l2_boff + nk1;
    hipLaunchKernelGGL((k_l2_count<OUT, Rec>), dim3(grid), dim3(256), 0, st, g, b.map, nblocks,
                       b.l2_blk, rec, b.l2_cnt);
    hipLaunchKernelGGL(k_l2_scan, dim3((unsigned)nk1), dim3(4 * kMaxFine), 0, st, b.map, b.eoff1, b.l2_boff,
                       b.l2_cnt, b.offsets, b.heavy);
    if (b.stage & kStageL2)
        hipLaunchKernelGGL((k_l2_scatter_staged<OUT, Rec, Out>), dim3(grid), dim3(kStageThreads),
                           0, st, g, b.map, b.eoff1, nblocks, b.l2_blk, b.l2_cnt, rec, ent);
    else
        hipLaunchKernelGGL((k_l2_scatter<OUT, Rec, Out>), dim3(grid), dim3(256), 0, st, g, b.map,
                           b.eoff1, nblocks, b.l2_blk, b.l2_cnt, rec, ent);
    return hipGetLastError();
}

template <typename Rec>
static void launch_l1_scatter_grid(bool global_l1, bool index_vis, size_t lds, hipStream_t st,
                                   long long n, long long F, long long P, const double* uu,
                                   const double* vv, const double* ww, const float* vr,
                                   const float* vi, const float* wt, const Geometry& g,
                                   const Buckets& b, Rec* rec)
{
    if (((b.stage & kStageL1) && !global_l1) || std::is_same<Rec, Entry32>::value) {
        auto k = index_vis ? k_l1_scatter_staged<Rec, true> : k_l1_scatter_staged<Rec, false>;
        hipLaunchKernelGGL(k, dim3((unsigned)b.nwg), dim3(kStageThreads), 0, st, n, F, P, uu, vv,
                           ww, vr, vi, wt, g, b.map, b.chunk, b.off1, b.base1, rec);
        return;
    }
    if constexpr (!std::is_same<Rec, Entry32>::value) {
        auto k = global_l1 ? (index_vis ? k_l1_scatter_grid<Rec, true, true>
                                        : k_l1_scatter_grid<Rec, true, false>)
                           : (index_vis ? k_l1_scatter_grid<Rec, false, true>
                                        : k_l1_scatter_grid<Rec, false, false>);
        hipLaunchKernelGGL(k, dim3((unsigned)b.nwg), dim3(256), lds, st, n, F, P, uu, vv, ww, vr,
                           vi, wt, g, b.map, b.chunk, b.off1, b.base1, rec);
    }
}

hipError_t bucket_sort_grid(int precision, long long n, long long F, long long P,
                            const double* uu, const double* vv, const double* ww, const float* vr,
                            const float* vi, const float* wt, const Geometry& g, const Buckets& b,
                            Entry64* rec, void* entries, hipStream_t st, bool index_vis)
{
    const size_t lds = b.global_l1 ? 0 : (size_t)b.map.nk1 * sizeof(unsigned);
    if (n > 0 && b.global_l1) {
        hipError_t e = fill_u32(b.base1, b.map.nk1, 0u, st);
        if (e != hipSuccess) return e;
    }
    if (b.one_level) {
        if (n > 0 && precision == LOFAR_FP64)
            launch_l1_scatter_grid<Entry64>(false, index_vis, lds, st, n, F, P, uu, vv, ww, vr, vi,
                                            wt, g, b, (Entry64*)entries);
        else if (n > 0)
            launch_l1_scatter_grid<Entry32>(false, index_vis, lds, st, n, F, P, uu, vv, ww, vr, vi,
                                            wt, g, b, (Entry32*)entries);
        return hipGetLastError();
    }
    if (precision == LOFAR_FP64) {
        if (n > 0)
            launch_l1_scatter_grid<Entry64>(b.global_l1, index_vis, lds, st, n, F, P, uu, vv, ww,
                                            vr, vi, wt, g, b, rec);
        return level2<kOutFp64>(g, b, (const Entry64*)rec, (Entry64*)entries, st);
    }
    Rec32* rec32 = (Rec32*)rec;  // the record buffer holds total_rec 32-byte records
    if (n > 0)
        launch_l1_scatter_grid<Rec32>(b.global_l1, index_vis, lds, st, n, F, P, uu, vv, ww, vr,
                                      vi, wt, g, b, rec32);
    return level2<kOutFp32>(g, b, (const Rec32*)rec32, (Entry32*)entries, st);
}

// A plan's visibilities: every sample's channel/polarisation-summed weighted visibility as
// k_l1_scatter_grid forms it, in the samples' order (coalesced; rounded to float for
// Entry32, as the entries hold it).  The gridder gathers each entry's by the sample index
// the sort left in its real part's slot; where it takes filled entries only (accumulation
// variants), k_plan_fill writes them, one 8- or 16-byte gather per entry.
template <typename V2, typename V>
__global__ __launch_bounds__(256) void k_plan_vis(long long n, long long F, long long P,
                                                  const V* vr, const V* vi, const float* wt,
                                                  V2* vis)
{
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double sr, si;
    sample_vis(i, F, P, vr, vi, wt, sr, si);
    V2 x;
    x.x = (decltype(x.x))sr;
    x.y = (decltype(x.y))si;
    vis[i] = x;
}

template <typename Ent, typename V2>
__global__ __launch_bounds__(256) void k_plan_fill(long long total, const Ent* pent, Ent* ent,
                                                   const V2* vis)
{
    const long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= total) return;
    ent[e] = entry_at(pent, vis, e);
}

size_t plan_vis_bytes(int precision, long long n)
{
    return (size_t)n * (precision == LOFAR_FP64 ? sizeof(double2) : sizeof(float2));
}

hipError_t plan_vis(int precision, long long n, long long F, long long P, const void* vr,
                    const void* vi, bool vis64, const float* wt, void* vis, hipStream_t st)
{
    if (n <= 0) return hipSuccess;
    const dim3 gs(blocks_for(n, 256));
    if (vis64 && precision != LOFAR_FP64) return hipErrorInvalidValue;
    if (vis64)
        hipLaunchKernelGGL((k_plan_vis<double2, double>), gs, dim3(256), 0, st, n, F, P,
                           (const double*)vr, (const double*)vi, wt, (double2*)vis);
    else if (precision == LOFAR_FP64)
        hipLaunchKernelGGL((k_plan_vis<double2, float>), gs, dim3(256), 0, st, n, F, P,
                           (const float*)vr, (const float*)vi, wt, (double2*)vis);
    else
        hipLaunchKernelGGL((k_plan_vis<float2, float>), gs, dim3(256), 0, st, n, F, P,
                           (const float*)vr, (const float*)vi, wt, (float2*)vis);
    return hipGetLastError();
}

hipError_t plan_fill(int precision, long long total, const void* pent, void* ent, const void* vis,
                     hipStream_t st)
{
    if (total <= 0) return hipSuccess;
    const dim3 grid(blocks_for(total, 256));
    if (precision == LOFAR_FP64)
        hipLaunchKernelGGL((k_plan_fill<Entry64, double2>), grid, dim3(256), 0, st, total,
                           (const Entry64*)pent, (Entry64*)ent, (const double2*)vis);
    else
        hipLaunchKernelGGL((k_plan_fill<Entry32, float2>), grid, dim3(256), 0, st, total,
                           (const Entry32*)pent, (Entry32*)ent, (const float2*)vis);
    return hipGetLastError();
}

hipError_t bucket_sort_home(long long n, const double* uu, const double* vv, const double* ww,
                            const float* wt1, const Geometry& g, const Buckets& b, DEntry* rec,
                            DEntry* entries, hipStream_t st)
{
    if (b.one_level) rec = entries;
    if (n > 0 && b.global_l1) {
        hipError_t e = fill_u32(b.base1, b.map.nk1, 0u, st);
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL(k_l1_scatter_home<true>, dim3((unsigned)b.nwg), dim3(256), 0, st, n,
                           uu, vv, ww, wt1, g, b.map, b.chunk, b.off1, b.base1, rec);
    } else if (n > 0 && (b.stage & kStageL1)) {
        hipLaunchKernelGGL(k_l1_scatter_home_staged, dim3((unsigned)b.nwg), dim3(kStageThreads),
                           0, st, n, uu, vv, ww, wt1, g, b.map, b.chunk, b.off1, b.base1, rec);
    } else if (n > 0) {
        hipLaunchKernelGGL(k_l1_scatter_home<false>, dim3((unsigned)b.nwg), dim3(256),
                           (size_t)b.map.nk1 * sizeof(unsigned), st, n, uu, vv, ww, wt1, g,
                           b.map, b.chunk, b.off1, b.base1, rec);
    }
    if (b.one_level) return hipGetLastError();
    return level2<kOutHome>(g, b, (const DEntry*)rec, entries, st);
}

}  // namespace lofar
