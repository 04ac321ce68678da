// Scans by minimizer bins: a scan's runs of equal k-mers without sorting its
// tuples.
//
// The reference sorts every tuple of a scan (sortKmerList, metapart.c:1494-1598)
// so that equal k-mers lie together; the filter (metapart.c:2270-2519) and the
// union (2520-2800) then only use the runs, not the order between them.  Here
// consecutive k-mer windows of a read that share their minimizer travel
// together as one 16-byte record (a "super-k-mer", about 10 windows at k = 31)
// to the bin of that minimizer, so equal k-mers meet in one bin, and one
// workgroup builds the runs of a bin in an LDS hash table, evaluates the
// filter on them and writes the labels of the runs to join.  Per window that
// moves about 2 x 2 bytes of records, a share of the 2-bit stream and the 4
// bytes of the labels of runs of two or more, where the radix passes move 13
// bytes per tuple and pass.
//
// Steps (one kernel each):
//   bin_scan     minimizers of every window from the 2-bit stream, the records
//                of a tile and its count per coarse bin; the largest k-mer of
//                every segment (the filter evaluates no last run of a segment)
//   bin_col_*    offsets of every (tile, coarse bin)
//   bin_scatter  records to their coarse bin
//   bin_group    inside a coarse bin: fine cells counted, neighbouring cells
//                cut into bins of about kBinAim windows, records to their bin
//   bin_runs     one workgroup per bin: windows expanded from the 2-bit stream,
//                runs in an LDS table, filter, labels of the runs to join
//   bin_runs_big the same for bins past the table's size, in hashed parts
//
// Measured, whole scan (mp_scan) of 12 M reads of 150 bases at k = 31, 1.44e9
// tuples: 23.5 ms against 67.7 by radix passes; 2.2 M reads of 60-125 bases at
// k = 21: 6.3 against 16.5; 2,500 reads of 100 bases: 0.28 against 0.54.
//
// What this path leaves to the radix sort (mp_sort.hip), see bins_apply():
// k below 20 or 32 (the reference's forward code quirk), 3-minimizer scans,
// reads with letters whose neighbour class the 2-bit code cannot give, scans
// in bucket parts, and inputs whose windows pile up in a few minimizers with
// too many k-mers for bin_runs_big to be the faster way.
#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <memory>
#include <vector>

#include "mp_internal.h"
#include "mp_kmer.h"

namespace mp {

constexpr int kNC = 1024;           // coarse bins
constexpr int kStepPos = 960;       // base positions a wave takes per step: 60 lanes x 16 (4 lanes look ahead)
constexpr int kStepRec = 480;       // records of a step (more: the radix path)
constexpr int kMaxRun = 31;         // windows per record
constexpr uint32_t kBinCap = 4096;  // windows of a bin that bin_runs takes; its table's slots
constexpr uint32_t kBinRec = 1024;  // records of such a bin
constexpr uint32_t kBinAim = kBinCap * 3 / 4;  // windows per bin aimed at, at most (fewer where records hold few)
constexpr int kRunThreads = 1024;
constexpr uint64_t kRunGrid = 1ull << 21;  // bins of a dispatch of bin_runs: fewer than 2^32 threads
constexpr int kBigRec = 64;         // records that bin_runs_big expands at once
constexpr int kBinWit = 8;          // witnesses per bin (bin_runs)
constexpr int kMaxSeg = 256;        // segments (samples of a batch)
constexpr int kStripes = 64;        // copies of the global counters, a cache line each
constexpr uint64_t kCellBases = 1200000000;  // bases from which a coarse bin has 8192 cells instead of 2048

struct BinRec {  // a super-k-mer: consecutive windows of one read with one minimizer
    uint64_t a;      // first window's base (40 bits) | windows << 40 (5) | flags << 45 (2) | cell << 47 (13)
    uint32_t label;
    uint32_t in;     // its windows in the bucket range, the last at bit 0 (scans of part of the buckets)
};
static_assert(kRunGrid * kRunThreads < (1ull << 32), "one dispatch");
static_assert(sizeof(BinRec) == 16, "one 16-byte access");
constexpr uint32_t kPrevN = 1, kNextN = 2;  // flags: no base before the first / after the last window ('N' class)

struct BinDesc {
    uint32_t rec0, nrec, nwin, smp;
};

struct BinCtl {  // device counters of a scan, cleared before it
    unsigned long long nvalid[kMaxSeg];  // windows without 'N' per sample of a batch
    unsigned long long kmax1[kMaxSeg];   // 1 + the largest k-mer of every segment (0: none)
    unsigned long long out;              // labels written (64-aligned per bin)
    unsigned long long big_win;          // windows of the big bins
    unsigned long long big_grp, big_most; // groups of kBigRec of their records: all, the largest bin's
    uint32_t nbin, nbig, err;
    uint32_t next[2];                    // bin_runs_big, and its CHECK: bins taken
    uint32_t pad;
    uint32_t found[kMaxSeg];             // live labels seen in the last segment (of the sample): kFoundOther, kFoundLast
    unsigned long long stat[kStripes][16];  // [0] runs, [1] zeroed; of bin_scan [2] records, [3] windows, [4] of them in range
};

struct BinScan {
    const uint32_t *packed;   // 2-bit stream as 32-bit halves
    const uint16_t *nmask;    // 'N' stream as 16-bit quarters
    const uint16_t *rstart;   // read starts, one bit per base, as nmask
    const uint64_t *base_off;
    uint64_t N, total;        // reads, bases
    int K, steps;             // wave steps per wave of a tile
    uint64_t nsteps;          // wave steps of the input
    uint32_t lo, hi;          // bucket range
    uint16_t *inr;            // windows in it, one bit per base, as nmask; nullptr: all are
    int T;                    // segments (plain) or samples (batch)
    const uint32_t *bounds;   // T + 1 bucket boundaries (plain)
    const uint64_t *first;    // T + 1 first read ids (batch), else nullptr
    const uint32_t *cbase;    // T + 1 first coarse bin of every sample (batch)
    int cell_bits;
    uint64_t *desc;           // kStepRec per step
    uint32_t *nrec, *erank;   // per step: records, reads that start before it
    uint32_t *cnt;            // tiles x kNC
    BinCtl *ctl;
};

__device__ __forceinline__ uint32_t fun32(uint32_t hi, uint32_t lo, int s)  // 32 bits of hi:lo from bit s, s < 32
{
    return s ? (hi << s) | (lo >> (32 - s)) : hi;
}

__device__ __forceinline__ uint32_t rc32(uint32_t x)  // reverse complement of 16 packed bases
{
    x = __builtin_bitreverse32(~x);
    return ((x >> 1) & 0x55555555u) | ((x & 0x55555555u) << 1);
}

// orders a wave's LDS writes before its following reads of other lanes' data
__device__ __forceinline__ void wave_lds_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// last i in [0, n) with first[i] <= x (first ascending, first[0] <= x)
template <typename A, typename V> __device__ __forceinline__ int last_le(const A *first, int n, V x)
{
    int lo = 0, hi = n - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (first[mid] <= x) lo = mid; else hi = mid - 1;
    }
    return lo;
}

// minimizer hash -> (coarse bin of nc, cell): two multiplicative mixes, since
// minimizers are the low end of their own order
__device__ __forceinline__ void bin_of(uint32_t h, uint32_t nc, int cell_bits, uint32_t &coarse, uint32_t &cell)
{
    uint32_t g = h * 0x85EBCA6Bu;
    g ^= g >> 15;
    g *= 0xC2B2AE35u;
    coarse = __umulhi(g, nc);
    uint32_t q = (h ^ (h >> 16)) * 0x27D4EB2Fu;
    q ^= q >> 13;
    q *= 0x165667B1u;
    cell = q >> (32 - cell_bits);
}

// One wave takes 960 base positions per step, 16 per lane; lanes 60-63 only
// look ahead.  Everything of a position comes from the lane's own 16 bases and
// the next lanes' by shuffles: the M-mer hashes, their minimum over the W
// M-mers of the window, the window's validity (no 'N', one read) from bit
// masks.  A record starts where a valid window has another minimizer than the
// one before (or that is not valid), at the step's first position, and at the
// first position of a lane whose 16 windows are all valid without a start
// (about 2 % more records; it bounds a record to 16 + 15 windows).
// Bound by vector instructions.  A lane puts its windows' hashes and masks in
// LDS and only lists its record starts; the records are then made 64 at a time
// (a branch per window and lane before: 920 -> 670 instructions a step; 12 M
// reads 3.25 -> 2.56 ms).  The tiles' totals go to 64 copies of the counters:
// 529 k reads 0.36 -> 0.15 ms, of which 40,000 atomics on one line were most.
// A scan of part of the buckets makes only the records that hold a window in
// them: in one scan of 64 that is every sixth, and what is left holds a window
// at the least, so a bin of up to kBinRec windows never has more records than
// bin_runs takes.
// PART: the scan holds part of the buckets.
template <int M, int W, bool PART>
__global__ __launch_bounds__(256, 4) void bin_scan_kernel(BinScan P)
{
    __shared__ uint4 s_min[4][kWave][5];      // minimizer hashes of a lane's 16 windows (rows 80 bytes apart: no conflicts)
    __shared__ uint4 s_lane[4][kWave];        // what else a record needs of its lane
    __shared__ uint16_t s_start[4][kStepRec]; // the step's record starts: 16 lane + window
    __shared__ uint32_t s_cnt[kNC];
    __shared__ unsigned long long s_max[kMaxSeg];
    __shared__ uint32_t s_nv[kMaxSeg];        // batch: windows per sample
    __shared__ uint32_t s_all[3];             // records, windows, windows in range
    __shared__ uint32_t s_bnd[kMaxSeg + 1];
    __shared__ uint64_t s_first[kMaxSeg + 1];
    __shared__ uint32_t s_cb[kMaxSeg + 1];
    const uint32_t tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
    const bool batch = P.first != nullptr;
    for (uint32_t j = tid; j < kNC; j += 256) s_cnt[j] = 0;
    for (uint32_t j = tid; j < (uint32_t)P.T; j += 256) {
        s_max[j] = P.ctl->kmax1[j];
        s_nv[j] = 0;
    }
    if (tid < 3) s_all[tid] = 0;
    for (uint32_t j = tid; j <= (uint32_t)P.T; j += 256) {
        if (batch) {
            s_first[j] = P.first[j];
            s_cb[j] = P.cbase[j];
        } else {
            s_bnd[j] = P.bounds[j];
        }
    }
    __syncthreads();
    const int K = P.K;
    const uint64_t ws0 = ((uint64_t)blockIdx.x * 4 + wave) * P.steps;
    const uint64_t ws1 = min(ws0 + P.steps, P.nsteps);
    // reads that start before the wave's first position: a 64-way search
    uint64_t rank = 0;
    if (ws0 < ws1 && ws0 > 0) {
        const uint64_t pos = ws0 * kStepPos - 1;
        uint64_t lo = 0, n = P.N;
        while (n > 1) {
            const uint64_t st = (n + 63) / 64, i = lane * st;
            const bool le = i < n && P.base_off[lo + i] <= pos;
            const int c = __popcll(__ballot(le));  // lane 0 holds base_off[lo] <= pos
            lo += (uint64_t)(c - 1) * st;
            n = min(st, n - (uint64_t)(c - 1) * st);
        }
        rank = lo + 1;
    }
    const uint64_t nh = (P.total + 127) / 16;  // halves that the streams hold at the least
    uint32_t over = 0, nv = 0, nin = 0;
    const uint32_t lo12 = P.lo << 12, span = PART ? (P.hi << 12) - lo12 : ~0u;  // of the top 16 bases
    uint32_t rec_total = 0;
    for (uint64_t ws = ws0; ws < ws1; ws++) {
        const uint64_t p0 = ws * kStepPos, h = p0 / 16 + lane;
        const bool have = h < nh;
        const uint32_t X0 = have ? P.packed[h ^ 1] : 0u;
        const uint32_t ne = have ? (uint32_t)P.nmask[h ^ 3] | ((uint32_t)P.rstart[h ^ 3] << 16) : 0u;
        const uint32_t X1 = __shfl_down(X0, 1, kWave), X2 = __shfl_down(X0, 2, kWave);
        const uint32_t ne1 = __shfl_down(ne, 1, kWave), ne2 = __shfl_down(ne, 2, kWave);
        const uint32_t E = ne >> 16;
        // windows: no 'N' in [i, i + K), no read start in (i, i + K), and not a read of K bases
        uint32_t V;
        {
            const uint64_t n = ((uint64_t)(ne & 0xFFFF) << 48) | ((uint64_t)(ne1 & 0xFFFF) << 32) | ((uint64_t)(ne2 & 0xFFFF) << 16);
            const uint64_t e = ((uint64_t)(ne >> 16) << 48) | ((uint64_t)(ne1 >> 16) << 32) | ((uint64_t)(ne2 >> 16) << 16);
            uint64_t x = n | (e << 1);
            x |= x << 1;
            x |= x << 2;
            x |= x << 4;
            x |= x << 8;
            x |= x << (K - 17);  // positions i .. i + K - 2 (K - 1 >= 19)
            x |= n << (K - 1);
            x |= e & (e << K);
            V = (uint32_t)(~x >> 48);
            const uint64_t p = p0 + 16 * lane;
            const uint32_t in = p + 16 <= P.total ? 16u : p < P.total ? (uint32_t)(P.total - p) : 0u;
            V &= 0xFFFF0000u >> in;
            V &= 0xFFFF;
        }
        // hashes of the M-mers at the lane's positions and the W - 1 that follow
        uint32_t a[16 + W - 1];
        {
            const uint64_t fw = ((uint64_t)X0 << 32) | X1;
            const uint64_t rv = ((uint64_t)rc32(X1) << 32) | rc32(X0);
            constexpr uint32_t kM = (1u << (2 * M)) - 1;
#pragma unroll
            for (int j = 0; j < 16; j++) {
                const uint32_t f = (uint32_t)(fw >> (64 - 2 * (j + M))) & kM, r = (uint32_t)(rv >> (2 * j)) & kM;
                a[j] = (min(f, r) ^ 0x2545F49u) * 0x9E3779B1u;
            }
#pragma unroll
            for (int j = 0; j < W - 1; j++) a[16 + j] = __shfl_down(a[j % 16], 1 + j / 16, kWave);
        }
        // minima over W by doubling
        constexpr int kP = W >= 16 ? 16 : 8;
#pragma unroll
        for (int d = 1; d < kP; d <<= 1) {
#pragma unroll
            for (int j = 0; j + d < 16 + W - 1; j++) a[j] = min(a[j], a[j + d]);
        }
        if constexpr (W > kP) {
#pragma unroll
            for (int j = 0; j < 16; j++) a[j] = min(a[j], a[j + W - kP]);
        }
        uint32_t chg = 0;
        const uint32_t before = __shfl_up(a[15], 1, kWave);
#pragma unroll
        for (int j = 0; j < 16; j++) chg = chg + chg + (a[j] != (j ? a[j - 1] : before) ? 1u : 0u);
        const uint32_t Vb = __shfl_up(V, 1, kWave);
        const uint32_t Vn = __shfl_down(V, 1, kWave);
        const uint32_t Vo = lane < 60 ? V : 0u;
        uint32_t S = Vo & (chg | ~((V >> 1) | (lane ? (Vb & 1) << 15 : 0u)));
        if (Vo == 0xFFFF && S == 0) S = 0x8000;
        // 'N' class before the first window: that window is not valid
        uint32_t pv = (V >> 1) | ((Vb & 1) << 15);
        if (lane == 0) {
            bool prev_ok = false;
            if (p0 > 0 && !(E >> 15)) prev_ok = !((P.nmask[((p0 - 1) >> 4) ^ 3] >> (15 - ((p0 - 1) & 15))) & 1);
            pv = (V >> 1) | (prev_ok ? 0x8000u : 0u);
        }
        const uint32_t stop = (~Vo | S) & 0xFFFF;
        const uint32_t lead = stop ? (uint32_t)__builtin_clz(stop) - 16 : 16u;
        const uint32_t nxt = __shfl_down(lead, 1, kWave);
        const uint32_t nx7 = (Vn >> (15 - nxt)) & 1 ? 0u : kNextN;  // the window after a record that leaves the lane
        const uint32_t Eo = lane < 60 ? E : 0u;
        const uint32_t mine = (uint32_t)__popc(S) | ((uint32_t)__popc(Eo) << 16);
        const uint32_t inc = wave_incl(mine), exc = inc - mine;
        const uint32_t tot = __shfl(inc, kWave - 1, kWave);
        uint32_t at = exc & 0xFFFF;
        const uint32_t nr = tot & 0xFFFF;
        const bool fits = nr <= kStepRec;
        // the canonical k-mers' top 16 bases, by position; the windows in the bucket range
        const uint32_t Y0 = rc32(X2), Y1 = rc32(X1), Y2 = rc32(X0);
        const int zs = 2 * (33 - K);
        const uint32_t Z0 = fun32(Y0, Y1, zs), Z1 = fun32(Y1, Y2, zs);
        uint32_t I = 0xFFFF;
        if constexpr (PART) {
            I = 0;
#pragma unroll
            for (int j = 0; j < 16; j++) {
                const uint32_t c = min(fun32(X0, X1, 2 * j), fun32(Z0, Z1, 2 * (15 - j)));
                I = I + I + (c - lo12 < span ? 1u : 0u);
            }
            I &= Vo;
            nin += (uint32_t)__popc(I);
            if (lane < 60) P.inr[h ^ 3] = (uint16_t)I;
        }
        if (!fits) over = 1;
        if (fits) {
#pragma unroll
            for (int j = 0; j < 4; j++) s_min[wave][lane][j] = make_uint4(a[4 * j], a[4 * j + 1], a[4 * j + 2], a[4 * j + 3]);
            s_lane[wave][lane] = make_uint4((stop << 16) | V, (pv << 16) | E, nxt | (nx7 << 8) | (PART ? I << 16 : 0u), exc >> 16);
            for (uint32_t m = S; m;) {
                const uint32_t j = (uint32_t)__builtin_clz(m) - 16;
                m ^= 0x8000u >> j;
                s_start[wave][at++] = (uint16_t)(16 * lane + j);
            }
        }
        wave_lds_fence();
        uint32_t kept = fits && !PART ? nr : 0u;  // records with a window in range (counted below, by lane 0 in whole)
        if (fits) {
            uint64_t *out = P.desc + ws * kStepRec;
            for (uint32_t i = lane; i < nr; i += kWave) {
                const uint32_t o = s_start[wave][i], j = o & 15;
                const uint4 q = s_lane[wave][o >> 4];
                const uint32_t hash = ((const uint32_t *)s_min[wave][o >> 4])[j];
                const uint32_t qs = q.x >> 16, qv = q.x & 0xFFFF, rest = qs & ((0x8000u >> j) - 1);
                const uint32_t end = rest ? (uint32_t)__builtin_clz(rest) - 16 : 16 + (q.z & 31);  // past its last window
                uint32_t to = i;
                if constexpr (PART) {  // a record without a window in range is left out (it ends in its lane or the next)
                    const uint32_t in = ((q.z & 0xFFFF0000u) | (s_lane[wave][(o >> 4) + 1].z >> 16)) << j;
                    const bool keep = in >> (32 - (end - j));
                    const uint64_t m = __ballot(keep);
                    to = kept + (uint32_t)__popcll(m & lanemask_lt());
                    kept += (uint32_t)__popcll(m);
                    if (!keep) continue;
                }
                const uint32_t n7 = rest ? ((qv >> (15 - end)) & 1 ? 0u : kNextN) : (q.z >> 8) & 3;
                const uint32_t p7 = (q.y >> (31 - j)) & 1 ? 0u : kPrevN;
                const uint32_t rk = q.w + (uint32_t)__popc((q.y & 0xFFFF) >> (15 - j));
                const uint32_t misc = o | ((end - j) << 10) | ((p7 | n7) << 15) | (rk << 17);
                uint32_t c0 = 0, nc = kNC;
                if (batch) {
                    const int s = last_le(s_first, P.T, rank + (misc >> 17) - 1);
                    c0 = s_cb[s];
                    nc = s_cb[s + 1] - c0;
                    atomicAdd(&s_nv[s], (misc >> 10) & 31);
                }
                uint32_t coarse, cell;
                bin_of(hash, nc, P.cell_bits, coarse, cell);
                coarse += c0;
                atomicAdd(&s_cnt[coarse], 1u);
                out[to] = (uint64_t)misc | ((uint64_t)coarse << 32) | ((uint64_t)cell << 42);
            }
        }
        rec_total += kept;
        if (lane == 0) {
            P.nrec[ws] = kept;
            P.erank[ws] = (uint32_t)rank;
        }
        // the largest k-mer of every segment: the top 16 bases first, the whole
        // k-mer only where they reach the largest seen
        {
            const int sh = 2 * K - 32;
            uint32_t cand = 0;
            if (!batch) {
                nv += (uint32_t)__popc(Vo);
                cand = I;
            }
            if (P.T == 1 && !batch) {
                const unsigned long long m1 = s_max[0];
                const uint32_t thr = m1 ? (uint32_t)((m1 - 1) >> sh) : 0u, top = PART ? lo12 + span - thr : 0u - thr;
                // [thr, end of the range); thr = 0 (nothing seen yet) or the end at 2^32: all from thr on
                bool any = false;
#pragma unroll
                for (int j = 0; j < 16; j++) {
                    const uint32_t c = min(fun32(X0, X1, 2 * j), fun32(Z0, Z1, 2 * (15 - j)));
                    any |= c - thr <= top - 1;
                }
                if (!any) cand = 0;
                else {
#pragma unroll
                    for (int j = 0; j < 16; j++)
                        if (min(fun32(X0, X1, 2 * j), fun32(Z0, Z1, 2 * (15 - j))) < thr) cand &= ~(0x8000u >> j);
                }
            } else if (batch) {
                // the sample of the lane's windows, when they all lie in one read's sample
                const uint64_t r0 = rank + (exc >> 16);  // reads that start before the lane
                const int s0 = last_le(s_first, P.T, r0 + (E >> 15) - (r0 + (E >> 15) ? 1 : 0));
                const bool one = rank + (inc >> 16) <= s_first[s0 + 1];
                const unsigned long long m1 = s_max[s0];
                const uint32_t thr = one && m1 ? (uint32_t)((m1 - 1) >> sh) : 0u;
#pragma unroll
                for (int j = 0; j < 16; j++) {
                    const uint32_t c = min(fun32(X0, X1, 2 * j), fun32(Z0, Z1, 2 * (15 - j)));
                    if (c >= thr) cand |= 1u << (15 - j);
                }
            } else {
#pragma unroll 4
                for (int j = 0; j < 16; j++) {
                    const uint32_t f = (uint32_t)((((((uint64_t)X0 << 32) | X1) << (2 * j)) >> 32));
                    const uint32_t r = (uint32_t)((((((uint64_t)Z0 << 32) | Z1) << (2 * (15 - j))) >> 32));
                    const uint32_t c = min(f, r), b = c >> 12;
                    if (!((cand >> (15 - j)) & 1)) continue;
                    const int t = last_le(s_bnd, P.T, b);
                    const unsigned long long m1 = s_max[t];
                    if (m1 && c < (uint32_t)((m1 - 1) >> sh)) cand &= ~(0x8000u >> j);
                }
            }
            cand &= Vo;
            while (cand) {
                const int j = __builtin_clz(cand) - 16;
                cand &= ~(0x8000u >> j);
                const uint64_t hi64 = ((uint64_t)X0 << 32) | X1, lo64 = (uint64_t)X2 << 32;
                const uint64_t F = ((hi64 << (2 * j)) | ((lo64 >> 1) >> (63 - 2 * j))) >> (64 - 2 * K);
                const uint64_t R = revcomp(F, K);
                const uint64_t c = F < R ? F : R;
                int t = 0;
                if (batch) t = last_le(s_first, P.T, rank + (exc >> 16) + (uint32_t)__popc(E >> (15 - j)) - 1);
                else if (P.T > 1) t = last_le(s_bnd, P.T, (uint32_t)(c >> (2 * K - 20)));
                atomicMax(&s_max[t], (unsigned long long)c + 1);
            }
        }
        rank += tot >> 16;
        wave_lds_fence();
    }
    if (over) atomicOr(&P.ctl->err, 1u);
    if (!batch)
        for (int o = kWave / 2; o > 0; o >>= 1) {
            nv += __shfl_down(nv, o, kWave);
            nin += __shfl_down(nin, o, kWave);
        }
    if (lane == 0) {
        atomicAdd(&s_all[0], rec_total);
        if (nv) atomicAdd(&s_all[1], nv);
        if (nin) atomicAdd(&s_all[2], nin);
    }
    __syncthreads();
    for (uint32_t j = tid; j < kNC; j += 256) P.cnt[(uint64_t)blockIdx.x * kNC + j] = s_cnt[j];
    for (uint32_t j = tid; j < (uint32_t)P.T; j += 256) {
        if (s_max[j] > P.ctl->kmax1[j]) atomicMax(&P.ctl->kmax1[j], s_max[j]);
        if (batch && s_nv[j]) atomicAdd(&P.ctl->nvalid[j], (unsigned long long)s_nv[j]);
    }
    // (a counter's copies: thousands of atomics on one address take longer than a small scan)
    if (tid < 3 && s_all[tid]) atomicAdd(&P.ctl->stat[blockIdx.x % kStripes][2 + tid], (unsigned long long)s_all[tid]);
}

// ---------------------------------------------------------------- offsets of (tile, coarse bin)
constexpr int kColTiles = 32;

__global__ __launch_bounds__(kNC) void bin_col_sum_kernel(const uint32_t *__restrict__ cnt, uint32_t tiles,
                                                          uint32_t *__restrict__ csum)
{
    const uint32_t c = blockIdx.x, d = threadIdx.x, t0 = c * kColTiles, t1 = min(t0 + kColTiles, tiles);
    uint32_t s = 0;
    for (uint32_t t = t0; t < t1; t++) s += cnt[(uint64_t)t * kNC + d];
    csum[c * kNC + d] = s;
}

// csum to its exclusive prefix over the chunks, coarse[d] the first record of coarse bin d (kNC + 1 entries)
__global__ __launch_bounds__(kNC) void bin_col_scan_kernel(uint32_t *__restrict__ csum, uint32_t nchunk,
                                                           uint32_t *__restrict__ coarse)
{
    __shared__ uint32_t s_w[kNC / kWave];
    const uint32_t d = threadIdx.x, wave = d / kWave;
    uint32_t run = 0;
    constexpr int kU = 8;  // loads in flight a lane (4: 5 % slower)
    for (uint32_t c0 = 0; c0 < nchunk; c0 += kU) {
        uint32_t v[kU];
#pragma unroll
        for (int u = 0; u < kU; u++) v[u] = c0 + u < nchunk ? csum[(c0 + u) * kNC + d] : 0u;
#pragma unroll
        for (int u = 0; u < kU; u++) {
            if (c0 + u < nchunk) csum[(c0 + u) * kNC + d] = run;
            run += v[u];
        }
    }
    const uint32_t inc = wave_incl(run);
    if (__lane_id() == kWave - 1) s_w[wave] = inc;
    __syncthreads();
    uint32_t off = 0;
    for (uint32_t w = 0; w < wave; w++) off += s_w[w];
    coarse[d] = off + inc - run;
    if (d == kNC - 1) coarse[kNC] = off + inc;
}

// cnt to the first record of every (tile, coarse bin)
__global__ __launch_bounds__(kNC) void bin_col_apply_kernel(uint32_t *__restrict__ cnt, uint32_t tiles,
                                                            const uint32_t *__restrict__ csum,
                                                            const uint32_t *__restrict__ coarse)
{
    const uint32_t c = blockIdx.x, d = threadIdx.x, t0 = c * kColTiles, t1 = min(t0 + kColTiles, tiles);
    uint32_t run = coarse[d] + csum[c * kNC + d];
    for (uint32_t t = t0; t < t1; t++) {
        const uint32_t v = cnt[(uint64_t)t * kNC + d];
        cnt[(uint64_t)t * kNC + d] = run;
        run += v;
    }
}

// ---------------------------------------------------------------- records to their coarse bin
// A tile's records in batches, ordered by coarse bin in LDS, so that what a
// batch holds of a bin is written together and the next batch goes on in the
// same line.  (16 bytes at a time from 32 waves of a CU, a line was written
// back in parts: twice the bytes.)  Batches of 6144 records fill a CU's LDS and
// write 96 bytes of a bin at once: 140 M records of 12 M reads 3.18 -> 1.85 ms,
// 2.10 with 3072.  A tile of few steps holds little more than one such batch,
// and there two workgroups of 3072 on a CU overlap better: 4 scans of 2 M reads
// (40 steps, some 4000 records a tile) 2.28 -> 1.10 ms, 1.35 with 6144.  One
// scan, records made and moved, 3072 against 6144: 210 Mb 0.59, 0.63 ms, 450 Mb
// 1.21, 1.11, 900 Mb 2.38, 2.21, 1.8 Gb 4.78, 4.43; four scans 2.27, 2.52; 4.27,
// 4.42; 8.46, 8.40; 16.6, 16.8.
constexpr int kScThreads = 1024;
constexpr int kTileSteps = 512;  // wave steps of a tile at most
constexpr int kScLongTile = 32;  // wave steps per wave of a tile from which the batch is 6144

template <int kScItems>
__global__ __launch_bounds__(kScThreads) void bin_scatter_kernel(KParams G, const uint64_t *__restrict__ desc,
                                                                 const uint32_t *__restrict__ nrec,
                                                                 const uint32_t *__restrict__ erank,
                                                                 const uint32_t *__restrict__ offs, int steps,
                                                                 uint64_t nsteps, const uint64_t *__restrict__ inr,
                                                                 uint4 *__restrict__ rec)
{
    constexpr int kScBatch = kScItems * kScThreads;
    static_assert(kNC == kScThreads && kTileSteps <= kScThreads, "a bin and a step a lane");
    __shared__ uint4 s_rec[kScBatch];
    __shared__ uint16_t s_bin[kScBatch];
    __shared__ uint32_t s_n[kNC], s_at[kNC], s_to[kNC];  // of a batch: records, first place; then first place in rec less that
    __shared__ uint32_t s_first[kTileSteps + 1], s_rank[kTileSteps], s_w[kScThreads / kWave];
    const uint32_t tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
    // tiles of one XCD in one range: the partial lines of two neighbouring tiles meet in one L2
    const uint64_t g = gridDim.x, b = blockIdx.x, x = b & 7, per = g >> 3, rem = g & 7;
    const uint64_t tile = x * per + (x < rem ? x : rem) + (b >> 3);
    const uint64_t ws0 = tile * 4 * steps;
    const uint32_t ns = (uint32_t)min((uint64_t)(4 * steps), nsteps - ws0);
    auto prefix = [&](uint32_t v, uint32_t &total) {  // sum over the lanes before this one
        const uint32_t inc = wave_incl(v);
        __syncthreads();  // s_w is read until here
        if (lane == kWave - 1) s_w[wave] = inc;
        __syncthreads();
        const uint32_t t = wave_incl(s_w[lane % (kScThreads / kWave)]);
        total = (uint32_t)__builtin_amdgcn_readlane((int)t, kScThreads / kWave - 1);
        const uint32_t w = (uint32_t)__builtin_amdgcn_readfirstlane((int)wave);
        return inc - v + (w ? (uint32_t)__builtin_amdgcn_readlane((int)t, (int)w - 1) : 0u);
    };
    uint32_t all = 0;
    {
        const uint32_t v = tid < ns ? nrec[ws0 + tid] : 0u, at = prefix(v, all);
        if (tid < ns) {
            s_first[tid] = at;
            s_rank[tid] = erank[ws0 + tid];
        }
        if (tid == 0) s_first[ns] = all;
    }
    uint32_t cur = offs[tile * kNC + tid];
    s_n[tid] = 0;
    __syncthreads();
    for (uint32_t r0 = 0; r0 < all; r0 += kScBatch) {
        uint64_t v[kScItems];
        uint32_t st[kScItems];
#pragma unroll
        for (int i = 0; i < kScItems; i++) {
            const uint32_t r = r0 + i * kScThreads + tid;
            st[i] = ~0u;
            v[i] = 0;
            if (r >= all) continue;
            uint32_t lo = 0, hi = ns - 1;  // its step: the last with s_first <= r (steps without records share theirs)
            while (lo < hi) {
                const uint32_t mid = (lo + hi + 1) >> 1;
                if (s_first[mid] <= r) lo = mid; else hi = mid - 1;
            }
            st[i] = lo;
            v[i] = desc[(ws0 + lo) * kStepRec + (r - s_first[lo])];
        }
        uint32_t at[kScItems];  // bin | place in it << 10 (no record: ~0)
        uint4 x[kScItems];
#pragma unroll
        for (int i = 0; i < kScItems; i++) {
            at[i] = ~0u;
            if (st[i] == ~0u) continue;
            const uint32_t misc = (uint32_t)v[i], c = (uint32_t)(v[i] >> 32) & (kNC - 1);
            const uint64_t pos = (ws0 + st[i]) * kStepPos + (misc & 1023);
            const uint64_t a = pos | ((uint64_t)((misc >> 10) & 31) << 40) | ((uint64_t)((misc >> 15) & 3) << 45) |
                               (v[i] >> 42 << 47);
            uint32_t in = 0;
            if (inr) {
                const uint32_t o = (uint32_t)pos & 63;
                const uint64_t w = (inr[pos >> 6] << o) | ((inr[(pos >> 6) + 1] >> 1) >> (63 - o));
                in = (uint32_t)(w >> (64 - ((misc >> 10) & 31)));
            }
            x[i] = make_uint4((uint32_t)a, (uint32_t)(a >> 32), label_of(G, (uint64_t)s_rank[st[i]] + (misc >> 17) - 1), in);
            at[i] = c | (atomicAdd(&s_n[c], 1u) << 10);
        }
        __syncthreads();
        uint32_t n;
        const uint32_t mine = s_n[tid], first = prefix(mine, n);
        s_at[tid] = first;
        s_to[tid] = cur - first;
        cur += mine;
        s_n[tid] = 0;
        __syncthreads();
#pragma unroll
        for (int i = 0; i < kScItems; i++) {
            if (at[i] == ~0u) continue;
            const uint32_t c = at[i] & (kNC - 1), p = s_at[c] + (at[i] >> 10);
            s_rec[p] = x[i];
            s_bin[p] = (uint16_t)c;
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < kScItems; i++) {
            const uint32_t p = i * kScThreads + tid;
            if (p < n) rec[s_to[s_bin[p]] + p] = s_rec[p];
        }
        // (the next batch writes s_rec and s_to only behind two more barriers)
    }
}

// ---------------------------------------------------------------- bins of a coarse bin
// One workgroup per coarse bin: records and windows per cell in LDS, cells cut
// into bins where the running window count passes a multiple of `aim`, the
// records moved to their bin: where a lane can hold a bin's cursor (up to 1024
// bins), in batches ordered by bin in LDS, so that what a batch holds of a bin
// is written together (12 M reads 2.93 -> 2.43 ms, four scans of 2 M 1.29 ->
// 1.16), else one by one.  Written were 2.3 times the bytes, as the bins' open
// lines of an XCD's 32 workgroups are more than its cache.
// PART: a record's windows are those in the bucket range.
template <int NM, bool PART>
__global__ __launch_bounds__(1024) void bin_group_kernel(const uint4 *__restrict__ rec, const uint32_t *__restrict__ coarse,
                                                         const uint32_t *__restrict__ smp_of,
                                                         uint4 *__restrict__ out, BinDesc *__restrict__ bins,
                                                         BinDesc *__restrict__ big, uint32_t big_cap, uint32_t aim,
                                                         BinCtl *ctl)
{
    constexpr int kPer = NM / 1024;
    constexpr uint32_t kBatch = NM >= 8192 ? 4096 : 2048, kItems = kBatch / 1024;
    constexpr size_t kRoom = (NM + 1) * sizeof(uint64_t) > kBatch * sizeof(uint4) ? (NM + 1) * sizeof(uint64_t) : kBatch * sizeof(uint4);
    __shared__ unsigned long long s_h[NM];  // records << 32 | windows per cell; then the cell's bin
    __shared__ __align__(16) uint8_t s_room[kRoom];
    __shared__ uint16_t s_bin[kBatch];
    __shared__ uint32_t s_n[1024], s_at[1024], s_to[1024];
    uint64_t *const s_st = (uint64_t *)s_room;  // first record << 32 | first window of every bin; then its cursor
    __shared__ uint64_t s_w[16];
    __shared__ uint32_t s_wb[16], s_place[2];
    const uint32_t tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
    const uint32_t r0 = coarse[blockIdx.x], n = coarse[blockIdx.x + 1] - r0;
    if (n == 0) return;
    if (n >= (1u << 26)) {  // the window counts below are 32 bits: the radix path
        if (tid == 0) atomicOr(&ctl->err, 2u);
        return;
    }
    for (uint32_t j = tid; j < NM; j += 1024) s_h[j] = 0;
    __syncthreads();
    const uint2 *const r2 = (const uint2 *)(rec + r0);
    const uint32_t cmask = NM - 1;
    constexpr int kU = 8;  // loads in flight a lane (4: 5 % slower)
    for (uint32_t i0 = tid; i0 < n; i0 += kU * 1024) {
        uint32_t h[kU], in[kU];
#pragma unroll
        for (int u = 0; u < kU; u++) {
            const uint64_t at = 2 * (uint64_t)min(i0 + u * 1024, n - 1);
            h[u] = r2[at].y;
            in[u] = PART ? r2[at + 1].y : 0u;
        }
#pragma unroll
        for (int u = 0; u < kU; u++)
            if (i0 + u * 1024 < n)
                atomicAdd(&s_h[(h[u] >> 15) & cmask], (1ull << 32) | (PART ? (uint32_t)__popc(in[u]) : (h[u] >> 8) & 31));
    }
    __syncthreads();
    // prefix of (records, windows) over the cells, kPer consecutive cells a lane
    uint64_t v[kPer], sum = 0;
#pragma unroll
    for (int q = 0; q < kPer; q++) {
        v[q] = s_h[tid * kPer + q];
        sum += v[q];
    }
    uint64_t inc = sum;
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1) {
        const uint64_t o = __shfl_up(inc, d, kWave);
        if (lane >= (uint32_t)d) inc += o;
    }
    if (lane == kWave - 1) s_w[wave] = inc;
    __syncthreads();
    uint64_t run = inc - sum, total = 0;
    for (uint32_t w = 0; w < 16; w++) {
        if (w < wave) run += s_w[w];
        total += s_w[w];
    }
    // a cell starts a bin where its first window falls into another multiple of `aim` than its
    // predecessor's (cell - 1's first window is this cell's less that cell's windows), and a cell of
    // more than aim / 3 windows (a deep genome's) is a bin by itself: a bin of several cells holds
    // at most 4/3 aim windows, however deep its cells
    uint32_t lead = 0;
    uint64_t st[kPer];
    uint64_t prev = tid ? s_h[tid * kPer - 1] : 0;
    {
        uint64_t p = run;
#pragma unroll
        for (int q = 0; q < kPer; q++) {
            st[q] = p;
            const uint32_t w1 = (uint32_t)p, w0 = (uint32_t)p - (uint32_t)prev;
            if ((tid == 0 && q == 0) || w1 / aim != w0 / aim || (uint32_t)v[q] > aim / 3 || (uint32_t)prev > aim / 3)
                lead |= 1u << q;
            prev = v[q];
            p += v[q];
        }
    }
    const uint32_t nl = (uint32_t)__popc(lead), linc = wave_incl(nl);
    if (lane == kWave - 1) s_wb[wave] = linc;
    __syncthreads();  // also: every lane has read s_h
    uint32_t b = linc - nl, nb = 0;
    for (uint32_t w = 0; w < 16; w++) {
        if (w < wave) b += s_wb[w];
        nb += s_wb[w];
    }
#pragma unroll
    for (int q = 0; q < kPer; q++) {
        if ((lead >> q) & 1) s_st[b++] = st[q];
        s_h[tid * kPer + q] = b - 1;
    }
    if (tid == 0) s_st[nb] = total;
    __syncthreads();
    // the bins' entries: places in the lists for all of them at once, then per wave
    const uint32_t smp = smp_of ? smp_of[blockIdx.x] : 0u;
    auto entry = [&](uint32_t i, bool &small, bool &large) {
        BinDesc d{0, 0, 0, smp};
        if (i < nb) {
            const uint64_t s = s_st[i], e = s_st[i + 1];
            d.rec0 = r0 + (uint32_t)(s >> 32);
            d.nrec = (uint32_t)(e >> 32) - (uint32_t)(s >> 32);
            d.nwin = (uint32_t)e - (uint32_t)s;
        }
        small = d.nwin && d.nwin <= kBinCap && d.nrec <= kBinRec;
        large = d.nwin && !small;
        return d;
    };
    if (tid < 2) s_place[tid] = 0;
    __syncthreads();
    uint32_t ns = 0, nl2 = 0;
    for (uint32_t i0 = wave * kWave; i0 < nb; i0 += 1024) {
        bool small, large;
        (void)entry(i0 + lane, small, large);
        ns += (uint32_t)__popcll(__ballot(small));
        nl2 += (uint32_t)__popcll(__ballot(large));
    }
    if (lane == 0) {
        if (ns) atomicAdd(&s_place[0], ns);
        if (nl2) atomicAdd(&s_place[1], nl2);
    }
    __syncthreads();
    if (tid < 2 && s_place[tid]) s_place[tid] = atomicAdd(tid ? &ctl->nbig : &ctl->nbin, s_place[tid]);
    __syncthreads();
    for (uint32_t i0 = wave * kWave; i0 < nb; i0 += 1024) {
        bool small, large;
        const BinDesc d = entry(i0 + lane, small, large);
        const uint64_t ms = __ballot(small), ml = __ballot(large);
        uint32_t at = 0, al = 0;
        if (lane == 0 && ms) at = atomicAdd(&s_place[0], (uint32_t)__popcll(ms));
        if (lane == 0 && ml) al = atomicAdd(&s_place[1], (uint32_t)__popcll(ml));
        at = __shfl(at, 0, kWave);
        al = __shfl(al, 0, kWave);
        if (small) bins[at + (uint32_t)__popcll(ms & lanemask_lt())] = d;
        if (large) {
            const uint32_t q = al + (uint32_t)__popcll(ml & lanemask_lt());
            if (q < big_cap) big[q] = d;
            const unsigned long long groups = (d.nrec + kBigRec - 1) / kBigRec;
            atomicAdd(&ctl->big_win, (unsigned long long)d.nwin);
            atomicAdd(&ctl->big_grp, groups);
            atomicMax(&ctl->big_most, groups);
        }
    }
    __syncthreads();
    if (nb <= 1024) {  // in batches ordered by bin
        uint4 *const s_rec = (uint4 *)s_room;
        uint32_t cur = tid < nb ? r0 + (uint32_t)(s_st[tid] >> 32) : 0u;
        s_n[tid] = 0;
        __syncthreads();
        for (uint32_t q0 = 0; q0 < n; q0 += kBatch) {
            uint4 x[kItems];
            uint32_t at[kItems];  // bin | place in it << 10 (no record: ~0)
#pragma unroll
            for (uint32_t u = 0; u < kItems; u++) x[u] = rec[r0 + min(q0 + u * 1024 + tid, n - 1)];
#pragma unroll
            for (uint32_t u = 0; u < kItems; u++) {
                at[u] = ~0u;
                if (q0 + u * 1024 + tid >= n) continue;
                const uint32_t bi = (uint32_t)s_h[(x[u].y >> 15) & cmask];
                at[u] = bi | (atomicAdd(&s_n[bi], 1u) << 10);
            }
            __syncthreads();
            const uint32_t mine = s_n[tid], inc2 = wave_incl(mine);
            if (lane == kWave - 1) s_wb[wave] = inc2;
            __syncthreads();
            const uint32_t run2 = wave_incl(s_wb[lane % 16]), w = (uint32_t)__builtin_amdgcn_readfirstlane((int)wave);
            const uint32_t first = inc2 - mine + (w ? (uint32_t)__builtin_amdgcn_readlane((int)run2, (int)w - 1) : 0u);
            s_at[tid] = first;
            s_to[tid] = cur - first;
            cur += mine;
            s_n[tid] = 0;
            __syncthreads();
#pragma unroll
            for (uint32_t u = 0; u < kItems; u++) {
                if (at[u] == ~0u) continue;
                const uint32_t bi = at[u] & 1023, p = s_at[bi] + (at[u] >> 10);
                s_rec[p] = x[u];
                s_bin[p] = (uint16_t)bi;
            }
            __syncthreads();
            const uint32_t m = min(kBatch, n - q0);
#pragma unroll
            for (uint32_t u = 0; u < kItems; u++) {
                const uint32_t p = u * 1024 + tid;
                if (p < m) out[s_to[s_bin[p]] + p] = s_rec[p];
            }
            // (the next batch writes s_to, s_rec and s_bin only behind two more barriers)
        }
        return;
    }
    uint32_t *const s_cur = (uint32_t *)s_st;  // word 2 i + 1 of entry i: its first record, counted up
    for (uint32_t i0 = tid; i0 < n; i0 += kU * 1024) {
        uint4 x[kU];
#pragma unroll
        for (int u = 0; u < kU; u++) x[u] = rec[r0 + min(i0 + u * 1024, n - 1)];
#pragma unroll
        for (int u = 0; u < kU; u++)
            if (i0 + u * 1024 < n) {
                const uint32_t bi = (uint32_t)s_h[(x[u].y >> 15) & cmask];
                out[r0 + atomicAdd(&s_cur[2 * bi + 1], 1u)] = x[u];
            }
    }
}

// ---------------------------------------------------------------- runs of a bin
struct BinRuns {
    const uint64_t *packed;
    const uint4 *rec;
    const BinDesc *bins;
    uint32_t nbin;
    int K;
    int T, batch;
    const uint32_t *bounds;   // T + 1 bucket boundaries (plain)
    uint32_t last_lo;         // first bucket of the last segment that holds tuples
    const uint8_t *bad;       // CHECK
    uint8_t *filtered;
    uint32_t *lab_out;        // labels of the runs to join
    uint64_t *st_bits;        // run starts among them (zero before)
    uint64_t out_cap;         // labels that lab_out holds
    uint32_t *wit;            // kBinWit labels per bin (~0: none)
    uint64_t big_work;        // groups that a workgroup of bin_runs_big may visit
    BinCtl *ctl;
};

// windows of staged records, expanded
struct Window {
    uint64_t key;
    uint32_t cls;   // in class | out class << 3 (0-3, 7 'N')
};

// K bases and their neighbours from the 64 staged bases (index 0: the base
// before the record's first window), window o of the record
__device__ __forceinline__ Window expand(uint64_t hi, uint64_t lo, uint32_t o, bool p7, bool n7, int K)
{
    const uint64_t y = (hi << (2 * o)) | ((lo >> 1) >> (63 - 2 * o));
    const uint32_t pc = (uint32_t)(y >> 62);
    const uint64_t F = (y << 2) >> (64 - 2 * K);
    const uint32_t ni = 1 + o + (uint32_t)K;  // 21 .. 62
    const uint32_t nc = (uint32_t)((ni < 32 ? hi : lo) >> (62 - 2 * (ni & 31))) & 3;
    const uint64_t R = revcomp(F, K);
    const bool fwd = F < R;
    Window w;
    w.key = fwd ? F : R;
    // class of a base: bits 1-3 of its letter (A 0, C 1, T 2, G 3); the complement flips bit 1
    const uint32_t cp = p7 ? 7u : pc ^ (pc >> 1), cn = n7 ? 7u : nc ^ (nc >> 1);
    const uint32_t rp = p7 ? 7u : cp ^ 2, rn = n7 ? 7u : cn ^ 2;
    w.cls = fwd ? cn | (cp << 3) : rp | (rn << 3);
    return w;
}

// 64 bases from base b - 1 of the 2-bit stream (b = 0: an A before the first)
__device__ __forceinline__ void bases64(const uint64_t *__restrict__ packed, uint64_t b, uint64_t &hi, uint64_t &lo)
{
    const uint64_t s = b ? b - 1 : 0, i = s >> 5;
    const uint32_t o = 2 * (uint32_t)(s & 31);
    const uint64_t w0 = packed[i], w1 = packed[i + 1], w2 = packed[i + 2];
    hi = (w0 << o) | ((w1 >> 1) >> (63 - o));
    lo = (w1 << o) | ((w2 >> 1) >> (63 - o));
    if (b == 0) {
        lo = (lo >> 2) | (hi << 62);
        hi >>= 2;
    }
}

// multiply-add hash of a key's 24-bit pieces (24-bit products run at the full
// rate, 32-bit ones at a quarter of it); its top bits are the good ones
__device__ __forceinline__ uint32_t key_hash(uint64_t k)
{
    const uint32_t a = (uint32_t)k, b = (uint32_t)(k >> 24), c = (uint32_t)(k >> 48);
    return __umul24(a & 0xFFFFFF, 0xD1B54B) + __umul24(b & 0xFFFFFF, 0x9E3779) + __umul24(c, 0xB5297A5 & 0xFFFFFF);
}

constexpr uint64_t kNoKey = ~0ull;  // k <= 31: no k-mer

// slot of key in the table of kBinCap slots (linear probing from its hash);
// fresh: this lane put it there
__device__ __forceinline__ uint32_t table_slot(unsigned long long *tab, uint64_t key, uint32_t hash, bool &fresh)
{
    uint32_t s = hash >> 20;
    fresh = false;
    for (;;) {
        unsigned long long cur = __hip_atomic_load(&tab[s], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        if (cur == key) return s;
        if (cur == kNoKey) {
            cur = atomicCAS(&tab[s], kNoKey, (unsigned long long)key);
            if (cur == kNoKey) {
                fresh = true;
                return s;
            }
            if (cur == key) return s;
        }
        s = (s + 1) & (kBinCap - 1);
    }
}
static_assert(kBinCap == 4096, "12-bit slots");

// 1 + the last k-mer of the segment that key lies in
__device__ __forceinline__ uint64_t last_of(const BinRuns &P, uint64_t key, uint32_t smp)
{
    int t = 0;
    if (P.batch) t = (int)smp;
    else if (P.T > 1) t = last_le(P.bounds, P.T, (uint32_t)(key >> (2 * P.K - 20)));
    return P.ctl->kmax1[t];
}

// the filter's verdict on a run whose side `tl` branches (the other does not):
// the largest class (the lowest on ties) and whether the second largest count
// exceeds 0.2 of the run's length as the reference computes it in float
// (metapart.c:2356-2359, 2419): the rounded quotient exceeds 0.2 exactly when
// second * 2^27 > 26843545 * len (both below 2^24)
__device__ __forceinline__ void side_verdict(const uint32_t tl[4], uint32_t len, uint32_t &arg, bool &ratio)
{
    uint64_t b1 = 0, b2 = 0;
#pragma unroll
    for (int c = 0; c < 4; c++) {
        const uint64_t v = ((uint64_t)tl[c] << 2) | (uint32_t)(3 - c);
        b2 = max(b2, min(b1, v));
        b1 = max(b1, v);
    }
    arg = 3 - (uint32_t)(b1 & 3);
    const uint64_t second = b2 >> 2;
    ratio = len < (1u << 24) ? (second << 27) > 26843545ull * len
                             : (double)__fdiv_rn((float)(int)second, (float)(int)len) > 0.2;
}

// a side's tallies by 2-bit code, as bin_runs keeps them (the in side's codes are the complement's), in the
// order of the classes and back: class of a base is code ^ code >> 1, and the complement flips its bit 1
__device__ __forceinline__ void code_verdict(const uint32_t t[4], bool out, uint32_t len, uint32_t &arg, bool &ratio)
{
    const uint32_t a = t[0], b = t[1], c = t[2], d = t[3];
    const uint32_t tl[4] = {out ? a : d, out ? b : c, out ? d : a, out ? c : b};
    uint32_t cls;
    side_verdict(tl, len, cls, ratio);
    arg = out ? cls ^ (cls >> 1) : (0x4Bu >> (2 * cls)) & 3;  // 3, 2, 0, 1
}

// meta word of a slot, first the tallies ...
constexpr uint32_t kCntMask = 0xFFFF;  // tuples; 16 + c: in class c seen, 24 + c: out class c (7, 'N', is not counted)
// ... then the run's verdict: place of its labels (13 bits) and
constexpr uint32_t kRunJoin = 1u << 13, kRunSide = 1u << 14, kRunOut = 1u << 15, kRunWit = 1u << 31, kRunRatio = 1u << 28;
constexpr uint32_t kRunLast = kRunRatio;  // CHECK: the last run of the last segment
// kRunSide: one side branches (kRunOut: the out side), its tallies' number in 16-27, then kRunRatio and its
// largest class in 29-30

constexpr uint32_t kFoundOther = 1, kFoundLast = 2;  // BinCtl::found

// the lanes' f or'ed into *flag, where it is not seen there already
__device__ __forceinline__ void note_found(uint32_t f, uint32_t *flag)
{
    const uint32_t all = (__ballot(f & kFoundOther) ? kFoundOther : 0u) | (__ballot(f & kFoundLast) ? kFoundLast : 0u);
    if (all && __lane_id() == 0 && (all & ~*flag)) atomicOr(flag, all);
}

// LDS of bin_runs: the staged records are dead once every window is expanded
// into registers, so the table takes their place; its keys are dead once the
// runs are evaluated, and make room for the labels and the side tallies.
// A staged record: 64 bases from three before its first window, their reverse
// complement from 31 - K bases on with its words in reverse order, its label.
// Window o's base before it and its K bases are then two 32-bit funnel shifts
// by -2 o - 4 of three words from the word that bit 5 of 2 o + 2 names on, and
// its reverse strand's the same of the second sequence by 2 o + 2.
struct RunsRow {
    uint32_t fw[4], rc[4], lab;
};
struct RunsStage {
    RunsRow row[kBinRec];
    uint32_t map[kBinCap];  // window: its row's byte offset | 2 + 2 x its place in the record << 16 | 'N' flags
};
static_assert(sizeof(RunsRow) * kBinRec <= 0x10000, "16-bit offsets");
// a window's flags: no base before it or after it.  Bits 24 and 27 (in side, out side) where its strand is the
// canonical one, 28 and 31 where the other is: the sides change places
constexpr uint32_t kMapPrevN = (1u << 27) | (1u << 28), kMapNextN = (1u << 24) | (1u << 31);
struct RunsTable {
    unsigned long long key[kBinCap];
    uint32_t gap[kBinCap];      // (the tallies' end)
    uint32_t meta[kBinCap];
};
union RunsLds {
    RunsStage st;
    RunsTable tb;
    struct {
        uint32_t lab[kBinCap];      // labels in run order
        uint32_t tal[2 * kBinCap];  // 4 tallies of every branching side (a run of two tuples at the least)
    } out;
};

// Bound by vector instructions (83 % of the cycles): about 280 per 64 windows,
// against 380 with the windows' places found by bit scans and a probe loop per
// window, and 300 with 64-bit shifts per window (1.44e9 windows, k = 31: 16.9
// -> 12.6 ms; 512 lanes of 8 windows: 18.6).  4096 windows, a lane for 4, is
// what two workgroups per CU and 64 registers hold.
// CHECK: only note which live labels there are (the first-run quirk's test).
// PART: the scan holds part of the buckets; only the records' windows in them
// are laid out (4 scans of 2 M reads of 150 bases: 6.8 -> 3.4 ms against
// expanding all of them).
template <bool CHECK, bool PART>
__global__ __launch_bounds__(kRunThreads, 8) void bin_runs_kernel(BinRuns P)
{
    constexpr int kPer = kBinCap / kRunThreads;  // windows a lane, distinct k-mers a lane at most
    constexpr int kWaves = kRunThreads / kWave;
    __shared__ __align__(16) RunsLds U;
    __shared__ uint16_t s_list[kBinCap];               // slots in use
    __shared__ unsigned long long s_ob[kBinCap / 64];  // run starts among the labels
    __shared__ uint32_t s_sum[kWaves], s_nkey, s_red[2];
    __shared__ uint64_t s_out;
    const uint32_t tid = threadIdx.x, lane = tid % kWave, wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const BinDesc d = P.bins[blockIdx.x];
    const int K = P.K;
    static_assert(kBinRec <= kRunThreads, "a record a lane");
    const bool have = tid < d.nrec;
    uint4 rc = make_uint4(0u, 0u, 0u, 0u);
    uint64_t fh = 0, fl = 0;
    if (have) {
        rc = P.rec[d.rec0 + tid];
        bases64(P.packed, (((uint64_t)rc.y << 32) | rc.x) & ((1ull << 40) - 1), fh, fl);
    }
    const uint32_t L = (rc.y >> 8) & 31;  // 0 past the records
    const uint32_t nl = PART ? (uint32_t)__popc(rc.w) : L;
    const uint32_t inc = wave_incl(nl);
    if (lane == kWave - 1) s_sum[wave] = inc;
    if (tid < kBinCap / 64) s_ob[tid] = 0;
    if (tid < 2) s_red[tid] = 0;
    if (tid == 0) s_nkey = 0;
    __syncthreads();
    uint32_t o = inc - nl;
    if (wave > 0 && wave * kWave < d.nrec)  // lane w of the sum: windows of the waves up to w
        o += (uint32_t)__builtin_amdgcn_readlane((int)wave_incl(s_sum[lane % kWaves]), (int)wave - 1);
    if (have) {  // the records' windows laid end to end
        RunsRow &row = U.st.row[tid];
        const uint64_t rh = revcomp(fl, 32), rl = revcomp(fh, 32);
        const int sh = 2 * (31 - K);  // 0 .. 22
        const uint64_t a = fh >> 4, b = (fh << 60) | (fl >> 4), c = (rh << sh) | ((rl >> 1) >> (63 - sh)), e = rl << sh;
        row.fw[0] = (uint32_t)(a >> 32);
        row.fw[1] = (uint32_t)a;
        row.fw[2] = (uint32_t)(b >> 32);
        row.fw[3] = (uint32_t)b;
        row.rc[3] = (uint32_t)(c >> 32);
        row.rc[2] = (uint32_t)c;
        row.rc[1] = (uint32_t)(e >> 32);
        row.rc[0] = (uint32_t)e;
        row.lab = rc.z;
        const uint32_t f = (rc.y >> 13) & 3, at = tid * (uint32_t)sizeof(RunsRow);
        const uint32_t pn = (f & kPrevN) ? kMapPrevN : 0u, nn = (f & kNextN) ? kMapNextN : 0u;
        if constexpr (PART) {
            for (uint32_t m = rc.w << ((32 - L) & 31); m;) {
                const uint32_t q = (uint32_t)__builtin_clz(m);
                m &= ~(0x80000000u >> q);
                U.st.map[o++] = at | ((q + 1) << 17) | (q == 0 ? pn : 0u) | (q + 1 == L ? nn : 0u);
            }
        } else {
            uint32_t e = at | (2u << 16) | pn;
            for (uint32_t q = 0; q + 1 < L; q++) {
                U.st.map[o + q] = e;
                e = (e & 0x3FFFFF) + (2u << 16);
            }
            U.st.map[o + L - 1] = e | nn;
        }
    }
    __syncthreads();
    // every window's k-mer (from bit 61 down), neighbour codes and label
    uint64_t key[kPer];
    uint32_t lab[kPer], st[kPer];  // st: slot | place in its run << 12 | codes << 24
    bool tup[kPer];                // a window there
    const int kz = 62 - 2 * K;     // zero bits below a key
    const uint64_t kmask = (~0ull >> 2) >> kz << kz;
#pragma unroll
    for (int i = 0; i < kPer; i++) {
        const uint32_t j = i * kRunThreads + tid;
        tup[i] = j < d.nwin;
        if (tup[i]) {
            const uint32_t m = U.st.map[j], zs = m >> 16, ys = 0u - 2 - zs;  // (a shift takes the low five bits)
            const uint32_t *const row = (const uint32_t *)((const char *)&U.st + (m & 0xFFFF));
            const uint32_t *const yw = row + ((m >> 21) & 1);
            const uint32_t *const zw = yw + 4;
            lab[i] = row[8];
            const uint32_t y1 = yw[1], z1 = zw[1];
            const uint32_t yh = __builtin_amdgcn_alignbit(yw[0], y1, ys), yl = __builtin_amdgcn_alignbit(y1, yw[2], ys);
            const uint32_t zh = __builtin_amdgcn_alignbit(zw[2], z1, zs), zl = __builtin_amdgcn_alignbit(z1, zw[0], zs);
            // y: base before, K bases ...; z: complement of the base after, reverse complement of the K bases ...
            const uint64_t F = (((uint64_t)yh << 32) | yl) & kmask, R = (((uint64_t)zh << 32) | zl) & kmask;
            const bool fwd = F < R;
            key[i] = fwd ? F : R;
            const uint32_t u = (fwd ? zh : yh) >> 30, v = ((fwd ? yh : zh) >> 27) & 0x18;
            st[i] = ((u | v | ((m >> (fwd ? 22 : 26)) & 0x24)) << 24) | (key_hash(key[i]) >> 20);
        }
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < kPer; q++) {
        U.tb.key[q * kRunThreads + tid] = kNoKey;
        U.tb.meta[q * kRunThreads + tid] = 0;
    }
    __syncthreads();
    // into the table: the first probes of a lane's windows together, then the
    // ones that met another k-mer (a lane's next unsettled window per step, so
    // that a wave takes the longest sum over a lane's windows, not the sum of
    // its longest probes)
    uint32_t open = 0, fresh = 0;
#pragma unroll
    for (int i = 0; i < kPer; i++) {
        if (!tup[i]) continue;
        const uint64_t old = atomicCAS(&U.tb.key[st[i] & 0xFFF], kNoKey, (unsigned long long)key[i]);
        if (old == kNoKey) fresh |= 1u << i;
        else if (old != key[i]) open |= 1u << i;
    }
    while (__any(open != 0)) {
        if (open) {
            const uint32_t i = (uint32_t)__builtin_ctz(open);
            uint64_t k = key[0];
            uint32_t s = st[0];
#pragma unroll
            for (int q = 1; q < kPer; q++) {
                k = i == (uint32_t)q ? key[q] : k;
                s = i == (uint32_t)q ? st[q] : s;
            }
            const uint32_t n = (s + 1) & 0xFFF;
            const uint64_t old = atomicCAS(&U.tb.key[n], kNoKey, (unsigned long long)k);
            s = (s & ~0xFFFu) | n;
#pragma unroll
            for (int q = 0; q < kPer; q++) st[q] = i == (uint32_t)q ? s : st[q];
            if (old == kNoKey) fresh |= 1u << i;
            if (old == kNoKey || old == k) open &= open - 1;
        }
    }
    // counts, places and classes seen; the slots taken first to the list
    {
        const uint32_t nf = (uint32_t)__popc(fresh), fi = wave_incl(nf);
        uint32_t at = 0;
        if (lane == kWave - 1) at = atomicAdd(&s_nkey, fi);
        at = __shfl(at, kWave - 1, kWave) + fi - nf;
        uint32_t old[kPer];
#pragma unroll
        for (int i = 0; i < kPer; i++)
            if (tup[i]) old[i] = atomicAdd(&U.tb.meta[st[i] & 0xFFF], 1u);
#pragma unroll
        for (int i = 0; i < kPer; i++) {
            if (!tup[i]) continue;
            const uint32_t s = st[i] & 0xFFF;
            const uint32_t seen = (1u << (16 + ((st[i] >> 24) & 7))) | (1u << (24 + (st[i] >> 27)));
            if (seen & ~old[i]) atomicOr(&U.tb.meta[s], seen);
            if ((fresh >> i) & 1) s_list[at++] = (uint16_t)s;
            st[i] |= (old[i] & 0xFFF) << 12;
        }
    }
    __syncthreads();
    // every run: evaluated unless it is its segment's last
    const uint32_t nkey = s_nkey;
    uint32_t cnt[kPer], run[kPer], at[kPer];  // tuples; verdict; slot
    uint32_t add = 0, nz = 0, nlast = 0;
    const bool one = P.T == 1 || P.batch;
    const uint64_t lk = one ? P.ctl->kmax1[d.smp] : 0, last = lk ? (lk - 1) << kz : kNoKey;
    const uint64_t wit = max((uint64_t)P.last_lo << 42, (uint64_t)1);  // witnesses: from the last segment on, not k-mer 0
#pragma unroll
    for (int q = 0; q < kPer; q++) {
        cnt[q] = run[q] = at[q] = 0;
        if (q * kRunThreads >= nkey) continue;  // uniform
        const uint32_t x = q * kRunThreads + tid;
        if (x >= nkey) continue;
        const uint32_t s = s_list[x], m = U.tb.meta[s], c = m & kCntMask;
        const uint64_t k = U.tb.key[s];
        at[q] = s;
        cnt[q] = c;
        const bool is_last = one ? k == last : (k >> kz) + 1 == last_of(P, k >> kz, d.smp);
        const uint32_t mc = (m >> 16) & 0x0F0F, m2 = mc & ((mc | 0x1010) - 0x0101);
        const bool bi = m2 & 0xFF, bo = m2 >> 8;  // more than one class (the | keeps an empty side from borrowing)
        nlast += is_last;
        const bool zero = !is_last && bi && bo;
        nz += zero;
        uint32_t v = 0;
        if (!zero) {
            if (c >= 2 && k != 0) v |= kRunJoin;
            if (!is_last && (bi || bo)) v |= kRunSide | (bo ? kRunOut : 0u);
            if (k >= wit) v |= !is_last ? kRunWit : CHECK ? kRunLast : 0u;
        }
        run[q] = v;
        add += ((v & kRunJoin) ? c : 0u) | ((v & kRunSide) ? 1u << 16 : 0u);
    }
    const uint32_t ainc = wave_incl(add);
    if (lane == kWave - 1) s_sum[wave] = ainc;
    __syncthreads();  // also: every lane has read the keys
    uint32_t base = ainc - add, tot = 0;
#pragma unroll
    for (uint32_t w = 0; w < kWaves; w++) {
        if (w < wave) base += s_sum[w];
        tot += s_sum[w];
    }
    const uint32_t nout = tot & 0xFFFF, nside = tot >> 16, npad = (nout + 63) & ~63u;
    if (!CHECK && tid == 0) {
        s_out = npad ? atomicAdd(&P.ctl->out, (unsigned long long)npad) : 0;
        if (s_out + npad > P.out_cap) atomicOr(&P.ctl->err, 8u);
    }
#pragma unroll
    for (int q = 0; q < kPer; q++) {
        if (!cnt[q]) continue;
        uint32_t v = run[q];
        if (v & kRunJoin) {
            const uint32_t p = base & 0xFFFF;
            v |= p;
            if (!CHECK) atomicOr(&s_ob[p >> 6], 1ull << (p & 63));
            base += cnt[q];
        }
        if (v & kRunSide) {
            v |= (base >> 16) << 16;
            if (!CHECK) {  // the list's slots are in registers: the sides' slots and lengths take its place
                s_list[base >> 16] = (uint16_t)at[q];
                s_list[kBinCap / 2 + (base >> 16)] = (uint16_t)cnt[q];
            }
            base += 1u << 16;
        }
        U.tb.meta[at[q]] = v;
    }
    if (!CHECK)
        for (uint32_t j = tid; j < 4 * nside; j += kRunThreads) U.out.tal[j] = 0;
    __syncthreads();
    if constexpr (CHECK) {
        uint32_t f = 0;
#pragma unroll
        for (int i = 0; i < kPer; i++) {
            if (!tup[i]) continue;
            const uint32_t v = U.tb.meta[st[i] & 0xFFF];
            if ((v & (kRunWit | kRunLast)) && !P.bad[lab[i]]) f |= v & kRunWit ? kFoundOther : kFoundLast;
        }
        note_found(f, &P.ctl->found[P.batch ? d.smp : 0]);
        return;
    }
    uint32_t ver[kPer];
#pragma unroll
    for (int i = 0; i < kPer; i++) {
        ver[i] = 0;
        if (!tup[i]) continue;
        const uint32_t v = U.tb.meta[st[i] & 0xFFF];
        ver[i] = v;
        if (v & kRunJoin) U.out.lab[(v & 0x1FFF) + ((st[i] >> 12) & 0xFFF)] = lab[i];
        if (v & kRunSide) {
            const uint32_t c = (st[i] >> ((v & kRunOut) ? 27 : 24)) & 7;
            if (c < 4) atomicAdd(&U.out.tal[4 * ((v >> 16) & 0xFFF) + c], 1u);
        }
        if (i == 0 && wave < kBinWit) {
            const uint64_t wm = __ballot((v & kRunWit) != 0);
            if (wm && (wm & lanemask_lt()) == 0 && (v & kRunWit)) P.wit[blockIdx.x * kBinWit + wave] = lab[i];
        }
    }
    if (nside) {
        __syncthreads();
        for (uint32_t h = tid; h < nside; h += kRunThreads) {
            const uint32_t sl = s_list[h];
            const uint32_t v = U.tb.meta[sl];
            uint32_t arg;
            bool ratio;
            code_verdict(&U.out.tal[4 * h], (v & kRunOut) != 0, s_list[kBinCap / 2 + h], arg, ratio);
            U.tb.meta[sl] = v | (ratio ? kRunRatio : 0u) | (arg << 29);
        }
    }
    __syncthreads();
    if (nside) {
#pragma unroll
        for (int i = 0; i < kPer; i++) {
            if (!(ver[i] & kRunSide)) continue;
            const uint32_t v = U.tb.meta[st[i] & 0xFFF];
            const uint32_t c = (st[i] >> ((v & kRunOut) ? 27 : 24)) & 7;
            if ((v & kRunRatio) || c != ((v >> 29) & 3)) P.filtered[lab[i]] = 1;
        }
    }
    const uint64_t ob = s_out;
    const bool room = ob + npad <= P.out_cap;
    if (room)
        for (uint32_t j = tid; j < npad; j += kRunThreads) P.lab_out[ob + j] = j < nout ? U.out.lab[j] : 0u;
    if (room && tid * 64 < npad) {
        uint64_t m = s_ob[tid];
        if (tid * 64 + 64 > nout) m |= ~0ull << (nout & 63);  // the padding: runs of one
        P.st_bits[ob / 64 + tid] = m;
    }
    const uint64_t zm = __ballot(nz != 0);
    if (zm) {
        for (int o = kWave / 2; o > 0; o >>= 1) nz += __shfl_down(nz, o, kWave);
        if (lane == 0) atomicAdd(&s_red[1], nz);
    }
    if (nlast) atomicSub(&s_red[0], nlast);
    __syncthreads();
    if (tid < 2) {
        const uint32_t v = s_red[tid] + (tid == 0 ? nkey : 0u);
        if (v) atomicAdd(&P.ctl->stat[blockIdx.x % kStripes][tid], (unsigned long long)v);
    }
}

// A bin past the table.  Its windows go by once to count, once to place the
// labels and tally the branching sides and once to mark (records expanded again
// each time, kBigRec at once), whole where its distinct k-mers fit the table, as
// in a pile of few k-mers however deep, else in parts by the top bits of the
// k-mer's hash, a part split again when its k-mers overfill the table.
// A bin of many k-mers is visited once per part, which grows with its square:
// at the first overfull table the groups still to come are reckoned from the
// k-mers seen so far, and where they would pass P.big_work, or once a workgroup
// has visited so many, the scan goes by radix passes instead.
// PART: a record's windows in the bucket range alone are expanded.
constexpr int kBigThreads = 1024;
constexpr uint32_t kBigKeys = 2048;   // k-mers of a part; a group of records adds at most 64 x 31, which still fit
constexpr uint32_t kBigPart = kBigKeys * 3 / 4;  // and on average
constexpr int kBigDepth = 24;
constexpr int kBigGrid = 256;         // workgroups, one a CU; each takes the next bin
// What bin_runs_big may take is what the radix path does: a window of 25e6 in a
// ms, and of those in large bins, whose k-mers of thousands of copies it sorts
// group by group and evaluates by one lane, 200e3 at the most (measured 44e3
// where 40 k reads are of one 500 bp genome, 15e3 for 100 k of 5 kb, 117e3 where
// 2 % of 60 k reads are poly-G, 171e3 for 40 k amplicons with 200 pairs of
// flanks).  A visit of a group takes 2.0 to 2.7 us.  Against radix passes
// these take 93 -> 3.7, 803 -> 0.8 and 41 -> 1.2 ms; the amplicons (the table overfull
// at once) go on to the radix path after 0.3.
constexpr double kBigGroupMs = 0.0025;
constexpr double kRadixWin = 25e6, kRadixDeep = 200e3;
static_assert(kBigKeys + kBigRec * kMaxRun < kBinCap, "the table never fills");

template <bool CHECK, bool PART>
__global__ __launch_bounds__(kBigThreads) void bin_runs_big_kernel(BinRuns P)
{
    constexpr int kPer = kBinCap / kBigThreads;
    constexpr int kWaves = kBigThreads / kWave;
    __shared__ unsigned long long s_key[kBinCap];
    __shared__ uint32_t s_cnt[kBinCap], s_meta[kBinCap], s_base[kBinCap];
    __shared__ uint32_t s_tal[kBigKeys + kBigRec * kMaxRun][4];
    __shared__ ulonglong2 s_seq[kBigRec];
    __shared__ uint32_t s_lab[kBigRec], s_fl[kBigRec];
    __shared__ uint16_t s_map[kBigRec * kMaxRun];  // window: its record | its place in it << 6
    __shared__ uint32_t s_nwin, s_nkey, s_bin, s_stop, s_sumc[kWaves], s_sums[kWaves], s_red[2];
    __shared__ uint64_t s_out;
    const uint32_t tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
    const int K = P.K;
    uint64_t work = 0;  // groups visited
    for (;;) {
        __syncthreads();
        if (tid == 0) s_bin = atomicAdd(&P.ctl->next[CHECK ? 1 : 0], 1u);
        __syncthreads();
        const uint32_t bin = s_bin;
        if (bin >= P.nbin) break;
        const BinDesc d = P.bins[bin];
        if (tid < 2) s_red[tid] = 0;
        // the windows of records [g, g + kBigRec) of the part, fn(window, label, hash) per lane
        auto group = [&](uint32_t g, auto fn) {
            __syncthreads();
            const uint32_t nr = min((uint32_t)kBigRec, d.nrec - g);
            if (tid < kBigRec) {  // one wave
                uint32_t m = 0;  // its windows to expand, the first at bit 31
                if (tid < nr) {
                    const uint4 rc = P.rec[d.rec0 + g + tid];
                    uint64_t hi, lo;
                    bases64(P.packed, (((uint64_t)rc.y << 32) | rc.x) & ((1ull << 40) - 1), hi, lo);
                    const uint32_t L = (rc.y >> 8) & 31;
                    s_seq[tid] = make_ulonglong2(hi, lo);
                    s_lab[tid] = rc.z;
                    s_fl[tid] = ((rc.y >> 13) & 3) | (L << 2);
                    m = (PART ? rc.w : ~0u) << (32 - L);
                }
                const uint32_t n = (uint32_t)__popc(m), i = wave_incl(n);
                if (tid == kBigRec - 1) s_nwin = i;
                for (uint32_t o = i - n; m; o++) {
                    const uint32_t q = (uint32_t)__builtin_clz(m);
                    m &= ~(0x80000000u >> q);
                    s_map[o] = (uint16_t)(tid | (q << 6));
                }
            }
            __syncthreads();
            const uint32_t nw = s_nwin;
            for (uint32_t j = tid; j < nw; j += kBigThreads) {
                const uint32_t e = s_map[j], r = e & 63, o = e >> 6, fl = s_fl[r];
                const ulonglong2 sq = s_seq[r];
                const Window x = expand(sq.x, sq.y, o, o == 0 && (fl & kPrevN), o + 1 == fl >> 2 && (fl & kNextN), K);
                fn(x, s_lab[r], key_hash(x.key));
            }
            work++;
        };
        int depth = 0;
        uint32_t part = 0;
        for (;;) {
            auto mine = [&](uint32_t h) { return depth == 0 || (h * 0x9E3779B1u) >> (32 - depth) == part; };
            __syncthreads();
#pragma unroll
            for (int q = 0; q < kPer; q++) {
                s_key[q * kBigThreads + tid] = kNoKey;
                s_cnt[q * kBigThreads + tid] = 0;
                s_meta[q * kBigThreads + tid] = 0;
            }
            if (tid == 0) {
                s_nkey = 0;
                s_stop = ld_agent(&P.ctl->err);  // another workgroup gave up
            }
            uint32_t seen_grp = 0;  // groups up to the one that overfilled the table
            for (uint32_t g = 0; g < d.nrec; g += kBigRec) {
                group(g, [&](const Window &x, uint32_t, uint32_t h) {
                    if (!mine(h)) return;
                    bool fresh;
                    const uint32_t s = table_slot(s_key, x.key, h, fresh);
                    if (fresh) atomicAdd(&s_nkey, 1u);
                    const uint32_t ci = x.cls & 7, co = x.cls >> 3;
                    const uint32_t seen = (ci < 4 ? 1u << ci : 0u) | (co < 4 ? 16u << co : 0u);
                    atomicAdd(&s_cnt[s], 1u);
                    if (seen & ~__hip_atomic_load(&s_meta[s], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP))
                        atomicOr(&s_meta[s], seen);
                });
                __syncthreads();
                // uniform: s_stop is written before the part's first barrier, s_nkey next behind another
                if (s_stop) return;
                if (s_nkey > kBigKeys) {
                    seen_grp = g / kBigRec + 1;
                    break;
                }
                if (work > P.big_work) break;
            }
            uint64_t todo = work;
            if (seen_grp && depth == 0) {  // parts by the k-mers seen per group, three visits of all groups each
                const uint64_t all = (d.nrec + kBigRec - 1) / kBigRec;
                todo += all * 3 * ((uint64_t)s_nkey * all / ((uint64_t)seen_grp * kBigPart) + 1);
            }
            if (todo > P.big_work) {  // uniform
                if (tid == 0) atomicOr(&P.ctl->err, 16u);
                return;
            }
            if (seen_grp) {
                if (depth == kBigDepth) {  // one hash value holds too many k-mers: the radix path
                    if (tid == 0) atomicOr(&P.ctl->err, 4u);
                    return;
                }
                depth++;
                part <<= 1;
                continue;
            }
            // verdicts and places
            uint32_t cnt[kPer], run[kPer], addc = 0, adds = 0, nev = 0, nz = 0;
#pragma unroll
            for (int q = 0; q < kPer; q++) {
                const uint32_t s = q * kBigThreads + tid;
                cnt[q] = s_cnt[s];
                run[q] = 0;
                if (!cnt[q]) continue;
                const uint64_t key = s_key[s];
                const uint32_t m = s_meta[s];
                const bool is_last = key + 1 == last_of(P, key, d.smp);
                const bool bi = __popc(m & 15) > 1, bo = __popc((m >> 4) & 15) > 1;
                nev += !is_last;
                const bool zero = !is_last && bi && bo;
                nz += zero;
                uint32_t v = 0;
                if (!zero) {
                    if (cnt[q] >= 2 && key != 0) v |= kRunJoin;
                    if (!is_last && (bi || bo)) v |= kRunSide | (bo ? kRunOut : 0u);
                    if (key != 0 && (uint32_t)(key >> (2 * K - 20)) >= P.last_lo)
                        v |= !is_last ? kRunWit : CHECK ? kRunLast : 0u;
                }
                run[q] = v;
                if (v & kRunJoin) addc += cnt[q];
                if (v & kRunSide) adds++;
            }
            const uint32_t ic = wave_incl(addc), is = wave_incl(adds);
            if (lane == kWave - 1) {
                s_sumc[wave] = ic;
                s_sums[wave] = is;
            }
            __syncthreads();
            uint32_t bc = ic - addc, bs = is - adds, nout = 0, nside = 0;
            for (uint32_t w = 0; w < kWaves; w++) {
                if (w < wave) {
                    bc += s_sumc[w];
                    bs += s_sums[w];
                }
                nout += s_sumc[w];
                nside += s_sums[w];
            }
            if (!CHECK && tid == 0) s_out = atomicAdd(&P.ctl->out, (unsigned long long)((nout + 63) & ~63u));
            __syncthreads();
            const uint64_t ob = CHECK ? 0 : s_out;
            if (!CHECK && ob + ((nout + 63) & ~63u) > P.out_cap) {  // uniform
                if (tid == 0) atomicOr(&P.ctl->err, 8u);
                return;
            }
#pragma unroll
            for (int q = 0; q < kPer; q++) {
                if (!cnt[q]) continue;
                const uint32_t s = q * kBigThreads + tid;
                if (run[q] & kRunJoin) {
                    s_base[s] = bc;
                    if (!CHECK)
                        atomicOr((unsigned long long *)&P.st_bits[(ob + bc) >> 6], 1ull << ((ob + bc) & 63));
                    bc += cnt[q];
                }
                if (run[q] & kRunSide) {
                    run[q] |= bs << 16;
#pragma unroll
                    for (int c = 0; c < 4; c++) s_tal[bs][c] = 0;
                    bs++;
                }
                s_cnt[s] = 0;
                s_meta[s] = run[q];
            }
            if (!CHECK && tid < 64 && (nout & 63) && tid >= (nout & 63)) {  // the padding: runs of one
                const uint64_t p = ob + (nout & ~63u) + tid;
                P.lab_out[p] = 0;
                atomicOr((unsigned long long *)&P.st_bits[p >> 6], 1ull << (p & 63));
            }
            if constexpr (CHECK) {
                uint32_t f = 0;
                for (uint32_t g = 0; g < d.nrec; g += kBigRec)
                    group(g, [&](const Window &x, uint32_t lab, uint32_t h) {
                        if (!mine(h)) return;
                        bool fresh;
                        const uint32_t v = s_meta[table_slot(s_key, x.key, h, fresh)];
                        if ((v & (kRunWit | kRunLast)) && !P.bad[lab]) f |= v & kRunWit ? kFoundOther : kFoundLast;
                    });
                note_found(f, &P.ctl->found[P.batch ? d.smp : 0]);
            } else {
                for (uint32_t g = 0; g < d.nrec; g += kBigRec)
                    group(g, [&](const Window &x, uint32_t lab, uint32_t h) {
                        if (!mine(h)) return;
                        bool fresh;
                        const uint32_t s = table_slot(s_key, x.key, h, fresh), v = s_meta[s];
                        if (v & kRunJoin) P.lab_out[ob + s_base[s] + atomicAdd(&s_cnt[s], 1u)] = lab;
                        if (v & kRunSide) {
                            const uint32_t c = (x.cls >> ((v & kRunOut) ? 3 : 0)) & 7;
                            if (c < 4) atomicAdd(&s_tal[(v >> 16) & 0xFFF][c], 1u);
                        }
                        if ((v & kRunWit) && wave < kBinWit) P.wit[bin * kBinWit + wave] = lab;
                    });
                __syncthreads();
                if (nside) {
#pragma unroll
                    for (int q = 0; q < kPer; q++) {
                        if (!(run[q] & kRunSide)) continue;
                        const uint32_t h = (run[q] >> 16) & 0xFFF;
                        const uint32_t tl[4] = {s_tal[h][0], s_tal[h][1], s_tal[h][2], s_tal[h][3]};
                        uint32_t arg;
                        bool ratio;
                        side_verdict(tl, cnt[q], arg, ratio);
                        s_meta[q * kBigThreads + tid] = run[q] | (ratio ? kRunRatio : 0u) | (arg << 29);
                    }
                    for (uint32_t g = 0; g < d.nrec; g += kBigRec)
                        group(g, [&](const Window &x, uint32_t lab, uint32_t h) {
                            if (!mine(h)) return;
                            bool fresh;
                            const uint32_t v = s_meta[table_slot(s_key, x.key, h, fresh)];
                            if (!(v & kRunSide)) return;
                            const uint32_t c = (x.cls >> ((v & kRunOut) ? 3 : 0)) & 7;
                            if ((v & kRunRatio) || c != ((v >> 29) & 3)) P.filtered[lab] = 1;
                        });
                }
                for (int o = kWave / 2; o > 0; o >>= 1) {
                    nev += __shfl_down(nev, o, kWave);
                    nz += __shfl_down(nz, o, kWave);
                }
                if (lane == 0) {
                    atomicAdd(&s_red[0], nev);
                    atomicAdd(&s_red[1], nz);
                }
                __syncthreads();
                if (tid < 2) {
                    if (s_red[tid])
                        atomicAdd(&P.ctl->stat[bin % kStripes][tid], (unsigned long long)s_red[tid]);
                    s_red[tid] = 0;
                }
            }
            // the next part: up from every right half, then the right sibling
            while (depth && (part & 1)) {
                part >>= 1;
                depth--;
            }
            if (!depth) break;
            part |= 1;
        }
    }
}

// found[sample] where a witness's label lives; one flag write per wave, and
// none where the flag is seen set (thousands of accesses to one word serialise)
__global__ __launch_bounds__(256) void bin_witness_kernel(const uint32_t *__restrict__ wit, const BinDesc *__restrict__ bins,
                                                          uint64_t n, int batch, const uint8_t *__restrict__ bad, BinCtl *ctl)
{
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t l = i < n ? wit[i] : ~0u;
    const bool live = l != ~0u && !bad[l];
    const uint32_t s = live && batch ? bins[i / kBinWit].smp : 0u;
    uint64_t m = __ballot(live);
    while (m) {
        const int f = __builtin_ctzll(m);
        const uint32_t s0 = __shfl(s, f, kWave);
        if ((int)__lane_id() == f && !ctl->found[s0]) atomicOr(&ctl->found[s0], kFoundOther);
        m &= ~__ballot(live && s == s0);
    }
}

// reads that the filter left alive, per sample
__global__ __launch_bounds__(256) void bin_alive_kernel(const uint8_t *__restrict__ bad, const uint64_t *__restrict__ first,
                                                        int ns, uint64_t N, unsigned long long *__restrict__ alive)
{
    __shared__ uint32_t s_n[kMaxSeg];
    __shared__ uint64_t s_first[kMaxSeg + 1];
    for (int j = threadIdx.x; j <= ns; j += 256) s_first[j] = first[j];
    for (int j = threadIdx.x; j < ns; j += 256) s_n[j] = 0;
    __syncthreads();
    const uint64_t stride = (uint64_t)gridDim.x * 256;
    for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < N; i += stride)
        if (!bad[i]) atomicAdd(&s_n[last_le(s_first, ns, i)], 1u);
    __syncthreads();
    for (int j = threadIdx.x; j < ns; j += 256)
        if (s_n[j]) atomicAdd(&alive[j], (unsigned long long)s_n[j]);
}

// ---------------------------------------------------------------- host side
template <int M, int W>
static void launch_scan(mp_ctx *ctx, uint32_t tiles, const BinScan &P)
{
    auto *const kernel = P.inr ? bin_scan_kernel<M, W, true> : bin_scan_kernel<M, W, false>;
    hipLaunchKernelGGL(kernel, dim3(tiles), dim3(256), 0, ctx->stream, P);
}

// M-mers of 13 bases (33 M canonical values, far more than there are cells);
// shorter ones below k = 22, so that a window keeps 10 of them.  wide: of 15
// (0.5 G values), which spread the minimizers of a large input over more cells
// and make some more records.  Records, grouping and runs of one scan of 150-base
// reads, 13 against 15 bases: 210 Mb 2.47, 2.51 ms (k = 25 2.66, 2.82), 450 Mb
// 5.02, 4.95 (5.45, 5.74), 1.2 Gb 16.4, 15.0 (17.9, 16.7); four scans of 1.2 Gb
// 26.7, 27.1.  They cross between 0.2 and 1.2 Gb, later for smaller k.
constexpr uint64_t kWideBases = 200000000;
static int scan_launch(mp_ctx *ctx, uint32_t tiles, bool wide, const BinScan &P)
{
    switch (wide && P.K >= 25 ? 100 + P.K : P.K) {
    case 125: launch_scan<15, 11>(ctx, tiles, P); break;
    case 126: launch_scan<15, 12>(ctx, tiles, P); break;
    case 127: launch_scan<15, 13>(ctx, tiles, P); break;
    case 128: launch_scan<15, 14>(ctx, tiles, P); break;
    case 129: launch_scan<15, 15>(ctx, tiles, P); break;
    case 130: launch_scan<15, 16>(ctx, tiles, P); break;
    case 131: launch_scan<15, 17>(ctx, tiles, P); break;
    case 20: launch_scan<11, 10>(ctx, tiles, P); break;
    case 21: launch_scan<12, 10>(ctx, tiles, P); break;
    case 22: launch_scan<13, 10>(ctx, tiles, P); break;
    case 23: launch_scan<13, 11>(ctx, tiles, P); break;
    case 24: launch_scan<13, 12>(ctx, tiles, P); break;
    case 25: launch_scan<13, 13>(ctx, tiles, P); break;
    case 26: launch_scan<13, 14>(ctx, tiles, P); break;
    case 27: launch_scan<13, 15>(ctx, tiles, P); break;
    case 28: launch_scan<13, 16>(ctx, tiles, P); break;
    case 29: launch_scan<13, 17>(ctx, tiles, P); break;
    case 30: launch_scan<13, 18>(ctx, tiles, P); break;
    case 31: launch_scan<13, 19>(ctx, tiles, P); break;
    default: return ctx->fail(MP_EINVAL, "no minimizer kernel for k = %d", P.K);
    }
    MP_HIP(hipGetLastError());
    return 0;
}

// The radix path keeps: 3-minimizer scans, k outside 20..31, letters whose
// neighbour class the 2-bit code cannot give (ctx->plain_letters), more
// segments than the tables hold, and callers who ask for a form of the radix
// sort (a tile shape, a digit width, a captured chain, an MP_SORT_* switch).
bool bins_apply(const mp_ctx *ctx, int T)
{
    if (ctx->cfg.min3 || ctx->cfg.k < 20 || ctx->cfg.k > 31 || !ctx->plain_letters || ctx->arena) return false;
    if (T > kMaxSeg || ctx->cfg.sort_graph || ctx->cfg.sort_tile || ctx->cfg.sort_digit_bits) return false;
    for (const char *e : {"MP_SORT_TILE", "MP_SORT_LOOKBACK", "MP_SORT_XCD", "MP_SORT_STATUS64", "MP_SORT_GLOBAL",
                          "MP_SORT_DIGITS"})
        if (getenv(e)) return false;
    return ctx->total_bases > 0 && ctx->total_bases < (1ull << 38);
}

namespace {

// bytes that a scan of n tuples by radix passes holds in its first key buffer:
// the bins' records take no more of it
uint64_t key_room(uint64_t n) { return (n + 1) * 8 + (n + 1) / 2; }

}  // namespace

int bins_scan(mp_ctx *ctx, const BinJob &job, mp_scan_stats *st, std::vector<uint64_t> *tpos, uint64_t *n_out, bool *done)
{
    *done = false;
    const uint64_t N = ctx->N, tb = ctx->total_bases;
    const int K = ctx->cfg.k, T = job.T;
    const bool batch = job.first != nullptr;
    const uint64_t nsteps = (tb + kStepPos - 1) / kStepPos;
    uint64_t npos = 0;  // windows, those with 'N' too
    MP_HIP(hipMemcpyAsync(&npos, (const uint64_t *)ctx->pos_off.p + N, sizeof(npos), hipMemcpyDeviceToHost, ctx->stream));
    MP_HIP(hipStreamSynchronize(ctx->stream));
    *n_out = npos;
    const uint64_t desc_bytes = nsteps * kStepRec * sizeof(uint64_t);
    if (npos == 0 || (desc_bytes > key_room(npos) && desc_bytes > (64ull << 20))) return 0;  // mostly reads without windows
    // wave steps per wave: about 8192 tiles (their table of counts stays small), at least one step
    static_assert(4 * 128 <= kTileSteps, "a tile's steps");
    const int steps = (int)std::min<uint64_t>(128, (nsteps + 4 * 8192 - 1) / (4 * 8192));
    const uint32_t tiles = (uint32_t)((nsteps + 4 * (uint64_t)steps - 1) / (4 * (uint64_t)steps));
    const uint32_t chunks = (tiles + kColTiles - 1) / kColTiles;
    // cells of a few hundred windows.  One scan, 11 against 13 bits: 450 Mb 4.99, 4.96 ms, 750 Mb 8.4, 7.9, 1.2 Gb
    // 15.0, 13.1, 1.8 Gb 24.0, 21.1 (four scans 9.9, 10.0; 16.5, 16.3; 27.3, 26.7; 43.1, 41.0): they cross at 450 Mb
    const int cell_bits = tb > kCellBases ? 13 : 11;
    struct Cleanup {  // the snapshot serves the kernels of this scan (and a later dump, which sets it again)
        mp_ctx *c;
        ~Cleanup() { c->use_labsnap = false; }
    } cleanup{ctx};
    auto enough = [&](int rc, bool *ok) -> int {  // a buffer that does not fit the budget: the radix path may still
        *ok = rc == 0;
        if (rc == MP_ENOMEM) {
            ctx->err.clear();
            return 0;
        }
        return rc;
    };
    bool ok = true;
#define MP_ROOM(x)                 \
    do {                           \
        MP_TRY(enough((x), &ok));  \
        if (!ok) return 0;         \
    } while (0)
    MP_ROOM(read_starts(ctx));
    // tables: counts per tile, chunk sums, coarse bins, per step counts and ranks, the segments
    const uint64_t o_csum = (uint64_t)tiles * kNC * 4, o_coarse = o_csum + (uint64_t)chunks * kNC * 4,
                   o_nrec = o_coarse + (kNC + 1) * 4, o_rank = o_nrec + nsteps * 4, o_bnd = o_rank + nsteps * 4,
                   o_cb = o_bnd + (kMaxSeg + 1) * 4, o_smp = o_cb + (kMaxSeg + 1) * 4,
                   o_first = (o_smp + kNC * 4 + 7) & ~7ull, o_end = o_first + (kMaxSeg + 1) * 8;
    MP_ROOM(ensure(ctx, ctx->rts, o_end + 64));
    MP_ROOM(ensure(ctx, ctx->binctl, sizeof(BinCtl) + 64 * sizeof(uint64_t) + (kMaxSeg + 1) * sizeof(uint64_t)));
    MP_ROOM(ensure(ctx, ctx->keys[0], desc_bytes));
    const uint32_t lo = (uint32_t)std::min<uint64_t>(job.lo, MP_NBUCKETS), hi = (uint32_t)std::min<uint64_t>(job.hi, MP_NBUCKETS);
    const bool ranged = !batch && !(lo == 0 && hi == MP_NBUCKETS);
    if (ranged) MP_ROOM(ensure(ctx, ctx->adj[1], nsteps * (kStepPos / 8) + 64));
    // a small scan holds the radix path's tuple buffers too, so that falling back to it, or a dump, allocates nothing
    if (npos <= (1ull << 24)) {
        const uint64_t n = job.expected ? std::min(job.expected, npos) : npos;
        for (int b = 0; b < 2; b++) {
            MP_ROOM(ensure(ctx, ctx->keys[b], (n + 1) * sizeof(uint64_t)));
            MP_ROOM(ensure(ctx, ctx->lab[b], (n + 1) * sizeof(uint32_t)));
            MP_ROOM(ensure(ctx, ctx->adj[b], n + 16));
        }
    }
    uint8_t *const tb0 = (uint8_t *)ctx->rts.p;
    uint32_t *const d_cnt = (uint32_t *)tb0, *const d_csum = (uint32_t *)(tb0 + o_csum),
             *const d_coarse = (uint32_t *)(tb0 + o_coarse), *const d_nrec = (uint32_t *)(tb0 + o_nrec),
             *const d_rank = (uint32_t *)(tb0 + o_rank), *const d_bnd = (uint32_t *)(tb0 + o_bnd),
             *const d_cb = (uint32_t *)(tb0 + o_cb), *const d_smp = (uint32_t *)(tb0 + o_smp);
    uint64_t *const d_first = (uint64_t *)(tb0 + o_first);
    BinCtl *const d_ctl = (BinCtl *)ctx->binctl.p;
    static_assert(sizeof(BinCtl) % 8 == 0, "words");
    unsigned long long *const d_nbad = (unsigned long long *)((uint8_t *)ctx->binctl.p + sizeof(BinCtl));
    unsigned long long *const d_alive = d_nbad + 64;
    MP_TRY(fill_u32(ctx, d_ctl, 0, sizeof(BinCtl) / 4 + 2 * 64 + 2 * (kMaxSeg + 1)));
    // segments: bucket boundaries, or a batch's samples with their share of the coarse bins
    std::vector<uint32_t> seg(2 * (kMaxSeg + 1) + kNC, 0);
    uint32_t *const h_bnd = seg.data(), *const h_cb = h_bnd + kMaxSeg + 1, *const h_smp = h_cb + kMaxSeg + 1;
    if (batch) {
        const uint64_t reads = job.first[T];
        uint32_t c = 0;
        for (int i = 0; i < T; i++) {  // at least one each: T + (kNC - T) in all at most
            const uint64_t n = job.first[i + 1] - job.first[i];
            const uint32_t share = 1 + (uint32_t)((double)n / (double)reads * (double)(kNC - T));
            h_cb[i] = c;
            for (uint32_t q = 0; q < share && c < (uint32_t)kNC; q++) h_smp[c++] = (uint32_t)i;
        }
        h_cb[T] = c;
        MP_HIP(hipMemcpyAsync(d_first, job.first, sizeof(uint64_t) * (T + 1), hipMemcpyHostToDevice, ctx->stream));
    } else {
        for (int i = 0; i <= T; i++) h_bnd[i] = (uint32_t)std::min<uint64_t>(job.bounds[i], MP_NBUCKETS);
    }
    MP_HIP(hipMemcpyAsync(d_bnd, seg.data(), seg.size() * sizeof(uint32_t), hipMemcpyHostToDevice, ctx->stream));
    // labels as they stand before any union of the scan, kept for a later dump
    KParams G{};
    G.N = N;
    G.scan0 = job.s == 0;
    G.parent = (const uint32_t *)ctx->parent.p;
    G.bad = (const uint8_t *)ctx->bad.p;
    if (job.s > 0) {
        MP_ROOM(snapshot_labels(ctx, job.s));
        G.labels = (const uint32_t *)ctx->labsnap.p;
        // filtered reads before the scan: restored when the scan is refused below (sizes is free until mp_finish)
        MP_HIP(hipMemcpyAsync(ctx->sizes.p, ctx->filtered.p, N, hipMemcpyDeviceToDevice, ctx->stream));
    }
    hipEventRecord(ctx->pev[0], ctx->stream);
    BinScan S{};
    S.packed = (const uint32_t *)ctx->packed.p;
    S.nmask = (const uint16_t *)ctx->nmask.p;
    S.rstart = (const uint16_t *)ctx->rstart.p;
    S.base_off = (const uint64_t *)ctx->base_off.p;
    S.N = N;
    S.total = tb;
    S.K = K;
    S.steps = steps;
    S.nsteps = nsteps;
    S.lo = lo;
    S.hi = hi;
    S.inr = ranged ? (uint16_t *)ctx->adj[1].p : nullptr;
    S.T = T;
    S.bounds = d_bnd;
    S.first = batch ? d_first : nullptr;
    S.cbase = d_cb;
    S.cell_bits = cell_bits;
    S.desc = (uint64_t *)ctx->keys[0].p;
    S.nrec = d_nrec;
    S.erank = d_rank;
    S.cnt = d_cnt;
    S.ctl = d_ctl;
    MP_TRY(scan_launch(ctx, tiles, tb > kWideBases, S));
    hipLaunchKernelGGL(bin_col_sum_kernel, dim3(chunks), dim3(kNC), 0, ctx->stream, (const uint32_t *)d_cnt, tiles, d_csum);
    hipLaunchKernelGGL(bin_col_scan_kernel, dim3(1), dim3(kNC), 0, ctx->stream, d_csum, chunks, d_coarse);
    hipLaunchKernelGGL(bin_col_apply_kernel, dim3(chunks), dim3(kNC), 0, ctx->stream, d_cnt, tiles,
                       (const uint32_t *)d_csum, (const uint32_t *)d_coarse);
    MP_HIP(hipGetLastError());
    std::unique_ptr<BinCtl> hc(new BinCtl);
    MP_HIP(hipMemcpyAsync(hc.get(), d_ctl, sizeof(BinCtl), hipMemcpyDeviceToHost, ctx->stream));
    MP_HIP(hipStreamSynchronize(ctx->stream));  // also: seg is read by the copy above
    uint64_t nrec = 0, nwin = 0, nv = 0;  // records, windows, the scan's tuples
    for (int i = 0; i < kStripes; i++) {
        nrec += hc->stat[i][2];
        nwin += hc->stat[i][3];
        nv += hc->stat[i][ranged ? 4 : 3];
    }
    if (batch)
        for (int i = 0; i < T; i++) nv += hc->nvalid[i];
    // a range that holds every window (one scan up to the last bucket that is not empty) needs no choice of windows
    const bool part = ranged && nv < nwin;
    if (hc->err || nv == 0 || nrec >= (1ull << 32) || nrec * sizeof(BinRec) > ctx->keys[0].bytes ||
        (nrec * sizeof(BinRec) > key_room(npos) && nrec * sizeof(BinRec) > (64ull << 20)))
        return 0;
    if (batch) {
        tpos->assign(T + 1, 0);
        for (int i = 0; i < T; i++) {  // a plain run's range plan is degenerate without k-mers (mp_plan_ranges)
            if (hc->nvalid[i] == 0) return ctx->fail(MP_EPLAN, "sample %d has no k-mers to partition", i);
            (*tpos)[i + 1] = (*tpos)[i] + hc->nvalid[i];
        }
    }
    if (job.expected && nv != job.expected)  // before any read is marked
        return ctx->fail(MP_ECOUNT, "scan %d enumerated %llu tuples, the histogram sized %llu", job.s, (unsigned long long)nv,
                         (unsigned long long)job.expected);
    // the last segment that holds tuples: the first-run quirk can only show there
    uint32_t last_lo = 0;
    if (!batch)
        for (int i = 0; i < T; i++)
            if (hc->kmax1[i]) last_lo = h_bnd[i];
    // bins of at most kBinRec records, with room for the cell that passes the aim
    const uint32_t aim = (uint32_t)std::max<uint64_t>(512, std::min<uint64_t>(kBinAim, nv * (kBinRec * 3 / 4) / nrec));
    const uint64_t bin_cap = 7 * nv / aim + kNC + 64;  // a cell of more than aim / 3 windows starts two
    MP_ROOM(ensure(ctx, ctx->keys[1], nrec * sizeof(BinRec)));
    MP_ROOM(ensure(ctx, ctx->lab[1], bin_cap * (2 * sizeof(BinDesc) + kBinWit * sizeof(uint32_t) * 2)));
    BinDesc *const d_bins = (BinDesc *)ctx->lab[1].p, *const d_big = d_bins + bin_cap;
    uint32_t *const d_wit = (uint32_t *)(d_big + bin_cap);
    uint4 *const rec_a = (uint4 *)ctx->keys[1].p, *const rec_b = (uint4 *)ctx->keys[0].p;
    hipLaunchKernelGGL(steps >= kScLongTile ? bin_scatter_kernel<6> : bin_scatter_kernel<3>, dim3(tiles), dim3(kScThreads), 0, ctx->stream, G, (const uint64_t *)S.desc,
                       (const uint32_t *)d_nrec, (const uint32_t *)d_rank, (const uint32_t *)d_cnt, steps, nsteps,
                       (const uint64_t *)(part ? S.inr : nullptr), rec_a);
    MP_HIP(hipGetLastError());
    hipEventRecord(ctx->pev[1], ctx->stream);
    auto *const group = cell_bits == 13 ? (part ? bin_group_kernel<8192, true> : bin_group_kernel<8192, false>)
                                        : (part ? bin_group_kernel<2048, true> : bin_group_kernel<2048, false>);
    hipLaunchKernelGGL(group, dim3(kNC), dim3(1024), 0, ctx->stream, (const uint4 *)rec_a, (const uint32_t *)d_coarse,
                       (const uint32_t *)(batch ? d_smp : nullptr), rec_b, d_bins, d_big, (uint32_t)bin_cap, aim, d_ctl);
    MP_HIP(hipGetLastError());
    MP_HIP(hipMemcpyAsync(hc.get(), d_ctl, sizeof(BinCtl), hipMemcpyDeviceToHost, ctx->stream));
    MP_HIP(hipStreamSynchronize(ctx->stream));
    const uint64_t nbin = hc->nbin, nbig = hc->nbig;
    if (hc->err || nbin > bin_cap || nbig > bin_cap) return 0;
    // what bin_runs_big may take, and its three visits of every group at the least
    const double big_ms = nv / kRadixWin + hc->big_win / kRadixDeep + 0.5;
    const uint64_t big_work = (uint64_t)(big_ms / kBigGroupMs);
    if (3 * std::max<uint64_t>(hc->big_most, hc->big_grp / kBigGrid) > big_work) return 0;
    // labels of the runs to join: every bin's (and every part's of a big bin) padded to whole bitmap words
    const uint64_t out_cap = nv + 64 * nbin + 256 * nbig + hc->big_win / 8 + 4096;
    MP_ROOM(ensure(ctx, ctx->lab[0], out_cap * sizeof(uint32_t)));
    MP_ROOM(ensure(ctx, ctx->runbits, (out_cap / 64 + 2) * sizeof(uint64_t)));
    if (nbig) MP_TRY(fill_u32(ctx, ctx->runbits.p, 0, 2 * (out_cap / 64 + 2)));
    const uint64_t nwit = (nbin + nbig) * kBinWit;
    MP_TRY(fill_u32(ctx, d_wit, ~0u, nwit));
    BinRuns R{};
    R.packed = (const uint64_t *)ctx->packed.p;
    R.rec = rec_b;
    R.K = K;
    R.T = T;
    R.batch = batch ? 1 : 0;
    R.bounds = d_bnd;
    R.last_lo = last_lo;
    R.bad = (const uint8_t *)ctx->bad.p;
    R.filtered = (uint8_t *)ctx->filtered.p;
    R.lab_out = (uint32_t *)ctx->lab[0].p;
    R.st_bits = (uint64_t *)ctx->runbits.p;
    R.out_cap = out_cap;
    R.ctl = d_ctl;
    auto runs = [&](bool check) -> int {
        // a dispatch holds fewer than 2^32 threads, so past 4 M bins (some 6e9 windows) there are several
        for (uint64_t b0 = 0; b0 < nbin; b0 += kRunGrid) {
            R.bins = d_bins + b0;
            R.nbin = (uint32_t)std::min(kRunGrid, nbin - b0);
            R.wit = d_wit + b0 * kBinWit;
            const dim3 gs(R.nbin), ts(kRunThreads);
            auto *const kernel = check ? (part ? bin_runs_kernel<true, true> : bin_runs_kernel<true, false>)
                                       : (part ? bin_runs_kernel<false, true> : bin_runs_kernel<false, false>);
            hipLaunchKernelGGL(kernel, gs, ts, 0, ctx->stream, R);
            MP_HIP(hipGetLastError());
        }
        R.bins = d_big;
        R.nbin = (uint32_t)nbig;
        R.wit = d_wit + nbin * kBinWit;
        R.big_work = check ? ~0ull : big_work;  // (a check repeats the first visits)
        if (nbig) {
            auto *const kernel = check ? (part ? bin_runs_big_kernel<true, true> : bin_runs_big_kernel<true, false>)
                                       : (part ? bin_runs_big_kernel<false, true> : bin_runs_big_kernel<false, false>);
            hipLaunchKernelGGL(kernel, dim3((unsigned)std::min<uint64_t>(nbig, kBigGrid)), dim3(kBigThreads), 0, ctx->stream, R);
            MP_HIP(hipGetLastError());
        }
        return 0;
    };
    hipEventRecord(ctx->pev[2], ctx->stream);
    MP_TRY(runs(false));
    hipEventRecord(ctx->pev[3], ctx->stream);
    // in-range tuples and errors before any read is marked BAD
    MP_HIP(hipMemcpyAsync(hc.get(), d_ctl, sizeof(BinCtl), hipMemcpyDeviceToHost, ctx->stream));
    MP_HIP(hipStreamSynchronize(ctx->stream));
    uint64_t runs_n = 0, zeroed = 0;
    for (int i = 0; i < kStripes; i++) {
        runs_n += hc->stat[i][0];
        zeroed += hc->stat[i][1];
    }
    auto restore = [&]() -> int {
        if (job.s > 0) {
            MP_HIP(hipMemcpyAsync(ctx->filtered.p, ctx->sizes.p, N, hipMemcpyDeviceToDevice, ctx->stream));
            MP_HIP(hipStreamSynchronize(ctx->stream));
        }
        return 0;
    };
    if (hc->err) return restore();  // the radix path marks the same reads again
    hipEventRecord(ctx->ev[2], ctx->stream);
    MP_TRY(refilter_reads(ctx, d_nbad));
    // First-run quirk (metapart.c:2539-2616): it shows only where the last run
    // of the last segment (of every sample) is the only one left with a live
    // label, so any live label of another run there rules it out: witnesses
    // of every bin first, then all tuples.  Where the last run alone lives,
    // the radix path decides
    if (nwit)
        hipLaunchKernelGGL(bin_witness_kernel, dim3((unsigned)((nbin * kBinWit + 255) / 256 + 1)), dim3(256), 0, ctx->stream,
                           (const uint32_t *)d_wit, (const BinDesc *)d_bins, nbin * kBinWit, R.batch,
                           (const uint8_t *)ctx->bad.p, d_ctl);
    if (nbig)
        hipLaunchKernelGGL(bin_witness_kernel, dim3((unsigned)((nbig * kBinWit + 255) / 256)), dim3(256), 0, ctx->stream,
                           (const uint32_t *)(d_wit + nbin * kBinWit), (const BinDesc *)d_big, nbig * kBinWit, R.batch,
                           (const uint8_t *)ctx->bad.p, d_ctl);
    if (batch)
        hipLaunchKernelGGL(bin_alive_kernel, dim3((unsigned)std::min<uint64_t>((N + 255) / 256, 512)), dim3(256), 0, ctx->stream,
                           (const uint8_t *)ctx->bad.p, (const uint64_t *)d_first, T, N, d_alive);
    MP_HIP(hipGetLastError());
    unsigned long long nbad = 0;
    std::vector<unsigned long long> alive(T, 0);
    MP_HIP(hipMemcpyAsync(hc->found, d_ctl->found, sizeof(hc->found), hipMemcpyDeviceToHost, ctx->stream));
    MP_HIP(hipMemcpyAsync(&nbad, d_nbad, sizeof(nbad), hipMemcpyDeviceToHost, ctx->stream));
    if (batch)
        MP_HIP(hipMemcpyAsync(alive.data(), d_alive, sizeof(unsigned long long) * T, hipMemcpyDeviceToHost, ctx->stream));
    MP_HIP(hipStreamSynchronize(ctx->stream));
    if (!batch) alive[0] = N - nbad;
    auto open = [&](bool all_seen) {
        for (int i = 0; i < (batch ? T : 1); i++)
            if (alive[i] && !(hc->found[i] & kFoundOther) && (!all_seen || (hc->found[i] & kFoundLast))) return true;
        return false;
    };
    if (open(false)) {
        MP_TRY(runs(true));
        MP_HIP(hipMemcpyAsync(hc->found, d_ctl->found, sizeof(hc->found), hipMemcpyDeviceToHost, ctx->stream));
        MP_HIP(hipStreamSynchronize(ctx->stream));
        if (open(true)) return 0;
    }
    hipEventRecord(ctx->ev[3], ctx->stream);
    MP_TRY(union_label_runs(ctx, (const uint32_t *)ctx->lab[0].p, (const uint64_t *)ctx->runbits.p, hc->out, N - nbad));
    hipEventRecord(ctx->ev[4], ctx->stream);
    MP_HIP(hipStreamSynchronize(ctx->stream));
    float ms = 0, a = 0, b = 0, u = 0;
    hipEventElapsedTime(&ms, ctx->pev[0], ctx->pev[1]);
    hipEventElapsedTime(&a, ctx->pev[1], ctx->pev[3]);
    hipEventElapsedTime(&b, ctx->ev[2], ctx->ev[3]);
    hipEventElapsedTime(&u, ctx->ev[3], ctx->ev[4]);
    float r = 0;
    hipEventElapsedTime(&r, ctx->pev[2], ctx->pev[3]);
    st->ms_enumerate = ms;
    st->ms_sort = a;
    st->ms_sort_local = r;
    st->ms_filter = b;
    st->ms_union = u;
    st->sort_long_groups = nbig;
    st->evaluated_runs = runs_n;
    st->zeroed_runs = zeroed;
    st->bad_labels = nbad;
    st->quirk_segments = 0;
    *n_out = nv;
    *done = true;
    return 0;
#undef MP_ROOM
}

}  // namespace mp
