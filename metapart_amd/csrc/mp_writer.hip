// Partitioned FASTQ writer (writeOutput3, metapart.c:956-1066).
//
// The reference re-reads every chunk on T threads and fwrite()s each record
// (single-end) or record pair (interleaved) to FromTid<t>_ToRank<P(root)>,
// a pair again to P(root of mate) when the two roots differ.  Here every
// output item (record or pair, copy 0 or 1) gets its place and its byte offset
// in one output buffer, which holds the 16*T files back to back (each in chunk
// and record order), by counts per file and tile and two scans over them, and
// waves copy the record bytes.  The host then writes each file's slice.  A
// batch of samples (one chunk each) gets 16 files per sample, planned over
// each sample's own ids.
#include <sys/stat.h>

#include <algorithm>
#include <cerrno>
#include <cstring>
#include <string>
#include <vector>

#include "mp_internal.h"
#include "mp_gather.h"

namespace mp {

constexpr int kMaxFiles = 0xFFFF;

// Items (a record, or a pair, of one output file) in file order without a sort:
// a tile is consecutive reads of one group (the chunks of one writer thread, or
// a sample of a batch), so its items go to the group's 16 files alone.  One
// wave counts a tile's items and bytes per file, two scans over the counts in
// file order give every tile its places, and one wave goes over the tile again
// and writes them, each item's place after those before it in the tile.
// (Against items with their file as key, sorted by two byte passes, and the
// lengths gathered and scanned: 12 M reads 1.07 -> 0.25 ms of kernels, 2,500 0.25 -> 0.19 ms a call.)
struct WParams {
    const uint64_t *rec_off;
    const uint32_t *parent;
    const uint64_t *chunk_ids;  // C + 1
    const uint64_t *pair_from;  // per chunk: first record that starts pairs (or chunk end); nullptr: none does
    const uint64_t *W;          // 17 per group (batch) or once: running maxima of the plan
    const uint64_t *first;      // G + 1: the groups' first reads
    const uint32_t *tile0;      // G + 1: their first tiles
    int C, G, batch;
    uint32_t tile_reads, tiles;
    uint32_t *cnt;              // items and bytes per (file, tile)
    uint64_t *bytes;
    const uint64_t *cnt_off, *byte_off;  // scanned
    uint32_t *slot;             // 2 r or 2 r + 1 of every item, in file order
    uint64_t *off;              // and its byte offset
};

// first p with x < W[p + 1] (metapart.c:1011-1012), the last if there is none; W of running maxima
__device__ __forceinline__ uint32_t part_of(const uint64_t *W, uint64_t x)
{
    static_assert(MP_NPART == 16, "four steps");
    uint32_t p = 0;
#pragma unroll
    for (uint32_t d = 8; d; d >>= 1)
        if (x >= W[p + d]) p += d;
    return p;
}

// first record of chunk c whose end offset (within the chunk) reaches il_start:
// records before it are single, records from it on pair up (getNextFullRead,
// metapart.c:211-294: a second record is read when the first ends at or after
// interleaveStart).
__global__ void pair_from_kernel(const uint64_t *__restrict__ rec_off, const uint64_t *__restrict__ chunk_ids,
                                 const uint64_t *__restrict__ chunk_ofs, const int64_t *__restrict__ il, int C,
                                 uint64_t *__restrict__ out)
{
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= C) return;
    uint64_t lo = chunk_ids[c], hi = chunk_ids[c + 1];
    if (il[c] < 0) {
        out[c] = hi;
        return;
    }
    const uint64_t target = chunk_ofs[c] + (uint64_t)il[c];
    while (lo < hi) {  // first r with rec_off[r+1] >= target
        const uint64_t mid = (lo + hi) >> 1;
        if (rec_off[mid + 1] < target) lo = mid + 1; else hi = mid;
    }
    out[c] = lo;
}

// entry of (group, file p of the group, tile) in cnt and bytes: files in order, a file's tiles in order
__device__ __forceinline__ uint64_t file_entry(const WParams &P, uint32_t g, uint32_t p, uint32_t tile)
{
    const uint32_t t0 = P.tile0[g];
    return P.batch ? (uint64_t)t0 * MP_NPART + (uint64_t)p * (P.tile0[g + 1] - t0) + (tile - t0) : (uint64_t)p * P.tiles + tile;
}

constexpr int kWWaves = 4;

template <bool PLACE> __global__ __launch_bounds__(kWWaves *kWave) void items_kernel(WParams P)
{
    __shared__ uint64_t s_W[kWWaves][MP_NPART + 1];
    __shared__ unsigned long long s_bytes[kWWaves][MP_NPART];
    __shared__ uint32_t s_cnt[kWWaves][MP_NPART];
    const uint32_t lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
    const uint32_t tile = blockIdx.x * kWWaves + wave;
    const bool have = tile < P.tiles;
    uint32_t g = 0;
    if (have)
        for (uint32_t hi = (uint32_t)P.G - 1; g < hi;) {  // the last group with tile0 <= tile
            const uint32_t mid = (g + hi + 1) >> 1;
            if (P.tile0[mid] <= tile) g = mid; else hi = mid - 1;
        }
    const uint64_t id0 = P.batch ? P.first[g] : 0;
    if (lane <= MP_NPART) s_W[wave][lane] = P.W[(P.batch ? (size_t)g * (MP_NPART + 1) : 0) + lane];
    if (lane < MP_NPART) {
        s_bytes[wave][lane] = 0;
        s_cnt[wave][lane] = 0;
    }
    __syncthreads();
    const uint64_t *const W = s_W[wave];
    const uint64_t r0 = have ? P.first[g] + (uint64_t)(tile - P.tile0[g]) * P.tile_reads : 0;
    const uint64_t r1 = have ? min(r0 + P.tile_reads, P.first[g + 1]) : 0;
    uint64_t at = 0, byte = 0;  // PLACE: lane p's next item of file p, and its first byte
    if (PLACE && have && lane < MP_NPART) {
        const uint64_t e = file_entry(P, g, lane, tile);
        at = P.cnt_off[e];
        byte = P.byte_off[e];
    }
    for (uint64_t b = r0; b < r1; b += kWave) {
        const uint64_t r = b + lane;
        uint32_t f0 = MP_NPART, f1 = MP_NPART, len = 0;  // files of the group (MP_NPART: no item)
        if (r < r1) {
            uint64_t pf = ~0ull;
            if (P.pair_from) {
                int lo = 0, hi = P.C - 1;
                while (lo < hi) {
                    const int mid = (lo + hi + 1) >> 1;
                    if (P.chunk_ids[mid] <= r) lo = mid; else hi = mid - 1;
                }
                pf = P.pair_from[lo];
            }
            const uint64_t pu = P.parent[r];
            if (r < pf) {
                f0 = part_of(W, pu - id0);
                len = (uint32_t)(P.rec_off[r + 1] - P.rec_off[r]);
            } else if (((r - pf) & 1) == 0) {
                const uint64_t mate = (r & 1) == 0 ? r + 1 : r - 1;  // metapart.c:1013-1016
                const uint64_t pv = P.parent[mate];
                f0 = part_of(W, pu - id0);
                if (pu != pv) f1 = part_of(W, pv - id0);
                len = (uint32_t)(P.rec_off[r + 2] - P.rec_off[r]);
            }
        }
        if constexpr (!PLACE) {
            if (f0 < MP_NPART) {
                atomicAdd(&s_cnt[wave][f0], 1u);
                atomicAdd(&s_bytes[wave][f0], (unsigned long long)len);
            }
            if (f1 < MP_NPART) {
                atomicAdd(&s_cnt[wave][f1], 1u);
                atomicAdd(&s_bytes[wave][f1], (unsigned long long)len);
            }
        } else {
            uint32_t todo = (f0 < MP_NPART ? 1u << f0 : 0u) | (f1 < MP_NPART ? 1u << f1 : 0u);
            for (;;) {  // the files that the wave's items go to, one by one
                const uint64_t any = __ballot(todo != 0);
                if (!any) break;
                const uint32_t f = (uint32_t)__builtin_ctz((uint32_t)__builtin_amdgcn_readlane((int)todo, __builtin_ctzll(any)));
                todo &= ~(1u << f);
                // items before (128 at most) and the low and high halves of their lengths, in two 32-bit sums
                const uint32_t c = (f0 == f ? 1u : 0u) + (f1 == f ? 1u : 0u);
                const uint32_t lo = (c << 23) + c * (len & 0xFFFF), hi = c * (len >> 16);
                const uint32_t li = wave_incl(lo), hi_i = wave_incl(hi), le = li - lo, he = hi_i - hi;
                const uint64_t a0 = __shfl(at, (int)f, kWave), b0 = __shfl(byte, (int)f, kWave);
                if (c) {
                    uint64_t q = a0 + (le >> 23), o = b0 + (le & 0x7FFFFF) + ((uint64_t)he << 16);
                    if (f0 == f) {
                        P.slot[q] = (uint32_t)(2 * r);
                        P.off[q++] = o;
                        o += len;
                    }
                    if (f1 == f) {
                        P.slot[q] = (uint32_t)(2 * r + 1);
                        P.off[q] = o;
                    }
                }
                const uint32_t lt = (uint32_t)__builtin_amdgcn_readlane((int)li, kWave - 1);
                const uint32_t ht = (uint32_t)__builtin_amdgcn_readlane((int)hi_i, kWave - 1);
                if (lane == f) {
                    at += lt >> 23;
                    byte += (lt & 0x7FFFFF) + ((uint64_t)ht << 16);
                }
            }
        }
    }
    if constexpr (!PLACE) {
        __syncthreads();
        if (have && lane < MP_NPART) {
            const uint64_t e = file_entry(P, g, lane, tile);
            P.cnt[e] = s_cnt[wave][lane];
            P.bytes[e] = s_bytes[wave][lane];
        }
    } else if (blockIdx.x == 0 && threadIdx.x == 0) {  // the end of the last item
        const uint64_t e = (uint64_t)P.tiles * MP_NPART;
        P.off[P.cnt_off[e]] = P.byte_off[e];
    }
}

// source of item i (in file order): its record, or the first record of its pair
struct RecSrc {
    const uint64_t *rec_off;
    const uint32_t *slot;
    __device__ uint64_t operator()(uint64_t i) const { return rec_off[slot[i] >> 1]; }
};

// first item of every file (and the end), and the byte offset there
__global__ void file_bounds_kernel(WParams P, int T, int F, uint64_t *__restrict__ pos, uint64_t *__restrict__ byte)
{
    const int f = blockIdx.x * blockDim.x + threadIdx.x;
    if (f > F) return;
    uint64_t e = (uint64_t)P.tiles * MP_NPART;
    if (f < F) {
        const uint32_t g = P.batch ? f / MP_NPART : f % T, p = P.batch ? f % MP_NPART : f / T;
        e = file_entry(P, g, p, P.tile0[g]);
    }
    pos[f] = P.cnt_off[e];
    byte[f] = P.byte_off[e];
}

static int make_dirs(const std::string &path)
{
    std::string cur;
    for (size_t i = 0; i <= path.size(); i++) {
        if (i == path.size() || path[i] == '/') {
            if (!cur.empty() && mkdir(cur.c_str(), 0755) != 0 && errno != EEXIST) return -1;
        }
        if (i < path.size()) cur.push_back(path[i]);
    }
    return 0;
}

int write_partitions(mp_ctx *ctx, const char *out_prefix, int T, const uint64_t *W, const int64_t *il_start,
                     uint64_t *bytes_out)
{
    const uint64_t N = ctx->N;
    const int C = ctx->C;
    const bool batch = ctx->batch;
    const int F = MP_NPART * T * (batch ? C : 1);
    if (F >= kMaxFiles) return ctx->fail(MP_EINVAL, "too many output files");
    // writer items are numbered 2 r and 2 r + 1 in 32 bits
    if (2 * N > (uint64_t)UINT32_MAX)
        return ctx->fail(MP_EINVAL, "the writer takes at most 2,147,483,647 reads (%llu loaded)",
                         (unsigned long long)N);
    if (batch && (T != 1 || ctx->sample_W.size() != (size_t)C * (MP_NPART + 1)))
        return ctx->fail(MP_ESTATE, "batch output needs T = 1 and per-sample plans");
    std::vector<int64_t> il(C, -1);
    bool paired = false;
    if (il_start)
        for (int c = 0; c < C; c++) {
            il[c] = il_start[c];
            paired |= il[c] >= 0;
        }
    // groups and their tiles: at most some 8192, and 256 reads or more
    const int G = batch ? C : T, cpt = C / G;
    const uint32_t tile_reads = (uint32_t)((std::max<uint64_t>(256, N / 8192) + kWave - 1) / kWave * kWave);
    std::vector<uint64_t> first(G + 1);
    std::vector<uint32_t> tile0(G + 2, 0);
    for (int g = 0; g <= G; g++) first[g] = ctx->chunk_ids[(size_t)g * cpt];
    for (int g = 0; g < G; g++) tile0[g + 1] = tile0[g] + (uint32_t)((first[g + 1] - first[g] + tile_reads - 1) / tile_reads);
    const uint32_t tiles = tile0[G];
    // small device inputs, in one copy: W (running maxima), first, tile0, and for pairs the chunks
    const size_t nW = batch ? (size_t)C * (MP_NPART + 1) : (size_t)(MP_NPART + 1);
    std::vector<uint64_t> in;
    in.reserve(nW + 2 * (size_t)(G + 2) + 4 * (size_t)(C + 1));
    for (size_t i = 0; i < nW; i++) {
        const uint64_t w = batch ? ctx->sample_W[i] : W[i];
        in.push_back(i % (MP_NPART + 1) > 1 ? std::max(w, in.back()) : w);
    }
    const size_t i_first = in.size();
    in.insert(in.end(), first.begin(), first.end());
    const size_t i_tile = in.size();
    in.resize(i_tile + (G + 2) / 2);
    memcpy(&in[i_tile], tile0.data(), sizeof(uint32_t) * (G + 1));
    const size_t i_ids = in.size(), i_cofs = i_ids + (paired ? C + 1 : 0), i_il = i_cofs + (paired ? C + 1 : 0);
    if (paired) {
        in.insert(in.end(), ctx->chunk_ids.begin(), ctx->chunk_ids.begin() + C + 1);
        in.insert(in.end(), ctx->chunk_ofs.begin(), ctx->chunk_ofs.begin() + C + 1);
        in.insert(in.end(), il.begin(), il.end());
    }
    const size_t i_pf = in.size(), i_pos = i_pf + (paired ? C : 0), i_end = i_pos + 2 * (size_t)(F + 1);
    uint64_t *d_small = nullptr;
    MP_HIP(hipMallocAsync((void **)&d_small, i_end * sizeof(uint64_t), ctx->stream));
    MP_HIP(hipMemcpyAsync(d_small, in.data(), in.size() * sizeof(uint64_t), hipMemcpyHostToDevice, ctx->stream));
    if (paired) {
        hipLaunchKernelGGL(pair_from_kernel, dim3((C + 255) / 256), dim3(256), 0, ctx->stream,
                           (const uint64_t *)ctx->rec_off.p, (const uint64_t *)(d_small + i_ids),
                           (const uint64_t *)(d_small + i_cofs), (const int64_t *)(d_small + i_il), C, d_small + i_pf);
        MP_HIP(hipGetLastError());
        std::vector<uint64_t> pf(C);
        MP_HIP(hipMemcpyAsync(pf.data(), d_small + i_pf, sizeof(uint64_t) * C, hipMemcpyDeviceToHost, ctx->stream));
        MP_HIP(hipStreamSynchronize(ctx->stream));
        for (int c = 0; c < C; c++)
            if ((ctx->chunk_ids[c + 1] - pf[c]) & 1) {
                MP_HIP(hipFreeAsync(d_small, ctx->stream));
                return ctx->fail(MP_EINVAL, "chunk %d: interleaved part has an odd number of records", c);
            }
    }
    const uint64_t n_items = paired ? 2 * N : N, E = (uint64_t)tiles * MP_NPART;  // at most; entries
    MP_TRY(ensure(ctx, ctx->ilens[0], n_items * sizeof(uint32_t)));
    MP_TRY(ensure(ctx, ctx->wg_off, (n_items + 1) * sizeof(uint64_t)));
    MP_TRY(ensure(ctx, ctx->wg_cnt, (E + 1) * sizeof(uint32_t)));
    MP_TRY(ensure(ctx, ctx->items[0], 3 * (E + 2) * sizeof(uint64_t)));
    WParams P{};
    P.rec_off = (const uint64_t *)ctx->rec_off.p;
    P.parent = (const uint32_t *)ctx->parent.p;
    P.chunk_ids = d_small + i_ids;
    P.pair_from = paired ? d_small + i_pf : nullptr;
    P.W = d_small;
    P.first = d_small + i_first;
    P.tile0 = (const uint32_t *)(d_small + i_tile);
    P.C = C;
    P.G = G;
    P.batch = batch ? 1 : 0;
    P.tile_reads = tile_reads;
    P.tiles = tiles;
    P.cnt = (uint32_t *)ctx->wg_cnt.p;
    P.bytes = (uint64_t *)ctx->items[0].p;
    uint64_t *const cnt_off = P.bytes + E + 2, *const byte_off = cnt_off + E + 2;
    P.cnt_off = cnt_off;
    P.byte_off = byte_off;
    P.slot = (uint32_t *)ctx->ilens[0].p;
    P.off = (uint64_t *)ctx->wg_off.p;
    hipEventRecord(ctx->ev[0], ctx->stream);
    const dim3 gi((tiles + kWWaves - 1) / kWWaves), ti(kWWaves * kWave);
    if (tiles) hipLaunchKernelGGL(items_kernel<false>, gi, ti, 0, ctx->stream, P);
    MP_HIP(hipGetLastError());
    MP_TRY(scan_u32(ctx, P.cnt, cnt_off, E));
    MP_TRY(scan_u64(ctx, P.bytes, byte_off, E));
    if (tiles) hipLaunchKernelGGL(items_kernel<true>, gi, ti, 0, ctx->stream, P);
    hipLaunchKernelGGL(file_bounds_kernel, dim3((F + 256) / 256), dim3(256), 0, ctx->stream, P, T, F, d_small + i_pos,
                       d_small + i_pos + (F + 1));
    MP_HIP(hipGetLastError());
    std::vector<uint64_t> bounds(2 * (size_t)(F + 1));
    MP_HIP(hipMemcpyAsync(bounds.data(), d_small + i_pos, sizeof(uint64_t) * bounds.size(), hipMemcpyDeviceToHost, ctx->stream));
    MP_HIP(hipStreamSynchronize(ctx->stream));
    const uint64_t *const fpos = bounds.data(), *const fbyte = fpos + (F + 1);
    const uint64_t total = fbyte[F];
    const uint32_t *const slot = P.slot;
    const uint64_t *const off = P.off;
    MP_TRY(ensure(ctx, ctx->out, total + 64));
    const uint64_t real_items = fpos[F];
    if (real_items && total) {
        uint64_t *first = nullptr;
        MP_HIP(hipMallocAsync((void **)&first, ((total + kGBlock - 1) / kGBlock + 1) * sizeof(uint64_t), ctx->stream));
        const int rc = launch_gather(ctx, ctx->d_fq, ctx->fq_bytes, off, real_items, total, total,
                                     first, RecSrc{(const uint64_t *)ctx->rec_off.p, slot},
                                     CopySink{(uint8_t *)ctx->out.p});
        MP_HIP(hipFreeAsync(first, ctx->stream));
        MP_TRY(rc);
    }
    hipEventRecord(ctx->ev[1], ctx->stream);
    MP_HIP(hipFreeAsync(d_small, ctx->stream));
    MP_HIP(hipStreamSynchronize(ctx->stream));
    if (bytes_out) *bytes_out = total;
    if (!out_prefix) return 0;
    // host side: one file per (t, P), written from pinned staging
    std::vector<char> host(total ? total : 1);
    if (total) MP_HIP(hipMemcpy(host.data(), ctx->out.p, total, hipMemcpyDeviceToHost));
    for (int f = 0; f < F; f++) {
        const int smp = f / (MP_NPART * T), p = (f / T) % MP_NPART, t = f % T;
        std::string dir = std::string(out_prefix) + (batch ? "/sample" + std::to_string(smp) : std::string()) + "/Rank0";
        if (batch && p == 0 && make_dirs(dir)) return ctx->fail(MP_EIO, "cannot create %s", dir.c_str());
        std::string name = dir + "/FromTid" + std::to_string(t) + "_ToRank" + std::to_string(p) + ".paired.fastq";
        FILE *fp = fopen(name.c_str(), "wb");
        if (!fp) return ctx->fail(MP_EIO, "cannot create %s", name.c_str());
        const uint64_t a = fbyte[f], b = fbyte[f + 1];
        if (b > a && fwrite(host.data() + a, 1, b - a, fp) != b - a) {
            fclose(fp);
            return ctx->fail(MP_EIO, "short write to %s", name.c_str());
        }
        fclose(fp);
    }
    return 0;
}

}  // namespace mp
