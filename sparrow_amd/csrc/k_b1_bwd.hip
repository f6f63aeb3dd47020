// k_b1_bwd.hip -- B1 sparse-connection backward (ops/src/b1_pure.rs:410-490,
// 642-656; ops/src/kernels.rs:2401-2478, 3229-3275), bitwise.
//
// dw is elementwise: each connection (i, j) gets one update from its own
// neuron's dy and source activation. dx is a scatter: source s sums
// dy[i] * w[i][j] over every connection that reads it, in (i, j) ascending
// order (the reference's loop order; its fused AVX2 kernel keeps that order
// by scattering one lane at a time). The GPU keeps the order without
// atomics through a reverse index: the connections grouped by source, in
// ascending connection number e = i * k0 + j inside each source, as pairs
// (neuron i, weight bits), so one thread per source (or per (source, token))
// replays its connections in the reference's order.
#include <hipcub/hipcub.hpp>

#include "internal.hpp"

namespace vmlm {

// Rust's `f as usize` for the f32 ids of SparseConnW.src
__device__ __forceinline__ size_t b1_usize(float f) {
    return f > 0.0f ? (f >= 1.8446744e19f ? ~(size_t)0 : (size_t)f) : 0;
}

__global__ __launch_bounds__(256) void b1_iota_kernel(uint32_t *v, size_t n) {
    const size_t stride = (size_t)gridDim.x * 256;
    for (size_t e = (size_t)blockIdx.x * 256 + threadIdx.x; e < n; e += stride) v[e] = (uint32_t)e;
}

// off[s] = first position of source s in the sorted ids (binary search),
// s = 0 .. d; ids >= d sort after off[d] and are never replayed.
__global__ __launch_bounds__(256) void b1_rev_offsets_kernel(const uint32_t *keys, size_t E,
                                                             size_t d, uint32_t *off) {
    const size_t s = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (s > d) return;
    size_t lo = 0, hi = E;
    while (lo < hi) {
        const size_t mid = (lo + hi) / 2;
        if (keys[mid] < s) lo = mid + 1;
        else hi = mid;
    }
    off[s] = (uint32_t)lo;
}

// dw[e] += dy[e / k0] * x[src[e]] (f32 ids when srcf, else u32); an id past
// the source dimension sets the guard and skips the connection.
__global__ __launch_bounds__(256) void b1_bwd_dw_kernel(const float *dy, const float *x,
                                                        const float *srcf, const uint32_t *src,
                                                        size_t E, size_t k0, size_t d, float *dw,
                                                        int *guard) {
    const size_t stride = (size_t)gridDim.x * 256;
    for (size_t e = (size_t)blockIdx.x * 256 + threadIdx.x; e < E; e += stride) {
        const size_t s = srcf ? b1_usize(srcf[e]) : src[e];
        if (s >= d) {
            atomicOr(guard, 1);
            continue;
        }
        dw[e] = dw[e] + dy[e / k0] * x[s];
    }
}

// dx[s] += dy[i] * w[e] over source s's connections in ascending e.
__global__ __launch_bounds__(256) void b1_bwd_dx_kernel(const uint2 *__restrict__ pairs,
                                                        const uint32_t *__restrict__ off,
                                                        const float *__restrict__ dy, size_t d,
                                                        float *__restrict__ dx) {
    const size_t s = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (s >= d) return;
    float acc = dx[s];
    const uint32_t end = off[s + 1];
    // eight pairs and their dy values in flight ahead of the ordered sum
    for (uint32_t t = off[s]; t < end; t += 8) {
        uint2 p[8];
        float v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) p[u] = pairs[t + u < end ? t + u : end - 1];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = dy[p[u].x];
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (t + u < end) acc = acc + v[u] * __uint_as_float(p[u].y);
    }
    dx[s] = acc;
}

// t8 dw: eight lanes per connection, lane l the FMA chain over tokens
// p = l, l + 8, ... (ops/src/kernels.rs:3245-3262), then the chains folded in
// hsum256's order ((l0+l4)+(l1+l5)) + ((l2+l6)+(l3+l7)) and added to dw.
__global__ __launch_bounds__(256) void b1_bwd_t8_dw_kernel(const uint32_t *src, const float *xt,
                                                           const float *dyt, size_t t8, size_t E,
                                                           size_t k0, size_t d, float *dw,
                                                           int *guard) {
    const size_t g = ((size_t)blockIdx.x * 256 + threadIdx.x) / 8;  // connection
    const int l = threadIdx.x & 7;
    const bool live = g < E;
    const size_t e = live ? g : 0;
    const size_t s = src[e];
    const bool ok = live && s < d;
    if (live && !ok && l == 0) atomicOr(guard, 1);
    float acc = 0.0f;
    if (ok) {
        const float *dr = dyt + (e / k0) * t8, *xr = xt + s * t8;
        for (size_t p = l; p < t8; p += 8) acc = __builtin_fmaf(dr[p], xr[p], acc);
    }
    const int base = (threadIdx.x & 63) & ~7;
    float v[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) v[q] = __shfl(acc, base + q, 64);
    if (ok && l == 0) {
        const float s0 = v[0] + v[4], s1 = v[1] + v[5], s2 = v[2] + v[6], s3 = v[3] + v[7];
        dw[e] = dw[e] + ((s0 + s1) + (s2 + s3));
    }
}

// The same over 16-byte aligned rows, two lanes per connection: lane h holds
// the chains l = 4h .. 4h + 3 of the reference's eight, so a step of eight
// tokens is one 16-byte load of each row, and eight steps are in flight. The
// kernel is bound by the gather of x rows out of L2 (4 * E * t8 bytes); the
// one-lane-per-chain form above loads 4 bytes a lane, an eighth of a step.
// n = 1536, k0 = 32, t8 = 1024: 36 -> 25 us.
__global__ __launch_bounds__(256) void b1_bwd_t8_dw_v4_kernel(
    const uint32_t *__restrict__ src, const float *__restrict__ xt, const float *__restrict__ dyt,
    size_t t8, size_t E, uint32_t k0, size_t d, float *__restrict__ dw, int *guard) {
    const size_t g = ((size_t)blockIdx.x * 256 + threadIdx.x) / 2;  // connection
    const int h = threadIdx.x & 1;
    const bool live = g < E;
    const uint32_t e = live ? (uint32_t)g : 0u;
    const size_t s = src[e];
    const bool ok = live && s < d;
    if (live && !ok && h == 0) atomicOr(guard, 1);
    const float *dr = dyt + (size_t)(e / k0) * t8 + 4 * h, *xr = xt + (ok ? s : 0) * t8 + 4 * h;
    float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    size_t p = 0;
    for (; p + 64 <= t8; p += 64) {
        float4 a[8], b[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            a[u] = *(const float4 *)(dr + p + 8 * u);
            b[u] = *(const float4 *)(xr + p + 8 * u);
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            acc[0] = __builtin_fmaf(a[u].x, b[u].x, acc[0]);
            acc[1] = __builtin_fmaf(a[u].y, b[u].y, acc[1]);
            acc[2] = __builtin_fmaf(a[u].z, b[u].z, acc[2]);
            acc[3] = __builtin_fmaf(a[u].w, b[u].w, acc[3]);
        }
    }
    for (; p < t8; p += 8) {
        const float4 a = *(const float4 *)(dr + p), b = *(const float4 *)(xr + p);
        acc[0] = __builtin_fmaf(a.x, b.x, acc[0]);
        acc[1] = __builtin_fmaf(a.y, b.y, acc[1]);
        acc[2] = __builtin_fmaf(a.z, b.z, acc[2]);
        acc[3] = __builtin_fmaf(a.w, b.w, acc[3]);
    }
    // hsum256: l and l + 4 sit in neighbouring lanes
    float sm[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) sm[q] = acc[q] + dpp_mov<0xB1>(acc[q]);
    if (ok && h == 0) dw[e] = dw[e] + ((sm[0] + sm[1]) + (sm[2] + sm[3]));
}

// The same with the x rows through LDS: a wave takes up to 32 connections of
// one output, copies 64 tokens of their rows straight into its own LDS (four
// rows of 256 contiguous bytes an instruction, two chunks ahead) and reads
// them back in the chains' order. The kernel above fetches 32 bytes of each of
// 32 rows an instruction, two cycles a segment at the address unit, and a
// wave's lines leave the L1 between its visits: 25 us at n = 1536, k0 = 32, t8
// = 1024, here 13.8. Piece q of row r lies at q ^ 2 (r % 8): the sixteen lanes
// that read a step of eight rows cover all banks once.
constexpr int B1_DW_W = 2, B1_DW_NS = 3;           // waves of a workgroup, chunks in LDS
constexpr int B1_DW_CHUNK = 32 * 256 + 256;        // 32 rows of x, one of dy
__global__ __launch_bounds__(64 * B1_DW_W) void b1_bwd_t8_dw_lds_kernel(
    const uint32_t *__restrict__ src, const float *__restrict__ xt, const float *__restrict__ dyt,
    uint32_t t8, uint32_t n, uint32_t k0, float *__restrict__ dw, int *guard) {
    __shared__ __align__(16) uint8_t lds[B1_DW_W * B1_DW_NS * B1_DW_CHUNK];
    const int lane = threadIdx.x & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t grp = (k0 + 31) / 32, gw = blockIdx.x * B1_DW_W + wave, j = gw / grp;
    if (j >= n) return;  // whole waves; no barriers below
    const int c = lane >> 1, h = lane & 1;
    const uint32_t idx = gw % grp * 32 + c;
    const bool live = idx < k0;
    const size_t e = (size_t)j * k0 + (live ? idx : 0);
    const uint32_t s = src[e];
    const bool ok = live && s < n;
    if (live && !ok && h == 0) atomicOr(guard, 1);
    const uint32_t row = (ok ? s : 0u) * t8 * 4;  // bytes; n * t8 * 4 < 2^32
    // copy v: rows 4v + lane / 16, the lane bringing piece lane % 16 as placed
    uint32_t voff[8];
#pragma unroll
    for (int v = 0; v < 8; ++v) voff[v] = (uint32_t)__shfl((int)row, 8 * v + 2 * (lane >> 4), 64);
    const uint32_t pc[2] = {(uint32_t)((lane & 15) ^ (2 * (lane >> 4))),
                            (uint32_t)((lane & 15) ^ (2 * (lane >> 4) + 8))};
    const float *dr = dyt + (size_t)j * t8;
    const uint8_t *mine = lds + wave * (B1_DW_NS * B1_DW_CHUNK);
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane(lds_addr(mine));
    const uint32_t nch = (t8 + 63) / 64;
    auto issue = [&](uint32_t kt) {  // nine copies; tokens past the row's end repeat its last
        const uint32_t base = lds0 + kt % B1_DW_NS * B1_DW_CHUNK;
        uint32_t tb[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) tb[i] = 4 * min(kt * 64 + 4 * pc[i], t8 - 4);
#pragma unroll
        for (int v = 0; v < 8; ++v) dma16s(xt, voff[v] + tb[v & 1], base + v * 1024);
        if (lane < 16) dma16s(dr, 4 * min(kt * 64 + 4 * (uint32_t)lane, t8 - 4), base + 8192);
    };
    float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    issue(0);
    if (nch > 1) issue(1);
    for (uint32_t kt = 0; kt < nch; ++kt) {
        if (kt + 2 < nch) {
            __builtin_amdgcn_s_waitcnt(0xC07F);  // the reads of the chunk written next
            issue(kt + 2);
            __builtin_amdgcn_s_waitcnt(waitcnt_vm(18));
        } else if (kt + 1 < nch) {
            __builtin_amdgcn_s_waitcnt(waitcnt_vm(9));
        } else {
            __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));
        }
        asm volatile("" ::: "memory");
        const uint8_t *st = mine + kt % B1_DW_NS * B1_DW_CHUNK;
        auto step = [&](int u) {
            const float4 a = *(const float4 *)(st + 8192 + u * 32 + h * 16);
            const float4 b = *(const float4 *)(st + c * 256 + (u ^ (c & 7)) * 32 + h * 16);
            acc[0] = __builtin_fmaf(a.x, b.x, acc[0]);
            acc[1] = __builtin_fmaf(a.y, b.y, acc[1]);
            acc[2] = __builtin_fmaf(a.z, b.z, acc[2]);
            acc[3] = __builtin_fmaf(a.w, b.w, acc[3]);
        };
        const int steps = (int)min(t8 - kt * 64, 64u) / 8;
        if (steps == 8) {
#pragma unroll
            for (int u = 0; u < 8; ++u) step(u);
        } else {
            for (int u = 0; u < steps; ++u) step(u);
        }
    }
    // hsum256: l and l + 4 sit in neighbouring lanes
    float sm[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) sm[q] = acc[q] + dpp_mov<0xB1>(acc[q]);
    if (ok && h == 0) dw[e] = dw[e] + ((sm[0] + sm[1]) + (sm[2] + sm[3]));
}

// t8 dx: one thread per (source, token): dxt[s][p] = fma(dyt[i][p], w[e],
// dxt[s][p]) over the source's connections in ascending e.
__global__ __launch_bounds__(256) void b1_bwd_t8_dx_kernel(const uint2 *__restrict__ pairs,
                                                           const uint32_t *__restrict__ off,
                                                           const float *__restrict__ dyt,
                                                           size_t t8, size_t d,
                                                           float *__restrict__ dxt) {
    const size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (idx >= d * t8) return;
    const size_t s = idx / t8, p = idx % t8;
    float acc = dxt[idx];
    for (uint32_t t = off[s]; t < off[s + 1]; ++t) {
        const uint2 pr = pairs[t];
        acc = __builtin_fmaf(dyt[(size_t)pr.x * t8 + p], __uint_as_float(pr.y), acc);
    }
    dxt[idx] = acc;
}

// The same with the gather in LDS: a workgroup stages TB tokens of every dyt
// row (4 * TB * d bytes) and takes its share of the sources, TB / 4 lanes of
// four tokens per source; a step is one pair (the lanes of a source read the
// same 8 bytes), one 16-byte LDS read and four FMAs. Bound by the LDS reads
// (4 * E * t8 bytes, about two bank cycles each over random rows); out of L2
// the same gather took 51 us at n = 1536, k0 = 32, t8 = 1024, here 21 us.
// TB is the largest of 16, 8, 4 whose tile fits the 160 KiB.
constexpr int B1_DX_THREADS = 768;
constexpr size_t B1_DX_LDS = 160 * 1024;
template <int TB>
__global__ __launch_bounds__(B1_DX_THREADS) void b1_bwd_t8_dx_lds_kernel(
    const uint2 *__restrict__ pairs, const uint32_t *__restrict__ off,
    const float *__restrict__ dyt, size_t t8, int d, int per, float *__restrict__ dxt) {
    extern __shared__ float4 b1_dx_tile[];
    constexpr int Q = TB / 4, SRC = B1_DX_THREADS / Q;  // lanes per source, sources per pass
    const int tid = threadIdx.x, q = tid % Q;
    const size_t t0 = (size_t)blockIdx.x * TB;
    const size_t t = t0 + 4 * (size_t)q;
    const int s1 = min(d, ((int)blockIdx.y + 1) * per);
    // the first source's range, then its first pairs, while the tile arrives
    int s = (int)blockIdx.y * per + tid / Q;
    uint32_t c = 0, end = 0;
    if (s < s1) {
        c = off[s];
        end = off[s + 1];
    }
    // pairs c .. c + 3 of a source that ends at e (past it the last, not used)
    auto load_pairs = [&](uint32_t c, uint32_t e, uint2 (&p)[4]) {
#pragma unroll
        for (int u = 0; u < 4; ++u) p[u] = pairs[c + u < e ? c + u : e ? e - 1 : 0];
    };
    // stage row r's tokens t0 .. t0 + TB - 1 (t8 is a multiple of 8: a quad is
    // all in range or all out), eight pieces in flight
    const int npc = d * Q;
    for (int pc0 = 0; pc0 < npc; pc0 += B1_DX_THREADS * 8) {
        float4 v[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const int pc = pc0 + tid + k * B1_DX_THREADS, pcc = pc < npc ? pc : npc - 1;
            const size_t t = t0 + 4 * (size_t)(pcc % Q);
            v[k] = *(const float4 *)(dyt + (size_t)(pcc / Q) * t8 + (t < t8 ? t : 0));
        }
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const int pc = pc0 + tid + k * B1_DX_THREADS;
            if (pc < npc) b1_dx_tile[pc] = v[k];
        }
    }
    uint2 p[4];
    float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
    load_pairs(c, end, p);
    if (s < s1 && t < t8) acc = *(const float4 *)(dxt + (size_t)s * t8 + t);
    __syncthreads();
    if (t >= t8) return;
    while (s < s1) {
        const int sn = s + SRC;
        uint32_t nc = 0, nend = 0;
        float4 nacc = acc;
        if (sn < s1) {
            nc = off[sn];
            nend = off[sn + 1];
            nacc = *(const float4 *)(dxt + (size_t)sn * t8 + t);
        }
        for (; c < end; c += 4) {
            uint2 np[4];
            float4 v[4];
            load_pairs(c + 4, end, np);
#pragma unroll
            for (int u = 0; u < 4; ++u) v[u] = b1_dx_tile[p[u].x * Q + q];
#pragma unroll
            for (int u = 0; u < 4; ++u)
                if (c + u < end) {
                    const float w = __uint_as_float(p[u].y);
                    acc.x = __builtin_fmaf(v[u].x, w, acc.x);
                    acc.y = __builtin_fmaf(v[u].y, w, acc.y);
                    acc.z = __builtin_fmaf(v[u].z, w, acc.z);
                    acc.w = __builtin_fmaf(v[u].w, w, acc.w);
                }
#pragma unroll
            for (int u = 0; u < 4; ++u) p[u] = np[u];
        }
        *(float4 *)(dxt + (size_t)s * t8 + t) = acc;
        s = sn;
        c = nc;
        end = nend;
        acc = nacc;
        load_pairs(c, end, p);
    }
}

static unsigned bwd_blocks(size_t n) {
    size_t b = (n + 255) / 256;
    return (unsigned)(b < 1 ? 1 : b);
}

// ---------------------------------------------------------- reverse index
// A counting sort in three launches. The connections are cut into tiles of
// 1024, a workgroup of 16 waves each, one connection a lane.
//  1. b1_rev_count: the rank of each connection among those of its tile with
//     the same source (inside a wave by ballots over the id's bits, across
//     the waves by byte counts in LDS), and the tile's count per source.
//  2. b1_rev_prefix: per source, the counts of the tiles before each tile,
//     and the total.
//  3. b1_rev_scatter: every tile scans the totals in LDS (the offsets) and
//     writes its connections' pairs at offset + prefix + rank.
// Ascending order inside a source follows from the order of tiles, waves and
// lanes. Each launch is latency bound: 49152 connections of 1536 sources
// 55 -> 12 us against the 32-bit radix sort with its index fill, which is
// kept for the index sizes past the limits below.
constexpr int REV_TILE = 1024;
constexpr size_t REV_DMAX = 8192;             // LDS: 16 * d bytes (count), 4 * d (scatter)
constexpr size_t REV_TABLE = (size_t)4 << 20;  // tiles * d (10 bytes of workspace each at most)

static size_t rev_tiles(size_t E) { return (E + REV_TILE - 1) / REV_TILE; }
static bool rev_counts(size_t E, size_t d) {
    return d <= REV_DMAX && rev_tiles(E) * d <= REV_TABLE;
}

__global__ __launch_bounds__(REV_TILE) void b1_rev_count_kernel(const uint32_t *__restrict__ src,
                                                                uint32_t E, int d, int d4, int bits,
                                                                uint16_t *__restrict__ rank,
                                                                uint16_t *__restrict__ cnt) {
    extern __shared__ uint32_t rev_hist[];  // [16 waves][d4 / 4 words]: byte counts
    uint8_t *hist = (uint8_t *)rev_hist;
    const int tid = threadIdx.x, wave = tid >> 6;
    const uint32_t e = blockIdx.x * REV_TILE + tid;
    const uint32_t key = e < E ? src[e] : 0xffffffffu;
    for (int i = tid; i < 16 * (d4 / 4); i += REV_TILE) rev_hist[i] = 0;
    const bool ok = key < (uint32_t)d;
    unsigned long long m = __ballot(ok);
    for (int b = 0; b < bits; ++b) {
        const bool one = (key >> b) & 1;
        const unsigned long long bal = __ballot(one);
        m &= one ? bal : ~bal;
    }
    const int lower = __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                                __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0));
    const int all = __popcll(m);
    __syncthreads();
    if (ok && lower == all - 1) hist[wave * d4 + key] = (uint8_t)all;
    __syncthreads();
    if (ok) {
        int r = lower;
        for (int w = 0; w < wave; ++w) r += hist[w * d4 + key];
        rank[e] = (uint16_t)r;
    }
    // four sources a thread: byte counts summed as two pairs of 16 bits
    for (int i = tid; i < d4 / 4; i += REV_TILE) {
        uint32_t lo = 0, hi = 0;
#pragma unroll
        for (int w = 0; w < 16; ++w) {
            const uint32_t v = rev_hist[w * (d4 / 4) + i];
            lo += v & 0x00ff00ffu;
            hi += (v >> 8) & 0x00ff00ffu;
        }
        uint2 o;
        o.x = (lo & 0xffffu) | (hi << 16);
        o.y = (lo >> 16) | (hi & 0xffff0000u);
        *(uint2 *)(cnt + (size_t)blockIdx.x * d4 + 4 * i) = o;
    }
}

// 64 sources a workgroup; each of its 16 waves takes a run of tiles.
__global__ __launch_bounds__(1024) void b1_rev_prefix_kernel(const uint16_t *__restrict__ cnt,
                                                             int tiles, int d4,
                                                             uint32_t *__restrict__ base,
                                                             uint32_t *__restrict__ tot) {
    __shared__ uint32_t part[16][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int s = blockIdx.x * 64 + lane, sc = s < d4 ? s : d4 - 1;
    const int run = (tiles + 15) / 16, b0 = wave * run, b1 = min(tiles, b0 + run);
    uint32_t sum = 0;
#pragma unroll 8
    for (int t = b0; t < b1; ++t) sum += cnt[(size_t)t * d4 + sc];
    part[wave][lane] = sum;
    __syncthreads();
    uint32_t acc = 0;
    for (int w = 0; w < wave; ++w) acc += part[w][lane];
    if (s >= d4) return;
#pragma unroll 8
    for (int t = b0; t < b1; ++t) {
        base[(size_t)t * d4 + s] = acc;
        acc += cnt[(size_t)t * d4 + s];
    }
    if (wave == 15) tot[s] = acc;
}

__global__ __launch_bounds__(REV_TILE) void b1_rev_scatter_kernel(
    const uint32_t *__restrict__ src, const float *__restrict__ w, uint32_t E, uint32_t k0, int d,
    int d4, const uint16_t *__restrict__ rank, const uint32_t *__restrict__ base,
    const uint32_t *__restrict__ tot, uint32_t *__restrict__ off, uint2 *__restrict__ pairs) {
    extern __shared__ uint32_t rev_off[];  // [d4]
    __shared__ uint32_t wsum[16];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const uint32_t e = blockIdx.x * REV_TILE + tid;
    const uint32_t key = e < E ? src[e] : 0xffffffffu;
    const bool ok = key < (uint32_t)d;
    const uint32_t r = ok ? (uint32_t)rank[e] + base[(size_t)blockIdx.x * d4 + key] : 0u;
    const float we = ok ? w[e] : 0.0f;
    // exclusive scan of the totals (zero past d): each thread a run of sources
    const int run = (d4 + REV_TILE - 1) / REV_TILE, s0 = tid * run;
    uint32_t v[REV_DMAX / REV_TILE];
    uint32_t mine = 0;
#pragma unroll
    for (int i = 0; i < (int)(REV_DMAX / REV_TILE); ++i) {
        v[i] = i < run && s0 + i < d4 ? tot[s0 + i] : 0u;
        mine += v[i];
    }
    uint32_t inc = mine;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t t = __shfl_up(inc, o, 64);
        if (lane >= o) inc += t;
    }
    if (lane == 63) wsum[wave] = inc;
    __syncthreads();
    uint32_t at = inc - mine;
    for (int q = 0; q < wave; ++q) at += wsum[q];
#pragma unroll
    for (int i = 0; i < (int)(REV_DMAX / REV_TILE); ++i) {
        if (i < run && s0 + i < d4) rev_off[s0 + i] = at;
        at += v[i];
    }
    __syncthreads();
    if (ok) pairs[rev_off[key] + r] = make_uint2(e / k0, __float_as_uint(we));
    if (blockIdx.x == 0) {
        for (int i = tid; i < d; i += REV_TILE) off[i] = rev_off[i];
        // at: after the last thread's run, the total
        if (tid == REV_TILE - 1) off[d] = at;
    }
}

// the sort path's pairs: connection perm[t]'s neuron and weight
__global__ __launch_bounds__(256) void b1_rev_pairs_kernel(const uint32_t *perm, size_t E,
                                                           const float *w, size_t k0,
                                                           uint2 *pairs) {
    const size_t stride = (size_t)gridDim.x * 256;
    for (size_t t = (size_t)blockIdx.x * 256 + threadIdx.x; t < E; t += stride)
        pairs[t] = make_uint2((uint32_t)(perm[t] / k0), __float_as_uint(w[perm[t]]));
}

static size_t sort_temp_bytes(size_t E) {
    size_t bytes = 0;
    (void)hipcub::DeviceRadixSort::SortPairs(nullptr, bytes, (const uint32_t *)nullptr,
                                             (uint32_t *)nullptr, (const uint32_t *)nullptr,
                                             (uint32_t *)nullptr, (int)E, 0, 32, (hipStream_t)0);
    return bytes;
}
static size_t a16(size_t x) { return (x + 15) / 16 * 16; }
static size_t rev_d4(size_t d) { return (d + 3) / 4 * 4; }

// Workspace: the pairs and offsets, then the counting sort's ranks, counts,
// prefixes and totals, or the radix sort's ids, permutations and temporary
// storage (16-byte aligned pieces).
size_t b1_rev_work_bytes(size_t E, size_t d) {
    const size_t out = a16(E * 8 + 8) + a16((d + 1) * 4);
    if (rev_counts(E, d)) {
        const size_t table = rev_tiles(E) * rev_d4(d);
        return out + a16(E * 2) + a16(table * 2) + a16(table * 4) + a16(rev_d4(d) * 4);
    }
    return out + 3 * a16(E * 4 + 4) + a16(sort_temp_bytes(E) + 16);
}

struct RevIndex {
    uint2 *pairs;
    uint32_t *off;
};

static int build_rev(const uint32_t *src, const float *w, size_t E, size_t k0, size_t d, void *work,
                     RevIndex &r, hipStream_t st) {
    VMLM_GUARD(E <= 0x7fffffffu && d < 0xffffffffu, "B1 backward: %zu connections", E);
    char *p = (char *)work;
    auto take = [&](size_t bytes) {
        char *q = p;
        p += a16(bytes);
        return q;
    };
    r.pairs = (uint2 *)take(E * 8 + 8);
    r.off = (uint32_t *)take((d + 1) * 4);
    if (rev_counts(E, d)) {
        int rc;
        const size_t tiles = rev_tiles(E), d4 = rev_d4(d);
        uint16_t *rank = (uint16_t *)take(E * 2);
        uint16_t *cnt = (uint16_t *)take(tiles * d4 * 2);
        uint32_t *base = (uint32_t *)take(tiles * d4 * 4);
        uint32_t *tot = (uint32_t *)take(d4 * 4);
        int bits = 0;
        while (((size_t)1 << bits) < d) ++bits;
        if ((rc = allow_lds((const void *)b1_rev_count_kernel, 16 * d4, 16 * REV_DMAX))) return rc;
        b1_rev_count_kernel<<<tiles, REV_TILE, 16 * d4, st>>>(src, (uint32_t)E, (int)d, (int)d4,
                                                              bits, rank, cnt);
        VMLM_HIP_CHECK(hipGetLastError());
        b1_rev_prefix_kernel<<<cdiv(d4, 64), 1024, 0, st>>>(cnt, (int)tiles, (int)d4, base, tot);
        VMLM_HIP_CHECK(hipGetLastError());
        b1_rev_scatter_kernel<<<tiles, REV_TILE, 4 * d4, st>>>(src, w, (uint32_t)E, (uint32_t)k0,
                                                               (int)d, (int)d4, rank, base, tot,
                                                               r.off, r.pairs);
        VMLM_HIP_CHECK(hipGetLastError());
        return VMLM_OK;
    }
    uint32_t *keys = (uint32_t *)take(E * 4 + 4);
    uint32_t *iota = (uint32_t *)take(E * 4 + 4);
    uint32_t *perm = (uint32_t *)take(E * 4 + 4);
    size_t tb = sort_temp_bytes(E);
    b1_iota_kernel<<<bwd_blocks(E), 256, 0, st>>>(iota, E);
    VMLM_HIP_CHECK(hipGetLastError());
    VMLM_HIP_CHECK(
        hipcub::DeviceRadixSort::SortPairs(p, tb, src, keys, iota, perm, (int)E, 0, 32, st));
    b1_rev_offsets_kernel<<<bwd_blocks(d + 1), 256, 0, st>>>(keys, E, d, r.off);
    VMLM_HIP_CHECK(hipGetLastError());
    b1_rev_pairs_kernel<<<bwd_blocks(E), 256, 0, st>>>(perm, E, w, k0, r.pairs);
    VMLM_HIP_CHECK(hipGetLastError());
    return VMLM_OK;
}

int launch_b1_backward(const float *w, const float *srcf, const uint32_t *src, size_t n,
                       size_t k0, const float *dy, const float *x, float *dw, float *dx,
                       void *work, hipStream_t st) {
    const size_t E = n * k0, d = n;
    if (E == 0) return VMLM_OK;
    int rc;
    if (dw) {
        b1_bwd_dw_kernel<<<bwd_blocks(E), 256, 0, st>>>(dy, x, srcf, src, E, k0, d, dw,
                                                        guard_flag_ptr());
        VMLM_HIP_CHECK(hipGetLastError());
    }
    if (dx) {
        RevIndex r;
        if ((rc = build_rev(src, w, E, k0, d, work, r, st))) return rc;
        b1_bwd_dx_kernel<<<bwd_blocks(d), 256, 0, st>>>(r.pairs, r.off, dy, d, dx);
        VMLM_HIP_CHECK(hipGetLastError());
    }
    return VMLM_OK;
}

// The dx launch over TB-token tiles: as many source shares as fill the CUs
// (a share is a whole number of passes of B1_DX_THREADS / (TB / 4) sources).
template <int TB>
static int launch_t8_dx_lds(const RevIndex &r, const float *dyt, size_t t8, size_t d, float *dxt,
                            hipStream_t st) {
    const int rc = allow_lds((const void *)b1_bwd_t8_dx_lds_kernel<TB>, d * TB * 4, B1_DX_LDS);
    if (rc) return rc;
    const size_t blocks = (t8 + TB - 1) / TB, pass = B1_DX_THREADS / (TB / 4);
    const size_t passes = (d + pass - 1) / pass;
    size_t shares = blocks >= 256 ? 1 : 256 / blocks;
    if (shares > passes) shares = passes;
    const size_t per = (passes + shares - 1) / shares * pass;
    b1_bwd_t8_dx_lds_kernel<TB>
        <<<dim3((unsigned)blocks, cdiv(d, per)), B1_DX_THREADS, d * TB * 4, st>>>(
            r.pairs, r.off, dyt, t8, (int)d, (int)per, dxt);
    VMLM_HIP_CHECK(hipGetLastError());
    return VMLM_OK;
}

int launch_b1_backward_t8(const float *w, const uint32_t *src, const float *xt, const float *dyt,
                          size_t t8, size_t n, size_t k0, float *dxt, float *dw, void *work,
                          hipStream_t st) {
    VMLM_GUARD(t8 % 8 == 0, "B1_T8 backward: t8 = %zu is not a multiple of 8", t8);
    const size_t E = n * k0, d = n;
    if (E == 0 || t8 == 0) return VMLM_OK;
    RevIndex r;
    int rc = build_rev(src, w, E, k0, d, work, r, st);
    if (rc) return rc;
    const bool al = (((uintptr_t)xt | (uintptr_t)dyt) & 15) == 0;
    // whole groups of 32 connections, or nearly (a wave takes a group)
    const size_t grp = (k0 + 31) / 32;
    if (al && n * t8 <= 0x3fffffff && n * grp <= 0x3fffffff && k0 * 4 >= grp * 96)
        b1_bwd_t8_dw_lds_kernel<<<cdiv(n * grp, B1_DW_W), 64 * B1_DW_W, 0, st>>>(
            src, xt, dyt, (uint32_t)t8, (uint32_t)n, (uint32_t)k0, dw, guard_flag_ptr());
    else if (al)
        b1_bwd_t8_dw_v4_kernel<<<bwd_blocks(E * 2), 256, 0, st>>>(src, xt, dyt, t8, E, (uint32_t)k0,
                                                                  d, dw, guard_flag_ptr());
    else
        b1_bwd_t8_dw_kernel<<<bwd_blocks(E * 8), 256, 0, st>>>(src, xt, dyt, t8, E, k0, d, dw,
                                                               guard_flag_ptr());
    VMLM_HIP_CHECK(hipGetLastError());
    // rows in LDS need 16-byte aligned rows and a tile that fits; few tokens
    // take the narrower tile (more workgroups for the same work)
    if ((((uintptr_t)dyt | (uintptr_t)dxt) & 15) == 0 && d * 16 <= B1_DX_LDS) {
        if (d * 64 <= B1_DX_LDS && t8 > 8) return launch_t8_dx_lds<16>(r, dyt, t8, d, dxt, st);
        if (d * 32 <= B1_DX_LDS) return launch_t8_dx_lds<8>(r, dyt, t8, d, dxt, st);
        return launch_t8_dx_lds<4>(r, dyt, t8, d, dxt, st);
    }
    b1_bwd_t8_dx_kernel<<<bwd_blocks(d * t8), 256, 0, st>>>(r.pairs, r.off, dyt, t8, d, dxt);
    VMLM_HIP_CHECK(hipGetLastError());
    return VMLM_OK;
}

}  // namespace vmlm
