// k_direct.hip -- GEMM of f32 rows with int8 or bf16 weights in one launch,
// without a prepared copy of either operand.
//
// C[M,N] = A[M,K] . W[N,K]^T (* scale[n]) (ops/src/kernels.rs:1199-1287) for
// any K, row alignment and M: the shapes whose time is the launches and passes
// around the GEMM rather than the GEMM itself.
//
// A workgroup owns a 16 TM x 16 TN tile of C and its NW waves split K into runs
// of 64-wide blocks. A wave loads a block of its rows with consecutive lanes on
// consecutive addresses (at whatever alignment the rows have), the next block's
// while the current one is multiplied, and passes it through a wave-private LDS
// slot into the MFMA operand layout, lane (g, r) = row r, k 16g .. 16g + 15.
// (Loading that layout straight from memory puts 16 rows into each quarter of
// a load instruction; the address processing then bounds the kernel:
// 77 x 1537 x 1001 8.3 us that way, 6.6 this way, 64 x 5760 x 2304 25 and 16.)
// The f32 values are split into the three bf16 terms of split_bf16 in registers,
// int8 weights become bf16 exactly, and each block runs two
// v_mfma_f32_16x16x32_bf16 per term and 16 x 16 tile (the first and the second
// eight k of every lane). The waves' sums meet in LDS and are added in wave
// order. Only the last block of a row can be partial; its elements past K are
// loaded from K - 1 and replaced by zeros, and rows past M or N repeat the last
// one (never stored), so no load leaves the operands.
#include "internal.hpp"

namespace vmlm {

namespace {

typedef u32x4 u32x4_b __attribute__((aligned(1)));
typedef f32x4 f32x4_w __attribute__((aligned(4)));

__device__ __forceinline__ f32x4 dg_mfma(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
// Orders one wavefront's LDS writes before its following LDS reads of other
// lanes' data (LDS operations of a wavefront execute in order).
__device__ __forceinline__ void dg_wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

struct DirectParams {
    const float *A;
    const uint8_t *W;
    const float *scale;
    float *C;
    size_t lda, ldw, ldc;  // elements
    int M, N, K;
};

// The three bf16 terms of 16 values (split_bf16), as two MFMA operands each:
// t[h][s] = term s of values 8h .. 8h + 7. Finite values need no test per
// remainder; a first term with an all-ones exponent (a NaN, an infinity or a
// value that rounds to one) anywhere in the wave redoes the split with them.
__device__ __forceinline__ void dg_terms(const f32x4 (&v)[4], u32x4 (&t)[2][3]) {
    typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
    u16x2 top = {0, 0};
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            float a = v[2 * h + q / 2][2 * (q % 2)], b = v[2 * h + q / 2][2 * (q % 2) + 1];
#pragma unroll
            for (int s = 0; s < 3; ++s) {
                const uint32_t p = bf16x2_rne_bits(a, b);
                t[h][s][q] = p;
                if (s == 0)
                    top = __builtin_elementwise_max(
                        top, __builtin_bit_cast(u16x2, p & 0x7fff7fffu));
                a = a - __uint_as_float(p << 16);
                b = b - __uint_as_float(p & 0xffff0000u);
            }
        }
    const bool bad = top[0] >= 0x7f80 || top[1] >= 0x7f80;
    if (__ballot(bad)) {
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                uint32_t x[3], y[3];
                split_bf16<3>(v[2 * h + q / 2][2 * (q % 2)], x);
                split_bf16<3>(v[2 * h + q / 2][2 * (q % 2) + 1], y);
#pragma unroll
                for (int s = 0; s < 3; ++s) t[h][s][q] = x[s] | (y[s] << 16);
            }
    }
}

// A block of a 16-row f32 fragment is 16 rows x 256 bytes: load q brings rows
// 4q .. 4q + 3, 16 lanes a row, and in LDS piece c (16 bytes) of row R sits in
// slot c ^ R. int8: 16 x 64 bytes, one load, 4 lanes a row; bf16: 16 x 128
// bytes, two loads, 8 lanes a row; slots c ^ (R / 4 % 4) and c ^ (R / 2 % 8).
// Writes and fragment reads are then free of bank conflicts.
template <bool WI8>
struct DgW {
    static constexpr int LDS = WI8 ? 1024 : 2048;
    static constexpr int NL = WI8 ? 1 : 2;          // loads per block
    static constexpr int LPR = WI8 ? 4 : 8;         // lanes per row
    static constexpr int EPL = WI8 ? 16 : 8;        // elements per lane
};

// NW waves; D blocks of a run in flight.
template <bool WI8, int TM, int TN, int NW, int D>
__global__ __launch_bounds__(NW * 64) void gemm_direct_kernel(DirectParams p) {
    using W = DgW<WI8>;
    constexpr int ESZ = WI8 ? 1 : 2;
    constexpr int SLOT = TM * 4096 + TN * W::LDS;  // a wave's operand bytes
    constexpr int RED = TM * TN * 1024;            // a wave's sums
    __shared__ __attribute__((aligned(16))) uint8_t smem[NW * (SLOT > RED ? SLOT : RED)];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 4, r = lane & 15;
    const int m0 = (int)blockIdx.y * (16 * TM), n0 = (int)blockIdx.x * (16 * TN);

    // load layout: this lane's rows and the element of a block it starts at
    const int ak = 4 * (lane & 15), wk = (lane % W::LPR) * W::EPL;
    const float *ar[TM][4];
    const uint8_t *wr[TN][W::NL];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int row = m0 + 16 * i + 4 * q + (lane >> 4);
            ar[i][q] = p.A + (size_t)(row < p.M ? row : p.M - 1) * p.lda;
        }
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int q = 0; q < W::NL; ++q) {
            const int row = n0 + 16 * j + (16 / W::NL) * q + lane / W::LPR;
            wr[j][q] = p.W + (size_t)(row < p.N ? row : p.N - 1) * p.ldw * ESZ;
        }
    // the lane's LDS bytes of a wave's slot: where its loads go, and its
    // fragment's pieces (f32: 4 of 16 bytes, int8: one, bf16: two)
    uint8_t *slot = smem + (size_t)wave * SLOT;
    int aw[4], ard[4], ww[W::NL], wrd[W::NL];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int R = 4 * q + (lane >> 4);
        aw[q] = R * 256 + ((lane & 15) ^ R) * 16;
        ard[q] = r * 256 + ((4 * g + q) ^ r) * 16;
    }
#pragma unroll
    for (int q = 0; q < W::NL; ++q) {
        if constexpr (WI8) {
            const int R = lane >> 2;
            ww[q] = R * 64 + ((lane & 3) ^ ((R >> 2) & 3)) * 16;
            wrd[q] = r * 64 + (g ^ ((r >> 2) & 3)) * 16;
        } else {
            const int R = 8 * q + (lane >> 3);
            ww[q] = R * 128 + ((lane & 7) ^ ((R >> 1) & 7)) * 16;
            wrd[q] = r * 128 + ((2 * g + q) ^ ((r >> 1) & 7)) * 16;
        }
    }

    // one row of tiles: the second and third terms' products in an accumulator
    // of their own, and the first term's two halves of a block in one each: half
    // the roundings at the sum's magnitude, no more than the few-row GEMV's
    // shorter runs of k have (with the halves in one, 2 x 19728 x 1536 bf16 had a
    // relative error of 1.18e-7 against its 9.9e-8)
    constexpr int NA = TM == 1 ? 3 : 1;
    f32x4 acc[NA][TM][TN];
#pragma unroll
    for (int n = 0; n < NA; ++n)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) acc[n][i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    f32x4 a[D][TM][4];
    u32x4 w[D][TN][W::NL];
    auto load = [&](int b, f32x4 (&da)[TM][4], u32x4 (&dw)[TN][W::NL]) {
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int q = 0; q < W::NL; ++q)
                dw[j][q] = *(const u32x4_b *)(wr[j][q] + (size_t)(64 * b + wk) * ESZ);
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int q = 0; q < 4; ++q) da[i][q] = *(const f32x4_w *)(ar[i][q] + 64 * b + ak);
    };
    auto load_tail = [&](int b, f32x4 (&da)[TM][4], u32x4 (&dw)[TN][W::NL]) {
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int q = 0; q < W::NL; ++q) {
                u32x4 v = u32x4{0, 0, 0, 0};
#pragma unroll
                for (int e = 0; e < W::EPL; ++e) {
                    const int k = 64 * b + wk + e, kc = k < p.K ? k : p.K - 1;
                    const uint32_t x = WI8 ? (uint32_t)wr[j][q][kc]
                                           : (uint32_t)((const uint16_t *)wr[j][q])[kc];
                    const int bit = e * ESZ * 8;
                    v[bit / 32] |= (k < p.K ? x : 0u) << (bit % 32);
                }
                dw[j][q] = v;
            }
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int k = 64 * b + ak + e;
                    const float x = ar[i][q][k < p.K ? k : p.K - 1];
                    da[i][q][e] = k < p.K ? x : 0.0f;
                }
    };
    auto compute = [&](const f32x4 (&da)[TM][4], const u32x4 (&dw)[TN][W::NL]) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int q = 0; q < 4; ++q) *(f32x4 *)(slot + i * 4096 + aw[q]) = da[i][q];
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int q = 0; q < W::NL; ++q)
                *(u32x4 *)(slot + TM * 4096 + j * W::LDS + ww[q]) = dw[j][q];
        dg_wave_sync();
        u32x4 wf[TN][2];
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const uint8_t *s = slot + TM * 4096 + j * W::LDS;
            if constexpr (WI8) {
                i8x16_to_bf16(*(const u32x4 *)(s + wrd[0]), wf[j][0], wf[j][1]);
            } else {
                wf[j][0] = *(const u32x4 *)(s + wrd[0]);
                wf[j][1] = *(const u32x4 *)(s + wrd[1]);
            }
        }
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            f32x4 v[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) v[q] = *(const f32x4 *)(slot + i * 4096 + ard[q]);
            u32x4 t[2][3];
            dg_terms(v, t);
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int s = 0; s < 3; ++s)
#pragma unroll
                    for (int j = 0; j < TN; ++j) {
                        f32x4 &c = acc[s == 0 && NA > 1 ? h : NA - 1][i][j];
                        c = dg_mfma(t[h][s], wf[j][h], c);
                    }
        }
        dg_wave_sync();
    };
    // this wave's whole blocks [b0, b1), then, for the last wave, the partial one
    const int nb = p.K / 64, b0 = nb * wave / NW, b1 = nb * (wave + 1) / NW;
    if (b0 < b1) {
        // D blocks a turn, so that each buffer is a fixed set of registers;
        // the loads past the run repeat its last block and are not used
#pragma unroll
        for (int u = 0; u < D - 1; ++u) load(b0 + u < b1 ? b0 + u : b1 - 1, a[u], w[u]);
        for (int b = b0; b < b1; b += D) {
#pragma unroll
            for (int u = 0; u < D; ++u) {
                const int nx = b + u + D - 1;
                if (nx < b1) load(nx, a[(u + D - 1) % D], w[(u + D - 1) % D]);
                if (b + u < b1) compute(a[u], w[u]);
            }
        }
    }
    if (wave == NW - 1 && nb * 64 < p.K) {
        load_tail(nb, a[0], w[0]);
        compute(a[0], w[0]);
    }

    __syncthreads();  // every wave is done with its slot
    f32x4 *red = (f32x4 *)smem;  // [NW][TM * TN][64]
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
            red[(wave * TM * TN + i * TN + j) * 64 + lane] =
                NA > 1 ? (acc[0][i][j] + acc[NA / 2][i][j]) + acc[NA - 1][i][j] : acc[0][i][j];
    __syncthreads();
    // accumulator (4g + e, r) of a tile: four rows of one column per thread
    for (int u = tid; u < TM * TN * 64; u += NW * 64) {
        const int t = u >> 6, ln = u & 63;
        f32x4 s = red[u];
#pragma unroll
        for (int q = 1; q < NW; ++q) s = s + red[q * TM * TN * 64 + u];
        const int col = n0 + 16 * (t % TN) + (ln & 15);
        const int row = m0 + 16 * (t / TN) + 4 * (ln >> 4);
        if (col >= p.N) continue;
        const float sc = p.scale ? p.scale[col] : 1.0f;
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (row + e < p.M) p.C[(size_t)(row + e) * p.ldc + col] = p.scale ? s[e] * sc : s[e];
    }
}

template <bool WI8, int TM, int TN, int NW, int D>
int launch_tile(const DirectParams &p, hipStream_t st) {
    const dim3 grid(cdiv((size_t)p.N, 16 * TN), cdiv((size_t)p.M, 16 * TM));
    gemm_direct_kernel<WI8, TM, TN, NW, D><<<grid, NW * 64, 0, st>>>(p);
    VMLM_HIP_CHECK(hipGetLastError());
    return VMLM_OK;
}

// The tiles. Two blocks of loads in flight (D = 2) where one workgroup is alone
// on its CU; one block, four waves and half the registers where several
// workgroups of a large grid hide each other's loads. `lat`, `thr`: us per block
// of a run with one workgroup on a CU, and per workgroup with its share of the
// CU full; `res`: workgroups that share a CU in the fit (at 17 to 1000 rows, 1500
// to 11520 columns, K 768 to 5760, int8; with bf16 weights LDS holds 1, 3 and 2 of
// the last three, which would change the choice at 3 of 151 bf16 sizes drawn,
// slower at two). Over 273 sizes drawn the estimate is 0.55 to
// 1.05 of the time of a call among others, 0.75 at the median: it lacks the store
// of C and the rows that every column of tiles reads again (1456 x 2764 x 75 14.4
// against 21.5 us, 768 x 11520 x 369 41.5 against 64, 100 x 2304 x 5760 20.6 against
// 21.7). The tile it chooses is 5 % from the best of the seven in the mean.
struct Tile {
    int tm, tn, nw, res;
    double lat, thr;
};
constexpr Tile TILES[] = {{1, 1, 8, 2, 0.94, 0.69}, {1, 2, 8, 1, 1.05, 1.31},
                          {1, 4, 8, 1, 1.65, 2.33}, {1, 4, 4, 3, 1.07, 0.85},
                          {2, 2, 8, 2, 1.75, 2.00}, {2, 2, 4, 4, 1.15, 0.80},
                          {2, 4, 4, 3, 1.50, 1.55}};

template <bool WI8>
int launch_w(const DirectParams &p, const Tile &t, hipStream_t st) {
    switch (100 * t.tm + 10 * t.tn + t.nw) {
    case 118: return launch_tile<WI8, 1, 1, 8, 2>(p, st);
    case 128: return launch_tile<WI8, 1, 2, 8, 2>(p, st);
    case 148: return launch_tile<WI8, 1, 4, 8, 2>(p, st);
    case 144: return launch_tile<WI8, 1, 4, 4, 1>(p, st);
    case 228: return launch_tile<WI8, 2, 2, 8, 1>(p, st);
    case 224: return launch_tile<WI8, 2, 2, 4, 1>(p, st);
    default: return launch_tile<WI8, 2, 4, 4, 1>(p, st);
    }
}

const Tile &pick_tile(int M, int N, int K, bool wi8, double *us) {
    const Tile *best = &TILES[0];
    double least = 1e30;
    for (const Tile &t : TILES) {
        const long long wgs = (long long)cdiv(N, 16 * t.tn) * cdiv(M, 16 * t.tm);
        const long long k = (wgs + 255) / 256, full = k / t.res, rest = k % t.res;
        const double blocks = (double)((K + 63) / 64) / t.nw;
        auto round = [&](long long r) {  // r workgroups on the busiest CU
            return r == 0 ? 0.0 : k == 1 || r * t.thr < t.lat ? t.lat : r * t.thr;
        };
        const double c = (blocks < 1.0 ? 1.0 : blocks) * (full * round(t.res) + round(rest));
        if (c < least) {
            least = c;
            best = &t;
        }
    }
    // no less than the operands once from HBM
    const double bytes = (double)N * K * (wi8 ? 1 : 2) + 4.0 * M * K + 4.0 * M * N;
    *us = 2.0 + (least > bytes / 5e6 ? least : bytes / 5e6);
    return *best;
}

}  // namespace

double gemm_direct_us(int M, int N, int K, bool w_int8) {
    double us;
    pick_tile(M, N, K, w_int8, &us);
    return us;
}

int launch_gemm_direct(const GemmDirectArgs &a, hipStream_t st) {
    VMLM_GUARD(a.M >= 1 && a.N >= 1 && a.K >= 1 && a.M <= 1 << 20,
               "gemm direct: M=%d N=%d K=%d", a.M, a.N, a.K);
    DirectParams p;
    p.A = a.A;
    p.W = (const uint8_t *)a.W;
    p.scale = a.scale;
    p.C = a.C;
    p.lda = a.lda;
    p.ldw = a.ldw;
    p.ldc = a.ldc;
    p.M = a.M;
    p.N = a.N;
    p.K = a.K;
    double us;
    const Tile &t = pick_tile(a.M, a.N, a.K, a.w_int8, &us);
    return a.w_int8 ? launch_w<true>(p, t, st) : launch_w<false>(p, t, st);
}

}  // namespace vmlm
