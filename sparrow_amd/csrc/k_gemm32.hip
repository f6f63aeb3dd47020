// k_gemm32.hip -- f32 GEMM on the f32 matrix cores.
//
// C[m,n] (+)= A[m,k] . op(B), op(B) = B[n,k]^T (NT: gemm_nt,
// ops/src/kernels.rs:986-1015) or B[k,n] (NN: gemm, :406-419).
// v_mfma_f32_16x16x4f32 multiplies f32 operands exactly and accumulates in f32
// (only the summation order differs from the reference's FMA chains, inside the
// 1e-4 * RMS contract of the attention composition).
//
// BM x BN tiles, four waves of 2 x 2. 32- or 64-deep k-steps go straight from
// global memory into a two-stage LDS ring, the next step's copies in flight while
// one is multiplied (three stages, so fewer workgroups a CU, were 1 to 4 %
// slower), or, where the rows are not 16-byte aligned, through registers. An
// operand stored along k ([row][k]) keeps its 16-byte
// pieces swizzled by row against bank conflicts, and a lane
// (g, r) = (lane / 16, lane % 16) reads four consecutive k of row r, one for each
// of four MFMAs (MFMA e of a 16-deep group multiplies k = 4g + e: any assignment
// that both operands share gives the same products). An NN B ([k][col]) keeps
// piece c of row k in slot c ^ 4 (k / 4 % 4), so that the four groups' rows meet
// other banks. Elements past k are copied from a zero; rows and columns past m
// and n repeat the last and are not stored.
//
// The MFMA rate bounds large shapes (a 16 x 16 x 4 product takes a matrix core 32
// cycles; the clock settles near 2.1 GHz under them), so the tile is chosen for an
// even load of the CUs. Against a register-staged kernel of 32 x 32 tiles: 1000 x
// 2304 x 2304 NT 125 -> 105 us, 2048^3 176 -> 141 (122 TFLOP/s), 4096^3 1400 ->
// 1030, 1500 x 1537 x 1535 (rows off 16 bytes) 193 -> 88. A rotated order of the
// steps per tile (to spread the L2 channels of rows 9 KiB apart) changed nothing,
// and tiles in an order that shares an XCD's L2 neither (4096^3 1030 us with
// both). The divisions of that order, an address loaded before the first copy and
// LDS for two stages where there is one step cost a short k up to 0.8 us (500 x
// 2304 x 64 5.4 us with them, 4.6 without; 161 x 1536 x 64 NN 3.6 and 3.0). A grid
// of few tiles is split over k (grid z): each slice writes its partial tile to
// `part` [ks][m][n] and gemm_f32_reduce_kernel sums the slices in order
// (deterministic). A result over its own operands goes that way with one slice
// too: the product stores nothing over rows that another tile still reads.
#include "internal.hpp"

namespace vmlm {

namespace {

// k of a step: 64 for the smallest tile (its 32-deep steps are mostly barriers)
template <int BM, int BN>
constexpr int g32_k() {
    return BM == 32 && BN == 32 ? 64 : 32;
}

__device__ __attribute__((aligned(16))) float g32_zero[4];

typedef f32x4 f32x4_w __attribute__((aligned(4)));

// LDS row of an NN B's k-row (and back): 32 columns are half of the banks, so
// groups 2 and 3 of a 16-deep group take the row of the other half.
template <int BN>
__device__ __forceinline__ int nn_row(int k) {
    return BN == 32 ? k ^ ((k >> 3) & 1) : k;
}

struct G32Params {
    const float *A, *B;
    float *C, *part;
    int m, n, k, acc, kslice;
};

// NA accumulators a tile: MFMA s of a step adds to accumulator s % NA.
template <bool NT, bool VEC, int BM, int BN, int NA>
__global__ __launch_bounds__(256) void gemm_f32_kernel(G32Params p) {
    constexpr int KS = g32_k<BM, BN>(), ROW = KS * 4, PK = KS / 4;  // pieces of a row along k
    constexpr int A_BYTES = BM * ROW, B_BYTES = BN * ROW, STAGE = A_BYTES + B_BYTES;
    constexpr int A_INS = A_BYTES / 4096, B_INS = B_BYTES / 4096;  // pieces a lane copies a step
    constexpr int WM = BM / 2, WN = BN / 2, TM = WM / 16, TN = WN / 16;
    static_assert(A_INS >= 1 && B_INS >= 1 && TM >= 1 && TN >= 1, "tile too small");
    extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];  // two stages, or the only step's

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 1, wn = wave & 1, g = lane >> 4, r = lane & 15;
    const int m0 = (int)blockIdx.y * BM, n0 = (int)blockIdx.x * BN;
    const int kb = (int)blockIdx.z * p.kslice;
    const int ke = kb + p.kslice < p.k ? kb + p.kslice : p.k;
    const int nk = (ke - kb + KS - 1) / KS;
    // slot of piece c of row R (rows along k): 128-byte rows share the banks in
    // pairs, 256-byte rows each hold all of them
    auto slot = [](int R, int c) { return c ^ (KS == 32 ? (R >> 1) & 7 : R & 15); };

    // this lane's source of each copy at step 0, and its k within the step
    const float *as[A_INS], *bs[B_INS];
    int ak[A_INS], bk[B_INS], bn[B_INS];
#pragma unroll
    for (int q = 0; q < A_INS; ++q) {
        const int off = ((q * 4 + wave) * 64 + lane) * 16, R = off / ROW;
        ak[q] = slot(R, (off >> 4) & (PK - 1)) * 4;
        const int row = m0 + R;
        as[q] = p.A + (size_t)(row < p.m ? row : p.m - 1) * p.k + kb + ak[q];
    }
#pragma unroll
    for (int q = 0; q < B_INS; ++q) {
        const int off = ((q * 4 + wave) * 64 + lane) * 16;
        if constexpr (NT) {
            const int R = off / ROW;
            bk[q] = slot(R, (off >> 4) & (PK - 1)) * 4;
            bn[q] = 4;
            const int row = n0 + R;
            bs[q] = p.B + (size_t)(row < p.n ? row : p.n - 1) * p.k + kb + bk[q];
        } else {
            constexpr int PPR = BN / 4;  // pieces per k-row
            bk[q] = nn_row<BN>(off / (BN * 4));
            const int c = ((off >> 4) & (PPR - 1)) ^ ((4 * (bk[q] >> 2)) & (PPR - 1) & 12);
            // (columns past n: a piece of the row's start, not stored)
            bn[q] = p.n - (n0 + 4 * c);
            const int col = bn[q] > 0 ? n0 + 4 * c : 0;
            bs[q] = p.B + (size_t)(kb + bk[q]) * p.n + col;
        }
    }
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane(lds_addr(smem));
    const size_t bstep = NT ? KS : (size_t)KS * p.n;
    auto issue = [&](int kt) {  // rows of whole 16-byte pieces, straight into LDS
        const uint32_t sb = lds0 + (uint32_t)((kt & 1) * STAGE);
        auto copies = [&](auto piece) {
#pragma unroll
            for (int q = 0; q < A_INS; ++q)
                dma16(piece(as[q] + kt * KS, ak[q]), sb + (q * 4 + wave) * 1024);
#pragma unroll
            for (int q = 0; q < B_INS; ++q)
                dma16(piece(bs[q] + kt * bstep, bk[q]), sb + A_BYTES + (q * 4 + wave) * 1024);
        };
        const int left = ke - (kb + kt * KS);
        // (apart, so that a whole step does not wait for the zero's address)
        if (left >= KS) copies([](const float *src, int) { return src; });
        else copies([&](const float *src, int k) { return k < left ? src : g32_zero; });
    };
    // rows at any float: the pieces through registers, those that cross the end
    // of a row (the last step, an NN B's last columns) element by element
    f32x4 ra[A_INS], rb[B_INS];
    auto load = [&](int kt) {
        const int left = ke - (kb + kt * KS);
        const bool whole = left >= KS && (NT || n0 + BN <= p.n);
        auto piece = [&](const float *src, int valid) {
            f32x4 v = {0.f, 0.f, 0.f, 0.f};
            if (valid >= 4) v = *(const f32x4_w *)src;
            else
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (e < valid) v[e] = src[e];
            return v;
        };
#pragma unroll
        for (int q = 0; q < A_INS; ++q) {
            const float *src = as[q] + kt * KS;
            ra[q] = left >= KS ? *(const f32x4_w *)src : piece(src, left - ak[q]);
        }
#pragma unroll
        for (int q = 0; q < B_INS; ++q) {
            const float *src = bs[q] + kt * bstep;
            rb[q] = whole ? *(const f32x4_w *)src
                    : NT  ? piece(src, left - bk[q])
                          : piece(src, bk[q] < left ? bn[q] : 0);
        }
    };
    auto store = [&](int kt) {
        uint8_t *sb = smem + (kt & 1) * STAGE + (wave * 64 + lane) * 16;
#pragma unroll
        for (int q = 0; q < A_INS; ++q) *(f32x4 *)(sb + q * 4096) = ra[q];
#pragma unroll
        for (int q = 0; q < B_INS; ++q) *(f32x4 *)(sb + A_BYTES + q * 4096) = rb[q];
    };

    f32x4 acc[NA][TM][TN];
#pragma unroll
    for (int n = 0; n < NA; ++n)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) acc[n][i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto compute = [&](const uint8_t *sA) {
        const uint8_t *sB = sA + A_BYTES;
#pragma unroll
        for (int h = 0; h < KS / 16; ++h) {
            const int at = slot(r, 4 * h + g) * 16;  // rows 16 i + r alike
            f32x4 a[TM], b[TN];
#pragma unroll
            for (int i = 0; i < TM; ++i)
                a[i] = *(const f32x4 *)(sA + (wm * WM + 16 * i + r) * ROW + at);
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const int col = wn * WN + 16 * j + r;
                if constexpr (NT) {
                    b[j] = *(const f32x4 *)(sB + col * ROW + at);
                } else {
                    const int cs = (col >> 2) ^ ((4 * g) & (BN / 4 - 1) & 12);
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        b[j][e] = *(const float *)(sB + nn_row<BN>(16 * h + 4 * g + e) * (BN * 4) +
                                                   cs * 16 + (col & 3) * 4);
                }
            }
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int j = 0; j < TN; ++j) {
                        f32x4 &c = acc[(4 * h + e) % NA][i][j];
                        c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i][e], b[j][e], c, 0, 0, 0);
                    }
        }
    };
    if constexpr (VEC) issue(0);
    else load(0);
    for (int kt = 0; kt < nk; ++kt) {
        // step kt is in LDS, and every wave has read step kt - 1
        if constexpr (VEC) __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));
        else store(kt);
        __syncthreads();
        if (kt + 1 < nk) {
            if constexpr (VEC) issue(kt + 1);
            else load(kt + 1);
        }
        compute(smem + (kt & 1) * STAGE);
    }

    float *out = p.part ? p.part + (size_t)blockIdx.z * p.m * p.n : p.C;
    const bool add = p.acc && !p.part;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
#pragma unroll
            for (int w = 1; w < NA; w *= 2)
#pragma unroll
                for (int n = 0; n < NA; n += 2 * w) acc[n][i][j] = acc[n][i][j] + acc[n + w][i][j];
            const int col = n0 + wn * WN + 16 * j + r, row = m0 + wm * WM + 16 * i + 4 * g;
            if (col >= p.n) continue;
            float *o = out + (size_t)row * p.n + col;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if (row + e >= p.m) continue;
                o[(size_t)e * p.n] = add ? o[(size_t)e * p.n] + acc[0][i][j][e] : acc[0][i][j][e];
            }
        }
}

__global__ __launch_bounds__(256) void gemm_f32_reduce_kernel(const float *__restrict__ part,
                                                              int ks, size_t mn,
                                                              float *__restrict__ C, int acc) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= mn) return;
    // 16 slices in flight, then summed in order
    float v[16];
#pragma unroll
    for (int z = 0; z < 16; ++z) v[z] = part[(size_t)(z < ks ? z : ks - 1) * mn + i];
    float sum = v[0];
#pragma unroll
    for (int z = 1; z < 16; ++z)
        if (z < ks) sum += v[z];
    for (int z0 = 16; z0 < ks; z0 += 16) {
#pragma unroll
        for (int z = 0; z < 16; ++z) v[z] = part[(size_t)(z0 + z < ks ? z0 + z : ks - 1) * mn + i];
#pragma unroll
        for (int z = 0; z < 16; ++z)
            if (z0 + z < ks) sum += v[z];
    }
    C[i] = acc ? C[i] + sum : sum;
}

// The tile with the least work on the busiest CU: `f` weighs what a smaller tile
// copies per product (128 x 128: 129 TFLOP/s at 4096^3; 64 x 64 119, 32 x 64 107,
// 32 x 32 102), `one` what it loses alone on its CU (fewer accumulators to keep
// a matrix core busy). Then the k-slices, of 128 at least, that give a small
// grid about two workgroups per CU (the second launch costs six steps, eight
// where it reduces more: 32 x 256 x 448 6.2 -> 6.0 us, 64 x 1024 x 448 6.2 -> 6.5, 114 x
// 768 x 512 6.8 -> 7.0):
// 16 at most, from k = 16384 on one per 1024 of k and 64 at most (32 x 32 x 65536:
// 37 us with 16, 14.6 with 64).
struct Shape {
    int bm, bn, ks, sums;
};
Shape pick_tile(size_t m, size_t n) {
    struct Tile {
        int bm, bn;
        double f, one;
    };
    constexpr Tile tiles[] = {{128, 128, 1.0, 1.0}, {64, 64, 1.08, 1.1}, {32, 64, 1.17, 1.15},
                              {32, 32, 1.26, 1.0}};
    Shape best{32, 32, 1, 1};
    if ((size_t)cdiv(m, 32) * cdiv(n, 32) <= 256) return best;  // one round of the smallest
    double least = 1e300;
    for (const Tile &t : tiles) {
        const size_t wgs = (size_t)cdiv(m, t.bm) * cdiv(n, t.bn), per = (wgs + 255) / 256;
        const double load = (double)per * t.bm * t.bn * t.f * (per == 1 ? t.one : 1.0);
        if (load < least) {
            least = load;
            best.bm = t.bm;
            best.bn = t.bn;
        }
    }
    return best;
}
Shape pick_shape(size_t m, size_t n, size_t k) {
    Shape best = pick_tile(m, n);
    const size_t wgs = (size_t)cdiv(m, best.bm) * cdiv(n, best.bn), steps = (k + 63) / 64;
    if (wgs <= 128 && steps >= (wgs > 64 ? 10 : wgs > 32 ? 8 : 7)) {
        size_t ks = 512 / wgs;
        if (ks > steps / 2) ks = steps / 2;
        const size_t most = steps <= 256 ? 16 : steps / 16 < 64 ? steps / 16 : 64;
        if (ks > most) ks = most;
        best.ks = (int)ks;
    }
    // fewer than 128 tiles: eight accumulators, so that a run of k is no longer
    // for it than in slices of 64 (100 x 256 x 448, one slice: relative error
    // 3.8e-7 with one, 1.9e-7 with four, 1.4e-7 with eight; 0.1 us; 32 x 32 x
    // 65536 1.1e-6 with one and 16 slices, 4.0e-7 in 256, now 2.5e-7)
    if ((size_t)cdiv(m, 32) * cdiv(n, 32) < 128 && k >= 128) best.sums = 8;
    return best;
}

template <bool NT, bool VEC, int BM, int BN, int NA = 1>
int launch_tile(const G32Params &p, int ks, hipStream_t st) {
    const dim3 grid(cdiv((size_t)p.n, BN), cdiv((size_t)p.m, BM), ks);
    constexpr int KS = g32_k<BM, BN>(), stage = (BM + BN) * KS * 4;
    static_assert(2 * stage <= 64 * 1024, "");
    const int lds = (p.kslice < p.k ? p.kslice : p.k) <= KS ? stage : 2 * stage;
    gemm_f32_kernel<NT, VEC, BM, BN, NA><<<grid, 256, lds, st>>>(p);
    VMLM_HIP_CHECK(hipGetLastError());
    return VMLM_OK;
}
template <bool NT, bool VEC>
int launch_shape(const G32Params &p, const Shape &s, hipStream_t st) {
    if (s.bm == 128) return launch_tile<NT, VEC, 128, 128>(p, s.ks, st);
    if (s.bm == 64) return launch_tile<NT, VEC, 64, 64>(p, s.ks, st);
    if (s.bn == 64) return launch_tile<NT, VEC, 32, 64>(p, s.ks, st);
    if (s.sums > 1) return launch_tile<NT, VEC, 32, 32, 8>(p, s.ks, st);
    return launch_tile<NT, VEC, 32, 32>(p, s.ks, st);
}

}  // namespace

size_t gemm_f32_work_floats(size_t m, size_t n, size_t k, bool over) {
    const int ks = pick_shape(m, n, k).ks;
    return ks > 1 || over ? (size_t)ks * m * n : 0;
}

int launch_gemm_f32(const float *a, const float *b, float *c, size_t m, size_t n, size_t k,
                    bool acc, bool b_is_nt, hipStream_t st, float *work, bool over) {
    if (m == 0 || n == 0) return VMLM_OK;
    if (k == 0) {
        if (!acc) return launch_fill_zero(c, m * n * sizeof(float), st);
        return VMLM_OK;
    }
    VMLM_GUARD(m <= 0x7fffffffu && n <= 0x7fffffffu && k <= 0x7fffffc0u,
               "gemm f32: shape too large");
    VMLM_GUARD(work || !over, "gemm f32: a result over its operands needs the workspace");
    Shape s = pick_shape(m, n, k);
    if (!work) s.ks = 1;
    const size_t steps = (k + 63) / 64;
    G32Params p;
    p.A = a;
    p.B = b;
    p.C = c;
    p.m = (int)m;
    p.n = (int)n;
    p.k = (int)k;
    p.acc = acc ? 1 : 0;
    p.kslice = (int)((steps + s.ks - 1) / s.ks * 64);
    s.ks = (int)((k + p.kslice - 1) / p.kslice);
    p.part = s.ks > 1 || over ? work : nullptr;
    const bool vec = k % 4 == 0 && (b_is_nt || n % 4 == 0) && ((uintptr_t)a & 15) == 0 &&
                     ((uintptr_t)b & 15) == 0;
    const int rc = b_is_nt ? vec ? launch_shape<true, true>(p, s, st) : launch_shape<true, false>(p, s, st)
                           : vec ? launch_shape<false, true>(p, s, st) : launch_shape<false, false>(p, s, st);
    if (rc || !p.part) return rc;
    gemm_f32_reduce_kernel<<<cdiv(m * n, (size_t)256), 256, 0, st>>>(work, s.ks, m * n, c, p.acc);
    VMLM_HIP_CHECK(hipGetLastError());
    return VMLM_OK;
}

}  // namespace vmlm
