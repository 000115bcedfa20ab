// f32 GEMM kernels for gfx950: C[b][i, j] (beta ? += : =) sum_p A(i, p) B(p, j)
// with f32 operands, f32 products and f32 accumulation on the matrix cores
// (v_mfma_f32_32x32x2_f32: 256 FLOP per clock and CU, twice what unpacked
// vector FMAs reach).  Each operand is "K-contiguous" (its reduction dim is
// contiguous: p[row * ld + k]) or "MN-contiguous" (p[k * ld + row]), at any
// leading dim and 4-byte alignment.
//
// The MFMA takes one k from each half of the wave, and which k is the
// program's choice as long as A and B agree: lane half h holds the four
// consecutive k at 8 g + 4 h, so a 32-row fragment of an 8-deep k group is
// one 16-byte read per lane and feeds four MFMAs.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "launch.h"

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

// one problem as the kernels read it
struct f32_args {
    const float *a;
    size_t lda, sa;
    const float *b;
    size_t ldb, sb;
    float *c;
    size_t ldc, sc;
    int m, n, k, beta, tiles_n;
    int va, vb; // 16-byte loads along k (K-contiguous operands)
};

// block id -> tile: ids are dealt to the 8 XCDs round-robin, so consecutive
// tiles (which share operand panels) are regrouped onto one XCD and its L2
__device__ __forceinline__ int xcd_tile(int pid, int nb)
{
    return (nb & 7) == 0 ? (pid & 7) * (nb >> 3) + (pid >> 3) : pid;
}

// the four k values at k .. k + 3 of row `row` (in range); those at or past
// kend read zero
template <bool MN>
__device__ __forceinline__ f32x4 load_k4(const float *__restrict__ p, size_t ld, int row, int k, int kend, bool vec)
{
    f32x4 v = {0.0f, 0.0f, 0.0f, 0.0f};
    if constexpr (MN) {
        const float *q = p + (size_t)k * ld + row;
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (j < kend - k)
                v[j] = q[(size_t)j * ld];
    } else {
        const float *q = p + (size_t)row * ld + k;
        if (vec && 3 < kend - k)
            return *(const f32x4 *)q;
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (j < kend - k)
                v[j] = q[j];
    }
    return v;
}

// the same four values when they are known to lie below kend
template <bool MN>
__device__ __forceinline__ f32x4 load_k4_full(const float *__restrict__ p, size_t ld, int row, int k, bool vec)
{
    if constexpr (MN) {
        const float *q = p + (size_t)k * ld + row;
        return f32x4{q[0], q[ld], q[2 * ld], q[3 * ld]};
    } else {
        const float *q = p + (size_t)row * ld + k;
        if (vec)
            return *(const f32x4 *)q;
        return f32x4{q[0], q[1], q[2], q[3]};
    }
}

__device__ __forceinline__ f32x16 mfma_f32(float a, float b, const f32x16 &c)
{
    return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ f32x4 mfma_f32(float a, float b, const f32x4 &c)
{
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Tiled kernel: a block of WGM x WGN waves owns BM x BN of C, each wave
// (BM / WGM) x (BN / WGN) of it.  K-tiles of KB go global -> registers ->
// LDS, the next tile's loads in flight while the current one is computed,
// two LDS buffers and one barrier per tile.  In LDS a tile is
// [KB / 4][ROWS + 1] slots of four consecutive k of one row: fragment reads
// are 16 bytes per lane over consecutive rows (no bank conflicts).  Whole
// tiles load from a wave-uniform base plus a fixed 32-bit offset per lane,
// so the loop spends no vector ALU work on addresses; an MN-contiguous
// operand comes as 4 x 4 blocks (four 16-byte loads) transposed in registers,
// or with 4-byte loads when it is not 16-byte aligned.  Bound by the matrix
// cores: 4096^3 runs at 121 - 133 TFLOP/s of 157 (128 x 128 tiles), and
// 2048 x 1024 x 1024 in 44 - 50 us on 64 x 64 tiles (two blocks per CU), where
// the 64 x 64 vector-FMA kernel before it took 206 - 210 us.
template <int ROWS, int KB, int NT, bool MN, bool VEC>
struct F32Tile {
    static constexpr int KQ = KB / 4, NL = ROWS * KQ / NT, SLOTS = KQ * (ROWS + 1);
    static_assert(ROWS * KQ % NT == 0, "tile slots divide by the thread count");
    static constexpr bool BLK = MN && VEC; // 4 x 4 blocks
    static_assert(!BLK || NL % 4 == 0, "whole 4 x 4 blocks");
    uint32_t off[NL];
    // the slot that load q of this thread fills.  BLK: load q reads k row
    // 4 kq + q % 4 of the four C rows row & ~3 .. row | 3, and after the
    // transpose slot q % 4 of the block is C row `row`
    __device__ __forceinline__ static void at(int q, int tid, int &row, int &kq)
    {
        if (BLK) {
            const int i = (q >> 2) * NT + tid;
            row = i % (ROWS / 4) * 4 + (q & 3);
            kq = i / (ROWS / 4);
        } else if (MN) {
            const int i = q * NT + tid;
            row = i % ROWS;
            kq = i / ROWS;
        } else {
            const int i = q * NT + tid;
            row = i / KQ;
            kq = i % KQ;
        }
    }
    // rows past `extent` read row 0 of the tile (their results are never
    // stored); BLK has extent % 4 == 0, so a block is wholly in or out
    __device__ __forceinline__ void init(size_t ld, int row0, int extent, int tid)
    {
#pragma unroll
        for (int q = 0; q < NL; ++q) {
            int row, kq;
            at(q, tid, row, kq);
            if (BLK)
                off[q] = (uint32_t)(4 * kq + (q & 3)) * (uint32_t)ld * 4 + (row0 + (row & ~3) < extent ? row & ~3 : 0) * 4;
            else if (MN)
                off[q] = (uint32_t)(4 * kq) * (uint32_t)ld * 4 + (row0 + row < extent ? row : 0) * 4;
            else
                off[q] = (uint32_t)(row0 + row < extent ? row : 0) * (uint32_t)ld * 4 + 16 * kq;
        }
    }
    // a tile wholly below k
    __device__ __forceinline__ void load_fast(f32x4 (&r)[NL], const float *__restrict__ p, size_t ld, int row0,
                                              int k0) const
    {
        const char *base = (const char *)(MN ? p + (size_t)k0 * ld + row0 : p + (size_t)row0 * ld + k0);
#pragma unroll
        for (int q = 0; q < NL; ++q) {
            if (VEC) {
                r[q] = *(const f32x4 *)(base + off[q]);
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    r[q][j] = *(const float *)(base + (MN ? (size_t)j * ld * 4 : (size_t)j * 4) + off[q]);
            }
        }
    }
    // any tile: values at or past k read zero
    __device__ __forceinline__ static void load(f32x4 (&r)[NL], const float *__restrict__ p, size_t ld, int row0,
                                                int extent, int k0, int k, int tid)
    {
#pragma unroll
        for (int q = 0; q < NL; ++q) {
            int row, kq;
            at(q, tid, row, kq);
            if (BLK) {
                const int kk = k0 + 4 * kq + (q & 3), gr = row0 + (row & ~3) < extent ? row0 + (row & ~3) : row0;
                r[q] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
                if (kk < k)
                    r[q] = *(const f32x4 *)(p + (size_t)kk * ld + gr);
            } else {
                r[q] = load_k4<MN>(p, ld, row0 + row < extent ? row0 + row : row0, k0 + 4 * kq, k, VEC);
            }
        }
    }
    __device__ __forceinline__ static void store(const f32x4 (&r)[NL], f32x4 *lds, int tid)
    {
#pragma unroll
        for (int q = 0; q < NL; ++q) {
            int row, kq;
            at(q, tid, row, kq);
            const int b = q & ~3, i = q & 3;
            if constexpr (BLK)
                lds[kq * (ROWS + 1) + pos(row)] = f32x4{r[b][i], r[b + 1][i], r[b + 2][i], r[b + 3][i]};
            else
                lds[kq * (ROWS + 1) + row] = r[q];
        }
    }
    // place of a row within its slot row: a 4 x 4 block's writes are 64 bytes
    // apart, so every other 16 rows take another order of their fours
    __device__ __forceinline__ static int pos(int row) { return BLK ? row ^ ((row >> 4) & 3) : row; }
    // rows r0 .. r0 + 31 of the k group at slot row 2 g
    __device__ __forceinline__ static f32x4 frag(const f32x4 *lds, int r0, int g, int lane)
    {
        return lds[(2 * g + (lane >> 5)) * (ROWS + 1) + pos(r0 + (lane & 31))];
    }
};

//
// With KG = 2 the block has two groups of WGM x WGN waves: each computes the
// whole tile over half of every k-tile, group 0 stages A and group 1 B, and
// group 1's sums are added through LDS at the end.  Twice the waves per SIMD
// for the same LDS, so one group's MFMAs cover the other's waits: for 256
// blocks or fewer, one per CU, 1024 x 1024 x 2048 goes from 57 - 67 to 50 - 56
// us; with two blocks per CU it measured the same, and slower on 128 x 128.
template <int BM, int BN, int WGM, int WGN, int KB, int KG, bool TA, bool TB, bool VEC>
__global__ void __launch_bounds__(64 * WGM * WGN * KG) k_gemm_f32(f32_args g)
{
    constexpr int NT = 64 * WGM * WGN, FM = BM / WGM / 32, FN = BN / WGN / 32, KS = KB / 8, KW = KS / KG;
    using OA = F32Tile<BM, KB, NT, TA, VEC>;
    using OB = F32Tile<BN, KB, NT, !TB, VEC>;
    __shared__ __align__(64) f32x4 smem[2 * (OA::SLOTS + OB::SLOTS)];
    f32x4(*const sa)[OA::SLOTS] = (f32x4(*)[OA::SLOTS])smem;
    f32x4(*const sb)[OB::SLOTS] = (f32x4(*)[OB::SLOTS])(smem + 2 * OA::SLOTS);
    const float *__restrict__ A = g.a + (size_t)blockIdx.z * g.sa;
    const float *__restrict__ B = g.b + (size_t)blockIdx.z * g.sb;
    float *__restrict__ C = g.c + (size_t)blockIdx.z * g.sc;
    const int tile = xcd_tile((int)blockIdx.x, (int)gridDim.x);
    const int m0 = tile / g.tiles_n * BM, n0 = tile % g.tiles_n * BN;
    const int grp = KG == 1 ? 0 : __builtin_amdgcn_readfirstlane((int)threadIdx.x / NT);
    const int tid = threadIdx.x - grp * NT, lane = tid & 63, wave = tid >> 6;
    const int wm = wave / WGN * (BM / WGM), wn = wave % WGN * (BN / WGN);
    f32x16 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e)
                acc[i][j][e] = 0.0f;
    static_assert(KG == 1 || (KG == 2 && OA::NL == OB::NL && KS % 4 == 0), "one staging register set per group");
    OA ta;
    OB tb;
    if (KG == 1 || grp == 0)
        ta.init(g.lda, m0, g.m, tid);
    if (KG == 1 || grp == 1)
        tb.init(g.ldb, n0, g.n, tid);
    f32x4 ra[OA::NL], rb2[KG == 1 ? OB::NL : 1];
    f32x4(&rb)[OB::NL] = *(f32x4(*)[OB::NL])(KG == 1 ? (void *)rb2 : (void *)ra);
    const int kt = g.k / KB + (g.k % KB != 0);
    auto store = [&](int buf) {
        if (KG == 1 || grp == 0)
            OA::store(ra, sa[buf], tid);
        if (KG == 1 || grp == 1)
            OB::store(rb, sb[buf], tid);
    };
    auto load = [&](int t) {
        if (KG == 1 || grp == 0)
            OA::load(ra, A, g.lda, m0, g.m, t * KB, g.k, tid);
        if (KG == 1 || grp == 1)
            OB::load(rb, B, g.ldb, n0, g.n, t * KB, g.k, tid);
    };
    auto compute = [&](const f32x4 *ca, const f32x4 *cb, int s0, int s1) {
#pragma unroll
        for (int s = s0; s < s1; ++s) {
            f32x4 fa[FM], fb[FN];
#pragma unroll
            for (int i = 0; i < FM; ++i)
                fa[i] = OA::frag(ca, wm + 32 * i, grp * KW + s, lane);
#pragma unroll
            for (int j = 0; j < FN; ++j)
                fb[j] = OB::frag(cb, wn + 32 * j, grp * KW + s, lane);
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int i = 0; i < FM; ++i)
#pragma unroll
                    for (int j = 0; j < FN; ++j)
                        acc[i][j] = mfma_f32(fa[i][q], fb[j][q], acc[i][j]);
        }
    };
    if (kt) {
        load(0);
        store(0);
        __syncthreads();
    }
    // tiles whose successor lies wholly below k (32-bit lane offsets reach it
    // for leading dims under 2^22): no branch in the loop
    const int fast = g.lda < ((size_t)1 << 22) && g.ldb < ((size_t)1 << 22) ? g.k / KB - 1 : 0;
    int t = 0;
    for (; t < fast; ++t) {
        if (KG == 1 || grp == 0)
            ta.load_fast(ra, A, g.lda, m0, (t + 1) * KB);
        if (KG == 1 || grp == 1)
            tb.load_fast(rb, B, g.ldb, n0, (t + 1) * KB);
        compute(sa[t & 1], sb[t & 1], 0, KW * 3 / 4);
        store((t + 1) & 1);
        compute(sa[t & 1], sb[t & 1], KW * 3 / 4, KW);
        __syncthreads();
    }
    for (; t < kt; ++t) {
        if (t + 1 < kt)
            load(t + 1);
        compute(sa[t & 1], sb[t & 1], 0, KW);
        if (t + 1 < kt)
            store((t + 1) & 1);
        __syncthreads();
    }
    if constexpr (KG == 2) { // after the last tile's barrier the buffers are free
        f32x16 *part = (f32x16 *)smem;
        static_assert(FM * FN * NT * 64 <= (int)sizeof smem, "group 1's sums fit");
        if (grp) {
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int j = 0; j < FN; ++j)
                    part[(i * FN + j) * NT + tid] = acc[i][j];
        }
        __syncthreads();
        if (grp)
            return;
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j)
                acc[i][j] += part[(i * FN + j) * NT + tid];
    }
    // lane holds column lane % 32 of rows 8 (e / 4) + 4 (lane / 32) + e % 4
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) {
            const int col = n0 + wn + 32 * j + (lane & 31);
            if (col >= g.n)
                continue;
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int row = m0 + wm + 32 * i + (e >> 2) * 8 + (lane >> 5) * 4 + (e & 3);
                if (row < g.m) {
                    float *p = C + (size_t)row * g.ldc + col;
                    *p = g.beta ? *p + acc[i][j][e] : acc[i][j][e];
                }
            }
        }
}

// Small outputs: a block owns one T x T tile of C (T = 16 or 32) and its eight
// waves split the reduction, each streaming its k range from global memory
// straight into MFMA operands (no LDS, no barrier in the k-loop; 1024 / T k in
// flight ahead of the MFMAs).  The waves' partial tiles are added through LDS
// in wave order.  For outputs with too few 64 x 64 tiles for the chip, where
// one wave's serial reduction would be the whole time.  Bound by the chain of
// load latencies along a wave's k range, which is why T = 16 is the faster one
// while its blocks all run at once: 256 x 512 x 784 takes 7.9 - 8.8 us at
// T = 16, 10.1 - 11.3 at T = 32 and 21 - 24 us on 64 x 64 tiles (103 us on the
// vector-FMA kernel before them); 32 x 32 x 4096 12 - 17, 32 - 37 and 85 - 92.
constexpr int kSmWaves = 8, kSmUnroll = 4;

template <int T, bool TA, bool TB>
__device__ __forceinline__ void f32_small_block(const f32_args &g, const int tile, float (*part)[T][T + 1])
{
    constexpr int KS = 256 / T; // k per MFMA group: four from each T-lane part of the wave
    typedef float acc_t __attribute__((ext_vector_type(T * T / 64)));
    const float *__restrict__ A = g.a + (size_t)blockIdx.z * g.sa;
    const float *__restrict__ B = g.b + (size_t)blockIdx.z * g.sb;
    float *__restrict__ C = g.c + (size_t)blockIdx.z * g.sc;
    const int m0 = tile / g.tiles_n * T, n0 = tile % g.tiles_n * T;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // this wave's k range, whole groups of KS
    const int kw = g.k ? (g.k - 1) / (KS * kSmWaves) * KS + KS : 0;
    const int kb = wave * kw < g.k ? wave * kw : g.k;
    const int kend = g.k - kb > kw ? kb + kw : g.k;
    const int row = m0 + lane % T < g.m ? m0 + lane % T : g.m - 1;
    const int col = n0 + lane % T < g.n ? n0 + lane % T : g.n - 1;
    const int kh = 4 * (lane / T);
    acc_t acc;
#pragma unroll
    for (int e = 0; e < T * T / 64; ++e)
        acc[e] = 0.0f;
    auto mm = [&](const f32x4 &x, const f32x4 &y) {
#pragma unroll
        for (int q = 0; q < 4; ++q)
            acc = mfma_f32(x[q], y[q], acc);
    };
    constexpr int U = kSmUnroll;
    const int whole = kb + (kend - kb) / (KS * U) * (KS * U);
    f32x4 fa[2][U], fb[2][U];
    auto load = [&](int buf, int k) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            fa[buf][u] = load_k4_full<TA>(A, g.lda, row, k + KS * u + kh, g.va);
            fb[buf][u] = load_k4_full<!TB>(B, g.ldb, col, k + KS * u + kh, g.vb);
        }
    };
    int k = kb;
    if (k < whole) {
        load(0, k);
        for (; whole - k >= 2 * KS * U; k += 2 * KS * U) {
            load(1, k + KS * U);
#pragma unroll
            for (int u = 0; u < U; ++u)
                mm(fa[0][u], fb[0][u]);
            if (whole - k > 2 * KS * U)
                load(0, k + 2 * KS * U);
#pragma unroll
            for (int u = 0; u < U; ++u)
                mm(fa[1][u], fb[1][u]);
        }
        if (k < whole) {
#pragma unroll
            for (int u = 0; u < U; ++u)
                mm(fa[0][u], fb[0][u]);
            k += KS * U;
        }
    }
    for (; k < kend; k += KS)
        mm(load_k4<TA>(A, g.lda, row, k + kh, kend, g.va), load_k4<!TB>(B, g.ldb, col, k + kh, kend, g.vb));
#pragma unroll
    for (int e = 0; e < T * T / 64; ++e)
        part[wave][(e >> 2) * 8 + lane / T * 4 + (e & 3)][lane % T] = acc[e];
    __syncthreads();
    const int c = tid % T;
    if (n0 + c >= g.n)
        return;
#pragma unroll
    for (int r = tid / T; r < T; r += 64 * kSmWaves / T) {
        if (m0 + r >= g.m)
            break;
        float v = 0.0f;
#pragma unroll
        for (int w = 0; w < kSmWaves; ++w)
            v += part[w][r][c];
        float *p = C + (size_t)(m0 + r) * g.ldc + n0 + c;
        *p = g.beta ? *p + v : v;
    }
}

template <int T, bool TA, bool TB>
__global__ void __launch_bounds__(64 * kSmWaves) k_gemm_f32_small(f32_args g)
{
    __shared__ float part[kSmWaves][T][T + 1];
    f32_small_block<T, TA, TB>(g, xcd_tile((int)blockIdx.x, (int)gridDim.x), part);
}

// A dgrad d (A K-contiguous, B transposed) and a wgrad w (A transposed) in one
// grid: d's blocks, then w's
template <int T>
__global__ void __launch_bounds__(64 * kSmWaves) k_gemm_f32_small_pair(f32_args d, f32_args w, int nd)
{
    __shared__ float part[kSmWaves][T][T + 1];
    const int pid = (int)blockIdx.x;
    if (pid < nd)
        f32_small_block<T, false, true>(d, xcd_tile(pid, nd), part);
    else
        f32_small_block<T, true, false>(w, xcd_tile(pid - nd, (int)gridDim.x - nd), part);
}

template <int BM, int BN, int WGM, int WGN, int KB, int KG, bool VEC>
void launch_tiled_v(int ta, int tb, const f32_args &g, dim3 grid, hipStream_t s)
{
    const dim3 block(64 * WGM * WGN * KG);
    switch ((ta ? 2 : 0) | (tb ? 1 : 0)) {
    case 0: hipLaunchKernelGGL((k_gemm_f32<BM, BN, WGM, WGN, KB, KG, false, false, VEC>), grid, block, 0, s, g); break;
    case 1: hipLaunchKernelGGL((k_gemm_f32<BM, BN, WGM, WGN, KB, KG, false, true, VEC>), grid, block, 0, s, g); break;
    case 2: hipLaunchKernelGGL((k_gemm_f32<BM, BN, WGM, WGN, KB, KG, true, false, VEC>), grid, block, 0, s, g); break;
    default: hipLaunchKernelGGL((k_gemm_f32<BM, BN, WGM, WGN, KB, KG, true, true, VEC>), grid, block, 0, s, g); break;
    }
}

template <int BM, int BN, int WGM, int WGN, int KB, int KG = 1>
void launch_tiled(int ta, int tb, f32_args g, unsigned batch, hipStream_t s)
{
    g.tiles_n = (g.n + BN - 1) / BN;
    const dim3 grid((unsigned)((g.m + BM - 1) / BM) * (unsigned)g.tiles_n, 1, batch);
    if (g.va && g.vb)
        launch_tiled_v<BM, BN, WGM, WGN, KB, KG, true>(ta, tb, g, grid, s);
    else
        launch_tiled_v<BM, BN, WGM, WGN, KB, KG, false>(ta, tb, g, grid, s);
}

template <int T>
void launch_small(int ta, int tb, f32_args g, unsigned batch, hipStream_t s)
{
    g.tiles_n = (g.n + T - 1) / T;
    const dim3 grid((unsigned)((g.m + T - 1) / T) * (unsigned)g.tiles_n, 1, batch), block(64 * kSmWaves);
    switch ((ta ? 2 : 0) | (tb ? 1 : 0)) {
    case 0: hipLaunchKernelGGL((k_gemm_f32_small<T, false, false>), grid, block, 0, s, g); break;
    case 1: hipLaunchKernelGGL((k_gemm_f32_small<T, false, true>), grid, block, 0, s, g); break;
    case 2: hipLaunchKernelGGL((k_gemm_f32_small<T, true, false>), grid, block, 0, s, g); break;
    default: hipLaunchKernelGGL((k_gemm_f32_small<T, true, true>), grid, block, 0, s, g); break;
    }
}

size_t tiles_of(size_t m, size_t n, size_t batch, size_t t)
{
    return ((m + t - 1) / t) * ((n + t - 1) / t) * batch;
}

// The tile side of the split-over-waves kernel (16, 32), or of the tiled one
// (64, 128): the shortest of three plans, as rounds of two blocks per CU, a
// round of 512 blocks and one of at most 256 (one per CU, which runs a block
// faster but leaves the CU short of waves), in units of 39 us at k = 1024.
// Measured there: 128 x 128 tiles 137 and 95 us, 64 x 64 tiles 39 and 28 us
// (33 with one wave group), 32 x 32 tiles with the reduction split over the
// waves 25 and 14 us.  The last become 16 x 16 tiles while those are at most
// kSm16Max, four blocks per CU: 512 x 512 x 512 takes 9 us either way, smaller
// outputs 7 - 9 against 7 - 21 us, 784 x 512 x 256 (1568 blocks) 10 against 8.
constexpr size_t kSm16Max = 1024;
int tile_plan(size_t m, size_t n, size_t batch)
{
    auto cost = [&](size_t tile, double full, double half) {
        const size_t tiles = tiles_of(m, n, batch, tile), rem = tiles % 512;
        return (double)(tiles / 512) * full + (rem > 256 ? full : rem ? half : 0.0);
    };
    const double big = cost(128, 3.5, 2.4), mid = cost(64, 1.0, 0.7), small = cost(32, 0.64, 0.36);
    if (small <= mid && small <= big)
        return tiles_of(m, n, batch, 16) <= kSm16Max ? 16 : 32;
    return mid <= big ? 64 : 128;
}

// 16-byte loads hold for an operand whose fragments start on 16 bytes
// (K-contiguous: every row; MN-contiguous: every k, over whole 4-row groups)
int vec_ok(const float *p, size_t ld, size_t stride, bool mn, size_t rows)
{
    return !(((uintptr_t)p & 15) | (ld & 3) | (stride & 3) | (mn ? rows & 3 : 0));
}

template <int T>
void launch_pair(f32_args d, f32_args w, hipStream_t s)
{
    d.tiles_n = (d.n + T - 1) / T;
    w.tiles_n = (w.n + T - 1) / T;
    const unsigned nd = (unsigned)((d.m + T - 1) / T) * (unsigned)d.tiles_n,
                   nw = (unsigned)((w.m + T - 1) / T) * (unsigned)w.tiles_n;
    hipLaunchKernelGGL(k_gemm_f32_small_pair<T>, dim3(nd + nw), dim3(64 * kSmWaves), 0, s, d, w, (int)nd);
}

} // namespace

extern "C" int pgk_gemm_f32(int ta, int tb, size_t m, size_t n, size_t k, const float *a, size_t lda,
                            size_t stride_a, const float *b, size_t ldb, size_t stride_b, float *c, size_t ldc,
                            size_t stride_c, size_t batch, int beta, pgk_stream s)
{
    if (!m || !n || !batch)
        return 0;
    if (batch > 65535 || m > 0x7fffffff || n > 0x7fffffff || k > 0x7fffffff)
        return (int)hipErrorInvalidValue;
    const f32_args g = {a, lda, stride_a, b, ldb, stride_b, c, ldc, stride_c, (int)m, (int)n, (int)k, beta, 0,
                        vec_ok(a, lda, stride_a, ta, m), vec_ok(b, ldb, stride_b, !tb, n)};
    switch (tile_plan(m, n, batch)) {
    case 16: launch_small<16>(ta, tb, g, (unsigned)batch, (hipStream_t)s); break;
    case 32: launch_small<32>(ta, tb, g, (unsigned)batch, (hipStream_t)s); break;
    case 64:
        if (tiles_of(m, n, batch, 64) <= 256)
            launch_tiled<64, 64, 2, 2, 64, 2>(ta, tb, g, (unsigned)batch, (hipStream_t)s);
        else
            launch_tiled<64, 64, 2, 2, 64>(ta, tb, g, (unsigned)batch, (hipStream_t)s);
        break;
    default: launch_tiled<128, 128, 2, 2, 32>(ta, tb, g, (unsigned)batch, (hipStream_t)s); break;
    }
    return (int)hipGetLastError();
}

// Both on the split-over-waves kernel when each alone would be: a launch
// boundary (about 1.2 us between dependent kernels) less, and the blocks of
// the one fill the CUs that the other leaves idle.  Not when the shared tile
// is 32 x 32 and one of them would alone be at most 256 tiles of 16 x 16 over
// a reduction of more than 640: the larger tile's chain of load latencies then
// costs more than the launch (8192 x 64 x 64: 79 us in one launch, 26 in two;
// 752 x 424 x 66: 11.0 and 9.7), and up to there less (437 x 613 x 56: 7.2 and
// 8.5 us; 540 tiles at 711 x 189 x 1293: 27 and 37).
extern "C" int pgk_gemm_f32_pair_tile(size_t m, size_t n, size_t k)
{
    if (!m || !n || !k || m > 0x7fffffff || n > 0x7fffffff || k > 0x7fffffff || tile_plan(m, k, 1) > 32 ||
        tile_plan(k, n, 1) > 32)
        return 0;
    const size_t td = tiles_of(m, k, 1, 16), tw = tiles_of(k, n, 1, 16);
    if (td + tw <= kSm16Max)
        return 16;
    return (td <= 256 && n > 640) || (tw <= 256 && m > 640) ? 0 : 32;
}

extern "C" int pgk_gemm_f32_pair(size_t m, size_t n, size_t k, const float *a, const float *b, const float *g,
                                 float *da, int beta_a, float *db, int beta_b, pgk_stream s)
{
    const int tile = pgk_gemm_f32_pair_tile(m, n, k);
    if (!tile)
        return PGK_GEMM_NOT_PAIRED;
    const f32_args d = {g, n, 0, b, n, 0, da, k, 0, (int)m, (int)k, (int)n, beta_a, 0, vec_ok(g, n, 0, false, m),
                        vec_ok(b, n, 0, false, k)};
    const f32_args w = {a, k, 0, g, n, 0, db, n, 0, (int)k, (int)n, (int)m, beta_b, 0, vec_ok(a, k, 0, true, k),
                        vec_ok(g, n, 0, true, n)};
    if (tile == 16)
        launch_pair<16>(d, w, (hipStream_t)s);
    else
        launch_pair<32>(d, w, (hipStream_t)s);
    return (int)hipGetLastError();
}
