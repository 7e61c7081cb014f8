// Row-major f32 matrix products on the f16 matrix cores: C (+)= op(A) op(B)
// with every f32 operand written as two f16 terms,
//   x 2^s = hi + lo,  hi = f16(x 2^s),  lo = f16(x 2^s - hi),
// and hi hi + hi lo + lo hi accumulated in f32 (lo lo is below 2^-22 of a
// product).  s is chosen per row of op(A) and per column of op(B) so that the
// largest element lies in [2^14, 2^15): hi + lo then carries 23 bits of every
// element down to 2^-17 of its row's largest and an absolute error of 2^-40
// of it below that.
//
// Rows the two terms do not represent (an infinity or a NaN, or a row more
// than half of whose nonzero elements lie below 2^-22 of its largest) are
// counted while splitting, and their outputs are formed from the f32 operands
// in f32 (exact_dot) instead.
//
// Bound: the f16 matrix cores, three products of 2 M N K (a third of 2.5
// PFLOP/s; the same products cost 157 TFLOP/s at most as f32 ones).  Measured,
// M x N x K: 32768 x 10496 x 2048 3.34 ms, 421 TFLOP/s of f32 product (1.26
// PFLOP/s of f16, where hipBLASLt's f16 kernel runs the same amount at 1.38),
// against 9.45 ms (149) by hipBLASLt in f32; 8192 x 2048 x 10496 0.79 against
// 2.31 ms; 2048 x 10496 x 8192 0.82 against 3.08 ms.  Relative error against
// f64 (2-norm) at K = 2048: 5.1e-7, where the f32 product's is 8.1e-7 (four
// times more roundings of the running sum).
#include "split_gemm.hpp"

namespace gdn2 {
namespace {

typedef _Float16 halfx8 __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

constexpr int kFragRows = 32, kFragK = 16; // one MFMA 32x32x16 operand: 64 lanes x 8 f16 = 1 KB
constexpr int kFragH8 = 64;                // halfx8 per fragment

// What a row of a split operand records about its elements.
//   amax   bits of the largest magnitude (NaN > infinity > every finite value)
//   small  nonzero elements below 2^-22 of it;  nonzero  nonzero elements
__device__ __forceinline__ bool row_bad(const SplitStat &s) {
    return s.amax >= 0x7F800000u || 2 * s.small > s.nonzero;
}
// x = m 2^e with m in [1/2, 1): the split multiplies by 2^(15 - e)
__device__ __forceinline__ int row_exp(unsigned amax) {
    return amax == 0 || amax >= 0x7F800000u ? 15 : __builtin_amdgcn_frexp_expf(__builtin_bit_cast(float, amax));
}
__device__ __forceinline__ unsigned abs_bits(float x) { return __builtin_bit_cast(unsigned, x) & 0x7FFFFFFFu; }

__device__ __forceinline__ void split8(const float *x, int sh, halfx8 *hi, halfx8 *lo) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const float s = __builtin_ldexpf(x[j], sh);
        const _Float16 h = (_Float16)s;
        (*hi)[j] = h;
        (*lo)[j] = (_Float16)(s - (float)h);
    }
}

// 8 consecutive elements of a row (or column) from k0: 0 past n
__device__ __forceinline__ void load8(const float *p, int64_t k0, int64_t n, bool vec, float *x) {
    if (vec && k0 + 8 <= n) {
        const floatx4 a = *reinterpret_cast<const floatx4 *>(p + k0), b = *reinterpret_cast<const floatx4 *>(p + k0 + 4);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            x[j] = a[j];
            x[4 + j] = b[j];
        }
    } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) x[j] = k0 + j < n ? p[k0 + j] : 0.f;
    }
}

// Splits rows along their contiguous dimension.  A workgroup owns 8 rows;
// lane l of a wave handles row l % 8 and the 8 elements from 8 (l / 8), so a
// row is read in runs of 256 bytes and a fragment written in runs of 128.
// Up to HELD x 256 elements a row stay in registers between the search for
// the row's largest and the split; longer rows are read again (from L2).
template <int HELD>
__global__ __launch_bounds__(256) void split_rows_kernel(const float *__restrict__ src, int64_t ld, int64_t R, int64_t n,
                                                         int64_t KT, bool vec, halfx8 *__restrict__ dst,
                                                         SplitStat *__restrict__ stat) {
    __shared__ unsigned red[3][4][8];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r8 = lane & 7;
    const int64_t row = (int64_t)blockIdx.x * 8 + r8;
    const bool ok = row < R;
    const float *p = src + (ok ? row : 0) * ld;
    const int64_t ng = 2 * KT; // groups of 8 elements, padded to whole fragments
    const int g0 = wave * 8 + (lane >> 3);
    float x[HELD][8];
    unsigned mx = 0;
#pragma unroll
    for (int i = 0; i < HELD; ++i) {
        const int64_t g = g0 + 32 * i;
        load8(p, 8 * g, ok && g < ng ? n : 0, vec, x[i]);
#pragma unroll
        for (int j = 0; j < 8; ++j) mx = max(mx, abs_bits(x[i][j]));
    }
    for (int64_t g = g0 + 32 * HELD; g < ng; g += 32) {
        float y[8];
        load8(p, 8 * g, ok ? n : 0, vec, y);
#pragma unroll
        for (int j = 0; j < 8; ++j) mx = max(mx, abs_bits(y[j]));
    }
#pragma unroll
    for (int o = 8; o < 64; o <<= 1) mx = max(mx, (unsigned)__shfl_xor((int)mx, o, 64));
    if (lane < 8) red[0][wave][r8] = mx;
    __syncthreads();
    mx = max(max(red[0][0][r8], red[0][1][r8]), max(red[0][2][r8], red[0][3][r8]));
    const int e = row_exp(mx);
    // nonzero magnitudes below 2^-22 of the largest (0 when that underflows)
    const unsigned lim = abs_bits(__builtin_ldexpf(__builtin_bit_cast(float, mx), -22));
    unsigned small = 0, nz = 0;
    // fragment of this row: (row / 32, g / 2), lane (row % 32) + 32 (g % 2)
    halfx8 *d = dst + (row / kFragRows) * KT * 2 * kFragH8 + row % kFragRows;
    auto put = [&](const float *y, int64_t g) {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const unsigned a = abs_bits(y[j]);
            small += a != 0 && a < lim;
            nz += a != 0;
        }
        halfx8 hi, lo;
        split8(y, 15 - e, &hi, &lo);
        halfx8 *f = d + (g / 2) * 2 * kFragH8 + (g & 1) * 32;
        f[0] = hi;
        f[kFragH8] = lo;
    };
#pragma unroll
    for (int i = 0; i < HELD; ++i)
        if (g0 + 32 * i < ng) put(x[i], g0 + 32 * i);
    for (int64_t g = g0 + 32 * HELD; g < ng; g += 32) {
        float y[8];
        load8(p, 8 * g, ok ? n : 0, vec, y);
        put(y, g);
    }
#pragma unroll
    for (int o = 8; o < 64; o <<= 1) {
        small += __shfl_xor((int)small, o, 64);
        nz += __shfl_xor((int)nz, o, 64);
    }
    if (lane < 8) {
        red[1][wave][r8] = small;
        red[2][wave][r8] = nz;
    }
    __syncthreads();
    if (wave == 0 && lane < 8) {
        SplitStat s;
        s.amax = mx;
        s.small = red[1][0][r8] + red[1][1][r8] + red[1][2][r8] + red[1][3][r8];
        s.nonzero = red[2][0][r8] + red[2][1][r8] + red[2][2][r8] + red[2][3][r8];
        stat[row] = s;
    }
}

__global__ __launch_bounds__(256) void stat_clear_kernel(SplitStat *stat, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n) stat[i] = SplitStat{0, 0, 0};
}

// Largest magnitude per column over a block of rows (a thread per column).
__global__ __launch_bounds__(256) void col_max_kernel(const float *__restrict__ src, int64_t ld, int64_t R, int64_t n,
                                                      int64_t per, SplitStat *__restrict__ stat) {
    const int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (c >= R) return;
    const int64_t k0 = (int64_t)blockIdx.y * per, k1 = min(n, k0 + per);
    unsigned mx = 0;
#pragma unroll 16
    for (int64_t k = k0; k < k1; ++k) mx = max(mx, abs_bits(src[k * ld + c]));
    atomicMax(&stat[c].amax, mx);
}

// Splits the columns of src (operand row = column of src, its k = row of
// src).  A workgroup takes 64 columns and `per` rows (a multiple of 64): it
// stages 64 x 64 tiles through LDS (rows 65 floats apart) and writes 2 x 4
// fragments of each; a thread's column is the same in all of them, so the
// counts of the column's record are added once at the end.
__global__ __launch_bounds__(256) void split_cols_kernel(const float *__restrict__ src, int64_t ld, int64_t R, int64_t n,
                                                         int64_t KT, int64_t per, halfx8 *__restrict__ dst,
                                                         SplitStat *__restrict__ stat) {
    __shared__ float t[64][65];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t c0 = (int64_t)blockIdx.x * 64, c = c0 + lane;
    const int fr = wave >> 1, cc = fr * 32 + (lane & 31);
    const int64_t row = c0 + cc, rt = c0 / kFragRows + fr, RT = (R + kFragRows - 1) / kFragRows;
    const unsigned mx = row < R ? stat[row].amax : 0;
    const int sh = 15 - row_exp(mx);
    const unsigned lim = abs_bits(__builtin_ldexpf(__builtin_bit_cast(float, mx), -22));
    unsigned small = 0, nz = 0;
    const int64_t kb = (int64_t)blockIdx.y * per, ke = min(kb + per, KT * kFragK);
    float next[16];
    auto load = [&](int64_t k0) {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int64_t k = k0 + wave * 16 + i;
            next[i] = c < R && k < n ? src[k * ld + c] : 0.f;
        }
    };
    load(kb);
    for (int64_t k0 = kb; k0 < ke; k0 += 64) {
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 16; ++i) t[wave * 16 + i][lane] = next[i];
        __syncthreads();
        if (k0 + 64 < ke) load(k0 + 64); // in flight beside this tile's split
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int fk = (wave & 1) * 2 + u, kk = fk * 16 + 8 * (lane >> 5);
            const int64_t kt = k0 / kFragK + fk;
            if (rt >= RT || kt >= KT) continue;
            float y[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                y[j] = t[kk + j][cc];
                const unsigned a = abs_bits(y[j]);
                small += a != 0 && a < lim;
                nz += a != 0;
            }
            halfx8 hi, lo;
            split8(y, sh, &hi, &lo);
            halfx8 *f = dst + (rt * KT + kt) * 2 * kFragH8 + lane;
            f[0] = hi;
            f[kFragH8] = lo;
        }
    }
    small += __shfl_xor((int)small, 32, 64);
    nz += __shfl_xor((int)nz, 32, 64);
    if (lane < 32 && row < R) {
        if (small) atomicAdd(&stat[row].small, small);
        if (nz) atomicAdd(&stat[row].nonzero, nz);
    }
}

// One output element from the f32 operands, in f32 (see the file comment).
__device__ __forceinline__ float exact_dot(const SplitGemmParams &p, int64_t m, int64_t n) {
    const float *a = p.A + (p.ta ? m : m * p.lda), *b = p.B + (p.tb ? n * p.ldb : n);
    const int64_t sa = p.ta ? p.lda : 1, sb = p.tb ? 1 : p.ldb;
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
    int64_t k = 0;
    for (; k + 4 <= p.Kd; k += 4)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[j] = __builtin_fmaf(a[(k + j) * sa], b[(k + j) * sb], acc[j]);
    for (; k < p.Kd; ++k) acc[0] = __builtin_fmaf(a[k * sa], b[k * sb], acc[0]);
    return (acc[0] + acc[1]) + (acc[2] + acc[3]);
}

// Tile and share of the contraction of a workgroup.  Whole rounds of the chip
// take whole tiles; the tiles left over are cut along the contraction into
// `split` items each, whose partial sums reduce_kernel adds.  Workgroup b runs
// on XCD b % 8: each XCD walks a run of consecutive tiles, four tile rows deep,
// so that the tiles in flight there share their operand rows in its L2 (eight
// rows: 3294 against 3238 us at 32768 x 10496 x 2048, 102 against 97 us at
// 32768 x 2048 x 128; sixteen: 3508 and 125).
constexpr unsigned kTileRows = 4;
__device__ __forceinline__ void tile_of(const SplitGemmParams &p, unsigned u, int *mt, int *nt) {
    const unsigned per = kTileRows * p.ntn, g = u / per;
    const unsigned rows = min(kTileRows, p.ntm - g * kTileRows), v = u - g * per;
    *mt = (int)(g * kTileRows + v % rows);
    *nt = (int)(v / rows);
}

// Exponents of a tile's rows or columns, for the epilogue: kBadRow marks a row
// that the two terms do not represent.
constexpr int kBadRow = 1 << 16;
__device__ __forceinline__ int stat_exp(const SplitStat *st, int64_t r, int64_t n) {
    if (r >= n) return 0;
    const SplitStat s = st[r];
    return row_bad(s) ? kBadRow : row_exp(s.amax) - 15;
}

// Stores one 32 x 32 accumulator tile: lane l holds row m = l % 32 and, in
// groups of four, columns 8 q + 4 (l / 32) + (0..3).  ea: the row's exponent,
// eb: the columns' exponents, from n0.
__device__ __forceinline__ void store_tile(const SplitGemmParams &p, const floatx16 &acc, int64_t m, int64_t n0, int lane,
                                           int ea, const int *eb) {
    if (m >= p.M) return;
    const int cl = 4 * (lane >> 5);
    float *c = p.C + m * p.ldc + n0 + cl;
    const int left = (int)min((int64_t)32, p.N - n0) - cl; // columns of this lane's run
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int4 e4 = *reinterpret_cast<const int4 *>(eb + 8 * q + cl);
        const int e[4] = {ea + e4.x, ea + e4.y, ea + e4.z, ea + e4.w};
        floatx4 v;
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = __builtin_ldexpf(acc[4 * q + j], e[j]);
        if (p.vec_c && 8 * q + 4 <= left && max(max(e[0], e[1]), max(e[2], e[3])) < kBadRow / 2) {
            floatx4 *d = reinterpret_cast<floatx4 *>(c + 8 * q);
            if (p.beta != 0.f) v += p.beta * *d;
            *d = v;
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (8 * q + j < left && e[j] < kBadRow / 2)
                    c[8 * q + j] = p.beta != 0.f ? v[j] + p.beta * c[8 * q + j] : v[j];
        }
    }
}

// The outputs of a tile that the two-term operands do not give.
__device__ __forceinline__ void store_exact(const SplitGemmParams &p, int64_t m0, int64_t n0, int tm, int tn, int tid,
                                            int nthreads) {
    for (int e = tid; e < tm * tn; e += nthreads) {
        const int64_t m = m0 + e / tn, n = n0 + e % tn;
        if (m >= p.M || n >= p.N || !(row_bad(p.sa[m]) || row_bad(p.sb[n]))) continue;
        float *c = p.C + m * p.ldc + n;
        const float v = exact_dot(p, m, n);
        *c = p.beta != 0.f ? v + p.beta * *c : v;
    }
}

// Copies two consecutive fragments (2 KB) from src + lane 16 bytes into LDS at
// dst.  The builtin for global_load_lds would make the compiler wait for all
// copies in flight before each LDS read that could alias them; the kernel
// waits for exactly the stage it reads (vm_wait).  The instruction has no
// destination registers, its offset applies to both addresses, and nothing
// else in the kernel uses m0.
__device__ __forceinline__ void copy_pair(const void *src, unsigned lane16, unsigned dst) {
    asm volatile("s_mov_b32 m0, %0\n\t"
                 "s_nop 0\n\t"
                 "global_load_lds_dwordx4 %1, %2\n\t"
                 "global_load_lds_dwordx4 %1, %2 offset:1024"
                 :
                 : "s"(dst), "v"(lane16), "s"(src)
                 : "memory");
}
template <int N> __device__ __forceinline__ void vm_wait() {
    static_assert(N >= 0 && N < 64, "vmcnt is 6 bits");
    __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14));
}
// leaves vmcnt alone: the copies of later stages stay in flight across it
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_s_waitcnt(0xC07F); // lgkmcnt(0)
    asm volatile("s_barrier" ::: "memory");
}

// A TM x TN tile by WM x WN waves.  At 256 x 256 a wave's 128 x 64 part takes
// 24 matrix instructions (768 cycles) per stage of 16 elements against 12 KB
// of LDS reads, so that LDS is busy two thirds of the time that the cores are;
// the four stages of the ring are 128 KB.  128 x 128 (four waves, 64 KB, two
// workgroups a unit) is for products with too few tiles of 256.
template <int TM, int TN, int WM, int WN>
__global__ __launch_bounds__(64 * WM * WN) void split_gemm_kernel(SplitGemmParams p) {
    constexpr int NW = WM * WN, MT = TM / WM / 32, NT = TN / WN / 32;
    constexpr int FA = 2 * TM / 32, F = 2 * (TM + TN) / 32, PER = F / NW; // fragments a stage, a wave's copies
    constexpr int NS = 4;                                                  // ring of stages
    static_assert(PER == 4 && FA % PER == 0, "each wave copies two row tiles (hi, lo) of one operand");
    __shared__ halfx8 ring[NS][F * kFragH8];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wm = wave / WN, wn = wave % WN;

    const unsigned b = blockIdx.x;
    unsigned u;
    int k0 = 0, k1 = p.KT, item = -1;
    if (b < p.whole) {
        u = (b % 8) * (p.whole / 8) + b / 8; // whole is a multiple of 8
    } else {
        item = (int)(b - p.whole);
        u = p.whole + item / p.split;
        const unsigned s = item % p.split;
        k0 = 2 * (int)((unsigned)(p.KT / 2) * s / p.split);
        k1 = 2 * (int)((unsigned)(p.KT / 2) * (s + 1) / p.split);
    }
    int mt, nt;
    tile_of(p, u, &mt, &nt);

    // this wave's two row tiles (clamped: rows past the operand are not stored)
    const int f0 = wave * PER;
    const bool isa = f0 < FA;
    const int64_t rt0 = isa ? (int64_t)mt * (TM / 32) + f0 / 2 : (int64_t)nt * (TN / 32) + (f0 - FA) / 2;
    const int64_t rtn = isa ? p.rta : p.rtb;
    const halfx8 *base = static_cast<const halfx8 *>(isa ? p.fa : p.fb);
    const halfx8 *s0 = base + min(rt0, rtn - 1) * p.KT * 2 * kFragH8;
    const halfx8 *s1 = base + min(rt0 + 1, rtn - 1) * p.KT * 2 * kFragH8;
    const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) void *)(&ring[0][f0 * kFragH8]);
    auto issue = [&](int k) { // stages past the end repeat the last one into a slot nobody reads
        const int64_t o = (int64_t)min(k, k1 - 1) * 2 * kFragH8;
        const unsigned d = lds0 + ((k - k0) & (NS - 1)) * (F * 1024);
        copy_pair(s0 + o, lane * 16, d);
        copy_pair(s1 + o, lane * 16, d + 2048);
    };
    struct Ops {
        halfx8 a[MT][2], b[NT][2];
    };
    auto fetch = [&](int k, Ops &o) {
        const halfx8 *r = ring[(k - k0) & (NS - 1)];
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int h = 0; h < 2; ++h) o.b[j][h] = r[(FA + 2 * (wn * NT + j) + h) * kFragH8 + lane];
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int h = 0; h < 2; ++h) o.a[i][h] = r[(2 * (wm * MT + i) + h) * kFragH8 + lane];
    };
    floatx16 acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
    auto products = [&](const Ops &o) {
#pragma unroll
        for (int i = 0; i < MT; ++i) {
#pragma unroll
            for (int j = 0; j < NT; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(o.b[j][0], o.a[i][0], acc[i][j], 0, 0, 0);
#pragma unroll
            for (int j = 0; j < NT; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(o.b[j][1], o.a[i][0], acc[i][j], 0, 0, 0);
#pragma unroll
            for (int j = 0; j < NT; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(o.b[j][0], o.a[i][1], acc[i][j], 0, 0, 0);
        }
    };
    // Stage k + 1's operands are read from LDS and stage k + 3's copied into
    // it while stage k's products run; at the end of stage k every wave's
    // copies of stage k + 2 have landed (the four of k + 3 may still fly).
    // one LDS read every two products, none of them waited for until the next stage
    auto interleave = [&]() {
#pragma unroll
        for (int i = 0; i < 2 * (MT + NT); ++i) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
        __builtin_amdgcn_sched_group_barrier(0x008, 3 * MT * NT - 2 * (MT + NT), 0);
    };
    Ops x, y;
    issue(k0);
    issue(k0 + 1);
    issue(k0 + 2);
    vm_wait<4>();
    lds_barrier();
    fetch(k0, x);
    for (int k = k0; k < k1; k += 2) {
        issue(k + 3);
        fetch(k + 1, y);
        products(x);
        interleave();
        vm_wait<4>();
        lds_barrier();
        issue(k + 4);
        fetch(k + 2, x);
        products(y);
        interleave();
        vm_wait<4>();
        lds_barrier();
    }

    const int64_t m0 = (int64_t)mt * TM, n0 = (int64_t)nt * TN;
    if (item >= 0 && p.split > 1) { // partial sums, in accumulator order
        floatx4 *w = reinterpret_cast<floatx4 *>(p.part) + ((int64_t)item * NW + wave) * MT * NT * 4 * 64 + lane;
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j)
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    w[((i * NT + j) * 4 + q) * 64] = floatx4{acc[i][j][4 * q], acc[i][j][4 * q + 1],
                                                             acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
        return;
    }
    // the copies past the last stage have landed, and nobody reads the ring any more
    vm_wait<0>();
    lds_barrier();
    int *ex = reinterpret_cast<int *>(&ring[0][0]); // exponents of the tile's rows, then of its columns
    bool bad = false;
    for (int i = tid; i < TM + TN; i += 64 * NW) {
        ex[i] = i < TM ? stat_exp(p.sa, m0 + i, p.M) : stat_exp(p.sb, n0 + i - TM, p.N);
        bad |= ex[i] == kBadRow;
    }
    const bool any_bad = __syncthreads_or(bad);
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            const int lm = (wm * MT + i) * 32 + (lane & 31), ln = (wn * NT + j) * 32;
            store_tile(p, acc[i][j], m0 + lm, n0 + ln, lane, ex[lm], ex + TM + ln);
            __builtin_amdgcn_sched_barrier(0);
        }
    if (any_bad) store_exact(p, m0, n0, TM, TN, tid, 64 * NW);
}

template <int TM, int TN, int WM, int WN>
__global__ __launch_bounds__(64 * WM * WN) void reduce_kernel(SplitGemmParams p) {
    constexpr int NW = WM * WN, MT = TM / WM / 32, NT = TN / WN / 32;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, wm = wave / WN, wn = wave % WN;
    int mt, nt;
    tile_of(p, p.whole + blockIdx.x, &mt, &nt);
    const int64_t m0 = (int64_t)mt * TM, n0 = (int64_t)nt * TN;
    // grid.y: one 32 x 32 tile of each wave
    const int t = blockIdx.y, i = t / NT, j = t % NT;
    const floatx4 *w = reinterpret_cast<const floatx4 *>(p.part) +
                       (((int64_t)blockIdx.x * p.split * NW + wave) * MT * NT + t) * 4 * 64 + lane;
    floatx16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.f;
    for (unsigned s = 0; s < p.split; ++s)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const floatx4 v = w[(int64_t)s * NW * MT * NT * 4 * 64 + q * 64];
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[4 * q + r] += v[r];
        }
    const int64_t mb = m0 + (wm * MT + i) * 32, nb = n0 + (wn * NT + j) * 32;
    __shared__ int ex[NW][64]; // the tile's 32 rows, then its 32 columns
    const int e = lane < 32 ? stat_exp(p.sa, mb + lane, p.M) : stat_exp(p.sb, nb + lane - 32, p.N);
    ex[wave][lane] = e;
    __syncthreads();
    store_tile(p, acc, mb + (lane & 31), nb, lane, ex[wave][lane & 31], &ex[wave][32]);
    if (__any(e == kBadRow)) store_exact(p, mb, nb, 32, 32, lane, 64);
}

template <int TM, int TN, int WM, int WN> hipError_t launch_t(SplitGemmParams p, hipStream_t s) {
    const unsigned rest = p.ntm * p.ntn - p.whole;
    hipLaunchKernelGGL((split_gemm_kernel<TM, TN, WM, WN>), dim3(p.whole + rest * p.split), dim3(64 * WM * WN),
                       0, s, p);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || rest == 0 || p.split == 1) return e;
    hipLaunchKernelGGL((reduce_kernel<TM, TN, WM, WN>), dim3(rest, (TM / WM / 32) * (TN / WN / 32)),
                       dim3(64 * WM * WN), 0, s, p);
    return hipGetLastError();
}

// Stages of a contraction: whole 32-element pairs, so that the product loop
// takes two stages a turn.
int64_t stages(int64_t Kd) { return 2 * ((Kd + 2 * kFragK - 1) / (2 * kFragK)); }

size_t up256(size_t n) { return (n + 255) & ~(size_t)255; }

}  // namespace

size_t split_frag_bytes(int64_t rows, int64_t Kd) {
    const int64_t rt = (rows + kFragRows - 1) / kFragRows;
    return up256((size_t)(rt * stages(Kd)) * 2 * kFragH8 * sizeof(halfx8));
}
size_t split_stat_bytes(int64_t rows) { return up256(sizeof(SplitStat) * (size_t)((rows + 31) / 32 * 32)); }

hipError_t launch_split(const float *src, int64_t ld, bool trans, int64_t rows, int64_t Kd, void *frags, SplitStat *stat,
                        hipStream_t s) {
    const int64_t KT = stages(Kd), rpad = (rows + 31) / 32 * 32;
    if (!trans) {
        const bool vec = reinterpret_cast<uintptr_t>(src) % 16 == 0 && ld % 4 == 0;
        const dim3 grid((unsigned)(rpad / 8));
        if (Kd <= 1024)
            hipLaunchKernelGGL(split_rows_kernel<4>, grid, dim3(256), 0, s, src, ld, rows, Kd, KT, vec,
                               static_cast<halfx8 *>(frags), stat);
        else
            hipLaunchKernelGGL(split_rows_kernel<8>, grid, dim3(256), 0, s, src, ld, rows, Kd, KT, vec,
                               static_cast<halfx8 *>(frags), stat);
        return hipGetLastError();
    }
    hipLaunchKernelGGL(stat_clear_kernel, dim3((unsigned)((rpad + 255) / 256)), dim3(256), 0, s, stat, rpad);
    // about four workgroups a compute unit each, of at least 64 rows
    const auto share = [&](int64_t cols) {
        const int64_t blocks = std::max<int64_t>(1, 1024 / cols);
        return std::max<int64_t>(64, ((Kd + blocks - 1) / blocks + 63) / 64 * 64);
    };
    const int64_t cb = (rows + 255) / 256, mp = share(cb);
    hipLaunchKernelGGL(col_max_kernel, dim3((unsigned)cb, (unsigned)((Kd + mp - 1) / mp)), dim3(256), 0, s, src, ld,
                       rows, Kd, mp, stat);
    const int64_t sb = (rows + 63) / 64, sp = share(sb);
    hipLaunchKernelGGL(split_cols_kernel, dim3((unsigned)sb, (unsigned)((KT * kFragK + sp - 1) / sp)), dim3(256), 0, s,
                       src, ld, rows, Kd, KT, sp, static_cast<halfx8 *>(frags), stat);
    return hipGetLastError();
}

size_t plan_split_gemm(SplitGemmParams *p) {
    p->KT = (int)stages(p->Kd);
    p->rta = (p->M + 31) / 32;
    p->rtb = (p->N + 31) / 32;
    const auto tiles = [&](int t) { return ((p->M + t - 1) / t) * ((p->N + t - 1) / t); };
    // 256 x 256 tiles, one workgroup a compute unit, once they fill the chip
    // at least once; 128 x 128, two a unit, below
    p->tile = tiles(256) >= 192 ? 256 : 128;
    const int64_t slots = p->tile == 256 ? 256 : 512, T = tiles(p->tile);
    p->ntm = (unsigned)((p->M + p->tile - 1) / p->tile);
    p->ntn = (unsigned)((p->N + p->tile - 1) / p->tile);
    const int64_t whole = T / slots * slots, rest = T - whole;
    p->whole = (unsigned)whole;
    // the tiles left over: cut along the contraction to fill one more round,
    // in shares of at least 8 stages
    p->split = rest ? (unsigned)std::max<int64_t>(1, std::min<int64_t>(slots / rest, p->KT / 8)) : 1;
    return p->split > 1 ? sizeof(float) * (size_t)(rest * p->split) * p->tile * p->tile : 0;
}

hipError_t launch_split_gemm(const SplitGemmParams &p, hipStream_t s) {
    return p.tile == 256 ? launch_t<256, 256, 2, 4>(p, s) : launch_t<128, 128, 2, 2>(p, s);
}

}  // namespace gdn2
