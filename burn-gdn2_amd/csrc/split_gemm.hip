// Row-major f32 matrix products on the f16 matrix cores: C (+)= op(A) op(B)
// with every f32 operand written as two f16 terms,
//   x 2^s = hi + lo,  hi = f16(x 2^s),  lo = f16(x 2^s - hi),
// and hi hi + hi lo + lo hi accumulated in f32 (lo lo is below 2^-22 of a
// product).  s is chosen per row of op(A) and per column of op(B) so that the
// largest element lies in [2^14, 2^15): hi + lo then carries 23 bits of every
// element down to 2^-17 of its row's largest and an absolute error of 2^-40
// of it below that.
//
// What such small elements lose is checked for each output.  Splitting adds up
// the row's remainders |x 2^s - hi - lo| of elements below 2^-17 of its largest
// (SplitStat::lost, r); the other operand's elements are below 2^15, so an
// output's error from them is at most 2^15 (r_m + r_n) in the accumulator's
// units.  An output whose accumulator is not 2^18 times that is formed again
// from the f32 operands, with all their digits (redo_kernel).  The others have an error of at
// most 2^-18 of themselves from this, if all remainders were largest and of the
// sign that hurts (the bound of an f32 sum of 64 terms; it is about the square
// root of their number less), and of 2^-21 sum |x| |w| from the terms' 23 bits.
// Rows with an infinity or a NaN always fail the check.  Ordinary rows lose
// nothing or one element's 2^-26, which no output but one cancelled to 2^-23 of
// its size notices; rows of channels of sizes 2^17 and more apart, read by
// weights that fold or ignore that, fail it throughout.
//
// Bound: the f16 matrix cores, three products of 2 M N K (a third of 2.5
// PFLOP/s; the same products cost 157 TFLOP/s at most as f32 ones).  Measured,
// M x N x K: 32768 x 10496 x 2048 3.24 ms, 434 TFLOP/s of f32 product (1.30
// PFLOP/s of f16, where hipBLASLt's f16 kernel runs the same amount at 1.38),
// against 9.45 ms (149) by hipBLASLt in f32; 8192 x 2048 x 10496 0.79 against
// 2.31 ms; 2048 x 10496 x 8192 0.82 against 3.08 ms.  Relative error against
// f64 (2-norm) at K = 2048: 5.1e-7, where the f32 product's is 8.1e-7 (four
// times more roundings of the running sum).
#include "split_gemm.hpp"

#include "common.hpp"

namespace gdn2 {
namespace {

typedef _Float16 halfx8 __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

constexpr int kFragRows = 32, kFragK = 16; // one MFMA 32x32x16 operand: 64 lanes x 8 f16 = 1 KB
constexpr int kFragH8 = 64;                // halfx8 per fragment

// Elements below kSmall = 2^-17 of a row's largest, in its scale, lose what lies
// below f16's 2^-24; what they lose is counted in units of 2^-36 (rounded up,
// whole numbers so that the sum's order does not matter; a row of 2^20 elements
// stays below 2^32).  kLeast: the smallest accumulator that passes, a unit.
constexpr float kSmall = 0x1p-2f, kLostUnit = 0x1p36f, kLeast = 0x1p-3f; // 2^18 x 2^15 x 2^-36
// x = m 2^e with m in [1/2, 1): the split multiplies by 2^(15 - e)
__device__ __forceinline__ int row_exp(unsigned amax) {
    return amax == 0 || amax >= 0x7F800000u ? 15 : __builtin_amdgcn_frexp_expf(__builtin_bit_cast(float, amax));
}
__device__ __forceinline__ unsigned abs_bits(float x) { return __builtin_bit_cast(unsigned, x) & 0x7FFFFFFFu; }

// Splits eight elements; returns what they lose.
__device__ __forceinline__ unsigned split8(const float *x, int sh, halfx8 *hi, halfx8 *lo) {
    unsigned lost = 0;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const float s = __builtin_ldexpf(x[j], sh);
        const _Float16 h = (_Float16)s;
        const float r = s - (float)h;
        const _Float16 l = (_Float16)r;
        (*hi)[j] = h;
        (*lo)[j] = l;
        const unsigned u = (unsigned)(__builtin_fabsf(r - (float)l) * kLostUnit) + 1u;
        lost += x[j] != 0.f && __builtin_fabsf(s) < kSmall ? u : 0u;
    }
    return lost;
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
    __shared__ unsigned red[2][4][8];
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
    unsigned lost = 0;
    // fragment of this row: (row / 32, g / 2), lane (row % 32) + 32 (g % 2)
    halfx8 *d = dst + (row / kFragRows) * KT * 2 * kFragH8 + row % kFragRows;
    auto put = [&](const float *y, int64_t g) {
        halfx8 hi, lo;
        lost += split8(y, 15 - e, &hi, &lo);
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
    for (int o = 8; o < 64; o <<= 1) lost += __shfl_xor((int)lost, o, 64);
    if (lane < 8) red[1][wave][r8] = lost;
    __syncthreads();
    if (wave == 0 && lane < 8)
        stat[row] = SplitStat{mx, red[1][0][r8] + red[1][1][r8] + red[1][2][r8] + red[1][3][r8]};
}

__global__ __launch_bounds__(256) void stat_clear_kernel(SplitStat *stat, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n) stat[i] = SplitStat{0, 0};
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
// fragments of each; a thread's column is the same in all of them, so what the
// column loses is added to its record once at the end.
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
    unsigned lost = 0;
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
            for (int j = 0; j < 8; ++j) y[j] = t[kk + j][cc];
            halfx8 hi, lo;
            lost += split8(y, sh, &hi, &lo);
            halfx8 *f = dst + (rt * KT + kt) * 2 * kFragH8 + lane;
            f[0] = hi;
            f[kFragH8] = lo;
        }
    }
    lost += __shfl_xor((int)lost, 32, 64);
    if (lane < 32 && row < R && lost) atomicAdd(&stat[row].lost, lost);
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

// A row's or column's record for the epilogue: its exponent, and the smallest
// accumulator that its lost remainders allow (NaN, which no accumulator passes,
// for an infinity or a NaN).
struct RowInfo {
    int e;
    float least;
};
__device__ __forceinline__ RowInfo row_info(const SplitStat *st, int64_t r, int64_t n) {
    if (r >= n) return RowInfo{0, 0.f};
    const SplitStat s = st[r];
    return RowInfo{row_exp(s.amax) - 15, s.amax >= 0x7F800000u ? __builtin_nanf("") : (float)s.lost * kLeast};
}

__device__ __forceinline__ void put(const SplitGemmParams &p, float *c, float v) {
    *c = p.beta != 0.f ? v + p.beta * *c : v;
}

// A 32 x 32 accumulator tile: lane l holds row m = l % 32 and, in groups of
// four, columns 8 q + 4 (l / 32) + (0..3).  Its outputs that fail the check (bit
// 4 q + j); a: the row's record, b: the columns', from n0.
__device__ __forceinline__ unsigned check_tile(const SplitGemmParams &p, const floatx16 &acc, int64_t m, int64_t n0,
                                               int lane, RowInfo a, const RowInfo *b) {
    const int cl = 4 * (lane >> 5), left = m < p.M ? (int)min((int64_t)32, p.N - n0) - cl : 0;
    unsigned failed = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
            failed |= !(__builtin_fabsf(acc[4 * q + j]) >= a.least + b[8 * q + cl + j].least) && 8 * q + j < left
                          ? 1u << (4 * q + j) : 0u;
        __builtin_amdgcn_sched_barrier(0); // four columns' records at a time in registers
    }
    return failed;
}
// Stores its outputs but those of `skip`, times 2^(ea + eb).
__device__ __forceinline__ void store_tile(const SplitGemmParams &p, const floatx16 &acc, int64_t m, int64_t n0, int lane,
                                           int ea, const RowInfo *b, unsigned skip) {
    if (m >= p.M) return;
    const int cl = 4 * (lane >> 5);
    float *c = p.C + m * p.ldc + n0 + cl;
    const int left = (int)min((int64_t)32, p.N - n0) - cl; // columns of this lane's run
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        floatx4 v;
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = __builtin_ldexpf(acc[4 * q + j], ea + (b ? b[8 * q + cl + j].e : 0));
        if (p.vec_c && 8 * q + 4 <= left && !(skip >> (4 * q) & 15)) {
            floatx4 *d = reinterpret_cast<floatx4 *>(c + 8 * q);
            if (p.beta != 0.f) v += p.beta * *d;
            *d = v;
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (8 * q + j < left && !(skip >> (4 * q + j) & 1)) put(p, c + 8 * q + j, v[j]);
        }
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
        if (item % p.split == 0 && tid < 8) p.redo[u * 8 + tid] = 0;
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
    RowInfo *info = reinterpret_cast<RowInfo *>(&ring[0][0]); // of the tile's rows, then of its columns
    unsigned *failed = reinterpret_cast<unsigned *>(info + TM + TN) + wave * MT * NT * 64 + lane; // outputs to redo
    bool losses = false;
    unsigned flags = 0; // this wave's parts left to redo_kernel
    for (int i = tid; i < TM + TN; i += 64 * NW) {
        info[i] = i < TM ? row_info(p.sa, m0 + i, p.M) : row_info(p.sb, n0 + i - TM, p.N);
        losses |= !(info[i].least == 0.f);
    }
#pragma unroll
    for (int t = 0; t < MT * NT; ++t) failed[t * 64] = 0;
    if (__syncthreads_or(losses)) {
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j) {
                const int lm = (wm * MT + i) * 32 + (lane & 31), ln = (wn * NT + j) * 32;
                const unsigned f = check_tile(p, acc[i][j], m0 + lm, n0 + ln, lane, info[lm], info + TM + ln);
                failed[(i * NT + j) * 64] = f;
                if (__any(f != 0)) {
                    p.failed[((u * NW + wave) * MT * NT + i * NT + j) * 64 + lane] = (unsigned short)f;
                    flags |= 1u << (i * NT + j);
                }
            }
    }
    if (lane == 0) p.redo[u * 8 + wave] = (unsigned char)flags;
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            const int lm = (wm * MT + i) * 32 + (lane & 31), ln = (wn * NT + j) * 32;
            store_tile(p, acc[i][j], m0 + lm, n0 + ln, lane, info[lm].e, info + TM + ln, failed[(i * NT + j) * 64]);
            __builtin_amdgcn_sched_barrier(0);
        }
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
    __shared__ RowInfo info[NW][64]; // the tile's 32 rows, then its 32 columns
    const RowInfo own = lane < 32 ? row_info(p.sa, mb + lane, p.M) : row_info(p.sb, nb + lane - 32, p.N);
    info[wave][lane] = own;
    unsigned failed = 0;
    if (__syncthreads_or(!(own.least == 0.f))) {
        failed = check_tile(p, acc, mb + (lane & 31), nb, lane, info[wave][lane & 31], &info[wave][32]);
        if (__any(failed != 0)) { // left to redo_kernel
            const unsigned u = p.whole + blockIdx.x, byte = u * 8 + wave;
            p.failed[((u * NW + wave) * MT * NT + t) * 64 + lane] = (unsigned short)failed;
            if (lane == 0) atomicOr(reinterpret_cast<unsigned *>(p.redo) + byte / 4, 1u << (byte % 4 * 8 + t));
        }
    }
    store_tile(p, acc, mb + (lane & 31), nb, lane, info[wave][lane & 31].e, &info[wave][32], failed);
}

// The outputs that fail the check, from the f32 operands: bit t of p.redo[8 u + w]
// stands for part t of wave w of tile u (as the product kernel shares them out)
// with such outputs, which p.failed notes.  A workgroup of 2 x 2 waves takes a
// block of 128 x 128: a few of its outputs by f32 sums, else all of them with
// every operand as three bf16 terms
//   h = bf16(x),  m = bf16(x - h),  l = bf16(x - h - m),
// whose sum is x exactly, without a scale, and hh + hm + mh + mm + hl + lh in f32
// accumulators (the rest is below 2^-25 of a product).  An infinity goes into l
// alone, which meets the other operand's h alone, so that it gives what an f32
// product gives (a NaN where both operands are infinite); h is kept finite.
// 16 elements of the contraction a stage, two stages in LDS as fragments (a
// lane's eight elements in one place: lanes 0-31 of a row tile hold the first
// eight of their row, 32-63 the others), the loads of the two stages after them
// in registers: what bounds it is those loads' latency.
// Measured, layer training step of 4 x 2048 tokens, hidden 2048 (6.2 ms where
// nothing fails, 11.1 with f32 products throughout): a loss on the last token of
// each sequence 10.0 ms, with strong decays 10.9 (its 2048 x 10496 x 8192
// redone in 2.1-2.8 ms), a NaN token 10.7; a thread summing each output instead
// took 180 to 530.  5-14 us where next to nothing fails, 34 and 72 for two products
// of an ordinary backward of that layer.
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
constexpr int kRedoGrid = 512; // two workgroups a unit
template <int TM, int TN, int WM, int WN> __global__ __launch_bounds__(256, 2) void redo_kernel(SplitGemmParams p) {
    constexpr int NW = WM * WN, MT = TM / WM / 32, NT = TN / WN / 32; // of the product kernel
    constexpr int NB = TM / 128;                                     // blocks a tile side
    static_assert(TM == TN && NW <= 8 && MT * NT <= 8, "flags");
    __shared__ floatx4 lds[2][8][3][64]; // stage, row tiles of op(A) then of op(B), terms (or halves of eight)
    __shared__ unsigned few[32];         // local row and column of the outputs to sum
    __shared__ int count;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wm = wave >> 1, wn = wave & 1;
    const unsigned blocks = p.ntm * p.ntn * NB * NB;
    // A sum over rows reads 8 Kd bytes; over columns a cache line for each of 2 Kd
    // elements, so that four read what a block's products do
    const int max_few = p.ta || !p.tb ? 4 : 32;
    const bool vec_a = !p.ta && reinterpret_cast<uintptr_t>(p.A) % 16 == 0 && p.lda % 4 == 0;
    const bool vec_b = p.tb && reinterpret_cast<uintptr_t>(p.B) % 16 == 0 && p.ldb % 4 == 0;
    // row tile r and column tile c of a tile: the product kernel's wave and part
    auto wave_of = [](int r, int c) { return r / MT * WN + c / NT; };
    auto part_of = [](int r, int c) { return r % MT * NT + c % NT; };
    auto flags_of = [&](unsigned b) { // the 4 x 4 parts of block b
        unsigned long long f = 0;
        if (b < blocks) f = reinterpret_cast<const unsigned long long *>(p.redo)[b / (NB * NB)];
        const int q = b % (NB * NB), r0 = 4 * (q / NB), c0 = 4 * (q % NB);
        unsigned w = 0;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int r = r0 + i / 4, c = c0 + i % 4;
            w |= (unsigned)(f >> (8 * wave_of(r, c) + part_of(r, c)) & 1) << i;
        }
        return w;
    };
    for (unsigned first = blockIdx.x; first < blocks; first += 64 * kRedoGrid) {
        const unsigned mine = flags_of(first + lane * kRedoGrid);
        for (unsigned long long left = __ballot(mine != 0); left; left &= left - 1) {
            const int which = __ffsll(left) - 1;
            const unsigned b = first + which * kRedoGrid, u = b / (NB * NB), flags = __shfl((int)mine, which, 64);
            int mt, nt;
            tile_of(p, u, &mt, &nt);
            const int q = b % (NB * NB), r0 = 4 * (q / NB), c0 = 4 * (q % NB);
            const int64_t m0 = (int64_t)mt * TM + 32 * r0, n0 = (int64_t)nt * TN + 32 * c0;
            const int kd = (int)p.Kd; // (split products have at most 2^20)
            // the failed outputs of part (i, j) of this wave's 64 x 64
            auto failed_of = [&](int i, int j) -> unsigned {
                const int r = r0 + 2 * wm + i, c = c0 + 2 * wn + j;
                if (!(flags >> ((2 * wm + i) * 4 + 2 * wn + j) & 1)) return 0;
                return p.failed[((u * NW + wave_of(r, c)) * MT * NT + part_of(r, c)) * 64 + lane];
            };
            if (tid == 0) count = 0;
            __syncthreads(); // (and every wave is done with the block before)
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    for (unsigned f = failed_of(i, j); f; f &= f - 1) {
                        const int e = __ffs(f) - 1, at = atomicAdd(&count, 1);
                        const int lm = (2 * wm + i) * 32 + (lane & 31);
                        const int ln = (2 * wn + j) * 32 + 8 * (e >> 2) + 4 * (lane >> 5) + (e & 3);
                        if (at < 32) few[at] = lm << 16 | ln;
                    }
            __syncthreads();
            const int total = count;
            if (total <= max_few) {
                for (int i = wave; i < total; i += 4) { // a wave an output
                    const int64_t m = m0 + (few[i] >> 16), n = n0 + (few[i] & 0xFFFF);
                    const int64_t ka = p.ta ? p.lda : 1, kb = p.tb ? 1 : p.ldb;
                    const float *a = p.A + (p.ta ? m : m * p.lda) + lane * ka, *c = p.B + (p.tb ? n * p.ldb : n) + lane * kb;
                    float sum = 0.f;
#pragma unroll 8
                    for (int k = lane; k < kd; k += 64, a += 64 * ka, c += 64 * kb) sum = __builtin_fmaf(*a, *c, sum);
                    sum = wave_sum(sum);
                    if (lane == 0) put(p, p.C + m * p.ldc + n, sum);
                }
                continue;
            }
            float xs[2][2][8];
            auto load = [&](int k0, float (&x)[2][8]) { // waves 0-3: row tiles 0-3 of op(A), then of op(B)
                const int k = k0 + 8 * (lane >> 5);
#pragma unroll
                for (int u2 = 0; u2 < 2; ++u2) {
                    const bool trans = u2 ? !p.tb : p.ta;
                    const int64_t r = 32 * wave + (lane & 31), row = u2 ? min(n0 + r, p.N - 1) : min(m0 + r, p.M - 1);
                    const unsigned ld = (unsigned)(u2 ? p.ldb : p.lda), sk = trans ? ld : 1;
                    const float *src = (u2 ? p.B : p.A) + (trans ? row : row * ld);
                    if ((u2 ? vec_b : vec_a) && k0 + 16 <= kd) { // a row's elements as vectors
                        const floatx4 v0 = *reinterpret_cast<const floatx4 *>(src + k);
                        const floatx4 v1 = *reinterpret_cast<const floatx4 *>(src + k + 4);
#pragma unroll
                        for (int j = 0; j < 4; ++j) {
                            x[u2][j] = v0[j];
                            x[u2][4 + j] = v1[j];
                        }
                        continue;
                    }
#pragma unroll
                    for (int j = 0; j < 8; ++j) { // loads without branches: past the end the last element, dropped
                        const float v = src[(uint64_t)(unsigned)min(k + j, kd - 1) * sk];
                        x[u2][j] = k + j < kd ? v : 0.f;
                    }
                }
            };
            floatx16 acc[2][2];
            auto stage = [&](int buf, const float (&x)[2][8]) {
                constexpr float kMost = 0x1.FEp127f; // bf16's largest
#pragma unroll
                for (int u2 = 0; u2 < 2; ++u2) {
                    bf16x8 v[3];
#pragma unroll
                    for (int j = 0; j < 8; j += 2) {
                        floatx2 r = {x[u2][j], x[u2][j + 1]};
                        const bool inf0 = __builtin_isinf(r[0]), inf1 = __builtin_isinf(r[1]);
                        r = floatx2{inf0 ? 0.f : r[0], inf1 ? 0.f : r[1]};
#pragma unroll
                        for (int t = 0; t < 3; ++t) {
                            floatx2 y = r;
                            if (t == 0) // (a NaN becomes a number here and stays in the remainder)
                                y = floatx2{__builtin_amdgcn_fmed3f(r[0], -kMost, kMost), __builtin_amdgcn_fmed3f(r[1], -kMost, kMost)};
                            if (t == 2) y = floatx2{inf0 ? x[u2][j] : r[0], inf1 ? x[u2][j + 1] : r[1]};
                            const bf16x2 h = __builtin_convertvector(y, bf16x2);
                            v[t][j] = h[0];
                            v[t][j + 1] = h[1];
                            r = floatx2{r[0] - (float)h[0], r[1] - (float)h[1]};
                        }
                    }
#pragma unroll
                    for (int t = 0; t < 3; ++t) lds[buf][4 * u2 + wave][t][lane] = __builtin_bit_cast(floatx4, v[t]);
                }
            };
            auto products = [&](int buf) {
                bf16x8 a[2][3], c[2][3];
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int t = 0; t < 3; ++t) {
                        a[i][t] = __builtin_bit_cast(bf16x8, lds[buf][2 * wm + i][t][lane]);
                        c[i][t] = __builtin_bit_cast(bf16x8, lds[buf][4 + 2 * wn + i][t][lane]);
                    }
                constexpr int ta[6] = {2, 0, 1, 1, 0, 0}, tb[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
                for (int e = 0; e < 6; ++e)
#pragma unroll
                    for (int i = 0; i < 2; ++i)
#pragma unroll
                        for (int j = 0; j < 2; ++j)
                            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(c[j][tb[e]], a[i][ta[e]], acc[i][j], 0, 0, 0);
            };
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
            load(0, xs[0]);
            stage(0, xs[0]);
            load(16, xs[1]);
            __syncthreads();
            for (int k0 = 0; k0 < kd; k0 += 32) { // (past the end: zeros)
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    load(k0 + 16 * h + 32, xs[h]); // two stages ahead
                    __builtin_amdgcn_sched_barrier(0);
                    products(h);
                    stage(h ^ 1, xs[h ^ 1]);
                    __syncthreads();
                }
            }
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const unsigned f = failed_of(i, j);
                    if (__any(f != 0))
                        store_tile(p, acc[i][j], m0 + (2 * wm + i) * 32 + (lane & 31), n0 + (2 * wn + j) * 32, lane, 0,
                                   nullptr, ~f);
                }
        }
    }
}

template <int TM, int TN, int WM, int WN> hipError_t launch_t(SplitGemmParams p, hipStream_t s) {
    const unsigned rest = p.ntm * p.ntn - p.whole;
    hipLaunchKernelGGL((split_gemm_kernel<TM, TN, WM, WN>), dim3(p.whole + rest * p.split), dim3(64 * WM * WN),
                       0, s, p);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess && rest > 0 && p.split > 1) {
        hipLaunchKernelGGL((reduce_kernel<TM, TN, WM, WN>), dim3(rest, (TM / WM / 32) * (TN / WN / 32)),
                           dim3(64 * WM * WN), 0, s, p);
        e = hipGetLastError();
    }
    if (e != hipSuccess) return e;
    const unsigned blocks = p.ntm * p.ntn * (TM / 128) * (TN / 128);
    hipLaunchKernelGGL((redo_kernel<TM, TN, WM, WN>), dim3(std::min<unsigned>(blocks, kRedoGrid)), dim3(256), 0, s, p);
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
void split_redo_bytes(const SplitGemmParams &p, size_t *flags, size_t *failed) {
    const size_t tiles = (size_t)p.ntm * p.ntn;
    *flags = up256(8 * tiles);
    *failed = up256(tiles * p.tile * p.tile / 8);
}

hipError_t launch_split_gemm(const SplitGemmParams &p, hipStream_t s) {
    return p.tile == 256 ? launch_t<256, 256, 2, 4>(p, s) : launch_t<128, 128, 2, 2>(p, s);
}

}  // namespace gdn2
