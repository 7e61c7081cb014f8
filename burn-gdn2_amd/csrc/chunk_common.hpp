// Device helpers shared by the chunked forward (chunk.hip) and backward
// (chunk_bwd.hip) kernels: chunk geometry, MFMA fragment helpers, the
// range-checked row loads and the XCD-aware workgroup mapping.
#pragma once

#include "common.hpp"
#include "kernels.hpp"

namespace gdn2 {

constexpr int C = kChunk;   // chunk length of the kernels
constexpr int NT = C / 16;  // 16-row tiles per chunk

// Waves per workgroup of the sequential kernels (each wave owns 16 value
// columns): four when V and K are multiples of 64, else two (V = 32, 96 and
// K = 32, whose segment transitions P have 32 columns).
constexpr int inter_nwv(int K, int V) { return (V % 64 == 0 && K % 64 == 0) ? 4 : 2; }

// Rows [0, valid) of a row-strided f32 matrix (row stride rs, rowlen
// elements used per row) as a buffer resource.  The hardware's range check
// returns 0 for every load past the last valid row, which is the zero padding
// of a ragged last chunk (src/forward.rs:94-99), so a load needs neither a
// clamp nor a mask, and its offset is a 32-bit element index.  Requires
// rs >= rowlen and ((valid - 1) rs + rowlen) * 4 < 2^31 (checked on the host).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rows_rsrc(const float *base, int rs, int valid, int rowlen) {
    const int bytes = ((valid - 1) * rs + rowlen) * 4;
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(base), (short)0, bytes, 0x00020000);
}

__device__ __forceinline__ float bld1(__amdgpu_buffer_rsrc_t r, int idx) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, idx * 4, 0, 0));
}

// A store through a rows_rsrc resource: dropped past its last valid row.
__device__ __forceinline__ void bst1(__amdgpu_buffer_rsrc_t r, int idx, float v) {
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(int, v), r, idx * 4, 0, 0);
}

__device__ __forceinline__ floatx4 bld4(__amdgpu_buffer_rsrc_t r, int idx) {
    return __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(r, idx * 4, 0, 0));
}
// 16 bytes through a rows_rsrc resource (idx a multiple of 4 within a row):
// dropped past its last valid row.
__device__ __forceinline__ void bst4(__amdgpu_buffer_rsrc_t r, int idx, floatx4 v) {
    typedef int intx4 __attribute__((ext_vector_type(4)));
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(intx4, v), r, idx * 4, 0, 0);
}

__device__ __forceinline__ floatx4 mfma4(float4 a, floatx4 b, floatx4 c) {
    c = mfma16(a.x, b[0], c);
    c = mfma16(a.y, b[1], c);
    c = mfma16(a.z, b[2], c);
    c = mfma16(a.w, b[3], c);
    return c;
}

// D = X^T for an accumulator tile X, i.e. the A-operand layout of X
// (lane (g, r) gets X[r][4g..4g+3]): the accumulator is a valid A operand
// of X^T under the k = 4g + step labelling, multiplied by the identity.
// Exact in f32 (products with 1 and 0).
__device__ __forceinline__ floatx4 transpose16(floatx4 x, int lr, int lg) {
    floatx4 d = floatx4{0.f, 0.f, 0.f, 0.f};
    d = mfma16(x[0], lr == 4 * lg + 0 ? 1.f : 0.f, d);
    d = mfma16(x[1], lr == 4 * lg + 1 ? 1.f : 0.f, d);
    d = mfma16(x[2], lr == 4 * lg + 2 ? 1.f : 0.f, d);
    d = mfma16(x[3], lr == 4 * lg + 3 ? 1.f : 0.f, d);
    return d;
}

__device__ __forceinline__ floatx4 mfma4n(float4 a, floatx4 b, floatx4 c) {
    c = mfma16(-a.x, b[0], c);
    c = mfma16(-a.y, b[1], c);
    c = mfma16(-a.z, b[2], c);
    c = mfma16(-a.w, b[3], c);
    return c;
}

// Streaming store: the workspace is read back by chunk-inter much later, so
// keeping it out of L2 leaves room for the chunk's inputs, which chunk-intra
// reads more than once.
__device__ __forceinline__ void st_stream(floatx4 *dst, floatx4 v) { __builtin_nontemporal_store(v, dst); }

// Pins a loaded value in a register where it is loaded: the compiler would
// otherwise sink a load used only under a lane condition into a divergent
// branch with its own wait, serialising the loads of an unrolled loop.
__device__ __forceinline__ float pin(float x) {
    asm volatile("" : "+v"(x));
    return x;
}
__device__ __forceinline__ float2 pin(float2 x) {
    asm volatile("" : "+v"(x.x), "+v"(x.y));
    return x;
}

__device__ __forceinline__ floatx4 exp2v(floatx4 x) {
    return floatx4{fast_exp2(x[0]), fast_exp2(x[1]), fast_exp2(x[2]), fast_exp2(x[3])};
}

// The two steps of a 4 x 4 transpose among the four lanes of a quad, whose
// lane i holds row i (elements 0 .. 3): afterwards lane i holds column i.
// Step 1, partner i ^ 2 (dpp quad_perm [2, 3, 0, 1]): the lower two lanes
// trade elements 2, 3 for the partner's 0, 1.  Step 2, partner i ^ 1
// (quad_perm [1, 0, 3, 2]): the even lanes trade elements 1, 3 for the
// partner's 0, 2.  Every lane of the wave must be active.
template <int CTRL> __device__ __forceinline__ float quad_perm(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), CTRL, 0xF, 0xF, true));
}
__device__ __forceinline__ void quad_swap_halves(floatx4 &x, bool upper) { // upper = i & 2
    const float r0 = quad_perm<0x4E>(upper ? x[0] : x[2]), r1 = quad_perm<0x4E>(upper ? x[1] : x[3]);
    if (upper) {
        x[0] = r0;
        x[1] = r1;
    } else {
        x[2] = r0;
        x[3] = r1;
    }
}
__device__ __forceinline__ void quad_swap_pairs(floatx4 &x, bool odd) { // odd = i & 1
    const float r0 = quad_perm<0xB1>(odd ? x[0] : x[1]), r1 = quad_perm<0xB1>(odd ? x[2] : x[3]);
    if (odd) {
        x[0] = r0;
        x[2] = r1;
    } else {
        x[1] = r0;
        x[3] = r1;
    }
}

// ---------------------------------------------------------------------------
// f32 products on the bf16 matrix cores, for the segment summaries: an operand
// x is taken as three bf16 terms,
//   h = bf16(x),  m = bf16(x - h),  l = bf16(x - h - m),
// whose sum is x exactly (8 significant bits each, and the signs of the
// remainders, cover f32's 24), whatever its neighbours in the row are, and
// hh + hm + mh + mm + hl + lh are accumulated in f32: what is left out is below
// 2^-25 of a product, less than its rounding in f32.  bf16 has f32's exponents,
// so there is no scale; only remainders below 2^-133 are lost.  A 16x16x32
// step takes the fragments of two neighbouring 16x16 tiles of the contraction,
// k = 4 group + step in each, so that two f32 accumulator tiles are one second
// operand.  Six such steps (16 cycles each) stand for the eight 16x16x4 f32
// steps (32 cycles each) of the same contraction; splitting costs 5.5 vector
// instructions an element, so it pays where a workgroup splits an operand once
// for many columns.
//
// Infinities (h infinite, x - h not a number) and values that round to one do
// not split.  They show as an output that is not finite; such outputs are
// formed again from the f32 operands by f32 instructions (products).
// ---------------------------------------------------------------------------
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float floatx2 __attribute__((ext_vector_type(2)));

struct Terms {
    bf16x8 t[3]; // h, m, l
};
// Two tiles' four elements each as one 32-deep operand.
__device__ __forceinline__ Terms split_pair(floatx4 a, floatx4 b) {
    Terms r;
#pragma unroll
    for (int j = 0; j < 8; j += 2) {
        float x = j < 4 ? a[j & 3] : b[j & 3], y = j < 4 ? a[(j & 3) + 1] : b[(j & 3) + 1];
#pragma unroll
        for (int t = 0; t < 3; ++t) {
            const bf16x2 q = __builtin_convertvector(floatx2{x, y}, bf16x2);
            r.t[t][j] = q[0];
            r.t[t][j + 1] = q[1];
            x -= (float)q[0];
            y -= (float)q[1];
        }
    }
    return r;
}
// T accumulator tiles of a column block as T / 2 second operands.
template <int T> __device__ __forceinline__ void split_tiles(const floatx4 *x, Terms *r) {
#pragma unroll
    for (int t = 0; t < T; t += 2) r[t / 2] = split_pair(x[t], x[t + 1]);
}

// A first operand's terms in LDS: pair i of neighbouring tiles (f32 fragments
// 2 i and 2 i + 1 of it) lies at s[3 i], as h, m and l of 64 lanes each.
__device__ __forceinline__ void put_terms(floatx4 a, floatx4 b, floatx4 *s, int pair, int lane) {
    const Terms r = split_pair(a, b);
#pragma unroll
    for (int t = 0; t < 3; ++t) s[(pair * 3 + t) * 64 + lane] = __builtin_bit_cast(floatx4, r.t[t]);
}

// x (+)= A b with f32 instructions, A of R row tiles x T tiles in f32 fragments
// in (row tile, tile) order from s (tile columns K0 .. K1 - 1 of it).  A tile
// column's fragments are read during the products of the one before it.
template <int R, int T, int K0 = 0, int K1 = T>
__device__ __forceinline__ void products_f32(const floatx4 *s, int lane, const floatx4 *b, floatx4 *x) {
    floatx4 a[2][R];
    auto read = [&](int k) {
#pragma unroll
        for (int r = 0; r < R; ++r) a[k & 1][r] = s[(r * T + k) * 64 + lane];
    };
    read(K0);
#pragma unroll
    for (int k = K0; k < K1; ++k) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
#pragma unroll
            for (int r = 0; r < R; ++r) x[r] = mfma16(a[k & 1][r][i], b[k][i], x[r]);
            if (i == 0) {
                __builtin_amdgcn_sched_barrier(0);
                if (k + 1 < K1) read(k + 1);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    }
}

// x = A b for A of R row tiles x P pairs of tiles whose terms lie in LDS from s,
// and a column block b (f32 tiles, and their terms t); src: A's f32 fragments.
template <int R, int P>
__device__ __forceinline__ void products(const floatx4 *s, const floatx4 *src, int lane, const floatx4 *b, const Terms *t,
                                         floatx4 *x) {
    constexpr int RB = R < 4 ? R : 4; // row tiles (independent chains) at a time
    constexpr int ta[6] = {2, 0, 1, 1, 0, 0}, tb[6] = {0, 2, 1, 0, 1, 0};
    constexpr int F = R / RB * P;
    bf16x8 a[2][RB][3]; // a step's operands are read during the step before it
    auto read = [&](int f) {
#pragma unroll
        for (int r = 0; r < RB; ++r)
#pragma unroll
            for (int j = 0; j < 3; ++j)
                a[f & 1][r][j] = __builtin_bit_cast(bf16x8, s[(((f / P * RB + r) * P + f % P) * 3 + j) * 64 + lane]);
    };
    read(0);
#pragma unroll
    for (int r = 0; r < R; ++r) x[r] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int f = 0; f < F; ++f) {
        if (f + 1 < F) read(f + 1);
#pragma unroll
        for (int i = 0; i < 6; ++i)
#pragma unroll
            for (int r = 0; r < RB; ++r) {
                floatx4 &y = x[f / P * RB + r];
                y = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[f & 1][r][ta[i]], t[f % P].t[tb[i]], y, 0, 0, 0);
            }
        __builtin_amdgcn_sched_barrier(0);
    }
    float mx = 0.f;
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int i = 0; i < 4; ++i) mx = __builtin_elementwise_maximum(mx, __builtin_fabsf(x[r][i]));
    if (__builtin_expect(__any(!(mx < __builtin_inff())), 0)) { // (maximum() keeps a NaN)
#pragma unroll
        for (int r = 0; r < R; ++r) x[r] = floatx4{0.f, 0.f, 0.f, 0.f};
        products_f32<R, 2 * P>(src, lane, b, x);
    }
}

// Element idx of a wave-uniform array: one scalar base and a 32-bit offset per
// lane, where 64-bit lane addresses of many loads would take registers.
__device__ __forceinline__ floatx4 ld_uni(const floatx4 *base, unsigned idx) {
    return *reinterpret_cast<const floatx4 *>(reinterpret_cast<const char *>(base) + idx * 16u);
}

// Direct global -> LDS copy of one float4 per lane (global_load_lds_dwordx4):
// lane l of the calling wave writes wave_base[l]; wave_base is wave-uniform.
// The copy counts in vmcnt: wait with vm_wait0() before the barrier that
// publishes it.
__device__ __forceinline__ void lds_copy4(const floatx4 *src, floatx4 *wave_base) {
    __builtin_amdgcn_global_load_lds(static_cast<const void *>(src),
                                     (__attribute__((address_space(3))) void *)(wave_base), 16, 0, 0);
}
// Pulls the 128-byte line holding `line` toward this XCD's L2: a 4-byte copy
// into the calling lane's word of wave_slot (64 floats per wave, never read).
// It counts in vmcnt like lds_copy4, so a wait that must not cover it leaves
// it among the most recent operations (vm_wait<N>).
__device__ __forceinline__ void l2_touch(const void *line, float *wave_slot) {
    __builtin_amdgcn_global_load_lds(line, (__attribute__((address_space(3))) void *)(wave_slot), 4, 0, 0);
}
// s_waitcnt vmcnt(N): every vector memory operation of the wave but the N
// most recent has completed (they complete in issue order); expcnt and
// lgkmcnt are not waited on.
template <int N> __device__ __forceinline__ void vm_wait() {
    static_assert(N >= 0 && N < 64, "vmcnt is 6 bits");
    __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14));
}
__device__ __forceinline__ void vm_wait0() { vm_wait<0>(); }
// Workgroup barrier that leaves vmcnt alone (__syncthreads' fence would wait
// for every copy and touch in flight): lgkmcnt(0) completes this wave's LDS
// accesses, and the asm's memory clobber keeps the compiler from moving
// memory accesses across it.  The caller's vm_wait<N>() decides which
// global -> LDS copies have landed.
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_s_waitcnt(0xC07F); // lgkmcnt(0); vmcnt(63) and expcnt(7) are no-ops
    asm volatile("s_barrier" ::: "memory");
}

// Sequences are spread over the 8 XCDs (workgroup i runs on XCD i % 8) so
// that the V-slices of one sequence, which read the same W, M and Kd^T,
// land on the same XCD and share its L2.  Identity when the sequence count
// is not a multiple of 8.
__device__ __forceinline__ void inter_block(int blk, int nseq, int nvs, int *bh, int *vs) {
    if (nseq % 8 == 0) {
        const int x = blk % 8, j = blk / 8;
        *bh = x + 8 * (j / nvs);
        *vs = j % nvs;
    } else {
        *bh = blk / nvs;
        *vs = blk % nvs;
    }
}

// The chain of the segmented passes, X <- P_i X + Q_i for i = 0 .. nsteps - 1,
// on a workgroup of K / 16 waves that owns 16 value columns of one sequence:
// wave w holds rows 16 w .. of X, and the waves exchange X through LDS between
// steps.  The steps are a serial chain, so what counts is one step: K / 4
// dependent products a wave and one barrier.  A wave's rows of P_{i+1} and Q_{i+1} are
// requested as those of step i are used, and land during it.  Against a wave
// that walks all rows of its columns ((K / 16)^2 x 4 products a step): the
// forward's chain at T = 32768, 16 heads, K = V = 128 (12 segments) 76 -> 26
// us, at T = 1024, 4 heads of 64 13.4 -> 6.7; B = 4, T = 2048, 16 heads of
// 128 (one step) 27 -> 15 forward, 32 -> 12 backward.
// load(i, kb): this lane's A fragment of P_i, row tile w, columns 16 kb ..;
// slot(i): where Q_i lies and X of step i goes, row-major with row length V.
template <int K, class Load, class Slot>
__device__ __forceinline__ void chain_walk(floatx4 x, int nsteps, int V, int col, Load load, Slot slot) {
    constexpr int NKT = K / 16;
    __shared__ floatx4 sX[2][NKT * 64];
    const int lane = threadIdx.x & 63, lg = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const size_t o = (size_t)(16 * wave + 4 * lg) * V + col;
    floatx4 pa[NKT], q = {};
    auto load_q = [&](int i) {
        const float *Q = slot(i) + o;
#pragma unroll
        for (int r = 0; r < 4; ++r) q[r] = Q[(size_t)r * V];
    };
    if (nsteps > 0) {
#pragma unroll
        for (int kb = 0; kb < NKT; ++kb) pa[kb] = load(0, kb);
        load_q(0);
    }
    sX[0][wave * 64 + lane] = x;
    for (int i = 0; i < nsteps; ++i) {
        lds_barrier(); // X of step i - 1 is whole; the buffer that step i - 2 was read from is free
        const floatx4 *X = sX[i & 1];
        const int nx = min(i + 1, nsteps - 1); // (the last step's requests are not used)
        x = q;
        load_q(nx);
#pragma unroll
        for (int kb = 0; kb < NKT; ++kb) {
            const floatx4 b = X[kb * 64 + lane];
#pragma unroll
            for (int st = 0; st < 4; ++st) x = mfma16(pa[kb][st], b[st], x);
            pa[kb] = load(nx, kb);
        }
        sX[(i & 1) ^ 1][wave * 64 + lane] = x;
        float *Q = slot(i) + o;
#pragma unroll
        for (int r = 0; r < 4; ++r) Q[(size_t)r * V] = x[r];
    }
}

// Host side of the chunked forward, shared with the backward (chunk.hip).
gdn2_status chunk_setup(const gdn2_chunk_args *a, const char *who, bool need_out, ChunkParams *p);
// shorten: with the short segments (inter_segments), as gdn2_chunk_workspace_bytes
// sizes it; without them, the least a call takes.
size_t chunk_fwd_ws_bytes(const gdn2_chunk_args *a, bool shorten);
// Segments per sequence of the sequential kernels (1 = unsegmented).
int chunk_segments(int64_t seqs, int64_t K, int64_t V, int64_t NC, bool shorten);
void chunk_bind_ws(const gdn2_chunk_args *a, char *ws, bool shorten, ChunkParams *p);

}  // namespace gdn2
