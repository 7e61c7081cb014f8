// f32 matrix products on the f16 matrix cores (split_gemm.hip).
#pragma once

#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <cstddef>
#include <cstdint>

namespace gdn2 {

// What a row of a split operand records about its elements.
struct SplitStat {
    unsigned amax; // bits of the largest magnitude (NaN > infinity > every finite value)
    unsigned lost; // sum of what its small elements lose, in units of 2^-36 of its scale
};

struct SplitGemmParams {
    // C [M, N] (+)= op(A) [M, Kd] op(B) [Kd, N], row-major; ta: A is stored [Kd, M], tb: B is stored [N, Kd]
    const float *A, *B;
    float *C;
    int64_t lda, ldb, ldc, M, N, Kd;
    float beta;
    bool ta, tb, vec_c;    // vec_c: rows of C are 16-byte aligned
    const void *fa, *fb;   // the split operands: rows of op(A), columns of op(B)
    const SplitStat *sa, *sb;
    float *part;           // partial sums of the tiles cut along the contraction
    // the 32 x 32 parts whose outputs are formed again by redo_kernel, eight bytes
    // of flags a tile, and which outputs of them (16 bits a lane)
    unsigned char *redo;
    unsigned short *failed;
    // plan_split_gemm:
    int tile, KT;
    unsigned ntm, ntn, split, whole;
    int64_t rta, rtb;
};

// Bytes of a split operand of `rows` rows of Kd elements, and of its row records.
size_t split_frag_bytes(int64_t rows, int64_t Kd);
size_t split_stat_bytes(int64_t rows);
// Splits an operand: rows of src when !trans (its contiguous dimension is the
// contraction), columns of src when trans.
hipError_t launch_split(const float *src, int64_t ld, bool trans, int64_t rows, int64_t Kd, void *frags, SplitStat *stat,
                        hipStream_t s);
// Fills the plan of p from M, N, Kd; returns the bytes of `part`.
size_t plan_split_gemm(SplitGemmParams *p);
void split_redo_bytes(const SplitGemmParams &p, size_t *flags, size_t *failed);
hipError_t launch_split_gemm(const SplitGemmParams &p, hipStream_t s);

// A weight matrix as the second operand of split products, whose terms are kept
// between them.  Its owner says when the values change; the next product then
// splits it again, or, once a captured graph reads the terms, changed() does.
struct SplitWeight {
    const float *src = nullptr;       // [rows of the stored matrix, cols], row stride ld
    int64_t ld = 0, rows = 0, Kd = 0; // rows of the operand (N of the product) and its contraction
    bool trans = false;               // the operand's rows are src's columns
    void *frags = nullptr;            // allocated by the first product that uses it
    SplitStat *stat = nullptr;

    // The terms of the present values, for work on s; false: no memory for them
    // (a call that is being recorded allocates none).
    bool ready(hipStream_t s, bool recording, hipError_t *e) {
        *e = hipSuccess;
        if (!frags) {
            const size_t fb = split_frag_bytes(rows, Kd);
            void *buf = nullptr;
            if (recording || hipMalloc(&buf, fb + split_stat_bytes(rows)) != hipSuccess) {
                (void)hipGetLastError();
                return false;
            }
            frags = buf;
            stat = reinterpret_cast<SplitStat *>(static_cast<char *>(buf) + fb);
        }
        if (!fresh_) {
            *e = launch_split(src, ld, trans, rows, Kd, frags, stat, s);
            fresh_ = *e == hipSuccess && !recording; // (what is recorded runs with each replay)
        }
        recorded_ = recorded_ || recording;
        return true;
    }
    // The values have changed: returns whether a split was queued (on the null stream).
    bool changed(hipError_t *e) {
        *e = hipSuccess;
        fresh_ = false;
        if (!recorded_) return false;
        *e = launch_split(src, ld, trans, rows, Kd, frags, stat, nullptr);
        fresh_ = *e == hipSuccess;
        return true;
    }
    void destroy() {
        if (frags) (void)hipFree(frags);
        frags = nullptr;
        stat = nullptr;
        fresh_ = recorded_ = false;
    }

  private:
    bool fresh_ = false;    // the terms are those of the present values
    bool recorded_ = false; // a captured graph reads them
};

}  // namespace gdn2
