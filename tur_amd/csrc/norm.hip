// RmsNorm, the layer in front of the q / k / v and gate / up projections (reference: src/models/layers/norm.rs:81-93 builds
// candle_nn::RmsNorm from the dequantized F32 `weight` of the GGUF file; src/models/qwen3.rs applies it before the attention and
// MLP blocks).  y[r][c] = x[r][c] / sqrt(mean_c(x[r][c]^2) + eps) * weight[c], computed in f32 in candle's order: the sum of
// squares of the row, one square root, then per element a division and a multiplication.
#include "mfma_common.h"

namespace {

template <int XT> __device__ inline float ld_elem(const void *x, int64_t i) {
    if (XT == TURQ_ACT_F32) return ((const float *)x)[i];
    if (XT == TURQ_ACT_BF16) return __uint_as_float((uint32_t)((const uint16_t *)x)[i] << 16);
    _Float16 h;
    const uint16_t u = ((const uint16_t *)x)[i];
    __builtin_memcpy(&h, &u, 2);
    return (float)h;
}

// The kernels take a row of more than 512 columns in pieces of 8 neighbouring columns: thread t of a row's 256 holds the pieces t, t + 256, ... (PER of them
// in registers), loaded and stored 16 bytes at a time where the row allows it.  Bound by latency at decode sizes (one row is one
// chain load -> sum -> barrier -> divide -> store in a launch of 4 us) and by the memory system at prompt sizes.  With one element per load
// (2 bytes of a bf16 row) the chain of 16 loads per thread was the kernel: 8 rows of 4096 bf16 columns took 10.5 us, now 4.0 - 4.7.

// eight columns of a row from column col0 on, +0 past k
template <int XT> __device__ inline void ld_piece(const void *x, int64_t row_off, int64_t col0, int64_t k, bool vec, float (&v)[8]) {
    if (vec && col0 + 8 <= k) {
        const uint8_t *p = (const uint8_t *)x + (row_off + col0) * (XT == TURQ_ACT_F32 ? 4 : 2);
        if constexpr (XT == TURQ_ACT_F32) {
            const float4v lo = ((const float4v *)p)[0], hi = ((const float4v *)p)[1];
            v[0] = lo.x, v[1] = lo.y, v[2] = lo.z, v[3] = lo.w, v[4] = hi.x, v[5] = hi.y, v[6] = hi.z, v[7] = hi.w;
        } else {
            const uint4v u = *(const uint4v *)p;
            const uint32_t wd[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
            for (int j = 0; j < 4; j++) {
                if constexpr (XT == TURQ_ACT_BF16) {
                    v[2 * j] = __uint_as_float(wd[j] << 16);
                    v[2 * j + 1] = __uint_as_float(wd[j] & 0xFFFF0000u);
                } else {
                    const half2v hh = as_half2(wd[j]);
                    v[2 * j] = (float)hh.x;
                    v[2 * j + 1] = (float)hh.y;
                }
            }
        }
    } else {
#pragma unroll
        for (int e = 0; e < 8; e++) v[e] = col0 + e < k ? ld_elem<XT>(x, row_off + col0 + e) : 0.0f;
    }
}

// The pieces tid, tid + 256, ... of a row (+0 past k, and everywhere where !live) and, up to WPER of them, of its weight.  Where rows, weight and
// k allow 16-byte loads all of them are requested before the first is looked at: a weight that is first asked for behind the sum, as the
// store needs it, waits for HBM a second time, and pieces that are converted one by one a time each (three layers at 77 bf16 rows of 4096 columns,
// six such launches in 338 us: 5 us less; 1024 columns, one piece per thread: no difference).
template <int XT, int PER, int WPER>
__device__ inline void ld_pieces(const void *x, int64_t row_off, int64_t k, bool live, bool vec_x, const float *w, bool vec_w, int tid, float (&v)[PER][8],
                                 float (&wv)[WPER][8]) {
    static_assert(WPER <= PER);
    if (vec_x && vec_w && (k & 7) == 0) {
        constexpr int ES = XT == TURQ_ACT_F32 ? 4 : 2;
        uint4v raw[PER][ES / 2];
        float4v rw[WPER][2];
        const uint8_t *px = (const uint8_t *)x + (live ? row_off : 0) * ES;  // (the first row exists)
#pragma unroll
        for (int j = 0; j < PER; j++) {
            const int64_t col0 = ((int64_t)j * 256 + tid) * 8, at = col0 < k ? col0 : 0;
#pragma unroll
            for (int h = 0; h < ES / 2; h++) raw[j][h] = ((const uint4v *)(px + at * ES))[h];
        }
#pragma unroll
        for (int j = 0; j < WPER; j++) {
            const int64_t col0 = ((int64_t)j * 256 + tid) * 8, at = col0 < k ? col0 : 0;
            rw[j][0] = ((const float4v *)(w + at))[0], rw[j][1] = ((const float4v *)(w + at))[1];
        }
#pragma unroll
        for (int j = 0; j < PER; j++) {
            const bool on = live && ((int64_t)j * 256 + tid) * 8 < k;
#pragma unroll
            for (int e = 0; e < 8; e++) {
                if constexpr (XT == TURQ_ACT_F32) {
                    v[j][e] = on ? __uint_as_float(raw[j][e >> 2][e & 3]) : 0.0f;
                } else if constexpr (XT == TURQ_ACT_BF16) {
                    const uint32_t u = raw[j][0][e >> 1];
                    v[j][e] = on ? __uint_as_float(e & 1 ? u & 0xFFFF0000u : u << 16) : 0.0f;
                } else {
                    const half2v hh = as_half2(raw[j][0][e >> 1]);
                    v[j][e] = on ? (float)(e & 1 ? hh.y : hh.x) : 0.0f;
                }
            }
        }
#pragma unroll
        for (int j = 0; j < WPER; j++)
#pragma unroll
            for (int e = 0; e < 8; e++) wv[j][e] = rw[j][e >> 2][e & 3];
        return;
    }
#pragma unroll
    for (int j = 0; j < PER; j++) ld_piece<XT>(x, row_off, ((int64_t)j * 256 + tid) * 8, live ? k : 0, vec_x, v[j]);
#pragma unroll
    for (int j = 0; j < WPER; j++) ld_piece<TURQ_ACT_F32>(w, 0, ((int64_t)j * 256 + tid) * 8, k, vec_w, wv[j]);
}

__device__ inline bool vec_row(const void *p, int64_t ld, int elem_bytes) {
    return ((uintptr_t)p & 15) == 0 && ((ld * elem_bytes) & 15) == 0;
}

// sqrt(mean(x^2) + eps) of the row that a workgroup of four waves holds: s[j] = what a thread has of the squares of its piece j, summed up over
// the lanes of each wave and then over the blocks 4 j + wave in order - one fixed order, shared by the kernels below so that they
// agree to the bit (as sq4 says).  part: 4 PER floats, which it fills; of a row with more than 4 PER blocks `blocks` floats, those behind the first 4 PER
// already filled by the caller (part[b]: the sum of block b).  Every thread of the workgroup calls it.
template <int PER> __device__ inline float rms_of(const float (&s)[PER], int64_t k, float eps, float *part, int blocks = 0) {
#pragma unroll
    for (int j = 0; j < PER; j++) {
        const float t = sum64(s[j]);
        if ((threadIdx.x & 63) == 0) part[4 * j + ((threadIdx.x >> 6) & 3)] = t;
    }
    __syncthreads();
    float total = part[0];
#pragma unroll
    for (int b = 1; b < 4 * PER; b++) total += part[b];
    for (int b = 4 * PER; b < blocks; b++) total += part[b];
    return sqrtf(total / (float)k + eps);
}
// the squares of a piece of eight columns
__device__ inline float sq8(const float (&v)[8]) { return sq4(v[0], v[1], v[2], v[3]) + sq4(v[4], v[5], v[6], v[7]); }

// v / rms for many v against one rms, to the last bit: with r = 1 / rms correctly rounded, q = v * r corrected once by its own
// remainder is the correctly rounded quotient (P. Markstein, "Computation of elementary functions on the IBM RISC System/6000",
// 1990) as long as nothing over- or underflows on the way.  No |v| of a row exceeds sqrt(k) * rms; from 2^-60 on, against an rms between
// 2^-40 and 2^40, the quotient is at least 2^-100 and the remainder, a multiple of 2^-48 |v| or so, stays exact.  Pieces with a smaller element -
// a zero, whose sign the correction would lose, among them - and rows whose rms is an infinity, a NaN or outside that range take the plain
// division (asked once per piece: asked per element the kernel was 0.3 us longer at one row, a tenth).
struct RowDiv {
    float rms, r, least;  // least: the smallest |v| that is corrected (an infinity: none is)
    __device__ explicit RowDiv(float d) : rms(d), r(1.0f / d), least(d > 0x1p-40f && d < 0x1p40f ? 0x1p-60f : __builtin_inff()) {}
    __device__ void operator()(const float (&v)[8], float (&o)[8]) const {
        bool plain = false;
#pragma unroll
        for (int e = 0; e < 8; e++) plain |= !(__builtin_fabsf(v[e]) >= least);
        if (__builtin_amdgcn_ballot_w64(plain) != 0) {  // (one branch of the wave: the division gives the others the same quotients)
#pragma unroll
            for (int e = 0; e < 8; e++) o[e] = v[e] / rms;
        } else {
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const float q = v[e] * r;
                o[e] = __builtin_fmaf(__builtin_fmaf(-q, rms, v[e]), r, q);
            }
        }
    }
};

// rows of up to kShort columns: one workgroup of 256 threads per row, two elements t and t + 256 per thread.  A piece of eight columns per thread
// leaves three of the four waves without any: 128 columns (the heads of q and k) at 1 / 16384 rows 2.7 / 16.0 us, here 2.2 / 11.7; from 1024
// columns on the pieces are ahead (16384 bf16 rows 28.5 -> 20.0)
constexpr int64_t kShort = 512;
template <int XT> __device__ inline float short_square_sum(const void *x, int64_t xo, int64_t k, int tid, float (&v)[2]) {
    float s = 0.0f;
#pragma unroll
    for (int j = 0; j < 2; j++) {
        const int64_t c = (int64_t)j * 256 + tid;
        v[j] = c < k ? ld_elem<XT>(x, xo + c) : 0.0f;
        s = __builtin_fmaf(v[j], v[j], s);  // (columns past k add +0)
    }
    return s;
}
template <int XT, int YT>
__global__ void __launch_bounds__(256) rms_norm_short_kernel(const void *__restrict__ x, int64_t k, int64_t ldx, const float *__restrict__ w,
                                                             float eps, void *__restrict__ y, int64_t ldy) {
    __shared__ float part[4];
    const int tid = threadIdx.x;
    const int64_t row = blockIdx.x;
    float v[2];
    const float sq[1] = {short_square_sum<XT>(x, row * ldx, k, tid, v)};
    const float rms = rms_of(sq, k, eps, part);
#pragma unroll
    for (int j = 0; j < 2; j++) {
        const int64_t c = (int64_t)j * 256 + tid;
        if (c < k) turq_store_out<YT>(y, row * ldy + c, v[j] / rms * w[c]);
    }
}

// one workgroup of 256 threads per row; rows of up to 2048 * PER elements are read once (so y may be x whatever the two element
// types), longer rows, which only PER = 3 takes, are read again
template <int XT, int YT, int PER>
__global__ void __launch_bounds__(256) rms_norm_kernel(const void *__restrict__ x, int64_t k, int64_t ldx, const float *__restrict__ w,
                                                       float eps, void *__restrict__ y, int64_t ldy) {
    __shared__ float part[PER == 3 ? 32 : 4 * PER];
    const int tid = threadIdx.x;
    const int64_t row = blockIdx.x;
    const int64_t xo = row * ldx, yo = row * ldy;
    const bool vx = vec_row(x, ldx, XT == TURQ_ACT_F32 ? 4 : 2), vy = vec_row(y, ldy, YT == TURQ_ACT_F32 ? 4 : 2);
    const bool vw = ((uintptr_t)w & 15) == 0;
    float v[PER][8], wv[PER][8];
    ld_pieces<XT, PER, PER>(x, xo, k, true, vx, w, vw, tid, v, wv);
    float s[PER];
#pragma unroll
    for (int j = 0; j < PER; j++) s[j] = sq8(v[j]);  // (columns past k add +0: the sum is that of the columns that exist)
    // longer rows: blocks of 512 columns of their own up to 16384 columns, what lies behind is added to the first
    int j = PER;
    for (; PER == 3 && (int64_t)j * 2048 < k && j < 8; j++) {
        float t[8];
        ld_piece<XT>(x, xo, ((int64_t)j * 256 + tid) * 8, k, vx, t);
        const float b = sum64(sq8(t));
        if ((tid & 63) == 0) part[4 * j + (tid >> 6)] = b;
    }
    for (int64_t col0 = ((int64_t)j * 256 + tid) * 8; PER == 3 && col0 < k; col0 += 2048) {
        float t[8];
        ld_piece<XT>(x, xo, col0, k, vx, t);
        s[0] += sq8(t);
    }
    const RowDiv div(rms_of(s, k, eps, part, 4 * j));
    auto store = [&](int64_t col0, const float (&t)[8], const float (&tw)[8]) {
        if (col0 >= k) return;
        float o[8];
        div(t, o);
#pragma unroll
        for (int e = 0; e < 8; e++) o[e] *= tw[e];
        if (vy && col0 + 8 <= k) {
            turq_note_results<YT>(o);
            uint8_t *p = (uint8_t *)y + (yo + col0) * (YT == TURQ_ACT_F32 ? 4 : 2);
            if constexpr (YT == TURQ_ACT_F32) {
                ((float4v *)p)[0] = float4v{o[0], o[1], o[2], o[3]};
                ((float4v *)p)[1] = float4v{o[4], o[5], o[6], o[7]};
            } else if constexpr (YT == TURQ_ACT_BF16) {
                *(uint4v *)p = uint4v{turq_f2bf_x2(o[0], o[1]), turq_f2bf_x2(o[2], o[3]), turq_f2bf_x2(o[4], o[5]), turq_f2bf_x2(o[6], o[7])};
            } else {
                half8v h;
#pragma unroll
                for (int e = 0; e < 8; e++) h[e] = (_Float16)o[e];
                *(half8v *)p = h;
            }
        } else {
#pragma unroll
            for (int e = 0; e < 8; e++)
                if (col0 + e < k) turq_store_out<YT>(y, yo + col0 + e, o[e]);
        }
    };
#pragma unroll
    for (int j = 0; j < PER; j++) store(((int64_t)j * 256 + tid) * 8, v[j], wv[j]);
    for (int64_t col0 = ((int64_t)PER * 256 + tid) * 8; PER == 3 && col0 < k; col0 += 2048) {
        float t[8], tw[8];
        ld_piece<XT>(x, xo, col0, k, vx, t);
        ld_piece<TURQ_ACT_F32>(w, 0, col0, k, vw, tw);
        store(col0, t, tw);
    }
}

// The same rows written straight into the fragments of the prefill GEMM (the order act_prep32_kernel writes, see there): what
// rms_norm_kernel with an f32 output followed by that kernel would leave - the same sums in the same order, the same one rounding
// to f16 - without the launch and the round trip in between.  One workgroup per row (rows past m, to the end of a 32-row m-tile: zeros); a fragment
// block holds 16 bytes of each row next to each other, so neighbouring rows, which meet in a cache line, run on one XCD and meet in its L2.  Four rows per
// workgroup, which wrote 64 bytes together, kept 24 of 256 CUs at 77 rows: the layers of 4096 columns at 77 / 512 rows took 342 / 557 us with them
// and 329 / 552 now, those of 1024 columns at 300 rows 846 and 810, 4096 columns at 2048 rows the same.  A thread keeps its PER pieces of 8 columns in registers
// between the two passes (k <= 2048 * PER); the sub-block sums of the fragments (32 columns) are added up between the four neighbouring lanes that hold
// a sub-block.
template <int XT, bool Q8, int PER>
__global__ void __launch_bounds__(256) rms_norm_prep32_kernel(const void *__restrict__ x, int64_t m, int64_t k, int64_t ldx, const float *__restrict__ w,
                                                              float eps, int64_t ntc, half8v *__restrict__ frags) {
    __shared__ float part[4 * PER];
    const int tid = threadIdx.x;
    // workgroups of one XCD (blockIdx % 8) take neighbouring rows (the grid: a multiple of 32)
    const int64_t row = (int64_t)(blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
    const int64_t mt = row >> 5;
    const int r = (int)(row & 31);
    const bool live = row < m;
    const int64_t xo = row * ldx;
    const bool vx = vec_row(x, ldx, XT == TURQ_ACT_F32 ? 4 : 2), vw = ((uintptr_t)w & 15) == 0;
    constexpr int WPER = PER <= 2 ? PER : 1;  // (longer rows: eight waves share a SIMD up to 64 registers)
    float v[PER][8], wv[WPER][8];
    float s[PER];
    ld_pieces<XT, PER, WPER>(x, xo, k, live, vx, w, vw, tid, v, wv);
    if (PER == 1 && k <= kShort) {  // (the order of rms_norm_short_kernel)
        float sq[2];
        s[0] = short_square_sum<XT>(x, xo, live ? k : 0, tid, sq);
    } else {
#pragma unroll
        for (int j = 0; j < PER; j++) s[j] = sq8(v[j]);
    }
    const RowDiv div(rms_of(s, k, eps, part));
#pragma unroll
    for (int j = 0; j < PER; j++) {
        const int64_t piece = (int64_t)j * 256 + tid, col0 = piece * 8;
        if (col0 >= k) continue;  // (k is a multiple of 256: whole pieces, and whole groups of four lanes)
        if (j >= WPER) ld_piece<TURQ_ACT_F32>(w, 0, col0, k, vw, wv[0]);
        const float (&wj)[8] = wv[j < WPER ? j : 0];
        half8v h;
        float sum = 0.0f, f[8];
        div(v[j], f);
#pragma unroll
        for (int e = 0; e < 8; e++) {
            f[e] = live ? f[e] * wj[e] : 0.0f;
            h[e] = (_Float16)f[e];
            sum += (float)h[e];
        }
        turq_note_results<TURQ_ACT_F16>(f);
        const int64_t b = piece >> 5;
        const int cc = (int)(piece & 31);
        half8v *dst = frags + (mt * ntc + b) * (17 * 64);
        const int g32 = Q8 ? (cc >> 1) & 1 : cc >> 4, q = Q8 ? 2 * (cc >> 2) + (cc & 1) : cc & 15;
        dst[q * 64 + r + 32 * g32] = h;
        if (!Q8) {
            sum += __shfl_xor(sum, 1, 64);
            sum += __shfl_xor(sum, 2, 64);
            if ((tid & 3) == 0) {
                const int sb = (cc >> 2) & 3;
                const _Float16 hi = (_Float16)sum;
                const _Float16 lo = (_Float16)(sum - (float)hi);
                ((half2v *)&dst[16 * 64 + r + 32 * g32])[sb] = half2v{hi, lo};
            }
        }
    }
}

template <int XT, int YT>
hipError_t launch2(const void *x, int64_t m, int64_t k, int64_t ldx, const float *w, float eps, void *y, int64_t ldy, hipStream_t s) {
    if (k <= kShort) rms_norm_short_kernel<XT, YT><<<(unsigned)m, 256, 0, s>>>(x, k, ldx, w, eps, y, ldy);
    else if (k <= 2048) rms_norm_kernel<XT, YT, 1><<<(unsigned)m, 256, 0, s>>>(x, k, ldx, w, eps, y, ldy);
    else if (k <= 2 * 2048) rms_norm_kernel<XT, YT, 2><<<(unsigned)m, 256, 0, s>>>(x, k, ldx, w, eps, y, ldy);
    else rms_norm_kernel<XT, YT, 3><<<(unsigned)m, 256, 0, s>>>(x, k, ldx, w, eps, y, ldy);
    return hipGetLastError();
}

template <int XT>
hipError_t launch1(int yt, const void *x, int64_t m, int64_t k, int64_t ldx, const float *w, float eps, void *y, int64_t ldy, hipStream_t s) {
    switch (yt) {
    case TURQ_ACT_F32: return launch2<XT, TURQ_ACT_F32>(x, m, k, ldx, w, eps, y, ldy, s);
    case TURQ_ACT_BF16: return launch2<XT, TURQ_ACT_BF16>(x, m, k, ldx, w, eps, y, ldy, s);
    case TURQ_ACT_F16: return launch2<XT, TURQ_ACT_F16>(x, m, k, ldx, w, eps, y, ldy, s);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace

hipError_t turq_launch_rms_norm(const void *x, int x_dtype, int64_t m, int64_t k, int64_t ldx, const float *weight, float eps, void *y,
                                int y_dtype, int64_t ldy, hipStream_t stream) {
    if (m == 0 || k == 0) return hipSuccess;
    if (m > 0x7FFFFFFF) return hipErrorInvalidValue;
    switch (x_dtype) {
    case TURQ_ACT_F32: return launch1<TURQ_ACT_F32>(y_dtype, x, m, k, ldx, weight, eps, y, ldy, stream);
    case TURQ_ACT_BF16: return launch1<TURQ_ACT_BF16>(y_dtype, x, m, k, ldx, weight, eps, y, ldy, stream);
    case TURQ_ACT_F16: return launch1<TURQ_ACT_F16>(y_dtype, x, m, k, ldx, weight, eps, y, ldy, stream);
    default: return hipErrorInvalidValue;
    }
}

// frags: turq_act_prep32_bytes(m, k) bytes; k a multiple of 256 and at most 16384; dtype picks the fragment order (Q8_0 / K-quants)
hipError_t turq_launch_rms_norm_prep32(int dtype, const void *x, int x_dtype, int64_t m, int64_t k, int64_t ldx, const float *weight,
                                       float eps, void *frags, hipStream_t stream) {
    if (m == 0 || k == 0) return hipSuccess;
    if (k % 256 != 0 || k > 16384 || m > (1 << 26)) return hipErrorInvalidValue;
    const int64_t ntc = k / 256;
    const unsigned grid = (unsigned)((m + 31) / 32 * 32);
    const bool q8 = dtype == TURQ_Q8_0;
#define TURQ_NP32(XT, PER)                                                                                                           \
    if (q8) rms_norm_prep32_kernel<XT, true, PER><<<grid, 256, 0, stream>>>(x, m, k, ldx, weight, eps, ntc, (half8v *)frags);       \
    else rms_norm_prep32_kernel<XT, false, PER><<<grid, 256, 0, stream>>>(x, m, k, ldx, weight, eps, ntc, (half8v *)frags)
#define TURQ_NP32_X(XT)                                  \
    if (k <= 2048) { TURQ_NP32(XT, 1); }                 \
    else if (k <= 2048 * 2) { TURQ_NP32(XT, 2); }        \
    else if (k <= 2048 * 3) { TURQ_NP32(XT, 3); }        \
    else if (k <= 2048 * 6) { TURQ_NP32(XT, 6); }        \
    else { TURQ_NP32(XT, 8); }                           \
    break
    switch (x_dtype) {
    case TURQ_ACT_F32: TURQ_NP32_X(TURQ_ACT_F32);
    case TURQ_ACT_BF16: TURQ_NP32_X(TURQ_ACT_BF16);
    case TURQ_ACT_F16: TURQ_NP32_X(TURQ_ACT_F16);
    default: return hipErrorInvalidValue;
    }
#undef TURQ_NP32_X
#undef TURQ_NP32
    return hipGetLastError();
}

TURQ_NONFINITE_READER(turq_nonfinite_norm)
