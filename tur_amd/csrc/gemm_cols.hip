// Quantized matmul for prompt chunks whose tiles, one workgroup each, would leave the machine waiting: the columns (k) of a tile are
// shared out over the WAVES of its workgroup instead of its rows.
//
// Every wave holds the whole workgroup tile - MT x NT MFMA tiles of 32 x 32 - and walks its own super-blocks (256 columns): the
// activation fragments (prepared in 32-row A order by act_prep32_kernel and its relatives) and the packed weights come straight
// into registers, a lane's 16 bytes at a time, each 1 KiB instruction reading one contiguous KiB of fragments.  Nothing a wave
// reads is read by another wave of the workgroup, so there is no LDS and no barrier in the loop; the waves' sums meet in the LDS once
// at the end, in a fixed order.  Against gemm_kq_kernel (gemm_mfma.hip), whose waves share a ring of stages in the LDS: that one moves
// fewer bytes per flop and is the better kernel where its launch fills the machine for many super-blocks, but each of its stage
// boundaries waits for copies that left one stage earlier, which is what a launch of few tiles spends its time on.
//
// The loop exists in two forms.  Loads of a wave return in order, so a weight load that comes from HBM holds up every fragment load issued after it.  The weights of
// super-block b + 1 are therefore requested together, behind the fragments of the last stage of b: the first loads that are waited for
// behind them belong to super-block b + 1 itself.  That takes a second set of weight registers and two stages of fragments.  The TIGHT
// form requests every stage of the weights of b + 1 into the registers that the same stage of b has just left, and holds one stage
// of fragments, a step of which is requested again as soon as it is used: with it two workgroups of the 64 x 64 tile share a CU, so that one
// computes while the other waits for its first loads or stores its results.  What bounds these launches is the issue of one wave per
// SIMD: without any load in the loop they still take 60 - 90 % of their time, and an order of MFMAs and unpacking made by hand, deeper
// rings and more waves of smaller tiles changed nothing.  Two workgroups per CU do: Q8_0 6144 x 1024 at 300 rows 14.1 -> 10.9 us, 4096 x 4096 at
// 512 31.6 -> 27.2, Q4_K 24576 x 4096 at 256 84 -> 73; where there is only one workgroup per CU, the first form is ahead (Q4_K 4096 x 4096 at 77
// rows 13.5 against 14.9).
#include <hip/hip_ext.h>

#include <algorithm>
#include <climits>

#include "gemm_formats.h"
#include "tuning.h"

namespace {

constexpr int kMaxGroup = 4;
struct ColsGroup {
    const uint8_t *w[kMaxGroup];
    void *y[kMaxGroup];
    const float *bias[kMaxGroup];
    int64_t n[kMaxGroup], ldy[kMaxGroup];
    float wscale[kMaxGroup];
    int first[kMaxGroup];  // first n-block of the weight (INT_MAX: there is none)
    int second;            // weights from `second` on are of the kernel's second format
};
// the weight of a workgroup
struct ColsPick {
    const uint8_t *w;
    void *y;
    const float *bias;
    int64_t n, ldy;
    float wscale;
    int index, first;
};

// a lane's packed weights of one 32-row tile and one super-block, as the loads deliver them: the header, and the four stages in order;
// what two stages share comes with the second of them
template <int DT> struct WBlk;
// loads: `t` the lane's 16-row tile (scalar base + lane offset `o`), slot = r16 + 32 * g32
__device__ inline uint4v ld16(const uint8_t *base, uint32_t o) { return *(const uint4v *)(base + o); }

template <> struct WBlk<TURQ_Q4_K> {
    uint4v q[4], hd;
    __device__ void load_hdr(const uint8_t *p, uint32_t o, uint32_t r16, uint32_t) { hd = ld16(p, o + TiledFmt<TURQ_Q4_K>::kHDR + 16u * r16); }
    template <int KS> __device__ void load(const uint8_t *p, uint32_t o, uint32_t slot) {
        q[KS] = ld16(p, o + 16u * slot + (uint32_t)((KS & 1) * 1024 + (KS >> 1) * 256));
    }
    __device__ GFmt<TURQ_Q4_K>::Hdr hdr() const { return {hd}; }
    template <int KS> __device__ GFmt<TURQ_Q4_K>::Stage stage() const { return {q[KS]}; }
};
template <> struct WBlk<TURQ_Q5_K> {
    uint4v q[4], hd;
    uint2v hh[2];
    __device__ void load_hdr(const uint8_t *p, uint32_t o, uint32_t r16, uint32_t) { hd = ld16(p, o + TiledFmt<TURQ_Q5_K>::kHDR + 16u * r16); }
    template <int KS> __device__ void load(const uint8_t *p, uint32_t o, uint32_t slot) {
        q[KS] = ld16(p, o + 16u * slot + (uint32_t)((KS & 1) * 1024 + (KS >> 1) * 256));
        if constexpr (KS & 1) hh[KS >> 1] = *(const uint2v *)(p + (o + TiledFmt<TURQ_Q5_K>::kQH + 8u * slot + (uint32_t)((KS >> 1) * 128)));
    }
    __device__ GFmt<TURQ_Q5_K>::Hdr hdr() const { return {hd}; }
    template <int KS> __device__ GFmt<TURQ_Q5_K>::Stage stage() const { return {q[KS], hh[KS >> 1]}; }
};
template <> struct WBlk<TURQ_Q6_K> {
    uint4v ql[4], qh[2];
    uint32_t sc0, sc1, d16;
    __device__ void load_hdr(const uint8_t *p, uint32_t o, uint32_t r16, uint32_t slot) {
        using F = TiledFmt<TURQ_Q6_K>;
        sc0 = *(const uint32_t *)(p + (o + F::kSC + 4u * slot));
        sc1 = *(const uint32_t *)(p + (o + F::kSC + 4u * slot + 64u));
        d16 = *(const uint16_t *)(p + (o + F::kD + 2u * r16));
    }
    template <int KS> __device__ void load(const uint8_t *p, uint32_t o, uint32_t slot) {
        ql[KS] = ld16(p, o + 16u * slot + (uint32_t)((KS & 1) * 1024 + (KS >> 1) * 256));
        if constexpr (KS & 1) qh[KS >> 1] = ld16(p, o + TiledFmt<TURQ_Q6_K>::kQH + 16u * slot + (uint32_t)((KS >> 1) * 256));
    }
    __device__ GFmt<TURQ_Q6_K>::Hdr hdr() const { return {sc0, sc1, d16}; }
    template <int KS> __device__ GFmt<TURQ_Q6_K>::Stage stage() const { return {ql[KS], qh[KS >> 1]}; }
};
template <> struct WBlk<TURQ_Q8_0> {
    uint4v a[4], b[4], dd;
    __device__ void load_hdr(const uint8_t *p, uint32_t o, uint32_t r16, uint32_t) { dd = ld16(p, o + TiledFmt<TURQ_Q8_0>::kD + 16u * r16); }
    template <int KS> __device__ void load(const uint8_t *p, uint32_t o, uint32_t slot) {
        a[KS] = ld16(p, o + 16u * slot + (uint32_t)(KS * 1024));
        b[KS] = ld16(p, o + 16u * slot + (uint32_t)(KS * 1024 + 256));
    }
    __device__ GFmt<TURQ_Q8_0>::Hdr hdr() const { return {dd}; }
    template <int KS> __device__ GFmt<TURQ_Q8_0>::Stage stage() const { return {a[KS], b[KS]}; }
};

template <int MT> struct AStage { half8v f[MT][4]; };

// Four waves in every tile shape and form, and (first form) one stage of fragments in flight besides the one being used.  The sums of a result are then the
// same numbers in the same order whatever the tile (a weight alone and in a launch of this kernel with others agree to the bit).  Eight waves were up
// to 7 % faster on the 64-row tile and spill on the larger ones; three stages in flight measured 1 - 8 % slower than one (registers).
constexpr int W = 4, RA = 2;
// The waves meet in rounds of T tiles, rows of kPitch floats (rows r and r + 4, which a store of a wave writes, lie 16 banks apart).
constexpr int kPitch = 36;
template <int MT, int NT> struct Meet {
    static constexpr int T = MT * NT < 3 ? MT * NT : MT * NT == 4 || MT * NT == 8 ? 2 : 3;
    static constexpr int ROUNDS = (MT * NT + T - 1) / T;
    static constexpr int LDS = W * T * 32 * kPitch * 4;
};

// PAIR: gate and up of an MLP (weights 0 and 1, one shape), which take turns by 16-row tiles, and SiLU(gate) * up as down_proj's activation fragments
// for results: see gemm_kq_kernel, whose pair does the same.  The halves of a 32-column MFMA tile are the two products of the same 16 columns, so a
// lane's weights are those of one of the two, which takes a 64-bit address per 32-row tile.  Without the sub-block sums of the fragments, whose 32
// columns are two workgroups' in tiles of 32 and 96 rows of weights: for a down_proj of Q6_K or Q8_0, which read none (with Q4_K and Q5_K the products go
// through memory, also where a tile of 64 would hold whole sub-blocks).  These launches are 6 - 35 us, and what the pair saves is the
// 5 us launch between it and down_proj: whole MLPs Q8_0 1024 x 3072 at 34 / 300 rows 19.3 / 30.3 -> 16.5 / 25.0 us, Q5_K / Q6_K
// 4096 x 12288 at 77 rows 66.6 -> 62.2, at 180 rows 108 -> 96; nowhere slower (4096 x 12288 .. 5120 x 15360, 34 - 600 rows, every format).
template <int DT, int MT, int NT, bool TIGHT, bool PAIR>
__device__ __forceinline__ void cols_body(const ColsGroup &grp, const ColsPick &pick, int nb, int mb, int64_t k, const uint8_t *__restrict__ frags, int64_t m,
                                          int yt, int vec_out, uint8_t *lds) {
    using Fm = GFmt<DT>;
    using Wb = WBlk<DT>;
    constexpr int TB = TiledFmt<DT>::kTileBytes;
    constexpr bool SUMS = Fm::SUMS;
    const uint8_t *__restrict__ w = pick.w;
    const int64_t n = pick.n;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n32 = lane & 31, g32 = lane >> 5, r16 = n32 & 15, tsel = n32 >> 4;
    const int ntc = (int)(k / 256);
    const int64_t mtiles = (m + 31) / 32;
    const int nrt = (int)turq_tile_rows(n);
    // this wave's super-blocks
    const int b0 = ntc * wave / W, b1 = ntc * (wave + 1) / W;

    const uint8_t *a_src[MT];  // (m-tiles past the last: the last one again, never stored)
#pragma unroll
    for (int i = 0; i < MT; i++) {
        const int64_t mt = (int64_t)mb * MT + i;
        const uint64_t off = ((uint64_t)((mt < mtiles ? mt : mtiles - 1) * ntc * 17)) << 10;  // (wave-uniform: kept in scalar registers)
        a_src[i] = frags + (((uint64_t)__builtin_amdgcn_readfirstlane((uint32_t)(off >> 32)) << 32) | __builtin_amdgcn_readfirstlane((uint32_t)off));
    }
    const int tile0 = nb * NT * (PAIR ? 1 : 2);
    const uint8_t *w_src = w + (size_t)tile0 * ntc * TB;
    uint32_t w_off[NT];  // the lane's 16-row tile of every 32-row tile
    const uint8_t *w_lane[NT];  // (pair: its address)
#pragma unroll
    for (int j = 0; j < NT; j++) {
        int t = PAIR ? tile0 + j : tile0 + 2 * j + tsel;
        t = t < nrt ? t : nrt - 1;  // (row tiles past the end: the last one again, never stored)
        w_off[j] = PAIR ? 0u : (uint32_t)(t - tile0) * (uint32_t)ntc * (uint32_t)TB;
        w_lane[j] = PAIR ? (tsel ? grp.w[1] : grp.w[0]) + (size_t)t * ntc * TB : nullptr;
    }
    auto w_at = [&](int b, int j) { return (PAIR ? w_lane[j] : w_src) + (size_t)b * TB; };
    uint32_t lane16 = 16u * (uint32_t)lane;
    const uint32_t slot = (uint32_t)(r16 + 32 * g32);
    const _Float16 ws = (_Float16)(PAIR ? (tsel ? grp.wscale[1] : grp.wscale[0]) : pick.wscale);

    float16v acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < NT; j++)
#pragma unroll
            for (int e = 0; e < 16; e++) acc[i][j][e] = 0.0f;

    if constexpr (!TIGHT) {
        AStage<MT> ra[RA];
        half8v sf[MT];
        Wb wcur[NT], wnext[NT];
        auto load_a = [&](int b, auto KS) {
            constexpr int ks = decltype(KS)::value;
#pragma unroll
            for (int i = 0; i < MT; i++) {
                const uint8_t *p = a_src[i] + ((size_t)(b * 17 + 4 * ks) << 10);
#pragma unroll
                for (int st = 0; st < 4; st++) ra[ks % RA].f[i][st] = __builtin_bit_cast(half8v, ld16(p, lane16 + (uint32_t)(st * 1024)));
            }
            if constexpr (SUMS && ks == 3) {
#pragma unroll
                for (int i = 0; i < MT; i++) sf[i] = __builtin_bit_cast(half8v, ld16(a_src[i] + ((size_t)(b * 17 + 16) << 10), lane16));
            }
        };
        auto load_w = [&](Wb (&dst)[NT], int b) {
#pragma unroll
            for (int j = 0; j < NT; j++) {
                const uint8_t *p = w_at(b, j);
                dst[j].load_hdr(p, w_off[j], (uint32_t)r16, slot);
                static_for<4>([&](auto KS) { dst[j].template load<decltype(KS)::value>(p, w_off[j], slot); });
            }
        };
        auto block = [&](int b, int bn, auto MORE) {
            constexpr bool more = decltype(MORE)::value;
            typename Fm::Consts cs[NT];
#pragma unroll
            for (int j = 0; j < NT; j++) cs[j] = Fm::consts(wcur[j].hdr(), g32, ws);
            static_for<4>([&](auto KS) {
                constexpr int ks = decltype(KS)::value, ahead = ks + RA - 1;
                if constexpr (ahead < 4) load_a(b, std::integral_constant<int, ahead>{});
                else if constexpr (more) load_a(bn, std::integral_constant<int, (ahead & 3)>{});
                if constexpr (more && ks == 2) load_w(wnext, bn);
                __builtin_amdgcn_sched_barrier(0);
                static_for<4>([&](auto ST) {
                    constexpr int st = decltype(ST)::value;
                    half8v bop[NT];
#pragma unroll
                    for (int j = 0; j < NT; j++) bop[j] = Fm::template operand<ks, st>(wcur[j].template stage<ks>(), cs[j]);
#pragma unroll
                    for (int i = 0; i < MT; i++)
#pragma unroll
                        for (int j = 0; j < NT; j++) acc[i][j] = mfma32x32x16(ra[ks % RA].f[i][st], bop[j], acc[i][j]);
                });
                if constexpr (SUMS && ks == 3) {
#pragma unroll
                    for (int i = 0; i < MT; i++)
#pragma unroll
                        for (int j = 0; j < NT; j++) acc[i][j] = mfma32x32x16(sf[i], Fm::bmin(cs[j]), acc[i][j]);
                }
                __builtin_amdgcn_sched_barrier(0);
            });
            if constexpr (more) {
#pragma unroll
                for (int j = 0; j < NT; j++) wcur[j] = wnext[j];
            }
        };
        if (b0 < b1) {
            const int cnt = b1 - b0;
            int b = b0;
            load_w(wcur, b);
            static_for<RA - 1>([&](auto KS) { load_a(b, KS); });
            for (int i = 1; i < cnt; i++) {
                asm volatile("" : "+v"(lane16));
                const int bn = b + 1 == b1 ? b0 : b + 1;
                block(b, bn, std::true_type{});
                b = bn;
            }
            block(b, b, std::false_type{});
        }
    } else {
        constexpr int D = 4;  // steps of fragments in registers
        half8v ra[D][MT], sf[MT];
        Wb wc[NT];
        auto load_a = [&](int b, auto U) {  // step U of super-block b
            constexpr int u = decltype(U)::value;
#pragma unroll
            for (int i = 0; i < MT; i++)
                ra[u % D][i] = __builtin_bit_cast(half8v, ld16(a_src[i] + ((size_t)(b * 17 + (u & ~3)) << 10), lane16 + (uint32_t)((u & 3) * 1024)));
        };
        auto load_w = [&](int b, auto KS) {
#pragma unroll
            for (int j = 0; j < NT; j++) wc[j].template load<decltype(KS)::value>(w_at(b, j), w_off[j], slot);
        };
        auto load_h = [&](int b) {
#pragma unroll
            for (int j = 0; j < NT; j++) wc[j].load_hdr(w_at(b, j), w_off[j], (uint32_t)r16, slot);
        };
        auto block = [&](int b, auto MORE) {
            constexpr bool more = decltype(MORE)::value;
            typename Fm::Consts cs[NT];
#pragma unroll
            for (int j = 0; j < NT; j++) cs[j] = Fm::consts(wc[j].hdr(), g32, ws);
            if constexpr (more) load_h(b + 1);
            if constexpr (SUMS) {
#pragma unroll
                for (int i = 0; i < MT; i++) sf[i] = __builtin_bit_cast(half8v, ld16(a_src[i] + ((size_t)(b * 17 + 16) << 10), lane16));
            }
            static_for<4>([&](auto KS) {
                constexpr int ks = decltype(KS)::value;
                static_for<4>([&](auto ST) {
                    constexpr int st = decltype(ST)::value, u = 4 * ks + st;
                    half8v bop[NT];
#pragma unroll
                    for (int j = 0; j < NT; j++) bop[j] = Fm::template operand<ks, st>(wc[j].template stage<ks>(), cs[j]);
#pragma unroll
                    for (int i = 0; i < MT; i++)
#pragma unroll
                        for (int j = 0; j < NT; j++) acc[i][j] = mfma32x32x16(ra[u % D][i], bop[j], acc[i][j]);
                    if constexpr (u + D < 16) load_a(b, std::integral_constant<int, u + D>{});
                    else if constexpr (more) load_a(b + 1, std::integral_constant<int, (u + D) & 15>{});
                });
                if constexpr (SUMS && ks == 3) {
#pragma unroll
                    for (int i = 0; i < MT; i++)
#pragma unroll
                        for (int j = 0; j < NT; j++) acc[i][j] = mfma32x32x16(sf[i], Fm::bmin(cs[j]), acc[i][j]);
                }
                if constexpr (more) load_w(b + 1, KS);
                __builtin_amdgcn_sched_barrier(0);
            });
        };
        if (b0 < b1) {
            load_h(b0);
            // (in the order of the loop, whose waits the compiler counts for both ways into it)
            static_for<4>([&](auto KS) {
                if constexpr (decltype(KS)::value == 3) static_for<D>([&](auto U) { load_a(b0, U); });
                load_w(b0, KS);
            });
            __builtin_amdgcn_sched_barrier(0);
            int b = b0;
            for (int i = b1 - b0; i > 1; i--) {
                asm volatile("" : "+v"(lane16));
                block(b, std::true_type{});
                b++;
            }
            block(b, std::false_type{});
        }
    }

    // ---- the waves meet: thread t adds up, of every tile, the four columns 4 (t % 8) .. + 3 of row t / 8 ----
    // (stored as they lie: 16 or 8 bytes per lane.  With a lane's four values in one column, as the MFMA leaves them, the stores were 4 us of a
    // launch of eight tiles per workgroup and 3 us of one of four)
    using M = Meet<MT, NT>;
    if constexpr (PAIR) {
        // thread: half a 16-byte chunk, 32 rows of which lie next to each other in a step of the fragments
        const float inv_g = 1.0f / grp.wscale[0], inv_u = 1.0f / grp.wscale[1];
        const float *bg = grp.bias[0], *bu = grp.bias[1];
        float *red = (float *)lds;
        const int half = tid & 1, row_l = (tid >> 1) & 31, chunk = (tid >> 6) & 1;
        uint32_t bad = 0;
#pragma unroll
        for (int r = 0; r < M::ROUNDS; r++) {
            if (r) __syncthreads();
#pragma unroll
            for (int t = 0; t < M::T; t++) {
                if (r * M::T + t >= MT * NT) continue;
                const int i = (r * M::T + t) / NT, j = (r * M::T + t) % NT;
#pragma unroll
                for (int e = 0; e < 16; e++) red[((wave * M::T + t) * 32 + 8 * (e >> 2) + 4 * g32 + (e & 3)) * kPitch + n32] = acc[i][j][e];
            }
            __syncthreads();
            for (int t = tid >> 7; t < M::T; t += 2) {
                const int tile = r * M::T + t;
                const int64_t mt = (int64_t)mb * MT + tile / NT, col = ((int64_t)nb * NT + tile % NT) * 16 + 8 * chunk + 4 * half;
                if (tile >= MT * NT || mt >= mtiles || col >= n) continue;
                const int at_lds = (t * 32 + row_l) * kPitch + 8 * chunk + 4 * half;
                float4v sg = *(const float4v *)(red + at_lds), su = *(const float4v *)(red + at_lds + 16);
#pragma unroll
                for (int v = 1; v < W; v++) {
                    sg += *(const float4v *)(red + v * (M::T * 32 * kPitch) + at_lds);
                    su += *(const float4v *)(red + v * (M::T * 32 * kPitch) + at_lds + 16);
                }
                float g[4], u[4];
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    g[e] = (sg[e] * inv_g + (bg ? bg[col + e] : 0.0f)) + 0.0f;
                    u[e] = (su[e] * inv_u + (bu ? bu[col + e] : 0.0f)) + 0.0f;
                }
                _Float16 h[4];
                silu_mul_f16<4>(g, u, mt * 32 + row_l < m, h, bad);
                const int cc = (int)(col & 255) >> 3;
                const int fg = yt ? (cc >> 1) & 1 : cc >> 4, q = yt ? 2 * (cc >> 2) + (cc & 1) : cc & 15;
                uint8_t *dst = (uint8_t *)grp.y[0] + ((size_t)((mt * (n >> 8) + (col >> 8)) * 17 + q) << 10);
                *(uint2v *)(dst + 16 * (row_l + 32 * fg) + 8 * half) = uint2v{as_u32(half2v{h[0], h[1]}), as_u32(half2v{h[2], h[3]})};
            }
        }
        turq_note_flush(bad);
        return;
    }
    const float inv_ws = 1.0f / pick.wscale;  // (a power of two: exact)
    const float *bias = pick.bias;
    void *y = pick.y;
    const int64_t ldy = pick.ldy;
    const int ytb = yt & 0xFF;
    const float lim = turq_finite_limit(ytb);
    uint32_t bad = 0;
    const int64_t row_t = (int64_t)mb * MT * 32 + (tid >> 3), col_t = (int64_t)nb * NT * 32 + 4 * (tid & 7);
    float *red = (float *)lds;  // [wave][tile of the round][row][kPitch]
#pragma unroll
    for (int r = 0; r < M::ROUNDS; r++) {
        // with TURQ_OUT_ACCUMULATE: what y holds, requested together and ahead of the round, so that it arrives under the meeting
        float4v old[M::T];
#pragma unroll
        for (int t = 0; t < M::T; t++) {
            old[t] = float4v{0.0f, 0.0f, 0.0f, 0.0f};
            const int tile = r * M::T + t;
            if (tile >= MT * NT || !(yt & TURQ_OUT_ACCUMULATE)) continue;
            const int64_t row = row_t + tile / NT * 32, col = col_t + tile % NT * 32, at = row * ldy + col;
            if (row >= m || col >= n) continue;
            if (vec_out) {
                if (ytb == TURQ_ACT_F32) {
                    old[t] = *(const float4v *)((const float *)y + at);
                } else {
                    const uint2v u = *(const uint2v *)((const uint16_t *)y + at);
                    if (ytb == TURQ_ACT_BF16) {
                        old[t] = float4v{__uint_as_float(u.x << 16), __uint_as_float(u.x & 0xFFFF0000u), __uint_as_float(u.y << 16), __uint_as_float(u.y & 0xFFFF0000u)};
                    } else {
                        const half2v a = as_half2(u.x), c = as_half2(u.y);
                        old[t] = float4v{(float)a.x, (float)a.y, (float)c.x, (float)c.y};
                    }
                }
            } else {
#pragma unroll
                for (int e = 0; e < 4; e++)
                    if (col + e < n)
                        old[t][e] = ytb == TURQ_ACT_F32 ? turq_load_out<TURQ_ACT_F32>(y, at + e)
                                  : ytb == TURQ_ACT_BF16 ? turq_load_out<TURQ_ACT_BF16>(y, at + e) : turq_load_out<TURQ_ACT_F16>(y, at + e);
            }
        }
        if (r) __syncthreads();
#pragma unroll
        for (int t = 0; t < M::T; t++) {
            if (r * M::T + t >= MT * NT) continue;
            const int i = (r * M::T + t) / NT, j = (r * M::T + t) % NT;
            // lane (n32, g32), register e: row 8 (e / 4) + 4 g32 + e % 4 of column n32
#pragma unroll
            for (int e = 0; e < 16; e++) red[((wave * M::T + t) * 32 + 8 * (e >> 2) + 4 * g32 + (e & 3)) * kPitch + n32] = acc[i][j][e];
        }
        __syncthreads();
#pragma unroll
        for (int t = 0; t < M::T; t++) {
            const int tile = r * M::T + t;
            if (tile >= MT * NT) continue;
            const int at_lds = (t * 32 + (tid >> 3)) * kPitch + 4 * (tid & 7);
            float4v s = *(const float4v *)(red + at_lds);
#pragma unroll
            for (int v = 1; v < W; v++) s += *(const float4v *)(red + v * (M::T * 32 * kPitch) + at_lds);
            const int64_t row = row_t + tile / NT * 32, col = col_t + tile % NT * 32, at = row * ldy + col;
            if (row >= m || col >= n) continue;
            float o[4];
#pragma unroll
            for (int e = 0; e < 4; e++) o[e] = (s[e] * inv_ws + (bias && col + e < n ? bias[col + e] : 0.0f)) + old[t][e];
            if (vec_out) {
#pragma unroll
                for (int e = 0; e < 4; e++) turq_note_accum(o[e], lim, bad);
                if (ytb == TURQ_ACT_F32) {
                    *(float4v *)((float *)y + at) = float4v{o[0], o[1], o[2], o[3]};
                } else if (ytb == TURQ_ACT_BF16) {
                    *(uint2v *)((uint16_t *)y + at) = uint2v{turq_f2bf_x2(o[0], o[1]), turq_f2bf_x2(o[2], o[3])};
                } else {
                    *(uint2v *)((uint16_t *)y + at) = uint2v{as_u32(half2v{(_Float16)o[0], (_Float16)o[1]}), as_u32(half2v{(_Float16)o[2], (_Float16)o[3]})};
                }
            } else {
#pragma unroll
                for (int e = 0; e < 4; e++)
                    if (col + e < n) turq_store_any(y, ytb, at + e, o[e]);
            }
        }
    }
    turq_note_flush(bad);
}

// MINB: workgroups that are to share a CU (2: the tight form of the 64 x 64 tile in 256 registers; otherwise what the tile leaves)
template <int DTA, int DTB, int MT, int NT, bool TIGHT, int MINB, bool PAIR>
__global__ void __launch_bounds__(64 * W, MINB) gemm_cols_kernel(ColsGroup grp, int64_t k, const uint8_t *__restrict__ frags, int64_t m, int yt,
                                                           int nblocks_n, int nblocks_m, int vec_out) {
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    // consecutive logical ids run on one XCD (blockIdx % 8): the m-blocks of one n-block share its packed weights in that XCD's L2.  Also where
    // the workgroups are no multiple of 8 (the first XCDs have one more): with ids as they come there, Q8_0 18944 x 1024 at 300 rows (990
    // workgroups) took 47.3 us instead of 41.3
    const int nwg = nblocks_n * nblocks_m, xcd = (int)blockIdx.x & 7, extra = nwg & 7;
    const int lid = xcd * (nwg >> 3) + (xcd < extra ? xcd : extra) + ((int)blockIdx.x >> 3);
    const int mb = lid % nblocks_m, nb_all = lid / nblocks_m;
    ColsPick p{grp.w[0], grp.y[0], grp.bias[0], grp.n[0], grp.ldy[0], grp.wscale[0], 0, 0};
    if constexpr (!PAIR) {
#pragma unroll
        for (int i = 1; i < kMaxGroup; i++) {  // (selects, no branches)
            const bool in = nb_all >= grp.first[i];
            p.w = in ? grp.w[i] : p.w, p.y = in ? grp.y[i] : p.y, p.bias = in ? grp.bias[i] : p.bias, p.n = in ? grp.n[i] : p.n;
            p.ldy = in ? grp.ldy[i] : p.ldy, p.wscale = in ? grp.wscale[i] : p.wscale, p.index = in ? i : p.index, p.first = in ? grp.first[i] : p.first;
        }
    }
    const int nb = nb_all - p.first;
    if (DTA == DTB || p.index < grp.second) cols_body<DTA, MT, NT, TIGHT, PAIR>(grp, p, nb, mb, k, frags, m, yt, vec_out, lds);
    else cols_body<DTB, MT, NT, TIGHT, PAIR>(grp, p, nb, mb, k, frags, m, yt, vec_out, lds);
}

template <int DTA, int DTB, int MT, int NT, bool TIGHT = false, int MINB = 1, bool PAIR = false>
hipError_t launch_cols(const TurqGemmWeights &ws, int second, int64_t k, const void *frags, int64_t m, int yt, hipStream_t stream,
                       hipEvent_t ev_start, hipEvent_t ev_stop) {
    const auto kernel = gemm_cols_kernel<DTA, DTB, MT, NT, TIGHT, MINB, PAIR>;
    constexpr int LDS_BYTES = Meet<MT, NT>::LDS;
    static_assert(LDS_BYTES <= 64 * 1024, "no raised LDS limit");
    ColsGroup grp{};
    grp.second = second;
    for (int i = ws.count; i < kMaxGroup; i++) grp.first[i] = INT_MAX;
    const int es = (yt & 0xFF) == TURQ_ACT_F32 ? 4 : 2;
    int nbn = 0, vec_out = 1;  // rows of y can be written four aligned columns at a time (every weight of the launch, or none)
    for (int i = 0; i < ws.count; i++) {
        vec_out = vec_out && (uintptr_t)ws.y[i] % (4 * es) == 0 && ws.ldy[i] % 4 == 0 && ws.n[i] % 4 == 0;
        grp.w[i] = (const uint8_t *)ws.w[i];
        grp.y[i] = ws.y[i];
        grp.bias[i] = ws.bias[i];
        grp.n[i] = ws.n[i];
        grp.ldy[i] = ws.ldy[i];
        grp.wscale[i] = ws.wscale[i];
        grp.first[i] = nbn;
        if (PAIR) nbn = (int)((ws.n[i] + 16 * NT - 1) / (16 * NT));
        else nbn += (int)((ws.n[i] + 32 * NT - 1) / (32 * NT));
    }
    const int nbm = (int)((m + 32 * MT - 1) / (32 * MT));
    const dim3 grid((unsigned)(nbn * nbm)), block(64 * W);
    if (ev_start)
        hipExtLaunchKernelGGL(kernel, grid, block, LDS_BYTES, stream, ev_start, ev_stop, 0, grp, k, (const uint8_t *)frags, m, yt, nbn, nbm, vec_out);
    else
        kernel<<<grid, block, LDS_BYTES, stream>>>(grp, k, (const uint8_t *)frags, m, yt, nbn, nbm, vec_out);
    return hipGetLastError();
}

int64_t cols_workgroups(int tile, int count, const int64_t *n, int64_t m) {
    int64_t nbn = 0;
    for (int i = 0; i < count; i++) nbn += (n[i] + 32 * (tile % 10) - 1) / (32 * (tile % 10));
    return nbn * ((m + 32 * (tile / 10) - 1) / (32 * (tile / 10)));
}

template <int DTA, int DTB>
hipError_t launch_tile(int tile, const TurqGemmWeights &ws, int second, int64_t k, const void *frags, int64_t m, int yt, int64_t cus,
                       hipStream_t stream, hipEvent_t ev_start, hipEvent_t ev_stop) {
    switch (tile) {
#define TURQ_COLS(MT, NT, ...) launch_cols<DTA, DTB, MT, NT, ##__VA_ARGS__>(ws, second, k, frags, m, yt, stream, ev_start, ev_stop)
    case 11: return TURQ_COLS(1, 1);
    case 21: return TURQ_COLS(2, 1);
    case 31: return TURQ_COLS(3, 1);
    case 22:  // (more than one workgroup per CU: two of them at a time)
        if (cols_workgroups(22, ws.count, ws.n, m) > cus) return TURQ_COLS(2, 2, true, 2);
        return TURQ_COLS(2, 2);
    case 32: return TURQ_COLS(3, 2);
    case 23: return TURQ_COLS(2, 3);
    case 42: return TURQ_COLS(4, 2);
    case 33: return TURQ_COLS(3, 3, true);  // (the first form spills here)
#undef TURQ_COLS
    default: return hipErrorInvalidValue;
    }
}

// the pair's tiles: of those above, without two that the estimates hardly ever pick for two weights
constexpr int kPairTiles[] = {11, 21, 22, 32, 42, 33};
template <int DT>
hipError_t launch_pair(int tile, const TurqGemmWeights &ws, int64_t k, const void *frags, int64_t m, int yt, int64_t cus, hipStream_t stream,
                       hipEvent_t ev_start, hipEvent_t ev_stop) {
    const int64_t n2 = 2 * ws.n[0];
#define TURQ_COLS(MT, NT, TIGHT, MINB) launch_cols<DT, DT, MT, NT, TIGHT, MINB, true>(ws, 2, k, frags, m, yt, stream, ev_start, ev_stop)
    switch (tile) {
    case 11: return TURQ_COLS(1, 1, false, 1);
    case 21: return TURQ_COLS(2, 1, false, 1);
    case 22:
        if (cols_workgroups(22, 1, &n2, m) > cus) return TURQ_COLS(2, 2, true, 2);
        return TURQ_COLS(2, 2, false, 1);
    case 32: return TURQ_COLS(3, 2, false, 1);
    case 42: return TURQ_COLS(4, 2, false, 1);
    case 33: return TURQ_COLS(3, 3, true, 1);
    default: return hipErrorInvalidValue;
    }
#undef TURQ_COLS
}

// bytes of one row tile's super-blocks, the larger of the two formats'
size_t row_tile_bytes(int dtype_a, int dtype_b, int64_t k) {
    return (size_t)(k / 256) * (size_t)std::max(turq_tile_bytes(dtype_a), turq_tile_bytes(dtype_b));
}

}  // namespace

bool turq_gemm_cols_mixed(int dtype_a, int dtype_b) { return (dtype_a == TURQ_Q4_K || dtype_a == TURQ_Q5_K) && dtype_b == TURQ_Q6_K; }

// What one launch of this kernel takes: one round over the CUs is `base` plus `per` for every super-block of 256 columns, the latter `fill`
// longer on a chip that is full (L2 and clock); a further round costs `again` of that and `more` for the part of it that is there.  Fitted to
// 628 launches (n 1024 .. 24576, k 1024 .. 18944, 40 .. 512 rows, weights from HBM), with an error of 6 % and of 25 % at most.
struct ColsCost { int tile; double base, per[4], again, more, fill; };  // per: Q4_K, Q5_K, Q6_K, Q8_0
static constexpr ColsCost kColsCost[] = {
    {11, 2.58, {0.229, 0.270, 0.288, 0.277}, 0.51, 0.30, 0.33}, {21, 3.21, {0.375, 0.418, 0.433, 0.432}, 0.58, 0.31, 0.22},
    {31, 3.58, {0.489, 0.528, 0.540, 0.547}, 0.60, 0.29, 0.29}, {22, 4.58, {0.498, 0.594, 0.652, 0.591}, 0.88, 0.25, 0.31},
    {32, 5.48, {0.647, 0.748, 0.775, 0.721}, 0.79, 0.28, 0.43}, {23, 5.80, {0.674, 0.843, 0.929, 0.868}, 0.62, 0.41, 0.47},
    {42, 6.95, {0.789, 0.893, 0.880, 0.880}, 0.74, 0.30, 0.54}, {33, 7.00, {0.919, 1.062, 1.116, 1.467}, 0.61, 0.39, 0.53},
};
static constexpr ColsCost kColsPair = {22, 3.84, {0.604, 0.707, 0.741, 0.715}, 0.42, 0.41, 0.25};  // two workgroups per CU

// ... unless the activations are what takes the time: fragments larger than an XCD's 4 MB of L2 come from the memory side again for every 32 NT
// rows of weights, and only the n-blocks that an XCD works on at a time share them.  In launches of several rounds of the smaller tiles that goes at
// 2 (64 x 64: 2.4) TB/s for each such n-block and 6.8 at least (120 shapes of 40 .. 2040 rows in every tile: 32 x 32 took up to 2.5 times the line above
// at 8 MB of fragments and more, 64 x 64 up to 1.5; from 96 x 64 on the line holds).  Q8_0 2 x 2560 x 5376 at 1953 rows: 64 x 64 241 us, 128 x 64 183.
static double cols_frag_us(int tile, int64_t n_blocks, int64_t k, int64_t m, int64_t cus, double x) {
    const double frag_mb = 2e-6 * (double)m * (double)k;
    if (x <= 1.0 || frag_mb <= 4.2 || (tile / 10) * (tile % 10) > 4) return 0.0;
    const int per_cu = tile == 22 ? 2 : 3;
    const double at_once = (double)(cus / 8 * per_cu) / (double)((m + 32 * (tile / 10) - 1) / (32 * (tile / 10)));
    return (double)n_blocks * frag_mb / std::max(6.8, (tile == 22 ? 2.4 : 2.0) * at_once);
}

static double cols_us(int tile, int dtype_a, int dtype_b, int count, const int64_t *n, int64_t k, int64_t m, int64_t cus) {
    const auto fmt = [](int dt) { return dt == TURQ_Q4_K ? 0 : dt == TURQ_Q5_K ? 1 : dt == TURQ_Q6_K ? 2 : 3; };
    const int64_t wgs = cols_workgroups(tile, count, n, m);
    const double x = (double)wgs / (double)cus;
    const ColsCost *c = &kColsPair;
    if (tile != 22 || x <= 1.0)
        for (const ColsCost &t : kColsCost)
            if (t.tile == tile) c = &t;
    return std::max(turq_launch_model_us(c->base, std::max(c->per[fmt(dtype_a)], c->per[fmt(dtype_b)]) * (double)(k / 256), c->again, c->more, c->fill, x),
                    cols_frag_us(tile, wgs / ((m + 32 * (tile / 10) - 1) / (32 * (tile / 10))), k, m, cus, x));
}

// Whether a launch of one weight in 32 x 32 tiles that is more than one round over the CUs goes out as one of 64 x 32, two of them one under the other:
// the same sums in the same order, and one round instead of a second for half of the CUs.  By the estimates, which for these two are right to a few
// percent: Q6_K 4096 x 12288 at 65 - 96 rows 34.4 -> 27.4 us, 2048 x 6144 at 150 18.7 -> 17.0, Q5_K / Q4_K 4096 x 4096 at 77 13.4 / 11.9 -> 12.2 / 11.2; not of
// Q8_0, of which three workgroups on a CU lose less (1024 x 2048 at 300 rows 8.1 -> 8.3), nor for a handful of workgroups beyond the round, which the
// estimates do not see: 4096 columns at 46 rows, 32 x 32 / 64 x 32, 260 workgroups Q4_K 12.8 / 14.2, Q5_K 14.0 / 14.7, Q6_K 14.7 / 15.0, but 272 14.0 / 14.0, 15.7 / 14.6 and
// 16.5 / 15.1.
static bool two_under_another(int dtype, const int64_t *n, int64_t k, int64_t m, int64_t cus) {
    if (dtype == TURQ_Q8_0 || cols_workgroups(11, 1, n, m) <= cus + cus / 32 || cols_workgroups(21, 1, n, m) > cus) return false;
    return cols_us(21, dtype, dtype, 1, n, k, m, cus) < cols_us(11, dtype, dtype, 1, n, k, m, cus);
}

// The tile with which one weight goes through this kernel as far as single rounds over the CUs decide, 0: gemm_kq_kernel.
// A launch of one round takes about base + per_sb * super-blocks, one line for every format; a further round costs as much again without the
// launch itself, of the smallest tile, of which three workgroups share a CU, three fifths of it.  So the smallest tile that makes the launch one
// round is taken, and the smallest of all up to one and a half (K-quants: two of them per workgroup where that makes one round, two_under_another).  Against gemm_kq_kernel:
//   one or two MFMA tiles: Q4_K 1024 x 4096 at 40 / 300 / 512 rows 13.0 / 19.0 / 19.1 -> 6.6 / 9.3 / 10.7 us, 4096 x 4096 at 40 / 100 rows 19.2 /
//   22.6 -> 8.7 / 11.3, Q6_K 4096 x 12288 33 / 43 -> 23 / 29, Q8_0 2048 x 2048 15 -> 5.4 / 5.5;
//   three or four: K-quants from two super-blocks on (Q4_K 12288 x 256 at 48 rows 8.4 -> 9.4); Q8_0 2048 x 2048 at 300 / 512 rows 15.4 -> 8.5 / 10.2, Q4_K 4096 x 4096 at 256 24 -> 15;
//   six: from 12 super-blocks on (Q4_K 4096 x 4096 at 300 rows 23.4 -> 20.4, Q6_K 4096 x 12288 74 -> 51; with 4 super-blocks Q8_0 6144 x 1024
//   at 160 rows 11.1 -> 11.7);
//   eight: from 40 super-blocks on, Q6_K from 24 (512 rows, 4096 x 12288: Q4_K 66 -> 64, Q5_K 76 -> 69, Q6_K 81 -> 66; 4096 x 4096: Q4_K 26.3 -> 27.5).
// Q8_0, whose tile in gemm_kq_kernel is the narrow 128 x 64, takes whichever kernel has the smaller estimate, in any number of rounds
// (4096 x 4096 at 512 / 700 rows 31 / 53 -> 29 / 41, 4096 x 12288 at 1024 / 2048 rows 160 / 300 -> 126 / 283).
static int cols_tile_by_rounds(int dtype, int64_t n, int64_t k, int64_t m, int64_t cus, int compute_units) {
    static constexpr struct { int mt, nt; double base, per_sb; } kTiles[] = {{1, 1, 3.2, 0.40}, {2, 1, 4.0, 0.52}, {3, 1, 4.6, 0.60}, {2, 2, 5.2, 0.68},
                                                                             {3, 2, 6.2, 0.92}, {2, 3, 6.2, 0.92}, {4, 2, 7.0, 1.20}};
    const bool eight = dtype == TURQ_Q8_0;
    const int64_t ntc = k / 256;
    double best_us = eight ? turq_gemm_launch_us(dtype, 1, &n, k, m, compute_units) : 1e30;
    int best = 0;
    for (const auto &c : kTiles) {
        const int area = c.mt * c.nt;
        const int64_t wgs = cols_workgroups(10 * c.mt + c.nt, 1, &n, m);
        if (!eight) {
            if (wgs > (area == 1 ? cus + cus / 2 : cus)) continue;
            if (area == 4 && ntc < 2) continue;
            if (area > 4 && ntc < (area == 6 ? 12 : dtype == TURQ_Q6_K ? 24 : 40)) continue;
        }
        const double x = (double)wgs / (double)cus;
        const double rounds = x <= 1.0 ? 1.0 : area == 1 ? 1.0 + 0.6 * (x - 1.0) : (double)((wgs + cus - 1) / cus);
        const double est = kTurqLaunchUs + (c.base + c.per_sb * (double)ntc - kTurqLaunchUs) * rounds;
        if (est < best_us) {
            best = 10 * c.mt + c.nt;
            best_us = est;
        }
    }
    return best;
}

// The tile (10 * MT + NT) with which `count` weights of n[i] rows and k columns go through this kernel in one launch, 0 where the launch
// is gemm_kq_kernel's; *us: roughly what it takes.
//
// One weight: by the rounds, unless another tile's estimate over several rounds is a fifth (Q8_0: a quarter and a bit) below what that launch
// takes: the estimates err by up to that much, and launches of more than one round are where the rounds alone misjudge (at 300 rows, 128 x 128 -> two
// 64 x 64 workgroups per CU: Q4_K / Q5_K / Q6_K 6144 x 4096 36 / 42 / 40 -> 25 / 28 / 30 us, 6144 x 1024 13.3 / 15.0 / 14.6 -> 9.9 / 10.8 / 11.5; at 180
// rows, 128 x 128 -> 96 x 96: Q5_K 12288 x 4096 45 -> 32).  Not of one super-block, which is mostly epilogue and which the estimates were not
// fitted to (Q5_K 14336 x 256 at 645 rows 26 us by the rounds, 35 by the estimates; Q8_0 4096 x 256 twice at 1001 rows 25 and 30; from two super-blocks
// on the estimates are ahead in 9 of 10).
// Several weights, each of which is this kernel's alone: together, by the estimates, where that is less than one after the other (gate and up of
// an 8B model at 77 rows, Q5_K 2 x 12288 x 4096: 45 -> 34), of Q8_0 also where they are up to 5 % above it (41 pairs of 1 - 2 rounds that the estimates
// had up to 7 % above took 0.94 - 1.07 of that, on average 0.99).
int turq_gemm_cols_tile(int dtype_a, int dtype_b, int count, const int64_t *n, int64_t k, int64_t m, int compute_units, double *us) {
    const TurqTuning &t = turq_tuning();
    const bool kq_forced = t.gemm_wide >= 0 || t.gemm_low >= 0 || t.gemm_split >= 0 || t.gemm_kgroups != 0 || t.gemm_grid_2x2 || t.gemm_merge >= 0;
    if (us) *us = 0.0;
    if (t.gemm_cols == 0 || (t.gemm_cols < 0 && kq_forced)) return 0;
    if (!turq_dt_is_quant(dtype_a) || (dtype_b != dtype_a && !turq_gemm_cols_mixed(dtype_a, dtype_b))) return 0;
    if (count < 1 || count > kMaxGroup || m <= 0 || k <= 0 || k % 256 != 0) return 0;
    // a lane's offset to the last of its 16-row tiles is 32-bit, here and in gemm_kq_kernel, whose n-blocks of eight row tiles (Q8_0: four)
    // decide: columns that it refuses are not taken instead (six row tiles are the most of a workgroup here)
    if (row_tile_bytes(dtype_a, dtype_b, k) >= (1ull << 32) / (dtype_a == TURQ_Q8_0 ? 6 : 8)) return 0;
    if (t.gemm_cols > 0) return t.gemm_cols;
    const int64_t cus = compute_units > 0 ? compute_units : 256;
    int best = 0;
    double best_us = 0.0, least = 0.0;  // the launch to be beaten, and below what
    if (count == 1) {
        best = cols_tile_by_rounds(dtype_a, n[0], k, m, cus, compute_units);
        best_us = best ? cols_us(best, dtype_a, dtype_a, 1, n, k, m, cus) : turq_gemm_kq_us(dtype_a, n[0], k, m, compute_units);
        least = k < 512 ? 0.0 : best_us / (dtype_a == TURQ_Q8_0 ? 1.27 : 1.2);
    } else {
        for (int i = 0; i < count; i++) {
            double alone = 0.0;  // (of a mixed launch as if of the first format: the estimate only has to order)
            if (!turq_gemm_cols_tile(dtype_a, dtype_a, 1, n + i, k, m, compute_units, &alone)) return 0;
            least += alone;
        }
        if (dtype_a == TURQ_Q8_0) least *= 1.05;
    }
    for (const ColsCost &c : kColsCost) {
        const double est = cols_us(c.tile, dtype_a, dtype_b, count, n, k, m, cus);
        if (est < least) {
            best = c.tile;
            best_us = least = est;
        }
    }
    if (us && best) *us = best_us;
    // (The time stays that of 32 x 32, what several weights together are held against: of 60000 calls of two or three weights 19 change with the other, and
    // eight of those, some of which went out together only so, took 0.87 - 1.19 of the time.)
    if (count == 1 && best == 11 && two_under_another(dtype_a, n, k, m, cus)) best = 21;
    return best;
}

// frags: as for turq_launch_gemm_mfma, in the order of the formats (Q8_0, or the K-quants); weights from `second` on are of dtype_b
hipError_t turq_launch_gemm_cols(int dtype_a, int dtype_b, int second, int tile, const TurqGemmWeights &ws, int64_t k, const void *frags, int64_t m,
                                 int y_dtype, int compute_units, hipStream_t stream, hipEvent_t ev_start, hipEvent_t ev_stop) {
    if (ws.count < 1 || ws.count > kMaxGroup || k <= 0 || k % 256 != 0 || k / 256 > (1 << 20)) return hipErrorInvalidValue;
    int64_t n = 0;
    for (int i = 0; i < ws.count; i++) {
        if (ws.n[i] <= 0) return ws.count == 1 && ws.n[i] == 0 ? hipSuccess : hipErrorInvalidValue;
        if (!(ws.wscale[i] >= 6.103515625e-5f && ws.wscale[i] <= 32768.0f)) return hipErrorInvalidValue;
        n += ws.n[i];
    }
    if (m == 0) return hipSuccess;
    if (row_tile_bytes(dtype_a, second < ws.count ? dtype_b : dtype_a, k) * 2 * (size_t)(tile % 10) >= (1ull << 32)) return hipErrorInvalidValue;
    if ((n / 32 + ws.count) * ((m + 31) / 32) > 0x7FFFFFFF) return hipErrorInvalidValue;
#define TURQ_COLS_TILE(A, B) return launch_tile<A, B>(tile, ws, second, k, frags, m, y_dtype, compute_units > 0 ? compute_units : 256, stream, ev_start, ev_stop)
    if (dtype_a != dtype_b && second < ws.count) {
        if (dtype_a == TURQ_Q4_K && dtype_b == TURQ_Q6_K) TURQ_COLS_TILE(TURQ_Q4_K, TURQ_Q6_K);
        if (dtype_a == TURQ_Q5_K && dtype_b == TURQ_Q6_K) TURQ_COLS_TILE(TURQ_Q5_K, TURQ_Q6_K);
        return hipErrorInvalidValue;
    }
    switch (dtype_a) {
    case TURQ_Q4_K: TURQ_COLS_TILE(TURQ_Q4_K, TURQ_Q4_K);
    case TURQ_Q5_K: TURQ_COLS_TILE(TURQ_Q5_K, TURQ_Q5_K);
    case TURQ_Q6_K: TURQ_COLS_TILE(TURQ_Q6_K, TURQ_Q6_K);
    case TURQ_Q8_0: TURQ_COLS_TILE(TURQ_Q8_0, TURQ_Q8_0);
    default: return hipErrorInvalidValue;
    }
#undef TURQ_COLS_TILE
}

// The tile with which gate and up of n rows each go through this kernel as a pair, by the estimates; *us: what that takes.  0: there is none.
int turq_gemm_cols_pair_tile(int dtype, int down_dtype, int64_t n, int64_t k, int64_t m, int compute_units, double *us) {
    *us = 0.0;
    if (!turq_dt_is_quant(dtype) || (down_dtype != TURQ_Q6_K && down_dtype != TURQ_Q8_0)) return 0;
    if (n <= 0 || n % 256 != 0 || k <= 0 || k % 256 != 0 || m <= 0) return 0;
    const int64_t n2 = 2 * n;
    const int forced = turq_tuning().gemm_cols;
    int best = 0;
    for (const int tile : kPairTiles) {
        if (forced > 0 && tile != forced) continue;
        const double est = cols_us(tile, dtype, dtype, 1, &n2, k, m, compute_units > 0 ? compute_units : 256);
        if (!best || est < *us) {
            best = tile;
            *us = est;
        }
    }
    return best;
}

// gate and up (ws.w[0], ws.w[1]; one shape, n a multiple of 256) as a pair: down_proj's fragments, turq_act_prep32_bytes(m, n) bytes at ws.y[0]
hipError_t turq_launch_gemm_cols_pair(int dtype, int down_dtype, int tile, const TurqGemmWeights &ws, int64_t k, const void *frags, int64_t m,
                                      int compute_units, hipStream_t stream, hipEvent_t ev_start, hipEvent_t ev_stop) {
    if (ws.count != 2 || ws.n[0] != ws.n[1] || ws.n[0] <= 0 || ws.n[0] % 256 != 0 || k <= 0 || k % 256 != 0 || k / 256 > (1 << 20)) return hipErrorInvalidValue;
    if (down_dtype != TURQ_Q6_K && down_dtype != TURQ_Q8_0) return hipErrorInvalidValue;
    for (int i = 0; i < 2; i++)
        if (!(ws.wscale[i] >= 6.103515625e-5f && ws.wscale[i] <= 32768.0f)) return hipErrorInvalidValue;
    if (m == 0) return hipSuccess;
    if ((ws.n[0] / 16 + 1) * ((m + 31) / 32) > 0x7FFFFFFF) return hipErrorInvalidValue;
    const int64_t cus = compute_units > 0 ? compute_units : 256;
    const int q8_order = down_dtype == TURQ_Q8_0 ? 1 : 0;
    switch (dtype) {
    case TURQ_Q4_K: return launch_pair<TURQ_Q4_K>(tile, ws, k, frags, m, q8_order, cus, stream, ev_start, ev_stop);
    case TURQ_Q5_K: return launch_pair<TURQ_Q5_K>(tile, ws, k, frags, m, q8_order, cus, stream, ev_start, ev_stop);
    case TURQ_Q6_K: return launch_pair<TURQ_Q6_K>(tile, ws, k, frags, m, q8_order, cus, stream, ev_start, ev_stop);
    case TURQ_Q8_0: return launch_pair<TURQ_Q8_0>(tile, ws, k, frags, m, q8_order, cus, stream, ev_start, ev_stop);
    default: return hipErrorInvalidValue;
    }
}

TURQ_NONFINITE_READER(turq_nonfinite_gemm_cols)
