// What the matrix-matrix kernels (gemm_mfma.hip, gemm_cols.hip) share: the MFMA shape, the LDS reads of the former, and per format
// the way from a lane's packed weights to the f16 operands of v_mfma_f32_32x32x16_f16.
#pragma once
#include <type_traits>
#include <utility>

#include "layout.h"
#include "mfma_common.h"

namespace {

typedef float float16v __attribute__((ext_vector_type(16)));

constexpr uint32_t kMagic1024 = 0x64006400u;  // 1024.0: a nibble in mantissa bits 0..3 reads as 1024 + n
constexpr uint32_t kMagic64 = 0x54005400u;    // 64.0:   a nibble in mantissa bits 4..7 reads as 64 + n
constexpr uint32_t kMagic256 = 0x5C005C00u;   // 256.0:  a 6-bit value in mantissa bits 2..7 reads as 256 + q
constexpr int kCoherent = 16;                 // cache policy of buffer loads and stores that other XCDs must see: sc1, as device-scope atomics carry

template <int... I, typename F> __device__ inline void static_for_impl(std::integer_sequence<int, I...>, F &&f) {
    (f(std::integral_constant<int, I>{}), ...);
}
// f(integral_constant<int, 0>) ... f(integral_constant<int, N - 1>): loop indices usable as template arguments
template <int N, typename F> __device__ inline void static_for(F &&f) { static_for_impl(std::make_integer_sequence<int, N>{}, f); }

__device__ inline _Float16 h_from_bits(uint32_t bits16) {
    const uint16_t u = (uint16_t)bits16;
    _Float16 h;
    __builtin_memcpy(&h, &u, 2);
    return h;
}

__device__ inline float16v mfma32x32x16(half8v a, half8v b, float16v c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

// wait until at most N of this wave's LDS reads are outstanding
template <int N> __device__ inline void wait_lds() { asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(N) : "memory"); }
// a value read by lds_read128 may be used only after a wait; passing it through an (empty) volatile
// statement placed after that wait keeps its users from being scheduled ahead of the wait (the value it yields is a new one
// to the compiler, so no copy made earlier can stand in for it).  What the compiler could still do is copy or spill the
// register between the read and the wait; the build walks the device assembly of this file and fails if any instruction
// touches the destination of an LDS read before the wait that covers it, or if a kernel here spills (check_lds_waits.py).
template <typename T> __device__ inline void pin(T &v) { asm volatile("" : "+v"(v)); }

template <int OFF, typename T> __device__ inline void lds_read128(T &dst, uint32_t addr) {
    static_assert(sizeof(T) == 16 && OFF >= 0 && OFF < 65536, "one ds_read_b128");
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(dst) : "v"(addr), "n"(OFF));
}

template <int OFF> __device__ inline void lds_read64(uint2v &dst, uint32_t addr) {
    asm volatile("ds_read_b64 %0, %1 offset:%2" : "=v"(dst) : "v"(addr), "n"(OFF));
}
template <int OFF> __device__ inline void lds_read32(uint32_t &dst, uint32_t addr) {
    asm volatile("ds_read_b32 %0, %1 offset:%2" : "=v"(dst) : "v"(addr), "n"(OFF));
}
template <int OFF> __device__ inline void lds_read16(uint32_t &dst, uint32_t addr) {
    asm volatile("ds_read_u16 %0, %1 offset:%2" : "=v"(dst) : "v"(addr), "n"(OFF));
}

// SiLU(g) * u in f16, the values of silu_mul_kernel and act_prep32_kernel<.., GU> (zeros where !live), and the sum of the rounded values in
// order.  With one wave per SIMD the epilogue that calls this is bound by its vector instructions, so what is no finite number is looked
// for without a compare per element: bad is set where a product is not (x * 0 stays 0 for finite x), and the rounded values are counted only
// where their sum shows one that is not (no eight finite f16 values add up to an infinity).
template <int N> __device__ inline float silu_mul_f16(const float (&g)[N], const float (&u)[N], bool live, _Float16 (&h)[N], uint32_t &bad) {
    static_assert(N <= 8, "sums of finite values stay finite");
    float v[N], fin = 0.0f, sum = 0.0f;
#pragma unroll
    for (int e = 0; e < N; e++) {
        fin = __builtin_fmaf(g[e], 0.0f, fin);
        fin = __builtin_fmaf(u[e], 0.0f, fin);
        v[e] = live ? g[e] / (1.0f + expf(-g[e])) * u[e] : 0.0f;
        h[e] = (_Float16)v[e];
        sum += (float)h[e];
    }
    bad |= live && !(fin == 0.0f) ? 1u : 0u;
    if (__builtin_expect(!(__builtin_fabsf(sum) < __builtin_inff()), 0)) turq_note_results<TURQ_ACT_F16>(v);
    return sum;
}

template <int I> __device__ inline uint32_t word_of(uint4v v) { return I == 0 ? v.x : I == 1 ? v.y : I == 2 ? v.z : v.w; }


// ---- per-format pieces -------------------------------------------------------------------------------------
// A lane (n32, g32) of a 32-row B tile works on row r16 = n32 % 16 of 16-row tile n32 / 16 and on that tile's lane
// slots 2 g32 and 2 g32 + 1 (64 columns each).  Stage ks of a super-block covers the 32 columns of half (ks & 1) of
// slot 2 g32 + (ks >> 1): operand steps i = 4 (ks & 1) + st, st = 0..3, of that slot.
//   Stage   what a lane reads from the LDS for one stage and one 32-row tile (NSTG reads)
//   Hdr     what it reads once per super-block (NHDR reads)
//   Consts  packed-f16 constants derived from Hdr
//   `tile` is the LDS address of the lane's 16-row tile in the weight ring entry.
template <int DT> struct GFmt;

struct K4Consts {
    half2v s[4], s16[4], c1[4], c2[4];  // per sub-block u = ks: d*sc, d*sc/16, -1024*d*sc, -64*d*sc (both halves equal)
    half8v bmin;                        // -(dmin*m_u) twice each, against the (hi, lo) sums fragment
};

// constants of the lane's four sub-blocks u (sub-block 4 * g32 + u of the super-block) from a Q4_K / Q5_K header row
__device__ inline K4Consts k4_consts(uint4v hd, int g32, _Float16 ws) {
    // 24-bit groups of lane slots 2*g32 and 2*g32+1 inside the 96-bit field hd.y, hd.z, hd.w
    // (both candidates are computed and selected: a divergent branch would cost more than the two shifts)
    const uint32_t g0a = hd.y, g0b = __builtin_amdgcn_alignbit(hd.w, hd.z, 16);
    const uint32_t g1a = __builtin_amdgcn_alignbit(hd.z, hd.y, 24), g1b = hd.w >> 8;
    const uint32_t msk = (uint32_t)-g32;  // all ones for the upper lane half
    const uint32_t G0 = (g0a & ~msk) | (g0b & msk);
    const uint32_t G1 = (g1a & ~msk) | (g1b & msk);
    const half2v k1024 = splat2((_Float16)1024.0f);
    const half2v dd = splat2(h_from_bits(hd.x & 0xFFFFu) * ws);  // ws is a power of two: exact
    const half2v dm = splat2(-h_from_bits(hd.x >> 16) * ws);
    K4Consts c;
    half2v mn[2];
#pragma unroll
    for (int s = 0; s < 2; s++) {
        const uint32_t G = s ? G1 : G0;
        const half2v sc = as_half2((G & 0x3Fu) | ((G << 4) & 0x003F0000u) | kMagic1024) - k1024;
        mn[s] = (as_half2(((G >> 6) & 0x3Fu) | ((G >> 2) & 0x003F0000u) | kMagic1024) - k1024) * dm;
        const half2v dsc = sc * dd;  // (d*sc of half 0, d*sc of half 1), rounded to f16
        c.s[2 * s] = splat2(dsc.x);
        c.s[2 * s + 1] = splat2(dsc.y);
    }
#pragma unroll
    for (int u = 0; u < 4; u++) {
        c.s16[u] = c.s[u] * splat2((_Float16)0.0625f);
        c.c1[u] = c.s[u] * splat2((_Float16)-1024.0f);
        c.c2[u] = c.s[u] * splat2((_Float16)-64.0f);
    }
    c.bmin = half8v{mn[0].x, mn[0].x, mn[0].y, mn[0].y, mn[1].x, mn[1].x, mn[1].y, mn[1].y};
    return c;
}

template <> struct GFmt<TURQ_Q4_K> {
    using F = TiledFmt<TURQ_Q4_K>;
    static constexpr int NSTG = 1;
    static constexpr bool SUMS = true;
    struct Stage { uint4v q; };
    struct Hdr { uint4v hd; };
    using Consts = K4Consts;
    struct Addr { uint32_t q, h; };
    __device__ static Addr addr(uint32_t tile, int r16, int g32) {
        return Addr{tile + 16u * (uint32_t)(r16 + 32 * g32), tile + (uint32_t)F::kHDR + 16u * (uint32_t)r16};
    }
    // OFF = byte offset of the n-tile inside the ring entry (compile time)
    template <int KS, int OFF> __device__ static void read_stage(Stage &st, const Addr &a, uint32_t ring) {
        lds_read128<OFF + (KS & 1) * 1024 + (KS >> 1) * 256>(st.q, a.q + ring);
    }
    template <int OFF> __device__ static void read_hdr(Hdr &h, const Addr &a, uint32_t ring) { lds_read128<OFF>(h.hd, a.h + ring); }
    __device__ static void pin_stage(Stage &st) { pin(st.q); }
    __device__ static void pin_hdr(Hdr &h) { pin(h.hd); }
    __device__ static Consts consts(const Hdr &h, int g32, _Float16 ws) { return k4_consts(h.hd, g32, ws); }
    __device__ static half8v bmin(const Consts &c) { return c.bmin; }
    template <int KS, int ST> __device__ static half8v operand(const Stage &st, const Consts &c) {
        const uint32_t w = word_of<ST>(st.q), w8 = w >> 8;
        return make_half8(pk_fma(and_or_asm_h2(w, 0x000F000Fu, kMagic1024), c.s[KS], c.c1[KS]), pk_fma(and_or_asm_h2(w, 0x00F000F0u, kMagic64), c.s[KS], c.c2[KS]),
                          pk_fma(and_or_asm_h2(w8, 0x000F000Fu, kMagic1024), c.s[KS], c.c1[KS]),
                          pk_fma(and_or_asm_h2(w8, 0x00F000F0u, kMagic64), c.s[KS], c.c2[KS]));
    }
};

template <> struct GFmt<TURQ_Q5_K> {
    using F = TiledFmt<TURQ_Q5_K>;
    static constexpr int NSTG = 2;
    static constexpr bool SUMS = true;
    struct Stage { uint4v q; uint2v hh; };
    struct Hdr { uint4v hd; };
    using Consts = K4Consts;
    struct Addr { uint32_t q, hh, h; };
    __device__ static Addr addr(uint32_t tile, int r16, int g32) {
        return Addr{tile + 16u * (uint32_t)(r16 + 32 * g32), tile + (uint32_t)F::kQH + 8u * (uint32_t)(r16 + 32 * g32),
                    tile + (uint32_t)F::kHDR + 16u * (uint32_t)r16};
    }
    template <int KS, int OFF> __device__ static void read_stage(Stage &st, const Addr &a, uint32_t ring) {
        lds_read128<OFF + (KS & 1) * 1024 + (KS >> 1) * 256>(st.q, a.q + ring);
        lds_read64<OFF + (KS >> 1) * 128>(st.hh, a.hh + ring);  // the two high-bit dwords of the lane slot
    }
    template <int OFF> __device__ static void read_hdr(Hdr &h, const Addr &a, uint32_t ring) { lds_read128<OFF>(h.hd, a.h + ring); }
    __device__ static void pin_stage(Stage &st) { pin(st.q); pin(st.hh); }
    __device__ static void pin_hdr(Hdr &h) { pin(h.hd); }
    __device__ static Consts consts(const Hdr &h, int g32, _Float16 ws) { return k4_consts(h.hd, g32, ws); }
    __device__ static half8v bmin(const Consts &c) { return c.bmin; }
    template <int KS, int ST> __device__ static half8v operand(const Stage &st, const Consts &c) {
        // step i of the slot; with v = 4 i + t the packed register t, u = v >> 1: its two high bits sit in H0 (even t) at
        // bits (4 + u, 20 + u) or in H1 (odd t) at bits (8 + u, 24 + u): a rotate right by u puts them on bit 4 / 20
        // (+16 on a nibble at bits 0..3) or bit 8 / 24 (+16 on a nibble at bits 4..7 read with 16 units per step)
        constexpr uint32_t u0 = 2 * (4 * (KS & 1) + ST);
        const uint32_t w = word_of<ST>(st.q), w8 = w >> 8;
        uint32_t t0 = and_or_asm(w, 0x000F000Fu, kMagic1024);
        uint32_t t1 = and_or_asm(w, 0x00F000F0u, kMagic1024);
        uint32_t t2 = and_or_asm(w8, 0x000F000Fu, kMagic1024);
        uint32_t t3 = and_or_asm(w8, 0x00F000F0u, kMagic1024);
        t0 = and_or_asm(rotr32(st.hh.x, u0), 0x00100010u, t0);
        t1 = and_or_asm(rotr32(st.hh.y, u0), 0x01000100u, t1);
        t2 = and_or_asm(rotr32(st.hh.x, u0 + 1), 0x00100010u, t2);
        t3 = and_or_asm(rotr32(st.hh.y, u0 + 1), 0x01000100u, t3);
        return make_half8(pk_fma(as_half2(t0), c.s[KS], c.c1[KS]), pk_fma(as_half2(t1), c.s16[KS], c.c2[KS]),
                          pk_fma(as_half2(t2), c.s[KS], c.c1[KS]), pk_fma(as_half2(t3), c.s16[KS], c.c2[KS]));
    }
};

template <> struct GFmt<TURQ_Q6_K> {
    using F = TiledFmt<TURQ_Q6_K>;
    static constexpr int NSTG = 2;
    static constexpr bool SUMS = false;
    struct Stage { uint4v ql, qh; };
    struct Hdr { uint32_t sc0, sc1, d16; };  // the four int8 scales of lane slots 2 g32 and 2 g32 + 1; the row's d
    struct Consts { half2v s[8]; };          // per 16-column group of the lane's 128 columns: d*sc, rounded to f16
    struct Addr { uint32_t q, qh, sc, d; };
    __device__ static Addr addr(uint32_t tile, int r16, int g32) {
        const uint32_t slot = (uint32_t)(r16 + 32 * g32);
        return Addr{tile + 16u * slot, tile + (uint32_t)F::kQH + 16u * slot, tile + (uint32_t)F::kSC + 4u * slot,
                    tile + (uint32_t)F::kD + 2u * (uint32_t)r16};
    }
    template <int KS, int OFF> __device__ static void read_stage(Stage &st, const Addr &a, uint32_t ring) {
        lds_read128<OFF + (KS & 1) * 1024 + (KS >> 1) * 256>(st.ql, a.q + ring);
        lds_read128<OFF + (KS >> 1) * 256>(st.qh, a.qh + ring);  // all 64 high fields of the lane slot
    }
    template <int OFF> __device__ static void read_hdr(Hdr &h, const Addr &a, uint32_t ring) {
        lds_read32<OFF>(h.sc0, a.sc + ring);
        lds_read32<OFF + 64>(h.sc1, a.sc + ring);
        lds_read16<OFF>(h.d16, a.d + ring);
    }
    __device__ static void pin_stage(Stage &st) { pin(st.ql); pin(st.qh); }
    __device__ static void pin_hdr(Hdr &h) { pin(h.sc0); pin(h.sc1); pin(h.d16); }
    __device__ static Consts consts(const Hdr &h, int, _Float16 ws) {
        const float d = (float)h_from_bits(h.d16) * (float)ws;
        Consts c;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const int sc = (int)(int8_t)((i < 4 ? h.sc0 : h.sc1) >> (8 * (i & 3)));
            const _Float16 s = (_Float16)(d * (float)sc);
            c.s[i] = splat2(s);
        }
        return c;
    }
    __device__ static half8v bmin(const Consts &c) { return half8v{}; }
    template <int KS, int ST> __device__ static half8v operand(const Stage &st, const Consts &c) {
        // step i = 4 (KS & 1) + ST of the slot: low nibbles of register t at bits 2 + 4 t (and + 16), high fields at bits
        // 6 + 8 (i & 1) + 2 t (and + 16) of high dword i >> 1; scale group i >> 1 of the slot
        constexpr int i = 4 * (KS & 1) + ST;
        constexpr int grp = 4 * (KS >> 1) + (i >> 1);
        const uint32_t wl = word_of<ST>(st.ql);
        const uint32_t wh = word_of<(i >> 1)>(st.qh);
        half2v r[4];
#pragma unroll
        for (int t = 0; t < 4; t++) {
            const uint32_t lo = and_or_asm(t == 0 ? wl : rotr32(wl, 4 * t), 0x003C003Cu, kMagic256);
            const uint32_t hi_src = (8 * (i & 1) + 2 * t) == 0 ? wh : rotr32(wh, (uint32_t)(8 * (i & 1) + 2 * t));
            // (256 + q) - 288 = q - 32 exactly, then one rounding in the product; a fused form would need the constant
            // -288 * d * sc, which f16 cannot hold exactly (288 is not a power of two)
            r[t] = (as_half2(and_or_asm(hi_src, 0x00C000C0u, lo)) - splat2((_Float16)288.0f)) * c.s[grp];
        }
        return make_half8(r[0], r[1], r[2], r[3]);
    }
};

// Q8_0: the tile holds 8 blocks of 32 columns in four planes (plane i = blocks 2 i, 2 i + 1); stage ks is plane ks.  The lane
// reads its two lane slots (2 g32, 2 g32 + 1: 8 bytes per block each) and takes, per block, first the 8 columns of the one,
// then of the other: operand step st of the stage is block 2 ks + st / 2, slot st % 2 (the Q8_0 order of act_prep32_kernel).
// Bytes are q + 128 (tiled layout), read as 1024 + 128 + q in the mantissa of 1024.0; (t - 1152) is q exactly and q * d is
// rounded once.  The tiles are 4352 bytes: wave tile 2 x 1 (workgroup 128 x 64) keeps three super-blocks in the LDS.
template <> struct GFmt<TURQ_Q8_0> {
    using F = TiledFmt<TURQ_Q8_0>;
    static constexpr int NSTG = 2;
    static constexpr bool SUMS = false;
    struct Stage { uint4v a, b; };     // lane slots 2 g32 and 2 g32 + 1 of the plane: (block 2 ks: lo, hi), (block 2 ks + 1: lo, hi)
    struct Hdr { uint4v dd; };         // the row's 8 f16 block scales
    struct Consts { half2v s[8]; };
    struct Addr { uint32_t q, h; };
    __device__ static Addr addr(uint32_t tile, int r16, int g32) {
        return Addr{tile + 16u * (uint32_t)(r16 + 32 * g32), tile + (uint32_t)F::kD + 16u * (uint32_t)r16};
    }
    template <int KS, int OFF> __device__ static void read_stage(Stage &st, const Addr &a, uint32_t ring) {
        lds_read128<OFF + KS * 1024>(st.a, a.q + ring);
        lds_read128<OFF + KS * 1024 + 256>(st.b, a.q + ring);
    }
    template <int OFF> __device__ static void read_hdr(Hdr &h, const Addr &a, uint32_t ring) { lds_read128<OFF>(h.dd, a.h + ring); }
    __device__ static void pin_stage(Stage &st) { pin(st.a); pin(st.b); }
    __device__ static void pin_hdr(Hdr &h) { pin(h.dd); }
    __device__ static Consts consts(const Hdr &h, int, _Float16 ws) {
        const uint32_t dw[4] = {h.dd.x, h.dd.y, h.dd.z, h.dd.w};
        Consts c;
#pragma unroll
        for (int i = 0; i < 8; i++) c.s[i] = splat2(h_from_bits((i & 1) ? dw[i >> 1] >> 16 : dw[i >> 1] & 0xFFFFu) * ws);
        return c;
    }
    __device__ static half8v bmin(const Consts &) { return half8v{}; }
    template <int KS, int ST> __device__ static half8v operand(const Stage &st, const Consts &c) {
        constexpr int blk = 2 * KS + (ST >> 1);
        const uint4v src = (ST & 1) ? st.b : st.a;
        const uint32_t w0 = (ST >> 1) ? src.z : src.x, w1 = (ST >> 1) ? src.w : src.y;
        const half2v k1152 = splat2((_Float16)1152.0f);
        return make_half8((and_or_asm_h2(w0, 0x00FF00FFu, kMagic1024) - k1152) * c.s[blk],
                          (and_or_asm_h2(w0 >> 8, 0x00FF00FFu, kMagic1024) - k1152) * c.s[blk],
                          (and_or_asm_h2(w1, 0x00FF00FFu, kMagic1024) - k1152) * c.s[blk],
                          (and_or_asm_h2(w1 >> 8, 0x00FF00FFu, kMagic1024) - k1152) * c.s[blk]);
    }
};

}  // namespace
