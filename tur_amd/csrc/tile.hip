// GGUF block bytes -> the tiled layout (layout.h), on the device: what turq_tile_host does, for uploads.  The host's transform was
// three passes of host memory over every tensor (clear, transform, copy) and a fourth for the largest scale; here the bytes of the file go
// over the bus once and one pass of device memory does the rest.  Bound by that copy (a 28 MB tensor: 20 us here, over 1 ms for the bus).
// One wave per tile, lane L = r + 16 g makes what the layout keeps at lane L: it reads the row's 64 elements of group g (Q8_0: its 8 elements
// of every block) and stores 16 bytes per plane, a contiguous KiB per store of the wave.  Rows past n and blocks past k are zeros.
#include "layout.h"
#include "mfma_common.h"

namespace {

// COUNT bytes from an address of which only ALIGN is known
template <int COUNT, int ALIGN> __device__ inline void ld_bytes(const uint8_t *p, uint8_t (&v)[COUNT]) {
    static_assert(ALIGN == 16 || ALIGN == 2, "16-byte blocks or halves");
    if constexpr (ALIGN == 16) {
#pragma unroll
        for (int i = 0; i < COUNT / 16; i++) {
            const uint4v u = ((const uint4v *)p)[i];
            const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
            for (int b = 0; b < 16; b++) v[16 * i + b] = (uint8_t)(w[b >> 2] >> (8 * (b & 3)));
        }
    } else {
#pragma unroll
        for (int i = 0; i < COUNT / 2; i++) {
            const uint32_t u = ((const uint16_t *)p)[i];
            v[2 * i] = (uint8_t)u;
            v[2 * i + 1] = (uint8_t)(u >> 8);
        }
    }
}
__device__ inline uint32_t ld_u16(const uint8_t *p) { return *(const uint16_t *)p; }
// |value| of f16 bits, as bits of an f32 (they order like the values, NaNs above everything)
__device__ inline uint32_t abs_bits(uint32_t h) {
    _Float16 v;
    const uint16_t u = (uint16_t)(h & 0x7FFFu);
    __builtin_memcpy(&v, &u, 2);
    return __float_as_uint((float)v);
}
// the largest scale of a block: |d|, for Q4_K / Q5_K also |dmin| / 1024 (see turq_weight::max_scale)
template <int DT> __device__ inline uint32_t block_scale(const uint8_t *nat) {
    uint32_t s = abs_bits(ld_u16(nat + (DT == TURQ_Q6_K ? 208 : 0)));
    if (DT == TURQ_Q4_K || DT == TURQ_Q5_K) {
        const uint32_t dm = __float_as_uint(__uint_as_float(abs_bits(ld_u16(nat + 2))) * (1.0f / 1024.0f));
        s = s > dm ? s : dm;
    }
    return s;
}
__device__ inline void note_scale(uint32_t s, uint32_t *__restrict__ top) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        const uint32_t o = (uint32_t)__shfl_xor((int)s, off, 64);
        s = s > o ? s : o;
    }
    if ((threadIdx.x & 63) == 0 && s > __hip_atomic_load(top, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
        __hip_atomic_fetch_max(top, s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// rows [row0, row0 + rows) of the tensor (row0 a multiple of 16) lie at `nat`, their tiles start at `tiled`; every wave of the launch
// has a tile
template <int DT>
__global__ void __launch_bounds__(256) tile_kernel(const uint8_t *__restrict__ nat, int64_t rows, int64_t k, int64_t tiles, uint8_t *__restrict__ tiled,
                                                   uint32_t *__restrict__ top) {
    using F = TiledFmt<DT>;
    constexpr int BB = F::kBlockBytes;
    const int64_t ti = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (ti >= tiles) return;
    const int L = threadIdx.x & 63, r = L & 15, g = L >> 4;
    const int64_t ntc = turq_tile_cols(k), bpr = k / F::kBlockElems;
    const int64_t row = ti / ntc * 16 + r, tb = ti % ntc;
    const bool live = row < rows;
    uint8_t *tile = tiled + ti * F::kTileBytes;
    uint32_t scale = 0;
    if constexpr (DT == TURQ_Q8_0) {
        uint32_t dd[4] = {0, 0, 0, 0};
#pragma unroll
        for (int i = 0; i < 4; i++) {
            uint32_t w[4] = {0, 0, 0, 0};
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const int q = 2 * i + h;
                const int64_t b = 8 * tb + q;
                if (!live || b >= bpr) continue;
                const uint8_t *blk = nat + (row * bpr + b) * BB;
                uint8_t v[8];
                ld_bytes<8, 2>(blk + 2 + 8 * g, v);
#pragma unroll
                for (int j = 0; j < 8; j++) {
                    const int c = ((j & 1) << 1) | ((j >> 1) & 1);  // byte order {0, 2, 1, 3}
                    w[2 * h + (j >> 2)] |= (uint32_t)(v[j] ^ 0x80) << (8 * c);
                }
                if (g == 0) {
                    dd[q >> 1] |= ld_u16(blk) << (16 * (q & 1));
                    const uint32_t s = block_scale<DT>(blk);
                    scale = s > scale ? s : scale;
                }
            }
            ((uint4v *)(tile + 1024 * i))[L] = uint4v{w[0], w[1], w[2], w[3]};
        }
        if (g == 0) ((uint4v *)(tile + F::kD))[r] = uint4v{dd[0], dd[1], dd[2], dd[3]};
    } else {
        const uint8_t *blk = nat + (row * bpr + tb) * BB;
        if (live && g == 0) scale = block_scale<DT>(blk);
        uint32_t w[8] = {0, 0, 0, 0, 0, 0, 0, 0};
        if constexpr (DT == TURQ_Q6_K) {
            // elements 64 g + e: low nibbles in bytes 64 (g / 2) + e of ql (the upper ones for odd g), two high bits in byte
            // 32 (g / 2) + e % 32 of qh at bit 4 (g % 2) + 2 (e / 32)
            uint32_t H[4] = {0, 0, 0, 0}, sc = 0;
            if (live) {
                uint8_t ql[64], qh[32];
                ld_bytes<64, 2>(blk + 64 * (g >> 1), ql);
                ld_bytes<32, 2>(blk + 128 + 32 * (g >> 1), qh);
#pragma unroll
                for (int i = 0; i < 8; i++)
#pragma unroll
                    for (int j = 0; j < 8; j++) {
                        const int e = 8 * i + j;
                        w[i] |= turq_rotl32((ql[e] >> (4 * (g & 1))) & 15u, turq_q6_nibble_bit(j));
                        H[i >> 1] |= turq_rotl32((qh[e & 31] >> (4 * (g & 1) + 2 * (e >> 5))) & 3u, turq_q6_high_bit(i, j));
                    }
                sc = ld_u16(blk + 192 + 4 * g) | (ld_u16(blk + 194 + 4 * g) << 16);
            }
            ((uint4v *)(tile + F::kQH))[L] = uint4v{H[0], H[1], H[2], H[3]};
            ((uint32_t *)(tile + F::kSC))[L] = sc;
            if (g == 0) ((uint16_t *)(tile + F::kD))[r] = live ? (uint16_t)ld_u16(blk + 208) : (uint16_t)0;
        } else {
            // elements 64 g + e: byte 32 g + e % 32 of qs, the upper nibbles from e = 32 on; Q5_K: the fifth bit in byte e % 32 of qh at
            // bit 2 g + e / 32
            constexpr int QS = DT == TURQ_Q5_K ? 48 : 16;
            if (live) {
                uint8_t qs[32];
                ld_bytes<32, 16>(blk + QS + 32 * g, qs);
#pragma unroll
                for (int i = 0; i < 8; i++)
#pragma unroll
                    for (int j = 0; j < 8; j++) {
                        const int e = 8 * i + j;
                        w[i] |= (uint32_t)((qs[e & 31] >> (4 * (e >> 5))) & 15) << turq_q4_nibble_bit(j);
                    }
            }
            if constexpr (DT == TURQ_Q5_K) {
                uint32_t H[2] = {0, 0};
                if (live) {
                    uint8_t qh[32];
                    ld_bytes<32, 16>(blk + 16, qh);
#pragma unroll
                    for (int i = 0; i < 8; i++)
#pragma unroll
                        for (int j = 0; j < 8; j++) {
                            const int e = 8 * i + j;
                            H[(j >> 1) & 1] |= (uint32_t)((qh[e & 31] >> (2 * g + (e >> 5))) & 1) << turq_q5_high_bit(i, j);
                        }
                }
                ((uint2v *)(tile + F::kQH))[L] = uint2v{H[0], H[1]};
            }
            if (g == 0) {
                if (live) TileBlock<TURQ_Q4_K>::pack_hdr(blk, tile + F::kHDR + 16 * r);
                else ((uint4v *)(tile + F::kHDR))[r] = uint4v{0, 0, 0, 0};
            }
        }
        ((uint4v *)tile)[L] = uint4v{w[0], w[1], w[2], w[3]};
        ((uint4v *)(tile + 1024))[L] = uint4v{w[4], w[5], w[6], w[7]};
    }
    note_scale(scale, top);
}

template <int DT>
__global__ void __launch_bounds__(256) scale_kernel(const uint8_t *__restrict__ nat, int64_t blocks, uint32_t *__restrict__ top) {
    uint32_t s = 0;
    for (int64_t b = (int64_t)blockIdx.x * 256 + threadIdx.x; b < blocks; b += (int64_t)gridDim.x * 256) {
        const uint32_t t = block_scale<DT>(nat + b * TiledFmt<DT>::kBlockBytes);
        s = s > t ? s : t;
    }
    note_scale(s, top);
}

}  // namespace

// nat: the GGUF bytes of `rows` whole rows (device memory, 16-byte aligned, 64 bytes allocated past their end), from a row that is a multiple
// of 16; tiled: where their tiles go; top: bits of the largest block scale, raised by the launch
hipError_t turq_launch_tile(int dt, const void *nat, int64_t rows, int64_t k, void *tiled, uint32_t *top, hipStream_t stream) {
    if (!turq_dt_is_quant(dt) || rows < 0 || k < 0 || k % turq_dt_block_elems(dt) != 0) return hipErrorInvalidValue;
    const int64_t tiles = turq_tile_rows(rows) * turq_tile_cols(k);
    if (tiles == 0) return hipSuccess;
    if (tiles > (int64_t)4 * 0x7FFFFFFF) return hipErrorInvalidValue;
    const unsigned grid = (unsigned)((tiles + 3) / 4);
    switch (dt) {
    case TURQ_Q4_K: tile_kernel<TURQ_Q4_K><<<grid, 256, 0, stream>>>((const uint8_t *)nat, rows, k, tiles, (uint8_t *)tiled, top); break;
    case TURQ_Q5_K: tile_kernel<TURQ_Q5_K><<<grid, 256, 0, stream>>>((const uint8_t *)nat, rows, k, tiles, (uint8_t *)tiled, top); break;
    case TURQ_Q6_K: tile_kernel<TURQ_Q6_K><<<grid, 256, 0, stream>>>((const uint8_t *)nat, rows, k, tiles, (uint8_t *)tiled, top); break;
    default: tile_kernel<TURQ_Q8_0><<<grid, 256, 0, stream>>>((const uint8_t *)nat, rows, k, tiles, (uint8_t *)tiled, top); break;
    }
    return hipGetLastError();
}

// ... of a tensor that stays in GGUF order
hipError_t turq_launch_block_scale(int dt, const void *nat, int64_t blocks, uint32_t *top, hipStream_t stream) {
    if (!turq_dt_is_quant(dt)) return hipErrorInvalidValue;
    if (blocks == 0) return hipSuccess;
    const unsigned grid = (unsigned)((blocks + 255) / 256 < 2048 ? (blocks + 255) / 256 : 2048);
    switch (dt) {
    case TURQ_Q4_K: scale_kernel<TURQ_Q4_K><<<grid, 256, 0, stream>>>((const uint8_t *)nat, blocks, top); break;
    case TURQ_Q5_K: scale_kernel<TURQ_Q5_K><<<grid, 256, 0, stream>>>((const uint8_t *)nat, blocks, top); break;
    case TURQ_Q6_K: scale_kernel<TURQ_Q6_K><<<grid, 256, 0, stream>>>((const uint8_t *)nat, blocks, top); break;
    default: scale_kernel<TURQ_Q8_0><<<grid, 256, 0, stream>>>((const uint8_t *)nat, blocks, top); break;
    }
    return hipGetLastError();
}
