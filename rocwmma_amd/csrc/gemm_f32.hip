// f32 GEMM on the bf16 matrix instructions, 64 x 64 macro tiles.
//
// v_mfma_f32_16x16x4_f32 runs at a sixteenth of the rate of v_mfma_f32_16x16x32_bf16.  An f32 has 24 significant bits, a bf16
// eight: 2^16 x = h + m + l with three bf16, each the rounded value of what the ones before it leave, holds every f32 below 2^112 exactly (the smallest,
// 2^-149, becomes 2^-133, the last bit of a bf16).  Of the nine products of two such sums the six down to 2^-17 of the whole are multiplied,
//     h h'   and   h m' + m h' + m m' + h l' + l h',
// which leaves out up to 2^-24 of a product (|m| is up to 2^-8 of x, |l| 2^-17: m l' + l m'), and summed in f32 accumulators, the first one in one of its
// own, so that the long chain of roundings is that of one product in 32 instead of one in one.  Against 64 bits such a sum is closer than with the f32
// instructions (norm of the difference, uniform operands, every orientation alike): K = 512 4.0e-7 -> 0.71e-7, 2560 9.1e-7 -> 1.36e-7, 3584 10.7e-7 -> 1.6e-7;
// positive operands, K = 2560, 7.8e-7 -> 0.85e-7; two products other than zero 3.1e-8 -> 2.6e-8, four 4.0e-8 -> 2.7e-8.  One product, correctly rounded by the
// f32 instructions, 2.53e-8 -> 2.60e-8: within 0.96 ulp instead of 0.5, 4 % of them the neighbouring f32.
//
//   workgroup    four waves, two workgroups a CU.  Each wave multiplies the whole tile over its own slices of K (32 wide, every fourth one),
//                so that an operand element is taken apart once in a workgroup and no wave waits for another before the end
//   global->LDS  direct loads into the wave's own 16 KiB, one slice ahead: A's half is filled again as soon as A's pieces are in registers,
//                B's under the last block's matrix instructions
//   registers    2 x 64 of accumulators, 48 of A's pieces, 12 of a block of B's
//   end          the four partial tiles meet in LDS and are added in the order of the waves: first the sums of h h' alone, then those of the rest, so that no wave
//                rounds one to the other (sums of two products: 3.5e-8 with one rounding a wave).  It costs 0.5 us per round, 2560^3 210 -> 213 us,
//                2048 x 2048 x 640 37.0 -> 39.0 (40.4 with f32 instructions); each wave adding up a quarter in its registers takes as long.
//   not a number An infinite or missing value anywhere in a tile makes the sum of the products that is not finite (l of an infinity is NaN), and so
//                does an operand from 2^112 (5e33) or a sum from 2^96 (8e28) on.  Such a tile is multiplied again with the f32 instructions, each wave
//                its own slices of K (the kernel of fewer tiles sums K in one chain: other roundings, the same infinities and NaN but where a sum
//                overflows in between).  It costs both: 2560^3 213 us, 390 with one infinity in A, 480 with one in every row, 250 with f32 instructions alone.
//
// What bounds it: the board's power, then the vector instructions that take the operands apart (416 per 96 matrix instructions, which
// hide two each).  2560^3: 254 us with f32 instructions -> 213 (191 with all-zero operands, 213 with a softmax of wide logits, a quarter of whose values are below
// 2^-110; without the factor 2^16, whose multiplications are two of every thirteen vector instructions, 209, but 475 where tiles with such values were multiplied again).
// Tried: the same with v_mfma_f32_32x32x16_bf16, 1.1 times as long; the pieces by v_dot2c_f32_bf16 subtractions, 1.01 (a dot product takes the matrix
// pipe); the forming dealt out between the matrix instructions, 1.03; all eight products but l l' 1.11 to 1.18, no faster than the f32 instructions on
// most shapes; the waves of a SIMD at different priorities, 0.96 to 1.01.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "common.hpp"
#include "gemm_params.hpp"
#include "lds_dma.hpp"
#include "tile_map.hpp"

namespace
{
    using i32x4  = int __attribute__((ext_vector_type(4)));
    using f32x4  = float __attribute__((ext_vector_type(4)));
    using bf16x2 = __bf16 __attribute__((ext_vector_type(2)));
    using bf16x8 = __bf16 __attribute__((ext_vector_type(8)));
    using Params = r355::GemmTileParams;
    using r355::loadToLds;

    constexpr float    SCALE = 65536.0f; // no f32 has bits that are below the last one of bf16 after it
    constexpr uint32_t TILE = 64, WAVES = 4, THREADS = 256;
    constexpr uint32_t SLICE = 32, SLICE_BYTES = 128; // K of a slice: elements, bytes
    constexpr uint32_t CHUNK = 16, OPER = TILE * SLICE_BYTES; // 8 KiB of an operand per slice
    constexpr uint32_t BLOCKS = TILE / 16, LOADS = OPER / CHUNK / 64; // 4 blocks of 16 rows, 8 direct loads per operand and slice

    // (assembly with a memory clobber: the reads of what the direct loads bring must not move above the wait)
    template <uint32_t N>
    __device__ __forceinline__ void waitLoads()
    {
        asm volatile("s_waitcnt vmcnt(%0)" : : "n"(N) : "memory");
    }
    __device__ __forceinline__ void waitReads()
    {
        asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");
    }

    // Eight f32 times SCALE as three bf16 each
    struct Pieces
    {
        i32x4 h, m, l;
    };
    __device__ __forceinline__ uint32_t pack(float x0, float x1)
    {
        uint32_t w = __builtin_bit_cast(uint32_t, bf16x2{static_cast<__bf16>(x0), static_cast<__bf16>(x1)});
        asm volatile("" : "+v"(w)); // (a word like any other: its halves are taken apart by a shift and a mask, not rounded once more)
        return w;
    }
    __device__ __forceinline__ Pieces split(const float (&in)[8])
    {
        Pieces p;
#pragma unroll
        for(uint32_t e = 0; e < 4; ++e)
        {
            float          x0 = in[2u * e] * SCALE, x1 = in[2u * e + 1u] * SCALE;
            const uint32_t h = pack(x0, x1);
            x0 -= __builtin_bit_cast(float, h << 16), x1 -= __builtin_bit_cast(float, h & 0xFFFF0000u);
            const uint32_t m = pack(x0, x1);
            x0 -= __builtin_bit_cast(float, m << 16), x1 -= __builtin_bit_cast(float, m & 0xFFFF0000u);
            p.h[e] = static_cast<int>(h), p.m[e] = static_cast<int>(m), p.l[e] = static_cast<int>(pack(x0, x1));
        }
        return p;
    }
    __device__ __forceinline__ void multiply(f32x4& acc, i32x4 x, i32x4 y)
    {
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, x), __builtin_bit_cast(bf16x8, y), acc, 0, 0, 0);
    }

    __device__ __forceinline__ uint32_t swzK(uint32_t row)
    {
        return (row >> 1) & 7u;
    }
    __device__ __forceinline__ uint32_t swzMN(uint32_t krow)
    {
        return ((krow >> 2) & 3u) << 2;
    }

    // One operand of a wave: its direct loads and its reads
    template <bool KCONTIG>
    struct Operand
    {
        uint64_t panel; // first row (column) of the tile, K 0
        uint32_t ld, rows, off[KCONTIG ? 2 : 4], kByte, rd; // rows: K-contiguous, of the tile inside the matrix

        __device__ __forceinline__ void init(const char* base, uint32_t first, uint32_t ldElems, uint32_t valid, uint32_t lane)
        {
            ld = ldElems, rows = valid;
            panel = r355::uniformAddress(base + (KCONTIG ? (uint64_t)first * ld : (uint64_t)first) * 4u);
            const uint32_t t = lane & 15u, g = lane >> 4;
            if constexpr(KCONTIG)
            {
                const uint32_t r = lane >> 3; // load j: row 8 j + r, whose swizzle alternates with j
                kByte  = ((lane & 7u) ^ swzK(r)) * CHUNK;
                off[0] = r * ld * 4u + kByte;
                off[1] = r * ld * 4u + (kByte ^ 64u);
                rd     = t * SLICE_BYTES + (g ^ swzK(t)) * CHUNK;
            }
            else
            {
                const uint32_t r = lane >> 4; // load j: k-row 4 j + r, whose swizzle is that of j
#pragma unroll
                for(uint32_t j = 0; j < 4; ++j) // (columns past the last one: the first chunk instead)
                {
                    const uint32_t c = (lane & 15u) ^ (j << 2);
                    off[j]           = r * ld * 4u + (c * 4u < valid ? c : 0u) * CHUNK;
                }
                // element e of block i: k-row 4 g + e (+ 16 for e >= 4), column t of the block
                rd = 4u * g * (TILE * 4u) + g * 64u + (t >> 2) * CHUNK + (t & 3u) * 4u;
            }
        }
        // the direct loads of a slice with `valid` bytes of K, into LDS at `dst`
        __device__ __forceinline__ void issue(uint32_t slice, uint32_t valid, uint32_t dst) const
        {
            const uint64_t at = panel + (uint64_t)slice * (KCONTIG ? (uint64_t)SLICE_BYTES : (uint64_t)SLICE_BYTES * ld);
            // rows past the last one (K-contiguous) and k-rows past it lie outside the buffer: zeros
            const uint32_t records = KCONTIG ? (rows - 1u) * ld * 4u + valid : valid * ld;
            const i32x4    rsrc{static_cast<int>(static_cast<uint32_t>(at)), static_cast<int>(static_cast<uint32_t>(at >> 32) & 0xFFFFu),
                             static_cast<int>(records), 0x00020000};
            if constexpr(KCONTIG)
            {
                uint32_t even = off[0], odd = off[1];
                if(valid != SLICE_BYTES) // (uniform)
                    even = kByte >= valid ? 0x80000000u : even, odd = (kByte ^ 64u) >= valid ? 0x80000000u : odd;
#pragma unroll
                for(uint32_t j = 0; j < LOADS; ++j)
                    loadToLds(rsrc, j & 1u ? odd : even, j * 32u * ld, dst + j * 1024u);
            }
            else
            {
#pragma unroll
                for(uint32_t j = 0; j < LOADS; ++j)
                    loadToLds(rsrc, off[j & 3u], j * 16u * ld, dst + j * 1024u);
            }
        }
        __device__ __forceinline__ void read(const char* lds, uint32_t i, float (&x)[8]) const
        {
            if constexpr(KCONTIG)
            {
                const f32x4 v0 = *reinterpret_cast<const f32x4*>(lds + rd + i * 16u * SLICE_BYTES);
                const f32x4 v1 = *reinterpret_cast<const f32x4*>(lds + (rd ^ 64u) + i * 16u * SLICE_BYTES);
#pragma unroll
                for(uint32_t e = 0; e < 4; ++e)
                    x[e] = v0[e], x[4u + e] = v1[e];
            }
            else
            {
                // (the swizzle of k-rows 4 g .. 4 g + 3, and of those 16 further, is g: chunk 4 i + t / 4 lies in slot 4 (i ^ g) + t / 4)
                const char* q = lds + (rd ^ (i * 64u));
#pragma unroll
                for(uint32_t e = 0; e < 8; ++e)
                    x[e] = *reinterpret_cast<const float*>(q + (e < 4u ? e : 12u + e) * (TILE * 4u));
            }
        }
    };

    // (the order of K inside a slice is the operands' own business as long as both have the same one: lane group g holds K 4 g .. 4 g + 3 and
    // those 16 further, two 16-byte chunks of a K-contiguous row)
    template <bool A_KCONTIG, bool B_KCONTIG>
    __global__ void __launch_bounds__(THREADS) __attribute__((amdgpu_waves_per_eu(2, 2))) gemmF32Kernel(Params p)
    {
        __shared__ __attribute__((aligned(1024))) char lds[WAVES * 2u * OPER];
        static_assert(sizeof(lds) == r355::F32_TILES_LDS, "what a launch plan reports");
        uint32_t tm, tn;
        if(!r355::tileCoordRange(blockIdx.x, p.tilesM, p.tilesN, p.tileFirst, p.tileCount, false, tm, tn))
            return;
        const uint32_t tid = threadIdx.x, lane = tid & 63u, t = lane & 15u, g = lane >> 4;
        const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        const uint32_t m0 = tm * TILE, n0 = tn * TILE;
        // this workgroup row's slices of K
        const uint32_t total = (p.k - 1u) / SLICE + 1u, firstSlice = blockIdx.y * p.splitStages;
        const uint32_t left = total - firstSlice, count = p.splitStages != 0u && p.splitStages < left ? p.splitStages : left;
        const uint32_t end = firstSlice + count, lastBytes = (p.k - (total - 1u) * SLICE) * 4u;
        char* const    d   = p.d + blockIdx.y * p.splitStrideD;

        Operand<A_KCONTIG> a;
        Operand<B_KCONTIG> b;
        a.init(p.a, m0, p.lda, p.m - m0 < TILE ? p.m - m0 : TILE, lane);
        b.init(p.b, n0, p.ldb, p.n - n0 < TILE ? p.n - n0 : TILE, lane);
        char* const    mine = lds + wave * 2u * OPER;
        const uint32_t dstA = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) char*)lds)) + wave * 2u * OPER;
        const uint32_t dstB = dstA + OPER;
        auto validOf = [&](uint32_t s) { return s + 1u < total ? SLICE_BYTES : lastBytes; };

        f32x4 hi[BLOCKS][BLOCKS], lo[BLOCKS][BLOCKS];
        bool  exact = false;
        for(;;)
        {
#pragma unroll
            for(uint32_t i = 0; i < BLOCKS; ++i)
#pragma unroll
                for(uint32_t j = 0; j < BLOCKS; ++j)
                    hi[i][j] = lo[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            uint32_t s = firstSlice + wave;
            if(s < end)
            {
                a.issue(s, validOf(s), dstA);
                b.issue(s, validOf(s), dstB);
            }
            if(!exact)
            {
                for(; s < end; s += WAVES)
                {
                    const bool more = s + WAVES < end;
                    waitLoads<LOADS>(); // A of this slice
                    Pieces pa[BLOCKS];
#pragma unroll
                    for(uint32_t i = 0; i < BLOCKS; ++i)
                    {
                        float x[8];
                        a.read(mine, i, x);
                        pa[i] = split(x);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                    waitReads(); // the reads of A are done, its place may be filled again
                    if(more)
                    {
                        a.issue(s + WAVES, validOf(s + WAVES), dstA);
                        waitLoads<LOADS>(); // B of this slice
                    }
                    else
                        waitLoads<0>();
#pragma unroll
                    for(uint32_t j = 0; j < BLOCKS; ++j)
                    {
                        float x[8];
                        b.read(mine + OPER, j, x);
                        const Pieces pb = split(x);
                        if(j + 1u == BLOCKS)
                        {
                            waitReads();
                            if(more)
                                b.issue(s + WAVES, validOf(s + WAVES), dstB);
                        }
#pragma unroll
                        for(uint32_t i = 0; i < BLOCKS; ++i)
                        {
                            multiply(hi[i][j], pb.h, pa[i].h);
                            multiply(lo[i][j], pb.h, pa[i].m);
                        }
#pragma unroll
                        for(uint32_t i = 0; i < BLOCKS; ++i)
                            multiply(lo[i][j], pb.m, pa[i].h);
#pragma unroll
                        for(uint32_t i = 0; i < BLOCKS; ++i)
                            multiply(lo[i][j], pb.m, pa[i].m);
#pragma unroll
                        for(uint32_t i = 0; i < BLOCKS; ++i)
                            multiply(lo[i][j], pb.h, pa[i].l);
#pragma unroll
                        for(uint32_t i = 0; i < BLOCKS; ++i)
                            multiply(lo[i][j], pb.l, pa[i].h);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
            }
            else
            {
                for(; s < end; s += WAVES)
                {
                    waitLoads<0>();
                    float xa[BLOCKS][8];
#pragma unroll
                    for(uint32_t i = 0; i < BLOCKS; ++i)
                        a.read(mine, i, xa[i]);
#pragma unroll
                    for(uint32_t j = 0; j < BLOCKS; ++j)
                    {
                        float xb[8];
                        b.read(mine + OPER, j, xb);
#pragma unroll
                        for(uint32_t e = 0; e < 8; ++e)
#pragma unroll
                            for(uint32_t i = 0; i < BLOCKS; ++i)
                                hi[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(xb[e], xa[i][e], hi[i][j], 0, 0, 0);
                    }
                    waitReads();
                    if(s + WAVES < end)
                    {
                        a.issue(s + WAVES, validOf(s + WAVES), dstA);
                        b.issue(s + WAVES, validOf(s + WAVES), dstB);
                    }
                }
            }
            // the waves' partial tiles, 16 KiB each in the place of the wave's operands, chunk c of row r in slot c ^ r; the leading products first,
            // so that no wave rounds them to the rest of its own
            f32x4 sum[4];
            bool  finite = true;
#pragma unroll
            for(uint32_t part = 0; part < 2; ++part)
            {
                if(part != 0u)
                    __syncthreads();
#pragma unroll
                for(uint32_t i = 0; i < BLOCKS; ++i)
#pragma unroll
                    for(uint32_t j = 0; j < BLOCKS; ++j)
                    {
                        const uint32_t row = 16u * i + t, c = 4u * j + g;
                        *reinterpret_cast<f32x4*>(mine + row * (TILE * 4u) + ((c ^ (row & 15u)) * CHUNK)) = part == 0u ? hi[i][j] : lo[i][j];
                    }
                __syncthreads();
#pragma unroll
                for(uint32_t it = 0; it < 4; ++it)
                {
                    const uint32_t row = 16u * it + (tid >> 4), c = tid & 15u;
                    const char*    q = lds + row * (TILE * 4u) + ((c ^ (row & 15u)) * CHUNK);
                    f32x4          v[WAVES];
#pragma unroll
                    for(uint32_t w = 0; w < WAVES; ++w)
                        v[w] = *reinterpret_cast<const f32x4*>(q + w * 2u * OPER);
                    const f32x4 whole = (v[0] + v[1]) + (v[2] + v[3]);
                    sum[it]           = part == 0u ? whole : sum[it] + whole;
                }
            }
#pragma unroll
            for(uint32_t it = 0; it < 4; ++it)
#pragma unroll
                for(uint32_t e = 0; e < 4; ++e)
                    finite = finite && __builtin_isfinite(sum[it][e]);
            if(!exact && __syncthreads_or(!finite))
            {
                exact = true;
                continue;
            }
            const float alpha = static_cast<float>(p.alpha), beta = static_cast<float>(p.beta), unscale = exact ? 1.0f : 1.0f / (SCALE * SCALE);
#pragma unroll
            for(uint32_t it = 0; it < 4; ++it)
            {
                const uint32_t row = m0 + 16u * it + (tid >> 4), col = n0 + (tid & 15u) * 4u;
                if(row < p.m && col < p.n)
                {
                    f32x4 out = sum[it] * unscale * alpha;
                    if(beta != 0.0f)
                        out += beta * *reinterpret_cast<const f32x4*>(p.c + ((uint64_t)row * p.ldc + col) * 4u);
                    __builtin_nontemporal_store(out, reinterpret_cast<f32x4*>(d + ((uint64_t)row * p.ldd + col) * 4u));
                }
            }
            return;
        }
    }
} // namespace

namespace r355
{
    void gemmF32Tiles(bool aK, bool bK, uint32_t splits, const GemmTileParams& p, hipStream_t stream)
    {
        const dim3 grid((p.tileCount + 7u) / 8u * 8u, splits), block(THREADS);
        if(aK && bK)
            hipLaunchKernelGGL((gemmF32Kernel<true, true>), grid, block, 0, stream, p);
        else if(aK)
            hipLaunchKernelGGL((gemmF32Kernel<true, false>), grid, block, 0, stream, p);
        else if(bK)
            hipLaunchKernelGGL((gemmF32Kernel<false, true>), grid, block, 0, stream, p);
        else
            hipLaunchKernelGGL((gemmF32Kernel<false, false>), grid, block, 0, stream, p);
    }
} // namespace r355
