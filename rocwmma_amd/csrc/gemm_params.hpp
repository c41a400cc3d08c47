// What a macro-tile GEMM launch hands its kernels, shared by the translation units that hold them.
#ifndef R355_GEMM_PARAMS_HPP
#define R355_GEMM_PARAMS_HPP

#include "common.hpp"

namespace r355
{
    struct GemmTileParams
    {
        uint32_t    m, n, k;
        const char* a;
        const char* b;
        const char* c;
        char*       d;
        uint32_t    lda, ldb, ldc, ldd; // elements
        double      alpha, beta; // narrowed to the accumulator type in the epilogue
        uint32_t    tilesM, tilesN;
        // the launch covers tile indices [tileFirst, tileFirst + tileCount) of the tilesM x tilesN walk; with
        // tileQuad the walk is over tiles of twice the kernel's edge, four workgroups each (tile_map.hpp)
        uint32_t tileFirst, tileCount, tileQuad;
        // split-K (128 x 128 tile kernels): workgroup row blockIdx.y multiplies K stages [y * splitStages, (y + 1) * splitStages)
        // and writes its partial D (in the accumulator type) at d + y * splitStrideD bytes; 0 = the whole K in one workgroup
        uint32_t splitStages;
        uint64_t splitStrideD;
        // host side only: 16-bit operands on the 256 x 256 tile take the five-buffer K loop instead of the two-buffer one
        uint32_t deepPipeline;
        // experiment (R355_STAGGER_TICKS in the environment, 10 ns units; 0 = off): the first staggerBlocks workgroups - the
        // first round over the CUs - start 0, 1, 2 or 3 x stagger ticks late, by groups of CUs within each XCD, so that
        // the rounds' epilogues do not all store at once
        uint32_t stagger, staggerBlocks;
    };
    constexpr uint32_t F32_TILES_LDS = 65536; // bytes of a workgroup of the following
    // f32 GEMM on the bf16 matrix instructions, 64 x 64 tiles (gemm_f32.hip): a launch of p.tileCount tiles x `splits` shares of K
    void gemmF32Tiles(bool aK, bool bK, uint32_t splits, const GemmTileParams& p, hipStream_t stream);
    // Whether an f32 launch of 64 x 64 tiles takes that kernel: more workgroups than CUs, K shares of 16 stages (512 elements) at least.
    // 70 random shapes of 260 to 2900 workgroups and K from 512 to 3640: 0.98 to 1.30 times as fast, 1.11 in the geometric mean (493 tiles x 3080
    // 93.0 -> 79.3 us, 1521 x 1856 165 -> 140, 294 x 3632 in three shares 75.0 -> 67.4; below K = 640, 0.98 to 1.05: 510 x 548 19.7 -> 20.1, 896 x 512 31.9 -> 31.0).  A CU's
    // only workgroup has nothing that covers its loads: 207 tiles x 2128 36.3 -> 35.9, 132 x 1024 18.6 -> 19.5, 24 x 272 7.1 -> 9.3; short K is
    // latency and the partial tiles' meeting: 1024 x 64 8.0 -> 12.3.
    // Shares of K want 22: they are for few tiles, and one or two rounds of short ones are the partial tiles' meeting: 48 tiles x 5168 in ten shares of 17 stages
    // 22.2 -> 25.1, 27 x 7924 in sixteen of 16 21.6 -> 25.5, 186 x 2364 in four of 19 33.7 -> 34.9; 108 x 2868 in four of 23 27.8 -> 27.2.
    inline bool f32TilesOnBf16(uint64_t tiles, uint32_t splits, uint32_t stages)
    {
        return tiles * splits > computeUnits() && stages >= (splits > 1u ? 22u : 16u);
    }
} // namespace r355

#endif // R355_GEMM_PARAMS_HPP
