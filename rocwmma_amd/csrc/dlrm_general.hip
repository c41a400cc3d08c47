// DLRM dot interaction for the shapes the specialised kernels of dlrm.hip do not take: more than 32 features, or an
// embedding width other than 32 / 64 / 128 / 256 (the reference's own tests run m = 128, k = 128 and m = k = 1024 with a
// batch of 64: test/dlrm/test/dlrm_test_params.hpp:55-58).  Written on the fragment API as the reference's kernels are
// (test/dlrm/device/dlrm_dot_fwd.hpp:37-135, dlrm_dot_bwd.hpp:35-176), m and k multiples of 16 as there
// (dlrm_kernel_base_impl.hpp:146-151) - but without their global scratch: the forward kernels take the lower triangle
// out of an accumulator block through 1 KiB of the wave's LDS instead of a [batch][m][m] f32 buffer, and the backward
// kernels form each 16 x 16 block of S = T + T^T in LDS from the packed upstream triangle instead of reconstructing
// [batch][m][m] in memory first.  These kernels run one 16 x 16 block per wave, as in the reference, and the backward also several
// (register-blocked, so that a fragment feeds several matrix instructions); macro tiles (gemm_tiled.hip) take the shapes that
// they are faster on, by the timing models below.
#include <rocwmma/rocwmma.hpp>

#include "common.hpp"

using namespace rocwmma;

namespace
{
    constexpr uint32_t BLK = 16, WAVES = 4, THREADS = WAVES * 64;
    constexpr uint32_t GRID_BATCH = 65535; // samples per launch (the batch is grid dimension y or z)

    template <typename T>
    constexpr uint32_t blockK()
    {
        return sizeof(T) == 4 ? 4u : 16u; // the K depth of the 16 x 16 matrix instruction behind mma_sync
    }

    // Forward.  Wave p of sample blockIdx.y owns block (ti, tj), tj <= ti, of X X^T; p = ti (ti + 1) / 2 + tj.
    template <typename T>
    __global__ void __launch_bounds__(THREADS) dlrmFwdGeneral(const T* __restrict__ in, T* __restrict__ out, uint32_t m, uint32_t k,
                                                             uint32_t pairs)
    {
        constexpr uint32_t BK = blockK<T>();
        using FragA   = fragment<matrix_a, BLK, BLK, BK, T, row_major>;
        using FragB   = fragment<matrix_b, BLK, BLK, BK, T, col_major>;
        using FragAcc = fragment<accumulator, BLK, BLK, BK, float32_t>;
        __shared__ float block[WAVES][BLK * BLK];

        const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
        const uint32_t p    = blockIdx.x * WAVES + wave;
        if(p >= pairs)
            return;
        uint32_t ti = 0;
        while((ti + 1u) * (ti + 2u) / 2u <= p)
            ++ti;
        const uint32_t tj     = p - ti * (ti + 1u) / 2u;
        const uint64_t stride = (uint64_t)k + (uint64_t)m * (m - 1u) / 2u;
        const T*       x      = in + (uint64_t)blockIdx.y * m * k;
        T*             o      = out + (uint64_t)blockIdx.y * stride;

        if(p == 0u) // the bottom-MLP row
            for(uint32_t e = lane; e < k; e += 64u)
                o[e] = x[e];

        FragAcc acc;
        fill_fragment(acc, 0.0f);
        const T* pa = x + (uint64_t)ti * BLK * k; // rows of X
        const T* pb = x + (uint64_t)tj * BLK * k; // X^T as a col-major k x m matrix: column n is row n of X
        for(uint32_t kk = 0; kk < k; kk += BK)
        {
            FragA a;
            FragB b;
            load_matrix_sync(a, pa + kk, k);
            load_matrix_sync(b, pb + kk, k);
            mma_sync(acc, a, b, acc);
        }
        float* mine = block[wave];
        store_matrix_sync(mine, acc, BLK, mem_row_major);
        __builtin_amdgcn_wave_barrier(); // (LDS is in order within a wave: the reads below see the block)
#pragma unroll
        for(uint32_t i = 0; i < BLK * BLK / 64u; ++i)
        {
            const uint32_t e = i * 64u + lane, r = e / BLK, c = e % BLK;
            const uint64_t gi = (uint64_t)ti * BLK + r, gj = (uint64_t)tj * BLK + c;
            if(gj < gi)
                o[k + gi * (gi - 1u) / 2u + gj] = static_cast<T>(mine[e]);
        }
    }

    // Backward.  Wave (ti, kc) of sample blockIdx.z owns block (ti, kc) of the gradient S X; S(i, j) is the upstream
    // triangle's element (max, min) of i, j and zero on the diagonal.
    template <typename T>
    __global__ void __launch_bounds__(THREADS) dlrmBwdGeneral(const T* __restrict__ in, const T* __restrict__ upstream,
                                                             T* __restrict__ mlpGrad, T* __restrict__ inGrad, uint32_t m, uint32_t k)
    {
        constexpr uint32_t BK = blockK<T>();
        using FragA   = fragment<matrix_a, BLK, BLK, BK, T, row_major>;
        using FragB   = fragment<matrix_b, BLK, BLK, BK, T, row_major>;
        using FragAcc = fragment<accumulator, BLK, BLK, BK, float32_t>;
        __shared__ T     sBlock[WAVES][BLK * BLK];
        __shared__ float block[WAVES][BLK * BLK];

        const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
        const uint32_t kc   = blockIdx.x * WAVES + wave, ti = blockIdx.y;
        if(kc * BLK >= k)
            return;
        const uint64_t stride = (uint64_t)k + (uint64_t)m * (m - 1u) / 2u;
        const T*       x      = in + (uint64_t)blockIdx.z * m * k;
        const T*       up     = upstream + (uint64_t)blockIdx.z * stride;
        const T*       tril   = up + k;

        if(ti == 0u && lane < BLK) // bottom-MLP gradient: the first k values of the upstream row
            mlpGrad[(uint64_t)blockIdx.z * k + kc * BLK + lane] = up[kc * BLK + lane];

        FragAcc acc;
        fill_fragment(acc, 0.0f);
        T* s = sBlock[wave];
        for(uint32_t tj = 0; tj < m / BLK; ++tj)
        {
#pragma unroll
            for(uint32_t i = 0; i < BLK * BLK / 64u; ++i)
            {
                const uint32_t e = i * 64u + lane, r = e / BLK, c = e % BLK;
                const uint64_t gi = (uint64_t)ti * BLK + r, gj = (uint64_t)tj * BLK + c;
                const uint64_t hi = gi > gj ? gi : gj, lo = gi > gj ? gj : gi;
                s[e] = gi == gj ? static_cast<T>(0.0f) : tril[hi * (hi - 1u) / 2u + lo];
            }
            __builtin_amdgcn_wave_barrier();
            const T* pb = x + (uint64_t)tj * BLK * k + kc * BLK;
#pragma unroll
            for(uint32_t kk = 0; kk < BLK; kk += BK)
            {
                FragA a;
                FragB b;
                load_matrix_sync(a, s + kk, BLK);
                load_matrix_sync(b, pb + (uint64_t)kk * k, k);
                mma_sync(acc, a, b, acc);
            }
            __builtin_amdgcn_wave_barrier(); // the block of S is rewritten in the next trip
        }
        float* mine = block[wave];
        store_matrix_sync(mine, acc, BLK, mem_row_major);
        __builtin_amdgcn_wave_barrier();
        T* g = inGrad + (uint64_t)blockIdx.z * m * k + (uint64_t)ti * BLK * k + kc * BLK;
#pragma unroll
        for(uint32_t i = 0; i < BLK * BLK / 64u; ++i)
        {
            const uint32_t e = i * 64u + lane, r = e / BLK, c = e % BLK;
            g[(uint64_t)r * k + c] = static_cast<T>(mine[e]);
        }
    }

    // Backward for large launches: a wave owns NBI x NBK blocks of the gradient - row blocks ti0 .. ti0 + NBI - 1, column
    // blocks kc0 .. kc0 + NBK - 1 - and the four waves of a workgroup share ti0: the NBI blocks of S that a step needs
    // (gathers from the packed triangle with their index arithmetic, the expensive part) are formed once per workgroup,
    // one element per thread and block, in an LDS image that every wave reads, and each feeds NBK matrix instructions per
    // wave and K step.  The 16 rows of X that a step multiplies them with go the same way: the workgroup's 256 columns of
    // them are fetched with 128-bit loads into an LDS image, from which every wave takes its matrix_b fragments (16-bit
    // types: transposing reads) - a row-major matrix_b fragment straight from global memory is four 2-byte loads per lane.
    // Both images have two buffers, so a step costs one barrier; the gathers and the rows of X for step tj + 1 are in
    // flight while the matrix instructions of step tj run.  Below the diagonal a block's rows are contiguous in the
    // triangle, above it its columns are, and the threads are laid along whichever it is.
    template <typename T, uint32_t NBI, uint32_t NBK>
    __global__ void __launch_bounds__(THREADS) dlrmBwdGeneralBlocked(const T* __restrict__ in, const T* __restrict__ upstream,
                                                                    T* __restrict__ mlpGrad, T* __restrict__ inGrad, uint32_t m, uint32_t k)
    {
        constexpr uint32_t BK = blockK<T>(), KSTEPS = BLK / BK;
        static_assert(THREADS == BLK * BLK, "one thread per element of a block of S");
        using FragA   = fragment<matrix_a, BLK, BLK, BK, T, row_major>;
        using FragB   = fragment<matrix_b, BLK, BLK, BK, T, row_major>;
        using FragAcc = fragment<accumulator, BLK, BLK, BK, float32_t>;
        // (16-bit types.  f32 fragments are four 4-byte loads per lane either way, and the image - 33 KiB - costs more in
        // resident workgroups than it saves: 512 x 128 x 256 0.28 -> 0.32 ms with it; f32 takes its fragments from global memory)
        constexpr bool     STAGE_X = sizeof(T) == 2;
        constexpr uint32_t COLS = WAVES * NBK * BLK; // columns of X (and of the gradient) per workgroup
        constexpr uint32_t XLD  = COLS + 16u / sizeof(T); // row pitch of the image of X: 16 bytes of padding
        constexpr uint32_t CH   = 16u / sizeof(T), XLOADS = BLK * COLS / CH / THREADS; // elements per 128-bit load, loads per thread
        using i32x4             = int __attribute__((ext_vector_type(4)));
        __shared__ T     sBlock[2][NBI][BLK * BLK];
        __shared__ __attribute__((aligned(16))) T xBlock[STAGE_X ? 2 : 1][STAGE_X ? BLK * XLD : CH];
        __shared__ float block[WAVES][BLK * BLK];

        const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        const uint32_t col0 = blockIdx.x * COLS; // first column of the workgroup
        const uint32_t kc0  = (blockIdx.x * WAVES + wave) * NBK, ti0 = blockIdx.y * NBI;
        const uint32_t tilesK = k / BLK, tilesM = m / BLK;
        const bool     active = kc0 < tilesK; // (a wave without column blocks still gathers its share of S)
        const uint64_t stride = (uint64_t)k + (uint64_t)m * (m - 1u) / 2u;
        const T*       x      = in + (uint64_t)blockIdx.z * m * k;
        const T*       up     = upstream + (uint64_t)blockIdx.z * stride;
        const T*       tril   = up + k;

        if(ti0 == 0u && lane < BLK) // bottom-MLP gradient: the first k values of the upstream row
#pragma unroll
            for(uint32_t c = 0; c < NBK; ++c)
                if(kc0 + c < tilesK)
                    mlpGrad[(uint64_t)blockIdx.z * k + (kc0 + c) * BLK + lane] = up[(kc0 + c) * BLK + lane];

        FragAcc acc[NBI][NBK];
#pragma unroll
        for(uint32_t i = 0; i < NBI; ++i)
#pragma unroll
            for(uint32_t c = 0; c < NBK; ++c)
                fill_fragment(acc[i][c], 0.0f);

        T     sNext[NBI];
        i32x4 xNext[STAGE_X ? XLOADS : 1u];
        FragB bNext[STAGE_X ? 1u : KSTEPS][NBK];
        auto  place = [&](uint32_t i, uint32_t tj, uint32_t& r, uint32_t& c) {
            const bool upper = tj > ti0 + i;
            r = upper ? tid % BLK : tid / BLK;
            c = upper ? tid / BLK : tid % BLK;
        };
        auto fetch = [&](uint32_t tj) {
#pragma unroll
            for(uint32_t i = 0; i < NBI; ++i)
            {
                uint32_t r, c;
                place(i, tj, r, c);
                const uint64_t gi = (uint64_t)(ti0 + i < tilesM ? ti0 + i : ti0) * BLK + r, gj = (uint64_t)tj * BLK + c;
                const uint64_t hi = gi > gj ? gi : gj, lo = gi > gj ? gj : gi;
                sNext[i] = gi == gj ? static_cast<T>(0.0f) : tril[hi * (hi - 1u) / 2u + lo];
            }
            if constexpr(STAGE_X)
            {
#pragma unroll
                for(uint32_t j = 0; j < XLOADS; ++j) // rows tj * 16 ... of X, the workgroup's columns (k is a multiple of 16: whole pieces)
                {
                    const uint32_t piece = j * THREADS + tid, r = piece / (COLS / CH), c = col0 + (piece % (COLS / CH)) * CH;
                    if(c < k)
                        xNext[j] = *reinterpret_cast<const i32x4*>(x + ((uint64_t)tj * BLK + r) * k + c);
                }
            }
            else if(active)
            {
#pragma unroll
                for(uint32_t ks = 0; ks < KSTEPS; ++ks)
#pragma unroll
                    for(uint32_t c = 0; c < NBK; ++c) // (a column block past the end reads the last one again: its products are not used)
                        load_matrix_sync(bNext[ks][c],
                                         x + (uint64_t)tj * BLK * k + (uint64_t)(kc0 + c < tilesK ? kc0 + c : tilesK - 1u) * BLK + (uint64_t)ks * BK * k, k);
            }
        };
        fetch(0u);
        for(uint32_t tj = 0; tj < tilesM; ++tj)
        {
            T(*s)[BLK * BLK] = sBlock[tj & 1u];
            T* xs            = xBlock[STAGE_X ? tj & 1u : 0u];
            FragB bNow[STAGE_X ? 1u : KSTEPS][NBK];
#pragma unroll
            for(uint32_t i = 0; i < NBI; ++i)
            {
                uint32_t r, c;
                place(i, tj, r, c);
                s[i][r * BLK + c] = sNext[i];
            }
            if constexpr(STAGE_X)
            {
#pragma unroll
                for(uint32_t j = 0; j < XLOADS; ++j)
                {
                    const uint32_t piece = j * THREADS + tid, r = piece / (COLS / CH), c = (piece % (COLS / CH)) * CH;
                    if(col0 + c < k)
                        *reinterpret_cast<i32x4*>(xs + r * XLD + c) = xNext[j];
                }
            }
            else
            {
#pragma unroll
                for(uint32_t ks = 0; ks < KSTEPS; ++ks)
#pragma unroll
                    for(uint32_t c = 0; c < NBK; ++c)
                        bNow[ks][c] = bNext[ks][c];
            }
            // the one barrier of the step: these buffers are complete; the others, which the next step writes, were last read
            // in the step before this one, and every wave has finished that step to get here
            __syncthreads();
            if(tj + 1u < tilesM)
                fetch(tj + 1u);
            if(active)
#pragma unroll
                for(uint32_t ks = 0; ks < KSTEPS; ++ks)
                {
                    FragA a[NBI];
                    FragB b[NBK];
#pragma unroll
                    for(uint32_t i = 0; i < NBI; ++i)
                        load_matrix_sync(a[i], s[i] + ks * BK, BLK);
#pragma unroll
                    for(uint32_t c = 0; c < NBK; ++c)
                        if constexpr(STAGE_X)
                            load_matrix_sync(b[c], xs + ks * BK * XLD + ((kc0 + c < tilesK ? kc0 + c : tilesK - 1u) * BLK - col0), XLD);
                        else
                            b[c] = bNow[ks][c];
#pragma unroll
                    for(uint32_t i = 0; i < NBI; ++i)
#pragma unroll
                        for(uint32_t c = 0; c < NBK; ++c)
                            if(ti0 + i < tilesM && kc0 + c < tilesK)
                                mma_sync(acc[i][c], a[i], b[c], acc[i][c]);
                }
        }
        if(!active)
            return;
        float* mine = block[wave];
#pragma unroll
        for(uint32_t i = 0; i < NBI; ++i)
#pragma unroll
            for(uint32_t c = 0; c < NBK; ++c)
            {
                if(ti0 + i >= tilesM || kc0 + c >= tilesK)
                    continue;
                store_matrix_sync(mine, acc[i][c], BLK, mem_row_major);
                __builtin_amdgcn_wave_barrier();
                T* g = inGrad + (uint64_t)blockIdx.z * m * k + (uint64_t)(ti0 + i) * BLK * k + (uint64_t)(kc0 + c) * BLK;
#pragma unroll
                for(uint32_t q = 0; q < BLK * BLK / 64u; ++q)
                {
                    const uint32_t e = q * 64u + lane, r = e / BLK, cc = e % BLK;
                    g[(uint64_t)r * k + cc] = static_cast<T>(mine[e]);
                }
                __builtin_amdgcn_wave_barrier(); // the block is rewritten by the next one
            }
    }

#ifdef R355_DLRM_BLOCK_PER_WAVE // measurement build: the block-per-wave kernels for every shape
    constexpr bool ONLY_BLOCK_PER_WAVE = true;
#else
    constexpr bool ONLY_BLOCK_PER_WAVE = false;
#endif

    // Which kernel a launch runs is the cheapest by a timing model: microseconds as a linear function of the launch's workgroups
    // (or waves; `groups` in thousands on 256 CUs), their steps along K and one more term.  Fitted by least squares of the relative
    // error to launches of every kernel on the same random shapes, m from 32 to 1024, k from 16 to 1024, up to 12000 samples
    // (profiles/tile_choice_survey.md: how well the models do, and what the choices give on further shapes).  The tiles' constants of the 16-bit types were
    // fitted when their diagonal stages, and the forward's stores, took up to 1.5 times as long as now: on 665 further 16-bit shapes the choice takes
    // 1.010 (forward) and 1.033 (backward) times as long as the fastest of itself and the two tiles, 87 of them more than 3 % longer.
    struct LaunchTime
    {
        double fixed, step, group, groupStep, more;
        double operator()(double steps, double groups, double term) const
        {
            return fixed + step * steps + groups * (group + groupStep * steps) + more * term;
        }
    };
    double thousands(uint64_t groups)
    {
        return static_cast<double>(groups) / (4.0 * r355::computeUnits());
    }
    uint64_t tilesOf(uint32_t n, uint32_t edge)
    {
        return (n - 1u) / edge + 1u;
    }
    uint64_t triangle(uint64_t rows) // blocks or tiles on and below the diagonal
    {
        return rows * (rows + 1u) / 2u;
    }

    // Forward.  A block per wave (steps of one matrix instruction) has the shortest launch, pads nothing, and re-reads every row of X for
    // each block of the sample, from lines that collide in the caches where rows are multiples of 128 bytes (the last term: waves times
    // steps again).  Macro tiles (steps: stages of 128 bytes; the last term: megabytes of input and output) read a row once per 64 or 128
    // others but pad m to the tile's edge: with few features or a short K most of a tile is padding and fixed cost.  bf16 32 x 48 x 7174: 10.3 us a block
    // per wave, 21 on 64 x 64 tiles, 48 on 128 x 128 ones; f16 64 x 112 x 2687: 28, 13.3 and 24; bf16 176 x 576 x 428: 227, 28 and 32; f16
    // 1024 x 1024 x 64: 136 and 88 on tiles.  Beyond 160 features only small launches run a block per wave: its reads of the
    // rows of X then cost more than the model says (bf16 192 x 16 x 505: 15.6 us, modelled 11, 12.0 on 64 x 64 tiles).
    constexpr LaunchTime FWD_WAVE[2]  = {{2.70, 0.0415, 0.104, 0.124, 0.104}, {2.48, 0.0954, 0.135, 0.225, 0.00649}}; // 16-bit, f32
    constexpr LaunchTime FWD_64[2]    = {{3.38, 0.00367, 2.13, 0.564, 0.0370}, {3.49, 0.227, 1.95, 1.62, 0.0517}};
    constexpr LaunchTime FWD_128      = {3.88, 0.124, 5.27, 0.804, 0.0816}; // 16-bit: f32, bound by its matrix instructions, is faster on 64 x 64 throughout
    constexpr double     FWD_MARGIN   = 0.97; // a tile has to be ahead of the block per wave by that
    // The kernel of a launch, an r355_dlrm_kernel_id.  Up to 16 features a sample is a single block.  Leading dimensions beyond 8 MiB per row do not
    // fit the tile kernels' (dlrmFwdTiled in gemm_tiled.hip) 32-bit lane offsets.
    int forwardKernel(int32_t dtype, uint32_t m, uint32_t k, uint32_t batch)
    {
        const uint64_t rowBytes = (uint64_t)k * r355::dtypeBytes(dtype);
        if(ONLY_BLOCK_PER_WAVE || m <= BLK || rowBytes > (1u << 23))
            return R355_DLRM_KERNEL_BLOCK_PER_WAVE;
        const bool     wide  = dtype == R355_F32;
        const uint64_t waves = triangle(m / BLK) * batch, steps = k / (wide ? 4u : 16u), stages = (rowBytes + 127u) / 128u;
        const double   megabytes
            = 1e-6 * r355::dtypeBytes(dtype) * batch * (static_cast<double>(m) * k + 0.5 * m * (m - 1.0) + static_cast<double>(k));
        const double small = FWD_64[wide](stages, thousands(triangle(tilesOf(m, 64u)) * batch), megabytes);
        const double large = FWD_128(stages, thousands(triangle(tilesOf(m, 128u)) * batch), megabytes);
        const double tiles = wide || small < large ? small : large;
        if(m <= 160u || waves <= 5u * r355::computeUnits())
            if(FWD_WAVE[wide](steps, thousands(waves), rowBytes % 128u == 0u ? thousands(waves) * steps : 0.0) * FWD_MARGIN <= tiles)
                return R355_DLRM_KERNEL_BLOCK_PER_WAVE;
        // (a sample of more 64 x 64 tiles than a launch holds: f32, 370704 features and more, a result of 256 GiB)
        return tiles == small && triangle(tilesOf(m, 64u)) <= r355::MAX_GROUPS ? R355_DLRM_KERNEL_TILED_64 : R355_DLRM_KERNEL_TILED_128;
    }

    // Backward.  The fragment-API kernels are a block per wave and 2 x 4 blocks per wave (the register-blocked kernel; waves of 32 x 64 of the
    // gradient, workgroups of 32 x 256 that form S once); macro tiles pad m and the K of the product, which is m again, to 64 or 128.  f16 32 x 208 x 4021: 33 us register-blocked,
    // 45 on 64 x 64 tiles; f16 80 x 208 x 1410: 38 and 42; f16 112 x 48 x 1612: 44 and 15.5; f16 1024 x 256 x 4: 96 a block per wave, 11.8 on
    // 64 x 64; f16 992 x 464 x 27: 117 register-blocked, 69 on 64 x 64, 52 on 128 x 128 tiles; f16 1024 x 1024 x 64: 473, 328 and 222.
    // By f16, bf16, f32.  Steps: blocks of 16 rows (fragments), stages of 128 bytes of K (tiles); the last term: megabytes, for the
    // register-blocked kernel thousands of block products.
    constexpr LaunchTime BWD_WAVE[3]    = {{1.71, 0.538, 0.0, 0.195, 0.305}, {1.97, 0.543, 0.0, 0.187, 0.296}, {1.77, 0.735, 0.0, 0.303, 0.124}};
    constexpr LaunchTime BWD_BLOCKED[3] = {{2.87, 0.531, 1.02, 0.552, 0.0157}, {4.33, 0.481, 1.23, 0.551, 0.0171}, {3.27, 0.916, 1.28, 0.691, 0.142}};
    constexpr LaunchTime BWD_64[3]      = {{3.39, 0.247, 1.27, 0.827, 0.132}, {3.48, 0.221, 1.33, 0.808, 0.128}, {2.91, 0.5, 1.24, 2.11, 0.0614}};
    constexpr LaunchTime BWD_128[3]     = {{3.77, 0.998, 2.94, 1.81, 0.251}, {3.38, 1.31, 2.52, 1.69, 0.238}, {3.27, 1.83, 4.09, 7.22, 0.0915}};
    constexpr double     BWD_MARGIN[3]  = {0.96, 0.92, 0.98}; // a tile has to be ahead of the fragment kernels by that: the models' error there
    constexpr uint32_t   NBI = 2, NBK = 4; // blocks per wave of the register-blocked kernel
    // The kernel of a launch, an r355_dlrm_kernel_id.  The tile kernel (dlrmBwdTiled in gemm_tiled.hip) reads upstream and writes mlpGrad in 16-byte
    // pieces (`aligned`), and rows beyond 8 MiB do not fit its 32-bit lane offsets.  Where it cannot run, and up to 16 features, for which
    // the models are not fitted, the register-blocked kernel takes launches that leave every SIMD two of its waves.
    int backwardKernel(int32_t dtype, bool aligned, uint32_t m, uint32_t k, uint32_t batch)
    {
        const uint32_t es = r355::dtypeBytes(dtype), blocks = m / BLK, samples = batch < GRID_BATCH ? batch : GRID_BATCH;
        const uint64_t waves = tilesOf(k, NBK * BLK) * tilesOf(m, NBI * BLK); // of a sample, register-blocked
        if(ONLY_BLOCK_PER_WAVE)
            return R355_DLRM_KERNEL_BLOCK_PER_WAVE;
        if(m <= BLK || (uint64_t)k * es > (1u << 23) || !aligned)
            return waves * samples >= 8ull * r355::computeUnits() ? R355_DLRM_KERNEL_REGISTER_BLOCKED : R355_DLRM_KERNEL_BLOCK_PER_WAVE;
        const uint32_t type   = dtype == R355_F16 ? 0u : dtype == R355_BF16 ? 1u : 2u;
        const uint64_t stages = ((uint64_t)m * es + 127u) / 128u, rows = tilesOf(m, NBI * BLK) * batch;
        const double   megabytes = 1e-6 * es * batch * (2.0 * m * k + 0.5 * m * (m - 1.0) + static_cast<double>(k));
        const double   wave      = BWD_WAVE[type](blocks, thousands((uint64_t)blocks * (k / BLK) * batch), megabytes);
        const LaunchTime& t      = BWD_BLOCKED[type];
        const double   blocked   = t.fixed + t.step * blocks + t.group * thousands(waves * batch) + t.groupStep * blocks * thousands(rows * tilesOf(k, 256u))
                               + t.more * blocks * thousands(rows * (k / BLK));
        const double fragments = wave < blocked ? wave : blocked;
        const double small     = BWD_64[type](stages, thousands(tilesOf(m, 64u) * tilesOf(k, 64u) * batch), megabytes);
        const double large     = BWD_128[type](stages, thousands(tilesOf(m, 128u) * tilesOf(k, 128u) * batch), megabytes);
        if(fragments * BWD_MARGIN[type] <= (small < large ? small : large))
            return wave < blocked ? R355_DLRM_KERNEL_BLOCK_PER_WAVE : R355_DLRM_KERNEL_REGISTER_BLOCKED;
        return small <= large && tilesOf(m, 64u) * tilesOf(k, 64u) <= r355::MAX_GROUPS ? R355_DLRM_KERNEL_TILED_64 : R355_DLRM_KERNEL_TILED_128;
    }

    template <typename T>
    int fwd(const void* in, void* out, uint32_t m, uint32_t k, uint32_t batch, hipStream_t s)
    {
        const uint32_t tiles = m / BLK, pairs = tiles * (tiles + 1u) / 2u;
        const uint64_t stride = (uint64_t)k + (uint64_t)m * (m - 1u) / 2u;
        // the batch is a grid dimension of at most 65535: a larger one goes out in several launches on the same stream
        for(uint32_t first = 0; first < batch; first += GRID_BATCH)
        {
            const uint32_t count = batch - first < GRID_BATCH ? batch - first : GRID_BATCH;
            const dim3     grid((pairs + WAVES - 1u) / WAVES, count);
            const T*       src = static_cast<const T*>(in) + (uint64_t)first * m * k;
            T*             dst = static_cast<T*>(out) + (uint64_t)first * stride;
            hipLaunchKernelGGL((dlrmFwdGeneral<T>), grid, dim3(THREADS), 0, s, src, dst, m, k, pairs);
        }
        return r355::checkLaunch("dlrm_fwd (general)");
    }
    template <typename T>
    int bwd(const void* in, const void* up, void* mlp, void* grad, uint32_t m, uint32_t k, uint32_t batch, bool blocked, hipStream_t s)
    {
        const uint64_t stride = (uint64_t)k + (uint64_t)m * (m - 1u) / 2u;
        for(uint32_t first = 0; first < batch; first += GRID_BATCH)
        {
            const uint32_t count = batch - first < GRID_BATCH ? batch - first : GRID_BATCH;
            const T*           src = static_cast<const T*>(in) + (uint64_t)first * m * k;
            const T*           ups = static_cast<const T*>(up) + (uint64_t)first * stride;
            T*                 dm  = static_cast<T*>(mlp) + (uint64_t)first * k;
            T*                 dg  = static_cast<T*>(grad) + (uint64_t)first * m * k;
            if(blocked) // NBI x NBK blocks per wave
                hipLaunchKernelGGL((dlrmBwdGeneralBlocked<T, NBI, NBK>),
                                   dim3(((k / BLK + NBK - 1u) / NBK + WAVES - 1u) / WAVES, (m / BLK + NBI - 1u) / NBI, count), dim3(THREADS), 0,
                                   s, src, ups, dm, dg, m, k);
            else
                hipLaunchKernelGGL((dlrmBwdGeneral<T>), dim3((k / BLK + WAVES - 1u) / WAVES, m / BLK, count), dim3(THREADS), 0, s, src, ups, dm, dg,
                                   m, k);
        }
        return r355::checkLaunch("dlrm_bwd (general)");
    }

    int checkGeneral(const char* what, uint32_t m, uint32_t k, uint32_t batch)
    {
        if(m % BLK || k % BLK || m == 0u || k == 0u)
            return r355::fail(R355_ERR_BAD_SIZE,
                              "%s: m=%u, k=%u - beyond m <= 32 with k of 32, 64, 128 or 256 (f32: up to 128) both must be multiples of %u", what,
                              m, k, BLK);
        (void)batch; // any batch: beyond 65535 samples the launch is repeated (fwd / bwd above)
        return R355_OK;
    }
} // namespace

namespace r355
{
    int dlrmGeneralFwd(int32_t dtype, const void* in, void* out, uint32_t m, uint32_t k, uint32_t batch, hipStream_t s)
    {
        const int rc = checkGeneral("dlrm_fwd", m, k, batch);
        if(rc != R355_OK)
            return rc;
        const int kernel = forwardKernel(dtype, m, k, batch);
        if(kernel != R355_DLRM_KERNEL_BLOCK_PER_WAVE)
            return dlrmFwdTiled(dtype, in, out, m, k, batch, kernel == R355_DLRM_KERNEL_TILED_64 ? 64u : 128u, s);
        switch(dtype)
        {
        case R355_F16: return fwd<float16_t>(in, out, m, k, batch, s);
        case R355_BF16: return fwd<bfloat16_t>(in, out, m, k, batch, s);
        default: return fwd<float32_t>(in, out, m, k, batch, s);
        }
    }
    int dlrmGeneralKernel(int32_t dtype, bool backward, uint32_t m, uint32_t k, uint32_t batch, bool aligned16)
    {
        const int rc = checkGeneral(backward ? "dlrm_bwd" : "dlrm_fwd", m, k, batch);
        if(rc != R355_OK)
            return rc;
        return backward ? backwardKernel(dtype, aligned16, m, k, batch) : forwardKernel(dtype, m, k, batch);
    }
    int dlrmGeneralBwd(int32_t dtype, const void* in, const void* upstream, void* mlpGrad, void* inGrad, uint32_t m, uint32_t k,
                       uint32_t batch, hipStream_t s)
    {
        const int rc = checkGeneral("dlrm_bwd", m, k, batch);
        if(rc != R355_OK)
            return rc;
        const int kernel = backwardKernel(dtype, aligned(upstream, 16) && aligned(mlpGrad, 16), m, k, batch);
        if(kernel == R355_DLRM_KERNEL_TILED_64 || kernel == R355_DLRM_KERNEL_TILED_128)
            return dlrmBwdTiled(dtype, in, upstream, mlpGrad, inGrad, m, k, batch, kernel == R355_DLRM_KERNEL_TILED_64 ? 64u : 128u, s);
        const bool blocked = kernel == R355_DLRM_KERNEL_REGISTER_BLOCKED;
        switch(dtype)
        {
        case R355_F16: return bwd<float16_t>(in, upstream, mlpGrad, inGrad, m, k, batch, blocked, s);
        case R355_BF16: return bwd<bfloat16_t>(in, upstream, mlpGrad, inGrad, m, k, batch, blocked, s);
        default: return bwd<float32_t>(in, upstream, mlpGrad, inGrad, m, k, batch, blocked, s);
        }
    }
} // namespace r355
