// How a GEMV's rows are dealt out to workgroups and to launches: host arithmetic only, so that it can be checked without a device.
#ifndef R355_GEMV_ROWS_HPP
#define R355_GEMV_ROWS_HPP

#include <cstdint>

namespace r355
{
    // Waves and rows of a workgroup for a row-major A with rows below 128 KiB, {0, 0}: a wave per row, four to a workgroup (gemvRowMajor).  A row of a
    // few KiB wants as many waves as make one or two trips of it, so that its loads are all under way at once; a matrix from HBM wants two rows a workgroup,
    // which share x and keep as many loads more in flight; short rows by the ten thousands want four rows a wave.  168 random shapes from 256 to 16384
    // rows and columns, A in the memory-side cache or not: 1.03 times as long as the best of 13 combinations, where a wave per row takes 1.15 times
    // (f32 576 x 1780 from HBM 3.40 -> 2.81 us, 380 x 11964 10.9 -> 6.0, 8920 x 3796 26.4 -> 22.6, 9496 x 12800 87 -> 70; f64 2052 x 5680 25.7 -> 18.7), and
    // 1.02 on most shapes outside (f32 88 x 27708 18.2 -> 6.5, 390884 x 16 64 -> 35, 16384^2 160 -> 150).
    struct RowGroup
    {
        uint32_t waves, rows;
    };
    inline RowGroup rowGroup(uint32_t m, uint64_t rowBytes, uint32_t elemBytes)
    {
        const uint64_t bytes = rowBytes * m;
        if(rowBytes <= 2048u && m >= 16384u)
            return elemBytes == 8u && rowBytes < 256u ? RowGroup{0u, 0u} : RowGroup{1u, 4u}; // (f64 25772 x 24 5.0 -> 5.7)
        if(rowBytes <= 1024u)
            return {0u, 0u};
        if(rowBytes <= 5632u)
            return {1u, 1u};
        if(rowBytes <= 9344u)
            return {2u, 1u};
        if(bytes <= 23000000u)
            return {rowBytes < (64u << 10) ? 4u : 8u, 1u};
        return {bytes <= 165000000u ? 4u : 8u, 2u};
    }

    // Rows of one launch.  A launch's threads are counted in 32 bits: one of more runs what is left modulo 2^32 and reports success.  Col-major: 1024 threads for
    // 16 pieces of 16 bytes of a column, the form that many rows take; row-major: as rowGroup says, rows of 128 KiB and more at most sixteen waves for four.  More
    // rows than that go out in several launches of nearly the same size, each a whole number of 4096 rows, so that columns stay on the cache lines they are on.
    // (f32 row-major 2^24 + 64 x 2340, 157 GB: 512 threads for two rows are 2^32 + 16384.)
    inline uint32_t gemvLaunchRows(bool colMajor, uint32_t m, uint64_t rowBytes, uint32_t elemBytes)
    {
        RowGroup form{4u, 4u}; // (a wave per row)
        if(colMajor)
            form = {16u, 256u / elemBytes};
        else if(rowBytes >= (128u << 10))
            form = {16u, 4u};
        else if(const RowGroup group = rowGroup(m, rowBytes, elemBytes); group.waves != 0u)
            form = group;
        const uint64_t most = ((1ull << 32) - 1u) / (form.waves * 64u) * form.rows / 4096u * 4096u;
        const uint64_t launches = (m + most - 1u) / most, rows = ((m + launches - 1u) / launches + 4095u) / 4096u * 4096u;
        return launches == 1u ? m : static_cast<uint32_t>(rows);
    }
} // namespace r355

#endif // R355_GEMV_ROWS_HPP
