// Sweep launchers (row and column passes and their variants) for one resolution N; each
// sweeps_<N>.hip instantiates them so the resolutions compile in parallel.
#pragma once
#include "engine_internal.hpp"

namespace mse_rt {

// Blocks of a persistent kernel that stay resident per CU (HIP's occupancy query for that
// kernel, asked once), at most `cap`: the persistent sweeps size their grids to what runs
// at once, so no block waits for another to finish before it starts.
template <auto KERNEL>
int resident_per_cu(int block_threads, int cap) {
    static const int n = [&]() {
        int b = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&b, KERNEL, block_threads, 0) != hipSuccess) {
            (void)hipGetLastError();
            b = cap;
        }
        return std::max(1, std::min(b, cap));
    }();
    return n;
}

template <int N>
void row_pass_n(mse_engine* e, int mode, const float2* in, float2* out, int nlines_sets, size_t wave_stride,
                const mse::RowArgs& args, int variant) {
    using P0 = typename mse::PlanFor<N>::P;
    using P1 = typename mse::PlanHalfLanes<N>::P;
    using REG = std::true_type;
    using MEM = std::false_type;
    const bool step = mode == mse::ROW_IFFT_T_FFT;
    if (step && variant < 0) {
        // Rule: while every line of the grid takes one row at most, the plain kernel (its waves go
        // straight to the loads); beyond, the persistent one, which keeps a transmission row in
        // registers over the waves and prefetches.  With 12 elements per lane the plain kernel's
        // fourth wave per SIMD outweighs both up to some 65,000 rows.  Plain against persistent,
        // us: 256^2 one wave 4.2 / 4.8, 32 waves 8.4 / 9.0; 384^2 48 waves 22 / 24, 128 waves
        // 50 / 53; 512^2 one 4.8 / 5.2, 8 waves 9.3 / 10.0, 16 waves 14.9 / 14.0, 64 waves
        // 45 / 35; 768^2 8 waves 17.6 / 18.9, 64 waves 96 / 99, 128 waves 216 / 194; 1024^2 2
        // waves 10.4 / 10.8, 8 waves 25.2 / 25.2, 64 waves 208 / 147.
        using K = std::integral_constant<int, mse::BAND_STEP>;
        const int per_cu = resident_per_cu<mse::k_row_step_pipe<P0, K::value, mse::WaveSync, true>>(256, 8);
        const bool one_round = nlines_sets <= e->num_cus * per_cu * (256 / P0::L) / N;
        variant = one_round || (P0::E == 12 && (long long)N * nlines_sets <= 65536) ? 0 : 4;
    }
    // one row per line of the grid, out of place or with the non-persistent variants
    auto go = [&](auto plan, auto sync, auto twreg) {
        using PL = decltype(plan);
        using SY = decltype(sync);
        constexpr bool TR = decltype(twreg)::value;
        constexpr int WPE = TR ? 1 : 8;
        constexpr int LINES = 256 / PL::L;
        dim3 grid(N / LINES, nlines_sets);
        launch(e, PK_ROW, [&]() {
#define MSE_ROW_CASE(M, IO)                                                                                         \
    if (mode == mse::M && args.io == mse::IO) {                                                                     \
        mse::k_row<PL, mse::M, mse::IO, SY, TR, WPE><<<grid, 256, 0, e->stream>>>(in, out, wave_stride, e->tw.p, args); \
        return;                                                                                                     \
    }
            MSE_ROW_CASE(ROW_IFFT_T_FFT, BAND_FULL)
            MSE_ROW_CASE(ROW_IFFT_T_FFT, BAND_FIRST)
            MSE_ROW_CASE(ROW_IFFT_T_FFT, BAND_STEP)
            if constexpr (TR && std::is_same<SY, mse::WaveSync>::value && std::is_same<PL, P0>::value) {
                MSE_ROW_CASE(ROW_FFT, BAND_FULL)
                MSE_ROW_CASE(ROW_IFFT_WIDE, BAND_FULL)
                MSE_ROW_CASE(ROW_COPY, BAND_FULL)
                MSE_ROW_CASE(ROW_IFFT_INTENSITY, BAND_FULL)
                MSE_ROW_CASE(ROW_ADJ_SEED, BAND_FULL)
                MSE_ROW_CASE(ROW_ADJ, BAND_FULL)
                MSE_ROW_CASE(ROW_ADJ, BAND_STEP)
            }
#undef MSE_ROW_CASE
            throw Error(MSE_ERR_STATE, "row pass without a kernel");
        });
    };
    // the persistent pipelined kernel, in place
    auto go_pipe = [&](auto plan, auto twreg, auto m, auto io) {
        using PL = decltype(plan);
        constexpr bool TR = decltype(twreg)::value;
        constexpr int MD = decltype(m)::value, IO = decltype(io)::value;
        constexpr int LINES = 256 / PL::L;
        const int per_cu = resident_per_cu<mse::k_row_step_pipe<PL, IO, mse::WaveSync, TR, MD>>(256, 8);
        // whole groups of N lines; as few as the rounds over the sets need
        const int most = std::max(1, e->num_cus * per_cu * LINES / N);
        const int rounds = (nlines_sets + most - 1) / most;
        const int blocks = (nlines_sets + rounds - 1) / rounds * (N / LINES);
        launch(e, PK_ROW, [&]() {
            mse::k_row_step_pipe<PL, IO, mse::WaveSync, TR, MD><<<blocks, 256, 0, e->stream>>>(
                out, wave_stride, e->tw.p, args, nlines_sets);
        });
    };
    auto pipe_step = [&](auto plan, auto twreg) {
        using M = std::integral_constant<int, mse::ROW_IFFT_T_FFT>;
        if (args.io == mse::BAND_STEP)
            go_pipe(plan, twreg, M{}, std::integral_constant<int, mse::BAND_STEP>{});
        else if (args.io == mse::BAND_FIRST)
            go_pipe(plan, twreg, M{}, std::integral_constant<int, mse::BAND_FIRST>{});
        else
            go_pipe(plan, twreg, M{}, std::integral_constant<int, mse::BAND_FULL>{});
    };
    if ((mode == mse::ROW_FFT || mode == mse::ROW_IFFT) && in == out) {
        // one transform in place (the band limit of transmission functions): the persistent
        // pipelined kernel, whatever the tuned variant
        using FFT = std::integral_constant<int, mse::ROW_FFT>;
        using IFFT = std::integral_constant<int, mse::ROW_IFFT>;
        using FULL = std::integral_constant<int, mse::BAND_FULL>;
        if (mode == mse::ROW_FFT && args.io == mse::BAND_WRITE)
            go_pipe(P0{}, REG{}, FFT{}, std::integral_constant<int, mse::BAND_WRITE>{});
        else if (mode == mse::ROW_FFT)
            go_pipe(P0{}, REG{}, FFT{}, FULL{});
        else if (args.io == mse::BAND_READ)
            go_pipe(P0{}, REG{}, IFFT{}, std::integral_constant<int, mse::BAND_READ>{});
        else
            go_pipe(P0{}, REG{}, IFFT{}, FULL{});
        return;
    }
    if (step && variant >= 4 && in == out) {
        if constexpr (N <= 512) {  // half-lane lines keep the prefetch registers within budget up to 512
            if (variant == 5) return pipe_step(P1{}, REG{});
        }
        return variant == 6 ? pipe_step(P0{}, MEM{}) : pipe_step(P0{}, REG{});
    }
    if (step && variant == 1)
        go(P1{}, mse::WaveSync{}, REG{});
    else if (step && variant == 2)
        go(P0{}, mse::BlockSync{}, REG{});
    else if (step && variant == 3)
        go(P0{}, mse::WaveSync{}, MEM{});
    else
        go(P0{}, mse::WaveSync{}, REG{});
}

// returns the number of column tiles of the launch (detector partials per wave)
template <int N>
int col_pass_n(mse_engine* e, int mode, const float2* in, float2* out, int nsets, size_t wave_stride,
               const mse::ColArgs& args0, int kind, int variant) {
    using P0 = typename mse::PlanFor<N>::P;
    using P1 = typename mse::PlanHalfLanes<N>::P;
    using C16 = std::integral_constant<int, 16>;
    using C8 = std::integral_constant<int, 8>;
    using C4 = std::integral_constant<int, 4>;
    using C32 = std::integral_constant<int, 32>;
    using REG = std::true_type;
    using MEM = std::false_type;
    const bool prop = mode == mse::COL_PROP || mode == mse::COL_PROP_DETECT || mode == mse::COL_PROP_CONJ;
    const bool hot = mode == mse::COL_PROP || mode == mse::COL_PROP_DETECT || mode == mse::COL_COPY;
    const bool band = prop && args0.band_k >= 0;
    if (!hot) variant = 0;
    mse::ColArgs args = args0;
    if (mode == mse::COL_PROP && in == out && variant < 0) {
        // Rule: the narrowest tiles while they leave CUs idle, wider ones as the launch grows (a
        // narrow tile is a shorter chain of loads, transforms and stores, a wide one moves whole
        // 128-byte lines and shares a line's transfer with no other block); with 12 elements per
        // lane the lean kernel, whose four waves per SIMD need no prefetch registers (the
        // persistent one has two).  us per launch on the band, persistent with 4 / 8 / 16 columns
        // (the first two in XCD-aware order) / lean:
        //   256^2 one wave 4.5 / 5.0 / 5.6 / 6.1, 16 waves 6.1 / 6.4 / 6.5 / 7.0, 64 15.4 / 15.5 / 12.3 / 13.0
        //   384^2 one 6.5 / 7.2 / 9.1 / 8.3, 8 waves 8.4 / 8.1 / 9.9 / 9.2, 32 17.6 / 17.3 / 17.4 / 15.8
        //   512^2 one 5.8 / 6.4 / 9.8 / 8.7, 8 waves 9.2 / 10.3 / 11.5 / 10.7, 64 49 / 38.8 / 38.9 / 44
        //   768^2 one 8.4 / 10.5 / 27 / 9.0, 4 waves 12.3 / 12.2 / 30 / 11.2, 64 108 / 103 / 235 / 97, 128 255 / 252 / - / 198
        //   1024^2 one 10.3 / 12.1 / 33 / 11.3, 4 waves 22.4 / 20.8 / 42 / 17.9, 16 48 / 48 / 108 / 52, 64 188 / 176 / 407 / 228
        // (16 columns of the 12- and 16-element plans spill.)  In a loop, where the row pass comes
        // between and the waves are written through (us per slice, 4 / 8 / 16 columns / lean):
        //   256^2 16 waves 11.8 / 11.7 / 11.7 / 12.8, 32 16.6 / 15.0 / 16.0 / 18.7, 64 29.2 / 25.8 / 23.2 / 27.7
        //   384^2 4 waves 13.3 / 13.7 / 15.6 / 14.9, 8 17.1 / 15.8 / 17.4 / 17.0, 16 23.5 / 20.4 / 20.8 / 20.6
        //   512^2 8 waves 18.1 / 18.5 / 19.7 / 19.4, 16 32.7 / 29.0 / 29.2 / 28.6, 64 89.8 / 74.2 / 72.8 / 74.1
        //   768^2 one 16.4 / 18.6 / 36 / 17.5, 4 waves 25.1 / 23.5 / 43 / 22.4; 1024^2 8 waves 53.2 / 53.0 / 101 / 52.7
        const int k = band ? args.band_k : N / 2;
        const auto items = [&](int tc) { return (2 * (k / tc) + 2) * (long long)nsets; };
        const int cus = e->num_cus;
        if (2 * items(4) <= (P0::E <= 8 ? 6 : N == 384 ? 3 : 2) * cus)
            variant = 5;
        else if (N == 384)
            variant = items(16) <= cus ? 12 : 11;
        else if (N == 768)
            variant = 11;
        else if (N == 1024)
            variant = items(8) <= 2 * cus ? 11 : 12;
        else
            variant = items(16) < 3 * cus ? 12 : 7;
    }
    // the tiles of TC columns to visit: with a band, those that hold columns 0..K or N-K..N-1
    auto set_tiles = [&](int TC) {
        args.tile_lo = N / TC;
        args.tile_skip = 0;
        if (band || (mode == mse::COL_PROBE && args.band_k >= 0)) {
            const int hi = (N - args.band_k) / TC;
            args.tile_lo = args.band_k / TC + 1;
            args.tile_skip = std::max(0, hi - args.tile_lo);
        }
        args.n_tiles = N / TC - args.tile_skip;
        return args.n_tiles;
    };
    // one tile per block
    auto go = [&](auto plan, auto tc, auto sync, auto twreg) {
        using PL = decltype(plan);
        using SY = decltype(sync);
        constexpr bool TR = decltype(twreg)::value;
        constexpr int WPE = TR ? 1 : 8;
        constexpr int TC = decltype(tc)::value;
        constexpr int NT = TC * PL::L;
        dim3 grid(set_tiles(TC), nsets);
        launch(e, kind, [&]() {
#define MSE_COL_CASE(M, BAND)                                                                                         \
    if (mode == mse::M && band == BAND) {                                                                             \
        mse::k_col<PL, TC, mse::M, BAND, SY, TR, WPE><<<grid, NT, 0, e->stream>>>(in, out, wave_stride, e->tw.p, args); \
        return;                                                                                                       \
    }
            MSE_COL_CASE(COL_PROP, false)
            MSE_COL_CASE(COL_PROP, true)
            MSE_COL_CASE(COL_PROP_DETECT, false)
            MSE_COL_CASE(COL_PROP_DETECT, true)
            MSE_COL_CASE(COL_COPY, false)
            if constexpr (TR && std::is_same<SY, mse::WaveSync>::value && std::is_same<PL, P0>::value) {
                MSE_COL_CASE(COL_PROBE, false)
                MSE_COL_CASE(COL_FFT_DETECT, false)
                MSE_COL_CASE(COL_FFT_DIFF, false)
                MSE_COL_CASE(COL_PROP_CONJ, false)
                MSE_COL_CASE(COL_PROP_CONJ, true)
                MSE_COL_CASE(COL_CTEM_IMAGE, false)
                MSE_COL_CASE(COL_FILTER, false)
            }
#undef MSE_COL_CASE
            throw Error(MSE_ERR_STATE, "column pass without a kernel");
        });
    };
    if ((variant >= 7 || variant == 5) && mode == mse::COL_PROP && in == out) {
        // persistent blocks, at most `cap` per CU; the XCD-aware order takes a multiple of 8
        auto go_pipe = [&](auto plan, auto tc, auto twreg, auto xcd, auto bnd, int cap) {
            using PL = decltype(plan);
            constexpr bool TR = decltype(twreg)::value, XCD = decltype(xcd)::value, BAND = decltype(bnd)::value;
            constexpr int TC = decltype(tc)::value, NT = TC * PL::L;
            const int items = set_tiles(TC) * nsets;
            const int per_cu = resident_per_cu<mse::k_col_prop_pipe<PL, TC, BAND, mse::WaveSync, TR, 1, XCD>>(NT, cap / NT);
            int blocks = std::max(1, std::min(e->num_cus * per_cu, items));
            if (XCD) blocks = (blocks + 7) / 8 * 8;
            launch(e, kind, [&]() {
                mse::k_col_prop_pipe<PL, TC, BAND, mse::WaveSync, TR, 1, XCD><<<blocks, NT, 0, e->stream>>>(
                    out, wave_stride, e->tw.p, args, nsets);
            });
        };
        auto pipe = [&](auto plan, auto tc, auto twreg, auto xcd, int cap) {
            if (band)
                go_pipe(plan, tc, twreg, xcd, std::true_type{}, cap);
            else
                go_pipe(plan, tc, twreg, xcd, std::false_type{}, cap);
        };
        if constexpr (N <= 512) {  // half lanes: two blocks per CU
            if (variant == 8) {
                pipe(P1{}, C16{}, REG{}, std::false_type{}, 2048);
                return args.n_tiles;
            }
        }
        if (variant == 11 || variant == kLeanAlt) {  // lean: one tile per block, several blocks per CU
            constexpr int TC = N <= 512 ? 16 : 8;
            const int blocks = (set_tiles(TC) * nsets + 7) / 8 * 8;
            auto lean = [&](auto bnd, auto alt) {
                launch(e, kind, [&]() {
                    mse::k_col_prop_lean<P0, TC, decltype(bnd)::value, decltype(alt)::value>
                        <<<blocks, TC * P0::L, 0, e->stream>>>(out, wave_stride, e->tw.p, args, nsets);
                });
            };
            if constexpr (N == 768) {
                if (variant == kLeanAlt) {
                    if (band)
                        lean(std::true_type{}, std::true_type{});
                    else
                        lean(std::false_type{}, std::true_type{});
                    return args.n_tiles;
                }
            }
            if (band)
                lean(std::true_type{}, std::false_type{});
            else
                lean(std::false_type{}, std::false_type{});
            return args.n_tiles;
        }
        switch (variant) {
            case 5: pipe(P0{}, C4{}, REG{}, std::true_type{}, 2048); break;
            case 12: pipe(P0{}, C8{}, REG{}, std::true_type{}, 2048); break;
            case 13: pipe(P0{}, C16{}, REG{}, std::true_type{}, 2048); break;
            case 10: pipe(P0{}, C8{}, REG{}, std::false_type{}, 1024); break;  // no spills at 1024
            case 9: pipe(P0{}, C16{}, MEM{}, std::false_type{}, 1024); break;  // twiddles read at use
            default: pipe(P0{}, C16{}, REG{}, std::false_type{}, 1024); break;
        }
        return args.n_tiles;
    }
    // Rule: 8-column tiles where 16-column ones would leave CUs without a block (one wave at 512^2:
    // detectors 14.4 -> 7.0 us) and for the plans whose 1024-thread blocks spill.  Detector
    // partials are per tile: FP64 sums in another grouping.
    if (variant >= 7 || variant == 5 || variant < 0) variant = 0;
    const bool few = (N / 16) * nsets < e->num_cus, spills = P0::L == 64 && P0::E > 8;
    if (variant == 1)
        go(P1{}, C16{}, mse::WaveSync{}, REG{});
    else if (variant == 2)
        go(P0{}, C8{}, mse::WaveSync{}, REG{});
    else if (variant == 3)
        go(P0{}, C16{}, mse::BlockSync{}, REG{});
    else if (variant == 4)
        go(P0{}, C16{}, mse::WaveSync{}, MEM{});
    else if (variant == 6) {
        if constexpr (N <= 512)  // 32 columns exceed the 160 KiB LDS above 512 points
            go(P1{}, C32{}, mse::WaveSync{}, REG{});
        else
            go(P0{}, C16{}, mse::WaveSync{}, REG{});
    } else if (variant == 0 && mode != mse::COL_COPY && mode != mse::COL_PROP && (few || spills))
        go(P0{}, C8{}, mse::WaveSync{}, REG{});
    else
        go(P0{}, C16{}, mse::WaveSync{}, REG{});
    return args.n_tiles;
}

}  // namespace mse_rt

#define MSE_INSTANTIATE_SWEEPS(NN)                                                                          \
    template void mse_rt::row_pass_n<NN>(mse_engine*, int, const float2*, float2*, int, size_t,             \
                                         const mse::RowArgs&, int);                                        \
    template int mse_rt::col_pass_n<NN>(mse_engine*, int, const float2*, float2*, int, size_t,              \
                                        const mse::ColArgs&, int, int);
