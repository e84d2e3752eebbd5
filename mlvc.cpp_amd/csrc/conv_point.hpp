// 1x1 convs over flattened pixels on gfx950 MFMA.
//
//   D[p, oc] = bias[oc] + sum_k X[k, p] W[oc, k],  k = 16-channel step
//
// Same product order and rounding as conv_mfma_kernel (conv_kernel.hpp), so
// it gives the same bits. A 1x1 conv does 2 * oc / 2 bytes of arithmetic per
// input element at most, so over many pixels it is bound by HBM and over few
// by the latency of its loads; both want every byte of a tile in flight at
// once and as few instructions around it as possible:
//   * the tile of BN pixels x SC channels goes from HBM to LDS by LDS DMA, 16
//     bytes a lane, with no registers, no conversions and no LDS writes. LDS
//     holds it as it lies in memory, [channel][pixel];
//   * the MFMA fragment of a pixel wants 8 consecutive channels: the
//     transposing LDS read (ds_read_b64_tr_b16) delivers 4 of them per 8
//     bytes. 32 lanes read 64 bytes of 4 channel rows each; the rows' 64-byte
//     chunks are XOR-swizzled by row as they are loaded (at()), so the four
//     fall on different banks;
//   * weights (packed in fragment order, [ocb][c16][m-tile][lane][8]) go
//     straight to registers, a pass of SC channels at a time;
//   * the pixels are the MFMA's rows, so a lane ends up with 4 consecutive
//     pixels of one channel: the results go through LDS as 8-byte writes, 64
//     pixels of 32 channels at a time per wave, and leave as 16-byte pieces of
//     128-byte rows;
//   * with two buffers (NBUF) the next pass's X and W are requested before the
//     current pass is multiplied, one barrier a pass.
// 64->192 at 544x960 (267 MB): 85 us by conv_mfma_kernel, 66-69 here (4.0
// TB/s); 512->256 at 63x64: 17 and 5.6 us.
// Rows of any even number of pixels: LDS DMA needs 4-byte alignment only.
// Pixels past the image are other channels' pixels or zeros (range check);
// they are columns of D that are not stored.

#pragma once

#include "conv_kernel.hpp"

namespace mlvc_hip {
namespace conv {

// WM waves along the output channels (MT m-tiles of 32 each) x WN along the
// pixels (NT tiles of 32 each).
template <int WM_, int WN_, int MT_, int NT_, int SC_, int NBUF_, int OCC_>
struct PtCfg {
    static constexpr int WM = WM_, WN = WN_, MT = MT_, NT = NT_, SC = SC_, NBUF = NBUF_, OCC = OCC_;
    static constexpr int WAVES = WM * WN, kThreads = 64 * WAVES;
    static constexpr int BM = 32 * WM * MT, BN = 32 * WN * NT;
    static constexpr int KS = SC / 16;             // MFMA steps per pass
    static constexpr int PPR = BN / 8;             // 16-byte pieces per staged channel row
    static constexpr int X = SC * BN;              // halves per buffer
    static constexpr int DMA = X * 2 / 1024;       // 1 KB DMA instructions per pass
    static constexpr int DMA_W = (DMA + WAVES - 1) / WAVES;
    static constexpr int EPX = 32 * NT < 64 ? 32 * NT : 64;  // pixels per epilogue step
    static constexpr int EROW = EPX + 4;           // halves; 8-byte writes of 32 rows hit distinct banks
    static constexpr int E = WAVES * 32 * EROW;
    static constexpr int LDS0 = X > E ? X : E, LDS1 = NBUF > 1 ? X : 8;
    static_assert(SC % 16 == 0 && PPR <= 16 && 64 / PPR <= 16 && X * 2 % 1024 == 0, "whole DMA instructions within a 16-channel step");
    static_assert((LDS0 + LDS1) * 2 <= 160 * 1024, "LDS budget");
    // 64-byte chunks (32 pixels) per row and their swizzle.
    __device__ static constexpr int swz(int row) { return BN >= 128 ? row & 3 : BN == 64 ? (row >> 1) & 1 : 0; }
    // LDS offset (halves) of pixel p of staged channel row.
    __device__ static constexpr int at(int row, int p) { return row * BN + (((p >> 5) ^ swz(row)) << 5) + (p & 31); }
};

// MODE as epi_mode (0 none, 1 LeakyReLU in the max form), 2: any epilogue.
template <class C, bool CONCAT, int MODE>
__global__ __launch_bounds__(C::kThreads) __attribute__((amdgpu_waves_per_eu(C::OCC))) void conv_point_kernel(ConvArgs a)
{
    // The host pass only needs the stub, and does not know gfx950's LDS builtins.
#if defined(__HIP_DEVICE_COMPILE__)
    // Two arrays, so that the compiler sees which reads a DMA in flight can
    // touch (it waits for every DMA into the array it reads).
    __shared__ __attribute__((aligned(1024))) std::uint16_t lds0[C::LDS0];
    __shared__ __attribute__((aligned(1024))) std::uint16_t lds1[C::LDS1];
    typedef short s16x4 __attribute__((ext_vector_type(4)));
    typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

    // The wave number is uniform; saying so keeps the DMA's resources and LDS
    // addresses in scalar registers.
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave / C::WN, wn = wave % C::WN;
    const int item = xcd_order(blockIdx.x, a.nwg);
    // (Integer divisions run on the vector ALU: say that they are uniform too.)
    const int t = __builtin_amdgcn_readfirstlane(item / a.ocbs), b = __builtin_amdgcn_readfirstlane(t / a.tiles);
    const int ocb = item - t * a.ocbs, tile = t - b * a.tiles;
    const int px0 = tile * C::BN;
    const int hw = a.iw;  // flattened: one row
    const std::uint32_t hw2 = static_cast<std::uint32_t>(hw) * 2u;
    // CONCAT: channels from c1 on are x2's. The resource is picked by its
    // address and size (scalar selects), then built.
    const int c1 = CONCAT ? a.ic_split : a.ic;
    const std::uint64_t xp = reinterpret_cast<std::uint64_t>(a.x + static_cast<size_t>(b) * c1 * hw);
    const std::uint64_t xp2 = CONCAT ? reinterpret_cast<std::uint64_t>(a.x2 + static_cast<size_t>(b) * (a.ic - c1) * hw) : xp;
    auto resource = [&](bool second) {
        const std::uint64_t p = second ? xp2 : xp;
        const std::uint32_t lo = __builtin_amdgcn_readfirstlane(static_cast<std::uint32_t>(p)),
                            hi = __builtin_amdgcn_readfirstlane(static_cast<std::uint32_t>(p >> 32));
        return __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void*>(static_cast<std::uint64_t>(hi) << 32 | lo), 0,
                                                 __builtin_amdgcn_readfirstlane(static_cast<int>((second ? a.ic - c1 : c1) * hw2)),
                                                 kRawBufferFlags);
    };

    // Piece of this lane in a DMA instruction: channel row lane / PPR of the
    // instruction's rows, 8 pixels. Instructions start at rows whose swizzle
    // is that of row 0, so the lane's part of the offset is the same in all.
    const int drow = lane / C::PPR, dpx = (((((lane % C::PPR) >> 2) ^ C::swz(drow)) << 2) | (lane & 3)) * 8;
    const std::uint32_t doff = static_cast<std::uint32_t>(drow) * hw2 + static_cast<std::uint32_t>(px0 + dpx) * 2u;
    auto dma = [&](int cb, std::uint16_t* lds) {
#pragma unroll
        for (int i = 0; i < C::DMA_W; ++i) {
            const int j = wave + i * C::WAVES;
            if (C::DMA % C::WAVES != 0 && j >= C::DMA) continue;
            const int c0 = cb + j * (64 / C::PPR);
            const bool second = CONCAT && c0 >= c1;
            // The whole offset goes in the VGPR operand, which the range
            // check covers: pixels past the last channel's end read zeros.
            __builtin_amdgcn_raw_ptr_buffer_load_lds(resource(second),
                                                     (__attribute__((address_space(3))) void*)(lds + j * 512), 16,
                                                     static_cast<int>(doff + static_cast<std::uint32_t>(second ? c0 - c1 : c0) * hw2), 0, 0, 0);
        }
    };
    // Fragment (16-channel step s, m-tile): lane offset in the VGPR, the rest scalar.
    const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<std::uint16_t*>(a.w), 0, a.ocbs * a.nchunks * C::WM * C::MT * 1024, kRawBufferFlags);
    const int wfrag = (ocb * a.nchunks * C::WM + wm) * C::MT;
    u32x4 wreg[C::NBUF][C::KS][C::MT];
    auto weights = [&](int cb, int buf) {
#pragma unroll
        for (int ks = 0; ks < C::KS; ++ks)
#pragma unroll
            for (int mt = 0; mt < C::MT; ++mt)
                wreg[buf][ks][mt] = __builtin_amdgcn_raw_buffer_load_b128(
                    rw, lane * 16, (wfrag + (cb / 16 + ks) * C::WM * C::MT + mt) * 1024, 0);
    };

    dma(0, lds0);
    weights(0, 0);
    floatx16 acc[C::MT][C::NT];
#pragma unroll
    for (int mt = 0; mt < C::MT; ++mt) {
        const float bv = a.bias[ocb * C::BM + (wm * C::MT + mt) * 32 + (lane & 31)];
#pragma unroll
        for (int nt = 0; nt < C::NT; ++nt)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[mt][nt][r] = bv;
    }
    // Transposing reads of step ks, pixel tile n: lanes 0-31 channels 0-7 and
    // lanes 32-63 channels 8-15 of the step, 16 lanes per 16 pixels, 4
    // channels per read.
    const int trow = 8 * (lane >> 5) + ((lane & 15) >> 2), tcol = 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
    int taddr[C::NT];  // of step 0; a row's swizzle repeats every 4 rows
#pragma unroll
    for (int nt = 0; nt < C::NT; ++nt) taddr[nt] = C::at(trow, (wn * C::NT + nt) * 32 + tcol);
    auto pixels = [&](const std::uint16_t* lds, int ks, int nt) -> half8 {
        auto read = [&](int row) {
            return __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                                                 (__attribute__((address_space(3))) s16x4*)(lds + taddr[nt] + row * C::BN)));
        };
        const u32x2 lo = read(ks * 16), hi = read(ks * 16 + 4);
        return __builtin_bit_cast(half8, u32x4{lo[0], lo[1], hi[0], hi[1]});
    };
    auto compute = [&](const std::uint16_t* lds, const u32x4 (&w)[C::KS][C::MT]) {
        // The next pass's loads stay in front of the products, and the reads
        // one step ahead of them.
        __builtin_amdgcn_sched_barrier(0);
        half8 xv[2][C::NT];
#pragma unroll
        for (int nt = 0; nt < C::NT; ++nt) xv[0][nt] = pixels(lds, 0, nt);
#pragma unroll
        for (int ks = 0; ks < C::KS; ++ks) {
            if (ks + 1 < C::KS) {
#pragma unroll
                for (int nt = 0; nt < C::NT; ++nt) xv[(ks + 1) & 1][nt] = pixels(lds, ks + 1, nt);
            }
#pragma unroll
            for (int mt = 0; mt < C::MT; ++mt)
#pragma unroll
                for (int nt = 0; nt < C::NT; ++nt)
                    acc[mt][nt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xv[ks & 1][nt], __builtin_bit_cast(half8, w[ks][mt]),
                                                                         acc[mt][nt], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    auto landed = [&] {
        __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): this wave's DMA and weights
        __syncthreads();
    };
    landed();
    // One exit and one copy of each product loop: with a peeled last pass the
    // compiler keeps the accumulators twice and spills.
    if constexpr (C::NBUF == 1) {
        for (int cb = 0;;) {
            compute(lds0, wreg[0]);
            __syncthreads();  // every wave is done with the buffer
            if ((cb += C::SC) >= a.ic) break;
            dma(cb, lds0);
            weights(cb, 0);
            landed();
        }
    } else {
        for (int cb = C::SC;; cb += 2 * C::SC) {
            dma(cb, lds1);
            weights(cb, 1);
            compute(lds0, wreg[0]);
            landed();
            const bool more = cb + C::SC < a.ic;
            if (more) {
                dma(cb + C::SC, lds0);
                weights(cb + C::SC, 0);
            }
            compute(lds1, wreg[1]);
            landed();
            if (!more) break;
        }
    }

    // Epilogue, wave by wave: lane l holds channel l % 32, pixels 8j + 4 (l / 32) .. + 3 of a tile.
    const bool max_form = leaky_max_form(a.alpha);
    std::uint16_t* const es = lds0 + wave * 32 * C::EROW;
    constexpr int G = C::EPX / 8, STEPS = 32 * C::NT / C::EPX;
#pragma unroll
    for (int mt = 0; mt < C::MT; ++mt)
#pragma unroll
        for (int st = 0; st < STEPS; ++st) {
#pragma unroll
            for (int n = 0; n < C::EPX / 32; ++n)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const floatx16& v = acc[mt][st * (C::EPX / 32) + n];
                    *reinterpret_cast<u32x2*>(&es[(lane & 31) * C::EROW + n * 32 + 8 * j + 4 * (lane >> 5)]) =
                        u32x2{pack_f16(v[4 * j], v[4 * j + 1]), pack_f16(v[4 * j + 2], v[4 * j + 3])};
                }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
#pragma unroll MODE == 2 ? 1 : 32 * G / 64
            for (int i = 0; i < 32 * G / 64; ++i) {
                const int u = lane + 64 * i, ocl = u / G, g = u % G;
                const int oc = ocb * C::BM + (wm * C::MT + mt) * 32 + ocl;
                const int px = px0 + wn * C::NT * 32 + st * C::EPX + g * 8;
                const u32x2 lo = *reinterpret_cast<const u32x2*>(&es[ocl * C::EROW + g * 8]);
                const u32x2 hi = *reinterpret_cast<const u32x2*>(&es[ocl * C::EROW + g * 8 + 4]);
                u32x4 h{lo[0], lo[1], hi[0], hi[1]};
                if (oc >= a.oc || px >= hw) continue;
                const size_t o = (static_cast<size_t>(b) * a.oc + oc) * hw + px;
                if constexpr (MODE == 2) {
                    if (px + 8 <= hw) store_row8<u32x4_any>(a, h, o, max_form);
                    else store_row_part(a, h, o, hw - px);
                } else {
                    if constexpr (MODE == 1) {
#pragma unroll
                        for (int k = 0; k < 4; ++k) h[k] = leaky_h2(h[k], a.alpha, true);
                    }
                    if (px + 8 <= hw) {
                        *reinterpret_cast<u32x4_any*>(a.y + o) = h;
                    } else {  // a row's last, partial group
                        for (int k = 0; k < hw - px; ++k)
                            a.y[o + k] = static_cast<std::uint16_t>((k < 4 ? (k < 2 ? h[0] : h[1]) : (k < 6 ? h[2] : h[3])) >> (16 * (k & 1)));
                    }
                }
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
        }
#endif
}

template <class C, bool CONCAT>
void launch_point_mode(const ConvArgs& a, dim3 grid, hipStream_t s)
{
    if (a.epi == MLVC_EPI_NONE)
        hipLaunchKernelGGL((conv_point_kernel<C, CONCAT, 0>), grid, dim3(C::kThreads), 0, s, a);
    else if (a.epi == MLVC_EPI_LEAKY_RELU && epi_mode(1, a.alpha) == 1)
        hipLaunchKernelGGL((conv_point_kernel<C, CONCAT, 1>), grid, dim3(C::kThreads), 0, s, a);
    else
        hipLaunchKernelGGL((conv_point_kernel<C, CONCAT, 2>), grid, dim3(C::kThreads), 0, s, a);
}

template <class C>
void launch_point(const ConvArgs& a, dim3 grid, hipStream_t s)
{
    if (a.x2) launch_point_mode<C, true>(a, grid, s);
    else launch_point_mode<C, false>(a, grid, s);
}

// Split K in one workgroup: wave s sums the input channels [s * split_c, (s +
// 1) * split_c) of a BM x BN tile (split 0 seeded with the bias), the FP32
// partials meet in LDS, and the waves add them in split order, round and apply
// the epilogue: the sums of conv_mfma_kernel's split and
// conv_splitk_reduce_kernel, bit for bit, without the partials' trip through
// memory and the second launch. Splits are whole 64-channel halves: both are
// multiplied whole, so the host sends other splits (set by hand; the plan's
// are multiples of 64) to the two kernels. Few pixels and many channels are bound by
// latency, so each wave has 128 channels of X (DMA into LDS of its own, no
// barrier) and W in flight at once; with the usual split_c of 128 that is its
// whole share. 1024->256 at 23x40, 8 splits: 16.7 us in two kernels, 5.8 here.
template <int MT_, int NT_>
struct PtSplitCfg {
    static constexpr int MT = MT_, NT = NT_, BM = 32 * MT, BN = 32 * NT, MAX_SPLIT = 8;
    using Half = PtCfg<1, 1, MT, NT, 64, 1, 2>;    // 64 channels of the tile
    static constexpr int PART = MT * NT * 1024;    // floats per split
    static constexpr int HALF = Half::X;           // halves of X per wave and half
    static_assert(PART * 2 <= 2 * HALF || MT <= 2, "partials");
    // One wave's X (two halves), later its partials.
    static constexpr int WAVE = 2 * HALF > PART * 2 ? 2 * HALF : PART * 2;
};

template <class C>
__global__ __launch_bounds__(64 * C::MAX_SPLIT) __attribute__((amdgpu_waves_per_eu(2))) void conv_point_split_kernel(ConvArgs a)
{
#if defined(__HIP_DEVICE_COMPILE__)
    using H = typename C::Half;
    extern __shared__ __attribute__((aligned(1024))) std::uint16_t lds_all[];
    typedef short s16x4 __attribute__((ext_vector_type(4)));
    typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

    const int lane = threadIdx.x & 63, split = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int item = xcd_order(blockIdx.x, a.nwg);
    const int t = __builtin_amdgcn_readfirstlane(item / a.ocbs), b = __builtin_amdgcn_readfirstlane(t / a.tiles);
    const int ocb = item - t * a.ocbs, px0 = (t - b * a.tiles) * C::BN;
    const int hw = a.iw;
    const std::uint32_t hw2 = static_cast<std::uint32_t>(hw) * 2u;
    const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<std::uint16_t*>(a.x + static_cast<size_t>(b) * a.ic * hw), 0, static_cast<int>(a.ic * hw2), kRawBufferFlags);
    const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<std::uint16_t*>(a.w), 0, a.ocbs * a.nchunks * C::MT * 1024, kRawBufferFlags);
    std::uint16_t* const lds = lds_all + split * C::WAVE;
    const int drow = lane / H::PPR, dpx = (((((lane % H::PPR) >> 2) ^ H::swz(drow)) << 2) | (lane & 3)) * 8;
    const std::uint32_t doff = static_cast<std::uint32_t>(drow) * hw2 + static_cast<std::uint32_t>(px0 + dpx) * 2u;

    floatx16 acc[C::MT][C::NT];
#pragma unroll
    for (int mt = 0; mt < C::MT; ++mt) {
        const float bv = split == 0 ? a.bias[ocb * C::BM + mt * 32 + (lane & 31)] : 0.0f;
#pragma unroll
        for (int nt = 0; nt < C::NT; ++nt)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[mt][nt][r] = bv;
    }
    const int trow = 8 * (lane >> 5) + ((lane & 15) >> 2), tcol = 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
    int taddr[C::NT];
#pragma unroll
    for (int nt = 0; nt < C::NT; ++nt) taddr[nt] = H::at(trow, nt * 32 + tcol);

    u32x4 wreg[2][4][C::MT];
    auto fetch = [&](int c0, int half) {  // 64 channels
#pragma unroll
        for (int j = 0; j < H::DMA; ++j)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (__attribute__((address_space(3))) void*)(lds + half * C::HALF + j * 512), 16,
                                                     static_cast<int>(doff + static_cast<std::uint32_t>(c0 + j * (64 / H::PPR)) * hw2),
                                                     0, 0, 0);
#pragma unroll
        for (int ks = 0; ks < 4; ++ks)
#pragma unroll
            for (int mt = 0; mt < C::MT; ++mt)
                wreg[half][ks][mt] = __builtin_amdgcn_raw_buffer_load_b128(
                    rw, lane * 16, ((ocb * a.nchunks + c0 / 16 + ks) * C::MT + mt) * 1024, 0);
    };
    auto compute = [&](int half) {
#pragma unroll
        for (int ks = 0; ks < 4; ++ks)
#pragma unroll
            for (int nt = 0; nt < C::NT; ++nt) {
                u32x2 v[2];
#pragma unroll
                for (int e = 0; e < 2; ++e)
                    v[e] = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                                                         (__attribute__((address_space(3))) s16x4*)(lds + half * C::HALF + taddr[nt] +
                                                                                                    (ks * 16 + 4 * e) * C::BN)));
                const half8 xv = __builtin_bit_cast(half8, u32x4{v[0][0], v[0][1], v[1][0], v[1][1]});
#pragma unroll
                for (int mt = 0; mt < C::MT; ++mt)
                    acc[mt][nt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xv, __builtin_bit_cast(half8, wreg[half][ks][mt]),
                                                                         acc[mt][nt], 0, 0, 0);
            }
    };
    const int cend = min(a.ic, (split + 1) * a.split_c);
    for (int c = split * a.split_c; c < cend; c += 128) {
        fetch(c, 0);
        const bool second = c + 64 < cend;
        if (second) fetch(c + 64, 1);
        __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): this wave's own DMA; no other wave reads it
        __builtin_amdgcn_sched_barrier(0);
        compute(0);
        if (second) compute(1);
        __builtin_amdgcn_sched_barrier(0);
    }

    // Partials of (m-tile, pixel tile) u, registers 4j .. 4j + 3: 16 bytes a
    // lane, after this wave's last read of its X.
    float* const part = reinterpret_cast<float*>(lds_all);
#pragma unroll
    for (int mt = 0; mt < C::MT; ++mt)
#pragma unroll
        for (int nt = 0; nt < C::NT; ++nt)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const floatx16& v = acc[mt][nt];
                *reinterpret_cast<floatx4*>(&part[split * (C::WAVE / 2) + (((mt * C::NT + nt) * 4 + j) * 64 + lane) * 4]) =
                    floatx4{v[4 * j], v[4 * j + 1], v[4 * j + 2], v[4 * j + 3]};
            }
    __syncthreads();
    for (int u = split; u < C::MT * C::NT * 4; u += a.ksplit) {
        const int mt = u / (4 * C::NT), nt = (u / 4) % C::NT, j = u % 4;
        floatx4 v = *reinterpret_cast<const floatx4*>(&part[(u * 64 + lane) * 4]);
        for (int sp = 1; sp < a.ksplit; ++sp) {
            const floatx4 q = *reinterpret_cast<const floatx4*>(&part[sp * (C::WAVE / 2) + (u * 64 + lane) * 4]);
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] = v[i] + q[i];
        }
        const int oc = ocb * C::BM + mt * 32 + (lane & 31), px = px0 + nt * 32 + 8 * j + 4 * (lane >> 5);
        if (oc >= a.oc || px >= hw) continue;
        std::uint16_t h[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) h[i] = px + i < hw ? finish(a, v[i], b, oc, 0, px + i) : 0;
        const size_t o = (static_cast<size_t>(b) * a.oc + oc) * hw + px;
        if (px + 4 <= hw) {
            typedef u32x2 u32x2_any __attribute__((aligned(2)));
            *reinterpret_cast<u32x2_any*>(a.y + o) = u32x2{static_cast<std::uint32_t>(h[0]) | static_cast<std::uint32_t>(h[1]) << 16,
                                                           static_cast<std::uint32_t>(h[2]) | static_cast<std::uint32_t>(h[3]) << 16};
        } else {
            for (int i = 0; i < 4; ++i)
                if (px + i < hw) a.y[o + i] = h[i];
        }
    }
#endif
}

template <class C>
void launch_point_split(const ConvArgs& a, dim3, hipStream_t s)
{
    hipLaunchKernelGGL(conv_point_split_kernel<C>, dim3(static_cast<unsigned>(a.nwg)), dim3(64u * a.ksplit),
                       static_cast<unsigned>(a.ksplit * C::WAVE * 2), s, a);
}

// Variant entry: weights packed with kc = 16. Operands off 16 bytes and
// splits off 64 channels run the split of conv_mfma_kernel on the same tile
// and the reduce kernel.
template <class C>
constexpr Variant point_split_variant(const char* name)
{
    Variant v{name, C::BM, 1, C::BN, 1, 1, 1, 16, &launch_mfma<Cfg<C::BM, 1, C::BN, 1, 1, 1, 16, 0, false, 1, 1, 1>>,
              &launch_point_split<C>, nullptr};
    v.point_ic = 64;
    v.point_split = true;
    return v;
}
#define MLVC_VARIANT_PTK(MT, NT) point_split_variant<PtSplitCfg<MT, NT>>("mfma_ptk_t" #MT "x" #NT)

// Variant entry: weights packed with kc = 16. Operands off 16 bytes run the
// per-pixel staging of conv_mfma_kernel on the same tile and packed weights, at
// two waves per SIMD: with the registers of one (96->192 at 492x656 468 us, 64->96
// at 189x456 49) few loads are in flight on a full chip; 286 and 28 so.
template <class C>
constexpr Variant point_variant(const char* name)
{
    Variant v{name, C::BM, 1, C::BN, 1, 1, 1, 16, &launch_mfma<Cfg<C::BM, 1, C::BN, 1, 1, 1, 16, 0, false, C::WM, C::WN, 2>>,
              &launch_point<C>, nullptr};
    v.point_ic = C::SC * C::NBUF;
    return v;
}
#define MLVC_VARIANT_PT(WM, WN, MT, NT, SC, NBUF, OCC)                                                             \
    point_variant<PtCfg<WM, WN, MT, NT, SC, NBUF, OCC>>("mfma_pt_w" #WM "x" #WN "_t" #MT "x" #NT "_sc" #SC "_b" #NBUF \
                                                        "_occ" #OCC)

}  // namespace conv
}  // namespace mlvc_hip
