// bgs_kernels.hip -- gfx950 kernels of the SuBSENSE / LOBSTER frame step.
//
// The reference apply() is a raster-order loop (BackgroundSubtractorSuBSENSE.cpp:333-481,
// BackgroundSubtractorLOBSTER.cpp:459-576) in which a background pixel may write a sample of
// a neighbour; a neighbour later in raster order sees that sample in the same frame. The frame
// step below reproduces that order exactly without a sequential sweep:
//   describe : per pixel, everything that does not depend on other pixels' decisions
//              (LBSP, thresholds, RNG draws, diffusion target/slot/gates)       -> rec, desc_cur
//   match    : speculative ordered scan of the first samples (phase A); samples diffused in by
//              raster-earlier neighbours are applied under a guess of their decision (previous raw
//              mask)
//   match_seq: the scans that phase A cut (phase B), one lane per pixel or, for short lists, 16
//   fixpoint : pixels whose writers' decisions differ from the guess are re-matched, and the
//              change propagates through worklists until nothing changes. The writer graph is
//              acyclic (raster order), so the fix point is unique and equals the sequential result.
//   update   : FP32 maps (D_last, D_min, raw segm, T, v, R), raw mask, blink bookkeeping; each pixel
//              gathers, in raster order, the writes aimed at its samples from the 5x5 window
//              (self-update included); the last writer of a slot wins. No atomics. The launch also
//              holds the 3x3 closing with the zones' border components and the down-sampled cells.
//   post     : hole fill (union-find over the zones), erode 7x7, binary median k x k, dilate 7x7,
//              blink masks, final-segmentation averages, pending model reset
//   control  : LBSP LUT adaptation, model reset, caps (beside the zones' holes)
#include <hip/hip_runtime.h>

#include <cmath>

#include <algorithm>
#include <cstddef>
#include <type_traits>

#include "bgs_kernels.hpp"

namespace lvbgs {

constexpr int TW = 64, TH = 4, TPB = 256;  // per-pixel kernels: 64x4 tile, one pixel per thread

// Blocks are dispatched round-robin over the 8 XCDs; remap so each XCD gets a contiguous
// range of tiles (neighbouring tiles share halo lines in that XCD's L2).
LV_D int xcd_tile(int bid, int nblocks) {
    constexpr int X = 8;
    if (nblocks < X) return bid;
    const int xcd = bid % X, idx = bid / X, per = nblocks / X, rem = nblocks % X;
    return xcd * per + (xcd < rem ? xcd : rem) + idx;
}

LV_D uint32_t popc(uint32_t v) { return (uint32_t)__builtin_popcount(v); }
LV_D uint32_t absdiff(uint32_t a, uint32_t b) { return __builtin_amdgcn_sad_u8(a, b, 0u); }  // of bytes
LV_D float fmin_ref(float a, float b) { return (b < a) ? b : a; }  // std::min
LV_D float fmax_ref(float a, float b) { return (a < b) ? b : a; }  // std::max

// Sum of one value per lane over the wavefront, in lane 63 (DPP row shifts and broadcasts: six adds, no LDS).
LV_D uint32_t wave_sum_last(uint32_t x) {
    auto step = [&](auto ctrl, auto rows) {
        x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, decltype(ctrl)::value, decltype(rows)::value, 0xf, false);
    };
    using std::integral_constant;
    step(integral_constant<int, 0x111>{}, integral_constant<int, 0xf>{});  // row_shr:1
    step(integral_constant<int, 0x112>{}, integral_constant<int, 0xf>{});  // row_shr:2
    step(integral_constant<int, 0x114>{}, integral_constant<int, 0xf>{});  // row_shr:4
    step(integral_constant<int, 0x118>{}, integral_constant<int, 0xf>{});  // row_shr:8
    step(integral_constant<int, 0x142>{}, integral_constant<int, 0xa>{});  // row_bcast:15
    step(integral_constant<int, 0x143>{}, integral_constant<int, 0xc>{});  // row_bcast:31
    return x;
}

// Workgroup sums of K 32-bit values per thread (each below 2^24), added to stripe blockIdx % kStripes of K
// counter arrays. Every thread of the workgroup must call it, once per kernel.
template <int NT, int K>
LV_D void block_add(const uint32_t (&value)[K], unsigned long long* const (&stripes)[K]) {
    __shared__ uint32_t part[NT / 64][K];
    const int lane = (int)(threadIdx.x & 63u), wave = (int)(threadIdx.x >> 6);
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const uint32_t t = wave_sum_last(value[k]);
        if (lane == 63) part[wave][k] = t;
    }
    __syncthreads();
    if (threadIdx.x < (uint32_t)K) {
        uint32_t t = 0;
#pragma unroll
        for (int i = 0; i < NT / 64; ++i) t += part[i][threadIdx.x];
        unsigned long long* s = stripes[0];
#pragma unroll
        for (int k = 1; k < K; ++k) s = threadIdx.x == (uint32_t)k ? stripes[k] : s;
        if (t) atomicAdd(&s[blockIdx.x % kStripes], (unsigned long long)t);
    }
}
template <int NT>
LV_D void block_add(uint32_t value, unsigned long long* stripes) {
    const uint32_t v1[1] = {value};
    unsigned long long* const s1[1] = {stripes};
    block_add<NT, 1>(v1, s1);
}

LV_HD unsigned long long sum_stripes(const unsigned long long* s) {
    unsigned long long t = 0;
    for (int i = 0; i < kStripes; ++i) t += s[i];
    return t;
}

// frame number of the step in flight (m_nFrameIdx after its increment at the top of apply)
LV_D uint32_t cur_frame(const View& v) { return v.sc->frame_idx + 1u; }

// ----------------------------------------------------------------------------------------------
// sample planes
// ----------------------------------------------------------------------------------------------
// one sample record: 12 bytes (RGB) or 4 bytes (grey), a single load or store per sample
struct alignas(4) Rec12 {
    uint32_t w0, w1, w2;
};

// Tile-major sample layout: the N samples of each group of 64 consecutive pixels are contiguous
// (group g, sample s, lane p % 64), so a wavefront's ordered scan walks one compact region instead
// of N planes a frame apart.
LV_D size_t sample_index(const View& v, uint32_t s, uint32_t p) {
    return ((size_t)(p >> 6) * (uint32_t)v.N + s) * 64u + (p & 63u);
}

// A device pointer seen through the global address space. The pointers of a batch member's View are
// read from a table in device memory, so the compiler sees them as generic (flat) pointers; loads
// through address space 1 are global loads instead (an SGPR base with a 32-bit lane offset, and
// LDS waits that do not also wait for them).
template <typename T>
using gptr = __attribute__((address_space(1))) T*;
template <typename T>
LV_D gptr<T> G(T* p) {
    return (gptr<T>)p;
}

// element i of a per-pixel array, through a 32-bit byte offset: every per-pixel array is below 4 GiB (at most 2^28
// pixels of 6 bytes), so a load takes its base from scalar registers and its offset from one vector
// register, where a 64-bit index costs two or three vector adds per access
template <typename T, typename I>
LV_D gptr<T> at(T* base, I i) {
    return (gptr<T>)((gptr<const uint8_t>)base + (uint32_t)((uint32_t)i * (uint32_t)sizeof(T)));
}

// Stores element i unless every lane of the wavefront that is here holds the value already stored (old). Most of
// the state of a settled background pixel does not change from frame to frame (raw averages at 0, v at its
// floor, T at a cap, no blinks), and a row of 64 unchanged values need not be written; whole rows keep
// the store's lines whole.
template <typename T, typename I>
LV_D void store_changed(T* base, I i, T value, T old) {
    bool same;
    if constexpr (sizeof(T) == 4) same = __builtin_bit_cast(uint32_t, value) == __builtin_bit_cast(uint32_t, old);
    else same = value == old;
    if (__ballot(!same) != 0ull) *at(base, i) = value;
}

// wavefront-local LDS exchange: the lanes' stores above are visible to the loads below
LV_D void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// raw sample in registers: ra = record words 0-1 (RGB) or word 0 (grey), rb = word 2 (RGB)
template <int C>
LV_D void fetch_raw(const View& v, uint32_t s, uint32_t p, uint64_t& ra, uint32_t& rb) {
    const size_t idx = sample_index(v, s, p);
    if constexpr (C == 3) {
        const gptr<const uint32_t> q = G((const uint32_t*)v.sA) + idx * 3u;
        ra = (uint64_t)q[0] | ((uint64_t)q[1] << 32);
        rb = q[2];
    } else {
        ra = G((const uint32_t*)v.sA)[idx];
        rb = 0;
    }
}

// records of one pixel: sample s at rec_base(v, p) + s * 64 (tile-major layout)
LV_D const uint32_t* rec_base(const View& v, uint32_t p) {
    return (const uint32_t*)v.sA + sample_index(v, 0u, p) * (v.C == 3 ? 3u : 1u);
}

template <int C>
LV_D void fetch_at(const uint32_t* rec, uint64_t& ra, uint32_t& rb) {
    const gptr<const uint32_t> q = G(rec);
    if constexpr (C == 3) {
        ra = (uint64_t)q[0] | ((uint64_t)q[1] << 32);
        rb = q[2];
    } else {
        ra = q[0];
        rb = 0;
    }
}

template <int C>
LV_D void decode_raw(uint64_t ra, uint32_t rb, uint32_t col[C], uint32_t desc[C]) {
    if constexpr (C == 3) {
        desc[0] = (uint32_t)(ra & 0xFFFFu);
        desc[1] = (uint32_t)((ra >> 16) & 0xFFFFu);
        desc[2] = (uint32_t)((ra >> 32) & 0xFFFFu);
        col[0] = (uint32_t)((ra >> 48) & 0xFFu);
        col[1] = (uint32_t)(ra >> 56);
        col[2] = rb & 0xFFu;
    } else {
        desc[0] = (uint32_t)(ra & 0xFFFFu);
        col[0] = (uint32_t)((ra >> 16) & 0xFFu);
    }
}

template <int C>
LV_D void encode_raw(const uint32_t col[C], const uint32_t desc[C], uint64_t& ra, uint32_t& rb) {
    if constexpr (C == 3) {
        ra = (uint64_t)desc[0] | ((uint64_t)desc[1] << 16) | ((uint64_t)desc[2] << 32) | ((uint64_t)col[0] << 48) |
             ((uint64_t)col[1] << 56);
        rb = col[2];
    } else {
        ra = (uint64_t)desc[0] | ((uint64_t)col[0] << 16);
        rb = 0;
    }
}

template <int C>
LV_D void store_raw(const View& v, uint32_t s, uint32_t p, uint64_t ra, uint32_t rb) {
    const size_t idx = sample_index(v, s, p);
    // non-temporal: scattered single-record writes gain nothing from being kept in L2
    typedef uint32_t u32x3 __attribute__((ext_vector_type(3)));
    if constexpr (C == 3) {
        u32x3 w;
        w.x = (uint32_t)ra;
        w.y = (uint32_t)(ra >> 32);
        w.z = rb;
        __builtin_nontemporal_store(w, (gptr<u32x3>)((Rec12*)v.sA + idx));
    } else {
        __builtin_nontemporal_store((uint32_t)ra, G((uint32_t*)v.sA + idx));
    }
}

template <int C>
LV_D void store_sample(const View& v, uint32_t s, uint32_t p, const uint32_t col[C], const uint32_t desc[C]) {
    uint64_t ra;
    uint32_t rb;
    encode_raw<C>(col, desc, ra, rb);
    store_raw<C>(v, s, p, ra, rb);
}

// unaligned words of global memory (global accesses need no alignment on this device)
struct __attribute__((packed, aligned(1))) UnalignedU32 {
    uint32_t v;
};
struct __attribute__((packed, aligned(1))) UnalignedU16 {
    uint16_t v;
};
template <typename W, typename T>
LV_D auto peek(T* base, uint32_t byte) {
    return ((gptr<const W>)((gptr<const uint8_t>)base + byte))->v;
}
template <typename W, typename T, typename V>
LV_D void poke(T* base, uint32_t byte, V value) {
    ((gptr<W>)((gptr<uint8_t>)base + byte))->v = value;
}

// intra descriptors of pixel q, RGB as {d0 | d1 << 16, d2}, grey as {d0}
template <int C>
struct DescWords {
    uint32_t w0, w1;
};
template <int C>
LV_D DescWords<C> load_desc(const uint16_t* desc, uint32_t q) {
    if constexpr (C == 3) return {peek<UnalignedU32>(desc, 6u * q), peek<UnalignedU16>(desc, 6u * q + 4u)};
    else return {*at(desc, q), 0u};
}
// a pixel's sample record (the value it writes into samples) from its packed colour and descriptor words
template <int C>
LV_D void record_of(uint32_t colour, DescWords<C> d, uint64_t& ra, uint32_t& rb) {
    if constexpr (C == 3) {
        ra = (uint64_t)d.w0 | ((uint64_t)(d.w1 | colour << 16) << 32);
        rb = colour >> 16;
    } else {
        ra = (uint64_t)(d.w0 | colour << 16);
        rb = 0;
    }
}
// the packed colour of pixel q from global memory (bytes, so that nothing past the frame is read)
template <int C>
LV_D uint32_t load_colour(const uint8_t* frame, uint32_t q) {
    uint32_t w = 0;
#pragma unroll
    for (int c = 0; c < C; ++c) w |= (uint32_t)*at(frame, q * C + c) << (8 * c);
    return w;
}

// ----------------------------------------------------------------------------------------------
// LDS frame tile with a 2-pixel halo (the 5x5 LBSP patch)
// ----------------------------------------------------------------------------------------------
// RGB: one word per pixel (c0 | c1 << 8 | c2 << 16), so a tap is one LDS read for the three channels and a
// halo row one 3-byte-strided word load per pixel. Grey: bytes, loaded as words from 4 bytes left of the tile.
template <int C>
struct FrameTile;
template <>
struct FrameTile<3> {
    static constexpr int LW = TW + 4, LH = TH + 4;
    uint32_t px[LH][LW];
};
template <>
struct FrameTile<1> {
    static constexpr int LW = TW + 4, LH = TH + 4, OFF = 2, WORDS = 18, PITCH = 4 * WORDS;
    alignas(4) uint8_t px[LH][PITCH];
};

// a 32-bit word at any byte offset of a buffer of `total` bytes (4 at least), zeros outside it; the last bytes
// of a buffer come from its last whole word
template <typename I>
LV_D uint32_t word_at(const uint8_t* base, I off, I total) {
    const I o = word_place(off, total);
    const uint32_t w = sizeof(I) == 4 ? peek<UnalignedU32>(base, (uint32_t)o) : peek<UnalignedU32>(base + o, 0u);
    const I beyond = off - o;  // < 0: left of the buffer, > 0: bytes to drop
    return beyond < 0 || beyond > 3 ? 0u : w >> (8 * (int)beyond);
}

// Pixels left and right of the image come out as whatever lies beside them in the frame: no pixel of the ROI
// reaches them. I: the type of byte offsets.
template <int C, typename I = int>
LV_D void load_frame_tile(FrameTile<C>& t, const uint8_t* frame, int W, int H, int x0, int y0) {
    using T = FrameTile<C>;
    const I total = (I)W * H * C;
    if constexpr (C == 3) {
        auto put = [&](int r, int c) {
            const int gy = y0 + r - 2;
            t.px[r][c] = gy >= 0 && gy < H ? word_at(frame, ((I)gy * W + x0 + c - 2) * 3, total) & 0xFFFFFFu : 0u;
        };
        const int lx = (int)threadIdx.x % TW, ly = (int)threadIdx.x / TW;
#pragma unroll
        for (int k = 0; k < T::LH / TH; ++k) put(ly + TH * k, lx);
        if (threadIdx.x < 4u * T::LH) put((int)threadIdx.x / 4, TW + (int)threadIdx.x % 4);
    } else {
        const int r = (int)threadIdx.x / T::WORDS, l = (int)threadIdx.x % T::WORDS, gy = y0 + r - 2;
        if (r < T::LH) {
            const uint32_t w = gy >= 0 && gy < H ? word_at(frame, (I)gy * W + x0 - 4 + 4 * l, total) : 0u;
            *(uint32_t*)&t.px[r][4 * l] = w;
        }
    }
}

// packed colour of halo pixel (hx, hy)
LV_D uint32_t tile_colour(const FrameTile<3>& t, int hx, int hy) { return t.px[hy][hx]; }
LV_D uint32_t tile_colour(const FrameTile<1>& t, int hx, int hy) { return t.px[hy][FrameTile<1>::OFF + hx]; }

// packed 16 taps of every channel around tile-local (lx, ly) (centre coordinates, halo excluded). RGB: four
// pixel words become three tap words by a byte transposition (seven v_perm; 16 LDS reads and 28 permutes
// where single bytes took 48 reads and 36 shifts).
LV_D void tile_taps(const FrameTile<3>& t, int lx, int ly, uint32_t (&taps)[3][4]) {
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        uint32_t q[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) q[k] = t.px[ly + 2 + kLbspDY[4 * w + k]][lx + 2 + kLbspDX[4 * w + k]];
        // v_perm_b32(hi, lo): bytes 0-3 select lo's, 4-7 hi's
        const uint32_t a = __builtin_amdgcn_perm(q[1], q[0], 0x05010400u);  // q0.0 q1.0 q0.1 q1.1
        const uint32_t b = __builtin_amdgcn_perm(q[3], q[2], 0x05010400u);
        const uint32_t c = __builtin_amdgcn_perm(q[1], q[0], 0x0C0C0602u);  // q0.2 q1.2
        const uint32_t d = __builtin_amdgcn_perm(q[3], q[2], 0x0C0C0602u);
        taps[0][w] = __builtin_amdgcn_perm(b, a, 0x05040100u);
        taps[1][w] = __builtin_amdgcn_perm(b, a, 0x07060302u);
        taps[2][w] = __builtin_amdgcn_perm(d, c, 0x05040100u);
    }
}
LV_D void tile_taps(const FrameTile<1>& t, int lx, int ly, uint32_t (&taps)[1][4]) {
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        uint32_t acc = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k)
            acc |= (uint32_t)t.px[ly + 2 + kLbspDY[4 * w + k]][FrameTile<1>::OFF + lx + 2 + kLbspDX[4 * w + k]] << (8 * k);
        taps[0][w] = acc;
    }
}

template <int C>
LV_D void taps_from_global(const uint8_t* frame, int W, int x, int y, int c, uint32_t taps[4]) {
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        uint32_t acc = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int n = 4 * w + k;
            acc |= (uint32_t)*at(frame, ((y + kLbspDY[n]) * W + (x + kLbspDX[n])) * C + c) << (8 * k);
        }
        taps[w] = acc;
    }
}

// the threshold limits of every colour (a block of 256 threads)
LV_D void load_lut(LbspLimits* lut, const Scalars* sc) {
    static_assert(TPB == 256, "one entry per thread");
    const uint32_t k = threadIdx.x;
    lut[k] = lbsp_limits(k, *at(sc->lut, k));
}

// ----------------------------------------------------------------------------------------------
// per-pixel match context
// ----------------------------------------------------------------------------------------------
template <int C>
struct PxCtx {
    uint32_t cur[C], intra[C];
    uint32_t taps[C][4];                   // packed taps (byte k of word w = tap 4w+k)
    uint32_t t_sc, t_tot_col, t_tot_desc;  // SuBSENSE 3ch / LOBSTER 3ch thresholds
    uint32_t t_col, t_desc;                // 1ch thresholds
};

// SuBSENSE per-pixel thresholds from the previous unstable flag (SUB:355-359, 1ch :222-223). The reference
// computes them in size_t; a threshold is only compared with distances of at most 765, so bounds that are
// far above those (2^28 for the colour, 2^20 for the power of two) give the same tests in 32 bits: the
// parameters are below 2^24, so nothing overflows.
template <int C>
LV_D void subsense_thresholds(const View& v, float R, uint32_t unst_old, PxCtx<C>& px) {
    const float colf = R * (float)v.color_thr - (unst_old ? 0.0f : (float)(v.color_thr / 5u));
    const uint32_t col = (uint32_t)fminf(colf, 268435456.0f);
    const uint32_t shift = (uint32_t)floorf(R + 0.5f) & 63u;
    const uint32_t desc = (1u << (shift < 20u ? shift : 20u)) + v.desc_thr + unst_old * v.desc_thr;
    if constexpr (C == 1) {
        px.t_col = col / 2u;
        px.t_desc = desc;
        px.t_sc = px.t_tot_col = px.t_tot_desc = 0u;  // unused by the 1-channel test
    } else {
        px.t_tot_col = 3u * col;
        px.t_tot_desc = 3u * desc;
        px.t_sc = px.t_tot_col / 2u;
        px.t_col = px.t_desc = 0u;  // unused by the 3-channel test
    }
}

// LOBSTER fixed thresholds (LOB:485-488 1ch; :515-518 3ch)
template <int C>
LV_D void lobster_thresholds(const View& v, PxCtx<C>& px) {
    if constexpr (C == 1) {
        px.t_col = v.color_thr / 2u;
        px.t_desc = v.desc_thr;
        px.t_sc = px.t_tot_col = px.t_tot_desc = 0u;  // unused by the 1-channel test
    } else {
        px.t_tot_desc = v.desc_thr * 3u;
        px.t_tot_col = v.color_thr * 3u;
        px.t_sc = px.t_tot_col / 2u;   // colour, per channel
        px.t_desc = px.t_tot_desc / 2u;  // descriptor, per channel
    }
}

// one sample test; returns true on a match and accumulates the SuBSENSE distances
template <int C, int ALGO, int RS>
LV_D bool test_sample(const PxCtx<C>& px, const LbspLimits* lut, const uint32_t col[C], const uint32_t desc[C],
                      uint32_t& tot_desc, uint32_t& tot_sum) {
    if constexpr (ALGO == kSuBSENSE && C == 3) {
        // all colour tests first: a sample failing any of them fails whatever the descriptors say
        uint32_t cdv[3];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            cdv[c] = absdiff(px.cur[c], col[c]);
            if (cdv[c] > px.t_sc) return false;
        }
        uint32_t td = 0, ts = 0;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const uint32_t cd = cdv[c];
            const uint32_t inter = lbsp_threshold_packed(px.taps[c], lut[col[c]]);
            const uint32_t dd = (popc(px.intra[c] ^ desc[c]) + popc(inter ^ desc[c])) >> 1;
            uint32_t sum = (dd >> 1) * 15u + cd;
            sum = sum > 255u ? 255u : sum;
            if (sum > px.t_sc) return false;
            td += dd;
            ts += sum;
        }
        if (td > px.t_tot_desc || ts > px.t_tot_col) return false;
        tot_desc = td;
        tot_sum = ts;
        return true;
    } else if constexpr (ALGO == kSuBSENSE && C == 1) {
        const uint32_t cd = absdiff(px.cur[0], col[0]);
        if (cd > px.t_col) return false;
        const uint32_t inter = lbsp_threshold_packed(px.taps[0], lut[col[0]]);
        const uint32_t dd = (popc(px.intra[0] ^ desc[0]) + popc(inter ^ desc[0])) >> 1;
        if (dd > px.t_desc) return false;
        uint32_t sum = (dd >> 2) * 15u + cd;
        sum = sum > 255u ? 255u : sum;
        if (sum > px.t_col) return false;
        tot_desc = dd;
        tot_sum = sum;
        return true;
    } else if constexpr (ALGO == kLOBSTER && C == 3) {
        uint32_t cdv[3];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            cdv[c] = absdiff(px.cur[c], col[c]);
            if (cdv[c] > px.t_sc) return false;
        }
        uint32_t tc = 0, td = 0;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const uint32_t cd = cdv[c];
            const uint32_t inter = lbsp_threshold_packed(px.taps[c], lut[col[c]]);
            const uint32_t dd = popc(inter ^ desc[c]);
            if (dd > px.t_desc) return false;
            tc += cd;
            td += dd;
        }
        tot_desc = td;
        tot_sum = tc;
        return td <= px.t_tot_desc && tc <= px.t_tot_col;
    } else {
        const uint32_t cd = absdiff(px.cur[0], col[0]);
        if (cd > px.t_col) return false;
        const uint32_t inter = lbsp_threshold_packed(px.taps[0], lut[col[0]]);
        tot_desc = 0;
        tot_sum = 0;
        return popc(inter ^ desc[0]) <= px.t_desc;
    }
}

// raster-earlier neighbours that can diffuse into p (5x5 window): offsets in raster order
constexpr int kPredDX[12] = {-2, -1, 0, 1, 2, -2, -1, 0, 1, 2, -2, -1};
constexpr int kPredDY[12] = {-2, -2, -2, -2, -2, -1, -1, -1, -1, -1, 0, 0};

LV_D int pred_dx(uint32_t i) { return (int)(i % 5u) - 2; }
LV_D int pred_dy(uint32_t i) { return (int)(i / 5u) - 2; }

// free bits of a record that the tiles in LDS fold tests into
constexpr uint32_t kRecBg = 1u << 11;   // decided background
constexpr uint32_t kRecFwd = 1u << 12;  // fwd_gate
constexpr uint32_t kRecAny = 1u << 13;  // gate a or gate b

// static forward gate of a record whose target lies after the writer in raster order
LV_D bool fwd_gate(uint32_t r) { return rec_gate_a(r) || (rec_gate_b(r) && rec_ghost_fwd(r)); }

// Ordered scan s = 0..N-1 until REQ matches (SUB:366-395, LOB:480-495). Samples overwritten by
// applied writers are taken from the writer; the last writer in raster order wins. Two evaluation orders
// give the same result as the sequential loop:
//   scan_seq  : one lane per pixel, samples in order, KF loads in flight, up to `limit`, with
//               at most kRepl overwritten slots substituted from the thread's LDS entries;
//   scan_group: the kGroup lanes of a group evaluate kGroup consecutive samples of one pixel at once; the
//               matches are then taken in sample order up to the REQ-th.
constexpr int kGroup = 16;

struct ScanState {
    uint32_t good, s, md, ms;
};

template <int C>
LV_D ScanState scan_init() {
    return ScanState{0u, 0u, C * 16u, C * 255u};
}

// Overwritten slots of a pixel with their replacement values (the last applied writer's current
// value), kept per thread in LDS so the sequential scan's loop carries only a slot bitmap: a sample
// whose slot bit is set looks its slot up in the thread's entries. At most kRepl distinct slots;
// pixels with more (very rare) go to the fix point unmatched. w2 holds the record's last byte with the slot
// above it.
constexpr int kRepl = 4;
struct ReplLds {
    uint32_t w0[kRepl][TPB], w1[kRepl][TPB], w2[kRepl][TPB];
};

// one LDS table per kernel, whichever channel counts the kernel instantiates
LV_D ReplLds& repl_lds() {
    __shared__ ReplLds r;
    return r;
}

template <int C>
LV_D void raw_current(const View& v, const uint8_t* frame, uint32_t q, uint64_t& ra, uint32_t& rb) {
    record_of<C>(load_colour<C>(frame, q), load_desc<C>(v.desc_cur, q), ra, rb);
}

// Fills the thread's entries from the applied writers, the latest in raster order first (it owns
// its slot). Returns the slot bitmap (mod 64) and the entry count, or false beyond kRepl slots.
// rec_of(i) is the update record of predecessor i, colour_of(i, q) its packed colour.
template <int C, typename RecOf, typename ColourOf>
LV_D bool build_repl(const View& v, int x, int y, uint32_t applied, uint64_t& sbm, int& n, RecOf rec_of,
                     ColourOf colour_of) {
    ReplLds& R = repl_lds();
    const int t = (int)threadIdx.x;
    sbm = 0;
    n = 0;
    for (uint32_t m = applied; m;) {
        const int i = 31 - __builtin_clz(m);
        m &= ~(1u << i);
        const uint32_t q = (uint32_t)((y + pred_dy((uint32_t)i)) * v.W + (x + pred_dx((uint32_t)i)));
        const uint32_t sl = rec_slot_diff(rec_of(i));
        bool seen = false;
#pragma unroll
        for (int k = 0; k < kRepl; ++k) seen = seen || (k < n && R.w2[k][t] >> 8 == sl);
        if (seen) continue;
        if (n == kRepl) return false;
        uint64_t ra;
        uint32_t rb;
        record_of<C>(colour_of(i, q), load_desc<C>(v.desc_cur, q), ra, rb);
        R.w0[n][t] = (uint32_t)ra;
        R.w1[n][t] = (uint32_t)(ra >> 32);
        R.w2[n][t] = rb | sl << 8;
        sbm |= 1ull << (sl & 63u);
        ++n;
    }
    return true;
}

// One batch of KF loaded samples of a sequential scan (stops at the limit or at REQ matches).
template <int C, int ALGO, int RS, int KF>
LV_D void scan_batch(const LbspLimits* lut, const PxCtx<C>& px, uint64_t sbm, int nrep, ScanState& st, uint32_t limit,
                     uint32_t REQ, const uint64_t (&ra)[KF], const uint32_t (&rb)[KF]) {
    const ReplLds& R = repl_lds();
    const int t = (int)threadIdx.x;
#pragma unroll
    for (int j = 0; j < KF; ++j) {
        if (st.s >= limit || st.good >= REQ) break;
        uint64_t a = ra[j];
        uint32_t b = rb[j];
        if ((sbm >> (st.s & 63u)) & 1u) {
            for (int k = 0; k < nrep; ++k)
                if (R.w2[k][t] >> 8 == st.s) {
                    a = (uint64_t)R.w0[k][t] | ((uint64_t)R.w1[k][t] << 32);
                    b = R.w2[k][t];
                    break;
                }
        }
        uint32_t col[C], desc[C];
        decode_raw<C>(a, b, col, desc);
        uint32_t td = 0, ts = 0;
        if (test_sample<C, ALGO, RS>(px, lut, col, desc, td, ts)) {
            st.md = td < st.md ? td : st.md;
            st.ms = ts < st.ms ? ts : st.ms;
            ++st.good;
        }
        ++st.s;
    }
}

// speculative scan: a wavefront whose active lanes drop below kWaveCutLanes after at least
// kWaveCutMinSamples samples hands its remaining pixels to the continuation (measured on the
// 64-stream batch: phase A 2544 -> 2403 us, the whole step 8124 -> 8071 us)
constexpr int kWaveCutLanes = 16;
constexpr uint32_t kWaveCutMinSamples = 4;

// words between the records of two consecutive samples of a pixel
template <int C>
constexpr uint32_t kSampleStride = 64u * (C == 3 ? 3u : 1u);

// Sequential scan from st.s up to the limit. Unconditional loads (the sample planes are padded by
// kMaxFetch samples) at constant offsets from a running pointer keep all KF loads in flight together
// without address arithmetic.
template <int C, int ALGO, int RS, int KF>
LV_D void scan_seq(const View& v, const LbspLimits* lut, const PxCtx<C>& px, int x, int y, uint64_t sbm, int nrep,
                   ScanState& st, uint32_t limit) {
    const uint32_t p = (uint32_t)(y * v.W + x);
    const uint32_t REQ = (uint32_t)v.REQ;
    constexpr uint32_t kStride = kSampleStride<C>;
    const uint32_t* cur = rec_base(v, p) + st.s * kStride;
    while (st.s < limit && st.good < REQ) {
        // speculative phase: once few lanes of the wavefront still scan, their pixels go on in the
        // dense continuation instead of holding the whole wavefront (the cut never changes a result)
        if constexpr (RS != 0)
            if (st.s >= kWaveCutMinSamples && __popcll(__ballot(1)) < kWaveCutLanes) break;
        uint64_t ra[KF];
        uint32_t rb[KF];
#pragma unroll
        for (int j = 0; j < KF; ++j) fetch_at<C>(cur + j * kStride, ra[j], rb[j]);
        cur += KF * kStride;
        scan_batch<C, ALGO, RS, KF>(lut, px, sbm, nrep, st, limit, REQ, ra, rb);
    }
}

LV_D uint32_t pack_state(const ScanState& st) { return mres_pack(st.good, st.md, st.ms, st.s); }

LV_D ScanState unpack_state(uint32_t mr) {
    return ScanState{mr & 255u, mr >> 24, (mr >> 8) & 63u, (mr >> 14) & 1023u};
}

// Appends one value per calling lane that wants to (push) to a list: one atomic per wavefront on the
// list's counter. Must be called by the lanes of a wavefront together.
LV_D void wave_append(bool push, uint32_t value, uint32_t* counter, uint32_t* list) {
    const unsigned long long bal = __ballot(push);
    if (!bal) return;
    const int lane = (int)(threadIdx.x & 63u), leader = __ffsll((long long)bal) - 1;
    uint32_t base = 0;
    if (lane == leader) base = atomicAdd(counter, (uint32_t)__popcll(bal));
    base = (uint32_t)__shfl((int)base, leader, 64);
    if (push) G(list)[base + (uint32_t)__popcll(bal & ((1ull << lane) - 1ull))] = value;
}

// Worklist of fix-point iteration 1, filled by the match phases: split into kContStripes stripes like
// the continuation list (the pixels of tile b push to stripe b % kContStripes, at most one entry
// each, so a stripe holds at most cont_region entries). With one counter for all pushes its atomics
// were what the continuation spent its time on, 12 to 16 ns each: match_seq 575 -> 154 us on a 3840x2160
// frame with 36 K pushes, 211 -> 81 us at 1920x1080. A target may be listed twice (two changed writers):
// both items match it against the same decisions, or the one that saw the older ones is followed by
// another in the next iteration, which its changed writer pushes.
LV_D void push_first(const View& v, bool push, uint32_t t, uint32_t stripe) {
    wave_append(push, t, &v.sc->wl_first[stripe * kContStride], v.wl1 + (size_t)stripe * v.cont_region);
}

// worklist of iteration k >= 2: one counter (few entries)
LV_D void push_next(const View& v, bool push, uint32_t t, uint32_t k, uint32_t* wl_dst) {
    wave_append(push, t, &v.sc->wl_count[k % kWlRing], wl_dst);
}

// exclusive prefix of the kContStripes counters at cnt (kContStride words apart) into pre, by the
// first wavefront of the block; the caller synchronizes before reading pre
LV_D void stripe_prefix(const uint32_t* cnt, uint32_t* pre) {
    static_assert(kContStripes <= 64 && (kContStripes & (kContStripes - 1)) == 0, "one wavefront scans the stripe counts");
    if (threadIdx.x >= 64u) return;
    const int lane = (int)threadIdx.x;
    uint32_t c = lane < kContStripes ? G(cnt)[lane * kContStride] : 0u;
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t t = (uint32_t)__shfl_up((int)c, (unsigned)o, 64);
        if (lane >= o) c += t;
    }
    if (lane < kContStripes) pre[lane + 1] = c;
    if (lane == 0) pre[0] = 0u;
}
// item i of a striped list: the last stripe whose prefix is at most i
LV_D uint32_t stripe_of(const uint32_t* pre, uint32_t i) {
    uint32_t k = 0;
    for (uint32_t half = kContStripes / 2; half > 0; half >>= 1)
        if (pre[k + half] <= i) k += half;
    return k;
}

// forward target of p's own diffusion (if any): target after p in raster order with open gate
LV_D bool forward_target(const View& v, uint32_t r, int x, int y, uint32_t& t) {
    const uint32_t tg = rec_tgt(r);
    if (tg == kRecNone || !fwd_gate(r)) return false;
    const int dx = tgt_dx(tg), dy = tgt_dy(tg);
    if (!(dy > 0 || (dy == 0 && dx > 0))) return false;
    t = (uint32_t)((y + dy) * v.W + (x + dx));
    return *at(v.roi, t) != 0;
}

// draw % N, with the reciprocal of N laid out in the View
LV_D uint32_t mod_n(const View& v, uint32_t d) {
    const uint32_t q = __umulhi(d, v.n_mul) >> v.n_shift;
    return v.N == 1 ? 0u : d - q * (uint32_t)v.N;
}

// ----------------------------------------------------------------------------------------------
// describe: LBSP intra descriptors, unstable flag, RNG draws, update record (SUB:355-365,
// :406-449 / LOB:499-512). Writes desc_cur, rec; counts non-zero descriptors.
// ----------------------------------------------------------------------------------------------
template <int C, int ALGO>
LV_D void describe_body(const View& v, uint32_t bid, uint32_t nblk) {
    const uint8_t* frame = v.frame;
    const double lr = v.lr;
    __shared__ FrameTile<C> tile;
    __shared__ alignas(8) LbspLimits lut[256];
    const int ntx = (v.W + TW - 1) / TW;
    const int tid = (int)bid;
    const int x0 = (tid % ntx) * TW, y0 = (tid / ntx) * TH;
    if (bid == 0 && threadIdx.x == 0) {
        // per-frame counters consumed by later kernels of this step
        for (int i = 0; i < kWlRing; ++i) v.sc->wl_count[i] = 0;
        for (int i = 0; i < 8; ++i) v.sc->wl_work[i] = 0;
        v.sc->iters = 0;
    }
    if (bid == 0 && threadIdx.x < kContStripes) {
        v.sc->cont_cnt[threadIdx.x * kContStride] = 0;
        v.sc->wl_first[threadIdx.x * kContStride] = 0;
    }
    if (bid == 0 && threadIdx.x < kStripes) {
        v.sc->ex_part[threadIdx.x] = 0;
        v.sc->wr_part[threadIdx.x] = 0;
        v.sc->spec_part[threadIdx.x] = 0;
        v.sc->coop_part[threadIdx.x] = 0;
    }
    const int lx = threadIdx.x % TW, ly = threadIdx.x / TW, x = x0 + lx, y = y0 + ly;
    const bool inside = x < v.W && y < v.H;
    // the pixel's own state is loaded first, so these loads run alongside the tile's
    const uint32_t pp = inside ? (uint32_t)(y * v.W + x) : 0u;
    const uint8_t roi_p = *at(v.roi, pp);
    float Rv = 0.f, Tv = 0.f, d_lt = 0.f, d_st = 0.f;
    if constexpr (ALGO == kSuBSENSE) {
        Rv = *at(v.R, pp);
        Tv = *at(v.T, pp);
        d_lt = *at(v.RawLT, pp) - *at(v.FinLT, pp);
        d_st = *at(v.RawST, pp) - *at(v.FinST, pp);
    }
    load_frame_tile<C>(tile, frame, v.W, v.H, x0, y0);
    load_lut(lut, v.sc);
    __syncthreads();
    bool nz = false;
    if (inside) {
        const uint32_t p = pp;
        if (!roi_p) {
            *at(v.rec, p) = kRecNone;
        } else {
            uint32_t pc = 0;
            uint32_t intra[C];
            uint32_t taps[C][4];
            tile_taps(tile, lx, ly, taps);
            const uint32_t centre = tile_colour(tile, lx + 2, ly + 2);
#pragma unroll
            for (int c = 0; c < C; ++c) {
                const uint32_t ref = (centre >> (8 * c)) & 255u;
                intra[c] = lbsp_threshold_packed(taps[c], lut[ref]);
                pc += popc(intra[c]);
            }
            if constexpr (C == 3) {
                poke<UnalignedU32>(v.desc_cur, 6u * p, intra[0] | intra[1 % C] << 16);
                poke<UnalignedU16>(v.desc_cur, 6u * p + 4u, (uint16_t)intra[2 % C]);
            } else {
                *at(v.desc_cur, p) = (uint16_t)intra[0];
            }
            nz = pc >= (C == 1 ? 2u : 4u);
            const uint32_t frame_no = cur_frame(v);
            uint32_t d[4];
            draw4(v.seed_lo, v.seed_hi, v.stream_id, frame_no, PH_APPLY, 0, p, 0, d);
            // draw 4 (group 1) is the diffusion slot: drawn only when a diffusion gate is open
            auto diff_slot = [&]() {
                uint32_t d4[4];
                draw4(v.seed_lo, v.seed_hi, v.stream_id, frame_no, PH_APPLY, 0, p, 1, d4);
                return mod_n(v, d4[0]);
            };
            // learning rates beyond the exact range of divides31 (uniform; infinity among them)
            const bool slow = lr > (double)kDividesMax;
            uint32_t r;
            if constexpr (ALGO == kSuBSENSE) {
                const uint32_t unst_new = (Rv > 3.0f || d_lt > 0.1f || d_st > 0.1f) ? 1u : 0u;
                const bool use3 = v.use3x3 && !unst_new;
                bool self_bg, gate_a;
                if (slow) {
                    const uint64_t L = isinf(lr) ? ~0ull : (uint64_t)ceil(lr);
                    self_bg = mod64(d[0], L) == 0u;
                    gate_a = mod64(d[3], use3 ? L : L / 2u + 1u) == 0u;
                } else {
                    const uint32_t L = lr > 0 ? (uint32_t)ceil(lr) : (uint32_t)ceilf(Tv);
                    self_bg = divides31(d[0], L);
                    gate_a = divides31(d[3], use3 ? L : L / 2u + 1u);
                }
                const bool self_fg = v.sc->cooldown != 0u && (d[0] % 2u) == 0u;
                int tx, ty;
                neighbor_pos(d[2], use3, x, y, v.W, v.H, tx, ty);
                const uint32_t lcap = (uint32_t)v.sc->lower_cap;  // 1, 2 or 4
                const bool gate_b = (lcap & (lcap - 1u)) == 0u ? (d[3] & (lcap - 1u)) == 0u : d[3] % lcap == 0u;
                bool ghost_fwd = false;
                if (ty > y || (ty == y && tx > x)) {
                    const uint32_t t = (uint32_t)(ty * v.W + tx);
                    ghost_fwd = *at(v.RawST, t) > 0.995f && *at(v.MLD, t) < 0.010f;
                }
                const uint32_t tg = (uint32_t)((ty - y + 2) * 5 + (tx - x + 2));
                const uint32_t sd = (gate_a || gate_b) ? diff_slot() : 0u;
                r = tg | ((uint32_t)gate_a << 5) | ((uint32_t)gate_b << 6) | ((uint32_t)ghost_fwd << 7) |
                    ((uint32_t)self_bg << 8) | ((uint32_t)self_fg << 9) | (unst_new << 10) | (mod_n(v, d[1]) << 16) |
                    (sd << 24);
            } else {
                const uint64_t L = isinf(lr) ? ~0ull : (uint64_t)ceil(lr);
                const bool self_bg = slow ? mod64(d[0], L) == 0u : divides31(d[0], (uint32_t)L);
                const bool gate_a = slow ? mod64(d[2], L) == 0u : divides31(d[2], (uint32_t)L);
                int tx, ty;
                neighbor_pos(d[3], true, x, y, v.W, v.H, tx, ty);
                const uint32_t tg = (uint32_t)((ty - y + 2) * 5 + (tx - x + 2));
                const uint32_t sd = gate_a ? diff_slot() : 0u;
                r = tg | ((uint32_t)gate_a << 5) | ((uint32_t)self_bg << 8) | (mod_n(v, d[1]) << 16) | (sd << 24);
            }
            *at(v.rec, p) = r;
        }
    }
    if constexpr (ALGO == kSuBSENSE) block_add<TPB>(nz ? 1u : 0u, v.sc->nz_part);
}

// a pixel's per-frame match inputs, loaded together with the tile: intra descriptors of the current frame with
// the ROI and the previous unstable flag above the last one, and R
template <int C>
struct PxIn {
    uint32_t w[C == 3 ? 2 : 1];
    float R;
    LV_D uint32_t desc(int c) const { return (w[c / 2] >> (16 * (c & 1))) & 0xFFFFu; }
    LV_D bool roi() const { return (w[C == 3 ? 1 : 0] >> 16) & 1u; }
    LV_D uint32_t unst() const { return w[C == 3 ? 1 : 0] >> 24; }
};

template <int C, int ALGO>
LV_D PxIn<C> load_px_in(const View& v, uint32_t q, bool in) {
    PxIn<C> r;
    const uint8_t roi = *at(v.roi, q);
    const DescWords<C> d = load_desc<C>(v.desc_cur, q);
    uint32_t unst = 0;
    r.R = 0.f;
    if constexpr (ALGO == kSuBSENSE) {
        r.R = *at(v.R, q);
        unst = *at(v.unstable, q);
    }
    const uint32_t flags = (in && roi ? 1u << 16 : 0u) | unst << 24;
    if constexpr (C == 3) {
        r.w[0] = d.w0;
        r.w[1 % (C == 3 ? 2 : 1)] = d.w1 | flags;
    } else {
        r.w[0] = d.w0 | flags;
    }
    return r;
}

// the match context of tile-local pixel (lx, ly) from the LDS frame tile (complete behind a workgroup
// barrier) and the inputs
template <int C, int ALGO>
LV_D void build_ctx_staged(const View& v, const FrameTile<C>& tile, int lx, int ly, const PxIn<C>& in, PxCtx<C>& px) {
    const uint32_t centre = tile_colour(tile, lx + 2, ly + 2);
#pragma unroll
    for (int c = 0; c < C; ++c) {
        px.cur[c] = (centre >> (8 * c)) & 255u;
        px.intra[c] = in.desc(c);
    }
    tile_taps(tile, lx, ly, px.taps);
    if constexpr (ALGO == kSuBSENSE) subsense_thresholds<C>(v, in.R, in.unst(), px);
    else lobster_thresholds<C>(v, px);
}

// A match context in kCtxWords words (16-byte aligned): taps (12 words), packed centre colours and
// intra descriptors (3), thresholds (5). Written by the speculative match for the pixels it leaves
// to the continuation, which then reads it instead of rebuilding it from the frame.
template <int C>
LV_D void store_ctx(uint32_t* d, const PxCtx<C>& px) {
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    const gptr<u32x4> q = (gptr<u32x4>)d;
#pragma unroll
    for (int c = 0; c < C; ++c) q[c] = u32x4{px.taps[c][0], px.taps[c][1], px.taps[c][2], px.taps[c][3]};
    if constexpr (C == 3) {
        q[3] = u32x4{px.cur[0] | px.cur[1] << 8 | px.cur[2] << 16, px.intra[0] | px.intra[1] << 16, px.intra[2], px.t_sc};
        q[4] = u32x4{px.t_tot_col, px.t_tot_desc, px.t_col, px.t_desc};
    } else {
        q[3] = u32x4{px.cur[0], px.intra[0], 0u, px.t_sc};
        q[4] = u32x4{px.t_tot_col, px.t_tot_desc, px.t_col, px.t_desc};
    }
}

template <int C>
LV_D void load_ctx(const uint32_t* d, PxCtx<C>& px) {
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    const gptr<const u32x4> q = (gptr<const u32x4>)d;
#pragma unroll
    for (int c = 0; c < C; ++c) {
        const u32x4 t = q[c];
        px.taps[c][0] = t.x;
        px.taps[c][1] = t.y;
        px.taps[c][2] = t.z;
        px.taps[c][3] = t.w;
    }
    const u32x4 a = q[3], b = q[4];
#pragma unroll
    for (int c = 0; c < C; ++c) px.cur[c] = (a.x >> (8 * c)) & 255u;
    px.intra[0] = a.y & 0xFFFFu;
    if constexpr (C == 3) {
        px.intra[1 % C] = a.y >> 16;
        px.intra[2 % C] = a.z;
    }
    px.t_sc = a.w;
    px.t_tot_col = b.x;
    px.t_tot_desc = b.y;
    px.t_col = b.z;
    px.t_desc = b.w;
}

// the same context with the taps read from the frame in global memory
template <int C, int ALGO>
LV_D void build_ctx_global(const View& v, const uint8_t* frame, int x, int y, PxCtx<C>& px) {
    const uint32_t p = (uint32_t)(y * v.W + x);
#pragma unroll
    for (int c = 0; c < C; ++c) {
        px.cur[c] = *at(frame, p * C + c);
        px.intra[c] = *at(v.desc_cur, p * C + c);
    }
#pragma unroll
    for (int c = 0; c < C; ++c)
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            uint32_t acc = 0;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int n = 4 * w + k;
                acc |= (uint32_t)*at(frame, ((y + kLbspDY[n]) * v.W + (x + kLbspDX[n])) * C + c) << (8 * k);
            }
            px.taps[c][w] = acc;
        }
    if constexpr (ALGO == kSuBSENSE) subsense_thresholds<C>(v, *at(v.R, p), *at(v.unstable, p), px);
    else lobster_thresholds<C>(v, px);
}

// ----------------------------------------------------------------------------------------------
// group match: the kGroup lanes of a group work on one pixel. A scan that one lane runs as a chain of
// dependent loads (50 samples: 13 rounds of four) takes four rounds here, and the twelve records and
// decisions of the raster-earlier neighbours are read by twelve lanes at once.
// ----------------------------------------------------------------------------------------------
struct GroupLds {
    uint32_t taps[TPB / kGroup][12];
};

// Writers of p applied by the match: bit i of the result is set when predecessor i targets p with an
// open forward gate and its decision is background (CURRENT: the decisions of the fix point, else those of
// the previous frame). slot = the sample slot lane i's predecessor writes; turned (CURRENT) = the group
// has a candidate writer of a slot below `below` whose decision is not the guessed one. Every lane of the
// wavefront calls.
template <bool CURRENT>
LV_D uint32_t group_writers(const View& v, int x, int y, bool active, uint32_t& slot, uint32_t below, bool& turned) {
    const int lane = (int)(threadIdx.x & 63u), gbase = lane & ~(kGroup - 1);
    const uint32_t sub = (uint32_t)(lane & (kGroup - 1));
    bool on = false, other = false;
    slot = 0;
    if (active && sub < 12u) {
        const int dx = pred_dx(sub), dy = pred_dy(sub);
        const uint32_t q = (uint32_t)((y + dy) * v.W + (x + dx));
        const uint32_t r = *at(v.rec, q);
        const uint8_t guess = *at(v.last_raw, q);
        const uint8_t d = CURRENT ? __hip_atomic_load(&v.dec[q], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : guess;
        const bool writer = rec_tgt(r) == (uint32_t)((2 - dy) * 5 + (2 - dx)) && fwd_gate(r);
        slot = rec_slot_diff(r);
        on = writer && d == 0;
        other = writer && (d == 0) != (guess == 0) && slot < below;
    }
    if constexpr (CURRENT) turned = ((uint32_t)(__ballot(other) >> gbase) & 0xFFFu) != 0u;
    return (uint32_t)(__ballot(on) >> gbase) & 0xFFFu;
}

// Scans on from st.s to REQ matches or N samples. Every lane of the wavefront calls; the lanes of a group
// share px, x, y, applied and st.
template <int C, int ALGO>
LV_D void scan_group(const View& v, const uint8_t* frame, const LbspLimits* lut, const PxCtx<C>& px, int x, int y,
                     uint32_t applied, uint32_t slot, ScanState& st, bool active) {
    const uint32_t N = (uint32_t)v.N, REQ = (uint32_t)v.REQ;
    const int lane = (int)(threadIdx.x & 63u), gbase = lane & ~(kGroup - 1);
    const uint32_t p = active ? (uint32_t)(y * v.W + x) : 0u;
    bool done = !active || st.good >= REQ || st.s >= N;
    while (__ballot(!done) != 0ull) {
        const uint32_t s = st.s + (uint32_t)(lane - gbase);
        const bool mine = !done && s < N;
        // the last applied writer of this sample, if any
        int w = -1;
        for (uint32_t m = done ? 0u : applied; __ballot(m != 0u) != 0ull; m &= m - 1u) {
            const int i = m ? __builtin_ctz(m) : 0;
            const uint32_t si = (uint32_t)__shfl((int)slot, gbase + i, 64);
            if (m != 0u && si == s) w = i;
        }
        bool match = false;
        uint32_t td = 0, ts = 0;
        if (mine) {
            uint64_t ra;
            uint32_t rb;
            if (w >= 0) raw_current<C>(v, frame, (uint32_t)((y + pred_dy((uint32_t)w)) * v.W + x + pred_dx((uint32_t)w)), ra, rb);
            else fetch_raw<C>(v, s, p, ra, rb);
            uint32_t col[C], desc[C];
            decode_raw<C>(ra, rb, col, desc);
            match = test_sample<C, ALGO, 0>(px, lut, col, desc, td, ts);
        }
        // matches in sample order (few: at most REQ are taken)
        uint32_t bits = done ? 0u : (uint32_t)(__ballot(match) >> gbase) & ((1u << kGroup) - 1u);
        const uint32_t dist = td << 16 | ts;
        while (__ballot(bits != 0u) != 0ull) {
            const int i = bits ? __builtin_ctz(bits) : 0;
            const uint32_t d = (uint32_t)__shfl((int)dist, gbase + i, 64);
            if (bits) {
                bits &= bits - 1u;
                const uint32_t a = d >> 16, b = d & 0xFFFFu;
                st.md = a < st.md ? a : st.md;
                st.ms = b < st.ms ? b : st.ms;
                if (++st.good == REQ) {
                    st.s += (uint32_t)i + 1u;
                    bits = 0;
                    done = true;
                }
            }
        }
        if (!done) {
            st.s = st.s + kGroup < N ? st.s + kGroup : N;
            done = st.s >= N;
        }
    }
}

// the match context of the group's pixel from global memory: lane 4c+w packs tap word w of channel c
template <int C, int ALGO>
LV_D void group_ctx(const View& v, const uint8_t* frame, int x, int y, bool active, GroupLds& L, PxCtx<C>& px) {
    const uint32_t sub = threadIdx.x & (kGroup - 1), g = threadIdx.x / kGroup, p = (uint32_t)(y * v.W + x);
    if (active && sub < 4u * C) {
        const uint32_t w = sub & 3u, c = sub >> 2;
        // (dx + 2) | (dy + 2) << 4 of taps 4w .. 4w+3, one byte each
        constexpr auto code = [](int n) { return (uint32_t)((kLbspDX[n] + 2) | ((kLbspDY[n] + 2) << 4)); };
        constexpr auto codes = [code](int a) {
            return code(a) | code(a + 1) << 8 | code(a + 2) << 16 | code(a + 3) << 24;
        };
        constexpr uint32_t k0 = codes(0), k1 = codes(4), k2 = codes(8), k3 = codes(12);
        const uint32_t ks = w == 0u ? k0 : w == 1u ? k1 : w == 2u ? k2 : k3;
        uint32_t acc = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int dx = (int)((ks >> (8 * k)) & 15u) - 2, dy = (int)((ks >> (8 * k + 4)) & 15u) - 2;
            acc |= (uint32_t)*at(frame, ((y + dy) * v.W + (x + dx)) * C + c) << (8 * k);
        }
        L.taps[g][sub] = acc;
    }
    if (active) {
#pragma unroll
        for (int c = 0; c < C; ++c) {
            px.cur[c] = *at(frame, p * C + c);
            px.intra[c] = *at(v.desc_cur, p * C + c);
        }
        if constexpr (ALGO == kSuBSENSE) subsense_thresholds<C>(v, *at(v.R, p), *at(v.unstable, p), px);
        else lobster_thresholds<C>(v, px);
    }
    wave_sync();
#pragma unroll
    for (int c = 0; c < C; ++c)
#pragma unroll
        for (int w = 0; w < 4; ++w) px.taps[c][w] = L.taps[g][4 * c + w];
    wave_sync();  // read before the group's next pixel overwrites them
}

// ----------------------------------------------------------------------------------------------
// speculative match: raster-earlier writers assumed to decide as in the previous frame
// ----------------------------------------------------------------------------------------------
struct PredTile;
template <int C, int ALGO, int KF>
LV_D bool match_pixel(const View& v, const uint8_t* frame, const LbspLimits* lut, const FrameTile<C>& tile,
                      const PredTile& pred, const PxIn<C>& in, int lx, int ly, int x, int y, uint32_t p,
                      uint32_t seq_limit, uint32_t& examined, PxCtx<C>& px, bool& push, uint32_t& target);

// Records of the raster-earlier part of a tile's 5x5 neighbourhood (rows y0-2 .. y0+TH-1, columns x0-2 ..
// x0+TW+1) with the guess (background in the previous frame) and the forward gate folded into free bits, so
// that an applied writer is one masked compare.
struct PredTile {
    static constexpr int LW = TW + 4, LH = TH + 2;
    uint32_t rec[LH][LW];
};

LV_D void load_pred_tile(PredTile& t, const View& v, int x0, int y0) {
    auto put = [&](int r, int c) {
        const int gx = x0 + c - 2, gy = y0 + r - 2;
        uint32_t w = kRecNone;
        if (gx >= 0 && gx < v.W && gy >= 0 && gy < v.H) {
            const uint32_t q = (uint32_t)(gy * v.W + gx);
            w = *at(v.rec, q);
            w |= (*at(v.last_raw, q) == 0 ? kRecBg : 0u) | (fwd_gate(w) ? kRecFwd : 0u);
        }
        t.rec[r][c] = w;
    };
    const int lx = (int)threadIdx.x % TW, ly = (int)threadIdx.x / TW;
    put(ly, lx);
    if (ly < PredTile::LH - TH) put(ly + TH, lx);
    else if (threadIdx.x >= TPB - 4u * PredTile::LH)  // the last columns, by the threads without a second row
        put((TPB - 1 - (int)threadIdx.x) / 4, TW + (int)threadIdx.x % 4);
}

// candidate writers of tile-local pixel (lx,ly) whose guessed decision is background
LV_D uint32_t applied_writers_tile(const PredTile& t, int lx, int ly) {
    uint32_t m = 0;
#pragma unroll
    for (int i = 0; i < 12; ++i) {
        const uint32_t r = t.rec[ly + 2 + kPredDY[i]][lx + 2 + kPredDX[i]];
        const uint32_t code = (uint32_t)((2 - kPredDY[i]) * 5 + (2 - kPredDX[i]));
        m |= (r & (31u | kRecBg | kRecFwd)) == (code | kRecBg | kRecFwd) ? 1u << i : 0u;
    }
    return m;
}

// LDS of the phase-A match for frames of up to CMAX channels. A batch kernel instantiates the match
// for both channel counts and calls both with CMAX = 3, so they share one allocation (separate
// arrays per instantiation would cost ~5 KB of LDS and an occupancy level).
template <int CMAX>
struct MatchLds {
    union {
        FrameTile<CMAX> big;
        FrameTile<1> c1;
    } tile;
    PredTile pred;
    alignas(8) LbspLimits lut[256];
};

template <int CMAX>
LV_D MatchLds<CMAX>& match_lds() {
    __shared__ MatchLds<CMAX> m;
    return m;
}

template <int C, int CMAX>
LV_D FrameTile<C>& tile_of(MatchLds<CMAX>& m) {
    if constexpr (C == CMAX) return m.tile.big;
    else return m.tile.c1;
}

template <int C, int ALGO, int KF, int CMAX = C>
LV_D void match_body(const View& v, uint32_t bid, uint32_t nblk) {
    static_assert(C == CMAX || C == 1, "a match instantiation shares the LDS of CMAX channels");
    const uint8_t* frame = v.frame;
    const uint32_t seq_limit = v.seq_limit;
    MatchLds<CMAX>& L = match_lds<CMAX>();
    FrameTile<C>& tile = tile_of<C>(L);
    PredTile& pred = L.pred;
    LbspLimits* lut = L.lut;
    const int ntx = (v.W + TW - 1) / TW;
    const int x0 = ((int)bid % ntx) * TW, y0 = ((int)bid / ntx) * TH;
    // The tile's pixels stay with their threads: the scan is cut after a few samples, so foreground pixels
    // cost a wavefront little, and gathering them into shared wavefronts (two barriers, the inputs through LDS)
    // no longer pays (1391 -> 1344 us for a batch of 64 without it, 250 -> 240 us at 3840x2160).
    const int lx = (int)threadIdx.x % TW, ly = (int)threadIdx.x / TW, x = x0 + lx, y = y0 + ly;
    const bool inside = x < v.W && y < v.H;
    const uint32_t p = (uint32_t)(y * v.W + x);
    const PxIn<C> in = load_px_in<C, ALGO>(v, inside ? p : 0u, inside);
    load_frame_tile<C>(tile, frame, v.W, v.H, x0, y0);
    load_pred_tile(pred, v, x0, y0);
    load_lut(lut, v.sc);
    __syncthreads();
    uint32_t examined = 0;
    bool cont = false, push = false;
    uint32_t target = 0;
    PxCtx<C> px{};
    if (in.roi())
        cont = !match_pixel<C, ALGO, KF>(v, frame, lut, tile, pred, in, lx, ly, x, y, p, seq_limit, examined, px, push,
                                         target);
    // unfinished pixels go to the continuation with their context: one atomic per wavefront, on
    // this tile's stripe of the list (at most cont_region entries reach one stripe)
    const uint32_t k = bid % (uint32_t)kContStripes;
    push_first(v, push, target, k);
    const unsigned long long bal = __ballot(cont);
    if (bal) {
        const int lane = (int)(threadIdx.x & 63u), leader = __ffsll((long long)bal) - 1;
        uint32_t base = 0;
        if (lane == leader) base = atomicAdd(&v.sc->cont_cnt[k * kContStride], (uint32_t)__popcll(bal));
        base = (uint32_t)__shfl((int)base, leader, 64);
        const uint32_t j = base + (uint32_t)__popcll(bal & ((1ull << lane) - 1ull));
        if (cont) {
            G(v.cont)[(size_t)k * v.cont_region + j] = p;
            if (j < v.cont_ctx_region)
                store_ctx<C>(v.cont_ctx + ((size_t)k * v.cont_ctx_region + j) * kCtxWords, px);
        }
    }
    block_add<TPB>(examined, v.sc->spec_part);
}

// Phase A: sequential scan of at most v_seq_limit samples. Returns true when the pixel is final;
// otherwise its partial state is left in mres for phase B.
template <int C, int ALGO, int KF>
LV_D bool match_pixel(const View& v, const uint8_t* frame, const LbspLimits* lut, const FrameTile<C>& tile,
                      const PredTile& pred, const PxIn<C>& in, int lx, int ly, int x, int y, uint32_t p,
                      uint32_t seq_limit, uint32_t& examined, PxCtx<C>& px, bool& push, uint32_t& target) {
    // guess: raster-earlier writers decide as in the previous frame
    const uint32_t applied = applied_writers_tile(pred, lx, ly);
    uint64_t sbm;
    int nrep;
    ScanState st = scan_init<C>();
    const uint32_t N = (uint32_t)v.N;
    // more than kRepl overwritten slots (very rare): the pixel keeps its guess for now and goes to the first
    // fix-point worklist itself, where a group matches it against any number of writers.
    // The replacements are gathered before the context is built, so the two are not live together.
    auto rec_of = [&](int i) { return pred.rec[ly + 2 + pred_dy((uint32_t)i)][lx + 2 + pred_dx((uint32_t)i)]; };
    auto colour_of = [&](int i, uint32_t) { return tile_colour(tile, lx + 2 + pred_dx((uint32_t)i), ly + 2 + pred_dy((uint32_t)i)); };
    const uint32_t own = pred.rec[ly + 2][lx + 2];
    const uint8_t guess = (own & kRecBg) ? 0 : 1;
    const bool fits = build_repl<C>(v, x, y, applied, sbm, nrep, rec_of, colour_of);
    const uint32_t limit = !fits ? 0u : seq_limit < N ? seq_limit : N;
    build_ctx_staged<C, ALGO>(v, tile, lx, ly, in, px);
    scan_seq<C, ALGO, 1, KF>(v, lut, px, x, y, sbm, nrep, st, limit);
    examined = st.s;
    *at(v.mres, p) = pack_state(st);
    if (fits && st.good < (uint32_t)v.REQ && st.s < N) return false;
    const uint8_t fg = !fits ? guess : st.good < (uint32_t)v.REQ ? 1 : 0;
    *at(v.dec, p) = fg;
    push = fg != guess && forward_target(v, own, x, y, target);
    if (!fits) {
        push = true;
        target = p;
    }
    return true;
}

// candidate writers of p that were background in the previous frame, by one lane
LV_D uint32_t applied_writers_global(const View& v, int x, int y) {
    uint32_t m = 0;
#pragma unroll
    for (int i = 0; i < 12; ++i) {
        const uint32_t q = (uint32_t)((y + kPredDY[i]) * v.W + (x + kPredDX[i]));
        const uint32_t r = *at(v.rec, q);
        const uint32_t code = (uint32_t)((2 - kPredDY[i]) * 5 + (2 - kPredDX[i]));
        if (rec_tgt(r) == code && fwd_gate(r)) m |= 1u << i;
    }
    uint32_t applied = 0;
    for (; m; m &= m - 1) {
        const int i = __builtin_ctz(m);
        const uint32_t q = (uint32_t)((y + pred_dy((uint32_t)i)) * v.W + (x + pred_dx((uint32_t)i)));
        if (*at(v.last_raw, q) == 0) applied |= 1u << i;
    }
    return applied;
}

// decision of a finished scan: match result, raw decision; true when the decision differs from the
// speculative guess and the pixel has a forward target (for the first fix-point worklist)
template <int C>
LV_D bool finish_pixel(const View& v, uint32_t p, int x, int y, const ScanState& st, uint32_t& t) {
    *at(v.mres, p) = pack_state(st);
    const uint8_t fg = st.good < (uint32_t)v.REQ ? 1 : 0;
    *at(v.dec, p) = fg;
    const uint8_t guess = *at(v.last_raw, p) ? 1 : 0;
    return fg != guess && forward_target(v, *at(v.rec, p), x, y, t);
}

// push_first for lanes of different stripes: one append per stripe present in the wavefront
LV_D void push_first_mixed(const View& v, bool push, uint32_t t, uint32_t stripe) {
    unsigned long long bal = __ballot(push);
    while (bal) {
        const uint32_t s0 = (uint32_t)__shfl((int)stripe, __ffsll((long long)bal) - 1, 64);
        const bool mine = push && stripe == s0;
        push_first(v, mine, t, s0);
        bal &= ~__ballot(mine);
    }
}

// Phase B continues the scans phase A cut, over the dense list of unfinished pixels (its stripes walked in
// order), with the context phase A cached (rebuilt from global memory past a stripe's cache).
// Two forms, chosen by the length of the list: a group per pixel up to View::group_limit entries, where a
// lane per pixel leaves most of the chip idle behind chains of 13 dependent loads (it holds 20 K groups at once at
// this kernel's occupancy of 5: 256 CUs x 20 wavefronts x 4). Past it a lane per pixel does the same work with fewer
// instructions. Both sides are measured at kGroupLimit.
template <int C, int ALGO, int KF>
LV_D void match_seq_lanes(const View& v, const LbspLimits* lut, const uint32_t* s_pre, uint32_t n, uint32_t bid,
                          uint32_t nblk) {
    const uint8_t* frame = v.frame;
    uint32_t examined = 0;
    for (uint32_t i = bid * TPB + threadIdx.x; i < n; i += nblk * TPB) {
        const uint32_t k = stripe_of(s_pre, i);  // item i = entry j of stripe k
        const uint32_t j = i - s_pre[k];
        const uint32_t p = G(v.cont)[(size_t)k * v.cont_region + j];
        const int x = (int)(p % (uint32_t)v.W), y = (int)(p / (uint32_t)v.W);
        PxCtx<C> px;
        if (j < v.cont_ctx_region) load_ctx<C>(v.cont_ctx + ((size_t)k * v.cont_ctx_region + j) * kCtxWords, px);
        else build_ctx_global<C, ALGO>(v, frame, x, y, px);
        const uint32_t applied = applied_writers_global(v, x, y);
        uint64_t sbm;
        int nrep;
        auto rec_of = [&](int i) { return *at(v.rec, (y + pred_dy((uint32_t)i)) * v.W + (x + pred_dx((uint32_t)i))); };
        auto colour_of = [&](int, uint32_t q) { return load_colour<C>(frame, q); };
        // at most kRepl slots: phase A keeps the others (same writers, same guesses)
        (void)build_repl<C>(v, x, y, applied, sbm, nrep, rec_of, colour_of);
        ScanState st = unpack_state(*at(v.mres, p));
        const uint32_t s0 = st.s;
        scan_seq<C, ALGO, 0, KF>(v, lut, px, x, y, sbm, nrep, st, (uint32_t)v.N);
        examined += st.s - s0;
        uint32_t t = 0;
        const bool push = finish_pixel<C>(v, p, x, y, st, t);
        push_first_mixed(v, push, t, k);
    }
    block_add<TPB>(examined, v.sc->coop_part);
}

template <int C, int ALGO>
LV_D void match_seq_groups(const View& v, const LbspLimits* lut, const uint32_t* s_pre, uint32_t n, uint32_t bid,
                           uint32_t nblk) {
    const uint8_t* frame = v.frame;
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t step = nblk * (TPB / kGroup);
    uint32_t examined = 0;
    for (uint32_t i0 = (bid * TPB + (threadIdx.x & ~63u)) / kGroup; i0 < n; i0 += step) {  // uniform per wavefront
        const uint32_t i = i0 + lane / kGroup;
        const bool active = i < n;
        uint32_t k = 0, p = 0;
        PxCtx<C> px{};
        ScanState st = scan_init<C>();
        int x = 0, y = 0;
        if (active) {
            k = stripe_of(s_pre, i);
            const uint32_t j = i - s_pre[k];
            p = G(v.cont)[(size_t)k * v.cont_region + j];
            x = (int)(p % (uint32_t)v.W);
            y = (int)(p / (uint32_t)v.W);
            if (j < v.cont_ctx_region) load_ctx<C>(v.cont_ctx + ((size_t)k * v.cont_ctx_region + j) * kCtxWords, px);
            else build_ctx_global<C, ALGO>(v, frame, x, y, px);
            st = unpack_state(*at(v.mres, p));
        }
        uint32_t slot;
        bool turned;
        const uint32_t applied = group_writers<false>(v, x, y, active, slot, 0u, turned);
        const uint32_t s0 = st.s;
        scan_group<C, ALGO>(v, frame, lut, px, x, y, applied, slot, st, active);
        bool push = false;
        uint32_t t = 0;
        if (active && lane % kGroup == 0) {
            examined += st.s - s0;
            push = finish_pixel<C>(v, p, x, y, st, t);
        }
        push_first_mixed(v, push, t, k);
    }
    block_add<TPB>(examined, v.sc->coop_part);
}

template <int C, int ALGO, int KF>
LV_D void match_seq_body(const View& v, uint32_t bid, uint32_t nblk) {
    __shared__ alignas(8) LbspLimits lut[256];
    __shared__ uint32_t s_pre[kContStripes + 1];  // exclusive prefix of the stripe counts
    stripe_prefix(v.sc->cont_cnt, s_pre);
    load_lut(lut, v.sc);
    __syncthreads();
    const uint32_t n = s_pre[kContStripes];
    const bool groups = n <= v.group_limit;
    if (bid * (groups ? TPB / kGroup : TPB) >= n) return;  // uniform: no item reaches this block
    if (groups) match_seq_groups<C, ALGO>(v, lut, s_pre, n, bid, nblk);
    else match_seq_lanes<C, ALGO, KF>(v, lut, s_pre, n, bid, nblk);
}

// worklist of fix-point iteration k: entry i, and its entry count for every thread of the block (pre:
// the block's LDS, kContStripes + 1 words, holding the stripes' prefix of iteration 1; the block
// synchronizes in here)
LV_D uint32_t wl_item(const View& v, uint32_t k, const uint32_t* pre, uint32_t i) {
    if (k != 1u) return ((k & 1u) ? v.wl1 : v.wl0)[i];
    const uint32_t s = stripe_of(pre, i);
    return v.wl1[(size_t)s * v.cont_region + (i - pre[s])];
}
LV_D uint32_t wl_total(const View& v, uint32_t k, uint32_t* pre) {
    if (k != 1u)
        return __hip_atomic_load(&v.sc->wl_count[k % kWlRing], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    stripe_prefix(v.sc->wl_first, pre);
    __syncthreads();
    return pre[kContStripes];
}

// result of a fix-point re-match; true when the decision changed and the pixel has a forward target
LV_D bool rematch_done(const View& v, uint32_t p, int x, int y, const ScanState& st, uint32_t& t) {
    *at(v.mres, p) = pack_state(st);
    const uint8_t fg = st.good < (uint32_t)v.REQ ? 1 : 0;
    if (fg == *at(v.dec, p)) return false;
    __hip_atomic_store(&v.dec[p], fg, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return forward_target(v, *at(v.rec, p), x, y, t);
}

// Fix-point re-match of a wavefront's worklisted pixels i0 .. i0 + 64/kGroup - 1, one group each. In iteration 1
// a pixel whose wrongly guessed writers all write slots that its speculative scan never reached keeps its
// result (a background pixel examines 2 to 5 of 50 samples, so nine in ten do): only the records and decisions
// around it are read. A writer that turns later pushes the pixel again, and later iterations match in full.
template <int C, int ALGO>
LV_D void rematch(const View& v, const LbspLimits* lut, GroupLds& L, const uint32_t* pre, uint32_t n, uint32_t i0,
                  uint32_t k, uint32_t* wl_next) {
    const uint8_t* frame = v.frame;
    const uint32_t lane = threadIdx.x & 63u, i = i0 + lane / kGroup;
    bool active = i < n;
    const uint32_t p = active ? wl_item(v, k, pre, i) : 0u;
    const int x = (int)(p % (uint32_t)v.W), y = (int)(p / (uint32_t)v.W);
    // samples its result rests on; 0 = not matched yet
    const uint32_t seen = active && k == 1u ? *at(v.mres, p) >> 24 : 0u;
    uint32_t slot;
    bool turned;
    const uint32_t applied = group_writers<true>(v, x, y, active, slot, seen, turned);
    active = active && (seen == 0u || turned);
    if (__ballot(active) == 0ull) return;
    PxCtx<C> px{};
    group_ctx<C, ALGO>(v, frame, x, y, active, L, px);
    ScanState st = scan_init<C>();
    scan_group<C, ALGO>(v, frame, lut, px, x, y, applied, slot, st, active);
    bool push = false;
    uint32_t t = 0;
    if (active && lane % kGroup == 0) push = rematch_done(v, p, x, y, st, t);
    push_next(v, push, t, k + 1u, wl_next);
}

// fix-point iterations from k0 on in one workgroup (normally no work is left)
template <int C, int ALGO>
LV_D void fixpoint_tail(const View& v, const LbspLimits* lut, GroupLds& L, uint32_t* s_pre, uint32_t k0, uint32_t cap) {
    __shared__ uint32_t s_n;
    for (uint32_t k = k0;; ++k) {
        __syncthreads();
        const uint32_t total = wl_total(v, k, s_pre);
        if (threadIdx.x == 0) {
            s_n = total;
            if (s_n != 0) {
                if (k - k0 >= cap) {
                    atomicOr(&v.sc->err_flags, kErrFixpointCap);
                    __hip_atomic_store(v.h_err, kErrFixpointCap, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                    s_n = 0;
                } else {
                    __hip_atomic_store(&v.sc->wl_count[(k + 2) % kWlRing], 0u, __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
                    atomicAdd(&v.sc->iters, 1u);
                    atomicMax(&v.sc->max_iter_seen, k);
                    if (k < 8) v.sc->wl_work[k] = s_n;
                }
            }
        }
        __syncthreads();
        const uint32_t n = s_n;
        if (n == 0) break;
        uint32_t* wl_next = (k & 1u) ? v.wl0 : v.wl1;
        for (uint32_t i0 = (threadIdx.x & ~63u) / kGroup; i0 < n; i0 += TPB / kGroup)
            rematch<C, ALGO>(v, lut, L, s_pre, n, i0, k, wl_next);
        __threadfence();
    }
}

// Fix-point iteration k: worklist k -> worklist k+1 (k >= 1). LAST: the block that finishes last goes on with
// the iterations left (fixpoint_tail): blocks with work count themselves when done, behind a
// device-scope fence; nobody waits for another block. Batches end with a launch of one block per
// stream instead (TAIL): there the fences of thousands of blocks cost more (151 us) than the launch (20 us).
enum FixKind : int { kFixMore, kFixLast, kFixTail };
template <int C, int ALGO, int KIND>
LV_D void fixpoint_body(const View& v, uint32_t bid, uint32_t nblk, uint32_t k, uint32_t cap) {
    __shared__ alignas(8) LbspLimits lut[256];
    __shared__ GroupLds L;
    __shared__ uint32_t s_pre[kContStripes + 1];
    if constexpr (KIND == kFixTail) {
        load_lut(lut, v.sc);
        fixpoint_tail<C, ALGO>(v, lut, L, s_pre, k, cap);
    } else {
        // slot k+2 was last read by iteration k-2 (finished); it must be empty before iteration k+1
        // pushes into it, whether or not this iteration has work.
        if (bid == 0 && threadIdx.x == 0)
            __hip_atomic_store(&v.sc->wl_count[(k + 2) % kWlRing], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const uint32_t n = wl_total(v, k, s_pre);
        if (n == 0) return;
        if (bid == 0 && threadIdx.x == 0) {
            atomicAdd(&v.sc->iters, 1u);
            atomicMax(&v.sc->max_iter_seen, k);
            if (k < 8) v.sc->wl_work[k] = n;
        }
        constexpr uint32_t kPerBlock = TPB / kGroup;
        if (bid * kPerBlock >= n) return;  // uniform: no item reaches this block
        load_lut(lut, v.sc);
        __syncthreads();
        uint32_t* wl_next = (k & 1u) ? v.wl0 : v.wl1;
        for (uint32_t i0 = (bid * TPB + (threadIdx.x & ~63u)) / kGroup; i0 < n; i0 += nblk * kPerBlock)
            rematch<C, ALGO>(v, lut, L, s_pre, n, i0, k, wl_next);
        if constexpr (KIND == kFixLast) {
            __shared__ uint32_t s_done;
            const uint32_t blocks = (n + kPerBlock - 1) / kPerBlock, nwork = blocks < nblk ? blocks : nblk;
            __threadfence();
            __syncthreads();
            // the counter wraps back to zero with the last block
            if (threadIdx.x == 0) s_done = atomicInc(&v.sc->fix_done, nwork - 1u);
            __syncthreads();
            if (s_done != nwork - 1u) return;
            __threadfence();
            fixpoint_tail<C, ALGO>(v, lut, L, s_pre, k + 1u, cap);
        }
    }
}

// ----------------------------------------------------------------------------------------------
// SuBSENSE feedback maps (SUB:396-420, :451-480; 1ch :254-329), raw mask and blink bookkeeping
// (SUB:536-539). Whole image: pixels outside the ROI get raw = 0.
// ----------------------------------------------------------------------------------------------
// v / n as the IEEE quotient, from the correctly rounded reciprocal inv = 1 / n with one residual correction:
// equal to the division for every whole v < 2^16 and whole n <= 255 as well as 765 (checked exhaustively),
// three operations where the division takes about ten
LV_HD float quot(float v, float n, float inv) {
    const float q = v * inv;
    return __builtin_fmaf(__builtin_fmaf(-q, n, v), inv, q);
}

// A pixel's state of the previous frame, loaded ahead of the tile barrier. The last colour and descriptor are
// read as one and two words (a byte or two past them lies in the same allocation).
template <int C>
struct PxState {
    uint32_t last_color, last_desc[C == 3 ? 2 : 1];
    float mld, dlt, dst, rlt, rst, T, V, R;
    uint32_t mres;
    uint8_t roi, last_fg, blinks, last_raw, last_raw_blink;
};
template <int C>
LV_D void load_px_state(const View& v, uint32_t p, PxState<C>& s) {
    s.roi = *at(v.roi, p);
    s.mres = *at(v.mres, p);
    if constexpr (C == 3) {
        s.last_color = peek<UnalignedU32>(v.last_color, 3u * p);
        s.last_desc[0] = peek<UnalignedU32>(v.last_desc, 6u * p);
        s.last_desc[1 % (C == 3 ? 2 : 1)] = peek<UnalignedU16>(v.last_desc, 6u * p + 4u);
    } else {
        s.last_color = *at(v.last_color, p);
        s.last_desc[0] = *at(v.last_desc, p);
    }
    s.mld = *at(v.MLD, p);
    s.dlt = *at(v.DminLT, p);
    s.dst = *at(v.DminST, p);
    s.rlt = *at(v.RawLT, p);
    s.rst = *at(v.RawST, p);
    s.T = *at(v.T, p);
    s.V = *at(v.V, p);
    s.R = *at(v.R, p);
    s.last_fg = *at(v.last_fg, p);
    s.blinks = *at(v.blinks, p);
    s.last_raw = *at(v.last_raw, p);
    s.last_raw_blink = *at(v.last_raw_blink, p);
}

template <int C>
LV_D void store_last(const View& v, uint32_t p, const uint32_t cur[C], const uint32_t intra[C]) {
    if constexpr (C == 3) {
        poke<UnalignedU16>(v.last_color, 3u * p, (uint16_t)(cur[0] | cur[1] << 8));
        *at(v.last_color, 3u * p + 2u) = (uint8_t)cur[2 % C];
        poke<UnalignedU32>(v.last_desc, 6u * p, intra[0] | intra[1 % C] << 16);
        poke<UnalignedU16>(v.last_desc, 6u * p + 4u, (uint16_t)intra[2 % C]);
    } else {
        *at(v.last_color, p) = (uint8_t)cur[0];
        *at(v.last_desc, p) = (uint16_t)intra[0];
    }
}

// One pixel (p < npx) with its current colour, descriptor, record and decision. Returns p's samples examined
// (k_p); s.rst and s.mld become the updated values the model update's ghost test reads.
template <int C>
LV_D uint32_t feedback_pixel(const View& v, uint32_t p, PxState<C>& s, const uint32_t cur[C], const uint32_t intra[C],
                             bool unstable, bool fg) {
    uint32_t examined = 0;
    uint8_t raw = 0;
    if (s.roi) {
        const uint32_t frame_no = cur_frame(v);
        const uint32_t mvn = v.mv_avgs;
        const float aLT = 1.0f / (float)(frame_no < mvn ? frame_no : mvn);
        const float aST = 1.0f / (float)(frame_no < mvn / 4u ? frame_no : mvn / 4u);
        const uint32_t good = s.mres & 255u, md = (s.mres >> 8) & 63u, ms = (s.mres >> 14) & 1023u;
        examined = s.mres >> 24;
        constexpr float col_max = (float)(C * 255), desc_max = (float)(C * 16);
        constexpr float inv_col = 1.0f / col_max, inv_desc = 1.0f / desc_max;
        // D_last (SUB:396-397): L1dist<3> accumulates in uchar (wraps mod 256)
        uint32_t l1 = 0, hd = 0;
#pragma unroll
        for (int c = 0; c < C; ++c) {
            l1 = __builtin_amdgcn_sad_u8((s.last_color >> (8 * c)) & 255u, cur[c], l1);
            hd += popc(((s.last_desc[c / 2] >> (16 * (c & 1))) & 0xFFFFu) ^ intra[c]);
        }
        l1 &= 255u;
        const float nld = (quot((float)l1, col_max, inv_col) + quot((float)hd, desc_max, inv_desc)) / 2.0f;
        const float mld = s.mld * (1.0f - aST) + nld * aST;
        *at(v.MLD, p) = mld;
        float dlt = s.dlt, dst = s.dst, rlt = s.rlt, rst = s.rst;
        const uint32_t REQ = (uint32_t)v.REQ;
        float nmd = (quot((float)ms, col_max, inv_col) + quot((float)md, desc_max, inv_desc)) / 2.0f;
        if (fg) {
            nmd = fmin_ref(1.0f, nmd + (float)(REQ - good) / (float)REQ);
            raw = 255;
        }
        dlt = dlt * (1.0f - aLT) + nmd * aLT;
        dst = dst * (1.0f - aST) + nmd * aST;
        rlt = rlt * (1.0f - aLT);
        rst = rst * (1.0f - aST);
        if (fg) {
            rlt = rlt + aLT;
            rst = rst + aST;
        }
        *at(v.DminLT, p) = dlt;
        *at(v.DminST, p) = dst;
        store_changed(v.RawLT, p, rlt, s.rlt);
        store_changed(v.RawST, p, rst, s.rst);
        s.rst = rst;
        s.mld = mld;
        const float lcap = v.sc->lower_cap, ucap = v.sc->upper_cap;
        const float mn = fmin_ref(dlt, dst), mx = fmax_ref(dlt, dst);
        const bool last_fg = s.last_fg != 0;
        float T = s.T, V = s.V, R = s.R;
        // T += 0.5 / (mx * V) or T -= 0.25 * V / mx, one division for both
        const bool up = last_fg || (mn < 0.1f && raw);
        const float step = (up ? 0.5f : 0.25f * V) / (up ? mx * V : mx);
        if (up) {
            if (T < ucap) T += step;
        } else if (T > lcap) {
            T -= step;
        }
        if (T < lcap) T = lcap;
        else if (T > ucap) T = ucap;
        if (mx > 0.1f && s.blinks) {
            V += 1.0f;
        } else if (V > 0.1f) {
            V -= last_fg ? 0.1f / 4 : unstable ? 0.1f / 2 : 0.1f;
            if (V < 0.1f) V = 0.1f;
        }
        const float base = 1.0f + mn * 2.0f;
        if ((double)R < (double)base * (double)base) {  // std::pow(float,2) in double: an exact square
            R += 0.01f * (V - 0.1f);
        } else {
            R -= 0.01f / V;
            if (R < 1.0f) R = 1.0f;
        }
        store_changed(v.T, p, T, s.T);
        store_changed(v.V, p, V, s.V);
        store_changed(v.R, p, R, s.R);
        *at(v.unstable, p) = (uint8_t)unstable;
        store_last<C>(v, p, cur, intra);
    }
    const uint8_t cb = raw ^ s.last_raw;
    store_changed(v.blinks, p, (uint8_t)(cb | s.last_raw_blink), s.blinks);
    store_changed(v.last_raw_blink, p, cb, s.last_raw_blink);
    store_changed(v.last_raw, p, raw, s.last_raw);  // this frame's raw mask from here on
    return examined;
}

// ----------------------------------------------------------------------------------------------
// model update: every pixel of the inner rectangle gathers the writes aimed at its samples, in
// the raster order of the writers; the last write of each slot wins (SUB:406-449, LOB:498-512).
// ----------------------------------------------------------------------------------------------
// The tile's 5x5 neighbourhood in LDS, a wavefront per row: records with the tests of a write folded into their
// free bits (a writer is then one masked compare instead of two reads and four tests), and the writers' current
// colours and intra descriptors (the values they write) as the rows' bytes.
template <int C>
struct UpdateTile {
    static constexpr int LW = TW + 4, LH = TH + 4;
    static constexpr int DW = LW * 2 * C / 4;  // words of a descriptor row
    uint32_t rec[LH][LW];
    uint32_t desc[LH][DW];
    FrameTile<C> px;
};

// SuBSENSE: the feedback maps of the thread's pixel are updated in the same pass (they depend on the pixel
// alone), and the ghost test uses the new values from registers. LOBSTER: the raw mask (LOB:496-497,
// :554-555) and the last colour frame (LOB:580) are written in the same pass.
template <int C, int ALGO>
LV_D void update_body(const View& v, uint32_t bid, uint32_t nblk) {
    using Tile = UpdateTile<C>;
    __shared__ Tile t;
    constexpr int LW = Tile::LW, LH = Tile::LH, DW = Tile::DW;
    const int ntx = (v.W + TW - 1) / TW;
    const int x0 = ((int)bid % ntx) * TW, y0 = ((int)bid / ntx) * TH;
    const int lx = (int)threadIdx.x % TW, ly = (int)threadIdx.x / TW, x = x0 + lx, y = y0 + ly;
    const bool inside = x < v.W && y < v.H;
    const uint32_t p = inside ? (uint32_t)(y * v.W + x) : 0u;
    auto stage_rec = [&](int r, int c) {
        const int gx = x0 + c - 2, gy = y0 + r - 2;
        uint32_t w = kRecNone;
        if (gx >= 0 && gx < v.W && gy >= 0 && gy < v.H) {
            const uint32_t q = (uint32_t)(gy * v.W + gx);
            w = *at(v.rec, q);
            w |= (*at(v.dec, q) == 0 ? kRecBg : 0u) | (fwd_gate(w) ? kRecFwd : 0u) |
                 (rec_gate_a(w) || rec_gate_b(w) ? kRecAny : 0u);
        }
        t.rec[r][c] = w;
    };
    const int total = (int)v.npx * 2 * C;
#pragma unroll
    for (int k = 0; k < LH / 4; ++k) {
        const int r = ly + 4 * k, gy = y0 + r - 2;
        stage_rec(r, lx);
#pragma unroll
        for (int j = 0; j < (DW + 63) / 64; ++j) {
            const int w = lx + 64 * j;
            if (w < DW)
                t.desc[r][w] = gy >= 0 && gy < v.H
                                   ? word_at((const uint8_t*)v.desc_cur, (gy * v.W + x0 - 2) * 2 * C + 4 * w, total)
                                   : 0u;
        }
    }
    if (threadIdx.x < 4 * LH) stage_rec((int)threadIdx.x / 4, TW + (int)threadIdx.x % 4);
    load_frame_tile<C>(t.px, v.frame, v.W, v.H, x0, y0);
    PxState<C> s;
    if constexpr (ALGO == kSuBSENSE) load_px_state<C>(v, p, s);
    __syncthreads();
    auto colour = [&](int hx, int hy, int c) { return (tile_colour(t.px, hx, hy) >> (8 * c)) & 255u; };
    auto descriptor = [&](int hx, int hy, int c) { return (uint32_t)((const uint16_t*)t.desc[hy])[hx * C + c]; };
    const uint32_t own = t.rec[ly + 2][lx + 2];
    const bool own_bg = (own & kRecBg) != 0;
    uint32_t nw = 0, examined = 0;
    bool ghost_new = false;  // writers at or after p read p's updated maps (SUB:438-441)
    if (inside) {
        uint32_t cur[C], intra[C];
#pragma unroll
        for (int c = 0; c < C; ++c) {
            cur[c] = colour(lx + 2, ly + 2, c);
            intra[c] = descriptor(lx + 2, ly + 2, c);
        }
        if constexpr (ALGO == kSuBSENSE) {
            examined = feedback_pixel<C>(v, p, s, cur, intra, rec_unstable(own), !own_bg);
            ghost_new = s.rst > 0.995f && s.mld < 0.010f;
        } else {
            const bool roi = rec_tgt(own) != kRecNone;
            *at(v.last_raw, p) = roi && !own_bg ? 255 : 0;
            if (roi) examined = *at(v.mres, p) >> 24;
#pragma unroll
            for (int c = 0; c < C; ++c) *at(v.last_color, p * C + c) = (uint8_t)cur[c];
        }
    }
    if (x >= 2 && y >= 2 && x < v.W - 2 && y < v.H - 2) {
        // Writes landing on p, as bits in sequential order: writer j of the 5x5 window (raster order), bit j
        // for j < 12 and j + 1 from 12 on; bit 12 is p's self update
        const uint32_t late = 31u | kRecBg | (ghost_new ? kRecAny : 1u << 5);
        constexpr uint32_t early = 31u | kRecBg | kRecFwd;
        uint32_t wm = 0;
#pragma unroll
        for (int j = 0; j < 25; ++j) {
            const int dy = j / 5 - 2, dx = j % 5 - 2;
            const uint32_t r = t.rec[ly + 2 + dy][lx + 2 + dx];
            const uint32_t code = (uint32_t)((2 - dy) * 5 + (2 - dx));
            const bool hit = j < 12 ? (r & early) == (code | kRecBg | kRecFwd) : ((r ^ ~31u) & late) == code;
            wm |= hit ? 1u << (j < 12 ? j : j + 1) : 0u;
        }
        if (rec_tgt(own) != kRecNone && (own_bg ? rec_self_bg(own) : (ALGO == kSuBSENSE && rec_self_fg(own)))) wm |= 1u << 12;
        nw = (uint32_t)popc(wm);
        // in sequential order: a later write to the same slot overwrites the earlier one, as stores of one
        // lane to one address do
        while (wm) {
            const int b = __builtin_ctz(wm);
            wm &= wm - 1u;
            const int j = b < 12 ? b : b == 12 ? 12 : b - 1;
            const int hy = ly + j / 5, hx = lx + j % 5;
            const uint32_t r = t.rec[hy][hx];
            const uint32_t sl = b == 12 ? rec_slot_self(r) : rec_slot_diff(r);
            uint32_t col[C], desc[C];
#pragma unroll
            for (int c = 0; c < C; ++c) {
                col[c] = colour(hx, hy, c);
                desc[c] = descriptor(hx, hy, c);
            }
            store_sample<C>(v, sl, p, col, desc);
        }
    }
    // workload counters: sample writes (w_p) and samples examined (k_p)
    const uint32_t sums[2] = {nw, examined};
    unsigned long long* const to[2] = {v.sc->wr_part, v.sc->ex_part};
    block_add<TPB, 2>(sums, to);
}

// ----------------------------------------------------------------------------------------------
// post-processing (SUB:540-554, LOB:578). Masks are 0/255 bytes.
// ----------------------------------------------------------------------------------------------
constexpr int PW = 64, PH = 16;  // post-processing tile; 256 threads x 4 pixels

// --- hole fill (SUB:540-543) on 64x64 zones, one wavefront per zone --------------------------
// PreFlood = morphologyEx(raw, CLOSE, 3x3) = erode3(dilate3(raw)) with neutral borders (SUB:540);
// holes = its 0-pixels not 4-connected through 0-pixels to pixel (0,0) (floodFill + bitwise_not,
// SUB:541-543). Lane y of a zone's wavefront holds row y of the zone as a 64-bit mask (bit x =
// column x). A zone's 0-pixels split into components that touch the zone border, numbered per
// zone, and components inside it, which are holes. The border components of all zones are joined
// across zone edges by union-find; a border component is outside iff its root is the root of the
// component holding pixel (0,0).
// Each kernel is bound by one wavefront's chain of rounds, not by memory, so a round's lane shifts are DPP moves
// and a zone row comes in four loads. Shifts through the LDS crossbar and byte loads with a ballot per row: the
// update launch that holds the closing at 320x240 26.9 -> 9.2 us; holes 10.1 -> 6.5 us at 3840x2160, and of 64
// mixed streams 20.6 -> 12.9 us.
constexpr int ZS = 64;                  // zone side
constexpr int ZPB = TPB / 64;           // zones per block, one per wavefront
constexpr uint32_t kZoneComps = 128;    // border components per zone (at most 126 of 252 pixels)

LV_D uint64_t brev64(uint64_t x) {
    return ((uint64_t)__builtin_bitreverse32((uint32_t)x) << 32) | __builtin_bitreverse32((uint32_t)(x >> 32));
}
LV_D uint64_t lane_bcast(uint64_t x, int l) {
    return ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(x >> 32), l) << 32) |
           (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)x, l);
}
// lane - N (SHR) or lane + N (SHL) within the rows of 16 lanes, `fill` past the row's end, as DPP moves: a shift
// through the LDS crossbar takes an order of magnitude longer, and a flood is a chain of them
template <int CTRL, int ROWS = 0xf>
LV_D uint64_t dpp64(uint64_t x, uint32_t fill) {
    const int lo = __builtin_amdgcn_update_dpp((int)fill, (int)(uint32_t)x, CTRL, ROWS, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp((int)fill, (int)(uint32_t)(x >> 32), CTRL, ROWS, 0xf, false);
    return ((uint64_t)(uint32_t)hi << 32) | (uint32_t)lo;
}
constexpr int kRowShr = 0x110, kRowShl = 0x100, kRowBcast15 = 0x142, kRowBcast31 = 0x143;

// What the column fills of a zone need of its pixels z (lane y holds row y), computed once per zone: products
// of z over the window each scan step covers. Down the rows: in-row shifts of 1, 2, 4, 8 lanes, then from the
// last lane of the row before (broadcast 15) and of the first half (broadcast 31). Up the rows: the same shifts
// the other way, then from the first lane of the row after, row by row.
struct ColumnWindows {
    uint64_t z, d1, d2, d4, d15, d31, u1, u2, u4, u[3];
};
LV_D ColumnWindows column_windows(uint64_t z, int lane) {
    ColumnWindows w;
    w.z = z;
    w.d1 = z & dpp64<kRowShr + 1>(z, ~0u);
    w.d2 = w.d1 & dpp64<kRowShr + 2>(w.d1, ~0u);
    w.d4 = w.d2 & dpp64<kRowShr + 4>(w.d2, ~0u);
    w.d15 = w.d4 & dpp64<kRowShr + 8>(w.d4, ~0u);  // from the row's first lane to this one
    w.d31 = w.d15 & dpp64<kRowBcast15, 0xa>(w.d15, ~0u);
    w.u1 = z & dpp64<kRowShl + 1>(z, ~0u);
    w.u2 = w.u1 & dpp64<kRowShl + 2>(w.u1, ~0u);
    w.u4 = w.u2 & dpp64<kRowShl + 4>(w.u2, ~0u);
    const uint64_t u15 = w.u4 & dpp64<kRowShl + 8>(w.u4, ~0u);  // from this lane to the row's last one
#pragma unroll
    for (int r = 0; r < 3; ++r) w.u[r] = (lane >> 4) == r ? u15 : 0ull;
    return w;
}

// the runs of z along the row that hold a bit of s (s within z). Adding s to z carries through
// the run above each seed bit and z & ~(z + s) keeps the bits the carry cleared; the same on the
// bit-reversed row covers the run below.
LV_D uint64_t fill_row(uint64_t z, uint64_t zr, uint64_t s) {
    const uint64_t up = (z & ~(z + s)) | s;
    const uint64_t ur = brev64(up);
    return brev64((zr & ~(zr + ur)) | ur);
}
// the runs of z down and up the columns that hold a bit of s: segmented OR scans over the lanes
LV_D uint64_t fill_cols(const ColumnWindows& w, uint64_t g) {
    g |= w.z & dpp64<kRowShr + 1>(g, 0u);
    g |= w.d1 & dpp64<kRowShr + 2>(g, 0u);
    g |= w.d2 & dpp64<kRowShr + 4>(g, 0u);
    g |= w.d4 & dpp64<kRowShr + 8>(g, 0u);
    g |= w.d15 & dpp64<kRowBcast15, 0xa>(g, 0u);
    g |= w.d31 & dpp64<kRowBcast31, 0xc>(g, 0u);
    g |= w.z & dpp64<kRowShl + 1>(g, 0u);
    g |= w.u1 & dpp64<kRowShl + 2>(g, 0u);
    g |= w.u2 & dpp64<kRowShl + 4>(g, 0u);
    g |= w.u4 & dpp64<kRowShl + 8>(g, 0u);
    g |= w.u[2] & lane_bcast(g, 48);
    g |= w.u[1] & lane_bcast(g, 32);
    g |= w.u[0] & lane_bcast(g, 16);
    return g;
}
// the 4-connected components of z holding a bit of s; each round adds at least one bit or ends
LV_D uint64_t flood(const ColumnWindows& w, uint64_t zr, uint64_t s) {
    uint64_t f = s & w.z;
    while (true) {
        const uint64_t g = fill_cols(w, fill_row(w.z, zr, f));
        if (__ballot(g != f) == 0ull) return g;
        f = g;
    }
}

// The 64 bytes of a row from column x0 on as bits (set: not 0), zeros outside the image. Four 16-byte loads in
// place of 64 ballots over single bytes; bit 7 of (b & 127) + 127 | b tells whether byte b is set, and one product
// gathers the four bits of a word (bit 24 + i of the product is byte i's).
LV_D uint64_t mask_row(const uint8_t* m, int W, int H, int x0, int gy) {
    if (gy < 0 || gy >= H) return 0ull;
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    struct __attribute__((packed, aligned(1))) Quad {
        u32x4 v;
    };
    const int off = gy * W + x0, total = W * H;
    uint32_t q[16];
    if (off + 64 <= total) {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const u32x4 t = peek<Quad>(m, (uint32_t)(off + 16 * k));
            q[4 * k] = t.x, q[4 * k + 1] = t.y, q[4 * k + 2] = t.z, q[4 * k + 3] = t.w;
        }
    } else {
#pragma unroll
        for (int k = 0; k < 16; ++k) q[k] = word_at(m, off + 4 * k, total);
    }
    uint32_t b[2] = {0u, 0u};
#pragma unroll
    for (int k = 0; k < 16; ++k) {
        const uint32_t nz = ((((q[k] & 0x7F7F7F7Fu) + 0x7F7F7F7Fu) | q[k]) >> 7) & 0x01010101u;
        b[k >> 3] |= ((nz * 0x01020408u) >> 24 & 15u) << (4 * (k & 7));
    }
    const uint64_t bits = ((uint64_t)b[1] << 32) | b[0];
    return W - x0 >= ZS ? bits : bits & ((1ull << (W - x0)) - 1ull);
}

// raw bits of columns x0-2, x0-1, x0+64, x0+65 of row gy (bits 0..3)
LV_D uint32_t raw_halo(const uint8_t* raw, int W, int H, int x0, int gy) {
    if (gy < 0 || gy >= H) return 0u;
    const uint8_t* row = raw + (size_t)gy * (size_t)W;
    const int xs[4] = {x0 - 2, x0 - 1, x0 + ZS, x0 + ZS + 1};
    uint32_t h = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i)
        if (xs[i] >= 0 && xs[i] < W && row[xs[i]] != 0) h |= 1u << i;
    return h;
}
// 3-wide dilation along a row: core columns x0..x0+63 and the halo bits above -> dilated core and
// dilated halo (bit 0: column x0-1, bit 1: column x0+64)
LV_D void dilate3_row(uint64_t c, uint32_t h, uint64_t& d, uint32_t& dh) {
    d = c | (c << 1) | (uint64_t)((h >> 1) & 1u) | (c >> 1) | ((uint64_t)((h >> 2) & 1u) << 63);
    const uint32_t left = (h & 1u) | ((h >> 1) & 1u) | (uint32_t)(c & 1ull);
    const uint32_t right = (uint32_t)(c >> 63) | ((h >> 2) & 1u) | ((h >> 3) & 1u);
    dh = left | (right << 1);
}

// closing of the zone, its 0-pixels, and their border components
LV_D void zone_close_body(const View& v, uint32_t bid, uint32_t nblk) {
    __shared__ uint64_t s_d[ZPB][ZS + 4];   // row-dilated raw rows y0-2 .. y0+65
    __shared__ uint32_t s_dx[ZPB][ZS + 4];
    const int W = v.W, H = v.H;
    const int lane = (int)(threadIdx.x & 63u), wv = (int)(threadIdx.x >> 6);
    const int nzx = (W + ZS - 1) / ZS, nz = nzx * ((H + ZS - 1) / ZS);
    const int z = (int)bid * ZPB + wv;
    if (z >= nz) return;  // whole wavefronts only; nothing below synchronizes the block
    const int x0 = (z % nzx) * ZS, y0 = (z / nzx) * ZS;
    // the raw mask is the decisions (zero outside the ROI): they are final before the model update, so
    // this runs beside it
    const uint8_t* raw = v.dec;
    // raw rows y0-2 .. y0+65 as 64-bit masks: lane y has row y, lanes 0..3 also rows 64..67
    const uint64_t c0 = mask_row(raw, W, H, x0, y0 - 2 + lane);
    const uint64_t c1 = lane < 4 ? mask_row(raw, W, H, x0, y0 - 2 + ZS + lane) : 0ull;
    const uint32_t h0 = raw_halo(raw, W, H, x0, y0 - 2 + lane);
    const uint32_t h1 = lane < 4 ? raw_halo(raw, W, H, x0, y0 - 2 + ZS + lane) : 0u;
    {
        uint64_t d;
        uint32_t dh;
        dilate3_row(c0, h0, d, dh);
        s_d[wv][lane] = d;
        s_dx[wv][lane] = dh;
        dilate3_row(c1, h1, d, dh);
        if (lane < 4) {
            s_d[wv][ZS + lane] = d;
            s_dx[wv][ZS + lane] = dh;
        }
    }
    wave_sync();
    // lane y: zone row y = dilated-row index y+2; erosion over dilated rows y+1..y+3, each the OR
    // of three row-dilated rows; outside the image the dilation is 255 (neutral for the erosion)
    const uint64_t in_cols = W - x0 >= ZS ? ~0ull : ((1ull << (W - x0)) - 1ull);
    const uint32_t out_halo = (x0 == 0 ? 1u : 0u) | (x0 + ZS >= W ? 2u : 0u);
    uint64_t e = ~0ull;
    uint32_t ex = 3u;
#pragma unroll
    for (int a = 1; a <= 3; ++a) {
        const int r = lane + a, gy = y0 - 2 + r;
        uint64_t d = s_d[wv][r - 1] | s_d[wv][r] | s_d[wv][r + 1];
        uint32_t dx = s_dx[wv][r - 1] | s_dx[wv][r] | s_dx[wv][r + 1];
        if (gy < 0 || gy >= H) {
            d = ~0ull;
            dx = 3u;
        } else {
            d |= ~in_cols;
            dx |= out_halo;
        }
        e &= d;
        ex &= dx;
    }
    const uint64_t pre = e & ((e << 1) | (uint64_t)(ex & 1u)) & ((e >> 1) | ((uint64_t)(ex >> 1) << 63));
    const uint64_t zm = y0 + lane < H ? (~pre & in_cols) : 0ull;
    v.zbits[(size_t)z * ZS + lane] = zm;
    // border components in the order top row, left column, right column, bottom row
    const uint64_t zr = brev64(zm);
    const ColumnWindows win = column_windows(zm, lane);
    uint64_t remT = lane_bcast(zm, 0), remB = lane_bcast(zm, 63);
    uint64_t remL = __ballot((zm & 1ull) != 0), remR = __ballot((zm >> 63) != 0);
    uint32_t cT = 255u, cB = 255u, cL = 255u, cR = 255u, k = 0;
    while ((remT | remB | remL | remR) != 0ull) {
        uint64_t s;
        if (remT) s = lane == 0 ? 1ull << __builtin_ctzll(remT) : 0ull;
        else if (remL) s = lane == __builtin_ctzll(remL) ? 1ull : 0ull;
        else if (remR) s = lane == __builtin_ctzll(remR) ? 1ull << 63 : 0ull;
        else s = lane == 63 ? 1ull << __builtin_ctzll(remB) : 0ull;
        const uint64_t f = flood(win, zr, s);
        const uint64_t fT = lane_bcast(f, 0), fB = lane_bcast(f, 63);
        const uint64_t fL = __ballot((f & 1ull) != 0), fR = __ballot((f >> 63) != 0);
        if ((fT >> lane) & 1ull) cT = k;
        if ((fB >> lane) & 1ull) cB = k;
        if ((fL >> lane) & 1ull) cL = k;
        if ((fR >> lane) & 1ull) cR = k;
        remT &= ~fT;
        remB &= ~fB;
        remL &= ~fL;
        remR &= ~fR;
        ++k;
    }
    uint8_t* edge = v.zedge + (size_t)z * 256;
    edge[lane] = (uint8_t)cT;
    edge[64 + lane] = (uint8_t)cB;
    edge[128 + lane] = (uint8_t)cL;
    edge[192 + lane] = (uint8_t)cR;
    const uint32_t base = (uint32_t)z * kZoneComps;
    if ((uint32_t)lane < k) v.zpar[base + lane] = base + lane;
    if ((uint32_t)lane + 64u < k) v.zpar[base + lane + 64] = base + lane + 64;
    if (lane == 0) v.zcount[z] = k;
}

// Root of a node, with path halving. Every store replaces a parent by one of its ancestors, so parents stay
// below their nodes; a store that races with a union may drop the link that union made to the node, which the
// union then makes again between the old and the new parent (it goes on with the value it replaced).
LV_D uint32_t g_find(uint32_t* lab, uint32_t a) {
    while (true) {
        const uint32_t pa = __hip_atomic_load(&lab[a], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (pa == a) return a;
        const uint32_t ga = __hip_atomic_load(&lab[pa], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (ga != pa) __hip_atomic_store(&lab[a], ga, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        a = ga;
    }
}

// joins a < b; most pairs meet as roots, which one atomic links
LV_D void g_union(uint32_t* lab, uint32_t a, uint32_t b) {
    const uint32_t first = atomicMin(&lab[b], a);
    bool done = first == b;
    b = first;
    while (!done) {
        a = g_find(lab, a);
        b = g_find(lab, b);
        if (a < b) {
            const uint32_t old = atomicMin(&lab[b], a);
            done = old == b;
            b = old;
        } else if (b < a) {
            const uint32_t old = atomicMin(&lab[a], b);
            done = old == a;
            a = old;
        } else {
            done = true;
        }
    }
}

// joins the components facing each other across one zone edge (lane = position along the edge);
// a lane whose pair repeats the previous lane's leaves the union to that lane
LV_D void zone_link(uint32_t* par, uint32_t za, uint32_t zb, uint32_t a, uint32_t b, int lane) {
    const uint32_t pa = (uint32_t)__shfl_up((int)a, 1u, 64), pb = (uint32_t)__shfl_up((int)b, 1u, 64);
    const bool dup = lane > 0 && pa == a && pb == b;
    if (a != 255u && b != 255u && !dup) g_union(par, za * kZoneComps + a, zb * kZoneComps + b);
}

// unions across the right and bottom edges of every zone. Bound by chains of atomics across XCDs, so each edge
// has a wavefront: against one for both edges of a zone that first looked up both roots, 3840x2160 24.7 -> 19.9 us,
// 1920x1080 12.7 -> 10.0, 320x240 6.6 -> 5.0, 64 mixed streams 45.6 -> 27.4 us.
LV_D void zone_link_body(const View& v, uint32_t bid, uint32_t nblk) {
    const int lane = (int)(threadIdx.x & 63u), wv = (int)(threadIdx.x >> 6);
    const int nzx = (v.W + ZS - 1) / ZS, nzy = (v.H + ZS - 1) / ZS;
    const int z = ((int)bid * ZPB + wv) >> 1;
    const bool right = (wv & 1) == 0;
    if (z >= nzx * nzy || (right ? z % nzx + 1 == nzx : z / nzx + 1 == nzy)) return;
    const int z2 = right ? z + 1 : z + nzx;
    const uint8_t* e = v.zedge;
    zone_link(v.zpar, (uint32_t)z, (uint32_t)z2, e[(size_t)z * 256 + (right ? 192 : 64) + lane],
              e[(size_t)z2 * 256 + (right ? 128 : 0) + lane], lane);
}

// holes of a zone: its 0-pixels minus the flood from the border pixels of outside components
LV_D void zone_holes_body(const View& v, uint32_t bid, uint32_t nblk) {
    const int lane = (int)(threadIdx.x & 63u), wv = (int)(threadIdx.x >> 6);
    const int nzx = (v.W + ZS - 1) / ZS, nz = nzx * ((v.H + ZS - 1) / ZS);
    const int z = (int)bid * ZPB + wv;
    if (z >= nz) return;
    const uint64_t zm = v.zbits[(size_t)z * ZS + lane];
    const uint8_t* e = v.zedge + (size_t)z * 256;
    const uint32_t cT = e[lane], cB = e[64 + lane], cL = e[128 + lane], cR = e[192 + lane];
    const uint32_t k = v.zcount[z];
    const uint32_t c00 = v.zedge[0];  // component of pixel (0,0) in zone 0, 255 if it is foreground
    const uint32_t root = c00 == 255u ? 0xFFFFFFFFu : g_find(v.zpar, c00);
    const uint32_t base = (uint32_t)z * kZoneComps;
    const bool o0 = (uint32_t)lane < k && g_find(v.zpar, base + lane) == root;
    const bool o1 = (uint32_t)lane + 64u < k && g_find(v.zpar, base + lane + 64) == root;
    const uint64_t m0 = __ballot(o0), m1 = __ballot(o1);
    auto outside = [&](uint32_t c) {
        return c < 64u ? ((m0 >> c) & 1ull) != 0 : (c < 128u && ((m1 >> (c - 64u)) & 1ull) != 0);
    };
    const uint64_t sT = __ballot(outside(cT)), sB = __ballot(outside(cB));
    uint64_t s = (outside(cL) ? 1ull : 0ull) | (outside(cR) ? 1ull << 63 : 0ull);
    if (lane == 0) s |= sT;
    if (lane == 63) s |= sB;
    const uint64_t o = flood(column_windows(zm, lane), brev64(zm), s);
    v.hbits[(size_t)z * ZS + lane] = zm & ~o;
}

// Post-processing masks are 0/255 bytes; the median and dilation kernels below work on four pixels
// per 32-bit word. Words start at columns that are multiples of 4 (tile origins are), so when the
// row pitch W is too a word is one aligned load or store; other widths assemble bytes.

// bytes (gx..gx+3, gy) of a W x H byte image, `pad` for those outside it; gx % 4 == 0
LV_D uint32_t load_mask_word(const uint8_t* m, int W, int H, int gx, int gy, uint32_t pad) {
    const uint32_t fill = pad * 0x01010101u;
    if (gy < 0 || gy >= H || gx + 3 < 0 || gx >= W) return fill;
    const uint8_t* row = m + (size_t)gy * (size_t)W;
    if ((W & 3) == 0) return *(const uint32_t*)(row + gx);  // gx >= 0 and gx + 3 < W here
    uint32_t w = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int x = gx + i;
        w |= (x >= 0 && x < W ? (uint32_t)row[x] : pad) << (8 * i);
    }
    return w;
}

LV_D void store_mask_word(uint8_t* m, int W, int H, int gx, int gy, uint32_t w) {
    if (gy >= H || gx >= W) return;
    uint8_t* row = m + (size_t)gy * (size_t)W;
    if ((W & 3) == 0) {
        *(uint32_t*)(row + gx) = w;
        return;
    }
    for (int i = 0; i < 4 && gx + i < W; ++i) row[gx + i] = (uint8_t)(w >> (8 * i));
}

// the same into the caller's mask, which may have any alignment
LV_D void store_out_word(uint8_t* m, int W, int H, int gx, int gy, uint32_t w) {
    if (((uintptr_t)m & 3u) == 0) {
        store_mask_word(m, W, H, gx, gy, w);
        return;
    }
    if (gy >= H) return;
    for (int i = 0; i < 4 && gx + i < W; ++i) m[(size_t)gy * (size_t)W + gx + i] = (uint8_t)(w >> (8 * i));
}

// bits (gx..gx+31, gy) of a zone bitmap (gx % 32 == 0), zero outside the image
LV_D uint32_t zone_bits32(const uint64_t* bits, int W, int H, int gx, int gy) {
    if (gx < 0 || gy < 0 || gx >= W || gy >= H) return 0u;
    const size_t zi = (size_t)(gy / ZS) * (size_t)((W + ZS - 1) / ZS) + (size_t)(gx / ZS);
    return ((const uint32_t*)bits)[(zi * ZS + (size_t)(gy % ZS)) * 2 + (size_t)(gx % ZS / 32)];
}
// four bits -> four bytes of 0/255 (the products of the bits with 1, 2^7, 2^14, 2^21 never
// overlap, so bit i lands alone at bit 8i)
LV_D uint32_t expand4(uint32_t b) { return ((b * 0x00204081u) & 0x01010101u) * 255u; }

// byte window of two adjacent words: bytes s..s+3 of (lo, hi)
LV_D uint32_t bytes_at(uint32_t hi, uint32_t lo, uint32_t s) { return __builtin_amdgcn_alignbyte(hi, lo, s); }

// OR of the word whose bytes start 4 bytes into a, b, c and its shifts by up to 3 bytes either way: the 7-wide
// dilation of the 0/255 bytes of b along the row
LV_D uint32_t dilate7_word(uint32_t a, uint32_t b, uint32_t c) {
    return b | bytes_at(b, a, 1) | bytes_at(b, a, 2) | bytes_at(b, a, 3) | bytes_at(c, b, 1) | bytes_at(c, b, 2) |
           bytes_at(c, b, 3);
}

// mask = raw | holes | erode7(PreFlood); last_fg = medianBlur(mask, k) (SUB:544-547; LOB:578 uses
// the raw mask directly). Binary median with zero padding = majority count over the k x k window.
// Counts are kept one per byte (at most 13 per column and 169 per window, so no byte carries into
// the next) and the majority test adds 128 - need to every byte and keeps bit 7. Holes and erosion stay bits (32
// columns a word) until the counts, as the zones have them. Bound by its LDS passes: with bytes throughout, one row
// of column counts an item and counts over 13 columns whatever k is, 3840x2160 29.2 -> 20.0 us, 1920x1080 9.3 -> 6.4,
// 64 mixed streams 156 -> 106 us.
template <bool SUBSENSE>
LV_D void median_body(const View& v, uint32_t bid, uint32_t nblk) {
    constexpr int HM = 6, HE = 3;           // median halo (k <= 13), erosion halo
    constexpr int MWW = (PW + 16) / 4;      // mask words: columns x0-8 .. x0+PW+7
    constexpr int MH = PH + 2 * HM;         // mask rows: y0-6 .. y0+PH+5
    constexpr int EH = MH + 2 * HE;         // PreFlood rows: y0-9 .. y0+PH+8
    constexpr int BW = PW / 32 + 2;         // words of a row's bits: columns x0-32 .. x0+PW+31
    constexpr int OWW = PW / 4;             // output words per row
    static_assert(EH * BW <= TPB, "an item per thread");
    __shared__ uint32_t s_pre[EH][BW];
    __shared__ uint32_t s_eh[EH][BW];
    __shared__ uint32_t s_bits[MH][BW];
    __shared__ uint32_t s_mask[MH][MWW];
    __shared__ uint32_t s_col[PH][MWW];
    const int W = v.W, H = v.H;
    const int ntx = (W + PW - 1) / PW;
    const int tid = (int)bid;
    const int x0 = (tid % ntx) * PW, y0 = (tid / ntx) * PH;
    const int k = v.median_k, r = k / 2, need = (k * k + 1) / 2;
    if constexpr (SUBSENSE) {
        const int ly = (int)threadIdx.x / BW, j = (int)threadIdx.x % BW, gx = x0 + 32 * (j - 1);
        // PreFlood is set except at its 0-pixels, and set outside the image
        if (ly < EH) s_pre[ly][j] = ~zone_bits32(v.zbits, W, H, gx, y0 - HM - HE + ly);
        __syncthreads();
        // horizontal 7-erosion (the outer three columns of a row's bits are not used)
        if (ly < EH) {
            const uint32_t w = s_pre[ly][j], l = s_pre[ly][max(j - 1, 0)], r = s_pre[ly][min(j + 1, BW - 1)];
            uint32_t e = w;
#pragma unroll
            for (uint32_t a = 1; a <= (uint32_t)HE; ++a)
                e &= __builtin_amdgcn_alignbit(w, l, 32u - a) & __builtin_amdgcn_alignbit(r, w, a);
            s_eh[ly][j] = e;
        }
        __syncthreads();
        // holes | erosion inside the image; mask row ly is PreFlood row ly+3
        if (ly < MH) {
            const int gy = y0 - HM + ly, left = W - gx;
            uint32_t e = s_eh[ly][j];
#pragma unroll
            for (int a = 1; a <= 2 * HE; ++a) e &= s_eh[ly + a][j];
            const bool in = gx >= 0 && left > 0 && gy >= 0 && gy < H;
            const uint32_t image = !in ? 0u : left >= 32 ? ~0u : (1u << left) - 1u;
            s_bits[ly][j] = (zone_bits32(v.hbits, W, H, gx, gy) | e) & image;
        }
        __syncthreads();
    }
    // the mask as 0/1 bytes, zero outside the image
    for (int i = threadIdx.x; i < MH * MWW; i += TPB) {
        const int ly = i / MWW, j = i % MWW, b = 24 + 4 * j;
        uint32_t m = load_mask_word(v.last_raw, W, H, x0 - 8 + 4 * j, y0 - HM + ly, 0u);
        if constexpr (SUBSENSE) m |= expand4(s_bits[ly][b >> 5] >> (b & 31) & 15u);
        s_mask[ly][j] = m & 0x01010101u;
    }
    __syncthreads();
    // column counts over k rows, two rows an item: the second drops a row and takes in the next
    static_assert(PH % 2 == 0 && PH / 2 * MWW <= TPB, "an item per thread");
    if (threadIdx.x < PH / 2 * MWW) {
        const int ly = (int)threadIdx.x / MWW * 2, j = (int)threadIdx.x % MWW, a0 = HM + ly - r;
        uint32_t c = 0;
        for (int a = a0; a <= a0 + 2 * r; ++a) c += s_mask[a][j];
        s_col[ly][j] = c;
        s_col[ly + 1][j] = c - s_mask[a0][j] + s_mask[a0 + 2 * r + 1][j];
    }
    __syncthreads();
    // row counts over k columns: output word q (columns x0+4q..) starts at byte 4q+8 of the counts
    const uint32_t bias = (uint32_t)(128 - need) * 0x01010101u;
    for (int i = threadIdx.x; i < PH * OWW; i += TPB) {
        const int ly = i / OWW, q = i % OWW;
        uint32_t w[5];
#pragma unroll
        for (int u = 0; u < 5; ++u) w[u] = s_col[ly][q + u];
        auto from = [&](int b) { return b & 3 ? bytes_at(w[(b >> 2) + 1], w[b >> 2], (uint32_t)(b & 3)) : w[b >> 2]; };
        uint32_t s = w[2];
#pragma unroll
        for (int o = 1; o <= HM; ++o)
            if (o <= r) s += from(8 - o) + from(8 + o);  // uniform
        const uint32_t bits = ((s + bias) >> 7) & 0x01010101u;
        store_mask_word(v.last_fg, W, H, x0 + 4 * q, y0 + ly, bits * 255u);
        if constexpr (!SUBSENSE)
            if (v.out_mask) store_out_word(v.out_mask, W, H, x0 + 4 * q, y0 + ly, bits * 255u);
    }
    if constexpr (!SUBSENSE) {
        if (bid == 0 && threadIdx.x == 0) {  // end of the LOBSTER step
            v.sc->frame_idx += 1u;
            v.sc->epoch += 1u;
        }
    }
}

// What the pixels around a tile offer to refreshModel: colour and descriptor as a sample record, and
// whether they may be sampled. A 3-pixel halo covers getSamplePosition's 7x7 window (its clamping moves a
// position towards the pixel). A record serves up to 50 samples of each of the 49 pixels around it, so it is
// built once here (LOBSTER computes its descriptor) instead of per sample from global memory.
struct RefreshTile {
    static constexpr int LW = TW + 6, LH = TH + 6;
    uint32_t w0[LW * LH], w1[LW * LH], w2[LW * LH];  // w0 alone with one channel
    uint8_t ok[LW * LH];
    uint8_t pos[512];  // sample position of each draw % 512: dx + 3 | (dy + 3) << 4
};

struct DilateTile {
    static constexpr int H3 = 3;
    static constexpr int FWW = (PW + 8) / 4;  // last_fg words: columns x0-4 .. x0+PW+3
    static constexpr int LH = PH + 2 * H3;    // rows y0-3 .. y0+PH+2
    static constexpr int OWW = PW / 4;
    uint32_t fg[LH][FWW], h[LH][OWW];
};

// one allocation for the two kinds of work of the dilation launch, whichever channel counts it instantiates
// (a sum instead of a union takes as long: the dilation of 64 mixed streams 200 us either way)
union SweepLds {
    RefreshTile refresh;
    DilateTile dilate;
};
LV_D SweepLds& sweep_lds() {
    __shared__ SweepLds m;
    return m;
}

// dilate7(last_fg), blink masks (SUB:548-551), final-segmentation averages (SUB:553-554) and the
// output mask. addWeighted(.., CV_32F) is evaluated as the double-precision scalar form. Runs after the
// controller, which has advanced the frame index.
LV_D void dilate_final_body(const View& v, uint32_t bid, uint32_t nblk) {
    uint8_t* out_mask = v.out_mask;
    constexpr int H3 = DilateTile::H3, FWW = DilateTile::FWW, LH = DilateTile::LH, OWW = DilateTile::OWW;
    DilateTile& t = sweep_lds().dilate;
    auto& s_fg = t.fg;
    auto& s_h = t.h;
    const int W = v.W, H = v.H;
    const int ntx = (W + PW - 1) / PW;
    const int tid = (int)bid;
    const int x0 = (tid % ntx) * PW, y0 = (tid / ntx) * PH;
    for (int i = threadIdx.x; i < LH * FWW; i += TPB) {
        const int ly = i / FWW, wx = i % FWW;
        s_fg[ly][wx] = load_mask_word(v.last_fg, W, H, x0 - 4 + 4 * wx, y0 - H3 + ly, 0u);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < LH * OWW; i += TPB) {
        const int ly = i / OWW, q = i % OWW;
        s_h[ly][q] = dilate7_word(s_fg[ly][q], s_fg[ly][q + 1], s_fg[ly][q + 2]);
    }
    __syncthreads();
    const uint32_t frame_no = v.sc->frame_idx, mvn = v.mv_avgs;
    const float aLT = 1.0f / (float)(frame_no < mvn ? frame_no : mvn);
    const float aST = 1.0f / (float)(frame_no < mvn / 4u ? frame_no : mvn / 4u);
    const double alt = (double)(1.0f - aLT), blt = (1.0 / 255) * (double)aLT;
    const double ast = (double)(1.0f - aST), bst = (1.0 / 255) * (double)aST;
    for (int i = threadIdx.x; i < PH * OWW; i += TPB) {
        const int ly = i / OWW, q = i % OWW, gx = x0 + 4 * q, gy = y0 + ly;
        if (gx >= W || gy >= H) continue;
        uint32_t d = s_h[ly][q];
#pragma unroll
        for (int a = 1; a <= 2 * H3; ++a) d |= s_h[ly + a][q];
        const uint32_t inv = ~d, fg = s_fg[ly + H3][q + 1];
        const size_t p = (size_t)gy * W + gx;
        if ((W & 3) == 0) {
            uint32_t* const bl = (uint32_t*)v.blinks;
            uint32_t* const ldi = (uint32_t*)v.last_dil_inv;
            const uint32_t w = (uint32_t)(p >> 2), bl0 = *at(bl, w), ldi0 = *at(ldi, w);
            store_changed(bl, w, bl0 & ldi0 & inv, bl0);
            store_changed(ldi, w, inv, ldi0);
            typedef float f32x4 __attribute__((ext_vector_type(4)));
            const gptr<f32x4> lt = at((f32x4*)v.FinLT, w), st = at((f32x4*)v.FinST, w);
            const f32x4 a0 = *lt, b0 = *st;
            f32x4 a = a0, b = b0;
            const double f0 = (double)(fg & 255u), f1 = (double)((fg >> 8) & 255u);
            const double f2 = (double)((fg >> 16) & 255u), f3 = (double)(fg >> 24);
            a.x = (float)((double)a.x * alt + f0 * blt + 0.0);
            a.y = (float)((double)a.y * alt + f1 * blt + 0.0);
            a.z = (float)((double)a.z * alt + f2 * blt + 0.0);
            a.w = (float)((double)a.w * alt + f3 * blt + 0.0);
            b.x = (float)((double)b.x * ast + f0 * bst + 0.0);
            b.y = (float)((double)b.y * ast + f1 * bst + 0.0);
            b.z = (float)((double)b.z * ast + f2 * bst + 0.0);
            b.w = (float)((double)b.w * ast + f3 * bst + 0.0);
            typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
            auto differ = [](f32x4 m, f32x4 n) {
                const u32x4 d = __builtin_bit_cast(u32x4, m) ^ __builtin_bit_cast(u32x4, n);
                return (d.x | d.y | d.z | d.w) != 0u;
            };
            if (__ballot(differ(a, a0)) != 0ull) *lt = a;
            if (__ballot(differ(b, b0)) != 0ull) *st = b;
            if (out_mask) {
                if (((uintptr_t)out_mask & 3u) == 0) *(uint32_t*)(out_mask + p) = fg;  // caller's buffer
                else
                    for (int u = 0; u < 4; ++u) out_mask[p + u] = (uint8_t)(fg >> (8 * u));
            }
        } else {
            for (int u = 0; u < 4 && gx + u < W; ++u) {
                const size_t pu = p + u;
                const uint8_t iu = (uint8_t)(inv >> (8 * u)), fu = (uint8_t)(fg >> (8 * u));
                *at(v.blinks, pu) = (uint8_t)(*at(v.blinks, pu) & *at(v.last_dil_inv, pu) & iu);
                *at(v.last_dil_inv, pu) = iu;
                const double f = (double)fu;
                *at(v.FinLT, pu) = (float)((double)*at(v.FinLT, pu) * alt + f * blt + 0.0);
                *at(v.FinST, pu) = (float)((double)*at(v.FinST, pu) * ast + f * bst + 0.0);
                if (out_mask) out_mask[pu] = fu;
            }
        }
    }
}

// ----------------------------------------------------------------------------------------------
// frame-level controller (SUB:555-611)
// ----------------------------------------------------------------------------------------------
LV_D uint8_t sat_u8(float f) {
    const float r = rintf(f);  // round half to even, like cvRound
    return (uint8_t)(r < 0.f ? 0.f : r > 255.f ? 255.f : r);
}

LV_D bool ds_exact8(const View& v) { return v.W == 8 * v.dsW && v.H == 8 * v.dsH; }

template <int C>
LV_D void ds_update_cell(const View& v, uint32_t cell, const uint8_t m[C], uint32_t& contrib) {
    const uint32_t frame_no = cur_frame(v), mvn = v.mv_avgs;
    const float aL = 1.0f / (float)(frame_no < mvn ? frame_no : mvn);
    const float aS = 1.0f / (float)(frame_no < mvn / 4u ? frame_no : mvn / 4u);
    const float bL = 1.0f - aL, bS = 1.0f - aS;
    uint32_t best = 0;
    for (int c = 0; c < C; ++c) {
        const size_t di = (size_t)cell * C + c;
        const float lt = (float)m[c] * aL + v.dsLT[di] * bL;
        const float st = (float)m[c] * aS + v.dsST[di] * bS;
        v.dsLT[di] = lt;
        v.dsST[di] = st;
        const uint32_t d = (uint32_t)fabsf(st - lt);
        best = d > best ? d : best;
    }
    contrib = C == 1 ? best / 2u : best;
}

// channel sums of one cell row: the 8 pixels (8*C bytes) at `row`, read as C aligned 8-byte words
template <int C>
LV_D void cell_row_sum(const uint8_t* row, uint32_t sum[C]) {
    const uint2* q = (const uint2*)row;
#pragma unroll
    for (int j = 0; j < C; ++j) {
        const uint2 w = q[j];
#pragma unroll
        for (int b = 0; b < 8; ++b) sum[(8 * j + b) % C] += ((b < 4 ? w.x : w.y) >> (8 * (b & 3))) & 0xFFu;
    }
}

// resize(INTER_AREA, W/8 x H/8) + accumulateWeighted LT/ST + per-cell |ST-LT| (SUB:568-583), one
// thread per cell in raster order. Frame sizes that are multiples of 8 (an integer factor: the
// rounded 8x8 block mean) read each cell row as C 8-byte words (bytes when the frame is not 8-byte
// aligned), so a wavefront's loads cover contiguous runs of 64 cells; other sizes take the general
// area weights.
template <int C>
LV_D void downsample_body(const View& v, uint32_t bid, uint32_t nblk) {
    const uint8_t* frame = v.frame;
    uint32_t contrib = 0;
    const uint32_t ncell = (uint32_t)(v.dsW * v.dsH);
    const uint32_t cell = bid * TPB + threadIdx.x;
    if (cell < ncell && ds_exact8(v)) {
        const int dx = (int)(cell % (uint32_t)v.dsW), dy = (int)(cell / (uint32_t)v.dsW);
        uint32_t sum[C];
#pragma unroll
        for (int c = 0; c < C; ++c) sum[c] = 0;
        const uint8_t* cell0 = frame + ((size_t)dy * 8 * v.W + (size_t)dx * 8) * C;
        if (((uintptr_t)frame & 7u) == 0) {
#pragma unroll
            for (int r = 0; r < 8; ++r) cell_row_sum<C>(cell0 + (size_t)r * v.W * C, sum);
        } else {
            for (int r = 0; r < 8; ++r)
#pragma unroll
                for (int b = 0; b < 8 * C; ++b) sum[b % C] += cell0[(size_t)r * v.W * C + b];
        }
        uint8_t mc[C];
#pragma unroll
        for (int c = 0; c < C; ++c) mc[c] = sat_u8((float)sum[c] * (1.f / 64.f));
        ds_update_cell<C>(v, cell, mc, contrib);
    } else if (cell < ncell) {
        const int dx = (int)(cell % (uint32_t)v.dsW), dy = (int)(cell / (uint32_t)v.dsW);
        uint8_t mc[C];
        if (v.W % v.dsW == 0 && v.H % v.dsH == 0) {
            const int sx = v.W / v.dsW, sy = v.H / v.dsH;
            for (int c = 0; c < C; ++c) {
                int sum = 0;
                for (int yy = 0; yy < sy; ++yy)
                    for (int xx = 0; xx < sx; ++xx) sum += *at(frame, ((dy * sy + yy) * v.W + (dx * sx + xx)) * C + c);
                mc[c] = sat_u8((float)sum * (1.f / (float)(sx * sy)));
            }
        } else {
            const double sx = (double)v.W / v.dsW, sy = (double)v.H / v.dsH;
            const double yb = dy * sy, ye = (dy + 1) * sy, xb = dx * sx, xe = (dx + 1) * sx;
            double acc[C];
#pragma unroll
            for (int c = 0; c < C; ++c) acc[c] = 0.0;
            // Sides that are no multiple of 8: a cell covers 8 to 15 pixels a side, and all but the smallest images
            // have cells within kCols columns. These take the column weights once for all rows and channels and
            // a row's bytes as words (a column past the cell has weight 0, which adds nothing); the sums keep
            // raster order per channel. Bound by a thread's chain of loads: the update launch that holds the
            // cells at 721x577 37.7 us with byte loads per channel, 25.0 with words.
            constexpr int kCols = 10, kWords = (kCols * C + 3) / 4;
            const int total = (int)v.npx * C, x_end = min(v.W, (int)ceil(xe));
            if (x_end - (int)xb <= kCols) {
                double wx[kCols];
#pragma unroll
                for (int j = 0; j < kCols; ++j) {
                    const int xx = (int)xb + j;
                    wx[j] = xx < x_end ? fmin((double)(xx + 1), xe) - fmax((double)xx, xb) : 0.0;
                }
#pragma unroll 2
                for (int yy = (int)yb; yy < v.H && (double)yy < ye; ++yy) {
                    const double wy = fmin((double)(yy + 1), ye) - fmax((double)yy, yb);
                    uint32_t q[kWords];
#pragma unroll
                    for (int k = 0; k < kWords; ++k) q[k] = word_at(frame, (yy * v.W + (int)xb) * C + 4 * k, total);
#pragma unroll
                    for (int j = 0; j < kCols; ++j)
#pragma unroll
                        for (int c = 0; c < C; ++c) {
                            const int b = j * C + c;
                            acc[c] += (double)((q[b >> 2] >> (8 * (b & 3))) & 255u) * (wy * wx[j]);
                        }
                }
            } else {
                for (int yy = (int)yb; yy < v.H && (double)yy < ye; ++yy) {
                    const double wy = fmin((double)(yy + 1), ye) - fmax((double)yy, yb);
                    for (int xx = (int)xb; xx < x_end; ++xx) {
                        const double wx = fmin((double)(xx + 1), xe) - fmax((double)xx, xb);
                        for (int c = 0; c < C; ++c) acc[c] += (double)*at(frame, (yy * v.W + xx) * C + c) * (wy * wx);
                    }
                }
            }
#pragma unroll
            for (int c = 0; c < C; ++c) mc[c] = sat_u8((float)(acc[c] / (sx * sy)));
        }
        ds_update_cell<C>(v, cell, mc, contrib);
    }
    block_add<TPB>(contrib, v.sc->cd_part);
}

// single-workgroup decision: LUT adaptation, model reset, learning-rate caps, counters
LV_D void decide_body(const View& v, uint32_t bid, uint32_t nblk) {
    Scalars* sc = v.sc;
    __shared__ float s_ratio, s_last;
    __shared__ unsigned long long s_cd;
    if (threadIdx.x == 0) {
        s_ratio = (float)sum_stripes(sc->nz_part) / (float)v.n_roi;
        s_last = sc->last_nz_ratio;
        s_cd = sum_stripes(sc->cd_part);
    }
    __syncthreads();
    if (threadIdx.x < kStripes) {
        sc->nz_part[threadIdx.x] = 0;
        sc->cd_part[threadIdx.x] = 0;
    }
    const float ratio = s_ratio, last = s_last;
    const uint32_t t = threadIdx.x;
    uint8_t lut = sc->lut[t];
    if (ratio < 0.1f && last < 0.1f) {
        const float lb = (float)v.lbsp_offset + ceilf((float)t * v.rel_lbsp / 4.0f);
        if (lut > sat_u8(lb)) --lut;
    } else if (ratio > 0.5f && last > 0.5f) {
        const uint8_t ub = sat_u8((float)v.lbsp_offset + 255.0f * v.rel_lbsp);
        if (lut < ub) ++lut;
    }
    __syncthreads();
    sc->lut[t] = lut;
    if (threadIdx.x != 0) return;
    sc->last_nz_ratio = ratio;
    sc->refresh_pending = 0;
    if (v.lr_scaling) {
        const float cratio = (float)s_cd / (float)(v.dsW * v.dsH);
        const uint32_t thr = v.color_thr / 2u;  // FRAMELEVEL_MIN_COLOR_DIFF_THRESHOLD
        if (sc->auto_reset) {
            if (sc->frames_since_reset > 1000u) {
                sc->auto_reset = 0;
            } else if (cratio >= (float)thr && sc->cooldown == 0u) {
                sc->frames_since_reset = 0;
                sc->refresh_pending = 1;  // refreshModel(0.1f) + T := 1 (SUB:589-592)
                sc->refresh_frac = 0.1f;
                sc->refresh_force_fg = 0;
                sc->refresh_frame = cur_frame(v);
                sc->refresh_ev = sc->refresh_seq++;
                sc->cooldown = v.mv_avgs / 4u;
            } else {
                ++sc->frames_since_reset;
            }
        } else if (cratio >= (float)(thr * 2u)) {
            sc->frames_since_reset = 0;
            sc->auto_reset = 1;
        }
        if (cratio >= (float)(thr / 2u)) {
            const int k = (int)(cratio / 2.0f);  // x86 shifts by the count mod 32
            const int lo = 2 >> (k & 31), hi = 256 >> (k & 31);
            sc->lower_cap = (float)(lo > 1 ? lo : 1);
            sc->upper_cap = (float)(hi > 1 ? hi : 1);
        } else {
            sc->lower_cap = 2.0f;
            sc->upper_cap = 256.0f;
        }
        if (sc->cooldown > 0u) --sc->cooldown;
    }
    sc->frame_idx += 1u;
    sc->epoch += 1u;
}

// refreshModel (SUB:80-105; LOB:410-440) over the tiles bid, bid + nblk, ... reset: the automatic reset's, which
// also sets T := 1 everywhere (SUB:592). outside: pixels outside the ROI get zero samples
// (initialization writes every sample of the model, so that its memory need not be cleared first).
// Bound by the sample stores and the draws: with a table in LDS for the position (a walk of up to 48
// entries before) and the tile's records 1305 -> 126 us (4.4 TB/s) for the 553 MB of a
// 1280x720 RGB model.
template <int C, int ALGO>
LV_D void refresh_body(const View& v, uint32_t bid, uint32_t nblk, int reset, float frac, int force_fg, uint32_t frame,
                       uint32_t ev, int outside) {
    RefreshTile& t = sweep_lds().refresh;
    constexpr int LW = RefreshTile::LW, LH = RefreshTile::LH;
    const uint32_t N = (uint32_t)v.N;
    const uint32_t nref = frac < 1.0f ? (uint32_t)(frac * (float)N) : N;
    uint32_t start = 0;
    if (frac < 1.0f) {
        uint32_t d[4];
        draw4(v.seed_lo, v.seed_hi, v.stream_id, frame, PH_REFRESH, ev, 0xFFFFFFFFu, 0, d);
        start = d[0] % N;
    }
    for (uint32_t i = threadIdx.x; i < 512u; i += TPB) {
        int ox, oy;
        sample_offset_7x7(i, ox, oy);
        t.pos[i] = (uint8_t)((ox + 3) | ((oy + 3) << 4));
    }
    const uint32_t ntx = (uint32_t)((v.W + TW - 1) / TW), ntiles = ntx * (uint32_t)((v.H + TH - 1) / TH);
    for (uint32_t tile = bid; tile < ntiles; tile += nblk) {
        const int x0 = (int)(tile % ntx) * TW, y0 = (int)(tile / ntx) * TH;
        __syncthreads();  // the previous tile's readers are done
        for (int i = threadIdx.x; i < LW * LH; i += TPB) {
            const int gx = x0 - 3 + i % LW, gy = y0 - 3 + i / LW;
            t.ok[i] = 0;
            if (gx < 2 || gy < 2 || gx >= v.W - 2 || gy >= v.H - 2) continue;  // positions are clamped inside
            const size_t q = (size_t)gy * v.W + gx;
            uint32_t col[C], desc[C];
#pragma unroll
            for (int c = 0; c < C; ++c) {
                col[c] = *at(v.last_color, q * C + c);
                if constexpr (ALGO == kLOBSTER) {
                    uint32_t taps[4];
                    taps_from_global<C>(v.last_color, v.W, gx, gy, c, taps);
                    desc[c] = lbsp_threshold_sad(taps, col[c], *at(v.sc->lut, col[c]));
                } else {
                    desc[c] = *at(v.last_desc, q * C + c);
                }
            }
            uint64_t ra;
            uint32_t rb;
            encode_raw<C>(col, desc, ra, rb);
            t.w0[i] = (uint32_t)ra;
            if constexpr (C == 3) {
                t.w1[i] = (uint32_t)(ra >> 32);
                t.w2[i] = rb;
            }
            t.ok[i] = force_fg || !*at(v.last_fg, q);
        }
        __syncthreads();
        const int x = x0 + (int)threadIdx.x % TW, y = y0 + (int)threadIdx.x / TW;
        if (x >= v.W || y >= v.H) continue;
        const uint32_t p = (uint32_t)(y * v.W + x);
        if (reset) *at(v.T, p) = 1.0f;
        const bool in = *at(v.roi, p) != 0 && (force_fg || !*at(v.last_fg, p));
        const bool zero = outside && !*at(v.roi, p);
        if (!in && !zero) continue;
        uint32_t d[4], slot = start;
        for (uint32_t j = 0; j < nref; ++j) {
            if ((j & 3u) == 0) draw4(v.seed_lo, v.seed_hi, v.stream_id, frame, PH_REFRESH, ev, p, j >> 2, d);
            const uint32_t o = t.pos[d[j & 3u] & 511u];
            int sx = x + (int)(o & 15u) - 3, sy = y + (int)(o >> 4) - 3;
            clamp_coords(sx, sy, 2, v.W, v.H);
            const int li = in ? (sy - y0 + 3) * LW + (sx - x0 + 3) : 0;
            if (zero || t.ok[li]) {
                uint64_t ra = t.w0[li];
                uint32_t rb = 0;
                if constexpr (C == 3) {
                    ra |= (uint64_t)t.w1[li] << 32;
                    rb = t.w2[li];
                }
                store_raw<C>(v, slot, p, zero ? 0ull : ra, zero ? 0u : rb);
            }
            slot = slot + 1u == N ? 0u : slot + 1u;
        }
    }
}

// the automatic reset the controller asked for in this step, by the blocks of the dilation (a launch
// of its own, or blocks of their own, cost 9 to 30 us per step of a 64-stream batch with nothing pending)
template <int C>
LV_D void refresh_pending(const View& v, uint32_t bid, uint32_t nblk) {
    __syncthreads();  // the dilation's readers of the shared LDS are done
    refresh_body<C, kSuBSENSE>(v, bid, nblk, 1, v.sc->refresh_frac, v.sc->refresh_force_fg, v.sc->refresh_frame,
                               v.sc->refresh_ev, 0);
}

// initial descriptors of the LBSP base (LBS:31-63): strict bounds x>2 && y>2 && x<W-2 && y<H-2
template <int C>
LV_D void init_desc_body(const View& v, const uint8_t* img, uint32_t bid) {
    __shared__ FrameTile<C> tile;
    __shared__ alignas(8) LbspLimits lut[256];
    const int ntx = (v.W + TW - 1) / TW;
    const int x0 = ((int)bid % ntx) * TW, y0 = ((int)bid / ntx) * TH;
    load_frame_tile<C>(tile, img, v.W, v.H, x0, y0);
    load_lut(lut, v.sc);
    __syncthreads();
    const int lx = threadIdx.x % TW, ly = threadIdx.x / TW, x = x0 + lx, y = y0 + ly;
    if (x >= v.W || y >= v.H) return;
    const uint32_t p = (uint32_t)(y * v.W + x);
    const bool roi = *at(v.roi, p) != 0, in = roi && x > 2 && y > 2 && x < v.W - 2 && y < v.H - 2;
    uint32_t taps[C][4];
    tile_taps(tile, lx, ly, taps);
    const uint32_t centre = tile_colour(tile, lx + 2, ly + 2);
#pragma unroll
    for (int c = 0; c < C; ++c) {
        const uint32_t ref = (centre >> (8 * c)) & 255u;
        *at(v.last_desc, p * C + c) = (uint16_t)(in ? lbsp_threshold_packed(taps[c], lut[ref]) : 0u);
        *at(v.last_color, p * C + c) = (uint8_t)(roi ? ref : 0u);
    }
}

// getBackgroundImage / getBackgroundDescriptorsImage (SUB:614-649): float sum of v/N in sample
// order, then saturate_cast (round half to even)
template <int C, bool DESC>
LV_D void background_body(const View& v, void* out, uint32_t bid) {
    const uint32_t p = bid * TPB + threadIdx.x;
    if (p >= v.npx) return;
    float acc[C];
#pragma unroll
    for (int c = 0; c < C; ++c) acc[c] = 0.0f;
    const float fN = (float)v.N, inv = 1.0f / fN;
    const uint32_t* rec = rec_base(v, p);
#pragma unroll 5
    for (int s = 0; s < v.N; ++s, rec += kSampleStride<C>) {
        uint64_t ra;
        uint32_t rb;
        fetch_at<C>(rec, ra, rb);
        uint32_t col[C], desc[C];
        decode_raw<C>(ra, rb, col, desc);
#pragma unroll
        for (int c = 0; c < C; ++c) acc[c] += quot((float)(DESC ? desc[c] : col[c]), fN, inv);
    }
#pragma unroll
    for (int c = 0; c < C; ++c) {
        if constexpr (DESC) {
            const float r = rintf(acc[c]);
            ((uint16_t*)out)[(size_t)p * C + c] = (uint16_t)(r < 0.f ? 0.f : r > 65535.f ? 65535.f : r);
        } else {
            ((uint8_t*)out)[(size_t)p * C + c] = sat_u8(acc[c]);
        }
    }
}

// stand-alone LBSP map (LBSP::compute2, LBSP.cpp:102-123) with the absolute threshold t, through either form of
// the threshold test
template <int C, bool PACKED, int FORM>
__global__ void __launch_bounds__(TPB) k_lbsp_abs(const uint8_t* __restrict__ img, int W, int H, uint32_t t,
                                                uint16_t* __restrict__ out) {
    __shared__ FrameTile<C> tile;
    const int ntx = (W + TW - 1) / TW, nty = (H + TH - 1) / TH;
    const int tid = xcd_tile((int)blockIdx.x, ntx * nty);
    const int x0 = (tid % ntx) * TW, y0 = (tid / ntx) * TH;
    const int lx = threadIdx.x % TW, ly = threadIdx.x / TW, x = x0 + lx, y = y0 + ly;
    if constexpr (FORM == kLbspEmpty) {
        if (x < W && y < H)
            for (int c = 0; c < C; ++c) out[((size_t)y * W + x) * C + c] = 0;
        return;
    }
    load_frame_tile<C, std::conditional_t<FORM == kLbsp64, int64_t, int>>(tile, img, W, H, x0, y0);
    __syncthreads();
    if (x >= W || y >= H) return;
    const bool in = x >= 2 && y >= 2 && x < W - 2 && y < H - 2;
    uint32_t taps[C][4];
    tile_taps(tile, lx, ly, taps);
    const uint32_t centre = tile_colour(tile, lx + 2, ly + 2);
#pragma unroll
    for (int c = 0; c < C; ++c) {
        const uint32_t ref = (centre >> (8 * c)) & 255u;
        uint16_t d = 0;
        if (in) d = (uint16_t)(PACKED ? lbsp_threshold_packed(taps[c], lbsp_limits(ref, min(t, 255u))) : lbsp_threshold_sad(taps[c], ref, t));
        out[((size_t)y * W + x) * C + c] = d;
    }
}

// RNG self-check: draws of the apply stream for pixels [0, n)
__global__ void k_rng_probe(View v, uint32_t frame, uint32_t phase, uint32_t ev, uint32_t n, uint32_t* out) {
    const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n) return;
    uint32_t d[4];
    draw4(v.seed_lo, v.seed_hi, v.stream_id, frame, phase, ev, p, 0, d);
    for (int i = 0; i < 4; ++i) out[(size_t)p * 4 + i] = d[i];
}

// sticky device error bits of each stream of a step, gathered for one copy to the host
__global__ void k_gather_errors(const View* __restrict__ views, int n, uint32_t* __restrict__ out) {
    const int i = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (i < n) out[i] = __hip_atomic_load(&views[i].sc->err_flags, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// ==============================================================================================
// kernel entry points. Single stream: the View by value, block id remapped per XCD. Batched: every
// stream of the batch in one launch; a workgroup finds its stream in a per-kernel prefix table of
// block counts (after the XCD remap, so each stream's tiles stay together) and dispatches on the
// stream's channel count.
// ==============================================================================================
struct BatchArgs {
    const View* views;
    const uint32_t* prefix;  // ns+1 block offsets
    int ns;
};

// block bid of nblk of a grid
template <class F>
LV_D void for_batch_block(const BatchArgs& b, uint32_t bid, uint32_t nblk, F&& f) {
    const uint32_t lb = (uint32_t)xcd_tile((int)bid, (int)nblk);
    int lo = 0, hi = b.ns;
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (b.prefix[mid] <= lb) lo = mid;
        else hi = mid;
    }
    // private copy: the fields become uniform registers that stores to the model cannot alias
    const View v = b.views[lo];
    f(v, lb - b.prefix[lo], b.prefix[lo + 1] - b.prefix[lo]);
}

template <class F>
LV_D void for_batch_block(const BatchArgs& b, F&& f) {
    for_batch_block(b, blockIdx.x, gridDim.x, f);
}

// Several kernels take two or three kinds of work in one launch: the small, latency-bound kinds in the
// first blocks, so that they run beside the kind that fills the chip instead of before or after it with a
// launch of their own (4 to 5 us each on an idle chip).
#define LV_SINGLE_BID ((uint32_t)xcd_tile((int)blockIdx.x, (int)gridDim.x)), gridDim.x
// kernels over a list that may fill only the first blocks: in dispatch order, so every XCD gets a share
// (remapped, 700 busy blocks of 4096 would all run on two XCDs)
#define LV_LIST_BID blockIdx.x, gridDim.x

template <int C, int ALGO>
__global__ void __launch_bounds__(TPB) k_describe(View v) { describe_body<C, ALGO>(v, LV_SINGLE_BID); }
// 72 VGPRs at occupancy 7 fit both fetch depths without spilling
#define LV_MATCH_WAVES __attribute__((amdgpu_waves_per_eu(7)))
template <int C, int ALGO, int KF>
__global__ void __launch_bounds__(TPB) LV_MATCH_WAVES k_match(View v) { match_body<C, ALGO, KF>(v, LV_SINGLE_BID); }
// Phase B needs 96 VGPRs. A single stream's grid does not fill the chip at occupancy 6, and the scratch of a kernel
// that spills costs each launch more than the waves give (occupancy 6 against 5: 320x240 14.8 and 12.2 us,
// 3840x2160 128 and 124 us). A batch's grid does (64 mixed streams: 635 and 654 us).
template <int C, int ALGO, int KF>
__global__ void __launch_bounds__(TPB) __attribute__((amdgpu_waves_per_eu(5))) k_match_seq(View v) {
    match_seq_body<C, ALGO, KF>(v, LV_LIST_BID);
}
template <int C, int ALGO, int KIND>
__global__ void __launch_bounds__(TPB) k_fixpoint(View v, uint32_t k, uint32_t cap) {
    fixpoint_body<C, ALGO, KIND>(v, LV_LIST_BID, k, cap);
}

// the zones' closing and the frame-level cells beside the model update (SuBSENSE; nzone = ncell = 0 else)
template <int C, int ALGO>
__global__ void __launch_bounds__(TPB) __attribute__((amdgpu_waves_per_eu(7))) k_update(View v, uint32_t nzone, uint32_t ncell) {
    const uint32_t b = blockIdx.x, rest = gridDim.x - nzone - ncell;
    if constexpr (ALGO == kSuBSENSE) {
        if (b < nzone) {
            zone_close_body(v, b, nzone);
            return;
        }
        if (b < nzone + ncell) {
            downsample_body<C>(v, b - nzone, ncell);
            return;
        }
    }
    update_body<C, ALGO>(v, (uint32_t)xcd_tile((int)(b - nzone - ncell), (int)rest), rest);
}
__global__ void __launch_bounds__(TPB) k_zone_close(View v) { zone_close_body(v, LV_SINGLE_BID); }
__global__ void __launch_bounds__(TPB) k_zone_link(View v) { zone_link_body(v, LV_SINGLE_BID); }
// the frame controller (ndecide = 1) beside the zones' holes
__global__ void __launch_bounds__(TPB) k_zone_holes(View v, uint32_t ndecide) {
    if (blockIdx.x < ndecide) decide_body(v, 0u, 1u);
    else zone_holes_body(v, blockIdx.x - ndecide, gridDim.x - ndecide);
}
template <bool SUB>
__global__ void __launch_bounds__(TPB) k_median(View v) { median_body<SUB>(v, LV_SINGLE_BID); }
template <int C>
__global__ void __launch_bounds__(TPB) k_dilate_final(View v) {
    const uint32_t bid = (uint32_t)xcd_tile((int)blockIdx.x, (int)gridDim.x);
    const int pending = v.sc->refresh_pending;  // loaded before the tile, not behind its stores
    dilate_final_body(v, bid, gridDim.x);
    if (pending) refresh_pending<C>(v, bid, gridDim.x);
}
template <int C, int ALGO>
__global__ void __launch_bounds__(TPB) k_refresh(View v, float frac, int force_fg, uint32_t frame, uint32_t ev,
                                               int outside) {
    refresh_body<C, ALGO>(v, LV_SINGLE_BID, 0, frac, force_fg, frame, ev, outside);
}
template <int C>
__global__ void __launch_bounds__(TPB) k_init_desc(View v, const uint8_t* img) {
    init_desc_body<C>(v, img, (uint32_t)xcd_tile((int)blockIdx.x, (int)gridDim.x));
}
template <int C, bool DESC>
__global__ void __launch_bounds__(TPB) k_background(View v, void* out) { background_body<C, DESC>(v, out, blockIdx.x); }

// batched entry points (SuBSENSE; streams of 1 and 3 channels may be mixed)
#define LV_BATCH_C(body, ...)                                                                \
    for_batch_block(b, [&](const View& v, uint32_t bid, uint32_t nblk) {                     \
        if (v.C == 3) body<3 __VA_OPT__(, ) __VA_ARGS__>(v, bid, nblk);                       \
        else body<1 __VA_OPT__(, ) __VA_ARGS__>(v, bid, nblk);                                \
    })
__global__ void __launch_bounds__(TPB) kb_describe(BatchArgs b) { LV_BATCH_C(describe_body, kSuBSENSE); }
template <int KF>
__global__ void __launch_bounds__(TPB) LV_MATCH_WAVES kb_match(BatchArgs b) {
    LV_BATCH_C(match_body, kSuBSENSE, KF, 3);
}
template <int KF>
__global__ void __launch_bounds__(TPB) __attribute__((amdgpu_waves_per_eu(6))) kb_match_seq(BatchArgs b) {
    LV_BATCH_C(match_seq_body, kSuBSENSE, KF);
}
template <int KIND>
__global__ void __launch_bounds__(TPB) kb_fixpoint(BatchArgs b, uint32_t k, uint32_t cap) {
    for_batch_block(b, [&](const View& v, uint32_t bid, uint32_t nblk) {
        if (v.C == 3) fixpoint_body<3, kSuBSENSE, KIND>(v, bid, nblk, k, cap);
        else fixpoint_body<1, kSuBSENSE, KIND>(v, bid, nblk, k, cap);
    });
}
// The general path of the cells (ten column weights in doubles) for two channel counts makes this kernel spill 11
// VGPRs, 48 bytes of scratch a lane; without the cells it takes 72 VGPRs and none.
__global__ void __launch_bounds__(TPB) __attribute__((amdgpu_waves_per_eu(7))) kb_update(BatchArgs zone, uint32_t nzone, BatchArgs cell, uint32_t ncell,
                                                 BatchArgs tile) {
    const uint32_t b = blockIdx.x;
    if (b < nzone) {
        for_batch_block(zone, b, nzone, zone_close_body);
    } else if (b < nzone + ncell) {
        for_batch_block(cell, b - nzone, ncell, [&](const View& v, uint32_t bid, uint32_t nblk) {
            if (v.C == 3) downsample_body<3>(v, bid, nblk);
            else downsample_body<1>(v, bid, nblk);
        });
    } else {
        for_batch_block(tile, b - nzone - ncell, gridDim.x - nzone - ncell,
                        [&](const View& v, uint32_t bid, uint32_t nblk) {
                            if (v.C == 3) update_body<3, kSuBSENSE>(v, bid, nblk);
                            else update_body<1, kSuBSENSE>(v, bid, nblk);
                        });
    }
}
__global__ void __launch_bounds__(TPB) kb_zone_link(BatchArgs b) { for_batch_block(b, zone_link_body); }
__global__ void __launch_bounds__(TPB) kb_zone_holes(BatchArgs one, uint32_t none, BatchArgs zone) {
    if (blockIdx.x < none) for_batch_block(one, blockIdx.x, none, decide_body);
    else for_batch_block(zone, blockIdx.x - none, gridDim.x - none, zone_holes_body);
}
__global__ void __launch_bounds__(TPB) kb_median(BatchArgs b) { for_batch_block(b, median_body<true>); }
__global__ void __launch_bounds__(TPB) kb_dilate_final(BatchArgs b) {
    for_batch_block(b, [&](const View& v, uint32_t bid, uint32_t nblk) {
        const int pending = v.sc->refresh_pending;
        dilate_final_body(v, bid, nblk);
        if (!pending) return;
        if (v.C == 3) refresh_pending<3>(v, bid, nblk);
        else refresh_pending<1>(v, bid, nblk);
    });
}

// ==============================================================================================
// host-side launchers
// ==============================================================================================
static inline unsigned cdiv(size_t a, size_t b) { return (unsigned)((a + b - 1) / b); }

uint32_t cont_stripe_slots(int W, int H) {
    const size_t tiles = (size_t)cdiv(W, TW) * cdiv(H, TH);
    return (uint32_t)((tiles + kContStripes - 1) / kContStripes * TPB);
}

void kernel_grids(const View& v, const StepOptions& opt, uint32_t g[kNumGrids]) {
    g[kGridTile] = cdiv(v.W, TW) * cdiv(v.H, TH);
    g[kGridPost] = cdiv(v.W, PW) * cdiv(v.H, PH);
    g[kGridZone] = cdiv((size_t)cdiv(v.W, ZS) * cdiv(v.H, ZS), ZPB);
    g[kGridLink] = cdiv((size_t)2 * cdiv(v.W, ZS) * cdiv(v.H, ZS), ZPB);
    g[kGridCell] = !v.lr_scaling ? 0u : cdiv((size_t)v.dsW * v.dsH, TPB);
    g[kGridOne] = 1u;
    // single stream: a block per 1024 pixels (16 groups each; the worklists hold a few per cent of them)
    g[kGridFix] = opt.fixpoint_blocks > 0 ? (uint32_t)opt.fixpoint_blocks
                                          : std::max(32u, std::min(1024u, cdiv(v.npx, 1024)));
    if (opt.fix_px_per_block > 0) g[kGridFix] = std::min(g[kGridFix], cdiv(v.npx, (size_t)opt.fix_px_per_block));
    // single stream: a block per 256 pixels, at most what covers group_limit entries in one round
    g[kGridCont] = opt.cont_blocks > 0 ? (uint32_t)opt.cont_blocks
                                       : std::max(64u, std::min(kGroupLimit / (TPB / kGroup), cdiv(v.npx, TPB)));
    if (opt.cont_px_per_block > 0) g[kGridCont] = std::min(g[kGridCont], cdiv(v.npx, (size_t)opt.cont_px_per_block));
}

template <int C, int ALGO>
static void frame_step_t(const View& v, const StepOptions& opt, hipStream_t st) {
    uint32_t g[kNumGrids];
    kernel_grids(v, opt, g);
    if (opt.timed_stage == 2) (void)hipEventRecord(opt.ev_begin, st);
    hipLaunchKernelGGL((k_describe<C, ALGO>), dim3(g[kGridTile]), dim3(TPB), 0, st, v);
    if (opt.timed_stage == 1) (void)hipEventRecord(opt.ev_begin, st);
    if (opt.fetch_depth == 4) hipLaunchKernelGGL((k_match<C, ALGO, 4>), dim3(g[kGridTile]), dim3(TPB), 0, st, v);
    else hipLaunchKernelGGL((k_match<C, ALGO, 2>), dim3(g[kGridTile]), dim3(TPB), 0, st, v);
    if (opt.timed_stage == 1) (void)hipEventRecord(opt.ev_end, st);
    // phase B finishes the scans phase A cut; it exits at once when there are none
    if (opt.fetch_depth == 4) hipLaunchKernelGGL((k_match_seq<C, ALGO, 4>), dim3(g[kGridCont]), dim3(TPB), 0, st, v);
    else hipLaunchKernelGGL((k_match_seq<C, ALGO, 2>), dim3(g[kGridCont]), dim3(TPB), 0, st, v);
    // the second iteration's worklist is about a hundredth of the first's to a tenth: on small frames the tail, one
    // workgroup, takes it. Step with one / two launches, us: 320x240 81.2 / 82.1, 480x360 85.1 / 86.0, 640x480
    // 97.1 / 97.1, 800x600 116.2 / 116.7; but 960x540 grey 159.9 / 124.8, 880x660 232 / 165, 1280x720 305 / 190
    // with more change in the frame, so the line lies where one launch still gains.
    const uint32_t launches = opt.fixpoint_launches >= 0 ? (uint32_t)opt.fixpoint_launches : v.npx < 200000u ? 1u : 2u;
    const uint32_t cap = (uint32_t)opt.tail_cap;
    for (uint32_t k = 1; k < launches; ++k)
        hipLaunchKernelGGL((k_fixpoint<C, ALGO, kFixMore>), dim3(g[kGridFix]), dim3(TPB), 0, st, v, k, cap);
    if (launches) hipLaunchKernelGGL((k_fixpoint<C, ALGO, kFixLast>), dim3(g[kGridFix]), dim3(TPB), 0, st, v, launches, cap);
    else hipLaunchKernelGGL((k_fixpoint<C, ALGO, kFixTail>), dim3(1), dim3(TPB), 0, st, v, 1u, cap);
    constexpr bool kSub = ALGO == kSuBSENSE;
    const uint32_t nzone = kSub ? g[kGridZone] : 0u, ncell = kSub ? g[kGridCell] : 0u;
    if (opt.timed_stage == 3) (void)hipEventRecord(opt.ev_begin, st);
    hipLaunchKernelGGL((k_update<C, ALGO>), dim3(nzone + ncell + g[kGridTile]), dim3(TPB), 0, st, v, nzone, ncell);
    if (opt.timed_stage == 3) (void)hipEventRecord(opt.ev_end, st);
    if constexpr (kSub) {
        hipLaunchKernelGGL(k_zone_link, dim3(g[kGridLink]), dim3(TPB), 0, st, v);
        hipLaunchKernelGGL(k_zone_holes, dim3(1 + nzone), dim3(TPB), 0, st, v, 1u);
        hipLaunchKernelGGL((k_median<true>), dim3(g[kGridPost]), dim3(TPB), 0, st, v);
        hipLaunchKernelGGL((k_dilate_final<C>), dim3(g[kGridPost]), dim3(TPB), 0, st, v);
    } else {
        hipLaunchKernelGGL((k_median<false>), dim3(g[kGridPost]), dim3(TPB), 0, st, v);
    }
    if (opt.timed_stage == 2) (void)hipEventRecord(opt.ev_end, st);
}

void frame_step(const View& v, const StepOptions& opt, hipStream_t st) {
    if (v.algo == kSuBSENSE) {
        if (v.C == 3) frame_step_t<3, kSuBSENSE>(v, opt, st);
        else frame_step_t<1, kSuBSENSE>(v, opt, st);
    } else {
        if (v.C == 3) frame_step_t<3, kLOBSTER>(v, opt, st);
        else frame_step_t<1, kLOBSTER>(v, opt, st);
    }
}

// one SuBSENSE step of every stream of a batch; d_views holds the streams' Views (with their
// per-frame inputs), prefix[k] the (ns+1) block offsets of grid kind k, total[k] their sums
void batch_step(const View* d_views, int ns, const uint32_t* const prefix[kNumGrids], const uint32_t total[kNumGrids],
                const StepOptions& opt, hipStream_t st) {
    auto args = [&](int kind) { return BatchArgs{d_views, prefix[kind], ns}; };
    if (opt.timed_stage == 2) (void)hipEventRecord(opt.ev_begin, st);
    hipLaunchKernelGGL(kb_describe, dim3(total[kGridTile]), dim3(TPB), 0, st, args(kGridTile));
    if (opt.timed_stage == 1) (void)hipEventRecord(opt.ev_begin, st);
    if (opt.fetch_depth == 4) hipLaunchKernelGGL(kb_match<4>, dim3(total[kGridTile]), dim3(TPB), 0, st, args(kGridTile));
    else hipLaunchKernelGGL(kb_match<2>, dim3(total[kGridTile]), dim3(TPB), 0, st, args(kGridTile));
    if (opt.timed_stage == 1) (void)hipEventRecord(opt.ev_end, st);
    if (opt.fetch_depth == 4) hipLaunchKernelGGL(kb_match_seq<4>, dim3(total[kGridCont]), dim3(TPB), 0, st, args(kGridCont));
    else hipLaunchKernelGGL(kb_match_seq<2>, dim3(total[kGridCont]), dim3(TPB), 0, st, args(kGridCont));
    const uint32_t launches = (uint32_t)opt.fixpoint_launches, cap = (uint32_t)opt.tail_cap;
    for (uint32_t k = 1; k <= launches; ++k)
        hipLaunchKernelGGL(kb_fixpoint<kFixMore>, dim3(total[kGridFix]), dim3(TPB), 0, st, args(kGridFix), k, cap);
    hipLaunchKernelGGL(kb_fixpoint<kFixTail>, dim3(total[kGridOne]), dim3(TPB), 0, st, args(kGridOne), launches + 1u, cap);
    const uint32_t nzone = total[kGridZone], ncell = total[kGridCell], none = total[kGridOne];
    if (opt.timed_stage == 3) (void)hipEventRecord(opt.ev_begin, st);
    hipLaunchKernelGGL(kb_update, dim3(nzone + ncell + total[kGridTile]), dim3(TPB), 0, st, args(kGridZone), nzone,
                       args(kGridCell), ncell, args(kGridTile));
    if (opt.timed_stage == 3) (void)hipEventRecord(opt.ev_end, st);
    hipLaunchKernelGGL(kb_zone_link, dim3(total[kGridLink]), dim3(TPB), 0, st, args(kGridLink));
    hipLaunchKernelGGL(kb_zone_holes, dim3(none + nzone), dim3(TPB), 0, st, args(kGridOne), none, args(kGridZone));
    hipLaunchKernelGGL(kb_median, dim3(total[kGridPost]), dim3(TPB), 0, st, args(kGridPost));
    hipLaunchKernelGGL(kb_dilate_final, dim3(total[kGridPost]), dim3(TPB), 0, st, args(kGridPost));
    if (opt.timed_stage == 2) (void)hipEventRecord(opt.ev_end, st);
}

void launch_refresh(const View& v, float frac, int force_fg, uint32_t frame, uint32_t ev, int outside, hipStream_t st) {
    const dim3 g(cdiv(v.W, TW) * cdiv(v.H, TH)), t(TPB);
    if (v.algo == kSuBSENSE) {
        if (v.C == 3) hipLaunchKernelGGL((k_refresh<3, kSuBSENSE>), g, t, 0, st, v, frac, force_fg, frame, ev, outside);
        else hipLaunchKernelGGL((k_refresh<1, kSuBSENSE>), g, t, 0, st, v, frac, force_fg, frame, ev, outside);
    } else {
        if (v.C == 3) hipLaunchKernelGGL((k_refresh<3, kLOBSTER>), g, t, 0, st, v, frac, force_fg, frame, ev, outside);
        else hipLaunchKernelGGL((k_refresh<1, kLOBSTER>), g, t, 0, st, v, frac, force_fg, frame, ev, outside);
    }
}

void launch_init_desc(const View& v, const uint8_t* img, hipStream_t st) {
    const unsigned b = cdiv(v.W, TW) * cdiv(v.H, TH);
    if (v.C == 3) hipLaunchKernelGGL(k_init_desc<3>, dim3(b), dim3(TPB), 0, st, v, img);
    else hipLaunchKernelGGL(k_init_desc<1>, dim3(b), dim3(TPB), 0, st, v, img);
}

void launch_background(const View& v, uint8_t* out_img, hipStream_t st) {
    const unsigned b = cdiv(v.npx, TPB);
    if (v.C == 3) hipLaunchKernelGGL((k_background<3, false>), dim3(b), dim3(TPB), 0, st, v, (void*)out_img);
    else hipLaunchKernelGGL((k_background<1, false>), dim3(b), dim3(TPB), 0, st, v, (void*)out_img);
}
void launch_background_desc(const View& v, uint16_t* out_desc, hipStream_t st) {
    const unsigned b = cdiv(v.npx, TPB);
    if (v.C == 3) hipLaunchKernelGGL((k_background<3, true>), dim3(b), dim3(TPB), 0, st, v, (void*)out_desc);
    else hipLaunchKernelGGL((k_background<1, true>), dim3(b), dim3(TPB), 0, st, v, (void*)out_desc);
}

template <int C, bool PACKED>
static void lbsp_abs_t(const uint8_t* img, int W, int H, uint32_t t, uint16_t* out, hipStream_t st) {
    const dim3 g(cdiv(W, TW) * cdiv(H, TH)), b(TPB);
    switch (lbsp_form(W, H, C)) {
    case kLbspEmpty: hipLaunchKernelGGL((k_lbsp_abs<C, PACKED, kLbspEmpty>), g, b, 0, st, img, W, H, t, out); break;
    case kLbsp32: hipLaunchKernelGGL((k_lbsp_abs<C, PACKED, kLbsp32>), g, b, 0, st, img, W, H, t, out); break;
    case kLbsp64: hipLaunchKernelGGL((k_lbsp_abs<C, PACKED, kLbsp64>), g, b, 0, st, img, W, H, t, out); break;
    }
}
void launch_lbsp_abs(const uint8_t* img, int W, int H, int C, uint32_t t, uint16_t* out, bool packed, hipStream_t st) {
    // RGB tiles give their taps packed, so the per-tap form would take them apart again. A call, per-tap / packed,
    // us: RGB 1920x1080 29.2 / 27.9, 3840x2160 72.6 / 67.5; grey 1920x1080 18.7 / 20.3
    if (C == 3) lbsp_abs_t<3, true>(img, W, H, t, out, st);
    else (packed ? lbsp_abs_t<1, true> : lbsp_abs_t<1, false>)(img, W, H, t, out, st);
}

// the SuBSENSE hole-filling and median kernels alone, on a raw mask
void launch_postprocess_probe(const View& view, uint8_t* raw, hipStream_t st) {
    View v = view;
    v.dec = v.last_raw = raw;
    uint32_t g[kNumGrids];
    kernel_grids(v, StepOptions{}, g);
    hipLaunchKernelGGL(k_zone_close, dim3(g[kGridZone]), dim3(TPB), 0, st, v);
    hipLaunchKernelGGL(k_zone_link, dim3(g[kGridLink]), dim3(TPB), 0, st, v);
    hipLaunchKernelGGL(k_zone_holes, dim3(g[kGridZone]), dim3(TPB), 0, st, v, 0u);
    hipLaunchKernelGGL((k_median<true>), dim3(g[kGridPost]), dim3(TPB), 0, st, v);
}

void launch_gather_errors(const View* d_views, int n, uint32_t* d_out, hipStream_t st) {
    if (n > 0) hipLaunchKernelGGL(k_gather_errors, dim3(cdiv((size_t)n, 256)), dim3(256), 0, st, d_views, n, d_out);
}

void launch_rng_probe(const View& v, uint32_t frame, uint32_t phase, uint32_t ev, uint32_t n, uint32_t* out,
                      hipStream_t st) {
    hipLaunchKernelGGL(k_rng_probe, dim3(cdiv(n, 256)), dim3(256), 0, st, v, frame, phase, ev, n, out);
}

}  // namespace lvbgs
