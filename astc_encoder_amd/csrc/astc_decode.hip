// astc_decode.hip -- ASTC LDR decoder kernel (one lane per block).
//
// Decodes the single-partition LDR subset of the ASTC specification to RGBA8:
// any block size up to 12x12, any 2D weight grid up to the block size with the
// specification's bilinear infill, every weight and endpoint quantisation (bits,
// trits, quints), one or two weight planes, colour endpoint modes 0 / 4 / 8 / 12
// (LDR luminance, luminance+alpha, RGB, RGBA direct, with blue contraction), and
// LDR void-extent blocks.  Anything else (multiple partitions, HDR, reserved
// modes) decodes to the error colour magenta.  Each texel is
// ((C0 * (64 - w) + C1 * w + 32) >> 6) >> 8 with C = endpoint * 257.
// It decodes every block the encoder produces and is used to check encoded
// textures at throughput (PSNR) without a round trip to the host.
//
// 4x4 and 6x6 images run decode_kernel<4> / <6>, whose waves take 64 blocks in
// the encoder's two layouts (4x4 weight grid, one plane, 8-bit endpoints) through
// a straight-line path (decode_fixed) and any others through the general one;
// other block sizes run decode_kernel<0>, the general path alone.
#include "astc_internal.h"

namespace astc {

namespace {

constexpr int kDecThreads = 256;
constexpr int kMaxWeights = 64;

__device__ __forceinline__ uint32_t get_bits(uint64_t lo, uint64_t hi, int pos, int n) {
    uint64_t v;
    if (pos >= 64) v = hi >> (pos - 64);
    else if (pos == 0) v = lo;
    else v = (lo >> pos) | (hi << (64 - pos));
    return uint32_t(v) & ((1u << n) - 1u);
}

__device__ __forceinline__ int ise_bit_count(int q, int count) {
    const QuantLevel L = kQuantLevels[q];
    if (L.trits) return ((8 + 5 * L.bits) * count + 4) / 5;
    if (L.quints) return ((7 + 3 * L.bits) * count + 2) / 3;
    return L.bits * count;
}

// Decode `count` ISE values of method q starting at bit `pos`; value i goes to
// out[i * kDecThreads] (a per-lane column in LDS).
__device__ void ise_decode(uint64_t lo, uint64_t hi, int pos, int count, int q, const uint32_t* trit_lut,
                           const uint16_t* quint_lut, uint8_t* out) {
    const QuantLevel L = kQuantLevels[q];
    const int b = L.bits;
    if (L.trits) {
        for (int g = 0; g < count; g += 5) {
            uint32_t m[5] = {0, 0, 0, 0, 0}, T = 0;
            int tshift = 0;
            for (int i = 0; i < 5 && g + i < count; ++i) {
                const int tb = (i == 2 || i == 4) ? 1 : 2;
                m[i] = get_bits(lo, hi, pos, b);
                pos += b;
                T |= get_bits(lo, hi, pos, tb) << tshift;
                pos += tb;
                tshift += tb;
            }
            const uint32_t t = trit_lut[T];
            for (int i = 0; i < 5 && g + i < count; ++i)
                out[(g + i) * kDecThreads] = uint8_t((((t >> (i < 4 ? 8 * i : 28)) & 3u) << b) | m[i]);
        }
    } else if (L.quints) {
        for (int g = 0; g < count; g += 3) {
            uint32_t m[3] = {0, 0, 0}, Q = 0;
            int qshift = 0;
            for (int i = 0; i < 3 && g + i < count; ++i) {
                const int qb = i == 0 ? 3 : 2;
                m[i] = get_bits(lo, hi, pos, b);
                pos += b;
                Q |= get_bits(lo, hi, pos, qb) << qshift;
                pos += qb;
                qshift += qb;
            }
            const uint32_t t = quint_lut[Q];
            for (int i = 0; i < 3 && g + i < count; ++i)
                out[(g + i) * kDecThreads] = uint8_t((((t >> (3 * i)) & 7u) << b) | m[i]);
        }
    } else {
        for (int i = 0; i < count; ++i, pos += b) out[i * kDecThreads] = uint8_t(get_bits(lo, hi, pos, b));
    }
}

// ISE symbol -> 0..255 colour value (specification colour unquantisation)
__device__ uint32_t unquant_color(int q, uint32_t sym) {
    const QuantLevel L = kQuantLevels[q];
    const int b = L.bits;
    if (!L.trits && !L.quints) {  // bit replication to 8 bits
        uint32_t acc = 0;
        int n = 0;
        while (n < 8) {
            acc = (acc << b) | sym;
            n += b;
        }
        return acc >> (n - 8);
    }
    const uint32_t D = sym >> b, low = sym & ((1u << b) - 1u);
    const uint32_t a = low & 1u, bb = (low >> 1) & 1u, cc = (low >> 2) & 1u, dd = (low >> 3) & 1u,
                   ee = (low >> 4) & 1u, ff = (low >> 5) & 1u;
    const uint32_t A = a ? 0x1FFu : 0u;
    uint32_t B = 0, C = 0;
    if (L.trits) {
        switch (b) {
        case 1: C = 204; break;
        case 2: C = 93; B = (bb << 8) | (bb << 4) | (bb << 2) | (bb << 1); break;
        case 3: C = 44; B = (cc << 8) | (bb << 7) | (cc << 3) | (bb << 2) | (cc << 1) | bb; break;
        case 4: C = 22; B = (dd << 8) | (cc << 7) | (bb << 6) | (dd << 2) | (cc << 1) | bb; break;
        case 5: C = 11; B = (ee << 8) | (dd << 7) | (cc << 6) | (bb << 5) | (ee << 1) | dd; break;
        default: C = 5; B = (ff << 8) | (ee << 7) | (dd << 6) | (cc << 5) | (bb << 4) | ff; break;
        }
    } else {
        switch (b) {
        case 1: C = 113; break;
        case 2: C = 54; B = (bb << 8) | (bb << 3) | (bb << 2); break;
        case 3: C = 26; B = (cc << 8) | (bb << 7) | (cc << 2) | (bb << 1) | cc; break;
        case 4: C = 13; B = (dd << 8) | (cc << 7) | (bb << 6) | (dd << 1) | cc; break;
        default: C = 6; B = (ee << 8) | (dd << 7) | (cc << 6) | (bb << 5) | ee; break;
        }
    }
    const uint32_t T = (D * C + B) ^ A;
    return (A & 0x80u) | (T >> 2);
}

// ISE symbol -> 0..64 weight (specification weight unquantisation)
__device__ uint32_t unquant_weight(int q, uint32_t sym) {
    const QuantLevel L = kQuantLevels[q];
    const int b = L.bits;
    uint32_t v;
    if (!L.trits && !L.quints) {
        uint32_t acc = 0;
        int n = 0;
        while (n < 6) {
            acc = (acc << b) | sym;
            n += b;
        }
        v = acc >> (n - 6);
    } else if (b == 0) {
        return sym * (L.trits ? 32u : 16u);
    } else {
        const uint32_t D = sym >> b, low = sym & ((1u << b) - 1u);
        const uint32_t A = (low & 1u) ? 0x7Fu : 0u, bb = (low >> 1) & 1u, cc = (low >> 2) & 1u;
        uint32_t B = 0, C = 0;
        if (L.trits) {
            if (b == 1) C = 50;
            else if (b == 2) { C = 23; B = (bb << 6) | (bb << 2) | bb; }
            else { C = 11; B = (cc << 6) | (bb << 5) | (cc << 1) | bb; }
        } else {
            if (b == 1) C = 28;
            else { C = 13; B = (bb << 6) | (bb << 1) | bb; }
        }
        v = (A & 0x20u) | (((D * C + B) ^ A) >> 2);
    }
    return v > 32 ? v + 1 : v;
}

struct Mode { int ok, gw, gh, dual, quant; };

__device__ Mode decode_mode(uint32_t m) {
    Mode r{0, 0, 0, 0, 0};
    int R, H = (m >> 9) & 1, D = (m >> 10) & 1;
    if (m & 3u) {
        R = int(((m & 3u) << 1) | ((m >> 4) & 1u));
        const int A = (m >> 5) & 3, B = (m >> 7) & 3;
        switch ((m >> 2) & 3) {
        case 0: r.gw = B + 4; r.gh = A + 2; break;
        case 1: r.gw = B + 8; r.gh = A + 2; break;
        case 2: r.gw = A + 2; r.gh = B + 8; break;
        default:
            if (m & 0x100u) { r.gw = (B & 1) + 2; r.gh = A + 2; }
            else { r.gw = A + 2; r.gh = (B & 1) + 6; }
        }
    } else {
        if ((m & 0xFu) == 0) return r;
        R = int(((m >> 1) & 6u) | ((m >> 4) & 1u));
        const int A = (m >> 5) & 3, B = (m >> 9) & 3;
        switch ((m >> 7) & 3) {
        case 0: r.gw = 12; r.gh = A + 2; break;
        case 1: r.gw = A + 2; r.gh = 12; break;
        case 2: r.gw = A + 6; r.gh = B + 6; D = 0; H = 0; break;
        default: {
            const int s = (m >> 5) & 3;
            if (s == 0) { r.gw = 6; r.gh = 10; }
            else if (s == 1) { r.gw = 10; r.gh = 6; }
            else return r;
        }
        }
    }
    if (R < 2) return r;
    r.quant = (R - 2) + 6 * H;
    r.dual = D;
    r.ok = 1;
    return r;
}

struct DecodeArgs {
    const uint4* blocks;
    uint32_t* rgba;  // width * height texels
    int width, height, bw, bh, xblocks, nblocks;
    uint32_t xb_magic;  // block row of a block id (block_row)
    int xb_shift;
    const TritQuintDecodeTable* tables;
};

__device__ __forceinline__ void fill_block(const DecodeArgs& a, int x0, int y0, uint32_t c) {
    for (int t = 0; t < a.bh; ++t)
        for (int s = 0; s < a.bw; ++s) {
            const int x = x0 + s, y = y0 + t;
            if (x < a.width && y < a.height) a.rgba[(size_t)y * a.width + x] = c;
        }
}

// The 4-point weight grid's infill over DIM texels (specification, as the
// general path below): texel s takes grid points j and j + 1 with fraction f.
template <int DIM>
struct Infill {
    static constexpr int pos(int s) { return (((1024 + DIM / 2) / (DIM - 1)) * s * 3 + 32) >> 6; }
    static constexpr int j(int s) { return pos(s) >> 4; }
    static constexpr int f(int s) { return pos(s) & 15; }
    // the texel's weight factors on one grid row, byte k the factor (0..16) of
    // grid point k: row 0 is grid row j(t), row 1 the one below
    static constexpr uint32_t taps(int s, int t, int row) {
        const int fs = f(s), ft = f(t);
        const int w11 = (fs * ft + 8) >> 4, w10 = ft - w11, w01 = fs - w11, w00 = 16 - fs - ft + w11;
        const int left = row ? w10 : w00, right = row ? w11 : w01;
        return (uint32_t(left) << (8 * j(s))) | (j(s) < 3 ? uint32_t(right) << (8 * j(s) + 8) : 0u);
    }
};

// Four ISE symbols, one in each byte, to weights 0..64.  QUANT_6: table lookup by
// symbol.  QUANT_12: by trit and high bit, once for each low bit.
template <bool RGBA>
__device__ __forceinline__ uint32_t unquant_weights4(uint32_t trits, uint32_t bits) {
    if (RGBA) {
        constexpr uint32_t lo = uint32_t(unquant_weight_trit(1, 0)) | uint32_t(unquant_weight_trit(1, 1)) << 8 |
                                uint32_t(unquant_weight_trit(1, 2)) << 16 | uint32_t(unquant_weight_trit(1, 3)) << 24;
        constexpr uint32_t hi = uint32_t(unquant_weight_trit(1, 4)) | uint32_t(unquant_weight_trit(1, 5)) << 8;
        return __builtin_amdgcn_perm(hi, lo, trits << 1 | bits);
    }
    // table entries 0..2: symbols 4t + b0, entries 4..6: symbols 4t + 2 + b0
    constexpr auto tab = [](int b) {
        return uint32_t(unquant_weight_trit(2, b)) | uint32_t(unquant_weight_trit(2, 4 + b)) << 8 |
               uint32_t(unquant_weight_trit(2, 8 + b)) << 16;
    };
    const uint32_t sel = trits | (bits & 0x02020202u) << 1;
    const uint32_t odd = (bits & 0x01010101u) * 0xFFu;
    constexpr uint32_t lo0 = tab(0), hi0 = tab(2), lo1 = tab(1), hi1 = tab(3);
    return (__builtin_amdgcn_perm(hi1, lo1, sel) & odd) | (__builtin_amdgcn_perm(hi0, lo0, sel) & ~odd);
}

// A block in one of the encoder's layouts: weights in 5-value trit groups of
// QUANT_6 (RGBA) or QUANT_12 (RGB), endpoints as bytes from bit 17.
//
// Every step works on four bytes in a register: a group's trits come from one
// table word and its low bits from shifted masks, four weights are unquantised by
// byte permutes, a 6x6 texel's infill is two 4-byte dot products with constant
// factors, and a texel's channel is one multiply-add whose byte 2 is the result
// (4 ((C0 (64 - w) + C1 w) + 32) < 2^24).  A lane writes each texel row of its
// block with 16- and 8-byte stores, so a wave's stores cover whole spans of the
// image's rows.  4096x4096 RGBA 6x6: 57.3 -> 16.4 us a launch among others (4.6
// TB/s of blocks read and texels written, where a 1 GiB copy reaches 5.2), most
// of it memory traffic; the general path spent its time on per-weight loops over
// LDS bytes and on 4-byte stores.
template <int DIM, bool RGBA>
__device__ __forceinline__ void decode_fixed(const DecodeArgs& a, int x0, int y0, uint4 blk, const uint32_t* trit_lut) {
    constexpr int b = RGBA ? 1 : 2, kGroupBits = 5 * b + 8;
    constexpr uint32_t low = (1u << b) - 1u;
    const uint64_t stream =
        uint64_t(__builtin_bitreverse32(blk.w)) | uint64_t(__builtin_bitreverse32(blk.z)) << 32;
    uint32_t quad[3], rest_t = 0, rest_b = 0;  // four weights of each group; each group's fifth, and weight 15
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        const uint32_t G = uint32_t(stream >> (g * kGroupBits)) & ((1u << (g < 3 ? kGroupBits : b + 2)) - 1u);
        const uint32_t T = (G >> b & 0x3u) | (G >> (2 * b) & 0xCu) | (G >> (3 * b) & 0x10u) | (G >> (4 * b) & 0x60u) |
                           (G >> (5 * b) & 0x80u);
        const uint32_t t = trit_lut[T];
        if (g == 3) {
            rest_t |= (t & 3u) << 24;
            rest_b |= (G & low) << 24;
            break;
        }
        const uint32_t bits = (G & low) | (G << (6 - b) & low << 8) | (G << (12 - 2 * b) & low << 16) |
                              (G << (19 - 3 * b) & low << 24);
        quad[g] = unquant_weights4<RGBA>(t & 0x03030303u, bits);
        rest_t |= (t >> 28) << (8 * g);
        rest_b |= (G >> (4 * b + 7) & low) << (8 * g);
    }
    const uint32_t rest = unquant_weights4<RGBA>(rest_t, rest_b);
    // weights 4r .. 4r + 3 of grid row r
    const uint32_t row[4] = {quad[0], quad[1] << 8 | (rest & 0xFFu),
                             quad[1] >> 24 | (rest & 0xFF00u) | quad[2] << 16, quad[2] >> 16 | (rest & 0xFFFF0000u)};
    // endpoint bytes r0 r1 g0 g1 | b0 b1 a0 a1
    const uint32_t ex = blk.x >> 17 | blk.y << 15, ey = blk.y >> 17 | blk.z << 15;
    int base[4], d[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        const uint32_t pair = (c < 2 ? ex : ey) >> (16 * (c & 1));
        const int e0 = (c < 3 || RGBA) ? int(pair & 0xFFu) : 255, e1 = (c < 3 || RGBA) ? int(pair >> 8 & 0xFFu) : 255;
        base[c] = e0 * (4 * 257 * 64) + 4 * 32;
        d[c] = (e1 - e0) * (4 * 257);
    }
    const bool whole = x0 + DIM <= a.width;
    uint32_t* out = a.rgba + (size_t)y0 * a.width + x0;
#pragma unroll
    for (int t = 0; t < DIM; ++t) {
        if (y0 + t >= a.height) break;
        uint32_t px[DIM];
#pragma unroll
        for (int s = 0; s < DIM; ++s) {
            using I = Infill<DIM>;
            int w;
            if (DIM == 4) {  // a texel per grid point
                w = int(row[t & 3] >> (8 * (s & 3)) & 0xFFu);
            } else {
                uint32_t acc = __builtin_amdgcn_udot4(row[I::j(t)], I::taps(s, t, 0), 8u, false);
                if (I::taps(s, t, 1)) acc = __builtin_amdgcn_udot4(row[I::j(t) < 3 ? I::j(t) + 1 : 3], I::taps(s, t, 1), acc, false);
                w = int(acc >> 4);
            }
            uint32_t v[4];
#pragma unroll
            for (int c = 0; c < 4; ++c) v[c] = uint32_t(__mul24(d[c], w) + base[c]);
            px[s] = __builtin_amdgcn_perm(v[1], v[0], 0x0C0C0602u) | __builtin_amdgcn_perm(v[3], v[2], 0x06020C0Cu);
        }
        if (whole) {
            typedef uint32_t Four __attribute__((ext_vector_type(4), aligned(4)));
            typedef uint32_t Two __attribute__((ext_vector_type(2), aligned(4)));
            *reinterpret_cast<Four*>(out) = Four{px[0], px[1], px[2], px[3]};
            if (DIM == 6) *reinterpret_cast<Two*>(out + 4) = Two{px[DIM - 2], px[DIM - 1]};
        } else {
#pragma unroll
            for (int s = 0; s < DIM; ++s)
                if (x0 + s < a.width) out[s] = px[s];
        }
        out += a.width;
    }
}

// DIM: the image's square block size, or 0 for any size (the general path only).
template <int DIM>
__global__ void __launch_bounds__(kDecThreads) decode_kernel(DecodeArgs a) {
    __shared__ uint32_t trit_lut[256];
    __shared__ uint16_t quint_lut[128];
    __shared__ uint8_t wbuf[kMaxWeights * kDecThreads];
    __shared__ uint8_t ebuf[8 * kDecThreads];
    const int id = blockIdx.x * kDecThreads + threadIdx.x;
    uint4 blk = make_uint4(0, 0, 0, 0);
    if (id < a.nblocks) blk = a.blocks[id];  // in flight while the tables are staged
    for (int i = threadIdx.x; i < 256; i += blockDim.x) trit_lut[i] = a.tables->trits[i];
    for (int i = threadIdx.x; i < 128; i += blockDim.x) quint_lut[i] = a.tables->quints[i];
    __syncthreads();
    if (id >= a.nblocks) return;
    const int by = block_row(id, a.xb_magic, a.xb_shift), bx = id - by * a.xblocks;
    const int x0 = bx * a.bw, y0 = by * a.bh;
    if (DIM) {
        // mode, partition count and endpoint mode of the encoder's layouts; with
        // the second endpoint's colour sum the larger there is no blue contraction
        const uint32_t head = blk.x & 0x1FFFFu;
        const uint32_t ex = blk.x >> 17 | blk.y << 15, ey = blk.y >> 17 | blk.z << 15;
        const bool plain = __builtin_amdgcn_udot4(ex, 0x01000100u, __builtin_amdgcn_udot4(ey, 0x0100u, 0u, false), false) >=
                           __builtin_amdgcn_udot4(ex, 0x00010001u, __builtin_amdgcn_udot4(ey, 0x0001u, 0u, false), false);
        constexpr int kDim = DIM ? DIM : 4;
        const bool rgba = head == (kModeRGBA | CEM_LDR_RGBA_DIRECT << 13);
        const bool rgb = head == (kModeRGB | CEM_LDR_RGB_DIRECT << 13);
        // whole waves only: one that has other blocks too would run both paths (up to
        // 13% of a launch over such images)
        if (__all(plain && (rgba || rgb))) {
            if (rgba) decode_fixed<kDim, true>(a, x0, y0, blk, trit_lut);
            else decode_fixed<kDim, false>(a, x0, y0, blk, trit_lut);
            return;
        }
    }
    const uint64_t lo = uint64_t(blk.x) | uint64_t(blk.y) << 32, hi = uint64_t(blk.z) | uint64_t(blk.w) << 32;
    const uint32_t kError = 0xFFFF00FFu;  // magenta, alpha 255
    const uint32_t mode = uint32_t(lo) & 0x7FFu;
    if ((mode & 0x1FFu) == 0x1FCu) {
        if (mode & 0x200u) { fill_block(a, x0, y0, kError); return; }
        const uint32_t c = uint32_t((hi >> 8) & 0xFF) | uint32_t((hi >> 24) & 0xFF) << 8 |
                           uint32_t((hi >> 40) & 0xFF) << 16 | uint32_t((hi >> 56) & 0xFF) << 24;
        fill_block(a, x0, y0, c);
        return;
    }
    const Mode m = decode_mode(mode);
    const int parts = int((lo >> 11) & 3) + 1;
    const int nw = m.gw * m.gh * (m.dual ? 2 : 1);
    if (!m.ok || parts != 1 || m.gw > a.bw || m.gh > a.bh || nw > kMaxWeights) { fill_block(a, x0, y0, kError); return; }
    const int wbits = ise_bit_count(m.quant, nw);
    const int cem = int((lo >> 13) & 0xF);
    if (wbits < 24 || wbits > 96 || (cem != 0 && cem != 4 && cem != 8 && cem != 12)) {
        fill_block(a, x0, y0, kError);
        return;
    }
    const int nvals = 2 * ((cem >> 2) + 1);
    const int avail = 128 - 17 - wbits - (m.dual ? 2 : 0);
    int eq = -1;
    for (int q = QUANT_256; q >= QUANT_6; --q)
        if (ise_bit_count(q, nvals) <= avail) { eq = q; break; }
    if (eq < 0) { fill_block(a, x0, y0, kError); return; }

    uint8_t* ecol = ebuf + threadIdx.x;
    ise_decode(lo, hi, 17, nvals, eq, trit_lut, quint_lut, ecol);
    int v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = i < nvals ? int(unquant_color(eq, ecol[i * kDecThreads])) : 0;
    int e0[4], e1[4];
    if (cem == 0) {
        e0[0] = e0[1] = e0[2] = v[0]; e1[0] = e1[1] = e1[2] = v[1]; e0[3] = e1[3] = 255;
    } else if (cem == 4) {
        e0[0] = e0[1] = e0[2] = v[0]; e1[0] = e1[1] = e1[2] = v[1]; e0[3] = v[2]; e1[3] = v[3];
    } else {
        const int a0 = cem == 12 ? v[6] : 255, a1 = cem == 12 ? v[7] : 255;
        if (v[1] + v[3] + v[5] >= v[0] + v[2] + v[4]) {
            e0[0] = v[0]; e0[1] = v[2]; e0[2] = v[4]; e0[3] = a0;
            e1[0] = v[1]; e1[1] = v[3]; e1[2] = v[5]; e1[3] = a1;
        } else {  // blue contraction, endpoints swapped
            e0[0] = (v[1] + v[5]) >> 1; e0[1] = (v[3] + v[5]) >> 1; e0[2] = v[5]; e0[3] = a1;
            e1[0] = (v[0] + v[4]) >> 1; e1[1] = (v[2] + v[4]) >> 1; e1[2] = v[4]; e1[3] = a0;
        }
    }

    // weights: the stream runs downwards from bit 127
    uint8_t* wcol = wbuf + threadIdx.x;
    const uint64_t rlo = __builtin_bitreverse64(hi), rhi = __builtin_bitreverse64(lo);
    ise_decode(rlo, rhi, 0, nw, m.quant, trit_lut, quint_lut, wcol);
    for (int i = 0; i < nw; ++i) wcol[i * kDecThreads] = uint8_t(unquant_weight(m.quant, wcol[i * kDecThreads]));
    const int ccs = m.dual ? int(get_bits(lo, hi, 128 - wbits - 2, 2)) : -1;
    const int planes = m.dual ? 2 : 1;

    // bilinear infill of the weight grid (specification), then interpolation
    const int Ds = (1024 + a.bw / 2) / (a.bw - 1), Dt = (1024 + a.bh / 2) / (a.bh - 1);
    for (int t = 0; t < a.bh; ++t) {
        const int y = y0 + t;
        if (y >= a.height) break;
        const int gt = (Dt * t * (m.gh - 1) + 32) >> 6;
        const int jt = gt >> 4, ft = gt & 15;
        for (int s = 0; s < a.bw; ++s) {
            const int x = x0 + s;
            if (x >= a.width) break;
            const int gs = (Ds * s * (m.gw - 1) + 32) >> 6;
            const int js = gs >> 4, fs = gs & 15;
            const int v0 = js + jt * m.gw;
            const int w11 = (fs * ft + 8) >> 4, w10 = ft - w11, w01 = fs - w11, w00 = 16 - fs - ft + w11;
            int wt[2];
            for (int p = 0; p < planes; ++p) {
                auto W = [&](int idx) -> int {
                    const int i = idx * planes + p;
                    return i < nw ? int(wcol[i * kDecThreads]) : 0;
                };
                int acc = W(v0) * w00;
                if (w01) acc += W(v0 + 1) * w01;
                if (w10) acc += W(v0 + m.gw) * w10;
                if (w11) acc += W(v0 + m.gw + 1) * w11;
                wt[p] = (acc + 8) >> 4;
            }
            uint32_t out = 0;
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const int w = (c == ccs) ? wt[1] : wt[0];
                const int C = (e0[c] * 257 * (64 - w) + e1[c] * 257 * w + 32) >> 6;
                out |= uint32_t(C >> 8) << (8 * c);
            }
            a.rgba[(size_t)y * a.width + x] = out;
        }
    }
}

}  // namespace

hipError_t launch_decode(const TritQuintDecodeTable* d_tables, const void* blocks, void* rgba, int width, int height,
                         int bw, int bh, hipStream_t stream) {
    DecodeArgs a;
    a.blocks = static_cast<const uint4*>(blocks);
    a.rgba = static_cast<uint32_t*>(rgba);
    a.width = width;
    a.height = height;
    a.bw = bw;
    a.bh = bh;
    a.xblocks = (width + bw - 1) / bw;
    a.nblocks = a.xblocks * ((height + bh - 1) / bh);
    set_block_row_magic(a.xblocks, &a.xb_magic, &a.xb_shift);
    a.tables = d_tables;
    (void)hipGetLastError();  // report this launch's errors only, not an earlier call's
    const dim3 grid(unsigned((a.nblocks + kDecThreads - 1) / kDecThreads)), threads(kDecThreads);
    if (bw == 4 && bh == 4) hipLaunchKernelGGL(decode_kernel<4>, grid, threads, 0, stream, a);
    else if (bw == 6 && bh == 6) hipLaunchKernelGGL(decode_kernel<6>, grid, threads, 0, stream, a);
    else hipLaunchKernelGGL(decode_kernel<0>, grid, threads, 0, stream, a);
    return hipGetLastError();
}

}  // namespace astc
