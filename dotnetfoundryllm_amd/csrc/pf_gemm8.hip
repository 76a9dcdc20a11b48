// pf_gemm8.hip — the prefill GEMMs of tile-interleaved Q4_K / Q5_K / Q6_K / Q8_0 weights and of GGUF rows
// of whole 256-element blocks (those types, Q4_0 and F16): workgroups of eight waves (2 along the tokens x 4
// along the weight rows), each 32 TI tokens x 64 weight rows, so tiles of 64 or 128 tokens x 256 rows.
//
// Numerics: fp16 matrix cores on X's two planes (22 bits) and on exact integers of the weights:
//  - Q4_K, Q5_K: w = d (sc q) - dmin m; sc q is an integer below 2048, exact in fp16, so a product is two
//    MFMAs (x lo, x hi). A 256-element block's sum is scaled by its d in f32. Its min term is one more
//    MFMA whose K slice packs, per row, (v_g hi, v_g lo, v_g hi) for v_g = -dmin m_g against, per token,
//    the group sums (X_g hi, X_g hi, X_g lo); the group sums are stored times 2^-6 (to stay in fp16's
//    range) and v_g times 2^-wexp, which brings the matrix's largest into [2^14, 2^15) (launch_pf_wmax), so
//    the sums are held times 2^-(wexp + 6), d and the epilogue taking the factor. (v_g times a fixed 2^6
//    had left its two halves' range from dmin m = 2047 on.)
//  - Q6_K: w = d (sc q), |sc q| <= 4096: hi = fp16(sc q) and lo = sc q - hi (0 or +-1) hold it exactly;
//    x lo hi + x hi lo + x hi hi (the dropped x lo lo is below 2^-22 of a product), d per block.
//  - Q8_0, Q4_0: the code (Q4_0: minus 8), exact; two MFMAs, each 32-element block's sum scaled by its d.
//  - F16: the weight itself times a power of two that costs no bit; two MFMAs.
//
// The MFMA rounds its sums down, the same way for every output (Q8_0, 2048 columns: -4e-8 of the result's root
// mean square): in the forms of codes every other block (step, in the step-scaled forms) enters with its codes
// and its d negated, so that half of the sums err upwards (below 5e-9 since). Not in F16, whose total stays in
// the MFMA: -1.6e-8 at 2048 columns, -4e-8 at 8192, as its three products had; a total beside the block's sum
// ran 3.5% longer, one negated in place 2% (4096 wide, 2000 tokens). Nor do the min terms alternate, which
// enter the total by one MFMA a block: 6e-10 of Q4_K at 8192 columns.
//
// What bounds it: the matrix cores beside the card's power. A tile of 64 tokens x 128 rows on four waves
// (32 x 64 each, three workgroups per CU, one LDS stage, two barriers a step) issued 5.2 vector-ALU
// instructions per 16x16x32 MFMA, most of them the weights' decode, and moved 192 bytes of LDS per
// matrix cycle. With 128 x 256 tiles a decoded weight meets twice the tokens (2.4 vector-ALU
// instructions per MFMA), an operand read feeds four MFMAs instead of 2.7, and two LDS stages need one
// barrier a step; the global loads of X and weights run 3 (TI 2) or 9 (TI 1) steps ahead in registers.
// The residual and the token factors are read together: one value at a time, each store's loads had
// waited for the one before, 20 us per tile. Per launch, before and now: Q4_K 28672 x 4096 over 511
// tokens 336 -> 288 us (835 TFLOP/s of fp16 products), Q6_K 4096 x 14336 254 -> 177; Q5_K 37888 x 3584
// over 2047 tokens 1496 -> 1280; Q8_0 28672 x 3584 over 4096 tokens 2108 -> 1760 (955 TFLOP/s; a plain
// fp16 8192^3 product runs at 1157 on this card, its clock held at 1.6-1.8 GHz by power). Tiles of
// 256 x 128 were slower (X's planes, not the weights, are the larger operand): 376 us for the first.
// GGUF rows, before (dequantized, split hi / lo, three products, element loads) and now, two layers:
// F16 2048 wide over 300 tokens 1485 -> 399 us, Q5_K 2304 wide over 700 1852 -> 1076; Q4_0 4096 wide over
// 300 (one layer) 892 -> 610.
#include "pf_gemm8.hpp"

namespace fllm {

typedef float g8_f4 __attribute__((ext_vector_type(4)));
typedef _Float16 g8_h8 __attribute__((ext_vector_type(8)));
typedef _Float16 g8_h2 __attribute__((ext_vector_type(2)));
typedef uint32_t g8_u4 __attribute__((ext_vector_type(4)));
typedef uint32_t g8_u2 __attribute__((ext_vector_type(2)));
typedef __fp16 g8_p2 __attribute__((ext_vector_type(2)));

typedef __amdgpu_buffer_rsrc_t g8_rsrc;
// addresses are kept in range by the callers (clamped rows and blocks)
__device__ __forceinline__ g8_rsrc g8_buf(const void* p) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, -1, 0x00027000);
}
__device__ __forceinline__ g8_u4 g8_ld16(g8_rsrc r, uint32_t v, uint32_t s) { return __builtin_amdgcn_raw_buffer_load_b128(r, (int)v, (int)s, 0); }
__device__ __forceinline__ g8_u2 g8_ld8(g8_rsrc r, uint32_t v, uint32_t s) { return __builtin_amdgcn_raw_buffer_load_b64(r, (int)v, (int)s, 0); }
__device__ __forceinline__ uint32_t g8_ld4(g8_rsrc r, uint32_t v, uint32_t s) { return __builtin_amdgcn_raw_buffer_load_b32(r, (int)v, (int)s, 0); }
__device__ __forceinline__ uint32_t g8_ld2(g8_rsrc r, uint32_t v, uint32_t s) { return (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(r, (int)v, (int)s, 0); }
__device__ __forceinline__ int g8_ld1(g8_rsrc r, uint32_t v, uint32_t s) { return (int8_t)__builtin_amdgcn_raw_buffer_load_b8(r, (int)v, (int)s, 0); }

// K elements of a step; halves of a min-term row (three used 16-byte chunks)
constexpr int G8_BK = 32, G8_LDV = 24;

// ---- weights: what one thread stages per step, 8 elements (chunk c of 4) of group g of a row -----
// Blk: a row's values of a whole 256-element block; Raw: of one step. REG: bytes of a block's region of
// RG rows (tile-interleaved: 16; GGUF rows, form PF_FORM_ROWS + type: 1); s + o: the region's offset from
// the tile's first weight (buffer w, address p), n: the row in it. SC, what scales a sum: a block's d, a
// step's d, or nothing.
enum { G8_SC_BLOCK, G8_SC_STEP, G8_SC_NONE };
template <int TYPE> struct G8W;

__device__ __forceinline__ float g8_half(uint32_t h) { return (float)__builtin_bit_cast(_Float16, (uint16_t)h); }
// (1024 + code) sc - 1024 sc in one packed fma: exact, |sc code| < 2048
__device__ __forceinline__ uint32_t g8_scaled(uint32_t code, g8_h2 sc2, g8_h2 nb) {
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(__builtin_bit_cast(g8_h2, code | 0x64006400u), sc2, nb));
}
// codes of a step-scaled group: p + off, negated in the odd groups
__device__ __forceinline__ uint32_t g8_centred(uint32_t p, g8_h2 off, int g) {
    const g8_h2 v = __builtin_bit_cast(g8_h2, p);
    return __builtin_bit_cast(uint32_t, (g & 1) ? -off - v : v + off);
}
// the two nibbles of the low byte in bits 0-3 and 16-19
__device__ __forceinline__ uint32_t g8_nib(uint32_t x) { return ((x << 12) & 0x000F0000u) | (x & 0xFu); }

// the 6-bit scale of group g of a K-quant header (DecodeKScaleMin, Dequantizer.cs:506-521)
__device__ __forceinline__ uint32_t g8_scale(const g8_u4& h, int g) {
    if (g < 4) return (h.y >> (8 * g)) & 63u;
    return ((h.w >> (8 * (g - 4))) & 15u) | (((h.y >> (8 * (g - 4) + 6)) & 3u) << 4);
}
// the 6-bit mins of groups 2 c and 2 c + 1, in bytes 0 and 1
__device__ __forceinline__ uint32_t g8_mins(const g8_u4& h, int c) {
    const uint32_t z = h.z >> (16 * (c & 1)), w = h.w >> (16 * (c & 1));
    return (c < 2 ? z : (((w >> 4) & 0x0F0Fu) | ((z >> 2) & 0x3030u))) & 0x3F3Fu;
}

template <> struct G8W<FLLM_TYPE_Q4_K> {
    static constexpr int REG = 16 * 144, PLANES = 1, RG = 16, SC = G8_SC_BLOCK;
    struct Blk { g8_u4 hdr; };
    struct Raw { g8_u2 q; };
    __device__ static void load_blk(Blk& b, g8_rsrc w, const uint8_t*, uint32_t s, uint32_t o, uint32_t n) { b.hdr = g8_ld16(w, o + 16 * n, s + 2048); }
    __device__ static void load(Raw& r, g8_rsrc w, const uint8_t*, uint32_t s, uint32_t o, uint32_t n, uint32_t c, int g) {
        r.q = g8_ld8(w, o + 16 * n + 8 * (c >> 1), s + 256 * g);
    }
    // a half's dwords hold its bytes 0, 2, 4, 6 and 1, 3, 5, 7 (q4t_src_byte)
    __device__ static g8_u4 decode(const Raw& r, const Blk& b, int c, int g, float sign) {
        const _Float16 s = (_Float16)(sign * (float)g8_scale(b.hdr, g));
        const g8_h2 sc2 = {s, s}, nb = sc2 * g8_h2{(_Float16)-1024.0f, (_Float16)-1024.0f};
        const uint32_t x = r.q.x >> (16 * (c & 1)), y = r.q.y >> (16 * (c & 1));
        return g8_u4{g8_scaled(g8_nib(x), sc2, nb), g8_scaled(g8_nib(y), sc2, nb), g8_scaled(g8_nib(x >> 8), sc2, nb),
                          g8_scaled(g8_nib(y >> 8), sc2, nb)};
    }
};

template <> struct G8W<FLLM_TYPE_Q5_K> {
    static constexpr int REG = 16 * 176, PLANES = 1, RG = 16, SC = G8_SC_BLOCK;
    struct Blk { g8_u4 hdr; };
    struct Raw { uint32_t q, h; };
    __device__ static void load_blk(Blk& b, g8_rsrc w, const uint8_t*, uint32_t s, uint32_t o, uint32_t n) { b.hdr = g8_ld16(w, o + 16 * n, s + 2560); }
    __device__ static void load(Raw& r, g8_rsrc w, const uint8_t*, uint32_t s, uint32_t o, uint32_t n, uint32_t c, int g) {
        r.q = g8_ld4(w, o + 16 * n + 4 * c, s + 256 * g);
        r.h = g8_ld4(w, o + 8 * n, s + 2048 + 128 * (g & 3) + (g < 4 ? 0 : 4));
    }
    // element 16 hf + 4 by + j has its high bit at bit 8 by + 4 hf + j of h; pair (2 b, 2 b + 1) of
    // chunk c = 2 hf + (c & 1): bits p, p + 1 of the half (c & 1) of h >> 4 hf, p = 8 (b >> 1) + 2 (b & 1)
    __device__ static g8_u4 decode(const Raw& r, const Blk& b, int c, int g, float sign) {
        const _Float16 s = (_Float16)(sign * (float)g8_scale(b.hdr, g));
        const g8_h2 sc2 = {s, s}, nb = sc2 * g8_h2{(_Float16)-1024.0f, (_Float16)-1024.0f};
        const uint32_t h16 = (r.h >> (16 * (c & 1) + 4 * (c >> 1))) & 0x0F0Fu, z = h16 | (h16 << 15);
        return g8_u4{g8_scaled(g8_nib(r.q) | ((z << 4) & 0x00100010u), sc2, nb),
                          g8_scaled(g8_nib(r.q >> 8) | ((z << 2) & 0x00100010u), sc2, nb),
                          g8_scaled(g8_nib(r.q >> 16) | ((z >> 4) & 0x00100010u), sc2, nb),
                          g8_scaled(g8_nib(r.q >> 24) | ((z >> 6) & 0x00100010u), sc2, nb)};
    }
};

template <> struct G8W<FLLM_TYPE_Q8_0> {
    static constexpr int REG = 16 * 272, PLANES = 1, RG = 16, SC = G8_SC_STEP;
    struct Blk {};
    struct Raw { g8_u4 h; uint32_t d; };
    __device__ static void load_blk(Blk&, g8_rsrc, const uint8_t*, uint32_t, uint32_t, uint32_t) {}
    __device__ static void load(Raw& r, g8_rsrc w, const uint8_t*, uint32_t s, uint32_t o, uint32_t n, uint32_t c, int g) {
        r.h = g8_ld16(w, o + 1024 * (c >> 1) + 16 * n, s + (g < 4 ? 0 : 2048) + 256 * (g & 3));
        r.d = g8_ld2(w, o + 16 * n, s + 4096 + 4 * (g & 3) + (g < 4 ? 0 : 2));
    }
    // the code's byte as fp16 1024 + 128 + q (0x64 80 ^ byte), minus 1152
    __device__ static g8_u4 decode(const Raw& r, const Blk&, int c, int g, float) {
        const uint32_t s0 = (c & 1) ? 0x0C060C02u : 0x0C040C00u, s1 = (c & 1) ? 0x0C070C03u : 0x0C050C01u;
        const g8_h2 off = {(_Float16)-1152.0f, (_Float16)-1152.0f};
        auto pr = [&](uint32_t hi, uint32_t lo, uint32_t sel) {
            return g8_centred(__builtin_amdgcn_perm(hi, lo, sel) ^ 0x64806480u, off, g);
        };
        return g8_u4{pr(r.h.y, r.h.x, s0), pr(r.h.w, r.h.z, s0), pr(r.h.y, r.h.x, s1), pr(r.h.w, r.h.z, s1)};
    }
};

template <> struct G8W<FLLM_TYPE_Q6_K> {
    static constexpr int REG = 16 * 210, PLANES = 2, RG = 16, SC = G8_SC_BLOCK;
    struct Blk { uint32_t d; };
    struct Raw { uint32_t ql, qh; int sc; };
    __device__ static void load_blk(Blk& b, g8_rsrc w, const uint8_t*, uint32_t s, uint32_t o, uint32_t n) { b.d = g8_ld2(w, o + 2 * n, s + 3328); }
    __device__ static void load(Raw& r, g8_rsrc w, const uint8_t*, uint32_t s, uint32_t o, uint32_t n, uint32_t c, int g) {
        r.ql = g8_ld4(w, o + 16 * n + 4 * c, s + 256 * g);
        r.qh = g8_ld2(w, o + 16 * n + 2 * c, s + 2048 + 256 * (g & 3) + (g < 4 ? 0 : 8));
        r.sc = g8_ld1(w, o + 4 * n + (c >> 1), s + 3072 + 64 * (g & 3) + (g < 4 ? 0 : 2));
    }
    // hi and lo halves of the exact integer sc q
    __device__ static void decode2(const Raw& r, float sign, g8_u4& hi, g8_u4& lo) {
        const _Float16 s = (_Float16)(sign * (float)r.sc);
        const g8_h2 sc2 = {s, s}, off = {(_Float16)-1056.0f, (_Float16)-1056.0f};
        const uint32_t y = r.qh | (r.qh << 14);
        uint32_t hv[4], lv[4];
#pragma unroll
        for (int b = 0; b < 4; b++) {
            const uint32_t t = (b == 0 ? (y << 4) : (y >> (4 * b - 4))) & 0x00300030u;
            const g8_h2 q = __builtin_bit_cast(g8_h2, g8_nib(r.ql >> (8 * b)) | t | 0x64006400u) + off;
            const g8_h2 vh = q * sc2;
            hv[b] = __builtin_bit_cast(uint32_t, vh);
            lv[b] = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(q, sc2, -vh));
        }
        hi = g8_u4{hv[0], hv[1], hv[2], hv[3]};
        lo = g8_u4{lv[0], lv[1], lv[2], lv[3]};
    }
};

// ---- GGUF rows of whole 256-element blocks ----------------------------------------------------------
// loads of the formats whose blocks start at even addresses
struct __attribute__((packed, aligned(2))) G8P8 { uint32_t x, y; };
struct __attribute__((packed, aligned(2))) G8P4 { uint32_t x; };

template <> struct G8W<PF_FORM_ROWS + FLLM_TYPE_Q4_K> : G8W<FLLM_TYPE_Q4_K> {
    static constexpr int REG = 144, RG = 1;
    struct Raw { uint32_t q; };
    __device__ static void load_blk(Blk& b, g8_rsrc w, const uint8_t*, uint32_t s, uint32_t o, uint32_t) { b.hdr = g8_ld16(w, o, s); }
    __device__ static void load(Raw& r, g8_rsrc w, const uint8_t*, uint32_t s, uint32_t o, uint32_t, uint32_t c, int g) {
        r.q = g8_ld4(w, o + 4 * c, s + 16 + 16 * g);
    }
    __device__ static g8_u4 decode(const Raw& r, const Blk& b, int, int g, float sign) {
        const _Float16 s = (_Float16)(sign * (float)g8_scale(b.hdr, g));
        const g8_h2 sc2 = {s, s}, nb = sc2 * g8_h2{(_Float16)-1024.0f, (_Float16)-1024.0f};
        return g8_u4{g8_scaled(g8_nib(r.q), sc2, nb), g8_scaled(g8_nib(r.q >> 8), sc2, nb), g8_scaled(g8_nib(r.q >> 16), sc2, nb),
                     g8_scaled(g8_nib(r.q >> 24), sc2, nb)};
    }
};

template <> struct G8W<PF_FORM_ROWS + FLLM_TYPE_Q5_K> : G8W<FLLM_TYPE_Q5_K> {
    static constexpr int REG = 176, RG = 1;
    __device__ static void load_blk(Blk& b, g8_rsrc w, const uint8_t*, uint32_t s, uint32_t o, uint32_t) { b.hdr = g8_ld16(w, o, s); }
    __device__ static void load(Raw& r, g8_rsrc w, const uint8_t*, uint32_t s, uint32_t o, uint32_t, uint32_t c, int g) {
        r.q = g8_ld4(w, o + 4 * c, s + 48 + 16 * g);
        r.h = (uint8_t)g8_ld1(w, o + c, s + 16 + 4 * g);
    }
    // element j of the chunk has its high bit at bit j of h
    __device__ static g8_u4 decode(const Raw& r, const Blk& b, int, int g, float sign) {
        const _Float16 s = (_Float16)(sign * (float)g8_scale(b.hdr, g));
        const g8_h2 sc2 = {s, s}, nb = sc2 * g8_h2{(_Float16)-1024.0f, (_Float16)-1024.0f};
        const uint32_t z = r.h | (r.h << 15);
        return g8_u4{g8_scaled(g8_nib(r.q) | ((z << 4) & 0x00100010u), sc2, nb),
                     g8_scaled(g8_nib(r.q >> 8) | ((z << 2) & 0x00100010u), sc2, nb),
                     g8_scaled(g8_nib(r.q >> 16) | (z & 0x00100010u), sc2, nb),
                     g8_scaled(g8_nib(r.q >> 24) | ((z >> 2) & 0x00100010u), sc2, nb)};
    }
};

template <> struct G8W<PF_FORM_ROWS + FLLM_TYPE_Q6_K> : G8W<FLLM_TYPE_Q6_K> {
    static constexpr int REG = 210, RG = 1;
    __device__ static void load_blk(Blk& b, g8_rsrc, const uint8_t* __restrict__ p, uint32_t s, uint32_t o, uint32_t) {
        b.d = *(const uint16_t*)(p + s + 208 + o);
    }
    __device__ static void load(Raw& r, g8_rsrc, const uint8_t* __restrict__ p, uint32_t s, uint32_t o, uint32_t, uint32_t c, int g) {
        r.ql = ((const G8P4*)(p + s + 16 * g + (o + 4 * c)))->x;
        r.qh = *(const uint16_t*)(p + s + 128 + 8 * g + (o + 2 * c));
        r.sc = *(const int8_t*)(p + s + 192 + 2 * g + (o + (c >> 1)));
    }
};

template <> struct G8W<PF_FORM_ROWS + FLLM_TYPE_Q8_0> {
    static constexpr int REG = 272, PLANES = 1, RG = 1, SC = G8_SC_STEP;
    struct Blk {};
    struct Raw { uint32_t x, y, d; };
    __device__ static void load_blk(Blk&, g8_rsrc, const uint8_t*, uint32_t, uint32_t, uint32_t) {}
    __device__ static void load(Raw& r, g8_rsrc, const uint8_t* __restrict__ p, uint32_t s, uint32_t o, uint32_t, uint32_t c, int g) {
        const G8P8 v = *(const G8P8*)(p + s + 34 * g + 2 + (o + 8 * c));
        r.x = v.x;
        r.y = v.y;
        r.d = *(const uint16_t*)(p + s + 34 * g + o);
    }
    __device__ static g8_u4 decode(const Raw& r, const Blk&, int, int g, float) {
        const g8_h2 off = {(_Float16)-1152.0f, (_Float16)-1152.0f};
        auto pr = [&](uint32_t v, uint32_t sel) {
            return g8_centred(__builtin_amdgcn_perm(0u, v, sel) ^ 0x64806480u, off, g);
        };
        return g8_u4{pr(r.x, 0x0C010C00u), pr(r.x, 0x0C030C02u), pr(r.y, 0x0C010C00u), pr(r.y, 0x0C030C02u)};
    }
};

// code - 8 exactly (Dequantizer.cs:155-185); chunks 0, 1 are the low nibbles of bytes 0-7, 8-15, 2, 3 the high ones
template <> struct G8W<PF_FORM_ROWS + FLLM_TYPE_Q4_0> {
    static constexpr int REG = 144, PLANES = 1, RG = 1, SC = G8_SC_STEP;
    struct Blk {};
    struct Raw { uint32_t x, y, d; };
    __device__ static void load_blk(Blk&, g8_rsrc, const uint8_t*, uint32_t, uint32_t, uint32_t) {}
    __device__ static void load(Raw& r, g8_rsrc, const uint8_t* __restrict__ p, uint32_t s, uint32_t o, uint32_t, uint32_t c, int g) {
        const G8P8 v = *(const G8P8*)(p + s + 18 * g + 2 + (o + 8 * (c & 1)));
        r.x = v.x;
        r.y = v.y;
        r.d = *(const uint16_t*)(p + s + 18 * g + o);
    }
    __device__ static g8_u4 decode(const Raw& r, const Blk&, int c, int g, float) {
        const uint32_t x = (r.x >> (4 * (c >> 1))) & 0x0F0F0F0Fu, y = (r.y >> (4 * (c >> 1))) & 0x0F0F0F0Fu;
        const g8_h2 off = {(_Float16)-1032.0f, (_Float16)-1032.0f};
        auto pr = [&](uint32_t v, uint32_t sel) {
            return g8_centred(__builtin_amdgcn_perm(0u, v, sel) | 0x64006400u, off, g);
        };
        return g8_u4{pr(x, 0x0C010C00u), pr(x, 0x0C030C02u), pr(y, 0x0C010C00u), pr(y, 0x0C030C02u)};
    }
};

// the weights themselves, times a power of two that takes no bit (g8_f16_exp)
template <> struct G8W<PF_FORM_ROWS + FLLM_TYPE_F16> {
    static constexpr int REG = 512, PLANES = 1, RG = 1, SC = G8_SC_NONE;
    struct Blk {};
    struct Raw { g8_u4 v; };
    __device__ static void load_blk(Blk&, g8_rsrc, const uint8_t*, uint32_t, uint32_t, uint32_t) {}
    __device__ static void load(Raw& r, g8_rsrc w, const uint8_t*, uint32_t s, uint32_t o, uint32_t, uint32_t c, int g) {
        r.v = g8_ld16(w, o + 16 * c, s + 64 * g);
    }
    __device__ static g8_u4 decode(const Raw& r, g8_h2 s0, g8_h2 s1) {
        g8_u4 o;
#pragma unroll
        for (int i = 0; i < 4; i++) o[i] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(g8_h2, (uint32_t)r.v[i]) * s0 * s1);
        return o;
    }
};
// 2^e scales F16 weights up into fp16's normal range: e = -wexp brings the largest magnitude below 2^15,
// so no product overflows and every value, a subnormal one too, keeps its bits; never down (e >= 0)
__device__ __forceinline__ int g8_f16_exp(int wexp) { return wexp > 0 ? 0 : wexp < -30 ? 30 : -wexp; }

// 2^e for |e| <= 126, in scalar registers where e is (wexp is the segment's; a ldexpf holds a vector register
// through the loop)
__device__ __forceinline__ float g8_pow2(int e) { return __uint_as_float((uint32_t)(127 + e) << 23); }

// ---- tile ---------------------------------------------------------------------------------------
// LDS of a tile of BM tokens x BN rows: two stages of [X hi | X lo | W planes] rows of 32 halves
// (16-byte chunk c of row r at position c ^ ((r >> 2) & 2): a 16-row operand read is then free of
// bank conflicts), then the block's scales and min-term slices.
template <int TI, int TYPE>
struct G8T {
    static constexpr int BM = 64 * TI, BN = 256, P = G8W<TYPE>::PLANES;
    static constexpr bool MIN = TYPE % PF_FORM_ROWS == FLLM_TYPE_Q4_K || TYPE % PF_FORM_ROWS == FLLM_TYPE_Q5_K;
    static constexpr int STAGE = (2 * BM + P * BN) * G8_BK;  // halves
    static constexpr size_t lds = sizeof(_Float16) * (2 * (size_t)STAGE + (MIN ? (size_t)(BM + BN) * G8_LDV : 0)) +
                                  sizeof(float) * (2 * BN + BM);
};

template <int TI, int TYPE>
__device__ __forceinline__ void g8_tile(const PfGemm& a, const PfSeg& sg, int n0, int t0, _Float16* lds) {
    using W = G8W<TYPE>;
    using S = G8T<TI, TYPE>;
    constexpr int BM = S::BM, BN = S::BN, P = S::P, STAGE = S::STAGE;
    constexpr bool MIN = S::MIN, F16 = W::SC == G8_SC_NONE;
    constexpr int SC = W::SC;
    constexpr int XP = BM / 64, WC = BN / 128;
    _Float16* sav = lds + 2 * STAGE;                               // MIN: [BM][G8_LDV]
    _Float16* swv = sav + (MIN ? BM * G8_LDV : 0);                 // MIN: [BN][G8_LDV]
    float* sd = (float*)(swv + (MIN ? BN * G8_LDV : 0));           // d: [BN] of the block, Q8_0 [2][BN] of the step
    float* sxs = sd + 2 * BN;                                      // what undoes the scales: the tokens' xs times the weights'
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave >> 2, wn = wave & 3;

    // staging: thread tid takes 16-byte chunk tid & 3 of row tid >> 2 (+ 128 i); 32-bit offsets from the
    // tile's first token (of the hi or lo plane, uniform over a wave) and weight row
    const int ch = tid & 3, r0 = tid >> 2;
    const size_t plane = (size_t)a.T * a.ldh;
    g8_rsrc xb[XP];
    uint32_t xp[XP];
#pragma unroll
    for (int i = 0; i < XP; i++) {
        const int pl = (__builtin_amdgcn_readfirstlane(r0) + 128 * i) / BM, row = (r0 + 128 * i) % BM;
        const int t = t0 + row < a.T ? row : a.T - 1 - t0;  // rows past the prompt repeat its last one
        xb[i] = g8_buf(a.xh + pl * plane + (size_t)t0 * a.ldh);
        xp[i] = 2u * ((uint32_t)t * (uint32_t)a.ldh + 8u * ch);
    }
    const int NB = a.K >> 8;
    const uint8_t* wb0 = sg.w + (size_t)(n0 / W::RG) * NB * W::REG;
    const g8_rsrc wb = g8_buf(wb0);
    uint32_t wp[WC], wnn[WC];
#pragma unroll
    for (int i = 0; i < WC; i++) {
        const int row = r0 + 128 * i, n = n0 + row < sg.N ? row : sg.N - 1 - n0;
        wp[i] = (uint32_t)(n / W::RG) * (uint32_t)(NB * W::REG);
        wnn[i] = n % W::RG;
    }
    // row r0 + 128 i of a stage: the swizzle depends on r0 alone
    const int so = r0 * G8_BK + ((ch ^ ((r0 >> 2) & 2)) << 3);
    const float wsc = g8_pow2(-sg.wexp);  // |wexp| <= 120 (pf_wexp)
    const float msc = MIN ? g8_pow2(-sg.wexp - 6) : 1.0f;  // what the sums of the block-scaled forms are held times
    const int fe = F16 ? g8_f16_exp(sg.wexp) : 0;
    const _Float16 fh0 = (_Float16)ldexpf(1.0f, fe < 15 ? fe : 15), fh1 = (_Float16)ldexpf(1.0f, fe < 15 ? 0 : fe - 15);
    const g8_h2 fs0 = {fh0, fh0}, fs1 = {fh1, fh1};
    // min term: thread tid < 2 BM takes token tid >> 1's hi (even) or lo group sums
    const int vt = tid >> 1, vhl = tid & 1, G = a.K / 32;
    const g8_rsrc vb = g8_buf(a.xh + 2 * plane + (size_t)t0 * G);
    const uint32_t vp = 2u * (uint32_t)G * (uint32_t)(vhl * a.T + (t0 + vt < a.T ? vt : a.T - 1 - t0));

    // a step's global loads are issued PD + 1 steps ahead into rings of PD registers sets (a wave's loads
    // complete in issue order, so X and the weights share one distance)
    constexpr int PD = TI == 1 ? 8 : 2;
    g8_u4 xr[PD][XP], xv = g8_u4{0u, 0u, 0u, 0u};
    typename W::Raw raw[PD][WC];
    typename W::Blk blk_c[WC], blk_n[WC];

    const int b0 = (int)blockIdx.z * (a.kpart >> 8);
    const int b1 = b0 + (a.kpart >> 8) < NB ? b0 + (a.kpart >> 8) : NB;
    auto load_x = [&](g8_u4* x, int k) {
#pragma unroll
        for (int i = 0; i < XP; i++) x[i] = g8_ld16(xb[i], xp[i], 2u * (uint32_t)k);
    };
    auto store_x = [&](const g8_u4* x, int buf) {
#pragma unroll
        for (int i = 0; i < XP; i++) *(g8_u4*)(lds + buf * STAGE + so + 128 * G8_BK * i) = x[i];
    };
    auto load_w = [&](typename W::Raw* r, int kb, int g) {
#pragma unroll
        for (int i = 0; i < WC; i++) W::load(r[i], wb, wb0, (uint32_t)kb * W::REG, wp[i], wnn[i], ch, g);
    };
    auto load_b = [&](typename W::Blk* b, int kb) {
#pragma unroll
        for (int i = 0; i < WC; i++) W::load_blk(b[i], wb, wb0, (uint32_t)kb * W::REG, wp[i], wnn[i]);
    };
    auto store_w = [&](const typename W::Raw* r, const typename W::Blk* b, int buf, int g, float sign) {
#pragma unroll
        for (int i = 0; i < WC; i++) {
            _Float16* dst = lds + buf * STAGE + 2 * BM * G8_BK + so + 128 * G8_BK * i;
            if constexpr (F16) {
                *(g8_u4*)dst = W::decode(r[i], fs0, fs1);
            } else if constexpr (P == 2) {
                g8_u4 hi, lo;
                W::decode2(r[i], sign, hi, lo);
                *(g8_u4*)dst = hi;
                *(g8_u4*)(dst + BN * G8_BK) = lo;
            } else {
                *(g8_u4*)dst = W::decode(r[i], b[i], ch, g, sign);
            }
            if constexpr (SC == G8_SC_STEP) {
                if (ch == 0) sd[buf * BN + r0 + 128 * i] = g8_half(r[i].d) * ((g & 1) ? -wsc : wsc);
            }
        }
    };

    constexpr int MI = 2 * TI;  // 16 x 16 tiles of the wave: MI along the tokens, 4 along the rows
    g8_f4 acc[MI][4], blk[MI][4];
    const g8_f4 zero = {};
#pragma unroll
    for (int i = 0; i < MI; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) acc[i][j] = blk[i][j] = zero;

    const float wun = F16 ? g8_pow2(-fe) : SC == G8_SC_STEP ? g8_pow2(sg.wexp) : MIN ? g8_pow2(sg.wexp + 6) : 1.0f;
    if (tid < BM) sxs[tid] = a.xs[t0 + tid < a.T ? t0 + tid : a.T - 1] * wun;
    float sign = 1.0f;  // of the current block's codes and d: every other block enters negated
    load_b(blk_c, b0);
    if (MIN && vt < BM) xv = g8_ld16(vb, vp, 16u * b0);
    // in step order (the loop's waits count the loads behind a step's own)
#pragma unroll
    for (int st = 0; st < PD; st++) {
        __builtin_amdgcn_sched_barrier(0);
        load_x(xr[st], 256 * b0 + G8_BK * st);
        load_w(raw[st], b0, st);
    }
    __builtin_amdgcn_sched_barrier(0);
    store_x(xr[0], 0);
    store_w(raw[0], blk_c, 0, 0, sign);
    const int bp = PD < 8 || b0 + 1 == b1 ? b0 : b0 + 1;
    load_x(xr[0], 256 * bp + G8_BK * (PD & 7));
    load_w(raw[0], bp, PD & 7);
    __builtin_amdgcn_sched_barrier(0);
    __syncthreads();

    // operand addresses: lane l reads row l & 15, K chunk l >> 4 of the step
    const int l15 = lane & 15, lq = lane >> 4;
    const int oc = l15 * G8_BK + ((lq ^ ((l15 >> 2) & 2)) << 3);

    for (int kb = b0; kb < b1; kb++) {
        const int kn = kb + 1 < b1 ? kb + 1 : kb;
#pragma unroll
        for (int st = 0; st < 8; st++) {
            const int buf = st & 1;
            const _Float16* sx = lds + buf * STAGE;
            const _Float16* sw = sx + 2 * BM * G8_BK;
            g8_h8 ah[MI], al[MI], bh[4], bl[4];
#pragma unroll
            for (int i = 0; i < MI; i++) {
                const _Float16* p = sx + (32 * TI * wm + 16 * i) * G8_BK + oc;
                al[i] = *(const g8_h8*)(p + BM * G8_BK);
                ah[i] = *(const g8_h8*)p;
            }
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const _Float16* p = sw + (64 * wn + 16 * j) * G8_BK + oc;
                bh[j] = *(const g8_h8*)p;
            }
            float dj[4];
            if constexpr (SC == G8_SC_STEP) {
#pragma unroll
                for (int j = 0; j < 4; j++) dj[j] = sd[buf * BN + 64 * wn + 16 * j + l15];
            }
            __builtin_amdgcn_sched_barrier(0);
            // the next step's operands into the other stage, and the loads of the steps after it
            store_x(xr[(st + 1) % PD], buf ^ 1);
            store_w(raw[(st + 1) % PD], st < 7 ? blk_c : blk_n, buf ^ 1, (st + 1) & 7, st < 7 ? sign : -sign);
            if (st == 0 && SC == G8_SC_BLOCK) {
#pragma unroll
                for (int i = 0; i < WC; i++) {
                    const int row = r0 + 128 * i;
                    if constexpr (MIN) {
                        if (ch == 0) sd[row] = (sign * msc) * g8_half(blk_c[i].hdr.x & 0xFFFFu);
                        // v_g = -dmin m_g (exact in f32) of groups 2 ch, 2 ch + 1, times 2^-wexp, split
                        const float dm = g8_half(blk_c[i].hdr.x >> 16);
                        const uint32_t mn = g8_mins(blk_c[i].hdr, ch);
                        const float v0 = -(dm * (float)(mn & 0xFFu)) * wsc, v1 = -(dm * (float)(mn >> 8)) * wsc;
                        const g8_p2 h = __builtin_amdgcn_cvt_pkrtz(v0, v1);
                        const g8_p2 l = __builtin_amdgcn_cvt_pkrtz(v0 - (float)h[0], v1 - (float)h[1]);
                        uint32_t* dv = (uint32_t*)(swv + row * G8_LDV) + ch;
                        dv[0] = __builtin_bit_cast(uint32_t, h);
                        dv[4] = __builtin_bit_cast(uint32_t, l);
                        dv[8] = __builtin_bit_cast(uint32_t, h);
                    } else if constexpr (P == 2) {
                        if (ch == 0) sd[row] = sign * g8_half(blk_c[i].d);
                    }
                }
                if constexpr (MIN) {
                    // tokens: (X hi, X hi, X lo) against (v hi, v lo, v hi)
                    if (vt < BM) {
                        g8_u4* av = (g8_u4*)(sav + vt * G8_LDV);
                        if (vhl == 0) {
                            av[0] = xv;
                            av[1] = xv;
                        } else {
                            av[2] = xv;
                        }
                    }
                }
            }
            // past the part's end: its last block again, not used
            const int kp = kb + (st + 1 + PD) / 8 < b1 ? kb + (st + 1 + PD) / 8 : b1 - 1;
            load_x(xr[(st + 1) % PD], 256 * kp + G8_BK * ((st + 1 + PD) & 7));
            load_w(raw[(st + 1) % PD], kp, (st + 1 + PD) & 7);
            if (st == 1) load_b(blk_n, kn);
            if (MIN && st == 3 && vt < BM) xv = g8_ld16(vb, vp, 16u * kn);
            __builtin_amdgcn_sched_barrier(0);
            // x lo first: the small products meet small sums
#pragma unroll
            for (int i = 0; i < MI; i++)
#pragma unroll
                for (int j = 0; j < 4; j++)  // a block's sum starts from zero
                    blk[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(al[i], bh[j], (st == 0 && !F16) || SC == G8_SC_STEP ? zero : blk[i][j], 0, 0, 0);
            if constexpr (P == 2) {
                // read here, into the registers of the x lo operands
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int j = 0; j < 4; j++) bl[j] = *(const g8_h8*)(sw + (BN + 64 * wn + 16 * j) * G8_BK + oc);
#pragma unroll
                for (int i = 0; i < MI; i++)
#pragma unroll
                    for (int j = 0; j < 4; j++) blk[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah[i], bl[j], blk[i][j], 0, 0, 0);
            }
#pragma unroll
            for (int i = 0; i < MI; i++)
#pragma unroll
                for (int j = 0; j < 4; j++) blk[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah[i], bh[j], blk[i][j], 0, 0, 0);
            if constexpr (SC == G8_SC_STEP) {
#pragma unroll
                for (int i = 0; i < MI; i++)
#pragma unroll
                    for (int j = 0; j < 4; j++)
#pragma unroll
                        for (int e = 0; e < 4; e++) acc[i][j][e] = fmaf(dj[j], blk[i][j][e], acc[i][j][e]);
                // the sums stay in the step (the compiler had carried every step's blk to the block's end)
#pragma unroll
                for (int i = 0; i < MI; i++)
#pragma unroll
                    for (int j = 0; j < 4; j++) asm volatile("" : "+v"(acc[i][j]));
            } else if (st == 7 && !F16) {
                // the block's d times its sum, and its min term (one K slice: chunks 0, 1, 2 and zero)
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const float d = sd[64 * wn + 16 * j + l15];
#pragma unroll
                    for (int i = 0; i < MI; i++)
#pragma unroll
                        for (int e = 0; e < 4; e++) acc[i][j][e] = fmaf(d, blk[i][j][e], acc[i][j][e]);
                }
                if constexpr (MIN) {
                    const bool kz = lq == 3;
                    const int vo = kz ? 0 : 8 * lq;
                    const g8_h8 z8 = {};
                    g8_h8 av[MI], bv[4];
#pragma unroll
                    for (int i = 0; i < MI; i++) {
                        av[i] = *(const g8_h8*)(sav + (32 * TI * wm + 16 * i + l15) * G8_LDV + vo);
                        if (kz) av[i] = z8;
                    }
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        bv[j] = *(const g8_h8*)(swv + (64 * wn + 16 * j + l15) * G8_LDV + vo);
                        if (kz) bv[j] = z8;
                    }
#pragma unroll
                    for (int i = 0; i < MI; i++)
#pragma unroll
                        for (int j = 0; j < 4; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av[i], bv[j], acc[i][j], 0, 0, 0);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            __syncthreads();
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int i = 0; i < WC; i++) blk_c[i] = blk_n[i];
        sign = -sign;
    }

    // D lane l: column l & 15, rows 4 (l >> 4) + e. The residual values are loaded together, from
    // clamped addresses, before the first store.
    const bool add = a.add && blockIdx.z == 0;
    float* out = blockIdx.z == 0 ? sg.y
                                 : a.part + (size_t)(blockIdx.z - 1) * a.T * sg.ldy + (size_t)(sg.y - a.seg[0].y);
#pragma unroll
    for (int i = 0; i < MI; i++) {
        const int tb = t0 + 32 * TI * wm + 16 * i + 4 * lq;
        float old[4][4] = {};
        if (add) {
#pragma unroll
            for (int j = 0; j < 4; j++)
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const int t = tb + e, n = n0 + 64 * wn + 16 * j + l15;
                    old[j][e] = out[(size_t)(t < a.T ? t : a.T - 1) * sg.ldy + (n < sg.N ? n : sg.N - 1)];
                }
        }
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int n = n0 + 64 * wn + 16 * j + l15;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int t = tb + e;
                const float r = (F16 ? blk : acc)[i][j][e] * sxs[t - t0];  // exact
                if (t < a.T && n < sg.N) out[(size_t)t * sg.ldy + n] = add ? old[j][e] + r : r;
            }
        }
    }
}

template <int TI, int FORM>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void k_pf_gemm8(const PfGemm a) {
    extern __shared__ __attribute__((aligned(16))) _Float16 pf_ld8w[];
    int bx = blockIdx.x, si = 0;
    while (si + 1 < a.nseg && bx >= a.seg[si].tiles) bx -= a.seg[si++].tiles;
    const PfSeg& sg = a.seg[si];
    const int n0 = bx * 256, t0 = blockIdx.y * 64 * TI;
    if constexpr (FORM == PF_FORM_MIX) {
        if (sg.type == FLLM_TYPE_Q6_K) g8_tile<TI, FLLM_TYPE_Q6_K>(a, sg, n0, t0, pf_ld8w);
        else if (sg.type == FLLM_TYPE_Q5_K) g8_tile<TI, FLLM_TYPE_Q5_K>(a, sg, n0, t0, pf_ld8w);
        else if (sg.type == FLLM_TYPE_Q8_0) g8_tile<TI, FLLM_TYPE_Q8_0>(a, sg, n0, t0, pf_ld8w);
        else g8_tile<TI, FLLM_TYPE_Q4_K>(a, sg, n0, t0, pf_ld8w);
    } else {
        g8_tile<TI, FORM>(a, sg, n0, t0, pf_ld8w);
    }
}

template <int TI>
static PfKernel g8_form(int form) {
    // by the stage's planes and the min term: Q5_K as Q4_K, the others without either as Q8_0
    constexpr size_t l4 = G8T<TI, FLLM_TYPE_Q4_K>::lds, l6 = G8T<TI, FLLM_TYPE_Q6_K>::lds, l8 = G8T<TI, FLLM_TYPE_Q8_0>::lds;
    // us of one 256-element block of a wave of one workgroup per CU (two products a weight; Q6_K three)
    constexpr double u2 = TI == 2 ? 8.8 : 5.3, u3 = TI == 2 ? 12.6 : 7.7;
    switch (form) {
        case FLLM_TYPE_Q4_K: return {k_pf_gemm8<TI, FLLM_TYPE_Q4_K>, l4, 64 * TI, 256, 512, u2};
        case FLLM_TYPE_Q5_K: return {k_pf_gemm8<TI, FLLM_TYPE_Q5_K>, l4, 64 * TI, 256, 512, u2};
        case FLLM_TYPE_Q6_K: return {k_pf_gemm8<TI, FLLM_TYPE_Q6_K>, l6, 64 * TI, 256, 512, u3};
        case FLLM_TYPE_Q8_0: return {k_pf_gemm8<TI, FLLM_TYPE_Q8_0>, l8, 64 * TI, 256, 512, u2};
        case PF_FORM_MIX: return {k_pf_gemm8<TI, PF_FORM_MIX>, l4 > l6 ? l4 : l6, 64 * TI, 256, 512, u2};
        case PF_FORM_ROWS + FLLM_TYPE_Q4_K: return {k_pf_gemm8<TI, PF_FORM_ROWS + FLLM_TYPE_Q4_K>, l4, 64 * TI, 256, 512, u2};
        case PF_FORM_ROWS + FLLM_TYPE_Q5_K: return {k_pf_gemm8<TI, PF_FORM_ROWS + FLLM_TYPE_Q5_K>, l4, 64 * TI, 256, 512, u2};
        case PF_FORM_ROWS + FLLM_TYPE_Q6_K: return {k_pf_gemm8<TI, PF_FORM_ROWS + FLLM_TYPE_Q6_K>, l6, 64 * TI, 256, 512, u3};
        case PF_FORM_ROWS + FLLM_TYPE_Q8_0: return {k_pf_gemm8<TI, PF_FORM_ROWS + FLLM_TYPE_Q8_0>, l8, 64 * TI, 256, 512, u2};
        case PF_FORM_ROWS + FLLM_TYPE_Q4_0: return {k_pf_gemm8<TI, PF_FORM_ROWS + FLLM_TYPE_Q4_0>, l8, 64 * TI, 256, 512, u2};
        case PF_FORM_ROWS + FLLM_TYPE_F16: return {k_pf_gemm8<TI, PF_FORM_ROWS + FLLM_TYPE_F16>, l8, 64 * TI, 256, 512, u2};
        default: return {nullptr, 0, 0, 0, 0, 0.0};
    }
}
PfKernel pf_gemm8_kernel(int form, int bm) { return bm == 64 ? g8_form<1>(form) : g8_form<2>(form); }

}  // namespace fllm
