// fp32-activation reader of the reference's frontier backend on gfx950: the
// seven GGUF kinds of its frontier model (F32, BF16, Q8_0, Q6_K, IQ3_XXS,
// IQ4_NL, IQ4_XS), a bit-exact dequant, and y = W x with fp32 x for one
// weight or for a job table of many weights in one launch.
//
// Replaces frontier_dequant / frontier_matvec / frontier_multi_matvec
// (driver/kernels/frontier_quant.cu:12-93) and their CPU definition
// dequantize (driver/src/frontier_core.rs:73-106), behind Weights::linear and
// Weights::batch (driver/src/frontier_forward.rs:14-28, frontier_backend.rs).
//
// Arithmetic. Every decoded weight of these kinds is an integer code times an
// f32 block scale that is itself an exact product (fp16 d times a small
// integer, or a power-of-two fraction of one), so sum_i w_i x_i equals
// sum over scale groups of scale * sum(code * x) exactly. x is written out as
// base-256 integer digits, the digits' sums with the codes run on int8 matrix
// instructions and are exact, integer sub-scales multiply them exactly, and a
// double collects the blocks: the oracle's exact double sum up to ~2^-50
// relative, so both agree bit for bit except in rare rounding-boundary cases
// (<= 1 ulp). The order of a row's sums is fixed by its length alone, so the
// single-weight and job-table forms agree bit for bit always. F32 and BF16
// products are formed in double directly.
//
// Bound and choices (MI355X, HIP events over back-to-back launches, before ->
// after, "before" being five v_dot4 digit planes with 8-16 lanes a row):
//  * digits on the matrix core: v_dot4 needed 1.25 instructions and 5 bytes of
//    LDS per weight. v_mfma_i32_16x16x64_i8 takes all eight digits, of 1,024
//    weights in Q8_0 and of 512 in the other kinds, whose scale groups lie so that
//    each operand of codes goes out twice; an instruction reads 1 KB of digits, 1
//    and 2 bytes per weight, half or a quarter of it other than the zeros of a
//    foreign slice. What is left on the VALU is the unpacking of the codes (IQ4_XS
//    and IQ3_XXS: 122 instructions beside 8 products a step of 16 rows x 256
//    columns, 88 of them the code book), which bounds large IQ weights; Q6_K and
//    Q8_0 reach 5.9 and 5.3 TB/s at 151936 x 2560, of a 7.0 TB/s streaming read.
//  * 52000 x 2560: Q6_K 38.0 -> 21.4 us, IQ3_XXS 33.0 -> 17.2, IQ4_NL 31.0 ->
//    20.5, IQ4_XS 32.6 -> 17.1, Q8_0 30.0 -> 29.9. 256 x 16384: Q6_K 59.3 ->
//    13.6, Q8_0 34.4 -> 18.3. 640 x 2560: IQ3_XXS 10.2 -> 4.8. Q8_0 of 2560
//    columns and 70000 rows or more is 3 to 5% slower (37.0 -> 38.8 us), of 2048
//    or 4096 columns 6 to 12% faster.
//  * tiles of 16 rows are laid out at upload in the order in which a wave reads
//    them (whole kilobytes per load instruction); Q8_0 shares the int8 matvec's
//    row planes.
#include "uq_device.h"
#include "uq_internal.h"
#include "../../include/uq.h"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <string>
#include <vector>

namespace uq {
namespace {

// IQ4_NL / IQ4_XS code book (frontier_core.rs:67) and the IQ3_XXS grid
// (frontier_tables.rs:2-35, ggml's iq3xxs_grid): data of the format, from
// ggml (MIT licence, third_party/LICENSE.ggml).
__constant__ __attribute__((aligned(16))) int8_t c_iq4[16] = {-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113};
__constant__ uint32_t c_iq3_grid[256] = {
    0x04040404u, 0x04040414u, 0x04040424u, 0x04040c0cu, 0x04040c1cu, 0x04040c3eu, 0x04041404u, 0x04041414u,
    0x04041c0cu, 0x04042414u, 0x04043e1cu, 0x04043e2cu, 0x040c040cu, 0x040c041cu, 0x040c0c04u, 0x040c0c14u,
    0x040c140cu, 0x040c142cu, 0x040c1c04u, 0x040c1c14u, 0x040c240cu, 0x040c2c24u, 0x040c3e04u, 0x04140404u,
    0x04140414u, 0x04140424u, 0x04140c0cu, 0x04141404u, 0x04141414u, 0x04141c0cu, 0x04141c1cu, 0x04141c3eu,
    0x04142c0cu, 0x04142c3eu, 0x04143e2cu, 0x041c040cu, 0x041c043eu, 0x041c0c04u, 0x041c0c14u, 0x041c142cu,
    0x041c3e04u, 0x04240c1cu, 0x04241c3eu, 0x04242424u, 0x04242c3eu, 0x04243e1cu, 0x04243e2cu, 0x042c040cu,
    0x042c043eu, 0x042c1c14u, 0x042c2c14u, 0x04341c2cu, 0x04343424u, 0x043e0c04u, 0x043e0c24u, 0x043e0c34u,
    0x043e241cu, 0x043e340cu, 0x0c04040cu, 0x0c04041cu, 0x0c040c04u, 0x0c040c14u, 0x0c04140cu, 0x0c04141cu,
    0x0c041c04u, 0x0c041c14u, 0x0c041c24u, 0x0c04243eu, 0x0c042c04u, 0x0c0c0404u, 0x0c0c0414u, 0x0c0c0c0cu,
    0x0c0c1404u, 0x0c0c1414u, 0x0c14040cu, 0x0c14041cu, 0x0c140c04u, 0x0c140c14u, 0x0c14140cu, 0x0c141c04u,
    0x0c143e14u, 0x0c1c0404u, 0x0c1c0414u, 0x0c1c1404u, 0x0c1c1c0cu, 0x0c1c2434u, 0x0c1c3434u, 0x0c24040cu,
    0x0c24042cu, 0x0c242c04u, 0x0c2c1404u, 0x0c2c1424u, 0x0c2c2434u, 0x0c2c3e0cu, 0x0c34042cu, 0x0c3e1414u,
    0x0c3e2404u, 0x14040404u, 0x14040414u, 0x14040c0cu, 0x14040c1cu, 0x14041404u, 0x14041414u, 0x14041434u,
    0x14041c0cu, 0x14042414u, 0x140c040cu, 0x140c041cu, 0x140c042cu, 0x140c0c04u, 0x140c0c14u, 0x140c140cu,
    0x140c1c04u, 0x140c341cu, 0x140c343eu, 0x140c3e04u, 0x14140404u, 0x14140414u, 0x14140c0cu, 0x14140c3eu,
    0x14141404u, 0x14141414u, 0x14141c3eu, 0x14142404u, 0x14142c2cu, 0x141c040cu, 0x141c0c04u, 0x141c0c24u,
    0x141c3e04u, 0x141c3e24u, 0x14241c2cu, 0x14242c1cu, 0x142c041cu, 0x142c143eu, 0x142c240cu, 0x142c3e24u,
    0x143e040cu, 0x143e041cu, 0x143e0c34u, 0x143e242cu, 0x1c04040cu, 0x1c040c04u, 0x1c040c14u, 0x1c04140cu,
    0x1c04141cu, 0x1c042c04u, 0x1c04342cu, 0x1c043e14u, 0x1c0c0404u, 0x1c0c0414u, 0x1c0c1404u, 0x1c0c1c0cu,
    0x1c0c2424u, 0x1c0c2434u, 0x1c14040cu, 0x1c14041cu, 0x1c140c04u, 0x1c14142cu, 0x1c142c14u, 0x1c143e14u,
    0x1c1c0c0cu, 0x1c1c1c1cu, 0x1c241c04u, 0x1c24243eu, 0x1c243e14u, 0x1c2c0404u, 0x1c2c0434u, 0x1c2c1414u,
    0x1c2c2c2cu, 0x1c340c24u, 0x1c341c34u, 0x1c34341cu, 0x1c3e1c1cu, 0x1c3e3404u, 0x24040424u, 0x24040c3eu,
    0x24041c2cu, 0x24041c3eu, 0x24042c1cu, 0x24042c3eu, 0x240c3e24u, 0x24141404u, 0x24141c3eu, 0x24142404u,
    0x24143404u, 0x24143434u, 0x241c043eu, 0x241c242cu, 0x24240424u, 0x24242c0cu, 0x24243424u, 0x242c142cu,
    0x242c241cu, 0x242c3e04u, 0x243e042cu, 0x243e0c04u, 0x243e0c14u, 0x243e1c04u, 0x2c040c14u, 0x2c04240cu,
    0x2c043e04u, 0x2c0c0404u, 0x2c0c0434u, 0x2c0c1434u, 0x2c0c2c2cu, 0x2c140c24u, 0x2c141c14u, 0x2c143e14u,
    0x2c1c0414u, 0x2c1c2c1cu, 0x2c240c04u, 0x2c24141cu, 0x2c24143eu, 0x2c243e14u, 0x2c2c0414u, 0x2c2c1c0cu,
    0x2c342c04u, 0x2c3e1424u, 0x2c3e2414u, 0x34041424u, 0x34042424u, 0x34042434u, 0x34043424u, 0x340c140cu,
    0x340c340cu, 0x34140c3eu, 0x34143424u, 0x341c1c04u, 0x341c1c34u, 0x34242424u, 0x342c042cu, 0x342c2c14u,
    0x34341c1cu, 0x343e041cu, 0x343e140cu, 0x3e04041cu, 0x3e04042cu, 0x3e04043eu, 0x3e040c04u, 0x3e041c14u,
    0x3e042c14u, 0x3e0c1434u, 0x3e0c2404u, 0x3e140c14u, 0x3e14242cu, 0x3e142c14u, 0x3e1c0404u, 0x3e1c0c2cu,
    0x3e1c1c1cu, 0x3e1c3404u, 0x3e24140cu, 0x3e24240cu, 0x3e2c0404u, 0x3e2c0414u, 0x3e2c1424u, 0x3e341c04u,
};

constexpr int FWG = 256;
constexpr int FL_WG = 512;  // workgroup of the linear kernel

constexpr bool row_kind(uint32_t kind) { return kind == KIND_F32 || kind == KIND_BF16; }

// ---------------------------------------------------------------- dequant
// One value per thread from the GGUF bytes, the formulas and f32 multiply
// order of dequantize (frontier_core.rs:73-106).
__device__ __forceinline__ uint32_t rd16(const uint8_t* p) { return (uint32_t)p[0] | ((uint32_t)p[1] << 8); }
__device__ __forceinline__ uint32_t rd32(const uint8_t* p) { return rd16(p) | (rd16(p + 2) << 16); }

__device__ float dequant_value(uint32_t kind, const uint8_t* in, int64_t i) {
    switch (kind) {
    case KIND_F32: return uq_bits_f(rd32(in + 4 * i));
    case KIND_BF16: return uq_bits_f(rd16(in + 2 * i) << 16);
    case KIND_Q8_0: {
        const uint8_t* p = in + (i / 32) * 34;
        return uq_half((uint16_t)rd16(p)) * (float)(int8_t)p[2 + i % 32];
    }
    case KIND_IQ4_NL: {
        const uint8_t* p = in + (i / 32) * 18;
        const int j = (int)(i % 32), q = (p[2 + j % 16] >> (4 * (j / 16))) & 15;
        return uq_half((uint16_t)rd16(p)) * (float)c_iq4[q];
    }
    case KIND_IQ4_XS: {
        const uint8_t* p = in + (i / 256) * 136;
        const int j = (int)(i % 256), sb = j / 32;
        const int sc = ((p[4 + sb / 2] >> (4 * (sb % 2))) & 15) | (((rd16(p + 2) >> (2 * sb)) & 3) << 4);
        const int q = (p[8 + sb * 16 + j % 16] >> (4 * ((j % 32) / 16))) & 15;
        return (uq_half((uint16_t)rd16(p)) * (float)(sc - 32)) * (float)c_iq4[q];
    }
    case KIND_Q6_K: {
        const uint8_t* p = in + (i / 256) * 210;
        const int j = (int)(i % 256), sub = j / 128, l = j % 32, g = (j % 128) / 32;
        const int lo = p[sub * 64 + l + (g % 2) * 32], hi = p[128 + sub * 32 + l];
        const int q = (((lo >> (4 * (g / 2))) & 15) | (((hi >> (2 * g)) & 3) << 4)) - 32;
        const int sc = (int8_t)p[192 + sub * 8 + l / 16 + g * 2];
        return (uq_half((uint16_t)rd16(p + 208)) * (float)sc) * (float)q;
    }
    case KIND_IQ3_XXS: {
        const uint8_t* p = in + (i / 256) * 98;
        const int j = (int)(i % 256), sb = j / 32, g = (j % 32) / 8;
        const uint32_t aux = rd32(p + 66 + sb * 4), s7 = (aux >> (7 * g)) & 127;
        const uint32_t sg = s7 | ((uint32_t)(__popc(s7) & 1) << 7);
        const int idx = p[2 + sb * 8 + g * 2 + (j % 8) / 4];
        const uint32_t q = (c_iq3_grid[idx] >> (8 * (j % 4))) & 255;
        const float scale = uq_half((uint16_t)rd16(p)) * (0.5f + (float)(aux >> 28)) * 0.5f;
        return (scale * (float)q) * ((sg & (1u << (j % 8))) ? -1.0f : 1.0f);
    }
    }
    return __builtin_nanf("");
}

__global__ __launch_bounds__(FWG) void k_dequant(const uint8_t* __restrict__ in, float* __restrict__ out, uint32_t kind,
                                                 int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * FWG + threadIdx.x; i < n; i += (int64_t)gridDim.x * FWG)
        out[i] = dequant_value(kind, in, i);
}

// ---------------------------------------------------------------- layout repack / verify
// 16-entry code books as v_perm_b32 tables. A selector byte q < 8 picks byte q
// of the table; 8..11 give the sign of byte 1, 3, 5 or 7 (0x00 here, see below),
// 12 gives 0x00 and 13..15 give 0xFF. With the codes 0..7 in one table and 8..15
// in another, perm(first, q) ^ perm(second, q ^ 8) is the entry itself, or its
// complement for (q & 7) >= 5: the tables hold those entries complemented. That
// takes four instructions behind the masked nibbles where picking one of two
// table bytes by bit 3 took five. The order of the codes makes bytes 1, 3, 5 and
// 7 of both tables non-negative: values >= 0 at 1 and 3, values < 0
// (complemented) at 5 and 7.
struct Book {
    uint32_t t[4];
};
constexpr int BOOK_ORDER[16] = {0, 8, 1, 9, 10, 2, 11, 3, 4, 12, 5, 13, 14, 6, 15, 7};  // code -> place in ascending order
constexpr Book make_book(const int (&ascending)[16]) {
    Book b{};
    for (int q = 0; q < 16; q++) {
        const int v = ascending[BOOK_ORDER[q]], e = (q & 7) >= 5 ? ~v : v;
        b.t[q / 4] |= (uint32_t)(e & 255) << (8 * (q % 4));
    }
    return b;
}
constexpr int IQ4_VALUES[16] = {-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113};
constexpr int IQ3_VALUES[16] = {-62, -52, -44, -36, -28, -20, -12, -4, 4, 12, 20, 28, 36, 44, 52, 62};
constexpr Book IQ4_BOOK = make_book(IQ4_VALUES), IQ3_BOOK = make_book(IQ3_VALUES);
// place in ascending order -> code, four bits each
constexpr uint64_t book_codes() {
    uint64_t m = 0;
    for (int q = 0; q < 16; q++) m |= (uint64_t)q << (4 * BOOK_ORDER[q]);
    return m;
}
constexpr uint64_t book_places() {
    uint64_t m = 0;
    for (int q = 0; q < 16; q++) m |= (uint64_t)BOOK_ORDER[q] << (4 * q);
    return m;
}
__device__ __forceinline__ uint32_t nibble_of(uint64_t table, uint32_t i) { return (uint32_t)(table >> (4 * i)) & 15u; }
// both nibbles of a byte through a 16-entry table
__device__ __forceinline__ uint32_t recode(uint64_t table, uint32_t b) {
    return nibble_of(table, b & 15) | nibble_of(table, b >> 4) << 4;
}

struct LayoutArgs {
    int64_t m;
    int32_t kind, block_bytes, blocks;  // blocks per row
    int32_t steps, bps;                 // steps per row, blocks per step
    int32_t rec[3];                     // bytes of a tile's step in each plane
    int64_t dwords[3];                  // of each plane
    uint8_t* plane[3];
};

// Codes of values e .. e + 3 (e % 4 == 0) of 32-value block sb of an IQ3_XXS
// superblock, one a byte.
__device__ __forceinline__ uint32_t iq3_codes(const uint8_t* p, int sb, int e) {
    const uint32_t s7 = (rd32(p + 66 + 4 * sb) >> (7 * (e / 8))) & 127u;
    const uint32_t neg = (s7 | (uint32_t)(__popc(s7) & 1) << 7) >> (e % 8);
    const uint32_t levels = c_iq3_grid[p[2 + 8 * sb + e / 4]] >> 3;
    uint32_t v = 0;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const uint32_t level = (levels >> (8 * k)) & 7u;
        v |= nibble_of(book_codes(), (neg >> k) & 1u ? 7 - level : 8 + level) << (8 * k);
    }
    return v;
}

// Byte `at` of a tile's step in plane pl: what the block's bytes p (of the
// lane's or row's own block) put there.
__device__ uint32_t plane_byte(const LayoutArgs& a, const uint8_t* src, int pl, int64_t rec, int at) {
    const int64_t tile = rec / a.steps;
    const int t = (int)(rec - tile * a.steps);
    const int sixth = a.rec[FL_ROW] == 160 && pl == FL_ROW;  // 16 x 8 scale bytes, then 16 x 2 bytes of d
    int g = 0, r, o;  // lane group, row of the tile, byte of the record
    if (pl == FL_BODY) {
        const int lane = (at & 1023) >> 4;
        g = lane >> 4;
        r = lane & 15;
        o = 16 * (at >> 10) + (at & 15);
    } else if (pl == FL_LANE) {
        const int w = a.rec[FL_LANE] / 64, lane = at / w;
        g = lane >> 4;
        r = lane & 15;
        o = at - lane * w;
    } else if (sixth && at < 128) {
        r = at >> 3;
        o = at & 7;
    } else {
        r = (sixth ? at - 128 : at) >> 1;
        o = 8 + (at & 1);
    }
    const int64_t row = 16 * tile + r, b = (int64_t)t * a.bps + (a.bps > 1 ? g : 0);
    if (row >= a.m || b >= a.blocks) return 0;
    const uint8_t* p = src + (row * a.blocks + b) * a.block_bytes;
    switch (a.kind) {
    case KIND_IQ4_NL: return pl == FL_BODY ? recode(book_codes(), p[2 + o]) : p[o];
    case KIND_IQ4_XS:
        if (pl == FL_BODY) return recode(book_codes(), p[8 + 16 * (4 * (o >> 4) + g) + (o & 15)]);
        if (o >= 8) return p[o - 8];
        else {  // scale byte o: slice o >> 2, its block number o & 3
            const int sb = 2 * (o & 3) + (o >> 2);
            return (uint32_t)((int)((p[4 + sb / 2] >> (4 * (sb % 2))) & 15) + (int)(((rd16(p + 2) >> (2 * sb)) & 3) << 4) - 32) & 255u;
        }
    case KIND_IQ3_XXS:
        if (o >= 8) return p[o - 8];  // (the body: k_layout_repack)
        return 2 * (p[66 + 4 * (2 * (o & 3) + (o >> 2)) + 3] >> 4) + 1;
    default:  // Q6_K
        if (pl == FL_BODY)
            return o < 32 ? p[(g >> 1) * 64 + 32 * (o >> 4) + 16 * (g & 1) + (o & 15)]
                          : p[128 + (g >> 1) * 32 + 16 * (g & 1) + (o & 15)];
        return pl == FL_LANE ? p[192 + (g >> 1) * 8 + (g & 1) + 2 * o] : p[208 + o - 8];
    }
}

// One dword of a plane per thread, the planes one behind the other; rows past the
// last and columns past n are zero. The bytes of an IQ3_XXS body hold two codes
// each and are made four at a time, as their grid words and signs are shared.
__global__ __launch_bounds__(FWG) void k_layout_repack(const uint8_t* __restrict__ src, LayoutArgs a, int64_t total) {
    for (int64_t j = (int64_t)blockIdx.x * FWG + threadIdx.x; j < total; j += (int64_t)gridDim.x * FWG) {
        int64_t i = j;
        int pl = 0;
        while (i >= a.dwords[pl]) i -= a.dwords[pl++];
        const int64_t rec = 4 * i / a.rec[pl];
        const int at = (int)(4 * i - rec * a.rec[pl]);
        uint32_t v = 0;
        if (a.kind == KIND_IQ3_XXS && pl == FL_BODY) {
            const int64_t tile = rec / a.steps, row = 16 * tile + ((at >> 4) & 15);
            const int sb = 4 * (at >> 10) + ((at >> 8) & 3);
            const uint8_t* p = src + (row * a.blocks + (rec - tile * a.steps)) * a.block_bytes;
            if (row < a.m) v = iq3_codes(p, sb, at & 15) | iq3_codes(p, sb, 16 + (at & 15)) << 4;
        } else {
#pragma unroll 1
            for (int k = 0; k < 4; k++) v |= plane_byte(a, src, pl, rec, at + k) << (8 * k);
        }
        ((uint32_t*)a.plane[pl])[i] = v;
    }
}

// Byte o of block b of a row as the planes hold it (-1: no GGUF bytes give them).
__device__ int source_byte(const LayoutArgs& a, int64_t row, int64_t b, int o) {
    const int64_t rec = (row >> 4) * a.steps + b / a.bps;
    const int r = (int)(row & 15);
    // the body byte `at` of lane group g's record
    auto body = [&](int g, int at) {
        return (uint32_t)a.plane[FL_BODY][rec * a.rec[FL_BODY] + 1024 * (at >> 4) + 16 * (16 * g + r) + (at & 15)];
    };
    auto scale = [&](int sb) { return (int)(int8_t)a.plane[FL_ROW][rec * 160 + 8 * r + 4 * (sb & 1) + (sb >> 1)]; };
    switch (a.kind) {
    case KIND_IQ4_NL: {
        const int g = (int)(b % a.bps);
        if (o < 2) return a.plane[FL_LANE][rec * 128 + 2 * (16 * g + r) + o];
        return (int)recode(book_places(), body(g, o - 2));
    }
    case KIND_IQ4_XS:
        if (o < 2) return a.plane[FL_ROW][rec * 160 + 128 + 2 * r + o];
        if (o < 4) {  // scales_h: two high bits of blocks 4(o - 2) ..
            int v = 0;
            for (int k = 0; k < 4; k++) v |= (((scale(4 * (o - 2) + k) + 32) >> 4) & 3) << (2 * k);
            return v;
        }
        if (o < 8) return ((scale(2 * (o - 4)) + 32) & 15) | ((scale(2 * (o - 4) + 1) + 32) & 15) << 4;
        return (int)recode(book_places(), body(((o - 8) >> 4) & 3, 16 * ((o - 8) >> 6) + ((o - 8) & 15)));
    default: {  // Q6_K
        if (o < 128) return (int)body(2 * (o >> 6) + ((o >> 4) & 1), 16 * ((o >> 5) & 1) + (o & 15));
        if (o < 192) return (int)body(2 * ((o - 128) >> 5) + ((o >> 4) & 1), 32 + (o & 15));
        if (o < 208) {
            const int i = o - 192, g = 2 * (i >> 3) + (i & 1);
            return a.plane[FL_LANE][rec * 256 + 4 * (16 * g + r) + ((i & 7) >> 1)];
        }
        return a.plane[FL_ROW][rec * 32 + 2 * r + (o - 208)];
    }
    }
}

__global__ __launch_bounds__(FWG) void k_layout_verify(const uint8_t* __restrict__ src, LayoutArgs a, int64_t total,
                                                       unsigned* bad) {
    unsigned miss = 0;
    for (int64_t i = (int64_t)blockIdx.x * FWG + threadIdx.x; i < total; i += (int64_t)gridDim.x * FWG) {
        const int64_t blk = i / a.block_bytes, row = blk / a.blocks;
        miss += source_byte(a, row, blk - row * a.blocks, (int)(i - blk * a.block_bytes)) != (int)src[i];
    }
    if (miss) atomicAdd(bad, miss);
}

// An IQ3_XXS superblock from its planes, a 32-value block per thread: the eight grid
// words (the grid's entries are distinct, so one names its index), the signs with
// their parity, the scale, and with block 0 the two bytes of d. Byte by byte, with
// a search of the grid, 50000 x 2560 took 0.5 ms longer to upload.
__global__ __launch_bounds__(FWG) void k_iq3_verify(const uint8_t* __restrict__ src, LayoutArgs a, int64_t total,
                                                    unsigned* bad) {
    unsigned miss = 0;
    for (int64_t i = (int64_t)blockIdx.x * FWG + threadIdx.x; i < total; i += (int64_t)gridDim.x * FWG) {
        const int64_t blk = i >> 3, row = blk / a.blocks, rec = (row >> 4) * a.steps + (blk - row * a.blocks);
        const int sb = (int)(i & 7), r = (int)(row & 15);
        const uint8_t* p = src + blk * a.block_bytes;
        const uint8_t* rr = a.plane[FL_ROW] + rec * a.rec[FL_ROW];
        const uint4 b = *(const uint4*)(a.plane[FL_BODY] + rec * a.rec[FL_BODY] + 1024 * (sb >> 2) + 16 * (16 * (sb & 3) + r));
        const uint32_t v[4] = {b.x, b.y, b.z, b.w};
        uint32_t signs = 0;
#pragma unroll
        for (int q = 0; q < 8; q++) {
            uint32_t w = 0;
#pragma unroll
            for (int k = 0; k < 4; k++) {
                // place in ascending order: below 8 negative
                const uint32_t place = nibble_of(book_places(), (v[q & 3] >> (8 * k + 4 * (q >> 2))) & 15u);
                const uint32_t level = place < 8 ? 7 - place : place - 8;
                w |= (level == 7 ? 62u : 8 * level + 4) << (8 * k);
                signs |= (place < 8 ? 1u : 0u) << (4 * q + k);
            }
            miss += c_iq3_grid[p[2 + 8 * sb + q]] != w;
        }
        const int sc = (int)(int8_t)rr[8 * r + 4 * (sb & 1) + (sb >> 1)];
        uint32_t aux = (uint32_t)(sc >> 1) << 28;
        miss += (sc & 1) == 0;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const uint32_t neg = (signs >> (8 * k)) & 255u;
            miss += (unsigned)__popc(neg) & 1u;
            aux |= (neg & 127u) << (7 * k);
        }
        miss += aux != rd32(p + 66 + 4 * sb);
        if (sb == 0) miss += rd16(rr + 128 + 2 * r) != rd16(p);
    }
    if (miss) atomicAdd(bad, miss);
}

// F32 / BF16 rows against their copy
__global__ __launch_bounds__(FWG) void k_copy_verify(const uint4* __restrict__ src, const uint4* __restrict__ dst,
                                                     int64_t n, unsigned* bad) {
    unsigned miss = 0;
    for (int64_t i = (int64_t)blockIdx.x * FWG + threadIdx.x; i < n; i += (int64_t)gridDim.x * FWG) {
        const uint4 x = src[i], y = dst[i];
        miss += (x.x != y.x) + (x.y != y.y) + (x.z != y.z) + (x.w != y.w);
    }
    if (miss) atomicAdd(bad, miss);
}

// ---------------------------------------------------------------- fp32-x matvec
// Job of the launch (the FrontierJob of frontier_quant.cu:71-78 with the
// planes of an uploaded weight): rows [0, m) of one weight times x.
struct FJob {
    const uint8_t* body;  // tiles (or, for F32, BF16 and Q8_0, rows of `pitch` bytes)
    const uint8_t* lane;  // per-lane records of a tile's step
    const uint8_t* row;   // per-row records of a tile's step (Q8_0: the fp16 scale plane)
    const float* x;
    float* y;
    int64_t m, pitch;
    int32_t kind, n;
    int32_t wg0, wgs;  // first workgroup of the job (JobArgs::start), workgroups of the job
};

// ---- exact integer form of x
// x is staged in LDS as integers X_j with x_j = X_j * 2^(E - 188) in groups of
// 256 values: E = max(biased exponent of max|x_j|, 1), |X_j| < 2^62, exact when
// every element lies within 2^38 of the group's maximum (or has zeros in the
// bits that fall away). X_j is held as eight balanced base-256 digits. Four values
// with one among them that is not exact (wider range, or not finite) have digits 0
// and a bit in their group's `far`, the group one in `wide`; their products run in
// double from x itself.
//
// The dots run on v_mfma_i32_16x16x64_i8 with the weights of 16 rows as one
// operand and the digits as the other, so one instruction forms all eight
// digits' sums of two scale groups for 16 rows, where v_dot4 needed eight
// instructions a dword. The matrix core has 16 columns: eight digits of two
// scale groups (slices). A column belongs to one slice, so the digits of the
// other chunks in it are zeros.
//
// LDS: 16-value chunk c holds digit d as 16 bytes at XCHUNK*c + 16*d and 16 zero
// bytes behind the eighth, which the column lanes of another slice read. The
// stride of nine 16-byte slots spreads the staging's dword writes of one digit
// over all banks (eight slots would put eight chunks on one bank).
constexpr int XDIG = 8, XGROUP = 256, XCHUNK = 16 * (XDIG + 1);

struct XStage {
    const uint8_t* dig;
    const double* gexp;   // per group: 2^(E - 188)
    const uint64_t* far;  // per group: bit q: values 4q .. 4q + 3 run in double
    const float* xg;      // x in global memory (those values)
    const float* xf;      // F32 / BF16 weights: x as f32 in LDS
    uint64_t wide;        // bit g: group g has such values
    int n;
};

// Four bytes of each of four dwords, byte k of all four in out[k].
__device__ __forceinline__ void bytes_transposed(const uint32_t (&v)[4], uint32_t (&out)[4]) {
    const uint32_t a01 = __builtin_amdgcn_perm(v[1], v[0], 0x05010400u);
    const uint32_t a23 = __builtin_amdgcn_perm(v[3], v[2], 0x05010400u);
    const uint32_t b01 = __builtin_amdgcn_perm(v[1], v[0], 0x07030602u);
    const uint32_t b23 = __builtin_amdgcn_perm(v[3], v[2], 0x07030602u);
    out[0] = __builtin_amdgcn_perm(a23, a01, 0x05040100u);
    out[1] = __builtin_amdgcn_perm(a23, a01, 0x07060302u);
    out[2] = __builtin_amdgcn_perm(b23, b01, 0x05040100u);
    out[3] = __builtin_amdgcn_perm(b23, b01, 0x07060302u);
}

// The first groups of a wave, loaded ahead of its weights: loads return in
// order, and x behind the weights would wait for HBM.
constexpr int XAHEAD = 2;
__device__ __forceinline__ float4 load_group(const float* __restrict__ x, int n, int grp) {
    const int q = 64 * grp + ((int)threadIdx.x & 63);
    return ((const float4*)x)[4 * q < n ? q : n / 4 - 1];
}
__device__ __forceinline__ void load_ahead(const float* __restrict__ x, int n, float4 (&v)[XAHEAD]) {
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), nw = (int)blockDim.x >> 6;
#pragma unroll
    for (int r = 0; r < XAHEAD; r++) v[r] = load_group(x, n, wave + r * nw);
}

// Stages x of one job, one 256-value group per wave at a time, 4 values per
// lane; returns the wave's wide groups.
__device__ __forceinline__ uint64_t stage_x(const float* __restrict__ x, int n, const float4 (&ahead)[XAHEAD], uint8_t* dig,
                                            double* gexp, uint64_t* far) {
    const int lane = threadIdx.x & 63, nw = (int)blockDim.x >> 6, ng = (n + XGROUP - 1) / XGROUP;
    uint64_t wide = 0;
    const int first = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    auto group = [&](int grp, const float4& v4) {
        const int q = 64 * grp + lane;
        const float v[4] = {4 * q < n ? v4.x : 0.0f, 4 * q < n ? v4.y : 0.0f, 4 * q < n ? v4.z : 0.0f,
                            4 * q < n ? v4.w : 0.0f};
        const float amax = uq_group_max<64>(fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fmaxf(fabsf(v[2]), fabsf(v[3]))));
        int E = (int)((__builtin_bit_cast(uint32_t, amax) >> 23) & 255);
        bool ok = E < 255;  // (a NaN is not its own floor below)
        E = E < 1 ? 1 : (E > 254 ? 254 : E);
        const double up = __builtin_bit_cast(double, (uint64_t)(188 - E + 1023) << 52);
        uint32_t lo[4], hi[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            // X = x * 2^(188 - E) as 2^32 * h + l, 0 <= l < 2^32: exact where X is
            // whole. (l alone does not show it: just below zero it rounds to 2^32.)
            const double X = (double)v[k] * up, h = __builtin_floor(X * 0x1p-32), l = __builtin_fma(h, -0x1p32, X);
            ok = ok && X == __builtin_floor(X);
            // offset binary: digit d = byte d of (X + 0x8080808080808080) - 0x80
            const uint64_t Y = ((uint64_t)(uint32_t)(int)h << 32 | (uint32_t)l) + 0x8080808080808080ull;
            lo[k] = (uint32_t)Y ^ 0x80808080u;
            hi[k] = (uint32_t)(Y >> 32) ^ 0x80808080u;
        }
        uint32_t d[8];
        {
            uint32_t t[4];
            bytes_transposed(lo, t);
#pragma unroll
            for (int k = 0; k < 4; k++) d[k] = t[k];
            bytes_transposed(hi, t);
#pragma unroll
            for (int k = 0; k < 4; k++) d[4 + k] = t[k];
        }
        const uint64_t out = __builtin_amdgcn_ballot_w64(!ok);
        if (__builtin_expect(out != 0, 0)) {
            wide |= 1ull << grp;
            if (lane == 0) far[grp] = out;
#pragma unroll
            for (int k = 0; k < XDIG; k++) d[k] = ok ? d[k] : 0;
        }
        const int c = q >> 2;
#pragma unroll
        for (int k = 0; k < XDIG; k++) *(uint32_t*)(dig + XCHUNK * c + 16 * k + 4 * (q & 3)) = d[k];
        *(uint32_t*)(dig + XCHUNK * c + 16 * XDIG + 4 * (q & 3)) = 0;
        if (lane == 0) gexp[grp] = __builtin_bit_cast(double, (uint64_t)(E - 188 + 1023) << 52);
    };
#pragma unroll
    for (int r = 0; r < XAHEAD; r++)
        if (first + r * nw < ng) group(first + r * nw, ahead[r]);
#pragma unroll 1
    for (int grp = first + XAHEAD * nw; grp < ng; grp += nw) group(grp, load_group(x, n, grp));
    return wide;
}

typedef int v4i __attribute__((ext_vector_type(4)));
__device__ __forceinline__ v4i as_v4i(const uint32_t (&c)[4]) { return v4i{(int)c[0], (int)c[1], (int)c[2], (int)c[3]}; }
__device__ __forceinline__ v4i lds16(const uint8_t* p) { return *(const v4i*)p; }

// Lane roles. As an operand lane, lane l holds 16 codes of row l & 15 of the
// tile, of the chunk that its lane group g = l >> 4 stands for, and 16 bytes of
// column l & 15 = 8 * slice + digit of the digits. As a result lane it holds
// four digits (4 * (g & 1) ..) of slice g >> 1 for row l & 15. Pair p of a set
// of four chunks takes the chunks of lane groups 2p and 2p + 1 as its slices:
// column lanes whose chunk is not their slice's read its zeros.
struct Lane {
    int lane, row, g;
    int slot[2];  // byte offset in a chunk of the digit that this lane reads for pair p
    __device__ __forceinline__ Lane() {
        lane = (int)threadIdx.x & 63;
        row = lane & 15;
        g = lane >> 4;
#pragma unroll
        for (int p = 0; p < 2; p++) slot[p] = 16 * (g == 2 * p + (row >> 3) ? row & 7 : XDIG);
    }
};
// The value of lane groups (2p, 2p + 1) in the result lanes of slices (0, 1).
__device__ __forceinline__ void to_slices(uint32_t v, uint32_t (&out)[2]) {
    const auto a = __builtin_amdgcn_permlane16_swap(v, v, false, false);  // [0 0 2 2], [1 1 3 3]
    const auto b = __builtin_amdgcn_permlane32_swap(a[0], a[1], false, false);
    out[0] = b[0];
    out[1] = b[1];
}

// ---- per-kind steps
// A wave walks a tile of 16 rows in steps of VPS columns; U is what a lane
// loads for one step, NB how many steps are in flight. Two pay where the bytes
// per instruction are many (Q8_0 and Q6_K, 52000 x 2560: 35.8 -> 30.9 us, 25.2 ->
// 22.2; Q8_0 with three or four within 4% of it from n 2048 on, slower below); for
// short waves (one_kernel) the smaller code of one does. The IQ kinds have one: two
// make IQ4_XS and IQ3_XXS 3 to 15% slower to n 1024 (151936 rows 3% faster) and 9%
// slower to 4% faster at 2560, but 15% faster at n 8192 from 13000 rows on (IQ4_NL
// 24%; at 2560 1% slower to 9% faster), where a CU holds
// one workgroup. step() adds the step's products to the lane's four digit sums;
// chunk() gives 16 codes and their scale, column() their first column, for the
// products that run in double.

// 16 codes of a 32-value block of nibbles through a code book: the low nibbles
// are its values 0..15, the high ones 16..31.
__device__ __forceinline__ void book_codes16(const Book& k, const uint4& w, int half, uint32_t (&c)[4]) {
    const uint32_t v[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const uint32_t sel = (half ? v[q] >> 4 : v[q]) & 0x0F0F0F0Fu;
        c[q] = __builtin_amdgcn_perm(k.t[1], k.t[0], sel) ^ __builtin_amdgcn_perm(k.t[3], k.t[2], sel ^ 0x08080808u);
    }
}

// A step runs in phases, kept apart by scheduling barriers: the digits of all
// its products are read from LDS first, the codes are unpacked while those
// reads are out, then the products go out back to back and their sums are
// scaled. Left to itself the compiler reads each product's digits right before
// it, and a wave spends its time waiting for LDS.
__device__ __forceinline__ void phase() { __builtin_amdgcn_sched_barrier(0); }

__device__ __forceinline__ v4i mfma64(const v4i& x, const v4i& w, const v4i& c) {
    return __builtin_amdgcn_mfma_i32_16x16x64_i8(x, w, c, 0, 0, 0);
}

// Four 32-value blocks (lane group g: block 4t + g) with an fp16 scale each.
template <class T>
__device__ __forceinline__ void step_f16(const typename T::U& u, const Lane& ln, const XStage& xs, int t, double (&acc)[4]) {
    v4i x[2][2];
#pragma unroll
    for (int p = 0; p < 2; p++)
#pragma unroll
        for (int h = 0; h < 2; h++)
            x[p][h] = lds16(xs.dig + (2 * XCHUNK * ln.g + ln.slot[p]) + 8 * XCHUNK * t + h * XCHUNK);
    const double e = xs.gexp[t >> 1];
    phase();
    uint32_t c0[4], c1[4], sc[2];
    T::codes(u, 0, c0);
    T::codes(u, 1, c1);
    to_slices(__builtin_bit_cast(uint32_t, uq_half((uint16_t)u.d)), sc);
    const v4i w0 = as_v4i(c0), w1 = as_v4i(c1), z = {0, 0, 0, 0};
    v4i d[2];
#pragma unroll
    for (int p = 0; p < 2; p++) d[p] = mfma64(x[p][0], w0, z);
#pragma unroll
    for (int p = 0; p < 2; p++) d[p] = mfma64(x[p][1], w1, d[p]);
#pragma unroll
    for (int p = 0; p < 2; p++) {
        const double s = (double)uq_bits_f(sc[p]) * e;
#pragma unroll
        for (int i = 0; i < 4; i++) acc[i] = __builtin_fma((double)d[p][i], s, acc[i]);
    }
}

// Eight 32-value blocks of a superblock (lane group g: blocks g and 4 + g):
// products of the codes w with the digits x, each block's sums times its
// integer scale.
__device__ __forceinline__ void read_blocks(const Lane& ln, const XStage& xs, int t, v4i (&x)[2][2][2]) {
#pragma unroll
    for (int b = 0; b < 2; b++)
#pragma unroll
        for (int p = 0; p < 2; p++)
#pragma unroll
            for (int h = 0; h < 2; h++)
                x[b][p][h] = lds16(xs.dig + (2 * XCHUNK * ln.g + ln.slot[p]) + 16 * XCHUNK * t + (8 * b + h) * XCHUNK);
}
__device__ __forceinline__ void block_sums(const v4i (&x)[2][2][2], const v4i (&w)[2][2], const int (&sc)[2][2], int (&ia)[4]) {
    v4i d[2][2];
    const v4i z = {0, 0, 0, 0};
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
        for (int b = 0; b < 2; b++)
#pragma unroll
            for (int p = 0; p < 2; p++) d[b][p] = mfma64(x[b][p][h], w[b][h], h ? d[b][p] : z);
#pragma unroll
    for (int i = 0; i < 4; i++) {
        ia[i] = __mul24(sc[0][0], d[0][0][i]);
        ia[i] += __mul24(sc[0][1], d[0][1][i]);
        ia[i] += __mul24(sc[1][0], d[1][0][i]);
        ia[i] += __mul24(sc[1][1], d[1][1][i]);
    }
}

template <uint32_t K>
struct TK;

// Q8_0 shares the int8 matvec's row planes: a load instruction reads 64 bytes
// (two blocks) of each of the tile's rows, lane group g their chunk g, so the
// two halves of a block meet in one instruction and one column slice.
template <>
struct TK<KIND_Q8_0> {
    static constexpr int VPS = 128, CHUNKS = 2, NB = 2;
    struct U {
        uint4 a, b;
        uint32_t d;  // scale of block 4t + g
    };
    static __device__ __forceinline__ U load(const FJob& j, int64_t tile, int t, int lane) {
        const int64_t r = 16 * tile + (lane & 15), rr = r < j.m - 1 ? r : j.m - 1;
        const int c0 = VPS * t + 16 * (lane >> 4), c1 = c0 + 64, last = j.n - 16;
        const int8_t* p = (const int8_t*)j.body + rr * j.pitch;
        U u;
        u.a = *(const uint4*)(p + (c0 < last ? c0 : last));
        u.b = *(const uint4*)(p + (c1 < last ? c1 : last));
        const int b = 4 * t + (lane >> 4), nb = j.n / 32;
        const uint32_t d = ((const uint16_t*)j.row)[rr * nb + (b < nb ? b : nb - 1)];
        u.d = b < nb ? d : 0u;
        return u;
    }
    static __device__ __forceinline__ void step(const U& u, const Lane& ln, const XStage& xs, int t, double (&acc)[4]) {
        const int slot = 16 * ((ln.g >> 1) == (ln.row >> 3) ? ln.row & 7 : XDIG);
        v4i x[2];
#pragma unroll
        for (int p = 0; p < 2; p++) x[p] = lds16(xs.dig + (XCHUNK * ln.g + slot) + 8 * XCHUNK * t + 4 * XCHUNK * p);
        const double e = xs.gexp[t >> 1];
        phase();
        uint32_t sc[2];
        to_slices(__builtin_bit_cast(uint32_t, uq_half((uint16_t)u.d)), sc);
        const uint32_t c0[4] = {u.a.x, u.a.y, u.a.z, u.a.w}, c1[4] = {u.b.x, u.b.y, u.b.z, u.b.w};
        const v4i z = {0, 0, 0, 0};
        const v4i d[2] = {mfma64(x[0], as_v4i(c0), z), mfma64(x[1], as_v4i(c1), z)};
#pragma unroll
        for (int p = 0; p < 2; p++) {
            const double s = (double)uq_bits_f(sc[p]) * e;
#pragma unroll
            for (int i = 0; i < 4; i++) acc[i] = __builtin_fma((double)d[p][i], s, acc[i]);
        }
    }
    static __device__ __forceinline__ int column(const Lane& ln, int t, int k) { return VPS * t + 64 * k + 16 * ln.g; }
    static __device__ __forceinline__ double chunk(const U& u, const Lane& ln, int k, uint32_t (&c)[4]) {
        uint32_t sc[2];
        to_slices(u.d, sc);
        c[0] = k ? u.b.x : u.a.x, c[1] = k ? u.b.y : u.a.y, c[2] = k ? u.b.z : u.a.z, c[3] = k ? u.b.w : u.a.w;
        return (double)uq_half((uint16_t)sc[k]);
    }
};

template <>
struct TK<KIND_IQ4_NL> {
    static constexpr int VPS = 128, CHUNKS = 2, NB = 1;
    struct U {
        uint4 a;
        uint32_t d;
    };
    static __device__ __forceinline__ U load(const FJob& j, int64_t tile, int t, int lane) {
        const int64_t rec = tile * ((j.n + VPS - 1) / VPS) + t;
        return {*(const uint4*)(j.body + rec * 1024 + (uint32_t)(16 * lane)),
                *(const uint16_t*)(j.lane + rec * 128 + (uint32_t)(2 * lane))};
    }
    static __device__ __forceinline__ void codes(const U& u, int half, uint32_t (&c)[4]) { book_codes16(IQ4_BOOK, u.a, half, c); }
    static __device__ __forceinline__ void step(const U& u, const Lane& ln, const XStage& xs, int t, double (&acc)[4]) {
        step_f16<TK>(u, ln, xs, t, acc);
    }
    static __device__ __forceinline__ int column(const Lane& ln, int t, int k) { return VPS * t + 32 * ln.g + 16 * k; }
    static __device__ __forceinline__ double chunk(const U& u, const Lane&, int k, uint32_t (&c)[4]) {
        codes(u, k, c);
        return (double)uq_half((uint16_t)u.d);
    }
};

// The 256-value kinds: their sub-scales are small integers, so a step's digit
// sums stay integers (|sum| < 2^27) and meet the double only once, with d.
__device__ __forceinline__ void add_step(const int (&ia)[4], double s, double (&acc)[4]) {
#pragma unroll
    for (int i = 0; i < 4; i++) acc[i] = __builtin_fma((double)ia[i], s, acc[i]);
}

// IQ4_XS, and IQ3_XXS with its grid and signs written out as codes of 4 bits (the
// grid has eight levels): 35% more bytes than the grid indices, but those took
// two dozen LDS lookups a step, and the lookups bounded the kernel (152000 x
// 2560: 53 us against 43).
template <uint32_t K>
struct BookKind {
    static constexpr int VPS = 256, CHUNKS = 4, NB = 1;
    struct U {
        uint4 a, b;  // blocks g and 4 + g of the superblock
        uint32_t sc;  // scales of blocks s, 2 + s, 4 + s, 6 + s (s = g >> 1)
        uint32_t d;
    };
    static constexpr Book book() { return K == KIND_IQ4_XS ? IQ4_BOOK : IQ3_BOOK; }
    static constexpr float unit() { return K == KIND_IQ4_XS ? 1.0f : 0.25f; }  // IQ3: d (0.5 + s) / 2 = d/4 (2 s + 1)
    static __device__ __forceinline__ U load(const FJob& j, int64_t tile, int t, int lane) {
        const int64_t rec = tile * (j.n / VPS) + t;
        const uint8_t* p = j.body + rec * 2048;
        const uint32_t o = 16 * lane;
        const uint8_t* r = j.row + rec * 160;
        return {*(const uint4*)(p + o), *(const uint4*)(p + o + 1024),
                *(const uint32_t*)(r + (uint32_t)(8 * (lane & 15) + 4 * (lane >> 5))),
                *(const uint16_t*)(r + 128 + (uint32_t)(2 * (lane & 15)))};
    }
    static __device__ __forceinline__ double scale_d(const U& u) { return (double)(uq_half((uint16_t)u.d) * unit()); }
    static __device__ __forceinline__ void step(const U& u, const Lane& ln, const XStage& xs, int t, double (&acc)[4]) {
        v4i x[2][2][2];
        read_blocks(ln, xs, t, x);
        const double e = xs.gexp[t];
        phase();
        v4i w[2][2];
#pragma unroll
        for (int b = 0; b < 2; b++)
#pragma unroll
            for (int h = 0; h < 2; h++) {
                uint32_t c[4];
                book_codes16(book(), b ? u.b : u.a, h, c);
                w[b][h] = as_v4i(c);
            }
        auto sc = [&](int k) { return (int)(int8_t)(uint8_t)(u.sc >> (8 * k)); };
        const int si[2][2] = {{sc(0), sc(1)}, {sc(2), sc(3)}};
        int ia[4];
        block_sums(x, w, si, ia);
        add_step(ia, scale_d(u) * e, acc);
    }
    static __device__ __forceinline__ int column(const Lane& ln, int t, int k) {
        return VPS * t + 128 * (k >> 1) + 32 * ln.g + 16 * (k & 1);
    }
    static __device__ __forceinline__ double chunk(const U& u, const Lane& ln, int k, uint32_t (&c)[4]) {
        const int b = k >> 1, sh = 4 * (k & 1);
        const uint4 w = {(b ? u.b.x : u.a.x) >> sh, (b ? u.b.y : u.a.y) >> sh, (b ? u.b.z : u.a.z) >> sh,
                         (b ? u.b.w : u.a.w) >> sh};
        book_codes16(book(), w, 0, c);
        // this lane's own block 4b + g: lane groups 2p, 2p + 1 stand for slices 0, 1 of pair p,
        // and the scales of slice s sit in lane groups 2s and 2s + 1
        const int own = 2 * b + (ln.g >> 1);
        const uint32_t other = (uint32_t)__shfl((int)u.sc, ln.row + 32 * (ln.g & 1), 64);
        return scale_d(u) * (double)(int8_t)(uint8_t)(other >> (8 * own));
    }
};
template <>
struct TK<KIND_IQ4_XS> : BookKind<KIND_IQ4_XS> {};
template <>
struct TK<KIND_IQ3_XXS> : BookKind<KIND_IQ3_XXS> {};

// Q6_K unit g = 2*sub + h of a superblock: ql[sub*64 + 16h ..], ql[sub*64 + 32 + 16h ..],
// qh[sub*32 + 16h ..] (16 bytes each) and the 4 group scales sc[sub*8 + h + 2k]: chunk k
// holds columns 128*sub + 16h + 32k.
template <>
struct TK<KIND_Q6_K> {
    static constexpr int VPS = 256, CHUNKS = 4, NB = 2;
    struct U {
        uint4 l0, l1, h;
        uint32_t sc, d;
    };
    static __device__ __forceinline__ U load(const FJob& j, int64_t tile, int t, int lane) {
        const int64_t rec = tile * (j.n / VPS) + t;
        const uint8_t* p = j.body + rec * 3072;
        const uint32_t o = 16 * lane;
        return {*(const uint4*)(p + o), *(const uint4*)(p + o + 1024), *(const uint4*)(p + o + 2048),
                *(const uint32_t*)(j.lane + rec * 256 + (uint32_t)(4 * lane)),
                *(const uint16_t*)(j.row + rec * 32 + (uint32_t)(2 * (lane & 15)))};
    }
    static __device__ __forceinline__ void codes(const U& u, int k, uint32_t (&c)[4]) {
        const uint4& l = (k & 1) ? u.l1 : u.l0;
        const uint32_t lv[4] = {l.x, l.y, l.z, l.w}, hv[4] = {u.h.x, u.h.y, u.h.z, u.h.w};
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const uint32_t lo = (k < 2 ? lv[q] : lv[q] >> 4) & 0x0F0F0F0Fu;
            const uint32_t hs = k < 2 ? hv[q] << (4 - 2 * k) : hv[q] >> (2 * k - 4);
            // code - 32 as a signed byte: + 0x60 carries out of no byte, then flip bit 7
            c[q] = (((hs & 0x30303030u) | lo) + 0x60606060u) ^ 0x80808080u;
        }
    }
    static __device__ __forceinline__ void step(const U& u, const Lane& ln, const XStage& xs, int t, double (&acc)[4]) {
        v4i x[4][2];
#pragma unroll
        for (int k = 0; k < 4; k++)
#pragma unroll
            for (int p = 0; p < 2; p++)
                x[k][p] = lds16(xs.dig + (XCHUNK * (8 * (ln.g >> 1) + (ln.g & 1)) + ln.slot[p]) + 16 * XCHUNK * t + 2 * XCHUNK * k);
        const double e = xs.gexp[t];
        phase();
        uint32_t sc[2];
        to_slices(u.sc, sc);
        const v4i z = {0, 0, 0, 0};
        int ia[4] = {0, 0, 0, 0};
#pragma unroll
        for (int q = 0; q < 4; q += 2) {
            v4i d[2][2];
#pragma unroll
            for (int k = 0; k < 2; k++) {
                uint32_t c[4];
                codes(u, q + k, c);
                const v4i w = as_v4i(c);
#pragma unroll
                for (int p = 0; p < 2; p++) d[k][p] = mfma64(x[q + k][p], w, z);
            }
#pragma unroll
            for (int k = 0; k < 2; k++)
#pragma unroll
                for (int p = 0; p < 2; p++) {
                    const int s = (int)(int8_t)(uint8_t)(sc[p] >> (8 * (q + k)));
#pragma unroll
                    for (int i = 0; i < 4; i++) ia[i] += __mul24(s, d[k][p][i]);
                }
        }
        add_step(ia, (double)uq_half((uint16_t)u.d) * e, acc);
    }
    static __device__ __forceinline__ int column(const Lane& ln, int t, int k) {
        return VPS * t + 128 * (ln.g >> 1) + 16 * (ln.g & 1) + 32 * k;
    }
    static __device__ __forceinline__ double chunk(const U& u, const Lane&, int k, uint32_t (&c)[4]) {
        // (as codes(), for a k that is not known when compiling)
        const uint32_t lv[4] = {u.l0.x, u.l0.y, u.l0.z, u.l0.w}, lw[4] = {u.l1.x, u.l1.y, u.l1.z, u.l1.w};
        const uint32_t hv[4] = {u.h.x, u.h.y, u.h.z, u.h.w};
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const uint32_t lo = (((k & 1) ? lw[q] : lv[q]) >> (4 * (k >> 1))) & 0x0F0F0F0Fu;
            c[q] = ((((hv[q] >> (2 * k)) & 0x03030303u) << 4 | lo) + 0x60606060u) ^ 0x80808080u;
        }
        return (double)uq_half((uint16_t)u.d) * (double)(int8_t)(uint8_t)(u.sc >> (8 * k));
    }
};

// Products of step t that run in double, this lane's chunks of its row: those of
// x's far values, or (ALL) every one.
template <class T, bool ALL>
__device__ __forceinline__ double step_double(const typename T::U& u, const Lane& ln, const XStage& xs, int t) {
    double r = 0.0;
#pragma unroll 1
    for (int k = 0; k < T::CHUNKS; k++) {
        const int col = T::column(ln, t, k);
        uint32_t take = col < xs.n ? 15u : 0u;
        if (!ALL) take &= (uint32_t)(xs.far[t * T::VPS / XGROUP] >> ((col & (XGROUP - 1)) >> 2));
        if (__builtin_amdgcn_ballot_w64(take != 0) == 0) continue;
        uint32_t c[4];
        const double s = T::chunk(u, ln, k, c);
        if (take) {
            // ALL: weight by weight, as the products of an infinite scale have signs
            // of their own, which the sum of a chunk would hide
            double d[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const float4 x4 = *(const float4*)(xs.xg + col + 4 * q);
                const float xv[4] = {x4.x, x4.y, x4.z, x4.w};
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const double code = (double)(int)(int8_t)(uint8_t)(c[q] >> (8 * i));
                    d[i] = ALL ? __builtin_fma(s * code, (double)xv[i], d[i])
                               : __builtin_fma(code, (take >> q) & 1 ? (double)xv[i] : 0.0, d[i]);
                }
            }
            const double sum = (d[0] + d[1]) + (d[2] + d[3]);
            r = ALL ? r + sum : __builtin_fma(s, sum, r);
        }
    }
    return r;
}

// All products of a tile in double.
template <class T>
__device__ double tile_double(const FJob& j, int64_t tile, int S, const Lane& ln, const XStage& xs) {
    double r = 0.0;
#pragma unroll 1
    for (int t = 0; t < S; t++) r += step_double<T, true>(T::load(j, tile, t, ln.lane), ln, xs, t);
    return r;
}

// A tile's S steps fall into ns = min(8, S) column segments, which the eight
// waves of a workgroup share out: with ns = 8 wave w takes segment (w + i) mod 8
// of the workgroup's i-th tile, so that segments of unequal length even out,
// with fewer every eighth segment of all its tiles. The segments' sums meet in
// LDS, `dep` tiles at a time, and add up as a binary tree: a row's bits do not
// depend on the launch, the number of its workgroups or the other jobs.
constexpr int FL_SEGS = FL_WG / 64;

// A wave's place: step s of segment seg (which ends at `end`) of tile i.
struct Place {
    int S, ns, inv;  // inv: x / ns = x * inv >> 8 for x < 16
    int i, seg, s, end;
    __device__ __forceinline__ void enter() {
        s = ns == FL_SEGS ? seg * S >> 3 : seg;
        end = ns == FL_SEGS ? (seg + 1) * S >> 3 : seg + 1;
    }
    __device__ __forceinline__ Place(int wave, int steps) {
        S = steps;
        ns = S < FL_SEGS ? S : FL_SEGS;
        inv = 256 / ns + 1;
        i = wave * inv >> 8;
        seg = wave - i * ns;
        enter();
    }
    __device__ __forceinline__ void next() {
        if (ns == FL_SEGS) {
            i++;
            seg = (seg + 1) & (FL_SEGS - 1);
        } else {
            const int q = (seg + FL_SEGS) * inv >> 8;
            i += q;
            seg += FL_SEGS - q * ns;
        }
        enter();
    }
};

// Tiles wgi, wgi + wgs, ... of one job. `stage` (the staging of x with its
// barrier) runs once the wave's first loads are out. part: 2 x dep x FL_SEGS x
// 64 doubles.
template <class T, int NB, class F>
__device__ __forceinline__ void job_tiles(const FJob& j, int wgi, int dep, double* part, F&& stage) {
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int S = (j.n + T::VPS - 1) / T::VPS, ns = S < FL_SEGS ? S : FL_SEGS;
    const int tiles = (int)((j.m + 15) >> 4);
    const int count = (tiles - wgi + j.wgs - 1) / j.wgs;  // this workgroup's tiles
    const Lane ln;
    const double half = (ln.g & 1) ? 4294967296.0 : 1.0;  // digits 4..7 stand 2^32 higher
    // A fetch past the wave's last step reads one address in every lane instead
    // of being branched around: with the same loads on every path the
    // compiler's waits stay exact (a branch made them wait for every load).
    typename T::U buf[NB];
    Place f(wave, S);
    auto fetch = [&](typename T::U& b) {
        const bool on = f.i < count;
        b = T::load(j, on ? wgi + f.i * j.wgs : 0, on ? f.s : 0, on ? ln.lane : 0);
        if (++f.s >= f.end) f.next();
    };
#pragma unroll
    for (int b = 0; b < NB; b++) fetch(buf[b]);
    const XStage xs = stage();
    // Tiles [from, to) of the workgroup: one wave sums a tile's segments, then
    // its four lane groups. A zero digit times an infinite scale is NaN where the
    // row's own products are not: rows that are not finite, and only they, are
    // summed again wholly in double at the end, and NaN until then.
    bool again = false;
    auto sum_tiles = [&](int from, int to, int buffer) {
        __syncthreads();
        for (int i = from + wave; i < to; i += FL_SEGS) {
            double v[FL_SEGS];
#pragma unroll
            for (int k = 0; k < FL_SEGS; k++) {
                const double t = part[((buffer * dep + (i - from)) * FL_SEGS + k) * 64 + ln.lane];
                v[k] = k < ns ? t : 0.0;
            }
            const double top = ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
            const int64_t tile = wgi + (int64_t)i * j.wgs, row = 16 * tile + ln.row;
            const double sum = uq_swap32_sum(uq_swap16_sum(top));
            const bool finite = __builtin_fabs(sum) < __builtin_inf();
            again = again || !finite;
            if (ln.g == 0 && row < j.m) j.y[row] = finite ? (float)sum : __builtin_nanf("");
        }
    };
    auto combine = [&](const double (&acc)[4]) {
        double t = __builtin_fma(acc[3], 256.0, acc[2]);
        t = __builtin_fma(t, 256.0, acc[1]);
        return __builtin_fma(t, 256.0, acc[0]) * half;
    };
    Place p(wave, S);
    // (expected, so that the double branches lie behind the code that runs: a call of
    // a few microseconds is some 1% longer where it fetches instructions across them,
    // IQ4_XS 3001 x 2560 4.85 us for 4.79)
    if (__builtin_expect(xs.wide == 0, 1)) {
        double acc[4] = {0.0, 0.0, 0.0, 0.0};
        int base = 0, buffer = 0;
        // once the wave is past them, the workgroup sums the tiles from `base` on
        auto flush = [&]() {
            const int to = base + dep < count ? base + dep : count;
            sum_tiles(base, to, buffer);
            base = to;
            buffer ^= 1;
        };
        auto catch_up = [&]() {
#pragma unroll 1
            while (p.i >= base + dep && p.i < count) flush();
        };
        catch_up();
        while (p.i < count) {
#pragma unroll
            for (int b = 0; b < NB; b++) {
                // (a step past the last is skipped, its fetch is not: a loop left
                // from the middle would cost the waits their counts as well)
                const bool on = p.i < count;
                if (on) T::step(buf[b], ln, xs, p.s, acc);
                fetch(buf[b]);
                if (on && ++p.s == p.end) {
                    part[((buffer * dep + (p.i - base)) * FL_SEGS + p.seg) * 64 + ln.lane] = combine(acc);
#pragma unroll
                    for (int i = 0; i < 4; i++) acc[i] = 0.0;
                    p.next();
                    catch_up();
                }
            }
        }
#pragma unroll 1
        while (base < count) flush();
    } else {
        // x has far values: without the ring, as the loads of x would cost it the
        // exact waits. Each wave sums its own steps' products with them, chunks
        // without one left out. 49344 x 2560 with one such value in x / one in
        // each group, against one wave summing all products of a group with one:
        // Q8_0 65.6 -> 30.6 us / 254 -> 41.7, IQ3_XXS 43.6 -> 21.6 / 214 -> 33.3.
        // Where x is full of them it costs more: with one value in twenty / in two
        // Q8_0 82 / 82 us, Q6_K 68 / 68, IQ4_XS 54 / 56 (65 / 75, 60 / 54 and 64 / 73
        // with 32-value blocks of a range over 2^14 in double).
        int base = 0, buffer = 0;
        auto flush = [&]() {
            const int to = base + dep < count ? base + dep : count;
            sum_tiles(base, to, buffer);
            base = to;
            buffer ^= 1;
        };
#pragma unroll 1
        while (p.i < count) {
            if (p.i >= base + dep) {
                flush();
                continue;
            }
            double acc[4] = {0.0, 0.0, 0.0, 0.0}, more = 0.0;
#pragma unroll 1
            for (; p.s < p.end; p.s++) {
                const typename T::U u = T::load(j, wgi + p.i * j.wgs, p.s, ln.lane);
                if ((xs.wide >> (p.s * T::VPS / XGROUP)) & 1) more += step_double<T, false>(u, ln, xs, p.s);
                T::step(u, ln, xs, p.s, acc);
            }
            part[((buffer * dep + (p.i - base)) * FL_SEGS + p.seg) * 64 + ln.lane] = combine(acc) + more;
            p.next();
        }
#pragma unroll 1
        while (base < count) flush();
    }
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(again) == 0, 1)) return;
#pragma unroll 1
    for (int i = 0; i < count; i++) {
        if (((i % dep) & (FL_SEGS - 1)) != wave) continue;
        const int64_t tile = wgi + (int64_t)i * j.wgs, row = 16 * tile + ln.row;
        const bool redo = ln.g == 0 && row < j.m && j.y[row] != j.y[row];  // the lane's own stores
        if (__builtin_amdgcn_ballot_w64(redo) == 0) continue;
        const double sum = uq_swap32_sum(uq_swap16_sum(tile_double<T>(j, tile, S, ln, xs)));
        if (redo) j.y[row] = (float)sum;
    }
}

// ---- F32 / BF16 rows
// A lane owns units u = sub, sub + LPR, ... of a row; dot() returns the unit's
// products with x in double.
template <uint32_t K>
struct FK;

template <>
struct FK<KIND_F32> {
    static constexpr int WPU = 8, LPR = 64, CH = 4;
    struct U {
        uint4 a, b;
    };
    static __device__ U load(const FJob& j, int64_t row, int u) {
        const uint4* p = (const uint4*)(j.body + row * j.pitch) + 2 * u;
        return {p[0], p[1]};
    }
    static __device__ double dot(const U& v, const XStage& xs, int u) {
        const float* x = xs.xf + 8 * u;
        const float4 xa = ((const float4*)x)[0], xb = ((const float4*)x)[1];
        const float xv[8] = {xa.x, xa.y, xa.z, xa.w, xb.x, xb.y, xb.z, xb.w};
        const uint32_t w[8] = {v.a.x, v.a.y, v.a.z, v.a.w, v.b.x, v.b.y, v.b.z, v.b.w};
        double s[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int k = 0; k < 8; k++) s[k & 3] = __builtin_fma((double)uq_bits_f(w[k]), (double)xv[k], s[k & 3]);
        return (s[0] + s[1]) + (s[2] + s[3]);
    }
};

template <>
struct FK<KIND_BF16> {
    static constexpr int WPU = 8, LPR = 64, CH = 4;
    struct U {
        uint4 a;
    };
    static __device__ U load(const FJob& j, int64_t row, int u) {
        return {((const uint4*)(j.body + row * j.pitch))[u]};
    }
    static __device__ double dot(const U& v, const XStage& xs, int u) {
        const float* x = xs.xf + 8 * u;
        const float4 xa = ((const float4*)x)[0], xb = ((const float4*)x)[1];
        const float xv[8] = {xa.x, xa.y, xa.z, xa.w, xb.x, xb.y, xb.z, xb.w};
        const uint32_t w[4] = {v.a.x, v.a.y, v.a.z, v.a.w};
        double s[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int k = 0; k < 4; k++) {
            s[k] = __builtin_fma((double)uq_bits_f(w[k] << 16), (double)xv[2 * k], s[k]);
            s[k] = __builtin_fma((double)uq_bits_f(w[k] & 0xFFFF0000u), (double)xv[2 * k + 1], s[k]);
        }
        return (s[0] + s[1]) + (s[2] + s[3]);
    }
};

// Rows of one job for workgroup `wgi` of `wgc`: LPR lanes per row, 64/LPR
// rows per wave, row blocks wgi, wgi + wgc, ... A lane owns units u = sub +
// LPR*i of its row and walks them in chunks of CH units: the next chunk's
// loads (the same row's or the next row block's) are issued before the
// current chunk's dots. Per row the lane adds its units in order; the lane
// group sums in double and rounds once.
template <class T>
__device__ void job_rows(const FJob& j, int wgi, int wgc, const XStage& xs) {
    constexpr int LPR = T::LPR, CH = T::CH, RPW = 64 / LPR;
    const int RPB = RPW * (int)(blockDim.x / 64);  // rows per row block: the launch picks 256 or 512 threads
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, sub = lane % LPR, grp = lane / LPR;
    const int nu = j.n / T::WPU;
    const int nb = (nu + LPR - 1) / LPR;    // unit slots per lane and row
    const int nch = (nb + CH - 1) / CH;      // chunks per row
    const int64_t rblocks = (j.m + RPB - 1) / RPB;
    if (wgi >= rblocks) return;
    typename T::U buf[2][CH];
    // (row block, chunk) of the next fetch, advanced without division
    int64_t frb = wgi;
    int fc = 0;
    auto fetch = [&](typename T::U (&b)[CH]) {
        const int64_t row = frb * RPB + wave * RPW + grp;
        const int64_t rr = row < j.m ? row : j.m - 1;
#pragma unroll
        for (int k = 0; k < CH; k++) {
            const int u = sub + LPR * (fc * CH + k);
            if (fc * CH + k < nb) b[k] = T::load(j, rr, u < nu ? u : nu - 1);  // slot test is wave-uniform
        }
        if (++fc == nch) {
            fc = 0;
            frb += wgc;
        }
    };
    fetch(buf[0]);
    int64_t rb = wgi;
    int c = 0;
    double acc = 0.0;
    while (rb < rblocks) {
        // two chunks per trip so the chunk buffers keep fixed registers
#pragma unroll
        for (int h = 0; h < 2; h++) {
            if (rb < rblocks) {
                if (frb < rblocks) fetch(buf[h ^ 1]);
#pragma unroll
                for (int k = 0; k < CH; k++) {
                    const int u = sub + LPR * (c * CH + k);
                    if (c * CH + k < nb) {
                        const double d = T::dot(buf[h][k], xs, u < nu ? u : nu - 1);
                        acc = acc + (u < nu ? d : 0.0);
                    }
                }
                if (++c == nch) {
                    const int64_t row = rb * RPB + wave * RPW + grp;
                    const double sum = uq_group_sum<LPR>(acc);
                    if (row < j.m && sub == 0) j.y[row] = (float)sum;
                    acc = 0.0;
                    c = 0;
                    rb += wgc;
                }
            }
        }
    }
}

// Up to MAX_JOBS jobs per launch, passed by value in the kernel arguments
// (no device table to copy before the launch); longer tables take several
// launches, each row computed the same way.
constexpr int MAX_JOBS = 32;
struct Parts {
    int32_t dep, at;  // tiles whose segments meet at once; their place in LDS
};
struct JobArgs {
    Parts parts;
    int32_t start[MAX_JOBS];  // first workgroup of each job, ascending; past the last job INT32_MAX
    FJob job[MAX_JOBS];
};

// The workgroup's job and its place in it (-1: none). The arguments lie in host
// memory and the first read of each line takes about a microsecond, so the
// workgroup reads as few as it can one behind the other: with a grid row per job
// the job's record alone, otherwise all starts at once (a binary search over the
// jobs was five such reads).
__device__ __forceinline__ FJob find_job(const JobArgs& a, int* wgi) {
    int job = (int)blockIdx.y;
    if (gridDim.y == 1) {
        const int32_t s = a.start[threadIdx.x & (MAX_JOBS - 1)];
        job = __popc((uint32_t)__builtin_amdgcn_ballot_w64(s <= (int32_t)blockIdx.x)) - 1;
    }
    const FJob j = a.job[job];
    *wgi = gridDim.y == 1 ? (int)blockIdx.x - j.wg0 : ((int)blockIdx.x < j.wgs ? (int)blockIdx.x : -1);
    return j;
}
// Dynamic LDS of a job: the digits of x padded to whole groups, the group
// factors and the groups' far values (F32 / BF16 weights: x as f32).
__device__ __forceinline__ XStage stage_floats(const FJob& j, uint8_t* lds) {
    XStage xs{};
    xs.xf = (const float*)lds;
    xs.n = j.n;
    for (int i = threadIdx.x; i < j.n / 4; i += (int)blockDim.x) ((float4*)lds)[i] = ((const float4*)j.x)[i];
    __syncthreads();
    return xs;
}
__device__ __forceinline__ XStage stage_digits(const FJob& j, const float4 (&ahead)[XAHEAD], uint8_t* lds, uint64_t* wides) {
    const int ng = (j.n + XGROUP - 1) / XGROUP;
    uint8_t* const dig = lds;
    double* const gexp = (double*)(lds + XCHUNK * (XGROUP / 16) * ng);
    uint64_t* const far = (uint64_t*)(gexp + ng);
    const uint64_t wide = stage_x(j.x, j.n, ahead, dig, gexp, far);
    if ((threadIdx.x & 63) == 0) wides[threadIdx.x >> 6] = wide;
    __syncthreads();
    XStage xs{};
    xs.dig = dig;
    xs.gexp = gexp;
    xs.far = far;
    xs.xg = j.x;
    xs.n = j.n;
    uint64_t all = 0;
    for (int w = 0; w < (int)blockDim.x / 64; w++) all |= wides[w];
    // the same in every lane: a scalar mask
    xs.wide = (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)all) |
              (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(all >> 32)) << 32;
    return xs;
}
template <uint32_t K, int NB = 0>
__device__ __forceinline__ void run_job(const FJob& j, int wgi, const Parts& parts, uint8_t* lds, uint64_t* wides) {
    if constexpr (row_kind(K)) {
        const XStage xs = stage_floats(j, lds);
        job_rows<FK<K>>(j, wgi, j.wgs, xs);
    } else {
        float4 ahead[XAHEAD];
        load_ahead(j.x, j.n, ahead);
        job_tiles<TK<K>, NB ? NB : TK<K>::NB>(j, wgi, parts.dep, (double*)(lds + parts.at), [&]() { return stage_digits(j, ahead, lds, wides); });
    }
}

// One job, its record in the first lines of the arguments. Four waves per SIMD,
// two workgroups of a CU at work, for the tiled kinds. The row kinds use fewer
// registers by themselves, but under the same bound the compiler scheduled F32 with
// more waits for all loads in flight, and 100000 x 256 took 34.6 us for 30.5.
struct OneJob {
    Parts parts;
    FJob job;
};
template <uint32_t K, int NB = 0>
__global__ __launch_bounds__(FL_WG, row_kind(K) ? 1 : 4) void k_flinear_one(OneJob a) {
    extern __shared__ __attribute__((aligned(16))) uint8_t fl_lds[];
    __shared__ uint64_t wides[FL_SEGS];
    run_job<K, NB>(a.job, (int)blockIdx.x, a.parts, fl_lds, wides);
}

// A job table of F32 or BF16 weights: registers sized for that kind alone.
template <uint32_t K>
__global__ __launch_bounds__(FL_WG) void k_flinear_rows(JobArgs a) {
    extern __shared__ __attribute__((aligned(16))) uint8_t fl_lds[];
    int wgi;
    const FJob j = find_job(a, &wgi);
    if (wgi >= 0) run_job<K>(j, wgi, a.parts, fl_lds, nullptr);
}

// One launch over a job table of any kinds.
__global__ __launch_bounds__(FL_WG, 4) void k_flinear(JobArgs a) {
    extern __shared__ __attribute__((aligned(16))) uint8_t fl_lds[];
    __shared__ uint64_t wides[FL_SEGS];
    int wgi;
    const FJob j = find_job(a, &wgi);
    if (wgi < 0) return;
    switch (j.kind) {
    case KIND_F32: run_job<KIND_F32>(j, wgi, a.parts, fl_lds, wides); break;
    case KIND_BF16: run_job<KIND_BF16>(j, wgi, a.parts, fl_lds, wides); break;
    case KIND_Q8_0: run_job<KIND_Q8_0>(j, wgi, a.parts, fl_lds, wides); break;
    case KIND_IQ4_NL: run_job<KIND_IQ4_NL>(j, wgi, a.parts, fl_lds, wides); break;
    case KIND_IQ4_XS: run_job<KIND_IQ4_XS>(j, wgi, a.parts, fl_lds, wides); break;
    case KIND_Q6_K: run_job<KIND_Q6_K>(j, wgi, a.parts, fl_lds, wides); break;
    case KIND_IQ3_XXS: run_job<KIND_IQ3_XXS>(j, wgi, a.parts, fl_lds, wides); break;
    default: break;
    }
}

using OneKernel = void (*)(OneJob);
using TableKernel = void (*)(JobArgs);
// `few`: no wave has more than two steps.
OneKernel one_kernel(int32_t kind, bool few) {
    switch (kind) {
    case KIND_F32: return k_flinear_one<KIND_F32>;
    case KIND_BF16: return k_flinear_one<KIND_BF16>;
    case KIND_Q8_0: return few ? k_flinear_one<KIND_Q8_0, 1> : k_flinear_one<KIND_Q8_0>;
    case KIND_IQ4_NL: return k_flinear_one<KIND_IQ4_NL>;
    case KIND_IQ4_XS: return k_flinear_one<KIND_IQ4_XS>;
    case KIND_Q6_K: return few ? k_flinear_one<KIND_Q6_K, 1> : k_flinear_one<KIND_Q6_K>;
    }
    return k_flinear_one<KIND_IQ3_XXS>;
}
TableKernel table_kernel(const JobArgs& a, int count) {
    const int32_t k = a.job[0].kind;
    for (int i = 1; i < count; i++)
        if (a.job[i].kind != k) return k_flinear;
    return k == KIND_F32 ? k_flinear_rows<KIND_F32> : (k == KIND_BF16 ? k_flinear_rows<KIND_BF16> : k_flinear);
}

// Workgroups of an F32 / BF16 kernel resident per CU at `lds` dynamic bytes
// (occupancy query, cached per kernel and size).
int fl_resident(const void* kern, size_t lds) {
    struct Entry {
        const void* k;
        size_t lds;
        int n;
    };
    static Entry cache[64];
    static int used = 0;
    for (int i = 0; i < used; i++)
        if (cache[i].k == kern && cache[i].lds == lds) return cache[i].n;
    int n = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kern, FL_WG, lds) != hipSuccess || n <= 0) n = 1;
    if (n > 8) n = 8;
    if (used < 64) cache[used++] = Entry{kern, lds, n};
    return n;
}

size_t stage_bytes(uint32_t kind, int n) {
    if (kind == KIND_F32 || kind == KIND_BF16) return 4 * (size_t)n;
    const size_t ng = ((size_t)n + XGROUP - 1) / XGROUP;
    return (XCHUNK * (XGROUP / 16) + 8 + 8) * ng;
}

// Tiles whose segments meet at once: 32 KB of LDS, one where x takes more than
// 64 KB (n > 7168), so that the largest x (148 KB) still fits.
constexpr int FL_DEP = 4;
Parts plan_parts(size_t stage, size_t* lds) {
    const int at = (int)((stage + 15) & ~(size_t)15), dep = at <= 64 * 1024 ? FL_DEP : 1;
    *lds = (size_t)at + 2 * 8 * 64 * FL_SEGS * (size_t)dep;
    return {dep, at};
}

// Workgroups of a single weight of a tiled kind: one or two a CU (a third never
// paid). MI355X, HIP events, weights that rotate past the caches, us:
//  * Where LDS holds one (n > 5376) the second only waits: 32000 x 7168 with
//    256 / 512 workgroups Q8_0 46.4 / 49.9, Q6_K 35.4 / 38.1, IQ4_XS 32.4 / 35.1.
//  * The IQ kinds are bound by the VALU and need four waves per SIMD once there
//    are tiles enough: 13000 x 2560 (3.2 tiles a CU) IQ4_XS 7.3 / 7.9, 20000 9.2 /
//    8.7, 49344 20.1 / 16.2, 151936 52.8 / 40.4; 100000 x 256 8.7 / 7.1, 70000 7.0 /
//    6.9; 13000 x 4096 IQ4_NL 12.3 / 11.5.
//  * Q8_0 reads at the memory's rate with two waves per SIMD and two steps in
//    flight: 100000 x 2560 52.8 / 54.0, 151936 77.2 / 79.3, 40000 x 4096 33.8 /
//    35.3. Short rows leave a wave one step or two per tile: 151936 x 2048 65.5 /
//    63.5, 100000 x 1024 25.6 / 21.5, 18000 x 1536 (4.4 tiles a CU) 8.6 / 9.1.
//  * Q6_K is between: 100000 x 2560 36.9 / 38.6, 128256 x 3072 55.5 / 52.9, 100000 x
//    3072 45.4 / 46.9, x 1024 17.2 / 17.1, x 256 9.0 / 7.7, 49344 x 4096 30.0 / 28.6.
// All CUs get one where there are many tiles: 49344 rows as 238 workgroups of 13
// tiles / 256 of 12 or 13, Q8_0 29.8 / 29.0. With few tiles, and Q6_K always,
// whole shares cost less: 13000 x 7168 as 204 of 4 / 256 of 3 or 4, Q6_K 18.0 / 19.5,
// Q8_0 25.1 / 25.5.
int64_t single_wgs(uint32_t kind, int64_t n, int64_t tiles, size_t lds, int64_t cu) {
    const bool q8 = kind == KIND_Q8_0, q6 = kind == KIND_Q6_K;
    const bool fits = 2 * lds <= 160 * 1024;
    const int64_t from = n >= 4096 ? (q6 ? 7 : 3) : (n >= 1024 ? (q8 ? 5 : 4) : 3 + 1536 / n);  // tiles a CU
    const bool two = fits && tiles > from * cu && (q8 ? n < 2560 : (q6 ? n < 1024 || n >= 4096 : true));
    if (two) return std::min(tiles, 2 * cu);
    const int64_t nt = (tiles + cu - 1) / cu;
    return q6 || nt < 8 ? (tiles + nt - 1) / nt : cu;
}

// Instructions of a wave for 16 rows per column, and of the staging per column,
// in proportion to each other: the table planner's weights. Counted, not fitted;
// what they choose was held against 1 to 20 tiles a workgroup: 22 IQ3_XXS 640 x
// 2560 beside an F32 router 8.44 us (4 tiles; best 8.41), eight IQ4_XS 2560 x 2560
// 9.93 (9.90), a Q8_0 q|k|v 7.61 (7.61). Tables of very unequal row lengths are
// not at their best: 2560 x 16384 with six of 2560 x 512 (Q6_K) 39.2 (21.0 with 2).
constexpr double STAGE_COST = 0.55;
double step_cost(uint32_t kind) {
    switch (kind) {
    case KIND_Q8_0: return 0.5;
    case KIND_IQ4_NL: return 1.1;
    }
    return 0.9;
}

bool linear_kind(uint32_t kind) {
    switch (kind) {
    case KIND_F32:
    case KIND_BF16:
    case KIND_Q8_0:
    case KIND_IQ4_NL:
    case KIND_IQ4_XS:
    case KIND_Q6_K:
    case KIND_IQ3_XXS: return true;
    }
    return false;
}

}  // namespace

// Device layout of an uploaded frontier kind (the Q8_0 split is the matvec's:
// int8 plane + fp16 plane). Returns false for kinds without one.
bool frontier_layout(uint32_t kind, FrontierLayout& L) {
    L = FrontierLayout{};
    switch (kind) {
    case KIND_F32: L = {4, 16, 0, {}}; return true;
    case KIND_BF16: L = {8, 16, 0, {}}; return true;
    // lane group g: block 4t + g of step t, its scale in the lane plane
    case KIND_IQ4_NL: L = {32, 18, 128, {1024, 128, 0}}; return true;
    // lane group g: blocks g and 4 + g; row plane: 8 scale bytes of 16 rows, their d
    case KIND_IQ4_XS: L = {256, 136, 256, {2048, 0, 160}}; return true;
    case KIND_IQ3_XXS: L = {256, 98, 256, {2048, 0, 160}}; return true;
    // lane group g = 2*sub + h: its three 16-byte pieces and, in the lane plane, four scales
    case KIND_Q6_K: L = {256, 210, 256, {3072, 256, 32}}; return true;
    }
    return false;
}

size_t frontier_plane_bytes(const FrontierLayout& L, int plane, int64_t n, int64_t m) {
    if (!L.step_vals) return plane == FL_BODY ? (size_t)(n / L.block_vals * m) * L.block_bytes : 0;
    return (size_t)((m + 15) / 16) * ((n + L.step_vals - 1) / L.step_vals) * L.rec[plane];
}

static int grid_blocks(int64_t total) {
    const int64_t g = (total + FWG - 1) / FWG;
    return (int)std::min<int64_t>(std::max<int64_t>(g, 1), 65536);
}

void launch_layout(uint32_t kind, const uint8_t* src, int64_t n, int64_t m, const FrontierLayout& L,
                   uint8_t* const planes[3], unsigned* bad, hipStream_t s) {
    const int64_t total = n / L.block_vals * m * L.block_bytes;
    if (!L.step_vals) {
        (void)hipMemcpyAsync(planes[FL_BODY], src, (size_t)total, hipMemcpyDeviceToDevice, s);
        hipLaunchKernelGGL(k_copy_verify, dim3(grid_blocks(total / 16)), dim3(FWG), 0, s, (const uint4*)src,
                           (const uint4*)planes[FL_BODY], total / 16, bad);
        return;
    }
    LayoutArgs a{};
    a.m = m;
    a.kind = (int32_t)kind;
    a.block_bytes = L.block_bytes;
    a.blocks = (int32_t)(n / L.block_vals);
    a.steps = (int32_t)((n + L.step_vals - 1) / L.step_vals);
    a.bps = L.step_vals / L.block_vals;
    for (int i = 0; i < 3; i++) {
        a.rec[i] = L.rec[i];
        a.plane[i] = planes[i];
        a.dwords[i] = (int64_t)frontier_plane_bytes(L, i, n, m) / 4;
    }
    const int64_t dwords = a.dwords[0] + a.dwords[1] + a.dwords[2];
    hipLaunchKernelGGL(k_layout_repack, dim3(grid_blocks(dwords)), dim3(FWG), 0, s, src, a, dwords);
    if (kind == KIND_IQ3_XXS) {
        const int64_t subs = m * a.blocks * 8;
        hipLaunchKernelGGL(k_iq3_verify, dim3(grid_blocks(subs)), dim3(FWG), 0, s, src, a, subs, bad);
        return;
    }
    hipLaunchKernelGGL(k_layout_verify, dim3(grid_blocks(total)), dim3(FWG), 0, s, src, a, total, bad);
}

}  // namespace uq

using namespace uq;

namespace {

FJob make_job(const Weight& w, const float* x, float* y) {
    FJob j{};
    j.body = (const uint8_t*)w.qs;
    j.lane = w.sc;
    j.row = (const uint8_t*)w.d;
    j.x = x;
    j.y = y;
    j.m = w.m;
    j.kind = (int32_t)w.kind;
    j.n = (int32_t)w.n;
    switch (w.kind) {
    case KIND_F32: j.pitch = 4 * w.n; break;
    case KIND_BF16: j.pitch = 2 * w.n; break;
    case KIND_Q8_0: j.pitch = w.n; break;
    }
    return j;
}

int check_job_weight(const uq_weight_t w) {
    if (!w) return set_error(ERR_ARG, "linear: null weight");
    if (!linear_kind(w->w.kind))
        return set_error(ERR_QUANT_TYPE, "linear: the fp32-activation reader takes F32, BF16, Q8_0, Q6_K, IQ3_XXS, "
                                         "IQ4_NL or IQ4_XS weights (frontier_core.rs:53-58)");
    return OK;
}

int enqueue_jobs(const uq_linear_job* jobs, int count, hipStream_t s) {
    if (!jobs || count <= 0) return set_error(ERR_ARG, "linear: empty job table");
    for (int i = 0; i < count; i++) {
        if (int rc = check_job_weight(jobs[i].weight)) return rc;
        if (!jobs[i].x || !jobs[i].y) return set_error(ERR_ARG, "linear: null x or y");
        if ((uintptr_t)jobs[i].x & 15) return set_error(ERR_ARG, "linear: x must be 16-byte aligned");
    }
    for (int c0 = 0; c0 < count; c0 += MAX_JOBS) {
        JobArgs a;
        const int jobs_here = std::min(MAX_JOBS, count - c0);
        size_t lds = 0;
        bool rows_only = true;
        for (int i = 0; i < jobs_here; i++) {
            const Weight& w = jobs[c0 + i].weight->w;
            a.job[i] = make_job(w, jobs[c0 + i].x, jobs[c0 + i].y);
            lds = std::max(lds, stage_bytes(w.kind, (int)w.n));
            rows_only = rows_only && row_kind(w.kind);
        }
        const bool one = jobs_here == 1;
        const int64_t cu = cu_count();
        int64_t wg = 0;
        int threads = FL_WG;
        bool few = false;
        if (!rows_only) {
            a.parts = plan_parts(lds, &lds);
            int64_t tiles = 0;
            for (int i = 0; i < jobs_here; i++)
                if (!row_kind((uint32_t)a.job[i].kind)) tiles += (a.job[i].m + 15) / 16;
            // Tiles per workgroup. Of a table: from those that make one to four
            // workgroups a CU the fewest instructions that a CU runs one behind the
            // other, the staging of x in every workgroup among them. One workgroup a
            // CU (two waves per SIMD) leaves some of its time idle.
            const int64_t alone = one ? single_wgs((uint32_t)a.job[0].kind, a.job[0].n, tiles, lds, cu) : 0;
            int64_t best = one ? (tiles + alone - 1) / alone : 0;
            double least = 0.0;
            for (int c = 0; c < 8 && !one; c++) {
                const int64_t nt = (tiles + (c / 2 + 1) * cu - 1) / ((c / 2 + 1) * cu) + (c & 1);
                int64_t wgs = 0;
                double work = 0.0;
                for (int i = 0; i < jobs_here; i++) {
                    const FJob& j = a.job[i];
                    const int64_t w = row_kind((uint32_t)j.kind) ? (j.m + 7) / 8 : ((j.m + 15) / 16 + nt - 1) / nt;
                    wgs += w;
                    work += (double)w * ((double)nt * step_cost((uint32_t)j.kind) + STAGE_COST) * j.n;
                }
                const int64_t per_cu = (wgs + cu - 1) / cu;
                const double cost = work / (double)wgs * (double)per_cu * (per_cu == 1 ? 1.1 : 1.0);
                if (!best || cost < least) {
                    best = nt;
                    least = cost;
                }
            }
            const int64_t step_vals = a.job[0].kind == KIND_Q8_0 || a.job[0].kind == KIND_IQ4_NL ? 128 : 256;
            few = best * ((a.job[0].n + step_vals - 1) / step_vals) <= 2 * FL_SEGS;
            for (int i = 0; i < jobs_here; i++) {
                FJob& j = a.job[i];
                j.wg0 = (int32_t)wg;
                j.wgs = (int32_t)(one ? alone : (row_kind((uint32_t)j.kind) ? std::min<int64_t>((j.m + 7) / 8, 4 * cu)
                                                                            : ((j.m + 15) / 16 + best - 1) / best));
                wg += j.wgs;
            }
        } else {
            // F32 / BF16: as many workgroups as fit on the chip at once; where
            // 512-thread ones cannot fill it, 256-thread ones, twice as many
            for (int pass = 0; pass < 2; pass++) {
                const void* const kern = one ? (const void*)one_kernel(a.job[0].kind, false) : (const void*)table_kernel(a, jobs_here);
                const int64_t cap = cu * fl_resident(kern, lds) * (FL_WG / threads), rpb = threads / 64;
                wg = 0;
                for (int i = 0; i < jobs_here; i++) {
                    a.job[i].wg0 = (int32_t)wg;
                    a.job[i].wgs = (int32_t)std::min<int64_t>((a.job[i].m + rpb - 1) / rpb, cap);
                    wg += a.job[i].wgs;
                }
                if (pass == 0 && wg < 2 * cu) threads = FL_WG / 2;
                else break;
            }
        }
        if (wg > 0x7fffffff) return set_error(ERR_SHAPE, "linear: job table too large for one launch");
        static bool lds_set = false;
        if (!lds_set) {
            const void* const all[] = {
                (const void*)k_flinear, (const void*)k_flinear_rows<KIND_F32>, (const void*)k_flinear_rows<KIND_BF16>,
                (const void*)k_flinear_one<KIND_F32>, (const void*)k_flinear_one<KIND_BF16>,
                (const void*)k_flinear_one<KIND_Q8_0>, (const void*)k_flinear_one<KIND_Q8_0, 1>,
                (const void*)k_flinear_one<KIND_IQ4_NL>, (const void*)k_flinear_one<KIND_Q6_K, 1>,
                (const void*)k_flinear_one<KIND_IQ4_XS>, (const void*)k_flinear_one<KIND_Q6_K>,
                (const void*)k_flinear_one<KIND_IQ3_XXS>};
            for (const void* f : all)
                UQ_CHECK_HIP(hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize,
                                                 (int)(stage_bytes(KIND_Q8_0, 16384) + 16 * 64 * FL_SEGS)));
            lds_set = true;
        }
        if (one) {
            hipLaunchKernelGGL(one_kernel(a.job[0].kind, few), dim3((unsigned)wg), dim3(threads), lds, s,
                               (OneJob{a.parts, a.job[0]}));
        } else {
            int64_t widest = 0;
            for (int i = 0; i < MAX_JOBS; i++) {
                a.start[i] = i < jobs_here ? a.job[i].wg0 : 0x7fffffff;
                if (i < jobs_here) widest = std::max<int64_t>(widest, a.job[i].wgs);
            }
            // a grid row per job, as wide as the widest, unless that leaves more
            // than half of the workgroups without work
            const bool rows = widest * jobs_here <= 2 * wg;
            const dim3 grid = rows ? dim3((unsigned)widest, (unsigned)jobs_here) : dim3((unsigned)wg);
            hipLaunchKernelGGL(table_kernel(a, jobs_here), grid, dim3(threads), lds, s, a);
        }
        UQ_CHECK_HIP(hipGetLastError());
    }
    return OK;
}

}  // namespace


extern "C" {

int uq_dequantize(uint32_t kind, const void* bytes, size_t nbytes, int64_t n, float* out) {
    if (!uq_stream()) return set_error(ERR_ARG, "uq_init has not been called");
    if (!bytes || !out) return set_error(ERR_ARG, "dequantize: null pointer");
    const int64_t rb = row_bytes(kind, n);
    if (rb == ERR_QUANT_TYPE || kind == KIND_Q3_K || kind == KIND_Q4_K)
        return set_error(ERR_QUANT_TYPE, "dequantize: unsupported kind (frontier_core.rs:53-58)");
    if (rb < 0) return set_error(ERR_SHAPE, "dequantize: n is not a whole number of blocks");
    if ((int64_t)nbytes != rb) return set_error(ERR_SHAPE, "dequantize: byte count != row_bytes(kind, n)");
    hipStream_t s = (hipStream_t)uq_stream();
    const size_t in_bytes = ((size_t)rb + 255) & ~(size_t)255;
    void* stage = nullptr;
    if (int rc = staging_buffer(in_bytes + sizeof(float) * (size_t)n, &stage)) return rc;
    uint8_t* const din = (uint8_t*)stage;
    float* const dout = (float*)((char*)stage + in_bytes);
    hipError_t e = hipMemcpyAsync(din, bytes, (size_t)rb, hipMemcpyHostToDevice, s);
    if (e == hipSuccess) {
        hipLaunchKernelGGL(k_dequant, dim3(grid_blocks(n)), dim3(FWG), 0, s, din, dout, kind, n);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipMemcpyAsync(out, dout, sizeof(float) * (size_t)n, hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    if (e != hipSuccess) return set_error(ERR_DEVICE, std::string("dequantize: ") + hipGetErrorString(e));
    return OK;
}

int uq_linear_multi_dev(const uq_linear_job* jobs, int count, void* stream) {
    if (!uq_stream()) return set_error(ERR_ARG, "uq_init has not been called");
    return enqueue_jobs(jobs, count, stream ? (hipStream_t)stream : (hipStream_t)uq_stream());
}

int uq_linear_dev(uq_weight_t w, const float* x, float* y, void* stream) {
    const uq_linear_job j{w, x, y};
    return uq_linear_multi_dev(&j, 1, stream);
}

int uq_linear_batch(const uq_linear_job* jobs, int count) {
    if (!uq_stream()) return set_error(ERR_ARG, "uq_init has not been called");
    if (!jobs || count <= 0) return set_error(ERR_ARG, "linear_batch: empty job table");
    int64_t xs = 0, ys = 0;
    for (int i = 0; i < count; i++) {
        if (int rc = check_job_weight(jobs[i].weight)) return rc;
        if (!jobs[i].x || !jobs[i].y) return set_error(ERR_ARG, "linear_batch: null x or y");
        xs += jobs[i].weight->w.n;
        ys += jobs[i].weight->w.m;
    }
    hipStream_t s = (hipStream_t)uq_stream();
    const size_t x_bytes = (sizeof(float) * (size_t)xs + 255) & ~(size_t)255;
    void *stage = nullptr, *host = nullptr;
    if (int rc = host_buffer(x_bytes + sizeof(float) * (size_t)ys + 16, &host)) return rc;
    float* const hx = (float*)host;
    float* const hy = (float*)((char*)host + x_bytes);
    int64_t xo = 0, yo = 0;
    for (int i = 0; i < count; i++) {
        const int64_t n = jobs[i].weight->w.n;
        if (!copy_finite(hx + xo, jobs[i].x, n)) return set_error(ERR_NONFINITE, "linear_batch: input: non-finite value");
        xo += n;  // n % 8 == 0 keeps every x 32-byte aligned
    }
    const bool direct = ys <= HOST_DIRECT;
    if (int rc = staging_buffer(x_bytes + (direct ? 0 : sizeof(float) * (size_t)ys + 16), &stage)) return rc;
    float* const dx = (float*)stage;  // every workgroup of a job reads its x
    float* const dy = direct ? hy : (float*)((char*)stage + x_bytes);
    std::vector<uq_linear_job> dj((size_t)count);
    xo = 0;
    for (int i = 0; i < count; i++) {
        const Weight& w = jobs[i].weight->w;
        dj[(size_t)i] = uq_linear_job{jobs[i].weight, dx + xo, dy + yo};
        xo += w.n;
        yo += w.m;
    }
    launch_copy(dx, hx, sizeof(float) * (size_t)xs, s);
    const int rc = enqueue_jobs(dj.data(), count, s);
    if (rc == OK && !direct) launch_copy(hy, dy, sizeof(float) * (size_t)ys, s);
    hipError_t e = hipGetLastError();
    // a failed enqueue still leaves the copy above reading the pinned buffer
    const hipError_t es = wait_host();
    if (e == hipSuccess) e = es;
    if (e != hipSuccess) return set_error(ERR_DEVICE, std::string("linear_batch: ") + hipGetErrorString(e));
    if (rc != OK) return rc;
    yo = 0;
    bool finite = true;
    for (int i = 0; i < count; i++) {
        const int64_t m = jobs[i].weight->w.m;
        finite = copy_finite(jobs[i].y, hy + yo, m) && finite;
        yo += m;
    }
    return finite ? OK : set_error(ERR_NONFINITE, "linear_batch: output: non-finite value");
}

int uq_time_linear(const uq_weight_t* ws, int count, int reps, int warmup, double* total_ms) {
    if (!uq_stream()) return set_error(ERR_ARG, "uq_init has not been called");
    if (!ws || count <= 0 || reps <= 0 || warmup < 0 || !total_ms) return set_error(ERR_ARG, "time_linear: bad args");
    int64_t xs = 0, ys = 0;
    for (int i = 0; i < count; i++) {
        if (int rc = check_job_weight(ws[i])) return rc;
        xs += ws[i]->w.n;
        ys += ws[i]->w.m;
    }
    hipStream_t s = (hipStream_t)uq_stream();
    float *dx = nullptr, *dy = nullptr;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    UQ_CHECK_HIP(hipMalloc(&dx, sizeof(float) * (size_t)xs));
    hipError_t e = hipMalloc(&dy, sizeof(float) * (size_t)ys);
    if (e == hipSuccess) e = hipMemsetAsync(dx, 0, sizeof(float) * (size_t)xs, s);
    if (e == hipSuccess) e = hipEventCreate(&e0);
    if (e == hipSuccess) e = hipEventCreate(&e1);
    int rc = OK;
    std::vector<uq_linear_job> jobs((size_t)count);
    int64_t xo = 0, yo = 0;
    for (int i = 0; i < count; i++) {
        jobs[(size_t)i] = uq_linear_job{ws[i], dx + xo, dy + yo};
        xo += ws[i]->w.n;
        yo += ws[i]->w.m;
    }
    for (int r = 0; r < warmup + reps && e == hipSuccess && rc == OK; r++) {
        if (r == warmup) e = hipEventRecord(e0, s);
        for (int i = 0; i < count && rc == OK; i++) rc = enqueue_jobs(&jobs[(size_t)i], 1, s);
    }
    if (e == hipSuccess && rc == OK) e = hipEventRecord(e1, s);
    if (e == hipSuccess && rc == OK) e = hipEventSynchronize(e1);
    float ms = 0.0f;
    if (e == hipSuccess && rc == OK) e = hipEventElapsedTime(&ms, e0, e1);
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    (void)hipStreamSynchronize(s);
    (void)hipFree(dx);
    if (dy) (void)hipFree(dy);
    if (e != hipSuccess) return set_error(ERR_DEVICE, std::string("time_linear: ") + hipGetErrorString(e));
    if (rc != OK) return rc;
    *total_ms = ms;
    return OK;
}

int uq_time_linear_tables(const uq_linear_job* jobs, const int* sizes, int ntables, int reps, double* total_ms) {
    if (!uq_stream()) return set_error(ERR_ARG, "uq_init has not been called");
    if (!jobs || !sizes || ntables <= 0 || reps <= 0 || !total_ms) return set_error(ERR_ARG, "time_linear_tables: bad args");
    hipStream_t s = (hipStream_t)uq_stream();
    hipEvent_t e0 = nullptr, e1 = nullptr;
    UQ_CHECK_HIP(hipEventCreate(&e0));
    hipError_t e = hipEventCreate(&e1);
    int rc = OK;
    for (int r = 0; r <= reps && e == hipSuccess && rc == OK; r++) {  // round 0 untimed
        if (r == 1) e = hipEventRecord(e0, s);
        int off = 0;
        for (int t = 0; t < ntables && rc == OK; t++) {
            rc = enqueue_jobs(jobs + off, sizes[t], s);
            off += sizes[t];
        }
    }
    if (e == hipSuccess && rc == OK) e = hipEventRecord(e1, s);
    if (e == hipSuccess && rc == OK) e = hipEventSynchronize(e1);
    float ms = 0.0f;
    if (e == hipSuccess && rc == OK) e = hipEventElapsedTime(&ms, e0, e1);
    (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    if (e != hipSuccess) return set_error(ERR_DEVICE, std::string("time_linear_tables: ") + hipGetErrorString(e));
    if (rc != OK) return rc;
    *total_ms = ms;
    return OK;
}

int uq_linear(uq_weight_t w, const float* x, int64_t n, float* y, int64_t m) {
    if (!w) return set_error(ERR_ARG, "linear: null weight");
    if (w->w.n != n || w->w.m != m) return set_error(ERR_SHAPE, "linear: tensor shape != x/y lengths");
    const uq_linear_job j{w, x, y};
    return uq_linear_batch(&j, 1);
}

}  // extern "C"
