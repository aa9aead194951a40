// Prefill GEMM of the formats scaled per 32 weights: the 32-weight formats (Q8_0, IQ4_NL, MXFP4, Q4_0,
// Q4_1, Q5_0, Q5_1) and IQ4_XS, whose 32-weight sub-blocks have a scale each (K a multiple of 256; Q8_0,
// IQ4_NL and Q4_0 also of 32 only).
//
// Integer arithmetic as in hk's CPU kernels (src/quant/gemm.zig kernelLegacy 131-176, kernelK 180-236
// per sub-block for IQ4_XS): per block c, y += (dw[r,c]*da[t,c]) * I_c with the exact integer I_c: one
// 32x32x32 int8 MFMA yields a tile's I_c, then each output takes a convert, a multiply (dw*da) and an fma.
// IQ4_XS's sub-block scales are integers and its activations have one scale per 256: sum_c ls_c * I_c is
// taken in integers (one 24-bit multiply-add per output and block), the floats once per super-block.
// Q4_0 / Q5_0 weights enter as u - zp (kernelLegacy's acci - zp*s); Q4_1 / Q5_1 as u, plus the offset
// term sum_c m[r,c] * (da*s)[t,c] (kernelLegacy's has_m term) on bf16 MFMAs: m (an f16) is hi + lo exactly
// (8 + at most 3 significant bits), the token side hi + mid + lo (the activation buffer's a8_dsb plane);
// three 32x32x16 MFMAs pair (hi|mid) with m's hi and lo and the token lo with m's hi -- every partial
// product down to 2^-24 relative. Only the f32 summation order differs from the reference.
//
// That was 48 VALU instructions per MFMA, and issuing them is what bounds such a tile (a SIMD takes about
// 1.8 ns each and 7 ns per MFMA). Two thirds do: the MFMA starts from MAGIC = 0x4B400000 instead of zero, so
// that its result, read as a float, is f = 1.5 * 2^23 + I_c, and fma(f, dw, -1.5 * 2^23 * dw) is I_c * dw with
// one rounding (-1.5 * 2^23 * dw is exact: dw has at most 11 significant bits); the second fma takes da from
// one register for all 16 tokens of a lane's half by DPP broadcast, which also spares four LDS reads in five.
// K <= 512 keeps the three instructions: dw*da rounds first there, as in hk's CPU kernels, so that the sums of a few
// blocks are theirs almost to the bit and the next layer's int8 rounding falls the same way (a small Q8_0 network
// had twice as many logit rows off by an int8 step otherwise); it costs little, 14336 x 512 at 200 tokens 12.3
// against 11.7 us, at 1000 38.7 against 32.8, where K 768 has 50.6 against 44.0.
// Steps with a scale of 2^100 or more (infinite, NaN, huge E8M0 exponents) take the three instructions,
// and so do the tiles of 32 tokens, where latency bounds and the two measured the same (12-15 us a round of K 4096).
//
// The structure is that of mmg.hip: 32*NW rows x 32*TT tokens per workgroup, KS slices of K, the
// activations of a step (256 values) shared by a slice's row waves and double buffered, the weights
// private to a wave; the updates of one block run beside the MFMA of the next.
// Measured, against a ring of whole-step slots with one wave per SIMD in most tiles: Q8_0 14336 x 4096 at 512
// tokens 210 -> 102 us (113 with three instructions per output), 4096 x 4096 64 -> 36 us, at 16 tokens 31 -> 11
// us; Q4_0 4096 x 4096 at 200 tokens 92 -> 25 us; IQ4_XS 14336 x 4096 at 1000 tokens 201 -> 170 us. K tails: Q8_0
// 4864 x 896 at 333 tokens 21 -> 14 us (a kernel without overlap), Q4_0 264 -> 13 us (decode passes of 8 tokens).

#include "common.hpp"
#include "gemm_store.hpp"

namespace hkhip {
namespace mb {

typedef int v16i __attribute__((ext_vector_type(16)));
typedef int v4i __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));

template <int T> constexpr bool is_xs = T == HKHIP_IQ4_XS;
template <int T> constexpr uint32_t row_bytes() { return T == HKHIP_Q8_0 ? 256 : 128; } // per row and step

// Activations of one step: chunk c of token t at c ^ (t & 15); the scales per block and token, [8][TOK]
// (IQ4_XS: per token); Q4_1 / Q5_1: the tokens' 48 bytes of a8_dsb.
template <int T, int TOK> struct ASlot {
    int8_t a[TOK * 256];
    float da[is_xs<T> ? (TOK + 63) / 64 * 64 : 8 * TOK];
    uint8_t dsb[has_m(T) ? (TOK * 48 + 1023) / 1024 * 1024 : 16];
};
// One wave's 32 rows of one step: quants (16-byte piece c of row r at c ^ (r & 15), & 7 for 128 bytes),
// 16 bytes of scales per row (then 16 of offsets), the fifth-bit words; IQ4_XS: 8 bytes per row.
template <int T> struct WSlot {
    uint8_t q[32 * row_bytes<T>()];
    uint8_t s[is_xs<T> ? 256 : 1024];
    uint8_t h[has_qh(T) ? 1024 : 16];
};
template <int NW, int KS> constexpr int resident() { return NW * KS < 8 && KS < 4 ? 2 : 1; }
// Two weight buffers per wave for the 32-token tiles, whose steps are short, where they fit.
template <int T, int NW, int TT, int KS> constexpr int wbufs() {
    return TT == 1 && sizeof(ASlot<T, 32 * TT>) * 2 * KS + sizeof(WSlot<T>) * 2 * KS * NW <= 160 * 1024 / resident<NW, KS>() ? 2 : 1;
}
template <int T, int NW, int TT, int KS> struct Smem {
    ASlot<T, 32 * TT> a[KS][2];
    WSlot<T> w[KS * NW][wbufs<T, NW, TT, KS>()];
};

struct MbArgs {
    const uint8_t *w;
    const uint8_t *ws; // scale (side) plane
    uint32_t rows, cols, n;
    const int8_t *aqs;
    const float *ad;
    const uint8_t *adsb; // a8_dsb: [k/256][n][48 B]
    float *y;
    const float *bias;
    int mode;
    int wide; // y 16-byte aligned and rows a multiple of 4: whole tiles go out as 16-byte stores
    uint32_t rblocks, tblocks;
};

// acc[V0 + i] += x[i] * (ds of lane V0 + i of this lane's row of 16 lanes), i < 8: fused multiply-adds with a DPP
// broadcast. The s_nop covers the two wait states between a VALU write of ds and a DPP read of it.
template <int V0> __device__ __forceinline__ void fma8_bcast(v16f &acc, const float (&x)[8], float ds) {
    float y[8];
#pragma unroll
    for (int i = 0; i < 8; i++) y[i] = acc[V0 + i];
    asm("s_nop 1\n"
        "v_fmac_f32_dpp %0, %16, %8 row_newbcast:%17 row_mask:0xf bank_mask:0xf\n"
        "v_fmac_f32_dpp %1, %16, %9 row_newbcast:%18 row_mask:0xf bank_mask:0xf\n"
        "v_fmac_f32_dpp %2, %16, %10 row_newbcast:%19 row_mask:0xf bank_mask:0xf\n"
        "v_fmac_f32_dpp %3, %16, %11 row_newbcast:%20 row_mask:0xf bank_mask:0xf\n"
        "v_fmac_f32_dpp %4, %16, %12 row_newbcast:%21 row_mask:0xf bank_mask:0xf\n"
        "v_fmac_f32_dpp %5, %16, %13 row_newbcast:%22 row_mask:0xf bank_mask:0xf\n"
        "v_fmac_f32_dpp %6, %16, %14 row_newbcast:%23 row_mask:0xf bank_mask:0xf\n"
        "v_fmac_f32_dpp %7, %16, %15 row_newbcast:%24 row_mask:0xf bank_mask:0xf"
        : "+v"(y[0]), "+v"(y[1]), "+v"(y[2]), "+v"(y[3]), "+v"(y[4]), "+v"(y[5]), "+v"(y[6]), "+v"(y[7])
        : "v"(x[0]), "v"(x[1]), "v"(x[2]), "v"(x[3]), "v"(x[4]), "v"(x[5]), "v"(x[6]), "v"(x[7]), "v"(ds), "n"(V0), "n"(V0 + 1),
          "n"(V0 + 2), "n"(V0 + 3), "n"(V0 + 4), "n"(V0 + 5), "n"(V0 + 6), "n"(V0 + 7));
#pragma unroll
    for (int i = 0; i < 8; i++) acc[V0 + i] = y[i];
}
template <int V0> __device__ __forceinline__ void fma8(v16f &acc, const v16i &p, float ds, float dw, float mdw) {
    float x[8];
#pragma unroll
    for (int i = 0; i < 8; i++) x[i] = fmaf(__builtin_bit_cast(float, int(p[V0 + i])), dw, mdw);
    fma8_bcast<V0>(acc, x, ds);
}

// TAIL: K is not a multiple of 256. The last step's loads run past the row into the next one, or past
// the plane into the one behind it (every plane is followed by another, or by its 256-byte rounding),
// and the blocks past the row are left out; the scales, whose rows are then not 16-byte aligned, are read
// by ordinary loads.
template <int T, int NW, int TT, int KS, bool TAIL>
__global__ __launch_bounds__(NW * KS * 64, (NW * KS * resident<NW, KS>() / 4)) void mmb_kernel(MbArgs a) {
    constexpr int TOK = 32 * TT;
    constexpr bool xs = is_xs<T>, q8 = T == HKHIP_Q8_0, quick_t = !xs && TT > 1;
    constexpr uint32_t RB = row_bytes<T>(), PPR = RB / 16;
    static_assert(!TAIL || (!xs && !has_m(T) && !has_qh(T)), "K tails: scale-only formats");
    __shared__ __attribute__((aligned(16))) Smem<T, NW, TT, KS> S;
    const uint32_t tid = threadIdx.x, lane = tid & 63;
    const uint32_t wall = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t ks = wall / NW, wave = wall % NW; // K slice, row wave within the slice
    const uint32_t h = lane >> 5, j = lane & 31;
    const uint32_t K = a.cols, nbr = K / 32, nsb = (K + 255) / 256;

    // Workgroup -> (row block, token block); the token blocks of a row block run on one XCD so
    // its L2 serves the repeated weight reads (workgroups go round-robin over the 8 XCDs).
    uint32_t rb, tb;
    {
        const uint32_t i = blockIdx.x;
        if (a.rblocks % 8 == 0) {
            const uint32_t xcd = i % 8, k = i / 8;
            rb = xcd * (a.rblocks / 8) + k / a.tblocks;
            tb = k % a.tblocks;
        } else {
            rb = i / a.tblocks;
            tb = i % a.tblocks;
        }
    }
    const uint32_t r0 = rb * 32 * NW, t0 = tb * TOK, rw0 = r0 + 32 * wave;
    const uint32_t myrow = rw0 + j;
    auto clamp_row = [&](uint32_t r) { return r < a.rows ? r : a.rows - 1; };
    auto clamp_tok = [&](uint32_t t) { return t < a.n ? t : a.n - 1; };

    // ---- direct loads: per-lane 32-bit offsets from uniform bases (mmb_supports checks the range) ----
    constexpr uint32_t TPW = TOK / NW; // token rows per wave
    static_assert(TPW % 4 == 0, "token rows per wave");
    uint32_t aoff[TPW / 4];
#pragma unroll
    for (uint32_t i = 0; i < TPW / 4; i++) {
        const uint32_t tl = TPW * wave + 4 * i + lane / 16;
        aoff[i] = clamp_tok(t0 + tl) * K + 16 * ((lane % 16) ^ (tl & 15));
    }
    // Token scales: load i of wave m covers entries 64*(DAL*m + i) .. of [8][TOK]: block e / TOK, token
    // e % TOK; IQ4_XS: wave m < TOK/64 loads tokens 64m...
    constexpr uint32_t DAL = xs ? 1 : 8 * TOK / (64 * NW);
    uint32_t doff[DAL];
#pragma unroll
    for (uint32_t i = 0; i < DAL; i++) {
        const uint32_t e = 64 * (DAL * wave + i) + lane;
        doff[i] = xs ? clamp_tok(t0 + 64 * wave + lane) * nsb * 4 : clamp_tok(t0 + e % TOK) * nbr * 4 + 4 * (e / TOK);
    }
    auto issue_a = [&](uint32_t sb, ASlot<T, TOK> &A) {
        const int8_t *ga = a.aqs + 256 * sb;
        const uint8_t *gd = reinterpret_cast<const uint8_t *>(a.ad);
#pragma unroll
        for (uint32_t i = 0; i < TPW / 4; i++) load_lds16(ga, aoff[i], &A.a[(TPW * wave + 4 * i) * 256]);
        if constexpr (xs) {
            if (64 * wave < uint32_t(TOK)) load_lds4(gd + 4 * sb, doff[0], &A.da[64 * wave]);
        } else {
#pragma unroll
            for (uint32_t i = 0; i < DAL; i++) load_lds4(gd + 32 * sb, doff[i], &A.da[64 * (DAL * wave + i)]);
        }
        if constexpr (has_m(T)) { // the token range's 48-byte rows are contiguous: 1-KB chunks
            for (uint32_t m = wave; m < (TOK * 48 + 1023) / 1024; m += NW) {
                const uint32_t e = 1024 * m + 16 * lane;
                load_lds16(a.adsb + uint64_t(sb) * a.n * 48, clamp_tok(t0 + e / 48) * 48 + e % 48, &A.dsb[1024 * m]);
            }
        }
    };
    const uint32_t rowbytes = nbr * (q8 ? 32 : 16);
    uint32_t woff[RB / 32];
#pragma unroll
    for (uint32_t i = 0; i < RB / 32; i++) {
        const uint32_t P = 64 * i + lane, lr = P / PPR;
        woff[i] = clamp_row(rw0 + lr) * rowbytes + 16 * ((P % PPR) ^ (lr & (PPR - 1)));
    }
    const uint32_t srow = clamp_row(myrow);
    const SideGeom G = side_geom(T, nbr);
    // Side data: the blocks' eight f16 per row (lanes 32-63 the offsets, or a repeat); the fifth-bit
    // words of blocks 0-3 (lanes 0-31) and 4-7; IQ4_XS: lane L word L % 2 of row L / 2's header.
    const uint32_t soff = xs ? clamp_row(rw0 + lane / 2) * nsb * 8 + 4 * (lane % 2) : srow * G.stride + (h && has_m(T) ? G.m_off : 0);
    const uint32_t hoff = srow * G.stride + G.qh_off + 16 * h;
    constexpr int WB = wbufs<T, NW, TT, KS>();
    auto issue_w = [&](uint32_t sb, WSlot<T> &W) {
        const uint8_t *gw = a.w + uint64_t(sb) * RB;
#pragma unroll
        for (uint32_t i = 0; i < RB / 32; i++) load_lds16(gw, woff[i], &W.q[1024 * i]);
        if constexpr (xs)
            load_lds4(a.ws + 8 * sb, soff, &W.s[0]);
        else if constexpr (!TAIL)
            load_lds16(a.ws + 16 * sb, soff, &W.s[0]);
        if constexpr (has_qh(T)) load_lds16(a.ws + 32 * sb, hoff, &W.h[0]);
    };
    // TAIL: this lane's row's scales of a step (past the row: repeats of its last block's, not used).
    uint32_t sraw[TAIL ? 8 : 1];
    auto load_scales = [&](uint32_t sb) {
        const uint16_t *p = reinterpret_cast<const uint16_t *>(a.ws) + uint64_t(srow) * nbr;
#pragma unroll
        for (uint32_t c = 0; c < (TAIL ? 8 : 1); c++) sraw[c] = p[8 * sb + c < nbr ? 8 * sb + c : nbr - 1];
    };

    v16f acc[TT];
#pragma unroll
    for (int t = 0; t < TT; t++)
#pragma unroll
        for (int v = 0; v < 16; v++) acc[t][v] = 0.0f;

    // MAGIC: as the addend of the integer products it makes their sum, read as a float, 1.5 * 2^23 + I_c
    // (|I_c| < 2^22); kept in registers, it is no inline constant.
    v16i magic;
#pragma unroll
    for (int v = 0; v < 16; v++) magic[v] = 0x4B400000;
    if constexpr (quick_t) asm volatile("" : "+v"(magic));

    // Step st of slice ks is super-block ks + KS*st.
    const uint32_t nst = (nsb + KS - 1) / KS;
    auto sb_of = [&](uint32_t st) {
        const uint32_t sb = ks + KS * st;
        return sb < nsb ? sb : nsb - 1;
    };
    issue_a(sb_of(0), S.a[ks][0]);
    issue_w(sb_of(0), S.w[wall][0]);
    if constexpr (TAIL) load_scales(sb_of(0));
    __builtin_amdgcn_s_waitcnt(0x0F70); // vmcnt(0)
    __syncthreads();

    const uint32_t sw = j & 15;
    auto step = [&](uint32_t buf, uint32_t st) {
        ASlot<T, TOK> &A = S.a[ks][buf];
        const WSlot<T> &W = S.w[wall][WB == 2 ? buf : 0];
        const bool more = st + 1 < nst;
        if (more) {
            issue_a(sb_of(st + 1), S.a[ks][buf ^ 1]);
            if constexpr (WB == 2) issue_w(sb_of(st + 1), S.w[wall][buf ^ 1]);
        }
        // ---- operands: block c of this lane's row, its 16 weights of half h ----
        v4i wv[8];
        float dw[xs ? 1 : 8]; // IQ4_XS: the super-block's scale, and the sub-blocks' integers
        int ls[xs ? 8 : 1];
        v8bf m1, m2, m3;
        const uint8_t *blk = &W.q[RB * j];
        if constexpr (q8) {
#pragma unroll
            for (int c = 0; c < 8; c++) wv[c] = *reinterpret_cast<const v4i *>(blk + 16 * ((2 * c + h) ^ sw));
        } else {
            constexpr int TL = xs ? HKHIP_IQ4_NL : T; // IQ4_XS: IQ4_NL's codebook
            uint4 x[8], qh4[2] = {};
#pragma unroll
            for (int c = 0; c < 8; c++) x[c] = *reinterpret_cast<const uint4 *>(blk + 16 * (c ^ (j & 7)));
            if constexpr (has_qh(T)) {
                qh4[0] = *reinterpret_cast<const uint4 *>(&W.h[16 * j]);
                qh4[1] = *reinterpret_cast<const uint4 *>(&W.h[16 * (32 + j)]);
            }
            const uint32_t qh[8] = {qh4[0].x, qh4[0].y, qh4[0].z, qh4[0].w, qh4[1].x, qh4[1].y, qh4[1].z, qh4[1].w};
#pragma unroll
            for (int c = 0; c < 8; c++) {
                const uint32_t xw[4] = {x[c].x, x[c].y, x[c].z, x[c].w};
#pragma unroll
                for (int i = 0; i < 4; i++) wv[c][i] = int(low_bit_word<TL>(xw[i], qh[c], h, i));
            }
        }
        if constexpr (xs) {
            // ls_c = scales_l nibble | scales_h bits << 4, minus 32 (dequant.zig:443-447).
            const uint2 hd = *reinterpret_cast<const uint2 *>(&W.s[8 * j]);
            dw[0] = f16_bits_to_f32(hd.x & 0xFFFF);
#pragma unroll
            for (int c = 0; c < 8; c++) {
                const uint32_t lo = (hd.y >> (4 * c)) & 0xF, hi = (hd.x >> (16 + 2 * c)) & 3;
                ls[c] = int(lo | (hi << 4)) - 32;
            }
        } else if constexpr (TAIL) {
#pragma unroll
            for (int c = 0; c < 8; c++) dw[c] = block_scale<T>(sraw[c]);
            if (more) load_scales(sb_of(st + 1));
        } else {
            const uint4 s16 = *reinterpret_cast<const uint4 *>(&W.s[16 * j]);
            const uint32_t sw4[4] = {s16.x, s16.y, s16.z, s16.w};
#pragma unroll
            for (int c = 0; c < 8; c++) dw[c] = block_scale<T>((sw4[c / 2] >> (16 * (c & 1))) & 0xFFFF);
        }
        if constexpr (has_m(T)) {
            const uint4 m16 = *reinterpret_cast<const uint4 *>(&W.s[16 * (32 + j)]);
            const uint32_t mw4[4] = {m16.x, m16.y, m16.z, m16.w};
            uint32_t mh[4], ml[4];
#pragma unroll
            for (int q = 0; q < 4; q++) {
                uint32_t hi2[2], lo2[2];
#pragma unroll
                for (int e = 0; e < 2; e++) {
                    const float m = f16_bits_to_f32((mw4[q] >> (16 * e)) & 0xFFFF);
                    hi2[e] = __builtin_bit_cast(uint32_t, m) & 0xFFFF0000u;
                    lo2[e] = __builtin_bit_cast(uint32_t, m - __builtin_bit_cast(float, hi2[e]));
                }
                mh[q] = __builtin_amdgcn_perm(hi2[1], hi2[0], 0x07060302u);
                ml[q] = __builtin_amdgcn_perm(lo2[1], lo2[0], 0x07060302u);
            }
            m1 = __builtin_bit_cast(v8bf, make_uint4(mh[0], mh[1], mh[2], mh[3]));
            m2 = __builtin_bit_cast(v8bf, make_uint4(ml[0], ml[1], ml[2], ml[3]));
            m3 = h ? v8bf{} : m1;
        }
        if constexpr (WB == 1) {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); // the reads are done: the bytes may be overwritten
            if (more) issue_w(sb_of(st + 1), S.w[wall][0]);
        }
        const uint32_t sb = ks + KS * st;
        if (KS > 1 && sb >= nsb) { // a slice past its last super-block keeps its loads in step
            __builtin_amdgcn_s_waitcnt(0x0F70);
            __syncthreads();
            return;
        }

        const uint32_t mytok = 8 * (lane % 16 / 4) + 4 * h + lane % 4; // the token of output lane % 16
        const int8_t *abase = &A.a[j * 256];
        v4i av[4];
        // Chunk c of tile t (c >= 8: of the next tile) into the ring of four operands.
        auto load_a = [&](int t, int c) {
            av[c % 4] = *reinterpret_cast<const v4i *>(abase + 32 * (t + c / 8) * 256 + 16 * ((2 * (c % 8) + h) ^ sw));
        };
        // Block c's integers into tile t: this lane's 16 outputs are tokens 32t + 8g + 4h + (0..3).
        int isum[xs ? 16 : 1];
        auto update = [&](const v16i &p, int t, int c, bool quick) __attribute__((always_inline)) {
            if constexpr (xs) {
                // |I_c| <= 32*127*127 < 2^23: 24-bit products; the sum of the eight stays below 2^28.
#pragma unroll
                for (int v = 0; v < 16; v++) isum[v] = c ? __mul24(p[v], ls[c]) + isum[v] : __mul24(p[v], ls[0]);
                if (c < 7) return;
            }
            if constexpr (quick_t)
                if (quick) { // p holds MAGIC + I_c, the bits of the float 1.5 * 2^23 + I_c
                    const float ds = A.da[c * TOK + 32 * t + mytok];
                    const float mdw = -12582912.0f * dw[c]; // exact: dw has at most 11 significant bits
                    fma8<0>(acc[t], p, ds, dw[c], mdw);
                    fma8<8>(acc[t], p, ds, dw[c], mdw);
                    return;
                }
            const float4 *dap = reinterpret_cast<const float4 *>(&A.da[(xs ? 0 : c * TOK) + 32 * t + 4 * h]);
#pragma unroll
            for (int g = 0; g < 4; g++) {
                const float4 dv = dap[2 * g];
                const float ds[4] = {dv.x, dv.y, dv.z, dv.w};
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const int v = 4 * g + e;
                    acc[t][v] = fmaf((float)(xs ? isum[xs ? v : 0] : p[v]), dw[xs ? 0 : c] * ds[e], acc[t][v]);
                }
            }
        };
#pragma unroll
        for (int c = 0; c < 4; c++) load_a(0, c);
        const uint32_t nb = TAIL && nbr - 8 * sb < 8 ? nbr - 8 * sb : 8;
        // Blocks past the row (the same for the whole slice), a short K (see above), or a scale whose product with
        // MAGIC is not finite.
        bool odd = (TAIL && nb < 8) || K <= 512;
        if constexpr (quick_t) {
            bool nan = false;
#pragma unroll
            for (int c = 0; c < 8; c++) nan |= !(__builtin_fabsf(dw[c]) < 0x1p100f);
            odd |= __builtin_amdgcn_ballot_w64(nan) != 0;
        }
        if ((TAIL || quick_t) && odd) {
#pragma unroll
            for (int t = 0; t < TT; t++)
#pragma unroll
                for (int c = 0; c < 8; c++) {
                    if (uint32_t(c) < nb) update(__builtin_amdgcn_mfma_i32_32x32x32_i8(av[c % 4], wv[c], v16i{}, 0, 0, 0), t, c, false);
                    if (c < 4 || t + 1 < TT) load_a(t, c + 4);
                    __builtin_amdgcn_sched_barrier(0);
                }
        } else {
            v16i p[2];
#pragma unroll
            for (int t = 0; t < TT; t++)
#pragma unroll
                for (int c = 0; c < 8; c++) {
                    p[c % 2] = __builtin_amdgcn_mfma_i32_32x32x32_i8(av[c % 4], wv[c], quick_t ? magic : v16i{}, 0, 0, 0);
                    if (c < 4 || t + 1 < TT) load_a(t, c + 4);
                    if (c > 0)
                        update(p[(c + 1) % 2], t, c - 1, true);
                    else if (t > 0)
                        update(p[1], t - 1, 7, true);
                    __builtin_amdgcn_sched_barrier(0);
                }
            update(p[1], TT - 1, 7, true);
        }
        if constexpr (has_m(T)) {
#pragma unroll
            for (int t = 0; t < TT; t++) {
                const uint8_t *tm = &A.dsb[48 * (32 * t + j)];
                const v8bf a12 = __builtin_bit_cast(v8bf, *reinterpret_cast<const uint4 *>(tm + 16 * h));
                const v8bf a3 = __builtin_bit_cast(v8bf, *reinterpret_cast<const uint4 *>(tm + 32));
                acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a12, m1, acc[t], 0, 0, 0);
                acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a12, m2, acc[t], 0, 0, 0);
                acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a3, m3, acc[t], 0, 0, 0);
            }
        }
        __builtin_amdgcn_s_waitcnt(0x0F70); // vmcnt(0): the next super-block is in LDS
        __syncthreads();
    };
    for (uint32_t st = 0; st < nst; st += 2) {
        step(0, st);
        if (st + 1 < nst) step(1, st + 1);
    }

    // The loads of the last step have landed and every wave is past its barrier: the LDS is free.
    float *red = reinterpret_cast<float *>(&S);
    if constexpr (KS > 1) { // slices 1.. leave their tiles in the LDS; slice 0 adds them in order
        static_assert((KS - 1) * NW * TT * 4096 <= sizeof(S), "reduction space");
        if (ks > 0) {
#pragma unroll
            for (int t = 0; t < TT; t++)
#pragma unroll
                for (int v = 0; v < 16; v++) red[((((ks - 1) * NW + wave) * TT + t) * 16 + v) * 64 + lane] = acc[t][v];
        }
        __syncthreads();
        if (ks == 0) {
#pragma unroll
            for (int k = 1; k < KS; k++)
#pragma unroll
                for (int t = 0; t < TT; t++)
#pragma unroll
                    for (int v = 0; v < 16; v++) acc[t][v] += red[((((k - 1) * NW + wave) * TT + t) * 16 + v) * 64 + lane];
        }
        __syncthreads(); // the partial tiles are read: the space takes the output staging
        if (ks > 0) return;
    }
    static_assert(NW * 4096 <= sizeof(S), "output staging space");
    const float bias_r = (a.bias && myrow < a.rows) ? a.bias[myrow] : 0.0f;
#pragma unroll
    for (int t = 0; t < TT; t++) {
        const uint32_t tk0 = t0 + 32 * t;
        if (a.wide && rw0 + 32 <= a.rows && tk0 + 32 <= a.n)
            gemm_store_tile_wide(red + 1024 * wave, acc[t], bias_r, a.y, a.rows, rw0, tk0, a.mode);
        else
            gemm_store_tile(acc[t], bias_r, a.y, a.rows, a.n, myrow, tk0, a.mode);
    }
}

template <int T, int NW, int TT, int KS, bool TAIL> hipError_t launch_cfg(const MbArgs &a0, hipStream_t s) {
    static_assert(sizeof(Smem<T, NW, TT, KS>) <= 160 * 1024 / resident<NW, KS>(), "LDS");
    MbArgs a = a0;
    a.rblocks = (a.rows + 32 * NW - 1) / (32 * NW);
    a.tblocks = (a.n + 32 * TT - 1) / (32 * TT);
    hipLaunchKernelGGL((mmb_kernel<T, NW, TT, KS, TAIL>), dim3(a.rblocks * a.tblocks), dim3(NW * KS * 64), 0, s, a);
    return hipGetLastError();
}

// The tile whose rounds of workgroups cost least, as in mmg.hip: rounds of what is resident at once (one
// workgroup per CU, two for the tiles of four waves with at most two K slices), each its steps plus its
// ends. In tenths of a us, measured for Q8_0 and IQ4_NL at 1024-14336 rows, K 896 and 4096, 16-1000 tokens (a
// round of K 4096: <4,2,2> 30-36 us, <4,2,1> 58 (half 40), <2,1,4> 12-15, <2,1,2> 23 (half 15), <1,1,4> 11.5).
// <8,4,1> is for IQ4_XS, whose updates leave it the registers (a round 80 us; 14336 x 4096 at 512 tokens 89 us
// against 98 of <4,2,1>); the others would spill (145 us).
template <int T, bool TAIL = false> hipError_t launch_fmt(const MbArgs &a, hipStream_t s) {
    constexpr uint32_t CUS = 256;
    struct Tile {
        uint32_t nw, tt, ks, resident, step, half; // step, half: tenths of a us per step
    };
    const Tile tiles[6] = {{8, 4, 1, 1, 49, 49}, {4, 2, 2, 1, 41, 41}, {4, 2, 1, 2, 35, 24},
                           {2, 1, 4, 1, 31, 31}, {2, 1, 2, 2, 25, 16}, {1, 1, 4, 1, 24, 24}};
    const uint32_t nsb = (a.cols + 255) / 256;
    uint64_t best = ~0ull;
    int pick = 0;
    for (int i = is_xs<T> ? 0 : 1; i < 6; i++) {
        const Tile &c = tiles[i];
        const uint64_t grid = uint64_t((a.rows + 32 * c.nw - 1) / (32 * c.nw)) * ((a.n + 32 * c.tt - 1) / (32 * c.tt));
        const uint64_t cap = CUS * c.resident, rest = grid % cap, steps = (nsb + c.ks - 1) / c.ks;
        const uint64_t ends = c.ks > 1 ? 15 : 10;
        const uint64_t cost = grid / cap * (steps * c.step + ends) + (rest == 0 ? 0 : steps * (rest <= CUS ? c.half : c.step) + ends);
        if (cost < best) best = cost, pick = i;
    }
    if constexpr (is_xs<T>)
        if (pick == 0) return launch_cfg<T, 8, 4, 1, false>(a, s);
    switch (pick) {
    case 1: return launch_cfg<T, 4, 2, 2, TAIL>(a, s);
    case 2: return launch_cfg<T, 4, 2, 1, TAIL>(a, s);
    case 3: return launch_cfg<T, 2, 1, 4, TAIL>(a, s);
    case 4: return launch_cfg<T, 2, 1, 2, TAIL>(a, s);
    default: return launch_cfg<T, 1, 1, 4, TAIL>(a, s);
    }
}

} // namespace mb

bool mmb_supports(int t, uint32_t rows, uint32_t cols, uint32_t n) {
    if ((t != HKHIP_IQ4_XS && !legacy32(t)) || rows == 0 || n == 0 || cols == 0 || cols % 32) return false;
    if (cols % 256 != 0 && t != HKHIP_Q8_0 && t != HKHIP_IQ4_NL && t != HKHIP_Q4_0) return false;
    // 32-bit per-lane byte offsets: quant plane, side plane and activations.
    const WLayout W = weight_layout(t, rows, cols);
    return W.total < (1ull << 32) && uint64_t(n) * cols < (1ull << 32);
}

hipError_t launch_mmb(int t, const uint8_t *w, uint32_t rows, uint32_t cols, const uint8_t *xq, uint32_t n, float *y,
                      const float *bias, int mode, hipStream_t s) {
    if (!mmb_supports(t, rows, cols, n)) return hipErrorInvalidValue;
    const WLayout W = weight_layout(t, rows, cols);
    const ActLayout A = act_layout(n, cols);
    const bool kq = t == HKHIP_IQ4_XS;
    mb::MbArgs a{};
    a.w = w;
    a.ws = w + W.scale_off;
    a.rows = rows;
    a.cols = cols;
    a.n = n;
    a.aqs = reinterpret_cast<const int8_t *>(xq + (kq ? A.k_qs : A.a8_qs));
    a.ad = reinterpret_cast<const float *>(xq + (kq ? A.k_d : A.a8_d));
    a.adsb = xq + A.a8_dsb;
    a.y = y;
    a.bias = bias;
    a.mode = mode;
    a.wide = (reinterpret_cast<uintptr_t>(y) % 16 == 0 && rows % (mode == HKHIP_SILU_MUL ? 8 : 4) == 0) ? 1 : 0;
    const bool tail = cols % 256 != 0;
    switch (t) {
    case HKHIP_Q8_0: return tail ? mb::launch_fmt<HKHIP_Q8_0, true>(a, s) : mb::launch_fmt<HKHIP_Q8_0>(a, s);
    case HKHIP_IQ4_NL: return tail ? mb::launch_fmt<HKHIP_IQ4_NL, true>(a, s) : mb::launch_fmt<HKHIP_IQ4_NL>(a, s);
    case HKHIP_Q4_0: return tail ? mb::launch_fmt<HKHIP_Q4_0, true>(a, s) : mb::launch_fmt<HKHIP_Q4_0>(a, s);
    case HKHIP_MXFP4: return mb::launch_fmt<HKHIP_MXFP4>(a, s);
    case HKHIP_Q4_1: return mb::launch_fmt<HKHIP_Q4_1>(a, s);
    case HKHIP_Q5_0: return mb::launch_fmt<HKHIP_Q5_0>(a, s);
    case HKHIP_Q5_1: return mb::launch_fmt<HKHIP_Q5_1>(a, s);
    default: return mb::launch_fmt<HKHIP_IQ4_XS>(a, s);
    }
}

} // namespace hkhip
