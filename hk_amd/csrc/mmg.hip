// Prefill GEMM of the super-block formats whose group scales fold into int8 weights: Q4_K, Q5_K, Q6_K,
// Q3_K and Q2_K (K a multiple of 256).
//
// Integer arithmetic as in hk's CPU kernels (src/quant/gemm.zig kernelK 180-236 with the canonical
// unpack of unpack.zig; dotCanonK, vecdot.zig:686-705): per row r, token t and super-block b the
// products of the 256 weights are one exact integer, scaled once in f32.
//  * Q6_K: w = sc*(q - 32) in [-4096, 4096] as two int8 planes, 4*w = 256*H + L (q6k_planes); the
//    two MFMA chains give (H-sum << 8) + L-sum = 4*I, and y += (d/4)*da * that.
//  * Q4_K: the 6-bit scale sc = 8*sh + sl, planes sh*q and sl*q (each at most 105: one packed 16-bit
//    multiply makes four weights); I = 8 * (sh-sum) + (sl-sum). Q5_K: sc*q <= 1953 = 256*H + L. The
//    mins are J = sum_s mn[s]*bsum32[s], an integer below 2^22 whose factors are exact bf16 integers
//    once bsum32 = 64*u + v (the activation buffer's k_mb plane): one 32x32x16 bf16 MFMA yields J
//    exactly in f32; y += da*(d*I - dmin*J).
//  * Q3_K: w = sc*(q - 4), sc in [-32, 31], q in [0, 7]: -w lies in [-128, 124], one int8 plane,
//    looked up: a group's eight products are two registers, a byte permute picks four at once.
//    y += -d*da * sum.
//  * Q2_K: sc*q <= 45, one plane (a packed 16-bit multiply makes four weights, no carries). The
//    group mins are a K = 16 product, J = sum_g mn[g]*bsum[g], with |bsum| <= 2032 and mn <= 15 both
//    exact in f16: one 32x32x16 f16 MFMA yields J exactly in f32; y += da*(d*I - dmin*J).
// Only the f32 summation order over super-blocks differs from the reference.
//
// Structure. A workgroup owns 32*NW rows x 32*TT tokens; its NW*KS waves are KS slices of K, slice
// k taking super-blocks k, k + KS, ... (partial tiles are added in LDS in slice order at the end).
// What bounds it is the VALU work of building the planes (Q6_K: ~3.3 instructions per weight) beside
// the MFMAs, so a SIMD needs two waves, one building while the other multiplies, and the LDS has
// to hold eight waves' operands: the activations of a super-block are shared by a slice's row
// waves and double buffered, but the weights are private to a wave and need one buffer only. A
// wave reads its rows' block from it into registers, and once those reads have returned the
// next block's loads go out into the same bytes, landing under the MFMAs.
// Inside a wave the order is fixed (sched_barrier): each MFMA is followed by a share of the VALU work
// that does not depend on it. Measured on this GPU, a SIMD's two waves take the larger of 16.5 ns per
// MFMA and 7 ns per MFMA plus 1.8 ns per VALU instruction: at 128 tokens per wave Q6_K's ~64 MFMAs and
// ~740 VALU instructions per super-block are VALU-bound.
// Measured at 512 tokens: Q3_K 14336 x 4096 30.6 ms (decode passes of 8 tokens on float-decoded
// weights) -> 53 us, Q2_K 57 us (1050 TOPS); Q6_K, against a tile that rebuilt its planes every 64
// tokens with one wave per SIMD, 14336 x 4096 169 -> 82 us, 4096 x 14336 152 -> 105 us, at 100 tokens
// 90 -> 44 us, 1024 x 4096 29.4 -> 15.9 us; Q4_K, against a tile with weights loaded row by row into registers
// and the mins on three bf16 MFMAs, 14336 x 4096 83 -> 73 us, 28672 x 4096 170 -> 158 us (and half the
// error against float64: 2.0e-7 -> 0.9e-7); Q5_K 14336 x 4096 108 -> 89 us, 4096 x 14336 147 -> 105 us, 4096 x
// 4096 at 100 tokens 38 -> 15 us. (A three-slot ring with the barrier moved inside the step and
// the planes built one super-block ahead was no faster, 109 -> 114 us at 4096 x 14336: neither the
// barrier nor the loads' latency is what bounds it.)
// MFMA roles: A = activations (tokens as M), B = weights (rows as N); output lane l holds row l%32
// and tokens 8*(v/4) + 4*(l/32) + v%4.

#include "common.hpp"
#include "gemm_store.hpp"
#include <type_traits>

namespace hkhip {
namespace mg {

typedef int v16i __attribute__((ext_vector_type(16)));
typedef int v4i __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef unsigned short us2 __attribute__((ext_vector_type(2)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef short v8s __attribute__((ext_vector_type(8)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));

// RB: quant-plane bytes per row and super-block; SB: side bytes.
template <int T> struct Fmt;
template <> struct Fmt<HKHIP_Q6_K> {
    static constexpr uint32_t RB = 208, SB = 0; // its f16 d per block goes as the aligned word holding it
    static constexpr int planes = 2;
};
template <> struct Fmt<HKHIP_Q3_K> {
    static constexpr uint32_t RB = 96, SB = 16;
    static constexpr int planes = 1;
};
template <> struct Fmt<HKHIP_Q2_K> {
    static constexpr uint32_t RB = 64, SB = 20;
    static constexpr int planes = 1;
};
template <> struct Fmt<HKHIP_Q4_K> {
    static constexpr uint32_t RB = 144, SB = 0;
    static constexpr int planes = 2;
};
template <> struct Fmt<HKHIP_Q5_K> {
    static constexpr uint32_t RB = 176, SB = 0;
    static constexpr int planes = 2;
};
// Formats with a min per 32 weights.
template <int T> constexpr bool has_mins = T == HKHIP_Q4_K || T == HKHIP_Q5_K;

// Activations of one super-block: chunk c of token t at c ^ (t & 15), token scales, and (Q2_K) the
// tokens' sixteen 16-value sums.
template <int T, int TOK> struct ASlot {
    int8_t a[TOK * 256];
    float da[(TOK + 63) / 64 * 64];
    int16_t bs[T == HKHIP_Q2_K || has_mins<T> ? TOK * 16 : 8]; // Q4_K, Q5_K: k_mb's 16 bf16
};
// One wave's 32 rows of one super-block.
template <int T> struct WSlot {
    uint8_t q[32 * Fmt<T>::RB];
    uint8_t s[T == HKHIP_Q6_K ? 256 : Fmt<T>::SB ? (32 * Fmt<T>::SB + 1023) / 1024 * 1024 : 16];
};
// Two workgroups share a CU's LDS and SIMDs in the tiles of four waves with at most two K slices.
template <int NW, int KS> constexpr int resident() { return NW * KS < 8 && KS < 4 ? 2 : 1; }
// Weight buffers per wave: two, so that the next block's loads go out at the start of a step, for the
// 32-token tiles, whose steps are too short for them otherwise, and for Q4_K (6144 x 14336 at 512 tokens 139
// -> 131 us; the other formats' larger tiles measured the same or, Q3_K, up to 10 % slower so), where
// they fit.
template <int T, int NW, int TT, int KS> constexpr int wbufs() {
    return (TT == 1 || T == HKHIP_Q4_K) &&
                   sizeof(ASlot<T, 32 * TT>) * 2 * KS + sizeof(WSlot<T>) * 2 * KS * NW <= 160 * 1024 / resident<NW, KS>()
               ? 2
               : 1;
}
template <int T, int NW, int TT, int KS> struct Smem {
    ASlot<T, 32 * TT> a[KS][2];
    WSlot<T> w[KS * NW][wbufs<T, NW, TT, KS>()];
};

struct MgArgs {
    const uint8_t *w;
    const uint8_t *ws; // side plane
    uint32_t rows, cols, n;
    const int8_t *aqs;
    const float *ad;
    const int16_t *abs;
    const uint8_t *amb; // k_mb: per token and super-block 64*u and v of its sub-block sums as bf16
    float *y;
    const float *bias;
    int mode;
    int wide; // y 16-byte aligned and rows a multiple of 4: whole tiles go out as 16-byte stores
    uint32_t rblocks, tblocks;
};

__device__ __forceinline__ uint4 ld16(const void *p) { return *reinterpret_cast<const uint4 *>(p); }
__device__ __forceinline__ uint32_t pk_mul(uint32_t a, uint32_t b) {
    return __builtin_bit_cast(uint32_t, __builtin_bit_cast(us2, a) * __builtin_bit_cast(us2, b));
}

// One lane's share of a super-block (its row's half h: 16 weights of every 32), raw.
template <int T> struct Raw;
template <> struct Raw<HKHIP_Q6_K> {
    uint4 ql[2][2], qh[2], sc;
    uint32_t d;
};
template <> struct Raw<HKHIP_Q3_K> {
    uint4 q[2], hm, side; // side: scales[12], d
};
template <> struct Raw<HKHIP_Q4_K> {
    uint4 hd, q[4];
};
template <> struct Raw<HKHIP_Q5_K> {
    uint4 hd, q[4], x; // x: the fifth bits
};
template <> struct Raw<HKHIP_Q2_K> {
    uint4 q[2];
    uint32_t sc[4], dm;
};

template <int T, int NW, int TT, int KS>
__global__ __launch_bounds__(NW * KS * 64, (NW * KS * resident<NW, KS>() / 4)) void mmg_kernel(MgArgs a) {
    using F = Fmt<T>;
    constexpr int TOK = 32 * TT;
    constexpr bool q6 = T == HKHIP_Q6_K, q3 = T == HKHIP_Q3_K, q2 = T == HKHIP_Q2_K, q4 = T == HKHIP_Q4_K,
                   q5 = T == HKHIP_Q5_K, km = has_mins<T>;
    __shared__ __attribute__((aligned(16))) Smem<T, NW, TT, KS> S;
    const uint32_t tid = threadIdx.x, lane = tid & 63;
    const uint32_t wall = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t ks = wall / NW, wave = wall % NW; // K slice, row wave within the slice
    const uint32_t h = lane >> 5, j = lane & 31;
    const uint32_t K = a.cols, nsb = K / 256;

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

    // ---- direct loads: per-lane 32-bit offsets from uniform bases (mmg_supports checks the range) ----
    constexpr uint32_t TPW = TOK / NW; // token rows per wave
    static_assert(TPW % 4 == 0, "token rows per wave");
    uint32_t aoff[TPW / 4];
#pragma unroll
    for (uint32_t i = 0; i < TPW / 4; i++) {
        const uint32_t tl = TPW * wave + 4 * i + lane / 16;
        aoff[i] = clamp_tok(t0 + tl) * K + 16 * ((lane % 16) ^ (tl & 15));
    }
    // Token scales: wave m < TOK/64 loads tokens 64m..; Q2_K's sums: wave m loads tokens 32m...
    const uint32_t doff = clamp_tok(t0 + 64 * wave + lane) * nsb * 4;
    const uint32_t boff = clamp_tok(t0 + 32 * wave + lane / 2) * nsb * 32 + 16 * (lane & 1); // 32 bytes per super-block
    auto issue_a = [&](uint32_t sb, ASlot<T, TOK> &A) {
        const int8_t *ga = a.aqs + 256 * sb;
#pragma unroll
        for (uint32_t i = 0; i < TPW / 4; i++) load_lds16(ga, aoff[i], &A.a[(TPW * wave + 4 * i) * 256]);
        if (64 * wave < uint32_t(TOK)) load_lds4(reinterpret_cast<const uint8_t *>(a.ad) + 4 * sb, doff, &A.da[64 * wave]);
        if constexpr (q2 || km) {
            const uint8_t *gb = km ? a.amb : reinterpret_cast<const uint8_t *>(a.abs);
#pragma unroll
            for (uint32_t b = 0; b < (TT + NW - 1) / NW; b++) {
                const uint32_t m = wave + NW * b;
                const uint32_t o = b == 0 ? boff : clamp_tok(t0 + 32 * m + lane / 2) * nsb * 32 + 16 * (lane & 1);
                if (m < uint32_t(TT)) load_lds16(gb + 32 * sb, o, &A.bs[512 * m]);
            }
        }
    };
    // Weights: the wave's area is its 32 rows' RB bytes back to back, 1 KB (64 lanes x 16 bytes) per
    // load; the last part of a KB goes as words (Q6_K) or fills it exactly.
    constexpr uint32_t W16 = 32 * F::RB / 1024, W4 = (32 * F::RB - 1024 * W16) / 256;
    static_assert(1024 * W16 + 256 * W4 == 32 * F::RB, "weight pieces");
    uint32_t woff[W16 + W4];
#pragma unroll
    for (uint32_t i = 0; i < W16; i++) {
        const uint32_t P = 64 * i + lane;
        woff[i] = clamp_row(rw0 + P / (F::RB / 16)) * nsb * F::RB + 16 * (P % (F::RB / 16));
    }
#pragma unroll
    for (uint32_t i = 0; i < W4; i++) {
        const uint32_t Wd = 256 * W16 + 64 * i + lane;
        woff[W16 + i] = clamp_row(rw0 + Wd / (F::RB / 4)) * nsb * F::RB + 4 * (Wd % (F::RB / 4));
    }
    const uint32_t srow = clamp_row(myrow);
    // Side data: Q6_K the word holding the row's f16 d (lanes 32-63 repeat lanes 0-31); Q3_K 16 bytes
    // per row, likewise; Q2_K 20 bytes per row as words, word e = 64*i + lane of the 160 (the lanes
    // past them repeat the last).
    uint32_t soff[q2 ? 3 : 1];
    if constexpr (q2) {
#pragma unroll
        for (uint32_t i = 0; i < 3; i++) {
            const uint32_t e = 64 * i + lane < 160 ? 64 * i + lane : 159;
            soff[i] = clamp_row(rw0 + e / 5) * nsb * 20 + 4 * (e % 5);
        }
    } else {
        soff[0] = q6 ? srow * nsb : srow * nsb * 16; // (unused by Q4_K and Q5_K)
    }
    constexpr int WB = wbufs<T, NW, TT, KS>();
    auto issue_w = [&](uint32_t sb, WSlot<T> &W) {
        const uint8_t *gw = a.w + uint64_t(sb) * F::RB;
#pragma unroll
        for (uint32_t i = 0; i < W16; i++) load_lds16(gw, woff[i], &W.q[1024 * i]);
#pragma unroll
        for (uint32_t i = 0; i < W4; i++) load_lds4(gw, woff[W16 + i], &W.q[1024 * W16 + 256 * i]);
        if constexpr (q6) {
            load_lds4(a.ws, ((soff[0] + sb) >> 1) << 2, &W.s[0]);
        } else if constexpr (q3) {
            load_lds16(a.ws + 16 * sb, soff[0], &W.s[0]);
        } else if constexpr (q2) {
#pragma unroll
            for (uint32_t i = 0; i < 3; i++) load_lds4(a.ws + 20 * sb, soff[i], &W.s[256 * i]);
        }
    };

    v16f acc[TT];
#pragma unroll
    for (int t = 0; t < TT; t++)
#pragma unroll
        for (int v = 0; v < 16; v++) acc[t][v] = 0.0f;

    // Step st of slice ks is super-block ks + KS*st (loads past the end repeat the last one).
    const uint32_t nst = (nsb + KS - 1) / KS;
    auto sb_of = [&](uint32_t st) {
        const uint32_t sb = ks + KS * st;
        return sb < nsb ? sb : nsb - 1;
    };
    issue_a(sb_of(0), S.a[ks][0]);
    issue_w(sb_of(0), S.w[wall][0]);
    __builtin_amdgcn_s_waitcnt(0x0F70); // vmcnt(0)
    __syncthreads();

    const uint32_t sw = j & 15;
    auto step = [&](uint32_t buf, uint32_t st) {
        ASlot<T, TOK> &A = S.a[ks][buf];
        const uint32_t sb = sb_of(st);
        const WSlot<T> &W = S.w[wall][WB == 2 ? buf : 0];
        const bool more = st + 1 < nst;
        if (more) {
            issue_a(sb_of(st + 1), S.a[ks][buf ^ 1]);
            if constexpr (WB == 2) issue_w(sb_of(st + 1), S.w[wall][buf ^ 1]);
        }
        // This lane's row half, raw; then the buffer is free for the next super-block.
        Raw<T> R;
        const uint8_t *blk = &W.q[F::RB * j];
        if constexpr (q6) {
#pragma unroll
            for (int n = 0; n < 2; n++) {
#pragma unroll
                for (int pp = 0; pp < 2; pp++) R.ql[n][pp] = ld16(blk + 64 * n + 32 * pp + 16 * h);
                R.qh[n] = ld16(blk + 128 + 32 * n + 16 * h);
            }
            R.sc = ld16(blk + 192);
            R.d = *reinterpret_cast<const uint32_t *>(&W.s[4 * j]);
        } else if constexpr (q3) {
            R.hm = ld16(blk + 16 * h);
            R.q[0] = ld16(blk + 32 + 16 * h);
            R.q[1] = ld16(blk + 64 + 16 * h);
            R.side = ld16(&W.s[16 * j]);
        } else if constexpr (km) {
            R.hd = ld16(blk);
#pragma unroll
            for (int p = 0; p < 4; p++) R.q[p] = ld16(blk + (q5 ? 48 : 16) + 32 * p + 16 * h);
            if constexpr (q5) R.x = ld16(blk + 16 + 16 * h);
        } else {
            R.q[0] = ld16(blk + 16 * h);
            R.q[1] = ld16(blk + 32 + 16 * h);
            const uint32_t *sd = reinterpret_cast<const uint32_t *>(&W.s[20 * j]);
#pragma unroll
            for (int i = 0; i < 4; i++) R.sc[i] = sd[i];
            R.dm = sd[4];
        }
        if constexpr (WB == 1) {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); // the reads are done: the bytes may be overwritten
            if (more) issue_w(sb_of(st + 1), S.w[wall][0]);
        }
        if (KS > 1 && ks + KS * st >= nsb) { // a slice past its last super-block keeps its loads in step
            __builtin_amdgcn_s_waitcnt(0x0F70);
            __syncthreads();
            return;
        }

        // ---- operands: chunk c = 32 weights, this lane's 16 of them ----
        v4i P[F::planes][8];
        float d;
        v8h mn;           // Q2_K: mins of groups 8h..8h+7
        v8bf mb;          // Q4_K, Q5_K: the sub-blocks' mins
        uint32_t scl = 0, sch = 0; // Q4_K, Q5_K: the sub-blocks' scales, a byte each
        float ndmin = 0.0f;
        if constexpr (q6) {
            d = 0.25f * f16_bits_to_f32(((soff[0] + sb) & 1) ? R.d >> 16 : R.d & 0xFFFF);
        } else if constexpr (q3) {
            d = -f16_bits_to_f32(R.side.w & 0xFFFF);
        } else if constexpr (km) { // the word unpack of vecdot.zig:461-474
            const uint32_t k1 = 0x3f3f3f3fu, k2 = 0x0f0f0f0fu, k3 = 0x03030303u;
            scl = R.hd.y & k1;
            sch = (R.hd.w & k2) | (((R.hd.y >> 6) & k3) << 4);
            const uint32_t mnl = R.hd.z & k1, mnh = ((R.hd.w >> 4) & k2) | (((R.hd.z >> 6) & k3) << 4);
            uint32_t w[4];
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const uint32_t src = q < 2 ? mnl : mnh, sh = 16 * (q & 1);
                const float e = (float)((src >> sh) & 0xFF), o = (float)((src >> (sh + 8)) & 0xFF);
                w[q] = __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, o), __builtin_bit_cast(uint32_t, e), 0x07060302u);
            }
            mb = __builtin_bit_cast(v8bf, make_uint4(w[0], w[1], w[2], w[3]));
            d = f16_bits_to_f32(R.hd.x & 0xFFFF);
            ndmin = -f16_bits_to_f32(R.hd.x >> 16);
        } else {
            const uint32_t m0 = h ? R.sc[2] : R.sc[0], m1 = h ? R.sc[3] : R.sc[1];
#pragma unroll
            for (int i = 0; i < 8; i++) mn[i] = (_Float16)(unsigned short)(((i < 4 ? m0 : m1) >> (8 * (i % 4) + 4)) & 0x0F);
            d = f16_bits_to_f32(R.dm & 0xFFFF);
            ndmin = -f16_bits_to_f32(R.dm >> 16);
        }
        // Planes of chunk c, words i0 .. i1.
        auto build = [&](auto cc) {
            constexpr int c = decltype(cc)::value, n = c / 4, p = c % 4;
            if constexpr (q6) {
                // Group 2c + h of chunk c = 4n + p is ql bytes 64n + 32(p&1) + 16h.. (nibble p>>1), qh
                // bytes 128 + 32n + 16h.. (bits 2p), scale byte 192 + 8n + 2p + h (dequant.zig's Q6_K order).
                const uint32_t scs[4] = {R.sc.x, R.sc.y, R.sc.z, R.sc.w};
                constexpr uint32_t sbyte = 8 * n + 2 * p; // + h
                const int sc = int(int8_t((scs[sbyte / 4] >> (8 * (sbyte % 4) + 8 * h)) & 0xFF));
                const uint32_t m = q6k_m(sc), k = q6k_k(sc);
                const uint4 l = R.ql[n][p & 1], hq = R.qh[n];
                const uint32_t qlw[4] = {l.x, l.y, l.z, l.w}, qhw[4] = {hq.x, hq.y, hq.z, hq.w};
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const uint32_t q = ((qlw[i] >> (4 * (p >> 1))) & 0x0F0F0F0Fu) | (((qhw[i] >> (2 * p)) & 0x03030303u) << 4);
                    int hp, lp;
                    q6k_planes(q, m, k, hp, lp);
                    P[0][c][i] = hp;
                    P[F::planes - 1][c][i] = lp;
                }
            } else if constexpr (q3) {
                // qs bytes 32n + 16h.. bits 2p, hmask bytes 16h.. bit c, scale index 2c + h: low nibble
                // of byte (2c + h) % 8 (c < 4) or its high nibble, top two bits from byte 8 + (2c + h) % 4
                // (q3kScales, dequant.zig:114-128).
                const uint32_t hw[4] = {R.hm.x, R.hm.y, R.hm.z, R.hm.w};
                const uint32_t nib = ((p < 2 ? R.side.x : R.side.y) >> (16 * (p % 2) + 4 * n + 8 * h)) & 0x0F;
                const uint32_t top = (R.side.z >> (16 * (p % 2) + 2 * (c / 2) + 8 * h)) & 3;
                const uint32_t s2 = (((nib | (top << 4)) - 32u) & 0xFFFFu) * 0x00010001u; // sc - 32 in both halves
                // The eight products -sc*(u - 4), u = 0..7, as bytes.
                const uint32_t p01 = pk_mul(s2, 0x00030004u), p23 = pk_mul(s2, 0x00010002u);
                const uint32_t p45 = pk_mul(s2, 0xFFFF0000u), p67 = pk_mul(s2, 0xFFFDFFFEu);
                const uint32_t T0 = __builtin_amdgcn_perm(p23, p01, 0x06040200u);
                const uint32_t T1 = __builtin_amdgcn_perm(p67, p45, 0x06040200u);
                const uint4 q4 = R.q[n];
                const uint32_t qw[4] = {q4.x, q4.y, q4.z, q4.w};
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const uint32_t hb = (c >= 2 ? hw[i] >> (c >= 2 ? c - 2 : 0) : hw[i] << (c < 2 ? 2 - c : 0)) & 0x04040404u;
                    P[0][c][i] = int(__builtin_amdgcn_perm(T1, T0, ((qw[i] >> (2 * p)) & 0x03030303u) | hb));
                }
            } else if constexpr (km) {
                // Sub-block c: nibble c % 2 of qs bytes 32(c/2) + 16h.., fifth bit c of qh bytes 16h...
                const uint32_t sc = ((c < 4 ? scl : sch) >> (8 * (c % 4))) & 0xFF;
                const uint4 q4v = R.q[c / 2];
                const uint32_t qw[4] = {q4v.x, q4v.y, q4v.z, q4v.w};
                if constexpr (q4) { // sc = 8*sh + sl: planes sh*q and sl*q, each at most 105
                    const uint32_t fh = (sc >> 3) * 0x00010001u, fl = (sc & 7) * 0x00010001u;
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const uint32_t q = (qw[i] >> (4 * (c % 2))) & 0x0F0F0F0Fu;
                        P[0][c][i] = int(pk_mul(q, fh));
                        P[F::planes - 1][c][i] = int(pk_mul(q, fl));
                    }
                } else { // sc*q <= 1953 = 256*H + L
                    const uint4 x = R.x;
                    const uint32_t xw[4] = {x.x, x.y, x.z, x.w}, m = sc * 0x00010001u;
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const uint32_t b5 = (c > 4 ? xw[i] >> (c > 4 ? c - 4 : 0) : xw[i] << (c < 4 ? 4 - c : 0)) & 0x10101010u;
                        int hp, lp;
                        q6k_planes(((qw[i] >> (4 * (c % 2))) & 0x0F0F0F0Fu) | b5, m, 0x00800080u, hp, lp);
                        P[0][c][i] = hp;
                        P[F::planes - 1][c][i] = lp;
                    }
                }
            } else {
                // qs bytes 32n + 16h.. bits 2p, scale byte 2c + h (dequant.zig:80-112).
                const uint32_t sc = (R.sc[c / 2] >> (16 * (c % 2) + 8 * h)) & 0x0F;
                const uint4 q4 = R.q[n];
                const uint32_t qw[4] = {q4.x, q4.y, q4.z, q4.w};
#pragma unroll
                for (int i = 0; i < 4; i++) P[0][c][i] = int(pk_mul((qw[i] >> (2 * p)) & 0x03030303u, sc * 0x00010001u));
            }
        };

        const int8_t *abase = &A.a[j * 256];
        v4i av[4];
        // Chunk c of tile t (c >= 8: of the next tile) into the ring of four operands.
        auto load_a = [&](int t, int c) {
            av[c % 4] = *reinterpret_cast<const v4i *>(abase + 32 * (t + c / 8) * 256 + 16 * ((2 * (c % 8) + h) ^ sw));
        };
#pragma unroll
        for (int c = 0; c < 4; c++) load_a(0, c);
        v16i comb = {};
        v16f jt = {}; // Q2_K: J; Q4_K, Q5_K: d*I - dmin*J
        // Outputs 2c, 2c + 1 of tile t's update: tokens 32t + 8g + 4h + (0..3), g = c / 2.
        auto update = [&](int t, int c) {
            const float2 dv = *reinterpret_cast<const float2 *>(&A.da[32 * t + 8 * (c / 2) + 4 * h + 2 * (c % 2)]);
            const float ds[2] = {dv.x, dv.y};
#pragma unroll
            for (int e = 0; e < 2; e++) {
                const int v = 2 * c + e;
                if constexpr (km)
                    acc[t][v] = fmaf(jt[v], ds[e], acc[t][v]);
                else if constexpr (q2)
                    acc[t][v] = fmaf(fmaf((float)comb[v], d, ndmin * jt[v]), ds[e], acc[t][v]);
                else
                    acc[t][v] = fmaf((float)comb[v], d * ds[e], acc[t][v]);
            }
        };
        build(std::integral_constant<int, 0>{});
        // The super-block's tiles one after another, as one interleaved stream: beside tile 0's MFMAs
        // the next chunk's planes are built, beside tile t's the update of tile t - 1 runs and the
        // operands of tile t + 1 are read into the registers just used.
#pragma unroll
        for (int t = 0; t < TT; t++) {
            v16i s0 = {}, s1 = {};
            auto chunk = [&](auto cc) {
                constexpr int c = decltype(cc)::value;
                s0 = __builtin_amdgcn_mfma_i32_32x32x32_i8(av[c % 4], P[0][c], s0, 0, 0, 0);
                if (t == 0) {
                    if constexpr (c < 7) build(std::integral_constant<int, c + 1>{});
                } else {
                    update(t - 1, c);
                }
                if constexpr (F::planes == 2) s1 = __builtin_amdgcn_mfma_i32_32x32x32_i8(av[c % 4], P[F::planes - 1][c], s1, 0, 0, 0);
                if (c < 4 || t + 1 < TT) load_a(t, c + 4);
                if constexpr (TT > 1 || !km) __builtin_amdgcn_sched_barrier(0);
            };
            chunk(std::integral_constant<int, 0>{});
            chunk(std::integral_constant<int, 1>{});
            chunk(std::integral_constant<int, 2>{});
            chunk(std::integral_constant<int, 3>{});
            chunk(std::integral_constant<int, 4>{});
            chunk(std::integral_constant<int, 5>{});
            chunk(std::integral_constant<int, 6>{});
            chunk(std::integral_constant<int, 7>{});
            if constexpr (q2) {
                const v8s b16 = *reinterpret_cast<const v8s *>(&A.bs[16 * (32 * t + j) + 8 * h]);
                v8h bh;
#pragma unroll
                for (int i = 0; i < 8; i++) bh[i] = (_Float16)b16[i];
                jt = __builtin_amdgcn_mfma_f32_32x32x16_f16(bh, mn, v16f{}, 0, 0, 0);
            }
            constexpr int shift = q4 ? 3 : 8;
#pragma unroll
            for (int v = 0; v < 16; v++) s0[v] = F::planes == 2 ? (s0[v] << shift) + s1[v] : s0[v];
            if constexpr (km) {
                __builtin_amdgcn_sched_barrier(0); // s1's registers are free for J's tile
                const uint4 b = ld16(&A.bs[16 * (32 * t + j) + 8 * h]);
                const v16f jm = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, b), mb, v16f{}, 0, 0, 0);
#pragma unroll
                for (int v = 0; v < 16; v++) jt[v] = fmaf((float)s0[v], d, ndmin * jm[v]);
            } else {
                comb = s0;
            }
        }
#pragma unroll
        for (int c = 0; c < 8; c++) update(TT - 1, c);
        __builtin_amdgcn_s_waitcnt(0x0F70); // vmcnt(0): the next super-block is in LDS
        __syncthreads();
    };
    for (uint32_t st = 0; st < nst; st += 2) {
        step(0, st);
        if (st + 1 < nst) step(1, st + 1);
    }

    // The loads of the last step have landed and every wave is past its barrier: the LDS is free. (Storing
    // each tile beside the next one's MFMAs in the last step spilled 200-330 registers in the large tile.)
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

template <int T, int NW, int TT, int KS> hipError_t launch_cfg(const MgArgs &a0, hipStream_t s) {
    static_assert(sizeof(Smem<T, NW, TT, KS>) <= 160 * 1024, "LDS");
    MgArgs a = a0;
    a.rblocks = (a.rows + 32 * NW - 1) / (32 * NW);
    a.tblocks = (a.n + 32 * TT - 1) / (32 * TT);
    hipLaunchKernelGGL((mmg_kernel<T, NW, TT, KS>), dim3(a.rblocks * a.tblocks), dim3(NW * KS * 64), 0, s, a);
    return hipGetLastError();
}

// The tile whose rounds of workgroups cost least. A round is what is resident at once: one workgroup per
// CU for the tiles of eight waves (LDS), two for those of four, whose barriers then drift apart. A
// round costs its super-block steps and its ends (launch or refill, sum over slices, stores), whatever
// the grid; a two-resident tile's last half round leaves its workgroups a SIMD per wave and costs less.
// In tenths of a us for Q4_K, measured at 1024-14336 rows, K 1024 and 4096, 36-700 tokens (a round of K 4096:
// <8,4,1> 60-66 us, <4,2,2> 22-26, <4,2,1> 41 (half 28), <2,1,4> 10-11, <2,1,2> 18 (half 11), <1,1,4> 8.6); the
// other formats' rounds are in the same ratios within 15 %.
template <int T> hipError_t launch_fmt(const MgArgs &a, hipStream_t s) {
    constexpr uint32_t CUS = 256;
    struct Tile {
        uint32_t nw, tt, ks, resident, step, half; // step, half: tenths of a us per super-block step
    };
    const Tile tiles[6] = {{8, 4, 1, 1, 37, 37}, {4, 2, 2, 1, 27, 27}, {4, 2, 1, 2, 25, 16},
                           {2, 1, 4, 1, 22, 22}, {2, 1, 2, 2, 21, 12}, {1, 1, 4, 1, 18, 18}};
    const uint32_t nsb = a.cols / 256;
    uint64_t best = ~0ull;
    int pick = 0;
    for (int i = 0; i < 6; i++) {
        const Tile &c = tiles[i];
        const uint64_t grid = uint64_t((a.rows + 32 * c.nw - 1) / (32 * c.nw)) * ((a.n + 32 * c.tt - 1) / (32 * c.tt));
        const uint64_t cap = CUS * c.resident, rest = grid % cap, steps = (nsb + c.ks - 1) / c.ks;
        const uint64_t ends = c.ks > 1 ? 15 : 10;
        const uint64_t cost = grid / cap * (steps * c.step + ends) + (rest == 0 ? 0 : steps * (rest <= CUS ? c.half : c.step) + ends);
        if (cost < best) best = cost, pick = i;
    }
    switch (pick) {
    case 0: return launch_cfg<T, 8, 4, 1>(a, s);
    case 1: return launch_cfg<T, 4, 2, 2>(a, s);
    case 2: return launch_cfg<T, 4, 2, 1>(a, s);
    case 3: return launch_cfg<T, 2, 1, 4>(a, s);
    case 4: return launch_cfg<T, 2, 1, 2>(a, s);
    default: return launch_cfg<T, 1, 1, 4>(a, s);
    }
}

} // namespace mg

bool mmg_supports(int t, uint32_t rows, uint32_t cols, uint32_t n) {
    if (t != HKHIP_Q6_K && t != HKHIP_Q3_K && t != HKHIP_Q2_K && t != HKHIP_Q4_K && t != HKHIP_Q5_K) return false;
    if (cols % 256 != 0 || rows == 0 || n == 0) return false;
    // 32-bit per-lane byte offsets: quant plane, side plane and activations.
    const WLayout W = weight_layout(t, rows, cols);
    return W.total < (1ull << 32) && uint64_t(n) * cols < (1ull << 32);
}

hipError_t launch_mmg(int t, const uint8_t *w, uint32_t rows, uint32_t cols, const uint8_t *xq, uint32_t n, float *y,
                      const float *bias, int mode, hipStream_t s) {
    if (!mmg_supports(t, rows, cols, n)) return hipErrorInvalidValue;
    const WLayout W = weight_layout(t, rows, cols);
    const ActLayout A = act_layout(n, cols);
    mg::MgArgs a{};
    a.w = w;
    a.ws = w + W.scale_off;
    a.rows = rows;
    a.cols = cols;
    a.n = n;
    a.aqs = reinterpret_cast<const int8_t *>(xq + A.k_qs);
    a.ad = reinterpret_cast<const float *>(xq + A.k_d);
    a.abs = reinterpret_cast<const int16_t *>(xq + A.k_bs);
    a.amb = xq + A.k_mb;
    a.y = y;
    a.bias = bias;
    a.mode = mode;
    a.wide = (reinterpret_cast<uintptr_t>(y) % 16 == 0 && rows % (mode == HKHIP_SILU_MUL ? 8 : 4) == 0) ? 1 : 0;
    switch (t) {
    case HKHIP_Q6_K: return mg::launch_fmt<HKHIP_Q6_K>(a, s);
    case HKHIP_Q4_K: return mg::launch_fmt<HKHIP_Q4_K>(a, s);
    case HKHIP_Q5_K: return mg::launch_fmt<HKHIP_Q5_K>(a, s);
    case HKHIP_Q3_K: return mg::launch_fmt<HKHIP_Q3_K>(a, s);
    default: return mg::launch_fmt<HKHIP_Q2_K>(a, s);
    }
}

} // namespace hkhip
