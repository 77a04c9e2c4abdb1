// NVFP4 rows against at most 16 activation rows on the bf16 matrix cores, gfx950.
//
// A few rows of one expert stream all its weights once, so what counts is that nothing but
// the stream and the decoding is on the path. The K dimension is split over the waves of a
// block and each wave keeps its slice of the activations in registers, as MFMA A operands in
// their bf16 terms, for every weight row it meets: no activation passes through LDS in the
// loop and no wave waits for another there. (Activations staged through LDS per K block, with
// the weights' loads in the operand layout or transposed through LDS, took 225-245 us for 512
// experts of 640 x 2560 with 10 rows each, whatever the occupancy: the loop was a chain of LDS
// reads, decoding and barriers. This form takes 147 to 158.)
//
//   - slice s of KS takes K columns [32 ST s, 32 ST (s + 1)); lane (r, q) (r = lane % 16, q =
//     lane / 16) holds the 8 ST columns from 32 ST s + 8 ST q on, of activation row r and of
//     weight row r: at step st both sides supply columns 8 st .. 8 st + 7 of the lane's run,
//     so every product pairs the same k and the steps add up to the plain dot product;
//   - a lane's run is 4 ST contiguous code bytes of its row and ST / 2 whole scale groups;
//     a group past K scales to 0;
//   - a wave's 16-row subtiles follow each other, four subtiles' loads in flight, coalesced and
//     then through a wave's own LDS area into the operand layout (loaded in that layout, 16
//     bytes of each of 64 lines an instruction, the stream alone took 137 us against 104);
//   - a subtile is ST decodings of 8 codes (e2m1 -> f32, times the e4m3 group scale, -> bf16:
//     exact) and TERMS x ST MFMAs, one accumulator a term;
//   - the slices' sums meet in LDS, 8 subtiles a wave at a time, added in slice order.
#pragma once

#include "stream.hpp"

namespace oom {

typedef __bf16 n4bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 n4bf16x2 __attribute__((ext_vector_type(2)));
typedef float n4f32x2 __attribute__((ext_vector_type(2)));
typedef float n4f4 __attribute__((ext_vector_type(4)));

// Two f32 values as packed bf16 (v_cvt_pk_bf16_f32, round to nearest even; exact for the weights
// here, which are bf16 values).
__device__ __forceinline__ uint32_t n4_cvt(float lo, float hi) {
    const n4f32x2 v = {lo, hi};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, n4bf16x2));
}

// Eight codes of one scale group (byte i: columns 2 i, 2 i + 1) times its scale, as bf16, exactly.
__device__ __forceinline__ n4bf16x8 n4_decode8(uint32_t cw, float sc) {
    const auto p0 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(cw, 1.0f, 0);
    const auto p1 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(cw, 1.0f, 1);
    const auto p2 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(cw, 1.0f, 2);
    const auto p3 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(cw, 1.0f, 3);
    return __builtin_bit_cast(n4bf16x8, make_uint4(n4_cvt(p0[0] * sc, p0[1] * sc), n4_cvt(p1[0] * sc, p1[1] * sc),
                                                   n4_cvt(p2[0] * sc, p2[1] * sc), n4_cvt(p3[0] * sc, p3[1] * sc)));
}

// The lane's activations as A operands: columns kq .. of the K floats at `row`. RAG: the run
// may pass K; what lies past it counts as zeros.
template <int TERMS, int ST>
struct RowsX {
    n4bf16x8 t[TERMS][ST];
    template <bool RAG>
    __device__ __forceinline__ void load(const float* row, int kq, int K) {
        const float* p = row + kq;
        // half of the run's loads at a time, all of a half in flight
#pragma unroll
        for (int h = 0; h < 2; h++) {
            float4 v[ST];
#pragma unroll
            for (int i = 0; i < ST; i++) {
                const int c = 4 * (h * ST + i);
                v[i] = *reinterpret_cast<const float4*>(RAG ? row + min(kq + c, K - 4) : p + c);
            }
            if constexpr (RAG) {
#pragma unroll
                for (int i = 0; i < ST; i++) {
                    const bool in = kq + 4 * (h * ST + i) < K;
                    v[i].x = in ? v[i].x : 0.0f;
                    v[i].y = in ? v[i].y : 0.0f;
                    v[i].z = in ? v[i].z : 0.0f;
                    v[i].w = in ? v[i].w : 0.0f;
                }
            }
#pragma unroll
            for (int j = 0; j < ST / 2; j++)
#pragma unroll
                for (int p = 0; p < TERMS; p++) {
                    float4 &a = v[2 * j], &b = v[2 * j + 1];
                    const uint32_t w0 = n4_cvt(a.x, a.y), w1 = n4_cvt(a.z, a.w), w2 = n4_cvt(b.x, b.y),
                                   w3 = n4_cvt(b.z, b.w);
                    t[p][h * (ST / 2) + j] = __builtin_bit_cast(n4bf16x8, make_uint4(w0, w1, w2, w3));
                    if (p + 1 < TERMS) {  // the remainder of a round to nearest: exact
                        a.x -= __uint_as_float(w0 << 16);
                        a.y -= __uint_as_float(w0 & 0xffff0000u);
                        a.z -= __uint_as_float(w1 << 16);
                        a.w -= __uint_as_float(w1 & 0xffff0000u);
                        b.x -= __uint_as_float(w2 << 16);
                        b.y -= __uint_as_float(w2 & 0xffff0000u);
                        b.z -= __uint_as_float(w3 << 16);
                        b.w -= __uint_as_float(w3 & 0xffff0000u);
                    }
                }
        }
    }
};

// LDS of a block: the waves' transposed codes, a batch's scales, the slices' sums.
struct RowsLds {
    __attribute__((aligned(16))) uint8_t codes[NR_WAVES][16 * 176];
    __attribute__((aligned(16))) uint8_t scales[NR_WAVES * 2560];
    n4f4 red[NR_WAVES][NR_BATCH][64];
};

// One projection's weights as a wave reads them: 16-row subtiles of its K slice. Loads are
// coalesced (ST lanes a row's 16 ST bytes, 64 / ST rows an instruction) and reach the operand
// layout through LDS; the batch's scales are one contiguous run a row group, loaded by the
// group's waves together one batch ahead.
template <int ST>
struct RowsW {
    static constexpr int RPI = 64 / ST, NI = (16 + RPI - 1) / RPI;  // rows an instruction, instructions a subtile
    static constexpr int CS = 16 * ST + 16;                         // LDS row stride of the codes
    static constexpr int NSC = 3;                                   // scale loads a lane a batch
    __amdgpu_buffer_rsrc_t cr, sr;
    unsigned crow, coff[NI], soff;
    int K, ks, slice;
    uint8_t *cw, *sb;         // this wave's codes, this row group's scales in LDS
    int cput, cget, sget;     // byte offsets of this lane's pieces
    int groups, sh;
    bool act;
    struct Ld {
        uint4 c[NI];
    };
    uint4 sv[NSC];
    // Codes at byte w_off and scales at s_off of record rec, n rows of K; row0: the group's
    // first row; the wave's place: slice of ks, wave index.
    __device__ __forceinline__ void init(RowsLds& lds, uint64_t rec, int64_t w_off, int64_t s_off, int n, int k, int row0,
                                         int lane, int wave, int slice_, int ks_log) {
        K = k;
        ks = 1 << ks_log;
        slice = slice_;
        cr = uniform_rsrc(rec + w_off, (int)((int64_t)n * K / 2));
        sr = uniform_rsrc(rec + s_off, (int)((int64_t)n * K / 16));
        crow = 8u * K;
        act = lane < RPI * ST;
        const int lr = lane / ST, lc = lane % ST;
#pragma unroll
        for (int i = 0; i < NI; i++)
            coff[i] = act && RPI * i + lr < 16 ? (unsigned)(row0 + RPI * i + lr) * (unsigned)(K / 2) +
                                                     16u * (unsigned)(ST * slice + lc)
                                               : (unsigned)OOB;
        soff = (unsigned)row0 * (unsigned)(K / 16) + 16u * (unsigned)(64 * slice + lane);
        const int r = lane & 15, q = lane >> 4, kq = 32 * ST * slice + 8 * ST * q;
        cw = lds.codes[wave];
        sb = lds.scales + ((wave >> ks_log) << ks_log) * 2560;
        cput = CS * lr + 16 * lc;
        cget = CS * r + 4 * ST * q;
        sget = r * (K / 16) + kq / 16;
        sh = sget & 3;
        sget &= ~3;
        groups = min(max((K - kq) / 16, 0), ST / 2);
    }
    // Loads of subtile i past the first (`on` false, past n and past the part: zeros).
    __device__ __forceinline__ void load(Ld& l, int i, bool on) const {
#pragma unroll
        for (int j = 0; j < NI; j++)
            l.c[j] = ld16(cr, (int)(on && coff[j] != (unsigned)OOB ? coff[j] + crow * (unsigned)i : (unsigned)OOB));
    }
    // Scale loads of the batch that starts i subtiles past the first: the group's 128 rows x
    // K / 16 bytes, 16 a lane and load.
    __device__ __forceinline__ void sload(int i, bool on) {
#pragma unroll
        for (int j = 0; j < NSC; j++)
            sv[j] = ld16(sr, (int)(on && 1024 * (ks * j + slice) < 8 * K
                                       ? soff + (unsigned)K * (unsigned)i + 1024u * (unsigned)(ks * j) : (unsigned)OOB));
    }
    __device__ __forceinline__ void sput(int lane) const {
#pragma unroll
        for (int i = 0; i < NSC; i++) {
            const int at = 16 * (64 * ks * i + 64 * slice + lane);
            if (at < 8 * K) *reinterpret_cast<uint4*>(sb + at) = sv[i];
        }
    }
    // A subtile's codes through LDS into the operand layout (the wave's LDS operations stay in
    // order, so one area serves subtile after subtile), with its scales (subtile i of the batch).
    struct Op {
        uint32_t w[ST], s[2];
    };
    __device__ __forceinline__ void stage(const Ld& l, int i, Op& o) const {
#pragma unroll
        for (int j = 0; j < NI; j++)
            if (act && cput + CS * RPI * j < CS * 16) *reinterpret_cast<uint4*>(cw + cput + CS * RPI * j) = l.c[j];
        wave_lds_order();
#pragma unroll
        for (int j = 0; j < ST / 2; j++) {
            const uint2 v = *reinterpret_cast<const uint2*>(cw + cget + 8 * j);
            o.w[2 * j] = v.x;
            o.w[2 * j + 1] = v.y;
        }
        const uint32_t* sp = reinterpret_cast<const uint32_t*>(sb + sget + K * i);
        o.s[0] = sp[0];
        o.s[1] = sp[1];
        wave_lds_order();
    }
    // x . w of a staged subtile over the wave's slice: lane holds x rows 4 (lane / 16) + j,
    // weight row lane % 16.
    template <int TERMS>
    __device__ __forceinline__ n4f4 dot(const Op& o, const RowsX<TERMS, ST>& x) const {
        const uint32_t(&w)[ST] = o.w;
        const uint32_t sl = o.s[0], sg = o.s[1];
        const uint32_t s0 = __builtin_amdgcn_alignbyte(sg, sl, sh), s1 = sg >> (8 * sh);
        n4f4 acc[TERMS];
#pragma unroll
        for (int gr = 0; gr < ST / 2; gr++) {
            float sc = gr == 0   ? __builtin_amdgcn_cvt_f32_fp8((int)s0, 0)
                       : gr == 1 ? __builtin_amdgcn_cvt_f32_fp8((int)s0, 1)
                       : gr == 2 ? __builtin_amdgcn_cvt_f32_fp8((int)s0, 2)
                       : gr == 3 ? __builtin_amdgcn_cvt_f32_fp8((int)s0, 3)
                                 : __builtin_amdgcn_cvt_f32_fp8((int)s1, 0);
            sc = gr < groups ? sc : 0.0f;
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const int st = 2 * gr + h;
                const n4bf16x8 b = n4_decode8(w[st], sc);
#pragma unroll
                for (int p = 0; p < TERMS; p++)
                    acc[p] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                        x.t[p][st], b, st ? acc[p] : n4f4{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
            }
        }
        n4f4 y = acc[TERMS - 1];  // the smallest terms first
#pragma unroll
        for (int p = TERMS - 2; p >= 0; p--) y += acc[p];
        return y;
    }
};

// The wave's share of a batch's subtiles, each the sum of its 1 << KSL slices in slice order:
// put(subtile of the batch, row groups one after the other; sum).
template <int KSL, typename Put>
__device__ __forceinline__ void rows_meet(const RowsLds& lds, int wave, int lane, Put put) {
    constexpr int KS = 1 << KSL, GROUPS = NR_WAVES >> KSL;
    constexpr int AT = KS < 4 ? KS : 4;  // reads in flight (the registers there are)
#pragma unroll 1
    for (int t = 0; t < GROUPS; t++) {
        const int gs = wave * GROUPS + t;
        const n4f4* p = &lds.red[(gs / NR_BATCH) << KSL][gs % NR_BATCH][lane];
        n4f4 y;
#pragma unroll
        for (int s = 0; s < KS; s += AT) {
            n4f4 v[AT];
#pragma unroll
            for (int i = 0; i < AT; i++) v[i] = p[(s + i) * NR_BATCH * 64];
#pragma unroll
            for (int i = 0; i < AT; i++) y = s + i ? y + v[i] : v[i];
        }
        put(gs, y);
    }
}

}  // namespace oom
