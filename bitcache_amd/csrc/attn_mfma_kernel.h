// Split-KV decode attention with the value phase on the matrix cores (gfx950).
//
// Same work decomposition and partial format as attn_split_kernel
// (attention.hip): grid.x = key split, grid.y = (b, kv head, query-head
// group), 4 wave64 per workgroup, 64-key tiles round-robin over the waves.
//
// Score phase (lane = key): XNOR popcount of the sign words, and the INT4
// residual dot directly on the stored two's-complement nibbles against the
// query in 24-bit fixed point: six balanced int4 digits for v_dot8_i32_i4
// (single heads) or three balanced int8 planes for an int8 MFMA (KMF below),
// of which a tile uses the top 16 bits unless a key's residual scale makes it
// a precise tile.
//
// Value phase: out[e] = sum_s a_s*(2*bit_se - 1) + b_s*n_se with a = p*sv,
// b = p*rs/7.  The V tile (sign bytes and code bytes of 64 keys) is copied to
// LDS with direct buffer loads, then ds_read_b64_tr_b4 transposes 16 keys x 16
// nibbles per 16-lane group so that each lane holds 16 keys of one dimension.
// int8 path (groups up to 4; I8 and R8 below): sign bits in place as int8
// elements, codes as 16 n, four keys per operation, the weights of each head
// as balanced 8-bit digit columns, v_mfma_i32_16x16x64_i8 with exact int32
// sums, flushed into a float bank on rescales.  fp16 path (groups of 8):
// nibbles (u = n + 8, the 8 b_s taken off at
// the end) and sign bits become exact fp16 subnormals (value * 2^(j-24) for
// bit position j < 10) with one mask per pair of keys, left in place (the
// power of two is folded into the weights of odd keys and into the
// accumulator of bit p), and v_mfma_f32_16x16x32_f16 accumulates dims x weight
// columns, (hi, lo) fp16 splits of a and b for each query head of the group;
// the fp32 accumulators are rescaled on running-max changes.
#pragma once

#include <math.h>

#include "attn.h"
#include "encode_row.h"

using bc::AttnArgs;
using bc::kLog2e;
using bc::MODE_ADAPTIVE;
using bc::MODE_BINARY;
using bc::MODE_COMP;
using bc::MODE_MIXED;

namespace {

typedef _Float16 h8_t __attribute__((ext_vector_type(8)));
typedef float f4_t __attribute__((ext_vector_type(4)));
typedef int v2i_t __attribute__((ext_vector_type(2)));
typedef int v4i_t __attribute__((ext_vector_type(4)));
typedef unsigned int v4u_t __attribute__((ext_vector_type(4)));
typedef unsigned int v3u_t __attribute__((ext_vector_type(3)));
typedef unsigned int v2u_t __attribute__((ext_vector_type(2)));
#define LDS_PTR(T, p) ((__attribute__((address_space(3))) T*)(p))

// Word 3 of a gfx9 buffer resource for raw byte-addressed loads (32-bit data
// format, no swizzle; with stride 0 a load past num_records returns zeros).
constexpr int kBufWord3 = 0x00020000;

// D/8 sign bytes at byte offset off of a buffer, as D/32 words: 16-byte loads
// and one of the 4, 8 or 12 bytes left (a row is dword-aligned).
template <int D, int AUX>
__device__ __forceinline__ SignWords<D> buf_signs(__amdgpu_buffer_rsrc_t r, int off) {
    SignWords<D> s;
#pragma unroll
    for (int i = 0; i < D / 128; i++) {
        const v4u_t v = __builtin_amdgcn_raw_buffer_load_b128(r, off + 16 * i, 0, AUX);
        s.w[4 * i + 0] = v[0]; s.w[4 * i + 1] = v[1]; s.w[4 * i + 2] = v[2]; s.w[4 * i + 3] = v[3];
    }
    constexpr int W0 = 4 * (D / 128), NL = D / 32 - W0;   // words left
    if constexpr (NL == 3) {
        const v3u_t v = __builtin_amdgcn_raw_buffer_load_b96(r, off + 4 * W0, 0, AUX);
        s.w[W0] = v[0]; s.w[W0 + 1] = v[1]; s.w[W0 + 2] = v[2];
    } else if constexpr (NL == 2) {
        const v2u_t v = __builtin_amdgcn_raw_buffer_load_b64(r, off + 4 * W0, 0, AUX);
        s.w[W0] = v[0]; s.w[W0 + 1] = v[1];
    } else if constexpr (NL == 1) {
        s.w[W0] = __builtin_amdgcn_raw_buffer_load_b32(r, off + 4 * W0, 0, AUX);
    }
    return s;
}

// The query of the INT4 residual dot as 24-bit fixed point:
// q_int = rint(q / step), step = max|q| / kQIntMax, written as six balanced
// int4 digits (q_int = sum_j d_j 16^j, d_j in [-8, 7]) or three balanced int8
// planes (q_int = p0 + 256 p1 + 65536 p2).  A tile's dots use the top 16 bits
// (digits 2..5, planes 1..2: q_int / 256 within 0.53, i.e. 16-bit fixed point
// of step 256*step) unless a key of the tile could see a score error above
// kPrecNats from it; then the low digits / plane are added (an fp32-level
// error).  kQIntMax leaves room below 7*(16^6 - 1)/15 = 7829367, the largest
// six-digit value, for the rounding of q / step.
constexpr float kQIntMax = 7800000.0f;
constexpr float kPrecNats = 1.0f / 2048.0f;

// How the K codes of a 16-key block are spread over the lanes for the int8
// MFMAs of the residual dot.  A key's row is D/16 units of 16 dims (8 bytes);
// one 16x16x64 MFMA takes four units of 16 keys, lane group q (lanes 16q ..
// 16q + 15, lane l%16 = key) holding one of them.  Whole 128-dim pieces are
// read as 16 bytes per lane (units 8p + 2q and 8p + 2q + 1: two MFMAs); the
// 32, 64 or 96 dims left as 8 bytes per lane (unit 8 kPieces + 4r + q; lane
// groups past the row repeat a unit of it against zero query operands).
template <int D>
struct KBlocks {
    static constexpr int kPieces = D / 128;                          // 16-byte loads
    static constexpr int kLeft = (D % 128) / 16;                     // units left: 0, 2, 4, 6
    static constexpr int kTails = (kLeft + 3) / 4;                   // 8-byte loads
    static constexpr int kLoads = kPieces + kTails;                  // loads of a block
    static constexpr int kMfma = 2 * kPieces + kTails;               // MFMAs of a block
    static constexpr int kWords = 4 * kPieces + 2 * kTails;          // code dwords per lane and block
    // the unit that MFMA m takes from lane group q (D/16 or more: none)
    static __device__ __forceinline__ int unit(int m, int q) {
        return m < 2 * kPieces ? 8 * (m >> 1) + 2 * q + (m & 1) : 8 * kPieces + 4 * (m - 2 * kPieces) + q;
    }
};

template <int D, int G, bool KMF>
struct QDigits {
    uint32_t signs[G][D / 32];
    // v_dot8 operands (per-key and linear code reads)
    int4 digits[KMF ? 1 : G][KMF ? 1 : D / 8];     // .x..w = balanced int4 digits 2..5 of q_int of elements 8w..8w+7 (nibble k = element 8w+k)
    int2 digits_lo[KMF ? 1 : G][KMF ? 1 : D / 8];  // digits 0..1
    // int8 MFMA B operands of the K residual dot: [MFMA][lane] (see the
    // kernel): planes 1, 2 (and plane 0 where the columns hold it), and
    // plane 0 for groups of more than 5 heads
    int4 bq[KMF ? KBlocks<D>::kMfma : 1][KMF ? 64 : 1];
    int4 bq_lo[(KMF && G > 5) ? KBlocks<D>::kMfma : 1][(KMF && G > 5) ? 64 : 1];
    float scale_q[G];             // sequential mean |q| (src/compensated_attention.cu:65-67)
    float dq[G];                  // step of the top 16 bits: 256 * step of q_int
    // bound on a key's score error (nats) from the top-16-bit dot, per unit of
    // its residual scale: 0.53 * max_g dq * D / sqrt(D)
    float prec_bound;
};

// Per-wave LDS, one __shared__ array per role (the compiler tracks LDS
// direct loads per array, so reading staging buffer i or the weights does not
// wait for the direct loads still landing in buffer i+1): V staging buffers
// (tile i is consumed while tile i+1 lands), each the tile's code bytes then
// its sign bytes; the (hi, lo) fp16 weight columns [part][2G][72 slots]; the
// K-side residual dots [64 keys][G] of GQA groups.  The epilogue reduces heads
// in batches through staging buffer 0.  Binary attention stages no codes.
template <int D, int G, bool RES, bool KMF>
struct WaveLds {
    static constexpr int kCodeBytes = RES ? 64 * D / 2 : 0;
    // Sign rows: 64-dim blocks of 8 bytes, as the transposed reads take them.
    // D % 64 == 32: rows padded to kSignStride and copied a dword per lane,
    // the pad words repeating the row's last word (their dims are dropped).
    // Otherwise whole KiB are copied (d = 64 and 192: the last one's second
    // half is unused).
    static constexpr bool kSignPad = D % 64 != 0;
    static constexpr int kSignStride = !kSignPad ? D / 8 : (D == 32 ? 8 : (D == 96 ? 16 : 32));
    static constexpr int kSignBytes = kSignPad ? 64 * kSignStride : (D / 8 + 15) / 16 * 1024;
    static constexpr int kStage = kCodeBytes + kSignBytes;
    // weight columns of 72 slots (64 used): the 16 lanes of a row group read
    // 16-byte runs of 16 columns without LDS bank conflicts
    static constexpr int kColSlots = 72;
    static constexpr int kWeightBytes = 2 * 2 * G * kColSlots * 2;
    static constexpr int kRdInts = KMF ? 64 * G : 4;
    // epilogue: heads per pass through staging buffer 0 ([parts][heads][D] floats)
    static constexpr int kEpiHeads = kStage / ((RES ? 2 : 1) * D * 4) < G ? kStage / ((RES ? 2 : 1) * D * 4) : G;
    static_assert(kEpiHeads >= 1, "staging buffer holds one head's partial sums");
};

// K-side data of one 64-key tile held in registers: sign words and scales of
// the lane's own key, and the lane's code pieces (see the kernel).
template <int D, bool KMF>
struct KRegs {
    static constexpr int kCodeWords = KMF ? 4 * KBlocks<D>::kWords : D / 8;
    SignWords<D> ks;              // (adaptive mode: the stored popcounts instead)
    uint32_t pcw[4];              // adaptive: the G popcounts of the lane's key
    uint32_t kc[kCodeWords];      // (adaptive mode: gathered later, selected keys)
    uint16_t sk, svv, rsk, rsv;   // raw fp16 scales (converted at use, so the
                                  // loads of the next tile are not waited on)
    uint32_t sel;                 // adaptive: bit g = head g selected the lane's key
};

// Eight INT4 codes of two dwords as the int8 MFMA operand 16*n (signed): low
// nibbles shifted up, high nibbles masked in place.
__device__ __forceinline__ v4i_t codes_i8(uint32_t x0, uint32_t x1) {
    return v4i_t{(int)((x0 << 4) & 0xF0F0F0F0u), (int)(x0 & 0xF0F0F0F0u), (int)((x1 << 4) & 0xF0F0F0F0u),
                 (int)(x1 & 0xF0F0F0F0u)};
}

// x through an empty asm: the compiler cannot split or re-associate it
__device__ __forceinline__ int opaque_int(int x) {
    asm volatile("" : "+v"(x));
    return x;
}

// (scale_q * scale_k) * (2pc - d)  (src/xnor_dot.cuh:30), two rounded products
// in every instance: a step that appends and a call that attends give the
// same bits
__device__ __forceinline__ float xnor_score(float scale_q, float scale_k, float mq) {
#pragma clang fp contract(off)
    return (scale_q * scale_k) * mq;
}

// 1 / f of a power of two between 2^-126 and 2^126
__device__ __forceinline__ float pow2_inv(float f) {
    return __builtin_bit_cast(float, 0x7F000000u - __builtin_bit_cast(uint32_t, f));
}

// a wave-uniform float, in a scalar register
__device__ __forceinline__ float uniform_f(float f) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, f)));
}

__device__ __forceinline__ uint16_t f2h_bits(float f) { return __builtin_bit_cast(uint16_t, (_Float16)f); }
__device__ __forceinline__ float h_bits2f(uint16_t h) { return (float)__builtin_bit_cast(_Float16, h); }

// slot position of key k (0..63) inside the weight columns: for MFMA half mh of
// group g4, slots (2t, 2t+1) hold keys (t, t+4) of the 8-key run.
__device__ __forceinline__ int slot_of(int k) {
    const int g4 = k >> 4, mh = (k >> 3) & 1, r = k & 7;
    return 16 * g4 + 8 * mh + ((r & 3) << 1) + (r >> 2);
}

// Slot of key k in the int8 weight columns: the 16 K-slots of lane group g4
// in the 16x16x64 int8 MFMA are the keys of that group's transposed sign
// read in register order, i.e. even then odd nibbles of its first word
// (keys 16g4 + 0..7), then of its second (keys 16g4 + 8..15).
__device__ __forceinline__ int slot8_of(int k) {
    const int g4 = k >> 4, hw = (k >> 3) & 1, r = k & 7;
    return 16 * g4 + 8 * hw + 4 * (r & 1) + (r >> 1);
}

// Adaptive mode packs the keys of a tile that some head selected into
// positions 0..n-1 of its residual data.  Position j sits in V staging row
// res_row(j): rows 16g + 0..7 feed MFMA half 0 and rows 16g + 8..15 half 1, so
// positions 0..31 are exactly the rows of half 0.  res_pos is the inverse.
__device__ __forceinline__ int res_row(int j) { return 16 * ((j >> 3) & 3) + 8 * (j >> 5) + (j & 7); }
__device__ __forceinline__ int res_pos(int row) { return 32 * ((row >> 3) & 1) + 8 * (row >> 4) + (row & 7); }
__device__ __forceinline__ int mbcnt64(uint64_t m) {
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

// Workgroup barrier for data exchanged through LDS only: this wave's LDS
// stores have completed (lgkmcnt), the compiler moves no memory access across
// it, and loads in flight (the first tile's, some into other LDS arrays) stay
// in flight.  A __syncthreads() would also wait for every direct-to-LDS load.
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0)
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// Query preparation of one workgroup (NT threads), spread over all threads:
// the query as floats and its sign words (a wave ballot per 64 elements);
// scale_q (sequential fp32 order, element 0 first) and the fixed-point step
// per head; q_int = rint(q / step) per element (in place of the floats); then
// the balanced int4 digit words (one (word, digit) pair per thread) and the
// int8 MFMA operand words (the fixed-point parts only for residual modes).
// Inlined in every instance: a call waits for every load in flight, the first
// tile's too (2048 MHA heads of 200 keys at d = 256: binary 20.4 us with a call,
// 16.5 inlined, compensated 49.6 and 43.4).
template <int D, int G, bool KMF, bool RES, int NT, int NQ>
__device__ __forceinline__ void prep_digits(const uint16_t (&qpre)[NQ], QDigits<D, G, KMF>& qd, float* qf) {
    const int tid = threadIdx.x, lane = tid & 63;
    uint32_t* signs = &qd.signs[0][0];   // [G * D / 32] words, bit b of word i = element 32i + b
    __shared__ float gmax[G * D / 32];   // max |q| of each 32-element group (one head's)
    // the three int8 planes of q_int per element (int8 MFMA operands)
    __shared__ __attribute__((aligned(8))) uint8_t pbytes[KMF ? 3 : 1][KMF ? G * D : 8];
    // floats, sign words (wave ballots) and max |q| per half wave (its 32
    // elements lie in one head); element tid + NT j was loaded into qpre[j]
    // (zero past the last one; a wave past it has nothing to do)
#pragma unroll
    for (int j = 0; j < NQ; j++) {
        const int i = tid + NT * j;
        if (i - lane >= G * D) break;   // (uniform)
        const float x = h2f(qpre[j]);
        const uint64_t bits = __ballot(x >= 0.0f);
        const float wm = half_max(fabsf(x));
        if (i < G * D) {
            qf[i] = x;
            if ((lane & 31) == 0) {
                signs[i / 32] = (uint32_t)(lane == 0 ? bits : bits >> 32);
                gmax[i / 32] = wm;
            }
        }
    }
    lds_barrier();
    if (tid < G) {
        // sequential fp32 order (element 0 first), eight float4 reads in
        // flight at a time
        float acc = 0.0f;
        const float4* q4 = (const float4*)&qf[tid * D];
#pragma unroll
        for (int c0 = 0; c0 < D / 4; c0 += 8) {
            float4 v[8];
#pragma unroll
            for (int u = 0; u < 8; u++) v[u] = q4[c0 + u];
#pragma unroll
            for (int u = 0; u < 8; u++) {
                acc += fabsf(v[u].x); acc += fabsf(v[u].y); acc += fabsf(v[u].z); acc += fabsf(v[u].w);
            }
        }
        qd.scale_q[tid] = acc / (float)D;
        float mx = 0.0f;
#pragma unroll
        for (int k = 0; k < D / 32; k++) mx = fmaxf(mx, gmax[tid * (D / 32) + k]);
        qd.dq[tid] = mx > 0.0f ? 256.0f * (mx / kQIntMax) : 256.0f;
    }
    lds_barrier();
    // binary attention needs only the sign words and scale_q
    if constexpr (!RES) return;
    if (tid == 0) {
        float m = 0.0f;
        for (int g = 0; g < G; g++) m = fmaxf(m, qd.dq[g]);
        qd.prec_bound = 0.53f * m * sqrtf((float)D);
    }
    // q_int over the floats (each thread converts the elements it reads) and
    // its balanced int8 planes, q_int = p0 + 256 p1 + 65536 p2, p_i in [-128, 127]
    int* qint = (int*)qf;
    for (int i = tid; i < G * D; i += NT) {
        const int t = (int)__builtin_rintf(qf[i] / (qd.dq[i / D] * (1.0f / 256.0f)));
        qint[i] = t;
        if constexpr (KMF) {
            const int p0 = ((t + 128) & 255) - 128;
            const int t1 = (t - p0) >> 8;
            const int p1 = ((t1 + 128) & 255) - 128;
            pbytes[0][i] = (uint8_t)p0;
            pbytes[1][i] = (uint8_t)p1;
            pbytes[2][i] = (uint8_t)((t1 - p1) >> 8);
        }
    }
    lds_barrier();
    if constexpr (!KMF) {
        // digit j of the 8 elements of word w: nibble k = element 8w + k (balanced
        // base 16: t = sum_j d_j 16^j, d_j in [-8, 7]).  Four threads per word
        // (a DPP quad), two elements each; the quad ORs its nibbles together.
        static_assert((G * D / 2) % 4 == 0, "whole quads per digit word");
        for (int e = tid; e < G * (D / 2); e += NT) {
            const int gw = e >> 2, q = e & 3, g = gw / (D / 8), w = gw % (D / 8);
            uint32_t word[6];
    #pragma unroll
            for (int j = 0; j < 6; j++) word[j] = 0u;
    #pragma unroll
            for (int k = 2 * q; k < 2 * q + 2; k++) {
                int t = qint[g * D + 8 * w + k];
    #pragma unroll
                for (int j = 0; j < 6; j++) {
                    const int d = ((t + 8) & 15) - 8;
                    word[j] |= ((uint32_t)d & 0xFu) << (4 * k);
                    t = (t - d) >> 4;
                }
            }
    #pragma unroll
            for (int j = 0; j < 6; j++) {
                word[j] |= dpp_u<0xB1>(word[j]);   // quad 1,0,3,2
                word[j] |= dpp_u<0x4E>(word[j]);   // quad 2,3,0,1
            }
            if (q == 0) {
                qd.digits[g][w] = make_int4((int)word[2], (int)word[3], (int)word[4], (int)word[5]);
                qd.digits_lo[g][w] = make_int2((int)word[0], (int)word[1]);
            }
        }
    }
    if constexpr (KMF) {
        // B operand words: column c = 2g + p (c < 2G) holds plane p + 1 of
        // head g, column 2G + g plane 0 of head g when 3G <= 16 (bq_lo column
        // 2g otherwise); slot s = 4r + j of lane group q for MFMA m holds dim
        // 16 unit(m, q) + 8 (r/2) + 2j + r%2, where the unpacked codes put
        // it: words r = 2rr, 2rr + 1 are the even and odd bytes of the 8
        // plane bytes at dim 16 unit + 8 rr (zeros past the row's units)
        constexpr bool LO_COLS = 3 * G <= 16;
        for (int e = tid; e < KBlocks<D>::kMfma * 64; e += NT) {
            const int m = e / 64, ln = e & 63;
            const int col = ln & 15, qg4 = ln >> 4;
            const int un = KBlocks<D>::unit(m, qg4);
            int gv = 0, pv = -1;   // the lane's column: plane pv of head gv (pv < 0: zeros)
            if (col < 2 * G) {
                gv = col >> 1;
                pv = (col & 1) ? 2 : 1;
            } else if (LO_COLS && col < 3 * G) {
                gv = col - 2 * G;
                pv = 0;
            }
            bool lo_col = !LO_COLS && col < 2 * G && !(col & 1);
            if (un >= D / 16) {
                pv = -1;
                lo_col = false;
            }
            int wd[4] = {0, 0, 0, 0}, wl[4] = {0, 0, 0, 0};
#pragma unroll
            for (int rr = 0; rr < 2; rr++) {
                const int at = gv * D + 16 * un + 8 * rr;
                if (pv >= 0) {
                    const bc_v2u x = *(const bc_v2u*)&pbytes[pv][at];
                    wd[2 * rr] = (int)__builtin_amdgcn_perm(x[1], x[0], 0x06040200u);
                    wd[2 * rr + 1] = (int)__builtin_amdgcn_perm(x[1], x[0], 0x07050301u);
                }
                if (lo_col) {
                    const bc_v2u x = *(const bc_v2u*)&pbytes[0][at];
                    wl[2 * rr] = (int)__builtin_amdgcn_perm(x[1], x[0], 0x06040200u);
                    wl[2 * rr + 1] = (int)__builtin_amdgcn_perm(x[1], x[0], 0x07050301u);
                }
            }
            qd.bq[m][ln] = make_int4(wd[0], wd[1], wd[2], wd[3]);
            if constexpr (!LO_COLS) qd.bq_lo[m][ln] = make_int4(wl[0], wl[1], wl[2], wl[3]);
        }
    }
    lds_barrier();
}

// Build-time switches; each default is the measured fastest on MI355X:
//   BC_MHA_WAVES   waves/SIMD the MHA compensated kernel's registers target (3)
//   BC_BIN_WAVES   the same for binary attention of groups up to 2 (5)
//   BC_ADAPT_WAVES the same for adaptive attention (2 where Occupancy::kAdaptTwo;
//                  its LDS holds two workgroups per CU at d = 128)
//   BC_LIN_V       V code tiles read as linear KiB runs (1) instead of per key
//   BC_MHA_PIPE / BC_ADAPT_PIPE / BC_GQA_PIPE  one-tile prefetch with two staging
//                  buffers for MHA (1), adaptive (1) and GQA compensated (0: one
//                  buffer keeps a third workgroup per CU) kernels
//   BC_NT_AUX      cache policy of the loads that cover whole KiB runs (K and V
//                  sign rows, the linear V code tile, the K code blocks): 2 = nontemporal (8-11% faster;
//                  lines that several loads share keep the default policy)
//   BC_NT_SCALES   cache policy of the 2-byte scale loads (0: default)
#ifndef BC_MHA_WAVES
#define BC_MHA_WAVES 3
#endif
#ifndef BC_LIN_V
#define BC_LIN_V 1
#endif
#ifndef BC_MHA_PIPE
#define BC_MHA_PIPE 1
#endif
#ifndef BC_ADAPT_PIPE
#define BC_ADAPT_PIPE 1
#endif
#ifndef BC_GQA_PIPE
#define BC_GQA_PIPE 0
#endif
#ifndef BC_BIN_WAVES
#define BC_BIN_WAVES 5
#endif
#ifndef BC_NT_AUX
#define BC_NT_AUX 2
#endif
#ifndef BC_NT_SCALES
#define BC_NT_SCALES 0
#endif
#ifndef BC_ADAPT_WAVES
#define BC_ADAPT_WAVES 2
#endif
template <int D, int G, int MODE>
struct Occupancy {
    // Compensated heads above d = 128: two waves where the tile's operands fit
    // 256 registers with next to no spilling (one wave's latencies are
    // exposed: 100 MB of cache, two against one: d = 256 MHA 38 / 61 us,
    // groups of 2 29 / 34; d = 224 groups of 4 36.5 / 40.6), one where they
    // do not (d = 256, groups of 4: 37.4 us at one, 47.0 at two)
    static constexpr bool kTwo = G <= 2 || (G == 4 && D <= 224) || D <= 160;
    // Adaptive heads: two up to d = 128 and for single heads of d = 160, whose
    // operands fit 256 registers (2048 heads of 800 keys 174 us at one, 121 at
    // two; 128 heads of 8000 keys 72 / 59); spilling costs the others what two
    // bring (d = 192 MHA, 2048 heads of 600 keys 177 / 145, 256 of 800 42 / 46)
    static constexpr bool kAdaptTwo = D <= 128 || (D == 160 && G == 1);
    static constexpr int kWaves =
        MODE == MODE_BINARY     ? (D <= 128 ? (G <= 2 ? BC_BIN_WAVES : 3) : 2)
        : MODE == MODE_ADAPTIVE ? (kAdaptTwo ? BC_ADAPT_WAVES : 1)
        : (G == 1 && D <= 128)  ? BC_MHA_WAVES
                                : (D <= 128 ? (G <= 4 && !BC_GQA_PIPE ? 3 : 2) : (kTwo ? 2 : 1));
};

// The K residual dots come from int8 MFMAs (see the kernel): every instance
// but the adaptive mode's single heads.
__host__ __device__ constexpr bool k_on_mfma(int G, int mode) {
    return mode != MODE_BINARY && (G > 1 || mode != MODE_ADAPTIVE);
}

// NW waves per workgroup (4, or 8 to 16 for a wide workgroup that takes all
// keys of its group: one split, no merge launch); wave w takes tiles w, w + NW,
// w + 2 NW, ... of the key range, and the epilogue merges the NW waves.
// APP: the workgroup whose key range holds the slot a.app_slot appends the
// token a.app_k / a.app_v there.
//
// The scalar arguments (14 dwords) come in registers with the wave (kernarg
// preloading: a launch's first read of its argument memory takes about a
// microsecond), so they are what the first loads' addresses need: the planes'
// bases (each blob's scales follow its signs or codes, whose capacity is
// kv_rows * kv_stride vectors) and the key range; plan packs the split's tiles
// (bits 0..16), whether the launch's groups come from a list (bit 17) and the
// head groups per kv head (bits 18..30).  Measured with it: one 64-key call
// 0.9 us less.
constexpr int kPlanList = 1 << 17, kPlanGroups = 18;
static_assert(((int64_t)bc::kMaxHeadGroups << kPlanGroups | (kPlanList - 1)) < ((int64_t)1 << 31), "the packed plan holds every count");
inline int pack_plan(const AttnArgs& a, int G) {
    return a.chunk / 64 | (a.group_list != nullptr ? kPlanList : 0) | (((a.Hq / a.Hkv) / G) << kPlanGroups);
}
#define BC_MFMA_ARGS(a, G)                                                                       \
    (a).q, (a).kb.signs, (a).vb.signs, (a).kr.codes, (a).vr.codes, (a).B * (a).Hkv, (a).S,       \
        (a).kv_stride, pack_plan(a, G), (a)
template <int D, int G, int MODE, int NW = 4, bool APP = false>
__global__ __launch_bounds__(NW * 64) __attribute__((amdgpu_waves_per_eu(Occupancy<D, G, MODE>::kWaves)))
void attn_mfma_kernel(const uint16_t* q, const uint8_t* k_signs, const uint8_t* v_signs,
                      const uint8_t* k_codes, const uint8_t* v_codes, int kv_rows, int S, int kv_stride,
                      int plan, AttnArgs a) {
    constexpr int NB = D / 16;   // nibble dim-blocks (16 dims each)
    constexpr int NH = (D + 63) / 64;   // sign blocks (64 dims each; D % 64 == 32: half of the last)
    constexpr int CW = D / 8;    // code dwords per key
    constexpr bool RES = MODE != MODE_BINARY;
    constexpr int SB = D / 8;    // sign bytes per key
    constexpr int CB = D / 2;    // code bytes per key
    // Code loads.  V codes: linear, load round i, lane l takes the 16 bytes at
    // i*1024 + 16*l of the tile (contiguous KiB); the adaptive mode gathers
    // only selected keys' rows.  K codes: in the key blocks of the int8 MFMAs
    // (KBlocks), or (adaptive single heads) the lane's own key's row.
    // every key's residual data is read (compensated, and mixed per-head modes)
    constexpr bool ALLRES = MODE == MODE_COMP || MODE == MODE_MIXED;
    constexpr int Q = D / 32;    // 16-byte pieces per code row
    constexpr bool Q_POW2 = (Q & (Q - 1)) == 0;
    // KMF: the K residual dots of all G heads come from one set of int8 MFMAs
    // (keys x dims times dims x (head, digit plane)); the lane holds code
    // pieces of 16 keys (KBlocks) instead of one key's row
    constexpr bool KMF = k_on_mfma(G, MODE);
    using KB = KBlocks<D>;
    constexpr bool LIN_V = BC_LIN_V && ALLRES;
    // Vector-memory operations issued per prefetched tile, counted at their
    // fewest (a load moves at most 16 bytes; planes are separate loads), so
    // waiting down to this many outstanding operations completes everything
    // issued before the prefetch and never less.
    constexpr int kSignDma = D % 64 != 0 ? WaveLds<D, G, RES, KMF>::kSignStride / 4 : (SB + 15) / 16;
    constexpr int kVDma = kSignDma + (ALLRES ? Q : 0);
    constexpr int kKLoads = (SB + 15) / 16 + (RES ? 4 + (KMF ? 4 * KB::kLoads : Q) : 2);
    constexpr int kPrefetchOps = kVDma + kKLoads;
    static_assert(kPrefetchOps + kVDma < 64, "vmcnt holds 6 bits");
    // GQA groups in compensated mode run without the one-tile prefetch: one
    // staging buffer and one K register set leave room for a third workgroup
    // per CU (measured faster), and above d = 128 single heads do too (a
    // second workgroup: Occupancy); adaptive mode keeps it
    constexpr bool PIPE = (G == 1 && BC_MHA_PIPE && (D <= 128 || !ALLRES)) ||
                          (MODE == MODE_ADAPTIVE && BC_ADAPT_PIPE) || BC_GQA_PIPE;
    using WL = WaveLds<D, G, RES, KMF>;
    using KR = KRegs<D, KMF>;
    // Groups up to 4: the sign-part value MFMAs run on int8 operands.  The
    // sign bits enter in place (element 2^p for bit p of a nibble, four keys
    // per AND instead of two fp16 elements) and each weight as an integer up
    // to 2^30 in four balanced 8-bit digit columns (columns 4g + j): the bytes
    // of w + 0x80808080, each less 128, so two operations give the packed
    // word.  The sums are exact in int32 accumulators.  A rescale (running max
    // or weight scale) flushes them, scaled, into a per-wave float bank in LDS
    // and restarts them at zero (flush8).
    // R8: the residual part too.  A code n enters as 16 n, eight codes in three
    // operations, its weight as digits of the same kind, and no offset is
    // needed for the codes' sign (fp16 codes are n + 8).  The sums are exact,
    // where fp32 accumulation in the matrix cores drops low bits of every
    // partial sum (the fp16 path at unit variance: 2.6e-4 to 2.9e-4 of the
    // output against 64 bits; the fp16 output's own rounding is 2.1e-4).
    constexpr bool I8 = G <= 4;
    constexpr bool R8 = I8 && RES;
    // int8 weights in LDS: a row per slot, 4 digit bytes per head (and part),
    // read back as columns by ds_read_b64_tr_b8 (16-byte rows; a shorter row
    // is read twice, its columns repeating).  Up to two heads, one row holds
    // the sign weights then the residual weights, so one operand serves both
    // parts; four heads take two 16-byte halves.
    constexpr int kWRow = G == 4 ? (R8 ? 32 : 16) : (G == 2 && R8 ? 16 : 8);
    constexpr int kResCol = (R8 && G <= 2) ? 4 * G : 0;   // first residual digit column
    // tiles whose sums int32 holds: a residual digit adds at most
    // 128 * 112 * 64 < 2^20 per tile
    constexpr int kMaxTiles8 = 2000;

    __shared__ QDigits<D, G, KMF> qd;
    __shared__ __attribute__((aligned(16))) uint8_t lds_st0[NW][WL::kStage];
    __shared__ __attribute__((aligned(16))) uint8_t lds_st1[NW][PIPE ? WL::kStage : 16];
    __shared__ __attribute__((aligned(16))) uint16_t lds_wts[NW][I8 ? 8 : WL::kWeightBytes / 2];
    __shared__ __attribute__((aligned(16))) uint8_t lds_w8[NW][I8 ? 64 * kWRow : 16];
    // (int8 path) per wave and head, the float sums of the keys before the
    // last rescale, [head][D]
    __shared__ __attribute__((aligned(16))) float lds_bank[NW][I8 ? G * D : 4];
    // the query as floats during its preparation (the bank is free until then)
    __shared__ __attribute__((aligned(16))) float lds_qf[I8 ? 4 : G * D];
    float* const qf = I8 ? &lds_bank[0][0] : lds_qf;
    __shared__ __attribute__((aligned(16))) int lds_rd[NW][WL::kRdInts];
    __shared__ __attribute__((aligned(16))) int lds_rdlo[NW][(KMF && G > 1 && 3 * G <= 16) ? WL::kRdInts : 1];
    __shared__ float wofs[NW][G];
    __shared__ float wm[NW][G], wlsum[NW][G], wsc[NW][G];
    // (groups of eight) the merge's factors per head: each wave's, maximum, total
    __shared__ float wfac[G == 8 ? NW : 1][G], wtot[G == 8 ? 2 : 1][G];

    const int split = blockIdx.x;
    // per-head modes: this launch's query-head groups come from its list
    int grow = blockIdx.y;
    if constexpr (MODE == MODE_BINARY || MODE == MODE_MIXED) {
        if (plan & kPlanList) {
            if (grow >= *a.group_count) return;
            grow = a.group_list[grow];
        }
    }
    // groups are numbered through batches, kv heads and the groups of a kv head
    const int nqg = plan >> kPlanGroups;
    const int bkv = grow / nqg;
    const int bhq0 = grow * G;   // first query head
    const int64_t cap = (int64_t)kv_rows * kv_stride;

    // the wave index is uniform: readfirstlane lets the compiler keep the tile
    // loop in scalar registers (a uniform loop, not an exec-masked one)
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int g4 = lane >> 4, lj = lane & 15;
    const int chunk = (plan & (kPlanList - 1)) * 64;
    const int key_begin = split * chunk;
    const int key_end = min(S, key_begin + chunk);
    const int64_t kv_base = (int64_t)bkv * kv_stride;
    const float isd2 = (1.0f / sqrtf((float)D)) * kLog2e;
    const int kown = lane;   // the key whose score this lane computes (tile-relative)
    // V code tiles of compensated mode (linear rows of CB bytes): the 16-byte
    // pieces of row k are stored at piece ^ vsw(k), vsw(k) = (k*CB/256) mod Q,
    // so the rows that one transposed read covers spread over the LDS banks;
    // the copy permutes the pieces within each row (same cache lines).  A
    // lane's transposed reads cover row = lane.  (Other piece counts: rows of
    // an odd number of pieces already start on distinct banks.)
    const int vsw = Q_POW2 ? ((lane * CB) >> 8) & (Q - 1) : 0;

    // Buffer resources over this workgroup's key range [key_begin, key_end)
    // of each plane: offsets are 32-bit and tile-relative, and a load of a key
    // past the range returns zeros (its weight is 0), so no lane clamps its
    // address and every lane issues the same loads (the wait counts stay exact)
    const int nk = max(key_end - key_begin, 0);   // (an empty split issues no loads)
    auto rsrc = [&](const void* plane, int rb) {
        return __builtin_amdgcn_make_buffer_rsrc(
            (void*)((const uint8_t*)plane + (kv_base + key_begin) * rb), (short)0, nk * rb, kBufWord3);
    };
    const __amdgpu_buffer_rsrc_t r_ks = rsrc(k_signs, SB), r_vs = rsrc(v_signs, SB);
    const __amdgpu_buffer_rsrc_t r_ksc = rsrc(k_signs + cap * SB, 2), r_vsc = rsrc(v_signs + cap * SB, 2);
    const __amdgpu_buffer_rsrc_t r_kc = rsrc(k_codes, CB), r_vc = rsrc(v_codes, CB);
    const __amdgpu_buffer_rsrc_t r_krs = rsrc(k_codes + cap * CB, 2), r_vrs = rsrc(v_codes + cap * CB, 2);
    // adaptive: stored popcounts of this group, one pack of G per key
    using Pack = bc::PcPack<bc::PcT<D>, G>;
    constexpr int kPack = (int)sizeof(Pack);
    static_assert(kPack <= 16, "one load per pack");
    const __amdgpu_buffer_rsrc_t r_pc = __builtin_amdgcn_make_buffer_rsrc(
        (void*)((const Pack*)a.pcs + (int64_t)grow * bc::pcs_stride(S) + key_begin), (short)0, nk * kPack, kBufWord3);
    // an offset past every range (the host keeps each range's bytes below
    // 2^31 - 4096): such a load returns zeros and moves no data
    constexpr int kOob = 0x7FFFF000;

    // ---------------- loads of one tile: K side into registers, V side to LDS
    // the lane's code pieces of key block kb (KBlocks), its key's row at byte
    // offset row (kOob: zeros)
    auto load_kblock = [&](KR& r, int kb, int row) {
        constexpr int aux = MODE == MODE_ADAPTIVE ? 0 : BC_NT_AUX;
#pragma unroll
        for (int pc = 0; pc < KB::kPieces; pc++) {
            const v4u_t c = __builtin_amdgcn_raw_buffer_load_b128(r_kc, row + 64 * pc + 16 * g4, 0, aux);
            const int i = kb * KB::kWords + 4 * pc;
            r.kc[i] = c[0]; r.kc[i + 1] = c[1]; r.kc[i + 2] = c[2]; r.kc[i + 3] = c[3];
        }
#pragma unroll
        for (int tl = 0; tl < KB::kTails; tl++) {
            // (a lane group past the row's units repeats the unit two back)
            constexpr int left = KB::kLeft;
            const int q = 4 * tl + 2 < left ? g4 : (g4 & 1);
            const v2u_t c = __builtin_amdgcn_raw_buffer_load_b64(r_kc, row + 64 * KB::kPieces + 32 * tl + 8 * q, 0, aux);
            const int i = kb * KB::kWords + 4 * KB::kPieces + 2 * tl;
            r.kc[i] = c[0]; r.kc[i + 1] = c[1];
        }
    };
    auto load_k = [&](KR& r, int t0) {
        const int tr = t0 - key_begin;      // tile offset in the range (keys)
        const int kk = tr + kown;
        if constexpr (MODE == MODE_ADAPTIVE) {
            // popcounts and the two binary scales; residual data is gathered
            // once the tile's selection is known
            if constexpr (kPack == 1) {
                r.pcw[0] = __builtin_amdgcn_raw_buffer_load_b8(r_pc, kk, 0, 0);
            } else if constexpr (kPack == 2) {
                r.pcw[0] = __builtin_amdgcn_raw_buffer_load_b16(r_pc, kk * 2, 0, 0);
            } else if constexpr (kPack == 4) {
                r.pcw[0] = __builtin_amdgcn_raw_buffer_load_b32(r_pc, kk * 4, 0, 0);
            } else if constexpr (kPack == 8) {
                const v2u_t v = __builtin_amdgcn_raw_buffer_load_b64(r_pc, kk * 8, 0, 0);
                r.pcw[0] = v[0]; r.pcw[1] = v[1];
            } else {
                const v4u_t v = __builtin_amdgcn_raw_buffer_load_b128(r_pc, kk * 16, 0, 0);
                r.pcw[0] = v[0]; r.pcw[1] = v[1]; r.pcw[2] = v[2]; r.pcw[3] = v[3];
            }
            r.sk = __builtin_amdgcn_raw_buffer_load_b16(r_ksc, kk * 2, 0, 0);
            r.svv = __builtin_amdgcn_raw_buffer_load_b16(r_vsc, kk * 2, 0, 0);
            r.rsk = 0;
            r.rsv = 0;
            return;
        }
        r.ks = buf_signs<D, BC_NT_AUX>(r_ks, kk * SB);
        r.sk = __builtin_amdgcn_raw_buffer_load_b16(r_ksc, kk * 2, 0, BC_NT_SCALES);
        r.svv = __builtin_amdgcn_raw_buffer_load_b16(r_vsc, kk * 2, 0, BC_NT_SCALES);
        r.rsk = 0;
        r.rsv = 0;
        // residual scales and K codes of every key (adaptive mode too: the
        // selection is known only after the scores, and these loads are the
        // ones worth prefetching; V codes are gathered for selected keys)
        if constexpr (RES) {
            r.rsk = __builtin_amdgcn_raw_buffer_load_b16(r_krs, kk * 2, 0, BC_NT_SCALES);
            r.rsv = __builtin_amdgcn_raw_buffer_load_b16(r_vrs, kk * 2, 0, BC_NT_SCALES);
            if constexpr (KMF) {
                // key block kb: key 16kb + l%16
#pragma unroll
                for (int kb = 0; kb < 4; kb++) load_kblock(r, kb, (tr + 16 * kb + lj) * CB);
            }
        }
    };
    // V tile to LDS: key k's sign row at k*SB; its code row at k*CB (linear,
    // pieces swizzled as above) or piece c at c*1024 + 16k (per key)
    auto issue_v = [&](int buf, int t0) {
        const int tr = t0 - key_begin;
        uint8_t* st_codes = buf ? lds_st1[wave] : lds_st0[wave];
        uint8_t* st_signs = st_codes + WL::kCodeBytes;
        if constexpr (WL::kSignPad) {
            // a dword per lane: RW lanes per row, 64 / RW rows per load
            constexpr int RW = WL::kSignStride / 4;
            const int w = min(lane % RW, SB / 4 - 1);
#pragma unroll
            for (int c = 0; c < RW; c++)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(r_vs, LDS_PTR(void, st_signs + c * 256), 4,
                                                         (tr + c * (64 / RW) + lane / RW) * SB + 4 * w, 0, 0, 0);
        } else {
            // whole KiB, and a half one at d = 64 and 192 (whose lanes 32..63
            // repeat lanes 0..31 into the half past the rows)
#pragma unroll
            for (int c = 0; c < SB / 16; c++)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(r_vs, LDS_PTR(void, st_signs + c * 1024), 16,
                                                         tr * SB + 16 * lane + c * 1024, 0, 0, BC_NT_AUX);
            if constexpr (SB % 16 != 0)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(r_vs, LDS_PTR(void, st_signs + SB / 16 * 1024), 16,
                                                         tr * SB + 16 * (lane & 31) + SB / 16 * 1024, 0, 0, 0);
        }
        if constexpr (ALLRES) {
#pragma unroll
            for (int c = 0; c < Q; c++)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(
                    r_vc, LDS_PTR(void, st_codes + c * 1024), 16,
                    LIN_V ? tr * CB + c * 1024 + 16 * (Q_POW2 ? lane ^ ((4 * c + (lane >> 4)) & (Q - 1)) : lane)
                          : (tr + lane) * CB + 16 * c, 0, 0, LIN_V ? BC_NT_AUX : 0);
        }
    };

    // The query's elements are loaded first, then the wave's first tile
    // (except in adaptive mode, whose first tile needs the selection), and the
    // query preparation runs while that tile is in flight: it waits only for
    // the older query loads, and its barriers wait for LDS traffic only.
    constexpr int NT = NW * 64;
    constexpr int NQ = (G * D + NT - 1) / NT;
    uint16_t qpre[NQ];
    {
        const uint16_t* qb = q + (int64_t)bhq0 * D;
#pragma unroll
        for (int j = 0; j < NQ; j++) {
            const int i = (int)threadIdx.x + NT * j;
            qpre[j] = i < G * D ? qb[i] : (uint16_t)0;
        }
    }
    int t = key_begin + wave * 64;
    const bool early = MODE != MODE_ADAPTIVE && t < key_end;
    KR ka, kb;
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (MODE != MODE_ADAPTIVE) {
        // without a first tile to fetch, the same loads address keys past the
        // range (a split holds fewer than 2^23 keys): zeros, no traffic, and
        // the same instructions on every path, so that the preparation's
        // wait for the query counts them exactly
        const int t_first = early ? t : key_begin + (1 << 23) + 1024;
        load_k(ka, t_first);
        issue_v(0, t_first);
    }
    __builtin_amdgcn_sched_barrier(0);
    // the appended token's slice of this lane (lane groups 0 and 1: K and V;
    // loaded by every wave, so that the wait for the query counts the same)
    constexpr int AL = D / 8;
    bc_v4u app_raw = {0u, 0u, 0u, 0u};
    if constexpr (APP) {
        app_raw = bc::load_row_slice((lane / AL == 1 ? a.app_v : a.app_k) + (int64_t)bkv * D, lane % AL);
        __builtin_amdgcn_sched_barrier(0);
    }
    prep_digits<D, G, KMF, RES, NT>(qpre, qd, qf);

    // In-place append: the wave that takes the slot's tile encodes the token's
    // K and V vectors (online-encode semantics: the residual against the fp32
    // mean) into LDS and stores them from there.  Nothing waits for the
    // stores: the wave's tile is loaded with the slot's old contents, and when
    // it is processed the token's score parts and dots (formed here, as a
    // tile's are) and its V row take their place.  No other wave reads the
    // slot (the host appends only with one query-head group per kv head), and
    // later launches see the token as after a separate encode.  (Encoding
    // first and then loading the tile is three dependent memory round trips:
    // 3 us of a 27 us step.)
    struct Token {
        uint32_t signs[2][D / 32];
        uint32_t codes[2][D / 8];
        uint16_t scale[2], rscale[2];
        float mq[G];             // 2 popcount - d of K against each query head
        int dot[G], dot_lo[G];   // K residual dots: planes 1 and 2, plane 0
    };
    __shared__ Token token[1];
    int app_t0 = -1;   // (wave-uniform) the slot's tile, if it is this wave's
    if constexpr (APP) {
        static_assert(bc::append_dim(D) && MODE != MODE_ADAPTIVE && MODE != MODE_MIXED, "append");
        const int slot = a.app_slot, tile = (slot - key_begin) >> 6;
        if (slot >= key_begin && slot < key_end && tile % NW == wave) {
            app_t0 = key_begin + 64 * tile;
            const int grp = lane / AL;
            const int kv = grp == 1;
            const bc::EncodeDst dst{(uint8_t*)token->signs[kv], &token->scale[kv],
                                    RES ? (uint8_t*)token->codes[kv] : nullptr, &token->rscale[kv]};
            bc::encode_row_slice<D, RES ? bc::ENC_FUSED_FP32 : bc::ENC_BINARY>(app_raw, lane % AL, grp < 2, dst, 0);
            __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0)
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
            if (lane < G) {
                int pc = 0;
#pragma unroll
                for (int w = 0; w < D / 32; w++) pc += __builtin_popcount(~(qd.signs[lane][w] ^ token->signs[0][w]));
                token->mq[lane] = (float)(2 * pc - D);
            }
            if constexpr (RES) {
                // (every key of the block is the token)
                v4i_t acc = v4i_t{0, 0, 0, 0}, accl = v4i_t{0, 0, 0, 0};
#pragma unroll
                for (int m = 0; m < KB::kMfma; m++) {
                    const int un = min(KB::unit(m, g4), D / 16 - 1);
                    const v4i_t av = codes_i8(token->codes[0][2 * un], token->codes[0][2 * un + 1]);
                    acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(*(const v4i_t*)&qd.bq[m][lane], av, acc, 0, 0, 0);
                    if constexpr (3 * G > 16)
                        accl = __builtin_amdgcn_mfma_i32_16x16x64_i8(*(const v4i_t*)&qd.bq_lo[m][lane], av, accl, 0, 0, 0);
                }
                if (lj == 0) {
#pragma unroll
                    for (int h = 0; h < 2; h++)
                        if (2 * g4 + h < G) {
                            token->dot[2 * g4 + h] = acc[2 * h] + 256 * acc[2 * h + 1];
                            if constexpr (3 * G > 16) token->dot_lo[2 * g4 + h] = accl[2 * h];
                        }
                    if constexpr (3 * G <= 16) {
#pragma unroll
                        for (int g = 0; g < G; g++)
                            if (g4 == (2 * G + g) / 4) token->dot_lo[g] = acc[(2 * G + g) % 4];
                    }
                }
            }
            // (the attention arguments hold the cache planes read-only)
            const int64_t at = kv_base + slot;
#pragma unroll
            for (int v = 0; v < 2; v++) {
                const BinPlanes& bp = v ? a.vb : a.kb;
                const ResPlanes& rp = v ? a.vr : a.kr;
                if (lane < D / 32) ((uint32_t*)(bp.signs + at * SB))[lane] = token->signs[v][lane];
                if (lane == 0) ((uint16_t*)bp.scales)[at] = token->scale[v];
                if constexpr (RES) {
                    if (lane < D / 8) ((uint32_t*)(rp.codes + at * CB))[lane] = token->codes[v][lane];
                    if (lane == 0) ((uint16_t*)rp.scales)[at] = token->rscale[v];
                }
            }
        }
    }

    // weight column owned by this lane in the MFMA B operand, and its head
    const int my_col = lj;
    // (int8 columns: 4 per head, repeating past the last; fp16: 2 per head)
    const int my_head = I8 ? (my_col >> 2) % G : my_col >> 1;
    const int my_rhead = R8 ? my_head : my_col >> 1;
    const int bcol = my_col < 2 * G ? my_col : (my_col & 1);

    // weight columns [2 parts][2G cols][72 slots]: this lane's store slot in
    // column 0, and its B-operand read position in column bcol.  The lane
    // offsets go through an opaque copy so that every access is one constant
    // offset from a base that the compiler ties to lds_wts (accesses it cannot
    // tie to one array wait for all direct loads in flight, the prefetch too)
    uint16_t* wsl = &lds_wts[0][0] + opaque_int(wave * (WL::kWeightBytes / 2) + slot_of(kown));
    const uint16_t* wrd = &lds_wts[0][0] + opaque_int(wave * (WL::kWeightBytes / 2) + bcol * WL::kColSlots + 16 * g4);
    // int8 weights: this lane's key's row, and the row halves it reads for the
    // sign and residual operands (slots 16 g4 + 0..7; the next eight follow)
    uint8_t* w8st = &lds_w8[0][0] + opaque_int(I8 ? (wave * 64 + slot8_of(kown)) * kWRow : 0);
    const uint8_t* w8rd = &lds_w8[0][0] + opaque_int(I8 ? (wave * 64 + 16 * g4 + (lj >> 1)) * kWRow + (kWRow >= 16 ? 8 * (lj & 1) : 0) : 0);
    int* rdl = lds_rd[wave];          // [64 keys][G] residual dots
    int* rdlo = lds_rdlo[wave];       // their plane-0 parts (precise tiles)

    constexpr int kRes0 = 2 * G;   // first fp16 residual weight column
    // softmax reference per head, lowered lazily: weights p = 2^(s - m) stay
    // <= 2^kTau, and the accumulators are rescaled only when a score passes
    // m + kTau (the result does not depend on m)
    constexpr int kTauI = 8;
    constexpr float kTau = (float)kTauI;
    float m[G], mlim[G], lsum[G], off[G];
#pragma unroll
    for (int g = 0; g < G; g++) {
        m[g] = -INFINITY;
        mlim[g] = -INFINITY;
        lsum[g] = 0.0f;
        off[g] = 0.0f;
    }
    f4_t cs[I8 ? 1 : NH][4];   // sign part: [block][p] rows = dims 64h + 4m + p
    v4i_t ci[I8 ? NH : 1][4];  // (int8 path) the same, per digit column
    f4_t cn[R8 ? 1 : NB];      // residual part: rows = dims 16db + m
    v4i_t cr[R8 ? NB : 1];     // (int8 path) the same, per digit column
#pragma unroll
    for (int h = 0; h < (I8 ? 1 : NH); h++)
#pragma unroll
        for (int p = 0; p < 4; p++) cs[h][p] = f4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int h = 0; h < (I8 ? NH : 1); h++)
#pragma unroll
        for (int p = 0; p < 4; p++) ci[h][p] = v4i_t{0, 0, 0, 0};
#pragma unroll
    for (int d = 0; d < (R8 ? 1 : NB); d++) cn[d] = f4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int d = 0; d < (R8 ? NB : 1); d++) cr[d] = v4i_t{0, 0, 0, 0};

    // (int8 path) a head's digit columns are one lane quad; the quad's first
    // lane owns the head's rows.  digits(): d0 + 256 d1 + 65536 d2 + 2^24 d3
    // of the quad (each lane scales its own digit, then a quad sum)
    const bool owner8 = I8 && my_col < 4 * G && (my_col & 3) == 0;
    const bool rowner8 = R8 && my_col >= kResCol && my_col < kResCol + 4 * G && (my_col & 3) == 0;
    auto digits = [&](int c, float dscale) {
        float v = (float)c * dscale;
        v += dpp_f<0xB1>(v);
        return v + dpp_f<0x4E>(v);
    };
    // the lane's factor 256^digit (formed where it is used: one register less
    // in the tile loop)
    auto digit_scale = [&] {
        return __builtin_bit_cast(float, 0x3F800000u + ((uint32_t)(opaque_int(lane) & 3) << 26));
    };
    // flush8: bank = (bank + integer sums) * f, the integer sums restart at 0
    auto bank_at = [&] {
        return &lds_bank[0][0] + (I8 ? (wave * G + ((opaque_int(lane) & 15) >> 2) % G) * D : 0);
    };
    bool banked = false;   // (wave-uniform) the bank holds values
    int live8 = 0;         // (wave-uniform) tiles in the integer sums
    auto flush8 = [&](float f) {
        const float dscale = digit_scale();
        float* const bank = bank_at();
#pragma unroll
        for (int h = 0; h < NH; h++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                // (accumulator p carries 2^p: bit p read in place)
                float t[4];
#pragma unroll
                for (int p = 0; p < 4; p++) {
                    t[p] = digits(ci[h][p][i], dscale) * (1.0f / (float)(1 << p));
                    ci[h][p][i] = 0;
                }
                if (owner8 && (64 * h + 16 * g4 < D)) {
                    float4* bp = (float4*)&bank[64 * h + 4 * (4 * g4 + i)];
                    float4 b = banked ? *bp : make_float4(0.f, 0.f, 0.f, 0.f);
                    *bp = make_float4((b.x + t[0]) * f, (b.y + t[1]) * f, (b.z + t[2]) * f, (b.w + t[3]) * f);
                }
            }
        if constexpr (R8) {
            // (other lanes add to what the sign part's owners have stored)
            __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0)
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
            // (codes as 16 n)
#pragma unroll
            for (int d = 0; d < NB; d++) {
                float t[4];
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    t[i] = digits(cr[d][i], dscale) * (1.0f / 16.0f);
                    cr[d][i] = 0;
                }
                if (rowner8) {
                    float4* bp = (float4*)&bank[16 * d + 4 * g4];
                    const float4 b = *bp;
                    *bp = make_float4(b.x + t[0] * f, b.y + t[1] * f, b.z + t[2] * f, b.w + t[3] * f);
                }
            }
        }
        banked = true;
        live8 = 0;
    };

    // fp16 path: weights enter the MFMAs as w * 2^wexp (hi + lo), wexp chosen so
    // the largest possible weight sits near 2^14: no overflow, and weights down
    // to ~2^-30 of the largest keep their contribution (undone exactly in the
    // epilogue)
    constexpr int kWTop = 14;
    int wexp = 0;
    bool have_wexp = false;
    float wlim = 0.0f;
    // int8 path: weights enter as integers round(p f es), es a power of two per
    // head.  es is planned from the weights themselves, not from the largest V
    // scale a key may have: the integer step is then 2^-24 to 2^-31 of the
    // largest weighted value since the head's last plan, whatever the rows that
    // carry no weight are (a plan for the largest scale: one key 12 nats above
    // 65536 others, one V row in 256 of 32 times the magnitude: 6.5e-3 of the
    // output, planned from the weights 2e-4).  A weight past kW8Max, whose
    // digits no longer fit, replans its head, and so does a move of the head's
    // reference (which flushes the sums anyway): the tile's largest weight to
    // [2^24, 2^25), so that it may grow 64 times before the next flush.  A flush
    // waits for the loads in flight; scores of unit variance grow 8 times past
    // a wave's first tile in 10 to 19% of the waves (d = 64, 96, 256: +8% of the
    // kernel's time with 2^28 here), 64 times in less than 1%.  The step is far
    // below the rounding of the fp16 output (2.1e-4): weights to 2^24, 2e-5 of
    // it with one key 9 to 16 nats above 32768 others.
    // Without any weight es stays at 2^60, below the last bit of any output.
    constexpr float kW8Max = 2139000000.0f;   // <= 0x7F7F7F7F
    constexpr int kW8Top = 25;
    constexpr float kEsMax = 1152921504606846976.0f;   // 2^60
    float es[G];
#pragma unroll
    for (int g = 0; g < G; g++) es[g] = kEsMax;

    uint32_t thresh[G];
    int cutoff[G];
    float thr_floor[G], thr_value[G];   // the threshold as float bounds
    if constexpr (MODE == MODE_ADAPTIVE) {
#pragma unroll
        for (int g = 0; g < G; g++) {
            thresh[g] = a.thresh[bhq0 + g];
            cutoff[g] = a.cutoff[bhq0 + g];
            thr_floor[g] = key_floor(thresh[g]);
            thr_value[g] = key_value(thresh[g]);
        }
    }
    // mixed mode: which heads of the group add their residual
    bool hmode[G];
#pragma unroll
    for (int g = 0; g < G; g++) hmode[g] = true;
    if constexpr (MODE == MODE_MIXED) {
#pragma unroll
        for (int g = 0; g < G; g++) hmode[g] = a.head_mode[bhq0 + g] != 0;
    }

    // query digits of a single head in scalar registers for the whole loop
    // (uniform operands of v_dot8) when codes are read per key, and the int8
    // MFMA B operands of the K residual dot (loop invariant)
    int sdig[(RES && !KMF) ? CW : 1][4];
    // (groups of four and more, and appending: read per tile, the registers are full)
    constexpr bool BQ_LDS = KMF && ALLRES && (G >= 4 || APP);
    v4i_t bq[KMF && !BQ_LDS ? KB::kMfma : 1];
    if constexpr (RES && !KMF) {
#pragma unroll
        for (int w = 0; w < CW; w++) {
            const int4 dg = qd.digits[0][w];
            sdig[w][0] = __builtin_amdgcn_readfirstlane(dg.x);
            sdig[w][1] = __builtin_amdgcn_readfirstlane(dg.y);
            sdig[w][2] = __builtin_amdgcn_readfirstlane(dg.z);
            sdig[w][3] = __builtin_amdgcn_readfirstlane(dg.w);
        }
    }
    if constexpr (KMF && !BQ_LDS) {
#pragma unroll
        for (int m = 0; m < KB::kMfma; m++) {
            const int4 w = qd.bq[m][lane];
            bq[m] = v4i_t{w.x, w.y, w.z, w.w};
        }
    }

    // ---------------- adaptive mode: a tile's selection, from its stored
    // popcounts and K scales, and the loads of its residual data: the residual
    // scales per key (lane = key), the K codes and V codes of the selected keys
    // at their compacted positions (K codes to registers, V codes to staging
    // buffer buf with the V signs).  Unselected keys and the positions past
    // the selected ones load from past the range (zeros, no traffic), so the
    // loads issue without branches.
    auto gather = [&](KR& r, int t0, int buf) {
        const int s = t0 + kown;
        const bool valid = s < key_end;
        const float sk = h2f(r.sk);
        uint32_t selmask = 0;
        // selected: above the threshold, or equal to it at an index up to the
        // cutoff (ties are taken lowest index first); compared as exact float
        // scores unless a lane of the wave has a non-finite scale
        const bool fast = __ballot(!finite_scale(sk)) == 0ull;
        const float sk2 = 2.0f * sk, nd = -(float)D * sk;
#pragma unroll
        for (int g = 0; g < G; g++) {
            constexpr int bits = 8 * (int)sizeof(bc::PcT<D>);
            constexpr int per_word = 32 / bits;
            const int pc = (int)((r.pcw[g / per_word] >> (bits * (g % per_word))) & ((1u << bits) - 1u));
            bool above, tie;
            if (fast) {
                const float sc = fmaf((float)pc, sk2, nd);
                above = sc > thr_floor[g];
                tie = sc == thr_value[g];
            } else {
                const uint32_t key = ordered_key(sk * (float)(2 * pc - D));
                above = key > thresh[g];
                tie = key == thresh[g];
            }
            const bool sel = above || (tie && s <= cutoff[g]);
            selmask |= (sel && valid) ? (1u << g) : 0u;
        }
        r.sel = selmask;
        issue_v(buf, t0);
        uint8_t* st_codes = buf ? lds_st1[wave] : lds_st0[wave];
        const uint64_t selany = __ballot(selmask != 0u);
        const int nsel = __builtin_popcountll(selany);
        const int tr = t0 - key_begin;
        const bool mine = selmask != 0u;
        const int kk = tr + kown;
        // compacted positions: key s goes to position mbcnt (selected) or to
        // n + its rank among the others; key_at = the key at position lane
        const int mb = mbcnt64(selany);
        const int key_at = __builtin_amdgcn_ds_permute(4 * (mine ? mb : nsel + lane - mb), lane);
        r.rsk = __builtin_amdgcn_raw_buffer_load_b16(r_krs, mine ? kk * 2 : kOob, 0, 0);
        r.rsv = __builtin_amdgcn_raw_buffer_load_b16(r_vrs, mine ? kk * 2 : kOob, 0, 0);
        if constexpr (KMF) {
            // key block kb: position 16kb + l%16
#pragma unroll
            for (int kb = 0; kb < 4; kb++) {
                const int j = 16 * kb + lj;
                const int key = __builtin_amdgcn_ds_bpermute(4 * j, key_at);
                load_kblock(r, kb, j < nsel ? (tr + key) * CB : kOob);
            }
        } else {
#pragma unroll
            for (int i = 0; i < Q; i++) {
                const v4u_t c = __builtin_amdgcn_raw_buffer_load_b128(r_kc, mine ? kk * CB + 16 * i : kOob, 0, 0);
                r.kc[4 * i] = c[0]; r.kc[4 * i + 1] = c[1]; r.kc[4 * i + 2] = c[2]; r.kc[4 * i + 3] = c[3];
            }
        }
        // V codes: staging row lane holds position res_pos(lane)
        const int jv = res_pos(lane);
        const int vkey = __builtin_amdgcn_ds_bpermute(4 * jv, key_at);
#pragma unroll
        for (int c = 0; c < Q; c++)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(r_vc, LDS_PTR(void, st_codes + c * 1024), 16,
                                                     jv < nsel ? (tr + vkey) * CB + 16 * c : kOob, 0, 0, 0);
    };

    // ---------------- one tile: scores, online softmax, value MFMAs
    auto process = [&](const KR& r, int t0, int buf) {
        uint8_t* st_codes = buf ? lds_st1[wave] : lds_st0[wave];
        uint8_t* st_signs = st_codes + WL::kCodeBytes;
        const int s = t0 + kown;
        const bool valid = s < key_end;
        // this tile's K registers: the younger operations are this tile's V
        // loads and the whole next-tile prefetch.  An explicit count keeps the
        // compiler from draining the queue (with direct-to-LDS loads pending it
        // would wait for zero).
        if constexpr (MODE != MODE_ADAPTIVE && PIPE) {
            constexpr int n = kVDma + kPrefetchOps;
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_s_waitcnt((n & 0xF) | ((n >> 4) << 14) | (0x7 << 4) | (0xF << 8));
            __builtin_amdgcn_sched_barrier(0);
        }
        const float sk = h2f(r.sk);
        float svv = h2f(r.svv);
        float rsk = h2f(r.rsk), rsv = h2f(r.rsv);
        uint32_t kc[KR::kCodeWords];
        if constexpr (RES) {
#pragma unroll
            for (int w = 0; w < KR::kCodeWords; w++) kc[w] = r.kc[w];
        }
        float xd[G];
        uint32_t selmask = 0;
#pragma unroll
        for (int g = 0; g < G; g++) {
            int pc = 0;
            if constexpr (MODE == MODE_ADAPTIVE) {
                // stored by the selection passes (same popcount as below)
                constexpr int bits = 8 * (int)sizeof(bc::PcT<D>);
                constexpr int per_word = 32 / bits;
                pc = (int)((r.pcw[g / per_word] >> (bits * (g % per_word))) & ((1u << bits) - 1u));
            } else {
#pragma unroll
                for (int w = 0; w < D / 32; w++) pc += __builtin_popcount(~(qd.signs[g][w] ^ r.ks.w[w]));
            }
            const float mq = (float)(2 * pc - D);
            xd[g] = xnor_score(qd.scale_q[g], sk, mq);
        }
        // (APP) the token's score parts and scales in place of the slot's key
        const bool has_token = APP && t0 == app_t0;
        if constexpr (APP) {
            if (has_token && opaque_int(lane) == a.app_slot - t0) {
                svv = h2f(token->scale[1]);
                if constexpr (RES) {
                    rsk = h2f(token->rscale[0]);
                    rsv = h2f(token->rscale[1]);
                }
#pragma unroll
                for (int g = 0; g < G; g++) xd[g] = xnor_score(qd.scale_q[g], h2f(token->scale[0]), token->mq[g]);
            }
        }
        // adaptive: the tile's compacted residual positions (as in gather):
        // nsel selected keys, the lane's key at position rpos
        int nsel = 64, rpos = kown;
        if constexpr (MODE == MODE_ADAPTIVE) {
            selmask = r.sel;
            const uint64_t selany = __ballot(selmask != 0u);
            const int mb = mbcnt64(selany);
            nsel = __builtin_popcountll(selany);
            rpos = selmask != 0u ? mb : nsel + lane - mb;
        }
        if constexpr (MODE == MODE_ADAPTIVE) {
            if (a.selected != nullptr && valid) {
#pragma unroll
                for (int g = 0; g < G; g++)
                    a.selected[(int64_t)(bhq0 + g) * S + s] = (selmask >> g) & 1u;
            }
        }

        // residual dot on the raw int4 codes: sum_i q_int_i * n_i per head, in
        // units of the top-16-bit step dq (racc, exact integers; in a precise
        // tile the float bits of that plus the low digits' part / 256)
        int racc[G];
#pragma unroll
        for (int g = 0; g < G; g++) racc[g] = 0;
        // precise tile: some key's score could move by more than kPrecNats
        // from the top 16 bits alone (uniform over the wave)
        const bool prec = RES && __ballot(rsk * qd.prec_bound > kPrecNats) != 0ull;
        if constexpr (KMF) {
          // key blocks holding codes: all four, or (adaptive) the blocks of
          // the nsel compacted positions
          const int nkb = (nsel + 15) >> 4;
          if (nkb > 0) {
            // codes as int8 16*n (signed): low nibbles via x << 4, high nibbles in
            // place; each half of a piece is one 16x16x64 MFMA of (head, digit
            // plane) rows x 64 dims times 64 dims x 16 keys (columns of keys whose
            // codes were not loaded are never used)
            // Lane l holds rows 4(l/16) + i = (head 2(l/16) + i/2, plane i%2 + 1)
            // of position 16kb + l%16: both planes of a head sit in one lane, and
            // q_int dot * 16 / 256 = plane1 + 256 plane2 goes to rdl[position][head].
            // Plane 0 of a precise tile (q_int dot * 16 = 65536 plane2 +
            // 256 plane1 + plane0): groups of more than 5 heads take it from a
            // second B operand (LDS) into the same lanes and store the float
            // bits of the sum; smaller groups have it in rows 2G + g (below)
            constexpr bool LO_COLS = 3 * G <= 16;
            v4i_t acc[4];
            v4i_t bt[KB::kMfma];   // this tile's B operands
            const int lz = BQ_LDS ? opaque_int(lane) : 0;   // (read per tile, not hoisted)
#pragma unroll
            for (int m = 0; m < KB::kMfma; m++) {
                if constexpr (BQ_LDS) bt[m] = *(const v4i_t*)&qd.bq[m][lz];
                else bt[m] = bq[m];
            }
#pragma unroll
            for (int kb = 0; kb < 4; kb++) {
                if (kb >= nkb) break;
                acc[kb] = v4i_t{0, 0, 0, 0};
                v4i_t accl = v4i_t{0, 0, 0, 0};
#pragma unroll
                for (int m = 0; m < KB::kMfma; m++) {
                    const v4i_t av = codes_i8(kc[kb * KB::kWords + 2 * m], kc[kb * KB::kWords + 2 * m + 1]);
                    acc[kb] = __builtin_amdgcn_mfma_i32_16x16x64_i8(bt[m], av, acc[kb], 0, 0, 0);
                    if (!LO_COLS && prec) {
                        const int4 w = qd.bq_lo[m][lane];
                        accl = __builtin_amdgcn_mfma_i32_16x16x64_i8(v4i_t{w.x, w.y, w.z, w.w}, av, accl, 0, 0, 0);
                    }
                }
                if constexpr (G == 1) {
                    // (rows 0 and 1 of the first lane group; plane 0 in row 2)
                    const int v = acc[kb][0] + 256 * acc[kb][1];
                    if (lane < 16)
                        rdl[16 * kb + lj] = prec ? __builtin_bit_cast(int, (float)v + (float)acc[kb][2] * (1.0f / 256.0f)) : v;
                } else if (lane < 8 * G) {
                    int2 v = make_int2(acc[kb][0] + 256 * acc[kb][1], acc[kb][2] + 256 * acc[kb][3]);
                    if (!LO_COLS && prec)
                        v = make_int2(__builtin_bit_cast(int, (float)v.x + (float)accl[0] * (1.0f / 256.0f)),
                                      __builtin_bit_cast(int, (float)v.y + (float)accl[2] * (1.0f / 256.0f)));
                    *(int2*)&rdl[(16 * kb + lj) * G + 2 * g4] = v;
                }
            }
            if (G > 1 && LO_COLS && prec && g4 == G / 2) {
                // plane 0 (q_int dot * 16 = 65536 plane2 + 256 plane1 + plane0)
                // to rdlo[position][head]: rows 2G + g of the same MFMAs (lane
                // group G/2, i = g)
#pragma unroll
                for (int kb = 0; kb < 4; kb++) {
                    if (kb >= nkb) break;
#pragma unroll
                    for (int g = 0; g < (LO_COLS && G > 1 ? G : 1); g++) rdlo[(16 * kb + lj) * G + g] = acc[kb][g];
                }
            }
            if constexpr (APP) {
                // (APP) the token's dots over the slot's, after them
                if (has_token) {
                    const int rel = a.app_slot - t0, g = opaque_int(lane);
                    if (g < G) {
                        const int v = token->dot[g], vl = token->dot_lo[g];
                        const bool joined = prec && (G == 1 || !LO_COLS);   // (one float, as above)
                        rdl[rel * G + g] = joined ? __builtin_bit_cast(int, (float)v + (float)vl * (1.0f / 256.0f)) : v;
                        if (G > 1 && LO_COLS) rdlo[rel * G + g] = vl;
                    }
                }
            }
            __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
            // kept x16: the factor is folded into the score's scale below
            // (lanes past the written positions read values they never use)
            if constexpr (G % 4 == 0) {
#pragma unroll
                for (int g = 0; g < G; g += 4) {
                    const int4 v = *(const int4*)&rdl[rpos * G + g];
                    racc[g] = v.x; racc[g + 1] = v.y; racc[g + 2] = v.z; racc[g + 3] = v.w;
                }
            } else {
#pragma unroll
                for (int g = 0; g < G; g++) racc[g] = rdl[rpos * G + g];
            }
            if (G > 1 && LO_COLS && prec) {
#pragma unroll
                for (int g = 0; g < G; g++)
                    racc[g] = __builtin_bit_cast(int, (float)racc[g] + (float)rdlo[rpos * G + g] * (1.0f / 256.0f));
            }
          }
        } else if constexpr (RES) {
            // (adaptive single heads: the lane's own key)
            int s0 = 0, s1 = 0, s2 = 0, s3 = 0;
#pragma unroll
            for (int w = 0; w < CW; w++) {
                s0 = __builtin_amdgcn_sdot8(sdig[w][0], (int)kc[w], s0, false);
                s1 = __builtin_amdgcn_sdot8(sdig[w][1], (int)kc[w], s1, false);
                s2 = __builtin_amdgcn_sdot8(sdig[w][2], (int)kc[w], s2, false);
                s3 = __builtin_amdgcn_sdot8(sdig[w][3], (int)kc[w], s3, false);
            }
            racc[0] = s0 + 16 * s1 + 256 * s2 + 4096 * s3;
            if (prec) {
                int l0 = 0, l1 = 0;
#pragma unroll
                for (int w = 0; w < CW; w++) {
                    const int2 dl = qd.digits_lo[0][w];
                    l0 = __builtin_amdgcn_sdot8(dl.x, (int)kc[w], l0, false);
                    l1 = __builtin_amdgcn_sdot8(dl.y, (int)kc[w], l1, false);
                }
                racc[0] = __builtin_bit_cast(int, (float)racc[0] + (float)(l0 + 16 * l1) * (1.0f / 256.0f));
            }
        }
        float sc[G];
#pragma unroll
        for (int g = 0; g < G; g++) {
            float score = xd[g];
            bool use_res = MODE == MODE_COMP;
            if constexpr (MODE == MODE_ADAPTIVE) use_res = (selmask >> g) & 1u;
            if constexpr (MODE == MODE_MIXED) use_res = hmode[g];
            // the dot in units of dq (the matrix-core dots come x16, an exact
            // power of two; in a precise tile they are float bits already)
            const float rd = prec ? __builtin_bit_cast(float, racc[g]) : (float)racc[g];
            if (RES && use_res)
                score = fmaf(rd, qd.dq[g] * (rsk * (KMF ? 1.0f / 112.0f : 1.0f / 7.0f)), score);
            sc[g] = valid ? score * isd2 : -INFINITY;
        }

        // (fp16 path) weight scale: weights are p * wb * 2^wexp with p <= 2^kTau,
        // so the plan holds while every wb <= wlim = 2^(kWTop - kTau - wexp); it is
        // redone (one wave max) only when a key exceeds it, and then only lowered
        if constexpr (!I8) {
            // (a scale that is not finite takes no part: the heads that read it are
            // NaN whatever the plan, a head that reads only the key's other part
            // needs its weights planned all the same)
            const float wa = 2.0f * fabsf(svv), wr = fabsf(rsv) * (1.0f / 7.0f);
            const float wb = valid ? fmaxf(wa < INFINITY ? wa : 0.0f, wr < INFINITY ? wr : 0.0f) : 0.0f;
            if (__ballot(wb > wlim) != 0ull) {
                const float wmx = wave_max(wb);
                const int e = kWTop - kTauI - (int)ceilf(log2f(wmx));
                if (have_wexp) {
                    // a larger weight than planned (e < wexp): bring the sums down
                    const float f = ldexpf(1.0f, e - wexp);
#pragma unroll
                    for (int h = 0; h < (I8 ? 0 : NH); h++)
#pragma unroll
                        for (int p = 0; p < 4; p++) cs[h][p] *= f;
#pragma unroll
                    for (int d = 0; d < (I8 ? 0 : NB); d++) cn[d] *= f;
#pragma unroll
                    for (int g = 0; g < G; g++) off[g] *= f;
                }
                wexp = e;
                have_wexp = true;
                wlim = ldexpf(1.0f, kWTop - kTauI - wexp);
            }
        }

        // online softmax; (hi, lo) fp16 weights, or the digits of the integer
        // weights, to LDS in MFMA slot order
        float lane_alpha = 1.0f;   // the factor of the lane's head's sums so far
        bool any_rescale = false;
        // the value operands of odd rows come out 16x larger (see the MFMA
        // loops below): their weights carry 1/16 so that every product is exact
        // (the residual row of a key is its compacted position's row, of the
        // parity of rpos); the int8 elements carry no such factor
        const float kfac = (!I8 && (kown & 1)) ? 0.0625f : 1.0f;
        const float kfac_res = (!I8 && (rpos & 1)) ? 0.0625f : 1.0f;
        // per-key factors shared by the heads: sign weight a2 = p * fa, residual
        // weight b = p * fb; (fp16) the offset sum_s (a_s + 8 b_s) grows by p * fo
        const float fa = I8 ? 2.0f * svv : ldexpf(2.0f * svv * kfac, wexp);
        const float fb = !RES ? 0.0f : I8 ? rsv * (1.0f / 7.0f) : ldexpf(rsv * (1.0f / 7.0f) * kfac_res, wexp);
        const float fo_bin = I8 ? 0.0f : ldexpf(svv, wexp);
        const float fo_res = (RES && !I8) ? ldexpf(svv + rsv * (8.0f / 7.0f), wexp) : fo_bin;
        // residual weights go to the slot of the key's residual position
        // (adaptive: compacted; unselected keys write zeros to the positions
        // past nsel, so every slot a residual MFMA reads is written)
        uint16_t* wres = wsl;
        uint8_t* w8res = w8st;
        if constexpr (MODE == MODE_ADAPTIVE && I8)
            w8res = &lds_w8[0][0] + opaque_int((wave * 64 + slot8_of(res_row(rpos))) * kWRow);
        else if constexpr (MODE == MODE_ADAPTIVE)
            wres = &lds_wts[0][0] + opaque_int(wave * (WL::kWeightBytes / 2) + slot_of(res_row(rpos)));
        // does head g take the key's residual
        auto with_res = [&](int g) {
            if constexpr (MODE == MODE_MIXED) return hmode[g];
            if constexpr (MODE == MODE_ADAPTIVE) return (bool)((selmask >> g) & 1u);
            return MODE == MODE_COMP;
        };
        // (int8 path) p es per head, its sign and residual weights plus 1/2, and
        // the heads whose reference moved
        float ps[G], wsig[G], wresid[G], wtop = 0.0f;
        uint32_t moved = 0u;
#pragma unroll
        for (int g = 0; g < G; g++) {
            // the reference m[g] moves only when a score passes m[g] + kTau
            if (__ballot(sc[g] > mlim[g]) != 0ull) {
                const float mn = uniform_f(fmaxf(m[g], wave_max(sc[g])));
                const float alpha = __builtin_amdgcn_exp2f(m[g] - mn);   // 0 when m was -inf
                lsum[g] *= alpha;
                off[g] *= alpha;
                if (my_head == g) lane_alpha = alpha;
                any_rescale = true;
                moved |= 1u << g;
                m[g] = mn;
                mlim[g] = mn + kTau;
            }
            const float p = valid ? __builtin_amdgcn_exp2f(sc[g] - m[g]) : 0.0f;
            lsum[g] += p;
            if constexpr (I8) {
                ps[g] = p * es[g];
                wsig[g] = fmaf(ps[g], fa, 0.5f);
                wtop = fmaxf(wtop, fabsf(wsig[g]));
                if constexpr (RES) {
                    wresid[g] = fmaf(ps[g], with_res(g) ? fb : 0.0f, 0.5f);
                    wtop = fmaxf(wtop, fabsf(wresid[g]));
                }
            } else {
                const float a2 = p * fa;
                const float bv = with_res(g) ? p * fb : 0.0f;
                // the offset a + 8 b of each key, taken off at the end: the (hi, lo)
                // pairs carry ~22 bits, a zero-mean difference
                off[g] = fmaf(p, with_res(g) ? fo_res : fo_bin, off[g]);
                const uint16_t a2h = f2h_bits(a2);
                const uint16_t a2l = f2h_bits(a2 - h_bits2f(a2h));
                wsl[(0 * 2 * G + 2 * g) * WL::kColSlots] = a2h;
                wsl[(0 * 2 * G + 2 * g + 1) * WL::kColSlots] = a2l;
                if constexpr (RES) {
                    const uint16_t bh = f2h_bits(bv);
                    const uint16_t bl = f2h_bits(bv - h_bits2f(bh));
                    wres[(kRes0 + 2 * g) * WL::kColSlots] = bh;
                    wres[(kRes0 + 2 * g + 1) * WL::kColSlots] = bl;
                }
            }
        }
        uint32_t dsig[G], dres[G];   // (int8 path) packed digits
        if constexpr (I8) {
            if (moved != 0u || __ballot(wtop >= kW8Max) != 0ull) {
                // (weights that are not finite take no part: their head is NaN,
                // below, and the group's other heads do not have them)
                uint32_t wmx[G];
#pragma unroll
                for (int g = 0; g < G; g++) {
                    float w = fabsf(wsig[g]) < INFINITY ? fabsf(wsig[g]) : 0.0f;
                    if constexpr (RES) w = fmaxf(w, fabsf(wresid[g]) < INFINITY ? fabsf(wresid[g]) : 0.0f);
                    wmx[g] = __builtin_bit_cast(uint32_t, w);
                }
                wave_umax(wmx);
#pragma unroll
                for (int g = 0; g < G; g++) {
                    if ((moved >> g & 1u) || wmx[g] >= __builtin_bit_cast(uint32_t, kW8Max)) {
                        // the largest weight is in [2^(e - 1), 2^e), e = its exponent
                        // field - 126; 2^kW8Top-e by its own exponent field
                        const int e = (int)(wmx[g] >> 23) - 126;
                        const float en = fminf(es[g] * __builtin_bit_cast(float, (uint32_t)(127 + kW8Top - e) << 23), kEsMax);
                        const float f = uniform_f(en * pow2_inv(es[g]));
                        es[g] = uniform_f(en);
                        ps[g] *= f;
                        off[g] *= f;
                        wsig[g] = fmaf(ps[g], fa, 0.5f);
                        if constexpr (RES) wresid[g] = fmaf(ps[g], with_res(g) ? fb : 0.0f, 0.5f);
                        if (my_head == g) lane_alpha *= f;
                        any_rescale = true;
                    }
                }
            }
            // a V scale that is not finite has no integer weight: it makes the
            // offset, so the output of the heads that read it, NaN, as the sums
            // of the fp16 path are
            if (__ballot(!(fabsf(svv) + (RES ? fabsf(rsv) : 0.0f) < INFINITY)) != 0ull) {
#pragma unroll
                for (int g = 0; g < G; g++) off[g] += svv * 0.0f + (with_res(g) ? rsv * 0.0f : 0.0f);
            }
#pragma unroll
            for (int g = 0; g < G; g++) {
                // (truncation after adding 1/2 rounds; a scale that is negative, as no
                // encoder writes one, rounds up)
                const int w = (int)wsig[g];
                // the offset a = a2 / 2 of each key, taken off at the end: half the
                // rounded weight, so that the key's sum stays +-a of one a (half
                // the unrounded one moves every dimension of the head the same
                // way, by the rounding errors of all keys)
                off[g] = fmaf(0.5f, (float)w, off[g]);
                // balanced digits
                dsig[g] = ((uint32_t)w + 0x80808080u) ^ 0x80808080u;
                if constexpr (RES) dres[g] = ((uint32_t)(int)wresid[g] + 0x80808080u) ^ 0x80808080u;
            }
        }
        if constexpr (I8 && G == 4) {
            *(v4u_t*)w8st = v4u_t{dsig[0], dsig[1], dsig[2], dsig[3]};
            if constexpr (R8) *(v4u_t*)(w8res + 16) = v4u_t{dres[0], dres[1], dres[2], dres[3]};
        } else if constexpr (I8 && G == 2) {
            if constexpr (R8 && ALLRES) {
                *(v4u_t*)w8st = v4u_t{dsig[0], dsig[1], dres[0], dres[1]};
            } else {
                *(v2u_t*)w8st = v2u_t{dsig[0], dsig[1]};
                if constexpr (R8) *(v2u_t*)(w8res + 8) = v2u_t{dres[0], dres[1]};
            }
        } else if constexpr (I8) {
            if constexpr (R8 && ALLRES) {
                *(v2u_t*)w8st = v2u_t{dsig[0], dres[0]};
            } else {
                *(uint32_t*)w8st = dsig[0];
                if constexpr (R8) *(uint32_t*)(w8res + 4) = dres[0];
            }
        }
        if constexpr (I8) {
            // the integer sums so far move to the float bank, scaled by this
            // tile's factors (rare: a score passed m + kTau, a weight kW8Max, or
            // the residual sums are full)
            if (live8 > 0 && (any_rescale || (R8 && live8 >= kMaxTiles8))) flush8(lane_alpha);
        } else if (any_rescale) {
            if (my_head >= G) lane_alpha = 1.0f;
#pragma unroll
            for (int h = 0; h < NH; h++)
#pragma unroll
                for (int p = 0; p < 4; p++) cs[h][p] *= lane_alpha;
#pragma unroll
            for (int d = 0; d < NB; d++) cn[d] *= lane_alpha;
        }

        // this tile's V data must be in LDS: everything but the next tile's
        // loads (the youngest kPrefetchOps vector-memory operations) completes
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (MODE != MODE_ADAPTIVE && PIPE) {
            constexpr int n = kPrefetchOps;
            __builtin_amdgcn_s_waitcnt((n & 0xF) | ((n >> 4) << 14) | (0x7 << 4) | (0xF << 8));
        } else if constexpr (MODE != MODE_ADAPTIVE) {
            __builtin_amdgcn_s_waitcnt(0);
        }
        // (adaptive mode: the compiler waits for this staging buffer's loads)
        if constexpr (APP) {
            if (has_token) {   // the token's V row over the slot's
                const int rel = a.app_slot - t0, ln = opaque_int(lane);
                if (ln < SB / 4) ((uint32_t*)(st_signs + WL::kSignStride * rel))[ln] = token->signs[1][ln];
                if constexpr (RES) {
                    const int sw = Q_POW2 ? ((rel * CB) >> 8) & (Q - 1) : 0;
                    if (ln < CB / 4)
                        ((uint32_t*)(st_codes + CB * rel + 16 * ((ln >> 2) ^ sw)))[ln & 3] = token->codes[1][ln];
                }
            }
        }
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the weight stores above
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");

        // B operands: (hi, lo) weight columns (lanes of unused columns read
        // columns 0/1 again, their output columns are never read back), or
        // the digit columns of the int8 rows
        h8_t bsig[2], bres[2];
        v4i_t b8 = v4i_t{0, 0, 0, 0}, b8r = v4i_t{0, 0, 0, 0};
        if constexpr (I8) {
            auto columns = [&](const uint8_t* at) {
                const v2i_t lo = __builtin_amdgcn_ds_read_tr8_b64_v2i32(LDS_PTR(v2i_t, at));
                const v2i_t hi = __builtin_amdgcn_ds_read_tr8_b64_v2i32(LDS_PTR(v2i_t, at + 8 * kWRow));
                return v4i_t{lo.x, lo.y, hi.x, hi.y};
            };
            b8 = columns(w8rd);
            b8r = b8;
            if constexpr (R8 && G == 4) b8r = columns(w8rd + 16);
        } else {
#pragma unroll
            for (int mh = 0; mh < 2; mh++) {
                bsig[mh] = *(const h8_t*)&wrd[8 * mh];
                if constexpr (RES) bres[mh] = *(const h8_t*)&wrd[kRes0 * WL::kColSlots + 8 * mh];
                else bres[mh] = bsig[mh];
            }
        }

        // all transposed reads of the tile first (they retire in order while
        // the MFMAs of earlier blocks run)
        const int row_key = 16 * g4 + lj;  // this lane addresses row (key) lj of its group
        // MFMA halves that hold residual positions (adaptive: ceil(nsel / 32))
        const int nmh = (nsel + 31) >> 5;
        v2i_t wsg[NH];
#pragma unroll
        for (int h = 0; h < NH; h++)
            wsg[h] = __builtin_amdgcn_ds_read_tr4_b64_v2i32(LDS_PTR(v2i_t, st_signs + WL::kSignStride * row_key + 8 * h));
        v2i_t wrs[RES ? NB : 1];
        if constexpr (RES) {
            if (nmh > 0) {
#pragma unroll
                for (int db = 0; db < NB; db++) {
                    const uint8_t* rp = LIN_V ? st_codes + CB * row_key + 16 * ((db >> 1) ^ vsw) + 8 * (db & 1)
                                              : st_codes + (db >> 1) * 1024 + 16 * row_key + 8 * (db & 1);
                    wrs[db] = __builtin_amdgcn_ds_read_tr4_b64_v2i32(LDS_PTR(v2i_t, rp));
                }
            }
        }

        // sign part: rows = dims 64h + 4*lj + p
        if constexpr (I8) {
            // int8: the lane's 16 keys (first word keys 0..7, second 8..15,
            // nibble r = key r) as bytes holding bit p of their nibble in
            // place (element 2^p): even nibbles from the word, odd ones from
            // the word >> 4, one AND per four keys; all 64 keys in one MFMA
#pragma unroll
            for (int h = 0; h < NH; h++) {
                const uint32_t x = (uint32_t)wsg[h].x, y = (uint32_t)wsg[h].y;
                const uint32_t x4 = x >> 4, y4 = y >> 4;
#pragma unroll
                for (int p = 0; p < 4; p++) {
                    const uint32_t msk = 0x01010101u << p;
                    const v4i_t av = v4i_t{(int)(x & msk), (int)(x4 & msk), (int)(y & msk), (int)(y4 & msk)};
                    ci[h][p] = __builtin_amdgcn_mfma_i32_16x16x64_i8(av, b8, ci[h][p], 0, 0, 0);
                }
            }
            live8++;
        }
#pragma unroll
        for (int h = 0; h < (I8 ? 0 : NH); h++) {
#pragma unroll
            for (int mh = 0; mh < 2; mh++) {
                // x holds nibble r of key r (r = 0..3) and of key r + 4 (bits
                // 16 + 4r): pair word k keeps bit p of keys k and k + 4 in place,
                // an fp16 subnormal 2^(4(k&1) + p - 24); keys 2, 3 via x >> 8
                const uint32_t x = (uint32_t)(mh ? wsg[h].y : wsg[h].x);
                const uint32_t y = x >> 8;
#pragma unroll
                for (int p = 0; p < 4; p++) {
                    uint32_t pw[4];
                    pw[0] = x & (0x00010001u << p);
                    pw[1] = x & (0x00100010u << p);
                    pw[2] = y & (0x00010001u << p);
                    pw[3] = y & (0x00100010u << p);
                    const h8_t av = __builtin_bit_cast(h8_t, pw);
                    cs[h][p] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av, bsig[mh], cs[h][p], 0, 0, 0);
                }
            }
        }

        // residual part: rows = dims 16db + lj
        auto res_mfma = [&](int db, int mh) {
            // u = n + 8 in place: keys k, k + 4 at 4(k&1) (odd keys 16x)
            const uint32_t x = (uint32_t)(mh ? wrs[db].y : wrs[db].x) ^ 0x88888888u;
            const uint32_t y = x >> 8;
            uint32_t pw[4];
            pw[0] = x & 0x000F000Fu;
            pw[1] = x & 0x00F000F0u;
            pw[2] = y & 0x000F000Fu;
            pw[3] = y & 0x00F000F0u;
            const h8_t av = __builtin_bit_cast(h8_t, pw);
            cn[db] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av, bres[mh], cn[db], 0, 0, 0);
        };
        if constexpr (MODE == MODE_ADAPTIVE && R8) {
            // positions 0..31 are the first words, the second ones only past 32
            if (nmh == 1) {
#pragma unroll
                for (int db = 0; db < NB; db++) {
                    const uint32_t x = (uint32_t)wrs[db].x;
                    const v4i_t av = v4i_t{(int)((x << 4) & 0xF0F0F0F0u), (int)(x & 0xF0F0F0F0u), 0, 0};
                    cr[db] = __builtin_amdgcn_mfma_i32_16x16x64_i8(av, b8r, cr[db], 0, 0, 0);
                }
            } else if (nmh == 2) {
#pragma unroll
                for (int db = 0; db < NB; db++)
                    cr[db] = __builtin_amdgcn_mfma_i32_16x16x64_i8(codes_i8((uint32_t)wrs[db].x, (uint32_t)wrs[db].y), b8r, cr[db], 0, 0, 0);
            }
        } else if constexpr (MODE == MODE_ADAPTIVE) {
            // half 0 when any key is selected, half 1 only past 32 of them
#pragma unroll
            for (int mh = 0; mh < 2; mh++) {
                if (mh >= nmh) break;
#pragma unroll
                for (int db = 0; db < NB; db++) res_mfma(db, mh);
            }
        } else if constexpr (R8) {
            // int8: the lane's 16 keys of dimension 16db + lj as bytes 16 n,
            // in the sign part's slot order
#pragma unroll
            for (int db = 0; db < NB; db++)
                cr[db] = __builtin_amdgcn_mfma_i32_16x16x64_i8(codes_i8((uint32_t)wrs[db].x, (uint32_t)wrs[db].y), b8r, cr[db], 0, 0, 0);
        } else if constexpr (RES) {
#pragma unroll
            for (int db = 0; db < NB; db++) {
                res_mfma(db, 0);
                res_mfma(db, 1);
            }
        }
        // the staging buffer is refilled two tiles later: its reads retire here
        __builtin_amdgcn_s_waitcnt(0xC07F);
        __builtin_amdgcn_wave_barrier();
    };

    // ---------------- software-pipelined tile loop: tile i+1 loads in flight
    // while tile i computes (two register sets, two LDS staging buffers).  The
    // prefetch after a wave's last tile addresses the tile past the range: its
    // loads return zeros and move no data, and no load sits behind a branch.  Every iteration of the two-tile
    // loop starts with no load in flight: the compiler follows direct loads to
    // LDS per staging buffer only within an iteration (across the back edge it
    // would wait for all of them at the first staging-buffer read), so the
    // prefetch issued before an iteration's second tile lands by its end.
    if constexpr (MODE == MODE_ADAPTIVE) {
        // popcounts and binary scales two tiles ahead, selection and residual
        // gathers one tile ahead; each iteration (two tiles) starts with no
        // load in flight and every load has a tile of compute to land
        if (t < key_end) {
            KR ra, rb, rc, rd;
            load_k(ra, t);
            load_k(rb, t + NW * 64);
            gather(ra, t, 0);
            __builtin_amdgcn_s_waitcnt(0);
            for (;;) {
                const int t1 = t + NW * 64;
                gather(rb, t1, 1);
                load_k(rc, t + 2 * NW * 64);
                load_k(rd, t + 3 * NW * 64);
                process(ra, t, 0);
                if (t1 >= key_end) break;
                // ra is free: it takes the popcounts and scales of tile t + 512
                // and receives that tile's residual gathers
                ra.pcw[0] = rc.pcw[0]; ra.pcw[1] = rc.pcw[1]; ra.pcw[2] = rc.pcw[2]; ra.pcw[3] = rc.pcw[3];
                ra.sk = rc.sk;
                ra.svv = rc.svv;
                gather(ra, t + 2 * NW * 64, 0);
                process(rb, t1, 1);
                t += 2 * NW * 64;
                if (t >= key_end) break;
                __builtin_amdgcn_s_waitcnt(0);
                rb.pcw[0] = rd.pcw[0]; rb.pcw[1] = rd.pcw[1]; rb.pcw[2] = rd.pcw[2]; rb.pcw[3] = rd.pcw[3];
                rb.sk = rd.sk;
                rb.svv = rd.svv;
            }
            __builtin_amdgcn_s_waitcnt(0);
            __builtin_amdgcn_wave_barrier();
        }
    } else if (!PIPE) {
        bool issued = early;   // (the first tile's loads went out before the preparation)
        for (; t < key_end; t += NW * 64) {
            if (!issued) {
                load_k(ka, t);
                issue_v(0, t);
            }
            issued = false;
            process(ka, t, 0);
        }
        __builtin_amdgcn_s_waitcnt(0);
        __builtin_amdgcn_wave_barrier();
    } else if (t < key_end) {
        if (!early) {
            load_k(ka, t);
            issue_v(0, t);
        }
        __builtin_amdgcn_s_waitcnt(0);
        for (;;) {
            int tp = t + NW * 64;
            load_k(kb, tp);
            issue_v(1, tp);
            process(ka, t, 0);
            t += NW * 64;
            if (t >= key_end) break;
            tp = t + NW * 64;
            load_k(ka, tp);
            issue_v(0, tp);
            process(kb, t, 1);
            t += NW * 64;
            if (t >= key_end) break;
            __builtin_amdgcn_s_waitcnt(0);
        }
        // the last prefetch still writes LDS that the epilogue reuses
        __builtin_amdgcn_s_waitcnt(0);
        __builtin_amdgcn_wave_barrier();
    }

    // ---------------- epilogue: per wave, per head: acc[e] = ((cs + cn) * unit - off) * 2^-wexp,
    // then the four waves' partials are merged.  Heads pass through staging
    // buffer 0 kEpiHeads at a time ([parts][kEpiHeads][D] floats per wave).
    constexpr int HP = WL::kEpiHeads;
    const float two24 = 16777216.0f;
    // the wave's reference, sums and weight scale per head (published by the
    // first barrier below)
#pragma unroll
    for (int g = 0; g < G; g++) {
        const float l_w = wave_sum63(lsum[g]);
        const float o_w = wave_sum63(off[g]);
        if (lane == 63) {
            wm[wave][g] = m[g];
            wlsum[wave][g] = l_w;
            wofs[wave][g] = o_w;
            wsc[wave][g] = I8 ? pow2_inv(es[g]) : ldexpf(1.0f, -wexp);
        }
    }
    // groups of eight form the merge's factors once per head (one barrier more;
    // the first below publishes them), not for each of its elements: binary 64
    // groups of 200 keys, d = 256, 15.7 -> 14.5 us, compensated 21.2 -> 20.4
    // (smaller groups form them per element and save the barrier)
    if constexpr (G == 8) {
        lds_barrier();
        if (threadIdx.x < G) {
            const int g = threadIdx.x;
            float M = -INFINITY, L = 0.0f;
#pragma unroll
            for (int w = 0; w < NW; w++) M = fmaxf(M, wm[w][g]);
#pragma unroll
            for (int w = 0; w < NW; w++) {
                const float f = wm[w][g] != -INFINITY ? __builtin_amdgcn_exp2f(wm[w][g] - M) : 0.0f;
                if (wm[w][g] != -INFINITY) L += f * wlsum[w][g];
                wfac[w][g] = f * wsc[w][g];
            }
            wtot[0][g] = M;
            wtot[1][g] = L;
        }
    }
    float* accw = (float*)lds_st0[wave];
    const float dscale = digit_scale();
    const float* const bank = bank_at();
    // hi + lo columns are adjacent lanes (col 2g, 2g+1); the even lane writes.
    // int8 path: the digit columns of a head are one lane quad; its first
    // lane writes
    const bool writer = I8 ? owner8 : (my_col < 2 * G && (my_col & 1) == 0);
    // the sign part's unit: 2^-24 (fp16 subnormal elements) or 1 (int8)
    const float sunit = I8 ? 1.0f : two24;
    for (int g0 = 0; g0 < G; g0 += HP) {
        const int hs = my_head - g0;   // this lane's head slot in the batch
        const bool wr = writer && hs >= 0 && hs < HP;
        const int rhs = my_rhead - g0;
        const bool rwr = (R8 ? rowner8 : my_col < 2 * G && (my_col & 1) == 0) && rhs >= 0 && rhs < HP;
        if (g0 > 0) __syncthreads();   // the previous batch has been read
        // hi + lo: the neighbour lane's column by DPP (quad_perm [1,0,3,2]),
        // all sums first, then the stores under one branch
        float sv[I8 ? 1 : NH][4][4];
        float nv[RES ? NB : 1][4];
        if constexpr (I8) {
            // one 64-dim block at a time (accumulator p carries 2^p: bit p
            // read in place)
#pragma unroll
            for (int h = 0; h < NH; h++) {
#pragma unroll
                for (int p = 0; p < 4; p++)
#pragma unroll
                    for (int i = 0; i < 4; i++) sv[0][p][i] = digits(ci[h][p][i], dscale);
                if (wr && 64 * h + 16 * g4 < D) {
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        // plus the banked sums of the keys before the last rescale
                        float4 b = make_float4(0.f, 0.f, 0.f, 0.f);
                        if (banked) b = *(const float4*)&bank[64 * h + 4 * (4 * g4 + i)];
                        const float bb[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
                        for (int p = 0; p < 4; p++)
                            accw[(0 * HP + hs) * D + 64 * h + 4 * (4 * g4 + i) + p] =
                                sv[0][p][i] * (1.0f / (float)(1 << p)) + bb[p];
                    }
                }
            }
        } else {
#pragma unroll
            for (int h = 0; h < NH; h++)
#pragma unroll
                for (int p = 0; p < 4; p++)
#pragma unroll
                    for (int i = 0; i < 4; i++)
                        // accumulator p carries 2^p (bit p read in place)
                        sv[h][p][i] = (cs[h][p][i] + dpp_f<0xB1>(cs[h][p][i])) * (1.0f / (float)(1 << p));
        }
        if constexpr (RES) {
#pragma unroll
            for (int d = 0; d < NB; d++)
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    if constexpr (R8) nv[d][i] = digits(cr[d][i], dscale) * (1.0f / 16.0f);   // (codes as 16 n)
                    else nv[d][i] = cn[d][i] + dpp_f<0xB1>(cn[d][i]);
                }
        }
        if (wr) {
#pragma unroll
            for (int h = 0; h < (I8 ? 0 : NH); h++) {
                if (64 * h + 16 * g4 >= D) continue;   // (the half block past d)
#pragma unroll
                for (int p = 0; p < 4; p++)
#pragma unroll
                    for (int i = 0; i < 4; i++)
                        accw[(0 * HP + hs) * D + 64 * h + 4 * (4 * g4 + i) + p] = sv[I8 ? 0 : h][p][i];
            }
        }
        if constexpr (RES) {
            if (rwr) {
#pragma unroll
                for (int d = 0; d < NB; d++)
#pragma unroll
                    for (int i = 0; i < 4; i++)
                        accw[(1 * HP + rhs) * D + 16 * d + 4 * g4 + i] = nv[d][i];
            }
        }
        __syncthreads();
        const int nh = min(HP, G - g0);
        for (int i = threadIdx.x; i < nh * D; i += blockDim.x) {
            const int hs2 = i / D, e = i % D, g = g0 + hs2;
            // the maximum M over the waves, each wave's factor 2^(m_w - M)
            // (0 for a wave without keys) and the total l
            float mw[NW], M = -INFINITY, accv = 0.0f, L = 0.0f;
            if constexpr (G == 8) {
                M = wtot[0][g];
                L = wtot[1][g];
            } else {
#pragma unroll
                for (int w = 0; w < NW; w++) {
                    mw[w] = wm[w][g];
                    M = fmaxf(M, mw[w]);
                }
            }
#pragma unroll
            for (int w = 0; w < NW; w++) {
                const float* aw = (const float*)lds_st0[w];
                float v = aw[(0 * HP + hs2) * D + e];
                if (RES) v += aw[(1 * HP + hs2) * D + e];
                if constexpr (G == 8) {
                    const float f = wfac[w][g];
                    accv += f != 0.0f ? (v * sunit - wofs[w][g]) * f : 0.0f;
                } else {
                    const bool live = mw[w] != -INFINITY;
                    const float f = live ? __builtin_amdgcn_exp2f(mw[w] - M) : 0.0f;
                    accv += live && f != 0.0f ? (v * sunit - wofs[w][g]) * (f * wsc[w][g]) : 0.0f;
                    if (live) L += f * wlsum[w][g];
                }
            }
            if (a.out != nullptr) {
                // one split: the output itself, normalised as the merge of a
                // single partial would (factor 1, sum l)
                a.out[(int64_t)(bhq0 + g) * D + e] = f2h(L > 0.0f ? accv * (1.0f / L) : 0.0f);
            } else {
                float* dst = a.ws + ((int64_t)(bhq0 + g) * a.n_splits + split) * (D + 2);
                dst[2 + e] = accv;
                if (e == 0) {
                    dst[0] = M;
                    dst[1] = L;
                }
            }
        }
    }
}

// Wide workgroups (one split per group, the output written directly): MHA
// binary attention at d = 64, 128, 256 with 8 waves; false for any other
// request.
template <int D>
bool launch_wide(int mode, int G, const AttnArgs& a, dim3 grid, hipStream_t st, int nw) {
    if constexpr (D == 64 || D == 128 || D == 256) {
        if (mode == MODE_BINARY && G == 1 && nw == 8) {
            hipLaunchKernelGGL((attn_mfma_kernel<D, 1, MODE_BINARY, 8>), grid, dim3(8 * 64), 0, st, BC_MFMA_ARGS(a, 1));
            return true;
        }
    }
    return false;
}

template <int D, int G>
void launch_dg(int mode, const AttnArgs& a, dim3 grid, hipStream_t st) {
    if constexpr (bc::append_dim(D)) {
        if (a.app_k != nullptr) {
            if (mode == MODE_BINARY)
                hipLaunchKernelGGL((attn_mfma_kernel<D, G, MODE_BINARY, 4, true>), grid, dim3(256), 0, st, BC_MFMA_ARGS(a, G));
            else
                hipLaunchKernelGGL((attn_mfma_kernel<D, G, MODE_COMP, 4, true>), grid, dim3(256), 0, st, BC_MFMA_ARGS(a, G));
            return;
        }
    }
    if (mode == MODE_BINARY)
        hipLaunchKernelGGL((attn_mfma_kernel<D, G, MODE_BINARY>), grid, dim3(256), 0, st, BC_MFMA_ARGS(a, G));
    else if (mode == MODE_COMP)
        hipLaunchKernelGGL((attn_mfma_kernel<D, G, MODE_COMP>), grid, dim3(256), 0, st, BC_MFMA_ARGS(a, G));
    else if (mode == MODE_MIXED)
        hipLaunchKernelGGL((attn_mfma_kernel<D, G, MODE_MIXED>), grid, dim3(256), 0, st, BC_MFMA_ARGS(a, G));
    else
        hipLaunchKernelGGL((attn_mfma_kernel<D, G, MODE_ADAPTIVE>), grid, dim3(256), 0, st, BC_MFMA_ARGS(a, G));
}

template <int D, int G>
int occupancy_dg(int mode) {
    int n = 0;
    hipError_t e;
    if (mode == MODE_BINARY)
        e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, attn_mfma_kernel<D, G, MODE_BINARY>, 256, 0);
    else if (mode == MODE_COMP)
        e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, attn_mfma_kernel<D, G, MODE_COMP>, 256, 0);
    else if (mode == MODE_MIXED)
        e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, attn_mfma_kernel<D, G, MODE_MIXED>, 256, 0);
    else
        e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, attn_mfma_kernel<D, G, MODE_ADAPTIVE>, 256, 0);
    return e == hipSuccess ? n : 0;
}

}  // namespace

namespace bc {

template <int D>
bool mfma_launch(int mode, int G, const AttnArgs& a, dim3 grid, hipStream_t st, int nw) {
    if (a.app_k != nullptr && (!append_dim(D) || mode == MODE_ADAPTIVE || mode == MODE_MIXED)) return false;
    if (nw != 4) return launch_wide<D>(mode, G, a, grid, st, nw);
    switch (G) {
        case 8: launch_dg<D, 8>(mode, a, grid, st); break;
        case 4: launch_dg<D, 4>(mode, a, grid, st); break;
        case 2: launch_dg<D, 2>(mode, a, grid, st); break;
        default: launch_dg<D, 1>(mode, a, grid, st); break;
    }
    return true;
}

template <int D>
int mfma_occupancy(int mode, int G) {
    switch (G) {
        case 8: return occupancy_dg<D, 8>(mode);
        case 4: return occupancy_dg<D, 4>(mode);
        case 2: return occupancy_dg<D, 2>(mode);
        default: return occupancy_dg<D, 1>(mode);
    }
}

}  // namespace bc
