// Matvecs over more activation columns than the dot4 kernels or the int8-MFMA
// classes do best (rq_cols_*, either weight layout, rq_params.h) and the fused
// gate/up front half of a gated FFN (rq_colsglu_*, the dot4 layout); on the
// same weight sources the f16 GEMM route's kernels for short prompts
// (rq_gemm_*, at the end). Which calls come
// here, and both sides' times: use_cols and gemm_fused in rq_host.cpp.
//
// What bounds them. Every weight is read once, so a launch cannot be faster
// than its bytes, which none is close to (counters below). The work beside
// it is per (row, 32-element block, column): the block's exact dot has to be
// scaled by the activation block's own scale before it is summed. With
// int8 MFMAs (K = 64, two blocks) that took half-empty operands and three
// VALU instructions per block dot, conversion, sub-block scale and sum, which
// bounded everything past 8 columns. Here a block is one
// v_mfma_f32_16x16x32_f16: K is exactly the block, and the weight operand
// holds sc q (Q4_K), the codes times their integer sub-block scale,
// which f16 represents exactly, so that the f32 result is the exact integer
// sc * dot (|sum| < 2^24) and one v_fma_mix_f32 with the f16 scale of the
// activation block is all that is left per entry. Q6_K's sc (q - 32) needs 13
// bits: it is the sum of two exact operands, 8 sc ((q >> 3) - 4) and
// sc (q & 7), in two MFMAs over one accumulator. The operands cost 9 to 26
// VALU per 16 rows x 32 elements and are shared by every column.
//
// Split. A workgroup takes RT tiles of 16 rows and all columns (CG groups of
// 16); its eight waves take the row's super-blocks in turn (wave w: s % 8 ==
// w) and meet in a pairwise LDS sum. The order of every sum depends on
// k alone: a column's result is the same at every column count, row count,
// tile split and in both layouts.
//
// Weights. MFMA layout: a lane's 16 bytes are loaded as stored (1 KB per wave
// instruction) and v_permlane32_swap hands each half of a window to all four
// k-groups. Dot4 layout: the workgroup loads eight super-blocks of its rows
// (128 contiguous bytes per row and chunk) through registers into LDS, from
// where each wave reads its own super-block; the copy's slots are permuted by
// row so that the 16 rows a wave reads together lie in different banks.
//
// Activations. Each wave stages the half super-block it works on in LDS of
// its own (no barrier), a column's 128 bytes as one line; a lane then holds
// column lane % 16: the same half swap, and two instructions per two codes
// into f16.
//
// Measured (us, replayed launches over weights beyond the caches; before:
// the dot4 kernels in groups of 8 columns, the int8-MFMA classes):
//   Q4_K 4096 x 4096, dot4 layout, 16 / 64 columns    17.6 / 70.2 -> 7.5 / 16.4
//   Q4_K 14336 x 4096, dot4 layout, 16 / 32           36.7 / 73.0 -> 15.7 / 20.2
//   Q6_K 4096 x 14336, MFMA layout, 16 / 32 / 64      21.7 / 37.7 / 72.8 -> 18.5 / 25.7 / 42.9
//   Q4_K q, k and Q6_K v of width 5120, dot4, 43      211 -> 46 (one launch for six, and the Q8_1 pass)
// Counters of 14336 x 4096 at 16 columns, dot4 layout: 3.87 M VALU
// instructions, 44% of the issue cycles of the CUs that hold a workgroup (Q6_K
// 4096 x 14336 at 32, MFMA layout: 51%), MFMA busy 9 to 13%; the rest is the
// loads' latency (one step in flight, one workgroup per CU) and LDS.

#include "rq_device.h"

#include <type_traits>

typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef u32 v2u __attribute__((ext_vector_type(2)));

extern __shared__ __attribute__((aligned(16))) char cols_lds[];

#define RQ_LAY_DOT4 0
#define RQ_LAY_MFMA 1

__device__ __forceinline__ h2 as_h2(u32 v) { return __builtin_bit_cast(h2, v); }
__device__ __forceinline__ h2 splat(_Float16 v) { return h2{v, v}; }
__device__ __forceinline__ u32 dw(const int4& v, int i) { return (u32)(i == 0 ? v.x : i == 1 ? v.y : i == 2 ? v.z : v.w); }

// An operand register set: eight f16 of one row or column.
struct Op {
    h2 r[4];
    __device__ __forceinline__ h8 v() const { return __builtin_bit_cast(h8, *this); }
};

__device__ __forceinline__ v4f mfma(const Op& a, const Op& b, v4f c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a.v(), b.v(), c, 0, 0, 0);
}

// The k order of an operand. A lane of k-group g holds, of a 32-element
// block, elements 0-7, 16-23, 8-15, 24-31 for g = 0, 1, 2, 3, as two dwords
// u0, u1 of four bytes each; register 2i + p holds bytes p and p + 2 of
// dword i. Weights and activations follow it alike, so that the products
// pair up.
//
// Both halves of a 64-element window as loaded (16 bytes at 16 g): after the
// swap, x is block 0's two dwords of every k-group, y block 1's.
struct Win {
    u32 x[2], y[2];
};
__device__ __forceinline__ Win win_of(const int4& w) {
    const auto a = __builtin_amdgcn_permlane32_swap((u32)w.x, (u32)w.z, false, false);
    const auto b = __builtin_amdgcn_permlane32_swap((u32)w.y, (u32)w.w, false, false);
    return Win{{a[0], b[0]}, {a[1], b[1]}};
}

// A constant kept in a vector register, so that (x & mask) ^ key is one
// instruction: at most one of its operands can be a scalar or a literal.
__device__ __forceinline__ u32 vconst(u32 v) {
    __asm__ volatile("" : "+v"(v));
    return v;
}
struct Masks {
    u32 byte, low, high;  // Q6_K: byte, fields q & 7, q >> 3
};
template <int FMT>
__device__ __forceinline__ Masks masks() {
    Masks m;
    m.byte = vconst(0x00FF00FFu);
    m.low = FMT == RQ_FMT_Q8_0 ? m.byte : vconst(FMT == RQ_FMT_Q6_K ? 0x001C001Cu : 0x000F000Fu);
    m.high = FMT == RQ_FMT_Q8_0 ? m.byte : vconst(FMT == RQ_FMT_Q6_K ? 0x00E000E0u : 0x00F000F0u);
    return m;
}

// Signed bytes as exact f16: 1024 + (128 + v) from the byte and the exponent
// bits, less 1152.
__device__ __forceinline__ Op bytes_op(u32 u0, u32 u1, u32 M) {
    constexpr u32 K = 0x64806480u;
    const h2 off = splat((_Float16)-1152.f);
    Op o;
    o.r[0] = as_h2((u0 & M) ^ K) + off;
    o.r[1] = as_h2(((u0 >> 8) & M) ^ K) + off;
    o.r[2] = as_h2((u1 & M) ^ K) + off;
    o.r[3] = as_h2(((u1 >> 8) & M) ^ K) + off;
    return o;
}

// Masked fields of a dword pair's bytes as a x + b in f16 (a single rounding,
// exact for every use below): x = (byte & mask) ^ flip in an f16 of exponent
// 2^10, i.e. 1024 + the field.
__device__ __forceinline__ Op fields_op(u32 u0, u32 u1, u32 mask, u32 key, h2 a, h2 b) {
    Op o;
    o.r[0] = __builtin_elementwise_fma(as_h2((u0 & mask) ^ key), a, b);
    o.r[1] = __builtin_elementwise_fma(as_h2(((u0 >> 8) & mask) ^ key), a, b);
    o.r[2] = __builtin_elementwise_fma(as_h2((u1 & mask) ^ key), a, b);
    o.r[3] = __builtin_elementwise_fma(as_h2(((u1 >> 8) & mask) ^ key), a, b);
    return o;
}

__device__ __forceinline__ _Float16 ubyte_h(u32 w, int i) { return (_Float16)(u16)((w >> (8 * i)) & 0xFFu); }
__device__ __forceinline__ float half_at(u32 w, int i) { return (float)as_h2(w)[i]; }

template <int FMT>
struct ColsFmt {
    static constexpr int C = FMT == RQ_FMT_Q8_0 ? 17 : FMT == RQ_FMT_Q6_K ? 13 : 9;  // dot4 chunks
    static constexpr bool NIB = FMT == RQ_FMT_Q4_K || FMT == RQ_FMT_Q4_0;
    static constexpr int L = NIB ? 2 : FMT == RQ_FMT_Q6_K ? 3 : 4;  // MFMA-layout code loads per super-block
    static constexpr bool BLOCK_D = FMT == RQ_FMT_Q4_0 || FMT == RQ_FMT_Q8_0;  // f16 scale per block, none per super-block
};

// A wave's weights of one 16-row tile and half a super-block (four blocks):
// the code dwords of each block in operand order (Q6_K: still packed, with
// the dwords its fourth window gathers from), and the scales.
template <int FMT>
struct HalfW {
    u32 u[4][2];   // blocks' dwords
    u32 sc, mn;    // Q4_K: the four blocks' scales and mins (row n)
    u32 sc6[2];    // Q6_K: the eight sub-block scales (row n)
    u32 dd;        // Q4_K: f16 d, dmin of row n
    u32 d[4][2];   // rows 4 g + e (OWN: [0] only, row n): d (Q4_K / Q6_K: [e][0] low half) or the four blocks' d (Q4_0 / Q8_0)
};

__device__ __forceinline__ void q4k_half(const int4& h, int hb, u32& sc, u32& mn) {
    if (hb == 0) {
        sc = (u32)h.y & 0x3F3F3F3Fu;
        mn = (u32)h.z & 0x3F3F3F3Fu;
    } else {
        sc = ((u32)h.w & 0x0F0F0F0Fu) | (((u32)h.y >> 2) & 0x30303030u);
        mn = (((u32)h.w >> 4) & 0x0F0F0F0Fu) | (((u32)h.z >> 2) & 0x30303030u);
    }
    // (Kept whole: folded into its uses, the mask became an AND per byte.)
    __asm__ volatile("" : "+v"(sc), "+v"(mn));
}

// Q6_K's fourth window from the dwords of the first three (2-bit pieces into
// bits 7..2 of each byte).
__device__ __forceinline__ u32 q6_fourth(u32 a, u32 b, u32 c) {
    return ((a & 0x03030303u) << 2) | ((b & 0x03030303u) << 4) | ((c & 0x03030303u) << 6);
}

// ---------------------------------------------------------------------------
// Weight sources.

// Rows of the workgroup: row r of its 16 RT (GLU: the first half gate's, the
// second up's, the same rows of both).
template <int RT, bool GLU>
struct ColsRows {
    RqColsTarget t0, t1;
    int row0;
    __device__ __forceinline__ const RqColsTarget& target(int tile) const { return GLU && tile >= RT / 2 ? t1 : t0; }
    __device__ __forceinline__ int row(int r) const {
        return row0 + (GLU && r >= 8 * RT ? r - 8 * RT : r);
    }
};

// Dot4 layout: eight super-blocks of every row at a time, through registers
// into LDS.
template <int FMT, int RT, bool GLU>
struct Dot4Source {
    static constexpr int C = ColsFmt<FMT>::C, ROWS = 16 * RT, ITEMS = C * ROWS * 8;
    static constexpr int NQ = (ITEMS + RQ_COLS_THREADS - 1) / RQ_COLS_THREADS;
    static constexpr int BYTES = ITEMS * 16 + (FMT == RQ_FMT_Q6_K ? ROWS * 16 : 0);  // LDS
    int4 q[NQ];
    u32 tail;

    // Slot t of row r holds super-block 8 it + (t ^ swz(r)): the 16 rows a
    // wave reads at one super-block then lie in 16 different 16-byte banks
    // (rows are 128 bytes apart).
    static __device__ __forceinline__ int swz(int r) { return (r >> 1) & 7; }

    __device__ __forceinline__ void load(const RqColsParams& P, const ColsRows<RT, GLU>& W, int it) {
        const int tid = threadIdx.x, lr = P.lr, S = P.S;
#pragma unroll
        for (int i = 0; i < NQ; i++) {
            const int item = tid + i * RQ_COLS_THREADS;
            if (ITEMS % RQ_COLS_THREADS != 0 && i == NQ - 1 && item >= ITEMS) break;
            const int r = (item >> 3) % ROWS, c = item / (8 * ROWS);
            const int s = min(8 * it + ((item & 7) ^ swz(r)), S - 1);
            const RqColsTarget& T = W.target(GLU && r >= 8 * RT ? RT - 1 : 0);
            const int row = min(W.row(r), T.n - 1);
            const int64_t slot = (((int64_t)(row >> lr) * C + c) << lr) * S + (row & ((1 << lr) - 1)) * S + s;
            q[i] = ld16_nt(T.a + slot * 16);
        }
        if constexpr (FMT == RQ_FMT_Q6_K) {
            if (tid < 8 * ROWS) {
                const int r = tid >> 3, s = min(8 * it + ((tid & 7) ^ swz(r)), S - 1);
                const RqColsTarget& T = W.target(GLU && r >= 8 * RT ? RT - 1 : 0);
                const int64_t slot = (int64_t)min(W.row(r), T.n - 1) * S + s;
                tail = gmem((const u16*)T.b)[slot];
            }
        }
    }
    __device__ __forceinline__ void store() const {
        const int tid = threadIdx.x;
#pragma unroll
        for (int i = 0; i < NQ; i++) {
            const int item = tid + i * RQ_COLS_THREADS;
            if (ITEMS % RQ_COLS_THREADS != 0 && i == NQ - 1 && item >= ITEMS) break;
            *(int4*)(cols_lds + item * 16) = q[i];
        }
        if constexpr (FMT == RQ_FMT_Q6_K)
            if (tid < 8 * ROWS) *(u16*)(cols_lds + ITEMS * 16 + tid * 2) = (u16)tail;
    }
    // LDS bytes of chunk c of row r, super-block s.
    static __device__ __forceinline__ const char* at(int c, int r, int s) {
        return cols_lds + ((c * ROWS + r) * 8 + ((s & 7) ^ swz(r))) * 16;
    }
    // Block b's two dwords of half hb. NIB: the low nibbles of a chunk's bytes
    // are elements 0-15, the high ones 16-31, so k-groups 0 and 2 take the low,
    // 1 and 3 the high nibbles of its first and second eight bytes. Q8_0: a
    // chunk per 16 elements. Q6_K: block b of window 2 hb (b < 2) or 2 hb + 1,
    // window w's blocks in chunks 1 + 4 w .. 4 + 4 w, window 3 gathered from
    // the three others'.
    __device__ __forceinline__ void codes(int t, int s, int hb, int b, u32 (&u)[2]) const {
        const int lane = threadIdx.x & 63, g = lane >> 4, r = 16 * t + (lane & 15);
        auto get = [&](int c) { return *(const uint2*)(at(c, r, s) + 8 * (g >> 1)); };
        uint2 v;
        if constexpr (ColsFmt<FMT>::NIB) {
            v = get(1 + 4 * hb + b);
        } else if constexpr (FMT == RQ_FMT_Q8_0) {
            v = get(1 + 2 * (4 * hb + b) + (g & 1));
        } else {
            const int c = 1 + 2 * (b & 1) + (g & 1);
            if (hb == 0 || b < 2) {
                v = get(c + 4 * (2 * hb + (b >> 1)));
            } else {
                const uint2 x = get(c), y = get(c + 4), z = get(c + 8);
                v = make_uint2(q6_fourth(x.x, y.x, z.x), q6_fourth(x.y, y.y, z.y));
            }
        }
        u[0] = v.x;
        u[1] = v.y;
    }
    // The half's scales, and (CODES) its blocks' codes; OWN: d of row n alone.
    template <bool OWN = false, bool CODES = true>
    __device__ __forceinline__ HalfW<FMT> half(int t, int s, int hb) const {
        const int lane = threadIdx.x & 63, g = lane >> 4, n = lane & 15, r = 16 * t + n;
        HalfW<FMT> h;
        if constexpr (CODES)
#pragma unroll
            for (int b = 0; b < 4; b++) codes(t, s, hb, b, h.u[b]);
        if constexpr (FMT == RQ_FMT_Q4_K) {
            const int4 hd = *(const int4*)at(0, r, s);
            q4k_half(hd, hb, h.sc, h.mn);
            h.dd = (u32)hd.x;
        }
        if constexpr (FMT == RQ_FMT_Q6_K) {
            const uint2 v = *(const uint2*)(at(0, r, s) + 8 * hb);
            h.sc6[0] = v.x;
            h.sc6[1] = v.y;
        }
#pragma unroll
        for (int e = 0; e < (OWN ? 1 : 4); e++) {
            const int re = OWN ? r : 16 * t + 4 * g + e;
            if constexpr (ColsFmt<FMT>::BLOCK_D) {
                const uint2 v = *(const uint2*)(at(0, re, s) + 8 * hb);
                h.d[e][0] = v.x;
                h.d[e][1] = v.y;
            } else if constexpr (FMT == RQ_FMT_Q4_K) {
                h.d[e][0] = *(const u32*)at(0, re, s);
            } else {
                h.d[e][0] = *(const u16*)(cols_lds + ITEMS * 16 + (re * 8 + ((s & 7) ^ swz(re))) * 2);
            }
        }
        return h;
    }
};

// MFMA layout: a super-block's loads straight into registers.
template <int FMT, int RT, bool GLU>
struct MfmaSource {
    static constexpr int L = ColsFmt<FMT>::L;
    static constexpr int BYTES = 0;  // LDS
    int4 cv[RT][L], hv[RT];
    u32 dv[RT];

    __device__ __forceinline__ void load(const RqColsParams& P, const ColsRows<RT, GLU>& W, int s) {
#pragma unroll
        for (int t = 0; t < RT; t++) load_tile(P, W, t, s);
    }
    __device__ __forceinline__ void load_tile(const RqColsParams& P, const ColsRows<RT, GLU>& W, int t, int s) {
        const u32 lane = threadIdx.x & 63, n = lane & 15;
        const RqColsTarget& T = W.target(t);
        const int tile = min(W.row(16 * t) >> 4, T.tiles - 1);
        const int64_t sb = (int64_t)tile * P.S2 + s;
        // Wave-uniform bases and 32-bit lane offsets: scalar addresses.
        const u8* cb = T.a + sb * L * 1024;
#pragma unroll
        for (int j = 0; j < L; j++) cv[t][j] = ld16_nt(cb + j * 1024 + lane * 16u);
        hv[t] = ld16_nt(T.b + sb * 256 + n * 16u);
        if constexpr (FMT == RQ_FMT_Q6_K) {
            const u32 DS = (u32)(P.S2 + 7) & ~7u;
            const u8* dp = T.b + (int64_t)T.tiles * P.S2 * 256 + (int64_t)tile * 32 * DS + 2 * s;
            dv[t] = *gmem((const u16*)(dp + n * DS * 2u));
        }
    }
    // The tile's registers hold nothing any more (without this the values
    // would stay live around the loop where no further load follows).
    __device__ __forceinline__ void drop_tile(int t) {
#pragma unroll
        for (int j = 0; j < L; j++)
            __asm__ volatile("" : "=v"(cv[t][j].x), "=v"(cv[t][j].y), "=v"(cv[t][j].z), "=v"(cv[t][j].w));
        __asm__ volatile("" : "=v"(hv[t].x), "=v"(hv[t].y), "=v"(hv[t].z), "=v"(hv[t].w));
        if constexpr (FMT == RQ_FMT_Q6_K) __asm__ volatile("" : "=v"(dv[t]));
    }
    template <bool OWN = false, bool CODES = true>
    __device__ __forceinline__ HalfW<FMT> half(int t, int s, int hb) const {
        (void)s;
        const int lane = threadIdx.x & 63, g = lane >> 4;
        HalfW<FMT> h;
        auto put = [&](int b, const int4& v) {
            const Win w = win_of(v);
#pragma unroll
            for (int j = 0; j < 2; j++) {
                h.u[b][j] = w.x[j];
                h.u[b + 1][j] = w.y[j];
            }
        };
        if constexpr (ColsFmt<FMT>::NIB) {
            put(0, cv[t][hb]);  // blocks 0, 1: low nibbles; 2, 3: high nibbles of the same dwords
#pragma unroll
            for (int j = 0; j < 2; j++) {
                h.u[2][j] = h.u[0][j];
                h.u[3][j] = h.u[1][j];
            }
        } else if constexpr (FMT == RQ_FMT_Q8_0) {
            put(0, cv[t][2 * hb]);
            put(2, cv[t][2 * hb + 1]);
        } else {
            put(0, cv[t][hb == 0 ? 0 : 2]);
            if (hb == 0) {
                put(2, cv[t][1]);
            } else {
                const int4 &a = cv[t][0], &b = cv[t][1], &c = cv[t][2];
                put(2, make_int4((int)q6_fourth(a.x, b.x, c.x), (int)q6_fourth(a.y, b.y, c.y),
                                 (int)q6_fourth(a.z, b.z, c.z), (int)q6_fourth(a.w, b.w, c.w)));
            }
        }
        if constexpr (FMT == RQ_FMT_Q4_K) {
            q4k_half(hv[t], hb, h.sc, h.mn);
            h.dd = (u32)hv[t].x;
        }
        if constexpr (FMT == RQ_FMT_Q6_K) {
            h.sc6[0] = dw(hv[t], 2 * hb);
            h.sc6[1] = dw(hv[t], 2 * hb + 1);
        }
        if constexpr (OWN) {
            h.d[0][0] = ColsFmt<FMT>::BLOCK_D ? dw(hv[t], 2 * hb) : FMT == RQ_FMT_Q4_K ? (u32)hv[t].x : dv[t];
            h.d[0][1] = ColsFmt<FMT>::BLOCK_D ? dw(hv[t], 2 * hb + 1) : 0u;
            return h;
        }
        // Rows 4 g + e of the tile sit in lanes 4 g + e.
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int src = (4 * g + e) * 4;
            if constexpr (ColsFmt<FMT>::BLOCK_D) {
                h.d[e][0] = (u32)__builtin_amdgcn_ds_bpermute(src, (int)dw(hv[t], 2 * hb));
                h.d[e][1] = (u32)__builtin_amdgcn_ds_bpermute(src, (int)dw(hv[t], 2 * hb + 1));
            } else {
                h.d[e][0] = (u32)__builtin_amdgcn_ds_bpermute(src, FMT == RQ_FMT_Q4_K ? hv[t].x : (int)dv[t]);
            }
        }
        return h;
    }
};

// ---------------------------------------------------------------------------

// Block b's weight operand(s) from its half super-block: sc q (Q4_K), q - 8
// (Q4_0), q (Q8_0), or the two parts of sc (q - 32) (Q6_K).
template <int FMT, int LAY>
__device__ __forceinline__ void weight_op(const HalfW<FMT>& h, int b, const Masks& mk, Op& o, Op& o2) {
    const int g = (threadIdx.x & 63) >> 4;
    const u32 u0 = h.u[b][0], u1 = h.u[b][1];
    if constexpr (ColsFmt<FMT>::NIB) {
        // Q4_0 subtracts its offset 8; Q4_K's would make sc * 1032 inexact
        // (13 bits), so its codes stay unsigned.
        constexpr float kBase = FMT == RQ_FMT_Q4_0 ? 1032.f : 1024.f;
        _Float16 sc = (_Float16)1.f;
        if constexpr (FMT == RQ_FMT_Q4_K) sc = ubyte_h(h.sc, b);
        if constexpr (LAY == RQ_LAY_DOT4) {
            // The lane's nibble to bits 3..0; high ones are stored XOR 8.
            const int sh = 4 * (g & 1);
            const u32 key = 0x64006400u | ((g & 1) ? 0x00080008u : 0u);
            o = fields_op(u0 >> sh, u1 >> sh, mk.low, key, splat(sc), splat(sc * (_Float16)-kBase));
        } else if (b < 2) {
            o = fields_op(u0, u1, mk.low, 0x64006400u, splat(sc), splat(sc * (_Float16)-kBase));
        } else {
            // 1024 + 16 q, stored XOR 8 in the high nibble.
            o = fields_op(u0, u1, mk.high, 0x64806480u, splat(sc * (_Float16)0.0625f),
                          splat(sc * (_Float16)(960.f - kBase)));
        }
    } else if constexpr (FMT == RQ_FMT_Q8_0) {
        o = bytes_op(u0, u1, mk.byte);
    } else {
        // The lane's elements lie in sub-block 2b + g % 2 (k-groups 0 and 2
        // the first 16, 1 and 3 the last). With u = q XOR 32 in bits 7..2:
        // bits 7..5 less the flip are q >> 3, bits 4..2 q & 7.
        const u32 w = b < 2 ? h.sc6[0] : h.sc6[1];
        const int i = 2 * (b & 1) + (g & 1);
        const _Float16 s4 = (_Float16)(int16_t)(int8_t)(w >> (8 * i)) * (_Float16)0.25f;
        o = fields_op(u0, u1, mk.high, 0x64806480u, splat(s4), splat(s4 * (_Float16)-1152.f));
        o2 = fields_op(u0, u1, mk.low, 0x64006400u, splat(s4), splat(s4 * (_Float16)-1024.f));
    }
}

// Activations of half a super-block as loaded: CG groups of 16 columns, a
// lane's 16 bytes of columns lane / 8 and 8 + lane / 8.
template <int CG>
struct XRaw {
    int4 w[CG][2];
};
__device__ __forceinline__ int cols_dstride(int S) { return 16 * S + 8; }

template <int FMT, int LAY, int RT, int CG, bool GLU>
__device__ __forceinline__ void cols_body(const RqColsParams& P, const ColsRows<RT, GLU>& W) {
    const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, n = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int S = P.S, k = P.k;
    using Source =
        typename std::conditional<LAY == RQ_LAY_DOT4, Dot4Source<FMT, RT, GLU>, MfmaSource<FMT, RT, GLU>>::type;

    // LDS: the dot4 layout's weights, each wave's staged activations, the
    // columns' scales. Columns past the last repeat it (their sums are not
    // stored).
    constexpr int XCOL = RQ_COLS_XCOL, XGROUP = 16 * XCOL;
    char* xl = cols_lds + Source::BYTES + wave * (CG * XGROUP);
    char* dl = cols_lds + Source::BYTES + RQ_COLS_PARTS * CG * XGROUP;
    const int ds = cols_dstride(S), nb = k >> 5;
    // A half super-block of a column is 128 contiguous bytes, one cache line:
    // eight columns per load. (Loaded as the operands need it, 64 bytes of
    // each of 16 columns, every line was looked up twice, and at widths of
    // 4096 all 16 lines fell in two sets of the L1 and were fetched twice.)
    u32 xoff[CG][2];
#pragma unroll
    for (int cg = 0; cg < CG; cg++)
#pragma unroll
        for (int i = 0; i < 2; i++) xoff[cg][i] = (u32)min(16 * cg + 8 * i + (lane >> 3), P.m - 1) * (u32)k;
    auto xload = [&](int s, int hb, XRaw<CG>& x) {
        const u32 o = min(256u * s + 128u * hb + 16u * (lane & 7), (u32)k - 16u);
#pragma unroll
        for (int cg = 0; cg < CG; cg++)
#pragma unroll
            for (int i = 0; i < 2; i++) x.w[cg][i] = ld16((const u8*)P.xq + (xoff[cg][i] + o));
    };
    auto xstore = [&](const XRaw<CG>& x) {
#pragma unroll
        for (int cg = 0; cg < CG; cg++)
#pragma unroll
            for (int i = 0; i < 2; i++)
                *(int4*)(xl + cg * XGROUP + (8 * i + (lane >> 3)) * XCOL + 16 * (lane & 7)) = x.w[cg][i];
    };

    v4f acc[RT][CG];
#pragma unroll
    for (int t = 0; t < RT; t++)
#pragma unroll
        for (int cg = 0; cg < CG; cg++) acc[t][cg] = v4f{0.f, 0.f, 0.f, 0.f};
    const Masks mk = masks<FMT>();
    Op ones;
#pragma unroll
    for (int i = 0; i < 4; i++) ones.r[i] = splat((_Float16)1.f);

    // Loads in flight: each half's activations go out as soon as the one
    // before it has been staged, the next weights as soon as their registers
    // are free. Waits are in issue order, so an activation load must never
    // stand behind weight loads that are needed later than it.
    XRaw<CG> xr;
    const int nit = (S + 7) >> 3;
    const int s0 = min(wave, S - 1);
    Source src;
    xload(s0, 0, xr);
    for (int c = wave; c < 16 * CG; c += RQ_COLS_PARTS) {
        const u16* d = P.xd + (int64_t)min(c, P.m - 1) * nb;
        for (int b = lane; b < 8 * S; b += 64) {
            const u16 v = gmem(d)[min(b, nb - 1)];
            *(u16*)(dl + c * ds + 2 * b) = b < nb ? v : (u16)0;
        }
    }
    src.load(P, W, LAY == RQ_LAY_DOT4 ? 0 : s0);
    if constexpr (LAY == RQ_LAY_MFMA) __syncthreads();  // the scales are staged

    for (int it = 0; it < nit; it++) {
        const int s = 8 * it + wave;
        const int sn = min(s + 8, S - 1);
        if constexpr (LAY == RQ_LAY_DOT4) {
            if (it > 0) __syncthreads();  // the last super-blocks' reads are done
            src.store();
            __syncthreads();
        }
        if (s >= S) {  // the wave has no super-block in this step, the last
            if constexpr (LAY == RQ_LAY_DOT4) continue;  // (to the barriers)
            break;
        }
#pragma unroll
        for (int hb = 0; hb < 2; hb++) {
            if (!sgpr_value(1)) continue;
            Op xo[4][CG];
            u32 dx[CG][2];
            float sx[CG];  // Q4_K: dx * (sum of codes) of column n, block g
            xstore(xr);
#pragma unroll
            for (int cg = 0; cg < CG; cg++) {
                const uint2 dv = *(const uint2*)(dl + (16 * cg + n) * ds + 16 * s + 8 * hb);
                dx[cg][0] = dv.x;
                dx[cg][1] = dv.y;
#pragma unroll
                for (int w = 0; w < 2; w++) {
                    const Win v = win_of(*(const int4*)(xl + cg * XGROUP + n * XCOL + 64 * w + 16 * g));
                    xo[2 * w][cg] = bytes_op(v.x[0], v.x[1], mk.byte);
                    xo[2 * w + 1][cg] = bytes_op(v.y[0], v.y[1], mk.byte);
                }
                if constexpr (FMT == RQ_FMT_Q4_K) {
                    // Every row of a product with ones holds the sum.
                    float sum[4];
#pragma unroll
                    for (int b = 0; b < 4; b++) sum[b] = mfma(ones, xo[b][cg], v4f{0.f, 0.f, 0.f, 0.f})[0];
                    const float lo = (g & 1) ? sum[1] : sum[0], hi = (g & 1) ? sum[3] : sum[2];
                    u32 dp = dx[cg][0], dq = dx[cg][1];
                    // (Opaque, or the choice becomes one of addresses, in scratch.)
                    __asm__ volatile("" : "+v"(dp), "+v"(dq));
                    dp = (g & 2) ? dq : dp;
                    sx[cg] = h2f((dp >> (16 * (g & 1))) & 0xFFFFu) * ((g & 2) ? hi : lo);
                }
            }
            if (hb == 0) {
                xload(s, 1, xr);
                if constexpr (LAY == RQ_LAY_DOT4)
                    if (it + 1 < nit) src.load(P, W, it + 1);
            } else if (s + 8 < S) {
                xload(sn, 0, xr);
            }
            // A block's products are issued, then the next block's operand is
            // made while they run, then their results are scaled and summed:
            // scheduled freely, the compiler put each product's results right
            // behind it and waited out the matrix pipe every time. Each tile
            // is a basic block of its own (an opaque branch, always taken),
            // or the compiler holds several tiles' values at once and spills.
#pragma unroll
            for (int t = 0; t < RT; t++) {
                if (!sgpr_value(1)) continue;
                const HalfW<FMT> h = src.half(t, s, hb);
                if constexpr (LAY == RQ_LAY_MFMA)
                    if (hb == 1) {
                        if (s + 8 < S)
                            src.load_tile(P, W, t, sn);
                        else
                            src.drop_tile(t);
                    }
                Op o, o2;
                weight_op<FMT, LAY>(h, 0, mk, o, o2);
                v4f sum[CG];
#pragma unroll
                for (int b = 0; b < 4; b++) {
                    v4f D[CG];
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int cg = 0; cg < CG; cg++) {
                        D[cg] = v4f{0.f, 0.f, 0.f, 0.f};
                        if constexpr (FMT == RQ_FMT_Q6_K) D[cg] = mfma(o2, xo[b][cg], D[cg]);
                    }
#pragma unroll
                    for (int cg = 0; cg < CG; cg++) D[cg] = mfma(o, xo[b][cg], D[cg]);
                    if constexpr (FMT == RQ_FMT_Q4_K) {
                        // The mins' terms -dmin m dx sum(x) of the half's four
                        // blocks, a 16 x 4 x 16 product.
                        if (b == 3) {
                            const float c = -half_at(h.dd, 1) * (float)((h.mn >> (8 * g)) & 0xFFu);
#pragma unroll
                            for (int cg = 0; cg < CG; cg++)
                                acc[t][cg] = __builtin_amdgcn_mfma_f32_16x16x4f32(c, sx[cg], acc[t][cg], 0, 0, 0);
                        }
                    }
                    __builtin_amdgcn_sched_barrier(0);
                    if (b < 3) weight_op<FMT, LAY>(h, b + 1, mk, o, o2);
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int cg = 0; cg < CG; cg++) {
                        const float dxb = half_at(dx[cg][b >> 1], b & 1);
#pragma unroll
                        for (int e = 0; e < 4; e++) {
                            // (Q4_0, Q8_0: the product of two f16 scales is exact.)
                            const float f = ColsFmt<FMT>::BLOCK_D ? half_at(h.d[e][b >> 1], b & 1) * dxb : dxb;
                            sum[cg][e] = b == 0 ? D[cg][e] * f : fmaf(D[cg][e], f, sum[cg][e]);
                        }
                    }
                }
#pragma unroll
                for (int cg = 0; cg < CG; cg++)
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        acc[t][cg][e] = ColsFmt<FMT>::BLOCK_D ? acc[t][cg][e] + sum[cg][e]
                                                              : fmaf(sum[cg][e], half_at(h.d[e][0], 0), acc[t][cg][e]);
            }
        }
    }

    // ---- The eight waves' sums, added pairwise. A lane's four rows of
    // one column are one 16-byte slot; slot n of (tile t, k-group g) sits at n
    // XOR (4 t + g), so that the row quads of a column lie in different banks.
    __syncthreads();
    v4f* part = (v4f*)cols_lds;
#pragma unroll
    for (int t = 0; t < RT; t++)
#pragma unroll
        for (int cg = 0; cg < CG; cg++)
            part[((wave * RT + t) * CG + cg) * 64 + 16 * g + (n ^ ((4 * t + g) & 15))] = acc[t][cg];
    __syncthreads();
    auto total = [&](int t, int gg, int c) {
        v4f v[RQ_COLS_PARTS];
#pragma unroll
        for (int w = 0; w < RQ_COLS_PARTS; w++)
            v[w] = part[((w * RT + t) * CG + (c >> 4)) * 64 + 16 * gg + ((c & 15) ^ ((4 * t + gg) & 15))];
#pragma unroll
        for (int d = 1; d < RQ_COLS_PARTS; d *= 2)
#pragma unroll
            for (int w = 0; w < RQ_COLS_PARTS; w += 2 * d) v[w] += v[w + d];
        return v[0];
    };
    if constexpr (!GLU) {
        const RqColsTarget& T = W.t0;
        for (int it = tid; it < CG * 16 * 4 * RT; it += RQ_COLS_THREADS) {
            const int c = it / (4 * RT), q = it % (4 * RT);
            const int row = W.row0 + 4 * q;
            if (c >= P.m || row >= T.n) continue;
            const v4f v = total(q >> 2, q & 3, c);
            float* o = T.out + (int64_t)c * T.n + row;
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (row + e < T.n) gmem(o)[e] = v[e];
        }
    } else {
        // h = act(gate) * up of the workgroup's 32 rows: eight lanes hold a
        // column's Q8_1 block (whole 8-lane groups stay active).
        for (int it = tid; it < CG * 16 * 8; it += RQ_COLS_THREADS) {
            const int c = it >> 3, q = it & 7;
            const v4f gs = total(q >> 2, q & 3, c), us = total(2 + (q >> 2), q & 3, c);
            float h[4];
#pragma unroll
            for (int e = 0; e < 4; e++) h[e] = act_apply(P.act, gs[e]) * us[e];
            const int64_t t = ((int64_t)c * W.t0.n + W.row0) / 4 + q;
            const bool in = c < P.m;
            if (P.hf && in) {
#pragma unroll
                for (int e = 0; e < 4; e++) gmem(P.hf)[4 * t + e] = h[e];
            }
            if (P.hq) q8_emit4(h, t, in, P.hq, P.hd, P.hs);
        }
    }
}

// The workgroup's target, picked by value (sgpr_value, rq_device.h).
__device__ __forceinline__ RqColsTarget cols_target(const RqColsParams& P, int ti) {
    RqColsTarget T;
#define RQ_PICK(f)                                                                                        \
    {                                                                                                     \
        const auto v0 = sgpr_value(P.t[0].f), v1 = sgpr_value(P.t[1].f), v2 = sgpr_value(P.t[2].f);       \
        T.f = ti == 0 ? v0 : ti == 1 ? v1 : v2;                                                           \
    }
    RQ_PICK(a) RQ_PICK(b) RQ_PICK(out) RQ_PICK(n) RQ_PICK(wg_start) RQ_PICK(fmt) RQ_PICK(tiles)
#undef RQ_PICK
    return T;
}

template <int FMT, int LAY, int RT, int CG>
__device__ __forceinline__ void cols_matvec(const RqColsParams& P) {
    const int blk = blockIdx.x;
    ColsRows<RT, false> W;
    W.t0 = cols_target(P, P.count > 2 && blk >= P.t[2].wg_start ? 2 : P.count > 1 && blk >= P.t[1].wg_start ? 1 : 0);
    W.row0 = (blk - W.t0.wg_start) * 16 * RT;
    if constexpr (FMT == RQ_FMT_MIX_K) {
        if (W.t0.fmt == RQ_FMT_Q4_K)
            cols_body<RQ_FMT_Q4_K, LAY, RT, CG, false>(P, W);
        else
            cols_body<RQ_FMT_Q6_K, LAY, RT, CG, false>(P, W);
    } else {
        cols_body<FMT, LAY, RT, CG, false>(P, W);
    }
}

template <int FMT, int CG>
__device__ __forceinline__ void cols_glu(const RqColsParams& P) {
    ColsRows<4, true> W;
    W.t0 = P.t[0];
    W.t1 = P.t[1];
    W.row0 = blockIdx.x * 32;
    cols_body<FMT, RQ_LAY_DOT4, 4, CG, true>(P, W);
}

#define RQ_COLS(NAME, FMT, LN, LAY, RT, CG)                                                                        \
    extern "C" __global__ __launch_bounds__(RQ_COLS_THREADS) void rq_cols_##NAME##_##LN##_##RT##x##CG(RqColsParams p) { \
        cols_matvec<FMT, LAY, RT, CG>(p);                                                                          \
    }
#define RQ_COLS_SET(NAME, FMT, LN, LAY)  \
    RQ_COLS(NAME, FMT, LN, LAY, 1, 1)    \
    RQ_COLS(NAME, FMT, LN, LAY, 1, 2)    \
    RQ_COLS(NAME, FMT, LN, LAY, 1, 3)    \
    RQ_COLS(NAME, FMT, LN, LAY, 1, 4)    \
    RQ_COLS(NAME, FMT, LN, LAY, 2, 1)    \
    RQ_COLS(NAME, FMT, LN, LAY, 2, 2)    \
    RQ_COLS(NAME, FMT, LN, LAY, 2, 3)
#define RQ_COLS_ALL(NAME, FMT)                    \
    RQ_COLS_SET(NAME, FMT, d, RQ_LAY_DOT4)        \
    RQ_COLS(NAME, FMT, d, RQ_LAY_DOT4, 4, 1)      \
    RQ_COLS_SET(NAME, FMT, m, RQ_LAY_MFMA)
// (4 x 2 of Q8_0 would not fit the LDS.)
#define RQ_COLS_4X2(NAME, FMT) RQ_COLS(NAME, FMT, d, RQ_LAY_DOT4, 4, 2)
#define RQ_COLS_GLU(NAME, FMT, CG)                                                                          \
    extern "C" __global__ __launch_bounds__(RQ_COLS_THREADS) void rq_colsglu_##NAME##_##CG(RqColsParams p) { \
        cols_glu<FMT, CG>(p);                                                                               \
    }
#define RQ_COLS_FMT(NAME, FMT) \
    RQ_COLS_ALL(NAME, FMT)     \
    RQ_COLS_GLU(NAME, FMT, 1)  \
    RQ_COLS_GLU(NAME, FMT, 2)

RQ_COLS_FMT(q4_0, RQ_FMT_Q4_0)
RQ_COLS_FMT(q8_0, RQ_FMT_Q8_0)
RQ_COLS_FMT(q4_k, RQ_FMT_Q4_K)
RQ_COLS_FMT(q6_k, RQ_FMT_Q6_K)
RQ_COLS_ALL(q4_k_q6_k, RQ_FMT_MIX_K)
RQ_COLS_4X2(q4_0, RQ_FMT_Q4_0)
RQ_COLS_4X2(q4_k, RQ_FMT_Q4_K)
RQ_COLS_4X2(q6_k, RQ_FMT_Q6_K)
RQ_COLS_4X2(q4_k_q6_k, RQ_FMT_MIX_K)

// ---------------------------------------------------------------------------
// The f16 GEMM route for short prompts (rq_gemm_<fmt>_<layout>): out[a][r] =
// sum over k of f16(x) f16(w), accumulated in f32, with the weights
// dequantized in registers: no f16 copy of the weight is written and read
// back (3.6 times a weight's Q4_K bytes, whose 27 us for 14336 x 4096 were
// half of the call up to a few hundred columns).
//
// Same split as the matvecs above: 32 rows and 96 or 128 columns per
// workgroup, its eight waves on the row's super-blocks in turn, their sums
// added pairwise. A weight operand (32 elements of 16 rows) takes about 38
// VALU and is used by six or eight v_mfma_f32_16x16x32_f16 of 16 cycles, so
// fewer columns per workgroup would dequantize more than they multiply, and
// more rows would leave the chip short of workgroups (64 rows by 64 columns:
// 14336 x 4096 at 128 columns 45 us against 38). What is left is bound by the
// reads of x, 1 KB per wave and two products (510 MB of reads from L2 for 14336
// x 4096 at 128 columns, 14 TB/s, by counters; VALU issue 27%, MFMA busy 17%),
// not by VALU or by the loads in flight: 16 % fewer
// VALU instructions took 1 to 3 % off some shapes and put as much on others
// (128 columns 36.5 -> 35.9 us, 96 30.6 -> 31.4), and loads two to four
// blocks ahead on top gained 5 % at most (Q6_K 4096 x 14336 at 128: 57.4 ->
// 54.7) and lost up to 10 (Q4_0 11008 x 4096 at 96: 29.3 -> 32.2). A value is
// evaluated in f32 and rounded to f16 once, as the dequantization to a copy
// does. x comes from rq_x16_tiles in the operands' own order: one load per
// wave, 1 KB contiguous, per block and column group.
//
// Us per call of the route, copy + rocBLAS -> these, dot4 / MFMA layout: Q4_K
// 14336 x 4096 at 96 columns 55.8 -> 34.4 / 62.5 -> 30.5, at 128 59.9 -> 38.0
// / 64 -> 35.7, at 256 75.5 -> 65.1 / 77 -> 62.1; Q6_K 4096 x 14336 at 128
// 69 -> 57 / 57; Q4_K 4096 x 4096 at 128 38.8 -> 20.0 / 19.4.

// Block b's weight operand: f16 of the dequantized values.
template <int FMT, int LAY>
__device__ __forceinline__ Op value_op(const HalfW<FMT>& h, const u32 (&u)[2], int b, const Masks& mk) {
    const int g = (threadIdx.x & 63) >> 4;
    const u32 u0 = u[0], u1 = u[1];
    // The codes q, exact in f16: as q (Q8_0, Q4_K), q - 8 (Q4_0) or 4 (q - 32)
    // (Q6_K).
    Op q;
    if constexpr (ColsFmt<FMT>::NIB) {
        // The nibble to bits 7..4 of its byte: 1024 + 16 q.
        u32 v[2][2];
        u32 key = 0x64006400u;
#pragma unroll
        for (int i = 0; i < 2; i++) {
            if constexpr (LAY == RQ_LAY_DOT4) {
                const int sh = 4 * (~g & 1);
                v[i][0] = u[i] << sh;
                v[i][1] = u[i] >> (8 - sh);
                key = 0x64006400u | ((g & 1) ? 0x00800080u : 0u);  // high nibbles are stored XOR 8
            } else if (b < 2) {
                v[i][0] = u[i] << 4;
                v[i][1] = u[i] >> 4;
            } else {
                v[i][0] = u[i];
                v[i][1] = u[i] >> 8;
                key = 0x64806480u;
            }
        }
#pragma unroll
        for (int i = 0; i < 4; i++) {
            q.r[i] = as_h2((v[i >> 1][i & 1] & mk.high) ^ key);
            q.r[i] = __builtin_elementwise_fma(q.r[i], splat((_Float16)0.0625f),
                                               splat((_Float16)(FMT == RQ_FMT_Q4_0 ? -72.f : -64.f)));
        }
    } else {
        q = bytes_op(FMT == RQ_FMT_Q6_K ? u0 & 0xFCFCFCFCu : u0, FMT == RQ_FMT_Q6_K ? u1 & 0xFCFCFCFCu : u1, mk.byte);
    }
    if constexpr (ColsFmt<FMT>::BLOCK_D) {
        // One rounding of the exact product of a code and an f16 scale.
        const float d = half_at(h.d[0][b >> 1], b & 1);
        Op o;
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int j = 0; j < 2; j++) o.r[i][j] = (_Float16)((float)q.r[i][j] * d);
        return o;
    } else {
        float s, m = 0.f;
        if constexpr (FMT == RQ_FMT_Q4_K) {
            s = half_at(h.d[0][0], 0) * (float)((h.sc >> (8 * b)) & 0xFFu);
            m = -half_at(h.d[0][0], 1) * (float)((h.mn >> (8 * b)) & 0xFFu);
        } else {
            const u32 w = b < 2 ? h.sc6[0] : h.sc6[1];
            s = half_at(h.d[0][0], 0) * (float)(int8_t)(w >> (8 * (2 * (b & 1) + (g & 1)))) * 0.25f;
        }
        Op o;
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int j = 0; j < 2; j++) {
                // Q6_K: an exact product. Q4_K: d sc q and dmin m are exact,
                // their difference need not be, and the copy rounds it to f32
                // and then to f16: the f32 value passes the empty asm, as in
                // pack32_f16, or part of the values become v_fma_mix to f16,
                // one rounding (another value where the f32 is an f16 tie).
                float v;
                if constexpr (FMT == RQ_FMT_Q4_K) {
                    v = fmaf((float)q.r[i][j], s, m);
                    __asm__ volatile("" : "+v"(v));
                } else {
                    v = (float)q.r[i][j] * s;
                }
                o.r[i][j] = (_Float16)v;
            }
        return o;
    }
}

template <int FMT, int LAY, int RT, int CG>
__device__ __forceinline__ void gemm_body(const RqGemmParams& P) {
    const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, n = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // The column chunks of one row block run on one XCD (workgroups go to the
    // XCDs in turn), so that its L2 serves all but the first read of the
    // weights.
    const int blk = blockIdx.x, per = 8 * P.chunks;
    const int rb = (blk / per) * 8 + (blk & 7), chunk = (blk % per) >> 3;
    if (rb >= P.row_blocks) return;
    ColsRows<RT, false> W;
    W.t0 = P.t;
    W.row0 = rb * 16 * RT;
    RqColsParams C;  // what the weight sources read
    C.lr = P.lr;
    C.S = P.S;
    C.S2 = P.S2;
    using Source =
        typename std::conditional<LAY == RQ_LAY_DOT4, Dot4Source<FMT, RT, false>, MfmaSource<FMT, RT, false>>::type;
    const int S = P.S, nb = P.k >> 5, groups = P.groups;
    const int g0 = chunk * CG;
    // Column group g0 + c (past the last: the last again, unused).
    u32 goff[CG];
#pragma unroll
    for (int c = 0; c < CG; c++) goff[c] = (u32)min(g0 + c, groups - 1) * 1024u + lane * 16u;
    auto xload = [&](int kb, Op (&x)[CG]) {
        const u8* p = (const u8*)P.x + (int64_t)min(kb, nb - 1) * groups * 1024;
#pragma unroll
        for (int c = 0; c < CG; c++) x[c] = __builtin_bit_cast(Op, ld16(p + goff[c]));
    };

    v4f acc[RT][CG];
#pragma unroll
    for (int t = 0; t < RT; t++)
#pragma unroll
        for (int c = 0; c < CG; c++) acc[t][c] = v4f{0.f, 0.f, 0.f, 0.f};
    const Masks mk = masks<FMT>();
    const int nit = (S + 7) >> 3;
    const int s0 = min(wave, S - 1);
    // A block's activations are loaded one block ahead (two to four gained 5 %
    // at most and lost up to 10, see above).
    Op x[2][CG];
    Source src;
    xload(8 * s0, x[0]);
    src.load(C, W, LAY == RQ_LAY_DOT4 ? 0 : s0);

    for (int it = 0; it < nit; it++) {
        const int s = 8 * it + wave;
        if constexpr (LAY == RQ_LAY_DOT4) {
            if (it > 0) __syncthreads();  // the last super-blocks' reads are done
            src.store();
            __syncthreads();
        }
        if (s >= S) {  // the wave has no super-block in this step, the last
            if constexpr (LAY == RQ_LAY_DOT4) continue;  // (to the barriers)
            break;
        }
#pragma unroll
        for (int hb = 0; hb < 2; hb++) {
            if (!sgpr_value(1)) continue;
            // (Dot4 layout: the codes come from LDS block by block.)
            constexpr bool LATE = LAY == RQ_LAY_DOT4;
            HalfW<FMT> h[RT];
            u32 u[2][RT][2];
#pragma unroll
            for (int t = 0; t < RT; t++) {
                h[t] = src.template half<true, !LATE>(t, s, hb);
                if constexpr (LATE) src.codes(t, s, hb, 0, u[0][t]);
            }
#pragma unroll
            for (int b = 0; b < 4; b++) {
                const int kb = 8 * s + 4 * hb + b, ahead = 4 * hb + b + 1;
                // Past the super-block's end: the wave's next one's blocks.
                xload(ahead < 8 ? 8 * s + ahead : 8 * min(s + 8, S - 1) + ahead - 8, x[ahead & 1]);
                if constexpr (LATE) {
                    if (hb == 0 && b == 0 && it + 1 < nit) src.load(C, W, it + 1);
                    if (b < 3)
#pragma unroll
                        for (int t = 0; t < RT; t++) src.codes(t, s, hb, b + 1, u[(b + 1) & 1][t]);
                }
                if (!sgpr_value(1) || kb >= nb) continue;  // (past a partial super-block's end)
#pragma unroll
                for (int t = 0; t < RT; t++) {
                    const Op o = value_op<FMT, LAY>(h[t], LATE ? u[b & 1][t] : h[t].u[b], b, mk);
#pragma unroll
                    for (int c = 0; c < CG; c++) acc[t][c] = mfma(o, x[b & 1][c], acc[t][c]);
                }
            }
            if constexpr (LAY == RQ_LAY_MFMA)
                if (hb == 1) {
#pragma unroll
                    for (int t = 0; t < RT; t++) {
                        if (s + 8 < S)
                            src.load_tile(C, W, t, s + 8);
                        else
                            src.drop_tile(t);
                    }
                }
        }
    }

    // The eight waves' sums, as in cols_body.
    __syncthreads();
    v4f* part = (v4f*)cols_lds;
#pragma unroll
    for (int t = 0; t < RT; t++)
#pragma unroll
        for (int c = 0; c < CG; c++)
            part[((wave * RT + t) * CG + c) * 64 + 16 * g + (n ^ ((4 * t + g) & 15))] = acc[t][c];
    __syncthreads();
    for (int it = tid; it < CG * 16 * 4 * RT; it += RQ_COLS_THREADS) {
        const int c = it / (4 * RT), q = it % (4 * RT), t = q >> 2, gg = q & 3;
        const int row = W.row0 + 4 * q, col = 16 * g0 + c;
        if (col >= P.m || row >= W.t0.n) continue;
        v4f v[RQ_COLS_PARTS];
#pragma unroll
        for (int w = 0; w < RQ_COLS_PARTS; w++)
            v[w] = part[((w * RT + t) * CG + (c >> 4)) * 64 + 16 * gg + ((c & 15) ^ ((4 * t + gg) & 15))];
#pragma unroll
        for (int d = 1; d < RQ_COLS_PARTS; d *= 2)
#pragma unroll
            for (int w = 0; w < RQ_COLS_PARTS; w += 2 * d) v[w] += v[w + d];
        float* o = W.t0.out + (int64_t)col * W.t0.n + row;
#pragma unroll
        for (int e = 0; e < 4; e++)
            if (row + e < W.t0.n) gmem(o)[e] = v[0][e];
    }
}

#define RQ_GEMM(NAME, FMT, LN, LAY, RT, CG)                                                                        \
    extern "C" __global__ __launch_bounds__(RQ_COLS_THREADS) void rq_gemm_##NAME##_##LN##_##RT##x##CG(RqGemmParams p) { \
        gemm_body<FMT, LAY, RT, CG>(p);                                                                            \
    }
#define RQ_GEMM_FMT(NAME, FMT)                 \
    RQ_GEMM(NAME, FMT, d, RQ_LAY_DOT4, 2, 6)   \
    RQ_GEMM(NAME, FMT, d, RQ_LAY_DOT4, 2, 8)   \
    RQ_GEMM(NAME, FMT, m, RQ_LAY_MFMA, 2, 6)   \
    RQ_GEMM(NAME, FMT, m, RQ_LAY_MFMA, 2, 8)
RQ_GEMM_FMT(q4_0, RQ_FMT_Q4_0)
RQ_GEMM_FMT(q8_0, RQ_FMT_Q8_0)
RQ_GEMM_FMT(q4_k, RQ_FMT_Q4_K)
RQ_GEMM_FMT(q6_k, RQ_FMT_Q6_K)

// x f32 [m][k] -> f16 (round to nearest even) in the operand order of
// rq_gemm_*: per 32-element block and group of 16 columns (zeros past m) 1 KB,
// lane 16 g + c holding column c's elements of k-group g (win_of's order, each
// dword's bytes 0, 2, 1, 3). A workgroup takes 8 blocks of a group: a thread
// converts 16 consecutive elements, 16 threads a column's 1 KB, and the
// operands leave through LDS as whole kilobytes. (A thread per lane of the
// result, reading 32 bytes of each of 16 columns, took 5.1 us for 128 columns
// of 4096.)
extern "C" __global__ __launch_bounds__(RQ_THREADS) void rq_x16_tiles(RqX16Params p) {
    __shared__ int4 lds[8 * 65];  // (a block's 64 pieces and one of skew)
    const int tid = threadIdx.x, c = tid >> 4, e = tid & 15, kb0 = blockIdx.x / p.groups * 8;
    const int grp = blockIdx.x - blockIdx.x / p.groups * p.groups;
    const int kb = kb0 + (e >> 1), col = grp * 16 + c;
    int4 v[2] = {make_int4(0, 0, 0, 0), make_int4(0, 0, 0, 0)};
    if (col < p.m && kb < p.nb) {
        const float* src = p.x + (int64_t)col * 32 * p.nb + 32 * kb + 16 * (e & 1);
        const auto pair = [](int a, int b) {
            return (int)((u32)f2h(__int_as_float(a)) | ((u32)f2h(__int_as_float(b)) << 16));
        };
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const int4 a = ld16(src + 8 * i), b = ld16(src + 8 * i + 4);
            v[i] = make_int4(pair(a.x, a.z), pair(a.y, a.w), pair(b.x, b.z), pair(b.y, b.w));
        }
    }
    // Elements 0-7 and 8-15 of a half block: k-groups e % 2 and 2 + e % 2.
#pragma unroll
    for (int i = 0; i < 2; i++) lds[(e >> 1) * 65 + 16 * ((e & 1) + 2 * i) + c] = v[i];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const int b = (tid >> 6) + 4 * i;
        if (kb0 + b < p.nb) st16(p.y + (((int64_t)(kb0 + b) * p.groups + grp) * 64 + (tid & 63)) * 8, lds[b * 65 + (tid & 63)]);
    }
}
