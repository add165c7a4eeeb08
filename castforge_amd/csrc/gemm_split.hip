// Quantized-weight products of small and mid-sized M on one bf16 MFMA per product (NF4: two), K
// split over the waves of a workgroup: y[m, n] = sum_k x[m, k] W[n, k] for INT4 (groups of 32, 64 or
// a multiple of 64), INT8, NF4 (M > 16) and the GGUF Q4_0 / Q8_0 planes.
//
// The weight operand is the exact integer (q - z, q or q - 8) as bf16 and x is the bf16 it is, as
// in prefill_i4_kernel; each 64-wide chunk (32-wide where the format scales every 32) sums into a
// fresh f32 partial that its scale multiplies into the total (eval.rs:1465-1507 with the
// dequantized weights of eval.rs:1145-1179).
//
// `qsplit_kernel<FMT, I, J, NW, S>`: workgroup tile 32 I (n) x 32 J (m).  Every wave computes the
// whole tile over its own 64-wide K chunks (wave w: chunks w, w + NW, ..) and the NW partial tiles
// are summed through LDS in wave order.  The prefill kernels walk K in barriered steps, 0.7 to
// 1.9 us of latency per 64 or 128 of K however small the problem; here nothing is shared between
// waves until the end, so there is no barrier in the loop:
//   * x: each wave keeps a ring of S stages of 32 J rows x 128 bytes, filled by buffer -> LDS loads
//     (8 rows x 128 bytes each; 16-byte pieces at piece ^ ((row >> 1) & 7), so sixteen rows read at
//     one piece cover the 256-byte bank window; rows past M read 0: the row is in the vector offset, which
//     the range check covers whatever it does with the scalar one);
//   * W: each lane loads its row's codes of the chunk into registers (a ring of S sets) and decodes
//     them there: no code is decoded twice within a workgroup, because the waves' chunks differ.
#include <algorithm>
#include <atomic>
#include <cstdlib>
#include <cstring>

#include "../../include/castforge_hip.h"
#include "cfh_common.hpp"

namespace cfh {

// what the one-MFMA prefill kernel takes for M x N, in rounds of 128-row tiles (gemm_prefill.hip)
double prefill_cost(int fmt, bool rows96, int64_t m, int64_t n);

namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef __amdgpu_buffer_rsrc_t rsrc_t;

// numbers as in gemm_prefill.hip; FMT_I8S: INT8 with a partial per chunk (any finite x)
enum Fmt { FMT_INT4 = 0, FMT_INT8 = 1, FMT_NF4 = 2, FMT_Q4G = 3, FMT_Q8G = 4, FMT_I4G32 = 5, FMT_I8S = 7 };
template <int FMT> constexpr bool kBytes = FMT == FMT_INT8 || FMT == FMT_I8S || FMT == FMT_Q8G;  // 8-bit codes
template <int FMT> constexpr bool kRowScale = FMT == FMT_INT8 || FMT == FMT_I8S;                 // one f32 scale per row

// The weight operand is the integer times 2^-kShift, undone in the scale: a partial of 64 (32)
// products then stays below the largest |x|, so it is finite for every finite x, and the smallest
// products (bf16 subnormal x) still have their last bit at or above 2^-149.
template <int FMT> constexpr int kShift = FMT == FMT_INT8 || FMT == FMT_NF4 ? 0 : FMT == FMT_I8S ? 14 : FMT == FMT_Q8G ? 13 : 11;

constexpr int kXcds = 8;
constexpr int kChunk = 64;          // K elements of a chunk
constexpr int kXRow = kChunk * 2;   // bytes of x per row and chunk
constexpr int kCopies = 16;         // of the NF4 decode table

struct QsProb {
    const uint16_t *x;
    const void *codes, *scales;
    const uint32_t *zeros;
    void *y;
    int N, K;
    int group;       // INT4
    int per_row;     // INT8: 1 per-channel scales, 0 per-tensor
    int y_vec;       // N % 4 == 0 and y 16-byte aligned
    int tile_begin;  // first workgroup of this problem
};

struct QsArgs {
    QsProb p[CFH_MAX_BATCH];
    int count, M, tiles_m, y_bf16;
    int tiles;       // workgroups of all problems
};

__device__ __forceinline__ rsrc_t make_rsrc(const void *base, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), static_cast<short>(0), static_cast<int>(bytes), 0x00020000);
}

// Waits until at most N vector-memory loads are outstanding and every LDS read has returned, and
// keeps memory accesses on their side of the wait (the compiler does not order LDS reads against
// the builtin: it has moved reads of a stage above the wait for the loads that fill it).
template <int N>
__device__ __forceinline__ void wait_vm_fence() {
    __builtin_amdgcn_s_waitcnt(vmcnt_imm(N) & ~(15 << 8));
    asm volatile("" ::: "memory");
}

__device__ __forceinline__ uint32_t pack_hi16(float a, float b) {
    return __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u);
}

// piece c of row r of an x stage
__device__ __forceinline__ int xswz(int r, int c) { return c ^ ((r >> 1) & 7); }

template <int FMT> constexpr bool fold32() { return FMT == FMT_Q4G || FMT == FMT_Q8G || FMT == FMT_I4G32; }
// vector-memory loads of one chunk per 32 weight rows: codes, scales, zero points
template <int FMT> constexpr int w_loads() { return kRowScale<FMT> || FMT == FMT_NF4 ? 2 : FMT == FMT_INT4 ? 1 : FMT == FMT_I4G32 ? 4 : 3; }

// One lane's codes and scales of a chunk (its row of 32, its half h of the MFMA's K).
template <int FMT>
struct WSet {
    uint4 w[kBytes<FMT> ? 2 : 1];
    uint32_t s, z;
};

// Which 8 k of the chunk MFMA step kk of half h takes (as the x piece index).  Formats that scale
// every 32 keep both halves of a step inside one 32-wide block: k = 32 (kk / 2) + 16 h + 8 (kk % 2);
// the others read each half's codes in one run: k = 32 h + 8 kk.
template <int FMT>
__device__ __forceinline__ int piece_of(int kk, int h) {
    return fold32<FMT>() ? 4 * (kk >> 1) + 2 * h + (kk & 1) : 4 * h + kk;
}

struct WAddr {
    rsrc_t rw, rs, rz;
    uint32_t vw, vs, vz;  // this lane's row offsets (row block 0)
    uint32_t row_w, row_s, row_z;  // bytes of 32 rows
};

template <int FMT>
__device__ __forceinline__ void load_w(const WAddr &A, int i, int c, int cpg, WSet<FMT> &r) {
    const uint32_t vw = A.vw + i * A.row_w, vs = A.vs + i * A.row_s;
    if constexpr (kRowScale<FMT>) {
        // bytes 32 h .. 32 h + 31 of the row's 64
        r.w[0] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(A.rw, vw, c * 64, 0));
        r.w[1] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(A.rw, vw + 16, c * 64, 0));
    } else if constexpr (FMT == FMT_Q8G) {
        // parts 2 h and 2 h + 1 of the 64-byte chunk: 8 bytes of each of its two blocks
        r.w[0] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(A.rw, vw, c * 64, 0));
        r.w[1] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(A.rw, vw + 16, c * 64, 0));
        r.s = __builtin_amdgcn_raw_buffer_load_b32(A.rs, vs, c * 4, 0);
    } else if constexpr (FMT == FMT_Q4G) {
        // the 64-byte chunk holds four blocks (two of these K chunks): 4 bytes of each block in
        // each of the parts 2 h, 2 h + 1
        const int o = (c >> 1) * 64 + (c & 1) * 8;
        const uint2 p = __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(A.rw, vw, o, 0));
        const uint2 q = __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(A.rw, vw + 16, o, 0));
        r.w[0] = make_uint4(p.x, q.x, p.y, q.y);  // step order: block, then part
        r.s = __builtin_amdgcn_raw_buffer_load_b32(A.rs, vs, c * 4, 0);
    } else if constexpr (FMT == FMT_I4G32) {
        // words 2 h, 2 h + 1 of each group of four
        const uint2 p = __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(A.rw, vw, c * 32, 0));
        const uint2 q = __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(A.rw, vw + 16, c * 32, 0));
        r.w[0] = make_uint4(p.x, p.y, q.x, q.y);
        r.s = __builtin_amdgcn_raw_buffer_load_b32(A.rs, vs, c * 4, 0);
        r.z = __builtin_amdgcn_raw_buffer_load_b32(A.rz, A.vz + i * A.row_z, (c >> 2) * 4, 0);
    } else if constexpr (FMT == FMT_NF4) {
        r.w[0] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(A.rw, vw, c * 32, 0));
        r.s = __builtin_amdgcn_raw_buffer_load_b32(A.rs, vs, (c >> cpg) * 4, 0);  // cpg: log2 of chunks per block
    } else {
        r.w[0] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(A.rw, vw, c * 32, 0));
    }
}

// Opaque constants: kept in registers, so that the masks fold into v_and_or_b32 and the multiplier
// of v_fma_mix_f32 stays one.
struct DecodeK {
    uint32_t m0, m1, c0, c1;
    float unit;  // 2^-kShift
};

// 8 codes (k order) -> unit (q - z) as bf16, exact; ce = -unit (1024 + z), co = -unit (64 + z).  Even nibbles become
// the f16 1024 + q, odd ones (at mantissa bits 4..7) 64 + q; v_fma_mix_f32 subtracts exactly.
__device__ __forceinline__ bf16x8_t decode4(uint32_t w, float ce, float co, const DecodeK &K) {
    typedef _Float16 h2_t __attribute__((ext_vector_type(2)));
    const uint32_t w8 = w >> 8;
    const h2_t p0 = __builtin_bit_cast(h2_t, (w & K.m0) | K.c0), p1 = __builtin_bit_cast(h2_t, (w & K.m1) | K.c1);
    const h2_t p2 = __builtin_bit_cast(h2_t, (w8 & K.m0) | K.c0), p3 = __builtin_bit_cast(h2_t, (w8 & K.m1) | K.c1);
    const float q0 = __builtin_fmaf(static_cast<float>(p0.x), K.unit, ce), q4 = __builtin_fmaf(static_cast<float>(p0.y), K.unit, ce);
    const float q1 = __builtin_fmaf(static_cast<float>(p1.x), K.unit, co), q5 = __builtin_fmaf(static_cast<float>(p1.y), K.unit, co);
    const float q2 = __builtin_fmaf(static_cast<float>(p2.x), K.unit, ce), q6 = __builtin_fmaf(static_cast<float>(p2.y), K.unit, ce);
    const float q3 = __builtin_fmaf(static_cast<float>(p3.x), K.unit, co), q7 = __builtin_fmaf(static_cast<float>(p3.y), K.unit, co);
    return __builtin_bit_cast(bf16x8_t, make_uint4(pack_hi16(q0, q1), pack_hi16(q2, q3), pack_hi16(q4, q5), pack_hi16(q6, q7)));
}

// 8 signed bytes -> unit q as bf16: f16 1024 + (q + 128) from the byte, minus 1152 times unit.
__device__ __forceinline__ bf16x8_t decode8s(uint32_t a, uint32_t b, const DecodeK &K) {
    typedef _Float16 h2_t __attribute__((ext_vector_type(2)));
    const float c = -1152.0f * K.unit;
    const h2_t a0 = __builtin_bit_cast(h2_t, (a & K.m1) ^ K.c1), a1 = __builtin_bit_cast(h2_t, ((a >> 8) & K.m1) ^ K.c1);
    const h2_t b0 = __builtin_bit_cast(h2_t, (b & K.m1) ^ K.c1), b1 = __builtin_bit_cast(h2_t, ((b >> 8) & K.m1) ^ K.c1);
    const float q0 = __builtin_fmaf(static_cast<float>(a0.x), K.unit, c), q2 = __builtin_fmaf(static_cast<float>(a0.y), K.unit, c);
    const float q1 = __builtin_fmaf(static_cast<float>(a1.x), K.unit, c), q3 = __builtin_fmaf(static_cast<float>(a1.y), K.unit, c);
    const float q4 = __builtin_fmaf(static_cast<float>(b0.x), K.unit, c), q6 = __builtin_fmaf(static_cast<float>(b0.y), K.unit, c);
    const float q5 = __builtin_fmaf(static_cast<float>(b1.x), K.unit, c), q7 = __builtin_fmaf(static_cast<float>(b1.y), K.unit, c);
    return __builtin_bit_cast(bf16x8_t, make_uint4(pack_hi16(q0, q1), pack_hi16(q2, q3), pack_hi16(q4, q5), pack_hi16(q6, q7)));
}

// 8 signed bytes -> q as bf16: one sign-extending byte conversion per code (12 instructions against 18).
__device__ __forceinline__ bf16x8_t decode8(uint32_t a, uint32_t b) {
    float v[8];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        v[j] = static_cast<float>(static_cast<int8_t>(a >> (8 * j)));
        v[4 + j] = static_cast<float>(static_cast<int8_t>(b >> (8 * j)));
    }
    return __builtin_bit_cast(bf16x8_t, make_uint4(pack_hi16(v[0], v[1]), pack_hi16(v[2], v[3]), pack_hi16(v[4], v[5]), pack_hi16(v[6], v[7])));
}

// XL: 1 KB loads of x per chunk (8 rows each), the size of a stage: 4 J, or fewer where M <= 8 XL.
// lv: the lane's offset in loads 0 and 1; a later pair's rows are 32 K bytes further each.
template <int XL>
__device__ __forceinline__ void issue_x(rsrc_t rx, uint8_t *__restrict__ dst, const int (&lv)[2], int K, int c) {
#pragma unroll
    for (int t = 0; t < XL; ++t)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (__attribute__((address_space(3))) void *)(dst + t * 1024), 16,
                                                 lv[t & 1] + (t >> 1) * 32 * K, c * kXRow, 0, 0);
}

// One chunk: refill stage `nxt` and set `wn` (used in the previous step) with chunk c_next, wait
// for chunk c, decode and multiply.  `cur` and `nxt` differ: the reads need not wait for the refill.
template <int FMT, int I, int J, int S, int XL>
__device__ __forceinline__ void chunk_step(const uint8_t *__restrict__ cur, uint8_t *__restrict__ nxt, bool refill, rsrc_t rx,
                                           const int (&lv)[2], int K, const WAddr &A, const uint32_t *__restrict__ sz, int cpg, int c,
                                           int c_next, int fr, int h,
                                           const DecodeK &D, const float (&rs)[I][2], const WSet<FMT> (&w)[I], WSet<FMT> (&wn)[I], floatx16 (&tot)[I][J]) {
    constexpr int kLoads = XL + w_loads<FMT>() * I;
    const int xr = XL < 4 * J ? min(fr, 8 * XL - 1) : fr;  // a lane past the staged rows repeats the last
    wait_vm_fence<63>();  // the previous step's reads of `nxt` returned
    if (refill) {
        issue_x<XL>(rx, nxt, lv, K, c_next);
#pragma unroll
        for (int i = 0; i < I; ++i) load_w<FMT>(A, i, c_next, cpg, wn[i]);
    }
    wait_vm_fence<(S - 1) * kLoads>();
    constexpr float kUp = static_cast<float>(1 << kShift<FMT>);
    float ce[I], co[I], sc[I];
    if constexpr (FMT == FMT_Q4G) {
#pragma unroll
        for (int i = 0; i < I; ++i) ce[i] = -1032.0f * D.unit, co[i] = -72.0f * D.unit;
    }
    if constexpr (FMT == FMT_INT4) {
        const uint32_t *row = sz + c / cpg * (32 * I) + fr;
#pragma unroll
        for (int i = 0; i < I; ++i) {
            const uint32_t v = row[32 * i];
            const float z = static_cast<float>(v >> 16);
            ce[i] = -(1024.0f + z) * D.unit;
            co[i] = -(64.0f + z) * D.unit;
            sc[i] = f16_to_f32(static_cast<uint16_t>(v)) * kUp;
        }
    }
    floatx16 part[I][J];
    static_for<4>([&](auto KK) {
        constexpr int kk = decltype(KK)::value;
        bf16x8_t xf[J];
#pragma unroll
        for (int j = 0; j < J; ++j)
            xf[j] = *reinterpret_cast<const bf16x8_t *>(cur + (32 * j + xr) * kXRow + xswz(xr, piece_of<FMT>(kk, h)) * 16);
        if constexpr (FMT == FMT_I4G32 && (kk & 1) == 0) {
            const int nib = 2 * (c & 3) + (kk >> 1);
#pragma unroll
            for (int i = 0; i < I; ++i) {
                const float z = static_cast<float>((w[i].z >> (4 * nib)) & 15u);
                ce[i] = -(1024.0f + z) * D.unit;
                co[i] = -(64.0f + z) * D.unit;
            }
        }
#pragma unroll
        for (int i = 0; i < I; ++i) {
            bf16x8_t wf, wl;
            if constexpr (FMT == FMT_NF4) {
                // the table's row of a code byte holds, per copy, the T_hi pair and the T_lo pair
                const uint4 q = w[i].w[0];
                const uint32_t word = kk == 0 ? q.x : kk == 1 ? q.y : kk == 2 ? q.z : q.w;
                uint32_t hi[4], lo[4];
#pragma unroll
                for (int b = 0; b < 4; ++b) {
                    const uint2 e = *reinterpret_cast<const uint2 *>(sz + ((word >> (8 * b)) & 0xFFu) * (2 * kCopies) + 2 * (fr % kCopies));
                    hi[b] = e.x, lo[b] = e.y;
                }
                wf = __builtin_bit_cast(bf16x8_t, make_uint4(hi[0], hi[1], hi[2], hi[3]));
                wl = __builtin_bit_cast(bf16x8_t, make_uint4(lo[0], lo[1], lo[2], lo[3]));
            } else if constexpr (FMT == FMT_INT8) {
                const uint4 q = w[i].w[kk >> 1];
                wf = (kk & 1) ? decode8(q.z, q.w) : decode8(q.x, q.y);
            } else if constexpr (FMT == FMT_I8S) {
                const uint4 q = w[i].w[kk >> 1];
                wf = (kk & 1) ? decode8s(q.z, q.w, D) : decode8s(q.x, q.y, D);
            } else if constexpr (FMT == FMT_Q8G) {
                const uint4 q = w[i].w[kk & 1];  // part 2 h + kk % 2, block kk / 2
                wf = (kk >> 1) ? decode8s(q.z, q.w, D) : decode8s(q.x, q.y, D);
            } else {
                const uint4 q = w[i].w[0];
                wf = decode4(kk == 0 ? q.x : kk == 1 ? q.y : kk == 2 ? q.z : q.w, ce[i], co[i], D);
            }
            // a fresh partial where a scale begins
            constexpr bool kStart = FMT == FMT_INT8 ? false : fold32<FMT>() ? (kk & 1) == 0 : kk == 0;
#pragma unroll
            for (int j = 0; j < J; ++j) {
                if constexpr (FMT == FMT_INT8) {
                    tot[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xf[j], wf, tot[i][j], 0, 0, 0);
                } else if constexpr (kStart) {
                    const floatx16 zero{};
                    part[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xf[j], wf, zero, 0, 0, 0);
                } else {
                    part[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xf[j], wf, part[i][j], 0, 0, 0);
                }
                if constexpr (FMT == FMT_NF4) part[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xf[j], wl, part[i][j], 0, 0, 0);
            }
        }
        if constexpr (FMT != FMT_INT8 && (fold32<FMT>() ? (kk & 1) == 1 : kk == 3)) {
#pragma unroll
            for (int i = 0; i < I; ++i) {
                if constexpr (FMT == FMT_NF4) sc[i] = __uint_as_float(w[i].s);
                if constexpr (fold32<FMT>()) sc[i] = f16_to_f32(static_cast<uint16_t>(kk == 1 ? (w[i].s & 0xFFFFu) : (w[i].s >> 16))) * kUp;
#pragma unroll
                for (int j = 0; j < J; ++j)
#pragma unroll
                    for (int e = 0; e < 16; ++e) {
                        // INT8: the row's scale and 2^kShift, split so that neither factor overflows
                        const float p = FMT == FMT_I8S ? part[i][j][e] * rs[i][1] : part[i][j][e];
                        tot[i][j][e] = __builtin_fmaf(FMT == FMT_I8S ? rs[i][0] : sc[i], p, tot[i][j][e]);
                    }
            }
        }
    });
}

// The NF4 table of QLoRA, as the evaluator's f32 values.  In LDS: for each code byte (two codes),
// kCopies copies of its T_hi = RNE(T) and T_lo = RNE(T - T_hi) bf16 pairs, the operand words of two MFMAs
// (16 copies: 32 KB, lanes r and r + 16 share one, so a read takes at most two passes).
__constant__ float kNf4S[16] = {
    -1.0f, -0.6961928009986877f, -0.5250730514526367f, -0.39491748809814453f,
    -0.28444138169288635f, -0.18477343022823334f, -0.09105003625154495f, 0.0f,
    0.07958029955625534f, 0.16093020141124725f, 0.24611230194568634f, 0.33791524171829224f,
    0.44070982933044434f, 0.5626170039176941f, 0.7229568362236023f, 1.0f};

// LDS of a workgroup: the x rings and the tile's `groups` scales and zero points (INT4) or the decode
// table (NF4), later the waves' partial tiles.
template <int FMT, int I, int J, int NW, int S, int XL>
constexpr int64_t lds_bytes(int64_t groups) {
    const int64_t ring = NW * S * XL * 1024 + (FMT == FMT_INT4 ? groups * 32 * I * 4 : FMT == FMT_NF4 ? 256 * kCopies * 8 : 0), sums = NW * 32 * J * (32 * I + 4) * 4;
    return ring > sums ? ring : sums;
}
constexpr int64_t kLdsMax = 160 * 1024;

template <int FMT, int I, int J, int NW, int S, int XL>
__global__ __launch_bounds__(64 * NW) void qsplit_kernel(QsArgs g) {
    constexpr int kBN = 32 * I, kBM = 32 * J, kStage = XL * 1024;
    extern __shared__ __align__(16) uint8_t lds[];
    int pid = blockIdx.x, pi = 0;
    while (pi + 1 < g.count && pid >= g.p[pi + 1].tile_begin) ++pi;
    const QsProb &a = g.p[pi];
    pid -= a.tile_begin;
    // each XCD owns a contiguous run of each problem's tiles, in groups of up to 8 m tiles of one W panel
    // (their x rows stay in the XCD's L2).  A run of the whole batch's tiles instead, longest K first, gave one
    // XCD all of a layer's W_down (the seven matrices, us, whole batch / each problem: INT4 at M = 8 54 / 37,
    // INT8 87 / 61; Q8_0 at M = 40 143 / 93; NF4 at M = 64 122 / 71).
    {
        const int tiles = (pi + 1 < g.count ? g.p[pi + 1].tile_begin : g.tiles) - a.tile_begin;
        const int per_xcd = tiles / kXcds, full = per_xcd * kXcds;
        if (pid < full) pid = (pid % kXcds) * per_xcd + pid / kXcds;
    }
    const int M = g.M, N = a.N, K = a.K;
    const int tiles_n = (N + kBN - 1) / kBN;
    const int span = 8 * tiles_n, first_m = pid / span * 8, gm = min(8, g.tiles_m - first_m);
    const int m0 = (first_m + pid % span % gm) * kBM, n0 = pid % span / gm * kBN;
    const int lane = threadIdx.x & 63, fr = lane & 31, h = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);

    const rsrc_t rx = make_rsrc(a.x + static_cast<int64_t>(m0) * K, static_cast<uint32_t>(min(kBM, M - m0)) * K * 2);
    int lv[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) lv[u] = (8 * u + (lane >> 3)) * K * 2 + xswz(8 * u + (lane >> 3), lane & 7) * 16;
    WAddr A;
    const int row_bytes = kBytes<FMT> ? K : K / 2;
    // scales per row: GGUF planes 8 ceil(K / 32 / 8), INT4 8 ceil(G / 8)
    // (NF4: f32 absmax, K / block)
    const int G = FMT == FMT_INT4 || FMT == FMT_I4G32 ? K / a.group : K / 32;
    const int ZW = (G + 7) / 8, GP = ZW * 8;
    const uint32_t nv = static_cast<uint32_t>(min(kBN, N - n0));
    A.rw = make_rsrc(static_cast<const uint8_t *>(a.codes) + static_cast<int64_t>(n0) * row_bytes, nv * row_bytes);
    const int NB = FMT == FMT_NF4 ? K / a.group : 0;  // absmax blocks per row
    A.rs = FMT == FMT_NF4 ? make_rsrc(static_cast<const float *>(a.scales) + static_cast<int64_t>(n0) * NB, nv * NB * 4)
                          : make_rsrc(static_cast<const uint16_t *>(a.scales) + static_cast<int64_t>(n0) * (kRowScale<FMT> ? 0 : GP),
                                      kRowScale<FMT> ? 0 : nv * GP * 2);
    constexpr bool kZeros = FMT == FMT_INT4 || FMT == FMT_I4G32;
    A.rz = make_rsrc(a.zeros + static_cast<int64_t>(n0) * (kZeros ? ZW : 0), kZeros ? nv * ZW * 4 : 0);
    A.vw = fr * row_bytes + (FMT == FMT_INT4 || FMT == FMT_NF4 ? 16 : FMT == FMT_I4G32 ? 8 : 32) * h;
    A.vs = FMT == FMT_NF4 ? fr * NB * 4 : fr * GP * 2;
    A.vz = fr * ZW * 4;
    A.row_w = 32 * row_bytes;
    A.row_s = FMT == FMT_NF4 ? 32 * NB * 4 : 32 * GP * 2;
    A.row_z = 32 * ZW * 4;
    const int cpg = FMT == FMT_INT4 ? a.group / kChunk : FMT == FMT_NF4 ? __builtin_ctz(static_cast<uint32_t>(a.group / kChunk)) : 1;

    auto opaque = [](uint32_t v) __attribute__((always_inline)) {
        asm("" : "+v"(v));
        return v;
    };
    // 4-bit: nibbles at bits 0..3 and 4..7 of each half, f16 1024 and 64; 8-bit: bytes, f16 1024 + 128
    const DecodeK D{opaque(0x000F000Fu), opaque(kBytes<FMT> ? 0x00FF00FFu : 0x00F000F0u), opaque(0x64006400u),
                    opaque(kBytes<FMT> ? 0x64806480u : 0x54005400u), __uint_as_float(opaque((127u - kShift<FMT>) << 23))};
    const float *sp = static_cast<const float *>(a.scales);
    float rs[I][2];
    if constexpr (FMT == FMT_I8S) {
#pragma unroll
        for (int i = 0; i < I; ++i) {
            const int n = n0 + 32 * i + fr;
            const float v = n < N ? sp[a.per_row ? n : 0] : 0.f, up = static_cast<float>(1 << kShift<FMT>);
            const bool large = fabsf(v) >= 0x1p100f;
            rs[i][0] = large ? v : v * up;
            rs[i][1] = large ? up : 1.0f;
        }
    }

    floatx16 tot[I][J];
#pragma unroll
    for (int i = 0; i < I; ++i)
#pragma unroll
        for (int j = 0; j < J; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) tot[i][j][e] = 0.f;

    const int chunks = K / kChunk;
    const int n_own = chunks > wave ? (chunks - wave + NW - 1) / NW : 0;
    uint8_t *ring = lds + wave * S * kStage;
    auto c_of = [&](int t) { return wave + NW * t; };
    WSet<FMT> ws[S][I];
    static_for<S - 1>([&](auto TI) {
        constexpr int t = decltype(TI)::value;
        if (t < n_own) {
            asm volatile("" ::: "memory");  // the waits count whole chunks
            issue_x<XL>(rx, ring + t * kStage, lv, K, c_of(t));
#pragma unroll
            for (int i = 0; i < I; ++i) load_w<FMT>(A, i, c_of(t), cpg, ws[t][i]);
        }
    });
    // INT4: every group's scale (f16, low half) and zero point of the tile's rows, [group][row], once
    // per workgroup.  A lane-per-row load of two bytes costs the L1 as much as one of sixteen; loaded
    // per chunk they took a quarter of the time of 64 x 64 tiles.
    uint32_t *sz = reinterpret_cast<uint32_t *>(lds + NW * S * kStage);
    if constexpr (FMT == FMT_INT4) {
        for (int o = threadIdx.x; o < kBN * ZW; o += 64 * NW) {
            const int r = o / ZW, g8 = o - r * ZW;
            const uint4 d = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(A.rs, r * GP * 2 + g8 * 16, 0, 0));
            const uint32_t z = __builtin_amdgcn_raw_buffer_load_b32(A.rz, (r * ZW + g8) * 4, 0, 0);
            const uint32_t dw[4] = {d.x, d.y, d.z, d.w};
#pragma unroll
            for (int q = 0; q < 8; ++q)
                if (8 * g8 + q < G) sz[(8 * g8 + q) * kBN + r] = ((dw[q >> 1] >> (16 * (q & 1))) & 0xFFFFu) | ((z >> (4 * q)) & 15u) << 16;
        }
        __syncthreads();
    }
    if constexpr (FMT == FMT_NF4) {
        for (int o = threadIdx.x; o < 256 * kCopies; o += 64 * NW) {
            const int v = o / kCopies;
            const float t0 = kNf4S[v & 15], t1 = kNf4S[v >> 4];
            const uint32_t hi = f32x2_to_bf16x2_rne(t0, t1);
            const uint32_t lo = f32x2_to_bf16x2_rne(t0 - __uint_as_float(hi << 16), t1 - __uint_as_float(hi & 0xFFFF0000u));
            *reinterpret_cast<uint2 *>(sz + 2 * o) = make_uint2(hi, lo);
        }
        __syncthreads();
    }
    int t0 = 0;
    for (; t0 + 2 * S - 2 < n_own; t0 += S)
        static_for<S>([&](auto SI) {
            constexpr int s = decltype(SI)::value, p = (s + S - 1) % S;
            chunk_step<FMT, I, J, S, XL>(ring + s * kStage, ring + p * kStage, true, rx, lv, K, A, sz, cpg, c_of(t0 + s),
                                     c_of(t0 + s + S - 1), fr, h, D, rs, ws[s], ws[p], tot);
        });
    for (; t0 < n_own; t0 += S)
        static_for<S>([&](auto SI) {
            constexpr int s = decltype(SI)::value, p = (s + S - 1) % S;
            const int t = t0 + s;
            if (t < n_own) {
                if (t + S - 1 >= n_own) wait_vm_fence<0>();  // fewer than S - 1 chunks follow
                chunk_step<FMT, I, J, S, XL>(ring + s * kStage, ring + p * kStage, t + S - 1 < n_own, rx, lv, K, A, sz, cpg,
                                         c_of(t), c_of(t + S - 1), fr, h, D, rs, ws[s], ws[p], tot);
            }
        });

    // ---- sum of the waves' tiles: tot[i][j] reg 4 g + q holds m = 32 j + 8 g + 4 h + q, n = 32 i + fr ----
    __syncthreads();  // every wave is done with its ring (all of its loads were waited for)
    constexpr int kRow = kBN + 4;
    float *sums = reinterpret_cast<float *>(lds);
#pragma unroll
    for (int i = 0; i < I; ++i)
#pragma unroll
        for (int j = 0; j < J; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e)
                sums[(wave * kBM + 32 * j + 8 * (e >> 2) + 4 * h + (e & 3)) * kRow + 32 * i + fr] = tot[i][j][e];
    __syncthreads();
#pragma unroll 2
    for (int o = threadIdx.x; o < kBM * kBN / 4; o += 64 * NW) {
        const int ml = o / (kBN / 4), nl = o % (kBN / 4) * 4;
        const int m = m0 + ml, n = n0 + nl;
        if (m >= M || n >= N) continue;
        float4 v = *reinterpret_cast<const float4 *>(sums + ml * kRow + nl);
#pragma unroll
        for (int w = 1; w < NW; ++w) {
            const float4 p = *reinterpret_cast<const float4 *>(sums + (w * kBM + ml) * kRow + nl);
            v.x += p.x, v.y += p.y, v.z += p.z, v.w += p.w;
        }
        float r[4] = {v.x, v.y, v.z, v.w};
        if constexpr (FMT == FMT_INT8) {
#pragma unroll
            for (int q = 0; q < 4; ++q) r[q] *= sp[a.per_row ? min(n + q, N - 1) : 0];
        }
        const int64_t at = static_cast<int64_t>(m) * N + n;
        if (a.y_vec) {
            if (g.y_bf16)
                *reinterpret_cast<uint2 *>(static_cast<uint16_t *>(a.y) + at) = make_uint2(f32x2_to_bf16x2_rne(r[0], r[1]), f32x2_to_bf16x2_rne(r[2], r[3]));
            else
                *reinterpret_cast<float4 *>(static_cast<float *>(a.y) + at) = make_float4(r[0], r[1], r[2], r[3]);
        } else {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                if (n + q < N) {
                    if (g.y_bf16) static_cast<uint16_t *>(a.y)[at + q] = f32_to_bf16_rne(r[q]);
                    else static_cast<float *>(a.y)[at + q] = r[q];
                }
            }
        }
    }
}

int64_t int4_groups(const QsProb &p) { return p.K / p.group; }

template <int FMT, int I, int J, int NW, int S, int XL>
void launch_x(QsArgs a, hipStream_t st) {
    int64_t lds = 0, tiles = 0;
    a.tiles_m = (a.M + 32 * J - 1) / (32 * J);
    for (int i = 0; i < a.count; ++i) {
        lds = std::max(lds, lds_bytes<FMT, I, J, NW, S, XL>(FMT == FMT_INT4 ? int4_groups(a.p[i]) : 0));
        a.p[i].tile_begin = static_cast<int>(tiles);
        tiles += static_cast<int64_t>(a.tiles_m) * ((a.p[i].N + 32 * I - 1) / (32 * I));
    }
    require(lds <= kLdsMax && tiles <= 0x7fffffff, "qsplit_kernel: LDS or tiles");
    a.tiles = static_cast<int>(tiles);
    static std::atomic<uint64_t> done{0};  // devices whose dynamic-LDS limit is raised (bit = ordinal < 64)
    int dev = 0;
    check_hip(hipGetDevice(&dev), "hipGetDevice");
    const uint64_t bit = dev < 64 ? (uint64_t{1} << dev) : 0;
    const auto kern = qsplit_kernel<FMT, I, J, NW, S, XL>;
    if (bit == 0 || !(done.load(std::memory_order_acquire) & bit)) {
        check_hip(hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, kLdsMax),
                  "hipFuncSetAttribute(qsplit_kernel)");
        done.fetch_or(bit, std::memory_order_acq_rel);
    }
    kern<<<dim3(static_cast<unsigned>(tiles)), dim3(64 * NW), static_cast<size_t>(lds), st>>>(a);
    check_launch("qsplit_kernel");
}

// Fewest rows that reach a 32-row tile of 32 I columns (qsplit_ok, launch_fmt): x stages for fewer are not built.
template <int FMT, int I>
constexpr int kMinRows = FMT == FMT_Q4G || FMT == FMT_Q8G ? 33 : FMT == FMT_NF4 || (FMT == FMT_I8S && I == 2) ? 17 : 2;

template <int FMT, int I, int J, int NW, int S>
void launch(const QsArgs &a, hipStream_t st) {
    if constexpr (J == 1) {
        if constexpr (kMinRows<FMT, I> <= 16) {
            if (a.M <= 8) return launch_x<FMT, I, J, NW, S, 1>(a, st);
            if (a.M <= 16) return launch_x<FMT, I, J, NW, S, 2>(a, st);
        }
        launch_x<FMT, I, J, NW, S, 4>(a, st);
    } else {
        launch_x<FMT, I, J, NW, S, 4 * J>(a, st);
    }
}

int64_t tiles_of(const QsArgs &a, int64_t bn, int64_t bm) {
    int64_t t = 0;
    for (int i = 0; i < a.count; ++i) t += (a.M + bm - 1) / bm * ((a.p[i].N + bn - 1) / bn);
    return t;
}
double rounds(int64_t tiles) { return static_cast<double>((tiles + cu_count() - 1) / cu_count()); }

// Rounds of 64 x 64 tiles that a round of 64 (n) x 128 takes the time of, and that a round of the one-MFMA
// prefill kernel's 256 (n) x 128 tiles takes, however few they are.
struct Costs {
    double r128, rpf;
};
Costs costs(int fmt, int64_t group) {
    if (fmt == FMT_INT8) return {1.5, 3.1};
    if (fmt == FMT_Q4G) return {1.75, 4.0};
    if (fmt == FMT_Q8G) return {1.75, 4.6};
    return group == 32 ? Costs{1.65, 3.5} : Costs{1.95, 4.0};
}

// Whether a problem of the kernel's runs on it.  By the problem alone, so that a batch gives the bits of
// one call per problem:
//   * up to 64 rows always; NF4 up to one 64 x 64 tile per CU, beyond which nf4_mfma_kernel's cheaper decode
//     decides (K = 4096 at M = 17 / 64, us there / here: n = 16384 27.7 / 17.2, 37 / 25; n = 17000 27.6 /
//     29.3, 37 / 42);
//   * above, where the one-MFMA prefill kernel does not cost less (INT4, 4096 x 4096 at M = 512: 33 us here
//     against 59; 11008 x 4096 at M = 512: 92 against 68; 4096 x 11008 at M = 603: 104 against 123); NF4 always.
bool chosen(int fmt, const QsArgs &a) {
    if (fmt == FMT_NF4) return a.M > 64 || tiles_of(a, 64, 64) <= cu_count();
    if (a.M <= 64 || tiles_of(a, 32, 64) <= cu_count()) return true;
    const Costs c = costs(fmt, a.p[0].group);
    const double here = std::min(rounds(tiles_of(a, 64, 64)), c.r128 * rounds(tiles_of(a, 64, 128)));
    const bool rows96 = fmt != FMT_INT8 && (fmt != FMT_INT4 || (a.p[0].group != 64 && a.p[0].group != 32));
    return here <= c.rpf * prefill_cost(fmt, rows96, a.M, a.p[0].N);
}

// The tile by the number of workgroups (us per round of 256 workgroups at K = 4096, INT4 / INT8 /
// Q8_0): 32 x 32 up to one tile per CU (8 / 9 / 11), three for M <= 32 (n = 20000, 625 tiles, at M = 8
// 16.9 / 24.0; as 64 x 32 20.0 / 32.1), INT8 at M <= 16 always (the per-row form decodes twice as long:
// n = 131072 119 against 136); then 64 (n) x 32 for M <= 32 (INT4 n = 32000 at M = 24 26.0; as 32 x 32
// 29.7); 32 (n) x 64 up to one per CU (12 / 12 / 14); then 64 x 64 (18 / 18 / 23 a round) or, above
// M = 64, 64 (n) x 128 (35 / 28 / 40) where its rounds cost less.  Every shape up to M = 64 sums the same
// chunks in the same order.
template <int FMT, int FMT_SMALL>
void launch_fmt(const QsArgs &a, hipStream_t st) {
    const int64_t cus = cu_count(), t32 = tiles_of(a, 32, 32);
    if (t32 <= (a.M <= 32 ? 3 * cus : cus) || (FMT == FMT_INT8 && a.M <= 16)) {
        launch<FMT_SMALL, 1, 1, 8, 2>(a, st);
    } else if (a.M <= 32) {
        if constexpr (kMinRows<FMT_SMALL, 2> <= 32) launch<FMT_SMALL, 2, 1, 8, 2>(a, st);
        else require(false, "qsplit_kernel: GGUF planes from 33 rows on");
    } else if (a.M <= 64) {
        if (tiles_of(a, 32, 64) <= cus) launch<FMT_SMALL, 1, 2, 8, 2>(a, st);
        else launch<FMT_SMALL, 2, 2, 8, 2>(a, st);
    } else if (tiles_of(a, 32, 64) <= cus) {
        launch<FMT, 1, 2, 8, 2>(a, st);
    } else if (rounds(tiles_of(a, 64, 64)) <= costs(FMT == FMT_I4G32 ? FMT_INT4 : FMT, a.p[0].group).r128 * rounds(tiles_of(a, 64, 128))) {
        launch<FMT, 2, 2, 8, 2>(a, st);
    } else {
        launch<FMT, 2, 4, 4, 2>(a, st);
    }
}

// NF4 (two MFMAs per product), us per round of 256 workgroups at K = 4096: 32 x 32 tiles up to one per CU
// (10), 64 (n) x 32 beyond for M <= 32 (16), 32 (n) x 64 up to one per CU (14), then 64 x 64 (23 a round),
// which holds to the largest M (4096 x 4096 at M = 64 / 512 / 4096 12 / 49 / 322 us, nf4_mfma_kernel 36 /
// 49 / 326; 4096 x 11008 at M = 4096 766 / 997).  All sum the same chunks in the same order.
void launch_nf4(const QsArgs &a, hipStream_t st) {
    const int64_t cus = cu_count();
    if (tiles_of(a, 32, 32) <= cus) launch<FMT_NF4, 1, 1, 8, 2>(a, st);
    else if (a.M <= 32) launch<FMT_NF4, 2, 1, 8, 2>(a, st);
    else if (tiles_of(a, 32, 64) <= cus) launch<FMT_NF4, 1, 2, 8, 2>(a, st);
    else launch<FMT_NF4, 2, 2, 8, 2>(a, st);
}

void launch_any(int fmt, const QsArgs &a, hipStream_t st) {
    if (fmt == FMT_INT8) launch_fmt<FMT_INT8, FMT_I8S>(a, st);
    else if (fmt == FMT_NF4) launch_nf4(a, st);
    else if (fmt == FMT_Q4G) launch_fmt<FMT_Q4G, FMT_Q4G>(a, st);
    else if (fmt == FMT_Q8G) launch_fmt<FMT_Q8G, FMT_Q8G>(a, st);
    else if (a.p[0].group == 32) launch_fmt<FMT_I4G32, FMT_I4G32>(a, st);
    else launch_fmt<FMT_INT4, FMT_INT4>(a, st);
}

QsProb prob(const uint16_t *x, int64_t n, int64_t k, int64_t group, const void *codes, const void *scales,
            const uint32_t *zeros, int per_row, void *y) {
    return QsProb{x, codes, scales, zeros, y, static_cast<int>(n), static_cast<int>(k), static_cast<int>(group), per_row,
                  (n % 4 == 0 && aligned(y, 16)) ? 1 : 0, 0};
}

}  // namespace

// Whether qsplit_kernel takes a problem of M = m >= 2 rows.  The variables that choose a prefill
// kernel keep M > 16 off it (NF4: CASTFORGE_NF4_MFMA=0 alone).
bool qsplit_ok(int fmt, const uint16_t *x, int64_t m, int64_t n, int64_t k, int64_t group, const void *codes, const void *scales) {
    if (fmt != FMT_INT4 && fmt != FMT_INT8 && fmt != FMT_NF4 && fmt != FMT_Q4G && fmt != FMT_Q8G) return false;
    // GGUF up to 32 rows: the skinny kernel, for single calls too, so that a batch gives their bits (Q8_0 / Q4_0
    // at M = 8, us there / here: W_gate and W_up in one launch 36 / 41, 26 / 34; a layer's seven matrices 71 / 75,
    // 50 / 59; one 4096 x 4096 14 / 11, 11 / 10)
    if ((fmt == FMT_Q4G || fmt == FMT_Q8G) && m <= 32) return false;
    // NF4: M > 16 (a partial reaches 64 |x|; up to 16 rows the skinny kernels take any finite x), blocks a
    // power of two; CASTFORGE_NF4_MFMA=0 keeps it on the skinny / prefill kernels (for comparison)
    if (fmt == FMT_NF4) {
        if (m < 17 || k < 256 || group < kChunk || (group & (group - 1)) != 0 || k % group != 0) return false;
        const char *e = std::getenv("CASTFORGE_NF4_MFMA");
        if (e && std::strcmp(e, "0") == 0) return false;
    }
    if (m < 2 || n < 1 || k < kChunk || k % kChunk != 0) return false;
    if (m > 0x7fffffff || n > 0x7fffffff) return false;
    // 32-bit buffer offsets over one tile's rows of x (128) and of codes (64)
    if (int64_t{128} * k * 2 >= (int64_t{1} << 31)) return false;
    if (!aligned(x, 16) || !aligned(codes, 16) || !aligned(scales, fmt == FMT_INT8 || fmt == FMT_NF4 ? 4 : 16)) return false;
    if (fmt == FMT_Q4G && (group != 32 || k % 128 != 0)) return false;
    if (fmt == FMT_Q8G && group != 32) return false;
    if (fmt == FMT_INT4) {
        if (k % group != 0 || (group != 32 && group % kChunk != 0)) return false;
        // groups of 64 and more: the largest tile's scales and zero points next to the x rings, up to 128 groups
        // (K = 8192 in groups of 64); longer rows stay on the skinny and prefill kernels
        if (group != 32 && lds_bytes<FMT_INT4, 2, 2, 8, 2, 8>(k / group) > kLdsMax) return false;
    }
    if (fmt != FMT_NF4 && m > 16 && (std::getenv("CASTFORGE_PREFILL_I4") || std::getenv("CASTFORGE_PREFILL_TILE"))) return false;
    return true;
}

// Whether qsplit_kernel runs a problem, alone or in a batch.
bool qsplit_takes(int fmt, const uint16_t *x, int64_t m, int64_t n, int64_t k, int64_t group, const void *codes, const void *scales) {
    if (!qsplit_ok(fmt, x, m, n, k, group, codes, scales)) return false;
    QsArgs a{};
    a.p[0].N = static_cast<int>(n), a.p[0].K = static_cast<int>(k), a.p[0].group = static_cast<int>(group);
    a.count = 1, a.M = static_cast<int>(m);
    return chosen(fmt, a);
}

// Runs a product on qsplit_kernel; false where the kernel does not take it or another is faster.
bool qsplit_try(int fmt, const uint16_t *x, int64_t m, int64_t n, int64_t k, int64_t group, const void *codes,
                const void *scales, const uint32_t *zeros, int per_row, void *y, int y_bf16, hipStream_t st) {
    if (!qsplit_takes(fmt, x, m, n, k, group, codes, scales)) return false;
    QsArgs a{};
    a.p[0] = prob(x, n, k, group, codes, scales, zeros, per_row, y);
    a.count = 1, a.M = static_cast<int>(m), a.y_bf16 = y_bf16;
    launch_any(fmt, a, st);
    return true;
}

// One launch over up to CFH_MAX_BATCH INT8 / INT4 / NF4 / GGUF problems of one format and group (INT4:
// whole multiples of 64) with the same M (2..64), each one that qsplit_takes.
void qsplit_batch(int fmt, int64_t m, int count, const uint16_t *const *x, const int64_t *n, const int64_t *k,
                  const int64_t *group, const void *const *codes, const void *const *scales, const uint32_t *const *zeros,
                  const int *per_row, void *const *y, int y_bf16, hipStream_t st) {
    require(count >= 1 && count <= CFH_MAX_BATCH && m >= 2 && m <= 64, "qsplit_batch: 1..CFH_MAX_BATCH problems, M = 2..64");
    QsArgs a{};
    // longest K first: the workgroups that run longest are not left for the end
    int order[CFH_MAX_BATCH];
    for (int i = 0; i < count; ++i) order[i] = i;
    std::stable_sort(order, order + count, [&](int p, int q) { return k[p] > k[q]; });
    for (int i = 0; i < count; ++i) {
        const int o = order[i];
        a.p[i] = prob(x[o], n[o], k[o], group[o], codes[o], scales[o], zeros[o], per_row[o], y[o]);
    }
    a.count = count, a.M = static_cast<int>(m), a.y_bf16 = y_bf16;
    launch_any(fmt, a, st);
}

}  // namespace cfh
