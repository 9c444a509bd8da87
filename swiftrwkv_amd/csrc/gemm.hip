// Quantised projections of a parallel (prefill) pass on the gfx950 matrix
// cores: sb6 (4, 5 or 6-bit codes) and sym (8 or 6-bit codes).
//
// The reference's long pass dequantises the whole matrix to the fp16 base
// type and runs an fp16 matmul, casting the result back to the input type
// (X070Backbone.baseMatmul, Sources/RWKVGen/X070Backbone.swift:337-356,
// 733-739; the dequant of RwkvqDequant.swift:116-140 (sb6) and :350-388,
// 442-466 (sym, whose fp16 branch computes in half)).  Here the dequant
// happens in the GEMM's operand path (quant_gemm_kernel; gemm_ks_kernel for
// passes of few output tiles), or, for larger ones, once per matrix into a
// workspace that dense_tiles_kernel then multiplies (gemm_route).  Per
// element the numbers are the reference's: the weight is exactly what the
// dequant kernels store in fp16 — sb6 fp16(fma(code, half(qs·d), half(qm·dm))),
// sym fp16((code − bias)·half(qs·d)) — the input is rounded to fp16, products
// accumulate in fp32 on v_mfma_f32_16x16x32_f16, and the sum is rounded to
// fp16 (the fp16 matmul's output) before the epilogue.
//
// quant_gemm_kernel.  A workgroup of 4 waves computes a 128 (input rows) × 128 (output
// features) tile in stages of 64 columns (two 32-column units); two
// workgroups share a CU.  The input tile is staged in LDS as fp16
// (double-buffered; rows padded to 144 B so the 16 lanes of a row group read
// distinct banks).  Wave w owns 32 output features — its own weight rows,
// which no other wave of the workgroup reads — and all 128 input rows: 8 × 2
// tiles of 16 × 16 accumulators.  Each lane dequantises the 8 weights that
// are its MFMA B operand (row 16j + (lane & 15), columns 8·(lane >> 4) .. +7
// of a unit) straight from the packed bytes, so a weight is decoded once per
// workgroup.  The next stage's input and weight bytes are loaded into
// registers before the current stage's products, so one barrier per stage
// separates LDS reuse.
//
// Operand layout of v_mfma_f32_16x16x32_f16 (lane l, g = l >> 4, i = l & 15):
// A[m = i][k = 8g .. 8g+7], B[k = 8g .. 8g+7][n = i]; D[m = 4g + r][n = i],
// r = 0..3.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "launch.h"

namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int BK = 64;            // columns per stage: two sb6 units
constexpr int DKS = 64;           // columns per stage of the dense kernels
constexpr int LDS_ROW = BK + 8;   // halves per staged row (144 B)

__device__ __forceinline__ float f16f(uint32_t bits16) {
    return (float)__builtin_bit_cast(_Float16, (uint16_t)(bits16 & 0xffffu));
}
__device__ __forceinline__ float hround(float x) { return (float)(_Float16)x; }

struct GemmArgs {
    const void* x;        // inputs [groups][M][lda] (fp32 or fp16)
    int64_t lda, x_gstride;
    const uint8_t* q;     // codes: sb6 K3 qblk [N][IN/32·(16+4·xbits)], sym qblk (interleaved)
    const uint8_t* s1;    // sb6 qsqm [N][IN/32·2] / sym qs [N][IN/16]
    const uint16_t* s2;   // sb6 ddm [N][IN/256·2] / sym d [N][IN/256]
    void* y;              // [M][ldy]: fp32 (epilogues 0, 1) or fp16 (epilogue 2)
    int64_t ldy;
    int M, N, K, out_per;
    float* part;          // splits > 1: the fp32 partial sums [splits][M][N]
    int splits;           // K ranges quant_gemm_kernel divides a tile's stages into
};

// The epilogue of one output: fp16 rounding of the fp32 sum (the fp16
// matmul's output), then store (fp32), add into y (fp32) or relu² (fp16).
template <int EP>
__device__ __forceinline__ void store_out(void* y, int64_t idx, float acc) {
    const float v = hround(acc);
    if constexpr (EP == 0) {
        reinterpret_cast<float*>(y)[idx] = v;
    } else if constexpr (EP == 1) {
        float* p = reinterpret_cast<float*>(y) + idx;
        *p = *p + v;
    } else {
        const float rl = fmaxf(v, 0.0f);
        reinterpret_cast<_Float16*>(y)[idx] = (_Float16)(rl * rl);
    }
}

// store_out of four consecutive outputs, 4-element aligned.
template <int EP>
__device__ __forceinline__ void store_out4(void* y, int64_t idx, f32x4 acc) {
#pragma unroll
    for (int c = 0; c < 4; ++c) acc[c] = hround(acc[c]);
    if constexpr (EP == 2) {
        typedef _Float16 half4 __attribute__((ext_vector_type(4)));
        half4 h;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const float rl = fmaxf(acc[c], 0.0f);
            h[c] = (_Float16)(rl * rl);
        }
        *reinterpret_cast<half4*>(reinterpret_cast<_Float16*>(y) + idx) = h;
    } else {
        f32x4* p = reinterpret_cast<f32x4*>(reinterpret_cast<float*>(y) + idx);
        *p = EP == 1 ? *p + acc : acc;
    }
}

// 4 bits → the low bit of 4 bytes (RwkvqSb6GEMV.swift:58-67 multiply spread).
__device__ __forceinline__ uint32_t spread4(uint32_t nib) { return (nib * 0x00204081u) & 0x01010101u; }

// Byte E of w as a float (v_cvt_f32_ubyteE).
template <int E>
__device__ __forceinline__ float ubyte(uint32_t w) {
    return (float)((w >> (8 * E)) & 0xffu);
}

// Eight code bytes (c0: columns 0..3, c1: 4..7 of the lane's 8) as
// fp16(fma(code, s, m)): the product and the sum are exact in fp32 for every
// format here, so the one rounding is the fp16 one.
__device__ __forceinline__ half8 bytes8_fma(uint32_t c0, uint32_t c1, float s, float m) {
    half8 h;
    h[0] = (_Float16)fmaf(ubyte<0>(c0), s, m);
    h[1] = (_Float16)fmaf(ubyte<1>(c0), s, m);
    h[2] = (_Float16)fmaf(ubyte<2>(c0), s, m);
    h[3] = (_Float16)fmaf(ubyte<3>(c0), s, m);
    h[4] = (_Float16)fmaf(ubyte<0>(c1), s, m);
    h[5] = (_Float16)fmaf(ubyte<1>(c1), s, m);
    h[6] = (_Float16)fmaf(ubyte<2>(c1), s, m);
    h[7] = (_Float16)fmaf(ubyte<3>(c1), s, m);
    return h;
}

// Weight formats.  A lane (row `row`, column group gq of 8) loads the bytes
// of its 8 columns of the stage's two units u, u + 1 (Raw) and decodes unit
// q ∈ {0, 1} into its B operand.
//
// sb6 (gs 32, super-block 8 units): unit = 16 B of nibbles (byte c: column c
// low, c + 16 high) ‖ 4 B qh ‖ 4 B qh2 (bit c: bit 4 / 5 of column c) for
// 4 + XB bit codes; qsqm (qs, qm − 31) per unit; ddm (d, dm) fp16 per
// super-block (the K3 layout, RwkvqFile.swift:189-212).
template <int XB>
struct Sb6W {
    static constexpr int UB = 16 + 4 * XB;
    static constexpr int SPS = 2;   // s2 halves per super-block
    struct Codes {
        uint2 nib[2];
        uint32_t hi[2][XB > 0 ? XB : 1];
    };
    struct Raw {
        Codes c;
        uint32_t sm;   // qsqm of units u, u + 1
        uint32_t dd;   // ddm of their super-block
    };
    // a row's codes of units u, u + 1, at unit u's bytes
    __device__ static Codes load_codes(const uint8_t* pq, int gq) {
        Codes r;
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const uint8_t* b = pq + q * UB;
            // 4-byte aligned only for a 20-byte unit: two dword loads
            const uint32_t* w = reinterpret_cast<const uint32_t*>(b + 8 * (gq & 1));
            r.nib[q] = make_uint2(w[0], w[1]);
#pragma unroll
            for (int e = 0; e < XB; ++e) r.hi[q][e] = *reinterpret_cast<const uint32_t*>(b + 16 + 4 * e);
        }
        return r;
    }
    __device__ static Raw load(const GemmArgs& g, int64_t row, int u, int gq) {
        const int NU = g.K >> 5, NSB = g.K >> 8;
        Raw r;
        r.c = load_codes(g.q + (row * NU + u) * UB, gq);
        r.sm = *reinterpret_cast<const uint32_t*>(g.s1 + (row * NU + u) * 2);
        r.dd = *reinterpret_cast<const uint32_t*>(g.s2 + (row * NSB + (u >> 3)) * 2);
        return r;
    }
    // a unit's scale word for decode(): (half(qs·d), half(qm·dm)) from its qsqm and its super-block's ddm
    __device__ static uint32_t scale(uint32_t sm, uint32_t dd) {
        const _Float16 s = (_Float16)((float)(sm & 0xffu) * f16f(dd));
        const _Float16 m = (_Float16)((float)(int8_t)((sm >> 8) & 0xffu) * f16f(dd >> 16));
        return (uint32_t)__builtin_bit_cast(uint16_t, s) | ((uint32_t)__builtin_bit_cast(uint16_t, m) << 16);
    }
    __device__ static uint32_t load_scale(const GemmArgs& g, int64_t row, int u) {
        const int NU = g.K >> 5, NSB = g.K >> 8;
        return scale(*reinterpret_cast<const uint16_t*>(g.s1 + (row * NU + u) * 2),
                     *reinterpret_cast<const uint32_t*>(g.s2 + (row * NSB + (u >> 3)) * 2));
    }
    __device__ static half8 decode(const Codes& r, int q, int gq, float s, float m) {
        const int shift = (gq >> 1) * 4;   // columns 16..31 in the high nibbles
        const uint32_t c0 = (r.nib[q].x >> shift) & 0x0F0F0F0Fu, c1 = (r.nib[q].y >> shift) & 0x0F0F0F0Fu;
        if constexpr (XB == 0) {
            // a 4-bit code byte read as fp8 E4M3 is code·2^-9 exactly: two
            // codes widen per instruction and s carries the 2^9
            s *= 512.0f;
            const auto p0 = __builtin_amdgcn_cvt_pk_f32_fp8((int)c0, false);
            const auto p1 = __builtin_amdgcn_cvt_pk_f32_fp8((int)c0, true);
            const auto p2 = __builtin_amdgcn_cvt_pk_f32_fp8((int)c1, false);
            const auto p3 = __builtin_amdgcn_cvt_pk_f32_fp8((int)c1, true);
            half8 h;
            h[0] = (_Float16)fmaf(p0[0], s, m);
            h[1] = (_Float16)fmaf(p0[1], s, m);
            h[2] = (_Float16)fmaf(p1[0], s, m);
            h[3] = (_Float16)fmaf(p1[1], s, m);
            h[4] = (_Float16)fmaf(p2[0], s, m);
            h[5] = (_Float16)fmaf(p2[1], s, m);
            h[6] = (_Float16)fmaf(p3[0], s, m);
            h[7] = (_Float16)fmaf(p3[1], s, m);
            return h;
        } else {
            uint32_t a = c0, b = c1;
#pragma unroll
            for (int e = 0; e < XB; ++e) {
                const uint32_t h8 = (r.hi[q][e] >> (8 * gq)) & 0xffu;   // bits of columns 8gq .. 8gq+7
                a |= spread4(h8 & 0xFu) << (4 + e);
                b |= spread4(h8 >> 4) << (4 + e);
            }
            return bytes8_fma(a, b, s, m);
        }
    }
    // decode with a scale word of scale()
    __device__ static half8 decode_scaled(const Codes& r, int q, int gq, uint32_t sw) {
        return decode(r, q, gq, f16f(sw), f16f(sw >> 16));
    }
    __device__ static half8 dequant(const Raw& r, int q, int gq) {
        return decode_scaled(r.c, q, gq, scale(r.sm >> (16 * q), r.dd));
    }
};

// sym (gs = super-block = 16 columns, RwkvqFile.swift:437-449 interleave):
// 8-bit: 32 int8 codes per unit (byte c = column c); 6-bit: 24 B per unit —
// words 0..3 nibbles (register order l0, l1, h0, h1 | l2, l3, h2, h3: word
// 2·(c / 16) + (c / 4) % 2, low nibbles for c % 8 < 4), word 4 qh, word 5 qh2,
// codes stored + 32.  qs int8 per 16 columns, d fp16 per 256 columns;
// w = (code − bias)·half(qs·d).
template <int BITS>
struct SymW {
    static constexpr int UB = BITS == 8 ? 32 : 24;
    static constexpr int SPS = 1;
    struct Codes {
        uint2 c[2];
        uint32_t hi[2][BITS == 8 ? 1 : 2];
    };
    struct Raw {
        Codes c;
        uint32_t qs;   // the four 16-column scales of units u, u + 1
        uint32_t d;    // super-block scale (fp16)
    };
    __device__ static Codes load_codes(const uint8_t* pq, int gq) {
        Codes r;
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const uint8_t* b = pq + q * UB;
            if constexpr (BITS == 8) {
                r.c[q] = *reinterpret_cast<const uint2*>(b + 8 * gq);
            } else {
                r.c[q] = *reinterpret_cast<const uint2*>(b + 8 * (gq >> 1));
                r.hi[q][0] = *reinterpret_cast<const uint32_t*>(b + 16);
                r.hi[q][1] = *reinterpret_cast<const uint32_t*>(b + 20);
            }
        }
        return r;
    }
    __device__ static Raw load(const GemmArgs& g, int64_t row, int u, int gq) {
        const int NU = g.K >> 5, NSB = g.K >> 8;
        Raw r;
        r.c = load_codes(g.q + (row * NU + u) * UB, gq);
        r.qs = *reinterpret_cast<const uint32_t*>(g.s1 + (row * NU + u) * 2);
        r.d = g.s2[row * NSB + (u >> 3)];
        return r;
    }
    // a unit's scale word: half(qs·d) of its columns 0..15 and 16..31
    __device__ static uint32_t scale(uint32_t qs, uint32_t d) {
        const _Float16 a = (_Float16)((float)(int8_t)(qs & 0xffu) * f16f(d));
        const _Float16 b = (_Float16)((float)(int8_t)((qs >> 8) & 0xffu) * f16f(d));
        return (uint32_t)__builtin_bit_cast(uint16_t, a) | ((uint32_t)__builtin_bit_cast(uint16_t, b) << 16);
    }
    __device__ static uint32_t load_scale(const GemmArgs& g, int64_t row, int u) {
        const int NU = g.K >> 5, NSB = g.K >> 8;
        return scale(*reinterpret_cast<const uint16_t*>(g.s1 + (row * NU + u) * 2), g.s2[row * NSB + (u >> 3)]);
    }
    __device__ static half8 decode(const Codes& r, int q, int gq, float s) {
        if constexpr (BITS == 8) {
            // int8 codes as unsigned bytes code + 128: (u − 128)·s exactly
            return bytes8_fma(r.c[q].x ^ 0x80808080u, r.c[q].y ^ 0x80808080u, s, -128.0f * s);
        } else {
            const int shift = (gq & 1) * 4;
            uint32_t a = (r.c[q].x >> shift) & 0x0F0F0F0Fu, b = (r.c[q].y >> shift) & 0x0F0F0F0Fu;
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const uint32_t h8 = (r.hi[q][e] >> (8 * gq)) & 0xffu;
                a |= spread4(h8 & 0xFu) << (4 + e);
                b |= spread4(h8 >> 4) << (4 + e);
            }
            return bytes8_fma(a, b, s, -32.0f * s);
        }
    }
    __device__ static half8 decode_scaled(const Codes& r, int q, int gq, uint32_t sw) {
        return decode(r, q, gq, f16f(sw >> (16 * (gq >> 1))));
    }
    __device__ static half8 dequant(const Raw& r, int q, int gq) {
        return decode(r.c, q, gq, hround((float)(int8_t)((r.qs >> (8 * (2 * q + (gq >> 1)))) & 0xffu) * f16f(r.d)));
    }
};

// MT × 16 input rows × (4 waves × NT × 16) output features per workgroup.
// A stage's inputs: thread t stages row t / TPR, EPT consecutive columns.
template <class F, typename TA, int EP, int MT, int NT>
__global__ __launch_bounds__(256, 2) void quant_gemm_kernel(GemmArgs g) {
    constexpr int BM = 16 * MT, BN = 64 * NT;
    constexpr int TPR = 256 / BM;        // staging threads per row
    constexpr int EPT = BK / TPR;        // columns per staging thread
    constexpr int AV = EPT * sizeof(TA) / 16;   // 16-byte loads per staging thread
    __shared__ __attribute__((aligned(16))) _Float16 As[2][BM][LDS_ROW];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int gq = lane >> 4, li = lane & 15;
    // Workgroups are dealt to the 8 XCDs round-robin (id mod 8), each XCD with
    // its own L2: XCD x takes a contiguous run of the (row block, feature
    // block, K range) order, so an input block is read into one L2, or two.
    const int ntn = g.N / BN, S = g.splits;
    const int total = ((g.M + BM - 1) / BM) * ntn * S;
    const int xcd = blockIdx.x & 7, loc = blockIdx.x >> 3;
    const int t = xcd * (total >> 3) + min(xcd, total & 7) + loc;   // the tile's place in that order
    const int kz = t % S, tile_n = (t / S) % ntn, tile_m = t / (S * ntn);
    const int n0 = tile_n * BN;
    const int m0 = tile_m * BM;
    const int nst = g.K / BK;
    const int st0 = (int)((int64_t)kz * nst / S), st1 = (int)((int64_t)(kz + 1) * nst / S);

    // input rows of this tile come from the matrix group its output features belong to
    const TA* xg = reinterpret_cast<const TA*>(g.x) + (int64_t)(n0 / g.out_per) * g.x_gstride;
    const int srow = threadIdx.x / TPR, scol = (threadIdx.x % TPR) * EPT;
    const TA* xrow = xg + (int64_t)min(m0 + srow, g.M - 1) * g.lda + scol;

    const int nb = n0 + wave * (16 * NT) + li;   // weight row of tile j: nb + 16 j

    auto load_a = [&](int st) {
        uint4 a[AV];
        const uint4* p = reinterpret_cast<const uint4*>(xrow + st * BK);
#pragma unroll
        for (int e = 0; e < AV; ++e) a[e] = p[e];
        struct R { uint4 v[AV]; } r;
#pragma unroll
        for (int e = 0; e < AV; ++e) r.v[e] = a[e];
        return r;
    };
    auto store_a = [&](int buf, const auto& a) {
        _Float16* d = &As[buf][srow][scol];
        if constexpr (sizeof(TA) == 4) {
#pragma unroll
            for (int e = 0; e < AV / 2; ++e) {
                const uint4 p = a.v[2 * e], q = a.v[2 * e + 1];
                half8 h;
                h[0] = (_Float16)__uint_as_float(p.x); h[1] = (_Float16)__uint_as_float(p.y);
                h[2] = (_Float16)__uint_as_float(p.z); h[3] = (_Float16)__uint_as_float(p.w);
                h[4] = (_Float16)__uint_as_float(q.x); h[5] = (_Float16)__uint_as_float(q.y);
                h[6] = (_Float16)__uint_as_float(q.z); h[7] = (_Float16)__uint_as_float(q.w);
                *reinterpret_cast<half8*>(d + 8 * e) = h;
            }
        } else {
#pragma unroll
            for (int e = 0; e < AV; ++e) *reinterpret_cast<uint4*>(d + 8 * e) = a.v[e];
        }
    };
    using Raw = typename F::Raw;
    struct BRaw {
        Raw t[NT];
    };
    auto load_b = [&](int st) {
        BRaw b;
#pragma unroll
        for (int j = 0; j < NT; ++j) b.t[j] = F::load(g, nb + 16 * j, st * 2, gq);
        return b;
    };
    auto dequant = [&](const BRaw& b, int q, half8* bop) {
#pragma unroll
        for (int j = 0; j < NT; ++j) bop[j] = F::dequant(b.t[j], q, gq);
    };
    // MT × NT MFMAs of unit q of the staged buffer
    f32x4 acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto products = [&](int buf, int q, const half8* bop) {
#pragma unroll
        for (int i = 0; i < MT; ++i) {
            const half8 aop = *reinterpret_cast<const half8*>(&As[buf][16 * i + li][32 * q + 8 * gq]);
#pragma unroll
            for (int j = 0; j < NT; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(aop, bop[j], acc[i][j], 0, 0, 0);
        }
    };

    auto ar = load_a(st0);
    BRaw bcur = load_b(st0);
    store_a(0, ar);
    half8 b0[NT], b1[NT];
    dequant(bcur, 0, b0);
    __syncthreads();

    // Per stage: the next stage's bytes are requested first; unit 0's
    // products run while unit 1 is decoded, unit 1's while the next stage's
    // unit 0 is (one MFMA, one VALU instruction, alternately).
    for (int st = st0; st < st1; ++st) {
        const int buf = (st - st0) & 1;
        const bool more = st + 1 < st1;
        BRaw bnxt = bcur;
        if (more) {
            ar = load_a(st + 1);
            bnxt = load_b(st + 1);
        }
        dequant(bcur, 1, b1);
        products(buf, 0, b0);
#pragma unroll
        for (int k = 0; k < MT * NT; ++k) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);   // one MFMA
            __builtin_amdgcn_sched_group_barrier(0x002, 1, 0);   // one VALU
        }
        if (more) dequant(bnxt, 0, b0);
        products(buf, 1, b1);
#pragma unroll
        for (int k = 0; k < MT * NT; ++k) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, 1, 0);
        }
        if (more) store_a(buf ^ 1, ar);
        bcur = bnxt;
        __syncthreads();
    }

    if (S > 1) {   // this K range's fp32 sums; gemm_split_reduce adds the ranges and applies the epilogue
        float* part = g.part + (int64_t)kz * g.M * g.N;
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = m0 + 16 * i + 4 * gq + r;
                if (row >= g.M) continue;
#pragma unroll
                for (int j = 0; j < NT; ++j) part[(int64_t)row * g.N + nb + 16 * j] = acc[i][j][r];
            }
        return;
    }
#pragma unroll
    for (int i = 0; i < MT; ++i) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = m0 + 16 * i + 4 * gq + r;
            if (row >= g.M) continue;
#pragma unroll
            for (int j = 0; j < NT; ++j) store_out<EP>(g.y, (int64_t)row * g.ldy + nb + 16 * j, acc[i][j][r]);
        }
    }
}

// The K ranges of a split launch summed in range order (a fixed order: the
// result does not depend on which workgroup finished first), then the
// epilogue of the one-range kernel: fp16 rounding, store / add / relu².
// Thread i takes 4 consecutive outputs of one row (N is a multiple of 128).
template <int EP>
__global__ __launch_bounds__(256) void gemm_split_reduce(const float* __restrict__ part, int S, int M, int N,
                                                         void* y, int64_t ldy) {
    const int64_t n4 = (int64_t)M * N / 4;
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n4) return;
    const float4* p = reinterpret_cast<const float4*>(part) + i;
    float4 a = p[0];
    for (int k = 1; k < S; ++k) {
        const float4 b = p[(int64_t)k * n4];
        a.x += b.x; a.y += b.y; a.z += b.z; a.w += b.w;
    }
    const int64_t row = 4 * i / N, col = 4 * i % N;
    const float v[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
    for (int c = 0; c < 4; ++c) store_out<EP>(y, row * ldy + col + c, v[c]);
}

// ── few output tiles: the K sum split over the waves of a workgroup ──
//
// A pass of a few hundred rows has few output tiles, and a tile whose K stages
// run one after another waits on memory once per stage.  Here a workgroup is
// one tile of 16·MT × 16·NT outputs and its W waves take K / W columns each.
// A wave works alone: it moves 128 columns at a time (its input rows and its
// weight rows' packed bytes) through its own LDS region, so no barrier stands
// in the K loop (a wave's LDS operations run in order, so what it stages is
// there for its own reads), with the next 128 columns' loads in registers meanwhile; the
// W partial tiles meet in LDS at the end, summed in wave order
// (deterministic), where the epilogue is applied.  One launch.
//
// Why through LDS: an MFMA operand wants lane l to hold row l & 15, and a load
// in that shape has every lane in another cache line (measured ~50 cycles per
// load instruction and CU, against 16 for one whose lanes run along a row:
// 128 rows × 768 × 3072 took 11.8 µs that way, 7.0 like this, on 32 × 16 tiles).
// Past a tile's start its time is its bytes through the CU's one memory path
// (18 KB per 64 × 32 × 128 step) beside as long a stretch of decoding.
// The scale words of the wave's rows go through its region too, four steps at
// a time (read per step they would cost as many cache lines as the codes).
constexpr int KS_COLS = 2 * BK;            // columns per step: four units
constexpr int KS_PAD = 4;                  // partial tiles: row padding (floats)
constexpr size_t KS_LDS = 160 * 1024;      // a gfx950 workgroup's LDS
constexpr int KS_AROW = KS_COLS * 2 + 16;  // LDS bytes per staged input row: an odd number of 16-byte chunks
// steps per block of scale words, and LDS bytes per weight row of them (an odd number of chunks)
constexpr int ks_ssteps(int nt) { return nt == 4 ? 2 : 4; }
constexpr int ks_srow(int nt) { return ks_ssteps(nt) * 16 + 16; }

struct KsArgs {
    GemmArgs g;
    int ep;    // epilogue (store_out)
    int vec;   // y rows take aligned 4-wide stores
};

// LDS bytes per staged weight row: the four units' bytes in an odd number of
// 16-byte chunks, so 16 rows' reads at one column fall on distinct banks.
constexpr int ks_brow(int unit_bytes) { return 16 * ((4 * unit_bytes / 16) | 1); }
constexpr int ks_wave_lds(int unit_bytes, int mt, int nt) {
    return 16 * mt * KS_AROW + 16 * nt * (ks_brow(unit_bytes) + ks_srow(nt));
}

template <class F, typename TA, int MT, int NT, int MAXW>
__global__ __launch_bounds__(64 * MAXW) void gemm_ks_kernel(KsArgs ka) {
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];   // W wave regions, then the partial tiles
    const GemmArgs& g = ka.g;
    constexpr int BM = 16 * MT, BN = 16 * NT, LS = BN + KS_PAD, SS = ks_ssteps(NT), SR = ks_srow(NT);
    constexpr int AC = KS_COLS * (int)sizeof(TA) / 16;   // 16-byte chunks per input row and step
    constexpr int AL = BM * AC / 64;                     // input loads per lane
    constexpr int BC = 4 * F::UB / 16;                   // chunks per weight row and step
    constexpr int BL = (BN * BC + 63) / 64;              // weight loads per lane
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int W = blockDim.x >> 6;
    const int gq = lane >> 4, li = lane & 15;
    // an XCD takes a contiguous run of tiles, row blocks fastest: the row
    // blocks of a weight panel share one L2
    const int tm = (g.M + BM - 1) / BM, total = tm * (g.N / BN);
    const int xcd = blockIdx.x & 7, loc = blockIdx.x >> 3;
    const int t = xcd * (total >> 3) + min(xcd, total & 7) + loc;
    const int m0 = (t % tm) * BM, n0 = (t / tm) * BN;
    const int steps = g.K / KS_COLS, NU = g.K >> 5;
    const int p0 = wave * steps / W, p1 = (wave + 1) * steps / W;   // W <= steps: at least one step each

    unsigned char* const mine = lds + wave * ks_wave_lds(F::UB, MT, NT);
    unsigned char* const mb = mine + BM * KS_AROW;
    unsigned char* const ms = mb + BN * ks_brow(F::UB);

    // Uniform bases (tile, step) plus a 32-bit offset per load.
    const char* xt = reinterpret_cast<const char*>(reinterpret_cast<const TA*>(g.x) +
                                                   (int64_t)(n0 / g.out_per) * g.x_gstride + (int64_t)m0 * g.lda);
    const uint8_t* qt = g.q + (int64_t)n0 * NU * F::UB;
    uint32_t xo[AL], bo[BL];
#pragma unroll
    for (int e = 0; e < AL; ++e) {
        const int id = lane + 64 * e, row = id / AC, c = id % AC;
        xo[e] = (uint32_t)(min(row, g.M - 1 - m0) * (int)g.lda * (int)sizeof(TA) + 16 * c);
    }
#pragma unroll
    for (int e = 0; e < BL; ++e) {
        const int id = min(lane + 64 * e, BN * BC - 1), row = id / BC, c = id % BC;
        bo[e] = (uint32_t)(row * NU * F::UB + 16 * c);
    }
    u32x4 ra[AL], rb[BL];
    auto load = [&](int p) __attribute__((always_inline)) {
        const char* xs = xt + (int64_t)p * (KS_COLS * (int)sizeof(TA));
        const uint8_t* qs = qt + (int64_t)p * (4 * F::UB);
#pragma unroll
        for (int e = 0; e < BL; ++e) rb[e] = *reinterpret_cast<const u32x4*>(qs + bo[e]);
#pragma unroll
        for (int e = 0; e < AL; ++e) ra[e] = *reinterpret_cast<const u32x4*>(xs + xo[e]);
    };
    auto stage = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < BL; ++e) {
            const int id = min(lane + 64 * e, BN * BC - 1);
            *reinterpret_cast<u32x4*>(mb + id / BC * ks_brow(F::UB) + id % BC * 16) = rb[e];
        }
#pragma unroll
        for (int e = 0; e < AL; ++e) {
            const int id = lane + 64 * e, row = id / AC, c = id % AC;
            unsigned char* const r = mine + row * KS_AROW;
            if constexpr (sizeof(TA) == 2) {
                *reinterpret_cast<u32x4*>(r + 16 * c) = ra[e];
            } else {
                typedef _Float16 half4 __attribute__((ext_vector_type(4)));
                half4 h;
                h[0] = (_Float16)__uint_as_float(ra[e].x); h[1] = (_Float16)__uint_as_float(ra[e].y);
                h[2] = (_Float16)__uint_as_float(ra[e].z); h[3] = (_Float16)__uint_as_float(ra[e].w);
                *reinterpret_cast<half4*>(r + 8 * c) = h;
            }
        }
    };
    // Scale words of steps p .. p + 3 of the wave's rows: lane → (row, step),
    // its four units' bytes and their super-block's fp16 scales.
    constexpr int SL = BN * SS / 64;
    const int NSB = g.K >> 8;
    uint2 rs[SL];
    uint32_t rd[SL];
    auto load_scales = [&](int p) __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < SL; ++e) {
            const int id = lane + 64 * e, row = n0 + id / SS, st = min(p + id % SS, steps - 1);
            rs[e] = *reinterpret_cast<const uint2*>(g.s1 + ((int64_t)row * NU + 4 * st) * 2);
            const uint16_t* d = g.s2 + ((int64_t)row * NSB + (st >> 1)) * F::SPS;
            if constexpr (F::SPS == 2) rd[e] = *reinterpret_cast<const uint32_t*>(d);
            else rd[e] = *d;
        }
    };
    auto stage_scales = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < SL; ++e) {
            const int id = lane + 64 * e;
            u32x4 w;
            w[0] = F::scale(rs[e].x, rd[e]);
            w[1] = F::scale(rs[e].x >> 16, rd[e]);
            w[2] = F::scale(rs[e].y, rd[e]);
            w[3] = F::scale(rs[e].y >> 16, rd[e]);
            *reinterpret_cast<u32x4*>(ms + id / SS * SR + id % SS * 16) = w;
        }
    };
    f32x4 acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto products = [&](int p) __attribute__((always_inline)) {
        u32x4 sw[NT];
#pragma unroll
        for (int j = 0; j < NT; ++j)
            sw[j] = *reinterpret_cast<const u32x4*>(ms + (16 * j + li) * SR + (p - p0) % SS * 16);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            typename F::Codes cd[NT];
#pragma unroll
            for (int j = 0; j < NT; ++j) cd[j] = F::load_codes(mb + (16 * j + li) * ks_brow(F::UB) + 2 * h * F::UB, gq);
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                half8 b[NT];
#pragma unroll
                for (int j = 0; j < NT; ++j) {
                    const uint32_t s = h == 0 ? (q == 0 ? sw[j].x : sw[j].y) : (q == 0 ? sw[j].z : sw[j].w);
                    b[j] = F::decode_scaled(cd[j], q, gq, s);
                }
#pragma unroll
                for (int i = 0; i < MT; ++i) {
                    const half8 a = *reinterpret_cast<const half8*>(mine + (16 * i + li) * KS_AROW +
                                                                    (4 * (2 * h + q) + gq) * 16);
#pragma unroll
                    for (int j = 0; j < NT; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b[j], acc[i][j], 0, 0, 0);
                }
            }
        }
    };
    load_scales(p0);
    load(p0);
    auto next_scales = [&](int p) __attribute__((always_inline)) {
        if ((p - p0) % SS != 0) return;
        stage_scales();
        load_scales(p + SS);
    };
    // the last step is peeled, so no input or code load is repeated
    for (int p = p0; p < p1 - 1; ++p) {
        next_scales(p);
        stage();
        load(p + 1);
        products(p);
    }
    next_scales(p1 - 1);
    stage();
    products(p1 - 1);
    __syncthreads();   // the staging LDS becomes the partial tiles

    float* const part = reinterpret_cast<float*>(lds);   // [W][BM][LS]
    float* const own = part + wave * (BM * LS);
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) own[(16 * i + 4 * gq + r) * LS + 16 * j + li] = acc[i][j][r];
    __syncthreads();
    for (int q = threadIdx.x; q < BM * BN / 4; q += blockDim.x) {
        const int row = q / (BN / 4), col = q % (BN / 4) * 4;
        const float* src = part + row * LS + col;
        f32x4 v = *reinterpret_cast<const f32x4*>(src);
        for (int k = 1; k < W; ++k) v += *reinterpret_cast<const f32x4*>(src + k * (BM * LS));
        if (m0 + row >= g.M) continue;
        const int64_t at = (int64_t)(m0 + row) * g.ldy + n0 + col;
        if (!ka.vec) {
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                if (ka.ep == 0) store_out<0>(g.y, at + c, v[c]);
                else if (ka.ep == 1) store_out<1>(g.y, at + c, v[c]);
                else store_out<2>(g.y, at + c, v[c]);
            }
            continue;
        }
        if (ka.ep == 0) store_out4<0>(g.y, at, v);
        else if (ka.ep == 1) store_out4<1>(g.y, at, v);
        else store_out4<2>(g.y, at, v);
    }
}

// ── dequantised weights in operand order ──
//
// For a quantised matrix the workspace copy need not be row-major: it is
// written in the order the matrix cores read it, so the GEMM loads its weight
// operands straight into registers and only the inputs go through LDS.  Block
// (n16, u) of 16 rows × one 32-column unit is 1 KiB at index n16·(K/32) + u;
// lane gq·16 + li's 16 bytes are row 16·n16 + li, columns 32u + 8gq .. + 7.
// (The row-major kernel below is bound by LDS: per 64-column stage its eight
// waves read 192 KB and write 64 KB, ~2,560 cycles at 128 and 64 B per cycle
// against 2,048 of MFMA.)
template <class F>
__global__ __launch_bounds__(256) void dequant_tiles_kernel(GemmArgs g, _Float16* __restrict__ out) {
    const int NU = g.K >> 5, NSB = g.K >> 8;
    const int lane = threadIdx.x & 63, gq = lane >> 4, li = lane & 15;
    // one wave: 16 rows × half a super-block (four units)
    const int wv = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (wv >= (g.N >> 4) * 2 * NSB) return;
    const int n16 = wv / (2 * NSB), hb = wv - n16 * 2 * NSB, u0 = 4 * hb;
    const int64_t row = 16 * n16 + li;
    const uint2 sm = *reinterpret_cast<const uint2*>(g.s1 + (row * NU + u0) * 2);
    uint32_t dd;
    if constexpr (F::SPS == 2) dd = *reinterpret_cast<const uint32_t*>(g.s2 + (row * NSB + (hb >> 1)) * 2);
    else dd = g.s2[row * NSB + (hb >> 1)];
    const uint8_t* pq = g.q + (row * NU + u0) * F::UB;
    const typename F::Codes c[2] = {F::load_codes(pq, gq), F::load_codes(pq + 2 * F::UB, gq)};
    half8* o = reinterpret_cast<half8*>(out) + ((int64_t)n16 * NU + u0) * 64 + lane;
#pragma unroll
    for (int u = 0; u < 4; ++u)
        o[64 * u] = F::decode_scaled(c[u >> 1], u & 1, gq, F::scale((u < 2 ? sm.x : sm.y) >> (16 * (u & 1)), dd));
}

// The dense product over a weight in operand order.  Tile 16·WM·AM input rows
// × 16·WN·AN features, WM × WN waves, 64-column stages (two units).  Inputs:
// global → registers a stage ahead → LDS (rows of 128 B, chunk c of row r at
// c ^ (r & 7)), two buffers.  Weights: two stages of operands in registers,
// a unit's set reloaded as soon as its products are issued.  The weight is the
// MFMA's A operand and the input its B operand, so lane gq·16 + li ends with
// input row li, features 4gq .. 4gq + 3: four consecutive outputs to store.
// Per output the products and their order are quant_gemm_kernel's.
struct DenseTArgs {
    const void* x;       // [groups][M][lda], fp16 or fp32
    int64_t lda, x_gstride;
    const _Float16* w;   // operand order
    void* y;             // [M][ldy]
    int64_t ldy;
    int M, N, K, out_per;
    int vec;             // y rows take aligned 4-wide accesses
};

template <typename TA, int EP, int WM, int WN, int AM, int AN, int DP, int DA>
__global__ __launch_bounds__(64 * WM * WN, WM * WN > 4 ? 1 : 2) void dense_tiles_kernel(DenseTArgs g) {
    constexpr int XV = (int)sizeof(TA) / 2;   // 16-byte loads per chunk of 8 inputs
    constexpr int TM = 16 * WM * AM, TN = 16 * WN * AN;
    constexpr int RP = 8 * WM * WN;   // rows one pass of the workgroup's input loads covers
    constexpr int PX = TM / RP;       // input chunks per thread and stage
    __shared__ u32x4 lds[2][TM * 8];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int gq = lane >> 4, li = lane & 15;
    // Tiles in groups of 4 row blocks × every feature block, feature-major
    // within a group; XCD x (workgroups x, x + 8, ...) takes a contiguous run
    // of that order.
    const int ntm = (g.M + TM - 1) / TM, ntn = g.N / TN, total = ntm * ntn;
    const int xcd = blockIdx.x & 7, loc = blockIdx.x >> 3;
    const int t = xcd * (total >> 3) + min(xcd, total & 7) + loc;
    const int grp = t / (4 * ntn), first = 4 * grp, gm = min(4, ntm - first);
    const int rr = t - grp * 4 * ntn;
    const int m0 = (first + rr % gm) * TM, n0 = (rr / gm) * TN;
    const int NU = g.K >> 5, nst = g.K / DKS;

    const int c = tid & 7, r0 = tid >> 3;
    const int mrows = min(TM, g.M - m0);
    const TA* xt = reinterpret_cast<const TA*>(g.x) + (int64_t)(n0 / g.out_per) * g.x_gstride + (int64_t)m0 * g.lda;
    const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<TA*>(xt), 0, (int)(mrows * g.lda * (int)sizeof(TA)), 0x00020000);
    const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<_Float16*>(g.w + (int64_t)n0 * g.K), 0, (int)((int64_t)TN * g.K * 2), 0x00020000);
    uint32_t xo[PX];
#pragma unroll
    for (int p = 0; p < PX; ++p) xo[p] = (uint32_t)((min(r0 + RP * p, mrows - 1) * (int)g.lda + 8 * c) * (int)sizeof(TA));
    const int dst0 = r0 * 8 + (c ^ (r0 & 7));   // row r0 + RP·p: + 8·RP·p chunks, the same swizzle
    const int wm = wave % WM, wn = wave / WM;
    u32x4 v[DA][PX * XV];
    auto gload = [&](u32x4 (&d)[PX * XV], int st) __attribute__((always_inline)) {
        const uint32_t so = (uint32_t)(min(st, nst - 1) * DKS * (int)sizeof(TA));
#pragma unroll
        for (int p = 0; p < PX; ++p)
#pragma unroll
            for (int e = 0; e < XV; ++e)
                d[p * XV + e] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rx, xo[p] + 16 * e, so, 0));
    };
    auto swrite = [&](int buf, const u32x4 (&d)[PX * XV]) __attribute__((always_inline)) {
#pragma unroll
        for (int p = 0; p < PX; ++p) {
            if constexpr (XV == 1) {
                lds[buf][dst0 + 8 * RP * p] = d[p];
            } else {
                half8 h;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    h[e] = (_Float16)__uint_as_float(d[2 * p][e]);
                    h[4 + e] = (_Float16)__uint_as_float(d[2 * p + 1][e]);
                }
                lds[buf][dst0 + 8 * RP * p] = __builtin_bit_cast(u32x4, h);
            }
        }
    };
    half8 bq[DP][2][AN];   // [stage mod DP][unit][feature tile]
    const uint32_t wlane = (uint32_t)(lane * 16);
    auto wload = [&](half8 (&b)[AN], int st, int kk) __attribute__((always_inline)) {
        const int u = 2 * min(st, nst - 1) + kk;
#pragma unroll
        for (int j = 0; j < AN; ++j)
            b[j] = __builtin_bit_cast(half8, __builtin_amdgcn_raw_buffer_load_b128(
                                                 rw, wlane, (uint32_t)(((wn * AN + j) * NU + u) * 1024), 0));
    };
    f32x4 acc[AM][AN];
#pragma unroll
    for (int a = 0; a < AM; ++a)
#pragma unroll
        for (int b = 0; b < AN; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int ra = (16 * AM * wm + li) * 8;
    auto operands = [&](int buf, int kk, half8 (&av)[AM]) __attribute__((always_inline)) {
        const int ch = (4 * kk + gq) ^ (li & 7);
#pragma unroll
        for (int a = 0; a < AM; ++a) av[a] = __builtin_bit_cast(half8, lds[buf][ra + 128 * a + ch]);
    };
    auto products = [&](const half8 (&av)[AM], const half8 (&bv)[AN]) __attribute__((always_inline)) {
#pragma unroll
        for (int a = 0; a < AM; ++a)
#pragma unroll
            for (int b = 0; b < AN; ++b)
                acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(bv[b], av[a], acc[a][b], 0, 0, 0);
    };
    // Stage st, at place q of the unrolled DP (LDS buffer q & 1).  Unit 0's
    // products carry the reload of the unit-1 operands the previous stage
    // consumed, unit 1's the reload of unit 0's, the LDS write of the next
    // stage's inputs and the loads that refill their registers.
    auto stage = [&](int q, int st) __attribute__((always_inline)) {
        {
            half8 av[AM];
            operands(q & 1, 0, av);
            wload(bq[(q + DP - 1) % DP][1], st + DP - 1, 1);
            products(av, bq[q][0]);
            __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);   // DS reads
#pragma unroll
            for (int i = 0; i < AM; ++i) {
                __builtin_amdgcn_sched_group_barrier(0x008, AN, 0);   // MFMA
                if (i < AM - 2) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x020, (AN + AM - 1) / AM, 0);   // VMEM read
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        {
            half8 av[AM];
            operands(q & 1, 1, av);
            wload(bq[q][0], st + DP, 0);
            products(av, bq[q][1]);
            swrite((q & 1) ^ 1, v[(q + 1) % DA]);
            gload(v[(q + 1) % DA], st + 1 + DA);
            __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
#pragma unroll
            for (int i = 0; i < AM; ++i) {
                __builtin_amdgcn_sched_group_barrier(0x008, AN, 0);
                if (i < AM - 2) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x200, (PX + AM - 1) / AM, 0);        // DS write
                __builtin_amdgcn_sched_group_barrier(0x020, (AN + PX * XV + AM - 1) / AM, 0);   // VMEM read
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        __syncthreads();
    };

    // nst is a multiple of DP; loads past the last stage repeat it, and the
    // final LDS write lands in a buffer no later stage reads
    gload(v[0], 0);
#pragma unroll
    for (int d = 0; d < DP; ++d) {
        wload(bq[d][0], d, 0);
        if (d < DP - 1) wload(bq[d][1], d, 1);
    }
    swrite(0, v[0]);
#pragma unroll
    for (int d = 1; d <= DA; ++d) gload(v[d % DA], d);
    __syncthreads();
    for (int st = 0; st < nst; st += DP) {
#pragma unroll
        for (int q = 0; q < DP; ++q) stage(q, st + q);
    }

#pragma unroll
    for (int a = 0; a < AM; ++a) {
        const int row = m0 + 16 * (AM * wm + a) + li;
        if (row >= g.M) continue;
#pragma unroll
        for (int b = 0; b < AN; ++b) {
            const int64_t at = (int64_t)row * g.ldy + n0 + 16 * (AN * wn + b) + 4 * gq;
            if (!g.vec) {
#pragma unroll
                for (int r = 0; r < 4; ++r) store_out<EP>(g.y, at + r, acc[a][b][r]);
                continue;
            }
            store_out4<EP>(g.y, at, acc[a][b]);
        }
    }
}

// ── dense fp16 weights, row-major ──
//
// y = epilogue(fp16(x · wᵀ)) for x [groups][M][lda] fp16 and w [N][K] fp16
// (rows K-contiguous): a dense fp16 base (rwkv_f16_gemm), and quantised passes
// of many rows and a short K (gemm_route).
//
// A workgroup of 8 waves computes a 256 (input rows) × 256 (output features)
// tile in stages of 64 columns.  Both operands are staged in LDS as rows of
// 128 B whose 16-byte chunk c is stored at chunk c ^ (row & 7): the 8 lanes
// reading one chunk column of 8 consecutive rows (an MFMA operand) or
// writing 8 chunks of one row hit distinct banks.  Wave w takes input rows
// 128·(w & 1) .. +127 and features 64·(w >> 1) .. +63: 8 × 4 accumulator
// tiles of 16 × 16, 32 MFMAs per 32-column unit against 12 LDS operand reads
// (the fused kernel's waves: 16 MFMAs against 8).  Each thread moves 8
// chunks a stage (4 input rows, 4 weight rows) with buffer loads: one offset
// register per input row and one for the weights (the stage and the row
// group ride in the scalar offset), which leaves room at two waves per SIMD
// for two register sets.  The loop body is two stages, each set loaded
// during one stage's first unit and written to LDS during the next stage's
// second unit, so loads have more than a stage to land and no register is
// copied (a copy of a register whose load is in flight waits for the load).
// Loads, LDS writes and operand reads are spread between the MFMAs
// (sched_group_barrier): measured 0.42-0.51 of the fp16 peak at M = 8192
// against 0.38-0.43 with them grouped.
//
// Per output the products and their order are quant_gemm_kernel's
// (v_mfma_f32_16x16x32_f16 over the same 32-column units, first to last), so
// with w = the fp16 weight that kernel decodes, the result is its bitwise.
constexpr int DT = 256;         // dense tile: input rows = output features

struct DenseArgs {
    const _Float16* x;    // [groups][M][lda]
    int64_t lda, x_gstride;
    const _Float16* w;    // [N][K]
    void* y;              // [M][ldy]
    int64_t ldy;
    int M, N, K, out_per;
};

template <int EP>
__global__ __launch_bounds__(512, 1) void dense_gemm_kernel(DenseArgs g) {
    __shared__ uint4 lds[2][2 * DT * 8];   // per stage: 256 input rows then 256 weight rows, 8 chunks each
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int gq = lane >> 4, li = lane & 15;
    // Tiles in groups of 4 row blocks × every feature block, feature-major
    // within a group; XCD x (workgroups x, x + 8, ...) takes a contiguous run
    // of that order, so the 32 workgroups an XCD holds at once share 4 input
    // row blocks and 8 weight blocks in its L2.
    const int ntm = (g.M + DT - 1) / DT, ntn = g.N / DT, total = ntm * ntn;
    const int xcd = blockIdx.x & 7, loc = blockIdx.x >> 3;
    const int t = xcd * (total >> 3) + min(xcd, total & 7) + loc;
    const int grp = t / (4 * ntn), first = 4 * grp, gm = min(4, ntm - first);
    const int rr = t - grp * 4 * ntn;
    const int m0 = (first + rr % gm) * DT, n0 = (rr / gm) * DT;
    const int nst = g.K / DKS;

    // staging: thread → chunk c of rows r0 + 64p (p < 4 input rows, clamped
    // to the last row; p >= 4 weight rows), offsets from the tile's first row
    const int c = tid & 7, r0 = tid >> 3;
    const int mrows = min(DT, g.M - m0);
    const _Float16* xt = g.x + (int64_t)(n0 / g.out_per) * g.x_gstride + (int64_t)m0 * g.lda;
    const __amdgpu_buffer_rsrc_t rx =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<_Float16*>(xt), 0, (int)(mrows * g.lda * 2), 0x00020000);
    const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<_Float16*>(g.w + (int64_t)n0 * g.K), 0, (int)((int64_t)DT * g.K * 2), 0x00020000);
    uint32_t xo[4];
#pragma unroll
    for (int p = 0; p < 4; ++p) xo[p] = (uint32_t)((min(r0 + 64 * p, mrows - 1) * (int)g.lda + 8 * c) * 2);
    const uint32_t wo = (uint32_t)((r0 * g.K + 8 * c) * 2), wrow64 = (uint32_t)(64 * g.K * 2);
    const int dst0 = r0 * 8 + (c ^ (r0 & 7));   // row r0 + 64p: + 512p chunks, the same swizzle
    auto gload = [&](uint4 (&v)[8], int st) {
        const uint32_t so = (uint32_t)(min(st, nst - 1) * DKS * 2);
#pragma unroll
        for (int p = 0; p < 4; ++p)
            v[p] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rx, xo[p], so, 0));
#pragma unroll
        for (int p = 0; p < 4; ++p)
            v[4 + p] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rw, wo, so + p * wrow64, 0));
    };
    auto swrite = [&](int buf, const uint4 (&v)[8]) {
#pragma unroll
        for (int p = 0; p < 8; ++p) lds[buf][dst0 + 512 * p] = v[p];
    };

    const int wm = wave & 1, wn = wave >> 1;
    f32x4 acc[8][4];
#pragma unroll
    for (int a = 0; a < 8; ++a)
#pragma unroll
        for (int b = 0; b < 4; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
    // operand rows: li + 16·tile (row & 7 = li & 7 for every tile)
    const int ra = (128 * wm + li) * 8, rb = (DT + 64 * wn + li) * 8;
    // A 32-column unit: the B operands first, then the A operands (the
    // order the products use them)
    auto operands = [&](int buf, int kk, half8 (&av)[8], half8 (&bv)[4]) {
        const int ch = (4 * kk + gq) ^ (li & 7);
#pragma unroll
        for (int b = 0; b < 4; ++b) bv[b] = __builtin_bit_cast(half8, lds[buf][rb + 128 * b + ch]);
#pragma unroll
        for (int a = 0; a < 8; ++a) av[a] = __builtin_bit_cast(half8, lds[buf][ra + 128 * a + ch]);
    };
    auto products = [&](const half8 (&av)[8], const half8 (&bv)[4]) {
#pragma unroll
        for (int a = 0; a < 8; ++a)
#pragma unroll
            for (int b = 0; b < 4; ++b)
                acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av[a], bv[b], acc[a][b], 0, 0, 0);
    };
    // One stage: its two units from LDS buffer `buf`.  The first unit's
    // products carry the loads of a later stage into `ld`, the second's the
    // LDS write of the next stage's chunks from `wr`: six operand reads up
    // front, then per A operand its four MFMAs, the read of the A operand two
    // ahead and one load or write (register use stays at 256, no spills).
    auto stage = [&](int buf, uint4 (&ld)[8], int ldst, const uint4 (&wr)[8]) {
        {
            half8 av[8], bv[4];
            operands(buf, 0, av, bv);
            gload(ld, ldst);
            products(av, bv);
            __builtin_amdgcn_sched_group_barrier(0x100, 6, 0);   // DS reads
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                __builtin_amdgcn_sched_group_barrier(0x008, 4, 0);   // MFMA
                if (i < 6) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);   // VMEM read
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        {
            half8 av[8], bv[4];
            operands(buf, 1, av, bv);
            products(av, bv);
            swrite(buf ^ 1, wr);
            __builtin_amdgcn_sched_group_barrier(0x100, 6, 0);
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                __builtin_amdgcn_sched_group_barrier(0x008, 4, 0);
                if (i < 6) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);   // DS write
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        __syncthreads();
    };

    // nst is even; the last pair's loads repeat the last stage and its final
    // LDS write lands in a buffer no later stage reads
    uint4 va[8], vb[8];
    gload(va, 0);
    swrite(0, va);
    gload(va, 1);
    __syncthreads();
    for (int st = 0; st < nst; st += 2) {
        stage(0, vb, st + 2, va);
        stage(1, va, st + 3, vb);
    }

#pragma unroll
    for (int a = 0; a < 8; ++a) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = m0 + 128 * wm + 16 * a + 4 * gq + r;
            if (row >= g.M) continue;
#pragma unroll
            for (int b = 0; b < 4; ++b)
                store_out<EP>(g.y, (int64_t)row * g.ldy + n0 + 64 * wn + 16 * b + li, acc[a][b][r]);
        }
    }
}

// Which kernel a quantised pass takes when the caller gave a workspace, by
// shape and weight format alone: fp32 inputs take the same sums as fp16 ones
// (an input is rounded to fp16 either way, so equal values give equal results).
// Times in µs, fitted on MI355X to graph-timed calls of every kernel at 11,000
// points (1-16,400 rows, 256-26,900 × 256-14,800 matrices, all five formats;
// the pick is within 15 % of the fastest kernel at 95 of 100 fp16 points).  In
// x rounds of the 256 CUs:
//   * Waves splitting K (gemm_ks_kernel): workgroups of W waves share a CU as
//     LDS and registers allow (occ); a round of occ costs a start plus its K,
//     longer by rho for each workgroup more.  A wave's steps are whole, so K
//     counts half as it is and half rounded up to W waves.  Against one launch
//     with K ranges and their reduction: 128 rows × 3072 × 768 6.5 (13.1), 128
//     × 768 × 3072 7.0 (16.1), 16 × 4096 × 4096 7.6 (22.8).  Its weights are
//     decoded once per row block, so many row blocks favour:
//   * the dense route (dequant_tiles_kernel + dense_tiles_kernel): the dequant
//     (a launch plus its bytes), the output's bytes, then per 64-column stage
//     the latency of one tile or the rate of a full CU.  Against the same: 1001
//     × 3072 × 1024 21.7 (32.9), 4096 × 1024 × 4096 44.7 (134).
//   * the dense route over row-major weights (rwkv_*_dequant +
//     dense_gemm_kernel; fp16 inputs): one round costs more, but each tile
//     starts and ends sooner, which tells for a short K: 8192 × 3072 × 256
//     31.9 (37.5 over operand order), 4177 × 12288 × 768 107 (117), 8192 ×
//     4096 × 1024 77 (78), 4096 × 4096 × 4096 126 (119).
//   * K ranges on 128 × 128 tiles (quant_gemm_kernel), where a tile's 128 rows
//     save a decode: 65-128 rows of 3584 features or more (98 × 10240 × 5888
//     sb6 4-bit 45 (52 split over waves), 128 × 14336 × 14336 sym 8-bit 148
//     (224); fewer features split over waves are faster throughout), and one
//     range, without a dequant, up to K = 1024 (512 × 12288 × 256 14.8 (18.5)).
struct GemmRoute {
    enum Kind { kRanges, kSplitWaves, kDense, kDenseRows } kind = kRanges;
    int tm = 128, tn = 128;   // the tile (kSplitWaves: with fp16 inputs; kDenseRows: that of kDense, for fp32 inputs)
    int parts = 1;            // what K is split over: ranges or waves
};

// Weight formats: sb6 by xbits, then sym 8- and 6-bit.
enum GemmFormat { kSb6 = 0, kSym8 = 3, kSym6 = 4, kFormats = 5 };

// K ranges of a launch on 128 × 128 tiles: one where the (row block, feature
// block) tiles already fill the chip; otherwise enough to reach about 384
// workgroups (two per CU hold 512), each range at least 3 stages of 64 columns.
int gemm_splits(int64_t M, int64_t N, int64_t K) {
    const int64_t tiles = ((M + 127) / 128) * (N / 128);
    if (tiles >= 160) return 1;
    const int64_t want = (384 + tiles - 1) / tiles, most = K / BK / 3;
    return (int)std::max<int64_t>(1, std::min(want, most));
}

// The dense kernel's shapes (x rows lda halves apart, group g at x + g·x_gstride).
bool dense_shape_ok(int64_t M, int64_t OUT, int64_t IN, int64_t out_per, int64_t lda) {
    return M >= 1 && M <= ((int64_t)1 << 24) && OUT >= DT && OUT % DT == 0 && OUT <= ((int64_t)1 << 30) &&
           out_per >= DT && out_per % DT == 0 && OUT % out_per == 0 && IN >= 2 * DKS && IN % (2 * DKS) == 0 &&
           lda >= IN && lda % 8 == 0 && (int64_t)DT * lda * 2 < ((int64_t)1 << 31) &&
           ((M + DT - 1) / DT) * (OUT / DT) < ((int64_t)1 << 31);
}

// Bytes of workspace a route uses.
int64_t route_bytes(const GemmRoute& r, int64_t M, int64_t N, int64_t K) {
    if (r.kind == GemmRoute::kDense || r.kind == GemmRoute::kDenseRows) return N * K * 2;   // the fp16 weight
    return r.kind == GemmRoute::kRanges && r.parts > 1 ? r.parts * M * N * 4 : 0;
}

// The fastest route within `bytes` of workspace.
GemmRoute gemm_route(int fmt, int64_t M, int64_t N, int64_t K, int64_t out_per, int64_t lda, int64_t bytes) {
    const double steps = (double)K / KS_COLS, st = (double)K / DKS;
    const double nk = (double)N * (double)K / 1e6, mn = (double)M * (double)N / 1e6;
    const auto rounds = [&](int tm, int tn) { return (double)((M + tm - 1) / tm) * (double)(N / tn) / 256; };
    GemmRoute best;
    double cost = 1e30;
    const auto offer = [&](double c, const GemmRoute& r) {
        if (c >= cost || route_bytes(r, M, N, K) > bytes) return;
        cost = c;
        best = r;
    };

    static const int unit_bytes[kFormats] = {Sb6W<0>::UB, Sb6W<1>::UB, Sb6W<2>::UB, SymW<8>::UB, SymW<6>::UB};
    struct Ks {
        int mt, nt, waves, many;   // waves per workgroup: one round of the CUs, more
        double a, rho, b[kFormats];
    };
    static const Ks ks[] = {{1, 1, 8, 8, 1.17, 1.00, {0.77, 0.96, 1.09, 0.89, 1.13}},
                            {2, 1, 12, 6, 1.19, 1.18, {1.00, 1.18, 1.29, 1.11, 1.40}},
                            {2, 2, 8, 8, 1.66, 0.94, {1.54, 1.93, 2.06, 1.66, 2.13}},
                            {4, 1, 8, 4, 1.62, 1.21, {1.33, 1.47, 1.59, 1.69, 1.60}},
                            {4, 2, 7, 7, 2.19, 1.42, {2.50, 2.88, 3.37, 2.88, 3.41}},
                            {4, 4, 6, 6, 2.10, 1.40, {5.12, 6.02, 7.66, 7.15, 7.65}}};
    for (const Ks& e : ks) {
        // offsets within a tile's input rows are 32-bit
        if ((int64_t)16 * e.mt * lda * 4 >= ((int64_t)1 << 31)) continue;
        const double x = rounds(16 * e.mt, 16 * e.nt);
        const int lds = ks_wave_lds(unit_bytes[fmt], e.mt, e.nt);
        int w = x > 1 ? e.many : e.waves;
        if (e.mt * e.nt == 1 && K >= 4096) w = 16;
        w = (int)std::min<int64_t>({(int64_t)w, K / KS_COLS, (int64_t)(KS_LDS / lds)});
        // 16 waves of up to 128 registers
        const int occ = std::max(1, std::min({(int)(KS_LDS / (w * lds)), 16 / w, 4}));
        const double kb = e.b[fmt] * (steps + std::ceil(steps / w) * w) / 16;
        const double whole = std::floor(x / occ), part = x - whole * occ;
        offer(2 + whole * (e.a + kb * (1 + e.rho * (occ - 1))) +
                  (part > 0 ? e.a + kb * (1 + e.rho * (std::ceil(part) - 1)) : 0.0),
              {GemmRoute::kSplitWaves, 16 * e.mt, 16 * e.nt, w});
    }

    struct Tile {
        int tm, tn;
        double start, dequant, out;   // dequant, out: per 10^6 weights, outputs
        double big;                   // per 10^6 weights past what the MALL holds of them
        double latency, rate;         // per stage: one tile alone, a tile on a full chip
    };
    const auto dense = [&](const Tile& t) {
        const double n = rounds(t.tm, t.tn), whole = std::floor(n), part = n - whole;
        return t.start + t.dequant * nk + t.big * std::max(0.0, nk - 128) + t.out * mn +
               st * (whole * t.rate + (part > 0 ? std::max(t.latency, t.rate * part) : 0.0));
    };
    static const Tile tiles[] = {{64, 64, 6.95, 0.62, 1.20, 1.00, 0.182, 0.185},
                                 {64, 128, 6.92, 0.66, 0.78, 1.03, 0.258, 0.314},
                                 {128, 128, 8.45, 0.60, 0.74, 0.72, 0.386, 0.434},
                                 {256, 256, 12.2, 0.64, 0.88, 0.62, 0.976, 1.35}};
    static const Tile row_major = {256, 256, 7.87, 0.62, 0.73, 0.50, 0.923, 1.46};
    const Tile* tile = nullptr;   // the fastest operand-ordered one
    double tile_cost = 1e30;
    for (const Tile& t : tiles) {
        if (N % t.tn || out_per % t.tn || (int64_t)t.tm * lda * 4 >= ((int64_t)1 << 31) ||
            (int64_t)t.tn * K * 2 >= ((int64_t)1 << 31))
            continue;
        const double c = dense(t);
        if (c >= tile_cost) continue;
        tile_cost = c;
        tile = &t;
    }
    if (tile) offer(tile_cost, {GemmRoute::kDense, tile->tm, tile->tn, 1});
    // row-major: 4 % faster at K = 1280, the same from 2304 to 4096, 2 % slower
    // beyond (medians over 1,300 passes); its dequant's thread index is 32-bit
    if (tile && K <= 2560 && dense_shape_ok(M, N, K, out_per, lda) && N * (K / 8) < INT32_MAX)
        offer(dense(row_major), {GemmRoute::kDenseRows, tile->tm, tile->tn, 1});

    const int64_t blocks = ((M + 127) / 128) * (N / 128);
    const int S = gemm_splits(M, N, K);
    if (S == 1 ? blocks >= 160 && K <= 1024 : M > 64 && M <= 128 && blocks >= 28) {
        static const double per_stage[kFormats] = {1.67, 2.24, 2.25, 1.66, 2.18};
        const double x = rounds(128, 128) * S, whole = std::floor(x / 2), part = x - 2 * whole;
        const double pitch = K % 2048 == 0 ? 1.21 : K % 1024 == 0 ? 1.09 : 1.0;   // its lanes are rows apart
        // a tie goes to the ranges
        offer((2.1 + (S > 1 ? 3.65 + 1.27 * S * mn : 0.45 * mn) +
               pitch * per_stage[fmt] * st / S *
                   (whole * 1.34 + (part > 0 ? 1 + 0.34 * std::max(0.0, part - 1) : 0.0))) *
                  (S > 1 ? 0.97 : 1.0),
              {GemmRoute::kRanges, 128, 128, S});
    }
    return best;
}

// Bytes of workspace that let a pass of this shape take its fastest route,
// whatever the format, for the entry points where NULL means one range: the
// split over waves touches none and asks for two ranges' fp32 sums, so that no
// shape that has a faster route is taken for one that has not.
int64_t gemm_workspace(int64_t M, int64_t N, int64_t K) {
    int64_t need = 0;
    for (int f = 0; f < kFormats; ++f) {
        const GemmRoute r = gemm_route(f, M, N, K, N, K, INT64_MAX);
        need = std::max(need, r.kind == GemmRoute::kSplitWaves ? 2 * M * N * 4 : route_bytes(r, M, N, K));
    }
    return need;
}

template <int EP>
void launch_dense_ep(const DenseArgs& g, hipStream_t s) {
    const int64_t tiles = (int64_t)((g.M + DT - 1) / DT) * (g.N / DT);
    rwkv::launch(dense_gemm_kernel<EP>, dim3((unsigned)tiles), dim3(512), s, g);
}

void launch_dense(const DenseArgs& g, int epilogue, hipStream_t s) {
    switch (epilogue) {
        case 0: launch_dense_ep<0>(g, s); break;
        case 1: launch_dense_ep<1>(g, s); break;
        default: launch_dense_ep<2>(g, s); break;
    }
}

// One tile shape: 128 × 128 with two workgroups per CU measured fastest
// (larger tiles cost occupancy: at one wave per SIMD the stage's loads are
// not hidden).
template <class F, typename TA, int EP>
void launch_gemm(const GemmArgs& g, hipStream_t s) {
    const int64_t blocks = (int64_t)((g.M + 127) / 128) * (g.N / 128) * g.splits;
    rwkv::launch(quant_gemm_kernel<F, TA, EP, 8, 2>, dim3((unsigned)blocks), dim3(256), s, g);
    if (g.splits > 1) {
        const int64_t n4 = (int64_t)g.M * g.N / 4;
        rwkv::launch(gemm_split_reduce<EP>, dim3((unsigned)((n4 + 255) / 256)), dim3(256), s, g.part, g.splits,
                     g.M, g.N, g.y, g.ldy);
    }
}

// y rows take aligned 4-wide accesses.
bool vec_rows(const GemmArgs& g, int epilogue) {
    return g.ldy % 4 == 0 && reinterpret_cast<uintptr_t>(g.y) % (epilogue == 2 ? 8 : 16) == 0;
}

template <class F, typename TA, int MT, int NT, int MAXW>
void launch_ks_tile(const KsArgs& a, int W, hipStream_t s) {
    constexpr int BM = 16 * MT, BN = 16 * NT;
    const int64_t blocks = (int64_t)((a.g.M + BM - 1) / BM) * (a.g.N / BN);
    const size_t lds = (size_t)W * std::max(BM * (BN + KS_PAD) * 4, ks_wave_lds(F::UB, MT, NT));
    rwkv::launch_lds(gemm_ks_kernel<F, TA, MT, NT, MAXW>, dim3((unsigned)blocks), dim3(64 * W), lds, s, a);
}

// The sums depend on the waves alone, not on the tile: fp32 inputs, whose
// staging takes twice the registers, run the same waves on another tile.
template <class F, typename TA>
void launch_ks(const GemmArgs& g, const GemmRoute& r, int epilogue, hipStream_t s) {
    const KsArgs a{g, epilogue, vec_rows(g, epilogue)};
    const int t = 10 * (r.tm / 16) + r.tn / 16, W = r.parts;
    if (t == 11) launch_ks_tile<F, TA, 1, 1, 16>(a, W, s);
    else if (t == 21) launch_ks_tile<F, TA, 2, 1, 12>(a, W, s);
    else if (t == 22) launch_ks_tile<F, TA, 2, 2, 8>(a, W, s);
    else if constexpr (sizeof(TA) == 4) {
        if (t == 41) launch_ks_tile<F, TA, 2, 2, 8>(a, W, s);
        else launch_ks_tile<F, TA, 2, 4, 8>(a, W, s);
    } else {
        if (t == 41) launch_ks_tile<F, TA, 4, 1, 8>(a, W, s);
        else if (t == 42) launch_ks_tile<F, TA, 4, 2, 8>(a, W, s);
        else launch_ks_tile<F, TA, 4, 4, 8>(a, W, s);
    }
}

template <typename TA, int EP, int WM, int WN, int AM, int AN, int DP, int DA>
void launch_tiles_shape(const DenseTArgs& g, hipStream_t s) {
    constexpr int TM = 16 * WM * AM, TN = 16 * WN * AN;
    rwkv::launch(dense_tiles_kernel<TA, EP, WM, WN, AM, AN, DP, DA>,
                 dim3((unsigned)((int64_t)((g.M + TM - 1) / TM) * (g.N / TN))), dim3(64 * WM * WN), s, g);
}

template <typename TA, int EP>
void launch_tiles_ep(const DenseTArgs& g, const GemmRoute& r, hipStream_t s) {
    switch (r.tm * r.tn) {
        case 64 * 64: launch_tiles_shape<TA, EP, 1, 4, 4, 1, 4, 4>(g, s); break;
        case 64 * 128: launch_tiles_shape<TA, EP, 1, 4, 4, 2, 4, 2>(g, s); break;
        case 128 * 128: launch_tiles_shape<TA, EP, 1, 4, 8, 2, 4, sizeof(TA) == 2 ? 2 : 1>(g, s); break;
        default: launch_tiles_shape<TA, EP, 2, 4, 8, 4, 2, 1>(g, s); break;     // 256 × 256
    }
}

template <typename TA>
void launch_tiles_ta(const DenseTArgs& a, const GemmRoute& r, int epilogue, hipStream_t s) {
    if (epilogue == 0) launch_tiles_ep<TA, 0>(a, r, s);
    else if (epilogue == 1) launch_tiles_ep<TA, 1>(a, r, s);
    else launch_tiles_ep<TA, 2>(a, r, s);
}

// The dense route: dequantise into the workspace (operand order), then multiply.
template <class F>
void launch_tiles(const GemmArgs& g, const GemmRoute& r, bool f16, void* workspace, int epilogue, hipStream_t s) {
    _Float16* w = reinterpret_cast<_Float16*>(workspace);
    const int64_t waves = (int64_t)(g.N / 16) * (g.K / 128);
    rwkv::launch(dequant_tiles_kernel<F>, dim3((unsigned)((waves + 3) / 4)), dim3(256), s, g, w);
    const DenseTArgs a{g.x, g.lda, g.x_gstride, w, g.y, g.ldy, g.M, g.N, g.K, g.out_per, vec_rows(g, epilogue)};
    f16 ? launch_tiles_ta<_Float16>(a, r, epilogue, s) : launch_tiles_ta<float>(a, r, epilogue, s);
}

template <class F>
void launch_gemm_ep(const GemmArgs& g, bool f16, int epilogue, hipStream_t s) {
    switch (epilogue) {
        case 0: f16 ? launch_gemm<F, _Float16, 0>(g, s) : launch_gemm<F, float, 0>(g, s); break;
        case 1: f16 ? launch_gemm<F, _Float16, 1>(g, s) : launch_gemm<F, float, 1>(g, s); break;
        default: f16 ? launch_gemm<F, _Float16, 2>(g, s) : launch_gemm<F, float, 2>(g, s); break;
    }
}

// Any kind but kDenseRows.
template <class F>
void launch_routed(GemmArgs g, const GemmRoute& r, bool f16, void* workspace, int epilogue, hipStream_t s) {
    if (r.kind == GemmRoute::kDense) {
        launch_tiles<F>(g, r, f16, workspace, epilogue, s);
    } else if (r.kind == GemmRoute::kSplitWaves) {
        f16 ? launch_ks<F, _Float16>(g, r, epilogue, s) : launch_ks<F, float>(g, r, epilogue, s);
    } else {
        g.part = reinterpret_cast<float*>(workspace);
        g.splits = r.parts;
        launch_gemm_ep<F>(g, f16, epilogue, s);
    }
}

// The dense route over row-major weights, once the workspace holds them.
void launch_rows(const GemmArgs& g, const void* workspace, int epilogue, hipStream_t s) {
    launch_dense(DenseArgs{reinterpret_cast<const _Float16*>(g.x), g.lda, g.x_gstride,
                           reinterpret_cast<const _Float16*>(workspace), g.y, g.ldy, g.M, g.N, g.K, g.out_per},
                 epilogue, s);
}

bool gemm_shape_ok(int64_t OUT, int64_t IN, int64_t out_per) {
    return OUT >= 128 && OUT % 128 == 0 && IN >= 256 && IN % 256 == 0 && out_per >= 128 && out_per % 128 == 0 &&
           OUT % out_per == 0 && OUT <= ((int64_t)1 << 30) && IN <= ((int64_t)1 << 24);
}

// Shared argument checks of the two entry points.
rwkv_status gemm_check(const char* who, const void* x, rwkv_dtype x_dt, int64_t M, int64_t lda,
                       int64_t x_group_stride, int64_t ldy, int64_t OUT, int64_t IN, int64_t out_per, int epilogue) {
    RWKV_REQUIRE(x_dt == RWKV_F32 || x_dt == RWKV_F16, RWKV_E_DTYPE, "%s: inputs must be f32 or f16", who);
    RWKV_REQUIRE(epilogue >= 0 && epilogue <= 2, RWKV_E_SHAPE, "%s: epilogue %d", who, epilogue);
    RWKV_REQUIRE(M >= 1 && M <= ((int64_t)1 << 24), RWKV_E_SHAPE, "%s: M (%lld) out of range", who, (long long)M);
    const int64_t groups = OUT / out_per;
    const int64_t xes = x_dt == RWKV_F32 ? 4 : 2;
    RWKV_REQUIRE(lda >= IN && lda % 8 == 0 && (groups == 1 || x_group_stride >= M * lda), RWKV_E_SHAPE,
                 "%s: lda (%lld) must be >= IN and a multiple of 8; groups need x_group_stride >= M·lda", who,
                 (long long)lda);
    RWKV_REQUIRE(ldy >= OUT && (epilogue == 2 ? ldy % 2 == 0 : true), RWKV_E_SHAPE, "%s: ldy (%lld) < OUT", who,
                 (long long)ldy);
    RWKV_REQUIRE((reinterpret_cast<uintptr_t>(x) % 16) == 0 && (x_group_stride * xes) % 16 == 0, RWKV_E_SHAPE,
                 "%s: inputs must be 16-byte aligned", who);
    RWKV_REQUIRE(((M + 127) / 128) * (OUT / 128) <= ((int64_t)1 << 26), RWKV_E_SHAPE,
                 "%s: %lld x %lld outputs exceed one launch", who, (long long)M, (long long)OUT);
    return RWKV_OK;
}

// A caller's workspace (checked before anything is launched): 16-byte aligned;
// `least` is what is refused below.
rwkv_status gemm_workspace_check(const char* who, int64_t least, const void* workspace, int64_t workspace_bytes) {
    RWKV_REQUIRE(workspace_bytes >= least && reinterpret_cast<uintptr_t>(workspace) % 16 == 0, RWKV_E_SHAPE,
                 "%s: workspace of %lld bytes (16-byte aligned) needed, %lld given", who, (long long)least,
                 (long long)workspace_bytes);
    return RWKV_OK;
}

// The least workspace of the entry points where NULL means one range: what
// gemm_workspace asks for, or what a caller may have sized by another rule, if
// that is less — the fp16 weight from 128 tiles of 256 × 256, else the sums of
// the K ranges that 128 × 128 tiles are split into, nothing for one range.  The
// route keeps within the bytes given.
int64_t gemm_workspace_least(int64_t M, int64_t N, int64_t K) {
    const int64_t S = gemm_splits(M, N, K);
    const bool dense = dense_shape_ok(M, N, K, N, K) && ((M + DT - 1) / DT) * (N / DT) >= 128;
    const int64_t other = dense ? N * K * 2 : S > 1 ? S * M * N * 4 : 0;
    return other ? std::min(other, gemm_workspace(M, N, K)) : 0;
}

// Route of a call with this much workspace (< 0: one K range).
GemmRoute entry_route(int fmt, rwkv_dtype x_dt, int64_t M, int64_t N, int64_t K, int64_t out_per, int64_t lda,
                      int64_t workspace_bytes) {
    GemmRoute r;
    if (workspace_bytes >= 0) r = gemm_route(fmt, M, N, K, out_per, lda, workspace_bytes);
    // row-major weights meet fp16 inputs only; operand order gives the same bits
    if (r.kind == GemmRoute::kDenseRows && x_dt != RWKV_F16) r.kind = GemmRoute::kDense;
    return r;
}

// The workspace an entry's call routes with: what NULL means is all that sets
// rwkv_*_gemm (one range) and rwkv_*_gemm_auto (no workspace) apart.
rwkv_status entry_workspace(const char* who, bool any, int64_t M, int64_t N, int64_t K, const void* workspace,
                            int64_t* workspace_bytes) {
    if (workspace == nullptr) {
        *workspace_bytes = any ? 0 : -1;
        return RWKV_OK;
    }
    return gemm_workspace_check(who, any ? 0 : gemm_workspace_least(M, N, K), workspace, *workspace_bytes);
}

rwkv_status sb6_gemm(const char* who, bool any, const void* x, rwkv_dtype x_dt, int64_t M, int64_t lda,
                     int64_t x_group_stride, const uint8_t* qblk, const uint8_t* qsqm, const uint16_t* ddm, void* y,
                     int64_t ldy, int64_t OUT, int64_t IN, int xbits, int64_t out_per, int epilogue, void* workspace,
                     int64_t workspace_bytes, void* stream) {
    RWKV_REQUIRE(x && qblk && qsqm && ddm && y, RWKV_E_NULL, "%s: null buffer", who);
    RWKV_REQUIRE(rwkv_sb6_gemm_applies(OUT, IN, xbits, out_per), RWKV_E_UNSUPPORTED,
                 "%s: xbits %d (0..2), OUT (%lld) and out_per (%lld) multiples of 128, IN (%lld) of 256", who, xbits,
                 (long long)OUT, (long long)out_per, (long long)IN);
    rwkv_status c = gemm_check(who, x, x_dt, M, lda, x_group_stride, ldy, OUT, IN, out_per, epilogue);
    if (c != RWKV_OK) return c;
    c = entry_workspace(who, any, M, OUT, IN, workspace, &workspace_bytes);
    if (c != RWKV_OK) return c;
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    const GemmArgs g{x, lda, x_group_stride, qblk, qsqm, ddm, y, ldy, (int)M, (int)OUT, (int)IN, (int)out_per, nullptr, 1};
    const bool f16 = x_dt == RWKV_F16;
    const GemmRoute r = entry_route(kSb6 + xbits, x_dt, M, OUT, IN, out_per, lda, workspace_bytes);
    if (r.kind == GemmRoute::kDense) rwkv::counters().sb6_dequant.fetch_add(1);
    if (r.kind == GemmRoute::kDenseRows) {
        c = rwkv_sb6_dequant(qblk, qsqm, ddm, workspace, RWKV_F16, OUT, IN, xbits, stream);
        if (c != RWKV_OK) return c;
        launch_rows(g, workspace, epilogue, s);
    } else if (xbits == 0) launch_routed<Sb6W<0>>(g, r, f16, workspace, epilogue, s);
    else if (xbits == 1) launch_routed<Sb6W<1>>(g, r, f16, workspace, epilogue, s);
    else launch_routed<Sb6W<2>>(g, r, f16, workspace, epilogue, s);
    RWKV_REQUIRE(hipGetLastError() == hipSuccess, RWKV_E_HIP, "%s: launch failed", who);
    rwkv::counters().sb6_gemm.fetch_add(1);
    rwkv::clear_error();
    return RWKV_OK;
}

rwkv_status sym_gemm(const char* who, bool any, const void* x, rwkv_dtype x_dt, int64_t M, int64_t lda,
                     int64_t x_group_stride, const uint8_t* qblk, const uint8_t* qs, const uint16_t* d, void* y,
                     int64_t ldy, int64_t OUT, int64_t IN, int bits, int64_t out_per, int epilogue, void* workspace,
                     int64_t workspace_bytes, void* stream) {
    RWKV_REQUIRE(x && qblk && qs && d && y, RWKV_E_NULL, "%s: null buffer", who);
    RWKV_REQUIRE(rwkv_sym_gemm_applies(OUT, IN, bits, out_per), RWKV_E_UNSUPPORTED,
                 "%s: %d-bit codes (8 or 6), OUT (%lld) and out_per (%lld) multiples of 128, IN (%lld) of 256", who,
                 bits, (long long)OUT, (long long)out_per, (long long)IN);
    rwkv_status c = gemm_check(who, x, x_dt, M, lda, x_group_stride, ldy, OUT, IN, out_per, epilogue);
    if (c != RWKV_OK) return c;
    c = entry_workspace(who, any, M, OUT, IN, workspace, &workspace_bytes);
    if (c != RWKV_OK) return c;
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    const GemmArgs g{x, lda, x_group_stride, qblk, qs, d, y, ldy, (int)M, (int)OUT, (int)IN, (int)out_per, nullptr, 1};
    const bool f16 = x_dt == RWKV_F16;
    const GemmRoute r = entry_route(bits == 8 ? kSym8 : kSym6, x_dt, M, OUT, IN, out_per, lda, workspace_bytes);
    if (r.kind == GemmRoute::kDense) rwkv::counters().sym_dequant.fetch_add(1);
    if (r.kind == GemmRoute::kDenseRows) {
        c = rwkv_sym_dequant(qblk, qs, d, workspace, RWKV_F16, OUT, IN, bits, stream);
        if (c != RWKV_OK) return c;
        launch_rows(g, workspace, epilogue, s);
    } else if (bits == 8) launch_routed<SymW<8>>(g, r, f16, workspace, epilogue, s);
    else launch_routed<SymW<6>>(g, r, f16, workspace, epilogue, s);
    RWKV_REQUIRE(hipGetLastError() == hipSuccess, RWKV_E_HIP, "%s: launch failed", who);
    rwkv::counters().sym_gemm.fetch_add(1);
    rwkv::clear_error();
    return RWKV_OK;
}

}  // namespace

extern "C" {

rwkv_status rwkv_quant_gemm_route(int sym, int bits, rwkv_dtype x_dt, int64_t M, int64_t OUT, int64_t IN,
                                  int64_t out_per, int64_t workspace_bytes, int32_t* route) {
    RWKV_REQUIRE(route, RWKV_E_NULL, "quant_gemm_route: null output");
    RWKV_REQUIRE(sym ? rwkv_sym_gemm_applies(OUT, IN, bits, out_per) : rwkv_sb6_gemm_applies(OUT, IN, bits, out_per),
                 RWKV_E_UNSUPPORTED, "quant_gemm_route: [%lld, %lld] bits %d out_per %lld not taken", (long long)OUT,
                 (long long)IN, bits, (long long)out_per);
    RWKV_REQUIRE(M >= 1 && M <= ((int64_t)1 << 24), RWKV_E_SHAPE, "quant_gemm_route: M (%lld) out of range", (long long)M);
    RWKV_REQUIRE(x_dt == RWKV_F32 || x_dt == RWKV_F16, RWKV_E_DTYPE, "quant_gemm_route: inputs are f32 or f16");
    const GemmRoute r = entry_route(sym ? (bits == 8 ? kSym8 : kSym6) : kSb6 + bits, x_dt, M, OUT, IN, out_per, IN,
                                    workspace_bytes);
    route[0] = r.kind;
    route[1] = r.kind == GemmRoute::kDenseRows ? DT : r.tm;
    route[2] = r.kind == GemmRoute::kDenseRows ? DT : r.tn;
    route[3] = r.parts;
    rwkv::clear_error();
    return RWKV_OK;
}

int64_t rwkv_quant_gemm_auto_workspace(int sym, int bits, int64_t M, int64_t OUT, int64_t IN, int64_t out_per) {
    if (M < 1 || M > ((int64_t)1 << 24) ||
        !(sym ? rwkv_sym_gemm_applies(OUT, IN, bits, out_per) : rwkv_sb6_gemm_applies(OUT, IN, bits, out_per)))
        return 0;
    const int fmt = sym ? (bits == 8 ? kSym8 : kSym6) : kSb6 + bits;
    return route_bytes(gemm_route(fmt, M, OUT, IN, out_per, IN, INT64_MAX), M, OUT, IN);
}

int64_t rwkv_quant_gemm_workspace(int64_t M, int64_t OUT, int64_t IN) {
    if (M < 1 || M > ((int64_t)1 << 24) || OUT < 128 || OUT % 128 != 0 || IN < 256 || IN % 256 != 0) return 0;
    return gemm_workspace(M, OUT, IN);
}

int rwkv_sb6_gemm_applies(int64_t OUT, int64_t IN, int xbits, int64_t out_per) {
    return xbits >= 0 && xbits <= 2 && gemm_shape_ok(OUT, IN, out_per);
}

rwkv_status rwkv_sb6_gemm(const void* x, rwkv_dtype x_dt, int64_t M, int64_t lda, int64_t x_group_stride,
                          const uint8_t* qblk, const uint8_t* qsqm, const uint16_t* ddm, void* y, int64_t ldy,
                          int64_t OUT, int64_t IN, int xbits, int64_t out_per, int epilogue, void* workspace,
                          int64_t workspace_bytes, void* stream) {
    return sb6_gemm("sb6_gemm", false, x, x_dt, M, lda, x_group_stride, qblk, qsqm, ddm, y, ldy, OUT, IN, xbits, out_per,
                    epilogue, workspace, workspace_bytes, stream);
}

rwkv_status rwkv_sb6_gemm_auto(const void* x, rwkv_dtype x_dt, int64_t M, int64_t lda, int64_t x_group_stride,
                               const uint8_t* qblk, const uint8_t* qsqm, const uint16_t* ddm, void* y, int64_t ldy,
                               int64_t OUT, int64_t IN, int xbits, int64_t out_per, int epilogue, void* workspace,
                               int64_t workspace_bytes, void* stream) {
    return sb6_gemm("sb6_gemm_auto", true, x, x_dt, M, lda, x_group_stride, qblk, qsqm, ddm, y, ldy, OUT, IN, xbits, out_per,
                    epilogue, workspace, workspace_bytes, stream);
}

int rwkv_sym_gemm_applies(int64_t OUT, int64_t IN, int bits, int64_t out_per) {
    return (bits == 8 || bits == 6) && gemm_shape_ok(OUT, IN, out_per);
}

rwkv_status rwkv_sym_gemm(const void* x, rwkv_dtype x_dt, int64_t M, int64_t lda, int64_t x_group_stride,
                          const uint8_t* qblk, const uint8_t* qs, const uint16_t* d, void* y, int64_t ldy,
                          int64_t OUT, int64_t IN, int bits, int64_t out_per, int epilogue, void* workspace,
                          int64_t workspace_bytes, void* stream) {
    return sym_gemm("sym_gemm", false, x, x_dt, M, lda, x_group_stride, qblk, qs, d, y, ldy, OUT, IN, bits, out_per,
                    epilogue, workspace, workspace_bytes, stream);
}

rwkv_status rwkv_sym_gemm_auto(const void* x, rwkv_dtype x_dt, int64_t M, int64_t lda, int64_t x_group_stride,
                               const uint8_t* qblk, const uint8_t* qs, const uint16_t* d, void* y, int64_t ldy,
                               int64_t OUT, int64_t IN, int bits, int64_t out_per, int epilogue, void* workspace,
                               int64_t workspace_bytes, void* stream) {
    return sym_gemm("sym_gemm_auto", true, x, x_dt, M, lda, x_group_stride, qblk, qs, d, y, ldy, OUT, IN, bits, out_per,
                    epilogue, workspace, workspace_bytes, stream);
}

int rwkv_f16_gemm_applies(int64_t M, int64_t OUT, int64_t IN, int64_t out_per) {
    return dense_shape_ok(M, OUT, IN, out_per, IN);
}

rwkv_status rwkv_f16_gemm(const void* x, int64_t M, int64_t lda, int64_t x_group_stride, const void* w, void* y,
                          int64_t ldy, int64_t OUT, int64_t IN, int64_t out_per, int epilogue, void* stream) {
    RWKV_REQUIRE(x && w && y, RWKV_E_NULL, "f16_gemm: null buffer");
    RWKV_REQUIRE(dense_shape_ok(M, OUT, IN, out_per, lda), RWKV_E_UNSUPPORTED,
                 "f16_gemm: M %lld, OUT (%lld) and out_per (%lld) multiples of 256, IN (%lld) of 128, lda (%lld) >= "
                 "IN and a multiple of 8",
                 (long long)M, (long long)OUT, (long long)out_per, (long long)IN, (long long)lda);
    rwkv_status c = gemm_check("f16_gemm", x, RWKV_F16, M, lda, x_group_stride, ldy, OUT, IN, out_per, epilogue);
    if (c != RWKV_OK) return c;
    RWKV_REQUIRE(reinterpret_cast<uintptr_t>(w) % 16 == 0, RWKV_E_SHAPE, "f16_gemm: weights must be 16-byte aligned");
    launch_dense(DenseArgs{reinterpret_cast<const _Float16*>(x), lda, x_group_stride,
                           reinterpret_cast<const _Float16*>(w), y, ldy, (int)M, (int)OUT, (int)IN, (int)out_per},
                 epilogue, reinterpret_cast<hipStream_t>(stream));
    RWKV_REQUIRE(hipGetLastError() == hipSuccess, RWKV_E_HIP, "f16_gemm: launch failed");
    rwkv::clear_error();
    return RWKV_OK;
}

}  // extern "C"
