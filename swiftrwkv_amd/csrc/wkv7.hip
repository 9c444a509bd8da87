// WKV-7 recurrence on gfx950: whole-sequence / chunk / training forward, the
// checkpointed backward, the one-token decode step and the tmix tail.
//
// Recurrence per (b, h), state S[i = value row, j = key column] (fp32):
//   sa_i = Σ_j S_ij a_j ;  S_ij ← w_j S_ij + v_i k_j + sa_i b_j ;  y_i = Σ_j S_ij r_j
// (Sources/RWKVKernel/WKV7.swift:207-224).
//
// Forward (one wave = 16 value rows × 64 key columns of one head, no LDS, no
// barrier).  Lane l owns row 16·blk + (l & 15) and the 16 key columns of
// column group g = l >> 4, holding those 16 state values in VGPRs for the
// whole sequence.  The 16 lanes of a DPP row share g, so each step vector
// (a, w, k, b, r) is held ONE value per lane (lane l keeps element 16g + (l & 15))
// and broadcast into the FMAs with DPP row_newbcast — a single global_load per
// vector per step, prefetched 8 steps ahead in a 16-slot register ring.  The
// four column-group partials of sa and y of a row (lanes l, l^16, l^32, l^48)
// are combined with v_permlane16_swap / v_permlane32_swap.  The next step's sa
// partial is accumulated inside the update loop, so a step is 5 FMAs per
// state element plus two lane swaps.
// The decode step, the chunk kernel and the training forward are this same
// kernel (T = 1 / emitted sa / emitted checkpoints), so they agree bitwise by
// construction (the reference's invariants WKV7SequenceTests,
// WKV7StateTests.swift:178-186, DecodeKernelTests.swift:27-39).
//
// Backward (the results of ckptBwdKernelV2, WKV7Train.swift:234-339).  Eight
// waves per head; wave q owns the value rows [8q, 8q+8) of the states and of
// dS, and the key columns [8q, 8q+8) of a second copy of dS.  Instead of
// reconstructing earlier states by dividing by w (which re-amplifies the
// forward's rounding by up to 1/w^15), each 16-step chunk's states are
// recomputed forward from the previous checkpoint (or h_in) with the stored sa
// in the forward's order of operations, and held in registers.  Step vectors
// are staged per chunk in LDS (coalesced loads issued one chunk ahead); dsa is
// the one quantity exchanged inside a step (one barrier per step); every
// output is summed over the eight waves from an LDS ring.
// Variant 1 is the reference's row-owned ckptBwdKernel (WKV7Train.swift:
// 99-205), which does divide by w: wkv7_bwd_rows_kernel below.
//
// All arithmetic is fp32 with a fixed summation order: launches are bitwise
// deterministic.

#include <hip/hip_runtime.h>

#include <type_traits>
#include <utility>

#include "launch.h"
#include "wkv7_step.h"

namespace {

using namespace rwkv_wkv;
constexpr int CH = 16;  // WKV7_CHUNK

template <int DT>
__device__ __forceinline__ float load1(const void* __restrict__ p, int64_t off) {
    if constexpr (DT == RWKV_F32) return reinterpret_cast<const float*>(p)[off];
    uint16_t h = reinterpret_cast<const uint16_t*>(p)[off];
    if constexpr (DT == RWKV_BF16) return __uint_as_float((uint32_t)h << 16);
    return (float)__builtin_bit_cast(_Float16, h);
}

template <int DT>
__device__ __forceinline__ void store1(void* __restrict__ p, int64_t off, float x) {
    if constexpr (DT == RWKV_F32) {
        reinterpret_cast<float*>(p)[off] = x;
    } else if constexpr (DT == RWKV_BF16) {
        reinterpret_cast<uint16_t*>(p)[off] = __builtin_bit_cast(uint16_t, (__bf16)x);
    } else {
        reinterpret_cast<uint16_t*>(p)[off] = __builtin_bit_cast(uint16_t, (_Float16)x);
    }
}

// Element off of p.
template <int DT>
__device__ __forceinline__ const void* at(const void* p, int64_t off) {
    return reinterpret_cast<const char*>(p) + off * (DT == RWKV_F32 ? 4 : 2);
}

// ─────────────────────────────── forward ───────────────────────────────
// Grid: 4 workgroups of one wave per (b, h); workgroup 4·(b·H + h) + blk owns
// value rows 16·blk .. 16·blk + 15.  Offsets inside one (b, h) sequence are
// 32-bit (the host checks T·H·64·4 < 2^32), so loads use an SGPR base.
template <int DT>
struct FwdIn {
    using E = typename std::conditional<DT == RWKV_F32, float, uint16_t>::type;
    const E* a;
    const E* w;
    const E* k;
    const E* b;
    const E* r;
    const E* v;
    __device__ __forceinline__ static float cvt(E x) {
        if constexpr (DT == RWKV_F32) return x;
        else if constexpr (DT == RWKV_BF16) return __uint_as_float((uint32_t)x << 16);
        else return (float)__builtin_bit_cast(_Float16, x);
    }
};

template <int DT, bool EMIT_SA, bool EMIT_CK>
__global__ __launch_bounds__(64) void wkv7_fwd_kernel(
    const void* __restrict__ r, const void* __restrict__ w, const void* __restrict__ k,
    const void* __restrict__ v, const void* __restrict__ a, const void* __restrict__ b,
    const float* __restrict__ h_in, float* __restrict__ out, float* __restrict__ h_out,
    float* __restrict__ sa_out, float* __restrict__ ckpt, int T, int H) {
    using In = FwdIn<DT>;
    using E = typename In::E;
    const int l = threadIdx.x;
    const int ri = l & 15, g = l >> 4;
    // Workgroups are dealt round-robin to the 8 XCDs (each with its own L2):
    // when the grid allows, the four waves of a head get ids congruent mod 8,
    // so they share one XCD and each step vector is fetched from HBM once.
    int bh, blk;
    if ((gridDim.x & 31) == 0) {
        const int id = blockIdx.x, xcd = id & 7, slot = id >> 3;
        bh = (slot >> 2) * 8 + xcd;
        blk = slot & 3;
    } else {
        bh = blockIdx.x >> 2;
        blk = blockIdx.x & 3;
    }
    const int bi = bh / H, hi = bh - bi * H;
    const int row = 16 * blk + ri;
    const uint32_t vidx = 16 * g + ri;   // step-vector element this lane broadcasts
    const uint32_t strideT = (uint32_t)H * D;
    const int64_t base0 = ((int64_t)bi * T * H + hi) * D;
    const int64_t sbase = (int64_t)bh * D * D + (int64_t)row * D + 16 * g;
    const int NC = T / CH;
    In in{reinterpret_cast<const E*>(a) + base0, reinterpret_cast<const E*>(w) + base0,
          reinterpret_cast<const E*>(k) + base0, reinterpret_cast<const E*>(b) + base0,
          reinterpret_cast<const E*>(r) + base0, reinterpret_cast<const E*>(v) + base0};
    float* const outp = out + base0;
    float* const sap = EMIT_SA ? sa_out + base0 : nullptr;

    float S[2][16];
    if (h_in) {
        const float4* src = reinterpret_cast<const float4*>(h_in + sbase);
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            const float4 f = src[m];
            S[0][4 * m] = f.x; S[0][4 * m + 1] = f.y; S[0][4 * m + 2] = f.z; S[0][4 * m + 3] = f.w;
        }
    } else {
#pragma unroll
        for (int c = 0; c < 16; ++c) S[0][c] = 0.0f;
    }

    // ring slot: a, w, k, b, r (broadcast sources), v (own row), as raw elements
    E ring[CH][6];
    // Buffer addressing: a descriptor per input (SGPRs), the per-lane part a
    // fixed VGPR offset, the per-step part a scalar offset — no per-load VALU.
    const uint32_t esz = (uint32_t)sizeof(E);
    const uint32_t span = (uint32_t)T * strideT * esz - (uint32_t)hi * D * esz;   // bytes from this head's base
    const uint32_t voff = vidx * esz, roff = (uint32_t)row * esz;
    auto rsrc = [&](const void* p, uint32_t n) { return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)n, 0x00020000); };
    const __amdgpu_buffer_rsrc_t ra = rsrc(in.a, span), rw = rsrc(in.w, span), rk_ = rsrc(in.k, span),
                                 rb = rsrc(in.b, span), rr = rsrc(in.r, span), rv = rsrc(in.v, span);
    auto ld = [&](__amdgpu_buffer_rsrc_t rs, uint32_t vo, uint32_t so) -> E {
        if constexpr (sizeof(E) == 2) return (E)__builtin_amdgcn_raw_buffer_load_b16(rs, vo, so, 0);
        else return __builtin_bit_cast(E, __builtin_amdgcn_raw_buffer_load_b32(rs, vo, so, 0));
    };
    auto fetch = [&](E (&slot)[6], int t) __attribute__((always_inline)) {
        const uint32_t so = (uint32_t)min(t, T - 1) * strideT * esz;
        slot[0] = ld(ra, voff, so);
        slot[1] = ld(rw, voff, so);
        slot[2] = ld(rk_, voff, so);
        slot[3] = ld(rb, voff, so);
        slot[4] = ld(rr, voff, so);
        slot[5] = ld(rv, roff, so);
    };
    const uint32_t ospan = (uint32_t)T * strideT * 4u - (uint32_t)hi * D * 4u;
    const __amdgpu_buffer_rsrc_t ro_ = rsrc(outp, ospan), rs_ = rsrc(EMIT_SA ? sap : outp, ospan);
    const uint32_t orow = (uint32_t)row * 4u;
#pragma unroll
    for (int s = 0; s < 8; ++s) fetch(ring[s], s);

    float p = 0.0f;
    fwd_dot16(S[0], In::cvt(ring[0][0]), p);
    float y = 0.0f;   // partial y of the previous step, reduced and stored one step late

    // one step at chunk position s (compile-time) and time t
    auto step = [&](auto sc, int t, int c) __attribute__((always_inline)) {
        constexpr int s = decltype(sc)::value;
        // Steps stay in program order (no store sinking / load hoisting across
        // them), so every wait for a prefetched value is a small exact count.
        __builtin_amdgcn_sched_barrier(0);
        fetch(ring[(s + 8) & (CH - 1)], t + 8);
        float sa = p;
        rowsum4_pair(sa, y);   // sa of step t, y of step t - 1
        // y of step t - 1 (at t = 0 a placeholder at row 0, overwritten next
        // step); the four lanes of a row store the same bits
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, y), ro_, orow,
                                              (uint32_t)max(t - 1, 0) * strideT * 4u, 0);
        y = 0.0f;
        p = 0.0f;
        const E* sl = ring[s];
        fwd_update16(S[s & 1], S[(s + 1) & 1], In::cvt(sl[2]), In::cvt(sl[3]), In::cvt(sl[1]), In::cvt(sl[4]),
                     In::cvt(ring[(s + 1) & (CH - 1)][0]), In::cvt(sl[5]), sa, y, p);
        const uint32_t so = (uint32_t)t * strideT * 4u;
        if constexpr (EMIT_SA) __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, sa), rs_, orow, so, 0);
        if constexpr (EMIT_CK && s == CH - 1) {
            float4* dst = reinterpret_cast<float4*>(ckpt + ((int64_t)bh * NC + c) * D * D + (int64_t)row * D + 16 * g);
#pragma unroll
            for (int m = 0; m < 4; ++m)
                dst[m] = make_float4(S[0][4 * m], S[0][4 * m + 1], S[0][4 * m + 2], S[0][4 * m + 3]);
        }
    };
    auto body = [&](int c, int n) __attribute__((always_inline)) {
        const int t0 = c * CH;
        [&]<int... s>(std::integer_sequence<int, s...>) {
            ((n > s ? step(std::integral_constant<int, s>{}, t0 + s, c) : void()), ...);
        }(std::make_integer_sequence<int, CH>{});
    };
    auto body_full = [&](int c) __attribute__((always_inline)) {
        const int t0 = c * CH;
        [&]<int... s>(std::integer_sequence<int, s...>) {
            (step(std::integral_constant<int, s>{}, t0 + s, c), ...);
        }(std::make_integer_sequence<int, CH>{});
    };
    // Branch-free chunks.  The first one is peeled so the loop is entered
    // with the same outstanding loads and stores as its back edge: the wait
    // counts at the loop head stay exact instead of draining everything.
    if (NC > 0) body_full(0);
    for (int c = 1; c < NC; ++c) body_full(c);
    const int tail = T - NC * CH;
    if (tail) body(NC, tail);
    y = rowsum4(y);
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, y), ro_, orow, (uint32_t)(T - 1) * strideT * 4u, 0);

    float4* dst = reinterpret_cast<float4*>(h_out + sbase);
    if (tail & 1) {
#pragma unroll
        for (int m = 0; m < 4; ++m) dst[m] = make_float4(S[1][4 * m], S[1][4 * m + 1], S[1][4 * m + 2], S[1][4 * m + 3]);
    } else {
#pragma unroll
        for (int m = 0; m < 4; ++m) dst[m] = make_float4(S[0][4 * m], S[0][4 * m + 1], S[0][4 * m + 2], S[0][4 * m + 3]);
    }
}

// Forward, four-row layout: 16 workgroups of one wave per (b, h); workgroup
// 16·(b·H + h) + blk owns value rows 4·blk .. 4·blk + 3.  Each lane loads
// element l of the step vectors (a 256-byte coalesced row per vector and
// step) and its row's v; otherwise the step is wkv7_fwd_kernel's.
template <int DT, bool EMIT_SA, bool EMIT_CK>
__global__ __launch_bounds__(64) void wkv7_fwd4_kernel(
    const void* __restrict__ r, const void* __restrict__ w, const void* __restrict__ k,
    const void* __restrict__ v, const void* __restrict__ a, const void* __restrict__ b,
    const float* __restrict__ h_in, float* __restrict__ out, float* __restrict__ h_out,
    float* __restrict__ sa_out, float* __restrict__ ckpt, int T, int H) {
    using In = FwdIn<DT>;
    using E = typename In::E;
    const int l = threadIdx.x;
    const int ri = l & 3, g = l >> 2;
    // the sixteen waves of a head on one XCD when the grid allows
    int bh, blk;
    if ((gridDim.x & 127) == 0) {
        const int id = blockIdx.x, xcd = id & 7, slot = id >> 3;
        bh = (slot >> 4) * 8 + xcd;
        blk = slot & 15;
    } else {
        bh = blockIdx.x >> 4;
        blk = blockIdx.x & 15;
    }
    const int bi = bh / H, hi = bh - bi * H;
    const int row = 4 * blk + ri;
    const uint32_t strideT = (uint32_t)H * D;
    const int64_t base0 = ((int64_t)bi * T * H + hi) * D;
    const int64_t sbase = (int64_t)bh * D * D + (int64_t)row * D + 4 * g;
    const int NC = T / CH;
    In in{reinterpret_cast<const E*>(a) + base0, reinterpret_cast<const E*>(w) + base0,
          reinterpret_cast<const E*>(k) + base0, reinterpret_cast<const E*>(b) + base0,
          reinterpret_cast<const E*>(r) + base0, reinterpret_cast<const E*>(v) + base0};
    float* const outp = out + base0;
    float* const sap = EMIT_SA ? sa_out + base0 : nullptr;

    float S[2][4];
    if (h_in) {
        const float4 f = *reinterpret_cast<const float4*>(h_in + sbase);
        S[0][0] = f.x; S[0][1] = f.y; S[0][2] = f.z; S[0][3] = f.w;
    } else {
#pragma unroll
        for (int c = 0; c < 4; ++c) S[0][c] = 0.0f;
    }

    E ring[CH][6];
    const uint32_t esz = (uint32_t)sizeof(E);
    const uint32_t span = (uint32_t)T * strideT * esz - (uint32_t)hi * D * esz;
    const uint32_t voff = (uint32_t)l * esz, roff = (uint32_t)row * esz;
    auto rsrc = [&](const void* p, uint32_t n) { return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)n, 0x00020000); };
    const __amdgpu_buffer_rsrc_t ra = rsrc(in.a, span), rw = rsrc(in.w, span), rk_ = rsrc(in.k, span),
                                 rb = rsrc(in.b, span), rr = rsrc(in.r, span), rv = rsrc(in.v, span);
    auto ld = [&](__amdgpu_buffer_rsrc_t rs, uint32_t vo, uint32_t so) -> E {
        if constexpr (sizeof(E) == 2) return (E)__builtin_amdgcn_raw_buffer_load_b16(rs, vo, so, 0);
        else return __builtin_bit_cast(E, __builtin_amdgcn_raw_buffer_load_b32(rs, vo, so, 0));
    };
    auto fetch = [&](E (&slot)[6], int t) __attribute__((always_inline)) {
        const uint32_t so = (uint32_t)min(t, T - 1) * strideT * esz;
        slot[0] = ld(ra, voff, so);
        slot[1] = ld(rw, voff, so);
        slot[2] = ld(rk_, voff, so);
        slot[3] = ld(rb, voff, so);
        slot[4] = ld(rr, voff, so);
        slot[5] = ld(rv, roff, so);
    };
    const uint32_t ospan = (uint32_t)T * strideT * 4u - (uint32_t)hi * D * 4u;
    const __amdgpu_buffer_rsrc_t ro_ = rsrc(outp, ospan), rs_ = rsrc(EMIT_SA ? sap : outp, ospan);
    const uint32_t orow = (uint32_t)row * 4u;
#pragma unroll
    for (int st = 0; st < 8; ++st) fetch(ring[st], st);

    float p = 0.0f;
    fwd_dot4(S[0], In::cvt(ring[0][0]), p);
    float y = 0.0f;   // partial y of the previous step, reduced and stored one step late

    auto step = [&](auto sc, int t, int c) __attribute__((always_inline)) {
        constexpr int s = decltype(sc)::value;
        __builtin_amdgcn_sched_barrier(0);
        fetch(ring[(s + 8) & (CH - 1)], t + 8);
        float sa = p;
        rowsum16_pair(sa, y);
        // y of step t - 1 (at t = 0 a placeholder at row 0, overwritten next
        // step); the sixteen lanes of a row store the same bits
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, y), ro_, orow,
                                              (uint32_t)max(t - 1, 0) * strideT * 4u, 0);
        y = 0.0f;
        p = 0.0f;
        const E* sl = ring[s];
        fwd_update4(S[s & 1], S[(s + 1) & 1], In::cvt(sl[2]), In::cvt(sl[3]), In::cvt(sl[1]), In::cvt(sl[4]),
                    In::cvt(ring[(s + 1) & (CH - 1)][0]), In::cvt(sl[5]), sa, y, p);
        const uint32_t so = (uint32_t)t * strideT * 4u;
        if constexpr (EMIT_SA) __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, sa), rs_, orow, so, 0);
        if constexpr (EMIT_CK && s == CH - 1) {
            *reinterpret_cast<float4*>(ckpt + ((int64_t)bh * NC + c) * D * D + (int64_t)row * D + 4 * g) =
                make_float4(S[0][0], S[0][1], S[0][2], S[0][3]);
        }
    };
    auto body = [&](int c, int n) __attribute__((always_inline)) {
        const int t0 = c * CH;
        [&]<int... s>(std::integer_sequence<int, s...>) {
            ((n > s ? step(std::integral_constant<int, s>{}, t0 + s, c) : void()), ...);
        }(std::make_integer_sequence<int, CH>{});
    };
    auto body_full = [&](int c) __attribute__((always_inline)) {
        const int t0 = c * CH;
        [&]<int... s>(std::integer_sequence<int, s...>) {
            (step(std::integral_constant<int, s>{}, t0 + s, c), ...);
        }(std::make_integer_sequence<int, CH>{});
    };
    if (NC > 0) body_full(0);
    for (int c = 1; c < NC; ++c) body_full(c);
    const int tail = T - NC * CH;
    if (tail) body(NC, tail);
    y = rowsum16(y);
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, y), ro_, orow, (uint32_t)(T - 1) * strideT * 4u, 0);

    const int fs = tail & 1;
    *reinterpret_cast<float4*>(h_out + sbase) = make_float4(S[fs][0], S[fs][1], S[fs][2], S[fs][3]);
}

// ─────────────────────────────── backward ───────────────────────────────
constexpr int BQ = 8;     // waves per head
constexpr int NVEC = 8;   // staged step vectors: r w k v a b dy sa
constexpr int NOUT = 6;   // dr dw dk db dv da

// Variant 2, the default.
//
// Eight waves per head.  Wave q holds the value rows 8q .. 8q + 7 of the state
// S and of dS (lane = key column), and the key columns 8q .. 8q + 7 of a second
// copy of dS (lane = value row): every sum is then a sum over registers, of the
// wave's eight rows or columns, and the waves' partials meet in LDS — dsa = dS·b
// in every step (the recurrence; one barrier per step), the six outputs a step
// later.  Lane l stands for element (l + 8q) mod 64, so lanes 0 .. 7 hold the
// wave's own rows' values of every step vector.
//
// The rank-1 updates and the sums over rows run on v_mfma_f32_4x4x1_16b_f32:
// its A operand, four lanes broadcast to all (cbsz 4), is four rows' values,
// its B operand 64 lanes.  One instruction (8 cycles) adds a row value ⊗ 64
// columns to four registers, twice the vector ALU's rate, or one register's
// share to two weighted sums, at its rate.  The fp32 matrix operations and the
// vector ALU do not run side by side, and changing between them costs about
// ten cycles, so a step keeps them in two groups (the scheduling barriers).
// A chunk's 17 states are in registers (136 of 234), computed once: two windows
// of eight steps repeat half of them.
//
// What bounds it: with 256 heads, one per CU, mostly the issue of both waves of
// a SIMD (0.35 of its cycles matrix, 0.29 vector instructions; loading the next
// step's vectors early changes nothing), then the step's exchange through LDS.  8 × 4096 × 32 heads, bf16: 3.9 ms with the
// vector ALU alone, whose products all take a broadcast operand, 3.0 ms so.  Four waves
// of 16 rows (one per SIMD, half the LDS traffic): 4.7 ms.
using f32x4 = __attribute__((ext_vector_type(4))) float;

// c + a[4·BLK .. 4·BLK + 3] ⊗ b: register r, lane l: lane 4·BLK + r of `a` times b's lane l.
template <int BLK>
__device__ __forceinline__ f32x4 outer4(float a, float b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_4x4x1f32(a, b, c, 4, BLK, 0);
}
// A matrix's eight rows (or columns) of the wave as registers.
struct Rows8 {
    f32x4 lo, hi;
};
__device__ __forceinline__ Rows8 outer8(float a, float b, const Rows8& c) {
    return {outer4<0>(a, b, c.lo), outer4<1>(a, b, c.hi)};
}
// Σ_j X0[j]·M_j and Σ_j X1[j]·M_j: X's lane 2j + x holds X_x[j].
struct Pair {
    float x0, x1;
};
__device__ __forceinline__ Pair dots8(float X, const Rows8& M) {
    f32x4 e = {0.f, 0.f, 0.f, 0.f}, o = {0.f, 0.f, 0.f, 0.f};
    e = outer4<0>(X, M.lo[0], e);
    o = outer4<0>(X, M.lo[1], o);
    e = outer4<1>(X, M.lo[2], e);
    o = outer4<1>(X, M.lo[3], o);
    e = outer4<2>(X, M.hi[0], e);
    o = outer4<2>(X, M.hi[1], o);
    e = outer4<3>(X, M.hi[2], e);
    o = outer4<3>(X, M.hi[3], o);
    return {e[0] + o[2], e[1] + o[3]};
}

// W_j·M_j, W's lane ≡ j (mod 8) of every 16-lane row (not inline assembly: the
// compiler places the wait between the matrix cores' write of M and this read).
template <int J>
__device__ __forceinline__ float bcast(float x) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x150 + J, 0xf, 0xf, true));
}
__device__ __forceinline__ Rows8 scale8(float W, const Rows8& M) {
    return {{bcast<0>(W) * M.lo[0], bcast<1>(W) * M.lo[1], bcast<2>(W) * M.lo[2], bcast<3>(W) * M.lo[3]},
            {bcast<4>(W) * M.hi[0], bcast<5>(W) * M.hi[1], bcast<6>(W) * M.hi[2], bcast<7>(W) * M.hi[3]}};
}

// The 8 waves' partials of one element (stride D floats), and their sum, pairwise.
struct Parts {
    float x[8];
    __device__ __forceinline__ explicit Parts(const float* p) {
#pragma unroll
        for (int i = 0; i < 8; ++i) x[i] = p[i * D];
    }
    __device__ __forceinline__ float sum() const {
        return ((x[0] + x[1]) + (x[2] + x[3])) + ((x[4] + x[5]) + (x[6] + x[7]));
    }
};

template <int DT, int GT>
__global__ __launch_bounds__(512) void wkv7_bwd_kernel(
    const void* __restrict__ r, const void* __restrict__ w, const void* __restrict__ k,
    const void* __restrict__ v, const void* __restrict__ a, const void* __restrict__ b,
    const float* __restrict__ h_in, const float* __restrict__ ckpt, const float* __restrict__ sa,
    const float* __restrict__ dout, const float* __restrict__ dhout, void* __restrict__ g_dr,
    void* __restrict__ g_dw, void* __restrict__ g_dk, void* __restrict__ g_dv, void* __restrict__ g_da,
    void* __restrict__ g_db, float* __restrict__ dh_in, int T, int H) {
    __shared__ float stage[2][NVEC][CH][D];        // step vectors of a chunk, fp32
    __shared__ float dsa_part[2][BQ][D];           // [parity][wave][row]
    __shared__ float ring[4][NOUT][BQ][D];         // output partials of the last steps

    const int tid = threadIdx.x;
    const int l = tid & 63;
    const int q = __builtin_amdgcn_readfirstlane(tid >> 6);    // rows (columns) 8q .. 8q+7
    const uint32_t e = (l + 8 * q) & 63;                       // the lane's element
    const int jw = 8 * q + (l & 7);                            // scale8's row
    const int jx = 8 * q + ((l >> 1) & 7);                     // dots8's row
    const bool odd = l & 1;
    const int bh = blockIdx.x;
    const int bi = bh / H, hi = bh - bi * H;
    const int64_t strideT = (int64_t)H * D;
    const int64_t base0 = ((int64_t)bi * T * H + hi) * D;
    const int64_t hb = (int64_t)bh * D * D;
    const int NC = T / CH;

    // chunk staging: thread covers 16 floats of the chunk's 8 × 16 × 64 block
    float stg[16];
    const uint32_t so = (uint32_t)((tid >> 6) * strideT + l), so8 = (uint32_t)(8 * strideT);
    auto stage_load = [&](int c) {
        const int64_t off = base0 + c * CH * strideT;
#pragma unroll
        for (int m = 0; m < 16; ++m) {   // vector m / 2, step 8·(m % 2) + wave
            const uint32_t o = so + (m & 1) * so8;
            switch (m >> 1) {
                case 0: stg[m] = load1<DT>(at<DT>(r, off), o); break;
                case 1: stg[m] = load1<DT>(at<DT>(w, off), o); break;
                case 2: stg[m] = load1<DT>(at<DT>(k, off), o); break;
                case 3: stg[m] = load1<DT>(at<DT>(v, off), o); break;
                case 4: stg[m] = load1<DT>(at<DT>(a, off), o); break;
                case 5: stg[m] = load1<DT>(at<DT>(b, off), o); break;
                case 6: stg[m] = (dout + off)[o]; break;
                default: stg[m] = (sa + off)[o];
            }
        }
    };
    auto stage_store = [&](int c) {
#pragma unroll
        for (int m = 0; m < 16; ++m) stage[c & 1][m >> 1][8 * (m & 1) + (tid >> 6)][l] = stg[m];
    };

    Rows8 dT, dR;   // dS[8q + j, e] and dS[e, 8q + j]
    const Rows8 zero = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
    dT = dR = zero;
    if (dhout) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            dT.lo[j] = dhout[hb + (int64_t)(8 * q + j) * D + e];
            dT.hi[j] = dhout[hb + (int64_t)(8 * q + 4 + j) * D + e];
        }
        dR.lo = *reinterpret_cast<const f32x4*>(dhout + hb + (int64_t)e * D + 8 * q);
        dR.hi = *reinterpret_cast<const f32x4*>(dhout + hb + (int64_t)e * D + 8 * q + 4);
    }

    // the state before a chunk, loaded a chunk ahead
    auto load_state = [&](int c) __attribute__((always_inline)) {
        const float* const src = c > 0 ? ckpt + hb * NC + (int64_t)(c - 1) * D * D : h_in ? h_in + hb : nullptr;
        Rows8 S = zero;
        if (src) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                S.lo[j] = (src + 8 * q * D)[j * D + e];
                S.hi[j] = (src + 8 * q * D)[(4 + j) * D + e];
            }
        }
        return S;
    };
    Rows8 Sst = load_state(NC - 1);
    stage_load(NC - 1);
    stage_store(NC - 1);

    // Outputs of the step in a ring slot: 6 × 64 sums of 8 partials, 48 per
    // wave so every wave carries the same share between two barriers; the
    // steps go out last to first, so the lane's address moves down by one.
    const int fidx = q * (NOUT * D / BQ) + min(l, NOUT * D / BQ - 1);   // output index owned by this lane (l < 48)
    const int fo = fidx >> 6, fcol = fidx & 63;
    constexpr int64_t gsz = GT == RWKV_F32 ? 4 : 2;
    char* fout = reinterpret_cast<char*>(fo == 0 ? g_dr : fo == 1 ? g_dw : fo == 2 ? g_dk : fo == 3 ? g_db : fo == 4 ? g_dv : g_da) +
                 (base0 + (T - 1) * strideT + fcol) * gsz;
    auto flush = [&](const Parts& p) __attribute__((always_inline)) {
        if (l < NOUT * D / BQ) store1<GT>(fout, 0, p.sum());
        fout -= strideT * gsz;
    };
    auto flush_parts = [&](int slot) __attribute__((always_inline)) { return Parts(&ring[slot][fo][0][fcol]); };

    for (int c = NC - 1; c >= 0; --c) {
        __syncthreads();   // chunk c staged; every read of the other buffer is done
        if (c > 0) stage_load(c - 1);
        const float (*st)[CH][D] = stage[c & 1];

        // the forward's state update: fma(w, S, fma(sa, b, v·k))
        auto advance = [&](int s, const Rows8& S) __attribute__((always_inline)) {
            const Rows8 n = outer8(st[7][s][e], st[5][s][e], outer8(st[3][s][e], st[2][s][e], zero));
            const float wi = st[1][s][e];
            return Rows8{S.lo * wi + n.lo, S.hi * wi + n.hi};
        };
        Rows8 h[CH + 1];   // h[s] = state before step s of the chunk
        h[0] = Sst;
#pragma unroll
        for (int s = 0; s < CH; ++s) h[s + 1] = advance(s, h[s]);
        if (c > 0) Sst = load_state(c - 1);
        float dr = dots8(st[6][CH - 1][jx], h[CH]).x0;   // the coming step's dr partial
#pragma unroll
        for (int s = CH - 1; s >= 0; --s) {
            const int par = s & 1, slot = s & 3;
            const float re = st[0][s][e], we = st[1][s][e], ae = st[4][s][e], dye = st[6][s][e];
            const float bk = st[odd ? 2 : 5][s][jx], vs = st[odd ? 7 : 3][s][jx], wj = st[1][s][jw];
            // dS gains dy rᵀ; the wave's columns' share of dsa (and dv) and, from its rows, dk and db
            dR = outer8(re, dye, dR);
            dT = outer8(dye, re, dT);
            __builtin_amdgcn_sched_barrier(0);
            const Pair ds_dv = dots8(bk, dR);
            const Pair kb = dots8(vs, dT);
            __builtin_amdgcn_sched_barrier(0);
            dsa_part[par][q][e] = ds_dv.x0;
            const Rows8 tR = scale8(wj, dR);
            const f32x4 pw = dT.lo * h[s].lo + dT.hi * h[s].hi;
            ring[slot][0][q][e] = dr;
            ring[slot][1][q][e] = (pw[0] + pw[1]) + (pw[2] + pw[3]);
            ring[slot][2][q][e] = kb.x0;
            ring[slot][3][q][e] = kb.x1;
            ring[slot][4][q][e] = ds_dv.x1;
            const Rows8 tT = {dT.lo * we, dT.hi * we};
            const float dyx = st[6][s > 0 ? s - 1 : 0][jx];
            __syncthreads();
            const Parts pd(&dsa_part[par][0][e]), pf = flush_parts((s + 1) & 3);
            const float dsa = pd.sum();
            const float dsx = __shfl(dsa, (l >> 1) & 7, 64);
            __builtin_amdgcn_sched_barrier(0);
            dR = outer8(ae, dsa, tR);
            dT = outer8(dsa, ae, tT);
            const Pair ar = dots8(odd ? dyx : dsx, h[s]);
            __builtin_amdgcn_sched_barrier(0);
            ring[slot][5][q][e] = ar.x0;
            dr = ar.x1;
            if (s < CH - 1 || c < NC - 1) flush(pf);   // the step after this one's
        }
        if (c > 0) stage_store(c - 1);
    }
    __syncthreads();
    flush(flush_parts(0));
    *reinterpret_cast<f32x4*>(dh_in + hb + (int64_t)e * D + 8 * q) = dR.lo;
    *reinterpret_cast<f32x4*>(dh_in + hb + (int64_t)e * D + 8 * q + 4) = dR.hi;
}

// ─────────────────────────────── backward, row-owned (variant 1) ───────────────────────────────
// The scheme of ckptBwdKernel (WKV7Train.swift:99-205): one wave per (b, h),
// lane i owns value row i of the state S and of its gradient C = dL/dS, both
// in VGPRs.  Each chunk starts from the state after it (the checkpoint) and
// walks its steps backward, recovering the state before a step by dividing
// by w: S_{t-1} = (S_t − v kᵀ − sa bᵀ) ⊘ w.  Per step (t descending)
//   C += dy rᵀ;  dsa = C b;  dv = C k
//   dr = S_tᵀ dy;  dw = Σ_i C ⊙ S_{t-1};  dk = Cᵀ v;  da = S_{t-1}ᵀ dsa;  db = Cᵀ sa
//   C ← C diag(w) + dsa aᵀ
// The column sums (over the lanes' rows, in row order) go through one LDS
// transpose per step: every lane writes its row of the five products as a
// column, lane j sums row j (16-byte reads).  A chunk's step vectors (and 1/w) are staged in LDS;
// the next chunk's values and checkpoint row are loaded while this one runs.
// Dividing by w amplifies the forward's rounding by up to Π 1/w over a chunk,
// the reason the default (variant 2) recomputes the states instead.
constexpr int kBwdRowsTS = D + 4;   // LDS row stride of the transposed products (16-byte rows)
constexpr int kBwdRowsLds = (CH * 8 * D + 5 * D * kBwdRowsTS) * 4;   // bytes of LDS

template <int DT, int GT>
__global__ __launch_bounds__(64) void wkv7_bwd_rows_kernel(
    const void* __restrict__ r, const void* __restrict__ w, const void* __restrict__ k,
    const void* __restrict__ v, const void* __restrict__ a, const void* __restrict__ b,
    const float* __restrict__ h_ckpt, const float* __restrict__ sa, const float* __restrict__ d_out,
    const float* __restrict__ d_h_out, void* __restrict__ dr, void* __restrict__ dw, void* __restrict__ dk,
    void* __restrict__ dv, void* __restrict__ da, void* __restrict__ db, float* __restrict__ dh_in, int T, int H) {
    extern __shared__ __attribute__((aligned(16))) float lds[];
    float* sv = lds;                   // [CH][8][64]: r, w, k, a, b, 1/w, v, sa of the chunk's steps
    float* acc = lds + CH * 8 * D;     // [5][64][68]: the five products transposed (column j of lane i's row at [j][i])
    constexpr int TS = kBwdRowsTS, AS = D * TS;   // row stride, floats per product matrix
    const int i = threadIdx.x;
    const int bh = blockIdx.x, bi = bh / H, hi = bh - bi * H;
    const int NC = T / CH;
    auto elem = [&](int c, int t) { return (((int64_t)bi * T + (int64_t)c * CH + t) * H + hi) * D + i; };
    const int64_t hb = (int64_t)bh * D * D + (int64_t)i * D;

    float C[D], hr[D];
#pragma unroll
    for (int q = 0; q < D / 4; ++q) {
        const float4 f = d_h_out ? reinterpret_cast<const float4*>(d_h_out + hb)[q] : make_float4(0.f, 0.f, 0.f, 0.f);
        C[4 * q] = f.x; C[4 * q + 1] = f.y; C[4 * q + 2] = f.z; C[4 * q + 3] = f.w;
    }
    // the chunk's per-lane values: r, w, k, a, b, v, sa, dy per step, and its
    // checkpoint row; fetched one chunk ahead (clamped at chunk 0: its values
    // again, unused)
    float pf[CH][8];
    float4 ph[D / 4];
    auto fetch = [&](int c) {
#pragma unroll
        for (int t = 0; t < CH; ++t) {
            const int64_t e = elem(c, t);
            pf[t][0] = load1<DT>(r, e);
            pf[t][1] = load1<DT>(w, e);
            pf[t][2] = load1<DT>(k, e);
            pf[t][3] = load1<DT>(a, e);
            pf[t][4] = load1<DT>(b, e);
            pf[t][5] = load1<DT>(v, e);
            pf[t][6] = sa[e];
            pf[t][7] = d_out[e];
        }
        const float4* src = reinterpret_cast<const float4*>(h_ckpt + ((int64_t)bh * NC + c) * D * D + (int64_t)i * D);
#pragma unroll
        for (int q = 0; q < D / 4; ++q) ph[q] = src[q];
    };
    fetch(NC - 1);
    for (int c = NC - 1; c >= 0; --c) {
        float dyc[CH];
#pragma unroll
        for (int t = 0; t < CH; ++t) {
            float* V = sv + t * 8 * D;
            V[0 * D + i] = pf[t][0];
            V[1 * D + i] = pf[t][1];
            V[2 * D + i] = pf[t][2];
            V[3 * D + i] = pf[t][3];
            V[4 * D + i] = pf[t][4];
            V[5 * D + i] = 1.0f / pf[t][1];
            V[6 * D + i] = pf[t][5];
            V[7 * D + i] = pf[t][6];
            dyc[t] = pf[t][7];
        }
#pragma unroll
        for (int q = 0; q < D / 4; ++q) {
            hr[4 * q] = ph[q].x; hr[4 * q + 1] = ph[q].y; hr[4 * q + 2] = ph[q].z; hr[4 * q + 3] = ph[q].w;
        }
        fetch(max(c - 1, 0));
        __syncthreads();
#pragma unroll 1
        for (int t = CH - 1; t >= 0; --t) {
            const float* V = sv + t * 8 * D;
            // the step vectors are the same for every lane: 16-byte broadcast reads
            const float4* V4 = reinterpret_cast<const float4*>(V);
            auto vec = [&](int q, int j4) { return V4[q * (D / 4) + j4]; };
            const float dy = dyc[t], vi = V[6 * D + i], sai = V[7 * D + i];
#pragma unroll
            for (int j4 = 0; j4 < D / 4; ++j4) {
                const float4 rr = vec(0, j4);
                C[4 * j4] = fmaf(dy, rr.x, C[4 * j4]);
                C[4 * j4 + 1] = fmaf(dy, rr.y, C[4 * j4 + 1]);
                C[4 * j4 + 2] = fmaf(dy, rr.z, C[4 * j4 + 2]);
                C[4 * j4 + 3] = fmaf(dy, rr.w, C[4 * j4 + 3]);
            }
            float dsa = 0.0f, dvv = 0.0f;
#pragma unroll
            for (int j4 = 0; j4 < D / 4; ++j4) {
                const float4 bb = vec(4, j4), kk = vec(2, j4);
                dsa = fmaf(C[4 * j4], bb.x, dsa);
                dvv = fmaf(C[4 * j4], kk.x, dvv);
                dsa = fmaf(C[4 * j4 + 1], bb.y, dsa);
                dvv = fmaf(C[4 * j4 + 1], kk.y, dvv);
                dsa = fmaf(C[4 * j4 + 2], bb.z, dsa);
                dvv = fmaf(C[4 * j4 + 2], kk.z, dvv);
                dsa = fmaf(C[4 * j4 + 3], bb.w, dsa);
                dvv = fmaf(C[4 * j4 + 3], kk.w, dvv);
            }
            const int64_t e = elem(c, t);
            store1<GT>(dv, e, dvv);
            float* col = acc + i;   // lane i writes element i of every transposed row
#pragma unroll
            for (int j4 = 0; j4 < D / 4; ++j4) {
                const float4 kk = vec(2, j4), bb = vec(4, j4), iw = vec(5, j4);
                const float kv[4] = {kk.x, kk.y, kk.z, kk.w}, bv[4] = {bb.x, bb.y, bb.z, bb.w};
                const float wv[4] = {iw.x, iw.y, iw.z, iw.w};
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const int j = 4 * j4 + u;
                    col[j * TS] = dy * hr[j];
                    hr[j] = (hr[j] - vi * kv[u] - sai * bv[u]) * wv[u];
                    col[AS + j * TS] = C[j] * hr[j];
                    col[2 * AS + j * TS] = C[j] * vi;
                    col[3 * AS + j * TS] = dsa * hr[j];
                    col[4 * AS + j * TS] = sai * C[j];
                }
            }
            __syncthreads();
            // column i of each product is row i of its transpose: 16-byte
            // reads, summed over the lanes' rows in order
            float gs[5] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int m = 0; m < 5; ++m) {
                const float4* tr = reinterpret_cast<const float4*>(acc + m * AS + i * TS);
#pragma unroll
                for (int s4 = 0; s4 < D / 4; ++s4) {
                    const float4 f = tr[s4];
                    gs[m] += f.x;
                    gs[m] += f.y;
                    gs[m] += f.z;
                    gs[m] += f.w;
                }
            }
            store1<GT>(dr, e, gs[0]);
            store1<GT>(dw, e, gs[1]);
            store1<GT>(dk, e, gs[2]);
            store1<GT>(da, e, gs[3]);
            store1<GT>(db, e, gs[4]);
#pragma unroll
            for (int j4 = 0; j4 < D / 4; ++j4) {
                const float4 ww = vec(1, j4), aa = vec(3, j4);
                C[4 * j4] = fmaf(C[4 * j4], ww.x, dsa * aa.x);
                C[4 * j4 + 1] = fmaf(C[4 * j4 + 1], ww.y, dsa * aa.y);
                C[4 * j4 + 2] = fmaf(C[4 * j4 + 2], ww.z, dsa * aa.z);
                C[4 * j4 + 3] = fmaf(C[4 * j4 + 3], ww.w, dsa * aa.w);
            }
            __syncthreads();
        }
    }
#pragma unroll
    for (int q = 0; q < D / 4; ++q)
        reinterpret_cast<float4*>(dh_in + hb)[q] = make_float4(C[4 * q], C[4 * q + 1], C[4 * q + 2], C[4 * q + 3]);
}

// ─────────────────────────────── tmix tail ───────────────────────────────

// y·g rounded to fp32, then converted to TO: for fp16 the fp32 output's
// value rounded once more.  The empty asm keeps the fp32 product: without it
// the compiler folds multiply and conversion into one v_fma_mixlo_f16, which
// rounds the exact product straight to fp16.
template <typename TO>
__device__ __forceinline__ TO tail_out(float y, float g) {
    float o = y * g;
    asm("" : "+v"(o));
    return (TO)o;
}

// One wave per (row, head), four to a workgroup; the output fp32, or fp16
// (TO = _Float16: the rounding the fp16 long pass of o_proj applies to its
// input, so the projection reads the same values from half the bytes).
template <typename TO>
__global__ __launch_bounds__(256) void wkv_tail_kernel(
    const float* __restrict__ wkv, const float* __restrict__ r, const float* __restrict__ k,
    const float* __restrict__ v, const float* __restrict__ rk, const float* __restrict__ lnw,
    const float* __restrict__ lnb, const float* __restrict__ g, TO* __restrict__ out,
    int NH, int H, int S, float eps) {
    const int tg = blockIdx.x * 4 + (threadIdx.x >> 6);   // row * H + head
    if (tg >= NH) return;   // whole waves; no barrier below
    const int h = tg % H;
    const int64_t base = (int64_t)tg * S, hb = (int64_t)h * S;
    const int lane = threadIdx.x & 63;
    if (S == 64) {
        // one element per lane, every load issued up front; the operations
        // of the loops below for their single pass, so the same bits
        const int64_t i = base + lane, j = hb + lane;
        const float wv = wkv[i], rv = r[i], kv = k[i], vv = v[i], gv = g[i];
        const float rkv = rk[j], lw = lnw[j], lb = lnb[j];
        float t1 = 0.0f;
        t1 += wv;
        const float mean = wave_total(t1) / 64.0f;
        const float d = wv - mean;
        const float inv = 1.0f / sqrtf(wave_total(fmaf(d, d, 0.0f)) / 64.0f + eps);
        const float dp = wave_total(fmaf(rv * kv, rkv, 0.0f));
        const float y = fmaf(dp, vv, fmaf((wv - mean) * inv, lw, lb));
        out[i] = tail_out<TO>(y, gv);
        return;
    }
    float s1 = 0.0f;
    for (int e = lane; e < S; e += 64) s1 += wkv[base + e];
    const float mean = wave_total(s1) / (float)S;
    float s2 = 0.0f;
    for (int e = lane; e < S; e += 64) {
        const float d = wkv[base + e] - mean;
        s2 = fmaf(d, d, s2);
    }
    const float inv = 1.0f / sqrtf(wave_total(s2) / (float)S + eps);
    float dp = 0.0f;
    for (int e = lane; e < S; e += 64) dp = fmaf(r[base + e] * k[base + e], rk[hb + e], dp);
    dp = wave_total(dp);
    for (int e = lane; e < S; e += 64) {
        const float nrm = (wkv[base + e] - mean) * inv;
        const float y = fmaf(dp, v[base + e], fmaf(nrm, lnw[hb + e], lnb[hb + e]));
        out[base + e] = tail_out<TO>(y, g[base + e]);
    }
}

// ─────────────────────────────── decode: step + tail in one launch ───────────────────────────────
// One workgroup per (row, head): four waves (sixteen-row layout) or sixteen
// (four-row layout, B·H < 256), each the T = 1 path of the forward kernel for
// its rows (head_step16 / head_step4: the same operations, so state and wkv
// are bitwise those of rwkv_wkv7_step); the head's 64 wkv values meet in LDS
// and wave 0 applies the tail with wkv_tail_kernel's operation sequence for
// S = 64 (head_tail).
template <bool R4>
__global__ __launch_bounds__(R4 ? 1024 : 256) void wkv7_step_tail_kernel(
    const float* __restrict__ r, const float* __restrict__ w, const float* __restrict__ k,
    const float* __restrict__ v, const float* __restrict__ a, const float* __restrict__ b,
    const float* __restrict__ h_in, float* __restrict__ h_out, const float* __restrict__ rk,
    const float* __restrict__ lnw, const float* __restrict__ lnb, const float* __restrict__ g,
    float* __restrict__ wkv_out, float* __restrict__ out, int H, float eps) {
    __shared__ float ys[D];
    const int blk = threadIdx.x >> 6, l = threadIdx.x & 63;
    const int bh = blockIdx.x;
    const int hi = bh % H;
    const int64_t base0 = (int64_t)bh * D;   // [B, H, 64]
    const int64_t hb = (int64_t)bh * D * D;
    const int row = R4 ? step4_row(blk, l) : step16_row(blk, l);
    const float A = a[base0 + l], W = w[base0 + l], K = k[base0 + l], Bv = b[base0 + l];
    const float R = r[base0 + l], V = v[base0 + row];
    const float* hin = h_in ? h_in + hb : nullptr;
    float S[R4 ? 4 : 16];
    if constexpr (R4) load_state4(hin, blk, l, S);
    else load_state16(hin, blk, l, S);
    // the tail's other inputs (wave 0; r and k of column l are R and K) do not
    // depend on the step: loaded with the state, not after the barrier
    const int64_t e = base0 + l, he = (int64_t)hi * D + l;
    float tv = 0.0f, trk = 0.0f, tlnw = 0.0f, tlnb = 0.0f, tg = 0.0f;
    if (blk == 0) {   // uniform per wave
        tv = v[e];
        trk = rk[he];
        tlnw = lnw[he];
        tlnb = lnb[he];
        tg = g[e];
    }
    float y;
    if constexpr (R4) y = head_step4_regs(S, h_out + hb, blk, l, A, W, K, Bv, R, V);
    else y = head_step16_regs(S, h_out + hb, blk, l, A, W, K, Bv, R, V);
    if ((R4 ? (l >> 2) : (l >> 4)) == 0) {
        ys[row] = y;
        if (wkv_out) wkv_out[base0 + row] = y;
    }
    __syncthreads();
    if (blk == 0) out[e] = head_tail(ys[l], R, K, tv, trk, tlnw, tlnb, tg, eps);
}

// ─────────────────────────────── host dispatch ───────────────────────────────
rwkv_status launch_status(const char* what) {
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        rwkv::set_error("%s: %s", what, hipGetErrorString(e));
        return RWKV_E_HIP;
    }
    rwkv::clear_error();
    return RWKV_OK;
}

template <bool SA, bool CK>
rwkv_status launch_fwd(const void* r, const void* w, const void* k, const void* v, const void* a, const void* b,
                       rwkv_dtype dt, const float* h_in, float* out, float* h_out, float* sa_out, float* ck,
                       int64_t B, int64_t T, int64_t H, void* stream) {
    const bool rows4 = use_rows4(B * H);
    dim3 grid((unsigned)(B * H * (rows4 ? 16 : 4))), block(64);   // one wave per 4 / 16 value rows
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
#define RWKV_FWD(DTV)                                                                                        \
    if (rows4)                                                                                               \
        rwkv::launch(wkv7_fwd4_kernel<DTV, SA, CK>, grid, block, st, r, w, k, v, a, b, h_in, out, h_out, sa_out, \
                     ck, (int)T, (int)H);                                                                    \
    else                                                                                                     \
        rwkv::launch(wkv7_fwd_kernel<DTV, SA, CK>, grid, block, st, r, w, k, v, a, b, h_in, out, h_out, sa_out,  \
                     ck, (int)T, (int)H)
    switch (dt) {
        case RWKV_F32: RWKV_FWD(RWKV_F32); break;
        case RWKV_BF16: RWKV_FWD(RWKV_BF16); break;
        case RWKV_F16: RWKV_FWD(RWKV_F16); break;
    }
#undef RWKV_FWD
    return launch_status("wkv7 forward launch");
}

rwkv_status check_wkv_common(const void* r, const void* w, const void* k, const void* v, const void* a,
                             const void* b, int dt, int64_t B, int64_t T, int64_t H) {
    RWKV_REQUIRE(r && w && k && v && a && b, RWKV_E_NULL, "wkv7: r/w/k/v/a/b must be non-null");
    RWKV_REQUIRE(rwkv::dtype_ok(dt), RWKV_E_DTYPE, "wkv7: input dtype code %d not in {f32, bf16, f16}", dt);
    RWKV_REQUIRE(B >= 1 && H >= 1, RWKV_E_SHAPE, "wkv7: B (%lld) and H (%lld) must be >= 1", (long long)B, (long long)H);
    RWKV_REQUIRE(T >= 1, RWKV_E_SHAPE, "wkv7: T (%lld) must be >= 1", (long long)T);
    RWKV_REQUIRE(B * H * 4 <= INT32_MAX && T * H * 64 * 4 < ((int64_t)1 << 32) && B * T * H * 64 <= (int64_t)1 << 46,
                 RWKV_E_SHAPE, "wkv7: B·T·H too large (one sequence must stay under 2^32 bytes)");
    return RWKV_OK;
}

}  // namespace

extern "C" {

int rwkv_wkv7_head_size(void) { return D; }
int rwkv_wkv7_chunk(void) { return CH; }

rwkv_status rwkv_wkv7_seq_fwd(const void* r, const void* w, const void* k, const void* v, const void* a,
                              const void* b, rwkv_dtype in_dt, const float* h_in, float* out, float* h_out,
                              int64_t B, int64_t T, int64_t H, void* stream) {
    rwkv_status s = check_wkv_common(r, w, k, v, a, b, in_dt, B, T, H);
    if (s != RWKV_OK) return s;
    RWKV_REQUIRE(out && h_out, RWKV_E_NULL, "wkv7_seq_fwd: out and h_out must be non-null");
    s = launch_fwd<false, false>(r, w, k, v, a, b, in_dt, h_in, out, h_out, nullptr, nullptr, B, T, H, stream);
    if (s == RWKV_OK) rwkv::counters().seq_fwd++;
    return s;
}

rwkv_status rwkv_wkv7_chunk_fwd(const void* r, const void* w, const void* k, const void* v, const void* a,
                                const void* b, rwkv_dtype in_dt, const float* h_in, float* out, float* h_out,
                                float* sa_out, int64_t B, int64_t T, int64_t H, void* stream) {
    rwkv_status s = check_wkv_common(r, w, k, v, a, b, in_dt, B, T, H);
    if (s != RWKV_OK) return s;
    RWKV_REQUIRE(T == CH, RWKV_E_SHAPE, "wkv7_chunk_fwd: T (%lld) must equal CHUNK %d", (long long)T, CH);
    RWKV_REQUIRE(h_in && out && h_out && sa_out, RWKV_E_NULL, "wkv7_chunk_fwd: h_in/out/h_out/sa_out must be non-null");
    s = launch_fwd<true, false>(r, w, k, v, a, b, in_dt, h_in, out, h_out, sa_out, nullptr, B, T, H, stream);
    if (s == RWKV_OK) rwkv::counters().chunk_fwd++;
    return s;
}

rwkv_status rwkv_wkv7_train_fwd(const void* r, const void* w, const void* k, const void* v, const void* a,
                                const void* b, rwkv_dtype in_dt, const float* h_in, float* out, float* h_out,
                                float* sa_out, float* h_ckpt, int64_t B, int64_t T, int64_t H, void* stream) {
    rwkv_status s = check_wkv_common(r, w, k, v, a, b, in_dt, B, T, H);
    if (s != RWKV_OK) return s;
    RWKV_REQUIRE(T % CH == 0, RWKV_E_SHAPE, "wkv7_train_fwd: T (%lld) must be a multiple of CHUNK %d", (long long)T, CH);
    RWKV_REQUIRE(out && h_out && sa_out && h_ckpt, RWKV_E_NULL, "wkv7_train_fwd: out/h_out/sa_out/h_ckpt must be non-null");
    s = launch_fwd<true, true>(r, w, k, v, a, b, in_dt, h_in, out, h_out, sa_out, h_ckpt, B, T, H, stream);
    if (s == RWKV_OK) rwkv::counters().train_fwd++;
    return s;
}

rwkv_status rwkv_wkv7_step(const void* r, const void* w, const void* k, const void* v, const void* a,
                           const void* b, rwkv_dtype in_dt, const float* h_in, float* out, float* h_out,
                           int64_t B, int64_t H, void* stream) {
    rwkv_status s = check_wkv_common(r, w, k, v, a, b, in_dt, B, 1, H);
    if (s != RWKV_OK) return s;
    RWKV_REQUIRE(out && h_out, RWKV_E_NULL, "wkv7_step: out and h_out must be non-null");
    s = launch_fwd<false, false>(r, w, k, v, a, b, in_dt, h_in, out, h_out, nullptr, nullptr, B, 1, H, stream);
    if (s == RWKV_OK) rwkv::counters().step++;
    return s;
}

rwkv_status rwkv_wkv7_train_bwd(const void* r, const void* w, const void* k, const void* v, const void* a,
                                const void* b, rwkv_dtype in_dt, const float* h_in, const float* h_ckpt,
                                const float* sa, const float* d_out, const float* d_h_out, void* dr, void* dw,
                                void* dk, void* dv, void* da, void* db, rwkv_dtype g_dt, float* dh_in, int64_t B,
                                int64_t T, int64_t H, int variant, void* stream) {
    rwkv_status s = check_wkv_common(r, w, k, v, a, b, in_dt, B, T, H);
    if (s != RWKV_OK) return s;
    RWKV_REQUIRE(T % CH == 0, RWKV_E_SHAPE, "wkv7_train_bwd: T (%lld) must be a multiple of CHUNK %d", (long long)T, CH);
    RWKV_REQUIRE(h_ckpt && sa && d_out && dr && dw && dk && dv && da && db && dh_in, RWKV_E_NULL,
                 "wkv7_train_bwd: checkpoints, sa, d_out, gradients and dh_in must be non-null");
    RWKV_REQUIRE(rwkv::dtype_ok(g_dt), RWKV_E_DTYPE, "wkv7_train_bwd: gradient dtype code %d not in {f32, bf16, f16}", g_dt);
    RWKV_REQUIRE(variant == 1 || variant == 2, RWKV_E_UNSUPPORTED, "wkv7_train_bwd: variant %d not in {1, 2}", variant);
    dim3 grid((unsigned)(B * H)), block(512);
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
#define RWKV_BWD_LAUNCH(DT, GT)                                                                          \
    rwkv::launch(wkv7_bwd_kernel<DT, GT>, grid, block, st, r, w, k, v, a, b, h_in, h_ckpt, sa, \
                       d_out, d_h_out, dr, dw, dk, dv, da, db, dh_in, (int)T, (int)H)
#define RWKV_BWD_GT(DT)                                         \
    switch (g_dt) {                                                  \
        case RWKV_F32: RWKV_BWD_LAUNCH(DT, RWKV_F32); break;   \
        case RWKV_BF16: RWKV_BWD_LAUNCH(DT, RWKV_BF16); break; \
        case RWKV_F16: RWKV_BWD_LAUNCH(DT, RWKV_F16); break;   \
    }
#define RWKV_BWD_DT()                                  \
    switch (in_dt) {                                      \
        case RWKV_F32: RWKV_BWD_GT(RWKV_F32); break;   \
        case RWKV_BF16: RWKV_BWD_GT(RWKV_BF16); break; \
        case RWKV_F16: RWKV_BWD_GT(RWKV_F16); break;   \
    }
#define RWKV_ROWS_LAUNCH(DT, GT)                                                                              \
    rwkv::launch_lds(wkv7_bwd_rows_kernel<DT, GT>, dim3((unsigned)(B * H)), dim3(64), (size_t)kBwdRowsLds, st, r, \
                     w, k, v, a, b, h_ckpt, sa, d_out, d_h_out, dr, dw, dk, dv, da, db, dh_in, (int)T, (int)H)
#define RWKV_ROWS_GT(DT)                                           \
    switch (g_dt) {                                                \
        case RWKV_F32: RWKV_ROWS_LAUNCH(DT, RWKV_F32); break;   \
        case RWKV_BF16: RWKV_ROWS_LAUNCH(DT, RWKV_BF16); break; \
        case RWKV_F16: RWKV_ROWS_LAUNCH(DT, RWKV_F16); break;   \
    }
    if (variant == 2) {
        RWKV_BWD_DT()
    } else {
        switch (in_dt) {
            case RWKV_F32: RWKV_ROWS_GT(RWKV_F32); break;
            case RWKV_BF16: RWKV_ROWS_GT(RWKV_BF16); break;
            case RWKV_F16: RWKV_ROWS_GT(RWKV_F16); break;
        }
    }
#undef RWKV_ROWS_GT
#undef RWKV_ROWS_LAUNCH
#undef RWKV_BWD_DT
#undef RWKV_BWD_GT
#undef RWKV_BWD_LAUNCH
    s = launch_status("wkv7 backward launch");
    if (s == RWKV_OK) rwkv::counters().train_bwd++;
    return s;
}

rwkv_status rwkv_wkv7_step_tail(const float* r, const float* w, const float* k, const float* v, const float* a,
                                const float* b, const float* h_in, float* h_out, const float* rk, const float* lnw,
                                const float* lnb, const float* g, float* wkv_out, float* out, int64_t B, int64_t H,
                                float eps, void* stream) {
    RWKV_REQUIRE(r && w && k && v && a && b && h_out && rk && lnw && lnb && g && out, RWKV_E_NULL,
                 "wkv7_step_tail: null buffer");
    RWKV_REQUIRE(B >= 1 && H >= 1 && B * H <= INT32_MAX, RWKV_E_SHAPE, "wkv7_step_tail: bad B (%lld) / H (%lld)",
                 (long long)B, (long long)H);
    if (use_rows4(B * H))
        rwkv::launch(wkv7_step_tail_kernel<true>, dim3((unsigned)(B * H)), dim3(1024),
                     reinterpret_cast<hipStream_t>(stream), r, w, k, v, a, b, h_in, h_out, rk, lnw, lnb, g, wkv_out,
                     out, (int)H, eps);
    else
        rwkv::launch(wkv7_step_tail_kernel<false>, dim3((unsigned)(B * H)), dim3(256),
                     reinterpret_cast<hipStream_t>(stream), r, w, k, v, a, b, h_in, h_out, rk, lnw, lnb, g, wkv_out,
                     out, (int)H, eps);
    rwkv_status s = launch_status("wkv7_step_tail launch");
    if (s == RWKV_OK) rwkv::counters().step_tail++;
    return s;
}

int rwkv_wkv_tail_applies(int64_t S) { return S > 0 && S % 32 == 0; }

rwkv_status rwkv_wkv_tail_to(const float* wkv, const float* r, const float* k, const float* v, const float* rk,
                             const float* lnw, const float* lnb, const float* g, void* out, rwkv_dtype out_dt,
                             int64_t N, int64_t H, int64_t S, float eps, void* stream) {
    RWKV_REQUIRE(wkv && r && k && v && rk && lnw && lnb && g && out, RWKV_E_NULL, "wkv_tail: null buffer");
    RWKV_REQUIRE(out_dt == RWKV_F32 || out_dt == RWKV_F16, RWKV_E_DTYPE, "wkv_tail: output dtype %d not f32/f16",
                 (int)out_dt);
    RWKV_REQUIRE(rwkv_wkv_tail_applies(S), RWKV_E_SHAPE, "wkv_tail: S=%lld is not a multiple of 32", (long long)S);
    RWKV_REQUIRE(N >= 1 && H >= 1 && N * H <= INT32_MAX - 3 && S <= 1 << 20, RWKV_E_SHAPE, "wkv_tail: bad N/H/S");
    const dim3 grid((unsigned)((N * H + 3) / 4)), block(256);
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    if (out_dt == RWKV_F16)
        rwkv::launch(wkv_tail_kernel<_Float16>, grid, block, st, wkv, r, k, v, rk, lnw, lnb, g,
                     reinterpret_cast<_Float16*>(out), (int)(N * H), (int)H, (int)S, eps);
    else
        rwkv::launch(wkv_tail_kernel<float>, grid, block, st, wkv, r, k, v, rk, lnw, lnb, g,
                     reinterpret_cast<float*>(out), (int)(N * H), (int)H, (int)S, eps);
    rwkv_status s = launch_status("wkv_tail launch");
    if (s == RWKV_OK) rwkv::counters().tail++;
    return s;
}

rwkv_status rwkv_wkv_tail(const float* wkv, const float* r, const float* k, const float* v, const float* rk,
                          const float* lnw, const float* lnb, const float* g, float* out, int64_t N, int64_t H,
                          int64_t S, float eps, void* stream) {
    return rwkv_wkv_tail_to(wkv, r, k, v, rk, lnw, lnb, g, out, RWKV_F32, N, H, S, eps, stream);
}

}  // extern "C"
