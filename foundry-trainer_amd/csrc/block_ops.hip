// Memory-bound kernels of foundry-spike's double-stream LoRA block (the
// pieces around the attention and the frozen linears):
//   LayerNorm-modulation   y = (1 + scale) * LN(x) + shift    (lib.rs:60-71)
//   its backward           dx = dres + rstd*(dn - mean(dn) - n*mean(dn*n)),
//                          dn = dy * (1 + scale)
//   gated residual         y = x + g * b, g broadcast over rows
//                          (throughput.rs:552-572)
//   tanh-GELU and its derivative (the c4 block's MLP activation; the
//                          reference block uses SwiGLU, lib.rs:293-297)
//   SiLU                   of the conditioning vector (throughput.rs:297-324)
//   AdamW step             lib.rs:477-510, operation for operation
// All are HBM-bound: rows move with 16-byte vector accesses, statistics are
// f32, results are rounded once to the storage type.
#include <math.h>

#include <type_traits>

#include "fa_device.hpp"
#include "fa_kernels.hpp"
#include "fa_lds.hpp"

namespace fa {
namespace {

// 8 consecutive elements <-> f32 (bf16: one 16-byte access, f32: two)
__device__ __forceinline__ void load8(const bf16 *p, float v[8]) {
    const bf16x8 a = as_bf16x8(ld_global_16(p));
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = (float)a[j];
}
__device__ __forceinline__ void load8(const float *p, float v[8]) {
    const f32x4 a = __builtin_bit_cast(f32x4, ld_global_16(p));
    const f32x4 b = __builtin_bit_cast(f32x4, ld_global_16(p + 4));
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        v[j] = a[j];
        v[4 + j] = b[j];
    }
}
__device__ __forceinline__ void store8(bf16 *p, const float v[8]) {
    bf16x8 a;
#pragma unroll
    for (int j = 0; j < 8; ++j) a[j] = f32_to_bf16(v[j]);
    *reinterpret_cast<bf16x8 *>(p) = a;
}
__device__ __forceinline__ void store8(float *p, const float v[8]) {
    *reinterpret_cast<f32x4 *>(p) = f32x4{v[0], v[1], v[2], v[3]};
    *reinterpret_cast<f32x4 *>(p + 4) = f32x4{v[4], v[5], v[6], v[7]};
}

// The same past the caches' allocation: for streams far larger than the L2s
// that nothing reads again soon.
__device__ __forceinline__ void load8nt(const bf16 *p, float v[8]) {
    const bf16x8 a = as_bf16x8(__builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(p)));
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = (float)a[j];
}
__device__ __forceinline__ void load8nt(const float *p, float v[8]) {
    const f32x4 a = __builtin_nontemporal_load(reinterpret_cast<const f32x4 *>(p));
    const f32x4 b = __builtin_nontemporal_load(reinterpret_cast<const f32x4 *>(p + 4));
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        v[j] = a[j];
        v[4 + j] = b[j];
    }
}
__device__ __forceinline__ void store8nt(bf16 *p, const float v[8]) {
    bf16x8 a;
#pragma unroll
    for (int j = 0; j < 8; ++j) a[j] = f32_to_bf16(v[j]);
    __builtin_nontemporal_store(as_u32x4(a), reinterpret_cast<u32x4 *>(p));
}
__device__ __forceinline__ void store8nt(float *p, const float v[8]) {
    __builtin_nontemporal_store(f32x4{v[0], v[1], v[2], v[3]}, reinterpret_cast<f32x4 *>(p));
    __builtin_nontemporal_store(f32x4{v[4], v[5], v[6], v[7]}, reinterpret_cast<f32x4 *>(p + 4));
}

// x rounded to the storage type T, back in f32
template <typename T>
__device__ __forceinline__ float round_to(float x) {
    return (float)(T)x;
}

// Sum over the wave, the same value in every lane: within each 16-lane row by
// DPP (partners lane^1, lane^2, then the mirrors within 8 and within 16 lanes;
// each step adds a disjoint group's partial, so every lane of a row ends with
// the same sum), then rows by lane^16 and lane^32 exchanges.
template <int CTRL>
__device__ __forceinline__ float dpp_f32(float x) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, 0xF, 0xF, false));
}
__device__ __forceinline__ float wave_sum(float s) {
    s += dpp_f32<0xB1>(s);   // quad_perm [1,0,3,2]
    s += dpp_f32<0x4E>(s);   // quad_perm [2,3,0,1]
    s += dpp_f32<0x141>(s);  // row_half_mirror
    s += dpp_f32<0x140>(s);  // row_mirror
    s += __shfl_xor(s, 16, 64);
    return sum_xor32(s);
}

// One wave per row; lane l holds elements k*512 + 8*l .. +8 for k < MAXCH.
// GATED: the row is first the gated residual x + g * b, rounded to T as the
// gated-residual op rounds it (the same fma), stored to sum (and sum2), and
// the statistics are those of the rounded sum: the bits of the gated
// residual followed by this kernel on its output.
template <typename T, int MAXCH, bool GATED>
__global__ __launch_bounds__(256) void ln_mod_fwd_kernel(LnModParams p) {
    const int lane = threadIdx.x & 63;
    const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= p.N) return;
    const int C = p.C;
    const T *x = static_cast<const T *>(p.x) + row * p.ldx;
    float v[MAXCH][8];
    float s = 0.f;
#pragma unroll
    for (int k = 0; k < MAXCH; ++k) {
        const int e = k * 512 + lane * 8;
        if (e < C) {
            load8(x + e, v[k]);
            if constexpr (GATED) {
                float gv[8], bv[8];
                load8(static_cast<const T *>(p.g) + e, gv);
                load8(static_cast<const T *>(p.b) + row * p.ldb + e, bv);
#pragma unroll
                for (int j = 0; j < 8; ++j) v[k][j] = round_to<T>(__builtin_fmaf(gv[j], bv[j], v[k][j]));
                store8(static_cast<T *>(p.sum) + row * p.ldsum + e, v[k]);
                if (p.sum2) store8(static_cast<T *>(p.sum2) + row * p.ldsum2 + e, v[k]);
            }
#pragma unroll
            for (int j = 0; j < 8; ++j) s += v[k][j];
        }
    }
    const float mean = wave_sum(s) / (float)C;
    float q = 0.f;
#pragma unroll
    for (int k = 0; k < MAXCH; ++k) {
        const int e = k * 512 + lane * 8;
        if (e < C) {
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const float d = v[k][j] - mean;
                q += d * d;
            }
        }
    }
    const float var = wave_sum(q) / (float)C;
    const float den = sqrtf(var + p.eps);
    const float inv = 1.f / den;
    const T *shift = static_cast<const T *>(p.shift), *scale = static_cast<const T *>(p.scale);
    T *y = static_cast<T *>(p.y) + row * p.ldy;
#pragma unroll
    for (int k = 0; k < MAXCH; ++k) {
        const int e = k * 512 + lane * 8;
        if (e < C) {
            float sh[8], sc[8], o[8];
            load8(shift + e, sh);
            load8(scale + e, sc);
#pragma unroll
            for (int j = 0; j < 8; ++j) o[j] = (v[k][j] - mean) * inv * (sc[j] + 1.f) + sh[j];
            store8(y + e, o);
        }
    }
    if (lane == 0 && p.mean) {
        p.mean[row] = mean;
        p.rstd[row] = 1.f / den;
    }
}

// Elements e .. e + 7 of a row as they lie in memory, through its buffer
// descriptor: past the row's end they read as zero.
struct RawBf16 {
    u32x4 w;
};
struct RawF32 {
    u32x4 w, w2;
};
__device__ __forceinline__ void load_raw(__amdgpu_buffer_rsrc_t rs, int e, RawBf16 &r) {
    r.w = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, e * 2, 0, 0));
}
__device__ __forceinline__ void load_raw(__amdgpu_buffer_rsrc_t rs, int e, RawF32 &r) {
    r.w = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, e * 4, 0, 0));
    r.w2 = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, e * 4 + 16, 0, 0));
}
__device__ __forceinline__ float raw_at(const RawBf16 &r, int j) { return (float)as_bf16x8(r.w)[j]; }
__device__ __forceinline__ float raw_at(const RawF32 &r, int j) {
    return j < 4 ? __builtin_bit_cast(f32x4, r.w)[j] : __builtin_bit_cast(f32x4, r.w2)[j - 4];
}
// Keeps r as it is (the compiler may not carry values derived from it across).
__device__ __forceinline__ void raw_keep(RawBf16 &r) { asm volatile("" : "+v"(r.w)); }
__device__ __forceinline__ void raw_keep(RawF32 &r) { asm volatile("" : "+v"(r.w), "+v"(r.w2)); }

// Backward, one wave (and workgroup) per row: lane l holds elements
// k*512 + 8*l .. +8 for k < MAXCH and sums them in that order, then the wave
// its lanes, so a row's bits depend on no launch shape.
//
// HBM-bound.  All of a row's operands, the residual's gradient among them, are
// loaded before any is used and stay in storage form (x and dy are widened
// again after the sums): 91 VGPRs for a bf16 row of 3072, so five waves per
// SIMD hold a 4608-row grid in one round (101 and four with GATE_OUT; held to
// five it spills and takes 35.2 us).  4608 x 3072 bf16 from cold HBM 31.1 ->
// 27.2 us (4.2 TB/s), with GATE_OUT 38.9 -> 32.0 (4.4), against loads chunk by
// chunk as the sums need them.  A row spread over six waves took 25.2 and
// 30.0, but adds in another order: dx then differs in bf16 roundings.
//
// GATE_OUT: also gdx = g * dx, from dx as rounded to T (the same fma as the
// gated-residual op with no x), the gradient through a gated branch whose
// output fed this layer norm's input.
template <typename T, int MAXCH, bool GATE_OUT>
__global__ __launch_bounds__(64) void ln_mod_bwd_kernel(LnModParams p) {
    // each product and sum below rounds by itself, but for the fmas written out
#pragma clang fp contract(off)
    using Raw = std::conditional_t<sizeof(T) == 2, RawBf16, RawF32>;
    const int lane = threadIdx.x;
    const int64_t row = blockIdx.x;
    const int C = p.C;
    const uint32_t bytes = (uint32_t)C * sizeof(T);
    const T *dres = static_cast<const T *>(p.dres);
    const __amdgpu_buffer_rsrc_t xrs = make_rsrc(static_cast<const T *>(p.x) + row * p.ldx, bytes);
    const __amdgpu_buffer_rsrc_t yrs = make_rsrc(static_cast<const T *>(p.dy) + row * p.lddy, bytes);
    const __amdgpu_buffer_rsrc_t rrs = make_rsrc(dres ? dres + row * p.ldres : dres, dres ? bytes : 0u);
    const __amdgpu_buffer_rsrc_t srs = make_rsrc(p.scale, bytes), grs = make_rsrc(p.g, bytes);
    Raw x[MAXCH], dy[MAXCH], res[MAXCH], sc, sc1;
#pragma unroll
    for (int k = 0; k < MAXCH; ++k) {
        load_raw(xrs, k * 512 + lane * 8, x[k]);
        load_raw(yrs, k * 512 + lane * 8, dy[k]);
    }
#pragma unroll
    for (int k = 0; k < MAXCH; ++k) load_raw(rrs, k * 512 + lane * 8, res[k]);
    load_raw(srs, lane * 8, sc);
    __builtin_amdgcn_sched_barrier(0);  // the compiler would move most of them down to their uses
    const float mean = p.mean[row], rstd = p.rstd[row];
    float a = 0.f, b = 0.f;
    // elements past C have dy = 0 and change neither sum
#pragma unroll
    for (int k = 0; k < MAXCH; ++k) {
        load_raw(srs, (k + 1) % MAXCH * 512 + lane * 8, sc1);  // at last chunk 0's again, for the results
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const float g = raw_at(sc, j) + 1.f, d = raw_at(dy[k], j);
            const float n = (raw_at(x[k], j) - mean) * rstd;
            a = __builtin_fmaf(g, d, a);
            b = __builtin_fmaf(g * d, n, b);
        }
        sc = sc1;
        __builtin_amdgcn_sched_barrier(0);
    }
    const float ma = wave_sum(a) / (float)C, mb = wave_sum(b) / (float)C;
    Raw gt;
    if constexpr (GATE_OUT) load_raw(grs, lane * 8, gt);
    T *dx = static_cast<T *>(p.dx) + row * p.lddx, *gdx = static_cast<T *>(p.gdx) + row * p.ldgdx;
#pragma unroll
    for (int k = 0; k < MAXCH; ++k) {
        raw_keep(x[k]);
        raw_keep(dy[k]);
        float o[8], go[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const float n = (raw_at(x[k], j) - mean) * rstd, dn = (raw_at(sc, j) + 1.f) * raw_at(dy[k], j);
            o[j] = __builtin_fmaf(rstd, __builtin_fmaf(-mb, n, dn - ma), raw_at(res[k], j));
            if constexpr (GATE_OUT) go[j] = __builtin_fmaf(raw_at(gt, j), round_to<T>(o[j]), 0.f);
        }
        // the next vectors before this chunk's stores: the wait for them then leaves the stores in flight
        __builtin_amdgcn_sched_barrier(0);
        if (k + 1 < MAXCH) {
            load_raw(srs, (k + 1) * 512 + lane * 8, sc);
            if constexpr (GATE_OUT) load_raw(grs, (k + 1) * 512 + lane * 8, gt);
        }
        if (lane * 8 < C - k * 512) {
            store8(dx + k * 512 + lane * 8, o);
            if constexpr (GATE_OUT) store8(gdx + k * 512 + lane * 8, go);
        }
        __builtin_amdgcn_sched_barrier(0);
    }
}

// Elementwise over an [N, C] view, 8 elements per thread (C % 8 == 0).
// op 0: y = x + g * b (x may be null: y = g * b);  1: y = gelu(b);
// op 2: y = x * gelu'(b) (x = upstream gradient);  3: y = silu(b)
// gelu(u) = u/2 * (1 + tanh(z)), z = k0 * (u + k1 u^3), evaluated as
// u * sigmoid(2z) (the same function: (1 + tanh z) / 2 = sigmoid(2z)) with one
// exp2 and one reciprocal; gelu'(u) = sg + 2 u sg (1 - sg) k0 (1 + 3 k1 u^2),
// sg = sigmoid(2z).
constexpr float kGeluK0 = 0.7978845608028654f;  // sqrt(2/pi)
constexpr float kGeluK1 = 0.044715f;

// sigmoid(2 k0 (u + k1 u^3)) of the tanh-GELU
__device__ __forceinline__ float gelu_sigmoid(float u) {
    const float z2 = (2.f * kGeluK0) * (u + kGeluK1 * u * u * u);
    return __builtin_amdgcn_rcpf(1.f + exp2_fast(-kLog2e * z2));
}

// Grid: x over 128-lane groups of a row's 8-element chunks, y over rows
// (striding by gridDim.y), so no lane divides to find its row.  Results, and
// what the GELU gradient reads last, go past the caches: with GELU and its
// gradient at 4096 x 9216 bf16 between the block's layer norms from cold HBM,
// the four launches 114 -> 102 us.
constexpr int kEltLanes = 128;
template <typename T, int OP>
__global__ __launch_bounds__(kEltLanes) void elementwise_kernel(EltParams p) {
    const int e = (blockIdx.x * kEltLanes + threadIdx.x) * 8;
    if (e >= p.C) return;
    const T *g = static_cast<const T *>(p.g);
    for (int64_t row = blockIdx.y; row < p.N; row += gridDim.y) {
        float bv[8], o[8];
        const T *b = static_cast<const T *>(p.b) + row * p.ldb + e;
        if constexpr (OP == 2)
            load8nt(b, bv);  // the pre-activation's last use
        else
            load8(b, bv);
        if constexpr (OP == 0) {
            float gv[8], xv[8];
            load8(g + e, gv);
            if (p.x) {
                load8(static_cast<const T *>(p.x) + row * p.ldx + e, xv);
            } else {
#pragma unroll
                for (int j = 0; j < 8; ++j) xv[j] = 0.f;
            }
#pragma unroll
            for (int j = 0; j < 8; ++j) o[j] = __builtin_fmaf(gv[j], bv[j], xv[j]);
        } else if constexpr (OP == 1) {
#pragma unroll
            for (int j = 0; j < 8; ++j) o[j] = bv[j] * gelu_sigmoid(bv[j]);
        } else if constexpr (OP == 2) {
            float xv[8];
            load8nt(static_cast<const T *>(p.x) + row * p.ldx + e, xv);
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const float u = bv[j];
                const float sg = gelu_sigmoid(u);
                const float d = sg + (2.f * kGeluK0) * u * (sg - sg * sg) * (1.f + (3.f * kGeluK1) * u * u);
                o[j] = xv[j] * d;
            }
        } else {
#pragma unroll
            for (int j = 0; j < 8; ++j) o[j] = bv[j] / (1.f + exp2_fast(-kLog2e * bv[j]));
        }
        store8nt(static_cast<T *>(p.y) + row * p.ldy + e, o);
    }
}

// SwiGLU over [N, C] views, 8 elements per thread.  Forward: y = T(T(silu(g))
// * u).  Backward: du = T(dy * T(silu(g))), dg = T(T(dy * u) * silu'(g)) with
// silu'(g) = s (1 + g (1 - s)), s = 1 / (1 + e^-g); T() = round to storage.
// The grid is the elementwise kernel's (a form that strode over all elements
// divided a 64-bit index by the row length on each), and what the backward
// reads last and both write goes past the caches: 4608 x 9216 bf16 from cold
// HBM 54 -> 50 -> 44 us forward (5.8 TB/s), 81 -> 74 -> 63 us backward (6.7 TB/s),
// and the layer-norm backward after it 27 -> 22.
template <typename T, bool BWD>
__global__ __launch_bounds__(kEltLanes) void swiglu_kernel(SwigluParams p) {
    const int e = (blockIdx.x * kEltLanes + threadIdx.x) * 8;
    if (e >= p.C) return;
    for (int64_t row = blockIdx.y; row < p.N; row += gridDim.y) {
        float gv[8], uv[8], o[8];
        const T *gate = static_cast<const T *>(p.gate) + row * p.ldg + e, *up = static_cast<const T *>(p.up) + row * p.ldu + e;
        if constexpr (BWD) {
            load8nt(gate, gv);
            load8nt(up, uv);
        } else {
            load8(gate, gv);
            load8(up, uv);
        }
        if constexpr (!BWD) {
#pragma unroll
            for (int j = 0; j < 8; ++j) o[j] = round_to<T>(gv[j] / (1.f + exp2_fast(-kLog2e * gv[j]))) * uv[j];
        } else {
            float dv[8], du[8];
            load8nt(static_cast<const T *>(p.dy) + row * p.lddy + e, dv);
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const float g = gv[j];
                const float sg = 1.f / (1.f + exp2_fast(-kLog2e * g));
                const float silu = round_to<T>(g / (1.f + exp2_fast(-kLog2e * g)));
                du[j] = dv[j] * silu;
                o[j] = round_to<T>(dv[j] * uv[j]) * (sg * (1.f + g * (1.f - sg)));
            }
            store8nt(static_cast<T *>(p.dup) + row * p.lddup + e, du);
        }
        store8nt(static_cast<T *>(p.y) + row * p.ldy + e, o);
    }
}

// AdamW, weight decay 0, in the reference's operation order:
//   m' = m*b1 + g*(1-b1);  v' = v*b2 + (g*g)*(1-b2)
//   p' = p - ((m' * ibc1) / (sqrt(v' * ibc2) + eps)) * lr
// each product / sum rounded separately (contraction off for the
// expressions written here), IEEE sqrt and division, p' rounded to T.
template <typename T, typename H>
__device__ __forceinline__ void adamw_elem(T *w, const float *grad, float *mm, float *vv, int64_t i, const H &h) {
#pragma clang fp contract(off)
    const float g = grad[i];
    const float m = mm[i] * h.b1 + g * h.one_m_b1;
    const float gg = g * g;
    const float v = vv[i] * h.b2 + gg * h.one_m_b2;
    const float mhat = m * h.ibc1;
    const float den = sqrtf(v * h.ibc2) + h.eps;
    const float delta = (mhat / den) * h.lr;
    w[i] = (T)((float)w[i] - delta);
    mm[i] = m;
    vv[i] = v;
}

template <typename T>
__global__ __launch_bounds__(256) void adamw_kernel(AdamwParams p) {
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < p.n; i += (int64_t)gridDim.x * 256)
        adamw_elem(static_cast<T *>(p.param), p.grad, p.m, p.v, i, p);
}

// Several tensors of one AdamW step in one launch: tensor k owns blocks
// [block0[k], block0[k + 1]) and strides over its elements with them.  Same
// per-element arithmetic as adamw_kernel, so the same bits.
template <typename T>
__global__ __launch_bounds__(256) void adamw_many_kernel(AdamwMany p) {
    const int b = blockIdx.x;
    int k = 0;
    while (k + 1 < p.count && p.block0[k + 1] <= b) ++k;
    const int nb = p.block0[k + 1] - p.block0[k];
    T *w = static_cast<T *>(p.param[k]);
    for (int64_t i = (int64_t)(b - p.block0[k]) * 256 + threadIdx.x; i < p.n[k]; i += (int64_t)nb * 256)
        adamw_elem(w, p.grad[k], p.m[k], p.v[k], i, p);
}

// Strided 2D copies of several small arrays in one launch: view k owns
// blocks [block0[k], block0[k + 1]) and strides over its rows * cols elements.
template <typename E>
__global__ __launch_bounds__(256) void copy2d_many_kernel(Copy2dMany p) {
    const int b = blockIdx.x;
    int k = 0;
    while (k + 1 < p.count && p.block0[k + 1] <= b) ++k;
    const int nb = p.block0[k + 1] - p.block0[k];
    const int cols = p.cols[k];
    const int64_t n = (int64_t)p.rows[k] * cols;
    const E *src = static_cast<const E *>(p.src[k]);
    E *dst = static_cast<E *>(p.dst[k]);
    for (int64_t i = (int64_t)(b - p.block0[k]) * 256 + threadIdx.x; i < n; i += (int64_t)nb * 256) {
        const int64_t r = i / cols, c = i - r * cols;
        dst[r * p.dst_rs[k] + c * p.dst_cs[k]] = src[r * p.src_rs[k] + c * p.src_cs[k]];
    }
}

inline int elt_grid(int64_t n8) {
    const int64_t blocks = (n8 + 255) / 256;
    return (int)(blocks < 4096 ? (blocks > 0 ? blocks : 1) : 4096);
}

}  // namespace

// MAXCH (512-element chunks per row): 2 up to C = 1024, 6 up to 3072 (the
// blocks' width: fewer registers, so a whole 4608-row grid is resident in one
// round), 8 up to 4096.
template <typename T, bool F>
static hipError_t ln_fwd_t(const LnModParams &p, hipStream_t s) {
    const dim3 grid((unsigned)((p.N + 3) / 4)), block(256);
    if (p.C <= 1024)
        hipLaunchKernelGGL((ln_mod_fwd_kernel<T, 2, F>), grid, block, 0, s, p);
    else if (p.C <= 3072)
        hipLaunchKernelGGL((ln_mod_fwd_kernel<T, 6, F>), grid, block, 0, s, p);
    else
        hipLaunchKernelGGL((ln_mod_fwd_kernel<T, 8, F>), grid, block, 0, s, p);
    return hipGetLastError();
}
template <typename T, bool F>
static hipError_t ln_bwd_t(const LnModParams &p, hipStream_t s) {
    const dim3 grid((unsigned)p.N), block(64);
    if (p.C <= 1024)
        hipLaunchKernelGGL((ln_mod_bwd_kernel<T, 2, F>), grid, block, 0, s, p);
    else if (p.C <= 3072)
        hipLaunchKernelGGL((ln_mod_bwd_kernel<T, 6, F>), grid, block, 0, s, p);
    else
        hipLaunchKernelGGL((ln_mod_bwd_kernel<T, 8, F>), grid, block, 0, s, p);
    return hipGetLastError();
}
template <typename T>
static hipError_t ln_fwd_t(const LnModParams &p, hipStream_t s) {
    return p.b ? ln_fwd_t<T, true>(p, s) : ln_fwd_t<T, false>(p, s);
}
template <typename T>
static hipError_t ln_bwd_t(const LnModParams &p, hipStream_t s) {
    return p.gdx ? ln_bwd_t<T, true>(p, s) : ln_bwd_t<T, false>(p, s);
}

hipError_t launch_ln_mod_fwd(const LnModParams &p, int dtype, hipStream_t s) {
    return dtype == 0 ? ln_fwd_t<bf16>(p, s) : ln_fwd_t<float>(p, s);
}
hipError_t launch_ln_mod_bwd(const LnModParams &p, int dtype, hipStream_t s) {
    return dtype == 0 ? ln_bwd_t<bf16>(p, s) : ln_bwd_t<float>(p, s);
}

// Grid over an [N, C] view, C % 8 == 0: about 64K workgroups in all, at most
// 65535 row groups.
static dim3 rows_grid(int N, int C) {
    const unsigned gx = (unsigned)((C / 8 + kEltLanes - 1) / kEltLanes);
    int64_t gy = ((int64_t)1 << 16) / gx;
    if (gy > N) gy = N;
    if (gy > 65535) gy = 65535;
    if (gy < 1) gy = 1;
    return dim3(gx, (unsigned)gy);
}

template <typename T>
static hipError_t elt_t(const EltParams &p, int op, hipStream_t s) {
    const dim3 grid = rows_grid(p.N, p.C), block(kEltLanes);
    switch (op) {
        case 0: hipLaunchKernelGGL((elementwise_kernel<T, 0>), grid, block, 0, s, p); break;
        case 1: hipLaunchKernelGGL((elementwise_kernel<T, 1>), grid, block, 0, s, p); break;
        case 2: hipLaunchKernelGGL((elementwise_kernel<T, 2>), grid, block, 0, s, p); break;
        default: hipLaunchKernelGGL((elementwise_kernel<T, 3>), grid, block, 0, s, p); break;
    }
    return hipGetLastError();
}
hipError_t launch_elementwise(const EltParams &p, int op, int dtype, hipStream_t s) {
    return dtype == 0 ? elt_t<bf16>(p, op, s) : elt_t<float>(p, op, s);
}

template <typename T>
static hipError_t swiglu_t(const SwigluParams &p, bool bwd, hipStream_t s) {
    const dim3 grid = rows_grid(p.N, p.C), block(kEltLanes);
    if (bwd)
        hipLaunchKernelGGL((swiglu_kernel<T, true>), grid, block, 0, s, p);
    else
        hipLaunchKernelGGL((swiglu_kernel<T, false>), grid, block, 0, s, p);
    return hipGetLastError();
}
hipError_t launch_swiglu(const SwigluParams &p, bool bwd, int dtype, hipStream_t s) {
    return dtype == 0 ? swiglu_t<bf16>(p, bwd, s) : swiglu_t<float>(p, bwd, s);
}

hipError_t launch_adamw_many(AdamwMany p, int dtype, hipStream_t s) {
    int blocks = 0;
    for (int k = 0; k < p.count; ++k) {
        p.block0[k] = blocks;
        const int64_t nb = (p.n[k] + 255) / 256;
        blocks += (int)(nb < 1024 ? nb : 1024);
    }
    p.block0[p.count] = blocks;
    const dim3 grid(blocks), block(256);
    if (dtype == 0)
        hipLaunchKernelGGL((adamw_many_kernel<bf16>), grid, block, 0, s, p);
    else
        hipLaunchKernelGGL((adamw_many_kernel<float>), grid, block, 0, s, p);
    return hipGetLastError();
}

hipError_t launch_copy2d_many(Copy2dMany p, int elt_bytes, hipStream_t s) {
    int blocks = 0;
    for (int k = 0; k < p.count; ++k) {
        p.block0[k] = blocks;
        const int64_t nb = ((int64_t)p.rows[k] * p.cols[k] + 255) / 256;
        blocks += (int)(nb < 256 ? nb : 256);
    }
    p.block0[p.count] = blocks;
    if (elt_bytes == 2)
        hipLaunchKernelGGL(copy2d_many_kernel<uint16_t>, dim3(blocks), dim3(256), 0, s, p);
    else
        hipLaunchKernelGGL(copy2d_many_kernel<uint32_t>, dim3(blocks), dim3(256), 0, s, p);
    return hipGetLastError();
}

hipError_t launch_adamw(const AdamwParams &p, int dtype, hipStream_t s) {
    const dim3 grid(elt_grid(p.n)), block(256);
    if (dtype == 0)
        hipLaunchKernelGGL((adamw_kernel<bf16>), grid, block, 0, s, p);
    else
        hipLaunchKernelGGL((adamw_kernel<float>), grid, block, 0, s, p);
    return hipGetLastError();
}

}  // namespace fa
