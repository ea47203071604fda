// f32 attention for gfx950 (FA_DTYPE_F32): the forward and the recomputing
// backward of foundry-spike's attn_fwd / AttnBwd::bwd (crates/foundry-spike/
// src/lib.rs:131-149, 216-263) with exact f32 products and f32 accumulation
// on v_mfma_f32_32x32x2_f32; P and dS stay f32, as in the reference's f32 run.
//
// What bounds these kernels is that instruction: 4096 flop in 64 clocks per
// SIMD (154 TF/s measured for an 8192^3 f32 GEMM).  It needs one operand read
// of 4 bytes per lane and 64 clocks, so LDS bandwidth and VALU have slack;
// what matters is that every SIMD always has an MFMA to issue.  Hence:
//   - Tiles of 32 rows go HBM/L2 -> LDS by 16-byte DMA and are read by
//     ds_read_b128: one read feeds four MFMAs.  The MFMA's k (or its m, for a
//     transposed operand) may be any permutation of the features as long as
//     both operands (or the store) agree, so a lane takes the 4 consecutive
//     features of a 16-byte chunk as 4 k-steps, or as its row of D / 32
//     output tiles.
//   - Each tile has one buffer.  A phase that reads one tile is 4096 clocks
//     at D = 128 (64 MFMAs), longer than a tile's load, so the tile a phase
//     has released is refilled while the next phase reads the other tile.
//   - A workgroup is 4 waves: RW waves of 32 rows each (queries in the
//     forward and dQ, keys in dK/dV) times CW groups that each stream every
//     CW-th 32-row block of the other side, their partial results merged
//     through LDS in a fixed order.  More groups make the unit of work per CU
//     smaller (32 rows at CW = 4) so that grids of few rows still fill the
//     chip evenly; fewer groups share each tile among more waves.
// Measured at B1 H24 S1536 D128, against one wave per 32 rows with 4-byte
// guarded loads and no overlap: forward 2647 -> 294 us (99 TF/s), dK/dV 4050
// -> 552 us (105 TF/s), dQ 2724 -> 430 us recomputing S and dP, about 140 us
// from the stored dS; forward and backward 9870 -> 973 us.  What remains is
// the last of 4.5 rounds of workgroups (10%), each workgroup's first loads and
// merge (about 10 us of 60), and the softmax VALU work between products.
#include <math.h>

#include <type_traits>

#include "fa_device.hpp"
#include "fa_kernels.hpp"
#include "fa_lds.hpp"

namespace fa {
namespace {

// A 32-row tile of D f32 features in LDS: 16-byte chunk c of row r sits at
// chunk c ^ (r % 16).  Row reads (32 rows at one chunk per lane half) then
// touch 16 distinct chunk columns (all 64 banks) per 16 lanes, and reads along
// a row stay a permutation of that row.
template <int D>
struct F32Tile {
    static constexpr int CH = D / 4;                // chunks per row
    static constexpr int ROWB = D * 4;              // bytes per row
    static constexpr int BYTES = 32 * ROWB;
    static constexpr int INSTS = BYTES / 1024;      // wave-instructions per tile
};

template <int D>
__device__ __forceinline__ uint32_t chunk_off(int row, int c) {
    return (uint32_t)(row * F32Tile<D>::ROWB + ((c ^ (row & 15)) << 4));
}

// Rows row0 .. row0+31 of a [S][D] view (row stride ss) into a tile, wave w of
// the NW that share it.  Through a buffer descriptor over the tile's rows: its
// base is 64-bit, the offsets inside it 32-bit, rows past S read as zero, and
// an instruction costs one XOR (its chunk keys) beside the load.  A tile that
// spans 4 GiB or more (WIDE, row strides of kWideStride elements on) takes
// 64-bit lane addresses instead, with rows past S read from row S - 1: callers
// mask keys past S and give queries past S an LSE of +inf, so either content
// is unused.
constexpr int64_t kWideStride = 1 << 25;
template <int D, int NW, bool WIDE>
__device__ __forceinline__ void tile_issue(const float *base, int64_t ss, int row0, int S, char *dst, int w, int lane) {
    using T = F32Tile<D>;
    static_assert(T::INSTS % NW == 0, "tile split over waves");
    constexpr int RPI = 64 / T::CH;  // rows per instruction
    if constexpr (!WIDE) {
        const int rows = min(32, S - row0);
        const __amdgpu_buffer_rsrc_t rs =
            make_rsrc(base + (int64_t)row0 * ss, rows > 0 ? (uint32_t)(((rows - 1) * ss + D) * 4) : 0u);
        const int lr = lane / T::CH;
        const uint32_t step = (uint32_t)(RPI * ss * 4), vrow = (uint32_t)(lr * ss * 4);
#pragma unroll
        for (int i = 0; i < T::INSTS / NW; ++i) {
            const int inst = i * NW + w;  // rows inst * RPI + lr; RPI is a power of two, so the keys' bits add as an XOR
            const uint32_t chunk = (uint32_t)((lane % T::CH) ^ lr ^ ((inst * RPI) & 15));
            buffer_to_lds_16(rs, dst + inst * 1024, vrow + (chunk << 4), (uint32_t)inst * step);
        }
    } else {
#pragma unroll
        for (int i = 0; i < T::INSTS / NW; ++i) {
            const int inst = i * NW + w, c = inst * 64 + lane;
            const int row = c / T::CH, logical = (c % T::CH) ^ (row & 15);
            const float *src = base + (int64_t)min(row0 + row, S - 1) * ss + logical * 4;
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)src,
                                             (__attribute__((address_space(3))) void *)(dst + inst * 1024), 16, 0, 0);
        }
    }
}

// This wave's DMA has landed and its LDS reads are done; with SHARED tiles,
// every wave of the workgroup is at the same point.
template <bool SHARED>
__device__ __forceinline__ void phase_sync() {
    if constexpr (SHARED)
        barrier_keep_dma<0>();
    else
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
}

__device__ __forceinline__ f32x4 ld_f32x4(const char *smem, uint32_t off) {
    return __builtin_bit_cast(f32x4, ld_lds_16(smem, (int)off));
}

// A product phase runs in steps of 8 MFMAs.  Each step reads the next step's
// operands before its own MFMAs, and nothing is scheduled across a step's end:
// left alone the compiler issues each read right before the MFMAs that use it
// and waits out the LDS latency, 100 of every 256 clocks in the one wave a
// SIMD holds.

// out[m][n] += sum_d tile[m][d] reg[n][d]: `reg` holds row n's chunks 2i + g.
// Two chains (even and odd chunks) so that no MFMA waits for the one before.
template <int D>
__device__ __forceinline__ f32x16 row_product(const char *tile, const f32x4 (&reg)[D / 8], int n, int g) {
    f32x16 a, b;
#pragma unroll
    for (int r = 0; r < 16; ++r) a[r] = b[r] = 0.f;
    f32x4 t0 = ld_f32x4(tile, chunk_off<D>(n, g)), t1 = ld_f32x4(tile, chunk_off<D>(n, 2 + g));
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < D / 8; i += 2) {
        f32x4 n0 = t0, n1 = t1;
        if (i + 2 < D / 8) {
            n0 = ld_f32x4(tile, chunk_off<D>(n, 2 * i + 4 + g));
            n1 = ld_f32x4(tile, chunk_off<D>(n, 2 * i + 6 + g));
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            a = mfma_32x32x2_f32(t0[e], reg[i][e], a);
            b = mfma_32x32x2_f32(t1[e], reg[i + 1][e], b);
        }
        t0 = n0;
        t1 = n1;
        __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) a[r] += b[r];
    return a;
}

// The D / 32 features n * D/32 .. of tile row `row` (a lane's operand in all
// D / 32 output tiles of a product over the tile's rows).
template <int D>
__device__ __forceinline__ void col_operand(const char *tile, int row, int n, float (&v)[D / 32]) {
    if constexpr (D == 128) {
        const f32x4 x = ld_f32x4(tile, chunk_off<D>(row, n));
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = x[e];
    } else {
        typedef float f32x2 __attribute__((ext_vector_type(2)));
        const f32x2 x = *reinterpret_cast<const f32x2 *>(tile + chunk_off<D>(row, n >> 1) + 8 * (n & 1));
        v[0] = x[0];
        v[1] = x[1];
    }
}

// acc[dt] += the product over the tile's 32 rows of x (element t: row
// acc_row(t)) and the rows' features n * D/32 + dt.  TILE_A: the tile is the A
// operand (features on the accumulator's rows), else x is.
template <int D, bool TILE_A>
__device__ __forceinline__ void col_product(const char *tile, const f32x16 &x, f32x16 (&acc)[D / 32], int lane) {
    constexpr int NT = D / 32, STEP = 8 / NT;  // tile rows per step and lane half
    const int n = lane & 31;
    float cur[STEP][NT], nxt[STEP][NT];
#pragma unroll
    for (int u = 0; u < STEP; ++u) col_operand<D>(tile, acc_row(u, lane), n, cur[u]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int t = 0; t < 16; t += STEP) {
#pragma unroll
        for (int u = 0; u < STEP; ++u) {
            if (t + STEP < 16) col_operand<D>(tile, acc_row(t + STEP + u, lane), n, nxt[u]);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < STEP; ++u)
#pragma unroll
            for (int dt = 0; dt < NT; ++dt)
                acc[dt] = TILE_A ? mfma_32x32x2_f32(cur[u][dt], x[t + u], acc[dt])
                                 : mfma_32x32x2_f32(x[t + u], cur[u][dt], acc[dt]);
#pragma unroll
        for (int u = 0; u < STEP; ++u)
#pragma unroll
            for (int dt = 0; dt < NT; ++dt) cur[u][dt] = nxt[u][dt];
        __builtin_amdgcn_sched_barrier(0);
    }
}

// Row `row` of a view into this lane's operand registers (chunks 2i + g).
template <int D>
__device__ __forceinline__ void load_rows(const float *base, int64_t ss, int row, int S, int g, f32x4 (&reg)[D / 8]) {
#pragma unroll
    for (int i = 0; i < D / 8; ++i)
        reg[i] = row < S ? __builtin_bit_cast(f32x4, ld_global_16(base + (int64_t)row * ss + (2 * i + g) * 4))
                         : f32x4{0.f, 0.f, 0.f, 0.f};
}

// NT consecutive floats (16- or 8-byte aligned).
template <int NT>
__device__ __forceinline__ void store_nt(float *p, const float (&v)[NT]) {
    if constexpr (NT == 4) {
        *reinterpret_cast<f32x4 *>(p) = f32x4{v[0], v[1], v[2], v[3]};
    } else {
        typedef float f32x2 __attribute__((ext_vector_type(2)));
        *reinterpret_cast<f32x2 *>(p) = f32x2{v[0], v[1]};
    }
}

// LDS of one workgroup: two arrays, one per streamed operand, each holding
// its CW groups' tiles (distinct objects, so that the compiler can tell the
// refill of one from the reads of the other).  After the loop the same bytes
// hold the waves' partial accumulators, D / 32 tiles at a time: waves 0 and 1
// in the first array, 2 and 3 in the second.
template <int D, int CW>
struct F32Lds {
    static constexpr int TILES = CW * F32Tile<D>::BYTES;
    static constexpr int PART = 2 * 16 * (D / 32) * 64 * 4;  // two waves' partials
    static_assert(CW == 1 || PART <= TILES, "partials fit in the tiles");
};

// Element (r, dt) of wave `wave`, lane `lane`.
template <int D>
__device__ __forceinline__ float *part_slot(char *a, char *b, int wave, int r, int dt, int lane) {
    return reinterpret_cast<float *>(wave < 2 ? a : b) + (((wave & 1) * 16 + r) * (D / 32) + dt) * 64 + lane;
}

// ---------------------------------------------------------------------------
// forward: a wave owns 32 queries (lane n) and streams key blocks.
//   S^T = K Q^T, P = exp2(s c - m c), O^T += V^T P^T
// Per block: S (K tile), refill K, softmax, P V (V tile), refill V.
// The exp2 reference m moves only when a block's maximum exceeds it by more
// than 2^8 in P, so most blocks rescale nothing (P <= 2^8 and l stay far from
// overflow, and f32 products keep their relative precision).
// ---------------------------------------------------------------------------
template <int D, int RW, int CW, bool WIDE = false>
__global__ __launch_bounds__(256, D == 128 && CW == 4 ? 1 : 2) void attn_fwd_f32_kernel(AttnFwdParams p) {
    using T = F32Tile<D>;
    constexpr int NT = D / 32;
    constexpr bool SHARED = RW > 1;
    __shared__ __align__(16) char ks[F32Lds<D, CW>::TILES], vs[F32Lds<D, CW>::TILES];
    __shared__ float ml[CW > 1 ? 2 * 4 * 32 : 1];  // merge: each wave's reference and row sum per query
    const int lane = threadIdx.x & 63, n = lane & 31, g = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int rw = wave % RW, cg = wave / RW;
    const int S = p.S, H = p.H;
    const int nq = (S + 32 * RW - 1) / (32 * RW);
    const int work = xcd_remap(blockIdx.x, gridDim.x);
    const int qt = work % nq, bh = work / nq;
    const int h = bh % H, b = bh / H;
    const float *kbase = static_cast<const float *>(p.k) + b * p.k_sb + h * p.k_sh;
    const float *vbase = static_cast<const float *>(p.v) + b * p.v_sb + h * p.v_sh;
    const uint8_t *keep = p.keep ? p.keep + (int64_t)b * S : nullptr;
    const int qi = (qt * RW + rw) * 32 + n;
    char *kt = ks + cg * T::BYTES, *vt = vs + cg * T::BYTES;

    tile_issue<D, RW, WIDE>(kbase, p.k_ss, cg * 32, S, kt, rw, lane);
    f32x4 qf[D / 8];
    load_rows<D>(static_cast<const float *>(p.q) + b * p.q_sb + h * p.q_sh, p.q_ss, qi, S, g, qf);
    f32x16 o[NT];
#pragma unroll
    for (int dt = 0; dt < NT; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[dt][r] = 0.f;
    float m_run = -INFINITY, m_sc = 0.f, l_run = 0.f;
    const float c = p.scale_log2;
    const int nkb = (S + 31) / 32, J = (nkb + CW - 1) / CW;
    phase_sync<SHARED>();
    tile_issue<D, RW, WIDE>(vbase, p.v_ss, cg * 32, S, vt, rw, lane);
    for (int j = 0; j < J; ++j) {
        const int k0 = (j * CW + cg) * 32;  // a group's padding block lies past S: all its keys are masked
        const bool kept = k0 + n < S && (!keep || keep[k0 + n]);
        f32x16 s = row_product<D>(kt, qf, n, g);
        phase_sync<SHARED>();
        tile_issue<D, RW, WIDE>(kbase, p.k_ss, k0 + CW * 32, S, kt, rw, lane);
        const uint32_t km = (uint32_t)__ballot(kept);
        if (km != ~0u) {
#pragma unroll
            for (int r = 0; r < 16; ++r)
                if (!((km >> acc_row(r, lane)) & 1)) s[r] = -INFINITY;
        }
        float mx = s[0];
#pragma unroll
        for (int r = 1; r < 16; ++r) mx = fmaxf(mx, s[r]);
        mx = max_xor32(mx);
        // m_run = -inf (no kept key yet): any finite maximum moves it
        if (__any(mx * c > (m_run == -INFINITY ? -INFINITY : m_sc + 8.f))) {
            const float m_new = fmaxf(m_run, mx);
            const float m_sc_new = m_new == -INFINITY ? 0.f : m_new * c;
            const float alpha = m_run == -INFINITY ? 0.f : exp2f(m_sc - m_sc_new);
            m_run = m_new;
            m_sc = m_sc_new;
            l_run *= alpha;
#pragma unroll
            for (int dt = 0; dt < NT; ++dt)
#pragma unroll
                for (int r = 0; r < 16; ++r) o[dt][r] *= alpha;
        }
        float psum = 0.f;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            s[r] = exp2f(s[r] * c - m_sc);
            psum += s[r];
        }
        l_run += psum;
        col_product<D, true>(vt, s, o, lane);
        phase_sync<SHARED>();
        tile_issue<D, RW, WIDE>(vbase, p.v_ss, k0 + CW * 32, S, vt, rw, lane);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the refills past the last block land before LDS is reused or freed

    // element (dt, r): feature acc_row(r) * NT + dt of query n
    float l_tot = sum_xor32(l_run);
    float *orow = static_cast<float *>(p.o) + b * p.o_sb + h * p.o_sh + (int64_t)qi * p.o_ss;
    float *lse = p.lse + (int64_t)bh * S + qi;
    if constexpr (CW == 1) {
        if (qi < S) {
            const float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                float v[NT];
#pragma unroll
                for (int dt = 0; dt < NT; ++dt) v[dt] = o[dt][r] * inv;
                store_nt<NT>(orow + acc_row(r, lane) * NT, v);
            }
            if (g == 0) *lse = l_tot > 0.f ? m_run * p.scale + logf(l_tot) : -INFINITY;
        }
    } else {
        // Groups merge as O = sum_k 2^(m_k - m) O_k / l, in group order; the
        // wave of group cg forms elements r in [cg * 16/CW, +16/CW).
        __syncthreads();  // every wave is done with the tiles
#pragma unroll
        for (int r = 0; r < 16; ++r)
#pragma unroll
            for (int dt = 0; dt < NT; ++dt) *part_slot<D>(ks, vs, wave, r, dt, lane) = o[dt][r];
        if (g == 0) {
            ml[wave * 32 + n] = m_run;
            ml[128 + wave * 32 + n] = l_tot;
        }
        __syncthreads();
        float mk[CW], m = -INFINITY;
#pragma unroll
        for (int k = 0; k < CW; ++k) {
            mk[k] = ml[(k * RW + rw) * 32 + n];
            m = fmaxf(m, mk[k]);
        }
        l_tot = 0.f;
        float wk[CW];
#pragma unroll
        for (int k = 0; k < CW; ++k) {
            wk[k] = mk[k] == -INFINITY ? 0.f : exp2f(mk[k] * c - m * c);
            l_tot += wk[k] * ml[128 + (k * RW + rw) * 32 + n];
        }
        if (qi < S) {
            const float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
#pragma unroll
            for (int rr = 0; rr < 16 / CW; ++rr) {
                const int r = cg * (16 / CW) + rr;
                float v[NT];
#pragma unroll
                for (int dt = 0; dt < NT; ++dt) {
                    float acc = 0.f;
#pragma unroll
                    for (int k = 0; k < CW; ++k) acc += wk[k] * *part_slot<D>(ks, vs, k * RW + rw, r, dt, lane);
                    v[dt] = acc * inv;
                }
                store_nt<NT>(orow + acc_row(r, lane) * NT, v);
            }
            if (g == 0 && cg == 0) *lse = l_tot > 0.f ? m * p.scale + logf(l_tot) : -INFINITY;
        }
    }
}

// Sum of the CW groups' partials of one accumulator array, in group order,
// through LDS; wave (rw, cg) forms elements r in [cg * 16/CW, +16/CW) and
// hands (r, the NT values) to `store`.  Without groups, its own elements.
template <int D, int RW, int CW, typename F>
__device__ __forceinline__ void merge_groups(const f32x16 (&acc)[D / 32], char *pa, char *pb, int wave, int lane, F &&store) {
    constexpr int NT = D / 32;
    if constexpr (CW == 1) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            float v[NT];
#pragma unroll
            for (int dt = 0; dt < NT; ++dt) v[dt] = acc[dt][r];
            store(r, v);
        }
    } else {
        const int rw = wave % RW, cg = wave / RW;
        __syncthreads();  // the tiles (or the previous array's partials) are no longer read
#pragma unroll
        for (int r = 0; r < 16; ++r)
#pragma unroll
            for (int dt = 0; dt < NT; ++dt) *part_slot<D>(pa, pb, wave, r, dt, lane) = acc[dt][r];
        __syncthreads();
#pragma unroll
        for (int rr = 0; rr < 16 / CW; ++rr) {
            const int r = cg * (16 / CW) + rr;
            float v[NT];
#pragma unroll
            for (int dt = 0; dt < NT; ++dt) {
                v[dt] = *part_slot<D>(pa, pb, rw, r, dt, lane);
#pragma unroll
                for (int k = 1; k < CW; ++k) v[dt] += *part_slot<D>(pa, pb, k * RW + rw, r, dt, lane);
            }
            store(r, v);
        }
    }
}

// ---------------------------------------------------------------------------
// dK / dV: a wave owns 32 keys (lane n, K and V rows in registers) and
// streams query blocks.  Per block: dP = dO V^T (dO tile), S = Q K^T (Q tile),
// P and dS, dV += P^T dO, refill dO, dK += dS^T Q, refill Q.
// DS: also store every block's unscaled dS for the dQ product (p.ds), as 32 x
// 32 f32 blocks [key][query] of 4 KiB, block (key / 32, query / 32) of a head
// at (key / 32) * ceil(S / 32) + query / 32.
// ---------------------------------------------------------------------------
constexpr int kDsBlock = 32 * 32;  // elements
template <int D, int RW, int CW, bool WIDE = false, bool DS = false>
__global__ __launch_bounds__(256, D == 128 ? 1 : 2) void attn_bwd_dkdv_f32_kernel(AttnBwdParams p) {
    using T = F32Tile<D>;
    constexpr int NT = D / 32;
    constexpr bool SHARED = RW > 1;
    __shared__ __align__(16) char qsm[F32Lds<D, CW>::TILES], osm[F32Lds<D, CW>::TILES];
    __shared__ __align__(16) float rowv[4 * 64];  // per wave: lse2, then delta of the block's queries
    const int lane = threadIdx.x & 63, n = lane & 31, g = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int rw = wave % RW, cg = wave / RW;
    const int S = p.S, H = p.H;
    const int nk = (S + 32 * RW - 1) / (32 * RW);
    const int work = xcd_remap(blockIdx.x, gridDim.x);
    const int kt = work % nk, bh = work / nk;
    const int h = bh % H, b = bh / H;
    const float *qbase = static_cast<const float *>(p.q) + b * p.q_sb + h * p.q_sh;
    const float *dobase = static_cast<const float *>(p.dout) + b * p.do_sb + h * p.do_sh;
    const float *lse2 = p.lse2 + (int64_t)bh * S, *delta = p.delta + (int64_t)bh * S;
    const int k0 = (kt * RW + rw) * 32, kj = k0 + n;
    const bool kept = kj < S && (!p.keep || p.keep[(int64_t)b * S + kj]);
    char *qs = qsm + cg * T::BYTES, *os = osm + cg * T::BYTES;

    tile_issue<D, RW, WIDE>(dobase, p.do_ss, cg * 32, S, os, rw, lane);
    f32x4 kf[D / 8], vf[D / 8];
    load_rows<D>(static_cast<const float *>(p.k) + b * p.k_sb + h * p.k_sh, p.k_ss, kj, S, g, kf);
    load_rows<D>(static_cast<const float *>(p.v) + b * p.v_sb + h * p.v_sh, p.v_ss, kj, S, g, vf);
    f32x16 dk[NT], dv[NT];
#pragma unroll
    for (int dt = 0; dt < NT; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) dk[dt][r] = dv[dt][r] = 0.f;
    const float c = p.scale_log2;
    const int nqb = (S + 31) / 32, J = (nqb + CW - 1) / CW;
    phase_sync<SHARED>();
    tile_issue<D, RW, WIDE>(qbase, p.q_ss, cg * 32, S, qs, rw, lane);
    for (int j = 0; j < J; ++j) {
        const int q0 = (j * CW + cg) * 32;
        // lane (n, 0) brings query q0 + n's lse2, lane (n, 1) its delta; past
        // S an lse2 of +inf makes P (and dS) zero
        float row = (g ? delta : lse2)[min(q0 + n, S - 1)];
        if (g == 0 && q0 + n >= S) row = INFINITY;
        f32x16 dp = row_product<D>(os, vf, n, g);
        phase_sync<SHARED>();  // the Q tile has landed
        rowv[wave * 64 + lane] = row;
        f32x16 s = row_product<D>(qs, kf, n, g);
#pragma unroll
        for (int grp = 0; grp < 4; ++grp) {
            // elements 4 grp .. +3 are queries 8 grp + 4 g .. +3
            const f32x4 l2 = *reinterpret_cast<const f32x4 *>(rowv + wave * 64 + grp * 8 + g * 4);
            const f32x4 dl = *reinterpret_cast<const f32x4 *>(rowv + wave * 64 + 32 + grp * 8 + g * 4);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int r = grp * 4 + e;
                const float pv = kept ? exp2f(s[r] * c - l2[e]) : 0.f;
                s[r] = pv;
                dp[r] = pv * (dp[r] - dl[e]);
            }
        }
        if constexpr (DS) {
            // elements 4 grp .. +3 of key n: queries 8 grp + 4 g .. +3.  A
            // key past S has zeros (kept is false) and stays inside its block;
            // a padding block of queries, or a wave past the last key, does not exist.
            if (q0 < S && k0 < S) {
                float *blk = static_cast<float *>(p.ds) +
                             (((int64_t)bh * nqb + k0 / 32) * nqb + q0 / 32) * kDsBlock + n * 32 + g * 4;
#pragma unroll
                for (int grp = 0; grp < 4; ++grp)
                    *reinterpret_cast<f32x4 *>(blk + grp * 8) =
                        f32x4{dp[grp * 4], dp[grp * 4 + 1], dp[grp * 4 + 2], dp[grp * 4 + 3]};
            }
        }
        col_product<D, false>(os, s, dv, lane);
        phase_sync<SHARED>();
        tile_issue<D, RW, WIDE>(dobase, p.do_ss, q0 + CW * 32, S, os, rw, lane);
        col_product<D, false>(qs, dp, dk, lane);
        phase_sync<SHARED>();  // the next dO tile has landed
        tile_issue<D, RW, WIDE>(qbase, p.q_ss, q0 + CW * 32, S, qs, rw, lane);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the refills past the last block

    // element (dt, r): key acc_row(r), feature n * NT + dt
    float *dkb = static_cast<float *>(p.dk) + b * p.dk_sb + h * p.dk_sh;
    float *dvb = static_cast<float *>(p.dv) + b * p.dv_sb + h * p.dv_sh;
    merge_groups<D, RW, CW>(dv, qsm, osm, wave, lane, [&](int r, float (&v)[NT]) {
        const int key = k0 + acc_row(r, lane);
        if (key < S) store_nt<NT>(dvb + (int64_t)key * p.dv_ss + n * NT, v);
    });
    merge_groups<D, RW, CW>(dk, qsm, osm, wave, lane, [&](int r, float (&v)[NT]) {
        const int key = k0 + acc_row(r, lane);
#pragma unroll
        for (int dt = 0; dt < NT; ++dt) v[dt] *= p.scale;
        if (key < S) store_nt<NT>(dkb + (int64_t)key * p.dk_ss + n * NT, v);
    });
}

// ---------------------------------------------------------------------------
// dQ: a wave owns 32 queries (lane n, Q and dO rows in registers) and streams
// key blocks.  Per block: dP^T = V dO^T (V tile), refill V, S^T = K Q^T,
// dS, dQ^T += K^T dS^T (K tile), refill K.
// ---------------------------------------------------------------------------
template <int D, int RW, int CW, bool WIDE = false>
__global__ __launch_bounds__(256, D == 128 ? 1 : 2) void attn_bwd_dq_f32_kernel(AttnBwdParams p) {
    using T = F32Tile<D>;
    constexpr int NT = D / 32;
    constexpr bool SHARED = RW > 1;
    __shared__ __align__(16) char ks[F32Lds<D, CW>::TILES], vs[F32Lds<D, CW>::TILES];
    const int lane = threadIdx.x & 63, n = lane & 31, g = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int rw = wave % RW, cg = wave / RW;
    const int S = p.S, H = p.H;
    const int nq = (S + 32 * RW - 1) / (32 * RW);
    const int work = xcd_remap(blockIdx.x, gridDim.x);
    const int qt = work % nq, bh = work / nq;
    const int h = bh % H, b = bh / H;
    const float *kbase = static_cast<const float *>(p.k) + b * p.k_sb + h * p.k_sh;
    const float *vbase = static_cast<const float *>(p.v) + b * p.v_sb + h * p.v_sh;
    const uint8_t *keep = p.keep ? p.keep + (int64_t)b * S : nullptr;
    const int qi = (qt * RW + rw) * 32 + n;
    char *kt = ks + cg * T::BYTES, *vt = vs + cg * T::BYTES;

    tile_issue<D, RW, WIDE>(vbase, p.v_ss, cg * 32, S, vt, rw, lane);
    f32x4 qf[D / 8], of[D / 8];
    load_rows<D>(static_cast<const float *>(p.q) + b * p.q_sb + h * p.q_sh, p.q_ss, qi, S, g, qf);
    load_rows<D>(static_cast<const float *>(p.dout) + b * p.do_sb + h * p.do_sh, p.do_ss, qi, S, g, of);
    float lse2 = INFINITY, dlt = 0.f;
    if (qi < S) {
        lse2 = p.lse2[(int64_t)bh * S + qi];
        dlt = p.delta[(int64_t)bh * S + qi];
    }
    f32x16 dq[NT];
#pragma unroll
    for (int dt = 0; dt < NT; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) dq[dt][r] = 0.f;
    const float c = p.scale_log2;
    const int nkb = (S + 31) / 32, J = (nkb + CW - 1) / CW;
    phase_sync<SHARED>();
    tile_issue<D, RW, WIDE>(kbase, p.k_ss, cg * 32, S, kt, rw, lane);
    for (int j = 0; j < J; ++j) {
        const int k0 = (j * CW + cg) * 32;
        const bool kept = k0 + n < S && (!keep || keep[k0 + n]);
        f32x16 dp = row_product<D>(vt, of, n, g);
        phase_sync<SHARED>();  // the K tile has landed, the V tile is no longer read
        tile_issue<D, RW, WIDE>(vbase, p.v_ss, k0 + CW * 32, S, vt, rw, lane);
        f32x16 s = row_product<D>(kt, qf, n, g);
        const uint32_t km = (uint32_t)__ballot(kept);
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            float pv = exp2f(s[r] * c - lse2);
            if (km != ~0u && !((km >> acc_row(r, lane)) & 1)) pv = 0.f;
            dp[r] = pv * (dp[r] - dlt);
        }
        col_product<D, true>(kt, dp, dq, lane);
        phase_sync<SHARED>();
        tile_issue<D, RW, WIDE>(kbase, p.k_ss, k0 + CW * 32, S, kt, rw, lane);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the refills past the last block

    // element (dt, r): feature acc_row(r) * NT + dt of query n
    float *row = static_cast<float *>(p.dq) + b * p.dq_sb + h * p.dq_sh + (int64_t)qi * p.dq_ss;
    merge_groups<D, RW, CW>(dq, ks, vs, wave, lane, [&](int r, float (&v)[NT]) {
#pragma unroll
        for (int dt = 0; dt < NT; ++dt) v[dt] *= p.scale;
        if (qi < S) store_nt<NT>(row + acc_row(r, lane) * NT, v);
    });
}

// ---------------------------------------------------------------------------
// dQ from the stored dS (B1 H24 S1536 D128: the backward 991 -> 689 us): dQ^T += K^T dS^T, one third of the recomputing
// kernel's products.  Both operands are whole rows (512 bytes of K and 128 of
// dS per lane half), so they come straight from memory into registers, a block
// ahead of the block being multiplied; no tile, no barrier before the merge.
// The same products in the same order as attn_bwd_dq_f32_kernel, so the same
// bits.
// ---------------------------------------------------------------------------
template <int D, int RW, int CW>
__global__ __launch_bounds__(256, 2) void attn_bwd_dq_ds_f32_kernel(AttnBwdParams p) {
    constexpr int NT = D / 32;
    __shared__ __align__(16) char pa[CW > 1 ? F32Lds<D, CW>::PART : 16], pb[CW > 1 ? F32Lds<D, CW>::PART : 16];
    const int lane = threadIdx.x & 63, n = lane & 31, g = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int rw = wave % RW, cg = wave / RW;
    const int S = p.S, H = p.H;
    const int nq = (S + 32 * RW - 1) / (32 * RW);
    const int work = xcd_remap(blockIdx.x, gridDim.x);
    const int qt = work % nq, bh = work / nq;
    const int h = bh % H, b = bh / H;
    const float *kbase = static_cast<const float *>(p.k) + b * p.k_sb + h * p.k_sh;
    const int q32 = qt * RW + rw, qi = q32 * 32 + n;
    const int nkb = (S + 31) / 32;
    const uint32_t kstep = (uint32_t)(p.k_ss * 4);  // launched for k_ss < kWideStride only
    // head bh's dS blocks of this wave's queries: block kb at kb * nkb
    const float *ds = static_cast<const float *>(p.ds) + ((int64_t)bh * nkb * nkb + q32) * kDsBlock;

    // Steps of half a block (8 of its 16 key pairs): two sets of 8 (NT + 1)
    // operands beside the 16 NT accumulators leave room for two or three
    // waves per SIMD, whose MFMAs cover the loads' latency.
    struct Operands {
        float k[8][NT], ds[8];  // element u of half hf: key acc_row(8 hf + u)
    };
    // Blocks of keys past S read as zero (a descriptor of no bytes)
    auto load = [&](int kb, int hf, Operands &x) {
        const int rows = min(32, S - kb * 32);
        const __amdgpu_buffer_rsrc_t krs =
            make_rsrc(kbase + (int64_t)kb * 32 * p.k_ss, rows > 0 ? (uint32_t)(((rows - 1) * p.k_ss + D) * 4) : 0u);
        const __amdgpu_buffer_rsrc_t srs =
            make_rsrc(ds + (int64_t)kb * nkb * kDsBlock, rows > 0 && q32 < nkb ? kDsBlock * 4u : 0u);
        const uint32_t kv = (uint32_t)(4 * g) * kstep + (uint32_t)(n * NT * 4), sv = (uint32_t)(4 * g * 32 + n) * 4;
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const uint32_t r = (uint32_t)(hf * 16 + (u >> 2) * 8 + (u & 3));  // acc_row(8 hf + u, lane) - 4 g
            x.ds[u] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(srs, sv, r * 128, 0));
            if constexpr (NT == 4) {
                const f32x4 v = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(krs, kv, r * kstep, 0));
#pragma unroll
                for (int e = 0; e < 4; ++e) x.k[u][e] = v[e];
            } else {
                typedef float f32x2 __attribute__((ext_vector_type(2)));
                const f32x2 v = __builtin_bit_cast(f32x2, __builtin_amdgcn_raw_buffer_load_b64(krs, kv, r * kstep, 0));
                x.k[u][0] = v[0];
                x.k[u][1] = v[1];
            }
        }
    };
    f32x16 dq[NT];
#pragma unroll
    for (int dt = 0; dt < NT; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) dq[dt][r] = 0.f;
    auto step = [&](int next, int next_half, const Operands &x, Operands &y) {
        load(next, next_half, y);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < 8; ++u)
#pragma unroll
            for (int dt = 0; dt < NT; ++dt) dq[dt] = mfma_32x32x2_f32(x.k[u][dt], x.ds[u], dq[dt]);
        __builtin_amdgcn_sched_barrier(0);
    };
    Operands x0, x1;
    load(cg, 0, x0);
    for (int kb = cg; kb < nkb; kb += CW) {
        step(kb, 1, x0, x1);
        step(kb + CW, 0, x1, x0);  // past the last block: zeros, not used
    }
    float *row = static_cast<float *>(p.dq) + b * p.dq_sb + h * p.dq_sh + (int64_t)qi * p.dq_ss;
    merge_groups<D, RW, CW>(dq, pa, pb, wave, lane, [&](int r, float (&v)[NT]) {
#pragma unroll
        for (int dt = 0; dt < NT; ++dt) v[dt] *= p.scale;
        if (qi < S) store_nt<NT>(row + acc_row(r, lane) * NT, v);
    });
}

// Groups per workgroup (1, 2 or 4): the busiest CU runs ceil(workgroups / CUs)
// workgroups of ceil(blocks / groups) blocks each, plus about a block's time
// per workgroup for its first loads and its merge.  Ties go to fewer groups
// (more waves share each tile).  Forward us with 1, 2 and 4 groups at D = 128:
// B1 H24 S1536 398, 311, 294; B2 H24 S1536 583, 496, 529; B1 H16 S4096 1011,
// 1027, 1169; B1 H8 S1024 142, 83, 50: the rule takes the fastest of each.
int f32_groups(int B, int H, int S) {
    const int64_t cus = device_cu_count(), nb = (S + 31) / 32;
    int best = 1;
    int64_t best_cost = -1;
    for (int cw : {1, 2, 4}) {
        const int64_t rows = 128 / cw, wgs = (int64_t)B * H * ((S + rows - 1) / rows);
        const int64_t cost = (wgs + cus - 1) / cus * ((nb + cw - 1) / cw + 1);
        if (best_cost < 0 || cost < best_cost) best = cw, best_cost = cost;
    }
    return best;
}

}  // namespace

// Calls f(D, RW, CW) as integral constants for a call's shape.
template <typename F>
void f32_shape(int D, int cw, F &&f) {
    auto go = [&](auto d) {
        if (cw == 1)
            f(d, std::integral_constant<int, 4>{}, std::integral_constant<int, 1>{});
        else if (cw == 2)
            f(d, std::integral_constant<int, 2>{}, std::integral_constant<int, 2>{});
        else
            f(d, std::integral_constant<int, 1>{}, std::integral_constant<int, 4>{});
    };
    if (D == 128)
        go(std::integral_constant<int, 128>{});
    else
        go(std::integral_constant<int, 64>{});
}

// Launches kern<D, RW, CW, ...>(p), one workgroup per RW * 32 rows.
#define FA_F32_GO(params, ...)                                                                       \
    hipLaunchKernelGGL((__VA_ARGS__),                                                                \
                       dim3((unsigned)((params).B * (params).H * (((params).S + 32 * RW - 1) / (32 * RW)))), dim3(256), 0, s, params)

hipError_t launch_attn_fwd_f32(const AttnFwdParams &p, int D, hipStream_t s) {
    const bool wide = p.k_ss >= kWideStride || p.v_ss >= kWideStride;
    f32_shape(D, wide ? 1 : f32_groups(p.B, p.H, p.S), [&](auto d, auto rw, auto cw) {
        constexpr int Dv = decltype(d)::value, RW = decltype(rw)::value, CW = decltype(cw)::value;
        if constexpr (CW == 1) {  // the only shape of tiles of 4 GiB or more
            if (wide) {
                FA_F32_GO(p, attn_fwd_f32_kernel<Dv, RW, CW, true>);
                return;
            }
        }
        FA_F32_GO(p, attn_fwd_f32_kernel<Dv, RW, CW>);
    });
    return hipGetLastError();
}

// The one-call backward with room for dS (p.ds) stores it in dK/dV and forms
// dQ from it; the separate phases, and tiles of 4 GiB or more, recompute it,
// so that dK/dV and dQ stay independent there.
hipError_t launch_attn_bwd_f32(const AttnBwdParams &p, int D, int phase, hipStream_t s) {
    if (phase == 0 || phase == 1) {
        const hipError_t e = launch_attn_bwd_delta_f32(p, D, s);
        if (e != hipSuccess || phase == 1) return e;
    }
    const bool wide = p.q_ss >= kWideStride || p.do_ss >= kWideStride || p.k_ss >= kWideStride || p.v_ss >= kWideStride;
    const bool ds = p.ds && phase == 0 && !wide;
    f32_shape(D, wide ? 1 : f32_groups(p.B, p.H, p.S), [&](auto d, auto rw, auto cw) {
        constexpr int Dv = decltype(d)::value, RW = decltype(rw)::value, CW = decltype(cw)::value;
        if (ds) {
            FA_F32_GO(p, attn_bwd_dkdv_f32_kernel<Dv, RW, CW, false, true>);
            FA_F32_GO(p, attn_bwd_dq_ds_f32_kernel<Dv, RW, CW>);
            return;
        }
        if constexpr (CW == 1) {
            if (wide) {
                if (phase != 3) FA_F32_GO(p, attn_bwd_dkdv_f32_kernel<Dv, RW, CW, true>);
                if (phase != 2) FA_F32_GO(p, attn_bwd_dq_f32_kernel<Dv, RW, CW, true>);
                return;
            }
        }
        if (phase != 3) FA_F32_GO(p, attn_bwd_dkdv_f32_kernel<Dv, RW, CW>);
        if (phase != 2) FA_F32_GO(p, attn_bwd_dq_f32_kernel<Dv, RW, CW>);
    });
    return hipGetLastError();
}

}  // namespace fa
