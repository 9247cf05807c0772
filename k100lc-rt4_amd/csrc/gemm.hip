// gemm.hip -- RT4 W4A8 prefill GEMM on gfx950 int8 matrix cores.
//
//   C[m][n] = Σ_g sa[g][m] * sb[g][n] * I[m][n][g],
//   I[m][n][g] = Σ_{k in group g} q8[m][k] * code[n][k]        (exact int32)
//
// with q8 the prefill activation codes (quant_rows_a8_k semantics, src/k_new.hip:
// 268-301: q8 = 16h + l), sa their per-(group, row) scale (`sc`), code the RT4 int4
// weights and sb the fp32 group-major weight scales (src/model.cpp:190-202).
//
// The reference computes this as two int4 x int4 passes over the digit planes h
// and l plus an add (k_gemm_i4_a8, src/k_gemm.hip:22-34; kernel gemm_w4a4,
// kernels/gemm_core.h:59-206).  Per group its integer content is
// 16*I_h + I_l = I exactly, so here the digits are recombined into int8 once
// and a single int8 contraction runs on v_mfma_i32_32x32x32_i8.
//
// Tiling.  Workgroup tile 32 RT activation rows x 256 weight rows, 8 waves; wave w
// owns weight rows (output columns) 32w..32w+31 and all the activation rows, i.e. RT
// 32 x 32 row tiles (four, unless M is small) sharing one weight fragment, so each wave
// unpacks only its own 32 weight rows.  One 128-wide K group ("unit" = one tile x one group)
// is four MFMA k-steps per row tile.  The int32 accumulators restart at every
// group and are folded into fp32:
//     facc += f32(acc) * S,   S = sa * sb,   acc = 16*I exactly (x16 nibble unpack),
// and the result is scaled by 1/16 once at the end (a power of two, so the bits
// equal those of scaling every term).  S is formed on the matrix core: one
// two-block fp32 outer product (v_mfma_f32_32x32x1_2b_f32) per pair of row tiles
// gives sa (x) sb for both in the accumulator layout of the int8 tiles (block b:
// the activation scales of row tile 2p + b from lanes 32b..32b+31, the weight
// scale of the lane's column in both halves).  Every element is one fp32
// product, so S is sa * sb correctly rounded, as the reference forms it
// (kernels/gemm_core.h:183).  Against four bf16 MFMAs on exact 3-part splits of
// both scales (the earlier form, within a few ulp) it drops the split work of
// every wave and one LDS pass per unit: C2 gate/up 143 -> 139 us, measured.
//
// What bounds this kernel on gfx950 is instruction issue: measured, a SIMD with
// two such waves issues about one instruction per 4 cycles whatever its kind
// (scalar, vector, LDS; an int8 MFMA takes about 16), with little overlap
// between the two waves, and the fold alone is two vector instructions per
// output per group (128 per wave per unit against 16 MFMAs).  So the
// loop is built for few instructions: every LDS read address is a per-lane
// register (moved on by one stage per unit, one add per register) plus the row
// tile as an immediate offset (a body unrolled over the four stages, which would
// make the stage an immediate too, spilled around the flush); the DMA
// sources are the kernel's scalar base pointers plus per-lane 32-bit offsets,
// moved on by one group per unit (advancing the scalar bases instead measured
// the same); tile bookkeeping is a few scalar counters.  The MFMAs of a row tile are interleaved one by one with the
// fold of the previous row tile (and with the unpack of the next k-step), in an
// order the compiler may not change (sched_barrier; every folded value also
// passes through an empty asm statement where it is formed, without which the
// compiler sinks three of the four folds of a unit past the barrier into one
// block and spills), so the matrix core and the vector ALU work at the same
// time and no fold waits for the MFMA just issued.
//
// Data movement.  Per unit the workgroup moves 16 KB of int8 activations, 16 KB
// of packed weights and the two scale vectors from global memory straight into
// LDS with global_load_lds_dwordx4 (no VGPR round trip), four stages deep (the
// unit three ahead is loading while a unit computes).  Each wave loads exactly
// the weight rows it reads; the activation tile is shared by all waves (one
// barrier per unit).  LDS layouts are XOR-swizzled for gfx950's 64-bank LDS: any
// 16 consecutive fragment rows of a ds_read_b128 hit 16 distinct 16-byte bank
// groups.
//
// Scheduling.  One persistent workgroup per CU.  With `rem` the tile count modulo the
// workgroup count, the first rem tiles are shared out by (tile, group) units, an equal
// contiguous range each; every workgroup then takes the same number of whole tiles.
// Whole tiles need no partial sums: at M=1024, N=17408, K=5120 (544 tiles) two of the
// three segments of a workgroup are whole, where equal ranges over all units ("stream-K"
// throughout) made two of three split: 64 MB of partials written and read back became 32
// (144 -> 127 us with the combining below; M=2048 262 -> 249).  A part of a tile goes to
// a workspace slot, and the parts are summed in range order, by gemm_combine_k or (INL, see
// gemm_plan) by the workgroup of the tile that counts in last: results do not depend on
// timing and no workgroup waits for another.  Workgroups of one XCD take neighbouring
// tiles (the same weights).
//
// Row tiles.  RT = 4 (128 rows) from 65 rows up; RT = 2 and 1 for up to 64 and 32 rows,
// whose units issue less (a unit of RT = 4 takes ~1.36 us here, RT = 2 0.87, RT = 1 0.60:
// the weight unpack, the barrier and the bookkeeping stay) and whose partials are half
// and a quarter of the size.  N=17408 K=5120, GEMM and combining launch, us: M=37 33.7 ->
// 16.2 + 4.9, of which the weights' one-pass read alone is 8.4; the 128-row form computed
// all 128 rows for any M.
#include "rt4_dev.h"
#include "rt4_internal.h"

namespace rt4 {
namespace {

typedef __attribute__((address_space(3))) void lds_void;
typedef unsigned v4u __attribute__((ext_vector_type(4)));
typedef float v32f __attribute__((ext_vector_type(32)));

constexpr int BN = 256;           // weight rows (output columns) per tile
constexpr int NT = 512;           // 8 waves
constexpr int NS = 4;             // LDS stages
constexpr int B_ST = BN * 64;     // packed weight tile per stage
constexpr int S_ST = 2048;        // sa (512 B) + sb (1024 B) + 512 B written by the two idle waves

// Sizes that depend on the row tiles per workgroup tile, RT = 1, 2 or 4 (32, 64 or 128
// activation rows).
template <int RT>
struct Tile {
    static constexpr int BM = 32 * RT;
    static constexpr int A_DMA = RT == 4 ? 2 : 1;         // activation DMA instructions per wave (8 rows each)
    static constexpr int A_ST = A_DMA * 8 * 1024;         // int8 activation rows per stage (64 for RT = 1 too:
                                                          // rows 32.. are loaded and not read)
    static constexpr int LDS_B = 0;                       // weight stages
    static constexpr int LDS_A = LDS_B + NS * B_ST;       // activation stages
    static constexpr int LDS_S = LDS_A + NS * A_ST;       // scale stages
    static constexpr int LDS_BYTES = LDS_S + NS * S_ST;
    static constexpr int DMA_PER_UNIT = A_DMA + 3;        // DMA instructions per wave per unit
    static constexpr int PART_FLOATS = NT * 16 * RT;      // one partial tile: 16 RT outputs per thread, [k][thread]
};

// Split-tile partials are written by buffer stores with the device-scope cache policy (sc1,
// that of agent-scope atomics): they write through the per-XCD L2 and are in memory once
// the writer's s_waitcnt has retired them.  gemm_combine_k, a launch of its own, reads them
// with plain loads; a workgroup that sums them in the same launch reads them with sc1, the
// coherent copy, all 4 RT loads of one part in flight together.
constexpr int kSc1 = 16;               // cache policy: sc1
constexpr int kRsrcW3 = 0x00020000;    // dword 3 of a buffer resource: 32-bit data format
template <int RT>
__device__ __forceinline__ __amdgpu_buffer_rsrc_t part_rsrc(float* part, int slot) {
    return __builtin_amdgcn_make_buffer_rsrc(part + (size_t)slot * Tile<RT>::PART_FLOATS, 0,
                                             Tile<RT>::PART_FLOATS * (int)sizeof(float), kRsrcW3);
}

// Per-lane byte offsets of this wave's DMA sources for one tile (relative to the
// unit's scalar bases), unchanged while the tile is.  LDS layouts:
//   A  [rows][8 x 16 B], 16-byte chunk c of row r stored at c ^ ((r >> 1) & 7); wave w
//      loads rows 8w.. (RT = 4: 16w.., two instructions), 8 rows x 128 B each
//   B  [256 rows][4 x 16 B] packed, chunk c of row r stored at c ^ ((r >> 2) & 3);
//      wave w loads rows 32w..32w+31, the ones it reads
//   S  sa[128] f32 (waves 0, 1), sb[256] f32 (waves 2..5); waves 6, 7 repeat an sb
//      load into the spare 512 B so that every wave issues the same count.
template <int RT>
struct DmaOff {
    uint32_t a[Tile<RT>::A_DMA], b[2], s;
};
template <int RT>
__device__ __forceinline__ DmaOff<RT> dma_offsets(int bm, int bn, int M, int N, int K, int w, int lane) {
    constexpr int A_DMA = Tile<RT>::A_DMA;
    DmaOff<RT> o;
#pragma unroll
    for (int t = 0; t < A_DMA; t++) {
        const int r = 8 * (A_DMA * w + t) + (lane >> 3);
        const int c = (lane & 7) ^ ((r >> 1) & 7);
        const int gr = min(bm + r, M - 1);
        o.a[t] = (uint32_t)gr * (uint32_t)K + c * 16;
    }
#pragma unroll
    for (int t = 0; t < 2; t++) {
        const int r = 32 * w + 16 * t + (lane >> 2);
        const int c = (lane & 3) ^ ((r >> 2) & 3);
        const int gr = min(bn + r, N - 1);
        o.b[t] = (uint32_t)gr * (uint32_t)(K >> 1) + c * 16;
    }
    if (w < 2)
        o.s = (uint32_t)min(bm + 64 * w + lane, M - 1) * 4u;
    else
        o.s = (uint32_t)min(bn + 64 * ((w - 2) & 3) + lane, N - 1) * 4u;
    return o;
}

// First unit of range b: floor(R b / Pr) with R = q Pr + r, in 32 bits (rem < 2^16 tiles,
// r and b < Pr <= the CU count).
__device__ __forceinline__ int range_start(const GemmSched& s, int b) {
    return s.q * b + (int)((unsigned)(s.r * b) / (unsigned)s.Pr);
}
// The range that holds unit u: an estimate, corrected to range_start(b) <= u < range_start(b + 1).
__device__ __forceinline__ int owner_of(const GemmSched& s, int u) {
    int b = (int)((float)u / ((float)s.q + (float)s.r / (float)s.Pr));
    b = min(max(b, 0), s.Pr - 1);
    while (range_start(s, b) > u) b--;
    while (range_start(s, b + 1) <= u) b++;
    return b;
}

// Tile coordinates of a unit, as the flush and the group-sum stores need them.
struct TileRef {
    int t, bm, bn, g;
};

template <int RT, bool GSUM, bool INL>
__global__ __launch_bounds__(NT, 1) void gemm_w4a8_k(const int8_t* __restrict__ A,
                                                     const uint32_t* __restrict__ W,
                                                     const float* __restrict__ sa,
                                                     const float* __restrict__ sb,
                                                     float* __restrict__ C,
                                                     int32_t* __restrict__ gsum,
                                                     float* __restrict__ part, int* __restrict__ cnt,
                                                     int M, int N, int K, GemmSched sch) {
    using TL = Tile<RT>;
    constexpr int BM = TL::BM, A_ST = TL::A_ST, DMA_PER_UNIT = TL::DMA_PER_UNIT;
    constexpr int LDS_A = TL::LDS_A, LDS_B = TL::LDS_B, LDS_S = TL::LDS_S;
    __shared__ __align__(16) unsigned char lds[TL::LDS_BYTES];
    __shared__ int s_last;
    const int lane = threadIdx.x & 63;
    const int w = uniform(threadIdx.x >> 6);
    const int lr = lane & 31, lh = lane >> 5;
    const int NG = K >> 7;
    const int P = gridDim.x;
    // b: this workgroup's number, consecutive ones on one XCD (workgroups are dealt to the
    // eight XCDs in turn).  rg: its range of the remainder tiles' units, -1 for none: b, or
    // (sch.spread) the ranges dealt evenly to the XCDs, consecutive ones on one XCD.
    const int x = (int)(blockIdx.x % 8u), j = (int)(blockIdx.x / 8u);
    const int b = P % 8 == 0 ? x * (P / 8) + j : (int)blockIdx.x;
    int rg = b < sch.Pr ? b : -1;
    if (sch.spread) {
        const int pq = sch.Pr >> 3, pr = sch.Pr & 7;
        rg = j < pq + (x < pr ? 1 : 0) ? x * pq + min(x, pr) + j : -1;
    }
    // This workgroup's work: its range [r0, r1) of the remainder tiles' units (the first
    // sch.rem tiles, shared by sch.Pr workgroups), then sch.full whole tiles, P apart.
    // rl_t, rl_e: the last remainder tile of the range and the group it ends before (-1:
    // no range).
    const int ntm = sch.ntm;
    const int r0 = rg >= 0 ? range_start(sch, rg) : 0, r1 = rg >= 0 ? range_start(sch, rg + 1) : 0;
    const int n = r1 - r0 + sch.full * NG;
    if (n == 0) return;
    const int rl_t = r1 > r0 ? (r1 - 1) / NG : -1, rl_e = r1 > r0 ? r1 - rl_t * NG : 0;
    const int t_first = r1 > r0 ? r0 / NG : sch.rem + b;
    const int g_first = r1 > r0 ? r0 - t_first * NG : 0;
    auto next_tile = [&](int t) __attribute__((always_inline)) -> int {
        return t < rl_t ? t + 1 : t < sch.rem ? sch.rem + b : t + P;
    };
    auto seg_end = [&](int t) __attribute__((always_inline)) -> int { return t == rl_t ? rl_e : NG; };

    // per-lane LDS read offsets into the current stage (next_stage moves them on);
    // the row tile is an immediate
    int ra[4];
#pragma unroll
    for (int ks = 0; ks < 4; ks++) ra[ks] = LDS_A + lr * 128 + (((4 * (ks >> 1) + 2 * lh + (ks & 1)) ^ ((lr >> 1) & 7)) * 16);
    int rb[2];
#pragma unroll
    for (int s2 = 0; s2 < 2; s2++) {
        const int r = 32 * w + lr;
        rb[s2] = LDS_B + r * 64 + (((2 * s2 + lh) ^ ((r >> 2) & 3)) * 16);
    }
    // sa of row 64p + lane (row tile 2p in lanes 0..31, 2p + 1 in lanes 32..63) at
    // rsa + 256p; sb of this lane's column at rsb
    int rsa = LDS_S + lane * 4, rsb = LDS_S + 512 + (32 * w + lr) * 4;
    // per-wave LDS destinations of the DMA (m0 = base + stage immediate)
    const uint32_t L = lds_addr(lds);
    const uint32_t dstA = L + LDS_A + TL::A_DMA * w * 1024, dstB = L + LDS_B + 2 * w * 1024;
    const uint32_t dstS = L + LDS_S + (w < 2 ? w * 256 : w < 6 ? 512 + (w - 2) * 256 : 1536);

    // facc[ii]: row tile ii (rows 32 ii..32 ii+31) x this wave's 32 columns; lane (lr, lh)
    // holds column 32w + lr, rows 32 ii + 8q + 4lh + e in register 4q + e.
    v16i facc[RT];
#pragma unroll
    for (int i = 0; i < RT; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) facc[i][r] = 0;

    const v16i zero16 = {};
    const v32f zero32f = {};
    auto unpack_ks = [&](v4i (&bu_)[4], const uint4 (&bp_)[2], int ks) {
        const uint4 p = bp_[ks >> 1];
        const uint32_t x0 = (ks & 1) ? p.z : p.x, x1 = (ks & 1) ? p.w : p.y;
        bu_[ks] = v4i{(int)even_x16(x0), (int)odd_x16(x0), (int)even_x16(x1), (int)odd_x16(x1)};
    };
    // Scale products of row tiles 2p and 2p + 1: the two-block outer product
    // (v_mfma_f32_32x32x1_2b_f32; block b takes its rows from lanes 32b..32b+31 and
    // its columns from the same lanes) of sa[64p + lane] and sb[this lane's column]
    // puts sa[row of register r] * sb[column] of tile 2p + b in register 16b + r,
    // the accumulator layout of the int8 tiles.
    auto scales2 = [&](float sa_pair, float sb_col) __attribute__((always_inline)) -> v32f {
        return __builtin_amdgcn_mfma_f32_32x32x1f32(sa_pair, sb_col, zero32f, 0, 0, 0);
    };
    auto slo = [](const v32f& v) __attribute__((always_inline)) -> v16f {
        return __builtin_shufflevector(v, v, 0, 1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15);
    };
    auto shi = [](const v32f& v) __attribute__((always_inline)) -> v16f {
        return __builtin_shufflevector(v, v, 16, 17, 18, 19, 20, 21, 22, 23, 24, 25, 26, 27, 28, 29, 30, 31);
    };
    // quarter q of the fold of row tile ii (registers 4q..4q+3)
    auto fold_q = [&](v16i& fa, const v16i& acc, const v16f& S, int ii, int q, const TileRef& x) __attribute__((always_inline)) {
#pragma unroll
        for (int r = 4 * q; r < 4 * q + 4; r++) {
            int v = __float_as_int(fmaf((float)acc[r], S[r], __int_as_float(fa[r])));
            asm volatile("" : "+v"(v));   // formed here, not sunk past the next MFMAs
            fa[r] = v;
        }
        if (GSUM && x.g >= 0) {
            const int nn = x.bn + 32 * w + lr;
#pragma unroll
            for (int r = 4 * q; r < 4 * q + 4; r++) {
                const int m = x.bm + 32 * ii + 8 * (r >> 2) + 4 * lh + (r & 3);
                if (m < M && nn < N) gsum[((size_t)m * N + nn) * NG + x.g] = acc[r] >> 4;
            }
        }
    };

    // C of the tile at (bm, bn) from f.  A wave whose columns all exist in a tile whose
    // rows all exist stores with the row as a scalar offset (one vector instruction per
    // value besides the store, where 64-bit addresses took four); edges go row by row
    // with the buffer's range check dropping the rows past M, and drain their stores.
    // (N passes through an empty asm: the row offsets are then formed here, in this
    // rare path, instead of being hoisted out of the loops into registers.)
    auto write_c = [&](const v16i (&f)[RT], int bm, int bn) __attribute__((always_inline)) {
        uint32_t Nb = (uint32_t)N * 4u;
        asm volatile("" : "+s"(Nb));
        const uint32_t nn = (uint32_t)(bn + 32 * w + lr);
        const int rows = min(M - bm, BM);
        const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
            reinterpret_cast<char*>(C) + (size_t)bm * Nb, 0, (int)((uint32_t)rows * Nb), kRsrcW3);
        const uint32_t vo = (uint32_t)(4 * lh) * Nb + nn * 4u;
        if (rows == BM && bn + 32 * w + 32 <= N) {
#pragma unroll
            for (int ii = 0; ii < RT; ii++)
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(__int_as_float(f[ii][r]) * 0.0625f), rs, vo,
                                                          (32 * ii + 8 * (r >> 2) + (r & 3)) * Nb, 0);
                    __builtin_amdgcn_sched_barrier(0);
                }
        } else {
            if (nn < (uint32_t)N) {
#pragma unroll
                for (int ii = 0; ii < RT; ii++)
                    if (32 * ii < rows) {
#pragma unroll
                        for (int r = 0; r < 16; r++) {
                            __builtin_amdgcn_raw_buffer_store_b32(
                                __float_as_uint(__int_as_float(f[ii][r]) * 0.0625f), rs,
                                vo + (32 * ii + 8 * (r >> 2) + (r & 3)) * Nb, 0, 0);
                            __builtin_amdgcn_sched_barrier(0);
                        }
                    }
            }
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        }
    };
    // End of this workgroup's segment of tile x.t: a whole tile is written out; a part
    // of one goes to its partial slot, 2 rg for this workgroup's first tile and 2 rg + 1 for
    // its last remainder tile, for gemm_combine_k or (INL) the tile's last contributor.  No
    // other workgroup is waited for.
    auto flush = [&](const TileRef& x, bool whole) __attribute__((always_inline)) {
        if (whole) {
            write_c(facc, x.bm, x.bn);
        } else {
            const __amdgpu_buffer_rsrc_t rs = part_rsrc<RT>(part, 2 * rg + (x.t == t_first ? 0 : 1));
#pragma unroll
            for (int ii = 0; ii < RT; ii++)
#pragma unroll
                for (int q = 0; q < 4; q++)
                    __builtin_amdgcn_raw_buffer_store_b128(
                        v4u{(unsigned)facc[ii][4 * q], (unsigned)facc[ii][4 * q + 1], (unsigned)facc[ii][4 * q + 2],
                            (unsigned)facc[ii][4 * q + 3]},
                        rs, threadIdx.x * 16, (4 * ii + q) * NT * 16, kSc1);
            if constexpr (INL) {
                // counted in for this tile once every wave's stores are in memory; the
                // workgroup that counts last sums the parts, in range order
                const int wf = owner_of(sch, x.t * NG), wl = owner_of(sch, x.t * NG + NG - 1);
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                __syncthreads();
                if (threadIdx.x == 0)
                    s_last = __hip_atomic_fetch_add(cnt + x.t, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == wl - wf;
                __syncthreads();
                if (s_last) {
                    const int slot_f = 2 * wf + (range_start(sch, wf) == x.t * NG ? 0 : 1);
#pragma unroll
                    for (int ii = 0; ii < RT; ii++)
#pragma unroll
                        for (int r = 0; r < 16; r++) facc[ii][r] = 0;
                    for (int v = wf; v <= wl; v++) {
                        const __amdgpu_buffer_rsrc_t ps = part_rsrc<RT>(part, v == wf ? slot_f : 2 * v);
                        v4u p[4 * RT];
#pragma unroll
                        for (int e = 0; e < 4 * RT; e++)
                            p[e] = __builtin_amdgcn_raw_buffer_load_b128(ps, threadIdx.x * 16, e * NT * 16, kSc1);
#pragma unroll
                        for (int e = 0; e < 4 * RT; e++)
#pragma unroll
                            for (int c = 0; c < 4; c++)
                                facc[e >> 2][4 * (e & 3) + c] = __float_as_int(
                                    __int_as_float(facc[e >> 2][4 * (e & 3) + c]) + __uint_as_float(p[e][c]));
                    }
                    write_c(facc, x.bm, x.bn);
                    if (threadIdx.x == 0)
                        __hip_atomic_store(cnt + x.t, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
            }
        }
#pragma unroll
        for (int ii = 0; ii < RT; ii++)
#pragma unroll
            for (int r = 0; r < 16; r++) facc[ii][r] = 0;
    };

    // ---- DMA side: the unit being loaded.  Its sources are the kernel arguments
    // (scalar bases) plus per-lane 32-bit offsets that hold the row, the chunk and
    // the group: each unit adds one group to them, a new tile recomputes them.
    int dt = t_first, dleft = seg_end(t_first) - g_first;
    int dtn = dt / ntm, dtm = dt - dtn * ntm;
    const void* sbase = (w < 2 ? (const void*)sa : (const void*)sb);
    const uint32_t s_step = (w < 2 ? (uint32_t)M : (uint32_t)N) * 4u;
    DmaOff<RT> off = dma_offsets<RT>(dtm * BM, dtn * BN, M, N, K, w, lane);
    // the group moves the (scalar) source bases; the per-lane offsets change per tile
    const char* bA = reinterpret_cast<const char*>(A) + (size_t)g_first * 128;
    const char* bW = reinterpret_cast<const char*>(W) + (size_t)g_first * 64;
    const char* bS = reinterpret_cast<const char*>(sbase) + (size_t)g_first * s_step;
    // DMA of the unit at the DMA side's position into stage st
    auto issue = [&](int st) __attribute__((always_inline)) {
        const uint32_t da = dstA + st * A_ST, db = dstB + st * B_ST, ds = dstS + st * S_ST;
        dma16<0>(off.a[0], bA, da);
        if constexpr (TL::A_DMA == 2) dma16<1024>(off.a[1], bA, da);
        dma16<0>(off.b[0], bW, db);
        dma16<1024>(off.b[1], bW, db);
        dma4<0>(off.s, bS, ds);
    };
    auto advance_dma = [&]() __attribute__((always_inline)) {
        if (--dleft == 0) {
            dt = next_tile(dt);
            dleft = seg_end(dt);
            dtn = dt / ntm;
            dtm = dt - dtn * ntm;
            off = dma_offsets<RT>(dtm * BM, dtn * BN, M, N, K, w, lane);
            bA = reinterpret_cast<const char*>(A);
            bW = reinterpret_cast<const char*>(W);
            bS = reinterpret_cast<const char*>(sbase);
        } else {
            bA += 128;
            bW += 64;
            bS += s_step;
        }
    };

    // ---- compute side: the tile of the current segment of units
    TileRef cur;
    auto set_tile = [&](int t) __attribute__((always_inline)) {
        const int tn = t / ntm;
        cur.t = t;
        cur.bm = (t - tn * ntm) * BM;
        cur.bn = tn * BN;
    };
    set_tile(t_first);
    cur.g = g_first;

    // prologue: DMA of units 0..3, then the fragments of unit 0
    issue(0);
    if (n > 1) { advance_dma(); issue(1); }
    if (n > 2) { advance_dma(); issue(2); }
    if (n > 3) { advance_dma(); issue(3); }
    if (n > 3) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(3 * DMA_PER_UNIT) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    v4i a_cur[4], a_nxt[4], bu[4];
    uint4 bp[2];
    // fragment reads: per-lane offsets into the current stage (moved on by one stage
    // per unit: one add per register) plus the row tile (an immediate).  The adds
    // are asm with the register tied in place: written in C, the compiler kept the
    // old and the new offsets alive together and spent 17 adds and 4 moves per
    // unit on the 8 updates (C2 gate/up 139 -> 138 us with them in place).
    auto next_stage = [&](int st_next) __attribute__((always_inline)) {
        const int da = st_next ? A_ST : -(NS - 1) * A_ST, db = st_next ? B_ST : -(NS - 1) * B_ST;
        const int ds = st_next ? S_ST : -(NS - 1) * S_ST;
#pragma unroll
        for (int ks = 0; ks < 4; ks++) asm volatile("v_add_u32 %0, %1, %0" : "+v"(ra[ks]) : "s"(da));
#pragma unroll
        for (int s2 = 0; s2 < 2; s2++) asm volatile("v_add_u32 %0, %1, %0" : "+v"(rb[s2]) : "s"(db));
        asm volatile("v_add_u32 %0, %1, %0" : "+v"(rsa) : "s"(ds));
        asm volatile("v_add_u32 %0, %1, %0" : "+v"(rsb) : "s"(ds));
    };
    auto read_a = [&](v4i (&dst)[4], int ii) __attribute__((always_inline)) {
#pragma unroll
        for (int ks = 0; ks < 4; ks++) dst[ks] = *reinterpret_cast<const v4i*>(lds + ra[ks] + ii * 4096);
    };
    auto read_b = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int s2 = 0; s2 < 2; s2++) bp[s2] = *reinterpret_cast<const uint4*>(lds + rb[s2]);
    };
    // the scale operands of a unit, read once its stage is valid (right after the
    // unit's barrier): sb of this wave's column and sa of the two row-tile pairs
    float sa2[2];
    float sbr;
    auto read_s = [&]() __attribute__((always_inline)) {
        sbr = *reinterpret_cast<const float*>(lds + rsb);
        sa2[0] = *reinterpret_cast<const float*>(lds + rsa);
        sa2[1] = *reinterpret_cast<const float*>(lds + rsa + 256);
    };
    read_a(a_cur, 0);
    read_b();
    read_s();

    // Software pipeline over row tiles: the MFMAs of row tile t run while tile t-1
    // is folded.  The last tile of a unit is folded during the first tile of the
    // next unit of the same segment; at the end of a segment it is folded there and
    // the segment is published.
    // Accumulators with fixed roles: row tiles 0 and 2 of a unit go to accA, tiles
    // 1 and 3 to accB, and a fold reads the one the MFMAs are not writing (no copies).
    v16i accA, accB;
    // Scale products: one buffer of two row tiles, (0, 1) from after row tile 0's
    // MFMAs (until then it holds tiles 2 and 3 of the previous unit, the last of which
    // is folded during row tile 0), (2, 3) from before the unit's barrier.
    v32f S2;
    // One row-tile step: the four MFMAs of tile (a, bu) into acc, each followed by a
    // quarter of the fold of the previous tile (prev into facc[fi], with its scale
    // products S, formed one row tile earlier) and, with UNPACK, by the unpack of
    // the next k-step's weights.
    auto step = [&](const v4i (&a)[4], v16i& acc, const v16i& prev, v16i& fa, int fi, const TileRef& fx,
                    bool do_unpack, const v16f& S) __attribute__((always_inline)) {
        if (do_unpack) unpack_ks(bu, bp, 0);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int ks = 0; ks < 4; ks++) {
            acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[ks], bu[ks], ks ? acc : zero16, 0, 0, 0);
            if (do_unpack && ks < 3) unpack_ks(bu, bp, ks + 1);
            fold_q(fa, prev, S, fi, ks, fx);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    int i = 0;   // the unit being computed
    // Wait for the DMA of unit i + 1: at most the two younger units' loads may be
    // pending (three units in flight).  Right after a flush its stores, at least 4 RT
    // per wave, are younger still and need not be waited for.  Near the end of the share
    // fewer units are in flight, and the group-sum variant stores as it goes: drain.
    auto wait_next = [&](bool flushed) __attribute__((always_inline)) {
        if (GSUM || i + 3 >= n) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        else if (flushed) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * DMA_PER_UNIT + 4 * RT) : "memory");
        else asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * DMA_PER_UNIT) : "memory");
    };
    // The end of a unit's reads: the next unit's data has landed and every wave has
    // issued its last read of this stage (the barrier waits for LDS reads); the stage is
    // refilled and the next unit's operands are read.
    auto turn = [&](v4i (&a_next)[4], bool flushed) __attribute__((always_inline)) {
        const int st = i & (NS - 1);
        wait_next(flushed);
        __syncthreads();
        if (i + 4 < n) {
            advance_dma();
            issue(st);
        }
        next_stage((st + 1) & (NS - 1));
        read_b();
        read_a(a_next, 0);
        read_s();
    };
    // One unit (one group of the current tile) from stage i % NS; `first`: no earlier
    // unit of this segment, so there is no last row tile awaiting its fold (accB and S2
    // are zero and the fold adds exact zeros).
    auto unit = [&](bool first) __attribute__((always_inline)) {
        const bool flushed = first && i > 0;
        TileRef x = cur;
        TileRef xprev = cur;
        if (GSUM) xprev.g = first ? -1 : cur.g - 1;   // -1: nothing to store
        // row tile 0, with the unpack of this unit's weights and the fold of the
        // previous unit's last tile
        read_a(a_nxt, 1);
        step(a_cur, accA, accB, facc[RT - 1], RT - 1, xprev, true, shi(S2));
        S2 = scales2(sa2[0], sbr);
        if constexpr (RT == 4) {
            // row tile 1, fold of tile 0
            read_a(a_cur, 2);
            step(a_nxt, accB, accA, facc[0], 0, x, false, slo(S2));
            // row tile 2, fold of tile 1
            read_a(a_nxt, 3);
            step(a_cur, accA, accB, facc[1], 1, x, false, shi(S2));
            S2 = scales2(sa2[1], sbr);   // before the barrier: sa2, sbr are refilled with the next unit's after it
        }
        turn(a_cur, flushed);
        // the last row tile, fold of the one before
        constexpr int F = RT >= 2 ? RT - 2 : 0;
        step(a_nxt, accB, accA, facc[F], F, x, false, slo(S2));
        ++i;
        if (GSUM) ++cur.g;
    };
    // RT = 1: one row tile per unit, the accumulators (and the scale products) taking
    // turns from unit to unit.
    auto unit1 = [&](v16i& acc, const v16i& prev, v32f& S, const v32f& Sprev, v4i (&a)[4], v4i (&a_next)[4],
                     bool first) __attribute__((always_inline)) {
        const bool flushed = first && i > 0;
        TileRef xprev = cur;
        if (GSUM) xprev.g = first ? -1 : cur.g - 1;
        S = scales2(sa2[0], sbr);
#pragma unroll
        for (int ks = 0; ks < 4; ks++) unpack_ks(bu, bp, ks);
        turn(a_next, flushed);
        step(a, acc, prev, facc[0], 0, xprev, false, slo(Sprev));
        ++i;
        if (GSUM) ++cur.g;
    };
    // segments: the units of one tile within this workgroup's share
    while (i < n) {
        const int len = seg_end(cur.t) - (i == 0 ? g_first : 0);
        if (GSUM) cur.g = i == 0 ? g_first : 0;
        accB = zero16;
        S2 = zero32f;
        TileRef xl = cur;
        if constexpr (RT == 1) {
            v32f S1 = zero32f;
            int k = 0;
            for (; k + 1 < len; k += 2) {
                unit1(accA, accB, S1, S2, a_cur, a_nxt, k == 0);
                unit1(accB, accA, S2, S1, a_nxt, a_cur, false);
            }
            if (GSUM) xl.g = cur.g - 1;
            if (k < len) {
                unit1(accA, accB, S1, S2, a_cur, a_nxt, k == 0);
                if (GSUM) xl.g = cur.g - 1;
#pragma unroll
                for (int q = 0; q < 4; q++) fold_q(facc[0], accA, slo(S1), 0, q, xl);
            } else {
#pragma unroll
                for (int q = 0; q < 4; q++) fold_q(facc[0], accB, slo(S2), 0, q, xl);
            }
        } else {
            for (int k = 0; k < len; k++) unit(k == 0);
            if (GSUM) xl.g = cur.g - 1;
            // the segment's last row tile, then publish the segment
#pragma unroll
            for (int q = 0; q < 4; q++) fold_q(facc[RT - 1], accB, shi(S2), RT - 1, q, xl);
        }
        flush(cur, len == NG);
        // the next unit's fragments, read again from its stage (still intact): the
        // copies read during the last unit are then dead across the flush, which
        // leaves the flush the registers it needs
        read_b();
        read_a(a_cur, 0);
        read_s();
        set_tile(next_tile(cur.t));
    }
}

// The split tiles: C = 1/16 of the sum of a tile's partials in range order.  Block
// (t, y) takes the 64 16-byte pieces 64 y.. of remainder tile t, one per thread: register
// quad y / 8 of the GEMM's wave y % 8, i.e. 8 rows x 32 columns.  Up to four
// contributors' loads are in flight per thread.  Bound by the partials' traffic: M=1024
// N=5120 K=5120, 54 MB read and 21 MB of C written, takes 12.4 us (6.0 TB/s; blocks of 256
// threads, two or four pieces a thread measure the same).
// Its own launch where tiles have many parts, and not the last contributor of each tile
// within the GEMM: that workgroup read up to 13 partials one after another (8.9-19 us at
// the end of a 20-34 us launch for 16-64 rows, 15.8 us at M=384 K=17408) while the others
// were done.  gemm_plan says where the last contributor does it.
template <int RT>
__global__ __launch_bounds__(64) void gemm_combine_k(const float* __restrict__ part, float* __restrict__ C, int M,
                                                      int N, int NG, GemmSched sch) {
    constexpr int PB = 4;
    const int t = blockIdx.x, tb = t * NG;
    const int wf = owner_of(sch, tb), wl = owner_of(sch, tb + NG - 1);
    if (wf == wl) return;                         // one workgroup's: already written
    const int slot_f = 2 * wf + (range_start(sch, wf) == tb ? 0 : 1);
    const int e = blockIdx.y * 64 + threadIdx.x;
    const float4* src = reinterpret_cast<const float4*>(part) + e;
    float4 f = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int v0 = wf; v0 <= wl; v0 += PB) {
        float4 p[PB];
#pragma unroll
        for (int j = 0; j < PB; j++) {
            const int v = min(v0 + j, wl);
            p[j] = src[(size_t)(v == wf ? slot_f : 2 * v) * (Tile<RT>::PART_FLOATS / 4)];
        }
#pragma unroll
        for (int j = 0; j < PB; j++)
            if (v0 + j <= wl) {
                f.x += p[j].x;
                f.y += p[j].y;
                f.z += p[j].z;
                f.w += p[j].w;
            }
    }
    // piece e: register quad k of thread e % NT of the GEMM's workgroup
    const int k = e / NT, w = (e % NT) >> 6, lr = e & 31, lh = (e >> 5) & 1;
    const int tn = t / sch.ntm, nn = tn * BN + 32 * w + lr;
    const int m = (t - tn * sch.ntm) * Tile<RT>::BM + 32 * (k >> 2) + 8 * (k & 3) + 4 * lh;
    if (nn >= N) return;
    float* c = C + (size_t)m * N + nn;
    if (m < M) c[0] = f.x * 0.0625f;
    if (m + 1 < M) c[(size_t)N] = f.y * 0.0625f;
    if (m + 2 < M) c[(size_t)N * 2] = f.z * 0.0625f;
    if (m + 3 < M) c[(size_t)N * 3] = f.w * 0.0625f;
}
}  // namespace

GemmPlan gemm_plan(int M, int N, int K, int cus) {
    GemmPlan p;
    const int NG = K / kGroup, ntn = (N + BN - 1) / BN, ncu = cus > 0 ? cus : 256;
    p.rt = M <= 32 ? 1 : M <= 64 ? 2 : 4;
    p.s.ntm = (M + 32 * p.rt - 1) / (32 * p.rt);
    const int ntiles = p.s.ntm * ntn;
    const long long T = (long long)ntiles * NG;
    p.P = T < ncu ? (int)T : ncu;
    p.s.full = ntiles / p.P;
    p.s.rem = ntiles - p.s.full * p.P;
    const int R = p.s.rem * NG;      // their units: rem < P, and one tile only where
                                     // K / 128 reaches 2^23 (the limits on M K and N K)
    // How many workgroups share the remainder tiles.  Every tile in S pieces on rem * S
    // workgroups (S = 1: whole tiles, nothing to combine), or equal ranges on all of them
    // (better balanced, but most workgroups then touch two tiles and leave two partials).
    // Cost in us: the longest share, at the time a unit takes, and for a split the
    // combining launch with its partials written and read.  Measured at M=1792 N=17408
    // K=1152 (952 tiles of 9 groups, 184 left over): equal ranges 83.3 us a call, whole
    // tiles 70.8.
    const double unit_us = p.rt == 1 ? 0.6 : p.rt == 2 ? 0.87 : 1.36;
    const double part_us = p.rt * (NT * 16 * sizeof(float)) / 4.5e6;
    p.s.Pr = p.s.rem;
    p.split = false;
    double best = NG * unit_us;
    const int smax = p.s.rem > 0 ? (p.P / p.s.rem < NG ? p.P / p.s.rem : NG) : 0;
    for (int S = 2; S <= smax; S++) {
        const double c = (NG + S - 1) / S * unit_us + 4.0 + (double)p.s.rem * S * part_us;
        if (c < best) {
            best = c;
            p.s.Pr = p.s.rem * S;
            p.split = true;
        }
    }
    if (R >= p.P && p.s.rem > 0 &&
        (double)((R + p.P - 1) / p.P) * unit_us + 4.0 + (double)(p.P + p.s.rem) * part_us < best) {
        p.s.Pr = p.P;
        p.split = true;
    }
    // Equal ranges of more than half a tile's groups: at most three parts a tile, and tiles
    // that are finished all through the launch, so the last contributor's sum hides behind
    // the others' work where a combining launch reads every partial (13 us) at the end.
    // Measured (us, combining launch -> in the launch, graph replayed): M=1024 N=5120
    // K=17408 136 -> 131, M=609 N=7395 K=7040 64.0 -> 60.7, M=200 N=17408 K=5120 45.7 -> 44.3.
    // With more parts it loses: M=1024 N=1024 K=5120 (8 parts) 23 -> 28, M=128 N=17408 K=5120
    // (68 tiles, 4 or 5) 31.0 -> 32.5.
    p.inline_combine = p.split && p.rt == 4 && p.s.Pr == p.P && 2 * p.s.rem > p.P;
    // Whether the ranges are spread over the XCDs.  On the first Pr workgroups they load
    // some XCDs with all of the shared tiles while the others idle or wait; but where they
    // are less than about three quarters of one XCD's workgroups, one XCD takes them as
    // fast and reads their operands once.  Measured (us, first workgroups -> spread):
    // M=1024 N=4096 K=256 (Pr 128) 11.4 -> 9.3, M=946 N=11400 K=128 (104) 14.9 -> 12.8,
    // M=512 N=18432 K=128 (32) 13.0 -> 12.1, N=17920 (24) 12.0 -> 11.8, N=17664 (20) 11.8 ->
    // 12.0, N=17408 (16) 11.2 -> 11.9.
    p.s.spread = p.P % 8 == 0 && p.s.Pr > 3 * p.P / 32;
    p.s.q = p.s.Pr > 0 ? R / p.s.Pr : 0;
    p.s.r = p.s.Pr > 0 ? R % p.s.Pr : 0;
    // Two partials of a 128-row tile per workgroup, whatever the tile and whether any is
    // split: what may be captured after an eager call then depends on the workgroup count
    // alone, which is the CU count from that many (tile, group) units up.
    p.part_bytes = (size_t)p.P * 2 * Tile<4>::PART_FLOATS * sizeof(float);
    return p;
}

hipError_t launch_gemm_w4a8(float* C, int32_t* gsum, const int8_t* A, const uint32_t* W,
                            const float* sa, const float* sb, int M, int N, int K, const GemmPlan& p,
                            float* part, int* cnt, hipStream_t st) {
#define RT4_GEMM_K(R, G, I) \
    hipLaunchKernelGGL((gemm_w4a8_k<R, G, I>), dim3(p.P), dim3(NT), 0, st, A, W, sa, sb, C, gsum, part, cnt, M, N, K, p.s)
#define RT4_GEMM(R)                      \
    if (gsum) RT4_GEMM_K(R, true, false); \
    else RT4_GEMM_K(R, false, false);     \
    if (p.split) hipLaunchKernelGGL(gemm_combine_k<R>, dim3(p.s.rem, 32 * R), dim3(64), 0, st, part, C, M, N, K / kGroup, p.s);
    if (p.rt == 1) {
        RT4_GEMM(1)
    } else if (p.rt == 2) {
        RT4_GEMM(2)
    } else if (p.inline_combine && cnt && !gsum) {
        RT4_GEMM_K(4, false, true);
    } else {
        RT4_GEMM(4)
    }
#undef RT4_GEMM
#undef RT4_GEMM_K
    return hipGetLastError();
}

// Zero the split counters of a workspace once, when it is (re)allocated.
__global__ void zero_i32_k(int* p, size_t n) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n) p[i] = 0;
}

hipError_t launch_zero_i32(int* p, size_t n, hipStream_t st) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(zero_i32_k, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, p, n);
    return hipGetLastError();
}

}  // namespace rt4
