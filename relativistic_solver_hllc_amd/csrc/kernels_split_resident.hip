// Split-precision contraction with the phase panel resident in LDS
// ("resident-panel" kernel), for cell-level state (one value per cell and
// direction, i.e. face-averaged intensities).
//
// The streaming kernel (kernels_split.hip) re-streams the whole panel through
// LDS for every 64 cells and synchronises its workgroup at every K-step; at
// 100 KB of LDS per workgroup only one workgroup fits a CU, so those barriers
// are exposed. Here each workgroup owns a fixed group of RBW row blocks (16 RBW
// output directions) and copies that slice of the panel for ALL K-steps into
// LDS once, then streams cells through it with no further barrier: persistent
// workgroups, one per CU. Two parts per row block are resident (hi and lo;
// hi and mid for the three-part form, whose lo part is read per K-step from
// L2, where every row group's slice of it stays): 2 KB per (K-step, row block),
// so five row blocks fit at M = 400 (130 KB) and the 25 row blocks of M = 400
// split into five groups without padding.
//
// Work split. The G row groups of a problem are served by G workgroups that
// sit on the same XCD (workgroup b runs on XCD b % 8) and walk the same
// sequence of 256-cell chunks, so a chunk's state is read from HBM once and
// from that XCD's L2 by the other G - 1. Each XCD owns a contiguous 1/8 of the
// chunks; within it, the floor(CUs per XCD / G) sets of G workgroups take
// chunks round-robin.
//
// Per wave (four waves, one per SIMD): four 16-cell tiles x RBW row blocks, so
// every A fragment read from LDS feeds four MFMAs per product; MFMAs are issued
// product-major so that no MFMA depends on the one before it; state vectors
// are prefetched K-steps ahead, across chunk boundaries too, with ordinary
// (L2-allocating) loads, since the other row groups of the XCD read the same
// vectors. Products and their order per (row block, tile) are those of the
// streaming kernel (each K-step's main hi*hi formed alone and added in FP32;
// cross hi*lo + lo*hi, and for three parts hi*lo, hi*mid, mid*mid, mid*hi,
// lo*hi), so the kernels give bit-identical results on the same state and
// panel.
#include "split_iter_res.hpp"

namespace rsh {

namespace {

// State prefetch depth in K-steps of the single-problem kernel (registers:
// XD x 4 tiles x parts x 4 VGPRs); the three-part form also prefetches the lo
// part of its panel slice kResLoXd K-steps ahead (RBW x 4 VGPRs each).
template <int NT>
constexpr int res_xd() { return NT == 2 ? 3 : 2; }
constexpr int kResLoXd = 1;

// STEPS > 0: the K-step count is a compile-time constant and the K loop is
// fully unrolled, so the state prefetch crosses no loop back-edge (where the
// compiler would otherwise wait for every outstanding load). STEPS = 0: any M.
// NL = parts of the panel slice resident in LDS (2); a three-part panel's lo
// part comes from global memory (L2), kResLoXd K-steps ahead.
template <int RBW, int FMT, int NT, int STEPS>
__global__ __launch_bounds__(64 * kRes4Waves) void split_resident_kernel(
    const v4u* __restrict__ state, int64_t n, int steps_rt, const float* __restrict__ cell_inv,
    const v4u* __restrict__ panel, const float* __restrict__ row_inv, void* __restrict__ out, int64_t ld, int rows,
    int out_f32, int groups, int sets, int64_t chunks) {
    typedef typename Fmt<FMT>::V V;
    constexpr int TT = kRes4Tiles;
    constexpr int NL = 2;
    constexpr int XD = res_xd<NT>();
    constexpr int XL = NT == 3 ? kResLoXd : 1;
    const int steps = STEPS > 0 ? STEPS : steps_rt;
    extern __shared__ v4u lds[];  // [steps][RBW][NL][64], then the row group's 16 RBW row scales
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // uniform: scalar tile bounds
    const int g = lane >> 4;
    const int xcd = blockIdx.x % kXcds;
    const int local = blockIdx.x / kXcds;
    const int set = local / groups;
    const int rg = local % groups;
    if (set >= sets) return;  // whole workgroup leaves together: no barrier below is skipped by part of it

    // 1. the row group's panel slice, all K-steps, parts 0 .. NL - 1, into LDS
    const int64_t slice = (int64_t)steps * RBW * NT * 64;  // the row group's panel, 16-byte vectors
    const v4u* __restrict__ src = panel + (int64_t)rg * slice;
    const int64_t units = (int64_t)steps * RBW * NL * 64;
    for (int64_t u = threadIdx.x; u < units; u += 64 * kRes4Waves) {
        const int64_t f = u >> 6;  // (s * RBW + rb) * NL + p
        lds[u] = src[((f / NL) * NT + f % NL) * 64 + (u & 63)];
    }
    const int row0 = rg * RBW * 16;
    // Row scales once per workgroup into LDS: scale loads from global memory in
    // every epilogue measurably broke the row groups' L2 sharing of the state.
    float* rscale = reinterpret_cast<float*>(lds + units);
    for (int r = threadIdx.x; r < RBW * 16; r += 64 * kRes4Waves)
        rscale[r] = row0 + r < rows ? row_inv[row0 + r] : 0.0f;
    __syncthreads();

    // The lo part of a three-part panel slice through one buffer descriptor; an
    // opaque zero in its offset, renewed per chunk, keeps the compiler from
    // hoisting all K-steps' loads out of the chunk loop (they would not fit).
    const __amdgpu_buffer_rsrc_t lo_rs =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<v4u*>(src), (short)0, (int)(slice * 16), kBufWord3);
    int lo_zero = 0;
    v4u plo[XL][RBW];
    auto load_lo = [&](auto slot_tag, int t) {
        if constexpr (NT == 3) {
            constexpr int sl = decltype(slot_tag)::value;
#pragma unroll
            for (int i = 0; i < RBW; i++)
                plo[sl][i] = __builtin_bit_cast(v4u, __builtin_amdgcn_raw_buffer_load_b128(
                                                         lo_rs, lane * 16 + lo_zero, ((t * RBW + i) * NT + 2) * 1024, 0));
        }
    };

    // 2. chunks of this XCD, round-robin over its sets
    const int64_t c_begin = chunks * xcd / kXcds, c_end = chunks * (xcd + 1) / kXcds;
    const int64_t tiles = (n + 15) / 16;
    const int64_t tile_units = (int64_t)steps * NT * 64;  // 16-byte vectors per 16-cell tile
    const int tile_bytes = (int)(tile_units * 16);

    // A chunk's state is read through one buffer descriptor: the uniform base and
    // the K-step offsets live in scalar registers, so a tile needs one VGPR
    // offset instead of a 64-bit address per K-step. Tiles past the end of the
    // state re-read the chunk's last tile (in range) and are not written.
    __amdgpu_buffer_rsrc_t xs;
    int xoff[TT];
    auto bind_chunk = [&](int64_t chunk) {
        const int64_t ct_chunk = chunk * kResChunkTiles;
        const int ntile = (int)(tiles - ct_chunk < kResChunkTiles ? tiles - ct_chunk : kResChunkTiles);
        xs = __builtin_amdgcn_make_buffer_rsrc(const_cast<v4u*>(state + ct_chunk * tile_units), (short)0,
                                               ntile * tile_bytes, kBufWord3);
#pragma unroll
        for (int q = 0; q < TT; q++) {
            const int tile = wave * TT + q;
            xoff[q] = (tile < ntile ? tile : ntile - 1) * tile_bytes + lane * 16;
        }
    };
    v4u xr[XD][TT][NT];
    auto load_x = [&](auto slot_tag, int t) {
        constexpr int sl = decltype(slot_tag)::value;
#pragma unroll
        for (int q = 0; q < TT; q++)
#pragma unroll
            for (int p = 0; p < NT; p++)
                xr[sl][q][p] = __builtin_bit_cast(
                    v4u, __builtin_amdgcn_raw_buffer_load_b128(xs, xoff[q] + p * 1024, t * NT * 1024, 0));
    };
    // First K-steps of a chunk. For every chunk after the first they are
    // issued before the previous chunk's result stores: loads and stores retire
    // through one in-order counter, so a load issued after the stores could
    // only be waited for together with all of them.
    auto prefetch_head = [&]() {
        asm volatile("v_mov_b32 %0, 0" : "=v"(lo_zero));
        static_for<0, XD>([&](auto u) {
            if (u.value < steps) load_x(u, u.value);
        });
        static_for<0, XL>([&](auto u) {
            if (u.value < steps) load_lo(u, u.value);
        });
    };

    int64_t chunk = c_begin + set;
    // hi fragments of the next K-step (res_mfma_step reads them a step ahead)
    V ahi[RBW];
#pragma unroll
    for (int i = 0; i < RBW; i++) ahi[i] = __builtin_bit_cast(V, lds[(i * NL) * 64 + lane]);
    if (chunk < c_end) {
        bind_chunk(chunk);
        prefetch_head();
    }
    for (; chunk < c_end; chunk += sets) {
        const int64_t ct0 = chunk * kResChunkTiles + wave * TT;
        // Cell scales now, ahead of the next chunk's prefetch: a load issued
        // after those could only be waited for together with all of them.
        float cinv[TT];
#pragma unroll
        for (int q = 0; q < TT; q++) {
            const int64_t cell = (ct0 + q) * 16 + (lane & 15);
            cinv[q] = cell_inv[cell < n ? cell : n - 1];
        }
        v4f accm[RBW][TT], accx[RBW][TT];
#pragma unroll
        for (int i = 0; i < RBW; i++)
#pragma unroll
            for (int q = 0; q < TT; q++) {
                accm[i][q] = v4f{0.f, 0.f, 0.f, 0.f};
                accx[i][q] = v4f{0.f, 0.f, 0.f, 0.f};
            }
        // K-step t with ring slot SL = t % XD and lo slot SLL = t % XL
        auto kstep = [&](auto slot_tag, auto lo_tag, const int t) {
            constexpr int sl = decltype(slot_tag)::value;
            constexpr int sll = decltype(lo_tag)::value;
            // Scheduling fence per K-step: in the unrolled loop the scheduler
            // would otherwise hoist every K-step's loads and run out of registers.
            __builtin_amdgcn_sched_barrier(0);
            V bx[TT][NT];
#pragma unroll
            for (int q = 0; q < TT; q++)
#pragma unroll
                for (int p = 0; p < NT; p++) bx[q][p] = __builtin_bit_cast(V, xr[sl][q][p]);
            V alo[RBW];
            if constexpr (NT == 3) {
#pragma unroll
                for (int i = 0; i < RBW; i++) alo[i] = __builtin_bit_cast(V, plo[sll][i]);
                if (t + XL < steps) load_lo(lo_tag, t + XL);
            }
            if (t + XD < steps) load_x(slot_tag, t + XD);
            const int tn = t + 1 < steps ? t + 1 : 0;  // the next chunk starts at K-step 0
            res_mfma_step<RBW, FMT, NT, TT, NL, true>(lds + (int64_t)t * RBW * NL * 64 + lane,
                                                lds + (int64_t)tn * RBW * NL * 64 + lane, ahi, bx, alo, accm, accx);
        };
        if constexpr (STEPS > 0) {
            static_for<0, STEPS>([&](auto t) {
                kstep(std::integral_constant<int, t.value % XD>{}, std::integral_constant<int, t.value % XL>{},
                      t.value);
            });
        } else {
            // XD and XL divide 6: blocks of six K-steps keep every ring slot a
            // compile-time constant
            static_assert(6 % XD == 0 && 6 % XL == 0, "ring depths must divide the unroll of six");
            for (int t = 0; t < steps; t += 6)
                static_for<0, 6>([&](auto u) {
                    if (t + u.value < steps)
                        kstep(std::integral_constant<int, u.value % XD>{},
                              std::integral_constant<int, u.value % XL>{}, t + u.value);
                });
        }
        __builtin_amdgcn_sched_barrier(0);
        if (chunk + sets < c_end) {
            bind_chunk(chunk + sets);
            prefetch_head();
        }
        __builtin_amdgcn_sched_barrier(0);

        // Epilogue: FP64 combination of the main and cross terms, exact scale
        // removal. Row scales are re-read from LDS per chunk: an opaque zero
        // offset keeps the compiler from hoisting them out of the chunk loop.
        // Lane pairs (cells 2c, 2c + 1 of a tile) swap half of their results
        // (swap_pair_lanes), so that a lane holds two adjacent cells of one row:
        // the even lane rows 4g, 4g + 1, the odd lane rows 4g + 2, 4g + 3. Each
        // store then writes two cells (16 bytes for FP64), half as many store
        // instructions as one cell per lane: with one cell per lane a chunk's
        // stores alone exceeded the wave's 63 outstanding memory operations.
        // Stores go through one buffer descriptor per row block (uniform base,
        // row offset h * ld in a scalar register, one VGPR offset per tile).
        int zoff;
        asm volatile("v_mov_b32 %0, 0" : "=v"(zoff));
        const float* __restrict__ rs = rscale + 4 * g + zoff;
        const int odd = lane & 1;
        auto store_all = [&](auto elem_tag, auto full_tag) {
            typedef decltype(elem_tag) OT;
            constexpr bool kFull = decltype(full_tag)::value;
            const int esz = (int)sizeof(OT);
            int voff[TT];
            bool ok1[TT], ok2[TT];
#pragma unroll
            for (int q = 0; q < TT; q++) {
                const int64_t cell0 = (ct0 + q) * 16 + (lane & 14);  // first cell of the lane pair
                ok1[q] = cell0 < n;
                ok2[q] = cell0 + 1 < n;
                voff[q] = (int)(((4 * g + 2 * odd) * ld + cell0) * esz);
            }
#pragma unroll
            for (int i = 0; i < RBW; i++) {
                const int rb_row = row0 + i * 16;
                if (!kFull && rb_row >= rows) break;
                const __amdgpu_buffer_rsrc_t os = __builtin_amdgcn_make_buffer_rsrc(
                    static_cast<OT*>(out) + (int64_t)rb_row * ld, (short)0, (int)(16 * ld * esz), kBufWord3);
                const v4f rsv = *reinterpret_cast<const v4f*>(rs + i * 16);  // this lane's 4 row scales
#pragma unroll
                for (int q = 0; q < TT; q++) {
                    OT v[4];
#pragma unroll
                    for (int r = 0; r < 4; r++)
                        v[r] = (OT)(split_value(accm[i][q][r], accx[i][q][r]) * (double)rsv[r] * (double)cinv[q]);
#pragma unroll
                    for (int h = 0; h < 2; h++) {
                        const OT recv = swap_pair_lanes(odd ? v[h] : v[2 + h]);
                        const OT first = odd ? recv : v[h];      // cell 2c
                        const OT second = odd ? v[2 + h] : recv;  // cell 2c + 1
                        if (!kFull && rb_row + 4 * g + 2 * odd + h >= rows) continue;
                        if ((ct0 + q + 1) * 16 <= n)  // whole tile inside the output (uniform branch)
                            store_cell_pair(first, second, true, true, os, voff[q], (int)(h * ld * esz));
                        else
                            store_cell_pair(first, second, ok2[q], ok1[q], os, voff[q], (int)(h * ld * esz));
                    }
                }
            }
        };
        const bool full = row0 + RBW * 16 <= rows;
        if (out_f32) {
            if (full) store_all(0.0f, std::true_type{});
            else store_all(0.0f, std::false_type{});
        } else {
            if (full) store_all(0.0, std::true_type{});
            else store_all(0.0, std::false_type{});
        }
    }
}

template <int RBW, int FMT, int NT, int STEPS>
hipError_t launch_res(int blocks, size_t lds_bytes, hipStream_t st, const v4u* state, int64_t n, int steps,
                      const float* cell_inv, const v4u* panel, const float* row_inv, void* out, int64_t ld, int rows,
                      int out_f32, int groups, int sets, int64_t chunks) {
    auto kern = split_resident_kernel<RBW, FMT, NT, STEPS>;
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(kern, dim3(blocks), dim3(64 * kRes4Waves), lds_bytes, st, state, n, steps, cell_inv, panel,
                       row_inv, out, ld, rows, out_f32, groups, sets, chunks);
    return hipGetLastError();
}

// The single-problem kernel (one wave per SIMD, 512 registers) holds five row blocks.
constexpr int kRes4MaxRbw = 5;
constexpr int kRes4LdsParts = 2;  // panel parts resident in LDS in the single-problem kernel

}  // namespace

// Row-group plan of a resident-panel kernel for output rows [0, rows) of an
// M-direction set: rb_per_pass = RBW row blocks per workgroup (largest slice
// that fits LDS, then balanced), passes = G row groups. grouped: the plan of
// the grouped iteration kernel (all parts of the slice in LDS), else that of
// the single-problem kernel (two parts in LDS). False if the kernel does not
// apply (G row groups do not fit one XCD's CUs).
bool plan_split_resident(int form, int m, int rows, int cus, SplitPlan* pl, int* sets, bool grouped) {
    const int nt = split_terms(form);
    const int steps = (m + 31) / 32;
    const int rb_need = (rows + 15) / 16;
    const int per_xcd = cus / kXcds;
    if (rb_need < 1) return false;
    int rbw = 0;
    if (grouped) {
        if (steps > kIterResMaxSteps) return false;
        rbw = iter_res_rbw(nt, steps, rb_need);
    } else {
        int rbw_max = kResLdsBytes / (steps * kRes4LdsParts * 1024 + 16 * 4);  // panel fragments + row scales
        if (rbw_max > kRes4MaxRbw) rbw_max = kRes4MaxRbw;
        if (rbw_max < 1) return false;
        const int g = (rb_need + rbw_max - 1) / rbw_max;
        rbw = (rb_need + g - 1) / g;
    }
    const int groups = (rb_need + rbw - 1) / rbw;
    if (groups > per_xcd) return false;
    pl->rb_per_pass = rbw;
    pl->passes = groups;
    pl->rb_total = rbw * groups;
    pl->steps = steps;
    *sets = per_xcd / groups;
    return true;
}

hipError_t launch_split_resident(int form, const void* d_state, int64_t n, const float* d_cell_inv,
                                 const void* d_panel, const float* d_row_inv, const SplitPlan& pl, int sets, int rows,
                                 void* d_out, int64_t ld, int out_f32, hipStream_t st) {
    if (n <= 0 || rows <= 0) return hipSuccess;
    const int nt = split_terms(form), fmt = split_fmt(form);
    const size_t lds_bytes = (size_t)pl.steps * pl.rb_per_pass * kRes4LdsParts * 1024 + (size_t)pl.rb_per_pass * 16 * 4;
    if (lds_bytes > (size_t)kResLdsBytes || pl.rb_per_pass > kRes4MaxRbw || sets < 1 || ld >= kSplitResidentMaxLd)
        return hipErrorInvalidValue;
    const int64_t tiles = (n + 15) / 16;
    const int64_t chunks = (tiles + kResChunkTiles - 1) / kResChunkTiles;
    const int blocks = kXcds * sets * pl.passes;
    const v4u* state = static_cast<const v4u*>(d_state);
    const v4u* panel = static_cast<const v4u*>(d_panel);
#define RSH_RES_S(RBW, FMT, NT, S)                                                                              \
    return launch_res<RBW, FMT, NT, S>(blocks, lds_bytes, st, state, n, pl.steps, d_cell_inv, panel, d_row_inv, \
                                       d_out, ld, rows, out_f32, pl.passes, sets, chunks)
    // Unrolled instances for the plans of M = 200, 400, 800 (7, 13, 25 K-steps).
#define RSH_RES(RBW, FMT, NT)                                                                   \
    {                                                                                           \
        if constexpr (RBW == 5) { if (pl.steps == 7) RSH_RES_S(RBW, FMT, NT, 7); }              \
        if constexpr (RBW == 5) { if (pl.steps == 13) RSH_RES_S(RBW, FMT, NT, 13); }            \
        if constexpr (RBW == 3) { if (pl.steps == 25) RSH_RES_S(RBW, FMT, NT, 25); }            \
        RSH_RES_S(RBW, FMT, NT, 0);                                                             \
    }
#define RSH_RES_FORMS(RBW)                           \
    case RBW:                                        \
        if (fmt == 0 && nt == 2) RSH_RES(RBW, 0, 2); \
        if (fmt == 1 && nt == 2) RSH_RES(RBW, 1, 2); \
        RSH_RES(RBW, 0, 3);
    switch (pl.rb_per_pass) {
        RSH_RES_FORMS(1) RSH_RES_FORMS(2) RSH_RES_FORMS(3) RSH_RES_FORMS(4) RSH_RES_FORMS(5)
        default:
            return hipErrorInvalidValue;
    }
#undef RSH_RES_FORMS
#undef RSH_RES
#undef RSH_RES_S
}

// Grouped iteration, resident-panel form: the plans of up to kIterResMaxSteps
// K-steps (split_iter_res.hpp). rb = RBW of the class, steps its K-steps.
bool iter_split_res_supported(int form, int rb, int steps) {
    const int nt = split_terms(form);
    if (steps < 1 || steps > kIterResMaxSteps) return false;
    return rb == iter_res_rbw(nt, steps, 2 * steps - 1) || rb == iter_res_rbw(nt, steps, 2 * steps);
}

// Plans that a caller may ask for by name (rsh_batch_set_split_kernel) and that
// have a four-wave form: M = 200, 400 and 800 with their neighbours. The others
// are taken by the automatic choice only.
bool iter_split_res_selectable(int steps) { return steps == 7 || steps == 13 || steps == 25; }

hipError_t launch_grouped_iter_split_res(bool launch, int form, int rb, int steps, int waves, int grid,
                                         const BatchProblem* d_probs, const BatchItem* d_items, const int* d_meta,
                                         int parity, hipStream_t st) {
    const IterResArgs a{launch, rb, steps, waves, grid, d_probs, d_items, d_meta, parity, st};
    switch (form) {
        case RSH_FORM_BF16X2: return steps <= 14 ? iter_res_range<0, 2, 1, 14>(a) : iter_res_range<0, 2, 15, 25>(a);
        case RSH_FORM_FP16X2: return steps <= 14 ? iter_res_range<1, 2, 1, 14>(a) : iter_res_range<1, 2, 15, 25>(a);
        case RSH_FORM_BF16X3: return steps <= 14 ? iter_res_range<0, 3, 1, 14>(a) : iter_res_range<0, 3, 15, 25>(a);
        default: return hipErrorInvalidValue;
    }
}

int iter_split_res_chunk_cells(int waves) { return waves * kResTiles * 16; }

int iter_split_res_grid(int waves, int cus) { return cus / kXcds * kXcds * (waves == 4 ? 2 : 1); }

}  // namespace rsh
