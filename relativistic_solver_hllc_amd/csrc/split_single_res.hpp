// Split-precision contraction with the phase panel resident in LDS: the
// single-problem kernel and the launcher of one (K-steps, row blocks) plan.
// Instantiated for every plan of a whole direction set of up to
// kSingleResMaxSteps K-steps by the kernels_res_*.hip files.
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
// Per wave: TT 16-cell tiles x RBW row blocks, so every A fragment read from LDS
// feeds TT MFMAs per product; MFMAs are issued
// product-major so that no MFMA depends on the one before it; state vectors
// are prefetched K-steps ahead, across chunk boundaries too, with ordinary
// (L2-allocating) loads, since the other row groups of the XCD read the same
// vectors. Products and their order per (row block, tile) are those of the
// streaming kernel (each K-step's main hi*hi formed alone and added in FP32;
// cross hi*lo + lo*hi, and for three parts hi*lo, hi*mid, mid*mid, mid*hi,
// lo*hi), so the kernels give bit-identical results on the same state and
// panel.
#pragma once

#include "split_res_core.hpp"

namespace rsh {

// Unrolled instances: M <= 32 * kSingleResMaxSteps = 800 directions.
constexpr int kSingleResMaxSteps = 25;
// One wave per SIMD, 512 registers: five row blocks.
constexpr int kRes4MaxRbw = 5;
constexpr int kRes4LdsParts = 2;  // panel parts resident in LDS
constexpr int kResLongSteps = 20;  // from these K-steps on a slice holds at most three row blocks

// Row blocks per workgroup for rb_need row blocks: the largest slice that fits
// LDS (panel fragments + row scales), then balanced; 0: not even one fits.
constexpr int single_res_rbw(int steps, int rb_need) {
    const int fit = kResLdsBytes / (steps * kRes4LdsParts * 1024 + 16 * 4);
    const int mx = fit < kRes4MaxRbw ? fit : kRes4MaxRbw;
    if (mx < 1) return 0;
    const int groups = (rb_need + mx - 1) / mx;
    return (rb_need + groups - 1) / groups;
}

struct SingleResArgs {
    int rbw, steps;
    int waves, tiles;  // per workgroup; 16-cell tiles per wave
    int blocks;
    size_t lds_bytes;
    hipStream_t st;
    const v4u* state;
    int64_t n;
    const float* cell_inv;
    const v4u* panel;
    const float* row_inv;
    void* out;
    int64_t ld;
    int rows, out_f32, nontemporal, groups, sets;
    int64_t chunks;
};

// State prefetch depth in K-steps of the single-problem kernel (registers:
// XD x 4 tiles x parts x 4 VGPRs); the three-part form also prefetches the lo
// part of its panel slice kResLoXd K-steps ahead (RBW x 4 VGPRs each).
template <int NT>
constexpr int res_xd() { return NT == 2 ? 3 : 2; }
constexpr int kResLoXd = 1;

// STEPS > 0: the K-step count is a compile-time constant and the K loop is
// fully unrolled, so the state prefetch crosses no loop back-edge (where the
// compiler would otherwise wait for every outstanding load). STEPS = 0: any M.
// us before and after the unrolled instances and the epilogue's choice of stores
// (FP32 results): 76,791 cells x 427 directions FP32 199 / 113, 100,000 x 500
// 251 / 166, 413,519 x 302 three parts 725 / 454, 60,000 x 640 three parts 405 / 287.
// NL = parts of the panel slice resident in LDS (2); a three-part panel's lo
// part comes from global memory (L2), kResLoXd K-steps ahead.
// W waves of TT 16-cell tiles: a chunk is 16 W TT cells. Forms: 8 waves x 2 tiles
// (two waves per SIMD: one's epilogue and adds overlap the other's MFMAs), 4 waves
// x 4 tiles (half the LDS reads per MFMA), 8 x 1 (few cells).
template <int RBW, int FMT, int NT, int STEPS, int W, int TT>
__global__ __launch_bounds__(64 * W) void split_resident_kernel(
    const v4u* __restrict__ state, int64_t n, int steps_rt, const float* __restrict__ cell_inv,
    const v4u* __restrict__ panel, const float* __restrict__ row_inv, void* __restrict__ out, int64_t ld, int rows,
    int out_f32, int nontemporal, int groups, int sets, int64_t chunks) {
    typedef typename Fmt<FMT>::V V;
    constexpr int CT = W * TT;  // tiles per chunk
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
    // kFill loads in flight per thread: one at a time cost a memory round trip each
    constexpr int kFill = 8, TH = 64 * W;
    for (int u0 = threadIdx.x; u0 < (int)units; u0 += kFill * TH) {
        v4u buf[kFill];
#pragma unroll
        for (int i = 0; i < kFill; i++) {
            const int u = u0 + i * TH < (int)units ? u0 + i * TH : (int)units - 1;
            const int f = u >> 6;  // (s * RBW + rb) * NL + p
            buf[i] = src[(int64_t)(f / NL * NT + f % NL) * 64 + (u & 63)];
        }
#pragma unroll
        for (int i = 0; i < kFill; i++)
            if (u0 + i * TH < (int)units) lds[u0 + i * TH] = buf[i];
    }
    const int row0 = rg * RBW * 16;
    // Row scales once per workgroup into LDS: scale loads from global memory in
    // every epilogue measurably broke the row groups' L2 sharing of the state.
    float* rscale = reinterpret_cast<float*>(lds + units);
    for (int r = threadIdx.x; r < RBW * 16; r += 64 * W)
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
        const int64_t ct_chunk = chunk * CT;
        const int ntile = (int)(tiles - ct_chunk < CT ? tiles - ct_chunk : CT);
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
        const int64_t ct0 = chunk * CT + wave * TT;
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
        auto store_all = [&](auto elem_tag, auto full_tag, auto aux_tag) {
            typedef decltype(elem_tag) OT;
            constexpr bool kFull = decltype(full_tag)::value;
            constexpr int kAux = decltype(aux_tag)::value;
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
                            store_cell_pair<kAux>(first, second, true, true, os, voff[q], (int)(h * ld * esz));
                        else
                            store_cell_pair<kAux>(first, second, ok2[q], ok1[q], os, voff[q], (int)(h * ld * esz));
                    }
                }
            }
        };
        const bool full = row0 + RBW * 16 <= rows;
        const auto stores = [&](auto elem_tag, auto aux_tag) {
            if (full) store_all(elem_tag, std::true_type{}, aux_tag);
            else store_all(elem_tag, std::false_type{}, aux_tag);
        };
        typedef std::integral_constant<int, 0> Plain;
        typedef std::integral_constant<int, kNontemporal> Nt;
        if (out_f32) {
            // single_res_nontemporal is for FP64 results but with long slices
            if constexpr (STEPS == 0 || STEPS >= kResLongSteps) {
                if (nontemporal) stores(0.0f, Nt{});
                else stores(0.0f, Plain{});
            } else {
                stores(0.0f, Plain{});
            }
        } else if (nontemporal) {
            stores(0.0, Nt{});
        } else {
            stores(0.0, Plain{});
        }
    }
}

template <int RBW, int FMT, int NT, int STEPS, int W, int TT>
hipError_t launch_res(const SingleResArgs& a) {
    auto kern = split_resident_kernel<RBW, FMT, NT, STEPS, W, TT>;
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)a.lds_bytes);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(kern, dim3(a.blocks), dim3(64 * W), a.lds_bytes, a.st, a.state, a.n, a.steps, a.cell_inv,
                       a.panel, a.row_inv, a.out, a.ld, a.rows, a.out_f32, a.nontemporal, a.groups, a.sets, a.chunks);
    return hipGetLastError();
}

// K-steps LO .. HI of one form; explicitly instantiated by the kernels_res_*.hip
// files. hipErrorNotFound: no unrolled instance of this plan, for instance that of a
// range of rows whose row blocks per workgroup are not the whole direction set's.
template <int FMT, int NT, int LO, int HI>
hipError_t single_res_range(const SingleResArgs& a);

template <int RBW, int FMT, int NT, int S>
hipError_t single_res_one(const SingleResArgs& a) {
    if (a.waves == 4) return launch_res<RBW, FMT, NT, S, 4, 4>(a);
    if constexpr (NT == 2) return launch_res<RBW, FMT, NT, S, 8, 2>(a);
    return hipErrorNotFound;
}

template <int FMT, int NT, int S, int HI>
hipError_t single_res_find(const SingleResArgs& a) {
    if (a.steps == S) {
        constexpr int r1 = single_res_rbw(S, 2 * S - 1), r2 = single_res_rbw(S, 2 * S);
        if (a.rbw == r1) return single_res_one<r1, FMT, NT, S>(a);
        if constexpr (r2 != r1) {
            if (a.rbw == r2) return single_res_one<r2, FMT, NT, S>(a);
        }
        return hipErrorNotFound;
    }
    if constexpr (S < HI) return single_res_find<FMT, NT, S + 1, HI>(a);
    return hipErrorNotFound;
}

#define RSH_SINGLE_RES_RANGE(FMT, NT, LO, HI)                            \
    namespace rsh {                                                      \
    template <>                                                          \
    hipError_t single_res_range<FMT, NT, LO, HI>(const SingleResArgs& a) { \
        return single_res_find<FMT, NT, LO, HI>(a);                      \
    }                                                                    \
    }

}  // namespace rsh
