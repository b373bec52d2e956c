// Grouped source iteration on split state, resident-panel form: the kernel and
// the launcher of one (K-steps, row blocks) plan. Instantiated for every plan
// of up to kIterResMaxSteps K-steps by the kernels_iter_res_*.hip files.
#pragma once

#include "split_res_core.hpp"

namespace rsh {

// Plans with an unrolled instance: M <= 32 * kIterResMaxSteps = 800 directions.
constexpr int kIterResMaxSteps = 25;

// Whether the panel slice is streamed through LDS by K-step (KS) instead of held
// whole. Held whole it bounds the row group; beyond 19 K-steps (two parts) or 13
// (three) a two-slot ring of K-steps leaves room for five row blocks. At 100,002
// cells, us per iteration, whole / streamed: two parts, 500 directions 224 / 285,
// 590 303 / 355; three parts, 350 directions 211 / 257, 400 281 / 286.
constexpr bool iter_res_k_streamed(int nt, int steps) { return steps > (nt == 2 ? 19 : 13); }
// Most row blocks per workgroup: eight waves, two per SIMD, hold five in 256
// registers; a whole slice of five fits LDS up to 15 (two parts) or 10 (three)
// K-steps, of four beyond.
constexpr int iter_res_max_rbw(int nt, int steps) {
    return !iter_res_k_streamed(nt, steps) && steps > (nt == 2 ? 15 : 10) ? 4 : 5;
}
// Row blocks per workgroup for rb_need row blocks: as few groups as fit, then balanced.
constexpr int iter_res_rbw(int nt, int steps, int rb_need) {
    const int mx = iter_res_max_rbw(nt, steps);
    const int groups = (rb_need + mx - 1) / mx;
    return (rb_need + groups - 1) / groups;
}
constexpr size_t iter_res_lds_bytes(int nt, int steps, int rbw) {
    return (size_t)(iter_res_k_streamed(nt, steps) ? 2 : steps) * rbw * nt * 1024 + (size_t)rbw * 16 * 4;
}

struct IterResArgs {
    bool launch;  // false: only set the kernel's dynamic-LDS limit
    int rb, steps, waves, grid;
    const BatchProblem* probs;
    const BatchItem* items;
    const int* meta;
    int parity;
    hipStream_t st;
};

// Source iteration I <- (1 - a) B + a S(I) on split state for a batch of
// problems, resident-panel form (the grouped counterpart of split_single_res.hpp).
// Work: meta = [problems of the class, row groups G, sets, chunks]. Workgroup b runs on
// XCD b % 8; the G workgroups of a set sit on one XCD and take one row group each
// of the same chunks at about the same time, so they share its L2 copy of the
// state. A class's chunks, one problem's after the other's (items[i].tile of them
// before problem i), are dealt to its 8 sets per set index in runs of equal length:
// dealt round-robin, every workgroup loaded a slice of every problem (28,790 and
// 34,497 cells x 194, two parts, 67 us an iteration, in runs 59;
// 10,368, 24,576, 48,000 and 3000 x 200 88 and 66). Every chunk of a class
// costs the same, so dealing them beforehand balances as well as a queue would,
// and a workgroup keeps its panel slice and its state prefetch running over all
// of its chunks of a problem: with items of 1-4 chunks from a queue, each one
// loaded the slice again and waited for its first state vectors. The slice (all
// K-steps) and the row scales go into LDS once per problem, then the chunks are
// swept as in split_resident_kernel (state prefetch across chunk boundaries,
// issued before the stores).
// KS (K-streamed panel, for long K ranges): the slice is not held whole; a
// two-slot LDS ring holds one K-step each, the next K-step's part of the slice
// is loaded into registers while the current one is multiplied, written into
// the other slot after it and published by an LDS-only barrier per K-step. The
// LDS then no longer bounds the row group: at M = 800 it holds 5 row blocks
// instead of 2 or 3, so each state fragment read from L2 feeds twice the MFMAs.
// The epilogue is that of the streaming grouped kernel (kernels_iter_split.hip): S in FP64 from
// the two accumulators and the exact scales, I_new = (1 - a) B + a S, the
// residual against the state the MFMAs consumed, I_new re-split into the other
// ping-pong buffer. Same products, same order: bit-identical to it.
template <int RBW, int FMT, int NT, int STEPS, int W, bool KS>
__global__ __launch_bounds__(64 * W, W == 4 ? 2 : 1) void grouped_iter_split_res_kernel(
    const BatchProblem* __restrict__ probs, const BatchItem* __restrict__ items, const int* __restrict__ meta,
    int parity) {
    typedef typename Fmt<FMT>::V V;
    typedef typename Fmt<FMT>::T T;
    // Chunk of CT 16-cell tiles, TT per wave: 8 waves x 2 tiles (one workgroup
    // per CU), or 4 waves x 2 tiles (two workgroups per CU, whose epilogues and
    // barriers are independent, so one's epilogue overlaps the other's MFMAs).
    constexpr int TT = kResTiles;
    constexpr int CT = W * TT;
    constexpr int XD = NT == 2 ? 3 : 2;  // shallower than the plain kernel: the epilogue needs the registers
    constexpr int steps = STEPS;
    constexpr int64_t units = (int64_t)steps * RBW * NT * 64;  // panel slice of a row group
    constexpr int SU = RBW * NT * 64;                          // one K-step of it
    constexpr int64_t lds_units = KS ? 2 * SU : units;
    // KS: 16-byte units of one K-step per thread (the last pass partial)
    constexpr int PER = (SU + 64 * W - 1) / (64 * W);
    extern __shared__ v4u lds[];  // [steps][RBW][NT][64] (KS: [2][RBW][NT][64]), then 16 RBW row scales
    float* rscale = reinterpret_cast<float*>(lds + lds_units);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // uniform: scalar tile offsets
    const int g = lane >> 4;
    const int cl = lane & 15;
    const int xcd = blockIdx.x % kXcds;
    const int nprobs = meta[0], groups = meta[1], sets = meta[2];
    const int set = blockIdx.x / kXcds / groups, rg = blockIdx.x / kXcds % groups;
    if (set >= sets) return;  // whole workgroup leaves together
    // this workgroup's run of the class's chunks: [lo, hi)
    const int slots = kXcds * sets, slot = set * kXcds + xcd, each = meta[3] / slots, over = meta[3] % slots;
    const int64_t lo = (int64_t)slot * each + (slot < over ? slot : over), hi = lo + each + (slot < over ? 1 : 0);
    constexpr int64_t tile_units = (int64_t)steps * NT * 64;
    constexpr int tile_bytes = (int)(tile_units * 16);
    for (int pi = 0; pi < nprobs; pi++) {
        const BatchItem item = items[pi];
        const BatchProblem& P = probs[item.problem];
        const int64_t n = P.n;
        const int64_t tiles = (n + 15) / 16;
        const int64_t chunks = (tiles + CT - 1) / CT;
        const int64_t c0 = lo > item.tile ? lo - item.tile : 0;
        const int64_t c1 = hi - item.tile < chunks ? hi - item.tile : chunks;
        if (c0 >= c1) continue;
        __syncthreads();  // every wave is done with the previous problem's LDS panel
        const int row0 = rg * RBW * 16;
        const v4u* __restrict__ src = static_cast<const v4u*>(P.spanel) + (int64_t)rg * units;
        // KS: the slice through a buffer descriptor (global loads, which an
        // LDS-only barrier does not wait for) and K-step 0 into ring slot 0.
        const __amdgpu_buffer_rsrc_t psrc =
            __builtin_amdgcn_make_buffer_rsrc(const_cast<v4u*>(src), (short)0, (int)(units * 16), kBufWord3);
        v4u preg[PER];
        auto panel_load = [&](int step) {
#pragma unroll
            for (int i = 0; i < PER; i++) {
                const int u = (int)threadIdx.x + i * 64 * W;
                if (SU % (64 * W) == 0 || u < SU)
                    preg[i] = __builtin_bit_cast(
                        v4u, __builtin_amdgcn_raw_buffer_load_b128(psrc, u * 16, step * SU * 16, 0));
            }
        };
        auto panel_store = [&](int slot) {
#pragma unroll
            for (int i = 0; i < PER; i++) {
                const int u = (int)threadIdx.x + i * 64 * W;
                if (SU % (64 * W) == 0 || u < SU) lds[slot * SU + u] = preg[i];
            }
        };
        if constexpr (KS) {
            panel_load(0);
            panel_store(0);
        } else {
            // eight loads in flight per thread (a load and its LDS store at a time
            // cost a memory round trip each: ~10 us for 70 KB)
            constexpr int B = 8, TH = 64 * W;
            v4u buf[B];
            for (int u0 = 0; u0 < (int)units; u0 += B * TH) {
#pragma unroll
                for (int i = 0; i < B; i++) {
                    const int u = u0 + i * TH + (int)threadIdx.x;
                    buf[i] = src[u < (int)units ? u : (int)units - 1];
                }
#pragma unroll
                for (int i = 0; i < B; i++) {
                    const int u = u0 + i * TH + (int)threadIdx.x;
                    if (u < (int)units) lds[u] = buf[i];
                }
            }
        }
        for (int r = threadIdx.x; r < RBW * 16; r += 64 * W)
            rscale[r] = row0 + r < P.m ? P.row_inv[row0 + r] : 0.0f;
        __syncthreads();

        const v4u* __restrict__ st_in = static_cast<const v4u*>(P.state[parity]);
        v4u* __restrict__ st_out = static_cast<v4u*>(P.state[parity ^ 1]);

        __amdgpu_buffer_rsrc_t xs;
        int xoff[TT];
        int64_t ntile_of_bound = 0;
        auto bind_chunk = [&](int64_t chunk) {
            const int64_t ct_chunk = chunk * CT;
            const int ntile = (int)(tiles - ct_chunk < CT ? tiles - ct_chunk : CT);
            ntile_of_bound = ntile;
            xs = __builtin_amdgcn_make_buffer_rsrc(const_cast<v4u*>(st_in + ct_chunk * tile_units), (short)0,
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
        auto prefetch_head = [&]() {
            static_for<0, XD>([&](auto u) {
                if (u.value < steps) load_x(u, u.value);
            });
        };
        RelMax rm;
        bind_chunk(c0);
        prefetch_head();
        int pc = 0;  // KS: ring slot of the chunk's K-step 0
        for (int64_t chunk = c0; chunk < c1; chunk++) {
            const int64_t ct0 = chunk * CT + wave * TT;
            float cinv[TT];
#pragma unroll
            for (int q = 0; q < TT; q++) {
                const int64_t cell = (ct0 + q) * 16 + cl;
                cinv[q] = P.cell_inv[cell < n ? cell : n - 1];
            }
            v4f accm[RBW][TT], accx[RBW][TT];
#pragma unroll
            for (int i = 0; i < RBW; i++)
#pragma unroll
                for (int q = 0; q < TT; q++) {
                    accm[i][q] = v4f{0.f, 0.f, 0.f, 0.f};
                    accx[i][q] = v4f{0.f, 0.f, 0.f, 0.f};
                }
            // KS: K-step t of this chunk sits in ring slot (t + pc) & 1 (with an
            // odd STEPS the parity flips from chunk to chunk); the step after
            // the last one is K-step 0 of the next chunk.
            const bool more_chunks = chunk + 1 < c1;
            static_for<0, STEPS>([&](auto tt) {
                constexpr int t = decltype(tt)::value;
                constexpr int sl = t % XD;
                __builtin_amdgcn_sched_barrier(0);
                // KS: the next K-step's panel load goes out before this step's
                // state prefetch, so that waiting for it (before its LDS store)
                // leaves the state loads in flight (one in-order counter).
                const bool next = KS && (t + 1 < STEPS || more_chunks);
                if constexpr (KS) {
                    if (next) panel_load((t + 1) % STEPS);
                }
                V bx[TT][NT];
#pragma unroll
                for (int q = 0; q < TT; q++)
#pragma unroll
                    for (int p = 0; p < NT; p++) bx[q][p] = __builtin_bit_cast(V, xr[sl][q][p]);
                if constexpr (t + XD < STEPS) load_x(std::integral_constant<int, sl>{}, t + XD);
                V ahi[RBW];
                if constexpr (KS) {
                    res_mfma_step<RBW, FMT, NT, TT, NT, false>(lds + ((t + pc) & 1) * SU + lane, nullptr, ahi, bx,
                                                               nullptr, accm, accx);
                    if (next) panel_store((t + 1 + pc) & 1);
                    lds_barrier();
                } else {
                    res_mfma_step<RBW, FMT, NT, TT, NT, false>(lds + (int64_t)t * RBW * NT * 64 + lane, nullptr, ahi,
                                                               bx, nullptr, accm, accx);
                }
            });
            // This chunk's state (old values) and the output chunk through buffer
            // descriptors (uniform base, 32-bit offsets), kept before the next
            // chunk's head is bound and requested ahead of this chunk's stores.
            const __amdgpu_buffer_rsrc_t xin = xs;
            const int ntile_cur = (int)ntile_of_bound;
            const __amdgpu_buffer_rsrc_t xout = __builtin_amdgcn_make_buffer_rsrc(
                st_out + chunk * CT * tile_units, (short)0, ntile_cur * tile_bytes, kBufWord3);
            __builtin_amdgcn_sched_barrier(0);
            if (more_chunks) {
                bind_chunk(chunk + 1);
                prefetch_head();
            }
            pc ^= STEPS & 1;
            __builtin_amdgcn_sched_barrier(0);
            int zoff;
            asm volatile("v_mov_b32 %0, 0" : "=v"(zoff));
            const float* __restrict__ rs = rscale + 4 * g + zoff;
            const double oma = P.one_minus_albedo, alb = P.albedo;  // in registers across the stores
            // Branch-free epilogue: every load is issued with an address that is
            // in range (cell clamped to the last cell, a padding row block to the
            // last real one), results of invalid positions are dropped by giving
            // their stores an offset past the buffer's range (the hardware
            // discards such stores) and by leaving them out of the residual. So
            // the whole epilogue is one basic block, and the scheduler overlaps the
            // loads of later (tile, row block) pairs with the arithmetic of earlier
            // ones instead of waiting for one memory round trip per pair.
            const int rb_last = (P.m + 15) / 16 - 1;  // last row block with rows
            constexpr int kDropped = 0x7FFF0000;      // store offset past any buffer's range
            // (tile q, row block i) pairs in order p = q * RBW + i; the loads of
            // pair p + LA are issued before the stores of pair p (the compiler
            // may not move a load above a store to another buffer: it cannot tell
            // that they do not alias). LA = 2 measured best at 4 and 5 row
            // blocks (with B in FP32; 4 was slower for three parts).
            constexpr int NPAIR = TT * RBW;
            constexpr int LA = RBW <= 3 ? 3 : 2;
            float bv[LA + 1][4];
            v2u oldraw[LA + 1][NT];
            auto pair_rb = [&](int i, bool& rb_ok) {
                const int rbg = rg * RBW + i;
                rb_ok = rbg <= rb_last;  // a padding row block has no rows and no state
                return rb_ok ? rbg : rb_last;
            };
            auto pair_voff = [&](int q, int rbe) {
                const int vlane = (2 * (rbe & 1) + (g >> 1)) * 16 + cl;
                return ((wave * TT + q) * (int)tile_units + vlane) * 16 + 8 * (g & 1);
            };
            auto load_pair = [&](auto pp) {
                constexpr int pi = decltype(pp)::value, q = pi / RBW, i = pi % RBW, buf = pi % (LA + 1);
                bool rb_ok;
                const int rbe = pair_rb(i, rb_ok);
                // the source term in output-tile order: this lane's 4 rows of its
                // cell are one 16-byte vector (the tile clamped into the array)
                const int64_t tq = ct0 + q < tiles ? ct0 + q : tiles - 1;
                const __amdgpu_buffer_rsrc_t bsrc = __builtin_amdgcn_make_buffer_rsrc(
                    const_cast<float*>(P.Bs) + (int64_t)rbe * tiles * 256, (short)0, (int)(tiles * 1024), kBufWord3);
                const v4f b4 = __builtin_bit_cast(
                    v4f, __builtin_amdgcn_raw_buffer_load_b128(bsrc, (int)((tq * 64 + lane) * 16), 0, 0));
#pragma unroll
                for (int r = 0; r < 4; r++) bv[buf][r] = b4[r];
                const int voff = pair_voff(q, rbe);
#pragma unroll
                for (int t = 0; t < NT; t++)
                    oldraw[buf][t] = __builtin_bit_cast(
                        v2u, __builtin_amdgcn_raw_buffer_load_b64(xin, voff, ((rbe >> 1) * NT + t) * 1024, 0));
            };
            static_for<0, (LA < NPAIR ? LA : NPAIR)>(load_pair);
            static_for<0, NPAIR>([&](auto pp) {
                constexpr int pi = decltype(pp)::value, q = pi / RBW, i = pi % RBW, buf = pi % (LA + 1);
                if constexpr (pi + LA < NPAIR) load_pair(std::integral_constant<int, pi + LA>{});
                const int tl = wave * TT + q;  // tile within the chunk
                const int64_t cell = (ct0 + q) * 16 + cl;
                bool rb_ok;
                const int rbe = pair_rb(i, rb_ok);
                // B rows exist up to the row block's end (the source array holds
                // whole row blocks, padding rows zero). A padding row (k >= M)
                // has zero panel rows, zero B and zero old state: nv = 0, parts
                // 0, residual term 0 / 0 = NaN, which fmax drops.
                const bool ok = tl < ntile_cur && cell < n && rb_ok;
                // The cell and row scales are powers of two, so scaling in FP32
                // is exact and commutes with every rounding below: the same
                // values as scaling in FP64, with four FP64 operations fewer per
                // result (FP64 runs at half the FP32 rate on the VALU).
                const float cif = cinv[q];
                const float csf = 1.0f / cif;  // power of two: exact
                T newp[NT][4];
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const float sc = rs[i * 16 + r] * cif;
                    const double S = split_value(accm[i][q][r] * sc, accx[i][q][r] * sc);
                    // explicit FMA: the same rounding in every split iteration kernel
                    const double nv = __builtin_fma(alb, S, oma * (double)bv[buf][r]);
                    float of = 0.0f;
#pragma unroll
                    for (int t = NT - 1; t >= 0; t--) {
                        T tmp[4];
                        __builtin_memcpy(tmp, &oldraw[buf][t], 8);
                        of += (float)tmp[r];
                    }
                    const double old = (double)(of * cif);
                    rm.add(old - nv, nv, ok);
                    T qp[NT];
                    split_parts<FMT, NT>((float)nv * csf, qp);
#pragma unroll
                    for (int t = 0; t < NT; t++) newp[t][r] = qp[t];
                }
                const int soff = ok ? pair_voff(q, rbe) : kDropped;
#pragma unroll
                for (int t = 0; t < NT; t++) {
                    v2u raw;
                    __builtin_memcpy(&raw, newp[t], 8);
                    __builtin_amdgcn_raw_buffer_store_b64(raw, xout, soff, ((rbe >> 1) * NT + t) * 1024, 0);
                }
            });
        }
        double res = rm.value();
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) res = fmax(res, __shfl_xor(res, off, 64));
        if (lane == 0 && res > 0.0)
            atomicMax(P.resid + parity, (unsigned long long)__double_as_longlong(res));
    }
}

template <int RBW, int FMT, int NT, int STEPS>
hipError_t iter_res_one(const IterResArgs& a) {
    constexpr bool KS = iter_res_k_streamed(NT, STEPS);
    constexpr size_t lds = iter_res_lds_bytes(NT, STEPS, RBW);
    static_assert(lds <= (size_t)kResLdsBytes, "the panel slice fits LDS");
    auto kern = grouped_iter_split_res_kernel<RBW, FMT, NT, STEPS, kResWaves, KS>;
    // the four-wave form where it was ever faster than the eight-wave one
    if constexpr (STEPS == 7 || STEPS == 13 || STEPS == 25) {
        if (a.waves == 4) kern = grouped_iter_split_res_kernel<RBW, FMT, NT, STEPS, 4, KS>;
    } else if (a.waves != kResWaves) {
        return hipErrorInvalidValue;
    }
    if (!a.launch)
        return hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                                   (int)lds);
    hipLaunchKernelGGL(kern, dim3(a.grid), dim3(64 * a.waves), lds, a.st, a.probs, a.items, a.meta, a.parity);
    return hipGetLastError();
}

// The plans of STEPS K-steps: M in (32 (STEPS - 1), 32 STEPS] has 2 STEPS - 1 or 2 STEPS row blocks.
template <int FMT, int NT, int STEPS>
hipError_t iter_res_steps(const IterResArgs& a) {
    constexpr int r1 = iter_res_rbw(NT, STEPS, 2 * STEPS - 1), r2 = iter_res_rbw(NT, STEPS, 2 * STEPS);
    if (a.rb == r1) return iter_res_one<r1, FMT, NT, STEPS>(a);
    if constexpr (r2 != r1) {
        if (a.rb == r2) return iter_res_one<r2, FMT, NT, STEPS>(a);
    }
    return hipErrorInvalidValue;
}

template <int I, int HI, typename F>
void iter_res_each(F&& f) {
    if constexpr (I <= HI) {
        f(std::integral_constant<int, I>{});
        iter_res_each<I + 1, HI>(f);
    }
}

// K-steps LO .. HI of one form; explicitly instantiated by the kernels_iter_res_*.hip files.
template <int FMT, int NT, int LO, int HI>
hipError_t iter_res_range(const IterResArgs& a);

#define RSH_ITER_RES_RANGE(FMT, NT, LO, HI)                                                        \
    namespace rsh {                                                                                \
    template <>                                                                                    \
    hipError_t iter_res_range<FMT, NT, LO, HI>(const IterResArgs& a) {                             \
        hipError_t e = hipErrorInvalidValue;                                                       \
        if (a.waves != 4 && a.waves != kResWaves) return e;                                        \
        iter_res_each<LO, HI>([&](auto s) {                                                        \
            constexpr int S = decltype(s)::value;                                                  \
            if (a.steps == S) e = iter_res_steps<FMT, NT, S>(a);                                   \
        });                                                                                        \
        return e;                                                                                  \
    }                                                                                              \
    }

}  // namespace rsh
