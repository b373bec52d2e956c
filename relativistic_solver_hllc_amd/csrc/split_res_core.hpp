// Device code shared by the resident-panel split kernels: the single-problem
// kernel (kernels_split_resident.hip) and the grouped source-iteration kernel
// (split_iter_res.hpp).
#pragma once

#include "mfma_split_core.hpp"

namespace rsh {

constexpr int kResWaves = 8;   // waves per workgroup of the grouped iteration kernel (2 per SIMD)
constexpr int kResTiles = 2;   // 16-cell tiles per wave of the grouped iteration kernel
constexpr int kXcds = 8;       // MI355X: 8 XCDs, workgroups dispatched round-robin
constexpr int kResLdsBytes = 160 * 1024;
// Buffer descriptor word 3 for raw (untyped) gfx9 buffer access: 32-bit data
// format, so that the hardware does not treat the descriptor as invalid.
constexpr int kBufWord3 = 0x00020000;

template <int I, int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_for<I + 1, N>(f);
    }
}

// Workgroup barrier that orders LDS only: it waits for this wave's LDS
// accesses, not for its global loads in flight (the state prefetch).
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// One K-step of MFMAs for TT tiles x RBW row blocks: A fragments of the parts
// resident in LDS from a_base (this lane's vector of the step's first
// fragment; NL parts per row block), the lo part of a three-part panel from
// alo when NL < NT, B from the state vectors in bx. A fragments of one part at
// a time (part-major), so that only RBW fragments are live. Product-major
// order: each round touches every (row block, tile) accumulator once, so an
// MFMA never waits for the previous result of its own accumulator. The main
// product hi*hi of the step is formed in fresh accumulators, one row block at a
// time (main_round), and added to accm with main_add. Products
// and their order per accumulator are those of the streaming kernel (cross:
// hi*lo + lo*hi; for three parts hi*lo, hi*mid, mid*mid, mid*hi, lo*hi).
//
// ahi (in/out): with AHEAD, ahi holds this step's hi fragments on entry, and
// the hi fragments of the K-step at a_next are read into it as soon as this
// step is done with its own (after the main products), so that the next step's
// first MFMAs do not wait for LDS. Without AHEAD, the step reads its own hi
// fragments first.
template <int RBW, int FMT, int NT, int TT, int NL, bool AHEAD>
__device__ __forceinline__ void res_mfma_step(const v4u* a_base, const v4u* a_next,
                                              typename Fmt<FMT>::V (&ahi)[RBW],
                                              const typename Fmt<FMT>::V (&bx)[TT][NT],
                                              const typename Fmt<FMT>::V* alo, v4f (&accm)[RBW][TT],
                                              v4f (&accx)[RBW][TT]) {
    typedef typename Fmt<FMT>::V V;
    V (&a)[RBW] = ahi;
    V am[RBW];  // second (and third) part
    auto fetch_into = [&](V(&dst)[RBW], const v4u* base, int p) {
#pragma unroll
        for (int i = 0; i < RBW; i++) dst[i] = __builtin_bit_cast(V, base[(i * NL + p) * 64]);
    };
    auto round = [&](const V(&af)[RBW], v4f (&acc)[RBW][TT], int pb) {
#pragma unroll
        for (int i = 0; i < RBW; i++)
#pragma unroll
            for (int q = 0; q < TT; q++) acc[i][q] = Fmt<FMT>::mfma(af[i], bx[q][pb], acc[i][q]);
    };
    // a holds the hi fragments. Software-pipelined over row blocks: row block
    // i's products are issued before row block i - 1's are added (so that the
    // adds do not wait for the MFMA just issued), and row block i's MFMAs are
    // ordered after row block i - 2's adds (order_after; two row blocks of
    // products in flight at most).
    auto main_round = [&]() {
        v4f ms[2][TT];
        static_for<0, RBW>([&](auto ii) {
            constexpr int i = decltype(ii)::value;
            order_after(a[i], accm[(i + 2 * RBW - 2) % RBW]);
#pragma unroll
            for (int q = 0; q < TT; q++) ms[i & 1][q] = Fmt<FMT>::mfma(a[i], bx[q][0], v4f{0.f, 0.f, 0.f, 0.f});
            if constexpr (i >= 1) {
#pragma unroll
                for (int q = 0; q < TT; q++) accm[i - 1][q] = main_add(accm[i - 1][q], ms[(i - 1) & 1][q]);
            }
        });
#pragma unroll
        for (int q = 0; q < TT; q++) accm[RBW - 1][q] = main_add(accm[RBW - 1][q], ms[(RBW - 1) & 1][q]);
    };
    if constexpr (!AHEAD) fetch_into(a, a_base, 0);
    fetch_into(am, a_base, 1);
    if constexpr (NT == 2) {
        round(a, accx, 1);
        main_round();
        if constexpr (AHEAD) fetch_into(a, a_next, 0);
        round(am, accx, 0);
    } else {
        round(a, accx, 2);
        round(a, accx, 1);
        main_round();
        if constexpr (AHEAD) fetch_into(a, a_next, 0);
        round(am, accx, 1);
        round(am, accx, 0);
        if constexpr (NL == 3) {
            fetch_into(am, a_base, 2);
        } else {
#pragma unroll
            for (int i = 0; i < RBW; i++) am[i] = alo[i];
        }
        round(am, accx, 0);
    }
}

}  // namespace rsh
