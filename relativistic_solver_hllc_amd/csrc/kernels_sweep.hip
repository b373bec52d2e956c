// Transport sweep (short characteristics) on the GPU: every direction walks its
// cells in upwind order and updates the intensities on the cells' out faces.
// Replaces the direction loop of MPI_CalculateIllumAsync
// (solve_module/illum/Illum_async.cpp:725-784) with CalculateIllumeOnInnerFace
// (:172-199), BoundaryConditions (solve_module/illum/illum_utils.cpp:407-471),
// GetCurIllum (:259-430, classes 0, 1, 2, 3, 10) and ReCalcIllum (:472-510).
//
// Parallel form. The reference runs one direction per OpenMP thread, each a
// sequential walk of sorted_id_cell. Here one workgroup owns one direction. The
// unit of work is one out face of a cell (three nodes, each traced back to an in
// face), one thread each; a pass is a set of cells whose upstream cells are all in
// earlier passes (sweep.cpp picks them), and passes follow one another with one
// LDS-only barrier each.
//
// Face values. The reference keeps three node values per face and only ever
// uses their mean ((c0 + c1 + c2) / 3, both when a downstream cell reads its in
// face and when ReCalcIllum stores the face intensity), so this kernel keeps that
// mean, computed in the same order. A pass writes its faces' values into an LDS
// ring of the last 16 passes, from which downstream nodes read them; an upstream
// value that has left the ring (host-coded) is read from the result. In the step
// after a pass, each of its cells' four values (own out faces, neighbours' out
// faces, boundary values) are gathered from the ring and stored to the new illum
// array [M][N][4] (the ReCalcIllum output layout), two lanes of 16 bytes per cell:
// every 32-byte cell is stored once and whole. A face out on both sides
// (|n . omega| <= eps) has two values; the later cell's in the given order also
// goes to the earlier cell's entry, at the end of the direction. The residual
// max |old - new| / new follows, with the reference's comparison (a NaN ratio
// never wins).
//
// Schedule. In step p a wave requests the by-cell values of pass p + 1, the
// records and s values of pass p + 2 and the codes of pass p's cells, then
// computes pass p, then stores the cells of pass p - 1. Vector memory completes in
// order, and step p + 1 uses the records requested in step p - 1 before it
// requests more: so every wave has completed its stores of step p - 2 when it
// enters step p. Pass q's cells are stored in step q + 1, complete before the
// barrier that ends step q + 3; a value is read from the result only when at least
// a ring's positions follow it (16 passes of full size, so q <= p - 16), requested
// in step p - 1 or later. Threads past a pass's end load its first record, so no
// branch surrounds a load and the wait counters stay exact; waves that hold only
// such threads skip the arithmetic.
//
// What bounds it. Up to ~50 directions a full pass takes 3 us, 2 of them its
// arithmetic (1024 faces of class 1 with two exponentials per node, the reference's
// expression); with a workgroup on every CU memory: 204 bytes per cell and
// direction, records and s values 80 of them, each added direction then costs its
// bytes at 5 TB/s. One thread per cell (up to nine nodes in a row, each wave
// executing all of them when one lane has three out faces), each lane storing its
// face values to both cells' entries 8 bytes at a time, took (us per sweep,
// cubes per edge x directions, class 1 or 10) 6 x 84: 143, 12 x 66: 306,
// 18 x 141: 756, 24 x 200: 1242, 32 x 400: 5800; this form 47, 120, 322, 1058, 5100.
// On the way, at 24 x 200: 8-byte stores to both entries 450 us of 1177; whole
// cells as two 16-byte stores per lane 1130, as two lanes 1095; the s values two
// passes ahead 1078; streamed arrays loaded past the caches 1060. Accumulating the
// residual with the stores instead of a pass at the end (185 us, 5.7 TB/s): 1237
// against 1095 (its gathers of old values wait).
#include "rsh_internal.hpp"

namespace rsh {

namespace {

// BoundaryConditions, non-Sphere build: OutSource (-3) -> 1, Free (-1),
// Lock (-2), InnerSource (-4) -> 0 (types are validated on the host).
__device__ inline double boundary_value(int type_bound) { return type_bound == -3 ? 1.0 : 0.0; }

// GetCurIllum of one class, in the reference's expression order.
template <int CLS>
__device__ inline double cur_illum(bool in_source, double s, double I_0, double S) {
    double Q, alpha, betta;
    if constexpr (CLS == 2) {
        const double ss = s * 388189 * 1e5;
        alpha = 1;
        Q = 1;
        const double I = I_0 * exp(-alpha * ss) + Q * (1 - exp(-alpha * ss)) / alpha;
        return I < 0 ? 0 : I;
    } else {
        if constexpr (CLS == 0) {
            // |x - (0.5, 0, 0)| < 0.05 at the node, evaluated on the host
            Q = 0; alpha = 2; betta = 1;
            if (in_source) { Q = 0; alpha = 0.5; betta = 0.5; }
        } else if constexpr (CLS == 1) {
            Q = 1; alpha = 1; betta = alpha / 2;
        } else if constexpr (CLS == 3) {
            alpha = 0; betta = alpha / 2; Q = 0;
        } else {  // 10
            Q = 0; alpha = 0.5; betta = 100;
        }
        const double k = alpha + betta;
        double I;
        if (k > 1e-10) I = (exp(-k * s) * (I_0 * k + (exp(k * s) - 1) * (Q + S * betta))) / k;
        else I = (1 - s * k) * (I_0 + s * (Q + S * betta));
        return I < 0 ? 0 : I;
    }
}

// What a thread needs for its face of a pass: the record, then the by-cell values.
struct PassRec {
    SweepFace f;
    double s[3];
    int first, cnt;  // the pass's faces
};
struct PassVal {
    double S;
    double far[3];  // upstream values no longer in the ring
};
// Half a cell whose four face values are complete: two values' codes.
struct DoneRec {
    int2 code;
    int cell;
    int cnt;  // halves: twice the pass's cells
};

// The pass table is read through the scalar cache (constant address space,
// uniform index): its loads retire on their own counter, so reading the next
// pass's first position never waits for the vector loads and stores in flight.
typedef const int32_t __attribute__((address_space(4)))* const_i32_ptr;

// Global-address-space view of a pointer read from the direction table, so
// that its loads are vector-memory loads (a generic "flat" load also counts on
// the scalar-load counter, and waiting for a scalar load would then wait for it).
template <typename T>
__device__ inline const __attribute__((address_space(1))) T* gptr(const T* p) {
    return (const __attribute__((address_space(1))) T*)p;
}

// Threads past a pass's end take its first record (ignored), so that no branch
// surrounds the loads.
__device__ inline int lane_of(int cnt) { return (int)threadIdx.x < cnt ? (int)threadIdx.x : 0; }

__device__ inline void load_rec(const SweepDirDev& d, int pi, PassRec& x) {
    typedef int32_t v4i __attribute__((ext_vector_type(4)));
    const const_i32_ptr pt = (const_i32_ptr)d.pass + 4 * pi;
    x.first = pt[0];
    x.cnt = pt[1];
    x.f = __builtin_bit_cast(SweepFace, __builtin_nontemporal_load(gptr(reinterpret_cast<const v4i*>(d.faces)) + x.first + lane_of(x.cnt)));
    const double* s3 = d.s3 + 3 * (int64_t)x.first + lane_of(x.cnt);
#pragma unroll
    for (int j = 0; j < 3; j++) x.s[j] = __builtin_nontemporal_load(gptr(s3) + j * x.cnt);
}

__device__ inline void load_done(const SweepDirDev& d, int pi, DoneRec& x) {
    typedef int32_t v2i __attribute__((ext_vector_type(2)));
    const const_i32_ptr pt = (const_i32_ptr)d.pass + 4 * pi;
    x.cnt = 2 * pt[3];
    const int64_t i = 2 * (int64_t)pt[2] + lane_of(x.cnt);
    x.code = __builtin_bit_cast(int2, __builtin_nontemporal_load(gptr(reinterpret_cast<const v2i*>(d.codes)) + i));
    x.cell = gptr(d.cells)[i >> 1];
}

__device__ inline bool is_far(int code) { return code <= kSweepFar; }
__device__ inline int64_t far_entry(int code) { return is_far(code) ? kSweepFar - code : 0; }

__device__ inline void load_val(const SweepDirDev& d, const PassRec& x, const double* __restrict__ Sk,
                                const double* fv, PassVal& y) {
    y.S = Sk[x.f.cell & kSweepCellMask];
    if (__builtin_amdgcn_ballot_w64(is_far(x.f.up[0]) || is_far(x.f.up[1]) || is_far(x.f.up[2]))) {
#pragma unroll
        for (int j = 0; j < 3; j++) y.far[j] = fv[far_entry(x.f.up[j])];
    }
}

// ReCalcIllum's per-entry term with the reference's comparison (a NaN ratio never wins).
__device__ inline void residual_term(double old, double cur, double& loc) {
    const double b = fabs(old - cur) / cur;
    if (b > loc) loc = b;
}

// Barrier that orders only LDS accesses: global stores may stay in flight across it.
__device__ inline void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

template <int CLS, int BLOCK>
__global__ __launch_bounds__(BLOCK) void sweep_kernel(const SweepDirDev* __restrict__ dirs, int64_t n,
                                                      const double* __restrict__ S, int64_t ld,
                                                      const double* __restrict__ old_illum, double* new_illum,
                                                      double* __restrict__ norm) {
    typedef double v2d __attribute__((ext_vector_type(2)));
    const int k = blockIdx.x;
    const SweepDirDev d = dirs[k];
    double* fv = new_illum + (int64_t)k * n * 4;
    const double* __restrict__ Sk = S + (int64_t)k * ld;
    const double* __restrict__ ok = old_illum ? old_illum + (int64_t)k * n * 4 : nullptr;
    constexpr int kRing = kSweepRing * BLOCK;
    __shared__ double ring[kRing];
    const int last = d.passes - 1;
    const int wave_first = __builtin_amdgcn_readfirstlane(threadIdx.x & ~63u);
    // A face value by its code (codes that are not in the ring read slot 0, ignored).
    auto value = [&](int code, double far) {
        const double r = ring[code >= 0 ? code : 0];
        return code >= 0 ? r : is_far(code) ? far : boundary_value(code == kSweepOne ? -3 : -1);
    };
    auto step = [&](PassRec& cur, PassVal& cv, PassRec& nx1, PassVal& nv, PassRec& nx2, DoneRec& done, DoneRec& ndone,
                    int pi) {
        load_val(d, nx1, Sk, fv, nv);
        load_rec(d, pi + 1 < last ? pi + 2 : last, nx2);
        load_done(d, pi, ndone);
        double far_x = 0, far_y = 0;
        if (__builtin_amdgcn_ballot_w64(is_far(done.code.x) || is_far(done.code.y))) {
            far_x = fv[far_entry(done.code.x)];
            far_y = fv[far_entry(done.code.y)];
        }
        if (wave_first < cur.cnt) {
            double I[3];
#pragma unroll
            for (int j = 0; j < 3; j++)
                I[j] = cur_illum<CLS>((cur.f.cell >> (29 + j)) & 1, cur.s[j], value(cur.f.up[j], cv.far[j]), cv.S);
            const double v = (I[0] + I[1] + I[2]) / 3;
            if ((int)threadIdx.x < cur.cnt) ring[(cur.first + (int)threadIdx.x) & (kRing - 1)] = v;
        }
        if (wave_first < done.cnt) {
            const v2d a = {value(done.code.x, far_x), value(done.code.y, far_y)};
            if ((int)threadIdx.x < done.cnt)
                *reinterpret_cast<v2d*>(fv + (int64_t)done.cell * 4 + 2 * (threadIdx.x & 1)) = a;
        }
        // every pass ends at a barrier: no wave runs more than a pass ahead, so
        // a ring slot is rewritten only after every read of its previous value
        lds_barrier();
    };
    PassRec ra, rb, rc;
    PassVal va = {}, vb = {};
    DoneRec da = {}, db = {};
    load_rec(d, 0, ra);
    load_rec(d, last < 1 ? last : 1, rb);
    load_val(d, ra, Sk, fv, va);
    // unrolled by six with the buffers taking turns: no register copy of a value
    // still in flight (which would wait for it)
    for (int pi = 0; pi < d.passes; pi += 6) {
        step(ra, va, rb, vb, rc, da, db, pi);
        if (pi + 1 >= d.passes) break;
        step(rb, vb, rc, va, ra, db, da, pi + 1);
        if (pi + 2 >= d.passes) break;
        step(rc, va, ra, vb, rb, da, db, pi + 2);
        if (pi + 3 >= d.passes) break;
        step(ra, vb, rb, va, rc, db, da, pi + 3);
        if (pi + 4 >= d.passes) break;
        step(rb, va, rc, vb, ra, da, db, pi + 4);
        if (pi + 5 >= d.passes) break;
        step(rc, vb, ra, va, rb, db, da, pi + 5);
    }
    // faces out on both sides: the earlier cell's entry takes the later cell's value
    if (d.fixes) {
        __syncthreads();
        for (int i = threadIdx.x; i < d.fixes; i += BLOCK) fv[gptr(d.fix)[2 * i]] = fv[gptr(d.fix)[2 * i + 1]];
    }
    // ReCalcIllum's residual over the direction's final entries (a separate
    // streaming pass measured faster than terms accumulated during the sweep).
    if (!ok) return;
    __syncthreads();
    double loc = -1;
    // one cell's four entries per thread as 16-byte loads (both arrays are
    // 16-byte aligned, checked on the host; 8-byte loads measured 0.42 ms
    // slower): the max is independent of the order, so this changes no result
    const v2d* __restrict__ ok2 = reinterpret_cast<const v2d*>(ok);
    const v2d* fv2 = reinterpret_cast<const v2d*>(fv);
    for (int64_t c = threadIdx.x; c < n; c += BLOCK) {
        const v2d a0 = ok2[2 * c], a1 = ok2[2 * c + 1], b0 = fv2[2 * c], b1 = fv2[2 * c + 1];
        residual_term(a0.x, b0.x, loc);
        residual_term(a0.y, b0.y, loc);
        residual_term(a1.x, b1.x, loc);
        residual_term(a1.y, b1.y, loc);
    }
    double* red = ring;
    red[threadIdx.x] = loc;
    __syncthreads();
    for (int w = BLOCK / 2; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w && red[threadIdx.x + w] > red[threadIdx.x]) red[threadIdx.x] = red[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) norm[k] = red[0];
}

}  // namespace

// Threads for `faces` out faces per level: fewer threads than that add passes, more
// idle ones (twice as many measured the same at 6 to 32 cubes per edge). More
// directions than CUs: two workgroups of 512 share a CU and hide each other's waits.
int sweep_block(int64_t faces, int m, int cus) {
    const int cap = m > cus ? 512 : 1024;
    int b = 128;
    while (b < faces && b < cap) b *= 2;
    return b;
}

hipError_t launch_sweep(int cls, int block, const SweepDirDev* d_dirs, int m, int64_t n, const double* d_S, int64_t ld,
                        const double* d_old, double* d_new, double* d_norm, hipStream_t st) {
    if (m <= 0 || n <= 0) return hipSuccess;
#define RSH_SWEEP(C, B)                                                                                            \
    if (cls == C && block == B) {                                                                                  \
        hipLaunchKernelGGL((sweep_kernel<C, B>), dim3((unsigned)m), dim3(B), 0, st, d_dirs, n, d_S, ld, d_old, d_new, \
                           d_norm);                                                                                \
        return hipGetLastError();                                                                                  \
    }
#define RSH_SWEEP_CLASS(C) RSH_SWEEP(C, 128) RSH_SWEEP(C, 256) RSH_SWEEP(C, 512) RSH_SWEEP(C, 1024)
    RSH_SWEEP_CLASS(0) RSH_SWEEP_CLASS(1) RSH_SWEEP_CLASS(2) RSH_SWEEP_CLASS(3) RSH_SWEEP_CLASS(10)
#undef RSH_SWEEP_CLASS
#undef RSH_SWEEP
    return hipErrorInvalidValue;
}

}  // namespace rsh
