// Radiation moments of the face intensities: energy, flux ("stream"), pressure
// tensor ("impuls") and the divergences of flux and pressure tensor, per cell,
// over all M directions. Replaces d_MakeIllumParam (cuda/cuda_kernel.cu:113-226)
// and its helpers IntegarteDirection / IntegarteDirection3Faces /
// IntegarteDirection9Faces (cuda/cuda_utils.cu:18-167).
//
// Every moment is a weighted sum over directions of one face intensity:
//   T_f[q] = sum_j psi[j][q] I[j][c][f],  psi[j][q] = phi_q(omega_j) w_j / F,
//   phi = (1, x, y, z, xx, xy, xz, yy, yz, zz)
// (ten functions: the pressure tensor is symmetric). That is a [10 x M] x
// [M x 4N] product with M = 400 against 4N = 6.3 M columns: 2.5 flop per byte
// of the intensity, so the kernel is HBM-bound (the intensity is read exactly
// once, 32 M bytes per cell) and runs on the FP64 VALU: psi is uniform across
// the wave and comes in through scalar loads as the SGPR operand of each
// v_fma_f64, the intensity is the vector operand, loaded with 16-byte loads.
//
// Thread mapping: FPT consecutive faces of one cell per thread (TPC = FACES /
// FPT threads per cell, adjacent lanes). The cell's face terms are combined
// with lane shuffles, then the first lane of the cell writes
//   energy    = (sum_f T_f[0]) / FACES
//   stream[k] = (sum_f T_f[1+k]) / FACES
//   impuls    = (sum_f T_f[4..9]) / FACES, expanded to 3x3 row-major
//   divstream = (sum_f (T_f[1..3] . n_f) area_f) / volume
//   divimpuls[h] = (sum_f (T_f[h,:] . n_f) area_f) / volume
// with the reference's layouts: normals[c][f][3], areas[c][f], volume[c].
#include "rsh_internal.hpp"

namespace rsh {

typedef double v2d_m __attribute__((ext_vector_type(2)));

// 128-thread workgroups and four rows in flight per thread: 72-74 % of the
// 8 TB/s HBM peak at 1.57 M cells x 400 directions (a pure streaming read of
// the same bytes: 88 %). Blocks of 64-1024 threads with 2-16 rows in flight
// measured 69-79 %, with the same configuration differing by up to 10 % from
// one process to the next, so none is reliably faster.
constexpr int kMomentBlock = 128;
constexpr int kMomentPipe = 4;

// Non-temporal loads: every face value is read exactly once, so it should not
// displace anything in the caches (plain loads measured 4-6 % slower).
template <int FPT>
__device__ inline void load_faces(const double* __restrict__ p, double (&v)[FPT]) {
    if constexpr (FPT == 4) {
        const v2d_m a = __builtin_nontemporal_load(reinterpret_cast<const v2d_m*>(p));
        const v2d_m b = __builtin_nontemporal_load(reinterpret_cast<const v2d_m*>(p + 2));
        v[0] = a.x; v[1] = a.y; v[2] = b.x; v[3] = b.y;
    } else if constexpr (FPT == 2) {
        const v2d_m a = __builtin_nontemporal_load(reinterpret_cast<const v2d_m*>(p));
        v[0] = a.x; v[1] = a.y;
    } else {
        v[0] = __builtin_nontemporal_load(p);
    }
}

template <int FPT>
__device__ inline void accumulate(const double* __restrict__ ps, const double (&v)[FPT],
                                  double (&acc)[FPT][kMomentFuncs]) {
#pragma unroll
    for (int q = 0; q < kMomentFuncs; q++) {
        const double w = ps[q];
#pragma unroll
        for (int f = 0; f < FPT; f++) acc[f][q] = __builtin_fma(w, v[f], acc[f][q]);
    }
}

template <int TPC>
__device__ inline double cell_sum(double x) {
#pragma unroll
    for (int off = 1; off < TPC; off <<= 1) x += __shfl_xor(x, off, 64);
    return x;
}

// Sums over the direction rows j0 .. j1 - 1 (at least one) of a thread's faces.
template <int FPT, int PIPE>
__device__ inline void sum_rows(const double* __restrict__ src, int64_t stride, int j0, int j1,
                                const double* __restrict__ psi, double (&acc)[FPT][kMomentFuncs]) {
#pragma unroll
    for (int f = 0; f < FPT; f++)
#pragma unroll
        for (int q = 0; q < kMomentFuncs; q++) acc[f][q] = 0.0;

    // Ring of PIPE direction rows in flight: row j + PIPE is requested while
    // row j is consumed (indices past the end re-read the last row, in bounds).
    double ring[PIPE][FPT];
#pragma unroll
    for (int u = 0; u < PIPE; u++) load_faces<FPT>(src + (int64_t)(j0 + u < j1 ? j0 + u : j1 - 1) * stride, ring[u]);
    // one pointer for the block's weights: with an index from j0 the compiler loaded row
    // after row, each with a wait of its own (132,030 cells x 115, one face 25.0 us for 24.1)
    const double* __restrict__ pj = psi + j0 * kMomentFuncs;
    int j = j0;
    for (; j + PIPE <= j1; j += PIPE, pj += PIPE * kMomentFuncs) {
#pragma unroll
        for (int u = 0; u < PIPE; u++) {
            double v[FPT];
#pragma unroll
            for (int f = 0; f < FPT; f++) v[f] = ring[u][f];
            const int jn = j + u + PIPE;
            load_faces<FPT>(src + (int64_t)(jn < j1 ? jn : j1 - 1) * stride, ring[u]);
            accumulate<FPT>(pj + u * kMomentFuncs, v, acc);
        }
    }
#pragma unroll
    for (int u = 0; u < PIPE; u++)
        if (j + u < j1) accumulate<FPT>(pj + u * kMomentFuncs, ring[u], acc);
}

// Sums of one cell: energy, flux, pressure tensor and the two divergences, each
// before its factor. The thread's FPT faces, then all lanes of the cell.
constexpr int kCellSums = 14;
template <int FACES, int FPT>
__device__ inline void cell_sums(const double (&acc)[FPT][kMomentFuncs], int64_t c, int fg, bool want_div,
                                 const double* __restrict__ normals, const double* __restrict__ areas,
                                 double (&x)[kCellSums]) {
    constexpr int TPC = FACES / FPT;
#pragma unroll
    for (int q = 0; q < kCellSums; q++) x[q] = 0.0;
#pragma unroll
    for (int f = 0; f < FPT; f++) {
        const double* a = acc[f];
#pragma unroll
        for (int q = 0; q < kMomentFuncs; q++) x[q] += a[q];
        if (want_div) {
            const int64_t cf = c * FACES + fg * FPT + f;
            const double nx = normals[3 * cf], ny = normals[3 * cf + 1], nz = normals[3 * cf + 2];
            const double ar = areas[cf];
            x[10] += (a[1] * nx + a[2] * ny + a[3] * nz) * ar;
            x[11] += (a[4] * nx + a[5] * ny + a[6] * nz) * ar;
            x[12] += (a[5] * nx + a[7] * ny + a[8] * nz) * ar;
            x[13] += (a[6] * nx + a[8] * ny + a[9] * nz) * ar;
        }
    }
    if constexpr (TPC > 1) {
#pragma unroll
        for (int q = 0; q < 10; q++) x[q] = cell_sum<TPC>(x[q]);
        if (want_div) {
#pragma unroll
            for (int q = 10; q < kCellSums; q++) x[q] = cell_sum<TPC>(x[q]);
        }
    }
}

struct MomentOut {
    double *energy, *stream, *impuls, *divstream, *divimpuls;
};

// Stores what one cell sum contributes to: q as in cell_sums.
template <int FACES>
__device__ inline void store_sum(const MomentOut& o, int64_t cell, int q, double x, double vol) {
    constexpr double inv_faces = 1.0 / FACES;  // FACES is 1 or 4: exact
    if (q == 0) {
        if (o.energy) o.energy[cell] = x * inv_faces;
    } else if (q < 4) {
        if (o.stream) o.stream[3 * cell + q - 1] = x * inv_faces;
    } else if (q < 10) {
        if (!o.impuls) return;
        // row-major 3x3 of the symmetric tensor (xx xy xz / xy yy yz / xz yz zz)
        const int r = q < 7 ? 0 : q < 9 ? 1 : 2, k = q < 7 ? q - 4 : q < 9 ? q - 6 : 2;
        o.impuls[9 * cell + 3 * r + k] = x * inv_faces;
        if (r != k) o.impuls[9 * cell + 3 * k + r] = x * inv_faces;
    } else if (q == 10) {
        if (o.divstream) o.divstream[cell] = x / vol;
    } else if (o.divimpuls) {
        o.divimpuls[3 * cell + q - 11] = x / vol;
    }
}

template <int FACES, int FPT, int PIPE>
__global__ __launch_bounds__(kMomentBlock) void moments_f64_kernel(
    const double* __restrict__ illum, int64_t n, int m, const double* __restrict__ psi,
    const double* __restrict__ normals, const double* __restrict__ areas, const double* __restrict__ volume,
    MomentOut out) {
    constexpr int TPC = FACES / FPT;
    const int64_t gid = (int64_t)blockIdx.x * kMomentBlock + threadIdx.x;
    const int64_t cell = gid / TPC;
    const int fg = (int)(gid % TPC);
    const bool active = cell < n;
    // Lanes past the last cell read the last cell (in bounds) and write nothing,
    // so every lane of a cell group takes part in the shuffles.
    const int64_t c = active ? cell : n - 1;
    double acc[FPT][kMomentFuncs], x[kCellSums];
    sum_rows<FPT, PIPE>(illum + c * FACES + fg * FPT, n * FACES, 0, m, psi, acc);
    const bool want_div = out.divstream || out.divimpuls;
    cell_sums<FACES, FPT>(acc, c, fg, want_div, normals, areas, x);
    if (!active || fg != 0) return;
    const double vol = want_div ? volume[cell] : 1.0;
#pragma unroll
    for (int q = 0; q < kCellSums; q++) store_sum<FACES>(out, cell, q, x[q], vol);
}

// Few cells: the directions are split over the SLICES waves of a workgroup, which
// all take the same 64 threads' faces; the slices' cell sums are added in order
// through LDS, one thread per sum. What bounds the plain kernel there is one
// thread's chain of rows (four in flight, ~0.5 us per round trip). us per call with
// 1 / 2 / 4 / 8 / 16 slices (cells x directions, two faces per thread):
//     528 x 294: 36.4 / 18.0 / 10.5 / 8.4 / 8.0    1733 x 265: 46.1 / 20.8 / 12.4 / 8.7 / 9.0
//    3762 x 73:  14.7 /  8.4 /  6.0 / 5.4 / 6.0    9000 x 400: 69.0 / 37.6 / 23.0 / 25.2 / 27.5
//   17170 x 294: 55.2 / 32.1 / 31.2 / 33.7 / 37.3  36000 x 200: 43.9 / 38.6 / 40.2 / 42.4 / 51.6
//   48000 x 200: 49.1 / 50.1 / 52.8 / 53.7 / 65.6  65536 x 200: 65.7 / 76.2 / 80.1 / 84.3 / 93.8
// Eight rows in flight instead of four: within 10 % either way.
template <int FACES, int FPT, int PIPE, int SLICES>
__global__ __launch_bounds__(64 * SLICES) void moments_f64_sliced_kernel(
    const double* __restrict__ illum, int64_t n, int m, const double* __restrict__ psi,
    const double* __restrict__ normals, const double* __restrict__ areas, const double* __restrict__ volume,
    MomentOut out) {
    constexpr int TPC = FACES / FPT, CELLS = 64 / TPC;
    __shared__ double part[SLICES][kCellSums][CELLS];
    const int lane = threadIdx.x & 63, slice = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t first = (int64_t)blockIdx.x * CELLS;
    const int fg = lane % TPC, cl = lane / TPC;
    const int64_t c = first + cl < n ? first + cl : n - 1;
    const bool want_div = out.divstream || out.divimpuls;
    // the host gives every slice at least one row: m >= SLICES
    const int j0 = (int)((int64_t)m * slice / SLICES), j1 = (int)((int64_t)m * (slice + 1) / SLICES);
    double acc[FPT][kMomentFuncs], x[kCellSums];
    sum_rows<FPT, PIPE>(illum + c * FACES + fg * FPT, n * FACES, j0, j1, psi, acc);
    cell_sums<FACES, FPT>(acc, c, fg, want_div, normals, areas, x);
    if (fg == 0) {
#pragma unroll
        for (int q = 0; q < kCellSums; q++) part[slice][q][cl] = x[q];
    }
    __syncthreads();
    for (int i = threadIdx.x; i < kCellSums * CELLS; i += 64 * SLICES) {
        const int q = i / CELLS;
        const int64_t cell = first + i % CELLS;
        if (cell >= n || (q >= 10 && !want_div)) continue;
        double sum = 0.0;
#pragma unroll
        for (int w = 0; w < SLICES; w++) sum += part[w][q][i % CELLS];
        store_sum<FACES>(out, cell, q, sum, q >= 10 ? volume[cell] : 1.0);
    }
}

// Slices of the directions: doubled while the chip has fewer than five waves per CU
// (1280) and a slice keeps at least eight rows, by the times above.
static int moment_slices(int64_t threads, int m) {
    const int64_t waves = (threads + 63) / 64;
    int s = 1;
    while (s < 16 && waves * s < 1280 && m >= 16 * s) s *= 2;
    return s;
}

hipError_t launch_moments_f64(const double* d_illum, int faces, int64_t n, int m, const double* d_psi,
                              const double* d_normals, const double* d_areas, const double* d_volume,
                              double* d_energy, double* d_stream, double* d_impuls, double* d_divstream,
                              double* d_divimpuls, int faces_per_thread, hipStream_t st) {
    if (n <= 0) return hipSuccess;
    const int fpt = faces == 1 ? 1 : faces_per_thread;
    const int64_t threads = n * (faces / fpt);
    const dim3 grid((unsigned)((threads + kMomentBlock - 1) / kMomentBlock)), block(kMomentBlock);
    const MomentOut out{d_energy, d_stream, d_impuls, d_divstream, d_divimpuls};
    const int slices = moment_slices(threads, m);
#define RSH_MOM_SLICED(FA, FP, S)                                                                                  \
    if (slices == S) {                                                                                             \
        hipLaunchKernelGGL((moments_f64_sliced_kernel<FA, FP, kMomentPipe, S>), dim3((unsigned)((threads + 63) / 64)), \
                           dim3(64 * S), 0, st, d_illum, n, m, d_psi, d_normals, d_areas, d_volume, out);          \
        return hipGetLastError();                                                                                  \
    }
#define RSH_MOM(FA, FP)                                                                                           \
    if (faces == FA && fpt == FP) {                                                                               \
        RSH_MOM_SLICED(FA, FP, 2)                                                                                 \
        RSH_MOM_SLICED(FA, FP, 4)                                                                                 \
        RSH_MOM_SLICED(FA, FP, 8)                                                                                 \
        RSH_MOM_SLICED(FA, FP, 16)                                                                                \
        hipLaunchKernelGGL((moments_f64_kernel<FA, FP, kMomentPipe>), grid, block, 0, st, d_illum, n, m, d_psi,  \
                           d_normals, d_areas, d_volume, out);                                                    \
        return hipGetLastError();                                                                                 \
    }
    RSH_MOM(1, 1)
    RSH_MOM(4, 4)
    RSH_MOM(4, 2)
    RSH_MOM(4, 1)
#undef RSH_MOM
#undef RSH_MOM_SLICED
    return hipErrorInvalidValue;
}

}  // namespace rsh
