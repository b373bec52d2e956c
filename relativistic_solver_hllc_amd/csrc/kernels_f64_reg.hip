// FP64 scattering integral for few cells: S[k][c] = sum_j P[k][j] sum_f I[j][c][f]
// with both MFMA operands loaded straight into registers.
//
// What bounds the LDS-panel kernel (kernels_f64.hip) below some tens of
// thousands of cells is not work but the length of one workgroup's chain: it
// gives 128 cells to a workgroup, so that 381 cells x 327 directions run on 3 of
// 256 CUs, each going through ~40 chunks of load, barrier and LDS at about 0.6 us
// on top of the MFMAs. Here the unit of work is one wave: a 16-cell tile and R
// row blocks (16 R output directions), all of K. A wave loads its face values
// and its slice of the phase panel itself (from L2 for all but the first wave
// that wants them), D j-steps ahead in a register ring; there is no LDS and no
// barrier, so waves advance independently and every SIMD can hold some.
//
// R is chosen per call (route_f64). Small R spreads a small problem over more
// SIMDs and shortens the chain of MFMAs; large R re-reads the faces less often.
// Units are numbered row group fastest, so that the four waves of a workgroup
// mostly share one cell tile and its face values in L1.
//
// Measured (us, this kernel / LDS-panel kernel): 381 x 327: 9 / 107; 1,000 x 400:
// 14 / 168; 2,958 x 200: 12 / 51; 5,000 x 302: 26 / 107; 10,000 x 400: 81 / 169;
// 24,576 x 200: 49 / 54; 24,576 x 400: 196 / 176 (the route takes the other).
// Per output the products are added in the same order (j ascending, one
// accumulator), so the results are those of the LDS-panel kernel bit for bit.
#include <algorithm>
#include <type_traits>

#include "mfma_f64_core.hpp"

namespace rsh {

namespace {

template <int I, int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_for<I + 1, N>(f);
    }
}

constexpr int kRegWaves = 4;  // independent waves per workgroup

// j-steps in flight per wave: 8 cover an L2 round trip with the MFMAs of few
// row blocks; more row blocks need fewer steps for the same time, and leave
// registers for fewer (two waves per SIMD).
constexpr int reg_depth(int r) { return r <= 5 ? 8 : r <= 7 ? 6 : 4; }

template <int R, int FACES>
__global__ __launch_bounds__(64 * kRegWaves, 2) void mfma_f64_reg_kernel(const double* __restrict__ illum, int64_t n,
                                                                         int64_t ldx, int m,
                                                                         const double* __restrict__ panel, int steps2,
                                                                         double* __restrict__ out, int64_t ld, int rows,
                                                                         unsigned groups, unsigned units) {
    constexpr int D = reg_depth(R);  // even
    constexpr int DP = D / 2;        // step pairs
    const int lane = threadIdx.x & 63;
    const int jr = lane >> 4;
    const unsigned unit = blockIdx.x * kRegWaves + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (unit >= units) return;
    const unsigned grp = unit % groups;
    const int64_t cell = (int64_t)(unit / groups) * 16 + (lane & 15);
    // Lanes past the last cell read the last cell and store nothing.
    const gcdouble_p xp = as_global(illum) + (cell < n ? cell : n - 1) * FACES;
    const gcv2d_p pp = (gcv2d_p)as_global(panel) + (int64_t)grp * steps2 * R * 64 + lane;
    const int64_t row = ldx * FACES;

    v4d acc[R];
#pragma unroll
    for (int i = 0; i < R; i++) acc[i] = v4d{0.0, 0.0, 0.0, 0.0};
    v2d ar[DP][R];        // panel ring: slot, row block -> the pair's two steps
    double xr[D][FACES];  // face ring: slot and step of the pair
    // Loads past the last pair or direction re-read the last one, in bounds.
    auto load = [&](auto slot, int sp) {
        constexpr int sl = decltype(slot)::value;
        const int s2 = sp < steps2 ? sp : steps2 - 1;
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const int j = 8 * s2 + 4 * u + jr;
            const gcdouble_p p = xp + (int64_t)(j < m ? j : m - 1) * row;
            if constexpr (FACES == 4) {
                const v2d a = ((gcv2d_p)p)[0], b = ((gcv2d_p)p)[1];
                xr[2 * sl + u][0] = a.x;
                xr[2 * sl + u][1 % FACES] = a.y;
                xr[2 * sl + u][2 % FACES] = b.x;
                xr[2 * sl + u][3 % FACES] = b.y;
            } else {
                xr[2 * sl + u][0] = p[0];
            }
        }
#pragma unroll
        for (int i = 0; i < R; i++) ar[sl][i] = pp[((int64_t)s2 * R + i) * 64];
    };
    auto mul = [&](auto slot, int sp) {
        constexpr int sl = decltype(slot)::value;
#pragma unroll
        for (int u = 0; u < 2; u++) {
            double v = xr[2 * sl + u][0];
#pragma unroll
            for (int f = 1; f < FACES; f++) v += xr[2 * sl + u][f];
            const double b = 8 * sp + 4 * u + jr < m ? v : 0.0;  // a repeated direction adds nothing, NaN included
#pragma unroll
            for (int i = 0; i < R; i++)
                acc[i] = __builtin_amdgcn_mfma_f64_16x16x4f64(u ? ar[sl][i].y : ar[sl][i].x, b, acc[i], 0, 0, 0);
        }
    };
    static_for<0, DP>([&](auto d) { load(d, d.value); });
    int sp = 0;
    for (; sp + DP <= steps2; sp += DP)
        static_for<0, DP>([&](auto d) {
            mul(d, sp + d.value);
            load(d, sp + d.value + DP);
            __builtin_amdgcn_sched_barrier(0);  // keep the ring: no load moves up past the slot's last use
        });
    static_for<0, DP>([&](auto d) {
        if (sp + d.value < steps2) mul(d, sp + d.value);
    });
    if (cell >= n) return;
    const int row0 = (int)grp * R * 16 + jr;
    double* ob = out + (int64_t)row0 * ld + cell;
#pragma unroll
    for (int i = 0; i < R; i++) {
#pragma unroll
        for (int r = 0; r < 4; r++)
            if (row0 + 16 * i + 4 * r < rows) ob[(int64_t)(16 * i + 4 * r) * ld] = acc[i][r];
    }
}

}  // namespace

bool f64_reg_rows_supported(int r) { return (r >= 1 && r <= 8) || r == 10; }

F64Plan plan_f64_reg(int m, int rows, int r) {
    F64Plan pl{};
    const int nrb = (rows + 15) / 16;
    pl.rb_per_pass = r;
    pl.passes = (nrb + r - 1) / r;
    pl.rb_total = pl.passes * r;
    pl.steps = (m + 7) / 8 * 2;
    pl.paired = true;
    return pl;
}

hipError_t launch_mfma_f64_reg(const double* d_illum, int faces, int64_t n, int64_t ldx, int m, const double* d_panel,
                               const F64Plan& pl, int rows, double* d_out, int64_t ld, hipStream_t st) {
    if (n <= 0 || rows <= 0) return hipSuccess;
    const int64_t units = (n + 15) / 16 * pl.passes;
    if (ldx < n || !pl.paired || (faces != 1 && faces != 4) || units > int64_t(0x7fffffff)) return hipErrorInvalidValue;
    const dim3 grid((unsigned)((units + kRegWaves - 1) / kRegWaves)), block(64 * kRegWaves);
#define RSH_REG(R)                                                                                                  \
    case R:                                                                                                         \
        if (faces == 4)                                                                                             \
            hipLaunchKernelGGL((mfma_f64_reg_kernel<R, 4>), grid, block, 0, st, d_illum, n, ldx, m, d_panel,        \
                               pl.steps / 2, d_out, ld, rows, (unsigned)pl.passes, (unsigned)units);               \
        else                                                                                                        \
            hipLaunchKernelGGL((mfma_f64_reg_kernel<R, 1>), grid, block, 0, st, d_illum, n, ldx, m, d_panel,        \
                               pl.steps / 2, d_out, ld, rows, (unsigned)pl.passes, (unsigned)units);               \
        break;
    switch (pl.rb_per_pass) {
        RSH_REG(1) RSH_REG(2) RSH_REG(3) RSH_REG(4) RSH_REG(5) RSH_REG(6) RSH_REG(7) RSH_REG(8) RSH_REG(10)
        default:
            return hipErrorInvalidValue;
    }
#undef RSH_REG
    return hipGetLastError();
}

// Which kernel and split an evaluation runs with. Costs in cycles of the
// busiest CU, fitted to the measured times of 21 sizes (300 to 1.57 M cells, 64
// to 800 directions, both face counts, every candidate below):
//   LDS panel, p passes of RB row blocks, 8-wave (128-cell) or 4-wave (64-cell)
//     workgroups: u waves per SIMD do u RB MFMAs of 64 cycles per j-step, and
//     chunk staging costs ~670 cycles per j-step where few waves per SIMD cannot
//     hide it. A pass beyond the least number re-reads the faces: 15 % of their
//     HBM time (4.8 TB/s) where they fit the 256 MB memory-side cache, else 40 %.
//     More, shorter passes fill the last round of workgroups better: 24,576 x 302
//     106.6 us in one pass of 8-wave workgroups, 86.6 in two of 4-wave ones;
//     48,963 x 400 cell-level 341 -> 272 (five); 50,000 x 302 214 against 235.
//   register-fed, R row blocks per wave: w waves per SIMD do w R MFMAs per j-step;
//     the CU's L1 delivers 4 w waves' faces and panel at 64 B/cycle, three quarters
//     of it beside the MFMAs' time; the first loads and the ring cost ~130 cycles
//     per j-step.
//   The register-fed kernel is never faster than the memory, faces and results at 10
//     TB/s from the caches (256 MB) or 5.5 from HBM (us: 40,000 cells, 47 of 368 rows
//     98, LDS panel 89; 40,000 x 32 10.4 / 9.0). With one face and fewer than four row
//     blocks it is left out beyond 32,768 cells, where its loads of 128 bytes a row fall
//     behind (52,862 x 25 8.8 / 7.0, 149,946 x 6 6.8 / 6.0). Up to four row blocks of all
//     directions, four faces, the memory bounds the LDS panel too, and fuller rounds
//     give nothing: eight waves (235,653 x 32 51, four waves 54; x 40 85 / 89; x 64 137 /
//     148; but 34,167 cells, 58 of 294 rows 74 / 68, 143,340 x 113 157 / 146).
F64Route route_f64(int m, int rows, int faces, int64_t n, int cus) {
    F64Route best{plan_f64(m, rows), 8, 2};
    const int nrb = (rows + 15) / 16;
    const double steps = (m + 3) / 4;
    const double face_bytes = 8.0 * faces * m * (double)n, bytes = face_bytes + 8.0 * rows * (double)n;
    const double memory = bytes / (bytes < 268e6 ? 10e12 : 5.5e12) * 2.4e9;
    const bool few_rows = nrb <= 4 && faces == 4 && 2 * rows > m;
    auto rounds = [&](int64_t wgs) { return (double)((wgs + cus - 1) / cus); };
    const int p0 = best.plan.passes;
    double cost = 0.0;
    for (int p = p0; p <= p0 + 4 && p <= nrb; p++) {
        const F64Plan pl = plan_f64(m, rows, (nrb + p - 1) / p);
        if (pl.passes != p) continue;
        const double again = (p - p0) * face_bytes * (face_bytes < 256e6 ? 0.15 : 0.4) / 4.8e12 * 2.4e9;
        for (int waves : {8, 4}) {
            if (waves == 4 && pl.rb_per_pass > kF64FourWaveMaxRb) continue;
            const double u = waves / 4 * rounds((n + 16 * waves - 1) / (16 * waves) * p);
            const double c = std::max(steps * (u * pl.rb_per_pass * 64 + 670), few_rows ? memory : 0.0) + again;
            // the first candidate unless another is clearly better
            if (cost == 0.0 || c < 0.97 * cost) {
                cost = c;
                best = F64Route{pl, waves, 2};
            }
        }
    }
    // never cheaper: every wave re-reads the faces and the panel
    if (n > (int64_t(1) << (faces == 1 && nrb < 4 ? 15 : 18))) return best;
    // 32-bit counts: at most 2^14 tiles, and nrb row groups
    const unsigned tiles = (unsigned)((n + 15) / 16), rb = (unsigned)nrb;
    double reg = 0.0;
    for (unsigned r = 1; r <= 10; r++) {
        if (!f64_reg_rows_supported((int)r)) continue;
        const unsigned units = tiles * ((rb + r - 1) / r);
        const double w = (units + kRegWaves * cus - 1) / (kRegWaves * cus);
        const double c = steps * (w * r * 64 + 0.75 * w * kRegWaves * (512.0 * faces + 512.0 * r) / 64 + 130);
        if (std::max(c, memory) < cost && (reg == 0.0 || c < reg)) {
            reg = c;
            best = F64Route{plan_f64_reg(m, rows, (int)r), 0, 0};
        }
        if (r >= rb) break;  // more row blocks per wave than there are
    }
    return best;
}

}  // namespace rsh
