// Resident-panel split kernels: plans, launchers and dispatch (the kernels are in
// split_single_res.hpp and split_iter_res.hpp).
#include "split_iter_res.hpp"
#include "split_single_res.hpp"

namespace rsh {

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
        rbw = single_res_rbw(steps, rb_need);
        if (rbw < 1) return false;
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

// Workgroup form of the single-problem kernel. Rounds = chunks of a form per set.
// 8 waves x 1 tile (128 cells) up to one round, three for three parts; beyond, two
// parts take 8 x 2, and 4 x 4 for FP64 results from four rounds on; three parts
// 4 x 4. us with 4 x 4 / 8 x 2 / 8 x 1 (cells x directions):
//   two parts 5000 x 400 20.4 / - / 13.4; 10,000 x 400 22.0 / 17.0 / -; 20,000 x 400 36.6 / 28.2 / -;
//     FP64 80,000 x 400 119 / 125, 100,000 x 500 195 / 204, 1,572,864 x 400 2000 / 2058 (FP32 80,000 x 400 103 / 99)
//   three parts 5000 x 302 23.8 / - / 14.2; 20,000 x 302 41 / 33 / 31; 413,519 x 302 454 / 517 / -
static void single_res_form(int nt, int64_t n, int sets, int out_f32, int* waves, int* tiles) {
    const int64_t slots = (int64_t)kXcds * sets;
    *waves = 8;
    *tiles = 1;
    if (n <= (nt == 2 ? 1 : 3) * 128 * slots) return;
    *tiles = 2;
    if (nt == 2 && (out_f32 || n < 4 * 256 * slots)) return;
    *waves = 4;
    *tiles = 4;
}

// Whether results are stored past the caches: FP64 where every 16 cells of a row fill
// whole 128-byte lines; a line stored in pieces has to meet in L2 (302 directions, three
// parts, us non-temporal / plain: 413,519 cells, odd rows, FP32 718 / 560, FP64 868 / 616;
// 393,216 cells FP32 458 / 422, FP64 490 / 500). And both kinds, pieces or not, where many
// row groups re-read a state that fits the 256 MB cache and plain results would push it
// out (long slices, 43,477 cells, us non-temporal / plain: 854 directions two parts 370 /
// 450, FP32 338 / 409, three parts 502 / 655; 80,001 x 640 two parts 288 / 328; but three
// parts, whose state does not fit, 501 / 440, and 20,001 x 854, all of which fits, 176 / 140).
static bool single_res_nontemporal(int nt, int64_t n, int steps, int rows, const void* out, int64_t ld, int out_f32) {
    if (!out_f32 && ld % 16 == 0 && reinterpret_cast<uintptr_t>(out) % 128 == 0) return true;
    const double state = 64.0 * nt * steps * (double)n, res = (out_f32 ? 4.0 : 8.0) * rows * (double)n, cache = 268e6;
    return steps >= kResLongSteps && state <= cache && state + res > cache;
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
    int waves, per_wave;
    single_res_form(nt, n, sets, out_f32, &waves, &per_wave);
    const int64_t chunks = (tiles + waves * per_wave - 1) / (waves * per_wave);
    const SingleResArgs a{pl.rb_per_pass, pl.steps, waves, per_wave, kXcds * sets * pl.passes, lds_bytes, st,
                          static_cast<const v4u*>(d_state), n, d_cell_inv, static_cast<const v4u*>(d_panel), d_row_inv,
                          d_out, ld, rows, out_f32,
                          single_res_nontemporal(nt, n, pl.steps, rows, d_out, ld, out_f32) ? 1 : 0, pl.passes, sets, chunks};
    if (per_wave > 1 && pl.steps <= kSingleResMaxSteps) {
        hipError_t e = hipErrorNotFound;
        switch (form) {
            case RSH_FORM_BF16X2: e = pl.steps <= 14 ? single_res_range<0, 2, 1, 14>(a) : single_res_range<0, 2, 15, 25>(a); break;
            case RSH_FORM_FP16X2: e = pl.steps <= 14 ? single_res_range<1, 2, 1, 14>(a) : single_res_range<1, 2, 15, 25>(a); break;
            default: e = pl.steps <= 14 ? single_res_range<0, 3, 1, 14>(a) : single_res_range<0, 3, 15, 25>(a); break;
        }
        if (e != hipErrorNotFound) return e;
    }
#define RSH_RES(RBW, FMT, NT) \
    return per_wave == 1 ? launch_res<RBW, FMT, NT, 0, 8, 1>(a) : launch_res<RBW, FMT, NT, 0, 4, 4>(a);
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
}

// Grouped iteration, resident-panel form: the plans of up to kIterResMaxSteps
// K-steps (split_iter_res.hpp). rb = RBW of the class, steps its K-steps.
bool iter_split_res_supported(int form, int rb, int steps) {
    const int nt = split_terms(form);
    if (steps < 1 || steps > kIterResMaxSteps) return false;
    return rb == iter_res_rbw(nt, steps, 2 * steps - 1) || rb == iter_res_rbw(nt, steps, 2 * steps);
}

// Plans that a caller may ask for by name (rsh_batch_set_split_kernel) and that
// have a four-wave form: M = 193 to 224, 385 to 416, 769 to 800, which were the only
// ones when the names were given. The others are taken by the automatic choice (and
// by the tuner's eight-wave candidate) only.
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
