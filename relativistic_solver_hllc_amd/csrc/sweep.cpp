// Host side of the transport sweep: validates the reference-format sweep
// structures of each direction (sorted_id_cell, face states, vec_x0 records),
// plans the passes of the direction, uploads everything once and launches the
// sweep kernel. Replaces ReadIllumGeometry's in-memory result
// (file_module/reader_bin.cpp:164-203) and the direction loop of
// MPI_CalculateIllumAsync (solve_module/illum/Illum_async.cpp:725-784).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <memory>
#include <mutex>
#include <string>
#include <vector>

#include "rsh_objects.hpp"
#include "rsh_scatter.h"

using namespace rsh;

struct rsh_sweep_s {
    int device = 0;
    int64_t n = 0;
    int m = 0;
    int block = 0;  // threads per direction, out faces per pass at most; from the first direction set
    // class 0's source test per cell, bit 3 f + j for node j of face f (|x -
    // (0.5, 0, 0)| < 0.05, GetCurIllum's expression); empty without nodes
    std::vector<uint16_t> node_in_source;
    std::vector<int32_t> pairs;  // host copy: validation, plans
    struct Dir {
        void* block = nullptr;  // one device allocation per direction
        SweepDirDev dev{};
        bool set = false;
    };
    std::vector<Dir> dirs;
    // Host arrays of one direction's plan, kept for the next one (a call takes a
    // set of its own: fresh pages would cost more than half of the planning) until
    // every direction is set; at most kSpare sets of about 125 bytes per cell.
    static constexpr size_t kSpare = 8;
    struct Cell {
        int32_t link;   // place in the given order; then, ready: the next cell of its list, taken: its first out face's position
        int32_t chain;  // cells in the longest chain before it; then in the longest one that still waits on it
        int32_t out0;   // out faces of the cells before it in the given order (three records each)
        uint8_t waits;  // cells it reads that are not taken yet
        uint8_t outs;   // bit f: face f is an out face
    };
    struct Work {
        std::vector<Cell> info;
        std::vector<int32_t> cells, pass, touched, old, open, fix;
        std::vector<uint64_t> marks, words;
        std::unique_ptr<char[]> image;  // what is uploaded
        size_t room = 0;
    };
    std::vector<std::unique_ptr<Work>> spare;  // capacity kSpare
    int unset = 0;  // directions not set
    SweepDirDev* d_table = nullptr;
    bool table_dirty = true;
    std::mutex mu;
};

namespace {

bool valid_bound(int32_t t) { return t >= RSH_BOUND_INNER_SOURCE && t <= RSH_BOUND_FREE; }

size_t align256(size_t b) { return (b + 255) & ~size_t(255); }

}  // namespace

extern "C" {

int rsh_sweep_create(int32_t device, int64_t n_cells, int32_t n_dirs, const int32_t* pairs, const double* nodes,
                     rsh_sweep* out) {
    if (!out || !pairs || n_cells <= 0 || n_dirs <= 0 || n_cells > INT32_MAX / 4)
        return fail(RSH_E_ARG, "invalid sweep size or null pointer");
    for (int64_t i = 0; i < n_cells * 4; i++) {
        const int32_t p = pairs[i];
        if (p >= 0 ? (p >= n_cells * 4 || p / 4 == i / 4 || pairs[p] != i) : !valid_bound(p))
            return fail(RSH_E_ARG, "pairs: entry " + std::to_string(i) +
                                       " is neither a symmetric neighbour face nor a boundary type -1..-4");
    }
    auto* s = new rsh_sweep_s();
    s->device = device;
    s->n = n_cells;
    s->m = n_dirs;
    s->pairs.assign(pairs, pairs + n_cells * 4);
    s->dirs.resize((size_t)n_dirs);
    s->unset = n_dirs;
    s->spare.reserve(rsh_sweep_s::kSpare);
    auto cleanup = [&](int rc) {
        rsh_sweep_destroy(s);
        return rc;
    };
    hipError_t e = hipSetDevice(device);
    if (e != hipSuccess) return cleanup(hip_fail(e, "hipSetDevice"));
    e = hipMalloc(&s->d_table, (size_t)n_dirs * sizeof(SweepDirDev));
    if (e != hipSuccess) return cleanup(hip_fail(e, "sweep: device allocation"));
    if (nodes) {
        s->node_in_source.assign((size_t)n_cells, 0);
        for (int64_t c = 0; c < n_cells; c++)
            for (int b = 0; b < 12; b++) {
                const double* x = nodes + (c * 12 + b) * 3;
                const double dx = x[0] - 0.5, dy = x[1] - 0.0, dz = x[2] - 0.0;
                if (std::sqrt(dx * dx + dy * dy + dz * dz) < 0.05) s->node_in_source[(size_t)c] |= (uint16_t)(1u << b);
            }
    }
    *out = s;
    return RSH_OK;
}

int rsh_sweep_destroy(rsh_sweep s) {
    if (!s) return RSH_OK;
    (void)hipSetDevice(s->device);
    for (auto& d : s->dirs)
        if (d.block) (void)hipFree(d.block);
    if (s->d_table) (void)hipFree(s->d_table);
    delete s;
    return RSH_OK;
}

int rsh_sweep_set_direction(rsh_sweep s, int32_t k, const int32_t* order, const int32_t* face_state,
                            const double* x0_s, const uint8_t* x0_face, int64_t n_records) {
    if (!s || k < 0 || k >= s->m || !order || !face_state || n_records < 0 || (n_records > 0 && (!x0_s || !x0_face)))
        return fail(RSH_E_ARG, "invalid direction, null pointer or record count");
    const int64_t n = s->n;
    const int32_t* pairs = s->pairs.data();
    struct Lease {  // a Work of this call, given back at its end (freed with the others once every direction is set)
        rsh_sweep s;
        std::unique_ptr<rsh_sweep_s::Work> w;
        explicit Lease(rsh_sweep sw) : s(sw) {
            std::lock_guard<std::mutex> lock(s->mu);
            if (!s->spare.empty()) {
                w = std::move(s->spare.back());
                s->spare.pop_back();
            }
            if (!w) w = std::make_unique<rsh_sweep_s::Work>();
        }
        ~Lease() {
            std::lock_guard<std::mutex> lock(s->mu);
            if (s->unset == 0) s->spare.clear();
            else if (s->spare.size() < rsh_sweep_s::kSpare) s->spare.push_back(std::move(w));
        }
    } lease(s);
    rsh_sweep_s::Work& w = *lease.w;
    // The loops below go through the cells in an order that is random in memory, over
    // arrays larger than L2: each fetches what the cells kAhead and 2 kAhead steps on
    // need (a third of the planning's time).
    constexpr int kAhead = 12;
    const auto cell_of = [](int32_t e) { return std::max(e, 0) >> 2; };
    auto& info = w.info;
    info.resize((size_t)n);
    int bad = 0;
    for (int64_t c = 0; c < n; c++) {
        bad |= face_state[c] & ~15;
        info[(size_t)c] = {-1, 0, 0, 0, (uint8_t)(~face_state[c] & 15)};
    }
    for (int64_t h = 0; h < n; h++) {
        const int32_t c = order[h];
        if (c < 0 || c >= n || info[(size_t)c].link >= 0) return fail(RSH_E_ARG, "order is not a permutation of the cells");
        info[(size_t)c].link = (int32_t)h;
    }
    if (bad) return fail(RSH_E_ARG, "face state outside 0..15");
    auto& fix = w.fix;
    fix.clear();
    int64_t r = 0;
    int32_t levels = 0;
    for (int64_t h = 0; h < n; h++) {
        const int32_t c = order[h];
        if (h + 2 * kAhead < n) {
            const int32_t a = order[h + 2 * kAhead], b = order[h + kAhead];
            __builtin_prefetch(pairs + 4 * (int64_t)a);
            __builtin_prefetch(&info[(size_t)a], 1);
            for (int f = 0; f < 4; f++) __builtin_prefetch(&info[(size_t)cell_of(pairs[b * 4 + f])]);
        }
        auto& I = info[(size_t)c];
        I.out0 = (int32_t)(r / 3);
        for (int f = 0; f < 4; f++) {
            const int32_t p = pairs[c * 4 + f];
            const bool in = !((I.outs >> f) & 1);
            if (!in) {
                for (int j = 0; j < 3; j++, r++) {
                    if (r >= n_records) return fail(RSH_E_ARG, "fewer x0 records than out-face nodes");
                    const int g = x0_face[r];
                    if (g > 3 || ((I.outs >> g) & 1))
                        return fail(RSH_E_ARG, "x0 record " + std::to_string(r) + " does not name an in face");
                }
            }
            if (p < 0) continue;
            const int32_t u = p / 4;
            const auto& U = info[(size_t)u];
            // Reads across an in face, and a face both cells treat as out
            // (written by both: the later one in the order wins), order u first.
            const bool both_out = !in && ((U.outs >> (p % 4)) & 1) && U.link < h;
            if (!in && !both_out) continue;
            if (both_out) fix.insert(fix.end(), {p, c * 4 + f});  // the later cell in the given order wins
            if (U.link > h)
                return fail(RSH_E_ARG, "order is not upwind: cell " + std::to_string(c) + " reads cell " +
                                           std::to_string(u) + " that comes later");
            I.chain = std::max(I.chain, U.chain + 1);
        }
        levels = std::max(levels, I.chain + 1);
    }
    if (r != n_records) return fail(RSH_E_ARG, "more x0 records than out-face nodes");
    // What a cell waits for, and the longest chain of cells behind it.
    for (auto& I : info) I.chain = 0;
    for (int64_t h = n - 1; h >= 0; h--) {
        const int32_t c = order[h];
        if (h >= 2 * kAhead) {
            const int32_t a = order[h - 2 * kAhead], b = order[h - kAhead];
            __builtin_prefetch(pairs + 4 * (int64_t)a);
            __builtin_prefetch(&info[(size_t)a], 1);
            for (int f = 0; f < 4; f++) __builtin_prefetch(&info[(size_t)cell_of(pairs[b * 4 + f])], 1);
        }
        auto& I = info[(size_t)c];
        for (int f = 0; f < 4; f++) {
            const int32_t q = pairs[c * 4 + f];
            if (((I.outs >> f) & 1) || q < 0) continue;
            I.waits++;
            int32_t& chain = info[(size_t)(q / 4)].chain;
            chain = std::max(chain, I.chain + 1);
        }
    }
    int block;
    {
        std::lock_guard<std::mutex> lock(s->mu);
        if (!s->block) s->block = sweep_block(n_records / 3 / levels, s->m, device_cus(s->device));
        block = s->block;
    }
    // Passes of at most block out faces and block / 2 cells whose upstream cells are in
    // earlier passes. Taken first: cells of a group of kLineCells that an earlier
    // pass touched, oldest group first (a 128-byte line of S, four of the result,
    // is finished while it is in L2); then the cell with the longest chain behind
    // it (fewest passes). Out faces have positions pass by pass, by cell and face.
    constexpr int32_t kLineCells = 16;
    const auto bits = [](unsigned x) { return (int32_t)(0x4332322132212110ull >> (4 * x) & 15); };  // of four: one digit each
    auto &cells = w.cells, &pass = w.pass;
    cells.clear();
    cells.reserve((size_t)n + 1);
    pass.clear();
    {
        // ready cells as lists: by the pass that touched their group, by their chain
        auto &touched = w.touched, &old = w.old, &open = w.open;
        touched.assign((size_t)(n / kLineCells + 1), -1);
        old.clear();
        open.assign((size_t)levels, -1);
        int32_t oldest = 0, longest = -1;
        auto push = [&](int32_t c) {
            const int32_t t = touched[(size_t)(c / kLineCells)], l = info[(size_t)c].chain;
            int32_t& head = t >= 0 ? old[(size_t)t] : open[(size_t)l];
            if (t >= 0) oldest = std::min(oldest, t);
            else longest = std::max(longest, l);
            info[(size_t)c].link = head;
            head = c;
        };
        auto top = [&]() -> int32_t* {
            while (oldest < (int32_t)old.size() && old[(size_t)oldest] < 0) oldest++;
            if (oldest < (int32_t)old.size()) return &old[(size_t)oldest];
            while (longest >= 0 && open[(size_t)longest] < 0) longest--;
            return longest >= 0 ? &open[(size_t)longest] : nullptr;
        };
        // a pass's cells in ascending order: marked in a bit set with a summary bit per
        // word (sorting them took a third of the planning)
        auto &marks = w.marks, &words = w.words;
        marks.assign((size_t)(n / 64 + 1), 0);
        words.assign((size_t)(n / 4096 + 1), 0);
        auto in_order = [&](auto&& f) {
            for (size_t y = 0; y < words.size(); y++)
                for (; words[y]; words[y] &= words[y] - 1) {
                    const size_t x = y * 64 + (size_t)__builtin_ctzll(words[y]);
                    for (; marks[x]; marks[x] &= marks[x] - 1) f((int32_t)(x * 64 + (size_t)__builtin_ctzll(marks[x])));
                }
        };
        for (int32_t c = (int32_t)n - 1; c >= 0; c--)
            if (!info[(size_t)c].waits) push(c);
        int32_t positions = 0;  // out faces so far
        for (int32_t p = 0; top(); p++) {
            const int32_t first = (int32_t)cells.size(), face0 = positions;
            int32_t cnt = 0, taken = 0;
            old.push_back(-1);
            for (int32_t* head; taken < block / 2 && (head = top()); taken++) {
                const int32_t c = *head;
                const auto& I = info[(size_t)c];
                if ((cnt += bits(I.outs)) > block) break;
                *head = I.link;
                int32_t& t = touched[(size_t)(c / kLineCells)];
                if (t < 0) t = p;
                marks[(size_t)c >> 6] |= uint64_t(1) << (c & 63);
                words[(size_t)c >> 12] |= uint64_t(1) << ((c >> 6) & 63);
            }
            in_order([&](int32_t c) {
                auto& I = info[(size_t)c];
                cells.push_back(c);
                I.link = positions;
                positions += bits(I.outs);
                for (unsigned left = I.outs; left; left &= left - 1) {
                    const int32_t q = pairs[c * 4 + __builtin_ctz(left)];
                    if (q < 0) continue;
                    auto& Q = info[(size_t)(q >> 2)];
                    if (!((Q.outs >> (q & 3)) & 1) && --Q.waits == 0) push(q >> 2);
                }
            });
            pass.insert(pass.end(), {face0, positions - face0, first, taken});
        }
        // one more, empty: the last pass's cells are stored in the step after it
        pass.insert(pass.end(), {positions, 0, (int32_t)n, 0});
    }
    const int32_t passes = (int32_t)(pass.size() / 4);
    // What the device gets, as one image: faces and codes with one record more than
    // used (threads without work load the one after the last).
    const size_t positions = (size_t)n_records / 3;
    const size_t b_faces = align256((positions + 1) * sizeof(SweepFace)), b_s3 = align256((positions + 1) * 24),
                 b_codes = align256((size_t)(n + 1) * 16), b_cells = align256((size_t)(n + 1) * 4),
                 b_pass = align256(pass.size() * 4), b_fix = align256(fix.size() * 4);
    const size_t bytes = b_faces + b_s3 + b_codes + b_cells + b_pass + b_fix;
    if (w.room < bytes) {
        w.image.reset();
        w.room = 0;
        w.image.reset(new char[bytes]);
        w.room = bytes;
    }
    SweepFace* const faces = reinterpret_cast<SweepFace*>(w.image.get());
    double* const s3 = reinterpret_cast<double*>(w.image.get() + b_faces);
    int32_t* const codes = reinterpret_cast<int32_t*>(w.image.get() + b_faces + b_s3);
    int32_t* const cells_out = reinterpret_cast<int32_t*>(w.image.get() + b_faces + b_s3 + b_codes);
    char* const tables = w.image.get() + b_faces + b_s3 + b_codes + b_cells;
    faces[positions] = SweepFace{0, {kSweepZero, kSweepZero, kSweepZero}};
    for (size_t j = 0; j < 3; j++) s3[3 * positions + j] = 0.0;
    for (size_t j = 0; j < 4; j++) codes[4 * (size_t)n + j] = kSweepZero;
    cells.push_back(0);
    std::memcpy(cells_out, cells.data(), cells.size() * 4);
    std::memcpy(tables, pass.data(), pass.size() * 4);
    if (!fix.empty()) std::memcpy(tables + b_pass, fix.data(), fix.size() * 4);
    // Code of a face value in a step: the position that it was written to (its own for
    // an out face, the neighbour's for an in face) while the ring holds it.
    const int32_t ring = block * kSweepRing;
    for (int32_t p = 0; p + 1 < passes; p++) {
        const int32_t* P = &pass[(size_t)p * 4];
        const int32_t first = P[0], cnt = P[1];
        // oldest positions in the ring in step p (node values) and in the step after it (cell values)
        const int32_t node_lo = first + cnt - ring, cell_lo = P[4] + P[5] - ring;
        double* s3_pass = s3 + 3 * (int64_t)first;
        for (int32_t i = P[2]; i < P[2] + P[3]; i++) {
            if (i + 2 * kAhead < n) {
                const int32_t ca = cells[(size_t)i + 2 * kAhead], cb = cells[(size_t)i + kAhead];
                const int64_t rb = 3 * (int64_t)info[(size_t)cb].out0;
                __builtin_prefetch(pairs + 4 * (int64_t)ca);
                __builtin_prefetch(&info[(size_t)ca]);
                __builtin_prefetch(x0_s + rb);
                __builtin_prefetch(x0_s + rb + 8);
                __builtin_prefetch(x0_face + rb);
                for (int f = 0; f < 4; f++) __builtin_prefetch(&info[(size_t)cell_of(pairs[cb * 4 + f])]);
            }
            const int32_t c = cells[(size_t)i];
            const rsh_sweep_s::Cell I = info[(size_t)c];
            int32_t node_code[4], *cell_code = codes + (int64_t)i * 4;
            for (int f = 0; f < 4; f++) {
                const int32_t q = pairs[c * 4 + f];
                const int32_t src = (I.outs >> f) & 1 ? c * 4 + f : q;  // < 0: a boundary's value
                const rsh_sweep_s::Cell& S = info[(size_t)cell_of(src)];
                const int32_t at = S.link + bits(S.outs & ((1u << (src & 3)) - 1u)), slot = at & (ring - 1),
                              far = kSweepFar - src;
                cell_code[f] = at >= cell_lo ? slot : far;
                node_code[f] = at >= node_lo ? slot : far;
                if (src < 0) cell_code[f] = node_code[f] = q == RSH_BOUND_OUT_SOURCE ? kSweepOne : kSweepZero;
            }
            SweepFace* F = faces + I.link;
            double* to = s3_pass + (I.link - first);
            const double* xs = x0_s + 3 * (int64_t)I.out0;  // records of the cell in out-face order
            const uint8_t* xf = x0_face + 3 * (int64_t)I.out0;
            const uint32_t in_source = s->node_in_source.empty() ? 0u : s->node_in_source[(size_t)c];
            for (unsigned left = I.outs; left; left &= left - 1, F++, to++) {
                F->cell = (uint32_t)c | ((in_source >> (3 * __builtin_ctz(left))) & 7u) << kSweepCellBits;
                for (int j = 0; j < 3; j++) {
                    F->up[j] = node_code[*xf++];
                    to[(int64_t)j * cnt] = *xs++;
                }
            }
        }
    }

    std::lock_guard<std::mutex> lock(s->mu);
    RSH_HIP_TRY(hipSetDevice(s->device));
    auto& d = s->dirs[(size_t)k];
    if (d.block) RSH_HIP_TRY(hipFree(d.block));
    d.block = nullptr;
    if (d.set) s->unset++;
    d.set = false;
    hipError_t e = hipMalloc(&d.block, bytes);
    if (e != hipSuccess) return hip_fail(e, "sweep: direction allocation");
    e = hipMemcpy(d.block, w.image.get(), bytes, hipMemcpyHostToDevice);
    if (e != hipSuccess) return hip_fail(e, "sweep: upload of a direction");
    char* const at = static_cast<char*>(d.block);
    d.dev.faces = reinterpret_cast<const SweepFace*>(at);
    d.dev.s3 = reinterpret_cast<const double*>(at + b_faces);
    d.dev.codes = reinterpret_cast<const int32_t*>(at + b_faces + b_s3);
    d.dev.cells = reinterpret_cast<const int32_t*>(at + b_faces + b_s3 + b_codes);
    d.dev.pass = reinterpret_cast<const int32_t*>(at + b_faces + b_s3 + b_codes + b_cells);
    d.dev.fix = reinterpret_cast<const int32_t*>(at + b_faces + b_s3 + b_codes + b_cells + b_pass);
    d.dev.passes = passes;
    d.dev.levels = levels;
    d.dev.fixes = (int32_t)(fix.size() / 2);
    d.set = true;
    s->unset--;
    s->table_dirty = true;
    return RSH_OK;
}

int rsh_sweep_levels(rsh_sweep s, int32_t k, int32_t* levels) {
    if (!s || k < 0 || k >= s->m || !levels) return fail(RSH_E_ARG, "invalid direction or null pointer");
    if (!s->dirs[(size_t)k].set) return fail(RSH_E_STATE, "direction not set");
    *levels = s->dirs[(size_t)k].dev.levels;
    return RSH_OK;
}

int rsh_sweep_run(rsh_sweep s, int32_t cls, const double* d_scattering, int64_t ld, const double* d_illum_old,
                  double* d_illum_new, double* d_norm, void* stream) {
    if (!s || !d_scattering || !d_illum_new || ld < s->n) return fail(RSH_E_ARG, "null pointer or ld < n_cells");
    if (cls != 0 && cls != 1 && cls != 2 && cls != 3 && cls != 10)
        return fail(RSH_E_UNSUPPORTED, "class_vtk must be 0, 1, 2, 3 or 10 (11 couples to the gas dynamics state)");
    if (cls == 0 && s->node_in_source.empty()) return fail(RSH_E_ARG, "class 0 needs the face nodes (rsh_sweep_create nodes)");
    if (d_illum_old && (d_illum_old == d_illum_new || !d_norm))
        return fail(RSH_E_ARG, "the residual needs distinct old and new arrays and a norm array");
    if ((reinterpret_cast<uintptr_t>(d_illum_new) | reinterpret_cast<uintptr_t>(d_illum_old)) & 15)
        return fail(RSH_E_ARG, "illum arrays must be 16-byte aligned");
    std::lock_guard<std::mutex> lock(s->mu);
    for (const auto& d : s->dirs)
        if (!d.set) return fail(RSH_E_STATE, "every direction needs rsh_sweep_set_direction first");
    RSH_HIP_TRY(hipSetDevice(s->device));
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (s->table_dirty) {
        std::vector<SweepDirDev> table;
        for (const auto& d : s->dirs) table.push_back(d.dev);
        RSH_HIP_TRY(hipMemcpy(s->d_table, table.data(), table.size() * sizeof(SweepDirDev), hipMemcpyHostToDevice));
        s->table_dirty = false;
    }
    RSH_HIP_TRY(launch_sweep(cls, s->block, s->d_table, s->m, s->n, d_scattering, ld, d_illum_old,
                             d_illum_new, d_norm, st));
    return RSH_OK;
}

}  // extern "C"
