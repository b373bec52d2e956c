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
    // set of its own: fresh pages would cost more than half of the planning).
    struct Work {
        std::vector<int64_t> x0_off;
        std::vector<int32_t> pos, level, waits, chain, entries, cells, pos_of, pass_of, pass, touched, next, old, open,
            codes, fix;
        std::vector<SweepFace> faces;
        std::vector<double> s3;
    };
    std::vector<std::unique_ptr<Work>> spare;
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
    auto cleanup = [&](int rc) {
        rsh_sweep_destroy(s);
        return rc;
    };
    if (hipSetDevice(device) != hipSuccess) return cleanup(fail(RSH_E_HIP, "hipSetDevice failed"));
    if (hipMalloc(&s->d_table, (size_t)n_dirs * sizeof(SweepDirDev)) != hipSuccess)
        return cleanup(fail(RSH_E_NOMEM, "sweep: device allocation failed"));
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
    struct Lease {  // a Work of this call, given back at its end
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
            s->spare.push_back(std::move(w));
        }
    } lease(s);
    rsh_sweep_s::Work& w = *lease.w;
    auto &pos = w.pos, &level = w.level;
    pos.assign((size_t)n, -1);
    level.assign((size_t)n, 0);
    for (int64_t h = 0; h < n; h++) {
        const int32_t c = order[h];
        if (c < 0 || c >= n || pos[(size_t)c] >= 0) return fail(RSH_E_ARG, "order is not a permutation of the cells");
        pos[(size_t)c] = (int32_t)h;
    }
    auto& x0_off = w.x0_off;
    x0_off.resize((size_t)n);
    int64_t r = 0;
    int32_t levels = 0;
    for (int64_t h = 0; h < n; h++) {
        const int32_t c = order[h];
        const int st = face_state[c];
        if (st < 0 || st > 15) return fail(RSH_E_ARG, "face state outside 0..15");
        x0_off[(size_t)c] = r;
        int32_t lv = 0;
        for (int f = 0; f < 4; f++) {
            const int32_t p = s->pairs[(size_t)(c * 4 + f)];
            const bool in = (st >> f) & 1;
            if (!in) {
                for (int j = 0; j < 3; j++, r++) {
                    if (r >= n_records) return fail(RSH_E_ARG, "fewer x0 records than out-face nodes");
                    const int g = x0_face[r];
                    if (g > 3 || !((st >> g) & 1))
                        return fail(RSH_E_ARG, "x0 record " + std::to_string(r) + " does not name an in face");
                }
            }
            if (p < 0) continue;
            const int32_t u = p / 4;
            // Reads across an in face, and a face both cells treat as out
            // (written by both: the later one in the order wins), order u first.
            const bool dep = in || (!((face_state[u] >> (p % 4)) & 1) && pos[(size_t)u] < h);
            if (!dep) continue;
            if (pos[(size_t)u] > h)
                return fail(RSH_E_ARG, "order is not upwind: cell " + std::to_string(c) + " reads cell " +
                                           std::to_string(u) + " that comes later");
            lv = std::max(lv, level[(size_t)u] + 1);
        }
        level[(size_t)c] = lv;
        levels = std::max(levels, lv + 1);
    }
    if (r != n_records) return fail(RSH_E_ARG, "more x0 records than out-face nodes");
    // Cells read by a cell, and the longest chain of cells that still waits on it.
    auto &waits = w.waits, &chain = w.chain;
    waits.assign((size_t)n, 0);
    chain.assign((size_t)n, 0);
    auto reads = [&](int32_t c, int f) { return ((face_state[c] >> f) & 1) && s->pairs[(size_t)(c * 4 + f)] >= 0; };
    for (int64_t h = n - 1; h >= 0; h--) {
        const int32_t c = order[h];
        for (int f = 0; f < 4; f++)
            if (reads(c, f)) {
                const int32_t u = s->pairs[(size_t)(c * 4 + f)] / 4;
                waits[(size_t)c]++;
                chain[(size_t)u] = std::max(chain[(size_t)u], chain[(size_t)c] + 1);
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
    auto &entries = w.entries, &cells = w.cells, &pos_of = w.pos_of, &pass_of = w.pass_of, &pass = w.pass;
    entries.clear();
    cells.clear();
    pass.clear();
    entries.reserve((size_t)n_records / 3);
    cells.reserve((size_t)n + 1);
    pos_of.assign((size_t)n * 4, -1);
    pass_of.resize((size_t)n);
    auto& cell_at = w.next;  // a cell taken is in no list any more
    cell_at.resize((size_t)n);
    auto out_faces = [&](int32_t c) { return 4 - __builtin_popcount((unsigned)face_state[c]); };
    {
        // ready cells as lists: by the pass that touched their group, by their chain
        auto &touched = w.touched, &next = w.next, &old = w.old, &open = w.open;
        touched.assign((size_t)(n / kLineCells + 1), -1);
        old.clear();
        open.assign((size_t)levels, -1);
        int32_t oldest = 0, longest = -1;
        auto push = [&](int32_t c) {
            const int32_t t = touched[(size_t)(c / kLineCells)], l = chain[(size_t)c];
            int32_t& head = t >= 0 ? old[(size_t)t] : open[(size_t)l];
            if (t >= 0) oldest = std::min(oldest, t);
            else longest = std::max(longest, l);
            next[(size_t)c] = head;
            head = c;
        };
        auto top = [&]() -> int32_t* {
            while (oldest < (int32_t)old.size() && old[(size_t)oldest] < 0) oldest++;
            if (oldest < (int32_t)old.size()) return &old[(size_t)oldest];
            while (longest >= 0 && open[(size_t)longest] < 0) longest--;
            return longest >= 0 ? &open[(size_t)longest] : nullptr;
        };
        for (int32_t c = (int32_t)n - 1; c >= 0; c--)
            if (!waits[(size_t)c]) push(c);
        for (int32_t p = 0; top(); p++) {
            const size_t first = cells.size();
            const int32_t face0 = (int32_t)entries.size();
            int32_t cnt = 0;
            old.push_back(-1);
            for (int32_t* head; (int32_t)(cells.size() - first) < block / 2 && (head = top());) {
                const int32_t c = *head;
                if ((cnt += out_faces(c)) > block) break;
                *head = next[(size_t)c];
                int32_t& t = touched[(size_t)(c / kLineCells)];
                if (t < 0) t = p;
                cells.push_back(c);
            }
            std::sort(cells.begin() + (int64_t)first, cells.end());
            for (size_t i = first; i < cells.size(); i++) {
                const int32_t c = cells[i];
                pass_of[(size_t)c] = p;
                cell_at[(size_t)c] = (int32_t)i;
                for (int f = 0; f < 4; f++)
                    if (!((face_state[c] >> f) & 1)) {
                        const int32_t q = s->pairs[(size_t)(c * 4 + f)];
                        pos_of[(size_t)(c * 4 + f)] = (int32_t)entries.size();
                        entries.push_back(c * 4 + f);
                        if (q >= 0 && reads(q / 4, q % 4) && --waits[(size_t)(q / 4)] == 0) push(q / 4);
                    }
            }
            pass.insert(pass.end(), {face0, (int32_t)entries.size() - face0, (int32_t)first, (int32_t)(cells.size() - first)});
        }
    }
    // one more, empty: the last pass's cells are stored in the step after it
    pass.insert(pass.end(), {(int32_t)entries.size(), 0, (int32_t)n, 0});
    const int32_t passes = (int32_t)(pass.size() / 4);
    // Code of an entry's value at step `step`: its own position's for an out face,
    // the neighbour's for an in face.
    const int64_t ring = (int64_t)block * kSweepRing;
    auto code_of = [&](int32_t e, int32_t step) -> int32_t {
        const int32_t up = s->pairs[(size_t)e];
        int32_t src = e;
        if ((face_state[e / 4] >> (e % 4)) & 1) {
            if (up < 0) return up == RSH_BOUND_OUT_SOURCE ? kSweepOne : kSweepZero;
            src = up;
        }
        const int64_t end = (int64_t)pass[(size_t)step * 4] + pass[(size_t)step * 4 + 1];
        return pos_of[(size_t)src] >= end - ring ? (int32_t)(pos_of[(size_t)src] & (ring - 1)) : kSweepFar - src;
    };
    // one record more than used: threads without work load the one after the last
    auto& faces = w.faces;
    auto& s3 = w.s3;
    auto &codes = w.codes, &fix = w.fix;
    faces.resize(entries.size() + 1);
    faces.back() = SweepFace{0, {kSweepZero, kSweepZero, kSweepZero}};
    s3.resize((entries.size() + 1) * 3);
    for (int j = 1; j <= 3; j++) s3[s3.size() - (size_t)j] = 0.0;
    codes.resize((size_t)(n + 1) * 4);
    for (int j = 1; j <= 4; j++) codes[codes.size() - (size_t)j] = kSweepZero;
    fix.clear();
    for (int64_t h = 0; h < n; h++) {
        const int32_t c = order[h], i = cell_at[(size_t)c], p = pass_of[(size_t)c];
        const int64_t first = pass[(size_t)p * 4], cnt = pass[(size_t)p * 4 + 1];
        int64_t r = x0_off[(size_t)c];  // records of the cell in out-face order
        for (int f = 0; f < 4; f++) {
            const int32_t e = c * 4 + f;
            codes[(size_t)i * 4 + (size_t)f] = code_of(e, p + 1);
            const int32_t at = pos_of[(size_t)e];
            if (at < 0) continue;
            SweepFace& F = faces[(size_t)at];
            F.cell = (uint32_t)c;
            if (!s->node_in_source.empty())
                F.cell |= (uint32_t)((s->node_in_source[(size_t)c] >> (3 * f)) & 7u) << kSweepCellBits;
            for (int j = 0; j < 3; j++, r++) {
                F.up[j] = code_of(c * 4 + x0_face[r], p);
                s3[(size_t)(first * 3 + j * cnt + at - first)] = x0_s[r];
            }
            // a face out on both sides: the later cell in the given order wins
            const int32_t q = s->pairs[(size_t)e];
            if (q >= 0 && pos_of[(size_t)q] >= 0 && pos[(size_t)(q / 4)] < pos[(size_t)c]) fix.insert(fix.end(), {q, e});
        }
    }
    cells.push_back(0);

    const size_t b_faces = align256(faces.size() * sizeof(SweepFace)), b_s3 = align256(s3.size() * 8),
                 b_pass = align256(pass.size() * 4), b_codes = align256(codes.size() * 4),
                 b_cells = align256(cells.size() * 4), b_fix = align256(fix.size() * 4);
    std::lock_guard<std::mutex> lock(s->mu);
    RSH_HIP_TRY(hipSetDevice(s->device));
    auto& d = s->dirs[(size_t)k];
    if (d.block) RSH_HIP_TRY(hipFree(d.block));
    d.block = nullptr;
    d.set = false;
    if (hipMalloc(&d.block, b_faces + b_s3 + b_pass + b_codes + b_cells + b_fix) != hipSuccess)
        return fail(RSH_E_NOMEM, "sweep: direction allocation failed");
    char* at = static_cast<char*>(d.block);
    auto put = [&](const void* src, size_t bytes, size_t room) {
        char* dst = at;
        at += room;
        return !bytes || hipMemcpy(dst, src, bytes, hipMemcpyHostToDevice) == hipSuccess ? dst : nullptr;
    };
    d.dev.faces = reinterpret_cast<const SweepFace*>(put(faces.data(), faces.size() * sizeof(SweepFace), b_faces));
    d.dev.s3 = reinterpret_cast<const double*>(put(s3.data(), s3.size() * 8, b_s3));
    d.dev.pass = reinterpret_cast<const int32_t*>(put(pass.data(), pass.size() * 4, b_pass));
    d.dev.codes = reinterpret_cast<const int32_t*>(put(codes.data(), codes.size() * 4, b_codes));
    d.dev.cells = reinterpret_cast<const int32_t*>(put(cells.data(), cells.size() * 4, b_cells));
    d.dev.fix = reinterpret_cast<const int32_t*>(put(fix.data(), fix.size() * 4, b_fix));
    if (!d.dev.faces || !d.dev.s3 || !d.dev.pass || !d.dev.codes || !d.dev.cells || !d.dev.fix)
        return fail(RSH_E_HIP, "sweep: upload of a direction failed");
    d.dev.passes = passes;
    d.dev.levels = levels;
    d.dev.fixes = (int32_t)(fix.size() / 2);
    d.set = true;
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
