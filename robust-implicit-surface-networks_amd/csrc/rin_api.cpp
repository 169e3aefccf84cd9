// C ABI over the device pipeline (declarations and conventions in include/rin.h).
#include <hip/hip_runtime.h>

#include <cstring>
#include <memory>
#include <mutex>
#include <string>
#include <vector>

#include "devmem.h"
#include "kernels/fetch.h"
#include "kernels/pipeline.h"
#include "rin.h"

struct rin_ctx {
    int device = 0;
    int n_cu = 256;
    void* scratch = nullptr;  // the allocation-free path's array on this device
    hipStream_t stream = nullptr;
    rin::DevMem mem;
    rin::HostStage stage;
    std::mutex mu;
    std::string err;
};
struct rin_grid {
    rin::Grid g;
};
struct rin_values {
    rin::Values v;
};
struct rin_result {
    rin::RunOut r;
};

namespace {

int fail(rin_ctx* c, int code, const std::string& msg) {
    if (c) c->err = msg;
    return code;
}

template <class F>
int guarded(rin_ctx* c, F&& f) {
    if (!c) return RIN_ERR_ARG;
    std::lock_guard<std::mutex> lock(c->mu);
    try {
        RIN_HIP(hipSetDevice(c->device));
        f();
        return RIN_OK;
    } catch (rin::HipError& e) {
        return fail(c, e.code == hipErrorOutOfMemory ? RIN_ERR_MEMORY : RIN_ERR_DEVICE, e.what());
    } catch (std::invalid_argument& e) {
        return fail(c, RIN_ERR_ARG, e.what());
    } catch (std::runtime_error& e) {
        const std::string w = e.what();
        if (w.find("active functions") != std::string::npos || w.find("capacity") != std::string::npos ||
            w.find("exceed") != std::string::npos)
            return fail(c, RIN_ERR_CAPACITY, w);
        if (w.find("not available") != std::string::npos) return fail(c, RIN_ERR_UNSUPPORTED, w);
        return fail(c, RIN_ERR_INTERNAL, w);
    } catch (std::exception& e) {
        return fail(c, RIN_ERR_INTERNAL, e.what());
    }
}

// an output array: `words` 64-bit words at dst
rin::PackCol col(rin::PackKind kind, uint64_t words, void* dst, const void* p0, const void* p1 = nullptr,
                 const void* p2 = nullptr, const void* p3 = nullptr, const void* p4 = nullptr) {
    rin::PackCol c;
    c.kind = kind;
    c.words = words;
    c.dst = dst;
    c.p[0] = p0;
    c.p[1] = p1;
    c.p[2] = p2;
    c.p[3] = p3;
    c.p[4] = p4;
    return c;
}

void fetch(rin_ctx* c, const std::vector<rin::PackCol>& cols) { c->stage.fetch(c->device, cols, c->stream); }

}  // namespace

extern "C" {

int rin_create(rin_ctx** out, int32_t device) {
    if (!out) return RIN_ERR_ARG;
    *out = nullptr;
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess || n == 0) return RIN_ERR_DEVICE;
    if (device < 0 || device >= n) return RIN_ERR_ARG;
    auto* c = new rin_ctx;
    c->device = device;
    if (hipSetDevice(device) != hipSuccess || hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess) {
        delete c;
        return RIN_ERR_DEVICE;
    }
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, device) == hipSuccess && prop.multiProcessorCount > 0)
        c->n_cu = prop.multiProcessorCount;
    try {
        c->scratch = rin::noalloc_scratch_address();
    } catch (std::exception&) {
        (void)hipStreamDestroy(c->stream);
        delete c;
        return RIN_ERR_DEVICE;
    }
    *out = c;
    return RIN_OK;
}

int rin_device_memory(rin_ctx* c, uint64_t* free_bytes, uint64_t* total_bytes) {
    if (!free_bytes || !total_bytes) return fail(c, RIN_ERR_ARG, "null argument");
    return guarded(c, [&] {
        size_t f = 0, t = 0;
        RIN_HIP(hipMemGetInfo(&f, &t));
        *free_bytes = f;
        *total_bytes = t;
    });
}

int rin_destroy(rin_ctx* c) {
    if (!c) return RIN_ERR_ARG;
    (void)hipSetDevice(c->device);
    (void)hipStreamSynchronize(c->stream);
    c->mem.trim();
    c->stage.release();
    (void)hipStreamDestroy(c->stream);
    delete c;
    return RIN_OK;
}

const char* rin_last_error(const rin_ctx* c) { return c ? c->err.c_str() : "null context"; }

int rin_grid_regular(rin_ctx* c, int32_t res, const double bmin[3], const double bmax[3], rin_grid** out) {
    if (!out || !bmin || !bmax) return fail(c, RIN_ERR_ARG, "null argument");
    return guarded(c, [&] {
        auto g = std::make_unique<rin_grid>();
        rin::grid_regular(c->mem, res, bmin, bmax, g->g, c->stream);
        RIN_HIP(hipStreamSynchronize(c->stream));
        *out = g.release();
    });
}

int rin_grid_explicit(rin_ctx* c, const double* pts, uint64_t V, const uint64_t* tets, uint64_t T, rin_grid** out) {
    if (!out || !pts || !tets) return fail(c, RIN_ERR_ARG, "null argument");
    return guarded(c, [&] {
        auto g = std::make_unique<rin_grid>();
        rin::grid_explicit(c->mem, pts, V, tets, T, g->g, c->stream);
        *out = g.release();
    });
}

int rin_grid_points(rin_ctx* c, const rin_grid* g, double* pts) {
    if (!g || !pts) return fail(c, RIN_ERR_ARG, "null argument");
    return guarded(c, [&] {
        RIN_HIP(hipMemcpyAsync(pts, g->g.pts.p, 24 * g->g.view.V, hipMemcpyDeviceToHost, c->stream));
        RIN_HIP(hipStreamSynchronize(c->stream));
    });
}

int rin_grid_release(rin_ctx* c, rin_grid* g) {
    return guarded(c, [&] {
        RIN_HIP(hipStreamSynchronize(c->stream));
        delete g;
    });
}

int rin_values_eval(rin_ctx* c, const rin_grid* g, const rin_func_desc* f, uint32_t F, rin_values** out) {
    if (!g || !f || !out) return fail(c, RIN_ERR_ARG, "null argument");
    static_assert(sizeof(rin_func_desc) == sizeof(rin::FuncDesc), "descriptor layout");
    return guarded(c, [&] {
        auto v = std::make_unique<rin_values>();
        rin::values_eval(c->mem, g->g, reinterpret_cast<const rin::FuncDesc*>(f), F, v->v, c->stream);
        *out = v.release();
    });
}

int rin_values_upload(rin_ctx* c, const rin_grid* g, const double* rm, uint32_t F, rin_values** out) {
    if (!g || !rm || !out) return fail(c, RIN_ERR_ARG, "null argument");
    return guarded(c, [&] {
        auto v = std::make_unique<rin_values>();
        rin::values_upload(c->mem, g->g, rm, F, v->v, c->stream);
        *out = v.release();
    });
}

int rin_eval_points(rin_ctx* c, const double* pts, uint64_t n, const rin_func_desc* f, uint32_t F, double* rm) {
    if ((!pts && n) || !f || (!rm && n)) return fail(c, RIN_ERR_ARG, "null argument");
    return guarded(c, [&] {
        rin::eval_points(c->mem, pts, n, reinterpret_cast<const rin::FuncDesc*>(f), F, rm, c->stream);
    });
}

int rin_eval_points_noalloc(rin_ctx* c, const double* pts, uint64_t n, const rin_func_desc* f, uint32_t F,
                            double* rm) {
    if ((!pts && n) || !f || (!rm && n)) return fail(c, RIN_ERR_ARG, "null argument");
    return guarded(c, [&] {
        rin::eval_points_noalloc(c->scratch, pts, n, reinterpret_cast<const rin::FuncDesc*>(f), F, rm, c->stream);
        RIN_HIP(hipStreamSynchronize(c->stream));
    });
}

int rin_values_download(rin_ctx* c, const rin_values* v, double* rm) {
    if (!v || !rm) return fail(c, RIN_ERR_ARG, "null argument");
    return guarded(c, [&] {
        rin::PackCol x = col(rin::PACK_ROWMAJOR, v->v.V * v->v.F, rm, v->v.vals.p);
        x.rows = v->v.F;
        x.stride = v->v.V;
        fetch(c, {x});
    });
}

int rin_values_release(rin_ctx* c, rin_values* v) {
    return guarded(c, [&] {
        RIN_HIP(hipStreamSynchronize(c->stream));
        delete v;
    });
}

int rin_run(rin_ctx* c, const rin_grid* g, const rin_values* v, uint32_t flags, rin_result** out) {
    if (!g || !v || !out) return fail(c, RIN_ERR_ARG, "null argument");
    *out = nullptr;
    if (v->v.grid_id != g->g.id) return fail(c, RIN_ERR_ARG, "the values were made on another grid");
    return guarded(c, [&] {
        auto r = std::make_unique<rin_result>();
        if (flags & RIN_FLAG_BATCHED) {
            try {
                if (flags & RIN_FLAG_MI)
                    rin::run_batched_mi(c->mem, g->g, v->v, flags, r->r, c->stream);
                else
                    rin::run_batched(c->mem, g->g, v->v, flags, r->r, c->stream, c->n_cu);
            } catch (rin::NeedsPlainForm& e) {
                // the plain form handles every tet the buckets cannot
                RIN_HIP(hipStreamSynchronize(c->stream));
                r = std::make_unique<rin_result>();
                rin::run_pipeline(c->mem, g->g, v->v, flags & ~(uint32_t)RIN_FLAG_BATCHED, r->r, c->stream);
                r->r.times.ms.insert(r->r.times.ms.begin(), {std::string("batched form fell back: ") + e.what(), 0.f});
            }
        } else {
            rin::run_pipeline(c->mem, g->g, v->v, flags, r->r, c->stream);
        }
        RIN_HIP(hipStreamSynchronize(c->stream));
        *out = r.release();
    });
}

int rin_result_sizes(rin_ctx* c, const rin_result* res, rin_sizes* s) {
    if (!res || !s) return fail(c, RIN_ERR_ARG, "null argument");
    const auto& r = res->r;
    s->n_tets = r.T;
    s->n_funcs = r.F;
    s->num_degenerate = r.num_degenerate;
    s->num_intersecting = r.num_intersecting;
    for (int i = 0; i < 3; ++i) s->bucket[i] = r.nb[i];
    s->n_func_in_tet = r.n_fit;
    s->n_verts = r.n_verts;
    s->n_faces = r.n_faces;
    s->n_face_verts = r.n_face_verts;
    s->n_tet_faces = r.n_tet_faces;
    s->n_vert_occ = r.n_vert_occ;
    s->n_face_occ = r.n_face_occ;
    s->n_face_occ_verts = r.n_face_occ_verts;
    s->n_cut[0] = r.n_cut34;
    s->n_cut[1] = r.n_cut58;
    s->n_rec_words = r.n_rec_words;
    for (int i = 0; i < 2; ++i) {
        s->cut_k_sum[i] = r.cut_k_sum[i];
        s->cut_words[i] = r.cut_words[i];
    }
    return RIN_OK;
}

int rin_result_csr(rin_ctx* c, const rin_result* res, uint64_t* fit, uint64_t* start) {
    if (!res || !fit || !start) return fail(c, RIN_ERR_ARG, "null argument");
    return guarded(c, [&] {
        const auto& r = res->r;
        rin::PackCol f = col(rin::PACK_U8, r.n_fit, fit, r.view.fit);
        fetch(c, {f, col(rin::PACK_U32, r.T + 1, start, r.view.csr_off)});
    });
}

int rin_result_verts(rin_ctx* c, const rin_result* res, uint64_t* rec11, double* xyz) {
    if (!res || !rec11 || !xyz) return fail(c, RIN_ERR_ARG, "null argument");
    return guarded(c, [&] {
        const auto& w = res->r.view;
        const uint64_t n = res->r.n_verts;
        fetch(c, {col(rin::PACK_VERT, 11 * n, rec11, w.v_tet, w.v_j, w.v_ss, w.v_sv, w.v_fn),
                  col(rin::PACK_F64, 3 * n, xyz, w.xyz)});
    });
}

int rin_result_faces(rin_ctx* c, const rin_result* res, uint64_t* vstart, uint64_t* verts, uint64_t* tfstart,
                     uint64_t* tf, uint64_t* func) {
    if (!res || !vstart || !verts || !tfstart || !tf || !func) return fail(c, RIN_ERR_ARG, "null argument");
    return guarded(c, [&] {
        const auto& r = res->r;
        const auto& w = r.view;
        const uint64_t nf = r.n_faces;
        fetch(c, {col(rin::PACK_U32, nf + 1, vstart, w.f_vstart), col(rin::PACK_U32, r.n_face_verts, verts, w.f_verts),
                  col(rin::PACK_U32, nf + 1, tfstart, w.f_tfstart),
                  col(rin::PACK_TET_FACE, 2 * r.n_tet_faces, tf, w.f_tf_tet, w.f_tf_local),
                  col(rin::PACK_U8_NONE, 2 * nf, func, w.f_func)});
    });
}

int rin_result_edge_count(rin_ctx* c, const rin_result* res, uint64_t* n_edges) {
    if (!res || !n_edges) return fail(c, RIN_ERR_ARG, "null argument");
    return guarded(c, [&] {
        auto& r = const_cast<rin_result*>(res)->r;  // the edges are cached in the result
        rin::compute_edges(c->mem, r, c->stream);
        *n_edges = r.n_edges;
    });
}

int rin_result_edges(rin_ctx* c, const rin_result* res, uint64_t* v12, uint64_t* start, uint64_t* occ,
                     uint64_t* edge_of) {
    if (!res || !v12 || !start || !occ || !edge_of) return fail(c, RIN_ERR_ARG, "null argument");
    return guarded(c, [&] {
        auto& r = const_cast<rin_result*>(res)->r;
        rin::compute_edges(c->mem, r, c->stream);
        const uint64_t NE = r.n_edges, NO = r.n_face_verts;
        fetch(c, {col(rin::PACK_U32, 2 * NE, v12, r.e_v12.p), col(rin::PACK_U32, NE + 1, start, r.e_start.p),
                  col(rin::PACK_EDGE_OCC, 2 * NO, occ, r.e_occ.p, r.e_face_of.p, r.view.f_vstart),
                  col(rin::PACK_U32, NO, edge_of, r.e_of_occ.p)});
    });
}

int rin_result_patch_count(rin_ctx* c, const rin_result* res, uint64_t* n_patches) {
    if (!res || !n_patches) return fail(c, RIN_ERR_ARG, "null argument");
    return guarded(c, [&] {
        auto& r = const_cast<rin_result*>(res)->r;  // the patches are cached in the result
        rin::compute_patches(c->mem, r, c->stream);
        *n_patches = r.n_patches;
    });
}

int rin_result_patches(rin_ctx* c, const rin_result* res, uint64_t* start, uint64_t* faces) {
    if (!res || !start || (!faces && res->r.n_faces)) return fail(c, RIN_ERR_ARG, "null argument");
    return guarded(c, [&] {
        auto& r = const_cast<rin_result*>(res)->r;
        rin::compute_patches(c->mem, r, c->stream);
        fetch(c, {col(rin::PACK_U32, r.n_patches + 1, start, r.p_start.p),
                  col(rin::PACK_U32, r.n_faces, faces, r.p_faces.p)});
    });
}

int rin_result_chain_count(rin_ctx* c, const rin_result* res, uint64_t* n_chains) {
    if (!res || !n_chains) return fail(c, RIN_ERR_ARG, "null argument");
    return guarded(c, [&] {
        auto& r = const_cast<rin_result*>(res)->r;  // the chains are cached in the result
        rin::compute_chains(c->mem, r, c->stream);
        *n_chains = r.n_chains;
    });
}

int rin_result_chains(rin_ctx* c, const rin_result* res, uint64_t* start, uint64_t* edges) {
    if (!res || !start) return fail(c, RIN_ERR_ARG, "null argument");
    return guarded(c, [&] {
        auto& r = const_cast<rin_result*>(res)->r;
        rin::compute_chains(c->mem, r, c->stream);
        fetch(c, {col(rin::PACK_U32, r.n_chains + 1, start, r.c_start.p)});
        const uint64_t n = start[r.n_chains];
        if (n && !edges) throw std::invalid_argument("null argument");
        if (n) fetch(c, {col(rin::PACK_U32, n, edges, r.c_edges.p)});
    });
}

int rin_result_records(rin_ctx* c, const rin_result* res, const uint64_t* tets, uint64_t n, uint64_t* rec_start,
                       uint16_t* words, uint64_t cap) {
    if (!res || (!tets && n) || !rec_start) return fail(c, RIN_ERR_ARG, "null argument");
    return guarded(c, [&] {
        const auto& r = res->r;
        if (!r.view.rec) throw std::invalid_argument("records were not kept (RIN_FLAG_KEEP_RECORDS)");
        rin::gather_records(c->mem, r, tets, n, rec_start, words, cap, c->stream);
    });
}

int rin_result_cut_counts(rin_ctx* c, const rin_result* res, uint64_t* counts) {
    if (!res || !counts) return fail(c, RIN_ERR_ARG, "null argument");
    return guarded(c, [&] {
        const auto& r = res->r;
        if (!r.view.cut_counts) throw std::invalid_argument("run was not RIN_FLAG_CUT_ONLY");
        fetch(c, {col(rin::PACK_U32, 3 * r.n_active, counts, r.view.cut_counts)});
    });
}

int rin_result_stage_times(rin_ctx* c, const rin_result* res, double* ms, int32_t cap) {
    if (!res) return fail(c, RIN_ERR_ARG, "null argument");
    const auto& t = res->r.times.ms;
    int n = 0;
    for (auto& e : t)
        if (n < cap && ms) ms[n++] = e.second;
    return (int)t.size();
}

const char* rin_result_stage_label(rin_ctx* c, const rin_result* res, int32_t i) {
    (void)c;
    if (!res || i < 0 || i >= (int)res->r.times.ms.size()) return "";
    return res->r.times.ms[i].first.c_str();
}

int rin_result_release(rin_ctx* c, rin_result* res) {
    return guarded(c, [&] {
        RIN_HIP(hipStreamSynchronize(c->stream));
        delete res;
    });
}

int rin_debug_cuts(rin_ctx* c, int32_t mi, const double* rows, const int32_t* ks, int32_t n, int32_t cap,
                   uint16_t* words, int32_t* lens) {
    if (!rows || !ks || !words || !lens || n < 0 || cap <= 8) return fail(c, RIN_ERR_ARG, "bad argument");
    return guarded(c, [&] { rin::debug_cuts(c->mem, mi, rows, ks, n, cap, words, lens, c->stream); });
}

int rin_debug_table_cuts(int32_t mode, const double* rows, int32_t n, int32_t cap, uint16_t* words, int32_t* lens) {
    if (!rows || !words || !lens || n < 0 || cap <= 8 || mode < 0 || mode > 3) return RIN_ERR_ARG;
    try {
        const int nr = mode == 0 ? 1 : (mode == 3 ? 3 : 2);
        for (int32_t i = 0; i < n; ++i) {
            const double* r = rows + (size_t)4 * nr * i;
            uint16_t* w = words + (size_t)cap * i;
            lens[i] = mode == 3   ? rin::debug_table_record_mi3(r, w, cap)
                      : mode == 2 ? rin::debug_table_record_mi2(r, w, cap)
                                  : rin::debug_table_record_ia(nr, r, w, cap);
        }
        return RIN_OK;
    } catch (std::exception&) {
        return RIN_ERR_INTERNAL;
    }
}

int rin_debug_copy(rin_ctx* c, uint64_t bytes, int32_t reps, double* ms) {
    if (!ms) return fail(c, RIN_ERR_ARG, "null argument");
    return guarded(c, [&] { *ms = rin::debug_copy(c->mem, bytes, reps, c->stream); });
}

int rin_debug_sqrt(rin_ctx* c, const double* in, uint64_t n, double* out) {
    if ((!in || !out) && n) return fail(c, RIN_ERR_ARG, "null argument");
    return guarded(c, [&] { rin::debug_sqrt(c->mem, in, n, out, c->stream); });
}

int rin_debug_scan(rin_ctx* c, int32_t fields, int32_t stride, const uint32_t* in, uint64_t n, uint64_t count,
                   uint32_t* out, uint32_t* totals) {
    if ((!in && n) || (!out && n) || !totals) return fail(c, RIN_ERR_ARG, "null argument");
    return guarded(c, [&] { rin::debug_scan(c->mem, fields, stride, in, n, count, out, totals, c->stream); });
}

}  // extern "C"
