// Batches (many sinograms over one resident matrix, mlem_batch_*) and the
// tile-shape autotuner (mlem_autotune).
#include "abi_internal.hpp"

using namespace mlem;
using namespace mlem::abi;

namespace {

// One iteration of the passes marked in `passes` on the batch's stream, up to
// b->group passes per launch.
int enqueue_batch_iteration(mlem_batch *b, const std::vector<uint8_t> &passes) {
    hipStream_t s = b->stream;
    const uint32_t BC = b->BC;
    for (uint32_t p = 0; p < b->passes;) {
        PassX fx{}, bx{};
        PassEpi fe{}, be{};
        for (; p < b->passes && fx.n < b->group; ++p) {
            if (!passes[p] || !b->pass[p]) continue;
            float *f = b->pass[p]->f.as<float>(), *ratio = b->pass[p]->ratio.as<float>();
            const uint32_t k = fx.n++;
            fx.x[k] = f;
            fe.ea[k].out = ratio;
            fe.ea[k].g = b->pass[p]->g.as<int32_t>();
            bx.x[k] = ratio;
            be.ea[k].norm = b->sens.as<float>();
            be.ea[k].f = f;
            be.ea[k].active = b->active.as<uint32_t>() + (size_t)p * BC;
        }
        fe.n = bx.n = be.n = fx.n;
        if (!fx.n) break;
        float *part = b->part.as<float>();
        HIPCHK(launch_tiled_spmv(b->tfp->plan, b->tfp->view, b->wfp->view, fx, part, BC, b->nt, EPI_RATIO, fe, s));
        HIPCHK(launch_tiled_spmv(b->tbp->plan, b->tbp->view, b->wbp->view, bx, part, BC, b->nt, EPI_UPDATE, be, s));
    }
    return MLEM_OK;
}

// A captured iteration holds the addresses of the passes and of the partial sums.
void drop_graph(mlem_batch *b) {
    if (b->gexec) (void)hipGraphExecDestroy(b->gexec);
    b->gexec = nullptr;
}

}  // namespace

namespace mlem {
namespace abi {

int batch_set_async(mlem_batch *b, uint32_t slot, const int32_t *g, const float *f0, uint64_t *allocated) {
    if (allocated) *allocated = 0;
    ARGCHK(b && g && f0, "mlem_batch_set: null argument");
    ARGCHK(slot < b->slots, "mlem_batch_set: slot %u >= %u", slot, b->slots);
    HIPCHK(hipSetDevice(b->m->device));
    const uint32_t p = slot / b->BC, q = slot % b->BC;
    const mlem_matrix *m = b->m;
    hipStream_t s = b->stream;
    if (!b->pass[p]) {  // first slot of this pass: its vectors, zero-filled (padding included)
        auto np = std::make_unique<BatchPass>();
        auto vectors = [&]() {
            hipError_t e = np->g.alloc(sizeof(int32_t) * b->rows_x * b->BC);
            if (e == hipSuccess) e = np->ratio.alloc(sizeof(float) * b->rows_x * b->BC);
            if (e == hipSuccess) e = np->f.alloc(sizeof(float) * b->cols_x * b->BC);
            return e;
        };
        hipError_t e = vectors();
        if (e == hipErrorOutOfMemory && b->group > 1) {  // the partial sums of one pass will do
            HIPCHK(hipStreamSynchronize(s));
            drop_graph(b);
            if (int st = batch_alloc_part(b, 1, 0)) return st;
            e = vectors();
        }
        HIPCHK(e);
        HIPCHK(launch_fill_u32(np->g.as<uint32_t>(), 0u, b->rows_x * b->BC, s));
        HIPCHK(launch_fill(np->ratio.as<float>(), 0.0f, b->rows_x * b->BC, s));
        HIPCHK(launch_fill(np->f.as<float>(), 0.0f, b->cols_x * b->BC, s));
        if (allocated) *allocated = np->g.bytes + np->ratio.bytes + np->f.bytes;
        b->pass[p] = std::move(np);
    }
    BatchPass &bp = *b->pass[p];
    // One staging vector serves both copies: the stream orders the second
    // copy after the first scatter.
    HIPCHK(hipMemcpyAsync(b->stage.p, g, sizeof(int32_t) * m->rows, hipMemcpyHostToDevice, s));
    if (b->row_order)  // the tiles hold A's rows in the matrix's row order: so do the counts
        HIPCHK(launch_ordered_put(bp.g.as<int32_t>() + q, b->BC, b->stage.p, b->row_order, m->rows, s));
    else
        HIPCHK(launch_strided_put(bp.g.as<int32_t>() + q, b->BC, b->stage.p, m->rows, s));
    HIPCHK(hipMemcpyAsync(b->stage.p, f0, sizeof(float) * m->cols, hipMemcpyHostToDevice, s));
    HIPCHK(launch_strided_put(bp.f.as<float>() + q, b->BC, b->stage.p, m->cols, s));
    HIPCHK(launch_fill_u32(b->active.as<uint32_t>() + slot, 1u, 1, s));
    b->active_host[slot] = 1;
    return MLEM_OK;
}

int batch_get_image_async(mlem_batch *b, uint32_t slot, float *f_out) {
    ARGCHK(b && f_out, "mlem_batch_get_image: null argument");
    ARGCHK(slot < b->slots, "mlem_batch_get_image: slot %u >= %u", slot, b->slots);
    const uint32_t p = slot / b->BC, q = slot % b->BC;
    ARGCHK(b->pass[p], "mlem_batch_get_image: slot %u was never set", slot);
    HIPCHK(hipSetDevice(b->m->device));
    HIPCHK(launch_strided_get(b->stage.p, b->pass[p]->f.as<float>() + q, b->BC, b->m->cols, b->stream));
    HIPCHK(hipMemcpyAsync(f_out, b->stage.p, sizeof(float) * b->m->cols, hipMemcpyDeviceToHost, b->stream));
    return MLEM_OK;
}

int batch_deactivate_async(mlem_batch *b, uint32_t slot) {
    ARGCHK(b, "mlem_batch_deactivate: null handle");
    ARGCHK(slot < b->slots, "mlem_batch_deactivate: slot %u >= %u", slot, b->slots);
    HIPCHK(hipSetDevice(b->m->device));
    b->active_host[slot] = 0;
    HIPCHK(launch_fill_u32(b->active.as<uint32_t>() + slot, 0u, 1, b->stream));
    return MLEM_OK;
}

int batch_move_slot_async(mlem_batch *b, uint32_t from, uint32_t to) {
    ARGCHK(b && from < b->slots && to < b->slots && from != to, "batch_move_slot: bad slots %u -> %u", from, to);
    const uint32_t BC = b->BC, pf = from / BC, qf = from % BC, pt = to / BC, qt = to % BC;
    ARGCHK(b->pass[pf] && b->pass[pt] && b->active_host[from] && !b->active_host[to],
           "batch_move_slot: slot %u is not active or slot %u is not free in an allocated pass", from, to);
    HIPCHK(hipSetDevice(b->m->device));
    hipStream_t s = b->stream;
    const uint32_t rows = b->m->rows, cols = b->m->cols;
    // The counts in the positions the tiles hold them (row order or not), and the image; the ratios are
    // recomputed from them by the next iteration.
    HIPCHK(launch_strided_get(b->stage.p, b->pass[pf]->g.as<int32_t>() + qf, BC, rows, s));
    HIPCHK(launch_strided_put(b->pass[pt]->g.as<int32_t>() + qt, BC, b->stage.p, rows, s));
    HIPCHK(launch_strided_get(b->stage.p, b->pass[pf]->f.as<float>() + qf, BC, cols, s));
    HIPCHK(launch_strided_put(b->pass[pt]->f.as<float>() + qt, BC, b->stage.p, cols, s));
    HIPCHK(launch_fill_u32(b->active.as<uint32_t>() + to, 1u, 1, s));
    HIPCHK(launch_fill_u32(b->active.as<uint32_t>() + from, 0u, 1, s));
    b->active_host[to] = 1;
    b->active_host[from] = 0;
    return MLEM_OK;
}

int batch_alloc_part(mlem_batch *b, uint32_t passes, uint64_t keep) {
    auto bytes = [&](const Tiled *t, const TileWorkDev *w) {
        return w->view.direct ? 0 : tiled_part_bytes(t->plan, w->view.nwg, b->BC);
    };
    const uint64_t one = std::max<uint64_t>(4, std::max(bytes(b->tfp, b->wfp), bytes(b->tbp, b->wbp)));
    // One right-hand side per pass: the blocked kernel takes one pass per launch.
    uint32_t n = b->BC == 1 ? 1u : std::max(1u, std::min(passes, kMaxPasses));
    b->part.reset();
    size_t free_b = 0;
    if (n > 1) HIPCHK(free_device_bytes(&free_b));
    while (n > 1 && n * one + keep > free_b) n = (n + 1) / 2;
    for (;; n = (n + 1) / 2) {
        const hipError_t e = b->part.alloc(n * one);
        b->group = n;
        if (e == hipSuccess) return MLEM_OK;
        if (n == 1 || e != hipErrorOutOfMemory) HIPCHK(e);
        (void)hipGetLastError();
    }
}

// The batch's tiles, work lists and partial sums.  Row slices may take more
// memory than the quads: where the batch would then find no room (in the
// budget, or on the device for all its passes) for what it holds with the
// quads, the larger ones built here are dropped and quads built instead.
static int batch_take_tiles(mlem_batch *b, uint32_t W, const uint32_t rows[2], const mlem_batch_opts &o,
                            uint64_t budget) {
    mlem_matrix *m = b->m;
    std::lock_guard<std::mutex> building(m->build_mu);
    std::set<mlem_matrix::TileKey> before;
    {
        std::lock_guard<std::mutex> lk(m->mu);
        for (const auto &t : m->tiles) before.insert(t.first);
    }
    // What the batch is still to hold: its passes, sensitivity, flags and staging vector.
    const uint64_t more = (uint64_t)b->passes * b->pass_bytes() + sizeof(float) * m->cols +
                          sizeof(uint32_t) * (uint64_t)b->passes * b->BC +
                          sizeof(float) * std::max<uint64_t>(m->rows, m->cols);
    auto build = [&](SliceUse use) -> int {
        if (int st = setup_tiled(m, 0, W, rows[0], o.values, b->BC, o.tile_groups, use, &b->tfp, &b->wfp, nullptr))
            return st;
        if (int st = setup_tiled(m, 1, W, rows[1], o.values, b->BC, o.tile_groups, use, &b->tbp, &b->wbp, nullptr))
            return st;
        // Under a budget one pass per launch: what several would add goes to requests.
        return batch_alloc_part(b, budget ? 1 : b->passes, more);
    };
    auto room = [&]() -> bool {
        if (!budget) {
            size_t free_b = 0;
            return free_device_bytes(&free_b) != hipSuccess || more <= free_b;
        }
        uint64_t held = 0;
        (void)mlem_matrix_info(m, nullptr, nullptr, nullptr, nullptr, &held);
        return held + b->part.bytes + more <= budget;
    };
    const int st = build(SliceUse::kAny);
    if (b->BC == 1 || m->tiles_only || (st != MLEM_OK && st != MLEM_ERR_OUT_OF_MEMORY)) return st;
    if (st == MLEM_OK) {
        bool larger = false;
        {
            std::lock_guard<std::mutex> lk(m->mu);
            for (const auto &t : m->tiles) larger = larger || (t.second->larger && !before.count(t.first));
        }
        if (!larger || room()) return MLEM_OK;
    }
    b->part.reset();
    {
        std::lock_guard<std::mutex> lk(m->mu);
        for (auto it = m->tiles.begin(); it != m->tiles.end();)
            it = it->second->larger && !before.count(it->first) ? m->tiles.erase(it) : std::next(it);
    }
    return build(SliceUse::kNotLarger);
}

int batch_create(mlem_matrix *m, uint32_t slots, const mlem_batch_opts *opts, uint64_t budget, mlem_batch **out) {
    ARGCHK(out, "mlem_batch_create: null out");
    *out = nullptr;
    ARGCHK(m && slots > 0, "mlem_batch_create: null matrix or no slots");
    mlem_batch_opts o;
    if (opts)
        o = *opts;
    else
        mlem_batch_opts_default(&o);
    const uint32_t BC = o.per_pass ? o.per_pass : 4u;
    ARGCHK(BC == 1 || BC == 4 || BC == 8, "mlem_batch_create: per_pass must be 1, 4 or 8");
    ARGCHK(o.values <= VAL_UF16, "mlem_batch_create: values must be 0 (f32), 1 (bf16), 2 (fp16) or 3 (uf16)");
    ARGCHK(m->has_T || m->tiles_only, "mlem_batch_create: the transpose must be resident (upload it or build it)");
    if (m->tiles_only) {
        ARGCHK(BC == m->tile_bc && (o.tile_width == 0 || o.tile_width == m->tile_W) &&
                   m->takes_rows(o.tile_rows) && (o.values == 0 || o.values == m->tile_vt),
               "mlem_batch_create: the matrix holds tiles of width %u and %u (A) and %u (A^T) rows with values %u for "
               "%u per pass",
               m->tile_W, m->tile_R[0], m->tile_R[1], m->tile_vt, m->tile_bc);
        o.tile_width = m->tile_W;
        o.values = m->tile_vt;
    }
    // Widths: 1024, 512 for 8 per pass (whose x of 1024 columns would leave
    // one workgroup per CU); default rows: setup_tiled, for FP and BP by itself.
    const uint32_t W = o.tile_width ? o.tile_width : (BC == 8 ? 512u : 1024u);
    ARGCHK(valid_tile_config(W, BC), "mlem_batch_create: no blocked kernel for width %u with %u per pass", W, BC);
    ARGCHK(o.tile_rows == 0 || valid_tile_rows(o.tile_rows),
           "mlem_batch_create: tile_rows must be 512 ... 16384 (a power of two)");
    ARGCHK(valid_stream_threads(o.tile_threads), "mlem_batch_create: tile_threads must be 0, 128, 256 or 512");
    HIPCHK(hipSetDevice(m->device));
    const uint32_t side_rows[2] = {o.tile_rows, o.tile_rows};
    auto b = std::make_unique<mlem_batch>();
    b->m = m;
    b->slots = slots;
    b->BC = BC;
    b->nt = o.tile_threads;
    b->use_graph = o.use_graph != 0;
    b->passes = (slots + BC - 1) / BC;
    b->rows_x = (m->rows + kTileXPad - 1) / kTileXPad * kTileXPad + kTileXPad;
    b->cols_x = (m->cols + kTileXPad - 1) / kTileXPad * kTileXPad + kTileXPad;
    HIPCHK(hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking));
    if (int st = batch_take_tiles(b.get(), W, m->tiles_only ? m->tile_R : side_rows, o, budget)) return st;
    if (b->tfp->ordered != b->tbp->ordered)  // a row order set from another thread between the two builds
        return set_err(MLEM_ERR_INVALID_ARGUMENT, "mlem_batch_create: the row order changed while the tiles were built");
    if (b->tfp->ordered) b->row_order = m->row_order.as<uint32_t>();
    const size_t per = (size_t)BC * b->passes;
    b->pass.resize(b->passes);  // passes are allocated when first used (batch_set_async)
    HIPCHK(b->sens.alloc(sizeof(float) * m->cols));
    HIPCHK(b->active.alloc(sizeof(uint32_t) * per));
    HIPCHK(b->stage.alloc(sizeof(float) * std::max<size_t>(1, std::max(m->rows, m->cols))));
    HIPCHK(launch_fill_u32(b->active.as<uint32_t>(), 0u, per, b->stream));
    b->active_host.assign(per, 0);
    if (o.values != VAL_F32)  // the quantized matrix's own sensitivity
        HIPCHK(hipMemcpyAsync(b->sens.p, b->tbp->sens.p, sizeof(float) * m->cols, hipMemcpyDeviceToDevice,
                              b->stream));
    else if (int st = sens_on_device(m, b->sens.as<float>(), nullptr, b->stream))
        return st;
    HIPCHK(hipStreamSynchronize(b->stream));
    (void)scratch_trim();
    m->users.fetch_add(1);
    *out = b.release();
    return MLEM_OK;
}

uint64_t batch_release_pass(mlem_batch *b, uint32_t p) {
    if (!b || p >= b->passes || !b->pass[p]) return 0;
    for (uint32_t q = 0; q < b->BC; ++q)
        if (b->active_host[(size_t)p * b->BC + q]) return 0;
    if (hipSetDevice(b->m->device) != hipSuccess || hipStreamSynchronize(b->stream) != hipSuccess) return 0;
    const uint64_t bytes = b->pass[p]->g.bytes + b->pass[p]->ratio.bytes + b->pass[p]->f.bytes;
    drop_graph(b);
    b->pass[p].reset();
    return bytes;
}

}  // namespace abi
}  // namespace mlem

// -------------------------------------------------------------- autotuner
namespace {

// The stream and events that candidates are timed with.
struct TuneClock {
    hipStream_t s = nullptr;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    ~TuneClock() {
        if (s) (void)hipStreamSynchronize(s);
        if (e0) (void)hipEventDestroy(e0);
        if (e1) (void)hipEventDestroy(e1);
        if (s) (void)hipStreamDestroy(s);
    }
};

// Times the candidates `passes` passes at a time; *short_of_memory: one of
// them, or the vectors, did not fit (with several passes nothing further is
// timed then).
int tune(mlem_matrix *m, uint32_t BC, uint32_t values, uint32_t passes, SliceUse use, mlem_tune_result *out,
         bool *short_of_memory) {
    int dev = 0, cus_i = 256;
    if (hipGetDevice(&dev) == hipSuccess)
        (void)hipDeviceGetAttribute(&cus_i, hipDeviceAttributeMultiprocessorCount, dev);
    const uint32_t cus = (uint32_t)std::max(1, cus_i);
    std::vector<std::pair<uint32_t, uint32_t>> shapes;  // (W, R)
    if (BC == 1)
        shapes = {{1024, 1024}, {1024, 2048}, {1024, 4096}, {2048, 1024}, {2048, 2048}};
    else if (BC == 4)
        shapes = {{512, 1024}, {1024, 512}, {1024, 1024}, {1024, 2048}, {512, 2048}};
    else
        shapes = {{512, 512}, {512, 1024}};
    const size_t rows_x = ((size_t)m->rows + kTileXPad - 1) / kTileXPad * kTileXPad + kTileXPad;
    const size_t cols_x = ((size_t)m->cols + kTileXPad - 1) / kTileXPad * kTileXPad + kTileXPad;
    DevBuf xf, xb, yf, yb;
    for (auto v : {std::make_pair(&xf, cols_x), std::make_pair(&xb, rows_x), std::make_pair(&yf, rows_x),
                   std::make_pair(&yb, cols_x)}) {
        const hipError_t e = v.first->alloc(sizeof(float) * v.second * BC * passes);
        *short_of_memory = *short_of_memory || e == hipErrorOutOfMemory;
        HIPCHK(e);
    }
    TuneClock c;
    HIPCHK(hipStreamCreateWithFlags(&c.s, hipStreamNonBlocking));
    HIPCHK(hipEventCreate(&c.e0));
    HIPCHK(hipEventCreate(&c.e1));
    HIPCHK(launch_fill(xf.as<float>(), 1.0f, cols_x * BC * passes, c.s));
    HIPCHK(launch_fill(xb.as<float>(), 1.0f, rows_x * BC * passes, c.s));
    // One side's time per launch (partials + reduce), mean of three after a warm-up.
    auto time_side = [&](const Tiled *t, const TileWorkDev *w, const DevBuf &part, const float *x, size_t x_pass,
                         float *y, uint32_t nt, double *ms) -> int {
        PassX px{};
        PassEpi pe{};
        for (uint32_t k = 0; k < passes; ++k) {
            px.x[k] = x + k * x_pass * BC;
            pe.ea[k].out = y + k * (size_t)t->plan.rows * BC;
        }
        px.n = pe.n = passes;
        for (int rep = 0; rep < 4; ++rep) {
            if (rep == 1) HIPCHK(hipEventRecord(c.e0, c.s));
            HIPCHK(launch_tiled_spmv(t->plan, t->view, w->view, px, part.as<float>(), BC, nt, EPI_PLAIN, pe, c.s));
        }
        HIPCHK(hipEventRecord(c.e1, c.s));
        HIPCHK(hipEventSynchronize(c.e1));
        float f = 0.0f;
        HIPCHK(hipEventElapsedTime(&f, c.e0, c.e1));
        *ms = f / 3.0;
        return MLEM_OK;
    };
    double best = 1e300;
    bool sliced = false;  // a shape kept both sides as row slices
    for (const auto &sh : shapes) {
        const uint32_t W = sh.first, R = sh.second;
        if (W == 512 && R == 2048 && sliced) continue;  // too tall for slices
        // The automatic runs where they are one per row block for a side.
        const bool direct = BC != 1 && (slices_direct(m->cols, W, R, m->rows, m->nnz, BC) ||
                                        slices_direct(m->rows, W, R, m->cols, m->nnz, BC));
        std::vector<uint32_t> groups;  // per CU, 0: automatic
        if (BC == 1) {
            groups = {16, 24, 32};
            if (default_tile_groups(m->nnz, values, 1) == 12 * cus) groups.push_back(12);
        } else if (W == 1024 && R == 512) {
            if (!direct) continue;  // small tiles pay where whole blocks are runs
            groups = {0};
        } else {
            groups = {4, 8, 16};
            if (direct) groups.push_back(0);
        }
        for (uint32_t g : groups) {
            const Tiled *t[2] = {};
            const TileWorkDev *w[2] = {};
            DevBuf part;  // FP and BP in turn
            int st = MLEM_OK;
            for (int side = 0; side < 2 && st == MLEM_OK; ++side)
                st = setup_tiled(m, side, W, R, values, BC, g * cus, use, &t[side], &w[side], nullptr);
            const bool slices = st == MLEM_OK && t[0]->plan.slices && t[1]->plan.slices;
            sliced = sliced || slices;
            if (slices && g == 16) continue;  // more runs than pay: 4 per CU beat 8 (default_tile_groups)
            if (st == MLEM_OK) {
                const hipError_t e = part.alloc(passes * std::max(tiled_part_bytes(t[0]->plan, w[0]->view.nwg, BC),
                                                                  tiled_part_bytes(t[1]->plan, w[1]->view.nwg, BC)));
                if (e == hipErrorOutOfMemory)
                    st = MLEM_ERR_OUT_OF_MEMORY;
                else
                    HIPCHK(e);
            }
            if (st == MLEM_ERR_OUT_OF_MEMORY) {
                *short_of_memory = true;
                if (passes > 1) return st;
            }
            if (st == MLEM_ERR_UNSUPPORTED || st == MLEM_ERR_OUT_OF_MEMORY) continue;  // does not suit or fit the matrix
            if (st != MLEM_OK) return st;
            // Work-items per workgroup of the block streams (128 was slower at
            // every shape timed on the 3D scanner matrix).
            for (uint32_t nt : {256u, 512u}) {
                if ((BC == 1 || slices) && nt != 512) continue;  // without effect
                double fp = 0, bp = 0;
                st = time_side(t[0], w[0], part, xf.as<float>(), cols_x, yf.as<float>(), BC == 1 ? 0 : nt, &fp);
                if (st == MLEM_OK)
                    st = time_side(t[1], w[1], part, xb.as<float>(), rows_x, yb.as<float>(), BC == 1 ? 0 : nt, &bp);
                if (st != MLEM_OK) return st;
                ++out->candidates;
                if (fp + bp < best) {
                    best = fp + bp;
                    out->tile_width = W;
                    out->tile_rows = R;
                    out->tile_groups = g * cus;
                    out->tile_threads = BC == 1 ? 0 : nt;
                    out->fp_ms = fp;
                    out->bp_ms = bp;
                }
            }
        }
    }
    return MLEM_OK;
}

}  // namespace

extern "C" {

// Times the blocked kernels of both sides over a few tile shapes and
// workgroup counts and reports the fastest.  Candidate tiles that did not
// exist before and were not chosen are freed again.
int mlem_autotune(mlem_matrix *m, uint32_t per_pass, uint32_t values, mlem_tune_result *out) {
    ARGCHK(m && out, "mlem_autotune: null argument");
    std::memset(out, 0, sizeof(*out));
    const uint32_t BC = per_pass ? per_pass : 1u;
    ARGCHK(BC == 1 || BC == 4 || BC == 8, "mlem_autotune: per_pass must be 1, 4 or 8");
    ARGCHK(values <= VAL_UF16, "mlem_autotune: values must be 0 (f32), 1 (bf16), 2 (fp16) or 3 (uf16)");
    ARGCHK(m->has_T, "mlem_autotune: the transpose must be resident");
    HIPCHK(hipSetDevice(m->device));
    std::lock_guard<std::mutex> building(m->build_mu);
    std::set<mlem_matrix::TileKey> before;
    {
        std::lock_guard<std::mutex> lk(m->mu);
        for (const auto &t : m->tiles) before.insert(t.first);
    }
    auto drop_others = [&]() {
        std::lock_guard<std::mutex> lk(m->mu);
        for (auto it = m->tiles.begin(); it != m->tiles.end();) {
            const auto &k = it->first;
            const bool chosen = out->candidates && std::get<1>(k) == out->tile_width &&
                                std::get<2>(k) == out->tile_rows && std::get<3>(k) == values &&
                                std::get<4>(k) == (BC > 1);
            it = (!before.count(k) && !chosen) ? m->tiles.erase(it) : std::next(it);
        }
    };
    // Batches of several passes share their launches, and taller tiles pay
    // then (683 M entries, one pass of 4 equal at 1024 and 2048 rows, four
    // 4110 against 3600 us): they are timed four passes at a time, each with
    // its own vectors, or one where that does not fit.
    bool short_of_memory = false;
    int st = tune(m, BC, values, BC == 1 ? 1u : 4u, SliceUse::kAny, out, &short_of_memory);
    if (short_of_memory && BC != 1) {
        std::memset(out, 0, sizeof(*out));
        drop_others();
        st = tune(m, BC, values, 1, SliceUse::kNotLarger, out, &short_of_memory);
    }
    drop_others();
    (void)scratch_trim();
    if (st != MLEM_OK) return st;
    if (!out->candidates) return set_err(MLEM_ERR_UNSUPPORTED, "mlem_autotune: no tile shape suits or fits this matrix");
    return MLEM_OK;
}

// ---------------------------------------------------------------- batches
void mlem_batch_opts_default(mlem_batch_opts *o) {
    if (!o) return;
    std::memset(o, 0, sizeof(*o));
    o->per_pass = 4;
}

int mlem_batch_create(mlem_matrix *m, uint32_t slots, const mlem_batch_opts *opts, mlem_batch **out) {
    return batch_create(m, slots, opts, 0, out);
}

int mlem_batch_set(mlem_batch *b, uint32_t slot, const int32_t *g, const float *f0) {
    if (int st = batch_set_async(b, slot, g, f0, nullptr)) return st;
    HIPCHK(hipStreamSynchronize(b->stream));  // g and f0 may be freed after the return
    return MLEM_OK;
}

int mlem_batch_deactivate(mlem_batch *b, uint32_t slot) { return batch_deactivate_async(b, slot); }

int mlem_batch_iterate(mlem_batch *b, uint32_t iters) {
    ARGCHK(b, "mlem_batch_iterate: null handle");
    if (!b->part.p) return set_err(MLEM_ERR_OUT_OF_MEMORY, "mlem_batch_iterate: the batch has lost its partial sums");
    HIPCHK(hipSetDevice(b->m->device));
    const uint32_t BC = b->BC;
    std::vector<uint8_t> passes(b->passes, 0);
    bool any = false;
    for (uint32_t p = 0; p < b->passes; ++p) {
        for (uint32_t q = 0; q < BC; ++q) passes[p] = passes[p] || b->active_host[(size_t)p * BC + q];
        any = any || passes[p];
    }
    if (!any || iters == 0) return MLEM_OK;
    if (!b->use_graph) {
        for (uint32_t it = 0; it < iters; ++it)
            if (int st = enqueue_batch_iteration(b, passes)) return st;
        return MLEM_OK;
    }
    if (!b->gexec || passes != b->graph_passes) {  // (re)capture for this set of passes
        if (b->gexec) {
            HIPCHK(hipStreamSynchronize(b->stream));
            HIPCHK(hipGraphExecDestroy(b->gexec));
            b->gexec = nullptr;
        }
        HIPCHK(hipStreamBeginCapture(b->stream, hipStreamCaptureModeThreadLocal));
        const int st = enqueue_batch_iteration(b, passes);
        hipGraph_t gr = nullptr;
        const hipError_t e2 = hipStreamEndCapture(b->stream, &gr);
        if (st != MLEM_OK) {
            if (gr) (void)hipGraphDestroy(gr);
            return st;
        }
        HIPCHK(e2);
        const hipError_t e3 = hipGraphInstantiate(&b->gexec, gr, nullptr, nullptr, 0);
        (void)hipGraphDestroy(gr);
        HIPCHK(e3);
        b->graph_passes = passes;
    }
    for (uint32_t it = 0; it < iters; ++it) HIPCHK(hipGraphLaunch(b->gexec, b->stream));
    return MLEM_OK;
}

int mlem_batch_sync(mlem_batch *b) {
    ARGCHK(b, "mlem_batch_sync: null handle");
    HIPCHK(hipSetDevice(b->m->device));
    HIPCHK(hipStreamSynchronize(b->stream));
    return MLEM_OK;
}

int mlem_batch_get_image(mlem_batch *b, uint32_t slot, float *f_out) {
    if (int st = batch_get_image_async(b, slot, f_out)) return st;
    HIPCHK(hipStreamSynchronize(b->stream));
    return MLEM_OK;
}

int mlem_batch_info(const mlem_batch *b, uint32_t *slots, uint32_t *per_pass, uint32_t *passes,
                    uint64_t *device_bytes) {
    ARGCHK(b, "mlem_batch_info: null handle");
    if (slots) *slots = b->slots;
    if (per_pass) *per_pass = b->BC;
    if (passes) *passes = b->passes;
    if (device_bytes) *device_bytes = b->device_bytes();
    return MLEM_OK;
}

int mlem_batch_layout(const mlem_batch *b, int side, mlem_tile_layout *out) {
    ARGCHK(b && out && (side == 0 || side == 1), "mlem_batch_layout: null argument or a side that is not 0 or 1");
    const Tiled *t = side ? b->tbp : b->tfp;
    const TileWorkDev *w = side ? b->wbp : b->wfp;
    const TilePlan &p = t->plan;
    out->kind = !p.quad ? 0u : !p.slices ? 1u : w->view.direct ? 3u : 2u;
    out->tile_width = p.W;
    out->tile_rows = p.R;
    out->runs = w->view.nwg;
    out->max_steps = p.slices ? p.most : 0u;
    out->entries = p.cap - 8;
    out->bytes = t->mem.bytes;
    return MLEM_OK;
}

void *mlem_batch_stream(mlem_batch *b) { return b ? b->stream : nullptr; }

int mlem_batch_destroy(mlem_batch *b) {
    if (!b) return MLEM_OK;
    (void)hipSetDevice(b->m->device);
    b->m->users.fetch_sub(1);
    delete b;
    return MLEM_OK;
}

}  // extern "C"
