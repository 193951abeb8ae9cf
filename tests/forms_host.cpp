// Host replay of the forms that the launchers of flux-interpolated-advection_amd/csrc/fia_kernels.hip
// choose by size and rule, where pass_host.cpp replays one form for every size.  The same __host__
// __device__ code that the kernels compile, driven the way the kernels drive it:
//   - WENO6 displacements by marched tiles (VertexMarch), with the kernel's buffer of z passes;
//   - the zero-velocity march in chunks of x planes, and the other zero-velocity kernels' rules;
//   - degenerate faces shared over lanes;
//   - the z stencil tables, and the table quadrature by bricks: rows of slots, box, staging, and the
//     pieces that read the box or the table; the quadrature of slots in parts (launch_slots);
//   - twisted faces' pieces in fixed records, and counted where those do not hold them.
// Not replayed: the scan kernels and the count kernels' sums (a plain scan here), the psi kernels' held
// columns (psi_body), and what one block's threads exchange through LDS or lane shuffles beyond the
// buffers named above.
//
// Fields, psi and tables lie in buffers with guards of 0xFF bytes (NaN) before and after, and the
// buffers themselves start as 0xFF: a read out of range or of an entry that nothing wrote makes the
// result NaN.  Each pass checks that the bricks visit every slot once.  Built by tests/test_forms_host.py
// with hipcc (optionally with AddressSanitizer); only the host code runs.
#include "pass_host.cpp"

namespace {

constexpr size_t kGuard = 4096;
template <class T> struct Guarded {
    std::vector<unsigned char> raw;
    T *p = nullptr;
    size_t n = 0;
    T *fill(size_t want) {
        raw.assign((want + 2 * kGuard) * sizeof(T) + alignof(T), 0xFF);
        const size_t at = (size_t)(raw.data() + kGuard * sizeof(T));
        p = (T *)((at + alignof(T) - 1) / alignof(T) * alignof(T));
        n = want;
        return p;
    }
    const T *copy(const T *from, size_t want) {
        memcpy((void *)fill(want), from, want * sizeof(T));
        return p;
    }
    bool guards_whole() const {
        const unsigned char *b = raw.data(), *e = b + raw.size(), *lo = (const unsigned char *)p,
                            *hi = (const unsigned char *)(p + n);
        return std::all_of(b, lo, [](unsigned char c) { return c == 0xFF; }) &&
               std::all_of(hi, e, [](unsigned char c) { return c == 0xFF; });
    }
};

enum { FS_TWISTED, FS_DEGEN, FS_SLOTS, FS_GEN_OVER, FS_TABLES, FS_BOX, FS_MEMORY, FS_GEN_MAX, kFormCols };

struct FormsCtx : HostCtx {
    Guarded<WenoHalf> tab[2];
    Guarded<float> disp_out[3];
    std::vector<double> forms;
};

struct Options {
    int weno_opt, tables;   // tables: 0 by the launcher's rule, 1 always, -1 never
    int zero_chunk;         // planes a chunk, 0: the launcher's
};

bool vertices_forms(FormsCtx &c, const CompGrid &g, const float *u, const float *v, const float *w, double dt_over_h,
                    int interp) {
    VertexParams p;
    memset(&p, 0, sizeof(p));
    p.g = g; p.u = u; p.v = v; p.w = w; p.dt_over_h = (float)dt_over_h; p.interp = interp;
    for (int a = 0; a < 3; ++a) p.disp[a] = c.disp_out[a].fill(g.lattice());
    if (interp == IM_WENO6) {
        const VertexTiles t(g);
        const WenoCoef wc(0.5f, 1.0f);
        constexpr int kThreads = kVtxTile * kVtxTile;
        parallel_for((long)t.blocks * 3, [&](long b) {
            std::vector<float> zs[2];
            for (auto &z : zs) z.assign((kVtxTile + 5) * kVtxTile, NAN);
            std::vector<VertexMarch> th;
            for (int tid = 0; tid < kThreads; ++tid)
                th.emplace_back(p, (int)(b % 3), (int)(b / 3), t.ty, t.tz, (int)t.chunk, tid);
            float yv[kThreads][6] = {};
            const VertexMarch &m = th[0];
            for (int pl = 0; pl < m.planes; ++pl) {
                std::vector<float> &rows = zs[pl & 1];
                float val[kThreads];
                for (int tid = 0; tid < kThreads; ++tid) {
                    const VertexMarch &h = th[tid];
                    const float *plane = h.plane(p, pl);
                    if (!(h.half[2] || h.half[1])) { val[tid] = plane[h.off[0]]; continue; }
                    val[tid] = h.pass(plane, 0u, wc);
                    if (!h.zy) continue;
                    rows[tid] = val[tid];
                    if (h.second) rows[tid + kThreads] = h.pass(plane, h.step, wc);
                }
                for (int tid = 0; tid < kThreads; ++tid) {
                    const VertexMarch &h = th[tid];
                    if (h.zy) val[tid] = VertexMarch::rows_pass(rows.data(), tid, wc);
                    if (h.x_pass(yv[tid], pl, val[tid], wc)) h.store(p, pl, val[tid]);
                }
            }
        });
    } else {
        parallel_for((long)g.lattice(), [&](long id) {
            if (interp == IM_LINEAR) vertex_body<IM_LINEAR>(p, id);
            else if (interp == IM_1DY_LINEAR) vertex_body<IM_1DY_LINEAR>(p, id);
            else vertex_body<-1>(p, id);
        });
    }
    for (int a = 0; a < 3; ++a)
        if (!c.disp_out[a].guards_whole()) {
            snprintf(c.msg, sizeof(c.msg), "displacements stored out of range");
            return false;
        }
    return true;
}

// the table quadrature of every slot, brick by brick; false with c.msg set if the bricks miss one
template <bool OPT> bool bricks_forms(FormsCtx &c, FaceParams &p, unsigned long long nslots, double st[kFormCols]) {
    const CompGrid &g = p.g;
    const long len = g.m[2] + kWenoPad, rq = (long)g.m[0] * g.m[1], rp = (long)g.m[0] * (g.m[1] + 1);
    WenoHalf *qt = c.tab[0].fill((size_t)(2 * rq * len)), *pt = c.tab[1].fill((size_t)(2 * rp * len));
    const long past = kBlock - 1;   // the last block's threads past the table
    parallel_for(rq * len + past, [&](long id) { weno_table_body<float, OPT>(p.q, rq, g.m[2], (double)p.kappa_q, qt, id); });
    parallel_for(rp * len + past, [&](long id) { weno_table_body<double, OPT>(p.psi, rp, g.m[2], (double)p.kappa_psi, pt, id); });
    if (!c.tab[0].guards_whole() || !c.tab[1].guards_whole()) {
        snprintf(c.msg, sizeof(c.msg), "table entries stored out of range");
        return false;
    }
    p.q_tab = qt; p.psi_tab = pt;
    const Bricks br(g);
    std::vector<unsigned char> seen(nslots, 0);
    std::atomic<long> boxed{0}, memory{0}, bad{0};
    parallel_for((long)br.count(), [&](long brick) {
        const BrickCells cells(g, br, (int)brick);
        int range[6] = {INT32_MAX, INT32_MAX, INT32_MAX, INT32_MIN, INT32_MIN, INT32_MIN};
        for (int t = 0; t < cells.vertices(); ++t) {
            int b[3];
            cells.bases(p, t, b);
            for (int a = 0; a < 3; ++a) {
                range[a] = std::min(range[a], b[a]);
                range[3 + a] = std::max(range[3 + a], b[a]);
            }
        }
        const BrickBox box(range, g.m[2]);
        std::vector<WenoHalf> win((size_t)kWinX * kWinY * 2 * kWinZ, WenoHalf{NAN, NAN, NAN, NAN});
        for (int t = 0; t < box.halves(); ++t) {
            int to;
            size_t from;
            if (!box.half_entry(g, t, to, from)) continue;
            if (to < 0 || (size_t)to >= win.size() || from >= c.tab[0].n) { ++bad; continue; }
            win[to] = qt[from];
        }
        unsigned long long start = 0;
        unsigned n = 0;
        const int rows = cells.rows(p, 0, start, n);
        if (rows > kBrickRows) ++bad;
        for (int r = 0; r < rows; ++r) {
            cells.rows(p, r, start, n);
            for (unsigned long long q = start; q < start + n; ++q) {
                if (q >= nslots || seen[q]++) { ++bad; continue; }
                const double ay = p.piece_ay[q];
                double val = 0.0;
                if (ay != 0.0) {
                    const double c3[3] = {p.piece_c[0][q], p.piece_c[1][q], p.piece_c[2][q]};
                    const PiecePoint t = piece_point<OPT>(p, c3);
                    const int at = box.corner(t, g.m[2]);
                    val = at >= 0 ? piece_flux_box<OPT>(p, t, ay, win.data() + at) : piece_flux_memory<OPT>(p, t, ay);
                    ++(at >= 0 ? boxed : memory);
                }
                p.piece_val[q] = val;
            }
        }
    });
    const long missed = (long)std::count(seen.begin(), seen.end(), 0);
    if (bad || missed) {
        snprintf(c.msg, sizeof(c.msg), "bricks: %ld bad entries, %ld slots of %llu missed", bad.load(), missed, nslots);
        return false;
    }
    st[FS_TABLES] = 1; st[FS_BOX] = (double)boxed; st[FS_MEMORY] = (double)memory;
    return true;
}

template <int RULE> void zero_forms(const FaceParams &p) {
    parallel_for((long)p.g.faces(1), [&](long id) { zero_velocity_face_body<false, RULE>(p, id); });
}

// do_faces of fia_api.hip with its launchers' forms
int faces_forms(FormsCtx &c, const CompGrid &g, const float *q, const double *psi, bool moving, FluxSetH &fs,
                const PassSpec &s, int fam_mask, double h, const Options &o) {
    double st[kFormCols] = {0};
    for (int f = 0; f < 3; ++f) {
        fs.f[f].ensure(g.faces(f));
        fs.c[f].ensure(g.faces(f));
        fs.m[f].ensure((fs.c[f].n + 31) / 32);
        memset((void *)fs.c[f].p, 0, fs.c[f].n * sizeof(double));
        memset((void *)fs.m[f].p, 0, fs.m[f].n * sizeof(unsigned));
    }
    const size_t nf = g.faces(0) + g.faces(1) + g.faces(2);
    c.twisted.ensure(nf);
    c.degen.ensure(nf);
    c.counters[0] = 0; c.counters[2] = 0;
    FaceParams p;
    memset(&p, 0, sizeof(p));
    p.g = g; p.q = q; p.psi = psi;
    for (int a = 0; a < 3; ++a) {
        p.disp[a] = moving ? c.disp_out[a].p : nullptr;
        p.flux[a] = fs.f[a].p;
        p.corr[a] = fs.c[a].p;
        p.corr_mask[a] = fs.m[a].p;
    }
    p.twisted = c.twisted.p; p.twisted_count = &c.counters[0]; p.error = &c.counters[1];
    p.degen = c.degen.p; p.degen_count = &c.counters[2];
    p.split = s.split; p.interp = s.interp; p.weno_opt = o.weno_opt; p.integral = s.integral; p.fam_mask = fam_mask;
    p.general_all = s.min_area < 1.0;
    p.fuse_value = !p.integral && (p.interp == FIA_INTERP_LINEAR || p.interp == FIA_INTERP_1DY_LINEAR);
    p.kappa_q = 1.0f;
    p.kappa_psi = (float)(h * h);
    p.min_area = s.min_area;
    p.gauss = gauss_table(s.ng);
    auto done = [&]() {
        c.forms.insert(c.forms.end(), st, st + kFormCols);
        return c.counters[1];
    };
    if (!moving && !p.general_all) {   // launch_zero_velocity_faces
        if (p.interp == IM_WENO6 && !p.weno_opt && !p.integral && zero_velocity_cuts_both(p)) {
            const int chunk = o.zero_chunk > 0 ? o.zero_chunk : (int)zero_velocity_chunk(g, kBlock), nx = g.m[0];
            parallel_for((long)(g.m[1] + 1) * g.m[2], [&](long row) {
                for (int i0 = 0; i0 < nx; i0 += chunk) zero_velocity_weno(p, (unsigned)row, i0, std::min(nx, i0 + chunk));
            });
        } else if (p.fuse_value) {
            zero_forms<kZeroValue>(p);
        } else {
            switch (p.interp == IM_WENO6 && p.weno_opt ? (int)IM_WENO6_OPT : p.interp) {
            case IM_LINEAR: zero_forms<IM_LINEAR>(p); break;
            case IM_WENO6: zero_forms<IM_WENO6>(p); break;
            case IM_1DY_LINEAR: zero_forms<IM_1DY_LINEAR>(p); break;
            case IM_1DY_WENO6: zero_forms<IM_1DY_WENO6>(p); break;
            default: zero_forms<IM_WENO6_OPT>(p); break;
            }
        }
        return done();
    }
    c.face_n.ensure(nf);
    c.face_start.ensure(nf);
    p.face_n = c.face_n.p;
    p.face_start = c.face_start.p;
    p.fam_base[0] = 0; p.fam_base[1] = g.faces(0); p.fam_base[2] = g.faces(0) + g.faces(1);
    parallel_for((long)g.faces(0), [&](long id) { face_count_body<0>(p, id); });
    parallel_for((long)g.faces(1), [&](long id) { face_count_body<1>(p, id); });
    parallel_for((long)g.faces(2), [&](long id) { face_count_body<2>(p, id); });
    const int n_twisted = c.counters[0], n_degen = c.counters[2];
    unsigned long long nslots = 0;
    for (size_t k = 0; k < nf; ++k) {
        c.face_start.p[k] = nslots;
        nslots += c.face_n.p[k];
    }
    for (int a = 0; a < 3; ++a) c.piece_c[a].ensure(nslots);
    c.piece_ay.ensure(nslots);
    c.piece_val.ensure(nslots);
    for (int a = 0; a < 3; ++a) p.piece_c[a] = c.piece_c[a].p;
    p.piece_ay = c.piece_ay.p;
    p.piece_val = c.piece_val.p;
    // twisted faces: kGenStride records a pair
    int over = GEN_FITS;
    bool strided = n_twisted > 0 && !p.general_all;
    const size_t pairs = 2 * (size_t)n_twisted;
    auto records = [&](size_t n) {
        for (int a = 0; a < 3; ++a) c.gen_c[a].ensure(n);
        c.gen_ay.ensure(n);
        c.gen_val.ensure(n);
        for (int a = 0; a < 3; ++a) p.gen_c[a] = c.gen_c[a].p;
        p.gen_ay = c.gen_ay.p;
        p.gen_val = c.gen_val.p;
    };
    if (strided) {
        c.gen_n.ensure(pairs);
        p.gen_n = c.gen_n.p;
        records(pairs * kGenStride);
        p.gen_stride = kGenStride;
        p.gen_over = &over;
        for (size_t k = 0; k < pairs; ++k) general_emit_pair(p, (int)(k >> 1), (int)(k & 1));
        if (over == GEN_FAILED) return c.counters[1];
    }
    auto seg = [&](auto famc, long id) {
        constexpr int F = decltype(famc)::value;
        const unsigned n = seg_face_body<F>(p, id);
        for (unsigned l = 0; l < n; ++l) seg_piece_body<F>(p, id, l);
    };
    if (fam_mask & 1) parallel_for((long)g.faces(0), [&](long id) { seg(std::integral_constant<int, 0>(), id); });
    if (fam_mask & 2) parallel_for((long)g.faces(1), [&](long id) { seg(std::integral_constant<int, 1>(), id); });
    if (fam_mask & 4) parallel_for((long)g.faces(2), [&](long id) { seg(std::integral_constant<int, 2>(), id); });
    const int lanes = 1 << face_share(n_degen);
    parallel_for((long)n_degen * lanes, [&](long t) { degenerate_pieces(p, (int)(t / lanes), (int)(t % lanes), lanes); });
    if (p.fuse_value) parallel_for(n_degen, [&](long t) { degenerate_value_body(p, (int)t); });
    else {
        size_t psi_halves = 0;
        const int qm = piece_quadrature_mode(p);
        const bool tables = qm == 1 && (o.tables > 0 || (o.tables == 0 && weno_table_halves(p, psi_halves) > 0));
        if (tables) {
            if (!(p.weno_opt ? bricks_forms<true>(c, p, nslots, st) : bricks_forms<false>(c, p, nslots, st))) return -1;
        } else {
            // launch_slots, in parts of a thousand slots
            constexpr unsigned long long kPart = 1009;
            parallel_for((long)((nslots + kPart - 1) / kPart), [&](long k) {
                const unsigned long long first = (unsigned long long)k * kPart, n = std::min(kPart, nslots - first);
                const FaceParams part = slots_from(p, first);
                for (unsigned long long slot = 0; slot < n; ++slot) {
                    int a = 0, b = 0, e = 0;
                    if (qm == 1 && p.weno_opt) piece_body<1, true>(part, slot, a, b, e);
                    else if (qm == 1) piece_body<1>(part, slot, a, b, e);
                    else if (qm == 2 && p.weno_opt) piece_body<2, true>(part, slot, a, b, e);
                    else if (qm == 2) piece_body<2>(part, slot, a, b, e);
                    else if (p.interp == IM_LINEAR) piece_body<kPieceLinear>(part, slot, a, b, e);
                    else piece_body<0>(part, slot, a, b, e);
                }
            });
        }
    }
    if (fam_mask & 1) parallel_for((long)g.faces(0), [&](long id) { face_sum_body<0>(p, id); });
    if (fam_mask & 2) parallel_for((long)g.faces(1), [&](long id) { face_sum_body<1>(p, id); });
    if (fam_mask & 4) parallel_for((long)g.faces(2), [&](long id) { face_sum_body<2>(p, id); });
    if (n_twisted > 0) {
        unsigned long long npieces = pairs * kGenStride;
        if (over == GEN_MORE) strided = false;
        if (!strided) {   // counted first
            c.gen_n.ensure(pairs);
            c.gen_start.ensure(pairs + 1);
            p.gen_stride = 0;
            p.gen_n = c.gen_n.p;
            p.gen_start = c.gen_start.p;
            for (size_t k = 0; k < pairs; ++k) general_count_pair(p, (int)(k >> 1), (int)(k & 1));
            if (c.counters[1] != 0) return c.counters[1];
            npieces = 0;
            for (size_t k = 0; k < pairs; ++k) {
                c.gen_start.p[k] = npieces;
                npieces += c.gen_n.p[k];
            }
            c.gen_start.p[pairs] = npieces;
            records(npieces);
            for (size_t k = 0; k < pairs; ++k) general_emit_pair(p, (int)(k >> 1), (int)(k & 1));
        }
        for (size_t k = 0; k < pairs; ++k) st[FS_GEN_MAX] = std::max(st[FS_GEN_MAX], (double)c.gen_n.p[k]);
        parallel_for((long)npieces, [&](long k) { general_piece_body(p, (unsigned long long)k); });
        parallel_for(n_twisted, [&](long t) { general_sum_body(p, (int)t); });
    }
    st[FS_TWISTED] = n_twisted; st[FS_DEGEN] = n_degen; st[FS_SLOTS] = (double)nslots; st[FS_GEN_OVER] = over;
    return done();
}

const double *psi_forms(FormsCtx &c, Guarded<double> &buf, const CompGrid &g, const float *q, int mode, int integral,
                        int ng) {
    PsiParams p;
    memset(&p, 0, sizeof(p));
    p.g = g; p.q = q; p.psi = buf.fill(g.psi_size()); p.mode = mode; p.integral = integral; p.kappa = 1.0f;
    p.gauss = gauss_table(ng);
    parallel_for((long)g.m[0] * g.m[2], [&](long col) { psi_body(p, col); });
    return buf.p;
}

struct Fields {
    Guarded<float> u, v, w, q;
    Guarded<double> psi;
    Fields(const CompGrid &g, const float *u_, const float *v_, const float *w_, const float *q_) {
        const size_t nx = g.n[0], ny = g.n[1], nz = g.n[2];
        u.copy(u_, (nx + 1) * ny * nz);
        v.copy(v_, nx * (ny + 1) * nz);
        w.copy(w_, nx * ny * (nz + 1));
        q.copy(q_, g.cells());
    }
};

int forms_step(FormsCtx &c, const CompGrid &g, const float *q_in, float *out, const float *u, const float *v, const float *w,
               double h, double dt, int interp, int use_integral, int ng, double min_area, int split_main, int split_err,
               const Options &o) {
    Fields f(g, u, v, w, q_in);
    int integral = use_integral ? 1 : 0, e;
    const int pm = psi_mode_for(interp, integral);
    PassSpec p1{split_main, interp, pm, 0, integral, ng, min_area};
    const double *psi = psi_forms(c, f.psi, g, f.q.p, p1.psi_mode, p1.integral, p1.ng);
    if (!vertices_forms(c, g, f.u.p, f.v.p, f.w.p, dt / h, p1.interp)) return -1;
    if ((e = faces_forms(c, g, f.q.p, psi, true, c.fsa, p1, 7, h, o)) != 0) return e;
    PassSpec p2{split_main, interp, FIA_PSI_CONST, 1, 0, ng, min_area};
    psi = psi_forms(c, f.psi, g, f.q.p, p2.psi_mode, p2.integral, p2.ng);
    if ((e = faces_forms(c, g, f.q.p, psi, false, c.fsb, p2, 2, h, o)) != 0) return e;
    Guarded<float> err;
    gather(g, c.fsb, nullptr, f.q.p, err.fill(g.cells()), 2, 2);
    PassSpec p3{split_err, FIA_INTERP_1DY_LINEAR, FIA_PSI_CONST, 0, 0, ng, min_area};
    psi = psi_forms(c, f.psi, g, err.p, p3.psi_mode, p3.integral, p3.ng);
    if (!vertices_forms(c, g, f.u.p, f.v.p, f.w.p, dt / h, p3.interp)) return -1;
    if ((e = faces_forms(c, g, err.p, psi, true, c.fsb, p3, 7, h, Options{0, -1, 0})) != 0) return e;
    gather(g, c.fsa, &c.fsb, nullptr, out, 1, 7);
    return 0;
}

void copy_forms(const FormsCtx &c, double *stats, int max_rows, int *rows) {
    const int n = (int)(c.forms.size() / kFormCols);
    *rows = n;
    memcpy(stats, c.forms.data(), sizeof(double) * kFormCols * std::min(n, max_rows));
}

// "WENO6-optimized" is WENO6 but for the quadrature points
int plain_interp(int interp, Options &o) {
    o.weno_opt = interp == FIA_INTERP_WENO6_OPTIMIZED;
    return o.weno_opt ? (int)FIA_INTERP_WENO6 : interp;
}

}  // namespace

extern "C" {

// whether the launcher gives the WENO6 integral pass of an nx x ny x nz cell grid the z stencil tables
int forms_takes_tables(int nx, int ny, int nz) {
    FaceParams p;
    memset(&p, 0, sizeof(p));
    p.g.init(-1, nx, ny, nz);
    p.interp = IM_WENO6;
    p.integral = 1;
    p.gauss = gauss_table(1);
    size_t psi_halves = 0;
    return weno_table_halves(p, psi_halves) > 0;
}

int forms_cols(void) { return kFormCols; }
void *forms_create(void) { return new FormsCtx(); }
void forms_destroy(void *c) { delete (FormsCtx *)c; }
const char *forms_message(void *c) { return ((FormsCtx *)c)->msg; }

// x planes per thread of the zero-velocity march on an nx x ny x nz cell grid, `block` threads a block
long forms_zero_chunk(int nx, int ny, int nz, int block) {
    CompGrid g;
    g.init(-1, nx, ny, nz);
    return (long)zero_velocity_chunk(g, block);
}

// fia_move_substances_3d in place; tables: 0 by the launcher's rule, 1 always, -1 never
int forms_move_substances(void *ctx, int nx, int ny, int nz, double h, float *rho, const float *u, const float *v,
                          const float *w, double dt, int split, int interp, int use_integral, int ng, double min_area,
                          int tables, int zero_chunk, double *stats, int max_rows, int *rows) {
    FormsCtx &c = *(FormsCtx *)ctx;
    c.forms.clear();
    c.counters[1] = 0;
    Options o{0, tables, zero_chunk};
    interp = plain_interp(interp, o);
    CompGrid g;
    g.init(-1, nx, ny, nz);
    const int e = forms_step(c, g, rho, rho, u, v, w, h, dt, interp, use_integral, ng, min_area, split, FIA_SPLIT_XZ_AXIS, o);
    copy_forms(c, stats, max_rows, rows);
    return e;
}

// one component of fia_advect_velocity_3d, into out
int forms_advect_velocity(void *ctx, int nx, int ny, int nz, double h, const float *u, const float *v, const float *w,
                          int comp, float *out, double dt, int interp, int use_integral, int ng, int tables, int zero_chunk,
                          double *stats, int max_rows, int *rows) {
    FormsCtx &c = *(FormsCtx *)ctx;
    c.forms.clear();
    c.counters[1] = 0;
    Options o{0, tables, zero_chunk};
    interp = plain_interp(interp, o);
    CompGrid g;
    g.init(comp, nx, ny, nz);
    const bool one_dy = interp == FIA_INTERP_1DY_LINEAR;
    const float *q = comp == 0 ? u : (comp == 1 ? v : w);
    const int e = forms_step(c, g, q, out, u, v, w, h, dt, interp, use_integral, ng, 1.0, velocity_split(comp, one_dy, false),
                             velocity_split(comp, false, true), o);
    copy_forms(c, stats, max_rows, rows);
    return e;
}

// one pass of q on component grid comp (-1: cells), in place
int forms_flux_pass(void *ctx, int comp, int nx, int ny, int nz, double h, float *q, const float *u, const float *v,
                    const float *w, double dt, int split, int interp, int psi_mode, int zero_velocity, int use_integral,
                    int ng, double min_area, int tables, int zero_chunk, double *stats, int max_rows, int *rows) {
    FormsCtx &c = *(FormsCtx *)ctx;
    c.forms.clear();
    c.counters[1] = 0;
    Options o{0, tables, zero_chunk};
    interp = plain_interp(interp, o);
    CompGrid g;
    g.init(comp, nx, ny, nz);
    Fields f(g, u, v, w, q);
    PassSpec s{split, interp, psi_mode, zero_velocity ? 1 : 0, use_integral ? 1 : 0, ng, min_area};
    const double *psi = psi_forms(c, f.psi, g, f.q.p, s.psi_mode, s.integral, s.ng);
    if (!zero_velocity && !vertices_forms(c, g, f.u.p, f.v.p, f.w.p, dt / h, interp)) return -1;
    const int fm = zero_velocity ? 2 : 7;
    const int e = faces_forms(c, g, f.q.p, psi, !zero_velocity, c.fsa, s, fm, h, o);
    if (e == 0) gather(g, c.fsa, nullptr, nullptr, q, 0, fm);
    copy_forms(c, stats, max_rows, rows);
    return e;
}

// the displacements of fia_backtrace_vertices on the lattice of component comp, three arrays in out:
// by the launcher's form, or (each = 1) vertex by vertex
int forms_vertices(void *ctx, int comp, int nx, int ny, int nz, const float *u, const float *v, const float *w,
                   double dt_over_h, int interp, int each, float *out) {
    FormsCtx &c = *(FormsCtx *)ctx;
    CompGrid g;
    g.init(comp, nx, ny, nz);
    std::vector<float> none(g.cells(), 0.0f);
    Fields f(g, u, v, w, none.data());
    if (each) {
        VertexParams p;
        memset(&p, 0, sizeof(p));
        p.g = g; p.u = f.u.p; p.v = f.v.p; p.w = f.w.p; p.dt_over_h = (float)dt_over_h; p.interp = interp;
        for (int a = 0; a < 3; ++a) p.disp[a] = out + (size_t)a * g.lattice();
        parallel_for((long)g.lattice(), [&](long id) { vertex_body(p, id); });
        return 0;
    }
    if (!vertices_forms(c, g, f.u.p, f.v.p, f.w.p, dt_over_h, interp)) return -1;
    for (int a = 0; a < 3; ++a) memcpy(out + (size_t)a * g.lattice(), c.disp_out[a].p, g.lattice() * sizeof(float));
    return 0;
}

}  // extern "C"
