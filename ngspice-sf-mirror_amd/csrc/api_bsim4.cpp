/*
 * C ABI of the BSIM4 device: model cards, instance sets and the
 * per-instance evaluation entry point.
 *
 * A set resolves every instance on the host (b4temp.c size / temperature
 * dependence), then splits the table columns: a field whose value is the
 * same for every instance of a model card becomes a per-model column, every
 * other field a per-instance column.  Only the per-instance columns cost
 * HBM traffic per evaluation.
 */
#include <algorithm>
#include <cstring>
#include <thread>
#include <unordered_map>
#include <vector>
#include "ngmi_internal.h"
#include "bsim4_setup.h"
#include "bsim4_eval.h"
#include "bsim4_dev.h"
#include "set_table.h"

namespace ngmi {
int launch_bsim4_eval(const B4Tab &tab, const B4Ckt &ck, const double *vterm,
                      double *const state[3], double *cache, double *stamp, double *rhs,
                      int *noncon, hipStream_t stream);

static const char *const kFieldNames[] = {
#define NGMI_X(f) #f,
    NGMI_B4_FIELDS(NGMI_X)
#undef NGMI_X
};

int field_index(const char *name)
{
    for (int f = 0; f < B4F__COUNT; f++)
        if (std::strcmp(kFieldNames[f], name) == 0) return f;
    return -1;
}

}  // namespace ngmi

using namespace ngmi;

struct ngmi_bsim4_model {
    B4Model m;
    bool ready = false;
};

struct ngmi_bsim4_set {
    std::vector<ngmi_bsim4_model *> models;   /* distinct cards, in first-use order */
    std::unordered_map<const ngmi_bsim4_model *, int> model_pos;
    std::vector<int> model_of;
    std::vector<B4Inst> inst;
    std::vector<double> rows;                 /* n x B4F__COUNT, after finalize */
    std::vector<int> code;
    int icols = 0, mcols = 0;
    SetRecords recs;
    std::vector<void *> dev;                  /* device buffers */
    size_t dev_bytes = 0;
    B4Tab tab{};
    bool final_ = false;

    void release()
    {
        for (void *p : dev) (void)hipFree(p);
        dev.clear();
        dev_bytes = 0;
    }
    template <class T>
    int upload(const std::vector<T> &v, const T **out)
    {
        const size_t bytes = std::max<size_t>(v.size(), 1) * sizeof(T);
        void *p = nullptr;
        NGMI_HIP(hipMalloc(&p, bytes));
        dev.push_back(p);
        dev_bytes += bytes;
        if (!v.empty()) NGMI_HIP(hipMemcpy(p, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice));
        *out = static_cast<const T *>(p);
        return NGMI_OK;
    }
};

namespace ngmi {

const B4Tab *set_table(const ngmi_bsim4_set *s) { return s && s->final_ ? &s->tab : nullptr; }

const SetRecords *set_records(const ngmi_bsim4_set *s) { return s && s->final_ ? &s->recs : nullptr; }

void set_tiles(const ngmi_bsim4_set *s, const std::vector<int> &at, std::vector<double> &tiles)
{
    const size_t ntile = (at.size() + B4_TILE - 1) / B4_TILE;
    const int nc = B4_NC_GEOM;
    tiles.assign(ntile * B4_TILE * (size_t)nc, 0.0);
    for (size_t i = 0; i < at.size(); i++) {
        if (at[i] < 0) continue;
        const double *row = &s->rows[(size_t)at[i] * B4F__COUNT];
        double *t = &tiles[(i / B4_TILE) * B4_TILE * nc + i % B4_TILE];
        for (int c = 0; c < nc; c++) t[(size_t)c * B4_TILE] = row[B4_IFIELDS[c]];
    }
}

/* the set's records: instances of one model card that differ only in the
 * per-instance fields share one, equal ones of several cards too */
static void build_records(const std::vector<double> &rows, const std::vector<int> &model_of, int nm,
                          const std::vector<char> &perinst, SetRecords &R)
{
    const size_t n = model_of.size();
    const int F = B4F__COUNT;
    R = SetRecords();
    std::vector<int> extra;   /* fields that vary within a card beyond the per-instance list */
    for (int f = 0; f < F; f++) {
        if (!perinst[f]) continue;
        if (B4_ICOL[f] < B4_NC_LD) R.nc = std::max(R.nc, B4_NC_LD);
        else if (B4_ICOL[f] < B4_NC_GEOM) R.nc = B4_NC_GEOM;
        else extra.push_back(f);
    }
    /* a card, or a card at one set of extra values, is a candidate; equal
     * candidates (in the fields read from records) are one record */
    auto hash = [](uint64_t h, uint64_t v) { return (h ^ v) * 0x9E3779B97F4A7C15ull + (h >> 29); };
    auto bits = [](double v) { uint64_t u; std::memcpy(&u, &v, 8); return u; };
    std::unordered_multimap<uint64_t, size_t> cand;      /* hash -> first instance of a candidate */
    std::unordered_multimap<uint64_t, int> by_content;   /* hash -> record */
    std::vector<int> cand_rec(n, -1), of_model(nm, -1);
    std::vector<size_t> rec_inst;
    R.rec_of.assign(n, -1);
    auto record_of = [&](size_t k) {
        const double *row = &rows[k * F];
        uint64_t h = 1;
        for (int f = 0; f < F; f++)
            if (B4_ICOL[f] >= R.nc) h = hash(h, bits(row[f]));
        const auto rg = by_content.equal_range(h);
        for (auto it = rg.first; it != rg.second; ++it) {
            const double *o = &rows[rec_inst[it->second] * F];
            bool same = true;
            for (int f = 0; f < F && same; f++)
                if (B4_ICOL[f] >= R.nc) same = bits(row[f]) == bits(o[f]);
            if (same) return it->second;
        }
        const int r = (int)rec_inst.size();
        rec_inst.push_back(k);
        by_content.emplace(h, r);
        return r;
    };
    /* records are not built for sets with more of them than this: 1.9 KB each,
     * a fraction of the columns' room */
    const size_t most = std::max<size_t>(4096, n / 8);
    for (size_t k = 0; k < n; k++) {
        int r = -1;
        if (extra.empty()) {
            int &m = of_model[model_of[k]];
            if (m < 0) m = record_of(k);
            r = m;
        } else {
            const double *row = &rows[k * F];
            uint64_t h = hash(2, (uint64_t)model_of[k]);
            for (int f : extra) h = hash(h, bits(row[f]));
            const auto rg = cand.equal_range(h);
            for (auto it = rg.first; it != rg.second && r < 0; ++it) {
                const double *o = &rows[it->second * F];
                bool same = model_of[it->second] == model_of[k];
                for (int f : extra) same = same && bits(row[f]) == bits(o[f]);
                if (same) r = cand_rec[it->second];
            }
            if (r < 0) {
                r = cand_rec[k] = record_of(k);
                cand.emplace(h, k);
            }
        }
        if (rec_inst.size() > most) {
            R.rec_of.clear();
            return;
        }
        R.rec_of[k] = r;
    }
    R.rec.resize(rec_inst.size() * F);
    for (size_t r = 0; r < rec_inst.size(); r++)
        std::copy(&rows[rec_inst[r] * F], &rows[rec_inst[r] * F] + F, &R.rec[r * F]);
    R.ok = true;
}

/* items (tile, record) over the tiles of `at`'s records: a tile is listed
 * once for each record among its lanes */
static void build_items(const std::vector<int> &rec_of, std::vector<int> &items)
{
    for (size_t t = 0; t * B4_TILE < rec_of.size(); t++) {
        const size_t b = t * B4_TILE, e = std::min(rec_of.size(), b + B4_TILE), i0 = items.size();
        for (size_t k = b; k < e; k++) {
            bool seen = false;
            for (size_t q = i0; q < items.size() && !seen; q += 2) seen = items[q + 1] == rec_of[k];
            if (!seen) {
                items.push_back((int)t);
                items.push_back(rec_of[k]);
            }
        }
    }
}

}  // namespace ngmi

extern "C" {

ngmi_bsim4_model *ngmi_bsim4_model_new(void) { return new ngmi_bsim4_model; }

void ngmi_bsim4_model_free(ngmi_bsim4_model *m) { delete m; }

int ngmi_bsim4_model_param(ngmi_bsim4_model *m, const char *name, double value)
{
    if (!m || !name) return NGMI_E_PANIC;
    if (m->m.set(name, value) != 0) {
        set_error("unknown BSIM4 model parameter '%s'", name);
        return NGMI_E_BADPARM;
    }
    m->ready = false;
    return NGMI_OK;
}

int ngmi_bsim4_model_setup(ngmi_bsim4_model *m, double tnom, double temp)
{
    if (!m) return NGMI_E_PANIC;
    if (m->m.finish(tnom, temp) != 0) {
        const char *why = m->m.check();
        set_error("BSIM4 model card not supported by the engine: %s", why ? why : "setup failed");
        return NGMI_E_UNSUPP;
    }
    m->ready = true;
    return NGMI_OK;
}

double ngmi_bsim4_model_get(const ngmi_bsim4_model *m, const char *what)
{
    if (!m || !what) return 0.0;
    if (!std::strcmp(what, "type")) return m->m.type;
    if (!std::strcmp(what, "coxe")) return m->m.coxe;
    if (!std::strcmp(what, "vtm")) return m->m.vtm;
    if (!std::strcmp(what, "vcrit")) return m->m.vcrit;
    return 0.0;
}

ngmi_bsim4_set *ngmi_bsim4_set_new(void) { return new ngmi_bsim4_set; }

void ngmi_bsim4_set_free(ngmi_bsim4_set *s)
{
    if (!s) return;
    s->release();
    delete s;
}

int ngmi_bsim4_set_add(ngmi_bsim4_set *s, ngmi_bsim4_model *const *models, int nmodels,
                       const int *model_idx, int n, const char *const *names, int nparams,
                       const double *params)
{
    if (!s || !models || n < 0 || (n > 0 && !model_idx)) return NGMI_E_PANIC;
    if (s->final_) {
        set_error("instance set already finalized");
        return NGMI_E_PANIC;
    }
    for (int k = 0; k < nmodels; k++) {
        if (!models[k] || !models[k]->ready) {
            set_error("model %d not set up (call ngmi_bsim4_model_setup first)", k);
            return NGMI_E_NOMOD;
        }
    }
    /* map caller model indices to set model indices */
    std::vector<int> local(nmodels, -1);
    const int first = (int)s->inst.size();
    for (int k = 0; k < n; k++) {
        const int mk = model_idx[k];
        if (mk < 0 || mk >= nmodels) {
            set_error("instance %d: model index %d out of range", k, mk);
            return NGMI_E_NOMOD;
        }
        if (local[mk] < 0) {
            auto it = s->model_pos.find(models[mk]);
            if (it == s->model_pos.end()) {
                s->models.push_back(models[mk]);
                local[mk] = (int)s->models.size() - 1;
                s->model_pos[models[mk]] = local[mk];
            } else {
                local[mk] = it->second;
            }
        }
        B4Inst in;
        in.model = &models[mk]->m;
        for (int j = 0; j < nparams; j++) {
            if (in.set(names[j], params[(size_t)j * n + k]) != 0) {
                set_error("unknown BSIM4 instance parameter '%s'", names[j]);
                s->inst.resize(first);
                s->model_of.resize(first);
                return -NGMI_E_BADPARM;
            }
        }
        in.defaults();
        if (const char *why = in.check()) {
            set_error("instance %d not supported by the engine: %s", first + k, why);
            s->inst.resize(first);
            s->model_of.resize(first);
            return -NGMI_E_UNSUPP;
        }
        s->inst.push_back(in);
        s->model_of.push_back(local[mk]);
    }
    return first;
}

}  // extern "C"

namespace ngmi {

/* resolves every instance and splits the columns; no device work */
static int set_resolve(ngmi_bsim4_set *s)
{
    const size_t n = s->inst.size();
    const int F = B4F__COUNT;
    const int nm = (int)s->models.size();
    s->rows.assign(n * F, 0.0);
    /* b4check clamps act on the first instance of each card: resolve those
     * first and in order, the rest in parallel */
    std::vector<char> done(n, 0);
    std::vector<char> seen(nm, 0);
    for (size_t k = 0; k < n; k++) {
        const int m = s->model_of[k];
        if (seen[m]) continue;
        seen[m] = 1;
        if (s->inst[k].resolve(&s->rows[k * F]) != 0) {
            set_error("instance %zu: effective channel length or width <= 0", k);
            return NGMI_E_PARMVAL;
        }
        done[k] = 1;
    }
    unsigned nt = std::max(1u, std::min(32u, std::thread::hardware_concurrency()));
    if (n < 4096) nt = 1;
    std::vector<int> bad(nt, -1);
    std::vector<std::thread> th;
    for (unsigned t = 0; t < nt; t++) {
        th.emplace_back([&, t]() {
            for (size_t k = t; k < n; k += nt) {
                if (done[k]) continue;
                if (s->inst[k].resolve(&s->rows[k * F]) != 0 && bad[t] < 0) bad[t] = (int)k;
            }
        });
    }
    for (auto &x : th) x.join();
    for (unsigned t = 0; t < nt; t++) {
        if (bad[t] >= 0) {
            set_error("instance %d: effective channel length or width <= 0", bad[t]);
            return NGMI_E_PARMVAL;
        }
    }
    /* column split */
    std::vector<char> perinst(F, 0);
    std::vector<size_t> firstOf(nm, (size_t)-1);
    for (size_t k = 0; k < n; k++)
        if (firstOf[s->model_of[k]] == (size_t)-1) firstOf[s->model_of[k]] = k;
    for (int f = 0; f < F; f++) {
        for (size_t k = 0; k < n && !perinst[f]; k++) {
            const double a = s->rows[k * F + f];
            const double b = s->rows[firstOf[s->model_of[k]] * F + f];
            if (std::memcmp(&a, &b, sizeof(double)) != 0) perinst[f] = 1;
        }
    }
    s->code.assign(F, 0);
    s->icols = s->mcols = 0;
    for (int f = 0; f < F; f++) s->code[f] = perinst[f] ? s->icols++ : ~(s->mcols++);
    build_records(s->rows, s->model_of, nm, perinst, s->recs);
    /* one selector word for the whole set lets the kernels compile the
     * selectors as constants */
    s->tab = B4Tab{};
    s->tab.flags = n ? (int)s->rows[B4F_flags] : -1;
    for (size_t k = 1; k < n && s->tab.flags >= 0; k++)
        if ((int)s->rows[k * F + B4F_flags] != s->tab.flags) s->tab.flags = -1;
    s->tab.n = (int64_t)n;
    s->tab.nm = nm;
    s->tab.mcols = s->mcols;
    s->final_ = true;
    return NGMI_OK;
}

int set_upload_columns(ngmi_bsim4_set *s)
{
    const size_t n = s->inst.size();
    const int F = B4F__COUNT, nm = (int)s->models.size();
    std::vector<size_t> firstOf(nm, (size_t)-1);
    for (size_t k = 0; k < n; k++)
        if (firstOf[s->model_of[k]] == (size_t)-1) firstOf[s->model_of[k]] = k;
    std::vector<double> itab((size_t)s->icols * n), mtab((size_t)s->mcols * std::max(nm, 1));
    for (int f = 0; f < F; f++) {
        if (s->code[f] >= 0) {
            double *dst = &itab[(size_t)s->code[f] * n];
            for (size_t k = 0; k < n; k++) dst[k] = s->rows[k * F + f];
        } else {
            /* model-major: one card's per-model values are contiguous, so
             * the few cards a workgroup reads stay in its L1 */
            for (int m = 0; m < nm; m++)
                if (firstOf[m] != (size_t)-1) mtab[(size_t)m * s->mcols + (~s->code[f])] = s->rows[firstOf[m] * F + f];
        }
    }
    s->tab.mode = B4T_COLUMNS;
    int rc;
    if ((rc = s->upload(itab, &s->tab.itab)) || (rc = s->upload(mtab, &s->tab.mtab)) ||
        (rc = s->upload(s->model_of, &s->tab.model_of)) || (rc = s->upload(s->code, &s->tab.code)))
        return rc;
    return NGMI_OK;
}

int set_finalize_host(ngmi_bsim4_set *s)
{
    if (!s) return NGMI_E_PANIC;
    const int rc = set_resolve(s);
    if (rc == NGMI_OK) s->release();
    return rc;
}

}  // namespace ngmi

extern "C" {

int ngmi_bsim4_set_finalize(ngmi_bsim4_set *s)
{
    int rc = set_finalize_host(s);
    if (rc) return rc;
    s->final_ = false;   /* until its tables are on the device */
    const SetRecords &R = s->recs;
    std::vector<int> items, at(s->inst.size());
    for (size_t k = 0; k < at.size(); k++) at[k] = (int)k;
    if (R.ok) build_items(R.rec_of, items);
    const size_t ntile = (at.size() + B4_TILE - 1) / B4_TILE, nit = items.size() / 2;
    constexpr size_t SIMDS = 1024;
    /* Lanes of one wavefront each with another of many records read 64 lines
     * where a column is a few; below two rounds of workgroups latency hides
     * that (65536 devices, 28397 records mixed, 57 us against columns' 61),
     * and in runs the lines are shared. 524288 devices mixed: 128 records 303
     * us against 324, 1024 records 337, 8192 records 366; 16385 in runs, 3
     * a tile, 289. */
    const bool scattered = ntile > SIMDS && R.rec.size() > (size_t)512 * B4F__COUNT && nit > 16 * ntile;
    if (!R.ok || scattered) {
        if ((rc = set_upload_columns(s))) return rc;
        s->final_ = true;
        return NGMI_OK;
    }
    /* Scalar records run a tile once per record in it; a record a lane runs
     * it once, with slower loads.  Worth it up to a third more workgroups
     * (524288 devices in runs of one record, 8192 tiles: 9196 items 237 us
     * against 280, 12235 items 297 against 281), and not for another round
     * of workgroups, one or two of which each of the 1024 SIMDs takes at a
     * time (40000 devices, 625 tiles: 688 items 44 us against 45, 1250 55
     * against 44; 131072, 2048 tiles: 2051 items 76 against 67). */
    const size_t round = ntile <= SIMDS ? SIMDS : ntile <= 2 * SIMDS ? 2 * SIMDS : nit;
    s->tab.mode = nit <= std::min(ntile + ntile / 3, round) ? B4T_UNIFORM : B4T_LANES;
    s->tab.nc = R.nc;
    s->tab.nitems = (int)nit;
    std::vector<double> tiles;
    set_tiles(s, at, tiles);
    if ((rc = s->upload(R.rec, &s->tab.rec)) || (rc = s->upload(tiles, &s->tab.itile)) ||
        (rc = s->upload(R.rec_of, &s->tab.rec_of)) || (rc = s->upload(items, &s->tab.items)))
        return rc;
    s->final_ = true;
    return NGMI_OK;
}

int ngmi_bsim4_set_size(const ngmi_bsim4_set *s) { return s ? (int)s->inst.size() : 0; }

double ngmi_bsim4_set_field(const ngmi_bsim4_set *s, int k, const char *field)
{
    if (!s || !s->final_ || k < 0 || (size_t)k >= s->inst.size()) return 0.0;
    const int f = field_index(field);
    if (f < 0) return 0.0;
    return s->rows[(size_t)k * B4F__COUNT + f];
}

int ngmi_bsim4_set_layout(const ngmi_bsim4_set *s, int *inst_cols, int *model_cols,
                          size_t *device_bytes)
{
    if (!s || !s->final_) return NGMI_E_PANIC;
    if (inst_cols) *inst_cols = s->icols;
    if (model_cols) *model_cols = s->mcols;
    if (device_bytes) *device_bytes = s->dev_bytes;
    return NGMI_OK;
}

int ngmi_bsim4_set_form(const ngmi_bsim4_set *s, int *form, int64_t *workgroups)
{
    static_assert(NGMI_FORM_COLUMNS == B4T_COLUMNS && NGMI_FORM_WAVE == B4T_UNIFORM && NGMI_FORM_LANE == B4T_LANES,
                  "the header's forms");
    if (!s || !s->final_) return NGMI_E_PANIC;
    if (form) *form = s->tab.mode;
    if (workgroups)
        *workgroups = s->tab.mode == B4T_UNIFORM ? s->tab.nitems : (s->tab.n + B4_TILE - 1) / B4_TILE;
    return NGMI_OK;
}

int ngmi_bsim4_eval(const ngmi_bsim4_set *s, const ngmi_ckt_scalars *c, const double *vterm,
                    double *const state[3], double *cache, double *stamp, double *rhs,
                    int *noncon, void *stream)
{
    if (!s || !s->final_ || !c || !state) {
        set_error("ngmi_bsim4_eval: set not finalized or missing arguments");
        return NGMI_E_PANIC;
    }
    if (c->order > 2 && c->method != 1) {
        set_error("ngmi_bsim4_eval keeps three state levels: Gear order %d needs more", c->order);
        return NGMI_E_UNSUPP;
    }
    B4Ckt ck;
    ck.mode = c->mode;
    ck.order = c->order;
    ck.method = c->method;
    for (int k = 0; k < 7; k++) ck.ag[k] = c->ag[k];
    ck.xfact = c->xfact;
    ck.gmin = c->gmin;
    ck.reltol = c->reltol;
    ck.abstol = c->abstol;
    return launch_bsim4_eval(s->tab, ck, vterm, state, cache, stamp, rhs, noncon,
                             (hipStream_t)stream);
}

}  // extern "C"
