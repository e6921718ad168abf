// Launch-shape selection for the fused ELL kernels (fields per thread, block size).
//
// A tuning table maps (kind, rows bucket, width, n_ops, fields, storage, field type,
// accumulation) to the shape measured fastest by rbfx_tune_spmm / the autotuner in the
// Python layer; the table lives in memory and can be saved/loaded as text so a run can reuse
// an earlier sweep. Without an entry the rules of default_shape decide.
#include <cstdio>
#include <map>
#include <mutex>
#include <tuple>

#include "rbfx_ell_common.h"

namespace {
using Key = std::tuple<int, int, int, int, int, int, int, int>;
std::map<Key, EllTune> g_table;
std::mutex g_mu;

int rows_bucket(int n) {
    int b = 0;
    while ((1 << (b + 1)) <= n) b++;
    return b;
}

Key make_key(const rbfx_ell* e, int F, int ft, int acc, int kind) {
    return Key(kind, rows_bucket(e->n_rows), e->width, e->n_ops, F, e->storage, ft, acc);
}

bool valid(int F, int fpt, int block) {
    if (fpt <= 0 || F % fpt) return false;
    if (fpt != 1 && fpt != 2 && fpt != 4 && fpt != 8) return false;
    if (block < 64 || block > 256 || block % 64) return false;
    return (F / fpt) <= block;
}

// An LDS-staged shape (share 4/5) holds for the operator set it was tuned on: another set with
// the same key may have no tile tables, other tiles or more nodes per tile than the LDS holds.
bool lds_shape_fits(const rbfx_ell* e, int F, int ft, int acc, int kind, const EllTune& c) {
    if (c.fpt <= 0 || F % c.fpt) return false;
    const int G = F / c.fpt;
    const size_t rec = (size_t)F * (ft == RBFX_F64 ? 8 : 4);
    bool ok = (kind == 0 || kind == 1) && e->lt > 0 && e->n_ops >= 3 && e->lt * G <= 512 && rec % 16 == 0 &&
              (size_t)e->k_max * rec <= (size_t)e->lds_limit;
    if (c.share == 5) ok = ok && c.fpt == 4 && G == 4 && e->storage != RBFX_F64 && ft == RBFX_F32 && acc == RBFX_F32;
    return ok;
}

// The shape of a set without a tuned entry. Times are of four RK4 stages, n = 31 or 50, FP64 / FP32.
EllTune default_shape(const rbfx_ell* e, int F, int ft, int acc, int kind) {
    const long long n = e->n_rows;
    const bool f64 = e->storage == RBFX_F64;
    const int cus = e->ctx->n_cu > 0 ? e->ctx->n_cu : 256;
    // LDS-staged gathers for a set with tile tables whose records fit the LDS (60,000 rows: 80 against
    // 106 us in FP64)
    if (e->lt > 0 && e->n_ops >= 3 && F == 16 && e->lt * 4 <= 512) {
        const size_t rec = (size_t)F * (ft == RBFX_F64 ? 8 : 4);
        if ((size_t)e->k_max * rec <= (size_t)e->lds_limit)
            return EllTune{4, e->lt * 4, 4, !f64 && ft == RBFX_F32 && acc == RBFX_F32 ? 5 : 4};
    }
    // One field of few rows: four lanes per row, while all waves of 16 rows are on the chip together
    // (two per SIMD in FP64, four in FP32). 4096 / 20,000 rows: 20.0 / 21.1 us in FP64 against 21.7 / 25.0
    // with a lane per row, 19.8 / 20.1 against 25.3 / 26.9 in FP32; at 40,000 rows 35.9 against 33.7 in
    // FP64, at 80,000 61 against 58 in FP32. Short stencils gain nothing (n = 17: 19.4 against 18.3). A
    // single operator's weights are loaded by all four lanes: not for long stencils (n = 101: 9.5 against
    // 9.0 us an apply) nor beyond two waves per SIMD (60,000 rows in FP32: 8.9 against 7.6).
    if (F == 1 && e->n_ops <= 4 && e->width >= 24 && n <= 128ll * cus * (f64 || e->n_ops == 1 ? 1 : 2) &&
        (e->n_ops > 1 || e->width <= 64))
        return EllTune{1, 64, 8, 6};
    const int max_acc = acc == RBFX_F64 ? 16 : 32;
    int fpt = 1, block, ub = 8;
    // 256-thread blocks keep neighbouring rows on one CU, 64-thread ones spread the last round of blocks over
    // all CUs: up to four waves per SIMD 64, unless 256-thread blocks fill at least 4/5 of their last round. One
    // field, rounds of 65,536 rows: 126,000 rows (1.92 rounds) 2-5% for 256, 250,000 (3.8) 0-4%; 70,000 (1.07) 19-42%
    // for 64, 100,000 (1.53) 4-6%, 160,000 (2.44) and 200,000 (3.05) 5-9%. 4096 rows: 22 against 29 us a step;
    // 320,000 rows x 3: 2-5% for 256.
    auto block_for = [&](long long lanes) {
        const long long round = 256ll * cus;
        return lanes >= 4 * round || (lanes > round && lanes % round * 5 >= round * 4) ? 256 : 64;
    };
    if (F == 1) {
        // Slots per memory round trip: 16 for a single operator (111 against 120 us with 4 at a million rows),
        // else 8 (4096 rows: 22 against 25), but 4 where 8 slots of FP64 weights leave few waves (an apply
        // of two operators, 100,000 rows: 17.8 against 18.5).
        block = block_for(n);
        if (kind == 0 && e->n_ops == 1) ub = 16;
        else if (kind == 0 && f64 && block == 64) ub = 4;
    } else {
        // Several fields: up to 4 per thread (16 FP64 or 32 FP32 sums at most), fewer loads of the indices
        // and weights, as long as there is a lane for each SIMD's wave with 4, and for three waves in eight
        // SIMDs with 2. Applies and stages, FP32 and FP64 have the line at the same place (8 fields, n = 17 to
        // 101: at 20,000 rows 2 ahead of 4 by 2-5%, at 40,000 4 ahead of 2 by 10-18%; 4 fields: at 20,000
        // 2 ahead of 1 by 2-14%, at 10,000 equal). Four FP64 fields in one lane lose to two lanes of two: 320,000
        // rows x 4, n = 50, 3 operators: 542-616 us a step against 522.
        for (int c : {4, 2})
            if (F % c == 0 && c * e->n_ops <= max_acc && n * (F / c) >= (c == 4 ? 256ll : 96ll) * cus &&
                !(f64 && c == 4 && F == 4)) {
                fpt = c;
                break;
            }
        block = block_for(n * (F / fpt));
        // 8 slots per round trip (4: 5-15% behind), but 4 for four FP64 fields of several operators, where
        // 8 leave few waves (80,000 rows x 8: 3-4% ahead), and for odd fields on short stencils (20,000
        // rows x 3, n = 17, FP64: 5.5 against 6.0 us an apply).
        if ((f64 && fpt == 4 && e->n_ops >= 3) || (fpt == 1 && F > 2 && e->width < 24 && n * F >= 192ll * cus)) ub = 4;
        // A row's fields stay in one block: rows of more lanes than it has take 256-thread blocks, and beyond
        // 256 lanes the most fields per thread, so that every field count up to 256 * 8 that divides finds a shape.
        if (F / fpt > block) block = 256;
        for (int c : {8, 4, 2})
            if (F / fpt > block && F % c == 0 && c * e->n_ops <= max_acc) {
                fpt = c;
                ub = 4;
            }
    }
    return EllTune{fpt, block, ub, 0};
}
}  // namespace

int rbfx_ell_pick(rbfx_ell* e, int F, int ft, int acc, int kind, EllTune* t) {
    {
        std::lock_guard<std::mutex> lk(g_mu);
        auto it = g_table.find(make_key(e, F, ft, acc, kind));
        if (it != g_table.end()) {
            EllTune c = it->second;
            if (c.share != 4 && c.share != 5) {
                *t = c;
                return RBFX_OK;
            }
            if (lds_shape_fits(e, F, ft, acc, kind, c)) {
                c.block = e->lt * (F / c.fpt);  // the block is this set's tile
                *t = c;
                return RBFX_OK;
            }
            // otherwise: the shape of a set without (fitting) tile tables, below
        }
    }
    *t = default_shape(e, F, ft, acc, kind);
    if (!valid(F, t->fpt, t->block) && t->share != 4 && t->share != 5)
        return rbfx_fail(e->ctx, RBFX_E_TOO_LARGE, "no launch shape for %d fields (at most 256*8)", F);
    return RBFX_OK;
}

extern "C" {

// Sets the launch shape used for (ell, n_fields, types, kind); kind 0 = SpMM, 1 = RK4 stage.
int rbfx_tune_set(rbfx_ell* e, int32_t kind, int32_t n_fields, int32_t field_type, int32_t accum, int32_t fpt, int32_t block,
                  int32_t batch, int32_t share) {
    if (!e) return RBFX_E_INVALID;
    if (share == 4 || share == 5) {  // LDS-staged gathers (rbfx_ell_build_local); the block is the tile
        const int G = fpt > 0 ? n_fields / fpt : 0;
        const size_t rec = (size_t)n_fields * (field_type == RBFX_F64 ? 8 : 4);
        bool ok = (kind == 0 || kind == 1) && e->lt > 0 && e->n_ops >= 3 && fpt > 0 && n_fields % fpt == 0 &&
                  ((fpt == 4 && G == 4) || (fpt == 8 && G == 2)) && (batch == 4 || batch == 8) &&
                  e->lt * G <= 512 && rec % 16 == 0 && (size_t)e->k_max * rec <= (size_t)e->lds_limit;
        // matrix-core multiply-adds: FP32 weights, fields and accumulation, 16 fields on 4 lanes
        if (share == 5)
            ok = ok && fpt == 4 && G == 4 && e->storage != RBFX_F64 && field_type == RBFX_F32 && accum == RBFX_F32;
        if (!ok)
            return rbfx_fail(e->ctx, RBFX_E_INVALID,
                             "tune_set: no LDS-staged shape for %d fields, fpt %d, batch %d (tile %d, %d nodes per tile)",
                             n_fields, fpt, batch, e->lt, e->k_max);
        std::lock_guard<std::mutex> lk(g_mu);
        g_table[make_key(e, n_fields, field_type, accum, kind)] = EllTune{fpt, e->lt * G, batch, share};
        return RBFX_OK;
    }
    if (share == 6) {  // one field on four lanes per row, 64-thread blocks
        if ((kind != 0 && kind != 1) || n_fields != 1 || fpt != 1 || block != 64 || batch != 8 || e->n_ops > 4)
            return rbfx_fail(e->ctx, RBFX_E_INVALID, "tune_set: share 6 takes one field, fpt 1, block 64, batch 8 and at most 4 operators");
        std::lock_guard<std::mutex> lk(g_mu);
        g_table[make_key(e, n_fields, field_type, accum, kind)] = EllTune{1, 64, 8, 6};
        return RBFX_OK;
    }
    // batch 16: the SpMV/SpMM kernel with one field per thread only
    const bool batch_ok = batch == 4 || batch == 8 || (batch == 16 && kind == 0 && fpt == 1 && share == 0);
    if (!valid(n_fields, fpt, block) || !batch_ok || share < 0 || share > 3)
        return rbfx_fail(e->ctx, RBFX_E_INVALID, "tune_set: invalid shape fpt %d block %d batch %d share %d for %d fields",
                         fpt, block, batch, share, n_fields);
    if (share) {
        int G = n_fields / fpt;
        if (kind != 1 || (G != 2 && G != 4) || fpt == 1 || batch % G)
            return rbfx_fail(e->ctx, RBFX_E_INVALID,
                             "tune_set: shared loads need the RK4 stage kernel, 2 or 4 lanes per row, fpt > 1 and a "
                             "batch divisible by them (fields %d, fpt %d, batch %d)", n_fields, fpt, batch);
        // pipelined cores (share 2, 3 = prefetch depth) exist for 3-4 operators and these shapes
        const bool pipe_ok = e->n_ops >= 3 && ((fpt == 4 && G == 4) || (fpt == 8 && G == 2) ||
                                               (share == 2 && ((fpt == 4 && G == 2) || (fpt == 2 && G == 4))));
        if (share >= 2 && !pipe_ok)
            return rbfx_fail(e->ctx, RBFX_E_INVALID, "tune_set: no pipelined core for %d operators, fpt %d, %d lanes, depth %d",
                             e->n_ops, fpt, G, share);
    }
    std::lock_guard<std::mutex> lk(g_mu);
    g_table[make_key(e, n_fields, field_type, accum, kind)] = EllTune{fpt, block, batch, share};
    return RBFX_OK;
}

int rbfx_tune_get(rbfx_ell* e, int32_t kind, int32_t n_fields, int32_t field_type, int32_t accum, int32_t* fpt, int32_t* block,
                  int32_t* batch, int32_t* share) {
    if (!e || !fpt || !block || !batch || !share) return RBFX_E_INVALID;
    EllTune t;
    int rc = rbfx_ell_pick(e, n_fields, field_type, accum, kind, &t);
    if (rc) return rc;
    *fpt = t.fpt;
    *block = t.block;
    *batch = t.ub;
    *share = t.share;
    return RBFX_OK;
}

int rbfx_tune_clear(void) {
    std::lock_guard<std::mutex> lk(g_mu);
    g_table.clear();
    return RBFX_OK;
}

}  // extern "C"
