/*
 * The launch planner of the host shim over many shapes, without a GPU: the
 * shim's source is compiled in, tensors are handles without weights, and no
 * launch is made. `plan_test scratch`: every launch that the no-allocation
 * entry point's rule accepts is made (its plans fit the scratch and a
 * workgroup's LDS), and as the plain entry point makes it (equal segments, so
 * equal bits). `plan_test capture`: every launch that fits a workspace of
 * that rule's size can be captured on a stream that holds just that, which
 * for short rows is nothing: plain and grouped, with the norm and SwiGLU.
 */
#include "../../my-inference-engine_amd/csrc/qmv_shim.cpp"

#include <cstdio>
#include <cstring>

namespace {

int g_failures = 0;

const int kFormats[] = {QMV_GGML_TYPE_Q8_0, QMV_GGML_TYPE_Q5_0, QMV_GGML_TYPE_Q4_K, QMV_GGML_TYPE_Q6_K};
const char *const kNames[] = {"Q8_0", "Q5_0", "Q4_K", "Q6_K"};
const int kRows[] = {1,     16,    64,    896,   1000,  3584,   4096,   8192,   8960,   18944,  32000,   37888,
                     65536, 98304, 128256, 151936, 152064, 200000, 262144, 300000, 524288, 1048576, 2000000};
const int kUnits[] = {1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15, 16, 17, 19, 20, 24, 28, 31, 32, 35, 38, 40, 56, 74, 112, 148};

QmvDeviceTensor tensor(int format, int rows, int units)
{
    QmvDeviceTensor t = {};
    t.ggml_type = (uint32_t)kFormats[format];
    qmv_geometry_of(t.ggml_type, &t.geo);
    t.rows = rows;
    t.cols = units * t.geo.unit_elements;
    t.blocks_per_row = t.cols / t.geo.block_elements;
    t.units = units;
    t.tiles = (rows + QMV_TILE_ROWS - 1) / QMV_TILE_ROWS;
    return t;
}

void fail(const char *what, const QmvDeviceTensor &t, int batch)
{
    ++g_failures;
    if (g_failures <= 40) printf("%s: %s %d x %d at %d positions\n", what, kNames[t.geo.format], t.rows, t.cols, batch);
}

/* LDS of a plan's workgroup, as launch_batch asks for it. */
bool lds_fits(const ChunkPlan &cp)
{
    if (!cp.batch) return true;
    const qmv::BatchParams &p = cp.bp;
    const int most = (p.units + p.segs - 1) / p.segs * p.chunk_segs;
    const size_t units = cp.bt_mode != QMV_BATCH_CHUNKS || most > p.units ? p.units : most, slots = 4 * cp.bt_nr;
    const size_t sums = cp.bt_mode == QMV_BATCH_DIRECT  ? (size_t)cp.waves * p.segs * slots * 16
                        : cp.bt_mode == QMV_BATCH_FUSED ? (size_t)p.segs * p.wg_groups * slots * 16 + slots
                                                        : 0;
    return (cp.bt_mode != QMV_BATCH_DIRECT || (cp.bt_r == 1 && !p.swiglu && !p.norm_w)) &&
           units * qmv::batch_stage_bytes(cp.fmt, cp.bt_nr) + sums * sizeof(float) <= 160 * 1024;
}

/* The order a launch adds its segments in. */
bool same_bits(const ChunkPlan &a, const ChunkPlan &b)
{
    if (a.batch != b.batch || a.rowdot != b.rowdot) return false;
    return a.batch ? a.bp.segs == b.bp.segs : a.p.positions == b.p.positions;
}

void check_scratch(const QmvDeviceTensor &t, int batch)
{
    QmvDeviceTensor *ts[1] = {const_cast<QmvDeviceTensor *>(&t)};
    float dummy = 0.0f, *out = &dummy; /* never dereferenced */
    const Epilogue epi;
    const WorkspaceNeed rule = workspace_rule(ts, 1, &dummy, batch, &out, epi);
    if (rule.partials > kScratchPartials || rule.counters > kScratchCounters) return;
    Cut cut;
    if (!scratch_cut(ts, 1, &dummy, batch, &out, &cut)) return fail("accepted by the rule but not planned", t, batch);
    ChunkPlan whole, piece;
    int b0 = 0;
    for (int i = 0; i < cut.pieces; ++i) {
        const int nb = piece_positions(batch, cut.pieces, i);
        if (!plan_chunk(ts, 1, &dummy, b0, nb, &out, epi, &piece, cut.room)) return fail("piece not planned", t, batch);
        if (piece.partials > kScratchPartials || piece.counters > kScratchCounters || !lds_fits(piece))
            return fail("piece over the scratch or LDS", t, batch);
        if (cut.room == SIZE_MAX) { /* the plain entry point launches the whole */
            if (!plan_chunk(ts, 1, &dummy, 0, batch, &out, epi, &whole) || (cut.pieces > 1 && !same_bits(whole, piece)))
                return fail("piece with other bits than the whole", t, batch);
        }
        b0 += nb;
    }
    if (b0 != batch) fail("pieces do not add up", t, batch);
}

void check_capture(const QmvDeviceTensor &t, int batch)
{
    const QmvDeviceTensor kv = tensor(t.geo.format, (t.rows + 7) / 8, t.units);
    QmvDeviceTensor *ts[3] = {const_cast<QmvDeviceTensor *>(&t), const_cast<QmvDeviceTensor *>(&kv),
                              const_cast<QmvDeviceTensor *>(&kv)};
    QmvDeviceTensor *pair[2] = {ts[0], ts[0]};
    float dummy = 0.0f, *out[3] = {&dummy, &dummy, &dummy};
    for (int form = 0; form < 5; ++form) {
        const bool swiglu = form >= 3, norm = form == 2 || form == 4;
        QmvDeviceTensor *const *tensors = swiglu ? pair : ts;
        const int count = swiglu ? 2 : form == 0 ? 1 : 3;
        Epilogue epi;
        epi.swiglu = swiglu;
        const WorkspaceNeed rule = workspace_rule(tensors, count, &dummy, batch, out, epi);
        ChunkPlan cp;
        if (norm) { /* as norm_then_group */
            epi.norm_w = &dummy;
            if (batch == 1 && plan_rowdot(tensors, count, &dummy, 0, out, epi, &cp)) continue;
            if (!plan_batch(tensors, count, &dummy, 0, batch, out, epi, &cp)) epi.norm_w = nullptr;
        }
        if (!plan_chunk(tensors, count, &dummy, 0, batch, out, epi, &cp)) { fail("not planned", t, batch); continue; }
        if (!lds_fits(cp)) fail("over LDS", t, batch);
        if (cp.partials <= rule.partials && cp.counters <= rule.counters) continue;
        Cut cut;
        if (!cut_within(tensors, count, &dummy, batch, out, epi, rule.partials, rule.counters, &cut)) {
            fail("cannot be captured", t, batch);
            continue;
        }
        for (int i = 0; i < cut.pieces; ++i)
            if (!plan_chunk(tensors, count, &dummy, 0, piece_positions(batch, cut.pieces, i), out, epi, &cp, cut.room) ||
                cp.partials > rule.partials || cp.counters > rule.counters || !lds_fits(cp))
                fail("piece over the workspace or LDS", t, batch);
    }
}

} // namespace

int main(int argc, char **argv)
{
    if (argc != 2) return 2;
    int launches = 0;
    for (int f = 0; f < 4; ++f)
        for (int rows : kRows)
            for (int units : kUnits)
                for (int batch = 1; batch <= QMV_MAX_BATCH; ++batch) {
                    const QmvDeviceTensor t = tensor(f, rows, units);
                    if (!strcmp(argv[1], "scratch")) check_scratch(t, batch);
                    else if (!strcmp(argv[1], "capture")) check_capture(t, batch);
                    else return 2;
                    ++launches;
                }
    printf("%d launches, %d failures\n", launches, g_failures);
    return g_failures != 0;
}
