// Plain FP64 form with the reference's rounding: built with
// -ffp-contract=off -DHOWMHD_EXACT=1 (true divisions, reference evaluation
// order), so every value equals the one a reference CPU run built without
// FMA contraction computes.  Also the FP64 sample collection of the learned
// indicator (labels from these WENO weights).
#include "stage.hpp"

#if !HOWMHD_EXACT
#error "step_exact.hip is built with HOWMHD_EXACT=1"
#endif

namespace howmhd {

int stage_fp64(howmhd_gpu_ctx* c, int iw, double dt) { return launch_stage<double>(c, iw, dt); }

// Synchronises.  The sweep tells the host where it queued a tile, and the
// IEEE-division launch runs only then: empty, it and the gap before it took 6 us
// of a collection at 64^3 (55 -> 49 us) and 2 us at 30x20x25 (26.6 -> 24.9).
int collect_fp64(howmhd_gpu_ctx* c, int dir, float* X, float* y, float* logits) {
    unsigned nb = 0;
    SweepArgs<double> a = sweep_args<double, SW_COLLECT>(c, 1, c->qbuf[c->qid[0]], 1u << dir, &nb);
    a.feat = X;
    a.label = y;
    a.logit = logits;
    a.stats = nullptr;
    *c->fixhost = 0u;
    launch_sweep<double, SW_COLLECT>(c, a, nb);
    HCHECK(c, hipGetLastError());
    HCHECK(c, hipStreamSynchronize(c->stream));
    if (*(volatile unsigned*)c->fixhost) {
        launch_recompute<double, SW_COLLECT>(c, a);
        HCHECK(c, hipGetLastError());
        HCHECK(c, hipStreamSynchronize(c->stream));
    }
    return HOWMHD_OK;
}

}  // namespace howmhd
