// Persistent path-tracker kernel: one path per lane, flattened endgame state machine.
//
// Compiled by hipRTC together with the generated system functions of one homotopy
// (HCG_N, HCG_KIND, sysG_* / sysF_*).  Each lane repeatedly takes a path index from a
// device work queue (atomic counter), tracks it with one tracker step per loop
// iteration; finished lanes of a wave write their PathResult records and take their next
// paths together (hcg_sched.h).
//
// Algorithm (restated from the reference, same arithmetic contract as the oracle):
//   tracker            src/tracker.jl:517-996     predictor  src/predictor.jl:124-371
//   Newton corrector   src/newton_corrector.jl:55-286
//   linear algebra     src/linear_algebra.jl:88-885   weighted norm  src/norm.jl:101-234
//   valuation          src/valuation.jl:38-228    endgame  src/endgame_tracker.jl:260-911
#pragma once
#include "hcg_arith.h"
#include "hcgpu_types.h"
#include "hcg_kargs.h"
#include "hcg_sched.h"
#include "hcg_mlp_infer.h"
#include "hcg_tracker_body.h"

extern "C" __global__ void __launch_bounds__(64, HCG_WAVES_PER_EU) hcg_track_kernel(hcg_kargs a) {
    __shared__ unsigned short mlp_lds[HCG_MLP_NPARAMS];
    const unsigned short* mw = stage_mlp(a.mlp, a.opts, mlp_lds);
    Lane L;
    lane_setup(L, a, mw);
    LaneTotals T = {0, 0, 0, 0.0};
    const int refill = refill_threshold(a.opts);
    int phase = 0;  // 0: idle, 1: tracking, 2: path k has ended and is not closed yet
    int k = -1;
    while ((int)threadIdx.x < a.lanes) {
        const unsigned long long fetch = wave_refill_mask(phase != 1, refill);
        // the rest of an ended path's last step runs beside the other lanes' steps
        if (phase == 1 || (fetch && phase == 2 && lane_unfinished(L))) lane_iter(L);
        if (phase == 1) {
            if (lane_ended(L)) phase = 2;
        } else if (fetch) {  // else wait for more idle lanes of this wave
            const int kn = wave_fetch(fetch, a.next_path);
            if (phase == 2) lane_close(L, a, k, T);
            phase = 0;
            k = kn;
            if (k >= a.npaths) break;
            if (lane_begin(L, a, k)) phase = lane_ended(L) ? 2 : 1;
        }
    }
    wave_add(&a.counters[0], (unsigned long long)T.steps);
    wave_add(&a.counters[1], (unsigned long long)T.newton);
    wave_add(&a.counters[2], (unsigned long long)T.flops);
    wave_add(&a.counters[3], (unsigned long long)T.lacc);
}
