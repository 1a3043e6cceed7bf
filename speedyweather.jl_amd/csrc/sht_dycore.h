// Launchers of the dry core's kernels (sht_dycore.hip).
#pragma once
#include "sht_internal.h"

namespace sht {

// Prognostic columns on the device: vorticity, divergence, temperature (E L columns each,
// member by member) and ln ps (E), columns of nharm coefficients one after another.
struct DryState {
    const float2 *vor, *div, *temp, *lnps;
};

int launch_dry_columns(const DevPlan *P, int nharm, const DryState &s, void *out, int L, int E, float radius,
                       void *stream);
int launch_dry_grid(const float *g, float *fields, const float *coslat_inv, const float *coriolis, int npoints, int L, int E,
                    float rinv, float r_dry, float kappa, void *stream);
int launch_dry_tendency(const DevPlan *P, int nharm, const void *s, const float2 *temp, const float *G, void *tend, int L,
                        int E, double radius, void *stream);
// The tendencies and the time step of a state in one kernel: S.now holds the state, S.prev the
// previous one where S.filter is set.
struct DryStep {
    DryState now, prev;
    const float *nu, *nu_div;
    float2 *now1, *next;
    float dt2, w1, w2;
    int filter;
};
int launch_dry_step(const DevPlan *P, int nharm, const void *s, const float *G, const DryStep &S, int L, int E,
                    double radius, void *stream);
int launch_dry_leapfrog(int nharm, const DryState &now, const DryState &prev, const void *tend, const float *nu,
                        const float *nu_div, void *now1, void *next, int L, int E, float dt2, float w1, float w2,
                        int filter, void *stream);

}  // namespace sht
