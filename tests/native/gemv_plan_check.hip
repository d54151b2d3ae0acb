// gemv_plan_check.hip -- the kernel a GEMV launch takes (kq_gemv_plan.h), for
// the CPU tests: it launches nothing.  Built by inferno_hip.build into
// tests/native/_build/libsdig_check.so.
#include "kq_gemv_plan.h"

extern "C" int norm_takes_wide_of(int type, int nblk, int outer, int ncu)
{
    return ihip::norm_takes_wide(type, nblk, outer, ncu);
}

// waves, ring slots and steps of k_gemv_mdig's instantiation, and its groups
extern "C" void mdig_plan_of(int type, int outer, int nstep, int ncu, int *out)
{
    const int groups = ihip::mdig_groups(outer, nstep, ncu);
    const ihip::MdPlan p = ihip::mdig_plan(type, nstep, groups);
    out[0] = p.nw;
    out[1] = p.d;
    out[2] = p.maxs;
    out[3] = groups;
}

extern "C" int gate_up_takes_wide_of(int type, int nblk, int outer, int ncu)
{
    return ihip::gate_up_takes_wide(type, nblk, outer, ncu);
}

extern "C" int b32_takes_wide_of(int type, int inner)
{
    return ihip::b32_takes_wide(type, inner);
}
