"""serve.footprint_bytes is an upper bound: the device memory that a batch
context takes, from its set-up to its converged solve, is no more than the
sum over the batch's requests, for both elements and precisions."""
import ctypes
import gc

import pytest

pytestmark = pytest.mark.gpu


def free_bytes():
    """Free device memory, by the HIP runtime that the library is linked to."""
    from tahoe_amd import api
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert api.lib().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


@pytest.mark.parametrize("form,precision", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("count,L", [(12, 48), (200, 16)])
def test_footprint_bounds_the_context(count, L, form, precision):
    from tahoe_amd import api, batch, rve, serve
    reqs = [rve.Request(i, L, form, 0.3, seed=40 + i) for i in range(count)]
    pk = batch.pack([r.problem() for r in reqs])
    api.init_device(0)
    gc.collect()                    # contexts that earlier tests left to the collector
    before = free_bytes()
    s = batch.make_solid(pk, formulation=form, precision=precision, precond=serve.precond_for(reqs[0]))
    try:
        batch.solve_one_step_partial(s, pk, s.opts(max_iterations=0, lin_rtol=1e-1, lin_maxit=20))
        used = before - free_bytes()
    finally:
        s.close()
    bound = sum(serve.footprint_bytes(r, precision) for r in reqs)
    print(f"# {count} x {L}^3 form {form} precision {precision}: {used / 1e9:.3f} GB of {bound / 1e9:.3f}", flush=True)
    assert used <= bound
    # (rows on the boundary are shorter: the bound is not far above either)
    assert used >= 0.7 * bound
