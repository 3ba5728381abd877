"""tune_spmv_xcd against a stand-in for the solver whose times the test
gives: the untuned product (-1, rows shared by waves) is among the
candidates, and the fastest pair of knobs is left in place."""
import pytest

from tahoe_amd import api, autotune


class Stub:
    def __init__(self, fastest):
        self.fastest = fastest
        self.knobs = {}

    def set_tuning(self, knob, value):
        self.knobs[knob] = value

    def timing_enable(self, on=True):
        pass

    timing_reset = synchronize = lambda self: None

    def timing(self):
        now = (self.knobs[api.TUNE_PCG_FUSED], self.knobs[api.TUNE_SPMV_XCD])
        return {"spmv_launches": 10, "spmv_ms": 1.0 if now == self.fastest else 2.0, "vector_ms": 0.5,
                "precond_ms": 0.0}


@pytest.mark.parametrize("fastest", [(1, -1), (0, -1), (0, 7), (1, 2)])
def test_fastest_product_is_left_in_place(fastest):
    s = Stub(fastest)
    t = autotune.tune_spmv_xcd(s, lambda: None)
    assert (s.knobs[api.TUNE_PCG_FUSED], s.knobs[api.TUNE_SPMV_XCD]) == fastest == (t["fused"], t["xcd"])
    assert len(t["ms_per_iteration"]) == 18


@pytest.mark.parametrize("nnd,mt,fused,precond,name", [
    (17 ** 3, "float", True, "jacobi", "k_split_spmv<float, 9>"), (64 * 640, "double", True, "block", "k_split_spmv<double, 5>"),
    (64 * 1536, "float", True, "jacobi", "k_split_spmv<float, 3>"), (17 ** 3, "float", True, "amg", None),
    (17 ** 3, "float", False, "jacobi", None), (64 * 1536 + 1, "float", False, "jacobi", None),
    (1 << 17, "double", False, "amg", "k_share_spmv<double>"), (129 ** 3, "float", False, "jacobi", "k_share_spmv<float>"),
    (129 ** 3, "double", False, "jacobi", None)])
def test_bench_names_the_untuned_product(nnd, mt, fused, precond, name):
    import bench
    assert bench.untuned_product(mt, fused, nnd, precond) == name
