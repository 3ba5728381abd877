"""bench.py's cube workload on a small cube: with the tuner off it runs the
untuned assembly, with a knob of the colour-ordered one that assembly, and
says which."""
import json

import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("more,assembly", [([], "rows"), (["--stiff-shape", "9"], "msr+expansion"),
                                           (["--assembly", "1"], "operator")])
def test_untuned_bench_runs_the_default_assembly(monkeypatch, capsys, more, assembly):
    import bench
    monkeypatch.setattr("sys.argv", ["bench.py", "--n", "8", "--steps", "2", "--warmup", "1", "--cpu-n", "0",
                                     "--correction", "0", "--autotune", "0", "--time-budget", "0"] + more)
    bench.bench_cube(bench.parse_args())
    line = json.loads(capsys.readouterr().out.strip().splitlines()[-1])
    assert line["config"]["newton_assembly"] == assembly and line["steps"] == 2
    assert line["config"]["spmv_variant"] == "rows shared" and line["config"]["pcg_fused"] is True
