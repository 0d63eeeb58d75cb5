"""The CPU entries of the bench line.  Without the reference's Eigen build the
timed baseline is recorded as skipped and the line still comes out, with the
matrix and the right-hand side compared with the oracle's assembly; a side that
is off is seen in the recorded difference."""
import json

import numpy as np
import pytest

import bench
import oracle as O


@pytest.mark.parametrize("planted", [0.0, 1e-3])
def test_line_without_the_reference(monkeypatch, planted):
    monkeypatch.setattr(O, "ref", lambda: None)
    orc = bench.OracleRun(2)
    vals, rhs = orc.assemble()
    vals = vals.copy()
    vals[5] += planted * np.abs(vals).max()
    x = np.zeros(orc.n_dofs)
    out = bench.cpu_block(2, 1e-10, {"fp64": x, "mixed": x}, vals, rhs, lambda *a: None)
    assert "not built" in out["cpu_baseline"]["skipped"] and "not built" in out["rel_err_vs_fp64_oracle"]["skipped"]
    assert out["matrix_rel_diff_vs_oracle"] == pytest.approx(planted, abs=1e-15)
    assert out["rhs_rel_diff_vs_oracle"] == 0.0
    json.dumps(bench.sig(out))
    with pytest.raises(RuntimeError, match="not built"):  # what needs the timed run still says so
        orc.run(1e-10, 1)
