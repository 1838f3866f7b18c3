"""Tuning overrides that change how the kernels move data but not what they
compute give the same bits as the defaults: the down-weight copies of 1 to
3 tokens (TFM_DS_PREFETCH=1), the grouped GEMM's tile rows and waves
(TFM_GGEMM_TILE, TFM_GGEMM_DOWN_TILE, TFM_GGEMM_WAVES: every tile adds the
products of an output in the same order), the router's two forms
(TFM_ROUTER_SPLIT_MAX_TOKENS), either grouping of the decode GEMV path
(TFM_DECODE_GROUPING=slots/workgroup) and the weight prefetch depth of 64-row
tiles of at most 16 rows (TFM_GGEMM_FEW_ROWS=0/2). TFM_GGEMM_SB_LAYOUT is said
to have no effect. The overrides are read once per process, so each runs in a
child process."""
import os
import subprocess
import sys

import numpy as np
import pytest

from tests._knob_cases import outputs
from tests._util import log

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def default_outputs(gpu):
    return outputs()


TILES = [{"TFM_GGEMM_TILE": "64", "TFM_GGEMM_WAVES": "4"}, {"TFM_GGEMM_TILE": "64", "TFM_GGEMM_WAVES": "8"},
         {"TFM_GGEMM_TILE": "96"}, {"TFM_GGEMM_TILE": "128", "TFM_GGEMM_WAVES": "4"},
         {"TFM_GGEMM_TILE": "128", "TFM_GGEMM_WAVES": "8"}, {"TFM_GGEMM_TILE": "256"}, {"TFM_GGEMM_WAVES": "4"},
         {"TFM_GGEMM_DOWN_TILE": "96", "TFM_GGEMM_WAVES": "8"}, {"TFM_GGEMM_DOWN_TILE": "256"}]


@pytest.mark.parametrize("env", [{"TFM_DS_PREFETCH": "1"}, {"TFM_DECODE_GROUPING": "slots"},
                                 {"TFM_DECODE_GROUPING": "workgroup"}, {"TFM_GGEMM_FEW_ROWS": "0"},
                                 {"TFM_GGEMM_FEW_ROWS": "2"}, {"TFM_GGEMM_SB_LAYOUT": "1"},
                                 {"TFM_ROUTER_SPLIT_MAX_TOKENS": "0"},
                                 {"TFM_ROUTER_SPLIT_MAX_TOKENS": "1000"}] + TILES,
                         ids=lambda e: ",".join(f"{k}={v}" for k, v in e.items()))
def test_override_gives_default_bits(default_outputs, env, tmp_path):
    log(f"override {env}")
    path = tmp_path / "out.npz"
    res = subprocess.run([sys.executable, "-m", "tests._knob_cases", str(path)], cwd=ROOT,
                         env={**os.environ, **env}, capture_output=True, text=True, timeout=110)
    assert res.returncode == 0, res.stderr[-2000:]
    got = np.load(path)
    for k, ref in default_outputs.items():
        if not k.startswith("topk_"):
            np.testing.assert_array_equal(got[k], ref, err_msg=k)
    if "TFM_GGEMM_SB_LAYOUT" in env:
        assert "TFM_GGEMM_SB_LAYOUT=1 has no effect" in res.stderr
    # A top-k kernel of its own: to 192 tokens by itself, and as the override says.
    split = int(env.get("TFM_ROUTER_SPLIT_MAX_TOKENS", 192))
    for name, T in (("olmoe", 32), ("granite", 64), ("olmoe", 300), ("granite", 1000)):
        assert got[f"topk_{name}_{T}_4"] == (1 if T <= split else 0), (name, T)
