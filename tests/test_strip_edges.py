"""The stage kernel's strips and segments at the sizes where their counts
change: the smallest marched panel, a panel one strip wide exactly and one
column more, the second and third strip, segments whose rows do not divide the
panel.  On the CPU the kernels run under AddressSanitizer against the oracle
(bars 1e-12 in FP64, 2e-5 in FP32); on the GPU one operator application
against the oracle, also at sizes whose segments have more rows."""
import os
import subprocess

import numpy as np
import pytest

from test_emu_kernels import emu_exe  # noqa: F401  (fixture)

EDGES = [(10, 42, 64), (11, 42, 64), (13, 21, 32), (63, 42, 32), (64, 42, 64), (122, 42, 32), (176, 21, 32)]


@pytest.mark.parametrize("N,order,prec", EDGES)
def test_strip_edges_under_asan(emu_exe, N, order, prec):  # noqa: F811
    env = dict(os.environ, ASAN_OPTIONS="detect_leaks=0:abort_on_error=0:halt_on_error=1")
    res = subprocess.run([emu_exe, "apply", str(N), str(order), str(prec), "1", str(N), "0"], capture_output=True,
                         text=True, timeout=600, env=env)
    out = res.stdout + res.stderr
    assert "AddressSanitizer" not in out, out[-4000:]
    assert res.returncode == 0 and res.stdout.rstrip().endswith("ok"), out[-4000:]


@pytest.mark.gpu
@pytest.mark.parametrize("N,order,prec", [(11, 42, 64), (63, 21, 64), (64, 42, 64), (121, 42, 64), (122, 42, 64),
                                          (173, 42, 64), (174, 42, 64), (178, 42, 64), (191, 42, 64), (200, 42, 64),
                                          (235, 42, 64), (236, 21, 64), (256, 21, 64), (260, 42, 32)])
def test_strip_edges_match_oracle(oracle_mod, N, order, prec):
    import ch_swe_amd as cs
    from oracle.swe_oracle import MESH_U, MESH_V, MESH_XY

    print(f"strip edges N={N} order={order} fp{prec}", flush=True)
    o = oracle_mod.Oracle(N, order)
    rng = np.random.default_rng(N)
    state = [rng.standard_normal(o.shape(m)) for m in (MESH_U, MESH_V, MESH_XY)]
    op = cs.create_linear_swm_operator(N, order, cs.FP64 if prec == 64 else cs.FP32)
    vin, vout = op.create_stvec(), op.create_stvec()
    vin.upload(*state)
    op.apply(vout, vin)
    for g, r in zip(vout.download(), o.apply(*state)):
        assert np.abs(g - r).max() / np.abs(r).max() < (1e-12 if prec == 64 else 2e-5)
