"""The streaming kernels as the device runs them by default (regrid with its
history behind the window, remap by pairs of fields, u/v walks with the
deepest-layer rule, Robert-Asselin u/v through the workspace), built for the
host, against the oracle, bitwise, over several steps on one state (the later
ones have massless bottom layers, whose points the u/v rule is about)."""
import ctypes

import pytest

import hostcheck_lib as hc
import hybgen_abi as abi
import oracle_lib as ol


def _step(P, d, m, n, raflag):
    lib = hc.lib()
    lib.hostcheck_stream_uv_fallback_points.restype = ctypes.c_int64
    assert lib.hostcheck_hybgen_stream_dev(ctypes.byref(P), ctypes.byref(d.fields()), m, n,
                                           raflag) == 0
    return lib.hostcheck_stream_uv_fallback_points()


@pytest.mark.parametrize("raflag", [0, 1])
@pytest.mark.parametrize("kdm,hybmap,ntracr,hybiso,extreme", [
    (4, 2, 0, 0.01, 0), (5, 3, 1, 0.01, 1), (7, 0, 2, 0.01, 0), (16, 2, 0, 0.01, 0),
    (22, 1, 3, 3.0, 1), (32, 2, 2, 0.01, 0), (41, 3, 0, 0.01, 0), (64, 2, 1, 0.01, 1),
])
def test_device_variants_match_oracle(kdm, hybmap, ntracr, hybiso, extreme, raflag):
    few = {"nsigma": kdm} if kdm < 16 else {}
    P, w = abi.workload_params("cfg1", idm=41, jdm=33, kdm=kdm, hybmap=hybmap, ntracr=ntracr,
                               trcflg=[2, 0, 0][:ntracr], **few)
    P.hybiso = hybiso
    got = abi.HostDomain(P).synth(abi.make_synth(P, w, seed=kdm, extreme=extreme))
    want = got.copy()
    for step in range(3):
        ol.run_oracle(want, m=1, n=2, raflag=raflag, threads=8)
        _step(P, got, 1, 2, raflag)
        df = ol.diff_domains(want, got)
        assert not df, f"step {step}: {df}"


@pytest.mark.parametrize("kdm,idm,jdm", [(16, 40, 30), (32, 150, 100), (22, 120, 90)])
def test_massless_bottoms_stay_in_the_walk(kdm, idm, jdm):
    P, w = abi.workload_params("cfg1", idm=idm, jdm=jdm, kdm=kdm, ntracr=0)
    d = abi.HostDomain(P).synth(abi.make_synth(P, w, seed=5))
    for _ in range(3):
        assert _step(P, d, 1, 2, 0) == 0


def test_robert_asselin_points_take_the_workspace():
    # stepped on one state, a sixth of the level-m points cannot go in place
    P, w = abi.workload_params("glbb", idm=100, jdm=80, kdm=41, ntracr=0)
    d = abi.HostDomain(P).synth(abi.make_synth(P, w, seed=5))
    want = d.copy()
    for _ in range(2):
        ol.run_oracle(want, m=1, n=2, raflag=1, threads=8)
        assert _step(P, d, 1, 2, 1) == 0
        assert not ol.diff_domains(want, d)


@pytest.mark.parametrize("kdm,hybmap,zlevel", [(4, 2, 0), (16, 1, 1), (27, 3, 0), (41, 2, 1),
                                               (64, 0, 0)])
def test_denfix_search_matches_oracle(kdm, hybmap, zlevel):
    few = {"nsigma": kdm} if kdm < 16 else {}
    P, w = abi.workload_params("cfg1", idm=43, jdm=31, kdm=kdm, hybmap=hybmap, ntracr=1,
                               ldenfix=1, **few)
    got = abi.HostDomain(P).synth(abi.make_synth(P, w, seed=kdm))
    if zlevel:
        ol.zlevel_start(got, seed=kdm)
    want = got.copy()
    for step in range(3):
        ol.run_oracle(want, m=1, n=2, threads=8)
        _step(P, got, 1, 2, 0)
        assert not ol.diff_domains(want, got), f"step {step}"
