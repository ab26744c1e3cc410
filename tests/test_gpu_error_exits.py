"""A call whose kernels read or write the engine's pinned staging waits for them also when it ends with an error: the next
call overwrites the staging or frees it.  The errors are reported by stand-ins on the host (tests/host/failing_calls.c);
every kernel runs as usual."""
import json
import os
import shutil
import subprocess
import sys

import pytest

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(shutil.which("gcc") is None, reason="no host compiler")]
HERE = os.path.dirname(os.path.abspath(__file__))

CHILD = """
import ctypes, json, sys
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
import numpy as np
import gw_analysis_tools_amd as G
from gw_analysis_tools_amd import workloads as W
f = 20. + np.arange(400) * 2.
psd = W.analytic_psd(f)
ev = G.Event(f, [np.full(400, 1e-23 + 2e-23j)] * 2, [psd] * 2, [0, 1])
P = W.injection_params(40)
p = G.Params.from_buffer_copy(P[0].tobytes())
calls = {
    "likelihoods": lambda: G.loglike_batch(ev, P, G.IMRPHENOMD),
    "waveform": lambda: G.fourier_waveform(f, p, G.IMRPHENOMD),
    "response": lambda: G.fourier_detector_response(f, p, 1, G.IMRPHENOMD),
    "detection": lambda: G.create_coherent_GW_detection(f, p, [0, 1], G.IMRPHENOMD),
    "maximised": lambda: G.maximized_loglike_batch(ev, P, G.IMRPHENOMD),
    "fisher": lambda: G.fisher_batch(ev, P, G.IMRPHENOMD, G.BASIS_PHENOMD_FULL, 11, epsilon=1e-6),
}
for name, call in calls.items():
    call()
    out = {"call": name}
    for kind, k in (("hipGetLastError", 0), ("hipGetLastError", 1), ("rocfft_execute", 0), ("hipEventRecord", 0)):
        good = call()
        shim.arm(kind.encode(), k)
        try:
            call()
            error = False
        except G.GWHError:
            error = True
        out[kind + str(k)] = [shim.failures(), error, shim.waits_since_failure()]
        shim.arm(b"", 0)
        again = call()
        out["same"] = bool(out.get("same", True) and np.array_equal(np.asarray(good), np.asarray(again)))
    print(json.dumps(out), flush=True)
"""


@pytest.fixture(scope="module")
def outcomes(tmp_path_factory):
    d = tmp_path_factory.mktemp("exits")
    shim = str(d / "failing_calls.so")
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", os.path.join(HERE, "host", "failing_calls.c"), "-o", shim, "-ldl"],
                   check=True, timeout=60)
    r = subprocess.run([sys.executable, "-c", CHILD, shim], capture_output=True, text=True, timeout=100,
                       cwd=os.path.dirname(HERE))
    assert r.returncode == 0, r.stdout + r.stderr
    return {o["call"]: o for o in map(json.loads, r.stdout.splitlines())}


@pytest.mark.parametrize("call", ["likelihoods", "waveform", "response", "detection", "maximised", "fisher"])
def test_calls_that_fail_wait_for_their_kernels(outcomes, call):
    o = outcomes[call]
    assert o.pop("same") and o.pop("call") == call
    assert o["hipGetLastError0"][0] == 1 and o["hipGetLastError1"][0] == 1
    if call == "maximised":
        assert o["rocfft_execute0"][0] == 1
    if call == "fisher":
        assert o["hipEventRecord0"][0] == 1
    for failed, error, waits in o.values():
        assert not failed or (error and waits > 0), o
