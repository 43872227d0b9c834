"""GPU test of the library GEMM's first call in a nearly full arena: its
workspace is never taken from memory that the call uses. A bf16 linear packs
its input into scratch, then asks for the 64 MB workspace; one child process
for each amount of room: neither fits, only the scratch fits, either fits but
not both, both fit. The call is right or reports SDH_ERR_OOM, and is right in
the last case."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

BODY = r"""
import sys
sys.path[:0] = [%r, %r, %r]
import numpy as np, sdhip
from oracle import Oracle, f32_to_bf16
from tolerances import assert_gemm
MB = 1 << 20
room = int(sys.argv[1])
be, orc = sdhip.Backend(), Oracle()
M, N, K = 8192, 512, 2048  # the packed input takes 32 MB
A = orc.randn((M, K), 1)
W = f32_to_bf16(orc.randn((N, K), 2, 0.0, 1.0 / np.sqrt(K))).reshape(N, K)
dA, dW, dC = be.array(A), be.array(W), be.empty((M, N))
keep, hold = be.malloc(room * MB), []
try:
    while True:
        hold.append(be.malloc(MB))
except sdhip.SdhError as e:
    assert e.status == sdhip.SDH_ERR_OOM, e
be.free(keep)
rows = np.arange(0, M, 61)
want, S = orc.gemm_nt_bf16(A[rows], W, None, None, False)
for i in range(2):
    be.call('sdh_zero', dC.ptr, dC.nbytes)
    try:
        be.gemm_nt_bf16(M, N, K, dA, K, dW, K, dC, N)
        assert_gemm(dC.download()[rows], want, S, K + 2, 'bf16 linear')
        print('right', flush=True)
    except sdhip.SdhError as e:
        assert e.status == sdhip.SDH_ERR_OOM, e
        print('reported', flush=True)
""" % (os.path.join(ROOT, "stablediffusion-cpp_amd"), os.path.join(ROOT, "oracle"), HERE)


@pytest.mark.parametrize("room", [20, 40, 70, 110])
def test_first_library_gemm(room):
    r = subprocess.run([sys.executable, "-u", "-c", BODY, str(room)], capture_output=True, text=True, timeout=100,
                       env=dict(os.environ, SDH_ARENA_MB="320", SDH_ARENA_LIMIT_MB="320"))
    print(r.stdout, r.stderr[-3000:])
    assert r.returncode == 0
    assert r.stdout.split() == ["right" if room == 110 else "reported"] * 2
