"""GPU test of what a program may capture after a smaller call: an op whose
own route needs no workspace and little scratch still sizes both for the calls
that take the other route, so they can be captured afterwards. In a child
process per pair, so that nothing else has sized them; replayed over new inputs."""
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
be, orc = sdhip.Backend(), Oracle()
what = sys.argv[1]

def linear32(M, N, K, dA, dW, dC):
    be.gemm_nt_f32(M, N, K, dA, K, dW, K, dC, N)
def linear16(M, N, K, dA, dW, dC):
    be.gemm_nt_bf16(M, N, K, dA, K, dW, K, dC, N)

if what in ('linear32', 'linear16', 'swiglu'):
    M, N, K = 100, 256, 512
    W = orc.randn((N, K), 2, 0.0, 1.0 / np.sqrt(K))
    if what != 'linear32':
        W = f32_to_bf16(W).reshape(N, K)
    dA, dW, dC = be.empty((M, K)), be.array(W), be.empty((M, N))
    op = linear32 if what == 'linear32' else linear16
    dA.upload(orc.randn((M, K), 1))
    if what == 'swiglu':
        y = be.empty((64, N))
        be.linear_swiglu(dA, dW, dW, y, 64, K, N)
    else:
        op(4, N, K, dA, dW, dC)  # a few rows
    be.capture_begin()
    op(M, N, K, dA, dW, dC)
    graph = be.capture_end()
    for i in range(4):
        A = orc.randn((M, K), 10 + i)
        dA.upload(A)
        be.call('sdh_zero', dC.ptr, dC.nbytes)
        be.graph_launch(graph)
        want, S = (orc.gemm_nt_f32 if what == 'linear32' else orc.gemm_nt_bf16)(A, W, None, None, False)
        assert_gemm(dC.download(), want, S, K + 2, '%%s replay %%d' %% (what, i))
        op(M, N, K, dA, dW, dC)
        be.synchronize()
else:
    N, Cin, Cout = 1, 64, 32
    w = orc.randn((Cout, Cin, 3, 3), 2, 0.0, 0.05)
    dw = be.array(w)
    small, large = 240, 300   # the patches of either are cut at 128 MB
    dx, out = be.randn((N, Cin, small, small), 3), be.empty((N, Cout, large, large))
    be.conv2d(dx, N, Cin, small, small, dw, Cout, 3, 3, None, 1, 1, out, small, small)
    dx = be.empty((N, Cin, large, large))
    be.capture_begin()
    be.conv2d(dx, N, Cin, large, large, dw, Cout, 3, 3, None, 1, 1, out, large, large)
    graph = be.capture_end()
    for i in range(3):
        x = orc.randn((N, Cin, large, large), 20 + i)
        dx.upload(x)
        be.call('sdh_zero', out.ptr, out.nbytes)
        be.graph_launch(graph)
        want, S = orc.conv2d(x, w, None, 1, 1)
        assert_gemm(out.download(), want, S, Cin * 9 + 2, 'conv replay %%d' %% i)
be.graph_destroy(graph)
print('captured ok', flush=True)
""" % (os.path.join(ROOT, "stablediffusion-cpp_amd"), os.path.join(ROOT, "oracle"), HERE)


@pytest.mark.parametrize("what", ["linear32", "linear16", "swiglu", "conv"])
def test_capture_after_a_smaller_call(what):
    r = subprocess.run([sys.executable, "-u", "-c", BODY, what], capture_output=True, text=True, timeout=100)
    print(r.stdout, r.stderr[-3000:])
    assert r.returncode == 0 and "captured ok" in r.stdout
