"""GPU tests of conv2d's patch-gather route, which runs where the implicit
GEMM's scratch cannot be had, in a child process whose arena holds exactly the
room that the patches need: the product of a chunk at sizes that the fp32
linear sends to its split operands on its own (many output channels; rows that
are not a multiple of 16 bytes; a second chunk and a second sample at an
unaligned place), eagerly and captured, and beside a live graph. 1x1 kernels, so float64 matrix
products on the host are the reference; within the fp32 summation bound."""
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
from oracle import Oracle
from tolerances import assert_gemm
MB = 1 << 20
be, orc = sdhip.Backend(), Oracle()

def fill(room):
    '''Leaves one free range of `room` megabytes in the arena.'''
    keep = be.malloc(room * MB)
    hold = []
    try:
        while True:
            hold.append(be.malloc(MB))
    except sdhip.SdhError as e:
        assert e.status == sdhip.SDH_ERR_OOM, e
    be.free(keep)
    return hold

def inputs(N, Cin, H, W, Cout, seed):
    x = orc.randn((N, Cin, H, W), seed)
    w = orc.randn((Cout, Cin, 1, 1), seed + 1, 0.0, 1.0 / np.sqrt(Cin))
    b = orc.randn((Cout,), seed + 2)
    return x, w, b

def check(got, x, w, b, what):
    N, Cin, H, W = x.shape
    w2 = w.reshape(len(w), Cin).astype(np.float64)
    for n in range(N):
        x2 = x[n].reshape(Cin, H * W).astype(np.float64)
        want = w2 @ x2 + b[:, None]
        S = np.abs(w2) @ np.abs(x2) + np.abs(b)[:, None]
        assert_gemm(got[n].reshape(want.shape), want, S, Cin + 2, '%%s, sample %%d' %% (what, n))

def conv(dx, x, dw, w, db, out):
    N, Cin, H, W = x.shape
    be.conv2d(dx, N, Cin, H, W, dw, len(w), 1, 1, db, 1, 0, out, H, W)

# the library GEMM's workspace, before the arena is full
be.gemm_nt_f32(64, 64, 64, be.randn((64, 64), 1), 64, be.randn((64, 64), 2), 64, be.empty((64, 64)), 64)
be.synchronize()

# N, Cin, H, W, Cout, room in MB: patches fit it, the split operands do not
for N, Cin, H, W, Cout, room in ((2, 65, 97, 95, 20, 3), (1, 68, 296, 292, 256, 28), (1, 68, 703, 703, 64, 140)):
    x, w, b = inputs(N, Cin, H, W, Cout, 9000 + H)
    dx, dw, db, out = be.array(x), be.array(w), be.array(b), be.empty((N, Cout, H, W))
    hold = fill(room)
    for i in range(2):
        be.call('sdh_zero', out.ptr, out.nbytes)
        conv(dx, x, dw, w, db, out)
        check(out.download(), x, w, b, 'gather %%s' %% (x.shape,))
    print('gather', x.shape, Cout, 'right', flush=True)
    for p in hold: be.free(p)
    del dx, dw, db, out

# captured: the block is the patches' size, and may not grow
N, Cin, H, W, Cout = 1, 65, 97, 95, 20
x, w, b = inputs(N, Cin, H, W, Cout, 9500)
dx, dw, db, out = be.array(x), be.array(w), be.array(b), be.empty((N, Cout, H, W))
hold = fill(3)
conv(dx, x, dw, w, db, out)
be.capture_begin()
conv(dx, x, dw, w, db, out)
graph = be.capture_end()
for i in range(3):
    x = orc.randn((N, Cin, H, W), 9510 + i)
    dx.upload(x)
    be.call('sdh_zero', out.ptr, out.nbytes)
    be.graph_launch(graph)
    check(out.download(), x, w, b, 'captured, replay %%d' %% i)
used = be.memory_stats()[1]
for i in range(5):  # with a graph alive: refused again each time, and nothing more held
    be.call('sdh_zero', out.ptr, out.nbytes)
    conv(dx, x, dw, w, db, out)
    check(out.download(), x, w, b, 'beside a graph')
    assert be.memory_stats()[1] == used
be.graph_destroy(graph)
print('gather route ok', flush=True)
""" % (os.path.join(ROOT, "stablediffusion-cpp_amd"), os.path.join(ROOT, "oracle"), HERE)


def test_gather_route():
    r = subprocess.run([sys.executable, "-u", "-c", BODY], capture_output=True, text=True, timeout=110,
                       env=dict(os.environ, SDH_ARENA_MB="900", SDH_ARENA_LIMIT_MB="900"))
    print(r.stdout, r.stderr[-3000:])
    assert r.returncode == 0 and "gather route ok" in r.stdout
