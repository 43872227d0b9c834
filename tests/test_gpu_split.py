"""GPU tests of the fp32 products on split fp16 operands (k_gemm_split.hip):
sdh_gemm_nt_f32 at sizes that it takes, and sdh_conv2d, against the float64
oracle within the rigorous fp32 summation bound, element by element: at the
edges of every tile, K remainders, parts of K, padding and strides; rows of
extreme scale; infinities and NaN (what fp32 gives); a run of pixels far
below the sample's largest value; a captured graph replayed after the scratch
block it uses has been outgrown; and an arena too small for the scratch."""
import os
import subprocess
import sys

import numpy as np
import pytest

from tolerances import assert_gemm

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


def run_gemm(be, orc, M, N, K, seed, lda=None, bias=True, acc=False, edit=None):
    lda = lda or K
    A = orc.randn((M, lda), seed)
    W = orc.randn((N, K), seed + 1, 0.0, 1.0 / np.sqrt(K))
    if edit:
        edit(A, W)
    b = orc.randn((N,), seed + 2) if bias else None
    c0 = orc.randn((M, N), seed + 3) if acc else None
    dC = be.array(c0) if acc else be.empty((M, N))
    be.gemm_nt_f32(M, N, K, be.array(A), lda, be.array(W), K, dC, N, be.array(b) if bias else None, acc)
    return dC.download(), A[:, :K], W, b, c0


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,lda,bias,acc", [
    (257, 300, 321, None, True, False),      # odd K and ld, 64 x 64 tiles
    (65, 63, 65, 70, False, True),           # one past a tile, one short, one past a step
    (16, 16, 64, None, True, True),          # the smallest that an unaligned call sends here
    (1024, 1032, 1000, 1004, True, True),    # 64 x 64 or 128 x 128, K not a multiple of 32
    (130, 4100, 2052, None, True, False),    # few rows
    (700, 260, 8192, None, False, False),    # parts of K
    (4097, 2049, 128, None, True, False),    # 128 x 128, one past the tiles (unaligned C rows)
    (3000, 5000, 160, None, True, True),     # 256 x 256 with remainders
    # rows that are not a multiple of 16 bytes: the split product at the sizes above that the library takes when aligned
    (1024, 1032, 1000, 1005, True, True), (130, 4100, 2052, 2053, True, False), (700, 260, 8191, None, False, False),
])
def test_gemm(be, orc, M, N, K, lda, bias, acc):
    got, A, W, b, c0 = run_gemm(be, orc, M, N, K, 4000 + M + K, lda, bias, acc)
    want, S = orc.gemm_nt_f32(A, W, b, c0, acc)
    assert_gemm(got, want, S, K + 2, f"split gemm {M}x{N}x{K}")


@pytest.mark.gpu
def test_gemm_rows_of_any_scale(be, orc):
    """Each row has its own exponent: 2^+-120, subnormal rows, a zero row, and
    rows whose values span 2^16 (the range that keeps every bit)."""
    def edit(A, W):
        A[::7] *= np.float32(2.0 ** 100)
        A[1::7] *= np.float32(2.0 ** -100)
        A[2] = np.float32(2.0 ** -140) * np.rint(A[2] * 100)  # subnormal, exact
        A[3] = 0
        A[4] *= np.float32(2.0) ** np.linspace(0, 16, A.shape[1]).astype(np.float32)
        W[5] *= np.float32(2.0 ** 20)
        W[6] *= np.float32(2.0 ** -20)

    got, A, W, b, _ = run_gemm(be, orc, 300, 333, 340, 4500, bias=False, edit=edit)
    want, S = orc.gemm_nt_f32(A, W, None, None, False)
    assert_gemm(got, want, S + 2.0 ** -126, 342, "rows of any scale")  # results below 2^-126 round to its grid


@pytest.mark.gpu
def test_gemm_infinities_and_nan(be, orc):
    """Rows that hold them give what fp32 gives; all others are untouched."""
    def edit(A, W):
        A[10, 3], A[11, 5], A[12, 7], A[12, 9] = np.inf, np.nan, np.inf, -np.inf
        W[200, 3] = -np.inf
        W[201] = 0
        W[:, 5][::2] = 0

    got, A, W, b, _ = run_gemm(be, orc, 300, 333, 340, 4600, edit=edit)
    with np.errstate(invalid="ignore"):
        want = A.astype(np.float64) @ W.astype(np.float64).T + b
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(got[np.isinf(want)], want[np.isinf(want)].astype(np.float32))
    fine = np.isfinite(want)
    with np.errstate(invalid="ignore"):
        S = np.abs(A.astype(np.float64)) @ np.abs(W.astype(np.float64)).T + np.abs(b)
    assert np.array_equal(np.isfinite(got), fine)
    assert_gemm(got[fine], want[fine], S[fine], 342, "beside rows that are not finite")


CONVS = [  # N, Cin, H, W, Cout, kh, kw, stride, pad
    (1, 1, 1, 1, 1, 1, 1, 1, 0), (3, 33, 17, 19, 65, 3, 3, 1, 1), (2, 64, 16, 16, 64, 3, 3, 1, 1),
    (1, 31, 12, 40, 129, 5, 3, 1, 2), (2, 70, 21, 23, 66, 3, 3, 2, 1), (1, 96, 9, 31, 40, 1, 3, 3, 2),
    (2, 40, 5, 5, 20, 3, 3, 1, 4),      # pixels that see padding only
    (1, 320, 33, 31, 100, 1, 1, 1, 0), (2, 260, 8, 8, 300, 3, 3, 1, 1),  # parts of K
    (1, 36, 300, 260, 257, 3, 3, 1, 1),  # 256 x 256 tiles over rows and runs of 256 pixels
    (1, 70, 200, 140, 128, 3, 3, 1, 1),  # 128 x 256
    (2, 4, 66, 62, 3, 3, 3, 1, 1),
]


@pytest.mark.gpu
@pytest.mark.parametrize("N,Cin,H,W,Cout,kh,kw,stride,pad", CONVS)
def test_conv(be, orc, N, Cin, H, W, Cout, kh, kw, stride, pad):
    x = orc.randn((N, Cin, H, W), 4700 + Cin + H) * np.exp2(np.arange(N, dtype=np.float32) * 9)[:, None, None, None]
    w = orc.randn((Cout, Cin, kh, kw), 4701 + Cout, 0.0, 1.0 / np.sqrt(Cin * kh * kw))
    b = orc.randn((Cout,), 4702)
    Ho, Wo = (H + 2 * pad - kh) // stride + 1, (W + 2 * pad - kw) // stride + 1
    out = be.empty((N, Cout, Ho, Wo))
    be.conv2d(be.array(x), N, Cin, H, W, be.array(w), Cout, kh, kw, be.array(b), stride, pad, out, Ho, Wo)
    want, S = orc.conv2d(x, w, b, stride, pad)
    assert_gemm(out.download(), want, S, Cin * kh * kw + 2, f"conv2d {x.shape} k{kh}x{kw} s{stride} p{pad}")


@pytest.mark.gpu
@pytest.mark.parametrize("special", [None, np.inf, np.nan])
def test_conv_far_pixels_and_specials(be, orc, special):
    """One value of 2^20 (or an infinity, or NaN) in a corner of an image whose
    far half lies at 2^-10: every output still within the fp32 bound of its own
    terms, and what sees the special value as fp32 has it."""
    N, Cin, H, W, Cout = 2, 40, 48, 50, 70
    x = orc.randn((N, Cin, H, W), 4800)
    x[:, :, H // 2:] *= np.float32(2.0 ** -10)
    x[1, 7, 2, 3] = 2.0 ** 20 if special is None else special
    w = orc.randn((Cout, Cin, 3, 3), 4801, 0.0, 0.05)
    b = np.zeros(Cout, np.float32)
    out = be.empty((N, Cout, H, W))
    be.conv2d(be.array(x), N, Cin, H, W, be.array(w), Cout, 3, 3, be.array(b), 1, 1, out, H, W)
    got = out.download()
    with np.errstate(invalid="ignore"):
        want, S = orc.conv2d(x, w, b, 1, 1)
    fine = np.isfinite(want)
    assert fine.sum() == want.size - (0 if special is None else 9 * Cout)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(got[np.isinf(want)], want[np.isinf(want)].astype(np.float32))
    assert_gemm(got[fine], want[fine], S[fine], Cin * 9 + 2, f"conv2d beside {special}")


@pytest.mark.gpu
@pytest.mark.parametrize("N,Sq,Skv,heads,kvh,d,causal", [
    (1, 450, 450, 1, 1, 512, False), (2, 70, 65, 4, 2, 160, True), (1, 333, 77, 8, 8, 160, False),
    (2, 257, 301, 6, 3, 130, True), (1, 129, 2100, 2, 1, 256, False), (1, 40, 4100, 1, 1, 200, True),
    (1, 33, 16390, 1, 1, 144, False),  # the widest softmax rows
])
@pytest.mark.parametrize("out16", [False, True])
def test_wide_attention(be, orc, N, Sq, Skv, heads, kvh, d, causal, out16):
    """Head dimensions above 128 through the score matrix: odd sizes, grouped
    heads, several samples, more keys than queries; the bar of the other routes."""
    q, k, v = (orc.randn(s, 5000 + i + d) for i, s in enumerate(((N, Sq, heads * d), (N, Skv, kvh * d), (N, Skv, kvh * d))))
    out = sdhip_array(be, (N, Sq, heads * d), out16)
    call = be.attention_bf16 if out16 else be.attention
    call(be.array(q), be.array(k), be.array(v), out, N, Sq, Skv, heads, kvh, d, causal)
    want = orc.attention(q, k, v, heads, causal, kvh)
    got = out.download()
    if out16:
        from oracle import bf16_to_f32

        got = bf16_to_f32(got).reshape(want.shape)
    bound = 1e-4 + (2.0 ** -8 * np.abs(want) if out16 else 0)  # bf16: half a step, 2^-9, and its neighbour
    assert np.all(np.abs(got - want) <= bound), float(np.max(np.abs(got - want) - bound))


def sdhip_array(be, shape, bits16):
    import sdhip

    return sdhip.DArray(be, shape, dtype=np.uint16 if bits16 else np.float32)


@pytest.mark.gpu
def test_wide_attention_specials(be, orc):
    """A query and a key with NaN, a value channel with an infinity: what they
    touch is not finite, as in fp32; the rest is untouched."""
    S, d = 150, 160
    q, k, v = (orc.randn((1, S, 2 * d), 5100 + i) for i in range(3))
    q[0, 20, 5] = np.nan        # row 20 of head 0
    k[0, 100, d + 3] = np.nan   # head 1: rows 100 and on, by the causal mask
    v[0, 50, 7] = np.inf        # head 0, channel 7: rows 50 and on
    out = be.empty((1, S, 2 * d))
    be.attention(be.array(q), be.array(k), be.array(v), out, 1, S, S, 2, 2, d, True)
    got = out.download()
    bad = np.zeros((1, S, 2 * d), bool)
    bad[0, 20, :d] = bad[0, 100:, d:] = bad[0, 50:, 7] = True
    assert np.array_equal(~np.isfinite(got), bad)
    assert np.all(got[0, [r for r in range(50, S) if r != 20], 7] == np.inf)
    q[0, 20, 5] = k[0, 100, d + 3] = v[0, 50, 7] = 0
    want = orc.attention(q, k, v, 2, True, 2)
    assert np.max(np.abs(got - want)[~bad]) <= 1e-4


@pytest.mark.gpu
def test_graph_keeps_its_scratch(be, orc):
    """A graph holds the scratch block of its capture: the block lives on when
    a larger one replaces it, and replays over new inputs stay right."""
    M, N, K = 1000, 1100, 1008
    W = orc.randn((N, K), 4901, 0.0, 1.0 / np.sqrt(K))
    dA, dW, dC = be.empty((M, K)), be.array(W), be.empty((M, N))
    be.gemm_nt_f32(M, N, K, dA.upload(orc.randn((M, K), 4900)), K, dW, K, dC, N)
    be.capture_begin()
    be.gemm_nt_f32(M, N, K, dA, K, dW, K, dC, N)
    graph = be.capture_end()
    try:
        x = be.randn((1, 64, 512, 512), 4902)
        y = be.empty((1, 64, 512, 512))
        w = be.randn((64, 64, 3, 3), 4903)
        for i in range(3):
            A = orc.randn((M, K), 4910 + i)
            dA.upload(A)
            be.conv2d(x, 1, 64, 512, 512, w, 64, 3, 3, None, 1, 1, y, 512, 512)
            be.graph_launch(graph)
            be.conv2d(x, 1, 64, 512, 512, w, 64, 3, 3, None, 1, 1, y, 512, 512)
            want, S = orc.gemm_nt_f32(A, W, None, None, False)
            assert_gemm(dC.download(), want, S, K, f"replay {i}")
    finally:
        be.graph_destroy(graph)


BODY = r"""
import sys
sys.path[:0] = [%r, %r, %r]
import numpy as np, sdhip
from oracle import Oracle
from tolerances import assert_gemm
MB = 1 << 20
be, orc = sdhip.Backend(), Oracle()
x = orc.randn((1, 64, 96, 96), 1); w = orc.randn((80, 64, 3, 3), 2, 0.0, 0.05); b = orc.randn((80,), 3)
A = orc.randn((2000, 1024), 4); W = orc.randn((600, 1024), 5, 0.0, 0.03)
dx, dw, db, dy = be.array(x), be.array(w), be.array(b), be.empty((1, 80, 96, 96))
dA, dW, dC = be.array(A), be.array(W), be.empty((2000, 600))
want, S = orc.conv2d(x, w, b, 1, 1)
wg, Sg = orc.gemm_nt_f32(A, W, None, None, False)
be.gemm_nt_f32(2000, 600, 1024, dA, 1024, dW, 1024, dC, 600)
assert_gemm(dC.download(), wg, Sg, 1026, 'gemm')
# what is left of the arena falls in turn below every size that the calls ask for
hold = []
for left in (0, 1, 2, 4, 8, 16):
    try:
        while True:
            hold.append(be.malloc(MB))
    except sdhip.SdhError as e:
        assert e.status == sdhip.SDH_ERR_OOM, e
    for _ in range(left):
        be.free(hold.pop())
    for f, n in ((lambda: be.conv2d(dx, 1, 64, 96, 96, dw, 80, 3, 3, db, 1, 1, dy, 96, 96), 'conv'),
                 (lambda: be.gemm_nt_f32(2000, 600, 1024, dA, 1024, dW, 1024, dC, 600), 'gemm')):
        be.call('sdh_zero', dy.ptr, dy.nbytes); be.call('sdh_zero', dC.ptr, dC.nbytes)
        try:
            f()
            if n == 'conv': assert_gemm(dy.download(), want, S, 578, 'conv with %%d MB left' %% left)
            else: assert_gemm(dC.download(), wg, Sg, 1026, 'gemm with %%d MB left' %% left)
            print(n, left, 'MB left: right', flush=True)
        except sdhip.SdhError as e:
            assert e.status == sdhip.SDH_ERR_OOM, e
            print(n, left, 'MB left: reported', flush=True)
for p in hold: be.free(p)
be.conv2d(dx, 1, 64, 96, 96, dw, 80, 3, 3, db, 1, 1, dy, 96, 96)
assert_gemm(dy.download(), want, S, 578, 'conv at the end')
print('small arena ok', flush=True)
""" % (os.path.join(ROOT, "stablediffusion-cpp_amd"), os.path.join(ROOT, "oracle"), HERE)


@pytest.mark.gpu
def test_small_arena():
    r = subprocess.run([sys.executable, "-u", "-c", BODY], capture_output=True, text=True, timeout=110,
                       env=dict(os.environ, SDH_ARENA_MB="160", SDH_ARENA_LIMIT_MB="160"))
    print(r.stdout, r.stderr[-3000:])
    assert r.returncode == 0 and "small arena ok" in r.stdout


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,acc", [
    (3000, 5000, 160, True), (4097, 2049, 128, False), (1024, 1033, 1000, False),  # 256, 128 and 64 wide tiles
    (700, 260, 8191, True),  # parts of K
])
def test_gemm_one_bad_row_and_column(be, orc, M, N, K, acc):
    """A NaN in a row of A and infinities in a row of W: the blocks of their
    results by fp32 FMAs, every other result untouched, also where C is added."""
    def edit(A, W):
        A[M // 2, K // 3] = np.nan
        W[N // 3] = np.abs(W[N // 3])
        W[N // 3, 5] = np.inf
        A[:, 5] = np.abs(A[:, 5]) + 0.1

    got, A, W, b, c0 = run_gemm(be, orc, M, N, K, 5200 + K, acc=acc, edit=edit)
    rows = np.unique(np.concatenate([np.arange(0, M, max(1, M // 50)), np.arange(M // 2 - 3, M // 2 + 4), [M - 1]]))
    A2 = A.copy()
    A2[M // 2, K // 3] = 0
    W2 = W.copy()
    W2[N // 3, 5] = 0
    want, S = orc.gemm_nt_f32(A2[rows], W2, b, c0[rows] if acc else None, acc)
    got = got[rows]
    at = list(rows).index(M // 2)
    assert np.all(np.isnan(got[at]))
    fine = np.ones(got.shape, bool)
    fine[at] = fine[:, N // 3] = False
    assert np.all(np.isposinf(np.delete(got[:, N // 3], at)))
    assert_gemm(got[fine], want[fine], S[fine], K + 2, f"beside bad rows {M}x{N}x{K}")


@pytest.mark.gpu
def test_conv_one_bad_pixel_in_parts(be, orc):
    """An infinity in one pixel and a NaN in one output channel's weights where
    K is cut into parts: nine pixels of every channel, all pixels of one."""
    N, Cin, H, W, Cout = 2, 260, 8, 8, 300
    x = orc.randn((N, Cin, H, W), 5300)
    w = orc.randn((Cout, Cin, 3, 3), 5301, 0.0, 0.02)
    want, S = orc.conv2d(x, w, None, 1, 1)
    x[1, 100, 3, 4] = np.inf
    w[77, 9, 1, 1] = np.nan
    out = be.empty((N, Cout, H, W))
    be.conv2d(be.array(x), N, Cin, H, W, be.array(w), Cout, 3, 3, None, 1, 1, out, H, W)
    got = out.download()
    bad = np.zeros(got.shape, bool)
    bad[:, 77] = True
    bad[1, :, 2:5, 3:6] = True
    assert np.array_equal(~np.isfinite(got), bad)
    assert np.all(np.isnan(got[:, 77]))
    assert_gemm(got[~bad], want[~bad], S[~bad], Cin * 9 + 2, "beside a bad pixel and channel")


def unlike_groups(orc, shape, axis, seed, spread, pattern):
    """Values whose channels (along axis) fall into a large and a small group,
    2^spread apart: interleaved, or two halves."""
    x = orc.randn(shape, seed)
    n = shape[axis]
    large = np.arange(n) % 2 == 0 if pattern == "interleaved" else np.arange(n) < n // 2
    scale = np.where(large, np.float32(2.0) ** spread, np.float32(1))
    return x * scale.reshape([-1 if i == axis else 1 for i in range(len(shape))]), large


@pytest.mark.gpu
@pytest.mark.parametrize("spread", [12, 20, 24, 28, 60])
@pytest.mark.parametrize("pattern", ["interleaved", "halves"])
@pytest.mark.parametrize("M,N,K", [(300, 333, 641), (2048, 1024, 640), (300, 260, 8191)])
def test_gemm_unlike_channels(be, orc, M, N, K, pattern, spread):
    """Rows whose channels differ by 2^spread, met by weights that ignore the
    large group in every other output and are its reciprocal in some: within
    the error of fp32 sums of the result's own terms. Bound: K roundings of
    2^-24 each of partial sums no larger than the result in the mean, which
    add up as their squares do, 2^-24 sqrt(K) of the result's norm."""
    def edit(A, W):
        scaled, large = unlike_groups(orc, A.shape, 1, 5400, spread, pattern)
        A[:] = scaled
        W[::2, large] = 0
        W[1::4, large] *= np.float32(2.0) ** -spread

    got, A, W, _, _ = run_gemm(be, orc, M, N, K, 5400 + K, bias=False, edit=edit)
    want = A.astype(np.float64) @ W.astype(np.float64).T
    for part in (np.s_[:, ::2], np.s_[:, 1::4], np.s_[:, 3::4]):
        err = np.linalg.norm(got[part] - want[part]) / np.linalg.norm(want[part])
        assert err <= 2.0 ** -24 * np.sqrt(K), (part, err)


@pytest.mark.gpu
@pytest.mark.parametrize("d", [160, 512])
def test_wide_attention_unlike_channels(be, orc, d):
    """Queries whose channels differ by 2^24 and keys that ignore the large
    ones, values of one channel spread by 2^24 over the keys: scores and
    outputs as fp32 gives them."""
    S = 200
    q, large = unlike_groups(orc, (1, S, d), 2, 5500, 24, "interleaved")
    k, v = orc.randn((1, S, d), 5501), orc.randn((1, S, d), 5502)
    k[:, :, large] = 0
    k[:, :, ~large] *= 2
    v[0, :, 7] *= np.where(np.arange(S) % 2 == 0, np.float32(2.0 ** 24), 1)
    out = be.empty((1, S, d))
    be.attention(be.array(q), be.array(k), be.array(v), out, 1, S, S, 1, 1, d, False)
    want = orc.attention(q, k, v, 1, False, 1)
    got = out.download()
    assert np.max(np.abs(np.delete(got - want, 7, 2))) <= 1e-4
    assert np.max(np.abs(got[..., 7] - want[..., 7])) <= 1e-5 * 2.0 ** 24


@pytest.mark.gpu
@pytest.mark.parametrize("spread", [12, 20, 28, 60])
@pytest.mark.parametrize("pattern", ["interleaved", "halves", "dim chunk"])
@pytest.mark.parametrize("N,Cin,H,W,Cout,k", [(1, 128, 20, 24, 70, 3), (3, 96, 9, 8, 66, 1), (2, 640, 8, 8, 260, 3)])
def test_conv_unlike_channels(be, orc, N, Cin, H, W, Cout, k, pattern, spread):
    """Channels that differ by 2^spread (within a chunk of 32, between chunks,
    one small chunk), met by weights that ignore the large ones, are their
    reciprocal, or are alike: the bound of test_gemm_unlike_channels."""
    if pattern == "dim chunk":
        x = orc.randn((N, Cin, H, W), 5600)
        large = np.arange(Cin) >= 32
        x[:, large] *= np.float32(2.0) ** spread
    else:
        x, large = unlike_groups(orc, (N, Cin, H, W), 1, 5600, spread, pattern)
    w = orc.randn((Cout, Cin, k, k), 5601, 0.0, 0.1)
    w[::3, large] = 0
    w[1::3, large] *= np.float32(2.0) ** -spread
    out = be.empty((N, Cout, H, W))
    be.conv2d(be.array(x), N, Cin, H, W, be.array(w), Cout, k, k, None, 1, k // 2, out, H, W)
    want, _ = orc.conv2d(x, w, None, 1, k // 2)
    got = out.download()
    for part in range(3):
        err = np.linalg.norm(got[:, part::3] - want[:, part::3]) / np.linalg.norm(want[:, part::3])
        assert err <= 2.0 ** -24 * np.sqrt(Cin * k * k), (part, err)


@pytest.mark.gpu
def test_conv_unlike_pixels(be, orc):
    """Image rows 2^26 apart inside one run of 256 pixels, a zero chunk of
    channels, a zero sample: each output within the error of its own terms."""
    N, Cin, H, W, Cout = 3, 96, 32, 16, 40
    x = orc.randn((N, Cin, H, W), 5700)
    x[:, :, 8:] *= np.float32(2.0 ** -26)
    x[:, 32:64] = 0
    x[2] = 0
    w = orc.randn((Cout, Cin, 3, 3), 5701, 0.0, 0.1)
    out = be.empty((N, Cout, H, W))
    be.conv2d(be.array(x), N, Cin, H, W, be.array(w), Cout, 3, 3, None, 1, 1, out, H, W)
    want, _ = orc.conv2d(x, w, None, 1, 1)
    got = out.download()
    assert np.all(got[2] == 0)
    for part in (np.s_[:2, :, :8], np.s_[:2, :, 9:]):
        err = np.linalg.norm(got[part] - want[part]) / np.linalg.norm(want[part])
        assert err <= 2.0 ** -24 * np.sqrt(Cin * 9), (part, err)


@pytest.mark.gpu
def test_conv_many_samples(be, orc):
    """More samples than the pack's table of exponents takes at once."""
    N, Cin, H, W, Cout = 700, 130, 3, 5, 24  # 5 chunks: 409 samples at a time, then 291
    x = orc.randn((N, Cin, H, W), 5800) * np.exp2(np.arange(N, dtype=np.float32) % 40)[:, None, None, None]
    w = orc.randn((Cout, Cin, 3, 3), 5801, 0.0, 0.03)
    b = orc.randn((Cout,), 5802)
    out = be.empty((N, Cout, H, W))
    be.conv2d(be.array(x), N, Cin, H, W, be.array(w), Cout, 3, 3, be.array(b), 1, 1, out, H, W)
    want, S = orc.conv2d(x, w, b, 1, 1)
    assert_gemm(out.download(), want, S, Cin * 9 + 2, "many samples")


@pytest.mark.gpu
@pytest.mark.parametrize("N,Cin,H,W,Cout,k", [(1, 70, 9, 11, 5, 1), (1, 2100, 3, 4, 9, 1), (2, 33, 6, 5, 7, 3),
                                              (1, 20, 24, 23, 6, 23), (1, 2000, 4, 4, 10, 3)])
def test_conv_weights_of_any_scale(be, orc, N, Cin, H, W, Cout, k):
    """Each output channel's weights have their own exponent, found per 32
    channels: 2^+-60, one large weight at the row's either end, zeros, subnormal
    weights, and rows that hold an infinity or NaN at either end."""
    x = orc.randn((N, Cin, H, W), 5900)
    w = orc.randn((Cout, Cin, k, k), 5901, 0.0, 0.1)
    flat = w.reshape(Cout, -1)
    flat[0] *= np.float32(2.0 ** 60)
    flat[1] *= np.float32(2.0 ** -60)
    flat[2, -1], flat[3, 0] = 1000, -1000
    flat[4] = 0
    bad = {}
    if Cout > 6:
        flat[5] = np.float32(2.0 ** -140) * np.rint(flat[5] * 1000)
    if Cout > 8:
        flat[7, -1], flat[8, 0] = np.inf, np.nan
        bad = {7, 8}
    out = be.empty((N, Cout, H, W))
    be.conv2d(be.array(x), N, Cin, H, W, be.array(w), Cout, k, k, None, 1, k // 2, out, H, W)
    got = out.download()
    with np.errstate(invalid="ignore"):
        want, S = orc.conv2d(x, w, None, 1, k // 2)
    for co in range(Cout):
        if co in bad:
            assert np.array_equal(np.isnan(got[:, co]), np.isnan(want[:, co]))
            assert not np.any(np.isfinite(got[:, co]) & ~np.isfinite(want[:, co]))
        else:
            assert_gemm(got[:, co], want[:, co], S[:, co] + 2.0 ** -126, Cin * k * k + 2, f"channel {co}")
