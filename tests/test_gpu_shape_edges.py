"""Kernels at the sizes where their tiles, vectors and splits end: each shape sits on or
next to an edge of the variant it reaches, against the CPU oracle (or numpy for exact
results)."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("needs a GPU", allow_module_level=True)

import aethermind_amd.native as N  # noqa: E402
import oracle_lib as O  # noqa: E402
from gpu_util import bf16_dev, bits_host, dev, empty, host, p, pack_weight, stream  # noqa: E402
from test_gpu_decode_shapes import act_rows, bf16_rne_bits, close, launched, rbf  # noqa: E402

L = N.lib()


@pytest.mark.parametrize("dt", [N.AM_DT_F32, N.AM_DT_BF16])
@pytest.mark.parametrize("n", [1, 7, 2048, 2049, 128256, 131073])
def test_argmax_vector_edges(n, dt):
    """Rows whose length is no whole number of 16-byte vectors (later rows then start
    unaligned), ties across blocks, NaN, infinities and an all-NaN row: the first index of
    the largest value, twice on one workspace."""
    rng = np.random.default_rng(n)
    x = rbf(rng.standard_normal((5, n), dtype=np.float32))
    x[1, :] = -np.inf
    x[2, rng.integers(0, n, 3)] = np.nan
    x[3, :] = np.nan
    for at in (n - 1, n // 2):  # equal maxima, the lower index wins
        x[4, at] = np.inf
    ref = [0 if np.isnan(r).all() else int(np.nanargmax(r)) for r in x]
    xd = dev(x) if dt == N.AM_DT_F32 else bf16_dev(bf16_rne_bits(x))
    wsb = L.am_gfx950_argmax_workspace_bytes(5)
    ws = torch.zeros(wsb, dtype=torch.uint8, device="cuda")
    for _ in range(2):
        out = torch.full((5,), -1, dtype=torch.int64, device="cuda")
        L.call("am_gfx950_argmax", N.ArgmaxArgs(p(xd), dt, 5, n, p(out), p(ws), wsb), stream())
        assert list(host(out)) == ref


@pytest.mark.parametrize("m,n,k", [(2, 1, 4), (16, 16, 16), (17, 33, 20), (48, 1376, 512), (31, 512, 1376),
                                   (257, 515, 8192), (600, 1027, 132)])
def test_linear_f32_rows(m, n, k):
    """fp32 rows x fp32 weights: both tile sizes, ragged rows, columns and k tails.  Bar:
    fp32 sums of k products in any order differ by at most k * 2^-24 of the sum of their
    magnitudes."""
    rng = np.random.default_rng(m * n + k)
    x = rng.standard_normal((m, k), dtype=np.float32)
    w = rng.standard_normal((n, k), dtype=np.float32)
    res = rng.standard_normal((m, n), dtype=np.float32)
    dw, keep = pack_weight(w, N.AM_WF_F32)
    xd, rd = dev(x), dev(res)
    out = empty((m, n), torch.float32)
    L.call("am_gfx950_linear", N.LinearArgs(p(xd), 0, m, dw, p(out), 0, None, 0), stream())
    assert launched().startswith("gemm_f32<"), launched()
    ref = x.astype(np.float64) @ w.astype(np.float64).T
    bar = k * 2.0 ** -24 * (np.abs(x).astype(np.float64) @ np.abs(w).astype(np.float64).T) + 1e-30
    assert (np.abs(host(out) - ref) <= bar).all()
    # in place on the residual: one more rounding, of the sum
    L.call("am_gfx950_linear", N.LinearArgs(p(xd), 0, m, dw, p(rd), 0, p(rd), 0), stream())
    assert (np.abs(host(rd) - (ref + res)) <= bar + 2.0 ** -23 * np.abs(ref + res)).all()
    del keep
