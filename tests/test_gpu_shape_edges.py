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
from gpu_util import bf16_dev, dev, host, p, stream  # noqa: E402
from test_gpu_decode_shapes import bf16_rne_bits, rbf  # noqa: E402

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
