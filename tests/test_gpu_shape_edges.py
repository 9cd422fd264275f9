"""Kernels at the sizes where their tiles, vectors and splits end: each shape sits on or
next to an edge of the variant it reaches, against the CPU oracle (or numpy for exact
results)."""

import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("needs a GPU", allow_module_level=True)

import aethermind_amd.native as N  # noqa: E402
import oracle_lib as O  # noqa: E402
from gpu_util import bf16_dev, dev, empty, host, p, pack_weight, stream, zeros  # noqa: E402
from test_gpu_decode_shapes import act_rows, bf16_rne_bits, launched, rbf  # noqa: E402

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
    magnitudes.  Small integers, whose sums are exact in any order: every bit."""
    rng = np.random.default_rng(m * n + k)
    xi, wi, ri = (rng.integers(-8, 9, s).astype(np.float32) for s in ((m, k), (n, k), (m, n)))
    di, keep = pack_weight(wi, N.AM_WF_F32)
    xd, rd, out = dev(xi), dev(ri), empty((m, n), torch.float32)
    ref = xi.astype(np.float64) @ wi.astype(np.float64).T
    L.call("am_gfx950_linear", N.LinearArgs(p(xd), 0, m, di, p(out), 0, None, 0), stream())
    L.call("am_gfx950_linear", N.LinearArgs(p(xd), 0, m, di, p(rd), 0, p(rd), 0), stream())
    assert np.array_equal(host(out), ref) and np.array_equal(host(rd), ref + ri)
    del keep
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


@pytest.mark.parametrize("m,n,k", [(48, 1376, 512), (48, 512, 1376), (300, 2048, 520), (17, 4096, 8192)])
def test_linear_f32_rows_error(m, n, k):
    """The fp32 GEMM's error against fp64 (both tile sizes) is no larger than that of the
    GEMV per row: rms over all elements, with 5% for the sampling of two rms of at least
    65,000 elements each (below 1%) and the elements that share an operand row."""
    rng = np.random.default_rng(k)
    x, w = (dev(rng.standard_normal(s, dtype=np.float32)) for s in ((m, k), (n, k)))
    dw, keep = pack_weight(host(w), N.AM_WF_F32)
    ref = x.double() @ w.double().T
    rms = []
    for mode in (0, 1):
        out = empty((m, n), torch.float32)
        L.call("am_gfx950_linear", N.LinearArgs(p(x), 0, m, dw, p(out), 0, None, mode), stream())
        assert launched().startswith("gemm_f32<" if mode == 0 else "gemv<"), launched()
        rms.append(float((out.double() - ref).square().mean().sqrt()))
    assert rms[0] <= 1.05 * rms[1], rms
    del keep


def exact_weight(rng, n, k, fmt, group=128):
    """A device weight of small integers with power-of-two scales (INT4: a zero one here and
    there), and its values: products with small integers sum exactly in fp32, in any order
    and from any partial sum that the kernels keep."""
    if fmt == N.AM_WF_INT4:
        codes = rng.integers(0, 256, (n, k // 2), dtype=np.uint8)
        sc = np.exp2(-rng.integers(4, 7, (n, k // group)).astype(np.float32)).astype(np.float16)
        sc[rng.random(sc.shape) < 0.03] = 0
        logical, scales = dev(codes), dev(sc.view(np.int16))
        data, dsc = zeros((n * k // 2,), torch.uint8), zeros((n * (k // group),), torch.int16)
        dw = N.Weight(p(data), p(dsc), n, k, fmt, group)
        L.call("am_gfx950_pack_int4", N.PackInt4Args(p(logical), p(scales), dw), stream())
        q = np.stack([codes & 15, codes >> 4], -1).reshape(n, k).astype(np.int8)
        w = dev(np.where(q > 7, q - 16, q).astype(np.int8)).double() * dev(np.repeat(sc.astype(np.float32), group, 1)).double()
        return dw, w, (logical, scales, data, dsc)
    if fmt == N.AM_WF_INT8:
        q = rng.integers(-127, 128, (n, k), dtype=np.int16)
        sc = np.exp2(-rng.integers(4, 7, n).astype(np.float32))
        data, dsc = dev((q + 128).astype(np.uint8)), dev(sc)
        return N.Weight(p(data), p(dsc), n, k, fmt, 0), dev(q).double() * dsc.double()[:, None], (data, dsc)
    w = rng.integers(-8, 9, (n, k)).astype(np.float32)
    dw, keep = pack_weight(w, fmt)
    return dw, dev(w).double(), keep


# (m, n, k, group): rows and columns on both sides of the 64- and 128-row tiles of every
# weight format, one k step, an odd number of groups, groups of one, two and four 64-value
# steps (the 256-row tile and the splits are pinned by test_prefill_gemm_exact)
TILE_SHAPES = [(1, 64, 128, 128), (65, 72, 384, 128), (256, 4104, 640, 128), (257, 16392, 384, 128),
               (513, 28680, 512, 256), (300, 8200, 1024, 64), (1030, 6152, 2048, 128)]


@pytest.mark.parametrize("shape", TILE_SHAPES)
@pytest.mark.parametrize("fmt", [N.AM_WF_INT4, N.AM_WF_INT8, N.AM_WF_BF16])
def test_prefill_gemm_tiles(shape, fmt):
    """Every element against the fp64 product of the dequantized weights.  Bar: half a
    bf16 ulp of the result (2^-8 relative, generously) and k * 2^-24 of the summed
    magnitudes for the fp32 sums."""
    m, n, k, group = shape
    rng = np.random.default_rng(m + n)
    w = rbf(rng.standard_normal((n, k), dtype=np.float32) * np.float32(0.02))
    if group <= k // 2:
        w[::7, :group] = 0.0  # whole groups of zero scale
        w[3::7, group:2 * group] *= 1e-3  # neighbouring groups of very different scales
    dw, keep = pack_weight(w, fmt, group)
    if fmt == N.AM_WF_INT4:
        pk, sc = O.quant_int4(w, group)
        w = O.dequant_int4(pk, sc, k, group)
    elif fmt == N.AM_WF_INT8:
        w = O.dequant_int8(*O.quant_int8(w))
    x = act_rows(7, m, k)
    xd, wd = bf16_dev(bf16_rne_bits(x)), dev(w)
    xt = dev(x).double()
    ref, mag = xt @ wd.double().T, xt.abs() @ wd.double().abs().T
    nbytes = L.am_gfx950_gemm_workspace_bytes(m, n, k, group if fmt == N.AM_WF_INT4 else 128)
    ws = torch.zeros(max(nbytes, 16), dtype=torch.uint8, device="cuda")
    for use_ws in (False, True):
        out = empty((m, n), torch.bfloat16)
        args = N.LinearArgs(p(xd), N.AM_DT_BF16, m, dw, p(out), N.AM_DT_BF16, None, 2)
        if use_ws and nbytes:
            args.workspace, args.workspace_bytes = p(ws), nbytes
        L.call("am_gfx950_linear", args, stream())
        err = (out.double() - ref).abs()
        bar = ref.abs() * 2.0 ** -8 + mag * (k * 2.0 ** -24) + 1e-30
        assert bool((err <= bar).all()), (launched(), float((err - bar).max()))
    del keep


# (epilogue, m, n, k), and the (tile rows, tile columns, splits) it reaches: all formats, or
# INT4 and INT8, then bf16.  Ragged rows and columns in every tile; the 8B down projection
# and chunks of its kind are where the 256-row tile and its splits are used.
ALL = (N.AM_WF_INT4, N.AM_WF_INT8, N.AM_WF_BF16)
EXACT_TILES = [("store", 100, 1032, 14336, (64, 64, 8)), ("residual", 65, 72, 2048, (64, 64, 2)),
               ("silu", 100, 2048, 4096, (64, 128, 4)), ("store", 300, 2168, 8192, (128, 128, 4)),
               ("residual", 515, 4104, 14336, (128, 256, 2), (256, 256, 4)), ("silu", 750, 28672, 512, (128, 256, 1)),
               ("store", 1030, 12296, 512, (256, 256, 1)), ("residual", 1030, 4088, 14336, (256, 256, 2)),
               ("silu", 1000, 28672, 512, (256, 256, 1))]


@pytest.mark.skipif(torch.cuda.get_device_properties(0).multi_processor_count != 256, reason="tiles of 256 CUs")
@pytest.mark.parametrize("case", EXACT_TILES, ids=lambda c: f"{c[0]}-{c[1]}-{c[2]}-{c[3]}")
@pytest.mark.parametrize("fmt", ALL)
def test_prefill_gemm_exact(case, fmt):
    """Operands whose sums are exact: a store is the rounded product to the bit, a residual
    the rounded sum, SiLU-Mul within a rounding and fp32 exponentials of the value from the
    rounded halves.  The launch's grid and name tell the tile; twice on one workspace."""
    epi, m, n, k = case[:4]
    bm, bn, splits = case[-1] if fmt == N.AM_WF_BF16 else case[4]
    rng = np.random.default_rng(m + n)
    dw, w, keep = exact_weight(rng, n, k, fmt)
    x, h = (rng.integers(-4, 5, sh).astype(np.float32) for sh in ((m, k), (m, n)))
    xd, acc = bf16_dev(bf16_rne_bits(x)), (dev(x).double() @ w.T).float().bfloat16()
    nbytes = L.am_gfx950_gemm_workspace_bytes(m, n, k, 128)
    ws = zeros((max(nbytes, 16),), torch.uint8)
    none = (N.vp * 3)(None, None, None)
    for _ in range(2):
        if epi == "silu":
            out = empty((m, n // 2), torch.bfloat16)
            none[0] = p(out)
            L.call("am_gfx950_prefill_linear", N.PrefillLinearArgs(p(xd), m, dw, N.AM_PREFILL_SILU_MUL, none, (N.i64 * 2)(0, 0),
                                                                   p(ws), nbytes, None), stream())
            gate, up = acc[:, :n // 2].double(), acc[:, n // 2:].double()
            ref = torch.nn.functional.silu(gate) * up
            # (where fp32's exponential overflows silu is below 2^-121, and 0)
            bar = ref.abs() * (2.0 ** -8 + 2.0 ** -20) + up.abs() * 2.0 ** -121
            over = int(((out.double() - ref).abs() > bar).sum())
            assert over == 0, over
        else:
            out = bf16_dev(bf16_rne_bits(h)).view(torch.bfloat16).view(m, n)
            res = p(out) if epi == "residual" else None
            L.call("am_gfx950_linear", N.LinearArgs(p(xd), N.AM_DT_BF16, m, dw, p(out), N.AM_DT_BF16, res, 2, p(ws), nbytes),
                   stream())
            ref = (dev(h) + acc.float()).bfloat16() if res else acc
            assert torch.equal(out, ref), int((out != ref).sum())
        info = N.last_launch()
        tiles = -(-m // bm) * -(-n // bn)
        assert f"bn={bn},splits={splits}>" in info.kernel.decode() and info.grid == tiles * splits, (info.kernel, info.grid)
        assert not bool(ws[:4096].any())
    del keep


@pytest.mark.parametrize("fmt", ALL)
def test_prefill_gemm_rope_largest_tile(fmt):
    """The q|k|v epilogue in the 256 x 256 tile with a ragged last row tile: bit for bit the
    column split, am_gfx950_rope and am_gfx950_kv_update."""
    m, start, cap, hq, hkv, d, H = 2049, 63, 2176, 32, 8, 128, 512
    rng = np.random.default_rng(12)
    dw, w, keep = exact_weight(rng, (hq + 2 * hkv) * d, H, fmt)
    xd = bf16_dev(bf16_rne_bits(rng.integers(-4, 5, (m, H)).astype(np.float32)))
    cd, sd = (dev(t) for t in O.rope_tables(cap, d, 10000.0))
    startd, posd = dev(np.array([start], np.int64)), torch.arange(start, start + m, dtype=torch.int64, device="cuda")
    planes = [zeros((hkv * cap * d,), torch.int16) for _ in range(4)]
    qf, q, k, v = (empty((m, c * d), torch.int16) for c in (hq, hq, hkv, hkv))
    r = N.PrefillRopeKv(p(cd), p(sd), cap, p(startd), p(planes[0]), p(planes[1]), hq, hkv, d, cap, None, None)
    L.call("am_gfx950_prefill_linear", N.PrefillLinearArgs(p(xd), m, dw, N.AM_PREFILL_QKV_ROPE_KV, (N.vp * 3)(p(qf), None, None),
                                                           (N.i64 * 2)(0, 0), None, 0, C.pointer(r)), stream())
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        assert "qkv_rope_kv,bn=256" in launched() and N.last_launch().grid == 9 * 24, launched()
    L.call("am_gfx950_prefill_linear", N.PrefillLinearArgs(p(xd), m, dw, N.AM_PREFILL_SPLIT, (N.vp * 3)(p(q), p(k), p(v)),
                                                           (N.i64 * 2)(hq * d, (hq + hkv) * d)), stream())
    L.call("am_gfx950_rope", N.RopeArgs(p(q), p(k), p(q), p(k), p(posd), p(cd), p(sd), m, hq, hkv, d, cap, N.AM_DT_BF16), stream())
    L.call("am_gfx950_kv_update", N.KvUpdateArgs(p(k), p(v), p(planes[2]), p(planes[3]), m, hkv, d, cap, 0, p(startd),
                                                 N.AM_DT_BF16, None, None), stream())
    assert torch.equal(qf, q) and torch.equal(planes[0], planes[2]) and torch.equal(planes[1], planes[3])
    acc = (xd.view(torch.bfloat16).view(m, H).double() @ w.T).float().bfloat16()
    assert torch.equal(v.view(torch.bfloat16), acc[:, (hq + hkv) * d:])
    del keep


@pytest.mark.parametrize("m,n,k,group", [(70, 256, 512, 128), (300, 512, 512, 64), (257, 16392, 384, 128),
                                         (1030, 12296, 512, 128)])
@pytest.mark.parametrize("size", [1.0, 2.0 ** 80])
def test_prefill_gemm_zero_scale_groups(m, n, k, group, size):
    """INT4 groups whose scale is zero but whose codes are not add nothing, in each tile:
    an output row of zero scales is exactly zero, and sums of any size stay what they were
    before the group.  Bar as above."""
    rng = np.random.default_rng(5)
    codes = rng.integers(0, 256, (n, k // 2), dtype=np.uint8)
    sc = (rng.random((n, k // group), dtype=np.float32) * 0.1).astype(np.float16)
    sc[::2, 0] = 0
    sc[::3, 2] = 0
    sc[1::4, -1] = -0.0
    sc[5::40, :] = 0
    logical, scales = dev(codes), dev(sc.view(np.int16))
    data = torch.zeros(n * k // 2, dtype=torch.uint8, device="cuda")
    dsc = torch.zeros(n * (k // group), dtype=torch.int16, device="cuda")
    dw = N.Weight(p(data), p(dsc), n, k, N.AM_WF_INT4, group)
    L.call("am_gfx950_pack_int4", N.PackInt4Args(p(logical), p(scales), dw), stream())
    q = np.stack([codes & 15, codes >> 4], -1).reshape(n, k).astype(np.int32)
    w = dev(np.where(q > 7, q - 16, q) * np.repeat(sc.astype(np.float64), group, 1))
    x = act_rows(8, m, k) * np.float32(size)
    xd, xt = bf16_dev(bf16_rne_bits(x)), dev(x).double()
    out = empty((m, n), torch.bfloat16)
    L.call("am_gfx950_linear", N.LinearArgs(p(xd), N.AM_DT_BF16, m, dw, p(out), N.AM_DT_BF16, None, 2), stream())
    ref = xt @ w.T
    bar = ref.abs() * 2.0 ** -8 + k * 2.0 ** -24 * (xt.abs() @ w.abs().T)
    err = (out.double() - ref).abs()
    assert bool((err <= bar).all()), (launched(), float((err - bar).max()))
    assert not bool(out[:, 5::40].any())


@pytest.mark.parametrize("fmt", [N.AM_WF_INT4, N.AM_WF_INT8, N.AM_WF_BF16])
def test_prefill_gemm_workspace_of_longer_chunk(fmt):
    """A short prompt splits K in the workspace of a session whose chunks are long enough
    never to split, to the bits of its own workspace's result."""
    m, n, k = 37, 1024, 14336
    rng = np.random.default_rng(37)
    dw, keep = pack_weight(rbf(rng.standard_normal((n, k), dtype=np.float32) * np.float32(0.02)), fmt)
    xd = bf16_dev(bf16_rne_bits(act_rows(9, m, k)))
    outs = []
    for rows in (m, 12288):
        nbytes = L.am_gfx950_gemm_workspace_bytes(rows, n, k, 128)
        ws = torch.zeros(max(nbytes, 16), dtype=torch.uint8, device="cuda")
        outs.append(empty((m, n), torch.bfloat16))
        args = N.LinearArgs(p(xd), N.AM_DT_BF16, m, dw, p(outs[-1]), N.AM_DT_BF16, None, 2, p(ws), nbytes)
        L.call("am_gfx950_linear", args, stream())
        assert "splits=8" in launched(), launched()
    assert torch.equal(outs[0], outs[1])
    del keep


@pytest.mark.parametrize("B,hkv", [(16, 8), (12, 8), (9, 8), (5, 8), (64, 8), (24, 2)])
@pytest.mark.parametrize("paged", [False, True])
def test_attention_decode_split_rounds(B, hkv, paged):
    """Batched decode grids whose splits are cut to one or two rounds of blocks (and more
    (row, head) pairs than CUs): contexts from one position to past the long-context
    threshold side by side, against fp64 attention.  Twice on one workspace."""
    g, d, cap = 4, 128, 4608
    hq = g * hkv
    rng = np.random.default_rng(B)
    lens = [1, 31, 64, 65, 777, 4095, 4096, 4097, 4608]
    pos = np.array([lens[i % len(lens)] - 1 for i in range(B)], np.int64)
    k, v = (torch.randn((B, hkv, cap, d), device="cuda", generator=torch.Generator("cuda").manual_seed(s)).to(torch.bfloat16)
            for s in (B, B + 1))
    q = torch.randn((B, hq * d), device="cuda", generator=torch.Generator("cuda").manual_seed(3)).to(torch.bfloat16)
    kd, vd, pages = k, v, None
    if paged:
        per = cap // 64
        table = torch.from_numpy(rng.permutation(B * per).astype(np.int32)).cuda().view(B, per)
        kd, vd = (torch.empty((B * per, hkv, 64, d), dtype=torch.bfloat16, device="cuda") for _ in range(2))
        for src, dst in ((k, kd), (v, vd)):
            dst[table.long().view(-1)] = src.view(B, hkv, per, 64, d).transpose(1, 2).reshape(B * per, hkv, 64, d)
        pages = C.pointer(N.KvPages(p(table), 64, per, B * per, None))
    posd = dev(pos)
    wsb = L.am_gfx950_attention_workspace_bytes(B, 1, hq, hkv, d, cap, 0)
    ws = torch.zeros(wsb, dtype=torch.uint8, device="cuda")
    for _ in range(2):
        out = empty((B, hq * d), torch.bfloat16)
        L.call("am_gfx950_attention", N.AttentionArgs(p(q), p(kd), p(vd), p(out), 1, hq, hkv, d, cap, 0, p(posd), B,
                                                      hkv * cap * d, 1, 0, p(ws), wsb, pages), stream())
        for r in range(B):
            n = int(pos[r]) + 1
            kr, vr = (t[r, :, :n].double().repeat_interleave(g, 0) for t in (k, v))
            sc = (kr * q[r].double().view(hq, 1, d)).sum(-1) / d ** 0.5
            ref = (torch.softmax(sc, -1).unsqueeze(-1) * vr).sum(1).view(-1)
            err = (out[r].double() - ref).abs()
            # a bf16 rounding of the output and P in bf16 hi + lo (2^-16 of the row's largest value)
            assert bool((err <= ref.abs() * 2.0 ** -8 + 2.0 ** -15 * vr.abs().max()).all()), (r, n)


@pytest.mark.parametrize("B,hkv", [(16, 8), (24, 8), (32, 8), (64, 8), (65, 8), (128, 8), (9, 24)])
@pytest.mark.parametrize("at", [0, -1])
def test_attention_decode_one_long_row(B, hkv, at):
    """One long context among short ones keeps its 8 splits whatever the batch (the records
    written to the workspace tell them; the short rows are one block each), against fp64
    attention.  Twice on one workspace, whose tickets are left zero."""
    g, d, cap, long = 4, 128, 4608, 4600
    hq, gen = g * hkv, torch.Generator("cuda").manual_seed(B)
    lens = [1 + (7 * r) % 60 for r in range(B)]
    lens[at] = long
    k, v = (torch.randn((B, hkv, cap, d), device="cuda", generator=gen).to(torch.bfloat16) for _ in range(2))
    q = torch.randn((B, hq * d), device="cuda", generator=gen).to(torch.bfloat16)
    posd = dev(np.array(lens, np.int64) - 1)
    wsb = L.am_gfx950_attention_workspace_bytes(B, 1, hq, hkv, d, cap, 0)
    tickets = 64 * -(-B * hkv * 4 // 256)
    for _ in range(2):
        ws = torch.full((wsb // 4,), 0x7FC0DEAD, dtype=torch.int32, device="cuda")
        ws[:tickets] = 0
        out = empty((B, hq * d), torch.bfloat16)
        L.call("am_gfx950_attention", N.AttentionArgs(p(q), p(k), p(v), p(out), 1, hq, hkv, d, cap, 0, p(posd), B,
                                                      hkv * cap * d, 1, 0, p(ws), wsb), stream())
        assert not bool(ws[:tickets].any())
        # a record: maximum, sum and d outputs of g heads
        assert int((ws[tickets:] != 0x7FC0DEAD).sum()) == 8 * hkv * g * (d + 2)
        for r in sorted({0, 1, B // 2, B - 1}):
            n = lens[r]
            kr, vr = (t[r, :, :n].double().repeat_interleave(g, 0) for t in (k, v))
            sc = (kr * q[r].double().view(hq, 1, d)).sum(-1) / d ** 0.5
            ref = (torch.softmax(sc, -1).unsqueeze(-1) * vr).sum(1).view(-1)
            err = (out[r].double() - ref).abs()
            # a bf16 rounding of the output and P in bf16 hi + lo (2^-16 of the row's largest value)
            assert bool((err <= ref.abs() * 2.0 ** -8 + 2.0 ** -15 * vr.abs().max()).all()), (r, n)


@pytest.mark.parametrize("m,n,k", [(6, 4096, 14336), (16, 40, 14336), (9, 17, 16384), (16, 128, 5632)])
@pytest.mark.parametrize("fmt", [N.AM_WF_INT4, N.AM_WF_INT8, N.AM_WF_BF16])
def test_batched_rows_past_lds(m, n, k, fmt):
    """Token rows that do not fit one block's LDS together run as one launch: Linear + Add
    in place and the fp32 store.  The operands' sums are exact, so the results are the
    rounded fp64 ones to the bit, and a k step lost or taken twice shows."""
    rng = np.random.default_rng(m + n)
    dw, w, keep = exact_weight(rng, n, k, fmt)
    x, h = (rng.integers(-4, 5, sh).astype(np.float32) for sh in ((m, k), (m, n)))
    xd, hd = bf16_dev(bf16_rne_bits(x)), bf16_dev(bf16_rne_bits(h))
    xt = dev(x).double()
    ref = xt @ w.T
    for step in range(0, k, 128):  # each step's share of every row and column is there to be missed
        share = xt[:, step:step + 128] @ w[:, step:step + 128].T
        present = (share != 0).any(0).double().mean(), (share != 0).any(1).all()
        assert float(present[0]) > 0.5 and bool(present[1])
    L.call("am_gfx950_fused_linear_residual", N.FusedLinearResidualArgs(p(xd), dw, p(hd), N.AM_DT_BF16, m), stream())
    assert launched().endswith(",xg>"), launched()
    want = (dev(h) + ref.float().bfloat16().float()).bfloat16()
    assert torch.equal(hd.view(torch.bfloat16).view(m, n), want)
    out = empty((m, n), torch.float32)
    L.call("am_gfx950_linear", N.LinearArgs(p(xd), N.AM_DT_BF16, m, dw, p(out), N.AM_DT_F32, None, 3), stream())
    assert launched().endswith(",xg>") and torch.equal(out.double(), ref)
    del keep


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("start", [0, 31])
def test_attention_prefill_two_key_groups(d, start):
    """The middle prefill shape, two key groups merged one column group at a time: blocks
    whose second group has no tile (the first positions), one tile less than the first, or
    as many, a ragged last block, and columns that see no key of a group."""
    hq, hkv, B, qb = 16, 4, 1, 32
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    S = (-(-cus // hkv) - 1) * qb + 5  # exactly enough blocks, the last of 5 positions
    cap = start + S + 3
    rng = np.random.default_rng(710 + d + start)
    q = rbf(rng.standard_normal((S, hq * d), dtype=np.float32))
    kc = rbf(rng.standard_normal((hkv, cap, d), dtype=np.float32))
    vc = rbf(rng.standard_normal((hkv, cap, d), dtype=np.float32))
    qd, kd, vd = (bf16_dev(bf16_rne_bits(x)) for x in (q, kc, vc))
    out = empty((S, hq * d), torch.int16)
    a = N.AttentionArgs(p(qd), p(kd), p(vd), p(out), S, hq, hkv, d, cap, start, None, 1, 0, 1, 0, None, 0)
    L.call("am_gfx950_attention", a, stream())
    assert launched() == f"attention_prefill<d={d},g=4,qb={qb}>"
    got = O.bf16_to_f32(host(out).view(np.uint16)).reshape(S, hq * d)
    for s in (0, 1, 4, 30, 31, 32, 33, 63, 64, 65, 95, 96, S - 6, S - 5, S - 1):
        ref = O.attention(np.ascontiguousarray(q[s:s + 1]), kc, vc, 1, hq, hkv, d, cap, start + s)[0]
        # P is held as bf16 hi + lo (2^-16 of a weight), the result rounded to bf16 (2^-9)
        bad = np.abs(got[s] - ref) > 2.0 ** -8 * np.abs(ref) + 1e-4 * np.abs(ref).max()
        assert not bad.any(), (s, np.argwhere(bad)[:8])


@pytest.mark.parametrize("m,B,starts", [(2, 1, [4094]), (17, 2, [0, 3000]), (37, 1, [600]), (37, 2, [218, 219]), (128, 1, [4000]), (130, 1, [255])])
@pytest.mark.parametrize("d,g", [(128, 4), (64, 8)])
@pytest.mark.parametrize("paged", [False, True])
def test_attention_prefill_split_keys(m, B, starts, d, g, paged):
    """Few prefill rows over a long context, the keys split over blocks: contexts below and
    at two splits' keys, surplus blocks, splits whose keys some columns do not see, ragged
    query blocks, two sequences; against fp64 attention.  The workspace serves a batched
    decode call between two prefill calls, and every ticket is zero after each."""
    hkv, cap = 4, 4608
    hq, gen = g * hkv, torch.Generator("cuda").manual_seed(m + B)
    k, v = (torch.randn((B, hkv, cap, d), device="cuda", generator=gen).to(torch.bfloat16) for _ in range(2))
    q = torch.randn((B, m, hq * d), device="cuda", generator=gen).to(torch.bfloat16)
    kd, vd, pages = k, v, None
    if paged:
        per = cap // 64
        table = torch.from_numpy(np.random.default_rng(m).permutation(B * per).astype(np.int32)).cuda().view(B, per)
        kd, vd = (torch.empty((B * per, hkv, 64, d), dtype=torch.bfloat16, device="cuda") for _ in range(2))
        for src, dst in ((k, kd), (v, vd)):
            dst[table.long().view(-1)] = src.view(B, hkv, per, 64, d).transpose(1, 2).reshape(B * per, hkv, 64, d)
        pages = C.pointer(N.KvPages(p(table), 64, per, B * per, None))
    posd = dev(np.array(starts, np.int64))
    wsb = max(L.am_gfx950_attention_workspace_bytes(B, s, hq, hkv, d, cap, 0) for s in (1, m))
    assert L.am_gfx950_attention_workspace_bytes(B, m, hq, hkv, d, cap, 0) >= L.am_gfx950_attention_workspace_bytes(B, 2, hq, hkv, d, cap, 0)
    ws = torch.zeros(wsb, dtype=torch.uint8, device="cuda")

    def call(rows, qt, out):
        L.call("am_gfx950_attention", N.AttentionArgs(p(qt), p(kd), p(vd), p(out), rows, hq, hkv, d, cap, 0, p(posd), B,
                                                      hkv * cap * d, 1, 0, p(ws), wsb, pages), stream())
        assert not bool(ws[:256].any())

    outs = []
    for _ in range(2):
        outs.append(empty((B, m, hq, d), torch.bfloat16))
        call(m, q, outs[-1])
        assert f"ks=2,splits={min(16, torch.cuda.get_device_properties(0).multi_processor_count // (B * hkv * -(-m // (64 // g))))}>" in launched()
        call(1, q, empty((B, hq, d), torch.bfloat16))
    assert torch.equal(outs[0], outs[1])
    for b in range(B):
        for s in sorted({0, 1, m // 2, m - 1}):
            n = starts[b] + s + 1
            kr, vr = (t[b, :, :n].double().repeat_interleave(g, 0) for t in (k, v))
            sc = (kr * q[b, s].double().view(hq, 1, d)).sum(-1) / d ** 0.5
            ref = (torch.softmax(sc, -1).unsqueeze(-1) * vr).sum(1)
            err = (outs[0][b, s].double() - ref).abs()
            # a bf16 rounding of the output and P in bf16 hi + lo (2^-16 of the row's largest value)
            assert bool((err <= ref.abs() * 2.0 ** -8 + 2.0 ** -15 * vr.abs().max()).all()), (b, s)
