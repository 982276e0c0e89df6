"""Kernel-level parity on the GPU through the C ABI: the MFMA GEMM and the
gated GeGLU GEMM against a CPU GEMM with the same f16 rounding points, on
the odd shapes of the reference's kernel tests
(crates/omg-wgpu/tests/matmul.rs:201-290, relative tolerance 2e-3) and on
the 270M configuration's shapes; the embedding gather bit-exact."""
from __future__ import annotations

import numpy as np
import pytest

import grande_amd as g
import oracle

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

DTYPES = [g.F16, g.Q8, g.Q4]


def weight(rng: np.random.Generator, n: int, k: int, dtype: int, name: str = "w") -> tuple[g.QTensor, np.ndarray]:
    """[n, k] weight in `dtype` and its dequantized values rounded to f16 —
    the kernel's rounding point (matmul.rs:178-199)."""
    v = rng.uniform(-1, 1, (n, k)).astype(np.float32)
    if dtype == g.F16:
        t = g.QTensor(name, g.F16, (n, k), v.astype(np.float16).view(np.uint8).ravel().copy(), np.zeros(0, np.uint8))
    else:
        data, scales = oracle.quantize(dtype, v)
        t = g.QTensor(name, dtype, (n, k), data, scales)
    return t, t.to_f32().astype(np.float16).astype(np.float32)


def gelu(x):
    return 0.5 * x * (1.0 + np.tanh(0.7978845608 * (x + 0.044715 * x ** 3)))


def dev(a: np.ndarray):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("m,n,k", [(23, 96, 64), (130, 200, 96), (64, 128, 32), (1, 640, 2048),
                                   (384, 1536, 640), (2384, 640, 2048), (257, 1152, 1152),
                                   (600, 1536, 4096), (1000, 640, 4128), (700, 1152, 1024), (1100, 1536, 640)])
def test_gemm_matches_cpu(m, n, k, dtype):
    rng = np.random.default_rng(m * n * k + dtype)
    x = (rng.uniform(-1, 1, (m, k)) * 4).astype(np.float16)
    t, wd = weight(rng, n, k, dtype)
    w = g.DeviceWeight(t)
    xd = dev(x)
    y = torch.zeros((m, n), dtype=torch.float32, device="cuda")
    w.gemm(xd.data_ptr(), k, m, y.data_ptr(), n)
    torch.cuda.synchronize()
    exp = x.astype(np.float32) @ wd.T
    got = y.cpu().numpy()
    worst = float(np.max(np.abs(got - exp) / np.maximum(np.abs(exp), 1.0)))
    assert worst < 2e-3, f"gemm {dtype} {m}x{n}x{k}: max rel diff {worst}"


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("m,n,k", [(23, 96, 64), (70, 100, 160), (384, 2048, 640), (2384, 2048, 640),
                                   (600, 256, 1184), (130, 8192, 96), (600, 8192, 96),
                                   (1, 96, 640), (40, 100, 1184), (64, 320, 2560)])
def test_gated_matches_cpu(m, n, k, dtype):
    rng = np.random.default_rng(7 * m * n * k + dtype)
    x = rng.uniform(-1, 1, (m, k)).astype(np.float16)
    tg, gd = weight(rng, n, k, dtype, "gate")
    tu, ud = weight(rng, n, k, dtype, "up")
    wg, wu = g.DeviceWeight(tg), g.DeviceWeight(tu)
    xd = dev(x)
    act = torch.zeros((m, n), dtype=torch.float16, device="cuda")
    wg.gemm_geglu(wu, xd.data_ptr(), k, m, act.data_ptr(), n)
    torch.cuda.synchronize()
    xf = x.astype(np.float32)
    exp = gelu(xf @ gd.T) * (xf @ ud.T)
    got = act.cpu().numpy().astype(np.float32)
    worst = float(np.max(np.abs(got - exp) / np.maximum(np.abs(exp), 1.0)))
    assert worst < 2e-3, f"gated {dtype} {m}x{n}x{k}: max rel diff {worst}"


def test_gemm_rows_are_independent_of_m():
    """A row's result does not depend on how many rows share the launch (no
    split-K, fixed k order): the basis of the bit-equal resident-prefix and
    isolation invariants."""
    rng = np.random.default_rng(5)
    n, k = 640, 2048
    t, _ = weight(rng, n, k, g.Q4)
    w = g.DeviceWeight(t)
    x = rng.uniform(-2, 2, (2384, k)).astype(np.float16)
    outs = []
    for m in (2384, 384, 17, 1):
        y = torch.zeros((m, n), dtype=torch.float32, device="cuda")
        xd = dev(x[:m])  # held until the launch has run
        w.gemm(xd.data_ptr(), k, m, y.data_ptr(), n)
        torch.cuda.synchronize()
        outs.append(y.cpu().numpy())
    for o in outs[1:]:
        assert np.array_equal(o, outs[0][:o.shape[0]])


@pytest.mark.parametrize("k", [640, 2560])
def test_gated_rows_are_independent_of_m(k):
    """The gated product's rows are the same bits whichever tile shape the
    launch's M selects (96-row tiles for long passes, 32-row tiles with a
    deeper ring for short ones, gate and up on paired waves for branch-sized
    ones): the basis of the bit-equal warm and isolated rows through the
    feed-forward."""
    rng = np.random.default_rng(11 + k)
    n = 512
    tg, _ = weight(rng, n, k, g.Q4, "gate")
    tu, _ = weight(rng, n, k, g.Q4, "up")
    wg, wu = g.DeviceWeight(tg), g.DeviceWeight(tu)
    x = rng.uniform(-1, 1, (2384, k)).astype(np.float16)
    outs = []
    for m in (2384, 513, 384, 64, 40, 1):
        act = torch.zeros((m, n), dtype=torch.float16, device="cuda")
        xd = dev(x[:m])  # held until the launch has run
        wg.gemm_geglu(wu, xd.data_ptr(), k, m, act.data_ptr(), n)
        torch.cuda.synchronize()
        outs.append(act.cpu().numpy())
    for o in outs[1:]:
        assert np.array_equal(o, outs[0][:o.shape[0]])


@pytest.mark.parametrize("dtype", DTYPES)
def test_embed_gather_bit_exact(dtype):
    """embed.wgsl:15-48 = reference.rs:182-189: x = deq(E[id]) * sqrt(d),
    bit-exact; the fused first norm within f16 rounding."""
    rng = np.random.default_rng(11 + dtype)
    vocab, d = 300, 640
    t, _ = weight(rng, vocab, d, dtype, "embed")
    w = g.DeviceWeight(t)
    ids = rng.integers(0, vocab, 97).astype(np.uint32)
    norm_w = (1.0 + rng.uniform(-0.5, 0.5, d)).astype(np.float32)
    scale = np.float32(np.sqrt(np.float32(d)))
    x = torch.zeros((ids.size, d), dtype=torch.float32, device="cuda")
    hn = torch.zeros((ids.size, d), dtype=torch.float16, device="cuda")
    idd, wd = dev(ids.view(np.int32)), dev(norm_w)
    w.embed_norm(idd.data_ptr(), ids.size, float(scale), wd.data_ptr(), 1e-6, x.data_ptr(), hn.data_ptr())
    torch.cuda.synchronize()
    deq = t.to_f32()  # exact dequantization, f32
    exp = (deq[ids] * scale).astype(np.float32)
    got = x.cpu().numpy()
    assert np.array_equal(got.view(np.uint32), exp.view(np.uint32)), "embedding gather is not bit-exact"
    ms = (exp.astype(np.float64) ** 2).mean(axis=1, keepdims=True)
    exp_h = exp / np.sqrt(ms + 1e-6) * norm_w
    assert np.max(np.abs(hn.cpu().numpy().astype(np.float32) - exp_h)) < 1e-2 * np.max(np.abs(exp_h))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("vocab,d,nrows,softcap", [(25000, 640, 12, 0.0), (1000, 64, 1, 30.0), (4097, 1152, 37, 0.0)])
def test_label_readout_matches_cpu(vocab, d, nrows, softcap, dtype):
    """logits = rows . deq(E)^T in f32 (softcap applied), then the label
    columns and log_sum_exp of the whole row (readout.rs:124-146,
    math.rs:13-17), against float64 on the dequantized weights: label
    logits within 1e-4 of the row scale, log-sum-exp within 1e-5."""
    rng = np.random.default_rng(vocab + d + nrows + dtype)
    t, _ = weight(rng, vocab, d, dtype, "embed")
    e = t.to_f32().astype(np.float64)
    rows = rng.uniform(-1, 1, (nrows, d)).astype(np.float32)
    labels = rng.choice(vocab, 26, replace=False).astype(np.uint32)
    w = g.DeviceWeight(t)
    out = torch.zeros((nrows, 27), dtype=torch.float32, device="cuda")
    lab = dev(labels.view(np.int32))
    rd = dev(rows)
    w.label_readout(rd.data_ptr(), nrows, lab.data_ptr(), 26, softcap, out.data_ptr())
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    z = rows.astype(np.float64) @ e.T
    if softcap > 0:
        z = softcap * np.tanh(z / softcap)
    m = z.max(1, keepdims=True)
    lse = (m + np.log(np.exp(z - m).sum(1, keepdims=True)))[:, 0]
    scale = np.maximum(np.abs(z).max(1), 1.0)
    assert np.max(np.abs(got[:, :26] - z[:, labels]) / scale[:, None]) < 1e-4
    assert np.max(np.abs(got[:, 26] - lse) / np.maximum(np.abs(lse), 1.0)) < 1e-5


def test_label_readout_odd_shapes_and_out_of_vocab_labels():
    """Widths that are not multiples of 4 (every row of the logits starts
    off the 16-byte grid) and an odd rows x vocab product (the partials sit
    past an odd count of floats) give the same label logits and log-sum-exp
    as an aligned shape's rows; a label id past the vocabulary reads
    nothing and gives NaN in its column only."""
    rng = np.random.default_rng(77)
    vocab, d, nrows = 1001, 64, 3
    t, _ = weight(rng, vocab, d, g.Q8, "embed")
    e = t.to_f32().astype(np.float64)
    rows = rng.uniform(-1, 1, (nrows, d)).astype(np.float32)
    labels = np.array([0, 5, vocab - 1, vocab, 77, 0xFFFFFFFF], np.uint32)
    w = g.DeviceWeight(t)
    out = torch.zeros((nrows, labels.size + 1), dtype=torch.float32, device="cuda")
    rd, lab = dev(rows), dev(labels.view(np.int32))  # held until the launch has run
    w.label_readout(rd.data_ptr(), nrows, lab.data_ptr(), labels.size, 0.0, out.data_ptr())
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    z = rows.astype(np.float64) @ e.T
    m = z.max(1, keepdims=True)
    lse = (m + np.log(np.exp(z - m).sum(1, keepdims=True)))[:, 0]
    ok = labels < vocab
    assert np.isnan(got[:, :-1][:, ~ok]).all()
    assert np.max(np.abs(got[:, :-1][:, ok] - z[:, labels[ok]])) < 1e-4 * max(1.0, np.abs(z).max())
    assert np.max(np.abs(got[:, -1] - lse) / np.maximum(np.abs(lse), 1.0)) < 1e-5


# The split-row readout's edges: row tiles of 32 (31, 32, 33, 65 rows), K
# stages of 64 (32: half a stage, 96: a half last stage, 1,312: past the
# converted chunks), column tiles of 32 / 128 / 256 (31, 257, 1,025, 31,000
# columns: two column tiles per wave), more labels than a tile scans.
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("vocab,d,nrows,nlabels", [(31, 32, 31, 3), (257, 96, 32, 26), (1025, 1312, 33, 600),
                                                   (31000, 64, 130, 26), (640, 4096, 65, 5)])
def test_split_readout_edges(vocab, d, nrows, nlabels, dtype):
    """The parts hold a row element exactly, products are exact, and a
    column's sums are f32 over d / 16 roundings of the high parts' sums (the
    lower parts' are 2^-11 of those) and d / 32 of the scaled blocks:
    2^-24 (2 + d / 8) of sum |x||w| bounds a logit's error (and the
    log-sum-exp's, plus its own few ulps).  Rows of very different magnitudes
    share a launch; with and without scratch the logits are the same bits."""
    rng = np.random.default_rng(vocab * 7 + d + nrows + dtype)
    t, _ = weight(rng, vocab, d, dtype, "embed")
    e = t.to_f32().astype(np.float64)
    rows = rng.standard_normal((nrows, d)).astype(np.float32)
    rows[0] *= 1e-20
    rows[nrows // 2] = 0.0
    rows[-1, ::7] *= 50.0
    labels = rng.integers(0, vocab, nlabels).astype(np.uint32)
    w = g.DeviceWeight(t)
    rd, lab = dev(rows), dev(labels.view(np.int32))
    outs = []
    for f in (w.label_readout, w.label_readout_noalloc):
        out = torch.full((nrows, nlabels + 1), float("nan"), dtype=torch.float32, device="cuda")
        f(rd.data_ptr(), nrows, lab.data_ptr(), nlabels, 0.0, out.data_ptr())
        torch.cuda.synchronize()
        outs.append(out.cpu().numpy())
    assert np.array_equal(outs[0], outs[1])
    z = rows.astype(np.float64) @ e.T
    bound = 2.0 ** -24 * (2 + d / 8) * (np.abs(rows).astype(np.float64) @ np.abs(e).T)
    assert (np.abs(outs[0][:, :-1] - z[:, labels]) <= bound[:, labels] + 1e-45).all()
    m = z.max(1)
    lse = m + np.log(np.exp(z - m[:, None]).sum(1))
    assert (np.abs(outs[0][:, -1] - lse) <= bound.max(1) + 1e-6 * np.maximum(1.0, np.abs(lse))).all()


# Split ahead of the product (one and two column tiles per wave, a half last
# stage) and in the workgroups (more labels than a tile scans, no scratch).
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("vocab,d,nrows,nlabels", [(300, 96, 40, 7), (31, 2560, 33, 3), (31000, 64, 140, 9),
                                                   (1400, 352, 70, 600)])
def test_readout_of_rows_with_an_outlier(vocab, d, nrows, nlabels, dtype):
    """Rows with one element 2^12 to 2^102 times the others, read out at
    columns whose weight there is zero: their logits are the sums of the
    small elements and stay f32 sums of f32 values, whatever the range of the
    row.  An f32 sum of d products rounds at most d times: 2^-24 d of
    sum |x||w|, the outlier adding nothing.  Rows with and without an outlier
    share row tiles; each row alone gives the same bits."""
    rng = np.random.default_rng(vocab * 3 + d + nrows + dtype)
    at = d // 3
    v = rng.uniform(-1, 1, (vocab, d)).astype(np.float32)
    v[::2, at] = 0.0
    if dtype == g.F16:
        t = g.QTensor("embed", g.F16, (vocab, d), v.astype(np.float16).view(np.uint8).ravel().copy(),
                      np.zeros(0, np.uint8))
    else:
        t = g.QTensor("embed", dtype, (vocab, d), *oracle.quantize(dtype, v))
    e = t.to_f32().astype(np.float64)
    assert (e[::2, at] == 0.0).all()
    rows = rng.standard_normal((nrows, d)).astype(np.float32)
    wide = [r for r in range(nrows) if r % 3]
    for i, r in enumerate(wide):
        rows[r, at] = (-1.0) ** i * 2.0 ** (12 + 90 * i / len(wide))
    labels = rng.choice(np.arange(0, vocab, 2), nlabels, replace=False).astype(np.uint32)
    w = g.DeviceWeight(t)
    lab = dev(labels.view(np.int32))

    def run(f, x):
        xd = dev(x)
        out = torch.full((len(x), nlabels + 1), float("nan"), dtype=torch.float32, device="cuda")
        f(xd.data_ptr(), len(x), lab.data_ptr(), nlabels, 0.0, out.data_ptr())
        torch.cuda.synchronize()
        return out.cpu().numpy()

    got = run(w.label_readout, rows)
    z = rows.astype(np.float64) @ e.T
    bound = 2.0 ** -24 * d * (np.abs(rows).astype(np.float64) @ np.abs(e).T)
    assert (np.abs(got[:, :-1] - z[:, labels]) <= bound[:, labels]).all()
    for r in (0, 1, nrows // 2, nrows - 1):
        assert np.array_equal(run(w.label_readout, rows[r:r + 1])[0], got[r])
    few = rows[:min(nrows, 4_000_000 // (vocab + 100))]
    assert np.array_equal(run(w.label_readout_noalloc, few), got[:len(few)])


def test_readout_of_an_infinite_weight():
    """An infinite f16 weight gives its column infinities of the row
    element's sign (NaN where that element is zero), as an f32 product does,
    and leaves every other column alone."""
    rng = np.random.default_rng(4)
    v = rng.uniform(-1, 1, (200, 96)).astype(np.float16)
    rows = (rng.integers(1, 64, (35, 96)) * rng.choice([-1, 1], (35, 96))).astype(np.float32)
    rows[5, 40] = 0.0
    lab = dev(np.arange(200, dtype=np.int32))
    rd = dev(rows)

    def run():
        w = g.DeviceWeight(g.QTensor("embed", g.F16, v.shape, v.view(np.uint8).ravel().copy(), np.zeros(0, np.uint8)))
        out = torch.zeros((35, 201), dtype=torch.float32, device="cuda")
        w.label_readout(rd.data_ptr(), 35, lab.data_ptr(), 200, 0.0, out.data_ptr())
        torch.cuda.synchronize()
        return out.cpu().numpy()[:, :200]

    ref = run()
    v[17, 40] = np.inf
    got = run()
    others = np.arange(200) != 17
    assert np.array_equal(got[:, others], ref[:, others])
    live = np.arange(35) != 5
    assert np.array_equal(got[live, 17], np.sign(rows[live, 40]) * np.inf) and np.isnan(got[5, 17])


def test_readout_of_non_finite_rows_and_streams():
    """An infinity or a NaN in a row stays in that row; calls on two streams
    in turn, one at a time, give the same rows."""
    rng = np.random.default_rng(9)
    vocab, d, nrows = 500, 128, 40
    t, _ = weight(rng, vocab, d, g.Q8, "embed")
    w = g.DeviceWeight(t)
    rows = rng.standard_normal((nrows, d)).astype(np.float32)
    labels = dev(np.arange(26, dtype=np.int32))
    streams = [torch.cuda.Stream() for _ in range(2)]

    def readout(r, s=None):
        rd = dev(r)
        out = torch.zeros((nrows, 27), dtype=torch.float32, device="cuda")
        torch.cuda.synchronize()
        w.label_readout(rd.data_ptr(), nrows, labels.data_ptr(), 26, 0.0, out.data_ptr(), s.cuda_stream if s else None)
        return rd, out

    ref = readout(rows)[1]
    other = readout(rows[::-1].copy())[1]
    held = [readout(rows if i % 2 == 0 else rows[::-1].copy(), streams[i % 2]) for i in range(8)]
    torch.cuda.synchronize()
    for i, (_, out) in enumerate(held):
        assert torch.equal(out, ref if i % 2 == 0 else other)
    bad = rows.copy()
    bad[3, 5], bad[17, 100] = np.inf, np.nan
    got = readout(bad)[1].cpu().numpy()
    torch.cuda.synchronize()
    live = [r for r in range(nrows) if r not in (3, 17)]
    assert np.array_equal(got[live], ref.cpu().numpy()[live])
    assert not np.isfinite(got[3, :26]).any() and np.isnan(got[17]).all()


class _Readouts:
    """Label readouts of one weight on inputs that are uploaded and outputs
    that are allocated before the first of them is queued."""

    def __init__(self, sizes, vocab=6000, d=512, nlabels=26):
        rng = np.random.default_rng(sum(sizes))
        self.t, _ = weight(rng, vocab, d, g.Q8, "embed")
        self.nlabels = nlabels
        self.labels = dev(np.arange(nlabels, dtype=np.int32))
        self.rows = [dev(rng.standard_normal((n, d)).astype(np.float32)) for n in sizes]
        self.out = [torch.zeros((n, nlabels + 1), dtype=torch.float32, device="cuda") for n in sizes]
        alone = g.DeviceWeight(self.t)
        self.want = []
        for i in range(len(sizes)):
            self.call(alone, i, None)
            torch.cuda.synchronize()
            self.want.append(self.out[i].clone())
            self.out[i].zero_()
        torch.cuda.synchronize()

    def call(self, w, i, stream):
        w.label_readout(self.rows[i].data_ptr(), len(self.rows[i]), self.labels.data_ptr(), self.nlabels, 0.0,
                        self.out[i].data_ptr(), stream)

    def check(self):
        torch.cuda.synchronize()
        for i, (got, want) in enumerate(zip(self.out, self.want)):
            assert torch.equal(got, want), f"call {i}"


def test_readout_scratch_of_overlapping_streams():
    """Calls with one weight queued in turn on three streams (the null stream
    among them) with nothing waited for in between, small and large ones so
    that the kept scratch is too small, in use elsewhere and handed on: each
    gives the rows it gives alone."""
    r = _Readouts([180, 3, 70, 200, 40, 1] * 6)
    w = g.DeviceWeight(r.t)
    streams = [None, torch.cuda.Stream().cuda_stream, torch.cuda.Stream().cuda_stream]
    for i in range(len(r.rows)):
        r.call(w, i, streams[i % 3])
    r.check()


def test_readout_scratch_grows_on_one_stream():
    """Small, large, small, larger on one stream without a wait: the larger
    block replaces the kept one behind the calls that still use it."""
    r = _Readouts([2, 120, 5, 64, 200, 33, 1, 230])
    w = g.DeviceWeight(r.t)
    s = torch.cuda.Stream().cuda_stream
    for i in range(len(r.rows)):
        r.call(w, i, s)
    r.check()


def test_readout_scratch_outlives_its_streams():
    """Streams made, used once and destroyed (a new one can have the handle
    of an old one): every call gives the rows it gives alone."""
    import ctypes
    hip = ctypes.CDLL("libamdhip64.so.7")
    r = _Readouts([150, 2, 90, 40] * 4)
    w = g.DeviceWeight(r.t)
    for i in range(len(r.rows)):
        s = ctypes.c_void_p()
        assert hip.hipStreamCreate(ctypes.byref(s)) == 0
        r.call(w, i, s.value)
        assert hip.hipStreamDestroy(s) == 0
    r.check()


def test_readout_under_capture():
    """A call that is being captured takes scratch of its own: the graph's
    replays give the eager rows, with eager calls on the kept scratch in
    between."""
    r = _Readouts([60, 100])
    w = g.DeviceWeight(r.t)
    r.call(w, 0, None)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        r.call(w, 1, torch.cuda.current_stream().cuda_stream)
    for _ in range(3):
        r.out[0].zero_()
        r.out[1].zero_()
        graph.replay()
        r.call(w, 0, None)
        r.check()


# Wide tiles: a 7,944-column product makes more than one round of tiles from
# a few dozen rows on, so the rows below pass through the short tiles and
# wide ones of several row-block counts (and columns past the last whole
# tile); K 96 and 160 end in half a stage, 320 and 640 have an odd and an even
# stage count.
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("k", [96, 160, 320, 640])
def test_wide_tiles_give_the_short_tiles_rows(k, dtype):
    """Products of one type are the same bits for a row whatever M selects
    (f32, both gated forms, bias + ReLU), and match a float64 product of the
    same f16 operands: f32 sums of K products bound the error by 2^-23 K of
    sum |x||w|, f16 outputs add half an ulp (2^-11)."""
    rng = np.random.default_rng(k + dtype)
    n = 7944
    (tg, gd), (tu, ud) = weight(rng, n, k, dtype, "gate"), weight(rng, n, k, dtype, "up")
    wg, wu = g.DeviceWeight(tg), g.DeviceWeight(tu)
    bias = rng.uniform(-1, 1, n).astype(np.float16)
    x = rng.uniform(-1, 1, (700, k)).astype(np.float16)
    bd = dev(bias)

    def run(m, kind):
        xd = dev(x[:m])
        y = torch.zeros((m, n), dtype=torch.float32 if kind == "f32" else torch.float16, device="cuda")
        if kind == "f32":
            wg.gemm(xd.data_ptr(), k, m, y.data_ptr(), n)
        elif kind == "relu":
            wg.gemm_bias_relu(xd.data_ptr(), k, m, bd.data_ptr(), y.data_ptr(), n)
        else:
            (wg.gemm_geglu if kind == "tanh" else wg.gemm_geglu_erf)(wu, xd.data_ptr(), k, m, y.data_ptr(), n)
        torch.cuda.synchronize()
        return y.cpu().numpy()

    xf = x.astype(np.float64)
    a, u = xf @ gd.T, xf @ ud.T
    bound = 2.0 ** -23 * k * (np.abs(xf) @ np.abs(gd).T)
    for kind in ("f32", "relu", "tanh", "erf"):
        full = run(700, kind)
        for m in (1, 33, 95, 130, 257, 480):
            assert np.array_equal(run(m, kind), full[:m]), f"{kind} rows at M {m}"
        got = full.astype(np.float64)
        if kind == "f32":
            assert (np.abs(got - a) <= bound + 1e-30).all()
        elif kind == "relu":
            z = np.maximum(a + bias, 0.0)
            assert (np.abs(got - z) <= bound + 2.0 ** -11 * np.abs(z) + 1e-7).all()
        else:
            from math import erf
            z = a[:40]
            z = (gelu(z) if kind == "tanh" else 0.5 * z * (1.0 + np.vectorize(erf)(z / np.sqrt(2.0)))) * u[:40]
            assert np.max(np.abs(got[:40] - z) / np.maximum(np.abs(z), 1.0)) < 2e-3


# 7,944 columns again, at the rows where the choice of a tile changes (and one
# past them): f32 32 x 128, 64 x 128, 96 x 128, 128 x 256 and with f16 weights
# 96 x 128, 128 x 128, 192 x 128; bias + ReLU on two and four waves, one to four
# wide row blocks, f16 64 x 64 up to 192 x 128; the gated products' paired, short
# and wide tiles, f16 64 to 192 rows.
TILE_ROWS = (1, 33, 65, 100, 129, 200, 257, 300, 385, 450, 513, 700, 769, 801, 1000, 1025)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("k,ldx,ldy,shift", [(96, 96, 7944, 0), (320, 336, 7956, 0), (160, 168, 7944, 4)])
def test_every_tile_gives_the_same_rows(k, ldx, ldy, shift, dtype):
    """A row's outputs are the same bits whatever M selects, with X rows
    further apart than K and with output rows or a base off the 16 bytes that
    the eight-column f16 stores want (they fall back to four columns: ldy
    7,956, or the base four columns in), and match float64: f32 sums of K
    products within 2^-23 K of sum |x||w|, f16 outputs half an ulp more.
    Columns past N stay as they were."""
    from math import erf
    rng = np.random.default_rng(7 * k + dtype)
    n, rows = 7944, 1090
    (tg, gd), (tu, ud) = weight(rng, n, k, dtype, "gate"), weight(rng, n, k, dtype, "up")
    wg, wu = g.DeviceWeight(tg), g.DeviceWeight(tu)
    bias = rng.uniform(-1, 1, n).astype(np.float16)
    x = rng.uniform(-1, 1, (rows, ldx)).astype(np.float16)
    bd, xd = dev(bias), dev(x)

    def run(m, kind):
        y = torch.full((m * ldy + 16,), 7.0, dtype=torch.float32 if kind == "f32" else torch.float16, device="cuda")
        at = 0 if kind == "f32" else shift
        p = y.data_ptr() + 2 * at
        if kind == "f32":
            wg.gemm(xd.data_ptr(), ldx, m, p, ldy)
        elif kind == "relu":
            wg.gemm_bias_relu(xd.data_ptr(), ldx, m, bd.data_ptr(), p, ldy)
        else:
            (wg.gemm_geglu if kind == "tanh" else wg.gemm_geglu_erf)(wu, xd.data_ptr(), ldx, m, p, ldy)
        torch.cuda.synchronize()
        y = y.cpu().numpy()
        assert (y[:at] == 7.0).all() and (y[at + m * ldy:] == 7.0).all()
        y = y[at:at + m * ldy].reshape(m, ldy)
        assert (y[:, n:] == 7.0).all(), f"{kind} columns past N at M {m}"
        return y[:, :n]

    xf = x[:, :k].astype(np.float64)
    a, mass = xf @ gd.T, np.abs(xf) @ np.abs(gd).T
    u = xf[:40] @ ud.T
    bound = 2.0 ** -23 * k * mass
    for kind in ("f32", "relu", "tanh", "erf"):
        full = run(rows, kind)
        for m in TILE_ROWS:
            assert np.array_equal(run(m, kind), full[:m]), f"{kind} rows at M {m}"
        got = full.astype(np.float64)
        if kind == "f32":
            assert (np.abs(got - a) <= bound + 1e-30).all()
        elif kind == "relu":
            z = np.maximum(a + bias, 0.0)
            assert (np.abs(got - z) <= bound + 2.0 ** -11 * np.abs(z) + 1e-7).all()
        else:
            z = a[:40]
            z = (gelu(z) if kind == "tanh" else 0.5 * z * (1.0 + np.vectorize(erf)(z / np.sqrt(2.0)))) * u
            assert np.max(np.abs(got[:40] - z) / np.maximum(np.abs(z), 1.0)) < 2e-3


@pytest.mark.parametrize("dtype", DTYPES)
def test_every_f32_tile_of_a_narrow_product(dtype):
    """2,560 columns, K 640: the rows where 64 x 128 of the short stages takes
    over again past its first round, the 96- and 128-row tiles and, f16, 192
    rows: the same bits as the longest launch's rows, and float64's within the
    bound of f32 sums."""
    rng = np.random.default_rng(50 + dtype)
    n, k, rows = 2560, 640, 3700
    t, wd = weight(rng, n, k, dtype)
    w = g.DeviceWeight(t)
    x = rng.uniform(-1, 1, (rows, k)).astype(np.float16)
    xd = dev(x)

    def run(m):
        y = torch.zeros((m, n), dtype=torch.float32, device="cuda")
        w.gemm(xd.data_ptr(), k, m, y.data_ptr(), n)
        torch.cuda.synchronize()
        return y.cpu().numpy()

    full = run(rows)
    for m in (500, 513, 769, 1153, 1601, 2401, 3201, 3649):
        assert np.array_equal(run(m), full[:m]), f"rows at M {m}"
    xf = x.astype(np.float64)
    assert (np.abs(full - xf @ wd.T) <= 2.0 ** -23 * k * (np.abs(xf) @ np.abs(wd).T)).all()


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("vocab,d,nrows,nlabels", [(200, 4096, 800, 5), (1000, 64, 40, 600), (900, 192, 33, 513)])
def test_readout_split_in_the_workgroups(vocab, d, nrows, nlabels, dtype):
    """Without scratch for the split rows (they do not fit the fixed array, or
    the full rows take it) the workgroups split the rows themselves, also with
    fewer K stages than they convert at once: the same bits as with scratch,
    and the logits the float64 ones within 2^-24 (2 + d / 8) of sum |x||w|."""
    rng = np.random.default_rng(vocab + d + nrows + dtype)
    t, _ = weight(rng, vocab, d, dtype, "embed")
    e = t.to_f32().astype(np.float64)
    rows = rng.standard_normal((nrows, d)).astype(np.float32)
    rows[nrows // 3, d // 2] = 2.0 ** 60  # a row of the f32 product
    labels = rng.choice(vocab, nlabels, replace=False).astype(np.uint32)
    w = g.DeviceWeight(t)
    rd, lab = dev(rows), dev(labels.view(np.int32))
    outs = []
    for f in (w.label_readout, w.label_readout_noalloc):
        out = torch.full((nrows, nlabels + 1), float("nan"), dtype=torch.float32, device="cuda")
        f(rd.data_ptr(), nrows, lab.data_ptr(), nlabels, 0.0, out.data_ptr())
        torch.cuda.synchronize()
        outs.append(out.cpu().numpy())
    assert np.array_equal(outs[0], outs[1])
    rows64 = rows.astype(np.float64)
    z = rows64 @ e.T
    bound = 2.0 ** -24 * (2 + d / 8) * (np.abs(rows64) @ np.abs(e).T)
    bound[nrows // 3] *= 8  # (its sums round once per product)
    assert (np.abs(outs[0][:, :-1] - z[:, labels]) <= bound[:, labels]).all()
