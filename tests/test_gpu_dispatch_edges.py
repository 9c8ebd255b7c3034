"""The branches that the sizes of a call choose between, at the sizes where they begin and end: each against dense
logits or gradients formed on the GPU in fp32 / fp64."""

import pytest
import torch

from _util import make_inputs

pytestmark = pytest.mark.gpu


def _lib():
    from cut_cross_entropy import _hip

    return _hip.load()


@pytest.mark.parametrize("shape", [(1, 256 * 255, 128), (40, 256 * 256 + 1, 128), (256, 256 * 257 - 5, 192), (257, 256 * 129, 128),
                                   (700, 256 * 90 + 7, 128), (1025, 256 * 66, 128)])
def test_lse_forward_of_few_rows_fills_the_chip(shape):
    """One to five row blocks against many classes: more than 64 vocabulary spans per row block (up to one span for
    each tile), all merged by the second kernel."""
    lib = _lib()
    dev = torch.device("cuda:0")
    N, V, D = shape
    e, c, _, _ = make_inputs(N, V, D, torch.bfloat16, seed=5)
    ed, cd = e.to(dev), c.to(dev)
    want = torch.logsumexp((ed.float() @ cd.float().T).double(), dim=1)
    lse = torch.full((N,), float("nan"), dtype=torch.float32, device=dev)
    ws = torch.full((lib.cce_lse_forward_workspace_bytes(N, V, D) // 4,), float("nan"), device=dev)
    st = lib.cce_lse_forward(
        ed.data_ptr(), cd.data_ptr(), None, None, lse.data_ptr(), None, None, ws.data_ptr(), ws.numel() * 4,
        N, N, V, D, ed.stride(0), cd.stride(0), cd.stride(1), 0.0, 0, torch.cuda.current_stream().cuda_stream)
    assert st == 0, lib.cce_error_string(st)
    # fp32 sums of D <= 192 products of magnitude about 1, and of up to 66000 exponentials: the bound of
    # test_lse_forward_spans_of_many_tiles
    assert torch.allclose(lse.double(), want, atol=2e-4, rtol=2e-5)


@pytest.mark.parametrize("shape,fp32_out", [((300, 9000, 128), False), ((300, 9000, 128), True), ((70, 20011, 192), False),
                                            ((1100, 33000, 320), False), ((9001, 200, 128), False), ((5000, 520, 64), False),
                                            ((2100, 2500, 64), False), ((2100, 2500, 64), True), ((9000, 9000, 64), False),
                                            ((9000, 70, 64), True)])
@pytest.mark.parametrize("gathered", [False, True])
@pytest.mark.parametrize("budget", [1 << 28, 0])
def test_backward_dense_cuts_long_reductions(shape, fp32_out, gathered, budget):
    """Few tiles with a long reduction: the unfiltered backward cuts the reduction into slots and adds them up.  dE cut
    (few rows, many classes; with less workspace over several chunks, or not at all), dC cut (a small vocabulary under many
    rows), both cut; the caller's fp32 dE is added to.  Against the formulas in fp64."""
    lib = _lib()
    dev = torch.device("cuda:0")
    N, V, D = shape
    e, c, t, _ = make_inputs(N, V, D, torch.bfloat16, seed=7, planted=False, c_std=0.3)
    ed, cd, td = e.to(dev), c.to(dev), t.to(dev)
    rows = torch.arange(N, device=dev)
    valids = None
    if gathered:
        rows = rows[torch.rand(N, generator=torch.Generator().manual_seed(3)).to(dev) < 0.8]
        valids = rows.to(torch.int32)
    B = rows.numel()
    g = torch.rand((N,), generator=torch.Generator().manual_seed(4)).to(dev) + 0.5
    logits = ed.double()[rows] @ cd.double().T
    lse = torch.logsumexp(logits, dim=1)
    dz = torch.exp(logits - lse[:, None])
    dz[torch.arange(B, device=dev), td[rows]] -= 1.0
    dz *= g[rows].double()[:, None]
    want_dc = dz.T @ ed.double()[rows]
    want_de = torch.zeros((N, D), dtype=torch.float64, device=dev)
    want_de[rows] = dz @ cd.double()
    gdt = torch.float32 if fp32_out else torch.bfloat16
    de = torch.zeros((N, D), dtype=gdt, device=dev)
    if fp32_out:
        de += 1.0
    dc = torch.full((V, D), float("nan"), dtype=gdt, device=dev)
    db = torch.full((V,), 0.5, device=dev)
    smallest = lib.cce_backward_dense_workspace_bytes(B, V, D, 0 if fp32_out else 1, 0)
    ws_bytes = lib.cce_backward_dense_workspace_bytes(B, V, D, 0 if fp32_out else 1, budget or 3 * smallest)
    ws = torch.full((ws_bytes // 4 + 64,), float("nan"), device=dev)
    p = lambda x: x.data_ptr() if x is not None else None
    st = lib.cce_backward_dense(
        p(ed), p(cd), None, p(lse.float()), p(g), 0, None, p(valids), p(td), p(de), p(dc), p(db),
        (ws.data_ptr() + 255) // 256 * 256, ws_bytes, N, B, V, D, D, D, 1, 1.0, int(fp32_out), int(fp32_out), 0, 0, 0.0, 0,
        torch.cuda.current_stream().cuda_stream)
    assert st == 0, lib.cce_error_string(st)
    torch.cuda.synchronize()
    # dz and a 16-bit result are rounded to 8 bits once each (2^-9 relative, on sums of terms of either sign: a
    # hundredth of the largest value of the row), fp32 results by dz alone
    if fp32_out:
        de -= 1.0
    assert torch.isfinite(de).all() and torch.isfinite(dc).all()
    for got, want in ((de, want_de), (dc, want_dc)):
        scale = want.abs().amax(dim=1, keepdim=True)
        assert ((got.double() - want).abs() <= 1e-2 * scale + 1e-2 * want.abs() + 1e-6).all()
        assert (got.double() - want).norm() <= 6e-3 * want.norm()
    # the column sums of dz, rounded to 8 significant bits before: each term off by half a unit in the last place, 2^-8 of it
    want_db, size = dz.sum(0), dz.abs().sum(0)
    assert ((db.double() - 0.5 - want_db).abs() <= 2.0**-8 * size + 1e-6).all()


def _fp32_case(N, V, D, keep, seed, softcap=None, bias=False, d_lse=False, strided=False):
    """(inputs, results in fp64) of one fp32 call, everything made on the GPU."""
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(seed)
    e = torch.randn((N, D), generator=g, device=dev)
    c = torch.randn((V, D + 4), generator=g, device=dev)[:, :D] if strided else torch.randn((V, D), generator=g, device=dev)
    c = c * (0.5 / D**0.5) if not strided else c.mul_(0.5 / D**0.5)
    t = torch.randint(0, V, (N,), generator=g, device=dev)
    b = torch.randn((V,), generator=g, device=dev) if bias else None
    w = torch.rand((N,), generator=g, device=dev) + 0.5
    h = torch.randn((N,), generator=g, device=dev) * 0.1 if d_lse else None
    rows = torch.arange(N, device=dev)
    valids = None
    if keep < 1.0:
        rows = rows[torch.rand((N,), generator=g, device=dev) < keep]
        valids = rows.to(torch.int32)
    return e, c, t, b, w, h, rows, valids


@pytest.mark.parametrize("shape,keep,extra", [
    ((1, 3, 1), 1.0, {}), ((65, 257, 65), 1.0, {"softcap": 5.0}), ((300, 9001, 123), 0.7, {"bias": True, "d_lse": True}),
    ((64, 256, 64), 1.0, {}), ((130, 600, 1000), 0.5, {"strided": True}), ((40, 33000, 2048), 1.0, {"bias": True}),
    ((6000, 300, 200), 0.9, {"d_lse": True, "softcap": 20.0}), ((1500, 1400, 96), 1.0, {"strided": True, "bias": True}),
    ((176000, 70, 4096), 1.0, {}), ((180000, 70, 4096), 0.98, {}),
    ((30000, 5000, 64), 1.0, {"bias": True}), ((30000, 1500, 4096), 0.95, {"softcap": 10.0, "d_lse": True, "bias": True}),
])
@pytest.mark.parametrize("terms", [6, 3])
def test_fp32_passes_abi(shape, keep, extra, terms):
    """cce_fp32_forward / cce_fp32_backward against fp64: widths that are no multiple of anything, one and several chunks
    of classes (33000 x 2048), cut reductions of dE and of dC, rows gathered or taken as they lie, more rows than 32-bit
    offsets reach in one copy (blocks of rows: two forward, seven backward), a classifier with gaps between its rows."""
    _check_fp32_passes(shape, terms, extra.get("softcap"), *_fp32_case(*shape, keep, 21, **extra))


@pytest.mark.parametrize("shape,keep,extra,past", [
    ((65, 257, 65), 1.0, {"softcap": 5.0}, "e"), ((300, 9001, 123), 0.7, {"bias": True, "d_lse": True}, "e"),
    ((300, 9001, 123), 0.7, {"bias": True, "d_lse": True}, "c"), ((130, 600, 1000), 0.5, {"strided": True}, "c"),
    ((40, 33000, 2048), 1.0, {"bias": True}, "last class"), ((40, 33000, 2048), 1.0, {"bias": True}, "e"),
    ((6000, 300, 200), 0.9, {"d_lse": True, "softcap": 20.0}, "e"), ((1500, 1400, 96), 1.0, {"strided": True, "bias": True}, "c"),
    ((176000, 70, 4096), 1.0, {}, "first row"), ((176000, 70, 4096), 1.0, {}, "last row"), ((180000, 70, 4096), 0.98, {}, "last row"),
    ((30000, 5000, 64), 1.0, {"bias": True}, "e"),
])
@pytest.mark.parametrize("terms", [6, 3])
def test_fp32_passes_abi_by_parts(shape, keep, extra, past, terms):
    """The same with a value past what halves of fp16 hold, so that the logits go by bf16 parts as well: in E or in C, in the last of
    several chunks of classes alone, in the first or the last block of rows alone."""
    e, c, t, bias, w, h, rows, valids = _fp32_case(*shape, keep, 21, **extra)
    if past in ("c", "last class"):
        e[:, 0] *= 1e-2
        c[-1, 0] = 16.5
    else:
        c[:, 0] *= 1e-2
        e[rows[0] if past in ("e", "first row") else rows[-1], 0] = 300.0
    _check_fp32_passes(shape, terms, extra.get("softcap"), e, c, t, bias, w, h, rows, valids)


def _check_fp32_passes(shape, terms, cap, e, c, t, bias, w, h, rows, valids):
    lib = _lib()
    dev = torch.device("cuda:0")
    N, V, D = shape
    B = rows.numel()
    p = lambda x: x.data_ptr() if x is not None else None
    lse = torch.full((B,), float("nan"), device=dev)
    nll = torch.full((B,), float("nan"), device=dev)
    stream = torch.cuda.current_stream().cuda_stream

    def workspace(nbytes):
        buf = torch.full((nbytes // 4 + 64,), float("nan"), device=dev)
        return buf, (buf.data_ptr() + 255) // 256 * 256

    n_ws = lib.cce_fp32_forward_workspace_bytes(B, V, D, terms)
    buf, ws = workspace(n_ws)
    st = lib.cce_fp32_forward(p(e), p(c), p(bias), p(valids), p(t), p(lse), p(nll), ws, n_ws, N, B, V, D, e.stride(0), c.stride(0),
                              1, 0, 0, cap or 0.0, terms, stream)
    assert st == 0, lib.cce_error_string(st)
    x = e.double()[rows] @ c.double().T + (bias.double() if bias is not None else 0.0)
    damp = 1.0
    if cap:
        th = torch.tanh(x / cap)
        x, damp = cap * th, 1.0 - th * th
    want_lse = torch.logsumexp(x, dim=1)
    # six terms: 2^-24 per product, fp32 sums of D of them and of V exponentials; three: 2^-16 of |e| |c| ~ sqrt(D) / 2
    # per logit (before the cap), of random sign over D
    tol = 4e-6 if terms == 6 else 4e-5
    assert torch.allclose(lse.double(), want_lse, atol=tol, rtol=2e-6)
    # plain fp32 whatever the number of terms: D roundings of terms of up to 1
    assert torch.allclose(nll.double(), want_lse - x[torch.arange(B, device=dev), t[rows]], atol=2e-5 + tol, rtol=2e-6)
    dz = torch.exp(x - want_lse[:, None]) * (w.double()[rows] + (h.double()[rows] if h is not None else 0.0))[:, None]
    dz[torch.arange(B, device=dev), t[rows]] -= w.double()[rows]
    dz *= damp
    del x
    want_de = torch.zeros((N, D), dtype=torch.float64, device=dev)
    want_de[rows] = dz @ c.double()
    want_dc, want_db = dz.T @ e.double()[rows], dz.sum(0)
    del dz, buf
    de = torch.zeros((N, D), device=dev)
    dc = torch.full((V, D), float("nan"), device=dev)
    db = torch.zeros((V,), device=dev)
    n_ws = lib.cce_fp32_backward_workspace_bytes(B, V, D, terms)
    buf, ws = workspace(n_ws)
    lse32 = want_lse.float()
    st = lib.cce_fp32_backward(p(e), p(c), p(bias), p(lse32), p(w), 0, p(h), p(valids), p(t), p(de), p(dc), p(db), ws, n_ws,
                               N, B, V, D, e.stride(0), c.stride(0), 1, D, D, 1.0, 0, 0, cap or 0.0, terms, stream)
    assert st == 0, lib.cce_error_string(st)
    torch.cuda.synchronize()
    # relative to the norm: 2^-24 per term of the sums (2^-16 with three terms), a few times that for what dz inherits
    # from the logits and from the rounding of lse to fp32
    # (dC sums up to 180000 rows in fp32, 16 per rounding: sqrt(11000) 2^-24)
    rel = 8e-6 if terms == 6 else 2e-4
    for name, got, want in (("dE", de, want_de), ("dC", dc, want_dc), ("dBias", db, want_db)):
        assert torch.isfinite(got).all(), name
        err = (got.double() - want).norm().item()
        assert err <= rel * want.norm().item() + 1e-6 * want.numel() ** 0.5 * 1e-2, (name, err, want.norm().item())
    ignored = torch.ones(N, dtype=torch.bool, device=dev)
    ignored[rows] = False
    assert (de[ignored] == 0).all()


@pytest.mark.parametrize("scalar,with_dlse", [(0, False), (0, True), (1, True), (1, False)])
def test_fp32_backward_of_one_row_whose_label_is_past_the_end(scalar, with_dlse):
    """One row, no list of rows and a shift: the row has no label, so its gradients are zeros whatever stands behind the one upstream
    gradient that there is."""
    lib = _lib()
    V, D = 300, 72
    e, c, t, _, _, _, _, _ = _fp32_case(1, V, D, 1.0, 3)
    lse = torch.logsumexp(e @ c.T, 1)
    w = torch.full((64,), float("nan"), device="cuda")
    h = torch.full((64,), 1e30, device="cuda")
    w[0] = h[0] = 1.0
    de, dc, db = torch.zeros((1, D), device="cuda"), torch.full((V, D), float("nan"), device="cuda"), torch.zeros((V,), device="cuda")
    n_ws = lib.cce_fp32_backward_workspace_bytes(1, V, D, 6)
    buf = torch.full((n_ws // 4 + 64,), float("nan"), device="cuda")
    ws = (buf.data_ptr() + 255) // 256 * 256
    p = lambda x: x.data_ptr()
    st = lib.cce_fp32_backward(p(e), p(c), None, p(lse), p(w), scalar, p(h) if with_dlse else None, None, p(t), p(de), p(dc), p(db), ws,
                               n_ws, 1, 1, V, D, D, D, 1, D, D, 1.0, 1, 0, 0.0, 6, torch.cuda.current_stream().cuda_stream)
    assert st == 0, lib.cce_error_string(st)
    assert (de == 0).all() and (dc == 0).all() and (db == 0).all()


def _fp32_gradients(e, c, t, b):
    """Gradients of linear_cross_entropy under uneven weights, and the same in fp64: (dE, dC, dBias), (dE, dC, dBias)."""
    from cut_cross_entropy import linear_cross_entropy

    N = e.size(0)
    w = torch.rand((N,), generator=torch.Generator(device="cuda").manual_seed(9), device="cuda") + 0.5
    for x in (e, c, b):
        x.requires_grad_(True)
    linear_cross_entropy(e, c, t, bias=b, reduction="none").backward(w)
    with torch.no_grad():
        x = e.double() @ c.double().T + b.double()
        dz = torch.softmax(x, dim=1)
        dz[torch.arange(N, device="cuda"), t] -= 1.0
        dz *= w.double()[:, None]
        return (e.grad, c.grad, b.grad), (dz @ c.double(), dz.T @ e.double(), dz.sum(0))


@pytest.mark.parametrize("size", [1e-4, 1e-6, 1e-8, 1e-12])
@pytest.mark.parametrize("which", ["e", "c", "columns of e", "columns of c"])
@pytest.mark.parametrize("shape", [(300, 3000, 200), (20, 700, 64)])
def test_fp32_gradients_of_small_operands(which, size, shape):
    """dC is proportional to E and dE to C: an operand, or a feature, that is small everywhere has gradients as exact, for their own
    size, as any other."""
    N, V, D = shape
    e, c, t, b, _, _, _, _ = _fp32_case(N, V, D, 1.0, 11, bias=True)
    small = e if which.endswith("e") else c
    if which.startswith("columns"):
        small[:, 3:9] *= size
    else:
        small *= size
    got, want = _fp32_gradients(e, c, t, b)
    for x, exact in zip(got[:2], want[:2]):
        assert torch.isfinite(x).all()
        # per column: fp32 sums of at most 3000 products (sqrt(3000) 2^-24 if all roundings met the largest sum), and what dz inherits
        # from logits and log-sum-exps of up to 16 rounded to fp32, 2^-20
        err, norm = (x.double() - exact).norm(dim=0), exact.norm(dim=0)
        assert (err <= 4e-6 * norm).all(), (err / norm).max().item()


@pytest.mark.parametrize("softcap", [7.0, 15.0, 30.0, None])
def test_fp32_probability_of_the_only_class_is_one(softcap):
    """One class: the log-sum-exp is its logit, and the backward finds it to be: a row that is sure of its label has no gradient."""
    from cut_cross_entropy import linear_cross_entropy

    N, D = 8192, 64
    top = softcap or 20.0
    e = (torch.linspace(0.1, 1.5, N, device="cuda") * top / D).repeat(D, 1).T.contiguous().requires_grad_(True)
    c = torch.ones((1, D), device="cuda")
    linear_cross_entropy(e, c, torch.zeros((N,), dtype=torch.int64, device="cuda"), softcap=softcap, reduction="sum").backward()
    x = e.detach().double().sum(1)
    if softcap:
        # either pass forms the soft-capped logit by a hardware exponential and a reciprocal, of one unit in the last place each, and by
        # the same rounded factor; what is left has no sign in common but for those
        th = torch.tanh(x / softcap)
        off = e.grad.double()[:, 0] / (1.0 - th * th)  # p - 1
        assert abs(off.mean()) <= 2.0**-24 * (softcap * th).mean()
    else:
        assert e.grad.double().square().mean().sqrt() <= 2.0**-23


@pytest.mark.parametrize("width", [64, 128, 65536])
def test_fp32_losses_of_small_logits_from_large_factors(width):
    """E ~ 1e-6 and C ~ 5: what is lost of a small operand meets a large one, and the losses, log 2 and a little, show it."""
    from cut_cross_entropy import linear_cross_entropy

    N, V = 500, 2
    g = torch.Generator(device="cuda").manual_seed(1)
    e = torch.randn((N, width), generator=g, device="cuda") * 1e-6
    c = torch.randn((V, width), generator=g, device="cuda").clamp_(-3, 3) * 5.0
    t = torch.randint(0, V, (N,), generator=g, device="cuda")
    loss = linear_cross_entropy(e, c, t, reduction="none")
    x = e.double() @ c.double().T
    want = torch.logsumexp(x, 1) - x[torch.arange(N, device="cuda"), t]
    # three roundings of half a unit of 2^-24 at most: of the loss (0.69), of the logarithm in base 2 and of the sum of two exponentials
    assert (loss.double() - want).square().mean().sqrt() <= 3**0.5 * 2.0**-25


def test_fp32_gradients_keep_all_bits_of_their_operands():
    """Few rows and a head that has not learnt: a row of dC is one row of E times a dz of about -1, a value next to one product."""
    for seed in range(4):
        g = torch.Generator(device="cuda").manual_seed(seed)
        e, c = torch.randn((16, 64), generator=g, device="cuda"), torch.randn((2000, 64), generator=g, device="cuda") * 0.02
        t = torch.randint(0, 2000, (16,), generator=g, device="cuda")
        got, want = _fp32_gradients(e, c, t, torch.zeros((2000,), device="cuda"))
        # two roundings to 24 bits, of dz and of the result, each 2^-24 / sqrt(3) at most as a root mean square, and what dz inherits
        assert (got[1].double() - want[1]).norm() <= 2.0**-23.5 * want[1].norm()


@pytest.mark.parametrize("gap", [10.0, 25.0, 40.0, 70.0])
@pytest.mark.parametrize("rows", [5, 300])
def test_fp32_gradients_of_improbable_classes(gap, rows):
    """Classes that no row expects: their rows of dC and their dBias are small, and as exact for their own size as their probabilities."""
    V, D = 3000, 200
    e, c, t, b, _, _, _, _ = _fp32_case(rows, V, D, 1.0, 12, bias=True)
    b[1000:2000] -= gap
    t %= 1000
    got, want = _fp32_gradients(e, c, t, b)
    # a probability e^-x inherits the roundings of its logit, of x and of x log2(e), half a unit of 2^-23 of gap + 16 each; sums of rows
    rel = 4 * 2.0**-24 * (gap + 16.0)
    dc, want_dc = got[1].double()[1000:2000], want[1][1000:2000]
    err, norm = (dc - want_dc).norm(dim=1), want_dc.norm(dim=1)
    assert (norm > 0).all() and (err <= rel * norm).all(), (err / norm).max().item()
    db, want_db = got[2].double()[1000:2000], want[2][1000:2000]
    assert ((db - want_db).abs() <= rel * want_db.abs()).all()


@pytest.mark.parametrize("where", ["inside", "e", "e, two chunks", "c", "early c", "late c", "upstream", "nan"])
@pytest.mark.parametrize("bias", [False, True])
def test_fp32_values_without_room_in_halves_go_by_parts(where, bias):
    """The largest values that halves of fp16 are used for and the smallest past them, in E, in C, in the first or the second of two chunks of C;
    upstream gradients further apart than one scale serves; one row of NaN.  Against fp64, rows of gradients of their own size."""
    from cut_cross_entropy import linear_cross_entropy

    dev = torch.device("cuda:0")
    N, V, D = (70, 45000, 2048) if where in ("e, two chunks", "early c", "late c") else (300, 700, 200)
    e, c, t, b, w, _, _, _ = _fp32_case(N, V, D, 1.0, 4, bias=bias)
    e[5, 3], c[:, 3] = (255.6 if where.startswith("e,") or where == "e" else 255.5), c[:, 3] * 1e-2
    c[0 if where == "early c" else V - 1, 2], e[:, 2] = (16.0 if where.endswith("c") else 15.96875), e[:, 2] * 1e-2
    if where == "upstream":
        w[7] = 1e-6
    if where == "nan":
        e[9, 11] = float("nan")
    for x in (e, c) + ((b,) if bias else ()):
        x.requires_grad_(True)
    loss, lse = linear_cross_entropy(e, c, t, bias=b, reduction="none", return_lse=True)
    loss.backward(w)
    with torch.no_grad():
        x = e.double() @ c.double().T + (b.double() if bias else 0.0)
        want_lse = torch.logsumexp(x, dim=1)
        rows = torch.arange(N, device=dev)
        want = want_lse - x[rows, t]
        dz = torch.exp(x - want_lse[:, None])
        dz[rows, t] -= 1.0
        dz *= w.double()[:, None]
        want_de, want_dc = dz @ c.double(), dz.T @ e.double()
    if where == "nan":
        ok = rows != 9
        assert lse[9].isnan() and loss[9].isnan() and e.grad[9].isnan().all() and c.grad.isnan().all()
        lse, want_lse, loss, want = lse[ok], want_lse[ok], loss[ok], want[ok]
        pairs = [(e.grad[ok], want_de[ok])]
    else:
        pairs = [(e.grad, want_de), (c.grad, want_dc)]
        if bias:  # sums that may cancel: what each dz inherits from its logit (of up to 10) and from lse rounded to fp32
            assert ((b.grad.double() - dz.sum(0)).abs() <= 4e-6 * dz.abs().sum(0)).all()
    # 2^-23 of |e| |c| <= 4 per logit, random over D, sums of V exponentials; the target logit by D roundings of fp32
    assert torch.allclose(lse.double(), want_lse, atol=4e-6, rtol=2e-6)
    assert torch.allclose(loss.double(), want, atol=2e-5, rtol=2e-6)
    for got, exact in pairs:
        # what dz inherits from the logits and from lse rounded to fp32, and fp32 sums; rows of a small upstream gradient as well
        err, size = (got.double() - exact).norm(dim=1), exact.norm(dim=1)
        assert (err <= 2e-5 * size + 1e-12).all(), (err / size).max().item()


@pytest.mark.parametrize("shape", [(1, 1), (1, 64), (3, 21), (1, 8192), (1, 8193), (7, 1171), (5, 5000)])
@pytest.mark.parametrize("keep", [0.0, 0.4, 1.0])
def test_valid_rows_kernel_matches_the_host(shape, keep):
    """One trip of 8192 positions and its edges, sequences that end inside a wave, nothing and everything ignored."""
    from cut_cross_entropy.utils import _build_flat_valids

    t = torch.randint(0, 50, shape, generator=torch.Generator().manual_seed(1))
    t[torch.rand(shape, generator=torch.Generator().manual_seed(2)) >= keep] = -100
    for shift in (0, 1, 3):
        if shift >= shape[1]:
            continue
        want = _build_flat_valids(t, -100, shift)
        got = _build_flat_valids(t.cuda(), -100, shift)
        assert (want is None) == (got is None)
        if want is not None:
            assert got.dtype == torch.int32 and torch.equal(got.cpu(), want)


@pytest.mark.parametrize("shape", [(127, 9), (255, 64), (256, 64), (257, 65), (511, 1000), (1000, 7), (8200, 70), (3000, 40003)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_bias_gradient_in_ranges_of_rows(shape, dtype):
    """Column sums of dz: one range of rows and several, of 128 rows and a few more, whole lines of 64 classes and parts of one."""
    from cut_cross_entropy import linear_cross_entropy

    (N, V), D = shape, 128
    g = torch.Generator(device="cuda").manual_seed(N + V)
    e = torch.randn((N, D), generator=g, device="cuda").to(dtype)
    c = (torch.randn((V, D), generator=g, device="cuda") * 0.1).to(dtype)
    bias = torch.randn((V,), generator=g, device="cuda").to(dtype).requires_grad_(True)
    t = torch.randint(0, V, (N,), generator=g, device="cuda")
    linear_cross_entropy(e, c, t, bias=bias, reduction="sum", impl="cce_exact").backward()
    dz = torch.softmax(e.double() @ c.double().T + bias.detach().double(), dim=1)
    dz[torch.arange(N, device="cuda"), t] -= 1.0
    # dz is rounded to the type (half a unit of 8 or 11 bits), or inherits from its fp32 logit and log-sum-exp, and is summed in fp32;
    # the result is rounded too
    unit = {torch.bfloat16: 2.0**-8, torch.float16: 2.0**-11, torch.float32: 4e-6}[dtype]
    bound = (unit + 4e-6) * dz.abs().sum(0) + unit * dz.sum(0).abs() + N * (2.0**-25 if dtype == torch.float16 else 0.0)
    assert ((bias.grad.double() - dz.sum(0)).abs() <= bound).all()


@pytest.mark.parametrize("rows", [2048, 8192, 65536])
def test_bias_gradient_of_one_large_entry_among_small_ones(rows):
    """Classes that are the label of one row and improbable in all others: their dBias is rounded with every partial sum that meets the
    large entry, so these are added as trees."""
    from cut_cross_entropy import linear_cross_entropy

    V, D = 64, 64
    bias = torch.zeros((V,), device="cuda")
    bias[0] = 17.0
    bias.requires_grad_(True)
    t = torch.zeros((rows,), dtype=torch.int64)
    t[torch.randperm(rows, generator=torch.Generator().manual_seed(1))[: V - 1]] = torch.arange(1, V)
    linear_cross_entropy(torch.zeros((rows, D), device="cuda"), torch.zeros((V, D), device="cuda"), t.cuda(), bias=bias,
                         reduction="sum").backward()
    want = rows * torch.softmax(bias.detach().double(), 0) - torch.bincount(t, minlength=V).cuda()
    # at most 2^-25 each: the entry; rows of a lane, 3 exchanges, 4 levels of waves, and of up to 64 ranges 8 in a row and 3 levels; the result
    per_lane = -(-rows // (64 * 512))
    assert (bias.grad.double() - want)[1:].square().mean().sqrt() <= (17 + per_lane) ** 0.5 * 2.0**-25 / 3**0.5


@pytest.mark.parametrize("shape", [(1, 16384), (1, 16385), (9, 7001), (40000, 2), (1, 32 * 8192), (1, 32 * 8192 + 1), (3, 200003)])
@pytest.mark.parametrize("keep", [0.0, 0.4, 1.0])
def test_valid_rows_of_several_workgroups_match_the_host(shape, keep):
    """8192 positions a workgroup, and several trips each past 32 of these; sequences that end anywhere in what a workgroup counts."""
    test_valid_rows_kernel_matches_the_host(shape, keep)


@pytest.mark.parametrize("shape,shift", [((2, 4), 4), ((2, 4), 5), ((0, 4), 4), ((2, 0), 1)])
def test_a_shift_past_the_sequences_is_refused(shape, shift):
    """With no label left to compare with there is no loss: an error on either device, and not a mean of nothing."""
    from cut_cross_entropy.utils import _build_flat_valids

    for device in ("cpu", "cuda"):
        with pytest.raises(RuntimeError):
            _build_flat_valids(torch.zeros(shape, dtype=torch.int64, device=device), -100, shift)


@pytest.mark.parametrize("shape,shift", [((2, 4), 4), ((2, 4), 5), ((0, 4), 4), ((2, 0), 1)])
@pytest.mark.parametrize("reduction", ["mean", "sum", "none"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_the_operator_refuses_a_shift_past_the_sequences(shape, shift, reduction, dtype):
    """The same through the operator itself, empty batches among them."""
    from cut_cross_entropy.cce import cce_linear_cross_entropy

    e = torch.randn(shape + (64,), device="cuda", dtype=dtype).requires_grad_(True)
    c = torch.randn((100, 64), device="cuda", dtype=dtype).requires_grad_(True)
    t = torch.zeros(shape, dtype=torch.int64, device="cuda")
    with pytest.raises(RuntimeError, match="No label lies shift="):
        cce_linear_cross_entropy(e, c, t, shift=shift, reduction=reduction, return_lse=True)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shape", [(2, 3, 8), (5, 256 * 70, 128), (130, 700, 123), (1000, 2000, 192)])
@pytest.mark.parametrize("softcap,bias,shift", [(None, False, 0), (15.0, True, 1)])
def test_loss_forward_matches_its_two_halves(dtype, shape, softcap, bias, shift):
    """cce_loss_forward against cce_lse_forward and cce_indexed_neg_dot on the same inputs: more spans than lanes, one
    span, a width the vector loads cannot take, targets that are no class of the shard."""
    from cut_cross_entropy.cce_lse_forward import cce_lse_forward_kernel, loss_forward
    from cut_cross_entropy.indexed_dot import indexed_neg_dot_forward_kernel

    N, V, D = shape
    e, c, t, b = make_inputs(N, V, D, dtype, seed=8, bias=bias)
    t = t * 2 - V // 2  # half of them outside [0, V)
    valids = torch.arange(0, N - shift, 3, dtype=torch.int32).cuda() if shift else None
    e, c, t, b = e.cuda(), c.cuda(), t.cuda(), b.cuda() if b is not None else None
    lse, nll, _ = loss_forward(e, c, b, t, valids, shift, softcap, 0, False)
    want = cce_lse_forward_kernel(e, c, b, valids, softcap)
    dot = indexed_neg_dot_forward_kernel(e, c, t, b, shift, valids, softcap, torch.float32)
    # the same sums in another order: fp32 rounding of quantities of up to 20
    assert torch.allclose(lse, want, atol=4e-6, rtol=4e-7)
    assert torch.allclose(nll, dot + want, atol=8e-6, rtol=1e-6)


@pytest.mark.parametrize("shape", [(1, 4000, 128), (33, 20000, 256), (200, 9000, 2432), (500, 40000, 128), (90, 30000, 4736)])
@pytest.mark.parametrize("fp32_out", [False, True])
@pytest.mark.parametrize("with_dlse,gathered", [(False, False), (True, True)])
def test_filtered_backward_of_few_rows_deals_its_trips(shape, fp32_out, with_dlse, gathered):
    """Few row groups: their trips are dealt to several workgroups with a slot each.  One row group (16 parts), parts that
    get no trip, one to three slices of D.  The same call with less workspace runs one workgroup per row group: the same
    sub-tiles survive, so dC has the same bits, and dE is the same sum in another order."""
    lib = _lib()
    dev = torch.device("cuda:0")
    N, V, D = shape
    g = torch.Generator(device=dev).manual_seed(17)
    c = torch.randn((V, D), generator=g, device=dev).mul_(0.02).bfloat16()
    t = torch.randint(0, V, (N,), generator=g, device=dev)
    other = torch.randint(0, V, (N,), generator=g, device=dev)
    gain = (30.0 / D) ** 0.5 / 0.02
    e = (gain * (c[t].float() + 0.9 * c[other].float()) * 0.2 + torch.randn((N, D), generator=g, device=dev) * 0.1).bfloat16()
    rows = torch.arange(N, device=dev)
    valids = None
    if gathered:
        rows = rows[torch.arange(N, device=dev) % 5 != 3]
        valids = rows.to(torch.int32)
    B = rows.numel()
    w = torch.rand((N,), generator=g, device=dev) + 0.5
    h = torch.randn((N,), generator=g, device=dev) * 0.1 if with_dlse else None
    p = lambda x: x.data_ptr() if x is not None else None
    stream = torch.cuda.current_stream().cuda_stream
    lse = torch.empty((B,), device=dev)
    tile_max = torch.empty((lib.cce_tile_stat_elems(B, V),), device=dev)
    n_ws = lib.cce_lse_forward_workspace_bytes(B, V, D)
    ws = torch.empty((n_ws // 8 + 1,), dtype=torch.int64, device=dev)
    st = lib.cce_lse_forward(p(e), p(c), None, p(valids), p(lse), None, p(tile_max), p(ws), n_ws, N, B, V, D, D, D, 1, 0.0, 0, stream)
    assert st == 0, lib.cce_error_string(st)
    most = lib.cce_backward_workspace_bytes(B, V, D)
    # (a row group's survivor bits, then the count and ids of the class groups left to the second dC pass)
    least = (B + 31) // 32 * (((V + 31) // 32 + 31) // 32) * 4 + (1 + (V + 31) // 32) * 4
    assert most > least  # this shape is dealt out
    gdt = torch.float32 if fp32_out else torch.bfloat16
    got = []
    for n_ws in (most, least):
        ws = torch.full((most // 4 + 1,), float("nan"), device=dev)
        de = torch.zeros((N, D), dtype=gdt, device=dev)
        dc = torch.full((V, D), float("nan"), dtype=gdt, device=dev)
        st = lib.cce_backward(
            p(e), p(c), None, p(lse), p(w), 0, p(h), p(valids), None, p(t), p(tile_max), p(de), p(dc), None, p(ws), n_ws, None,
            N, B, V, D, D, D, 1, 1.0, 2.0**-12, 1, 1, int(fp32_out), int(fp32_out), 0, 0, 0.0, 0, stream)
        assert st == 0, lib.cce_error_string(st)
        got.append((de, dc))
    torch.cuda.synchronize()
    assert torch.isfinite(got[0][0]).all() and torch.isfinite(got[0][1]).all() and got[0][0].abs().max() > 0
    assert torch.equal(got[0][1], got[1][1])
    # the slots are fp32 sums of the same products, 1e-6 of the row's largest apart; two such values on either side of a
    # rounding boundary of bf16 come out one unit in the last place apart, 2^-7 of the value at most
    a, b = got[0][0].double(), got[1][0].double()
    scale = b.abs().amax(dim=1, keepdim=True)
    assert ((a - b).abs() <= (2e-6 if fp32_out else 2.0**-7) * b.abs() + 4e-6 * scale).all()


def _columns_with_rubbish_behind(x, gap):
    """The same matrix as a view whose rows are followed by ``gap`` columns of NaN."""
    wide = torch.full((x.size(0), x.size(1) + gap), float("nan"), dtype=x.dtype, device=x.device)
    wide[:, : x.size(1)] = x
    return wide[:, : x.size(1)]


# One 16-byte piece past a whole stage of the logits (64) or of the ownership kernels (128), one short of it, both sides of
# the halves in between, and a width of two slices of the ownership kernels whose second one ends in a partial stage.
@pytest.mark.parametrize("width", [72, 120, 136, 184, 192, 200, 248, 264, 1000, 2312, 4664])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("path", ["sparse", "dense"])
def test_widths_of_whole_pieces_are_streamed_as_they_lie(monkeypatch, width, dtype, path):
    """A width that is a multiple of 8 gives, bit for bit, what the same matrices with zero columns up to a multiple of 128
    give (the unfiltered backward: within the rounding of its 16-bit results, since the plan of its reductions goes by the
    width), whatever stands behind the rows and in rows that do not count."""
    from cut_cross_entropy import cce_backward as bw
    from cut_cross_entropy import linear_cross_entropy

    monkeypatch.setattr(bw, "FILTERED_BACKWARD_PATH", path)
    N, V = 330, 1300
    e, c, t, bias = make_inputs(N, V, width, dtype, seed=width, invalid_frac=0.2, bias=True)
    e, c, t, bias = e.cuda(), c.cuda(), t.cuda(), bias.cuda()
    ep = torch.nn.functional.pad(e, (0, -width % 128)).requires_grad_(True)
    cp = torch.nn.functional.pad(c, (0, -width % 128)).requires_grad_(True)
    e = torch.where((t == -100)[:, None], torch.full_like(e, float("inf")), e).requires_grad_(True)
    c = _columns_with_rubbish_behind(c, 16).requires_grad_(True)

    def run(e, c):
        return linear_cross_entropy(e, c, t, bias=bias, softcap=20.0, reduction="sum", return_lse=True, impl="cce")

    (got, lse), (want, want_lse) = run(e, c), run(ep, cp)
    assert torch.equal(lse, want_lse)
    # (the target's logit is summed by another kernel, in the order of the width)
    assert abs(got.item() - want.item()) <= 1e-5 * abs(want.item())
    (got + 0.1 * lse.sum()).backward()
    (want + 0.1 * want_lse.sum()).backward()
    if path == "sparse":
        assert torch.equal(e.grad, ep.grad[:, :width]) and torch.equal(c.grad, cp.grad[:, :width])
    else:
        for a, b in ((e.grad, ep.grad), (c.grad, cp.grad)):
            b = b[:, :width].float()
            # both round sums of the same 16-bit dz: two roundings to the type, and fp32 sums in another order
            eps = torch.finfo(dtype).eps
            assert ((a.float() - b).abs() <= 2 * eps * b.abs() + 1e-3 * eps * b.abs().max()).all()
    assert (e.grad[t == -100] == 0).all()


@pytest.mark.parametrize("rows", [2048, 2049])
@pytest.mark.parametrize("moved", ["e", "c", "both"])
def test_packed_matrices_off_a_boundary_are_copied(rows, moved):
    """e or c packed, but starting off a 16-byte boundary, on both sides of the number of rows up to which a ragged
    width is streamed as it lies: the results of aligned matrices, bit for bit."""
    from cut_cross_entropy import linear_cross_entropy

    e, c, t, _ = make_inputs(rows, 300, 136, torch.bfloat16, seed=2)

    def off(x):
        flat = torch.empty((x.numel() + 1,), dtype=x.dtype, device="cuda")
        flat[1:] = x.flatten().cuda()
        return flat[1:].view(x.shape)

    results = []
    for which in ("", moved):
        ed = (off(e) if which in ("e", "both") else e.cuda()).requires_grad_(True)
        cd = (off(c) if which in ("c", "both") else c.cuda()).requires_grad_(True)
        loss = linear_cross_entropy(ed, cd, t.cuda(), impl="cce_exact")
        loss.backward()
        results.append((loss.detach(), ed.grad, cd.grad))
    # (the target's logit alone is summed by whatever kernel the alignment allows)
    assert abs(results[0][0] - results[1][0]) <= 1e-5 * abs(results[0][0])
    assert torch.equal(results[0][1], results[1][1]) and torch.equal(results[0][2], results[1][2])


@pytest.mark.parametrize("width", [1, 63, 64, 65, 123, 129, 1001])
@pytest.mark.parametrize("autocast", [False, True])
def test_other_widths_get_zero_columns(width, autocast):
    """Widths that are no multiple of 8 (or at most one stage) against the formulas in fp64; under autocast fp32 inputs are
    rounded and padded in one pass and their gradients come back in fp32, packed."""
    from cut_cross_entropy import linear_cross_entropy
    from oracle import dense_lce

    N, V = 140, 700
    e, c, t, _ = make_inputs(N, V, width, torch.bfloat16, seed=width, invalid_frac=0.2)
    given = torch.float32 if autocast else torch.bfloat16
    ed, cd = (x.to("cuda", given).requires_grad_(True) for x in (e, c))
    with torch.autocast("cuda", dtype=torch.bfloat16, enabled=autocast):
        loss = linear_cross_entropy(ed, cd, t.cuda(), reduction="sum", impl="cce_exact")
    loss.backward()
    eo, co = e.double().requires_grad_(True), c.double().requires_grad_(True)
    want, _ = dense_lce.dense_linear_cross_entropy(eo, co, t, reduction="sum")
    want.backward()
    assert abs(loss.item() - want.item()) <= 1e-5 * abs(want.item())
    for got, ref in ((ed.grad, eo.grad), (cd.grad, co.grad)):
        assert got.dtype == given and got.is_contiguous() and got.shape == ref.shape
        # dz and the result are rounded to bf16: 2^-9 of every product and of the sum
        assert (got.cpu().double() - ref).norm() <= 4e-3 * ref.norm()


@pytest.mark.parametrize("shape,shift", [((1, 1), 0), ((1, 1), 1), ((3, 85), 0), ((3, 85), 2), ((1, 257), 1), ((4, 64), 70), ((2, 5000), 1)])
@pytest.mark.parametrize("keep", [0.0, 0.5, 1.0])
def test_rows_to_batch_matches_the_library_chain(shape, shift, keep):
    from cut_cross_entropy.utils import _build_flat_valids, handle_reduction_none, rows_to_batch

    g = torch.Generator().manual_seed(sum(shape) + shift)
    t = torch.randint(0, 9, shape, generator=g)
    t[torch.rand(shape, generator=g) >= keep] = -100
    if shift >= shape[1]:
        valids = torch.empty((0,), dtype=torch.int32)
    else:
        valids = _build_flat_valids(t, -100, shift)
        if valids is None:
            valids = torch.arange(t.numel(), dtype=torch.int32)
    values = torch.randn((valids.numel(),), generator=g)
    got = rows_to_batch(t.size(), valids.cuda(), shift, values.cuda())
    assert torch.equal(got.cpu(), handle_reduction_none(t.size(), valids, shift, values))


@pytest.mark.parametrize("rows,classes", [(1, 1), (31, 256 * 32), (32, 2049 * 32), (33, 2048 * 32 - 5), (512 * 32, 700), (512 * 32 + 1, 33), (40000, 5000)])
def test_flagged_cells_are_counted_in_one_launch(rows, classes):
    """One workgroup and several row groups per workgroup, cells of one trip of the loop and more; the word the workgroups
    meet in is zero again for the next launch, and the form that adds to a caller's word counts the same."""
    lib = _lib()
    groups, cols = -(-rows // 32), -(-classes // 32)
    assert lib.cce_tile_stat_elems(rows, classes) == groups * cols
    g = torch.Generator().manual_seed(rows + classes)
    cells = torch.randn((groups, cols), generator=g)
    cells[:: 3, :: 5] = float("-inf")
    lse = torch.randn((rows,), generator=g) + 3.0
    eps = 0.05
    padded = torch.full((groups * 32,), float("inf"))
    padded[:rows] = lse
    log_eps = (torch.tensor(eps).log() - 0.01).item()
    margin = cells - padded.view(groups, 32).amin(1, keepdim=True) - log_eps
    sure, open_ = int((margin > 1e-5).sum()), int((margin.abs() <= 1e-5).sum())  # fp32 rounding of values below 16
    cells, lse = cells.cuda(), lse.cuda()
    scratch = torch.zeros((2,), dtype=torch.int64, device="cuda")
    answer = torch.full((1,), -1, dtype=torch.int64, pin_memory=True)
    stream = torch.cuda.current_stream()
    for _ in range(3):
        answer.fill_(-1)
        assert lib.cce_measure_flagged_cells(cells.data_ptr(), lse.data_ptr(), rows, classes, eps, scratch.data_ptr(),
                                             answer.data_ptr(), stream.cuda_stream) == 0
        stream.synchronize()
        assert sure <= answer.item() <= sure + open_
        assert scratch.tolist() == [0, 0]
    assert lib.cce_count_flagged_cells(cells.data_ptr(), lse.data_ptr(), rows, classes, eps, scratch.data_ptr(), stream.cuda_stream) == 0
    assert scratch[0].item() == answer.item()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows", [1, 63, 64, 65, 127, 128, 129])
@pytest.mark.parametrize("width,classes", [(128, 300), (136, 256 * 257), (192, 512), (200, 2000), (704, 256 * 600 + 1)])
def test_forward_of_few_rows_keeps_three_stages(dtype, rows, width, classes):
    """Up to 128 rows (waves with and without rows), the fewest stages of the ring of three and one less, partial last
    stages, tiles of one span and of several, a cut last tile: log-sum-exp, losses and the cells' maxima."""
    from cut_cross_entropy.cce_lse_forward import loss_forward

    g = torch.Generator().manual_seed(rows + width)
    e = torch.randn((rows + 5, width), generator=g).to(dtype).cuda()
    c = (torch.randn((classes, width), generator=g) * 0.1).to(dtype).cuda()
    t = torch.randint(0, classes, (rows + 5,), generator=g).cuda()
    valids = torch.arange(5, rows + 5, dtype=torch.int32).cuda()
    for softcap, bias in ((None, None), (20.0, None), (None, torch.randn((classes,), generator=g).to(dtype).cuda())):
        for _ in range(2):
            lse, nll, cells = loss_forward(e, c, bias, t, valids, 0, softcap, 0, True)
        x = e[5:].float() @ c.float().T
        if bias is not None:
            x += bias.float()
        if softcap is not None:
            x = softcap * torch.tanh(x / softcap)
        want = torch.logsumexp(x, 1)
        # fp32 sums of `width` products of values around 1 and 0.1, then of the classes' exponentials
        assert (lse - want).abs().max() < 2e-5 * max(1.0, want.abs().max().item())
        assert (nll - (want - x.gather(1, t[5:, None])[:, 0])).abs().max() < 1e-4
        rb, cb = -(-rows // 32), -(-classes // 32)
        padded = torch.full((rb * 32, cb * 32), float("-inf"), device="cuda")
        padded[:rows, :classes] = x
        top = padded.view(rb, 32, cb, 32).amax((1, 3))
        assert (cells.view(rb, cb) - top).abs().max() < 2e-4


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("softcap", [None, 30.0, 50.0])
@pytest.mark.parametrize("rows,width", [(40, 64), (70, 192), (300, 136), (300, 256), (130, 123)])
def test_a_row_that_is_not_a_number_says_so(dtype, softcap, rows, width):
    """A NaN in a row that counts: its log-sum-exp and its loss are NaN, also where its label is no class of the shard (the
    loss is then the log-sum-exp alone); every other row has the values it has beside a row of zeros."""
    from cut_cross_entropy import VocabParallelOptions, linear_cross_entropy

    classes, bad = 3000, 33
    e, c, t, _ = make_inputs(rows, classes, width, dtype, seed=rows)
    e[bad] = 0.0
    e, c, t = e.cuda(), c.cuda(), t.cuda()
    spoilt = e.clone()
    spoilt[bad, 7] = float("nan")
    for shard in (None, VocabParallelOptions(0, classes)):
        labels = t.clone()
        if shard is not None:
            labels[bad] = classes + 5
        got, want = (linear_cross_entropy(x, c, labels, softcap=softcap, reduction="none", return_lse=True, impl="cce",
                                          vocab_parallel_options=shard) for x in (spoilt, e))
        others = torch.arange(rows, device="cuda") != bad
        for x, y in zip(got, want):
            assert torch.isfinite(y).all()
            assert torch.isnan(x[bad]) and torch.equal(x[others], y[others])


@pytest.mark.parametrize("shape", [(1, 700, 64), (300, 2000, 200), (3000, 100, 72)])
@pytest.mark.parametrize("past", [False, True])
def test_fp32_column_sums_keep_their_bits_with_three_terms(shape, past):
    """dBias is a sum of fp32 values and no product: with operands of 8 significant bits, whose logits three terms give
    exactly, it is bit for bit what six terms give; the logits from halves of fp16, or with a value past those from bf16 parts."""
    lib = _lib()
    N, V, D = shape
    g = torch.Generator(device="cuda").manual_seed(N)
    e = torch.randn((N, D), generator=g, device="cuda").bfloat16().float()
    c = (torch.randn((V, D), generator=g, device="cuda") / D**0.5).bfloat16().float()
    t = torch.randint(0, V, (N,), generator=g, device="cuda")
    w = torch.rand((N,), generator=g, device="cuda") + 0.5
    if past:
        e[0, 0], c[:, 0] = 320.0, c[:, 0] / 64
    lse = torch.logsumexp((e.double() @ c.double().T), 1).float()
    p = lambda x: x.data_ptr()
    sums = []
    for terms in (6, 3):
        n_ws = lib.cce_fp32_backward_workspace_bytes(N, V, D, terms)
        buf = torch.full((n_ws // 4 + 64,), float("nan"), device="cuda")
        ws = (buf.data_ptr() + 255) // 256 * 256
        de, dc, db = torch.zeros((N, D), device="cuda"), torch.empty((V, D), device="cuda"), torch.zeros((V,), device="cuda")
        st = lib.cce_fp32_backward(p(e), p(c), None, p(lse), p(w), 0, None, None, p(t), p(de), p(dc), p(db), ws, n_ws, N, N, V, D,
                                   D, D, 1, D, D, 1.0, 0, 0, 0.0, terms, torch.cuda.current_stream().cuda_stream)
        assert st == 0, lib.cce_error_string(st)
        sums.append(db)
    assert torch.isfinite(sums[0]).all() and sums[0].abs().max() > 0 and torch.equal(*sums)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("which", ["e", "c", "both"])
@pytest.mark.parametrize("width", [5, 8, 72, 128])
def test_a_single_row_with_a_stride_of_its_own(dtype, which, width):
    """One row of e, or one class, whose stride says nothing (the transpose of a [D, 1] column): as if it were packed."""
    from cut_cross_entropy import linear_cross_entropy

    N, V = (1 if which in ("e", "both") else 9), (1 if which in ("c", "both") else 300)
    e, c, _, _ = make_inputs(N, V, width, dtype, seed=width)
    t = torch.randint(0, V, (N,), generator=torch.Generator().manual_seed(1)).cuda()

    def column(x, moved):
        return torch.as_strided(x.cuda().flatten().clone(), x.shape, (1, 1)) if moved else x.cuda()

    results = []
    for moved in (False, True):
        ed, cd = column(e, moved and which != "c").requires_grad_(True), column(c, moved and which != "e").requires_grad_(True)
        loss = linear_cross_entropy(ed, cd, t, impl="cce_exact")
        loss.backward()
        results.append((loss.detach(), ed.grad, cd.grad))
    for a, b in zip(*results):
        assert torch.isfinite(a).all() and torch.equal(a, b)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows", [129, 191, 192, 193, 300, 384, 385, 576])
@pytest.mark.parametrize("width,classes", [(128, 256), (136, 1000), (192, 256 * 40 + 1), (704, 256 * 130)])
def test_forward_in_blocks_of_192_rows(dtype, rows, width, classes):
    """Blocks of 192 rows where 256 would be padding or an emptier last round: the edges of the blocks and of the cells in them, gathered
    rows, partial stages, cut tiles, several tiles per span; log-sum-exp, losses and the cells' maxima."""
    from cut_cross_entropy.cce_lse_forward import loss_forward

    g = torch.Generator().manual_seed(rows + width)
    e = torch.randn((rows + 5, width), generator=g).to(dtype).cuda()
    c = (torch.randn((classes, width), generator=g) * 0.1).to(dtype).cuda()
    t = torch.randint(0, classes, (rows + 5,), generator=g).cuda()
    valids = torch.arange(5, rows + 5, dtype=torch.int32).cuda()
    for softcap, bias in ((None, None), (20.0, None), (50.0, torch.randn((classes,), generator=g).to(dtype).cuda())):
        lse, nll, cells = loss_forward(e, c, bias, t, valids, 0, softcap, 0, True)
        x = e[5:].float() @ c.float().T
        if bias is not None:
            x += bias.float()
        if softcap is not None:
            x = softcap * torch.tanh(x / softcap)
        want = torch.logsumexp(x, 1)
        # the bounds of test_forward_of_few_rows_keeps_three_stages: the same sums in fp32
        assert (lse - want).abs().max() < 2e-5 * max(1.0, want.abs().max().item())
        assert (nll - (want - x.gather(1, t[5:, None])[:, 0])).abs().max() < 1e-4
        rb, cb = -(-rows // 32), -(-classes // 32)
        padded = torch.full((rb * 32, cb * 32), float("-inf"), device="cuda")
        padded[:rows, :classes] = x
        top = padded.view(rb, 32, cb, 32).amax((1, 3))
        assert (cells.view(rb, cb) - top).abs().max() < 2e-4


@pytest.mark.parametrize("shape,shift", [((1, 1), 0), ((3, 85), 0), ((3, 85), 2), ((1, 257), 1), ((2, 2, 5), 4), ((2, 5000), 1)])
@pytest.mark.parametrize("keep", [0.0, 0.5, 1.0])
def test_rows_to_steps_and_back(shape, shift, keep):
    """Per-row values laid out without the first steps of each sequence, and their gradients padded with zeros again: what slicing
    the whole batch and autograd's way back through the slice give."""
    from cut_cross_entropy.utils import flat_valids, handle_reduction_none, rows_to_steps, steps_to_batch

    g = torch.Generator().manual_seed(sum(shape) + shift)
    t = torch.randint(0, 9, shape, generator=g)
    t[torch.rand(shape, generator=g) >= keep] = -100
    valids = flat_valids(t, -100, shift)
    if valids is None:
        valids = torch.arange(t.numel(), dtype=torch.int32)
    for sets in (1, 2, 3):
        values = [torch.randn((valids.numel(),), generator=g) if sets >> k & 1 else None for k in range(2)]
        got = rows_to_steps(t.size(), valids.cuda(), shift, *(None if v is None else v.cuda() for v in values))
        for v, out in zip(values, got):
            assert (v is None) == (out is None)
            if v is not None:
                assert torch.equal(out.cpu(), handle_reduction_none(t.size(), valids, shift, v)[..., shift:])
        back = steps_to_batch(t.size(), shift, *got)
        for out, flat in zip(got, back):
            if out is not None:
                want = torch.zeros(shape)
                want[..., shift:] = out.cpu()
                assert torch.equal(flat.cpu(), want.view(-1))


@pytest.mark.parametrize("shape", [(0,), (3, 0), (0, 5)])
@pytest.mark.parametrize("reduction", ["mean", "sum", "none"])
def test_no_labels_at_all(shape, reduction):
    """Batches without a position: nothing to sum, values in the (empty) batch shape, gradients of zeros."""
    from cut_cross_entropy.cce import cce_linear_cross_entropy

    e = torch.randn(shape + (64,), device="cuda", dtype=torch.bfloat16).requires_grad_(True)
    c = torch.randn((100, 64), device="cuda", dtype=torch.bfloat16).requires_grad_(True)
    t = torch.zeros(shape, dtype=torch.int64, device="cuda")
    loss, lse = cce_linear_cross_entropy(e, c, t, reduction=reduction, return_lse=True)
    assert lse.shape == shape and loss.shape == (shape if reduction == "none" else ())
    if reduction != "none":
        assert loss.isnan() if reduction == "mean" else loss.item() == 0.0
    (loss.sum() + lse.sum()).backward()
    assert e.grad.shape == e.shape and not c.grad.any()


@pytest.mark.parametrize("shape,shift", [((1,), 0), ((2, 1), 0), ((70,), 3), ((3, 85), 2), ((2, 3, 50), 1), ((1, 16384), 0), ((1, 16385), 0),
                                         ((5, 3277), 1), ((3, 1400001), 1)])
@pytest.mark.parametrize("reduction", ["mean", "sum", "none"])
@pytest.mark.parametrize("labels", ["some", "none", "all ignored", "not given"])
def test_z_loss_kernels_against_tensor_operations(shape, shift, reduction, labels):
    """One value, one workgroup, one value more than that, and more values than the workgroups take once; slices of longer sequences;
    what a masked position holds (NaN, infinities) stays out of the value.  Bits of the single squares and gradients; sums in
    fp64 rounded once, which is as near as fp32 gets."""
    from cut_cross_entropy import utils

    g = torch.Generator().manual_seed(sum(shape) + shift)
    whole = (torch.randn(shape, generator=g) * 3 + 9).cuda()
    t = torch.randint(0, 50, shape, generator=g)
    t[torch.rand(shape, generator=g) < 0.3] = -100
    if labels == "all ignored":
        t[...] = -100
    elif labels == "none":
        t.clamp_(min=0)
    t = None if labels == "not given" else t.cuda()
    n_masked = 0
    if labels == "some" and whole[..., shift:].numel() > 2:
        masked = (t[..., shift:] == -100).nonzero()
        n_masked = len(masked)
        if n_masked:
            whole[..., shift:][tuple(masked[0])] = float("inf")
            whole[..., shift:][tuple(masked[-1])] = float("nan")
    lse = whole[..., shift:].detach().requires_grad_(True)
    assert utils._z_loss_has_kernels(lse.detach(), t, shift, -100)
    out = utils.compute_z_loss(lse, t, shift, reduction=reduction)
    up = torch.rand(out.shape, generator=g).cuda() + 0.5
    (grad,) = torch.autograd.grad(out, lse, up, retain_graph=True)

    ref = lse.detach().requires_grad_(True)
    sq = ref.square()
    if t is not None:
        sq = sq.masked_fill(t[..., shift:] == -100, 0.0)
    if reduction == "none":
        assert torch.equal(out, sq) and out.shape == sq.shape
        want = sq
    else:
        total = sq.double().sum()
        counted = sq.numel() if t is None else (t[..., shift:] != -100).sum()
        want = total if reduction == "sum" else total.float() / counted
        assert torch.allclose(out.double(), want.double(), rtol=2e-7, atol=0, equal_nan=True) and out.shape == ()
    (want_grad,) = torch.autograd.grad(want.float(), ref, up)
    # (the reference divides where the kernel does; NaN under a mask stays NaN in a gradient: 0 x NaN)
    assert grad.shape == want_grad.shape and torch.allclose(grad, want_grad, rtol=2e-7, atol=0, equal_nan=True)

    # a graph of the gradient, and what the kernels are not for: the same function by tensor operations
    if whole.numel() < 1000 and not n_masked and labels != "all ignored":  # (0 / 0 has no tangent)
        (g1,) = torch.autograd.grad(out, lse, up, create_graph=True)
        assert torch.allclose(g1, want_grad, rtol=2e-7, atol=0, equal_nan=True)
        (g2,) = torch.autograd.grad(g1.sum(), lse)
        assert torch.allclose(g2 * lse.detach(), want_grad, rtol=1e-6, atol=0)
        plain = lse.detach()
        # several upstream gradients at once, which autograd batches without storage
        pair = torch.stack([up, 2 * up])
        (both,) = torch.autograd.grad(out, lse, pair, retain_graph=True, is_grads_batched=True)
        for one, k in zip(both, (1, 2)):
            assert torch.allclose(one, k * want_grad, rtol=4e-7, atol=0, equal_nan=True)
        import torch.autograd.forward_ad as fwAD

        with fwAD.dual_level():
            dual = utils.compute_z_loss(fwAD.make_dual(plain, torch.ones_like(plain)), t, shift, reduction=reduction)
            tangent = fwAD.unpack_dual(dual).tangent
        (all_ones,) = torch.autograd.grad(utils.compute_z_loss(lse, t, shift, reduction=reduction).sum(), lse)
        assert torch.allclose(tangent.sum(), all_ones.sum(), rtol=1e-5, atol=1e-5, equal_nan=True)
        pair = torch.vmap(lambda x: utils.compute_z_loss(x, t, shift, reduction=reduction))(torch.stack([plain, plain]))
        assert torch.allclose(pair[1], out.detach(), rtol=1e-6, atol=0, equal_nan=True)


@pytest.mark.parametrize("shape,shift", [((3, 85), 2), ((5, 3277), 1)])
@pytest.mark.parametrize("reduction", ["mean", "sum", "none"])
def test_labels_overwritten_after_the_z_loss(shape, shift, reduction):
    """A label buffer that the next batch is written to before the gradients are taken: those of the labels that the loss saw, also
    for a graph of the gradient and for several upstream gradients at once."""
    from cut_cross_entropy import utils

    g = torch.Generator().manual_seed(3)
    lse = (torch.randn(shape, generator=g) * 3 + 9).cuda()[:, shift:].detach().requires_grad_(True)
    t = torch.randint(0, 50, shape, generator=g)
    t[torch.rand(shape, generator=g) < 0.3] = -100
    t = t.cuda()
    masked = t[:, shift:] == -100
    sq = lse.square().masked_fill(masked, 0.0)
    want = sq if reduction == "none" else sq.sum() / (1 if reduction == "sum" else (~masked).sum())
    out = utils.compute_z_loss(lse, t, shift, reduction=reduction)
    t.copy_(torch.where(t == -100, 7, -100))
    up = torch.rand(out.shape, generator=g).cuda() + 0.5
    (want_grad,) = torch.autograd.grad(want, lse, up)
    (graphed,) = torch.autograd.grad(out, lse, up, create_graph=True)
    (both,) = torch.autograd.grad(out, lse, torch.stack([up, up]), retain_graph=True, is_grads_batched=True)
    (grad,) = torch.autograd.grad(out, lse, up)
    for got in (grad, graphed, both[0], both[1]):
        assert torch.allclose(got, want_grad, rtol=4e-7, atol=0)


@pytest.mark.parametrize("reduction", ["mean", "none"])
@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_upstream_gradients_that_are_lazily_negated(reduction, shift, dtype):
    """What sends the gradients of imaginary parts back through a conjugate sends views with the negative bit set: the same gradients
    as from plain tensors, of the loss, of the log-sum-exps and of the z-loss."""
    from cut_cross_entropy import linear_cross_entropy, utils

    class Negated(torch.autograd.Function):
        @staticmethod
        def forward(ctx, x):
            return x.clone()

        @staticmethod
        def backward(ctx, g):
            return torch._neg_view((-g).contiguous())

    g = torch.Generator().manual_seed(2)
    e0 = torch.randn((3, 40, 128), generator=g).to(dtype).cuda()
    c0 = (torch.randn((500, 128), generator=g) * 0.1).to(dtype).cuda()
    t = torch.randint(0, 500, (3, 40), generator=g).cuda()
    got = []
    for through in (lambda x: x.clone(), Negated.apply):
        e, c = e0.clone().requires_grad_(True), c0.clone().requires_grad_(True)
        loss, lse = linear_cross_entropy(e, c, t, shift=shift, reduction=reduction, return_lse=True)
        z = utils.compute_z_loss(lse, t, shift, reduction=reduction)
        (through(loss).sum() + 1e-2 * through(lse).sum() + 1e-2 * through(z).sum()).backward()
        got.append((e.grad, c.grad))
    assert got[0][0].any() and torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])


@pytest.mark.parametrize("reduction", ["mean", "sum", "none"])
def test_a_trace_of_the_z_loss_can_be_saved(reduction):
    """torch.jit.trace records tensor operations: the trace is saved, loaded and run on other labels and values."""
    import io

    from cut_cross_entropy import utils

    g = torch.Generator().manual_seed(1)
    lse, other = (torch.randn((3, 6), generator=g).cuda() + 5 for _ in range(2))
    t = torch.tensor([[0, -100, 1, 2, 3, 4, 5]] * 3).cuda()
    traced = torch.jit.trace(lambda x, labels: utils.compute_z_loss(x, labels, 1, reduction=reduction), (lse, t))
    file = io.BytesIO()
    torch.jit.save(traced, file)
    file.seek(0)
    loaded = torch.jit.load(file)
    for x, labels in ((lse, t), (other, t.roll(2, 1))):
        # at most 18 additions of one sign, in either order
        assert torch.allclose(loaded(x, labels), utils.compute_z_loss(x, labels, 1, reduction=reduction), rtol=18 * 2.0**-23, atol=0)


@pytest.mark.parametrize("layout", ["sliced", "permuted", "expanded", "several"])
@pytest.mark.parametrize("reduction", ["mean", "none"])
def test_z_loss_of_layouts_with_dimensions_of_one_entry(layout, reduction):
    """Dimensions of one entry between larger ones: layouts that one stride leads through and layouts that it does not, for the
    log-sum-exps and for the labels."""
    from cut_cross_entropy import utils

    def laid_out(x):
        x = x.cuda()
        return {"sliced": lambda: x.view(4, 1, 12, 8)[:, :, :5], "permuted": lambda: x[:160].view(5, 4, 1, 8).permute(1, 2, 0, 3),
                "expanded": lambda: x[:32].view(4, 1, 1, 8).expand(4, 1, 3, 8),
                "several": lambda: x.view(4, 1, 3, 1, 32)[:, :, 1:2, :, 1:9]}[layout]()

    g = torch.Generator().manual_seed(5)
    values = torch.randn((384,), generator=g) * 3 + 9
    labels = torch.randint(0, 50, (384,), generator=g)
    labels[torch.rand((384,), generator=g) < 0.3] = -100
    for lse, t in ((laid_out(values), laid_out(labels)), (laid_out(values).contiguous(), laid_out(labels)),
                   (laid_out(values), laid_out(labels).contiguous())):
        lse = lse.detach().requires_grad_(True)
        out = utils.compute_z_loss(lse, t, reduction=reduction)
        up = torch.rand(out.shape, generator=g).cuda() + 0.5
        (grad,) = torch.autograd.grad(out, lse, up)
        ref = lse.detach().contiguous().requires_grad_(True)
        sq = ref.square().masked_fill(t == -100, 0.0)
        want = sq if reduction == "none" else sq.sum() / (t != -100).sum()
        (want_grad,) = torch.autograd.grad(want, ref, up)
        # at most 384 fp32 additions of values of one sign in the reference
        assert torch.allclose(out, want, rtol=384 * 2.0**-24, atol=0) and torch.allclose(grad, want_grad, rtol=2e-7, atol=0)


@pytest.mark.parametrize("shape,budget", [((4744, 6303, 320), 7 << 20), ((5308, 4438, 128), 5 << 20), ((9380, 4245, 320), 16 << 20),
                                          ((10691, 3041, 192), 11 << 20)])
def test_cut_reductions_in_more_launches(monkeypatch, shape, budget):
    """Buffers in which the slots of a cut reduction fit only beside smaller chunks than whole reductions would take: dC cut chunk by
    chunk, dE cut block by block, several launches of either.  Against the formulas in fp64."""
    from cut_cross_entropy import cce_backward as bw
    from cut_cross_entropy import linear_cross_entropy

    monkeypatch.setattr(bw, "DENSE_DZ_BYTES", budget)
    monkeypatch.setattr(bw, "DENSE_DZ_MIN_CLASSES", 256)
    N, V, D = shape
    e, c, t, _ = make_inputs(N, V, D, torch.bfloat16, seed=9, planted=False, c_std=0.3)
    e, c, t = e.cuda().requires_grad_(True), c.cuda().requires_grad_(True), t.cuda()
    linear_cross_entropy(e, c, t, reduction="sum", impl="cce_exact").backward()
    p = torch.softmax(e.detach().double() @ c.detach().double().T, 1)
    p[torch.arange(N, device="cuda"), t] -= 1.0
    for got, want in ((e.grad, p @ c.detach().double()), (c.grad, p.T @ e.detach().double())):
        # dz and the result are rounded to bf16, 2^-9 of every product and of the sum: the bound of the cuts above
        assert torch.isfinite(got).all() and (got.double() - want).norm() <= 6e-3 * want.norm()


@pytest.mark.parametrize("shape", [(8200, 2500, 2432), (4500, 1000, 2312), (8192, 3000, 4736)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("few_labels", [False, True])
def test_gradients_kept_between_the_filtered_passes(monkeypatch, shape, dtype, few_labels):
    """Widths in slices: the dE pass keeps the gradients of surviving sub-tiles, slices after the first (a launch of their own from 256 row
    groups on) and the dC pass read them.  Candidates that all have a slot (the labels of 32 rows), a partial last stage, against the
    same call with a bias of zeros, for whose gradient everything is formed again.  (More candidates than slots: below.)"""
    from cut_cross_entropy import cce_backward as bw
    from cut_cross_entropy import linear_cross_entropy

    monkeypatch.setattr(bw, "FILTERED_BACKWARD_PATH", "sparse")
    N, V, D = shape
    g = torch.Generator(device="cuda").manual_seed(N + V)
    c = (torch.randn((V, D), generator=g, device="cuda") * 0.02).to(dtype)
    t = torch.randint(0, 40 if few_labels else V, (N,), generator=g, device="cuda")
    other = torch.randint(0, V, (N,), generator=g, device="cuda")
    gain = (30.0 / D) ** 0.5 / 0.02
    e = gain * (c[t].float() + 0.9 * c[other].float()) * 0.2 + torch.randn((N, D), generator=g, device="cuda") * 0.1
    e = e.to(dtype)
    got = []
    for bias in (None, torch.zeros((V,), dtype=dtype, device="cuda", requires_grad=True)):
        e1, c1 = e.clone().requires_grad_(True), c.clone().requires_grad_(True)
        linear_cross_entropy(e1, c1, t, bias=bias, softcap=50.0, reduction="sum", filter_eps=2.0**-9).backward()
        got.append((e1.grad.double(), c1.grad.double()))
    for a, b in zip(*got):
        assert torch.isfinite(a).all() and a.abs().max() > 0
        # dz is rounded to the type from logits summed in another order: 2^-9 (bf16) of single products, and of the results
        assert (a - b).norm() <= 2e-3 * b.norm()
        assert ((a - b).abs() <= 2e-2 * b.abs() + 2e-2 * b.abs().amax(dim=1, keepdim=True)).all()


@pytest.mark.parametrize("shape,likely", [((8200, 2500, 2432), 6), ((4500, 1900, 2312), 3), ((8192, 3000, 4736), 2), ((4500, 60000, 2432), 1)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_more_candidates_than_slots_for_kept_gradients(monkeypatch, shape, likely, dtype):
    """Rows with several likely classes: row groups with more candidates than the 40 slots beside groups with fewer, so that trips read
    kept gradients, form them again, and do either for some of their entries; and, with classes many against the rows, class groups of one
    or two survivors, which the light dC pass takes.  What each is here for is counted in plain torch.  Reference and bounds as above."""
    from cut_cross_entropy import cce_backward as bw
    from cut_cross_entropy import linear_cross_entropy
    from cut_cross_entropy.cce_lse_forward import loss_forward

    monkeypatch.setattr(bw, "FILTERED_BACKWARD_PATH", "sparse")
    N, V, D = shape
    eps, softcap, quota = 2.0**-9, 50.0, 40
    g = torch.Generator(device="cuda").manual_seed(N + V)
    c = (torch.randn((V, D), generator=g, device="cuda") * 0.02).to(dtype)
    # a logit of 12 for each of `likely` classes; every fourth row group has its labels alone, all in one sub-tile
    pick = torch.randint(0, V, (likely, N), generator=g, device="cuda")
    few = (torch.arange(N, device="cuda") // 32) % 4 == 0
    pick[:, few] = torch.randint(0, 32, (1, int(few.sum())), generator=g, device="cuda")
    t = pick[0].clone()
    e = torch.randn((N, D), generator=g, device="cuda") * 0.1
    for classes in pick:
        add = 12.0 / (D * 0.02**2) * c[classes].float()
        e += torch.where(few[:, None], add / likely, add)
    e = e.to(dtype)

    # candidates of a row group: sub-tiles whose largest logit can make a probability of eps in one of its rows, and those of its labels
    lse, _, tile_max = loss_forward(e, c, None, t, None, 0, softcap, 0, True)
    groups, blocks = -(-N // 32), -(-V // 32)
    low = torch.nn.functional.pad(lse, (0, groups * 32 - N), value=float("inf")).view(groups, 32).amin(1)
    candidate = tile_max.view(groups, blocks) - low[:, None] >= torch.log(torch.tensor(eps)).item()
    candidate[torch.arange(N, device="cuda") // 32, t // 32] = True
    per_group = candidate.sum(1)
    p = torch.exp(softcap * torch.tanh((e.float() @ c.float().T) / softcap) - lse[:, None])
    p[torch.arange(N, device="cuda"), t] -= 1.0
    p = torch.nn.functional.pad(p.abs(), (0, blocks * 32 - V, 0, groups * 32 - N)).view(groups, 32, blocks, 32).amax((1, 3)) >= eps
    if V < 10000:
        assert (per_group > quota).sum() > groups // 2 and (per_group <= quota).any()
        # survivors behind the last slot, and class groups whose list holds survivors of either kind
        late = p & candidate & (candidate.cumsum(1) > quota)
        assert (late.any(0) & (p & candidate & ~late).any(0)).sum() > 4
    else:
        light = ((p & candidate).sum(0) >= 1) & ((p & candidate).sum(0) <= 2)
        assert light.sum() > 500 and (p.sum(0) > 2).any()

    got = []
    for bias in (None, torch.zeros((V,), dtype=dtype, device="cuda", requires_grad=True)):
        e1, c1 = e.clone().requires_grad_(True), c.clone().requires_grad_(True)
        linear_cross_entropy(e1, c1, t, bias=bias, softcap=softcap, reduction="sum", filter_eps=eps).backward()
        got.append((e1.grad.double(), c1.grad.double()))
    for a, b in zip(*got):
        assert torch.isfinite(a).all() and a.abs().max() > 0
        assert (a - b).norm() <= 2e-3 * b.norm()
        assert ((a - b).abs() <= 2e-2 * b.abs() + 2e-2 * b.abs().amax(dim=1, keepdim=True)).all()


@pytest.mark.parametrize("shape,likely", [((1, 4000, 128), 1), ((33, 20000, 72), 1), ((300, 30000, 2432), 2), ((130, 9000, 2056), 1),
                                          ((90, 30000, 4736), 1), ((3200, 26000, 256), 4), ((64, 30000, 2056), 48)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_gradients_kept_where_few_row_groups_are_dealt_out(monkeypatch, shape, likely, dtype):
    """Row groups dealt to 2 - 16 workgroups keep the gradients of what survives too, 40 slots for each workgroup, in one slice of D or
    several; from 2048 columns on the light dC pass is in two slices, the last one partial (2056 = 1152 + 904); the last two shapes have row
    groups with more candidates than that, one of them for the light pass in two slices.  Against the same call with a bias of zeros, as above."""
    from cut_cross_entropy import _hip
    from cut_cross_entropy import cce_backward as bw
    from cut_cross_entropy import linear_cross_entropy
    from cut_cross_entropy.cce_lse_forward import loss_forward

    monkeypatch.setattr(bw, "FILTERED_BACKWARD_PATH", "sparse")
    N, V, D = shape
    eps, softcap = 2.0**-9, 50.0
    lib, groups, blocks = _hip.load(), -(-N // 32), -(-V // 32)
    words = -(-blocks // 32)
    kept = lib.cce_backward_keeping_workspace_bytes(N, V, D) - lib.cce_backward_unkept_workspace_bytes(N, V, D) - groups * words * 4
    quota = kept // (groups * 2048)
    assert quota >= 80 and quota % 40 == 0
    g = torch.Generator(device="cuda").manual_seed(N + V)
    c = (torch.randn((V, D), generator=g, device="cuda") * 0.02).to(dtype)
    pick = torch.randint(0, V, (likely, N), generator=g, device="cuda")
    t = pick[0].clone()
    e = torch.randn((N, D), generator=g, device="cuda") * 0.1
    for classes in pick:
        e += 12.0 / (D * 0.02**2) * c[classes].float()
    e = e.to(dtype)
    lse, _, tile_max = loss_forward(e, c, None, t, None, 0, softcap, 0, True)
    low = torch.nn.functional.pad(lse, (0, groups * 32 - N), value=float("inf")).view(groups, 32).amin(1)
    candidates = (tile_max.view(groups, blocks) - low[:, None] >= torch.log(torch.tensor(eps)).item()).sum(1)
    assert (candidates > quota).any() == (N in (64, 3200))

    got = []
    for bias in (None, torch.zeros((V,), dtype=dtype, device="cuda", requires_grad=True)):
        e1, c1 = e.clone().requires_grad_(True), c.clone().requires_grad_(True)
        linear_cross_entropy(e1, c1, t, bias=bias, softcap=softcap, reduction="sum", filter_eps=eps).backward()
        got.append((e1.grad.double(), c1.grad.double()))
    for a, b in zip(*got):
        assert torch.isfinite(a).all() and a.abs().max() > 0
        assert (a - b).norm() <= 2e-3 * b.norm()
        assert ((a - b).abs() <= 2e-2 * b.abs() + 2e-2 * b.abs().amax(dim=1, keepdim=True)).all()


@pytest.mark.parametrize("call,keeps", [("plain", True), ("frozen e", True), ("frozen c", False), ("bias", False), ("frozen bias", True),
                                        ("unfiltered c", False), ("unfiltered e", True), ("no filter", None)])
def test_room_for_kept_gradients_only_where_they_are_kept(monkeypatch, call, keeps):
    """Which calls bring the larger workspace.  With dE unfiltered the ownership kernels are left with dC, whose passes keep."""
    from cut_cross_entropy import _hip
    from cut_cross_entropy import cce_backward as bw
    from cut_cross_entropy import linear_cross_entropy

    monkeypatch.setattr(bw, "FILTERED_BACKWARD_PATH", "sparse")
    N, V, D = 1200, 1000, 2432
    lib, brought = _hip.load(), []
    least, most = lib.cce_backward_unkept_workspace_bytes(N, V, D), lib.cce_backward_workspace_bytes(N, V, D)
    assert most - least >= (N // 32) * 40 * 2048

    class Recorded:
        def __getattr__(self, name):
            if name == "cce_backward":
                return lambda *a: brought.append(a[15]) or lib.cce_backward(*a)
            return getattr(lib, name)

    monkeypatch.setattr(_hip, "load", lambda: Recorded())
    g = torch.Generator().manual_seed(4)
    e = torch.randn((N, D), generator=g).to(torch.bfloat16).cuda().requires_grad_(call != "frozen e")
    c = (torch.randn((V, D), generator=g) * 0.05).to(torch.bfloat16).cuda().requires_grad_(call != "frozen c")
    t = torch.randint(0, V, (N,), generator=g).cuda()
    bias = torch.zeros((V,), dtype=torch.bfloat16, device="cuda", requires_grad=call == "bias") if "bias" in call else None
    impl = {"unfiltered c": "cce_kahan_full_c", "unfiltered e": "cce_kahan_full_e", "no filter": "cce_exact"}.get(call, "cce")
    linear_cross_entropy(e, c, t, bias=bias, impl=impl).backward()
    if keeps is None:
        assert not brought
    else:
        (got,) = brought
        assert got >= most if keeps else least <= got < least + 16
    if keeps:  # the same gradient where everything is formed again (a bias of zeros that wants one); bound as above
        e1, c1 = e.detach().clone().requires_grad_(e.requires_grad), c.detach().clone().requires_grad_(True)
        linear_cross_entropy(e1, c1, t, bias=torch.zeros((V,), dtype=c.dtype, device="cuda", requires_grad=True), impl=impl).backward()
        for x, y in ((c, c1),) if call == "frozen e" else ((e, e1), (c, c1)):
            assert y.grad.any() and (x.grad.double() - y.grad.double()).norm() <= 2e-3 * y.grad.double().norm()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows", [129, 191, 192, 193, 300, 384, 385, 576])
@pytest.mark.parametrize("width,classes", [(128, 256), (136, 1000), (192, 256 * 40 + 1), (704, 256 * 130)])
def test_logit_gradients_in_blocks_of_192_rows(dtype, rows, width, classes):
    """The blocks of test_forward_in_blocks_of_192_rows in the kernel that forms dz: gathered rows, partial stages, cut tiles, several
    tiles per item, soft-cap and bias.  Seen through dBias (the sums of dz over the rows) and the two products."""
    from cut_cross_entropy import linear_cross_entropy

    g = torch.Generator().manual_seed(rows + width)
    e0 = torch.randn((rows + 5, width), generator=g).to(dtype).cuda()
    c0 = (torch.randn((classes, width), generator=g) * 0.1).to(dtype).cuda()
    b0 = torch.randn((classes,), generator=g).to(dtype).cuda()
    t = torch.randint(0, classes, (rows + 5,), generator=g).cuda()
    t[:5] = -100
    for softcap, biased in ((None, False), (20.0, True)):
        e, c, bias = (x.clone().requires_grad_(True) for x in (e0, c0, b0))
        nll = linear_cross_entropy(e, c, t, bias=bias if biased else None, softcap=softcap, reduction="none", impl="cce_exact")
        up = torch.rand(nll.shape, generator=torch.Generator().manual_seed(1)).cuda() + 0.5
        nll.backward(up.to(nll.dtype))
        z = e0.double() @ c0.double().T + (b0.double() if biased else 0.0)
        x = softcap * torch.tanh(z / softcap) if softcap else z
        dz = torch.softmax(x, 1)
        dz[5:].scatter_add_(1, t[5:, None], -torch.ones((rows, 1), dtype=torch.float64, device="cuda"))
        if softcap:
            dz *= 1 - (x / softcap) ** 2
        dz *= up.to(nll.dtype).double()[:, None]
        dz[:5] = 0.0
        # the bounds of test_backward_dense_cuts_long_reductions: dz and the results are rounded to 8 (11) bits once each
        for got, want in ((e.grad, dz @ c0.double()), (c.grad, dz.T @ e0.double())):
            scale = want.abs().amax(dim=1, keepdim=True)
            assert ((got.double() - want).abs() <= 1e-2 * scale + 1e-2 * want.abs() + 1e-6).all()
            assert (got.double() - want).norm() <= 6e-3 * want.norm()
        if biased:  # terms of 8 significant bits: half a unit in the last place is up to 2^-8 of each, and of their sum once more;
            # below 2^-14 a fp16 term is off by up to 2^-25 whatever its size
            want = dz.sum(0)
            tiny = (rows + 1) * 2.0**-25 if dtype == torch.float16 else 0.0
            assert ((bias.grad.double() - want).abs() <= 2.0**-8 * (dz.abs().sum(0) * 1.01 + want.abs()) + tiny + 1e-6).all()
