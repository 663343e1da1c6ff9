"""The whole-box forward kernel where its table, pieces and transposition can go wrong.

Against the direct kernels on the same inputs (their own oracle tests pin them): boxes of one
piece and of many (offsets of many voxels), boxes reaching past every face of the volume, unit
axes, partial tiles, windows of 1 to 160 taps (one to five taps per lane, the last partly
filled).  fp32: both sum the same products in fp32, the tiled weights in fixed point of 2^-30
per corner (at most 8 * 160 corners per output, |V| < 6): 1e-5.  bf16: the weights are rounded
to bf16 (2^-9) and so is the output: 2e-2 of the largest value.
"""

import pytest
import torch

pytestmark = pytest.mark.gpu

CASES = [
    # T, H, W, heads, window, offset std in voxels
    (1, 4, 4, 1, (1, 1, 1), 0.0),
    (7, 12, 12, 2, (3, 7, 7), 0.5),    # the usual box: one piece
    (9, 13, 21, 1, (3, 7, 7), 6.0),    # cut along several axes
    (5, 30, 33, 1, (3, 7, 7), 30.0),   # clamped onto every face, most of the volume
    (40, 5, 1, 1, (5, 7, 4), 9.0),     # a unit axis, a long one, 140 taps
    (1, 3, 70, 2, (1, 4, 40), 2.0),    # 160 taps, wide and flat
    (6, 1, 9, 1, (3, 1, 11), 1.0),     # 33 taps
    (2, 15, 18, 1, (3, 7, 7), 3.0),    # two frames: every box ends at the volume
    (1, 45, 60, 1, (3, 7, 7), 12.0),   # one frame, cut
    (14, 1, 90, 1, (3, 1, 7), 30.0),   # one row, cut
]


def _inputs(case, hd, dt):
    T, H, W, nh, win, std = case
    g = torch.Generator().manual_seed(5)
    N, K = T * H * W, win[0] * win[1] * win[2]
    q, k, v = (torch.randn(1, N, nh * hd, generator=g) for _ in range(3))
    # slot 0 moves x by W / 2 / max(T - 1, 1) voxels a unit, slot 2 z by T / 2 / max(W - 1, 1)
    unit = torch.tensor([max(T - 1, 1) / W, max(H - 1, 1) / H, max(W - 1, 1) / T]) * 2
    off = (torch.randn(1, N, nh * K, 3, generator=g) * std * unit).view(1, N, -1)
    return [t.to(dt).cuda() for t in (q, k, v, off)]


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("hd", [32, 64, 96, 128])
@pytest.mark.parametrize("case", CASES)
def test_box_forward_matches_direct(case, hd, dt):
    from megaslide_amd import dsa3d_core

    print(f"[box forward] {case} {hd} {dt}", flush=True)
    T, H, W, nh, win, _ = case
    ins = _inputs(case, hd, dt)
    with torch.no_grad():
        a, la = dsa3d_core(*ins, (T, H, W), nh, win, algo="tiled", return_lse=True)
        b, lb = dsa3d_core(*ins, (T, H, W), nh, win, algo="direct", return_lse=True)
    tol = 1e-5 if dt == torch.float32 else 2e-2
    assert (a.float() - b.float()).abs().max() <= tol * b.float().abs().max()
    assert (la - lb).abs().max() < 1e-4


@pytest.mark.parametrize("hd,dt", [(32, torch.bfloat16), (64, torch.bfloat16),
                                   (96, torch.bfloat16), (128, torch.bfloat16),
                                   (40, torch.bfloat16), (80, torch.float32)])
def test_infinite_value_reaches_who_samples_it(hd, dt):
    """A V row with one infinite element spoils that channel of the queries that sample it, and
    nothing else: as in the direct kernels, which gather what each query samples."""
    from megaslide_amd import dsa3d_core

    case = (5, 9, 11, 1, (3, 7, 7), 0.5)
    q, k, v, off = _inputs(case, hd, dt)
    v[0, (2 * 9 + 4) * 11 + 5, hd - 3] = float("inf")
    with torch.no_grad():
        out = dsa3d_core(q, k, v, off, case[:3], 1)
        ref = dsa3d_core(q, k, v, off, case[:3], 1, algo="direct")
    fin = torch.isfinite(ref)
    assert torch.equal(torch.isfinite(out), fin) and 0 < (~fin).sum() < ref.shape[1]
    assert (out[fin].float() - ref[fin].float()).abs().max() < 2e-2


def _grads(ins, extra, shape, nh, win, **kw):
    from megaslide_amd import dsa3d_core

    ts = [t.detach().clone().requires_grad_(True) for t in ins]
    es = [t.detach().clone().requires_grad_(True) for t in extra]
    ek, ev = es or (None, None)
    out = dsa3d_core(*ts, shape, nh, win, extra_k=ek, extra_v=ev, **kw)
    g = torch.Generator(device="cuda").manual_seed(8)
    dout = torch.randn(out.shape, generator=g, device="cuda").to(out.dtype)
    return [out.detach(), *torch.autograd.grad(out, ts + es, dout)]


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("hd", [8, 24, 40, 56, 72, 88, 104, 120])
@pytest.mark.parametrize("G,p", [(0, 0.0), (5, 0.0), (40, 0.3)])
def test_other_head_sizes_match_direct(hd, G, p, dt):
    """Multiples of 8 between the compiled head sizes (padded copies) against the direct kernels:
    both compute in fp32 (2e-5 of the largest value over sums of ~1,000 terms) and round bf16
    results once (2^-8)."""
    print(f"[padded head size] {hd} {G} {p} {dt}", flush=True)
    T, H, W, nh, win, _ = case = (4, 9, 10, 3, (3, 5, 5), 1.0)
    ins = _inputs(case, hd, dt)
    g = torch.Generator(device="cuda").manual_seed(6)
    extra = [torch.randn(1, G, nh * hd, generator=g, device="cuda").to(dt) for _ in range(2 * (G > 0))]
    kw = dict(dropout_p=p, dropout_seed=11)
    a = _grads(ins, extra, (T, H, W), nh, win, **kw)
    b = _grads(ins, extra, (T, H, W), nh, win, algo="direct", **kw)
    for x, y in zip(a, b):
        tol = 2e-5 if dt == torch.float32 else 2.0 ** -8
        assert (x.float() - y.float()).abs().max() <= tol * y.float().abs().max()


@pytest.mark.parametrize("hd,dt", [(32, torch.float32), (64, torch.bfloat16), (96, torch.float32),
                                   (128, torch.bfloat16)])
@pytest.mark.parametrize("p", [0.0, 0.4])
@pytest.mark.parametrize("case", CASES)
def test_box_backward_matches_direct(case, p, hd, dt):
    """The first backward kernel's tables, pieces and records: every gradient against the direct
    kernels (fp32: fixed-point tables of 2^-30 per corner; bf16: operands of 2^-9).  A one-tap
    window's dq and dk vanish identically: 1e-4 of the unit-variance inputs."""
    print(f"[box backward] {case} {hd} {dt} {p}", flush=True)
    T, H, W, nh, win, _ = case
    ins = _inputs(case, hd, dt)
    kw = dict(dropout_p=p, dropout_seed=3)
    a = _grads(ins, [], (T, H, W), nh, win, algo="tiled", **kw)
    b = _grads(ins, [], (T, H, W), nh, win, algo="direct", **kw)
    for x, y in zip(a, b):
        tol = 2e-5 if dt == torch.float32 else 2e-2
        bound = max(tol * y.float().abs().max().item(), 1e-4)
        assert (x.float() - y.float()).abs().max().item() <= bound


def test_more_workgroups_than_one_launch_axis_takes():
    """8.5 million tiles of one query: more workgroups of 512 threads than an axis of a launch
    holds.  One tap per query: the output is that tap's V sample, and dq, dk vanish."""
    from megaslide_amd import dsa3d_core

    B, T, nh, hd = 32, 4096, 65, 32
    g = torch.Generator(device="cuda").manual_seed(9)
    q, v, dout = (torch.randn(B, T, nh * hd, generator=g, device="cuda", dtype=torch.bfloat16)
                  for _ in range(3))
    off = torch.zeros(B, T, nh * 3, device="cuda", dtype=torch.bfloat16)
    res = []
    for algo in ("tiled", "direct"):
        vv = v.detach().requires_grad_(True)
        out = dsa3d_core(q, q, vv, off, (T, 1, 1), nh, (1, 1, 1), algo=algo)
        res.append((out.detach(), *torch.autograd.grad(out, vv, dout)))
    for x, y in zip(*res):
        assert (x - y).abs().max() <= 2e-2 * y.abs().max()


def test_padded_backward_does_without_its_copies(monkeypatch):
    """Where the padded copies' workspace does not fit the device, the backward takes the kernels
    that need none (the direct ones: equal up to the atomics' order, 2e-5 as above)."""
    case = (4, 9, 10, 3, (3, 5, 5), 1.0)
    ins = _inputs(case, 40, torch.float32)
    ref = _grads(ins, [], case[:3], 3, case[4], algo="direct")
    empty, failed = torch.empty, []

    def scarce(*args, **kw):
        if kw.get("dtype") == torch.uint8 and not failed:
            failed.append(args)
            raise torch.OutOfMemoryError("no room")
        return empty(*args, **kw)

    monkeypatch.setattr(torch, "empty", scarce)
    got = _grads(ins, [], case[:3], 3, case[4])
    assert failed
    for x, y in zip(got, ref):
        assert (x - y).abs().max() <= 2e-5 * y.abs().max()


@pytest.mark.parametrize("hd", [32, 64, 96, 128])
@pytest.mark.parametrize("case", [
    # units (pairs of 4 x 4 columns of a head) on both sides of the lines of 256 CUs
    (6, 4, 4, 102, (3, 5, 5), 0.5),
    (6, 4, 4, 103, (3, 5, 5), 0.5),
    (6, 4, 4, 128, (3, 5, 5), 0.5),
    (6, 4, 4, 129, (3, 5, 5), 0.5),
    # the streaming kernel's walks: its ring of frames, wide boxes, more than 256 frames
    (40, 4, 4, 136, (3, 7, 7), 0.5),
    (20, 8, 24, 24, (3, 3, 3), 4.0),
    (5, 13, 21, 12, (3, 7, 7), 1.5),
    (300, 4, 4, 130, (1, 3, 3), 0.5),
])
def test_both_second_backward_kernels_match_direct(case, hd):
    """bf16 gradients through the tile kernel (few columns) and the column-streaming one (many):
    operands of 2^-9 as above."""
    print(f"[second backward kernel] {case} {hd}", flush=True)
    T, H, W, nh, win, _ = case
    ins = _inputs(case, hd, torch.bfloat16)
    a = _grads(ins, [], (T, H, W), nh, win, algo="tiled")
    b = _grads(ins, [], (T, H, W), nh, win, algo="direct")
    for x, y in zip(a, b):
        assert (x.float() - y.float()).abs().max() <= 2e-2 * y.float().abs().max()


def test_cut_boxes_round_each_weight_once():
    """bf16: the weight of a voxel that two pieces of a cut box share is rounded once, as every
    other.  With q = 0 every tap weighs 1 / K, and a channel of V that is 1 at one voxel leaves
    that voxel's weight as the output: the direct kernels' fp32 weight, rounded.  A fixed-point
    weight is below that by less than one unit of 2^-30 a tap and corner: ~1e-8 of a bf16 step
    of at least 2^-17 (weights from 2^-9), so that the rounding differs for under 1 %."""
    from megaslide_amd import dsa3d_core

    T, H, W, nh, win, _ = case = (12, 16, 16, 1, (3, 7, 7), 1.3)
    hd, N = 128, 12 * 16 * 16
    q, _, _, off = _inputs(case, hd, torch.bfloat16)
    q.zero_()
    differ = total = 0
    for v0 in range(0, N, hd):
        v = torch.zeros(1, N, hd, device="cuda")
        n = min(hd, N - v0)
        v[0, torch.arange(v0, v0 + n), torch.arange(n)] = 1.0
        with torch.no_grad():
            out = dsa3d_core(q, q, v.bfloat16(), off, (T, H, W), nh, win)
            ref = dsa3d_core(q.float(), q.float(), v, off.float(), (T, H, W), nh, win,
                             algo="direct")
        big = ref >= 2.0 ** -9
        differ += (out != ref.bfloat16())[big].sum().item()
        total += big.sum().item()
    print(f"[cut boxes] {differ} of {total} weights rounded otherwise", flush=True)
    assert total > 10000 and differ < 0.01 * total


@pytest.mark.parametrize("shape", [(1, 1, 16384), (1, 2, 16390), (2, 16390, 1)])
def test_axes_beyond_the_tap_records(shape):
    """bf16 gradients on both sides of the longest axis that the column-streaming kernel's tap
    records address (enough columns for it in each): operands of 2^-9 as above."""
    print(f"[long axis] {shape}", flush=True)
    case = (*shape, 1, (1, 3, 5) if shape[2] > 1 else (2, 5, 1), 1.0)
    ins = _inputs(case, 32, torch.bfloat16)
    a = _grads(ins, [], shape, 1, case[4], algo="tiled")
    b = _grads(ins, [], shape, 1, case[4], algo="direct")
    for x, y in zip(a, b):
        assert (x.float() - y.float()).abs().max() <= 2e-2 * y.float().abs().max()


@pytest.mark.parametrize("hd,G", [(40, 0), (72, 0), (80, 60), (104, 0), (112, 160), (120, 60)])
def test_other_head_sizes_as_precise_as_direct(hd, G):
    """fp32 at padded head sizes: no result further from 64 bits than the direct kernels' (a
    tenth for the spread of such errors over inputs), the reference being the same direct
    kernels' inputs through the operator's definition in float64."""
    import perf.cases as cases

    case = cases._core("", 6, 12, 14, 3, hd, "fp32", 1, (3, 7, 7), 0.5, 0.0, True, G)
    exact = cases.exact(case, 4)
    q, k, v, off, ek, ev, dout = cases._core_inputs(case, 4)
    ins = [t.requires_grad_(True) for t in (q, k, v, off, ek, ev) if t is not None]

    def errors(**kw):
        from megaslide_amd import dsa3d_core
        out = dsa3d_core(q, k, v, off, (6, 12, 14), 3, extra_k=ek, extra_v=ev, **kw)
        res = (out.detach(), *torch.autograd.grad(out, ins, dout))
        return [((a.double() - b).norm() / b.norm()).item() for a, b in zip(res, exact)]

    padded, direct = errors(), errors(algo="direct")
    print(f"[precision] {hd} {G} {padded} {direct}", flush=True)
    assert all(p <= 1.1 * d for p, d in zip(padded, direct))


@pytest.mark.parametrize("what", ["k", "lowest k", "v and k", "huge v", "offsets"])
@pytest.mark.parametrize("hd,dt", [(40, torch.float32), (80, torch.bfloat16),
                                   (104, torch.float32), (24, torch.bfloat16)])
@pytest.mark.parametrize("std", [0.5, 6.0])  # boxes of one piece, of several
def test_other_head_sizes_sample_non_finite_values(what, hd, dt, std):
    """Padded head sizes where inputs are infinite or at the type's limit: the outputs that are
    finite in the oracle are so here, and equal (products in fp32, bf16 results of 2^-9).  An
    infinite score of one sign leaves a query its other taps."""
    from megaslide_amd import dsa3d_core
    from oracle.dsa3d_ref import dsa3d_core_ref

    case = (6, 9, 13, 2, (3, 7, 7), std)
    shape = case[:3]
    q, k, v, off = (t.cpu() for t in _inputs(case, hd, dt))
    g = torch.Generator().manual_seed(12)
    if "k" in what:
        worst = torch.finfo(dt).min if "lowest" in what else float("-inf")
        k[0, 300, 3] = worst
        k[0, 411, hd + 2] = -worst
    if what == "v and k":
        v[0, 305, 1] = float("nan")
        v[0, 400, hd + 1] = float("inf")
    if what == "huge v":
        v *= 1e30
    if what == "offsets":
        at = torch.randint(off.numel(), (200,), generator=g)
        off.view(-1)[at] = float("inf")
        off.view(-1)[at[:100]] = float("-inf")
    ref = dsa3d_core_ref(*(t.float() for t in (q, k, v, off)), shape, 2, case[4], 1.0).double()
    with torch.no_grad():
        out = dsa3d_core(*(t.cuda() for t in (q, k, v, off)), shape, 2).double().cpu()
    fin = torch.isfinite(ref)
    print(f"[non-finite, padded] {what} {hd} {dt} {std}: {(~fin).sum()} "
          f"{(torch.isfinite(out) != fin).sum()}", flush=True)
    if what == "lowest k":  # a score that overflows before its scaling may stay finite here
        assert torch.isfinite(out)[fin].all()
    else:
        assert torch.equal(torch.isfinite(out), fin)
    assert fin.sum() > 0.3 * fin.numel()
    tol = 1e-4 if dt == torch.float32 else 1e-2
    assert (out - ref)[fin].abs().max() <= tol * ref[fin].abs().max()


@pytest.mark.parametrize("what", ["k", "v", "dout", "dlse", "offsets", "huge"])
@pytest.mark.parametrize("hd,dt,p,G", [(40, torch.float32, 0.0, 0), (80, torch.bfloat16, 0.3, 20),
                                       (104, torch.float32, 0.2, 5), (24, torch.bfloat16, 0.0, 0)])
def test_other_head_sizes_differentiate_non_finite_values_as_direct(what, hd, dt, p, G):
    """Padded head sizes where an input or an incoming gradient is not finite, or at the type's
    limit: the gradients are the direct kernels', which these calls took before, finite where
    theirs are (equal up to the order of fp32 atomics, 2e-5, and one rounding to bf16)."""
    from megaslide_amd import dsa3d_core

    print(f"[non-finite gradients, padded] {what} {hd} {dt} {p} {G}", flush=True)
    case = (4, 9, 13, 3, (3, 5, 5), 0.8)
    shape = case[:3]
    ins = _inputs(case, hd, dt)
    g = torch.Generator().manual_seed(12)
    if G:
        ins += [torch.randn(1, G, 3 * hd, generator=g).to(dt).cuda() for _ in range(2)]
    dout = torch.randn(1, 4 * 9 * 13, 3 * hd, generator=g).to(dt).cuda()
    dlse = torch.randn(1, 4 * 9 * 13, 3, generator=g).cuda()
    if what == "k":
        ins[1][0, 200, 3] = float("inf")
    if what == "v":
        ins[2][0, 205, hd + 1] = float("nan")
    if what == "dout":
        dout[0, 77, 2 * hd] = float("nan")
        dout[0, 300, 5] = float("inf")
    if what == "dlse":
        dlse[0, 100, 1] = float("inf")
    if what == "offsets":
        at = torch.randint(ins[3].numel(), (300,), generator=g)
        for i, x in enumerate(("inf", "-inf", "nan")):
            ins[3].view(-1)[at[i::3].cuda()] = float(x)
    if what == "huge":
        ins[2] *= 1e30
        dout *= 1e-30

    def grads(**kw):
        ts = [t.detach().clone().requires_grad_(True) for t in ins]
        out, lse = dsa3d_core(*ts[:4], shape, 3, case[4], extra_k=ts[4] if G else None,
                              extra_v=ts[5] if G else None, dropout_p=p, dropout_seed=7,
                              return_lse=True, offset_scale=0.7, **kw)
        return torch.autograd.grad([out, lse], ts, [dout, dlse])

    some = 0
    for i, (x, y) in enumerate(zip(grads(), grads(algo="direct"))):
        x, y = x.double(), y.double()
        fin = torch.isfinite(y)
        if what == "k":  # (a first tap of -inf makes the direct forward's running sum NaN)
            assert torch.isfinite(x)[fin].all(), f"gradient {i}"
        else:
            assert torch.equal(torch.isfinite(x), fin), f"gradient {i}"
        some += fin.sum().item()
        if fin.any():
            tol = 2e-5 if dt == torch.float32 else 2.0 ** -8
            assert (x - y)[fin].abs().max() <= tol * y[fin].abs().max(), f"gradient {i}"
    assert some > 0.5 * sum(t.numel() for t in ins)


@pytest.mark.parametrize("dt,p,G", [(torch.float32, 0.2, 7), (torch.bfloat16, 0.0, 0)])
def test_padded_backward_over_groups_of_heads(dt, p, G):
    """More heads than the padded copies' workspace takes at once: the groups' gradients against
    the direct kernels' (tolerances as above; dropout's counters run over all heads)."""
    print(f"[groups of heads] {dt} {p} {G}", flush=True)
    case = (16, 24, 26, 19, (3, 7, 7), 0.5)
    ins = _inputs(case, 40, dt)
    g = torch.Generator(device="cuda").manual_seed(6)
    extra = [torch.randn(1, G, 19 * 40, generator=g, device="cuda").to(dt) for _ in range(2 * (G > 0))]
    kw = dict(dropout_p=p, dropout_seed=11)
    a = _grads(ins, extra, case[:3], 19, case[4], **kw)
    b = _grads(ins, extra, case[:3], 19, case[4], algo="direct", **kw)
    for x, y in zip(a, b):
        tol = 3e-5 if dt == torch.float32 else 2.0 ** -8
        assert (x.float() - y.float()).abs().max() <= tol * y.float().abs().max()


@pytest.mark.parametrize("hd,dt,inf", [
    *((hd, dt, inf) for inf in (False, True)
      for hd, dt in ((32, torch.bfloat16), (96, torch.bfloat16), (128, torch.bfloat16),
                     (72, torch.float32))),
    # (whole-head fp32 products have no plain-arithmetic pass)
    (64, torch.float32, False), (128, torch.float32, False)])
@pytest.mark.parametrize("G,p", [(20, 0.0), (128, 0.3), (200, 0.0), (0, 0.3)])
def test_cut_boxes_with_extra_keys_and_dropout(G, p, hd, dt, inf):
    """Boxes of several pieces together with extra keys and dropout, and with an infinite value in
    a V row (and one in an extra value: its weight reaches every query), which sends tiles to the
    plain-arithmetic pass: against the direct kernels, tolerances as above."""
    from megaslide_amd import dsa3d_core

    case = (9, 13, 21, 2, (3, 7, 7), 6.0)
    q, k, v, off = _inputs(case, hd, dt)
    g = torch.Generator().manual_seed(4)
    ek = ev = None
    if G:
        ek, ev = (torch.randn(1, G, 2 * hd, generator=g).to(dt).cuda() for _ in range(2))
    if inf:
        v[0, 1000, hd - 3] = float("inf")
        v[0, 1500, hd + 5] = float("-inf")
        if G:
            ev[0, G - 1, 2] = float("inf")
    kw = dict(extra_k=ek, extra_v=ev, dropout_p=p, dropout_seed=5)
    with torch.no_grad():
        out = dsa3d_core(q, k, v, off, case[:3], 2, **kw).double()
        ref = dsa3d_core(q, k, v, off, case[:3], 2, algo="direct", **kw).double()
    fin = torch.isfinite(ref)
    assert torch.equal(torch.isfinite(out), fin) and fin.all() == (not inf)
    tol = 1e-5 if dt == torch.float32 else 2e-2
    assert (out - ref)[fin].abs().max() <= tol * ref[fin].abs().max()


@pytest.mark.parametrize("hd,dt", [(64, torch.bfloat16), (96, torch.float32), (40, torch.bfloat16),
                                   (72, torch.float32)])
@pytest.mark.parametrize("std", [0.5, 6.0])
def test_strides_of_their_own(hd, dt, std):
    """q, k and v (and their gradients) with three different token strides, through the C entry
    points, equal the contiguous call bit for bit in the forward and up to the order of fp32
    atomics (2e-5; bf16 one rounding) in the backward."""
    import ctypes
    from megaslide_amd import _lib, dsa3d_core

    lib = _lib.load()
    case = (7, 9, 14, 3, (3, 5, 5), std)
    T, H, W, nh, win, _ = case
    ins = _inputs(case, hd, dt)
    N, D = T * H * W, nh * hd
    g = torch.Generator(device="cuda").manual_seed(8)
    dout = torch.randn(1, N, D, generator=g, device="cuda").to(dt)
    ts = [t.detach().clone().requires_grad_(True) for t in ins]
    ref, rlse = dsa3d_core(*ts, case[:3], nh, win, return_lse=True)
    grads = torch.autograd.grad(ref, ts, dout)

    strides = (D + 8, 2 * D, 3 * D + 16)
    wide = [torch.full((N, s), 7.0, dtype=dt, device="cuda") for s in strides]
    outs = [torch.full((N, s), 7.0, dtype=dt, device="cuda") for s in strides]
    for w, t in zip(wide, ins):
        w[:, :D] = t[0]
    desc = _lib.DsaDesc(1, T, H, W, nh, hd, *win, _lib.dtype_code(dt), *strides, 1.0, hd ** -0.5)
    out, lse = torch.empty_like(ref), torch.empty_like(rlse)
    stream = _lib.stream_handle(out.device)
    _lib.check(lib.msd_dsa3d_fwd(ctypes.byref(desc), *(w.data_ptr() for w in wide),
                                 ins[3].data_ptr(), None, None, out.data_ptr(), lse.data_ptr(),
                                 stream), "fwd")
    assert torch.equal(out, ref) and torch.equal(lse, rlse)
    size = lib.msd_dsa3d_bwd_best_workspace_size(ctypes.byref(desc))
    ws = torch.empty(size, dtype=torch.uint8, device="cuda")
    doff = torch.empty_like(ins[3])
    _lib.check(lib.msd_dsa3d_bwd(ctypes.byref(desc), *(w.data_ptr() for w in wide),
                                 ins[3].data_ptr(), None, None, out.data_ptr(), dout.data_ptr(),
                                 lse.data_ptr(), None, *(o.data_ptr() for o in outs),
                                 doff.data_ptr(), None, None, ws.data_ptr(), size, stream), "bwd")
    tol = 2e-5 if dt == torch.float32 else 2.0 ** -7
    for o, x in zip([w[:, :D] for w in outs] + [doff[0]], grads):
        assert (o.float() - x[0].float()).abs().max() <= tol * x.float().abs().max()
    for o in outs:  # nothing between the rows
        assert (o[:, D:] == 7.0).all()
