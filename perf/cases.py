"""Performance cases: what a program that uses this package has it do.

Each case is one pass through a public entry point (``dsa3d_core``,
``dwconv3d``, ``DiTBlock``) at a size from this repository's benchmark,
configurations or tests, or a generic one of the same range.  ``listed`` gives
the fixed cases, ``draw`` another of the same ranges; ``prepare`` makes what a
program holds before the call, ``run`` is the call, ``exact`` the same outputs
from plain torch in float64.
"""

from __future__ import annotations

import math

import torch
import torch.nn.functional as F

import megaslide_amd as ms

_DT = {"bf16": torch.bfloat16, "fp32": torch.float32}


def _core(name, T, H, W, heads, hd, dtype="bf16", B=1, window=(3, 7, 7), std=0.5, bias=0.0,
          train=True, extra=0):
    kt, kh, kw = window
    return {"name": name, "kind": "core", "B": B, "T": T, "H": H, "W": W, "heads": heads,
            "head_dim": hd, "kt": kt, "kh": kh, "kw": kw, "dtype": dtype, "std": std,
            "bias": bias, "train": train, "extra": extra}


def _conv(name, T, H, W, C, window, gelu, dtype="bf16", B=1):
    kt, kh, kw = window
    return {"name": name, "kind": "conv", "B": B, "T": T, "H": H, "W": W, "C": C, "kt": kt,
            "kh": kh, "kw": kw, "dtype": dtype, "gelu": gelu}


def listed():
    return [
        # one layer of a small fp32 model at inference: launches and latency count
        _core("core_fwd_tiny_fp32", 8, 16, 16, 4, 64, dtype="fp32", std=0.3, train=False),
        # one training layer of a 16-layer, 1,024-wide model at 2,048 tokens
        _core("core_train_small_bf16", 32, 8, 8, 16, 64, window=(3, 5, 5)),
        # fp32 training with offsets that often leave the volume, batch of two
        _core("core_train_fp32", 16, 32, 32, 8, 64, dtype="fp32", B=2, std=1.5),
        # a 256-frame clip at inference, and the same layer in training
        _core("core_fwd_long_bf16", 64, 32, 32, 16, 64, train=False),
        _core("core_train_long_bf16", 64, 32, 32, 16, 64),
        # a grid that no tile divides, trained offsets biased by up to 4 voxels per tap
        _core("core_train_ragged_bf16", 13, 45, 80, 16, 96, std=0.3, bias=4.0),
        # the largest layer: 131,072 tokens, 3,072 wide
        _core("core_train_large_bf16", 32, 64, 64, 24, 128, std=0.5),
        # hybrid attention: 128 register tokens that every query also attends to
        _core("core_train_registers_bf16", 16, 32, 32, 16, 64, extra=128),
        # a width of 1,280 over 16 heads: a head size that is no multiple of 32
        _core("core_train_hd80_bf16", 16, 16, 16, 16, 80, window=(3, 5, 5)),
        # the module's depthwise term in training, long clip
        _conv("dwconv7_train_bf16", 64, 32, 32, 1024, (3, 7, 7), False),
        # the offset net's depthwise conv and GELU in training, ragged grid
        _conv("dwconv3_gelu_train_bf16", 13, 45, 80, 1536, (3, 3, 3), True),
        # a whole transformer block's training step, fp32 as the module runs by default
        {"name": "block_train_fp32", "kind": "block", "B": 1, "T": 16, "H": 16, "W": 16,
         "heads": 8, "head_dim": 64, "kt": 3, "kh": 5, "kw": 5, "dtype": "fp32", "std": 0.5},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: an attention core in four of five, else a depthwise conv."""
    if rng.random() < 0.2:
        window = rng.choice([(3, 7, 7), (3, 5, 5), (3, 3, 3)])
        dtype = "bf16" if rng.random() < 0.7 else "fp32"
        while True:
            T, H, W = _log_int(rng, 2, 64), _log_int(rng, 6, 64), _log_int(rng, 6, 96)
            C = 8 * _log_int(rng, 8, 192)
            if 2 ** 17 <= T * H * W * C <= 2 ** 26:
                break
        c = _conv("", T, H, W, C, window, window == (3, 3, 3), dtype)
    else:
        dtype = "bf16" if rng.random() < 0.7 else "fp32"
        tiled = rng.random() < 0.8
        # head sizes of common widths; other multiples of 8 at sizes up to 2,048 tokens
        hd = rng.choice([32, 64, 64, 96, 128]) if tiled else rng.choice([24, 40, 48, 72, 80, 112])
        cap = 2 ** 25 if tiled else 2 ** 20
        if dtype == "fp32":
            cap //= 4
        while True:
            T, H, W = _log_int(rng, 2, 64), _log_int(rng, 6, 64), _log_int(rng, 6, 96)
            heads = _log_int(rng, 2, 24)
            if min(2 ** 17, cap // 8) <= T * H * W * heads * hd <= cap:
                break
        window = rng.choice([(3, 7, 7), (3, 7, 7), (3, 5, 5), (3, 3, 3)])
        std, bias = rng.choice([(0.3, 0.0), (0.5, 0.0), (1.5, 0.0), (0.3, 4.0)])
        extra = rng.choice([16, 77, 128]) if tiled and rng.random() < 0.15 else 0
        c = _core("", T, H, W, heads, hd, dtype, 1, window, std, bias, rng.random() < 0.75, extra)
    del c["name"]
    return c


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _randn(g, dt, *shape, std=1.0):
    return torch.randn(*shape, generator=g, device="cuda").mul_(std).to(dt)


def _window(c):
    return (c["kt"], c["kh"], c["kw"])


def _grid(c):
    return (c["T"], c["H"], c["W"])


def _sizes(c):
    N = c["T"] * c["H"] * c["W"]
    D = c["heads"] * c["head_dim"]
    K = c["kt"] * c["kh"] * c["kw"]
    return c["B"], N, D, K


def _core_inputs(c, seed):
    """q, k, v as unit-variance projections; offsets ~ N(0, std) around a bias per (head, tap)."""
    g, dt = _gen(seed), _DT[c["dtype"]]
    B, N, D, K = _sizes(c)
    q, k, v = (_randn(g, dt, B, N, D) for _ in range(3))
    C = c["heads"] * K * 3
    off = torch.randn(B, N, C, generator=g, device="cuda", dtype=torch.float32).mul_(c["std"])
    if c["bias"] > 0:
        off += (torch.rand(C, generator=g, device="cuda") * 2 - 1) * c["bias"]
    off = off.to(dt)
    dout = _randn(g, dt, B, N, D) if c["train"] else None
    ek = _randn(g, dt, B, c["extra"], D) if c["extra"] else None
    ev = _randn(g, dt, B, c["extra"], D) if c["extra"] else None
    return q, k, v, off, ek, ev, dout


def _conv_inputs(c, seed):
    g, dt = _gen(seed), _DT[c["dtype"]]
    B, N, C = c["B"], c["T"] * c["H"] * c["W"], c["C"]
    x, dy = _randn(g, dt, B, N, C), _randn(g, dt, B, N, C)
    w = _randn(g, dt, C, 1, *_window(c), std=1.0 / math.sqrt(math.prod(_window(c))))
    b = _randn(g, dt, C, std=0.02)
    return x, w, b, dy


class _BlockConfig:
    def __init__(self, c):
        self.hidden_size = c["heads"] * c["head_dim"]
        self.num_heads = c["heads"]
        self.dsa_kernel_size = _window(c)
        self.offset_scale = 1.0
        self.dropout = 0.0
        self.mlp_hidden_size = 4 * self.hidden_size
        self.use_text_conditioning = False


def _block_params(c, g):
    """Parameter values by name, Xavier-scaled, offsets of about std voxels."""
    _, _, D, K = _sizes(c)
    C = c["heads"] * K * 3

    def r(*shape, std):
        return torch.randn(*shape, generator=g, device="cuda") * std

    lin = 1.0 / math.sqrt(D)
    p = {}
    for n in ("norm1", "norm2"):
        p[n + ".weight"], p[n + ".bias"] = 1.0 + r(D, std=0.02), r(D, std=0.02)
    for n in ("q_proj", "k_proj", "v_proj", "out_proj"):
        p[f"attn.{n}.weight"], p[f"attn.{n}.bias"] = r(D, D, std=lin), r(D, std=0.02)
    p["attn.dw_conv.weight"] = r(D, 1, *_window(c), std=1.0 / math.sqrt(K))
    p["attn.dw_conv.bias"] = r(D, std=0.02)
    p["attn.offset_net.0.weight"] = r(D, 1, 3, 3, 3, std=0.2)
    p["attn.offset_net.0.bias"] = r(D, std=0.02)
    p["attn.offset_net.2.weight"] = r(C, D, 1, 1, 1, std=lin * c["std"])
    p["attn.offset_net.2.bias"] = r(C, std=c["std"])
    p["mlp.fc1.weight"], p["mlp.fc1.bias"] = r(4 * D, D, std=lin), r(4 * D, std=0.02)
    p["mlp.fc2.weight"], p["mlp.fc2.bias"] = r(D, 4 * D, std=lin / 2), r(D, std=0.02)
    return p


def _block_inputs(c, seed):
    g, dt = _gen(seed), _DT[c["dtype"]]
    B, N, D, _ = _sizes(c)
    params = _block_params(c, g)
    return params, _randn(g, dt, B, N, D), _randn(g, dt, B, N, D)


def prepare(case, seed):
    if case["kind"] == "core":
        q, k, v, off, ek, ev, dout = _core_inputs(case, seed)
        if case["train"]:
            for t in (q, k, v, off, ek, ev):
                if t is not None:
                    t.requires_grad_(True)
        return {"case": case, "q": q, "k": k, "v": v, "off": off, "ek": ek, "ev": ev,
                "dout": dout}
    if case["kind"] == "conv":
        x, w, b, dy = _conv_inputs(case, seed)
        for t in (x, w, b):
            t.requires_grad_(True)
        return {"case": case, "x": x, "w": w, "b": b, "dy": dy}
    params, x, dy = _block_inputs(case, seed)
    block = ms.DiTBlock(_BlockConfig(case))
    block = block.to(device="cuda", dtype=_DT[case["dtype"]])
    with torch.no_grad():
        for name, p in block.named_parameters():
            p.copy_(params[name])
    return {"case": case, "block": block, "params": dict(block.named_parameters()),
            "x": x.requires_grad_(True), "dy": dy}


def run(state):
    c = state["case"]
    if c["kind"] == "core":
        ins = [state["q"], state["k"], state["v"], state["off"]]
        if c["extra"]:
            ins += [state["ek"], state["ev"]]
        if not c["train"]:
            with torch.no_grad():
                return ms.dsa3d_core(*ins[:4], _grid(c), c["heads"], _window(c),
                                     extra_k=state["ek"], extra_v=state["ev"])
        out = ms.dsa3d_core(*ins[:4], _grid(c), c["heads"], _window(c), extra_k=state["ek"],
                            extra_v=state["ev"])
        return (out.detach(),) + torch.autograd.grad(out, ins, state["dout"])
    if c["kind"] == "conv":
        ins = (state["x"], state["w"], state["b"])
        y = ms.dwconv3d(*ins, _grid(c), act="gelu" if c["gelu"] else None)
        return (y.detach(),) + torch.autograd.grad(y, ins, state["dy"])
    y = state["block"](state["x"], _grid(c))
    grads = torch.autograd.grad(y, [state["x"], *state["params"].values()], state["dy"])
    # a common shift of every key leaves the softmax as it is, so this one gradient is zero
    # up to rounding and its value is noise
    named = dict(zip(state["params"], grads[1:]))
    named["attn.k_proj.bias"] = None
    return (y.detach(), grads[0], *(g for g in named.values() if g is not None))


def work(case):
    """Bytes: each input read once, each output written once.  Operations: per
    (query, head, key) the score and the weighted sum, 2 head_dim each, and
    five such products in training's backward (the recomputed score, dO.v, dq,
    dk, dv), sampling counted as free; per conv tap 2 a direction."""
    e = 2 if case["dtype"] == "bf16" else 4
    if case["kind"] == "conv":
        N, K = case["B"] * case["T"] * case["H"] * case["W"], math.prod(_window(case))
        ND = N * case["C"]
        # forward: x, y (GELU also keeps its input: not counted); backward: x, dy, dx
        return {"bytes": 5 * e * ND, "flops": 3 * 2 * K * ND}
    B, N, D, K = _sizes(case)
    R, nh, hd = B * N, case["heads"], case["head_dim"]
    C = nh * K * 3
    keys = K + case.get("extra", 0)
    train = case.get("train", True)
    byts = R * (e * (4 * D + C)) + (R * (e * (8 * D + 2 * C) + 4 * nh) if train else 0)
    flops = R * nh * keys * hd * (4 + (10 if train else 0))
    if case["kind"] == "block":
        # GEMMs: q, k, v, out, offsets, MLP; forward once, backward twice; both convs
        mm = 2 * R * D * (4 * D + C + 8 * D)
        flops += 3 * mm + 3 * 2 * R * D * (K + 27)
        weights = e * (4 * D * D + D * C + 8 * D * D)
        byts = e * R * D * 4 + 3 * weights
    return {"bytes": byts, "flops": flops}


def tolerance(case):
    """About four times the difference measured against ``exact``: bf16 at most 2.9e-3 (dk),
    fp32 at most 4.4e-7 in the core, sums in another order up to 1.1e-6 in the block.  The
    block's offsets are its own arithmetic's: one of its 3.7 million tap positions that
    another summation order puts across a voxel's edge changes that tap's gradient by its own
    size, 1 / sqrt(3.7e6) = 5e-4 of the gradient's norm."""
    if case["kind"] == "block":
        return {"rel": 2e-3}
    return {"rel": 1.2e-2 if case["dtype"] == "bf16" else 5e-6}


# ---------------------------------------------------------------------------
# float64 results
# ---------------------------------------------------------------------------

def _axis(n_pos, taps, offsets, S, div):
    """Sampling position of one axis: [n, K] lower corner, upper weight, and the mask of the
    unclamped positions.  The position is fp32, op by op, by definition of the operator
    (the corner a tap takes at a voxel's edge depends on that rounding).  Divisors are
    device tensors: a division by a Python number multiplies by its reciprocal on the GPU."""
    pos = n_pos.float()[:, None] + taps.float()[None, :]
    g = 2.0 * pos / torch.full_like(pos, max(S - 1, 1)) - 1.0
    if div > 0:
        g = g + offsets / torch.full_like(offsets, div)
    u = ((g + 1.0) * float(S) - 1.0) / 2.0
    c = u.clamp(0.0, float(S - 1))
    fl = c.floor()
    inside = (u > 0.0) & (u < float(S - 1))
    return fl.long(), (c - fl).double(), inside


def _core_exact(c, q, k, v, off, ek, ev, dout):
    """out and, with dout, dq, dk, dv, d offsets (and d extra keys, values) in float64."""
    B, N, D, K = _sizes(c)
    T, H, W = _grid(c)
    nh, hd = c["heads"], c["head_dim"]
    kt, kh, kw = _window(c)
    dev = q.device
    tap = torch.arange(K, device=dev)
    ci, cj, ck = tap // (kh * kw) - kt // 2, (tap // kw) % kh - kh // 2, tap % kw - kw // 2
    scale = 1.0 / math.sqrt(hd)
    f64 = dict(dtype=torch.float64, device=dev)
    out = torch.empty(B, N, D, **f64)
    grads = None
    if dout is not None:
        grads = [torch.zeros(B, N, D, **f64) for _ in range(3)]
        grads.append(torch.empty(B, N, nh, K, 3, **f64))
        if ek is not None:
            grads += [torch.zeros(ek.shape, **f64) for _ in range(2)]
    step = max(1, 2 ** 25 // (K * hd))
    for b in range(B):
        for h in range(nh):
            ch = slice(h * hd, (h + 1) * hd)
            kf, vf = k[b, :, ch].double(), v[b, :, ch].double()
            for n0 in range(0, N, step):
                n = torch.arange(n0, min(n0 + step, N), device=dev)
                o3 = off[b, n, h * K * 3:(h + 1) * K * 3].float().view(-1, K, 3)
                x0, fx, mx = _axis(n % W, ck, o3[..., 0], W, T - 1)
                y0, fy, my = _axis((n // W) % H, cj, o3[..., 1], H, H - 1)
                z0, fz, mz = _axis(n // (W * H), ci, o3[..., 2], T, W - 1)
                qf = q[b, n, ch].double()
                idx, wts, sc = [], [], []
                for dz in (0, 1):
                    for dy in (0, 1):
                        for dx in (0, 1):
                            i = (((z0 + dz).clamp_max(T - 1) * H + (y0 + dy).clamp_max(H - 1)) * W
                                 + (x0 + dx).clamp_max(W - 1))
                            ax = (fx if dx else 1 - fx, fy if dy else 1 - fy, fz if dz else 1 - fz)
                            idx.append(i)
                            wts.append(ax)
                            sc.append((kf[i] @ qf[:, :, None])[..., 0])
                s = sum(wx * wy * wz * t for (wx, wy, wz), t in zip(wts, sc)) * scale
                if ek is not None:
                    ekf, evf = ek[b, :, ch].double(), ev[b, :, ch].double()
                    s = torch.cat([s, qf @ ekf.t() * scale], 1)
                p = torch.softmax(s, 1)
                o = p[:, K:] @ evf if ek is not None else 0.0
                vc = [] if dout is not None else None
                gf = dout[b, n, ch].double() if dout is not None else None
                for i, (wx, wy, wz) in zip(idx, wts):
                    rows = vf[i]
                    o = o + ((p[:, :K] * wx * wy * wz)[:, None] @ rows)[:, 0]
                    if vc is not None:
                        vc.append((rows @ gf[:, :, None])[..., 0])
                out[b, n, ch] = o
                if dout is None:
                    continue
                dp = sum(wx * wy * wz * t for (wx, wy, wz), t in zip(wts, vc))
                if ek is not None:
                    dp = torch.cat([dp, gf @ evf.t()], 1)
                ds = p * (dp - (p * dp).sum(1, keepdim=True)) * scale
                dst, pt = ds[:, :K], p[:, :K]
                dq = ds[:, K:] @ ekf if ek is not None else 0.0
                du = [0.0, 0.0, 0.0]
                for j, (i, (wx, wy, wz)) in enumerate(zip(idx, wts)):
                    w = wx * wy * wz
                    dq = dq + ((dst * w)[:, None] @ kf[i])[:, 0]
                    grads[1][b, :, ch].index_add_(
                        0, i.reshape(-1), ((dst * w)[..., None] * qf[:, None]).reshape(-1, hd))
                    grads[2][b, :, ch].index_add_(
                        0, i.reshape(-1), ((pt * w)[..., None] * gf[:, None]).reshape(-1, hd))
                    t = dst * sc[j] + pt * vc[j]
                    sx, sy, sz = (1 if j & 1 else -1), (1 if j & 2 else -1), (1 if j & 4 else -1)
                    du[0] = du[0] + sx * wy * wz * t
                    du[1] = du[1] + sy * wx * wz * t
                    du[2] = du[2] + sz * wx * wy * t
                grads[0][b, n, ch] = dq
                for j, (m, S, div) in enumerate(((mx, W, T - 1), (my, H, H - 1), (mz, T, W - 1))):
                    grads[3][b, n, h, :, j] = du[j] * m * (0.5 * S / div if div > 0 else 0.0)
                if ek is not None:
                    grads[4][b, :, ch] += ds[:, K:].t() @ qf
                    grads[5][b, :, ch] += p[:, K:].t() @ gf
    if dout is None:
        return out
    grads[3] = grads[3].view(B, N, nh * K * 3)
    return (out, *grads)


def _conv_exact(c, x, w, b, dy):
    """y, dx, dw, db: the sum over taps of shifted slices, in float64."""
    B, (T, H, W), C = c["B"], _grid(c), c["C"]
    kt, kh, kw = _window(c)
    pad = (0, 0, kw // 2, kw // 2, kh // 2, kh // 2, kt // 2, kt // 2)
    xp = F.pad(x.view(B, T, H, W, C), pad).double()
    wf = w.double().view(C, kt * kh * kw)

    def taps():
        for j in range(kt * kh * kw):
            i0, i1, i2 = j // (kh * kw), (j // kw) % kh, j % kw
            yield j, (slice(None), slice(i0, i0 + T), slice(i1, i1 + H), slice(i2, i2 + W))

    z = b.double().expand(B, T, H, W, C).clone()
    for j, sl in taps():
        z += xp[sl] * wf[:, j]
    dz = dy.double().view(z.shape)
    y = z
    if c["gelu"]:
        cdf = 0.5 * (1.0 + torch.erf(z / math.sqrt(2.0)))
        y = z * cdf
        dz = dz * (cdf + z * torch.exp(-0.5 * z * z) / math.sqrt(2.0 * math.pi))
    dxp, dw = torch.zeros_like(xp), torch.empty_like(wf)
    for j, sl in taps():
        dxp[sl] += dz * wf[:, j]
        dw[:, j] = (xp[sl] * dz).sum((0, 1, 2, 3))
    dx = dxp[:, kt // 2:kt // 2 + T, kh // 2:kh // 2 + H, kw // 2:kw // 2 + W]
    return (y.reshape(x.shape), dx.reshape(x.shape), dw.view(w.shape), dz.sum((0, 1, 2, 3)))


def _block_exact(c, params, x, dy):
    """The block's output.  Its gradients have no float64 counterpart: the offsets' gradient
    jumps where a position crosses a voxel's edge, and the positions come from the block's
    own fp32 arithmetic."""
    p = {n: t.to(_DT[c["dtype"]]).double() for n, t in params.items()}
    B, N, D, K = _sizes(c)
    x = x.double()

    def norm(t, n):
        return F.layer_norm(t, (D,), p[n + ".weight"], p[n + ".bias"], 1e-6)

    def lin(t, n):
        return t @ p[n + ".weight"].flatten(1).t() + p[n + ".bias"]

    def conv(t, n, window, gelu):
        cc = {**c, "C": D, "kt": window[0], "kh": window[1], "kw": window[2], "gelu": gelu}
        return _conv_exact(cc, t, p[n + ".weight"], p[n + ".bias"], t)[0]

    a = norm(x, "norm1")
    off = lin(conv(a, "attn.offset_net.0", (3, 3, 3), True), "attn.offset_net.2")
    core = _core_exact({**c, "extra": 0}, lin(a, "attn.q_proj"), lin(a, "attn.k_proj"),
                       lin(a, "attn.v_proj"), off, None, None, None)
    x = x + lin(core, "attn.out_proj") + conv(a, "attn.dw_conv", _window(c), False)
    h = F.gelu(lin(norm(x, "norm2"), "mlp.fc1"))
    y = x + lin(h, "mlp.fc2")
    return (y,) + (None,) * len(p)  # dx and every parameter's gradient but k_proj.bias


def exact(case, seed):
    with torch.no_grad():
        if case["kind"] == "core":
            B, N, D, K = _sizes(case)
            if B * N * D * K > 2 ** 34:  # over about 20 seconds
                return None
            return _core_exact(case, *_core_inputs(case, seed))
        if case["kind"] == "conv":
            return _conv_exact(case, *_conv_inputs(case, seed))
        return _block_exact(case, *_block_inputs(case, seed))
