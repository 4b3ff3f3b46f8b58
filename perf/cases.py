"""Performance cases of the selective-scan framework: the work a user has it
do, through its public entry points.

Kinds (``case["op"]``):
  scan      a plain selective scan call, training (forward + VJP) or the
            inference-only ``metal`` mode, float32 or bf16 inputs
  conv      the direction-batched causal conv + SiLU, forward + backward
  norm      the pre-norm with its residual branch, forward + backward
  block     a Mamba block (plain, bidirectional or multi-directional),
            forward only or forward + backward
  encoder   a whole VisionMamba: one training step with AdamW, or a forward

Inputs follow the distributions of ``mlx_vision_mamba_amd.synthetic``: unit
normal activations, dt log-normal in about [1e-3, 1e-1], S4D-real A.
"""

import math

import torch
import torch.nn.functional as F

import mlx_vision_mamba_amd as mvm
from mlx_vision_mamba_amd import directions, gemm_tuning
from mlx_vision_mamba_amd.conv import causal_conv_silu
from mlx_vision_mamba_amd.norm import layer_norm
from mlx_vision_mamba_amd.optim import AdamW

DEV = "cuda"


def listed():
    return [
        # the scan of one d_model = 768 block on a 14x14 grid, trained: the
        # reference's single-block shape, bound by latency and launches
        {"name": "scan_single_train", "op": "scan", "train": True, "dtype": "float32",
         "B": 2, "L": 196, "D": 1536, "N": 16},
        # inference on a ragged batch: odd length, channels not a multiple of 64
        {"name": "scan_ragged_infer", "op": "scan", "train": False, "dtype": "bfloat16",
         "B": 3, "L": 1037, "D": 1000, "N": 16},
        # the long-sequence workload of the benchmark, bf16 activations
        {"name": "scan_long_train", "op": "scan", "train": True, "dtype": "bfloat16",
         "B": 8, "L": 16384, "D": 1536, "N": 16},
        # the conv of one VisionMamba-2D layer of the training step
        {"name": "conv_2d_train", "op": "conv", "B": 32, "L": 196, "K": 4, "D": 768, "W": 4},
        # the pre-norm of the same layer, its residual gradient added
        {"name": "norm_2d_train", "op": "norm", "rows": 6272, "E": 384},
        # one image through one block: the smallest call of a serving loop
        {"name": "block_single_infer", "op": "block", "block": "mamba", "train": False,
         "B": 1, "L": 196, "E": 384, "N": 16, "K": 1, "grid": ""},
        # the reference's single block, trained at batch 2
        {"name": "block_single_train", "op": "block", "block": "mamba", "train": True,
         "B": 2, "L": 196, "E": 768, "N": 16, "K": 1, "grid": ""},
        # odd sizes throughout: width, length, batch and a smaller state
        {"name": "block_bidir_ragged_train", "op": "block", "block": "bidirectional", "train": True,
         "B": 5, "L": 331, "E": 200, "N": 8, "K": 2, "grid": ""},
        # one layer of the benchmark's 2D training step
        {"name": "block_2d_train", "op": "block", "block": "multi", "train": True,
         "B": 32, "L": 196, "E": 384, "N": 16, "K": 4, "grid": "14x14"},
        # one layer of the 3D encoder on 16^3 patches, trained: the largest block
        {"name": "block_3d_train", "op": "block", "block": "multi", "train": True,
         "B": 4, "L": 4096, "E": 384, "N": 16, "K": 6, "grid": "16x16x16"},
        # the benchmark's whole 2D training step: forward, loss, backward, AdamW
        {"name": "encoder_2d_step", "op": "encoder", "train": True, "dim": 2, "B": 32, "img": 224,
         "patch": 16, "frames": 1, "E": 384, "depth": 6},
        # a forward of the 4D encoder: clips of 8 volumes of 64^3
        {"name": "encoder_4d_infer", "op": "encoder", "train": False, "dim": 4, "B": 2, "img": 64,
         "patch": 16, "frames": 8, "E": 384, "depth": 6},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["scan", "scan", "conv", "norm", "block", "block", "block", "encoder"])
    if op == "scan":
        D = _log(rng, 192, 1536)
        L = _log(rng, 100, 16384)
        B = max(1, min(_log(rng, 1, 32), 8 * 16384 * 1536 // (L * D)))
        return {"op": "scan", "train": rng.random() < 0.7,
                "dtype": rng.choice(["float32", "bfloat16"]) if B * L * D < 6e7 else "bfloat16",
                "B": B, "L": L, "D": D, "N": rng.choice([8, 13, 16, 16, 16])}
    if op == "conv":
        return {"op": "conv", "B": _log(rng, 1, 32), "L": _log(rng, 49, 512), "K": rng.choice([1, 2, 4, 6]),
                "D": _log(rng, 128, 1024), "W": rng.choice([3, 4, 4])}
    if op == "norm":
        return {"op": "norm", "rows": _log(rng, 196, 20000), "E": rng.choice([192, 200, 384, 384, 500, 768])}
    if op == "block":
        kind = rng.choice(["mamba", "bidirectional", "multi", "multi"])
        E = rng.choice([160, 200, 256, 384, 384])
        train = rng.random() < 0.7
        if kind == "multi":
            K = rng.choice([4, 6])
            dims = [rng.randint(7, 20) for _ in range(2)] if K == 4 else [rng.randint(4, 11) for _ in range(3)]
            L = math.prod(dims)
            return {"op": "block", "block": kind, "train": train, "B": max(1, min(_log(rng, 1, 40), 14000 // L)),
                    "L": L, "E": E, "N": 16, "K": K, "grid": "x".join(str(d) for d in dims)}
        L = _log(rng, 60, 1500)
        return {"op": "block", "block": kind, "train": train, "B": max(1, min(_log(rng, 1, 40), 14000 // L)),
                "L": L, "E": E, "N": rng.choice([8, 16, 16]), "K": 2 if kind == "bidirectional" else 1,
                "grid": ""}
    dim = rng.choice([2, 3])
    grid = rng.randint(8, 14) if dim == 2 else rng.randint(4, 6)
    return {"op": "encoder", "train": rng.random() < 0.5, "dim": dim, "B": rng.randint(1, 24 if dim == 2 else 8),
            "img": grid * 16, "patch": 16, "frames": 1, "E": rng.choice([192, 384]), "depth": rng.randint(2, 5)}


# ------------------------------------------------------------------ inputs

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _grid(case):
    return tuple(int(v) for v in case["grid"].split("x")) if case["grid"] else None


def _randomise(module, seed):
    """Weights that a trained model could hold: the norms' gains and biases,
    D and the biases away from their initial constants."""
    g = _gen(seed)
    with torch.no_grad():
        for name, p in module.named_parameters():
            if name.endswith("norm.weight") or name.endswith(".D") or name == "D":
                p.add_(torch.randn(p.shape, generator=g, device=DEV), alpha=0.1)
            elif name.endswith("norm.bias") or name.endswith("A_log"):
                p.add_(torch.randn(p.shape, generator=g, device=DEV), alpha=0.05)


def prepare(case, seed):
    g = _gen(seed)
    rn = lambda *s: torch.randn(*s, generator=g, device=DEV)  # noqa: E731
    op, st = case["op"], {"case": case}
    if op == "scan":
        B, L, D, N = case["B"], case["L"], case["D"], case["N"]
        dt = getattr(torch, case["dtype"])
        u = rn(B, L, D).to(dt)
        delta = F.softplus(rn(B, L, D) * 0.5 - 4.6)
        A = -torch.arange(1, N + 1, dtype=torch.float32, device=DEV).repeat(D, 1) * torch.exp(0.05 * rn(D, N))
        ins = [u, delta, A, rn(B, L, N).to(dt), rn(B, L, N).to(dt), 1.0 + 0.1 * rn(D)]
        st["in"] = [t.requires_grad_(case["train"]) for t in ins]
        st["dy"] = rn(B, L, D).to(dt) if case["train"] else None
    elif op == "conv":
        B, L, K, D, W = (case[k] for k in "BLKDW")
        # the conv reads the first half of the in_proj output
        xz = rn(B, L, K, 2 * D)
        st["in"] = [xz[..., :D].detach().requires_grad_(), (rn(K, D, W) * W ** -0.5).requires_grad_(),
                    (rn(K, D) * 0.1).requires_grad_()]
        order = torch.stack([torch.arange(L) if k % 2 == 0 else torch.arange(L).flip(0) for k in range(K)])
        st["tok"] = order.to(torch.int32).to(DEV)
        st["dy"] = rn(B, L, K, D)
    elif op == "norm":
        norm = torch.nn.LayerNorm(case["E"]).to(DEV)
        with torch.no_grad():
            norm.weight.add_(rn(case["E"]), alpha=0.1)
            norm.bias.add_(rn(case["E"]), alpha=0.1)
        st["norm"] = norm
        st["x"] = (rn(case["rows"], case["E"]) * 2 + 0.3).requires_grad_()
        st["dy"], st["dres"] = rn(case["rows"], case["E"]), rn(case["rows"], case["E"])
    elif op == "block":
        gemm_tuning.load()  # the recorded GEMM picks, as the benchmark loads them
        torch.manual_seed(seed)
        E, N = case["E"], case["N"]
        if case["block"] == "mamba":
            m = mvm.MambaBlock(E, d_state=N, scan_mode="hip")
        elif case["block"] == "bidirectional":
            m = mvm.BidirectionalMambaBlock(E, d_state=N, scan_mode="hip")
        else:
            m = mvm.MultiDirectionalMambaBlock(E, d_state=N, num_directions=case["K"], grid_shape=_grid(case),
                                               scan_mode="hip")
        st["m"] = m = m.to(DEV)
        _randomise(m, seed)
        st["x"] = rn(case["B"], case["L"], E).requires_grad_(case["train"])
        st["dy"] = rn(case["B"], case["L"], E) if case["train"] else None
        st["params"] = list(m.parameters())
    else:
        gemm_tuning.load()
        torch.manual_seed(seed)
        m = mvm.VisionMamba(img_size=case["img"], patch_size=case["patch"], in_channels=1, embed_dim=case["E"],
                            depth=case["depth"], input_dim=case["dim"], num_temporal_frames=case["frames"],
                            scan_mode="hip")
        st["m"] = m = m.to(DEV)
        _randomise(m, seed)
        space = (case["img"],) * min(case["dim"], 3)
        st["x"] = rn(case["B"], *((case["frames"],) if case["dim"] == 4 else ()), *space, 1)
        if case["train"]:
            st["opt"] = AdamW(m.parameters(), lr=1e-4)
            st["target"] = rn(case["B"], m.num_patches, case["E"])
    return st


# --------------------------------------------------------------------- run

def run(st):
    case = st["case"]
    op = case["op"]
    if op == "scan":
        if not case["train"]:
            return mvm.selective_scan_metal(*st["in"])
        y = mvm.selective_scan(*st["in"])
        return [y, *torch.autograd.grad(y, st["in"], st["dy"])]
    if op == "conv":
        y = causal_conv_silu(*st["in"], st["tok"])
        return [y, *torch.autograd.grad(y, st["in"], st["dy"])]
    if op == "norm":
        y, xr = layer_norm(st["x"], st["norm"], residual=True)
        return [y, *torch.autograd.grad([y, xr], [st["x"], st["norm"].weight, st["norm"].bias],
                                        [st["dy"], st["dres"]])]
    if op == "block":
        if not case["train"]:
            with torch.no_grad():
                return st["m"](st["x"])
        y = st["m"](st["x"])
        return [y, *torch.autograd.grad(y, [st["x"], *st["params"]], st["dy"])]
    if not case["train"]:
        with torch.no_grad():
            return st["m"](st["x"])
    opt = st["opt"]
    opt.zero_grad(set_to_none=True)
    y = st["m"](st["x"])
    F.mse_loss(y, st["target"]).backward()
    opt.step()
    # the moments hold every parameter's gradient (scaled by 1 - beta1 on the
    # first step), in the order of the parameters
    return [y, opt.exp_avg]


# ----------------------------------------------------------- work, accuracy

# operations of the scan per (batch, position, direction, channel, state):
# forward, and forward + VJP with its recomputed states
SCAN_FWD, SCAN_TRAIN = 8, 40


def _block_work(B, L, E, N, K, train, norm):
    din, R = 2 * E, math.ceil(E / 16)
    weights = K * (2 * din * E + din * (R + 2 * N) + din * R + din * E + din * (N + 4 + 3)) + (2 * E if norm else 0)
    macs = B * L * K * (2 * din * E + din * (R + 2 * N) + din * R + din * E)
    flops = 2 * macs * (3 if train else 1) + (SCAN_TRAIN if train else SCAN_FWD) * B * L * K * din * N
    return weights, flops


def work(case):
    op = case["op"]
    if op == "scan":
        B, L, D, N = case["B"], case["L"], case["D"], case["N"]
        s = 4 if case["dtype"] == "float32" else 2
        fwd = B * L * D * (2 * s + 4) + B * L * N * 2 * s + D * (N + 1) * 4
        vjp = B * L * D * (3 * s + 8) + B * L * N * 4 * s + D * (N + 1) * 8
        return {"bytes": fwd + (vjp if case["train"] else 0),
                "flops": B * L * D * N * (SCAN_TRAIN if case["train"] else SCAN_FWD)}
    if op == "conv":
        n = case["B"] * case["L"] * case["K"] * case["D"]
        return {"bytes": n * 4 * 5, "flops": n * (6 * case["W"] + 20)}
    if op == "norm":
        return {"bytes": case["rows"] * case["E"] * 4 * 6, "flops": case["rows"] * case["E"] * 20}
    if op == "block":
        w, fl = _block_work(case["B"], case["L"], case["E"], case["N"], case["K"], case["train"],
                            case["block"] != "mamba")
        x = case["B"] * case["L"] * case["E"]
        return {"bytes": 4 * (w * (2 if case["train"] else 1) + x * (4 if case["train"] else 2)), "flops": fl}
    g = case["img"] // case["patch"]
    K = {2: 4, 3: 6, 4: 8}[case["dim"]]
    L = g ** min(case["dim"], 3) * case["frames"]
    w, fl = _block_work(case["B"], L, case["E"], 16, K, case["train"], True)
    pix = case["patch"] ** min(case["dim"], 3)
    w, fl = w * case["depth"] + pix * case["E"], fl * case["depth"] + 4 * case["B"] * L * pix * case["E"]
    x = case["B"] * L * (pix + case["E"])
    # a training step also reads and writes both moments of every weight
    return {"bytes": 4 * (w * (7 if case["train"] else 1) + x * (2 if case["train"] else 1)), "flops": fl}


def tolerance(case):
    """About four times the largest error against 64 bits over the listed and
    24 drawn cases: scan float32 2.7e-7 (max 5.1e-6), bf16 results 1.7e-3
    (3.9e-3: their rounding), conv and norm 1.5e-7 (1.6e-6), block 2.4e-6
    (2.9e-5), encoder 1.4e-6 (1.9e-5; its training step repeats with updated
    weights, so twice that)."""
    op = case["op"]
    if op == "scan":
        return {"rel": 1.2e-6, "max": 2e-5} if case["dtype"] == "float32" else {"rel": 7e-3, "max": 1.6e-2}
    if op in ("conv", "norm"):
        return {"rel": 6e-7, "max": 7e-6}
    if op == "block":
        return {"rel": 1e-5, "max": 1.2e-4}
    return {"rel": 1.2e-5, "max": 1.6e-4} if case["train"] else {"rel": 6e-6, "max": 8e-5}


# ------------------------------------------------ the same results in 64 bits

class _Scan64(torch.autograd.Function):
    """y_t = C_t . h_t + D u_t, h_t = exp(delta_t A) h_{t-1} + delta_t u_t B_t
    and its gradients, position by position.  Shapes: u, delta (B, L, K, D);
    A (K, D, N); Bm, C (B, L, K, N); Dv (K, D); each direction in scan order."""

    @staticmethod
    def forward(ctx, u, delta, A, Bm, C, Dv):
        B, L, K, D = u.shape
        hs = u.new_empty(L, B, K, D, A.shape[-1])
        y = torch.empty_like(u)
        h = torch.zeros_like(hs[0])
        for t in range(L):
            h = torch.exp(delta[:, t, :, :, None] * A) * h
            h += (delta[:, t] * u[:, t])[..., None] * Bm[:, t, :, None, :]
            hs[t] = h
            y[:, t] = (h * C[:, t, :, None, :]).sum(-1) + Dv * u[:, t]
        ctx.save_for_backward(u, delta, A, Bm, C, Dv, hs)
        return y

    @staticmethod
    def backward(ctx, g):
        u, delta, A, Bm, C, Dv, hs = ctx.saved_tensors
        du, dd, dB, dC = (torch.empty_like(t) for t in (u, delta, Bm, C))
        dA, mu = torch.zeros_like(A), torch.zeros_like(hs[0])
        for t in range(u.shape[1] - 1, -1, -1):
            dl, ut, bt = delta[:, t], u[:, t], Bm[:, t, :, None, :]
            lam = mu + g[:, t, :, :, None] * C[:, t, :, None, :]
            mu = torch.exp(dl[..., None] * A) * lam
            lb = (lam * bt).sum(-1)
            dd[:, t], du[:, t] = lb * ut, lb * dl + Dv * g[:, t]
            if t:
                w = mu * hs[t - 1]
                dA += (dl[..., None] * w).sum(0)
                dd[:, t] += (w * A).sum(-1)
            dB[:, t] = (lam * (dl * ut)[..., None]).sum(-2)
            dC[:, t] = (g[:, t, :, :, None] * hs[t]).sum(-2)
        return du, dd, dA, dB, dC, (g * u).sum((0, 1))


def _conv64(x, w, b):
    """silu(causal depthwise conv) of (B, L, K, D) in scan order, w (K, D, W)."""
    L, W = x.shape[1], w.shape[-1]
    xp = F.pad(x, (0, 0, 0, 0, W - 1, 0))
    return F.silu(b + sum(xp[:, j:j + L] * w[..., j] for j in range(W)))


def _gather(x, order):
    """(B, L, K, X) with direction k's positions in the order order[k]."""
    return torch.gather(x, 1, order.t()[None, :, :, None].expand(x.shape))


def _mamba64(h, p, order, N):
    """Sum over directions of the Mamba block with stacked parameters p."""
    K, (B, L, _) = p["A_log"].shape[0], h.shape
    xz = torch.stack([F.linear(h, p["in_proj.weight"][k]) for k in range(K)], 2)
    x, z = _gather(xz, order).chunk(2, -1)
    x = _conv64(x, p["conv1d.weight"][:, :, 0], p["conv1d.bias"])
    proj = torch.stack([F.linear(x[:, :, k], p["x_proj.weight"][k]) for k in range(K)], 2)
    dt, Bm, C = proj.split([proj.shape[-1] - 2 * N, N, N], -1)
    dt = torch.stack([F.linear(dt[:, :, k], p["dt_proj.weight"][k], p["dt_proj.bias"][k]) for k in range(K)], 2)
    y = _Scan64.apply(x, F.softplus(dt), -torch.exp(p["A_log"]), Bm, C, p["D"]) * F.silu(z)
    y = _gather(y, torch.argsort(order, 1))
    return sum(F.linear(y[:, :, k], p["out_proj.weight"][k]) for k in range(K))


_KINDS = ("in_proj.weight", "conv1d.weight", "conv1d.bias", "x_proj.weight", "dt_proj.weight", "dt_proj.bias",
          "A_log", "D", "out_proj.weight")


def _block64(x, params, prefixes, norm, order, N):
    p = {k: torch.stack([params[f + k] for f in prefixes]) for k in _KINDS}
    if norm is None:
        return _mamba64(x, p, order, N)
    h = F.layer_norm(x, x.shape[-1:], params[norm + "weight"], params[norm + "bias"])
    return x + _mamba64(h, p, order, N)


def _order(K, L, grid):
    if K == 1:
        return torch.arange(L, device=DEV)[None]
    return directions.seq_to_tok_table(K, L, grid if K > 2 else None).long().to(DEV)


def exact(case, seed):
    op = case["op"]
    st = prepare(case, seed)
    dbl = lambda t: t.detach().double().requires_grad_()  # noqa: E731
    if op == "scan":
        if case["B"] * case["L"] * case["D"] * case["N"] > 4.1e9:
            return None
        ins = [dbl(t) for t in st["in"]]
        lift = [t.unsqueeze(d) for t, d in zip(ins, (2, 2, 0, 2, 2, 0))]
        with torch.set_grad_enabled(case["train"]):
            y = _Scan64.apply(*lift)[:, :, 0]
        return [y, *torch.autograd.grad(y, ins, st["dy"].double())] if case["train"] else y
    if op == "conv":
        x, w, b = ins = [dbl(t) for t in st["in"]]
        order = st["tok"].long()
        y = _gather(_conv64(_gather(x, order), w, b), torch.argsort(order, 1))
        return [y, *torch.autograd.grad(y, ins, st["dy"].double())]
    if op == "norm":
        x, w, b = ins = [dbl(t) for t in (st["x"], st["norm"].weight, st["norm"].bias)]
        y = F.layer_norm(x, x.shape[-1:], w, b, st["norm"].eps)
        return [y, *torch.autograd.grad([y, x * 1], ins, [st["dy"].double(), st["dres"].double()])]
    params = {n: dbl(p) for n, p in st["m"].named_parameters()}
    if op == "block":
        K, N = case["K"], case["N"]
        order = _order(K, case["L"], _grid(case))
        prefixes = {"mamba": [""], "bidirectional": ["forward_mamba.", "backward_mamba."]}.get(
            case["block"], ["mamba_blocks.%d." % k for k in range(K)])
        x = dbl(st["x"])
        with torch.set_grad_enabled(case["train"]):
            y = _block64(x, params, prefixes, None if case["block"] == "mamba" else "norm.", order, N)
        return [y, *torch.autograd.grad(y, [x, *params.values()], st["dy"].double())] if case["train"] else y
    dim, p, B = case["dim"], case["patch"], case["B"]
    g, K = case["img"] // p, {2: 4, 3: 6, 4: 8}[dim]
    grid = ((case["frames"],) if dim == 4 else ()) + (g,) * min(dim, 3)
    L = math.prod(grid)
    order = _order(K, L, grid)
    with torch.set_grad_enabled(case["train"]):
        x = st["x"].double()
        if dim == 4:
            x = x.flatten(0, 1)
        x = (F.conv2d if dim == 2 else F.conv3d)(x.movedim(-1, 1), params["patch_embed.proj.weight"],
                                                 params["patch_embed.proj.bias"], stride=p)
        x = x.flatten(2).transpose(1, 2).reshape(B, L, -1) + params["pos_embed"]
        for i in range(case["depth"]):
            x = _block64(x, params, ["blocks.%d.mamba_blocks.%d." % (i, k) for k in range(K)],
                         "blocks.%d.norm." % i, order, 16)
        y = F.layer_norm(x, x.shape[-1:], params["norm.weight"], params["norm.bias"])
    if not case["train"]:
        return y
    grads = torch.autograd.grad(F.mse_loss(y, st["target"].double()), list(params.values()))
    return [y, 0.1 * torch.cat([t.reshape(-1) for t in grads])]
