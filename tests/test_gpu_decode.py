"""Forward calls that read the weights as they are stored (no op-dtype copy):
few routes per expert (the weight-streaming kernel, fp32 or 16-bit weights),
and 16-bit weights with more routes (the long-K kernel on [k][n] rows).  Each
against the per-route products of the rounded operands in float64, at tile
edges of every size: rows around 16 per expert and past 64 of them, K with
partial 32-k steps, N with partial column tiles."""
import pytest
import torch

import cvmm_codex_amd.api as C

pytestmark = pytest.mark.gpu

_DT = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


def _case(T, k, E, D, H, op, weights, hot, seed):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(T, D, generator=g).to(_DT[op])
    keys = (torch.randn(E, D, H, generator=g) / D ** 0.5).to(_DT[weights])
    sel = torch.randint(0, E, (T, k), generator=g)
    if hot:
        sel[:, 0] = E - 1
    return x.cuda(), keys.cuda(), sel.cuda()


def _check(y, ref, tol=2e-2):
    # one rounding of a product of K rounded terms to the output type: u |y|
    # (2^-8 in bf16) plus fp32 sums; 2e-2 of the largest magnitude as in the
    # parity tests
    assert torch.isfinite(y.float()).all()
    err = ((y.double() - ref).abs().max() / ref.abs().max()).item()
    assert err <= tol, err


@pytest.mark.parametrize("op,weights", [("bf16", "fp32"), ("bf16", "bf16"), ("fp16", "fp32"), ("fp16", "fp16")])
@pytest.mark.parametrize("T,k,E,D,H,hot", [
    (1, 1, 1, 8, 8, False), (1, 8, 64, 1024, 128, False), (4, 8, 64, 128, 1024, False), (3, 2, 5, 40, 72, False),
    (17, 1, 1, 136, 136, False), (33, 8, 16, 200, 520, True), (65, 4, 8, 1000, 264, True), (64, 2, 3, 264, 64, False),
    (200, 4, 16, 96, 136, True), (130, 8, 128, 520, 40, True), (20, 4, 70, 1000, 1032, True)])
def test_forward_reads_the_stored_weights(T, k, E, D, H, hot, op, weights):
    x, keys, sel = _case(T, k, E, D, H, op, weights, hot, T + D)
    with torch.no_grad(), torch.autocast("cuda", dtype=_DT[op]):
        y = C.cvmm(x, C.cvmm_prepare_sel2(sel), keys)
        yg = C.cvmm_gelu(x, C.cvmm_prepare_sel2(sel), keys)
        w = torch.rand(T, k, device="cuda")
        xr = torch.randn(T, k, D, device="cuda").to(_DT[op])
        yw = C.cvmm(xr, C.cvmm_prepare_sel2(sel, w, route_input=True), keys)
    kd = keys.to(_DT[op]).double()
    ref = torch.stack([torch.stack([x[t].double() @ kd[sel[t, j]] for j in range(k)]) for t in range(T)])
    _check(y, ref)
    _check(yg, torch.nn.functional.gelu(ref))
    refw = torch.stack([sum(w[t, j].double() * (xr[t, j].double() @ kd[sel[t, j]]) for j in range(k)) for t in range(T)])
    _check(yw, refw)


@pytest.mark.parametrize("weights,D,H", [("bf16", 136, 128), ("fp16", 264, 72), ("bf16", 128, 136)])
def test_16_bit_weights_train_without_a_copy(weights, D, H):
    """Forward and grad-input both read the 16-bit weights in place (d_in >
    128) or one copy beside them: the gradients against float64 autograd."""
    T, k, E = 700, 2, 4
    x, keys, sel = _case(T, k, E, D, H, weights, weights, True, D)
    x.requires_grad_()
    keys.requires_grad_()
    gy = torch.randn(T, k, H, device="cuda").to(x.dtype)
    with torch.autocast("cuda", dtype=x.dtype):
        y = C.cvmm(x, C.cvmm_prepare_sel2(sel), keys)
    gx, gk = torch.autograd.grad(y, [x, keys], gy)
    xd, kd = x.detach().double().requires_grad_(), keys.detach().double().requires_grad_()
    rows = xd.repeat_interleave(k, 0)
    onehot = torch.nn.functional.one_hot(sel.reshape(-1), E).double()
    ref = sum(onehot[:, e:e + 1] * (rows @ kd[e]) for e in range(E)).view(T, k, H)
    rx, rk = torch.autograd.grad(ref, [xd, kd], gy.double())
    _check(y, ref.detach())
    _check(gx, rx)
    _check(gk, rk)
    assert gk.dtype == keys.dtype


def test_stored_weights_views_fall_back():
    """Transposed, strided and misaligned weights of the op dtype: same results."""
    T, k, E, D, H = 9, 2, 3, 136, 72
    x, keys, sel = _case(T, k, E, D, H, "bf16", "bf16", False, 5)
    flat = torch.zeros(keys.numel() + 1, dtype=keys.dtype, device="cuda")
    flat[1:] = keys.reshape(-1)
    views = [keys, keys.transpose(1, 2).contiguous().transpose(1, 2), flat[1:].view(E, D, H),
             torch.stack([keys, keys], -1)[..., 0]]
    outs = []
    with torch.no_grad(), torch.autocast("cuda", dtype=torch.bfloat16):
        for v in views:
            outs.append(C.cvmm(x, C.cvmm_prepare_sel2(sel), v))
    ref = torch.stack([torch.stack([x[t].double() @ keys[sel[t, j]].double() for j in range(k)]) for t in range(T)])
    for o in outs:
        _check(o, ref)


@pytest.mark.parametrize("T,k,E,D,H,weights", [
    (60, 2, 16, 128, 256, "bf16"),    # few routes: the weights are read as they are stored
    (400, 2, 16, 128, 200, "fp32"),   # an output of no whole 64-column tiles
    (1400, 8, 7, 100, 512, "fp32")])  # padded copies
def test_no_scaled_rows_are_made_where_none_are_kept(T, k, E, D, H, weights):
    """A weighted route-input forward that trains the weights makes the
    tensors of one that does not: no [R, d_in] rows that nothing fills."""
    _, keys, sel = _case(T, k, E, D, H, "bf16", weights, False, D)
    x = torch.randn(T, k, D, device="cuda").to(torch.bfloat16)
    w = torch.rand(T, k, device="cuda")

    def made(kv):
        for _ in range(2):
            with torch.autocast("cuda", dtype=torch.bfloat16):
                s = C.cvmm_prepare_sel2(sel, w, route_input=True)
                before = torch.cuda.memory_stats()["allocation.all.allocated"]
                C.cvmm(x, s, kv)
            n = torch.cuda.memory_stats()["allocation.all.allocated"] - before
        return n

    training, frozen = made(keys.clone().requires_grad_()), made(keys)
    assert training == frozen


@pytest.mark.parametrize("weights", ["fp32", "bf16"])
@pytest.mark.parametrize("E,D,H", [(8, 136, 128), (64, 1024, 512)])   # weights below and from 2^25 values
def test_atomic_sums_over_stored_weights(monkeypatch, E, D, H, weights):
    """The top-k sum by atomics copies small weights and reads large ones in place."""
    monkeypatch.setattr(C, "cvmm_atomic_reduce", True)
    T, k = 9, 3
    _, keys, sel = _case(T, k, E, D, H, "bf16", weights, False, E)
    x = torch.randn(T, k, D, device="cuda").to(torch.bfloat16)
    w = torch.rand(T, k, device="cuda")
    plan = C._eager_plan(keys, torch.bfloat16, T * k, False, False, False, True)
    assert plan.stored == (keys.numel() >= 1 << 25)
    with torch.no_grad(), torch.autocast("cuda", dtype=torch.bfloat16):
        y = C.cvmm(x, C.cvmm_prepare_sel2(sel, w, route_input=True), keys)
    kd = keys.to(torch.bfloat16).double()
    ref = torch.stack([sum(w[t, j].double() * (x[t, j].double() @ kd[sel[t, j]]) for j in range(k)) for t in range(T)])
    _check(y, ref)
