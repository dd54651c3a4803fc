"""Projections whose widths are not multiples of 8, large enough for the
padded operand copies (16-bit op, >= 1.34e8 products per launch, >= 16 routes
per expert): each kernel the copies reach (long-K and short-K products,
narrow and wide outputs, the weight gradient's tiles), row ends of every
remainder, token and route input, weighted or not, fp32 x and weights and
16-bit ones, ids outside the range, against the oracle."""
import pytest
import torch

import cvmm_codex_amd.api as C
from cvmm_codex_amd import _native as N
from tests import gpu_util as U

pytestmark = pytest.mark.gpu

_DT = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


def _run(T, K, D, H, E, weighted, route_input, xdt, kdt, op, hot):
    g = torch.Generator().manual_seed(T + D + H)
    x = torch.randn(*((T, K, D) if route_input else (T, D)), generator=g).to(_DT[xdt])
    keys = (torch.randn(E, D, H, generator=g) / D ** 0.5).to(_DT[kdt])
    sel = torch.randint(0, E, (T, K), generator=g)
    if hot:
        sel[torch.rand(T, K, generator=g) < 0.6] = 0
    w = torch.rand(T, K, generator=g) if weighted else None
    go = torch.randn(*((T, H) if weighted else (T, K, H)), generator=g).to(_DT[op])
    got = U.run_hip(x, keys, sel, w, go, route_input, True, amp_dtype=_DT[op])
    exp = U.run_oracle(x, keys, sel, w, go, route_input, True,
                       amp_dtype="float16" if op == "fp16" else "bfloat16")
    U.compare(got, exp, 2e-2)


@pytest.mark.parametrize("T,K,D,H", [
    (700, 4, 412, 130),     # long-K both ways, partial last pieces
    (1400, 8, 201, 63),     # narrow output, 1-column tails
    (1400, 8, 63, 201),     # short-K forward, long-K grad-input
    (5200, 8, 100, 33),     # short-K both ways
    (700, 8, 136, 181),     # only d_out off the grid
    (700, 8, 181, 128),     # only d_in off the grid
    (400, 2, 523, 321),     # 256-wide weight-gradient tiles' range
    (1400, 8, 100, 512),    # short-K forward whose padded output fills whole 64-column tiles (the kernel
    (1400, 8, 60, 1024),    # that can keep scaled route rows: here p.K != d_in, none are kept)
    (1400, 8, 126, 1020),
    (1400, 8, 64, 1020),    # the same with only d_out off the grid
    (1024, 4, 33, 1001),    # a K <= 64 product over groups of column tiles (weighted)
    (700, 8, 100, 250),     # an unweighted forward that stays with the general kernel
])
@pytest.mark.parametrize("weighted,route_input", [(False, False), (True, True), (True, False), (False, True)])
def test_padded_widths(T, K, D, H, weighted, route_input):
    _run(T, K, D, H, 7, weighted, route_input, "bf16", "fp32", "bf16", False)


@pytest.mark.parametrize("xdt,kdt,op", [("fp32", "fp32", "bf16"), ("bf16", "bf16", "bf16"), ("fp16", "fp32", "fp16"),
                                        ("fp16", "fp16", "fp16")])
@pytest.mark.parametrize("weighted", [False, True])
def test_padded_widths_storage_types(xdt, kdt, op, weighted):
    _run(900, 4, 409, 131, 5, weighted, weighted, xdt, kdt, op, False)


def test_padded_widths_hot_expert_splits():
    _run(2100, 8, 203, 75, 16, True, True, "bf16", "fp32", "bf16", True)


def test_padded_gelu_and_unrouted_rows():
    T, K, D, H, E = 700, 4, 412, 130, 7
    g = torch.Generator().manual_seed(3)
    x = torch.randn(T, D, generator=g).to(torch.bfloat16).cuda().requires_grad_()
    keys = (torch.randn(E, D, H, generator=g) / D ** 0.5).cuda().requires_grad_()
    sel = torch.randint(0, E, (T, K), generator=g)
    sel[torch.rand(T, K, generator=g) < 0.2] = E
    gy = torch.randn(T, K, H, generator=g).to(torch.bfloat16).cuda()
    with torch.autocast("cuda", dtype=torch.bfloat16):
        y = C.cvmm_gelu(x, C.cvmm_prepare_sel2(sel.cuda()), keys)
        ref = torch.nn.functional.gelu(C.cvmm(x, C.cvmm_prepare_sel2(sel.cuda()), keys))
    out = (sel >= E).cuda()
    assert bool((y[out] == 0).all())
    got = torch.autograd.grad(y, [x, keys], gy)
    exp = torch.autograd.grad(ref, [x, keys], gy)
    assert U.norm_rel(U.to_np(y), U.to_np(ref)) <= 2e-2
    for a, b in zip(got, exp):
        assert U.norm_rel(U.to_np(a), U.to_np(b)) <= 2e-2


def test_padded_strided_keys():
    """Weights stored transposed and with gaps, x rows with a row stride."""
    T, K, D, H, E = 700, 4, 411, 133, 7
    g = torch.Generator().manual_seed(9)
    xb = torch.randn(T, D + 5, generator=g).to(torch.bfloat16).cuda()
    keys = (torch.randn(E, D, H, generator=g) / D ** 0.5).cuda()
    sel = torch.randint(0, E, (T, K), generator=g).cuda()
    outs = []
    for kv in (keys, keys.transpose(1, 2).contiguous().transpose(1, 2), torch.stack([keys, keys], -1)[..., 0]):
        xl = xb[:, 3:3 + D].detach().requires_grad_()
        with torch.autocast("cuda", dtype=torch.bfloat16):
            y = C.cvmm(xl, C.cvmm_prepare_sel2(sel), kv)
        outs.append((y, *torch.autograd.grad(y.float().square().sum(), [xl])))
    for o in outs[1:]:
        for a, b in zip(o, outs[0]):
            assert torch.equal(a, b)


def test_padded_rows_are_not_kept():
    """A stream's first weight gradient of a large odd width leaves its tile
    counters and partials allocated, not the padded operand rows."""
    T, K, D, H, E = 6000, 8, 900, 259, 16
    lib = N.lib()
    R = T * K
    kept = lib.cvmm_bwd_w_workspace_bytes(R, E, D, H, N.BF16, 1)
    assert lib.cvmm_bwd_w_rows_bytes(T, R, R, E, D, H, N.BF16, 0) > 32 << 20
    g = torch.Generator().manual_seed(4)
    x = torch.randn(T, D, generator=g).to(torch.bfloat16).cuda()
    keys = torch.randn(E, D, H, generator=g).cuda().requires_grad_()
    sel = torch.randint(0, E, (T, K), generator=g).cuda()
    gy = torch.randn(T, K, H, generator=g).to(torch.bfloat16).cuda()
    torch.cuda.synchronize()
    with torch.cuda.stream(torch.cuda.Stream()):
        before = torch.cuda.memory_allocated()
        with torch.autocast("cuda", dtype=torch.bfloat16):
            y = C.cvmm(x, C.cvmm_prepare_sel2(sel), keys)
        gk = torch.autograd.grad(y, keys, gy)[0]
        del y, gk
        torch.cuda.synchronize()
        held = torch.cuda.memory_allocated() - before
    # (beside it the sort's scratch, at most 1 MiB)
    assert held <= kept + (1 << 20) + 4096
