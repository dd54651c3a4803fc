"""fp32 projections on the DMA-staged matrix-core kernels (from 1e8 products per
launch): partial k slices, partial column tiles, narrow outputs, empty and hot
experts, both weight orientations, weighted and not, the routing-weight
gradient, a split weight gradient; against the oracle in float64 at 1e-5 of
the largest value (fp32 sums of up to ~5000 terms: sqrt(5000) * 2^-24 = 4e-6
of the result's scale)."""
import pytest
import torch

import cvmm_codex_amd.api as C
from cvmm_codex_amd import _native as N
from tests import gpu_util as U

pytestmark = pytest.mark.gpu


def _run(T, K, D, H, E, weighted, route_input, hot=False, empty=False):
    g = torch.Generator().manual_seed(T + D + H + E)
    x = torch.randn(*((T, K, D) if route_input else (T, D)), generator=g)
    keys = torch.randn(E, D, H, generator=g) / D ** 0.5
    sel = torch.randint(0, max(1, E // 2) if empty else E, (T, K), generator=g)
    if hot:
        sel[torch.rand(T, K, generator=g) < 0.7] = E - 1
    w = torch.rand(T, K, generator=g) if weighted else None
    go = torch.randn(*((T, H) if weighted else (T, K, H)), generator=g)
    got = U.run_hip(x, keys, sel, w, go, route_input, False)
    exp = U.run_oracle(x, keys, sel, w, go, route_input, False)
    U.compare(got, exp, 1e-5)


@pytest.mark.parametrize("T,K,D,H,E", [
    (1030, 2, 1024, 64, 8),     # narrow output, one column tile
    (517, 8, 260, 132, 16),     # partial slices and tiles both ways
    (2100, 8, 132, 60, 5),      # narrow and partial
    (3000, 2, 68, 300, 3),      # few experts, many rows each
    (1200, 4, 36, 640, 9),      # short k
    (700, 1, 512, 512, 4),      # top-1
    (4100, 8, 64, 64, 33),      # 64 x 64 weight blocks
])
@pytest.mark.parametrize("weighted,route_input", [(False, False), (True, True), (True, False)])
def test_f32_projection(T, K, D, H, E, weighted, route_input):
    _run(T, K, D, H, E, weighted, route_input)


@pytest.mark.parametrize("weighted", [False, True])
def test_f32_empty_and_hot_experts(weighted):
    _run(600, 8, 256, 128, 70, weighted, weighted, hot=True, empty=True)


@pytest.mark.parametrize("D,H", [(512, 96), (96, 512), (260, 60)])
def test_f32_split_weight_gradient(D, H):
    lib = N.lib()
    assert lib.cvmm_tuning_set(N.TUNE_WGRAD_CHUNK, 256) == 0
    try:
        _run(max(700, 26_000_000 // (D * H)), 4, D, H, 4, False, False, hot=True)  # (>= 1e8 products)
        _run(700, 4, D, H, 4, True, False, hot=True)
    finally:
        lib.cvmm_tuning_set(N.TUNE_WGRAD_CHUNK, 0)


@pytest.mark.parametrize("chunk", [0, 32])
@pytest.mark.parametrize("weighted", [False, True])
def test_f32_weight_gradient_of_128_wide_tiles(weighted, chunk):
    """Eight 128 x 128 tiles per CU (512 experts of 256 x 256), whole experts
    and experts in chunks of 32 routes."""
    lib = N.lib()
    assert lib.cvmm_tuning_set(N.TUNE_WGRAD_CHUNK, chunk) == 0
    try:
        _run(500, 4, 256, 256, 512, weighted, weighted, hot=True)
    finally:
        lib.cvmm_tuning_set(N.TUNE_WGRAD_CHUNK, 0)


@pytest.mark.parametrize("E,R,D,H", [(1, 720, 512, 512), (2, 4096, 512, 256), (5, 4096, 132, 260), (9, 720, 512, 512),
                                     (63, 8192, 132, 132), (64, 8192, 132, 132)])
def test_f32_weight_gradient_orders(E, R, D, H):
    """Below 64 experts the tiles of a chunk spread over the XCDs, from there
    chunks are dealt to them; few routes per expert are split from 256 on.
    Both orders' bits are the same, and the built-in one's."""
    g = torch.Generator().manual_seed(E)
    x = torch.randn(R // 4, D, generator=g).cuda()
    keys = torch.randn(E, D, H, generator=g).cuda().requires_grad_()
    p = torch.arange(1, E + 1.).pow(-0.7)
    ids = torch.multinomial(p, R, replacement=True, generator=g).view(-1, 4).cuda()
    go = torch.randn(R // 4, 4, H, generator=g).cuda()
    lib = N.lib()
    y = C.cvmm(x, C.cvmm_prepare_sel2(ids), keys)
    out = []
    try:
        for order in (0, 1, 3):
            assert lib.cvmm_tuning_set(N.TUNE_WGRAD_ORDER, order) == 0
            out.append(torch.autograd.grad(y, keys, go, retain_graph=True)[0])
    finally:
        lib.cvmm_tuning_set(N.TUNE_WGRAD_ORDER, 0)
    assert torch.equal(out[0], out[1]) and torch.equal(out[0], out[2])
    rows = x.double().repeat_interleave(4, 0)
    flat, gd = ids.reshape(-1), go.double().reshape(R, H)
    ref = torch.stack([rows[flat == e].T @ gd[flat == e] for e in range(E)])
    assert ((out[0].double() - ref).abs().max() / ref.abs().max()).item() <= 1e-5


def test_f32_transposed_keys_and_unrouted_ids():
    T, K, D, H, E = 900, 4, 256, 136, 6
    g = torch.Generator().manual_seed(1)
    x = torch.randn(T, D, generator=g).cuda()
    keys = (torch.randn(E, D, H, generator=g) / D ** 0.5).cuda()
    sel = torch.randint(0, E, (T, K), generator=g)
    sel[torch.rand(T, K, generator=g) < 0.2] = E + 1
    res = []
    for kv in (keys, keys.transpose(1, 2).contiguous().transpose(1, 2)):
        xl = x.clone().requires_grad_()
        y = C.cvmm(xl, C.cvmm_prepare_sel2(sel.cuda()), kv)
        res.append((y, *torch.autograd.grad(y.square().sum(), [xl])))
    assert bool((res[0][0][(sel >= E).cuda()] == 0).all())
    for a, b in zip(*res):
        assert U.norm_rel(U.to_np(a), U.to_np(b)) <= 1e-5
