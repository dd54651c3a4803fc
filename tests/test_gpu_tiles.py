"""The routed GEMMs' tile schedule at the expert counts where its form
changes (register-held offsets up to 256 experts, two passes beyond), with
empty experts and ids outside the expert range, against the oracle."""
import pytest
import torch

import cvmm_codex_amd.api as C
from cvmm_codex_amd import _native as N
from tests import gpu_util as U

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("E", [1, 64, 65, 255, 256, 257, 700])
@pytest.mark.parametrize("D,H", [(136, 72), (64, 192)])   # long-K and small-K products
def test_tile_schedule_over_expert_counts(E, D, H):
    g = torch.Generator().manual_seed(E)
    T, K = 301, 4
    x = torch.randn(T, D, generator=g).to(torch.bfloat16)
    keys = torch.randn(E, D, H, generator=g) / D ** 0.5
    sel = torch.randint(0, max(1, E * 3 // 4), (T, K), generator=g)   # a quarter of the experts empty
    sel[:, 0] = 0                                                     # one hot expert
    go = torch.randn(T, K, H, generator=g).to(torch.bfloat16)
    got = U.run_hip(x, keys, sel, None, go, False, True)
    exp = U.run_oracle(x, keys, sel, None, go, False, True)
    U.compare(got, exp, 2e-2)


@pytest.mark.parametrize("E", [64, 257])
def test_surplus_tiles_zero_the_unrouted_rows(E):
    g = torch.Generator().manual_seed(E)
    T, K, D, H = 130, 3, 136, 72
    x = torch.randn(T, D, generator=g).to(torch.bfloat16).cuda()
    keys = (torch.randn(E, D, H, generator=g) / D ** 0.5).cuda()
    sel = torch.randint(0, E, (T, K), generator=g)
    sel[torch.rand(T, K, generator=g) < 0.3] = E + 5
    with torch.autocast("cuda", dtype=torch.bfloat16):
        y = C.cvmm(x, C.cvmm_prepare_sel2(sel.cuda()), keys)
    out_of_range = (sel >= E).cuda()
    assert bool((y[out_of_range] == 0).all())
    e = sel.clamp(max=E - 1).cuda()
    ref = torch.einsum("td,tkdh->tkh", x.float(), keys.to(torch.bfloat16).float()[e])
    err = ((y.float() - ref)[~out_of_range].abs().max() / ref.abs().max()).item()
    assert err <= 2e-2


@pytest.mark.parametrize("E", [1, 5, 16])
@pytest.mark.parametrize("load", ["even", "one_long", "one_empty"])
def test_weight_gradient_chunk_order(E, load):
    # 400 routes per expert: below the loads whose chunks are ordered by length
    g = torch.Generator().manual_seed(E)
    T, K, D, H = 100 * E, 4, 136, 128
    sel = (torch.arange(T * K) % E).view(T, K)
    if load == "one_long":
        sel[torch.rand(T, K, generator=g) < 0.5] = E - 1
    elif load == "one_empty":
        sel[sel == 0] = E // 2
    x = torch.randn(T, D, generator=g).to(torch.bfloat16)
    keys = torch.randn(E, D, H, generator=g) / D ** 0.5
    go = torch.randn(T, K, H, generator=g).to(torch.bfloat16)
    got = U.run_hip(x, keys, sel, None, go, False, True)
    exp = U.run_oracle(x, keys, sel, None, go, False, True)
    U.compare(got, exp, 2e-2)


def _dw64(x, ids, go, E):
    """dW[e] = sum over the routes of e of x^T go in float64."""
    order = torch.argsort(ids.reshape(-1), stable=True)
    rows = x.double()[order // ids.shape[1]].split(torch.bincount(ids.reshape(-1), minlength=E).tolist())
    g = go.double().reshape(-1, go.shape[-1])[order].split([r.shape[0] for r in rows])
    return torch.stack([a.T @ b for a, b in zip(rows, g)])


@pytest.mark.parametrize("E", [8, 9, 16, 64, 65, 128, 200, 256, 257])
@pytest.mark.parametrize("load,chunk", [("even", 0), ("uneven", 0), ("uneven", 256), ("one_long", 512)])
def test_weight_gradient_chunks_by_length(E, load, chunk):
    """800 routes per expert: with 9 to 256 experts of uneven loads the chunks
    run longest first (the rank spans one to four waves), split experts among
    them; other launches in expert order.  The bits of the tile-major order,
    which never sorts, and float64's sums within fp32's rounding of ~800
    terms."""
    g = torch.Generator().manual_seed(E)
    K, D, H = 4, 72, 136
    T = 200 * E
    ids = (torch.arange(T * K) % E).view(T, K)
    if load == "uneven":
        ids = torch.multinomial(1 + 1.5 * torch.rand(E, generator=g), T * K, replacement=True, generator=g).view(T, K)
        ids[ids == 1] = 0          # an empty expert
    elif load == "one_long":
        ids[torch.rand(T, K, generator=g) < 0.3] = E // 2
    x = torch.randn(T, D, generator=g).to(torch.bfloat16).cuda()
    keys = torch.randn(E, D, H, generator=g).cuda().requires_grad_()
    go = torch.randn(T, K, H, generator=g).to(torch.bfloat16).cuda()
    ids = ids.cuda()
    lib = N.lib()
    out = []
    assert lib.cvmm_tuning_set(N.TUNE_WGRAD_CHUNK, chunk) == 0
    try:
        for order in (0, 2):
            assert lib.cvmm_tuning_set(N.TUNE_WGRAD_ORDER, order) == 0
            with torch.autocast("cuda", dtype=torch.bfloat16):
                y = C.cvmm(x, C.cvmm_prepare_sel2(ids), keys)
            out.append(torch.autograd.grad(y, keys, go)[0])
    finally:
        lib.cvmm_tuning_set(N.TUNE_WGRAD_ORDER, 0)
        lib.cvmm_tuning_set(N.TUNE_WGRAD_CHUNK, 0)
    assert torch.equal(out[0], out[1])
    ref = _dw64(x, ids, go, E)
    assert ((out[0].double() - ref).abs().max() / ref.abs().max()).item() <= 1e-5


@pytest.mark.parametrize("T,k,E,D,H", [(64, 2, 8, 64, 1000), (300, 2, 8, 40, 136), (1024, 4, 8, 64, 2008),
                                       (40, 1, 70, 24, 520)])
def test_short_products_over_groups_of_column_tiles(T, k, E, D, H):
    """K <= 64 and N off the 64-column grid: the workgroups of a launch with
    few row tiles share out its column tiles."""
    g = torch.Generator().manual_seed(T + H)
    x = torch.randn(T, k, D, generator=g).to(torch.bfloat16)
    keys = torch.randn(E, D, H, generator=g) / D ** 0.5
    ids = torch.randint(0, E, (T, k), generator=g)
    w = torch.rand(T, k, generator=g)
    go = torch.randn(T, H, generator=g).to(torch.bfloat16)
    got = U.run_hip(x, keys, ids, w, go, True, True)
    exp = U.run_oracle(x, keys, ids, w, go, True, True)
    U.compare(got, exp, 2e-2)
