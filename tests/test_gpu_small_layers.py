"""GPU parity of single-token layers of about one block per CU.

Up to one gate/up and down block per CU the single-token kernel takes the
router inside; larger register-path layers keep the router launch (up to two
gate/up blocks per CU).  Shapes lie on both sides of that line (h / 4 down
blocks and 32-block groups of gate/up chunks against 256 CUs), with more
experts than wave lanes of a row and rows that only one-element loads take.
Selection and output are checked against the oracle, for new tokens one after
the other and for replays of a captured call.
"""
import pytest
import torch

from tests._helpers import assert_parity, oracle_rows

from warp_route import functional as F
from warp_route.synthetic import make_layer

pytestmark = pytest.mark.gpu

SHAPES = [(8, 256, 512, 2), (64, 256, 512, 6), (64, 16, 32, 1), (8, 512, 512, 2),
          (8, 516, 512, 2), (8, 896, 128, 1), (16, 512, 1024, 2), (7, 37, 101, 3),
          (64, 130, 250, 6)]


@pytest.mark.parametrize("xd", [torch.float32, torch.float16], ids=["xf32", "xf16"])
@pytest.mark.parametrize("shape", SHAPES, ids=["-".join(map(str, s)) for s in SHAPES])
def test_small_layer_token(cuda, shape, xd):
    E, h, I, k = shape
    print(f"[gpu] small layer {shape} {xd}", flush=True)
    tol = 2e-3 if xd == torch.float16 else 1e-4
    xs, gw, buf = make_layer(E, h, I, router_std=h ** -0.5, expert_std=0.05, seed=E + h + I, batch=4,
                             device=cuda, x_dtype=xd)
    rows = oracle_rows(xs, gw, buf, E, h, I, k, True)
    ids = torch.empty(k, dtype=torch.int32, device=cuda)
    ws = torch.empty(k, dtype=torch.float32, device=cuda)
    for x, row in zip(xs, rows):
        out = F.fused_moe(x, gw, buf, E, h, I, k, True, ids, ws)
        torch.cuda.synchronize()
        if row["robust"]:
            assert_parity(out, ids, ws, row, rel_tol=tol, label=f"{shape}")
    assert sum(r["robust"] for r in rows) >= 2
    x = xs[0].clone()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = F.fused_moe(x, gw, buf, E, h, I, k, True, ids, ws)
    for src, row in zip(xs, rows):
        x.copy_(src)
        eager = F.fused_moe(x, gw, buf, E, h, I, k, True)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager)
        if row["robust"]:
            assert_parity(out, ids, ws, row, rel_tol=tol, label=f"{shape} replay")
