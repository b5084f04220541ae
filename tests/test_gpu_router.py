"""GPU parity of the router and selection kernel (gate_topk) over its variants:
one, two and four experts per wave and round (up to 4, up to 8 and more experts),
one and two tokens per block (the second from one token per CU on), and router
rows in 16-byte pieces or single elements, shorter and longer than a block's
first round.

Ids and weights are those of the single-token op bit for bit (the same sums in
the same order), and the oracle's where rounding cannot change the selection.
"""
import pytest
import torch

from tests._helpers import f64

from oracle import moe_oracle as O
from warp_route import functional as F
from warp_route.synthetic import make_layer

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B", [1, 5, 257, 300])
@pytest.mark.parametrize("h", [37, 1000, 7168])
@pytest.mark.parametrize("E", [1, 2, 3, 4, 5, 7, 8, 9, 17, 64])
def test_gate_topk_variants(cuda, E, h, B):
    k, I, rn = min(E, 1 + E % 6), 8, bool(E % 2)
    xd = torch.float16 if (E + B) % 2 else torch.float32
    x, gw, buf = make_layer(E, h, I, router_std=h ** -0.5, seed=E + B, batch=B, device=cuda,
                            x_dtype=xd)
    print(f"[gpu] gate_topk E={E} h={h} B={B} {xd}", flush=True)
    ids, ws = F.gate_topk(x, gw, E, h, k, rn)
    torch.cuda.synchronize()
    rows = sorted({0, 1, B // 2, B - 2, B - 1} & set(range(B)))
    for b in rows:
        s_ids = torch.empty(k, dtype=torch.int32, device=cuda)
        s_ws = torch.empty(k, dtype=torch.float32, device=cuda)
        F.fused_moe(x[b], gw, buf, E, h, I, k, rn, s_ids, s_ws)
        assert torch.equal(s_ids, ids[b]) and torch.equal(s_ws, ws[b]), b
        if O.selection_is_robust(f64(gw), f64(x[b]), k):
            _, want, w = O.softmax_topk((f64(gw) @ f64(x[b])).astype("float32"), k, rn)
            assert ids[b].cpu().tolist() == want.tolist(), b
            assert abs(ws[b].cpu().double().numpy() - w).max() < 1e-5, b


# Either side of the line between the selection in the grouping launch and in the
# router launch: E <= 16 at 64 tokens, more experts at 24 + E h / 6144 (24, 32 and
# 64 here) tokens.
@pytest.mark.parametrize("E,h,B", [(16, 256, 64), (16, 256, 65), (17, 256, 24), (17, 256, 25),
                                   (64, 768, 32), (64, 768, 33), (64, 4096, 64), (64, 4096, 65)])
def test_batched_selection_is_gate_topk(cuda, E, h, B):
    k, I = 6, 128
    for xd in (torch.float32, torch.float16):
        x, gw, buf = make_layer(E, h, I, torch.float16, router_std=h ** -0.5, seed=B, batch=B,
                                device=cuda, gen_device=cuda, x_dtype=xd)
        want_ids, want_ws = F.gate_topk(x, gw, E, h, k, True)
        ids, ws = torch.empty_like(want_ids), torch.empty_like(want_ws)
        print(f"[gpu] batched selection E={E} h={h} B={B} {xd}", flush=True)
        F.batched_fused_moe(x, gw, buf, E, h, I, k, True, ids, ws)
        torch.cuda.synchronize()
        assert torch.equal(ids, want_ids) and torch.equal(ws, want_ws)
