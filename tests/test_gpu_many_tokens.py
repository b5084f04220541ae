"""GPU parity of batched calls with more than 64 tokens on an expert.  With more
than 32 (fp16, bf16), 48 (fp8) or 80 (MXFP4) pairs per expert on average the
many-token kernels (k_many_gu, k_many_dn) take them in equal passes of up to 160
tokens, five 16-token tiles per wave; else the 64-token kernels do, 64 per pass.

Batch sizes put an expert's count at, just below and just above each number of
tiles, the 64-token kernels' limit and one pass, so that every instantiation
and the second pass run, and the average at and just above each of its bounds.  Rows are checked against the oracle (a sample) and
against the single-token op (all: identical ids, outputs equal up to summation
order, 1e-5 of max|out|; bf16 and MXFP4 weights, whose batched operands are two
bf16 terms within 2^-18, at 5e-5, as for the smaller tiles); two calls agree
bit for bit.
"""
import pytest
import torch

from tests._helpers import assert_parity, assert_same_up_to_order, oracle_token

from warp_route import functional as F
from warp_route.synthetic import clustered_batch, make_layer

pytestmark = pytest.mark.gpu

F32, F16 = torch.float32, torch.float16
BF16, FP8, MX4 = torch.bfloat16, torch.float8_e4m3fn, torch.float4_e2m1fn_x2
WTYPES = {"f16": F16, "bf16": BF16, "fp8": FP8, "mxfp4": MX4}


@pytest.mark.parametrize("x_dtype", [F32, F16], ids=["xf32", "xf16"])
# Clustered on one pair of experts: close to B tokens on each.  E = 2 with
# k = 2: exactly B on both.  E = 8, k = 2: the average is B / 4.
@pytest.mark.parametrize("E,B", [(2, 65), (2, 81), (2, 96), (2, 97), (2, 128), (2, 129), (2, 160),
                                 (2, 161), (2, 321), (8, 128), (8, 129), (8, 192), (8, 193),
                                 (8, 200), (8, 320), (8, 321)])
@pytest.mark.parametrize("wd", WTYPES)
def test_many_tokens_every_row(cuda, wd, E, B, x_dtype):
    h, I, k, rn = (384, 640, 2, True) if B % 2 else (512, 256, 2, False)
    x, gw, buf = make_layer(E, h, I, WTYPES[wd], router_std=h ** -0.5, expert_std=0.05, seed=B,
                            batch=B, device=cuda, x_dtype=x_dtype)
    if E > 2:
        x = clustered_batch(gw, B, pair=(1, 6), alpha=4.0, seed=B, device=cuda).to(x_dtype)
    ids = torch.empty(B, k, dtype=torch.int32, device=cuda)
    ws = torch.empty(B, k, dtype=torch.float32, device=cuda)
    print(f"[gpu] many tokens {wd} {x_dtype} E={E} B={B}", flush=True)
    out = F.batched_fused_moe(x, gw, buf, E, h, I, k, rn, ids, ws)
    again = F.batched_fused_moe(x, gw, buf, E, h, I, k, rn)
    torch.cuda.synchronize()
    assert torch.equal(out, again)
    assert torch.bincount(ids.flatten().long()).max() > 64
    singles = []
    for b in range(B):
        s_ids = torch.empty(k, dtype=torch.int32, device=cuda)
        singles.append(F.fused_moe(x[b], gw, buf, E, h, I, k, rn, s_ids))
        assert torch.equal(s_ids, ids[b]), f"row {b} selection"
    tol = 2e-3 if x_dtype == F16 else 5e-5 if wd in ("bf16", "mxfp4") else 1e-5
    for b in range(B):
        assert_same_up_to_order(out[b], singles[b], f"{wd} E={E} B={B} row {b}", tol)
    for b in (0, 63, 64, B - 1):
        ref = oracle_token(x[b], gw, buf, E, h, I, k, rn)
        if ref["robust"]:
            assert_parity(out[b], ids[b], ws[b], ref, rel_tol=2e-3 if x_dtype == F16 else 1e-4,
                          label=f"{wd} E={E} B={B} row {b}")


def test_many_tokens_long_act_rows(cuda):
    """A pass whose act rows end more than 4 GiB past its first: the many-token
    kernels' 32-bit offsets do not reach, the 64-token kernels take the call."""
    E, h, I, k, B = 1, 128, 52864 * 128, 1, 160
    assert 160 * I * 4 > 159 * I * 4 > 1 << 32
    gen = torch.Generator(device=cuda).manual_seed(5)
    lay = F.weight_layout(E, h, I, MX4)
    buf = F.zeros_weights(lay["expert_stride"], MX4, cuda)
    raw = buf.view(torch.uint8)
    for part in raw.split(1 << 26):
        part.copy_(torch.randint(0, 256, (part.numel(),), generator=gen, device=cuda,
                                 dtype=torch.uint8))
    raw[lay["scale_offset"]:].fill_(122)  # 2^-5
    x = torch.randn(B, h, generator=gen, device=cuda)
    gw = torch.randn(E, h, generator=gen, device=cuda) * h ** -0.5
    print("[gpu] many tokens, act rows of 26 MiB", flush=True)
    out = F.batched_fused_moe(x, gw, buf, E, h, I, k)
    for b in (0, 63, 64, 127, 158, 159):
        single = F.fused_moe(x[b], gw, buf, E, h, I, k)
        torch.cuda.synchronize()
        # fp32 sums of 6.8 million columns, in other orders.
        assert_same_up_to_order(out[b], single, f"row {b}", 1e-3)
