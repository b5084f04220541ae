"""Batched calls in which some tokens have no finite logit (the uninitialised
padding rows of a decode batch).

Such a token selects expert 0 in all of its k slots, as in the single-token op,
so expert 0 can have more pairs than the batch has tokens: up to B k.  The
other rows' outputs must not depend on that.  The workspace first holds another
call's routing, act and partial sums, so that a kernel that leaves without
writing its part shows.
"""
import ctypes

import pytest
import torch

from tests._helpers import assert_same_up_to_order

from warp_route import capi
from warp_route import functional as F
from warp_route.synthetic import make_layer

pytestmark = pytest.mark.gpu

WTAG = {torch.float32: capi.WR_F32, torch.float16: capi.WR_F16, torch.bfloat16: capi.WR_BF16,
        torch.float8_e4m3fn: capi.WR_FP8_E4M3, torch.float4_e2m1fn_x2: capi.WR_MXFP4}


def batched(x, gw, buf, E, h, I, k, ids, ws, work):
    out = torch.zeros_like(x)
    a = capi.WrMoeArgs()
    a.gate_w, a.weight_buf = gw.data_ptr(), buf.data_ptr()
    a.weight_bytes = buf.numel() * buf.element_size()
    a.weight_dtype = WTAG[buf.dtype]
    a.act_dtype = capi.WR_F16 if x.dtype == torch.float16 else capi.WR_F32
    a.num_experts, a.hidden_dim, a.intermediate_dim, a.top_k = E, h, I, k
    a.renormalize, a.batch_size = 1, x.shape[0]
    a.x, a.out, a.topk_ids, a.topk_weights = (t.data_ptr() for t in (x, out, ids, ws))
    a.workspace, a.workspace_bytes = work.data_ptr(), work.numel()
    st = capi.call("wr_batched_fused_moe", a, torch.cuda.current_stream(x.device).cuda_stream)
    assert st == capi.WR_OK, capi.status_str(st)
    return out


# B, k, bad rows: expert 0 gets more than 32 pairs at B <= 32 (34, 36, 40 and 62
# of them), more than 64 at B <= 64, more than 16 at B = 16; then the sizes whose
# class the counts choose.
@pytest.mark.parametrize("B,k,nbad", [(16, 6, 12), (17, 2, 16), (20, 2, 17), (20, 6, 6), (32, 2, 20),
                                      (32, 2, 31), (40, 2, 33), (80, 2, 70), (80, 6, 3)])
@pytest.mark.parametrize("h,I", [(256, 384), (520, 1190)], ids=["aligned", "ragged"])
@pytest.mark.parametrize("wd", WTAG, ids=["f32", "f16", "bf16", "fp8", "mxfp4"])
def test_rows_beside_nonfinite_tokens(cuda, wd, h, I, B, k, nbad):
    E = 8
    if wd == torch.float4_e2m1fn_x2:
        h, I = (h + 31) // 32 * 32, (I + 31) // 32 * 32
    x_dtype = torch.float16 if (B + k) % 4 else torch.float32
    x, gw, buf = make_layer(E, h, I, wd, router_std=h ** -0.5, expert_std=0.05, seed=B + k, batch=B,
                            device=cuda, x_dtype=x_dtype)
    work = torch.zeros(capi.lib().wr_workspace_bytes(capi.WR_KIND_BATCHED, E, h, I, k, B),
                       dtype=torch.uint8, device=cuda)
    ids = torch.empty(B, k, dtype=torch.int32, device=cuda)
    ws = torch.empty(B, k, dtype=torch.float32, device=cuda)
    batched(x.flip(0).contiguous(), gw, buf, E, h, I, k, ids, ws, work)
    bad = torch.randperm(B, generator=torch.Generator().manual_seed(B))[:nbad].tolist()
    for i, b in enumerate(bad):
        x[b, i % h] = float("nan") if i % 2 else float("inf")
        x[b, (i + 1) % h] = float("nan")
    print(f"[gpu] non-finite tokens {wd} {x_dtype} h={h} I={I} k={k} B={B}", flush=True)
    out = batched(x, gw, buf, E, h, I, k, ids, ws, work)
    torch.cuda.synchronize()
    assert ids[bad].eq(0).all()
    tol = (2e-3 if x_dtype == torch.float16 else
           5e-5 if wd in (torch.bfloat16, torch.float4_e2m1fn_x2) else 1e-5)
    for b in range(B):
        if b in bad:
            assert not torch.isfinite(out[b]).any(), b
            continue
        s_ids = torch.empty(k, dtype=torch.int32, device=cuda)
        single = F.fused_moe(x[b], gw, buf, E, h, I, k, True, s_ids)
        assert torch.equal(s_ids, ids[b]), b
        assert_same_up_to_order(out[b], single, f"row {b}", tol)
