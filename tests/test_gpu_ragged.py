"""GPU parity of layers whose sizes are multiples of nothing.

Rows that are not whole, aligned 16-byte pieces (or, for batched calls, whole K
steps) are loaded with unaligned loads clamped to the row's end.  The
single-token and per-token kernels mask the columns that a clamped piece
repeats; the batched MFMA kernels (k_rag_gu, k_rag_dn) shift it into place.
Every row of every batched case is checked against the oracle and against the
single-token op (identical ids and weights, outputs equal up to summation
order: 1e-5 of max|out|, as for aligned layers; bf16 and MXFP4 weights too,
since ragged rows take x and act in three 16-bit terms, within 2^-24 of them).
"""
import pytest
import torch

from tests._helpers import assert_parity, assert_same_up_to_order, oracle_rows

from warp_route import functional as F
from warp_route.synthetic import make_layer

pytestmark = pytest.mark.gpu

F32, F16 = torch.float32, torch.float16
BF16, FP8, MX4 = torch.bfloat16, torch.float8_e4m3fn, torch.float4_e2m1fn_x2
WTYPES = [F32, F16, BF16, FP8, MX4]
WIDS = ["f32", "f16", "bf16", "fp8", "mxfp4"]


def check(x, gw, buf, E, h, I, k, rn, label):
    B = x.shape[0]
    ids = torch.empty(B, k, dtype=torch.int32, device=x.device)
    ws = torch.empty(B, k, dtype=torch.float32, device=x.device)
    print(f"[gpu] ragged {label}", flush=True)
    out = F.batched_fused_moe(x, gw, buf, E, h, I, k, rn, ids, ws)
    again = F.batched_fused_moe(x, gw, buf, E, h, I, k, rn)
    torch.cuda.synchronize()
    assert torch.equal(out, again)
    rows = oracle_rows(x, gw, buf, E, h, I, k, rn)
    robust = 0
    for b in range(B):
        s_ids = torch.empty(k, dtype=torch.int32, device=x.device)
        s_ws = torch.empty(k, dtype=torch.float32, device=x.device)
        single = F.fused_moe(x[b], gw, buf, E, h, I, k, rn, s_ids, s_ws)
        assert torch.equal(s_ids, ids[b]) and torch.equal(s_ws, ws[b]), f"{label} row {b} selection"
        assert_same_up_to_order(out[b], single, label=f"{label} row {b} vs single-token op")
        if rows[b]["robust"]:
            robust += 1
            assert_parity(out[b], ids[b], ws[b], rows[b],
                          rel_tol=2e-3 if x.dtype == F16 else 1e-4, label=f"{label} row {b}")
    assert 2 * robust >= B, f"{label}: {robust} of {B} rows robust"


# h and I: around one 16-byte piece, one below / above whole K steps of 64 and
# 128, odd, one of the two aligned; then layers large enough for the batched
# kernels from B = 16 on, and some at B = 2 (the small ones take them at the larger
# B and for the narrower types only).
SHAPES = [(8, 32, 96, 2), (5, 127, 129, 2), (20, 72, 40, 6), (8, 264, 520, 2),
          (2, 1151, 1025, 2), (3, 1025, 1151, 3), (2, 2047, 1536, 1), (2, 1536, 1990, 2),
          (12, 500, 1258, 3)]


def of_type(shape, wd):
    """MXFP4 rows are whole blocks of 32."""
    E, h, I, k = shape
    return (E, (h + 31) // 32 * 32, (I + 31) // 32 * 32, k) if wd == MX4 else shape


@pytest.mark.parametrize("B", [2, 16, 17, 70])
@pytest.mark.parametrize("shape", SHAPES, ids=["-".join(map(str, s)) for s in SHAPES])
@pytest.mark.parametrize("wd", WTYPES, ids=WIDS)
def test_ragged_batched_every_row(cuda, wd, shape, B):
    E, h, I, k = of_type(shape, wd)
    x_dtype = F16 if (h + B) % 2 else F32
    x, gw, buf = make_layer(E, h, I, wd, router_std=h ** -0.5, expert_std=0.05, seed=B, batch=B,
                            device=cuda, x_dtype=x_dtype)
    check(x, gw, buf, E, h, I, k, B % 2 == 0, f"{wd} {x_dtype} E={E} h={h} I={I} k={k} B={B}")


@pytest.mark.parametrize("hI", [(264, 520), (1025, 1415)], ids=str)
@pytest.mark.parametrize("wd", WTYPES, ids=WIDS)
def test_ragged_batched_error(cuda, wd, hI):
    """The batched kernels' sums are no further from 64 bits than the
    single-token op's.  The ratio of the two errors (2-norms over 96 rows, each
    row's error an independent sum of roundings) varies by a few per cent from
    seed to seed; the bound of 1.15 is above that, and below the 1.3 to 1.8 of a
    single chain of sums through a K step."""
    E, h, I, k = of_type((2, *hI, 1), wd)
    B = 96
    x, gw, buf = make_layer(E, h, I, wd, router_std=h ** -0.5, seed=h, batch=B, device=cuda)
    print(f"[gpu] ragged error {wd} h={h} I={I}", flush=True)
    out = F.batched_fused_moe(x, gw, buf, E, h, I, k, True)
    single = torch.stack([F.fused_moe(row, gw, buf, E, h, I, k, True) for row in x])
    torch.cuda.synchronize()
    ref = torch.stack([torch.from_numpy(r["out"])
                       for r in oracle_rows(x, gw, buf, E, h, I, k, True)])
    err, err_single = ((t.cpu().double() - ref).norm().item() for t in (out, single))
    assert err <= 1.15 * err_single, (err, err_single)


@pytest.mark.parametrize("x_dtype", [F32, F16], ids=["xf32", "xf16"])
@pytest.mark.parametrize("hI", [(15, 40), (17, 33), (255, 257), (257, 515), (770, 255), (260, 1030),
                                (1031, 261), (2049, 77), (77, 2049), (3001, 1027)], ids=str)
@pytest.mark.parametrize("wd", WTYPES, ids=WIDS)
def test_ragged_single_token(cuda, wd, hI, x_dtype):
    """One token: rows shorter than one piece, around the bounds between single
    elements and pieces (half a wave of pieces on average; fp8 a quarter for the
    shorter row), and of several rounds."""
    E, h, I, k = of_type((6, *hI, 3), wd)
    for seed in range(50):
        x, gw, buf = make_layer(E, h, I, wd, router_std=h ** -0.5, expert_std=0.05, seed=seed,
                                device=cuda, x_dtype=x_dtype)
        ref = oracle_rows(x.reshape(1, h), gw, buf, E, h, I, k, True)[0]
        if ref["robust"]:
            break
    ids = torch.empty(k, dtype=torch.int32, device=cuda)
    ws = torch.empty(k, dtype=torch.float32, device=cuda)
    print(f"[gpu] ragged token {wd} {x_dtype} h={h} I={I}", flush=True)
    out = F.fused_moe(x, gw, buf, E, h, I, k, True, ids, ws)
    torch.cuda.synchronize()
    assert_parity(out, ids, ws, ref, rel_tol=2e-3 if x_dtype == F16 else 1e-4, label=f"{wd} {hI}")


@pytest.mark.parametrize("what", ["weights", "x", "router"])
@pytest.mark.parametrize("wd", WTYPES, ids=WIDS)
def test_unaligned_pointers_of_aligned_sizes(cuda, wd, what):
    """The same kernels serve aligned sizes behind pointers that are not
    16-byte aligned (views into larger tensors)."""
    E, h, I, k, B = 4, 1152, 1280, 2, 20
    x, gw, buf = make_layer(E, h, I, wd, router_std=h ** -0.5, expert_std=0.05, seed=3, batch=B,
                            device=cuda)

    def off_by_one(t):
        flat = torch.empty(t.numel() + 1, dtype=torch.uint8 if t.element_size() == 1 else t.dtype,
                           device=cuda).view(t.dtype)
        v = flat[1:].view(t.shape)
        assert v.data_ptr() % 16 != 0
        (v.view(torch.uint8) if t.element_size() == 1 else v).copy_(
            t.view(torch.uint8) if t.element_size() == 1 else t)
        return v

    if what == "weights":
        buf = off_by_one(buf)
    elif what == "x":
        x = off_by_one(x)
    else:
        gw = off_by_one(gw)
    check(x, gw, buf, E, h, I, k, True, f"{wd} unaligned {what}")


@pytest.mark.parametrize("bad", [float("inf"), float("nan")], ids=["inf", "nan"])
@pytest.mark.parametrize("matrix", ["gate", "up", "down"])
@pytest.mark.parametrize("wd", [F32, F16, BF16, FP8], ids=WIDS[:4])
def test_ragged_rows_do_not_leak(cuda, wd, matrix, bad):
    """A non-finite weight reaches only the outputs that its row takes part in,
    exactly as in the single-token op: at the first column of a row, where the
    last K step of the row before it loads past that row's end, and at the end of
    the last row, which the rows past it in its tile repeat."""
    if wd == FP8 and bad == float("inf"):
        pytest.skip("E4M3 has no infinity")
    E, h, I, k, B = 4, 1131, 1077, 2, 20
    x, gw, buf = make_layer(E, h, I, wd, router_std=h ** -0.5, expert_std=0.05, seed=4, batch=B,
                            device=cuda)
    stride = buf.numel() // E
    n = h * I
    rows, cols = (h, I) if matrix == "down" else (I, h)
    base = ["gate", "up", "down"].index(matrix) * n
    # Expert 0: row 40, first column; expert 1: last row and column.
    for at in (0 * stride + base + 40 * cols, 1 * stride + base + rows * cols - 1):
        if wd == FP8:
            buf.view(torch.uint8)[at] = 0x7F  # NaN
        else:
            buf[at] = bad
    ids = torch.empty(B, k, dtype=torch.int32, device=cuda)
    print(f"[gpu] ragged leak {wd} {matrix} {bad}", flush=True)
    out = F.batched_fused_moe(x, gw, buf, E, h, I, k, False, ids)
    for b in range(B):
        single = F.fused_moe(x[b], gw, buf, E, h, I, k)
        torch.cuda.synchronize()
        assert torch.equal(torch.isfinite(out[b]), torch.isfinite(single)), b
    assert (~torch.isfinite(out)).any()
    clean = (ids >= 2).all(dim=1)
    assert clean.any() and torch.isfinite(out[clean]).all()
