"""The screened split encode gives fm_rvq_encode_split's codes bit for bit."""

from __future__ import annotations

import pytest
import torch

from fast_mimi_amd import _native as nat

pytestmark = pytest.mark.gpu
DEV = "cuda"


def encode(x, embeds, norms, embeds_t, nsem, T, screened):
    n, e, d = embeds.shape
    rows = x.shape[0]
    st = torch.cuda.current_stream().cuda_stream
    codes = torch.full((rows // T, n, T), -1, dtype=torch.int64, device=DEV)
    wsb = nat.library().fm_rvq_split_workspace_bytes(rows, d, e)
    ws = torch.empty((wsb + 3) // 4, device=DEV)
    args = [x.data_ptr(), x.shape[1], rows, T, d, e, nsem, n - nsem, embeds.data_ptr()]
    if screened:
        planes = torch.empty(n * e * d, dtype=torch.float16, device=DEV)
        info = torch.empty(n, 2, dtype=torch.int32, device=DEV)
        nat.call("fm_rvq_prepare_screen", embeds.data_ptr(), norms.data_ptr(), e, d, n, planes.data_ptr(),
                 info.data_ptr(), st)
        nat.call("fm_rvq_encode_split_screened", *args, norms.data_ptr(), planes.data_ptr(), info.data_ptr(),
                 codes.data_ptr(), n * T, st)
    else:
        nat.call("fm_rvq_encode_split", *args, embeds_t.data_ptr(), norms.data_ptr(), codes.data_ptr(), n * T,
                 ws.data_ptr(), wsb, st)
    torch.cuda.synchronize()
    return codes.cpu()


def books(emb):
    norms = emb.pow(2).sum(-1).contiguous()
    return emb.to(DEV), norms.to(DEV), emb.transpose(1, 2).contiguous().to(DEV)


@pytest.mark.parametrize("B,T,nsem,n,e", [(1, 1025, 1, 8, 2048), (16, 125, 1, 8, 2048), (3, 2700, 1, 32, 2048),
                                          (1, 2100, 2, 5, 1024), (2, 600, 0, 3, 2048), (2, 600, 3, 3, 2048),
                                          (1, 16400, 1, 4, 96), (1, 32800, 1, 2, 32), (1, 8300, 1, 3, 2048),
                                          (205, 5, 1, 3, 2048)])
def test_codes_equal_step_launches(B, T, nsem, n, e):
    g = torch.Generator().manual_seed(B * T + n + e)
    emb, norms, emb_t = books(torch.randn(n, e, 256, generator=g) / 16)
    x = (torch.randn(B * T, 512, generator=g) * torch.exp(torch.randn(B * T, 1, generator=g))).to(DEV)
    want = encode(x, emb, norms, emb_t, nsem, T, False)
    assert torch.equal(encode(x, emb, norms, emb_t, nsem, T, True), want)


HARD = ["ties", "cluster", "tiny", "huge", "zero_rows", "bad_rows", "bad_book", "mixed", "on_entries", "zero_book",
        "offset"]


@pytest.mark.parametrize("kind,e,rows", [(k, 2048, 1300) for k in HARD] +
                         [(k, e, rows) for k in ("cluster", "offset") for e, rows in ((1024, 2049), (512, 4100),
                                                                                     (32, 32769))])
def test_hard_inputs(kind, e, rows):
    """Equal and nearly equal entries, rows that are entries, scales near both
    ends of FP32, zero and non-finite rows and codebooks; near-ties also at the
    fewest rows a smaller codebook is accepted with."""
    g = torch.Generator().manual_seed(len(kind))
    n = 4
    emb = torch.randn(n, e, 256, generator=g) / 16
    x = torch.randn(rows, 512, generator=g)
    if kind == "ties":
        emb[:, 1024:] = emb[:, :1024].flip(1)
    elif kind == "cluster":
        emb = emb[:, :1] + 1e-4 * emb
    elif kind == "tiny":
        emb, x = emb * 1e-25, x * 1e-25
        x[::3] *= 1e-12
    elif kind == "huge":
        emb, x = emb * 1e17, x * 1e18
        x[::3] *= 1e15
    elif kind == "zero_rows":
        x[::2] = 0
    elif kind == "bad_rows":
        x[5, 3], x[40, 300], x[41, 511], x[1299, 0] = float("nan"), float("inf"), float("-inf"), float("nan")
    elif kind == "bad_book":
        emb[1, 700, 9], emb[2, 3, 4] = float("inf"), float("nan")
    elif kind == "mixed":
        emb *= 10.0 ** (8 * torch.rand(n, e, 1, generator=g) - 4)
        x *= 10.0 ** (8 * torch.rand(rows, 1, generator=g) - 4)
    elif kind == "on_entries":
        i = torch.randint(0, e, (rows,), generator=g)
        x = torch.cat([emb[0, i], emb[1, i] + emb[2, i.flip(0)]], 1)
    elif kind == "zero_book":
        emb[2] = 0
    elif kind == "offset":
        emb, x = emb + 3.0, x + 3.0
    emb, norms, emb_t = books(emb)
    x = x.contiguous().to(DEV)
    want = encode(x, emb, norms, emb_t, 1, rows, False)
    assert torch.equal(encode(x, emb, norms, emb_t, 1, rows, True), want)


def test_screen_rejects():
    """Calls whose FP32 sums the step launches order otherwise (few rows for the
    entries) and shapes without a screened form are refused."""
    t = torch.empty(4096, device=DEV)
    p = t.data_ptr()
    lib = nat.library()
    for rows, dim, e in ((1024, 256, 2048), (1100, 256, 1024), (1031, 256, 96), (1031, 256, 32), (2000, 128, 2048), (2000, 256, 2080), (2000, 256, 80), (2000, 256, 0)):
        assert not lib.fm_rvq_screen_supported(rows, dim, e)
    with pytest.raises(nat.NativeError, match="unsupported"):
        nat.call("fm_rvq_encode_split_screened", p, 512, 1024, 1024, 256, 2048, 1, 1, p, p, p, p, p, 2048, 0)
    with pytest.raises(nat.NativeError, match="unsupported"):
        nat.call("fm_rvq_encode_split_screened", p, 512, 1100, 1100, 256, 1024, 1, 1, p, p, p, p, p, 1024, 0)
    with pytest.raises(nat.NativeError, match="bad argument"):
        nat.call("fm_rvq_encode_split_screened", p, 512, 2000, 2000, 256, 2048, 1, 1, p, p, None, p, p, 2048, 0)
    with pytest.raises(nat.NativeError, match="unsupported"):
        nat.call("fm_rvq_prepare_screen", t.data_ptr(), t.data_ptr(), 4, 128, 1, t.data_ptr(), t.data_ptr(), 0)
    with pytest.raises(nat.NativeError, match="bad argument"):
        nat.call("fm_rvq_prepare_screen", t.data_ptr(), t.data_ptr(), 0, 256, 1, t.data_ptr(), t.data_ptr(), 0)
