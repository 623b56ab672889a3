"""The three-product fp16 form (FM_WEIGHTS_H3) against float64.

Tolerance: a product drops a1 b1 (at most 2^-22 |a b|) and each operand is
within 2^-23 of its value, so a sum of K products is within
(2^-22 + 2 * 2^-23) sum |a b| of the exact one plus the FP32 rounding of its
accumulation, which the FP32 and bf16x6 kernels are held to as 1e-5 sum |a b|;
the same 1e-5 holds here.  Row scales make that a per-row property, whatever
the magnitudes of the other rows.
"""

from __future__ import annotations

import math

import pytest
import torch
import torch.nn.functional as F

from fast_mimi_amd import MimiModel
from fast_mimi_amd import _native as nat
from fast_mimi_amd.config import MimiConfig
from fast_mimi_amd.runtime import _Conv, _ConvT, rope_tables
from oracle.mimi_oracle import causal_conv1d, causal_conv_transpose1d

pytestmark = pytest.mark.gpu
DEV = "cuda"
WS_BYTES = 64 << 20
FLAGS = nat.WEIGHTS_X6 | nat.WEIGHTS_H3


@pytest.fixture(scope="module")
def ws():
    return torch.empty(WS_BYTES // 4, device=DEV)


def stream():
    return torch.cuda.current_stream().cuda_stream


def with_planes(w):
    """W^T [N, K], then its bf16 planes, then its fp16 planes and row exponents."""
    rows, cols = w.shape
    n = w.numel()
    x6 = n + 3 * n // 2
    buf = torch.empty(x6 + n + rows, device=DEV)
    buf[:n].copy_(w.reshape(-1))
    nat.call("fm_split_weights", buf.data_ptr(), rows, cols, buf.data_ptr() + 4 * n, stream())
    nat.call("fm_split_weights_h3", buf.data_ptr(), rows, cols, buf.data_ptr() + 4 * x6, stream())
    torch.cuda.synchronize()
    return buf[:n].view(w.shape), buf[x6:]


def linear(x, w, ws, flags=FLAGS, res=None, scale=None):
    rows, k = x.shape
    n = w.shape[0]
    y = torch.full((rows, n), float("nan"), device=DEV)
    nat.call("fm_linear", x.data_ptr(), rows, k, w.data_ptr(), n, flags, None if res is None else res.data_ptr(),
             None if scale is None else scale.data_ptr(), y.data_ptr(), ws.data_ptr(), WS_BYTES, stream())
    torch.cuda.synchronize()
    return y


def close_dot(got, want, absref, rel=1e-5):
    worst = ((got.double() - want).abs() / (rel * absref + 1e-300)).max().item()
    assert worst <= 1.0, f"error {worst:.2f}x the per-element bound"


def test_split_weights_h3_layout():
    """Two fp16 pieces per weight, within 2^-22 of it, each row scaled so its
    largest magnitude lies in [2^13, 2^14); zero and tiny rows included."""
    g = torch.Generator().manual_seed(1)
    w = torch.randn(48, 80, generator=g) * torch.logspace(-30, 30, 48)[:, None]
    w[5] = 0
    _, planes = with_planes(w.to(DEV))
    n = w.numel()
    half = planes[:n].view(torch.float16).view(2, 5, 48, 16).permute(0, 2, 1, 3).reshape(2, 48, 80).cpu().double()
    s = planes[n:].view(torch.int32).cpu().double()
    top = half[0].abs().amax(1)
    assert torch.all((top >= 2 ** 13) & (top <= 2 ** 14) | (w.abs().amax(1) == 0))
    back = half.sum(0) * torch.exp2(-s)[:, None]
    assert torch.all((back - w.double()).abs() <= w.double().abs() * 2.0 ** -22 + w.abs().amax(1, keepdim=True) * 2.0 ** -38)
    with pytest.raises(nat.NativeError, match="unsupported"):
        nat.call("fm_split_weights_h3", planes.data_ptr(), 4, 24, planes.data_ptr(), stream())
    with pytest.raises(nat.NativeError, match="bad argument"):
        nat.call("fm_split_weights_h3", planes.data_ptr(), 0, 16, planes.data_ptr(), stream())


@pytest.mark.parametrize("rows,k,n,plan", [
    (1, 2048, 512, "<64,64,2,2,4,2"), (63, 64, 32, "<64,64,2,2,4,2"), (65, 1024, 1536, "<64,64,2,2,4,2"),
    (250, 2048, 4096, "<128,128,4,2,2,4"), (2500, 512, 512, "<64,64,2,2,4,2"), (1100, 512, 2048, "<64,64,2,2,2,4"), (2500, 96, 100, "<64,128,2,2,2,3"),
    (2500, 512, 1536, "<128,128,4,2,2,4"), (4000, 2048, 512, "<128,128,4,2,2,4"),
    (127, 48, 36, "<128,128,2,2,1,4"), (66000, 256, 128, "<128,128,2,2,1,4"), (16001, 512, 640, "<128,128,2,2,1,4"),
])
def test_linear_tiles(rows, k, n, plan, ws):
    """Each tile and K split, ragged rows and columns, against float64; no
    further from it (2-norm) than the FP32 / bf16x6 plan of the same call."""
    g = torch.Generator().manual_seed(rows + k + n)
    x = torch.randn(rows, k, generator=g).to(DEV)
    w, _ = with_planes((torch.randn(n, k, generator=g) / math.sqrt(k)).to(DEV))
    want = x.double() @ w.double().t()
    got = linear(x, w, ws)
    assert f"gemm_h3_kernel{plan}" in nat.last_gemm_plan(), nat.last_gemm_plan()
    close_dot(got, want, x.double().abs() @ w.double().abs().t())
    other = linear(x, w, ws, nat.WEIGHTS_X6)
    err, was = ((v.double() - want).norm() / want.norm() for v in (got, other))
    assert err <= max(1.1 * was, 1.5e-7), f"{err:.2e} against {was:.2e}"
    res, scale = torch.randn(rows, n, generator=g).to(DEV), torch.randn(n, generator=g).to(DEV)
    close_dot(linear(x, w, ws, FLAGS | nat.EPI_RES_SCALE, res, scale), res.double() + scale.double() * want,
              res.double().abs() + scale.double().abs() * (x.double().abs() @ w.double().abs().t()))


@pytest.mark.parametrize("rows,k,n,plan", [
    (160, 1024, 1536, "tiles=72 splits=4"), (1030, 2048, 512, "tiles=136 splits=3"), (250, 2048, 4096, "tiles=64 splits=8"),
    (1500, 1024, 1536, "tiles=144 splits=3"), (3000, 1024, 1536, "tiles=288 splits=1"), (4600, 2048, 512, "tiles=144 splits=3"),
    (8200, 2048, 512, "tiles=260 splits=1"), (8192, 2048, 512, "tiles=256 splits=2"), (776, 512, 640, "tiles=130 splits=3"),
    (1700, 512, 640, "tiles=270 splits=1"), (400, 512, 640, "tiles=70 splits=4"), (1, 2048, 512, "tiles=8 splits=16"),
    (2100, 2048, 512, "tiles=68 splits=5"), (2500, 2048, 512, "tiles=80 splits=4"), (1000, 1536, 256, "tiles=64 splits=8"),
    (8300, 1536, 256, "tiles=130 splits=3"), (100, 1088, 512, "tiles=16 splits=6"),
])
def test_splits_stay_resident(rows, k, n, plan, ws):
    """K splits never put more blocks into a launch than the chip holds at once
    (two per CU), any number of splits adds up, and short last splits too."""
    tiles, splits = (int(item.split("=")[1]) for item in plan.split())
    assert splits == 1 or tiles * splits <= 512
    g = torch.Generator().manual_seed(rows + k)
    x = torch.randn(rows, k, generator=g).to(DEV)
    w, _ = with_planes((torch.randn(n, k, generator=g) / math.sqrt(k)).to(DEV))
    got = linear(x, w, ws)
    assert "gemm_h3_kernel" in nat.last_gemm_plan() and plan in nat.last_gemm_plan(), nat.last_gemm_plan()
    close_dot(got, x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t())


@pytest.mark.parametrize("rows,plan", [
    (1, "gemm_h3_kernel<64,64,2,2,4,2,true> tiles=4 splits=8"), (1023, "gemm_h3_kernel<64,64,2,2,4,2,true> tiles=64 splits=8"),
    (1024, "gemm_x6d_kernel<"), (2176, "gemm_x6d_kernel<"), (2177, "gemm_h3_kernel<128,128,4,1,2,2,true> tiles=36 splits=8"),
    (8161, "gemm_h3_kernel<128,128,4,1,2,2,true> tiles=128 splits=4"), (32700, "gemm_h3_kernel<128,128,4,1,2,2,true> tiles=512 splits=1"),
    (32800, "gemm_h3_kernel<128,128,4,1,1,4,true> tiles=514 splits=1"),
])
def test_elu_on_load_tiles(rows, plan, ws):
    """The 512-channel residual block's k3 conv (256 columns, ELU on load) over
    its tiles and the gap that stays on the bf16 form."""
    g = torch.Generator().manual_seed(rows)
    x = torch.randn(rows, 512, generator=g).to(DEV)
    wt = torch.randn(256, 3 * 512, generator=g).to(DEV) / math.sqrt(1536)
    w, _ = with_planes(wt)
    b = torch.randn(256, generator=g).to(DEV)
    y = torch.full((rows, 256), float("nan"), device=DEV)
    nat.call("fm_conv1d", x.data_ptr(), 1, rows, 512, w.data_ptr(), b.data_ptr(), 256, 3, 1, 0, FLAGS | nat.ELU_IN, None,
             y.data_ptr(), rows, ws.data_ptr(), WS_BYTES, stream())
    torch.cuda.synchronize()
    assert plan in nat.last_gemm_plan(), nat.last_gemm_plan()
    a = F.pad(F.elu(x.double()), (0, 0, 2, 0))
    taps = torch.cat([a[j:j + rows] for j in range(3)], 1)
    close_dot(y, taps @ wt.double().t() + b.double(), taps.abs() @ wt.double().abs().t() + b.double().abs())


@pytest.mark.parametrize("rows,k,n", [(200, 512, 256), (2500, 512, 1536), (2500, 512, 512), (70000, 128, 128), (1100, 512, 2048)])
def test_row_scales(rows, k, n, ws):
    """Rows from 1e-30 to 1e30 side by side, rows that start with zeros, rows
    that grow by 2^60 along k and rows of zeros all keep their own relative
    accuracy; a row holding an inf or a NaN spoils only itself."""
    g = torch.Generator().manual_seed(rows + n)
    x = torch.randn(rows, k, generator=g)
    x *= 10.0 ** (60 * torch.rand(rows, 1, generator=g) - 30)
    x[3::7, :k // 2] = 0
    x[4::7] *= torch.exp2(torch.linspace(-40, 20, k))
    x[5::7] *= torch.exp2(torch.linspace(20, -40, k))
    x[6::7] = 0
    x[0, 5], x[64, k - 1], x[130, 0] = float("inf"), float("nan"), float("-inf")
    x = x.to(DEV)
    w, _ = with_planes((torch.randn(n, k, generator=g) / math.sqrt(k)).to(DEV))
    got = linear(x, w, ws)
    assert "gemm_h3_kernel" in nat.last_gemm_plan()
    bad = torch.zeros(rows, dtype=torch.bool, device=DEV)
    bad[[0, 64, 130]] = True
    assert not torch.isfinite(got[bad]).any()
    x, got = x[~bad], got[~bad]
    close_dot(got, x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t())
    assert torch.all(got[(x == 0).all(1)] == 0)


@pytest.mark.parametrize("B,cin,cout,stride,L", [(1, 1024, 512, 8, 26), (1, 128, 64, 4, 6240), (3, 256, 128, 5, 1001),
                                                 (2, 128, 64, 4, 40001), (1, 48, 16, 4, 777),
                                                 (1, 256, 128, 4, 131_500)])  # (over 256 MB written: streaming stores)
def test_conv_transpose1d(B, cin, cout, stride, L, ws):
    """Stride phases, batch seams inside a tile and the zero row before each clip."""
    g = torch.Generator().manual_seed(L)
    x = torch.randn(B, cin, L, generator=g)
    w, b = torch.randn(cin, cout, 2 * stride, generator=g) / math.sqrt(2 * cin), torch.randn(cout, generator=g)
    layer = _ConvT(w.to(DEV), b.to(DEV), stride)
    wp, _ = with_planes(layer.w)
    xd = x.transpose(1, 2).contiguous().to(DEV)
    y = torch.full((B, L * stride, cout), float("nan"), device=DEV)
    nat.call("fm_conv_transpose1d", xd.data_ptr(), B, L, cin, wp.data_ptr(), layer.b.data_ptr(), cout, layer.k,
             stride, FLAGS, None, y.data_ptr(), ws.data_ptr(), WS_BYTES, stream())
    torch.cuda.synchronize()
    assert "gemm_h3_kernel" in nat.last_gemm_plan()
    want = causal_conv_transpose1d(x.double(), w.double(), b.double(), stride)
    absref = causal_conv_transpose1d(x.double().abs(), w.double().abs(), b.double().abs(), stride)
    close_dot(y.cpu().transpose(1, 2), want, absref)


@pytest.mark.parametrize("B,cin,cout,k,L,y_len,flags", [
    (1, 512, 256, 3, 208, None, nat.ELU_IN | nat.EPI_ELU), (16, 512, 256, 3, 2000, None, nat.ELU_IN | nat.EPI_ELU),
    (3, 256, 512, 1, 700, None, nat.EPI_RES_ADD | nat.EPI_ELU), (2, 512, 1024, 7, 61, 50, nat.EPI_ELU),
    (4, 64, 128, 3, 20001, 19000, 0)])
def test_conv1d(B, cin, cout, k, L, y_len, flags, ws):
    """ELU on load, residual and ELU epilogues, cropped outputs."""
    g = torch.Generator().manual_seed(L + cin)
    x = torch.randn(B, cin, L, generator=g)
    w, b = torch.randn(cout, cin, k, generator=g) / math.sqrt(cin * k), torch.randn(cout, generator=g)
    res = torch.randn(B, cout, L, generator=g)
    y_len = L if y_len is None else y_len
    layer = _Conv(w.to(DEV), b.to(DEV))
    wp, _ = with_planes(layer.w)
    xd, rd = (t.transpose(1, 2).contiguous().to(DEV) for t in (x, res))
    y = torch.full((B, y_len, cout), float("nan"), device=DEV)
    nat.call("fm_conv1d", xd.data_ptr(), B, L, cin, wp.data_ptr(), layer.b.data_ptr(), cout, k, 1, 0, flags | FLAGS,
             rd.data_ptr(), y.data_ptr(), y_len, ws.data_ptr(), WS_BYTES, stream())
    torch.cuda.synchronize()
    assert "gemm_h3_kernel" in nat.last_gemm_plan()
    xin = F.elu(x.double()) if flags & nat.ELU_IN else x.double()
    want = causal_conv1d(xin, w.double(), b.double())
    absref = causal_conv1d(xin.abs(), w.double().abs(), b.double().abs())
    if flags & nat.EPI_RES_ADD:
        want, absref = want + res, absref + res.abs()
    if flags & nat.EPI_ELU:
        want = F.elu(want)
    close_dot(y.cpu().transpose(1, 2), want[..., :y_len], absref[..., :y_len])


@pytest.mark.parametrize("rows,per_seq,n,rope_cols", [(2500, 2500, 1536, 1024), (30000, 250, 1536, 1024),
                                                      (2500, 100, 512, 512), (100, 100, 1536, 1024)])
def test_linear_rope_equals_linear_then_rope(rows, per_seq, n, rope_cols, ws):
    """RoPE in the tile's epilogue, or after it where the tile cannot, equals
    fm_linear followed by fm_apply_rope bit for bit."""
    g = torch.Generator().manual_seed(rows + n)
    x = torch.randn(rows, 512, generator=g).to(DEV)
    w, _ = with_planes((torch.randn(n, 512, generator=g) / math.sqrt(512)).to(DEV))
    cos, sin = (t.to(DEV) for t in rope_tables(MimiConfig(), per_seq))
    want = linear(x, w, ws)
    nat.call("fm_apply_rope", want.data_ptr(), rows, n, rope_cols, 64, cos.data_ptr(), sin.data_ptr(), per_seq,
             stream())
    got = torch.full((rows, n), float("nan"), device=DEV)
    nat.call("fm_linear_rope", x.data_ptr(), rows, 512, w.data_ptr(), n, FLAGS, cos.data_ptr(), sin.data_ptr(),
             rope_cols, per_seq, got.data_ptr(), ws.data_ptr(), WS_BYTES, stream())
    torch.cuda.synchronize()
    assert torch.equal(got, want)


def block_reference(x, w1, b1, w2, b2):
    """float64 block output [B, C, L] and the scale its error is held to: the
    same sums on absolute values."""
    a = F.elu(x)
    hid = F.elu(causal_conv1d(a, w1, b1))
    ref = causal_conv1d(a.abs(), w1.abs(), b1.abs())
    return x + causal_conv1d(hid, w2, b2), x.abs() + causal_conv1d(ref, w2.abs(), b2.abs())


@pytest.mark.parametrize("C,B,L", [(64, 1, 1000), (64, 2, 129), (128, 1, 777), (128, 3, 1), (128, 2, 66), (256, 1, 2000),
                                   (256, 2, 33), (256, 1, 31)])
@pytest.mark.parametrize("kind", ["plain", "loud_quiet", "zero_channels", "tiny"])
def test_resblock(C, B, L, kind):
    """The fp16 residual block against float64, no further from it than the
    bf16 one; rows far below their neighbours, hidden channels of zero weight
    and whole inputs near 1e-25 (the block's scales are dynamic).  ELU as
    e^x - 1 adds an absolute error of a few 2^-24 to either form."""
    g = torch.Generator().manual_seed(C + L)
    x = torch.randn(B, C, L, generator=g)
    w1, b1 = torch.randn(C // 2, C, 3, generator=g) / math.sqrt(3 * C), 0.1 * torch.randn(C // 2, generator=g)
    w2, b2 = torch.randn(C, C // 2, 1, generator=g) / math.sqrt(C // 2), 0.1 * torch.randn(C, generator=g)
    if kind == "loud_quiet":
        x *= 10.0 ** (torch.arange(L) % 5 - 2)
    elif kind == "zero_channels":
        w1[::3] = 0
    elif kind == "tiny":
        x, b1, b2 = x * 1e-25, b1 * 0, b2 * 0
    c1, c2 = _Conv(w1.to(DEV), b1.to(DEV)), _Conv(w2.to(DEV), b2.to(DEV))
    (w1p, _), (w2p, _) = with_planes(c1.w), with_planes(c2.w)
    xd = x.transpose(1, 2).contiguous().to(DEV)
    want, absref = block_reference(*(t.double() for t in (x, w1, b1, w2, b2)))
    out = {}
    for flags in (FLAGS, nat.WEIGHTS_X6):
        y = torch.full_like(xd, float("nan"))
        nat.call("fm_resblock", xd.data_ptr(), B, L, C, w1p.data_ptr(), c1.b.data_ptr(), w2p.data_ptr(),
                 c2.b.data_ptr(), flags | nat.ACT_EXP, y.data_ptr(), stream())
        torch.cuda.synchronize()
        out[flags] = y.cpu().double().transpose(1, 2)
    # (FLAGS without bit 1 has no trailing ELU; the e^x - 1 error passes through both convs.)
    if kind != "tiny":
        close_dot(out[FLAGS], want, absref + 1.0)
    err, was = ((v - want).norm() for v in out.values())
    assert err <= 1.1 * was + 1e-7 * want.norm()


def run_block(x, w1, b1, w2, b2):
    """fm_resblock on the fp16 planes: [B, C, L] on the CPU."""
    B, C, L = x.shape
    c1, c2 = _Conv(w1.to(DEV), b1.to(DEV)), _Conv(w2.to(DEV), b2.to(DEV))
    (w1p, _), (w2p, _) = with_planes(c1.w), with_planes(c2.w)
    xd = x.transpose(1, 2).contiguous().to(DEV)
    y = torch.full_like(xd, float("nan"))
    nat.call("fm_resblock", xd.data_ptr(), B, L, C, w1p.data_ptr(), c1.b.data_ptr(), w2p.data_ptr(), c2.b.data_ptr(),
             FLAGS | nat.ACT_EXP, y.data_ptr(), stream())
    torch.cuda.synchronize()
    return y.cpu().transpose(1, 2)


@pytest.mark.parametrize("C,B,L", [(64, 1, 300), (64, 2, 127), (128, 1, 131), (128, 2, 64), (256, 1, 97), (256, 3, 5)])
@pytest.mark.parametrize("outlier", [False, True])
def test_resblock_rows_keep_their_own_accuracy(C, B, L, outlier):
    """Rows from 1e-12 to 1e12 side by side, each held to its own sums:
    positive inputs and first weights keep both ELUs exact, so only the
    contractions' 1e-5 of the sum of magnitudes is allowed (the residual's
    rounding, 2^-24, is within it).  ``outlier``: one hidden channel 1e4 above
    the others, whose second weights weigh it down again; the others then keep
    2^-39 * 2^6 * 1e4 = 1.2e-6 of what they are."""
    g = torch.Generator().manual_seed(C + L)
    x = torch.rand(B, C, L, generator=g) + 0.1
    x *= 10.0 ** (24 * torch.rand(B, 1, L, generator=g) - 12)
    x[:, :, L // 2:L // 2 + 4] = 0
    w1 = (torch.rand(C // 2, C, 3, generator=g) + 0.1) / (3 * C)
    w2 = torch.randn(C, C // 2, 1, generator=g) / math.sqrt(C // 2)
    if outlier:
        w1[1] *= 1e4
        w2[:, 1] *= 1e-4
    zero1, zero2 = torch.zeros(C // 2), torch.zeros(C)
    want, absref = block_reference(*(t.double() for t in (x, w1, zero1, w2, zero2)))
    close_dot(run_block(x, w1, zero1, w2, zero2), want, absref)


@pytest.mark.parametrize("C,L", [(64, 300), (128, 150), (256, 70)])
def test_resblock_rows_are_independent(C, L):
    """A loud, an infinite and a NaN row change the rows that read them (its own
    and the next two) and no bit of any other, before or after."""
    g = torch.Generator().manual_seed(C)
    x = torch.randn(1, C, L, generator=g)
    w1, b1 = torch.randn(C // 2, C, 3, generator=g) / math.sqrt(3 * C), 0.1 * torch.randn(C // 2, generator=g)
    w2, b2 = torch.randn(C, C // 2, 1, generator=g) / math.sqrt(C // 2), 0.1 * torch.randn(C, generator=g)
    plain = run_block(x, w1, b1, w2, b2)
    loud = x.clone()
    rows = (0, 20, L // 2, L - 1)
    loud[:, :, 0] *= 1e7
    loud[:, :, 20] *= 1e20
    loud[:, 3, L // 2] = float("inf")
    loud[:, 5, L - 1] = float("nan")
    got = run_block(loud, w1, b1, w2, b2)
    own = torch.ones(L, dtype=torch.bool)
    for r in rows:
        own[r:r + 3] = False
    assert torch.equal(got[..., own], plain[..., own])


@pytest.mark.parametrize("B,L,y_len", [(1, 1000, 1000), (2, 129, 100), (3, 33, 33), (1, 1, 1)])
def test_resblock64_conv(B, L, y_len):
    """The decoder's last block and waveform conv on fp16 weights."""
    g = torch.Generator().manual_seed(L)
    x = torch.randn(B, 64, L, generator=g)
    w1, b1 = torch.randn(32, 64, 3, generator=g) / math.sqrt(192), 0.1 * torch.randn(32, generator=g)
    w2, b2 = torch.randn(64, 32, 1, generator=g) / math.sqrt(32), 0.1 * torch.randn(64, generator=g)
    w3, b3 = torch.randn(1, 64, 3, generator=g) / math.sqrt(192), torch.randn(1, generator=g)
    c1, c2, c3 = (_Conv(w.to(DEV), b.to(DEV)) for w, b in ((w1, b1), (w2, b2), (w3, b3)))
    (w1p, _), (w2p, _) = with_planes(c1.w), with_planes(c2.w)
    xd = x.transpose(1, 2).contiguous().to(DEV)
    d = torch.empty(nat.library().fm_resblock64_conv_workspace_bytes(B, L) // 4, device=DEV)
    blk, _ = block_reference(*(t.double() for t in (x, w1, b1, w2, b2)))
    want = causal_conv1d(F.elu(blk), w3.double(), b3.double())[..., :y_len]
    errs = []
    for flags in (FLAGS, nat.WEIGHTS_X6):
        y = torch.full((B, y_len), float("nan"), device=DEV)
        nat.call("fm_resblock64_conv", xd.data_ptr(), B, L, w1p.data_ptr(), c1.b.data_ptr(), w2p.data_ptr(),
                 c2.b.data_ptr(), 1 | flags | nat.ACT_EXP, c3.w.data_ptr(), c3.b.data_ptr(), y_len, y.data_ptr(),
                 d.data_ptr(), d.numel() * 4, stream())
        torch.cuda.synchronize()
        errs.append((y.cpu().double()[:, None] - want).norm())
        assert (y.cpu().double()[:, None] - want).abs().max() <= 2e-5 * want.abs().max()
    assert errs[0] <= 1.1 * errs[1] + 1e-7 * want.norm()


@pytest.mark.parametrize("rows,k,n,ln,epi", [(250, 512, 1536, True, "rope"), (1, 512, 2048, True, "gelu"), (33, 512, 512, False, "res"),
                                             (512, 512, 2048, True, "gelu"), (17, 2048, 512, False, "res"), (250, 2048, 512, False, "res"),
                                             (16, 512, 64, False, "plain")])
@pytest.mark.parametrize("kind", ["plain", "scales"])
def test_row_linear(rows, k, n, ln, epi, kind):
    """The few-row projections on fp16 planes, each epilogue; rows of any
    magnitude side by side and k-ranges (one per wave) of any magnitude within a
    row, zero rows and rows with an inf."""
    g = torch.Generator().manual_seed(rows + k + n)
    x = torch.randn(rows, k, generator=g)
    if kind == "scales" and not ln:
        x *= 10.0 ** (40 * torch.rand(rows, 1, generator=g) - 20)
        x *= torch.exp2(torch.randint(-30, 30, (1, 8), generator=g).repeat_interleave(k // 8, 1).float())
        x[2::5] = 0
    x = x.to(DEV)
    w, _ = with_planes((torch.randn(n, k, generator=g) / math.sqrt(k)).to(DEV))
    gamma, beta = (1 + 0.1 * torch.randn(k, generator=g)).to(DEV), (0.1 * torch.randn(k, generator=g)).to(DEV)
    res, scale = torch.randn(rows, n, generator=g).to(DEV), torch.randn(n, generator=g).to(DEV)
    cos, sin = (t.to(DEV) for t in rope_tables(MimiConfig(), max(rows // 2, 1)))
    flags = FLAGS | {"gelu": nat.EPI_GELU, "res": nat.EPI_RES_SCALE}.get(epi, 0)
    rope_cols, per_seq = (1024, max(rows // 2, 1)) if epi == "rope" else (0, 1)
    y = torch.full((rows, n), float("nan"), device=DEV)
    nat.call("fm_row_linear", x.data_ptr(), rows, k, gamma.data_ptr() if ln else None, beta.data_ptr() if ln else None,
             1e-5, w.data_ptr(), n, flags, res.data_ptr() if epi == "res" else None,
             scale.data_ptr() if epi == "res" else None, cos.data_ptr() if rope_cols else None,
             sin.data_ptr() if rope_cols else None, rope_cols, per_seq, y.data_ptr(), stream())
    torch.cuda.synchronize()
    a = x.double()
    if ln:
        a = F.layer_norm(a, (k,), gamma.double(), beta.double(), 1e-5)
    want, absref = a @ w.double().t(), a.abs() @ w.double().abs().t()
    if epi == "gelu":
        want = F.gelu(want)
    elif epi == "res":
        want, absref = res.double() + scale.double() * want, res.double().abs() + scale.double().abs() * absref
    elif epi == "rope":
        pos = torch.arange(rows, device=DEV) % per_seq
        c, s = (t.double()[pos].repeat(1, rope_cols // 64) for t in (cos, sin))
        q = want[:, :rope_cols].view(rows, -1, 64)
        half = torch.cat((-q[..., 32:], q[..., :32]), -1).reshape(rows, -1)
        h2 = absref[:, :rope_cols].view(rows, -1, 64)
        want[:, :rope_cols] = want[:, :rope_cols] * c + half * s
        absref[:, :rope_cols] += torch.cat((h2[..., 32:], h2[..., :32]), -1).reshape(rows, -1)
    close_dot(y, want, absref)


@pytest.mark.parametrize("B,cin,cout,k,L,flags", [
    (1, 512, 1024, 7, 2, nat.EPI_ELU), (1, 512, 1024, 7, 250, nat.EPI_ELU), (2, 512, 1024, 7, 131, 0), (1, 512, 1024, 7, 265, 0),
    (1, 512, 256, 3, 208, nat.ELU_IN | nat.EPI_ELU), (1, 512, 256, 3, 2000, nat.ELU_IN | nat.EPI_ELU),
    (1, 256, 512, 1, 16, nat.EPI_RES_ADD | nat.EPI_ELU), (3, 256, 512, 1, 701, nat.EPI_RES_ADD)])
def test_conv1d_rows(B, cin, cout, k, L, flags):
    """The few-row convolutions on fp16 planes: one- and two-tile blocks, batch
    seams, ELU on load, residuals; quiet rows between loud ones."""
    g = torch.Generator().manual_seed(L + cin)
    x = torch.randn(B, cin, L, generator=g) * 10.0 ** (torch.arange(L) % 4 * 3 - 6)
    w, b = torch.randn(cout, cin, k, generator=g) / math.sqrt(cin * k), torch.randn(cout, generator=g)
    res = torch.randn(B, cout, L, generator=g)
    layer = _Conv(w.to(DEV), b.to(DEV))
    wp, _ = with_planes(layer.w)
    xd, rd = (t.transpose(1, 2).contiguous().to(DEV) for t in (x, res))
    y = torch.full((B, L, cout), float("nan"), device=DEV)
    nat.call("fm_conv1d_rows", xd.data_ptr(), B, L, cin, wp.data_ptr(), layer.b.data_ptr(), cout, cout, k, 1, 0,
             flags | FLAGS, rd.data_ptr(), y.data_ptr(), stream())
    torch.cuda.synchronize()
    xin = F.elu(x.double()) if flags & nat.ELU_IN else x.double()
    want = causal_conv1d(xin, w.double(), b.double())
    absref = causal_conv1d(xin.abs(), w.double().abs(), b.double().abs())
    if flags & nat.EPI_RES_ADD:
        want, absref = want + res, absref + res.abs()
    if flags & nat.EPI_ELU:
        want = F.elu(want)
    close_dot(y.cpu().transpose(1, 2), want, absref)
    with pytest.raises(nat.NativeError, match="unsupported"):
        nat.call("fm_conv1d_rows", xd.data_ptr(), B, L, cin, wp.data_ptr(), layer.b.data_ptr(), cout, cout, k, 1, 0,
                 nat.WEIGHTS_H3, rd.data_ptr(), y.data_ptr(), stream())


@pytest.mark.parametrize("kind,k,n,rows", [("row", 512, 1536, 26), ("row", 512, 512, 250), ("row", 2048, 512, 13),
                                           ("conv", 7, 1024, 26), ("conv", 7, 1024, 265), ("conv", 3, 256, 2000),
                                           ("conv", 1, 512, 40)])
@pytest.mark.parametrize("weight_exp", [0, -60, -100])
def test_few_rows_reach_the_ends_of_fp32(kind, k, n, rows, weight_exp):
    """Results of 2^100 and more, to which every partial product belongs, stay
    finite whatever the weights' own scale: a weight row's exponent (13 and up,
    more for small weights) must not meet a partial sum alone."""
    g = torch.Generator().manual_seed(rows + n)
    cin = k if kind == "row" else 256 if k == 1 else 512
    taps = 1 if kind == "row" else k
    x = torch.randn(1, cin, rows, generator=g) * 2.0 ** (112 if weight_exp == 0 else 120)
    w = torch.randn(n, cin, taps, generator=g) / math.sqrt(cin * taps) * 2.0 ** weight_exp
    layer = _Conv(w.to(DEV), torch.zeros(n, device=DEV))
    wp, _ = with_planes(layer.w)
    xd = x.transpose(1, 2).contiguous().to(DEV)
    y = torch.full((1, rows, n), float("nan"), device=DEV)
    if kind == "row":
        nat.call("fm_row_linear", xd.data_ptr(), rows, k, None, None, 1e-5, wp.data_ptr(), n, FLAGS, None, None, None,
                 None, 0, 1, y.data_ptr(), stream())
    else:
        nat.call("fm_conv1d_rows", xd.data_ptr(), 1, rows, cin, wp.data_ptr(), layer.b.data_ptr(), n, n, k, 1, 0, FLAGS,
                 None, y.data_ptr(), stream())
    torch.cuda.synchronize()
    want = causal_conv1d(x.double(), w.double(), torch.zeros(n, dtype=torch.float64))
    close_dot(y.cpu().transpose(1, 2), want, causal_conv1d(x.double().abs(), w.double().abs(),
                                                           torch.zeros(n, dtype=torch.float64)))


def test_every_packed_copy_is_read():
    """A few-row round trip reads each fragment-packed projection the runtime
    keeps: none beside the 16-bit planes that replace it."""
    model = MimiModel(MimiConfig(num_hidden_layers=2), device=DEV, use_graphs=False)
    rt = model.runtime()
    read = set()

    def call(name, *args):
        if name.startswith("fm_row_linear_packed"):
            read.add(args[6 if name == "fm_row_linear_packed" else 3].data_ptr())
        return type(rt)._call(rt, name, *args)

    rt._call = call
    model.decode(model.encode(torch.randn(1, 1, 24_000, device=DEV)).audio_codes)
    assert rt._packed and {t.data_ptr() for t in rt._packed.values()} == read


@pytest.mark.parametrize("kind,k,n,rows,fp16", [
    ("conv", 1, 512, 26, False), ("conv", 1, 512, 2000, False), ("conv", 3, 256, 1024, True), ("conv", 7, 1024, 26, True), ("conv", 7, 1024, 256, True),
    ("conv", 7, 1024, 257, False), ("conv", 7, 1024, 272, False), ("row", 512, 2048, 1, True), ("row", 512, 512, 1, True),
    ("row", 2048, 512, 1, True), ("rope", 512, 1536, 1, True), ("rope", 512, 1536, 512, True),
])
def test_few_rows_take_the_faster_form(kind, k, n, rows, fp16):
    """With both plane sets the call is the bf16 form bit for bit where that one
    is the faster, and the fp16 form elsewhere."""
    g = torch.Generator().manual_seed(rows + n)
    cin = k if kind != "conv" else 256 if k == 1 else 512
    taps = k if kind == "conv" else 1
    x = torch.randn(rows, cin, generator=g).to(DEV)
    w, _ = with_planes(torch.randn(n, cin * taps, generator=g).to(DEV))
    cos, sin = (t.to(DEV) for t in rope_tables(MimiConfig(), rows))
    out = []
    for flags in (FLAGS, nat.WEIGHTS_X6):
        y = torch.full((rows, n), float("nan"), device=DEV)
        if kind == "conv":
            nat.call("fm_conv1d_rows", x.data_ptr(), 1, rows, cin, w.data_ptr(), None, 0, n, k, 1, 0, flags, None,
                     y.data_ptr(), stream())
        else:
            rope = (cos.data_ptr(), sin.data_ptr(), 1024) if kind == "rope" else (None, None, 0)
            nat.call("fm_row_linear", x.data_ptr(), rows, cin, None, None, 1e-5, w.data_ptr(), n, flags, None, None,
                     *rope, rows, y.data_ptr(), stream())
        torch.cuda.synchronize()
        out.append(y)
    assert torch.isfinite(out[0]).all() and torch.equal(*out) != fp16


@pytest.mark.parametrize("kind,rows,k,n", [
    ("gemm", 240, 256, 256), ("gemm", 6240, 256, 256), ("gemm", 208, 1024, 1536), ("gemm", 1248, 512, 640),
    ("gemm", 1030, 2048, 512), ("gemm", 2500, 2048, 512), ("gemm", 300, 3584, 1024), ("gemm", 2600, 1536, 256),
    ("gemm", 9000, 256, 512), ("gemm", 70000, 256, 256), ("elu", 600, 1536, 256), ("elu", 2600, 1536, 256),
    ("elu", 33000, 1536, 256), ("conv", 26, 256, 512), ("conv", 26, 1536, 256), ("conv", 2000, 1536, 256),
    ("conv", 26, 3584, 1024), ("conv", 250, 3584, 1024), ("row", 26, 512, 2048), ("row", 250, 512, 1536),
    ("packed", 26, 512, 512), ("packed", 250, 2048, 512),
])
@pytest.mark.parametrize("spread", [0.0, 2.0])
def test_no_further_from_float64_than_before(kind, rows, k, n, spread, ws):
    """The 2-norm error of the fp16 form against float64 is at most that of the
    form it replaces at the same size: the bf16x6 or FP32 plan, and the
    fragment-packed FP32 kernel ("packed").  ``spread``: rows scaled by e^(2 z)."""
    g = torch.Generator(device=DEV).manual_seed(rows + k)
    taps = {"elu": 3, "conv": 1 if k == 256 else k // 512}.get(kind, 1)
    x = torch.randn(rows, k // taps, device=DEV, generator=g)
    x *= torch.exp(spread * torch.randn(rows, 1, device=DEV, generator=g))
    wt = torch.randn(n, k, device=DEV, generator=g) / math.sqrt(k)
    w, _ = with_planes(wt)
    packed = torch.empty_like(wt)
    nat.call("fm_pack_row_weights", wt.data_ptr(), n, k, packed.data_ptr(), stream())
    errs = []
    for flags in (FLAGS, nat.WEIGHTS_X6):
        y = torch.full((rows, n), float("nan"), device=DEV)
        if kind == "gemm":
            y = linear(x, w, ws, flags)
        elif kind == "elu":
            nat.call("fm_conv1d", x.data_ptr(), 1, rows, k // 3, w.data_ptr(), None, n, 3, 1, 0, flags | nat.ELU_IN, None,
                     y.data_ptr(), rows, ws.data_ptr(), WS_BYTES, stream())
        elif kind == "conv":
            nat.call("fm_conv1d_rows", x.data_ptr(), 1, rows, k // taps, w.data_ptr(), None, 0, n, taps, 1, 0, flags, None,
                     y.data_ptr(), stream())
        else:
            name, wp, f = "fm_row_linear", w, flags
            if kind == "packed" and flags != FLAGS:
                name, wp, f = "fm_row_linear_packed", packed, 0
            nat.call(name, x.data_ptr(), rows, k, None, None, 1e-5, wp.data_ptr(), n, f, None, None, None, None, 0, 1,
                     y.data_ptr(), stream())
        torch.cuda.synchronize()
        a = F.pad(F.elu(x.double()) if kind == "elu" else x.double(), (0, 0, taps - 1, 0))
        want = torch.cat([a[j:j + rows] for j in range(taps)], 1) @ wt.double().t()
        errs.append(((y.double() - want).norm() / want.norm()).item())
    assert errs[0] <= errs[1], f"{errs[0]:.3e} against {errs[1]:.3e}"
