"""The fp32 two-pass schedule (csrc/wgrad_f32.hpp) at the edges of its rules.

Against the float64 oracle at the repository's fp32 bar (1e-5): samples of one
row (||a||^2 ||b||^2), of 2..16 rows (fp64 row-Gram norms or direct ones, by
cost), 17 rows and more (direct); k-tiles that hold rows of several samples;
64- and 128-wide tiles with ragged edges; split contractions; more samples per
workgroup than it forms factors for; both layouts.
"""
import numpy as np
import pytest
import torch

from oracle import dp_clip as O
from oracle import philox
from tests._tol import assert_close, assert_elementwise

from flashdp4review_amd import _lib, core

pytestmark = pytest.mark.gpu
DEV = "cuda"

SHAPES = [  # B, K, M, N
    (1, 1, 1, 1),           # one value
    (5, 1, 70, 129),        # one row a sample, ragged 64-wide tiles
    (300, 1, 256, 320),     # several samples in every k-tile
    (2500, 1, 64, 64),      # more samples than a workgroup's factor table
    (7, 2, 131, 67),        # row Gram or direct, samples straddle k-tiles
    (64, 3, 512, 640),
    (33, 16, 640, 512),     # the row Gram's longest sample
    (33, 17, 320, 256),     # one row more: direct norms
    (3, 50, 70, 90),
    (4, 128, 768, 768),
    (2, 700, 300, 260),     # split contraction, rows not a multiple of a k-tile
    (8, 96, 1100, 1030),    # 128-wide tiles, ragged both ways
    (1, 4096, 129, 65),     # one long sample
]


def make(B, K, M, N, layout, seed=0):
    g = torch.Generator().manual_seed(seed)
    a = torch.randn((B, K, M) if layout == "tn" else (B, M, K), generator=g)
    b = torch.randn(B, K, N, generator=g) * (0.1 + torch.rand(B, 1, 1, generator=g))
    return a.to(DEV), b.to(DEV)


@pytest.mark.parametrize("layout", ["tn", "nn"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_f32_parity(shape, layout):
    B, K, M, N = shape
    a, b = make(B, K, M, N, layout)
    _, norms_ref, _ = O.wgrad_clip(a, b, 1.0, 1.0, layout)
    C = float(np.median(norms_ref)) * (1.0 if B > 1 else 0.5)
    ref, norms_ref, fac_ref = O.wgrad_clip(a, b, C, 1.0, layout)
    out, norms, fac = core.wgrad_clip(a, b, C, 1.0, layout=layout, return_stats=True)
    assert_close(out, ref, torch.float32, "sum")
    assert_elementwise(norms, norms_ref, torch.float32, "norms")
    assert_elementwise(fac, fac_ref, torch.float32, "factors")
    assert torch.equal(out, core.wgrad_clip(a, b, C, 1.0, layout=layout))


@pytest.mark.parametrize("K", [1, 2, 16])
def test_f32_cancelling_rows(K):
    """Rows that cancel: every pair's sum is 1e-3 of its terms, so the squared
    norm is 1e-6 of the Gram terms it is summed from (2e-16 each in fp64,
    6e-8 in fp32); the bound is the 1e-5 bar over the 1e-3 that fp32 inputs keep."""
    B, M, N = 6, 96, 160
    g = torch.Generator().manual_seed(4)
    a = torch.randn(B, K, M, generator=g)
    x = torch.randn(B, 1, N, generator=g).expand(B, K, N).contiguous()
    for k in range(1, K, 2):
        a[:, k] = -a[:, k - 1] * (1 + 1e-3)
    _, norms_ref, _ = O.wgrad_clip(a, x, 1.0, 1.0, "tn")
    _, norms, _ = core.wgrad_clip(a.to(DEV), x.to(DEV), 1.0, 1.0, return_stats=True)
    e = np.abs(norms.double().cpu().numpy() - norms_ref) / norms_ref
    assert e.max() <= 1e-5


@pytest.mark.parametrize("shape", [(6, 1, 96, 100), (6, 20, 96, 101)], ids=lambda s: "x".join(map(str, s)))
def test_f32_infinite_sample_is_left_out(shape):
    """A sample with an infinite entry in a has an infinite norm, so its factor
    is zero and it adds nothing, although its neighbours share its k-tiles."""
    B, K, M, N = shape
    a, b = make(B, K, M, N, "tn", seed=2)
    b[3] = b[3].abs() + 0.5  # (no zero times infinity in its norm)
    keep = [i for i in range(B) if i != 3]
    ref, _, _ = O.wgrad_clip(a[keep], b[keep], 1.0, 1.0, "tn")
    a[3] = a[3].abs() + 0.5
    a[3, 0, 5] = float("inf")
    out, norms, fac = core.wgrad_clip(a, b, 1.0, 1.0, return_stats=True)
    assert torch.isinf(norms[3]) and float(fac[3]) == 0.0
    assert_close(out, ref, torch.float32)


@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16], ids=str)
@pytest.mark.parametrize("shape", [(4, 64, 130, 96), (2, 640, 66, 101)], ids=lambda s: "x".join(map(str, s)))
def test_f32_noise_strides_and_least_workspace(shape, out_dtype):
    """The drawn noise in the sum pass's and in the split sum's epilogue, into a
    strided output, from strided operands; and the call in the least workspace
    that is accepted (fewer splits)."""
    B, K, M, N = shape
    a, b = make(B, K + 3, M + 5, N + 2, "tn", seed=5)
    a, b = a[:, 1:K + 1, 2:M + 2], b[:, 2:K + 2, 1:N + 1]
    wide = torch.zeros(M, N + 7, dtype=out_dtype, device=DEV)
    ref, _, _ = O.wgrad_clip(a, b, 1.0, 0.9, "tn")
    z = philox.normals(M * N, 77, 5).reshape(M, N)
    expect = ref / B + 0.01 * z
    core.wgrad_clip(a, b, 1.0, 0.9, out_scale=1.0 / B, noise_scale=0.01, noise_key=(77, 5),
                    out=wide[:, 3:N + 3])
    assert_close(wide[:, 3:N + 3], expect, out_dtype, "strided")
    assert torch.count_nonzero(wide[:, :3]) == 0 and torch.count_nonzero(wide[:, N + 3:]) == 0
    a, b = a.contiguous(), b.contiguous()
    L = _lib.lib()
    most = _lib.size_query(L.fdp_wgrad_clip_workspace_size, B, K, M, N, _lib.FDP_F32, 0)
    least = _lib.size_query(L.fdp_wgrad_clip_workspace_size, B, K, M, N, _lib.FDP_BF16, 0)
    outs = []
    for nbytes in (most, least):
        ws = torch.zeros(nbytes, dtype=torch.uint8, device=DEV)
        out = torch.empty(M, N, device=DEV)
        st = L.fdp_wgrad_clip(a.data_ptr(), b.data_ptr(), B, K, M, N, K * M, M, K * N, N,
                              _lib.LAYOUT_TN, _lib.FDP_F32, 1.0, 0.9, None, 1.0 / B, None, 0.0, None,
                              out.data_ptr(), N, _lib.FDP_F32, None, None, 0, ws.data_ptr(), nbytes,
                              _lib.stream_handle(torch.device(DEV, torch.cuda.current_device())))
        assert st == 0
        outs.append(out)
        assert_close(out, ref / B, torch.float32, f"{nbytes} bytes")


PAIR_SHAPES = [  # B, K, M, N: even batches, whole 16-deep k-tiles, 16-byte aligned rows
    (6, 16, 64, 64),        # one k-tile, part of one tile
    (6, 32, 192, 192),      # one whole tile
    (8, 48, 392, 520),      # ring wraps at three k-tiles, ragged tiles
    (8, 128, 196, 768),
    (24, 64, 200, 380),     # more pairs than load at once
    (72, 16, 64, 192),      # the largest batch: one block per region
    (8, 64, 1536, 1536),    # fills the device: the default route
]


@pytest.mark.parametrize("bias", [None, "a", "b"])
@pytest.mark.parametrize("shape", PAIR_SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_f32_paired(shape, bias):
    """The paired single pass on fp32 operands ("wide": wherever its plan
    applies): sum, norms and factors and the bias of either operand at the fp32
    bar, with the drawn noise, repeated bitwise, beside two-pass calls on the
    same workspace."""
    B, K, M, N = shape
    a, b = make(B, K, M, N, "tn", seed=7)
    _, norms_ref, _ = O.wgrad_clip(a, b, 1.0, 1.0, "tn")
    C = float(np.median(norms_ref))
    ref, norms_ref, fac_ref = O.wgrad_clip(a, b, C, 1.0, "tn")
    kw = dict(out_scale=1.0 / B, noise_scale=0.01, noise_key=(5, 9), single_pass="wide",
              return_stats=True, check=True)
    n = M if bias == "a" else N
    db = torch.empty(n, device=DEV)
    if bias is not None:
        kw.update(bias_out=db, bias_scale=0.25, bias_operand=bias, bias_noise_scale=0.02,
                  bias_noise_key=(6, 1))
    r = core.wgrad_clip(a, b, C, 1.0, **kw)
    expect = ref / B + 0.01 * philox.normals(M * N, 5, 9).reshape(M, N)
    assert_close(r[0], expect, torch.float32, "sum")
    assert_elementwise(r[1], norms_ref, torch.float32, "norms")
    assert_elementwise(r[2], fac_ref, torch.float32, "factors")
    first_db = db.clone()
    two = core.wgrad_clip(a, b, C, 1.0, out_scale=1.0 / B, two_pass=True)
    assert_close(two, ref / B, torch.float32, "two passes")
    again = core.wgrad_clip(a, b, C, 1.0, **kw)
    assert torch.equal(again[0], r[0])
    if bias is not None:
        u = (a if bias == "a" else b).double().cpu().numpy()
        nr = np.sqrt((u ** 2).sum((1, 2)))
        assert_elementwise(r[3], nr, torch.float32, "bias norms")
        fac = np.minimum(1.0, C / (nr + 1e-10))
        assert_close(first_db, 0.25 * (fac[:, None] * u.sum(1)).sum(0) + 0.02 * philox.normals(n, 6, 1),
                     torch.float32, "bias")
        assert torch.equal(first_db, db)


def test_f32_paired_strides_and_expiry(monkeypatch):
    """Samples two apart and rows inside wider ones, with infinities around; and a
    wait that gives up at once: NaN, an error, and a correct next call."""
    B, K, M, N = 6, 32, 64, 72
    wa = torch.full((2 * B, K, M + 8), float("inf"), device=DEV)
    wb = torch.full((2 * B, K, N + 4), float("inf"), device=DEV)
    a0, b0 = make(B, K, M, N, "tn", seed=8)
    a, b = wa[::2, :, 4:M + 4], wb[::2, :, :N]
    a.copy_(a0)
    b.copy_(b0)
    ref, _, _ = O.wgrad_clip(a0, b0, 1.0, 1.0, "tn")
    assert_close(core.wgrad_clip(a, b, 1.0, 1.0, single_pass="wide"), ref, torch.float32)
    monkeypatch.setenv("FDP_WGRAD_SPIN_LIMIT", "0")
    with pytest.raises(_lib.FlashDPError):
        core.wgrad_clip(a0, b0, 1.0, 1.0, single_pass="wide", check=True)
    monkeypatch.delenv("FDP_WGRAD_SPIN_LIMIT")
    out = core.wgrad_clip(a0, b0, 1.0, 1.0, single_pass="wide", check=True)
    assert_close(out, ref, torch.float32, "after the expiry")


@pytest.mark.parametrize("noclip", [False, True])
@pytest.mark.parametrize("layout", ["tn", "nn"])
def test_f32_samples_without_rows(layout, noclip):
    """K = 0: zero products, and every sample's statistics are still written."""
    B, M, N = 5, 70, 129
    a = torch.empty((B, 0, M) if layout == "tn" else (B, M, 0), device=DEV)
    b = torch.empty(B, 0, N, device=DEV)
    out, norms, fac = core.wgrad_clip(a, b, 1.0, 0.75, layout=layout, noclip=noclip,
                                      return_stats=True)
    assert torch.count_nonzero(out) == 0
    assert norms is None if noclip else torch.count_nonzero(norms) == 0
    assert torch.equal(fac.cpu(), torch.full((B,), 0.75))
