"""16-bit two-pass schedules beside the Gram one, at the edges of their rules
(csrc/wgrad_staged.hpp, prod_norm_kernel and the NN clipped sum of
csrc/wgrad_stream.hpp): rows that are not 16-byte aligned, operands narrower
than a 16-byte chunk, a contraction that fills no k-tile, exactly one, or
leaves a remainder; edge tiles of 128 x 256; grouped samples.

Against the float64 oracle on the same rounded operands: the products are
accumulated in fp32 and the fp32 output is not rounded, so fp32's bar holds
(K <= 300 terms: 300 * 2^-24 = 2e-5 of the largest partial sum at worst, and
random signs keep it below 1e-5 of the result).
"""
import numpy as np
import pytest
import torch

from oracle import dp_clip as O
from tests._tol import assert_close, assert_elementwise

from flashdp4review_amd import core

pytestmark = pytest.mark.gpu
DEV = "cuda"

SHAPES = [  # B, K, M, N
    (3, 5, 3, 2),          # rows shorter than a chunk
    (2, 33, 7, 300),       # operand a narrower than a chunk, two k-tiles
    (4, 32, 129, 257),     # one whole k-tile, odd widths, ragged tiles
    (3, 64, 128, 256),     # whole tiles and k-tiles (aligned)
    (2, 96, 130, 512),     # a ragged, b whole
    (3, 95, 261, 777),     # every edge ragged, the last k-tile too
    (5, 31, 1, 1),
    (16, 160, 200, 264),   # grouped samples, aligned
    (9, 300, 131, 513),
    # split Gram norms (TN): one and several Gram tiles a sample, ragged rows,
    # either operand the wider one, parts of unequal length
    (2, 128, 3001, 130),
    (3, 130, 70, 2049),
    (1, 257, 5003, 259),
]


def make(B, K, M, N, dtype, layout, seed=0):
    g = torch.Generator().manual_seed(seed)
    a = torch.randn((B, K, M) if layout == "tn" else (B, M, K), generator=g)
    b = torch.randn(B, K, N, generator=g) * (0.1 + torch.rand(B, 1, 1, generator=g))
    return a.to(dtype).to(DEV), b.to(dtype).to(DEV)


@pytest.mark.parametrize("layout", ["tn", "nn"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=str)
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_two_pass_parity(shape, dtype, layout):
    B, K, M, N = shape
    a, b = make(B, K, M, N, dtype, layout)
    _, norms_ref, _ = O.wgrad_clip(a, b, 1.0, 1.0, layout)
    C = float(np.median(norms_ref))
    ref, norms_ref, fac_ref = O.wgrad_clip(a, b, C, 1.0, layout)
    out, norms, fac = core.wgrad_clip(a, b, C, 1.0, layout=layout, out_dtype=torch.float32,
                                      two_pass=True, return_stats=True)
    assert_close(out, ref, torch.float32, "sum")
    assert_elementwise(norms, norms_ref, torch.float32, "norms")
    assert_elementwise(fac, fac_ref, torch.float32, "factors")
    # the same rows inside a wider allocation, one element off a 16-byte boundary,
    # with infinities in what lies around them
    def off(t):
        w = torch.full((t.shape[0], t.shape[1] + 2, t.shape[2] + 9), float("inf"), dtype=dtype,
                       device=DEV)
        v = w[:, 1:-1, 1:t.shape[2] + 1]
        v.copy_(t)
        return v
    o2, n2, _ = core.wgrad_clip(off(a), off(b), C, 1.0, layout=layout, out_dtype=torch.float32,
                                two_pass=True, return_stats=True)
    assert_close(o2, ref, torch.float32, "offset sum")
    assert_elementwise(n2, norms_ref, torch.float32, "offset norms")


def test_last_rows_of_an_allocation():
    """Operands that end with their allocation's last bytes (a whole 2 MB one):
    nothing past them is read as data."""
    B, K, M, N = 2, 40, 131, 133
    n = 1 << 20
    a, b = make(B, K, M, N, torch.bfloat16, "tn", seed=3)
    ref, _, _ = O.wgrad_clip(a, b, 1.0, 1.0, "tn")
    bufs = [torch.empty(n, dtype=torch.bfloat16, device=DEV) for _ in range(2)]
    views = []
    for t, w in zip((a, b), bufs):
        v = w[n - t.numel():].view(t.shape)
        v.copy_(t)
        views.append(v)
    out = core.wgrad_clip(*views, 1.0, 1.0, out_dtype=torch.float32, two_pass=True)
    assert_close(out, ref, torch.float32)


ROUTES = [  # B, K, M, N, whether the default is the two-pass schedule
    # several samples per workgroup in one launch (100 tiles): K of 64 and 65
    (6, 64, 1280, 1280, True),
    (6, 65, 1280, 1280, False),
    (5, 64, 1280, 1280, False),    # 500 workgroups, one sample each
    (7, 1, 1216, 1224, True),
    # several launches (21 samples each of 24 tiles; 4 of 289): K at the two limits
    (85, 400, 512, 768, True),
    (85, 401, 512, 768, False),
    (5, 600, 2120, 2120, True),
    (5, 601, 2120, 2120, False),
    # few Gram tiles: norms from the products; many: the Gram form
    (1, 22, 1472, 7232, True),
    (8, 150, 2240, 5120, True),
    (40, 70, 2048, 1024, True),
]


@pytest.mark.parametrize("route", ROUTES, ids=lambda s: "x".join(map(str, s[:4])))
def test_default_route(route):
    """The rule between the grouped single pass and the two passes, and the one
    between Gram and product norms: the oracle's result on either side."""
    B, K, M, N, two = route
    g = torch.Generator(DEV).manual_seed(B * K)
    a = torch.randn(B, K, M, generator=g, device=DEV).to(torch.bfloat16)
    b = torch.randn(B, K, N, generator=g, device=DEV).to(torch.bfloat16)
    # per-sample scales, powers of two: exact in bf16, and clipped and unclipped samples
    b *= torch.tensor([2.0 ** (i % 3) for i in range(B)], device=DEV).to(b.dtype).view(B, 1, 1)
    C = 2.0 * (K * M * N) ** 0.5
    ref = torch.zeros(M, N, dtype=torch.float64, device=DEV)
    norms_ref, fac_ref = [], []
    for i in range(B):
        G = a[i].double().t() @ b[i].double()
        norms_ref.append(G.norm())
        fac_ref.append((C / norms_ref[-1]).clamp(max=1.0))
        ref += fac_ref[-1] * G
    kw = dict(out_dtype=torch.float32, return_stats=True)
    out, norms, fac = core.wgrad_clip(a, b, C, 1.0, **kw)
    forced, _, _ = core.wgrad_clip(a, b, C, 1.0, two_pass=True, **kw)
    if two:
        assert torch.equal(out, forced)
        assert_close(out, ref.cpu().numpy(), torch.float32, "sum")
    else:  # the single pass parks its products in 16 bits
        assert_close(out, ref.cpu().numpy(), torch.bfloat16, "sum")
        assert_close(forced, ref.cpu().numpy(), torch.float32, "two-pass sum")
    assert_elementwise(norms, torch.stack(norms_ref).cpu().numpy(), torch.float32, "norms")
    assert_elementwise(fac, torch.stack(fac_ref).cpu().numpy(), torch.float32, "factors")
