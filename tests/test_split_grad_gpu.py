"""Feature gradients whose operands are split into two 16-bit halves (csrc/split_grad.hip) against float64.

Sizes at the edges of its tiles: pixels around multiples of 16 and 128, rows around multiples of 8, columns around
multiples of 32 and rows that are no multiple of 4 long (their weights are laid out anew), channels around the 64/128/256
they are padded to, tiles around the number of workgroups; and operands that have no halves, which it multiplies in fp32.
"""
import ctypes

import pytest
import torch

from separableflowthesis_amd import _lib
from tests._util import op_inputs

pytestmark = pytest.mark.gpu

# (B, H1, W1, H2, W2, C), B H1 W1 H2 W2 (C + 64) above the lines of split_grad_line() alone and combined; weight channels
SHAPES = [((1, 30, 82, 74, 35, 32), 1), ((3, 31, 64, 61, 36, 33), 4), ((1, 63, 65, 33, 65, 64), 3), ((1, 87, 91, 62, 32, 65), 2),
          ((1, 74, 64, 33, 68, 128), 4), ((6, 21, 43, 55, 36, 130), 1), ((2, 47, 48, 42, 36, 255), 3), ((2, 24, 49, 27, 97, 256), 2),
          ((1, 16, 8, 136, 240, 256), 4), ((2, 136, 120, 8, 24, 256), 4), ((2, 43, 47, 17, 100, 256), 6)]


# More tiles than workgroups (256), or as many: tiles of d_f1 x their steps, tiles of d_f2 x theirs.  Up to 48 steps a tile's
# sums stay in registers, above that what a workgroup has of it passes through its slot.
MANY_TILES = [((33, 32, 32, 64, 32, 32), 1),     # 264 x 64, 264 x 64
              ((32, 32, 32, 49, 32, 32), 2),     # 256 x 49, 224 x 64
              ((33, 24, 32, 64, 32, 64), 1),     # 198 x 64, 264 x 48
              ((33, 32, 32, 24, 64, 40), 1),     # 264 x 48, 198 x 64
              ((12, 64, 128, 49, 8, 33), 1),     # 768 x 49, 84 x 512: three tiles a workgroup
              ((12, 28, 28, 128, 128, 32), 1),   # 84 x 512, 768 x 49
              ((7, 61, 83, 51, 37, 100), 3)]     # 280 x 102, 98 x 317


def _tensors(device, dims, K, seed=0):
    B, H1, W1, H2, W2, C = dims
    f1, f2, g = op_inputs(*dims, seed=seed)
    r = lambda *s: torch.randn(*s, generator=g)
    x = dict(f1=f1, f2=f2, a_u=r(B, H1, W1, K, W2).softmax(-1), a_v=r(B, H1, W1, K, H2).softmax(-1), g_cu=r(B, H1, W1, K, H2),
             g_cv=r(B, H1, W1, K, W2), g_u=r(B, H1, W1, 2, H2), g_v=r(B, H1, W1, 2, W2))
    x["am_u"] = torch.randint(-1, W2 + 1, (B, H1, W1, 1, H2), generator=g, dtype=torch.int32)   # (one entry each side out of range)
    x["am_v"] = torch.randint(-1, H2 + 1, (B, H1, W1, 1, W2), generator=g, dtype=torch.int32)
    return {k: v.to(device) for k, v in x.items()}


def _run(x, both, add=None):
    from separableflowthesis_amd import MemorySaver as M
    if both:
        return M.fused_backward(x["f1"], x["f2"], x["am_u"], x["am_v"], x["g_u"], x["g_v"], x["a_u"], x["a_v"], x["g_cu"], x["g_cv"],
                                add_to_grad_fmap1=add)
    return M.compression_backward(x["f1"], x["f2"], x["a_u"], x["a_v"], x["g_cu"], x["g_cv"])[:2]


def _exact(x, both):
    """d_f1, d_f2 in 64 bits, dL/dS of one row of image 1 at a time."""
    d = {k: v.double() for k, v in x.items()}
    B, H1, W1, C = x["f1"].shape
    H2, W2 = x["f2"].shape[1:3]
    d1, d2 = torch.zeros_like(d["f1"]), torch.zeros_like(d["f2"])
    u, v = torch.arange(H2, device=d1.device), torch.arange(W2, device=d1.device)
    for b in range(B):
        for i in range(H1):
            G = torch.matmul(d["g_cu"][b, i].transpose(1, 2).contiguous(), d["a_u"][b, i]) + torch.matmul(d["a_v"][b, i].transpose(1, 2).contiguous(), d["g_cv"][b, i])
            if both:
                G += d["g_u"][b, i, :, 0, :, None] * (x["am_u"][b, i, :, 0, :, None] == v) + d["g_u"][b, i, :, 1, :, None] / W2
                G += d["g_v"][b, i, :, 0, None, :] * (x["am_v"][b, i, :, 0, None, :] == u[:, None]) + d["g_v"][b, i, :, 1, None, :] / H2
            G = G.reshape(W1, H2 * W2)
            d1[b, i] = G @ d["f2"][b].reshape(-1, C)
            d2[b] += (G.t().contiguous() @ d["f1"][b, i]).reshape(H2, W2, C)
    return d1, d2


def _rel(got, ref):
    return float((got.double() - ref).norm() / ref.norm())


class _Contraction:
    def __init__(self, mode):
        self.mode = mode

    def __enter__(self):
        self.old = _lib.load().sepcorr_set_contraction(self.mode)

    def __exit__(self, *a):
        _lib.load().sepcorr_set_contraction(self.old)


def _labels_of(fn):
    lib = _lib.load()
    lib.sepcorr_profile_enable(1)
    try:
        fn()
        torch.cuda.synchronize()
    finally:
        names, ms = ctypes.create_string_buffer(1 << 14), (ctypes.c_float * 256)()
        n = lib.sepcorr_profile_collect(names, len(names), ms, 256)
        lib.sepcorr_profile_enable(0)
    return set(names.value.decode().split("\n")[:n])


@pytest.mark.parametrize("both", [False, True], ids=["compression", "combined"])
@pytest.mark.parametrize("dims,K", SHAPES + MANY_TILES, ids=str)
def test_against_float64(device, dims, K, both):
    x = _tensors(device, dims, K, seed=K)
    got = []
    kind = "both" if both else "comp"
    assert {f"df1_{kind}_split", f"df2_{kind}_split"} <= _labels_of(lambda: got.extend(_run(x, both)))
    ref = _exact(x, both)
    # An operand's halves hold 22 bits (an error of 2^-23 of it at the most, 0.7e-7 in the mean), dL/dS itself is a sum of up to 15
    # fp32 terms, and at most 96 sums follow one another before they are put apart: 1.3e-7 to 1.9e-7 for d_f1 and up to
    # 3.3e-7 for d_f2 were seen; the fp32 kernels make 1.9e-7 to 2.4e-7 and 2e-7 to 9e-7.
    assert _rel(got[0], ref[0]) < 3e-7 and _rel(got[1], ref[1]) < 5e-7
    again = _run(x, both)
    assert torch.equal(got[0], again[0]) and torch.equal(got[1], again[1])
    if both:
        base = torch.randn(x["f1"].shape, device=device)
        added = _run(x, both, add=base.clone())[0]
        # (more than four weight channels come in two parts, the second of which is added to base + the first)
        assert torch.equal(added, base + got[0]) if K <= 4 else _rel(added, base.double() + got[0]) < 1e-6


@pytest.mark.parametrize("both", [False, True], ids=["compression", "combined"])
@pytest.mark.parametrize("what", ["avoided 12", "avoided 40", "one loud pixel", "small at random", "peaks", "masked", "tiny"])
def test_every_row_by_itself(device, what, both):
    """Rows of d_f2 that all attention avoids, or that only pixels with small gradients reach, and rows of d_f1 of such pixels."""
    B, H1, W1, H2, W2, C = dims = (1, 40, 53, 90, 56, 128)
    x = _tensors(device, dims, 3, seed=5)
    g = torch.Generator(device=device).manual_seed(6)
    zu, zv = (torch.randn(x[k].shape, generator=g, device=device) for k in ("a_u", "a_v"))
    size = torch.ones(B, H1, W1, 1, 1, device=device)
    if "avoided" in what:   # the last columns and rows
        zu[..., W2 // 2 + 1:] -= float(what.split()[1])
        zv[..., H2 // 2 + 1:] -= float(what.split()[1])
    else:                   # every pixel looks at its own place
        j, v = torch.arange(W1, device=device), torch.arange(W2, device=device)
        i, u = torch.arange(H1, device=device), torch.arange(H2, device=device)
        zu -= 5 * (v - j.clamp(max=W2 - 1)[:, None]).abs().clamp(max=4).view(1, 1, W1, 1, W2)
        zv -= 5 * (u - i.clamp(max=H2 - 1)[:, None]).abs().clamp(max=4).view(1, H1, 1, 1, H2)
    if what == "one loud pixel":   # (one product of dL/dS: a sum of several may cancel, and rows that have this pixel's alone show it)
        size[0, 11, 17] = 2.0 ** 40
        x["g_cu"][0, 11, 17, 1:] = 0
        x["g_cv"][0, 11, 17] = 0
    if what == "small at random": size = torch.exp2(-torch.randint(0, 41, size.shape, generator=g, device=device))
    if what == "masked":
        size[:, :13] = 0
        size[:, 20:, 9] = 2.0 ** -30
    if what == "tiny":
        size *= 2.0 ** -80
        x["f1"] *= 2.0 ** -20
    x["a_u"], x["a_v"] = zu.softmax(-1), zv.softmax(-1)
    for k in ("g_cu", "g_cv"): x[k] *= size
    for k in ("g_u", "g_v"): x[k] *= size * 2.0 ** -60   # (the rest of dL/dS is not to be covered by the averages)
    got = []
    kind = "both" if both else "comp"
    assert {f"df1_{kind}_split", f"df2_{kind}_split"} <= _labels_of(lambda: got.extend(_run(x, both)))
    ref = _exact(x, both)
    for a, r in zip(got, ref):
        # Halves hold 22 bits, the products of two low ones are left out: 3 2^-23 of a product at the most, 0.7e-7 in the mean, and
        # fp32 sums on top; up to 2.5e-7 of a row's length were seen, up to 3.1e-7 from the fp32 kernels.
        assert bool(((a.double() - r).norm(dim=-1) <= 6e-7 * r.norm(dim=-1)).all())


def test_sums_are_not_biased(device):
    """The 16-bit matrix instructions round down; the signs turned in every other row keep that out of the mean."""
    x = _tensors(device, (1, 16, 64, 136, 240, 256), 2)
    for got, ref in zip(_run(x, False), _exact(x, False)):
        err = got.double() - ref
        assert abs(float(err.mean())) < 0.05 * float(err.pow(2).mean().sqrt())


@pytest.mark.parametrize("what", ["f2 inf", "f1 nan", "g nan", "weight inf", "tiny", "huge", "one large", "zero gradients"])
@pytest.mark.parametrize("both", [False, True], ids=["compression", "combined"])
def test_operands_without_halves(device, what, both):
    # (two channels with the max/average terms: the fp32 kernels then take them in one pass too, and inf comes out alike)
    dims, K = ((4, 24, 49, 27, 52, 256), 2) if both else ((1, 41, 91, 62, 35, 65), 3)
    x = _tensors(device, dims, K)
    if what == "f2 inf": x["f2"][0, 3, 4, 5] = float("inf")
    if what == "f1 nan": x["f1"][0, 3, 4, 5] = float("nan")
    if what == "g nan": x["g_cu"][0, 3, 4, 1, 6] = float("nan")
    if what == "weight inf": x["a_v"][0, 3, 4, 1, 6] = float("inf")
    if what == "tiny": x["f1"] *= 1e-25
    if what == "huge": x["f2"] *= 1e25
    if what == "one large": x["f2"][0, 3, 4, 5] = 2.0 ** 24
    if what == "zero gradients":
        for k in ("g_cu", "g_cv", "g_u", "g_v"): x[k][:, :12] = 0
    got = _run(x, both)
    with _Contraction(0):
        ref = _run(x, both)
    for a, b in zip(got, ref):
        assert torch.equal(a.isnan(), b.isnan()) and torch.equal(a.isinf(), b.isinf())
        fin = b.isfinite()
        if fin.any():   # sums of the same fp32 products in another order
            assert float((a - b)[fin].double().norm()) <= 2e-6 * float(b[fin].double().norm())


@pytest.mark.parametrize("both", [False, True], ids=["compression", "combined"])
@pytest.mark.parametrize("dims,K", SHAPES + MANY_TILES, ids=str)
def test_fp32_contraction_against_float64(device, dims, K, both):
    x = _tensors(device, dims, K, seed=K)
    x["f2"][..., 0] *= 2.0 ** -20   # (a channel of small values beside one large one: more than one feature in 2048)
    x["f2"][:, 0, 0, 0] = 1
    got, ref = _run(x, both), _exact(x, both)
    # fp32 products, 128 of them in a register sum and up to a hundred such sums in another, dL/dS itself a sum of up to 15 fp32
    # terms: each rounding is 2^-25 of its sum in the mean, of a random walk of n terms about (n / 3)^0.5 of that in all, 2e-7 for
    # both sums together; 1.3e-7 to 2.7e-7 were seen
    assert _rel(got[0], ref[0]) < 4e-7 and _rel(got[1], ref[1]) < 4e-7
    again = _run(x, both)
    assert torch.equal(got[0], again[0]) and torch.equal(got[1], again[1])


def test_scratch_and_alignment(device):
    """Less scratch than the query gives, and weights at addresses that are no multiple of 16: the same gradients."""
    dims, K = (4, 24, 49, 27, 52, 256), 2
    x = _tensors(device, dims, K)
    ref = _run(x, False)
    y = dict(x)
    for k in ("a_u", "g_cv"):
        flat = torch.empty(x[k].numel() + 1, device=device)[1:]
        flat.copy_(x[k].flatten())
        y[k] = flat.view(x[k].shape)
    got = _run(y, False)
    assert all(_rel(a, b.double()) < 1e-6 for a, b in zip(got, ref))
    lib = _lib.load()
    n = lib.sepcorr_backward_workspace_bytes(*dims)
    ws = torch.empty(n, dtype=torch.uint8, device=device)
    d = [torch.empty_like(x[k]) for k in ("f1", "f2", "a_u", "a_v")]
    _lib.check(lib.sepcorr_compression_backward(*[x[k].data_ptr() for k in ("f1", "f2", "a_u", "a_v", "g_cu", "g_cv")],
                                                *[t.data_ptr() for t in d], *dims, K, ws.data_ptr(), n - 256,
                                                torch.cuda.current_stream().cuda_stream))
    with _Contraction(0):
        fp32 = _run(x, False)
    assert torch.equal(d[0], fp32[0]) and torch.equal(d[1], fp32[1])


def test_replayed_graph(device):
    x = _tensors(device, (4, 24, 49, 27, 52, 256), 4)
    ref = _run(x, True)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        _run(x, True)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = _run(x, True)
    for _ in range(3):
        out[0].zero_()
        out[1].zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out[0], ref[0]) and torch.equal(out[1], ref[1])
