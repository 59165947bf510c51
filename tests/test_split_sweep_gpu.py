"""Forward-type sweeps whose operands are split into two 16-bit halves (csrc/split_sweep.hip) against float64.

Sizes at the edges of its tiles: pixels around multiples of 128, columns around multiples of 32, channels around the
16/64/128/256 its channel steps are padded to, and pixels it cannot split (inf, NaN, magnitudes outside [2^-60, 2^61),
several channels far below the largest), which it multiplies in fp32.
"""
import ctypes

import pytest
import torch

from separableflowthesis_amd import _lib
from tests._util import assert_close, op_inputs

pytestmark = pytest.mark.gpu

# (B, H1, W1, H2, W2, C); all large enough for the split sweep: B H1 W1 H2 W2 (C + 64) of 1e9 and a little more
SHAPES = [(1, 50, 82, 74, 35, 32), (2, 40, 64, 61, 34, 33), (1, 63, 65, 33, 65, 64), (1, 51, 91, 62, 31, 65),
          (1, 36, 73, 33, 70, 128), (3, 21, 43, 55, 36, 130), (1, 47, 48, 42, 35, 255), (2, 24, 49, 27, 97, 256),
          (1, 96, 172, 401, 1, 96), (1, 48, 65, 11, 290, 48)]


def _labels_of(fn):
    """Labels of the kernels that fn() launches, by the library's own kernel timing."""
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


@pytest.mark.parametrize("dims", SHAPES, ids=str)
def test_sizes_take_the_split_sweep(device, dims):
    f1, f2 = (torch.randn(dims[0], *hw, dims[5], device=device) for hw in (dims[1:3], dims[3:5]))
    for argmax in (True, False):
        for scratch in (True, False):
            assert _labels_of(lambda: _max_avg(f1, f2, dims, scratch, argmax)) == {"fwd_maxavg_split"}


def test_three_channels_of_32_features_stay_fp32(device):
    from separableflowthesis_amd import MemorySaver
    B, H1, W1, H2, W2, C = dims = SHAPES[0]
    f1, f2 = (torch.randn(B, *hw, C, device=device) for hw in (dims[1:3], dims[3:5]))
    for K, labels in ((2, {"fwd_weighted_split"}), (3, {"fwd_weighted"}), (4, {"fwd_weighted_split"}), (7, {"fwd_weighted", "fwd_weighted_split"})):
        a_u, a_v = (torch.randn(B, H1, W1, K, n, device=device) for n in (W2, H2))
        got = []
        assert _labels_of(lambda: got.extend(MemorySaver.compression_forward(f1, f2, a_u, a_v))) == labels
        vol = _volume(f1.double(), f2.double())
        for k in range(K):
            assert torch.allclose(got[0][:, :, :, k].double(), (vol * a_u[:, :, :, k, None, :]).sum(4), rtol=1e-4, atol=1e-4)
            assert torch.allclose(got[1][:, :, :, k].double(), (vol * a_v[:, :, :, k, :, None]).sum(3), rtol=1e-4, atol=1e-4)


@pytest.mark.parametrize("mode,label", [("CONTRACT_FP32", "fwd_maxavg"), ("CONTRACT_BF16X3", "fwd_maxavg"), ("CONTRACT_SPLIT", "fwd_maxavg_split")])
def test_contraction_modes(device, mode, label):
    """fp32 products when they are asked for, also by the planes' mode where the planes do not apply (C = 128)."""
    from separableflowthesis_amd import MemorySaver
    dims = SHAPES[4]
    f1, f2, _ = op_inputs(*dims, seed=13)
    f1, f2 = f1.to(device), f2.to(device)
    previous = MemorySaver.set_contraction(getattr(MemorySaver, mode))
    try:
        assert previous == MemorySaver.CONTRACT_SPLIT
        for scratch in (True, False):
            assert _labels_of(lambda: _max_avg(f1, f2, dims, scratch)) == {label}
        B, H1, W1, H2, W2, _ = dims
        a_u, a_v = (torch.randn(B, H1, W1, 2, n, device=device) for n in (W2, H2))
        assert _labels_of(lambda: MemorySaver.compression_forward(f1, f2, a_u, a_v)) == {label.replace("maxavg", "weighted")}
    finally:
        MemorySaver.set_contraction(previous)


def _call(name, outs, ins, dims, scratch, extra=(), K=2):
    lib = _lib.load()
    h2, w2 = (ctypes.c_int * 1)(dims[3]), (ctypes.c_int * 1)(dims[4])
    n = lib.sepcorr_forward_levels_workspace_bytes(h2, w2, 1, *dims[:3], dims[5], K) if scratch else 0
    ws = torch.empty(max(n, 256), dtype=torch.uint8, device=ins[0].device)
    _lib.check(getattr(lib, name)(*(t.data_ptr() for t in ins), *(t.data_ptr() for t in outs), *dims, *extra,
                                  ws.data_ptr() if n else None, n, torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()


def _max_avg(f1, f2, dims, scratch=True, argmax=True):
    B, H1, W1, H2, W2, C = dims
    e = lambda *s, **k: torch.empty(*s, device=f1.device, **k)
    outs = [e(B, H1, W1, 2, H2), e(B, H1, W1, 2, W2)]
    if argmax:
        outs += [e(B, H1, W1, 1, H2, dtype=torch.int32), e(B, H1, W1, 1, W2, dtype=torch.int32)]
    _call("sepcorr_max_argmax_avg_forward" if argmax else "sepcorr_max_avg_forward", outs, [f1, f2], dims, scratch)
    return outs


def _volume(f1, f2):
    B, H1, W1, C = f1.shape
    return (f1.reshape(B, H1 * W1, C) @ f2.reshape(B, -1, C).transpose(1, 2).contiguous()).view(B, H1, W1, *f2.shape[1:3])


def _bound(f1, f2, extra=0):
    """Largest error of one product sum: 2^-21 of sum |a b| for what the halves do not hold, and one rounding of at most
    2^-24 of it per addition (three products per channel, `extra` additions of the reduction behind it)."""
    C = f1.shape[-1]
    return (8 + 3 * C + extra + 8) * 2.0 ** -24 * _volume(f1.double().abs(), f2.double().abs())


@pytest.mark.parametrize("dims", SHAPES, ids=str)
def test_max_argmax_avg(device, dims):
    f1, f2, _ = op_inputs(*dims, seed=5)
    vol, err = _volume(f1.double(), f2.double()), _bound(f1, f2, sum(dims[3:5]))
    out_u, out_v, am_u, am_v = (t.cpu() for t in _max_avg(f1.to(device), f2.to(device), dims))
    for out, am, d in ((out_u, am_u, 4), (out_v, am_v, 3)):
        worst = err.amax(d)
        assert ((out[:, :, :, 0] - vol.amax(d)).abs() <= worst).all()
        assert ((out[:, :, :, 1] - vol.mean(d)).abs() <= err.mean(d)).all()
        # the index points at a value that is the maximum but for the rounding of both
        at = vol.gather(d, am[:, :, :, 0].long().unsqueeze(d)).squeeze(d)
        assert (vol.amax(d) - at <= 2 * worst).all()
    plain = _max_avg(f1.to(device), f2.to(device), dims, argmax=False)
    assert torch.equal(plain[0].cpu(), out_u) and torch.equal(plain[1].cpu(), out_v)


@pytest.mark.parametrize("K", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("dims", SHAPES[1::2] + [(2, 45, 48, 46, 53, 64), (2, 45, 48, 46, 66, 40)], ids=str)
def test_weighted(device, dims, K):
    B, H1, W1, H2, W2, C = dims
    f1, f2, g = op_inputs(*dims, seed=6)
    a_u, a_v = torch.randn(B, H1, W1, K, W2, generator=g), torch.randn(B, H1, W1, K, H2, generator=g)
    outs = [torch.empty(B, H1, W1, K, H2, device=device), torch.empty(B, H1, W1, K, W2, device=device)]
    _call("sepcorr_compression_forward", outs, [t.to(device) for t in (f1, f2, a_u, a_v)], dims, True, (K,), K)
    vol, err = _volume(f1.double(), f2.double()), _bound(f1, f2, H2 + W2 + 2)
    for k in range(K):
        wu, wv = a_u[:, :, :, k, None, :].double(), a_v[:, :, :, k, :, None].double()
        assert ((outs[0][:, :, :, k].cpu() - (vol * wu).sum(4)).abs() <= (err * wu.abs()).sum(4)).all()
        assert ((outs[1][:, :, :, k].cpu() - (vol * wv).sum(3)).abs() <= (err * wv.abs()).sum(3)).all()


def _check_max_avg(got, f1, f2):
    """out_u, out_v, argmax_u, argmax_v against float64 element by element, products that fp32 cannot hold being inf."""
    C, lines = f1.shape[-1], sum(f2.shape[1:3])
    vol, err = _volume(f1.double(), f2.double()).float().double(), _bound(f1, f2, lines) + C * 2.0 ** -126   # (subnormals may be lost)
    err = torch.where(vol.isfinite(), err, torch.zeros_like(err))
    vol_max = torch.where(vol.isnan(), torch.full_like(vol, -float("inf")), vol)   # (NaN never wins)
    for out, am, d in ((got[0], got[2], 4), (got[1], got[3], 3)):
        best, mean, worst = vol_max.amax(d), vol.mean(d), err.amax(d)
        out_max, out_mean = out[:, :, :, 0].double(), out[:, :, :, 1].double()
        fin = best.isfinite()
        assert torch.equal(out_max[~fin], best[~fin]) and ((out_max - best).abs() <= worst)[fin].all()
        fin = mean.isfinite()
        assert torch.equal(out_mean[~fin].nan_to_num(12.0), mean[~fin].nan_to_num(12.0))
        assert ((out_mean - mean).abs() <= err.mean(d))[fin].all()
        at = vol_max.gather(d, am[:, :, :, 0].long().unsqueeze(d)).squeeze(d)
        assert ((at == best) | (best - at <= 2 * worst)).all()


# just inside and just outside of what has halves (a largest channel in [2^-60, 2^61)), far outside, and what is no number
@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan"), 0.0] + [2.0 ** e for e in (30, 60, 61, 100, -30, -60, -61, -100)])
@pytest.mark.parametrize("where", ["f1", "f2", "both"])
@pytest.mark.parametrize("C", [48, 256])
def test_pixels_without_halves(device, value, where, C):
    dims = (1, 50, 81, 62, 40, C)
    f1, f2, _ = op_inputs(*dims, seed=7)
    if where != "f2":
        f1[0, 3, 7] = value if abs(value) < 1 else f1[0, 3, 7]   # a whole tiny (or zero) pixel, or one large channel
        f1[0, 3, 7, 11] = value
    if where != "f1":
        f2[0, 30, 39] = value if abs(value) < 1 else f2[0, 30, 39]
        f2[0, 30, 39, 11] = value
    _check_max_avg([t.cpu() for t in _max_avg(f1.to(device), f2.to(device), dims)], f1, f2)


@pytest.mark.parametrize("dims", [(1, 48, 65, 41, 61, 100), (2, 48, 40, 41, 35, 255)], ids=str)
def test_whole_maps_without_halves(device, dims):
    """Every block in fp32: channels that are no multiple of a turn, pixels and columns that are no multiple of a block."""
    f1, f2, _ = op_inputs(*dims, seed=12)
    f1 *= 2.0 ** 70
    _check_max_avg([t.cpu() for t in _max_avg(f1.to(device), f2.to(device), dims)], f1, f2)


def _outlier(f1, f2, r, g):
    f1[..., 0], f2[..., 0] = 2.0 ** r, 0.0


def _outliers_on_both_sides(f1, f2, r, g):
    f1[..., 0], f2[..., 0] = 2.0 ** r, 0.0
    f1[..., 1], f2[..., 1] = 0.0, 2.0 ** r


def _channel_scales(f1, f2, r, g):
    s = 2.0 ** torch.randint(-r // 2, r // 2 + 1, f1.shape[-1:], generator=g)
    s[0] = 1.0
    f1 *= s
    f2 /= s


@pytest.mark.parametrize("C", [256, 64])
@pytest.mark.parametrize("mode", ["max_avg", 1, 4])
@pytest.mark.parametrize("change", [_outlier, _outliers_on_both_sides, _channel_scales])
def test_range_within_a_pixel(device, change, mode, C):
    """Channels of very different magnitude within a pixel.  None of the changes alters a product that is not zero, so the
    error (2-norm) stays what it is without them, but for the larger one of blocks that are multiplied in fp32: a sum of
    256 products is rounded 128 times there and 16 times (the small cross terms aside) with halves, which gives sqrt(8)
    times the error; 3 times is allowed."""
    dims = (1, 48, 64, 47, 64, C)
    B, H1, W1, H2, W2, _ = dims
    errors = {}
    for r in (None, 12, 18, 20, 22, 24, 27, 32, 48):
        f1, f2, g = op_inputs(*dims, seed=11)
        for f in (f1, f2):
            f[..., :2] = 0.0
        weights = [torch.randn(B, H1, W1, mode, n, generator=g) for n in (W2, H2)] if mode != "max_avg" else []
        if r is not None:
            change(f1, f2, r, g)
        vol = _volume(f1.double(), f2.double())
        if mode == "max_avg":
            out_u, out_v = (t.cpu().double() for t in _max_avg(f1.to(device), f2.to(device), dims)[:2])
            got = [out_u[:, :, :, 1], out_v[:, :, :, 1], out_u[:, :, :, 0], out_v[:, :, :, 0]]
            want = [vol.mean(4), vol.mean(3), vol.amax(4), vol.amax(3)]
        else:
            outs = [torch.empty(B, H1, W1, mode, n, device=device) for n in (H2, W2)]
            _call("sepcorr_compression_forward", outs, [t.to(device) for t in [f1, f2] + weights], dims, True, (mode,), mode)
            got = [t.cpu().double() for t in outs]
            want = [torch.stack([(vol * weights[0][:, :, :, k, None, :]).sum(4) for k in range(mode)], 3),
                    torch.stack([(vol * weights[1][:, :, :, k, :, None]).sum(3) for k in range(mode)], 3)]
        errors[r] = [((a - b).norm() / b.norm()).item() for a, b in zip(got, want)]
    print(errors)
    for r, error in errors.items():
        assert all(e <= 3 * e0 for e, e0 in zip(error, errors[None])), (r, error, errors[None])


@pytest.mark.parametrize("magnitude", [1.0, 2.0 ** -20])
def test_large_products_stay_finite(device, magnitude):
    """Products up to 2^126 and weights up to 2^112 come out finite where their sums are: an fmap2 channel of +-2^e beside
    features of `magnitude` (one of 2^120 has no halves and is multiplied in fp32)."""
    dims = (1, 50, 82, 74, 35, 32)
    B, H1, W1, H2, W2, C = dims
    f1, f2, g = op_inputs(*dims, seed=10)
    f1 = f1 * magnitude
    f1[..., 11] = magnitude
    for e, u, v in ((120, 30, 20), (100, 50, 33), (22, 60, 3)):
        f2[0, u, v, 11], f2[0, u + 5, v, 11] = 2.0 ** e, -2.0 ** e
    vol, err = _volume(f1.double(), f2.double()), _bound(f1, f2, H2 + W2)
    out_u, out_v = (t.cpu().double() for t in _max_avg(f1.to(device), f2.to(device), dims)[:2])
    for out, d in ((out_u, 4), (out_v, 3)):
        assert out.isfinite().all()
        assert ((out[:, :, :, 0] - vol.amax(d)).abs() <= err.amax(d)).all()
        assert ((out[:, :, :, 1] - vol.mean(d)).abs() <= err.mean(d)).all()
    # the weights take the place of the large features: the sums stay below 2^124
    f2.clamp_(-8, 8)
    a_u, a_v = (torch.randn(B, H1, W1, 4, n, generator=g) * 2.0 ** 112 for n in (W2, H2))
    vol, err = _volume(f1.double(), f2.double()), _bound(f1, f2, H2 + W2 + 2)
    for K in (1, 4):
        outs = [torch.empty(B, H1, W1, K, n, device=device) for n in (H2, W2)]
        ws = [a_u[:, :, :, :K].contiguous(), a_v[:, :, :, :K].contiguous()]
        _call("sepcorr_compression_forward", outs, [t.to(device) for t in [f1, f2] + ws], dims, True, (K,), K)
        for k in range(K):
            wu, wv = a_u[:, :, :, k, None, :].double(), a_v[:, :, :, k, :, None].double()
            assert ((outs[0][:, :, :, k].cpu() - (vol * wu).sum(4)).abs() <= (err * wu.abs()).sum(4)).all()
            assert ((outs[1][:, :, :, k].cpu() - (vol * wv).sum(3)).abs() <= (err * wv.abs()).sum(3)).all()


def test_without_scratch_the_same_bits(device):
    dims = SHAPES[7]
    f1, f2, _ = op_inputs(*dims, seed=9)
    for a, b in zip(_max_avg(f1.to(device), f2.to(device), dims), _max_avg(f1.to(device), f2.to(device), dims, scratch=False)):
        assert torch.equal(a, b)


def test_small_features_keep_their_accuracy(device):
    """Every pixel has a scale of its own: features of 1e-6 beside features of 1e6 lose nothing."""
    dims = (1, 48, 96, 30, 64, 64)
    f1, f2, g = op_inputs(*dims, seed=8)
    f1 *= 10.0 ** torch.randint(-6, 7, f1.shape[:3] + (1,), generator=g)
    f2 *= 10.0 ** torch.randint(-6, 7, f2.shape[:3] + (1,), generator=g)
    vol, err = _volume(f1.double(), f2.double()), _bound(f1, f2, sum(dims[3:5]))
    out_u, out_v = (t.cpu() for t in _max_avg(f1.to(device), f2.to(device), dims)[:2])
    assert ((out_u[:, :, :, 0] - vol.amax(4)).abs() <= err.amax(4)).all()
    assert ((out_v[:, :, :, 1] - vol.mean(3)).abs() <= err.mean(3)).all()


@pytest.mark.parametrize("dims", [(4, 64, 64, 64, 64, 128), (8, 32, 64, 33, 61, 100), (4, 64, 64, 16, 64, 64)], ids=str)
def test_dense_max_avg_backward_on_two_streams(device, dims):
    """Whole tiles and up to 128 channels: d_f1 and d_f2 run beside each other with the workspace that they would share
    otherwise.  The same bits as one after the other (as the library's kernel timing runs them)."""
    from separableflowthesis_amd import MemorySaver
    B, H1, W1, H2, W2, C = dims
    f1, f2 = (torch.randn(B, *hw, C, device=device) for hw in ((H1, W1), (H2, W2)))
    _, _, am_u, am_v = _max_avg(f1, f2, dims)
    g_u, g_v = (torch.randn(B, H1, W1, 2, n, device=device) for n in (H2, W2))
    previous = MemorySaver.set_max_avg_backward(MemorySaver.MAXAVG_DENSE)
    try:
        call = lambda: MemorySaver.max_argmax_avg_backward(f1, f2, am_u, am_v, g_u, g_v)
        serial = []
        _labels_of(lambda: serial.extend(call()))
        for _ in range(5):
            assert all(torch.equal(a, b) for a, b in zip(call(), serial))
    finally:
        MemorySaver.set_max_avg_backward(previous)


@pytest.mark.parametrize("K", [1, 3, 4])
@pytest.mark.parametrize("dims", [SHAPES[2], SHAPES[6], SHAPES[7], (2, 45, 48, 46, 66, 40)], ids=str)
def test_softmax_inside(device, dims, K):
    """Weights from logits and gradients of the logits, rows of odd length and of 2 more than a multiple of 4."""
    from separableflowthesis_amd import MemorySaver as ms
    B, H1, W1, H2, W2, C = dims
    f1, f2, g = op_inputs(*dims, seed=14)
    z_u, z_v = 3 * torch.randn(B, H1, W1, K, W2, generator=g), 3 * torch.randn(B, H1, W1, K, H2, generator=g)
    g_cu, g_cv = torch.randn(B, H1, W1, K, H2, generator=g), torch.randn(B, H1, W1, K, W2, generator=g)
    f1, f2, z_u, z_v, g_cu, g_cv = (t.to(device) for t in (f1, f2, z_u, z_v, g_cu, g_cv))
    labels = _labels_of(lambda: ms.compression_forward_from_logits(f1, f2, z_u, z_v))
    assert "fwd_weighted_split" in labels
    cu, cv, st_u, st_v = ms.compression_forward_from_logits(f1, f2, z_u, z_v)
    dz_u, dz_v = ms.compression_backward_from_logits(f1, f2, z_u, z_v, st_u, st_v, cu, cv, g_cu, g_cv, need_features=False)[2:]
    vol = _volume(f1.double(), f2.double())
    a_u, a_v = z_u.double().softmax(-1), z_v.double().softmax(-1)
    over_v = lambda w: torch.stack([(vol * w[:, :, :, k, None, :]).sum(4) for k in range(K)], 3)
    over_u = lambda w: torch.stack([(vol * w[:, :, :, k, :, None]).sum(3) for k in range(K)], 3)
    assert_close(cu.cpu(), over_v(a_u).cpu(), "compression_output_u")
    assert_close(cv.cpu(), over_u(a_v).cpu(), "compression_output_v")
    for got, a, d, name in ((dz_u, a_u, over_u(g_cu.double()), "d_logits_u"), (dz_v, a_v, over_v(g_cv.double()), "d_logits_v")):
        assert_close(got.cpu(), (a * (d - (a * d).sum(-1, keepdim=True))).cpu(), name, scale_atol=True)


def test_levels_with_pixels_without_halves(device):
    """Every level of a pyramid in one launch, pixels of image 1 and of each level that are multiplied in fp32."""
    from separableflowthesis_amd import MemorySaver as ms
    B, H, W, C = 2, 41, 67, 72
    f1, f2, _ = op_inputs(B, H, W, H, W, C, seed=15)
    levels = [f2[:, :H >> l, :W >> l].contiguous() for l in range(4)]
    f1[1, 20, 33, 5], f1[0, 40, 66, 71] = float("nan"), 2.0 ** 70
    for l, value in enumerate((float("inf"), 2.0 ** 64, float("nan"), 2.0 ** -70)):
        levels[l][l % 2, (H >> l) - 1, (W >> l) - 1] *= 2.0 ** -60 if value < 1 else 1.0
        levels[l][l % 2, (H >> l) - 1, (W >> l) - 1, 9] = value
    on_gpu = [t.to(device) for t in levels]
    got = []
    assert _labels_of(lambda: got.extend(ms.max_argmax_avg_forward_levels(f1.to(device), on_gpu))) == {"fwd_maxavg_levels_split"}
    for outs, f in zip(got, levels):
        _check_max_avg([t.cpu() for t in outs], f1, f)


@pytest.mark.parametrize("K", [0, 1, 2, 4])
def test_pixel_range_in_slabs(device, K):
    """With argmax and with four channels there is more of out_u's parts than one launch may leave in scratch (96 MiB): the
    pixel range is cut into two slabs (checked in float64 on the GPU)."""
    dims = (1, 199, 201, 61, 99, 32)
    B, H1, W1, H2, W2, C = dims
    f1, f2 = (torch.randn(B, *hw, C, device=device) for hw in (dims[1:3], dims[3:5]))
    if K:
        a_u, a_v = (torch.randn(B, H1, W1, K, n, device=device) for n in (W2, H2))
        outs = [torch.empty(B, H1, W1, K, n, device=device) for n in (H2, W2)]
        _call("sepcorr_compression_forward", outs, [f1, f2, a_u, a_v], dims, True, (K,), K)
    else:
        outs = _max_avg(f1, f2, dims)
    for rows in torch.arange(H1, device=device).split(25):
        vol = _volume(f1[:, rows].double(), f2.double())
        if K:
            for k in range(K):
                for out, w, d in ((outs[0], a_u[:, rows, :, k, None, :], 4), (outs[1], a_v[:, rows, :, k, :, None], 3)):
                    want = (vol * w).sum(d)
                    assert ((out[:, rows, :, k] - want).norm() <= 1e-6 * want.norm()).item()
        else:
            for out, am, d in ((outs[0], outs[2], 4), (outs[1], outs[3], 3)):
                assert ((out[:, rows, :, 0] - vol.amax(d)).norm() <= 1e-6 * vol.amax(d).norm()).item()
                assert ((out[:, rows, :, 1] - vol.mean(d)).norm() <= 1e-6 * vol.mean(d).norm()).item()
                at = vol.gather(d, am[:, rows, :, 0].long().unsqueeze(d)).squeeze(d)
                assert (vol.amax(d) - at <= 1e-5 * vol.amax(d)).all()


def _shifted(t):
    """A contiguous copy whose first element lies 4 bytes past a 256-byte boundary."""
    view = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)[1:].view(t.shape)
    view.copy_(t)
    assert view.data_ptr() % 8 == 4
    return view


@pytest.mark.parametrize("dims", [SHAPES[2], SHAPES[4], (2, 45, 48, 46, 64, 40), SHAPES[6]], ids=str)
def test_tensors_aligned_to_4_bytes(device, dims):
    B, H1, W1, H2, W2, C = dims
    f1, f2 = (torch.randn(B, *hw, C, device=device) for hw in (dims[1:3], dims[3:5]))
    e = lambda *s, **k: torch.empty(*s, device=device, **k)
    max_avg = [e(B, H1, W1, 2, H2), e(B, H1, W1, 2, W2), e(B, H1, W1, 1, H2, dtype=torch.int32), e(B, H1, W1, 1, W2, dtype=torch.int32)]
    calls = [("sepcorr_max_argmax_avg_forward", max_avg, [f1, f2], (), 2)]
    for K in (1, 2, 4):
        a_u, a_v = (torch.randn(B, H1, W1, K, n, device=device) for n in (W2, H2))
        calls.append(("sepcorr_compression_forward", [e(B, H1, W1, K, H2), e(B, H1, W1, K, W2)], [f1, f2, a_u, a_v], (K,), K))
    for name, outs, ins, extra, K in calls:
        _call(name, outs, ins, dims, True, extra, K)
        shifted = [_shifted(t) for t in outs]
        for t in shifted:
            t.fill_(7)
        _call(name, shifted, [_shifted(t) for t in ins], dims, True, extra, K)
        assert all(torch.equal(a, b) for a, b in zip(outs, shifted)), name


@pytest.mark.parametrize("dims", [SHAPES[1], SHAPES[5], SHAPES[7], (4, 48, 64, 48, 64, 256)], ids=str)
def test_workspaces_of_exactly_the_quoted_size(device, dims):
    """What each query gives is enough and nothing behind it is written."""
    from separableflowthesis_amd import MemorySaver
    lib, stream = _lib.load(), torch.cuda.current_stream().cuda_stream
    B, H1, W1, H2, W2, C = dims
    f1, f2 = (torch.randn(B, *hw, C, device=device) for hw in (dims[1:3], dims[3:5]))
    e = lambda *s, **k: torch.empty(*s, device=device, **k)
    P = lambda t: t.data_ptr()

    def guarded(n, call):
        ws = torch.full((n + 4096,), 0x5A, dtype=torch.uint8, device=device)
        _lib.check(call(P(ws), n))
        assert (ws[n:] == 0x5A).all()

    outs = [e(B, H1, W1, 2, H2), e(B, H1, W1, 2, W2), e(B, H1, W1, 1, H2, dtype=torch.int32), e(B, H1, W1, 1, W2, dtype=torch.int32)]
    n = lib.sepcorr_forward_workspace_bytes(*dims, 2)
    assert n > 0
    guarded(n, lambda ws, n: lib.sepcorr_max_avg_forward(P(f1), P(f2), P(outs[0]), P(outs[1]), *dims, ws, n, stream))
    guarded(n, lambda ws, n: lib.sepcorr_max_argmax_avg_forward(P(f1), P(f2), *(P(t) for t in outs), *dims, ws, n, stream))
    for K in (3, 7):
        a_u, a_v = (torch.randn(B, H1, W1, K, m, device=device) for m in (W2, H2))
        g_cu, g_cv = torch.randn_like(a_v), torch.randn_like(a_u)
        c_u, c_v, d_u, d_v, st_u, st_v = (torch.empty_like(t) for t in (a_v, a_u, a_u, a_v, a_u[..., :2], a_v[..., :2]))
        d_f1, d_f2 = torch.empty_like(f1), torch.empty_like(f2)
        guarded(lib.sepcorr_forward_workspace_bytes(*dims, K), lambda ws, n: lib.sepcorr_compression_forward_from_logits(
            P(f1), P(f2), P(a_u), P(a_v), P(c_u), P(c_v), P(st_u), P(st_v), 0, *dims, K, ws, n, stream))
        for feat in (0, 1):
            guarded(lib.sepcorr_compression_backward_from_logits_workspace_bytes(*dims, K, feat),
                    lambda ws, n: lib.sepcorr_compression_backward_from_logits(
                        P(f1), P(f2), P(a_u), P(a_v), P(st_u), P(st_v), P(c_u), P(c_v), P(g_cu), P(g_cv), P(d_f1) if feat else None,
                        P(d_f2) if feat else None, P(d_u), P(d_v), *dims, K, ws, n, stream))
        guarded(lib.sepcorr_backward_workspace_bytes(*dims), lambda ws, n: lib.sepcorr_compression_backward(
            P(f1), P(f2), P(a_u), P(a_v), P(g_cu), P(g_cv), P(d_f1), P(d_f2), P(d_u), P(d_v), *dims, K, ws, n, stream))
