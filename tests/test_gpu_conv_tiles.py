"""The f16 conv's tiles: every tile of a tap class against float64, at lengths around its tile edges, and
the same lanes alone and in a batch (another tile, the same bits: all tiles of a class sum an output in
one order). That the rows below reach every tile is held in test_conv_tile_choice.py."""
import pytest
import torch

from dtts import nlc

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    return torch.device("cuda:0")


def _inputs(lanes, length, cin, cout, k, dev):
    g = torch.Generator(device=dev)
    g.manual_seed(lanes * 1000003 + length * 101 + cin + cout + k)
    x = torch.randn((lanes, length, cin), generator=g, device=dev).half()
    w = (torch.randn((cout, k * cin), generator=g, device=dev) / (k * cin) ** 0.5).half()
    b = (torch.randn((cout,), generator=g, device=dev) * 0.1).half()
    return x, w, b


def _f64(x, w, b, k, dil):
    cin, length = x.shape[2], x.shape[1]
    x64, w64 = x.double(), w.double()
    y = b.double().expand(x.shape[0], length, -1).clone()
    for t in range(k):
        off = (k - 1 - t) * dil
        if off < length:
            for i in range(x.shape[0]):
                y[i, off:] += x64[i, : length - off] @ w64[:, t * cin:(t + 1) * cin].t().contiguous()
    return y


# f16 operands are exact in the products; an f32 sum of up to 5376 unit-scale terms in MFMA order is
# within 1e-4 of exact, and the result is rounded to f16 once: half an ulp, 2^-11 relative.
def _check(y, ref):
    bound = 2.0 ** -11 * 1.001 * ref.abs() + 1e-4
    assert torch.isfinite(y).all()
    assert ((y.double() - ref).abs() <= bound).all()


# lanes, length, cin, cout, k, dilation
ROWS = [
    # k <= 7: 128x32, 128x64, 128x96, 256x96, 512x96 and their edges; a run-time tap count
    (1, 1, 64, 96, 7, 1), (1, 25, 1024, 1536, 7, 1), (1, 127, 96, 96, 7, 9), (1, 129, 96, 64, 7, 9), (2, 200, 768, 768, 7, 3),
    (4, 250, 512, 1536, 7, 1), (1, 385, 192, 192, 7, 9), (8, 500, 384, 768, 7, 3), (4, 2001, 384, 768, 7, 3),
    (3, 3000, 384, 384, 7, 9), (24, 1025, 192, 768, 7, 1), (24, 2047, 96, 768, 7, 9), (2, 33, 64, 1024, 3, 1), (3, 511, 32, 32, 5, 2),
    (24, 501, 96, 192, 7, 9),
    # ... and the register-staged tiles of widths that are no multiple of 96
    (170, 100, 64, 64, 5, 1), (170, 257, 32, 32, 3, 2), (30, 701, 64, 160, 7, 9),
    # k = 2: 64x64, 128x128, 256x128, 128x96
    (1, 25, 1536, 6144, 2, 1), (1, 65, 96, 64, 2, 1), (4, 250, 768, 6144, 2, 1), (6, 1000, 768, 1920, 2, 1),
    (1, 1000, 384, 768, 2, 1), (2, 130, 192, 288, 2, 1),
    (400, 100, 96, 64, 2, 1),
    # k = 1: 64x64, 128x64, 128x128, 256x192, 256x256, 32-channel steps
    (1, 1, 64, 64, 1, 1), (1, 129, 256, 2048, 1, 1), (1, 701, 512, 2048, 1, 1), (5, 411, 512, 2048, 1, 1), (10, 325, 512, 3072, 1, 1),
    (1, 701, 256, 12288, 1, 1), (10, 1300, 512, 1024, 1, 1), (2, 515, 96, 96, 1, 1), (24, 5000, 384, 384, 1, 1), (1, 65, 32, 64, 1, 1),
    (1, 2043, 512, 4096, 1, 1), (3, 683, 256, 2048, 1, 1),
]


@pytest.mark.parametrize("lanes,length,cin,cout,k,dil", ROWS)
def test_tiles_against_float64(dev, lanes, length, cin, cout, k, dil):
    x, w, b = _inputs(lanes, length, cin, cout, k, dev)
    y = nlc.conv1d(x, w, b, k=k, dilation=dil)
    _check(y, _f64(x, w, b, k, dil))
    alone = nlc.conv1d(x[lanes - 1:].contiguous(), w, b, k=k, dilation=dil)
    assert torch.equal(alone[0], y[lanes - 1])


# lanes, length, channels, k, dilation
EPILOGUE = [
    (1, 200, 192, 7, 3), (7, 300, 192, 7, 9), (24, 129, 192, 7, 1), (24, 500, 192, 7, 9), (16, 1201, 192, 7, 3), (40, 801, 192, 7, 9),
    (4, 129, 192, 1, 1), (16, 1201, 192, 1, 1), (24, 300, 512, 1, 1), (16, 1201, 512, 1, 1), (24, 2001, 256, 1, 1),
]


@pytest.mark.parametrize("lanes,length,c,k,dil", EPILOGUE)
def test_small_tiles_epilogue_forms(dev, lanes, length, c, k, dil):
    """Residual, both outputs and the SnakeBetas on the tiles that few positions take, and on the larger
    ones, against the plain forms composed."""
    x, w, b = _inputs(lanes, length, c, c, k, dev)
    act = (torch.rand(c, device=dev) + 0.5, torch.rand(c, device=dev) + 0.5)
    pre, y = nlc.conv1d(x, w, b, k=k, dilation=dil, residual=x, snake_out=act, want_pre=True)
    _check(pre, _f64(x, w, b, k, dil) + x.double())
    p = pre.double()
    _check(y, p + act[1].double() * torch.sin(act[0].double() * p) ** 2)


@pytest.mark.parametrize("lanes,length,cin,cout,k,dil", [
    (24, 25, 1024, 1536, 7, 1), (48, 1000, 384, 384, 7, 1), (48, 800, 256, 512, 7, 1), (24, 25, 1536, 6144, 2, 1),
    (24, 1000, 384, 768, 2, 1), (48, 200, 768, 768, 1, 1), (24, 1000, 384, 384, 1, 1),
])
def test_activation_forms_alone_and_in_a_batch(dev, lanes, length, cin, cout, k, dil):
    """SnakeBeta, the residual and the activations round an output the same way on every tile of a class."""
    x, w, b = _inputs(lanes, length, cin, cout, k, dev)
    g = torch.Generator(device=dev)
    g.manual_seed(cout)
    act = (torch.rand(cout, generator=g, device=dev) + 0.5, torch.rand(cout, generator=g, device=dev) + 0.5)
    res = torch.randn((lanes, length, cout), generator=g, device=dev).half()
    scale = torch.rand(cout, generator=g, device=dev)
    for form in (dict(snake_out=act), dict(residual=res, snake_out=act, want_pre=True), dict(act="gelu"),
                 dict(residual=res, scale=scale)):
        one = {key: v[3:4].contiguous() if key == "residual" else v for key, v in form.items()}
        y, alone = nlc.conv1d(x, w, b, k=k, dilation=dil, **form), nlc.conv1d(x[3:4].contiguous(), w, b, k=k, dilation=dil, **one)
        for a, c in zip(y, alone) if isinstance(y, tuple) else ((y, alone),):
            assert torch.equal(a[3], c[0]), (list(form), int((a[3] != c[0]).sum()))
