"""GPU parity of the FK dip filter (sh_fkdip, hipFFT in float64) against
the numpy oracle.  The FFTs differ in summation order from numpy's, so the
bar is float64 rounding: max |gpu - oracle| <= 1e-11 * max |oracle| with the
oracle in float64.  numpy 2 transforms float32 input in float32 (the
reference's forward FFTs then round to single precision), so for float32
input the bar against the oracle run on that input is 1e-6."""
import numpy as np
import pytest

from oracle import fk_oracle as F

pytestmark = pytest.mark.gpu
TOL = 1e-11
TOL_F32_INPUT = 1e-6


@pytest.fixture(scope="module")
def fk():
    import torch
    from pyseistr_amd import _lib, fk
    assert torch.cuda.is_available()
    assert not _lib.missing_symbols()
    return fk


def _rel(a, b):
    return np.abs(a - b).max() / np.abs(b).max()


@pytest.mark.parametrize("shape,w", [((1000, 300), 0.02), ((256, 128), 0.005), ((513, 65), 0.3),
                                     ((100, 1), 5.0), ((1, 50), 0.05), ((2, 3), 0.4), ((64, 64), 0.45)])
@pytest.mark.parametrize("dt", [np.float64, np.float32])
def test_fkdip_matches_oracle(fk, shape, w, dt):
    d = np.random.default_rng(shape[0] + 7 * shape[1]).standard_normal(shape).astype(dt)
    got = fk.fkdip(d, w)
    ref = F.fkdip(d.astype(np.float64), w)
    assert got.shape == ref.shape and got.dtype == np.float64
    assert np.abs(ref).max() > 0  # the cone keeps something
    print(shape, w, dt.__name__, "rel err", _rel(got, ref))
    assert _rel(got, ref) <= TOL
    if dt == np.float32:
        assert _rel(got, F.fkdip(d, w)) <= TOL_F32_INPUT


@pytest.mark.parametrize("shape", [(1000, 300), (513, 65), (64, 64)])
def test_one_dimensional_transforms_agree(fk, monkeypatch, shape):
    """SH_FK_1D=1 runs the time and space transforms as separate batched 1-D
    transforms (the path taken anyway when an axis has one sample) instead
    of one 2-D real transform; both meet the float64 bar."""
    d = np.random.default_rng(shape[1]).standard_normal(shape)
    ref = F.fkdip(d, 0.03)
    two = fk.fkdip(d, 0.03)
    monkeypatch.setenv("SH_FK_1D", "1")
    one = fk.fkdip(d, 0.03)
    monkeypatch.delenv("SH_FK_1D")
    assert _rel(one, ref) <= TOL and _rel(two, ref) <= TOL


@pytest.mark.parametrize("n1", [65, 128, 129, 400, 513, 2048, 2500, 4097, 9001, 16384])
@pytest.mark.parametrize("n2", [33, 64, 90, 257, 600, 2000])
def test_transform_lengths(fk, n1, n2):
    """Every length of the three-kernel path along time (128 to 16384, the
    odd and even ends of a trace) against each along space (64 to 2048, with
    and without padding; 4096 is in the section above): the rounding of its
    log2(n) additions a value stays far below the bar."""
    if n1 * n2 > 10_000_000:
        n2 = n2 // 16 + 33
    d = np.random.default_rng(n1 + n2).standard_normal((n1, n2))
    for w in (0.03, 0.4):
        got, ref = fk.fkdip(d, w), F.fkdip(d, w)
        assert _rel(got, ref) <= TOL


def _long_double(d, w):
    """oracle.fk_oracle.fkdip in long double."""
    n1, n2 = d.shape
    nf, nk = F.nextpow2(n1), F.nextpow2(n2)
    h = nf // 2 + 1
    D = np.fft.fftshift(np.fft.fft(np.fft.fft(d.astype(np.longdouble), nf, 0)[:h], nk, 1), 1)
    assert D.dtype == np.clongdouble
    D = np.fft.ifft(np.fft.ifftshift(D * F.cone(h, nk, w), 1), nk, 1)
    full = np.concatenate([D, np.conj(np.flipud(D[1:-1]))])
    return np.real(np.fft.ifft(full, nf, 0))[:n1, :n2]


@pytest.mark.parametrize("shape", [(129, 33), (1000, 300), (2500, 600), (6000, 200)])
def test_error_against_long_double(fk, monkeypatch, shape):
    """Root mean square error of the three kernels and of the library's
    transforms against long double.  The four transforms have 2 log2(nf nk)
    levels of additions, each rounding a value by at most half an ulp (2^-53)
    in the mean square: the root of their number bounds the sum."""
    d = np.random.default_rng(shape[0]).standard_normal(shape)
    ref = _long_double(d, 0.05)
    scale = np.sqrt(np.mean(ref.astype(np.float64) ** 2))

    def err(x):
        return float(np.sqrt(np.mean((x - ref) ** 2))) / scale

    own = err(fk.fkdip(d, 0.05))
    monkeypatch.setenv("SH_FK_1D", "1")
    print(shape, "rms error: kernels", own, "library", err(fk.fkdip(d, 0.05)), flush=True)
    assert own <= np.sqrt(2 * np.log2(F.nextpow2(shape[0]) * F.nextpow2(shape[1]))) * 2.0**-53


def test_lengths_left_to_the_library(fk):
    """One step beyond the three kernels' range on each side."""
    for shape in [(64, 100), (16385, 40), (200, 32), (130, 4097)]:
        d = np.random.default_rng(shape[0]).standard_normal(shape)
        assert _rel(fk.fkdip(d, 0.1), F.fkdip(d, 0.1)) <= TOL


def test_repeated_and_resized_calls(fk):
    # the plans are cached per size: alternate sizes and repeat
    rng = np.random.default_rng(3)
    for shape in [(300, 200), (64, 48), (300, 200), (64, 48)]:
        d = rng.standard_normal(shape)
        ref = F.fkdip(d, 0.03)
        assert np.abs(fk.fkdip(d, 0.03) - ref).max() <= TOL * np.abs(ref).max()


def test_das_size_properties(fk):
    """A DAS-sized section, 8192 samples x 4096 channels (no padding): an
    open cone returns the input, and the filter is linear."""
    import torch
    n1, n2 = 8192, 4096
    g = torch.Generator(device="cuda").manual_seed(4)
    x = torch.randn(n1 * n2, generator=g, device="cuda", dtype=torch.float64)
    y = torch.randn(n1 * n2, generator=g, device="cuda", dtype=torch.float64)
    same = fk.fkdip_device(x, (n1, n2), 1e12)
    assert float((same - x).abs().max()) <= 1e-12 * float(x.abs().max())
    fx = fk.fkdip_device(x, (n1, n2), 0.02)
    fy = fk.fkdip_device(y, (n1, n2), 0.02)
    fxy = fk.fkdip_device(2.0 * x - 0.5 * y, (n1, n2), 0.02)
    assert float((fxy - (2.0 * fx - 0.5 * fy)).abs().max()) <= 1e-12 * float(fxy.abs().max())
    # the cone removes a real share of the noise's energy
    assert float(fx.norm()) < 0.9 * float(x.norm())


def test_errors(fk):
    with pytest.raises(ValueError):
        fk.fkdip(np.zeros((8, 8)), 0.0)
    with pytest.raises(ValueError):
        fk.fkdip(np.zeros(8), 0.1)
