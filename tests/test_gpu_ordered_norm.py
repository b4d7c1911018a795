"""The norms' sum of squares (ordered_sum.hpp): one wave adds the terms as the
serial loop of cpu::rms_from rounds them, whatever the terms are, so the norms
keep the oracle's bits."""
import numpy as np
import pytest

from decisive_amd import rocm
from tests import pplx_model
from tests.gpu_util import bits_equal, dev, empty, host
from tests.test_gpu_pplx import SMALL

pytestmark = pytest.mark.gpu
EPS = 1e-6


def _rows(kind, rows, d):
    rng = np.random.default_rng(d + rows)
    v = rng.standard_normal((rows, d))
    at = np.arange(d)
    if kind == "halves":  # squares of few bits: terms that are exact halves of the sum's ulp
        v = np.ldexp(rng.integers(0, 64, (rows, d)) * 2.0 + 1, -rng.integers(0, 14, (rows, d)))
    elif kind == "powers":
        v = np.ldexp(1.0, rng.integers(-12, 12, (rows, d)))
    elif kind == "growing":  # a binade every few terms
        v = np.ldexp(v, at // 32 % 120 - 60)
    elif kind == "falling":
        v = np.ldexp(v, 30 - at // 16 % 90)
    elif kind == "sparse":  # zeros, and jumps over many binades
        v = np.where(rng.random((rows, d)) < 0.01, v * 1e9, np.where(rng.random((rows, d)) < 0.5, 0.0, v))
    elif kind == "tiny":  # squares at and below the smallest normal float
        v = v * 2e-20
    elif kind == "overflow":  # the sum reaches infinity, every normed value 0
        v = v * 1e19
    return v.astype(np.float32)


@pytest.mark.parametrize("d", [64, 448, 512, 576, 1088, 2560, 8192])
@pytest.mark.parametrize("kind", ["normal", "halves", "powers", "growing", "falling", "sparse", "tiny", "overflow"])
def test_readout_norm_adds_in_row_order(ctx, oracle, kind, d):
    torch = pytest.importorskip("torch")
    rows, n = 9, 5
    rng = np.random.default_rng(1)
    packed = oracle.pack_g64(oracle.f32_to_bf16((rng.standard_normal((n, d)) * 0.02).astype(np.float32)), n, d, 8)
    w = ctx.upload(packed, rocm.Q8_G64_F32, n, d)
    hidden, norm = _rows(kind, rows, d), (rng.standard_normal(d) * 0.1).astype(np.float32)
    logits = empty((rows, n), torch.float32)
    ctx.readout(w, dev(norm), dev(hidden), rows, EPS, logits)
    got = host(ctx, logits)
    x = oracle.rmsnorm(hidden, norm, EPS, zero_centered=True)
    for r in range(rows):
        # the logits carry every group's scale, so an ulp of the row scale shows
        assert bits_equal(got[r], oracle.project(packed, 8, d, x[r], n)), r


@pytest.mark.parametrize("d,at", [(64, 0), (576, 300), (2560, 2559), (8192, 4100)])
@pytest.mark.parametrize("bad", [np.nan, -np.nan, np.inf, -np.inf])
def test_readout_norm_reports_nonfinite_rows(ctx, oracle, bad, d, at):
    """A NaN or infinite term takes the sum out of the last binade: the row's
    norm is not finite, as the serial loop's is not, and the next call is
    unaffected."""
    torch = pytest.importorskip("torch")
    packed = oracle.pack_g64(oracle.f32_to_bf16(np.full((3, d), 0.01, np.float32)), 3, d, 8)
    w = ctx.upload(packed, rocm.Q8_G64_F32, 3, d)
    norm, logits = np.zeros(d, np.float32), empty((4, 3), torch.float32)
    clean = _rows("normal", 4, d)
    rows = clean.copy()
    rows[2, at] = bad
    with pytest.raises(rocm.DzError, match="nonfinite readout activation"):
        ctx.readout(w, dev(norm), dev(rows), 4, EPS, logits)
    ctx.readout(w, dev(norm), dev(clean), 4, EPS, logits)
    want = oracle.project(packed, 8, d, oracle.rmsnorm(clean, norm, EPS, zero_centered=True)[2], 3)
    assert bits_equal(host(ctx, logits)[2], want)


@pytest.mark.parametrize("hidden", [192, 1024, 1088, 3072, 3136, 4096, 4160])
def test_quantizing_norm_of_every_row_width(ctx, oracle, hidden):
    """The codes' block holds 1024, 3072, 4096 or 8192 columns; each gives the
    bits of the norm and the quantizer run apart."""
    pytest.importorskip("torch")
    n = 19
    model = pplx_model.random_model(oracle, dict(SMALL, layers=1, hidden=hidden, ff=64), seed=hidden)
    p = pplx_model.load(ctx, rocm, model)
    out = {}
    for v in ("fused", "separate"):
        h = dev(_rows("falling", n, hidden))
        ctx.select_variant("norm", v)
        try:
            p.layer(0, h, n)
        finally:
            ctx.select_variant("norm", "fused")
        out[v] = host(ctx, h)
    p.close()
    assert np.isfinite(out["fused"]).all()
    assert np.array_equal(out["fused"].view(np.uint32), out["separate"].view(np.uint32))
