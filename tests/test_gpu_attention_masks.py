"""The one-pass attention kernel (kaun/lib/attention.ml:67-110 as one launch) over the forms its mask takes and at
the edges of its key tiles. The mask is read four bytes at a time where its keys are neighbours in memory and byte
by byte where they are not, and generated where it is causal: one mask in all of these forms gives the same bits.
Against float64: a probability is rounded to the dtype once and the output once, each to within 2^-8 (bfloat16;
float16 2^-11) of itself, so that a result is within twice that of the sum of probability times |v|; a tenth
more for the float32 sums, and 2^-25 |v| a key for float16 probabilities below its normal range."""

import numpy as np
import pytest

from helpers import decode, encode, logical, pair
from raven_amd import dtype as dt

pytestmark = pytest.mark.gpu
SIZES = [(1, 1, 64), (64, 64, 64), (65, 128, 64), (31, 129, 64), (130, 130, 64), (95, 95, 32), (130, 193, 32), (97, 300, 128)]


def reference(q, k, v, keep):
    s = np.where(keep, q @ k.swapaxes(-1, -2) * 0.125, -np.inf)
    p = np.exp(s - s.max(-1, keepdims=True))
    p = p / p.sum(-1, keepdims=True)
    return p @ v, p @ np.abs(v)


@pytest.mark.parametrize("d", [dt.bfloat16, dt.float16], ids=lambda d: d.name)
@pytest.mark.parametrize("sq,sk,hd", SIZES, ids=lambda n: str(n))
@pytest.mark.parametrize("causal", [False, True], ids=["random", "causal"])
def test_one_mask_in_all_its_forms(hip, oracle, monkeypatch, d, sq, sk, hd, causal):
    monkeypatch.delenv("NXH_ATTENTION", raising=False)
    rng = np.random.default_rng(sq * 1000 + sk + hd)
    outer = (2, 3)
    host = [encode(rng.standard_normal(outer + (n, hd)) * 1.5, d, oracle) for n in (sq, sk, sk)]
    q, k, v = (pair(x, d, hip, oracle)[0] for x in host)
    keep = np.tril(np.ones((sq, sk), bool)) if causal else rng.random((sq, sk)) < 0.6
    keep[:, 0] = True
    fill = dict(masked_value=float("-inf"))

    def run(stored, build):
        m = build(hip.reshape(hip.from_host(np.ascontiguousarray(stored), dt.bool_), stored.shape))
        m = hip.expand(hip.reshape(m, (1, 1, sq, sk)), outer + (sq, sk))
        return logical(hip.attention(q, k, v, 0.125, mask=m, **fill))

    got = run(keep, lambda t: t)
    wide = np.zeros((sq, sk + 6), bool)
    wide[:, 3:3 + sk] = keep
    forms = {"rows at odd bytes": run(wide, lambda t: hip.shrink(t, ((0, sq), (3, 3 + sk)))),
             "keys apart": run(keep.T, lambda t: hip.permute(t, (1, 0))),
             "keys backwards": run(keep[:, ::-1], lambda t: hip.flip(t, (False, True)))}
    if causal and sq == sk:
        forms["generated"] = logical(hip.attention(q, k, v, 0.125, causal=True, **fill))
    for name, other in forms.items():
        assert got.tobytes() == other.tobytes(), name
    want, size = reference(*(decode(x, d, oracle) for x in host), keep)
    unit = 2.0 ** (-8 if d is dt.bfloat16 else -11)
    assert np.all(np.abs(decode(got, d, oracle) - want) <= 1.1 * 2 * unit * size + 2.0 ** -25 * 6 * sk)


@pytest.mark.parametrize("heads,sq,hd", [(24, 64, 128), (27, 130, 128), (50, 70, 64)], ids=str)
def test_tiles_handed_out_in_groups(hip, oracle, monkeypatch, heads, sq, hd):
    """Keys and values of more heads than three times what the L2s hold: the same bits as a few heads at a time."""
    monkeypatch.delenv("NXH_ATTENTION", raising=False)
    rng = np.random.default_rng(heads)
    q, k, v = (pair(encode(rng.standard_normal((heads, n, hd)), dt.bfloat16, oracle), dt.bfloat16, hip, oracle)[0]
               for n in (sq, 8192, 8192))
    got = logical(hip.attention(q, k, v, 0.125))
    for first in range(0, heads, 9):
        last = min(first + 9, heads)
        part = [hip.shrink(t, ((first, last), (0, t.shape[1]), (0, hd))) for t in (q, k, v)]
        assert got[first:last].tobytes() == logical(hip.attention(*part, 0.125)).tobytes(), first


@pytest.mark.parametrize("hd", [0, 1, 8, 16, 96, 256])
@pytest.mark.parametrize("form", ["", "twopass"])
def test_other_head_dimensions_are_refused(hip, monkeypatch, hd, form):
    """None too, which no quotient on the way may meet."""
    monkeypatch.setenv("NXH_ATTENTION", form)
    t = hip.full(dt.bfloat16, (1, 1, 1, hd), 1.0)
    with pytest.raises(RuntimeError, match="head dimension must be 32, 64 or 128"):
        hip.attention(t, t, t, 0.125)
