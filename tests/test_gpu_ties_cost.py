"""Rows with many equal logits cost a small multiple of rows without (coarse logits, masks with a finite value): the whole
device works on them, not one workgroup. Times of the same call on the same shapes, side by side; the bounds leave a
factor of two over what was measured."""
import ctypes
import os
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))

from ferro_amd import workloads as W  # noqa: E402
from ferro_amd._lib import lib  # noqa: E402
import ferro_amd as F  # noqa: E402


@pytest.fixture(scope="module", autouse=True)
def gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    yield
    torch.cuda.synchronize()


def P(t):
    return ctypes.c_void_p(t.data_ptr())


def time_us(x, k, top_p=0.95, host=True, **kw):
    """Median over five blocks of eight calls; host: with a host copy of the parameters."""
    B, V = x.shape
    p = W.make_params(B, temperature=0.8, top_k=k, top_p=top_p, repetition_penalty=1.0)
    for f, v in kw.items():
        p[f] = v
    d = torch.from_numpy(x).cuda()
    dp = torch.from_numpy(p.view(np.uint8).copy()).cuda()
    u = torch.from_numpy(np.random.default_rng(1).random(B)).cuda()
    hist = torch.arange(B * 64, dtype=torch.int32, device="cuda")
    off = torch.arange(B + 1, dtype=torch.int64, device="cuda") * 64
    tok = torch.empty(B, dtype=torch.int32, device="cuda")
    ctx, st = F.sampler.Context(), torch.cuda.current_stream()

    def call():
        hp = [p.ctypes.data_as(ctypes.c_void_p)] if host else []
        rc = (lib().fs_sample_batch_hp if host else lib().fs_sample_batch)(
            ctx.h, P(d), V, B, V, P(hist), P(off), P(dp), *hp, P(u), P(tok), 0, None, None, None,
            ctypes.c_void_p(st.cuda_stream))
        assert rc == 0
    call()
    torch.cuda.synchronize()
    t = []
    for _ in range(5):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        for _ in range(8):
            call()
        b.record()
        b.synchronize()
        t.append(a.elapsed_time(b) * 1e3 / 8)
    assert F.device_error(ctx) == 0
    return sorted(t)[2]


def test_lists_of_equal_logits():
    rng = np.random.default_rng(2)
    x = (rng.standard_normal((32, 262144)) * 2).astype(np.float32)
    plain, coarse = time_us(x, 200), time_us(np.round(x), 200)
    assert coarse < 3.5 * plain, (plain, coarse)


@pytest.mark.parametrize("k", [65, 1000, 2048])
def test_bounds_of_equal_logits(k):
    """Masks that allow fewer than k tokens, coarse logits, rows of one value: 1.6 to 2.8 times a row without ties here
    (100 to 120 times when one workgroup selected such a row alone)."""
    rng = np.random.default_rng(2)
    x = (rng.standard_normal((32, 262144)) * 2).astype(np.float32)
    plain = time_us(x, k)
    few = rng.random(x.shape) < 1e-4
    for name, y in (("mask", np.where(few, x, -np.inf)), ("finite mask", np.where(few, x, -1e9)), ("one value", x * 0),
                    ("whole", np.round(x)), ("two", np.where(x > 1, 1.0, 0.0))):
        t = time_us(y.astype(np.float32), k)
        assert t < 6 * plain, (name, t, plain)


@pytest.mark.parametrize("V", [65536, 262144])
def test_every_token_of_few_values(V):
    """top_k = 0 on coarse logits and rows of one value: 0.18 to 0.63 times the call without host parameters, whose kernel
    took them before."""
    rng = np.random.default_rng(2)
    x = (rng.standard_normal((8, V)) * 2).astype(np.float32)
    for name, y in (("one value", x * 0), ("two", (x > 1).astype(np.float32)), ("whole", np.round(x))):
        t, fused = time_us(y, 0), time_us(y, 0, host=False)
        assert t < 1.2 * fused, (name, t, fused)
